"""The occupancy table script (csrc/tune_occupancy.py) and its table: one entry per kernel instance and degree triple."""
import importlib.util
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ictc-o3-hp-k100_amd", "csrc")


def _script():
    spec = importlib.util.spec_from_file_location("tune_occupancy", os.path.join(CSRC, "tune_occupancy.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def _remarks(name, spill, scratch):
    return (f"a.h:1:0: remark: Function Name: {name} [-Rpass]\na.h:1:0: remark:     VGPRs: 128 [-Rpass]\n"
            f"a.h:1:0: remark:     ScratchSize [bytes/lane]: {scratch} [-Rpass]\n"
            f"a.h:1:0: remark:     VGPRs Spill: {spill} [-Rpass]\n")


def test_instances_of_one_triple_are_kept_apart():
    tune = _script()
    args = "EvNS_8OperandsENS_8TangentsEPKlNS_3CsrEPKfPfi"
    text = (_remarks("_ZN4ictc17msg_bwd_x2_kernelINS_2TpILi3ELi3ELi3EEELb1EE" + args, 15, 64)
            + _remarks("_ZN4ictc17msg_bwd_x2_kernelINS_2TpILi3ELi3ELi3EEELb0EE" + args, 0, 0)
            + _remarks("_ZN4ictc14msg_fwd_kernelINS_2TpILi2ELi2ELi2EEEE" + args, 3, 16)
            + _remarks("_ZN4ictc19msg_bwd_edge_kernelINS_2TpILi2ELi2ELi2EEELb0ELb0EE" + args, 1, 8)
            + _remarks("_ZN4ictc18msg_bwd_src_kernelINS_2TpILi3ELi3ELi3EEELNS_8GateGradE3ELb1EE" + args, 34, 84))
    usage = tune.parse_usage(text)
    assert usage == {("kMsgBwdX2All", 3, 3, 3): [15, 64], ("kMsgBwdX2", 3, 3, 3): [0, 0], ("kMsgFwd", 2, 2, 2): [3, 16],
                     ("kMsgBwdEdge", 2, 2, 2): [1, 8]}
    with pytest.raises(RuntimeError, match="two instances"):
        tune.parse_usage(text + text)


def test_table_names_its_kinds():
    tune = _script()
    table = open(os.path.join(CSRC, "ictc_occupancy.h")).read()
    kinds = set(re.search(r"enum KernelKind \{([^}]*)\}", open(os.path.join(CSRC, "ictc_kernels.h")).read()).group(1)
                .replace(",", " ").split())
    assert kinds == set(tune.KINDS.values())
    entries = re.findall(r"Occupancy<(\w+), (\d), (\d), (\d)> \{ static constexpr int value = (\d)", table)
    assert len(entries) == len({e[:4] for e in entries}) and {e[0] for e in entries} <= kinds
    assert all(dict(((k, int(a), int(b), int(c)), int(v)) for k, a, b, c, v in entries)[key] == waves
               for key, waves in tune.MEASURED.items())
