"""Choose the occupancy (minimum waves per SIMD) of every TP / message kernel instance.

The generated CG code is straight-line; how many VGPRs the scheduler wants for
it depends on the degree triple in ways a size formula does not capture.  This
script compiles the kernel translation units once per candidate occupancy
(4, 3, 2, 1 waves per SIMD, i.e. 128, 168, 256, 512 registers per lane),
reads the compiler's resource-usage remarks, and picks for each (kernel and
its template flags, degree triple) the highest occupancy at which it compiles with at most
SPILL_BUDGET spilled VGPRs (a few spills outside the inner loop cost far less
than halving the waves that hide memory latency: measured on the cfg5
msg_bwd_edge<2,3,3>, 8 spills at 2 waves per SIMD ran 4.39 -> 2.90 ms).  The result is written to ``ictc_occupancy.h`` (committed) as
``Occupancy<kind, LI, LE, LO>`` specializations.  Run it after changing
``ictc_kernels.h`` or the generated tables; the build does not run it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
UNITS = ["tp_edge.hip", "msg_fwd.hip", "msg_bwd.hip", "tp_second.hip", "msg_second_rcv.hip", "msg_second_src.hip"]
# kernel and template flags -> table entry (the gate-tangent forms of msg_bwd_edge_kernel go by its plain form's entry,
# and the source-owned message adjoint fixes its own count from its register sizes)
KINDS = {("edge_fwd_kernel", "0"): "kEdgeFwd", ("edge_fwd_kernel", "1"): "kEdgeFwdMul",
         ("edge_bwd_kernel", "0"): "kEdgeBwd", ("edge_bwd_kernel", "1"): "kEdgeBwdMul",
         ("msg_fwd_kernel", ""): "kMsgFwd", ("msg_bwd_edge_kernel", "00"): "kMsgBwdEdge",
         ("msg_bwd_x_kernel", ""): "kMsgBwdX", ("edge_second_kernel", ""): "kEdgeSecond",
         ("msg_fwd2_kernel", "0"): "kMsgFwd2", ("msg_fwd2_kernel", "1"): "kMsgFwd2All",
         ("msg_bwd_edge2_kernel", ""): "kMsgBwdEdge2", ("msg_bwd_x2_kernel", "0"): "kMsgBwdX2",
         ("msg_bwd_x2_kernel", "1"): "kMsgBwdX2All"}
LEVELS = (4, 3, 2, 1)
SPILL_BUDGET = 8
# Measured exceptions (us over 357 k edges, 64 channels unless said otherwise): the source-owned second-order pass of
# (3,3,3) with both tangents 1,356 at 2 waves with 15 spilled VGPRs, 1,770 at 1 without; the receiver-owned one of
# (2,2,2) with all tangents 908 at 3 waves, 934 at 4 with 5 spilled (128 channels); the edge adjoint of (2,3,3) on
# [channel, magnetic] rows 378 at 3 waves, 386 at 4 with 8 spilled (30,011 edges of 128 channels).
MEASURED = {("kMsgBwdX2All", 3, 3, 3): 2, ("kMsgFwd2All", 2, 2, 2): 3, ("kEdgeBwdMul", 2, 3, 3): 3}
NAME = re.compile(r"Function Name: _ZN4ictc\d+(\w+?)INS_2TpILi(\d)ELi(\d)ELi(\d)EEE?((?:Lb[01]E)*)")


def parse_usage(text: str):
    """{(table entry, li, le, lo): [spilled VGPRs, scratch bytes]} of the compiler's remarks."""
    out, key = {}, None
    for line in text.splitlines():
        m = NAME.search(line)
        if m:
            kind = KINDS.get((m.group(1), re.sub("[^01]", "", m.group(5))))
            key = (kind, int(m.group(2)), int(m.group(3)), int(m.group(4))) if kind else None
            if key in out:
                raise RuntimeError(f"two instances of {key}")
            if key is not None:
                out[key] = [0, 0]
        elif key is not None and "VGPRs Spill:" in line:
            out[key][0] = int(line.split(":")[-1].split()[0])
        elif key is not None and "ScratchSize [bytes/lane]:" in line:
            out[key][1] = int(line.split(":")[-1].split()[0])
    return out


def _usage(unit: str, waves: int):
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", f"-DICTC_OCCUPANCY_PROBE={waves}", "-c", os.path.join(HERE, unit), "-o", os.devnull,
           "-Rpass-analysis=kernel-resource-usage"]
    text = subprocess.run(cmd, capture_output=True, text=True, cwd=HERE).stderr
    out = parse_usage(text)
    if not out:
        raise RuntimeError(f"no resource remarks for {unit} at {waves} waves:\n{text[-2000:]}")
    return out


def main(path=None):
    path = path or os.path.join(HERE, "ictc_occupancy.h")
    jobs = [(u, w) for u in UNITS for w in LEVELS]
    with cf.ThreadPoolExecutor(min(len(jobs), os.cpu_count() or 4)) as ex:
        results = dict(zip(jobs, ex.map(lambda j: _usage(*j), jobs)))
    choice = {}
    for (unit, w), usage in results.items():
        for key, (spill, scratch) in usage.items():
            # scratch without spills would be a stack array: never acceptable
            if spill <= SPILL_BUDGET and (scratch == 0 or spill > 0) and w > choice.get(key, 0):
                choice[key] = w
    choice.update(MEASURED)
    keys = {k for usage in results.values() for k in usage}
    lines = ["// Generated by tune_occupancy.py: minimum waves per SIMD per (kernel instance, degree triple),",
             f"// the highest of 4, 3, 2, 1 with at most {SPILL_BUDGET} spilled VGPRs, or a measured count.  Do not edit.", "#pragma once", ""]
    for key in sorted(keys):
        kind, li, le, lo = key
        w = choice.get(key, 1)
        if w == 4:
            continue   # the default
        lines.append(f"template <> struct Occupancy<{kind}, {li}, {le}, {lo}> {{ static constexpr int value = "
                     f"{w}; }};")
    with open(path, "w") as f:
        f.write("\n".join(lines) + "\n")
    print(f"{path}: {len(lines) - 4} non-default entries")


if __name__ == "__main__":
    main(*sys.argv[1:])
