"""The source-owned message adjoint reads its edges' rows through descriptors and offsets in scalar registers: the
compiler makes no loop over the lanes' values around a buffer access."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ictc-o3-hp-k100_amd", "csrc")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.skipif(not os.path.exists(os.path.join(CSRC, "generated", "ictc_tables.h")), reason="not built here")
def test_no_lane_loops_around_buffer_accesses(tmp_path):
    unit = tmp_path / "unit.hip"
    lines = [f'#include "{CSRC}/ictc_kernels.h"', "namespace ictc {"]
    for triple in ("1, 1, 1", "1, 2, 2", "2, 2, 2"):
        for grad in ("kNoGrad", "kStoreGrad", "kAddGrad", "kTangent"):
            lines.append(f"template __global__ void msg_bwd_src_kernel<Tp<{triple}>, {grad}, false>(Operands, const int64_t*, "
                         "Csr, const float*, float*, float*, float*, float*, const float*, float*, float*, int);")
    unit.write_text("\n".join(lines + ["}"]) + "\n")
    out = tmp_path / "unit.out"
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-munsafe-fp-atomics", "--cuda-device-only", "-S", str(unit), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    text = out.read_text()
    assert text.count("buffer_load") > 100 and text.count("buffer_store") > 10
    loops = re.findall(r"v_readfirstlane_b32[^;]*?s_and_saveexec_b64 [^;]*?buffer_(?:load|store)[^;]*?s_cbranch_execnz", text)
    assert not loops, loops[0]
