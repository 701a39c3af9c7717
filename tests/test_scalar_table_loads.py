"""The cell kernels read the FE tables, which are the same for every lane, with scalar
loads: a load of each lane instead costs the atomic assembly a quarter to a half of
its time. A store to global memory ahead of the cell work is enough to turn them
(the compiler can then not tell that the tables stay the same), and no output shows
it. So the assembly that the build's compiler makes is looked at: the loops over the
flux nodes and the quadrature points (the inner loops with the FP64 arithmetic) hold
scalar loads and no vector loads."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


@pytest.mark.parametrize("args", ["2, 3, 10, 15, 12, true, PH_BURGERS2D, SC_N", "2, 4, 9, 16, 8, false, PH_BURGERS2D, SC_LDA",
                                  "2, 3, 6, 10, 6, true, PH_EULER2D, SC_LDA"])
def test_cell_kernel_loops(args, tmp_path):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text('#include "rd_launch.hpp"\nnamespace pdrd {\n'
                   f"template __global__ void rd_cell_kernel<{args}>(CellArgs);\n}}\n")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-munsafe-fp-atomics", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "--cuda-device-only", "-S",
                    f"-I{ROOT}/pdekit_amd/csrc/hip", "-o", str(out), str(src)], check=True, stderr=subprocess.DEVNULL)
    blocks = re.split(r"\n(?=\.LBB)", out.read_text())
    loops = [b for b in blocks if "Inner Loop" in b.split("\n")[0] and b.count("v_fma_f64") >= 10]
    assert loops
    for b in loops:
        assert "s_load" in b and "global_load" not in b
