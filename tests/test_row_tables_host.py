"""The jump tables of the row updates (local.hip) assemble only if every case has the size by which
the jump multiplies: the tables alone are compiled with their own sizes and with others."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG_DIR

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
KERNEL = """
__global__ void use(double* p, int t) {
  d16 x, y;
  double g;
  for (int c = 0; c < 16; c++) { x[c] = p[c]; y[c] = p[16 + c]; }
  t = __builtin_amdgcn_readfirstlane(t) & 15;
  row_flip(x, p[32], p[33], p[34], t, g);
  row_add(y, x, g, t);
  row_update(x, g, t);
  for (int c = 0; c < 16; c++) { p[c] = x[c]; p[16 + c] = y[c]; }
}
"""


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
@pytest.mark.parametrize("old,new", [(None, None), ("DQMC_ROW_JUMP(156)", "DQMC_ROW_JUMP(152)"),
                                     ("DQMC_ROW_JUMP(132) DQMC_CASES16(DQMC_ADD)",
                                      "DQMC_ROW_JUMP(136) DQMC_CASES16(DQMC_ADD)"),
                                     ("DQMC_ROW_JUMP(132) DQMC_CASES16(DQMC_UPD)",
                                      "DQMC_ROW_JUMP(128) DQMC_CASES16(DQMC_UPD)")])
def test_case_sizes_are_checked(tmp_path, old, new):
    src = open(os.path.join(PKG_DIR, "csrc", "local.hip")).read()
    part = src[src.index("typedef double d16 "):src.index("// Both 16-lane rows of a pair")]
    if old:
        assert part.count(old) == 1
        part = part.replace(old, new)
    f = tmp_path / "tables.hip"
    f.write_text("#include <hip/hip_runtime.h>\n" + part + KERNEL)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-device-only", "-O3", "-std=c++17", "-Xclang",
                        "-target-feature", "-Xclang", "-packed-fp32-ops", "-c", str(f), "-o",
                        str(tmp_path / "tables.o")], capture_output=True, text=True, timeout=120)
    assert (r.returncode == 0) == (old is None), r.stderr[-2000:]
    if old:
        assert "size of a row case" in r.stderr
