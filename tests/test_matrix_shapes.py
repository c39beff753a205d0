"""Matrix instructions of one kernel have one shape: an instruction that adds to
what one of another shape (another number of passes) has just written was seen
to give wrong rows, unless other work happened to lie between."""
import os
import re
import shutil
import subprocess

import pytest

from binarytpm_amd import build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("name", ["conduct.hip", "aux.hip"])
def test_one_shape_per_kernel(name, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    out = tmp_path / "k.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC", "-Wall")]
    r = subprocess.run([HIPCC, *flags, "-S", "--offload-device-only", "-I", build.CSRC,
                        os.path.join(build.CSRC, name), "-o", str(out)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"^([A-Za-z_]\w*):.*?\n(.*?)^\.Lfunc_end", out.read_text(), re.M | re.S)
    shapes = {k: set(re.findall(r"v_mfma_\w+", body)) for k, body in kernels}
    assert any(shapes.values())
    assert {k: s for k, s in shapes.items() if len(s) > 1} == {}
