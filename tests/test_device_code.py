"""What the compiled kernels must look like, checked on their assembly (no
GPU needed: the sources are cross-compiled)."""
import os
import re
import subprocess

import pytest

from tbplas_amd import build


def _assembly(src, tmp_path):
    out = str(tmp_path / "k.s")
    r = subprocess.run([build.HIPCC, *build.COMMON, "--offload-device-only", "-S",
                        os.path.join(build.CSRC, src), "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    with open(out) as f:
        return f.read()


@pytest.mark.parametrize("src", ["tbg_ring_f64_v1_real.hip", "tbg_ring_f32_v2_cplx.hip"])
def test_resident_pass_loads_are_bounds_checked(src, tmp_path):
    """A buffer load's bound is compared with the lane's offset and the
    immediate one only: a scalar offset on top of them would let the lanes
    beyond a short block read beyond its tables."""
    loads = re.findall(r"^\s*buffer_load_\w+ [^,]+, [^,]+, s\[\d+:\d+\], (\S+)",
                       _assembly(src, tmp_path), re.M)
    assert len(loads) > 50
    assert {x.rstrip(",") for x in loads} == {"0"}
