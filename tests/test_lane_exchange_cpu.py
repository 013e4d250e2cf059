"""few_kernel's experts (kernels_lin.hip): lanes whose row did not choose an expert read the row of a lane that did.  What they read is multiplied into
columns that nobody stores, so no result can show a wrong row; the compiled kernel can."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_the_row_of_another_lane_is_read_from_a_lane_that_is_on(tmp_path):
    out = tmp_path / "lin.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", "-S",
                           "--offload-device-only", os.path.join(ROOT, "deepseek.cpp_amd", "csrc", "kernels_lin.hip"), "-o", str(out)], stderr=subprocess.DEVNULL)
    text = out.read_text()
    bodies = [b.split("s_endpgm\n.Lfunc_end")[0] for b in text.split("\n_Z10few_kernel")[1:]]
    assert len(bodies) == 3
    for body in bodies:
        # an exchange reads nothing of lanes that are off where it stands (the branch for the other lanes); a scalar read of a lane does not ask
        assert "ds_bpermute" not in body and "v_readlane" in body
