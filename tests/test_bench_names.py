"""The stage that bench.py reads off a profiler's kernel name, for the names of the kernels that the
built library holds."""
import os
import shutil
import subprocess

import pytest

import bench

LIB = os.path.join(os.path.dirname(os.path.abspath(bench.__file__)), "delta-block-lm_amd", "lib",
                   "libgdn2_amd.so")


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB) or not shutil.which("nm"):
        pytest.skip("the library is not built, or there is no nm")
    text = subprocess.run(["nm", "-C", LIB], check=True, capture_output=True, text=True).stdout
    return sorted({n.split(" ", 2)[2] for n in text.splitlines() if "_kernel<" in n})


# kernel, the position of its direction among the template arguments
@pytest.mark.parametrize("kernel,config,at", [("lr_scan", "LrCfg<", -1), ("fc_scan", "fc_scan_kernel<", 1),
                                              ("affine_scan", "affine_scan_kernel<", 0)])
def test_scan_directions(kernels, kernel, config, at):
    names = [n for n in kernels if f"::{kernel}_kernel<" in n and "__device_stub__" not in n]
    seen = set()
    for n in names:
        args = n.split(config, 1)[1].split(">", 1)[0].split(",")
        want = "adjoint_scan" if args[at].strip() == "true" else "state_scan"
        assert bench.kernel_stage(n) == (kernel, want), n
        seen.add(want)
    assert seen == {"state_scan", "adjoint_scan"}, names


@pytest.mark.parametrize("name,want", [
    ("void gdn2::lr_scan_kernel<gdn2::(anonymous namespace)::LrCfg<128, 64, 2, 2, true> >(gdn2::LrScanArgs)",
     ("lr_scan", "adjoint_scan")),
    ("void gdn2::lr_scan_kernel<gdn2::(anonymous namespace)::LrCfg<128, 64, 2, 3, false> >(gdn2::LrScanArgs)",
     ("lr_scan", "state_scan")),
    ("gdn2::wide_bgrad_kernel(gdn2::ChunkArgs)", ("wide_bgrad", "chunk_bgrad")),
    ("void gdn2::fs_prep_kernel<4, false, true>(gdn2::FcArgs)", ("fs_prep", "chunk_prep")),
    ("gdn2::hola_schedule_kernel(gdn2::HolaArgs)", ("hola_schedule", None)),
    ("Cijk_Ailk_Bjlk_BBS_BH", (None, None))])
def test_names(name, want):
    assert bench.kernel_stage(name) == want
