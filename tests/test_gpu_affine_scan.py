"""The chunk scans of the 64-wide bf16 kernels against the f64 oracle: chunk counts around
the ring's depth and the two-step loop, with decays so weak that the states of
all earlier chunks reach the last (a map applied with a wrong column shows).

Gate: 2e-2 (rms-floored), the bf16 gate of these kernels.
"""
import pytest

torch = pytest.importorskip("torch")

from gpu_util import TOL_BF16  # noqa: E402
from test_gpu_chunk_fs import _check, dk  # noqa: E402,F401
from test_gpu_scalar_decode import scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [64, 65, 192, 256, 257, 384, 450])
def test_chunk_counts(dk, T):  # noqa: F811
    p = scalar_problem(3 + T, 1, T, 3, 64, 64, masks=False)
    p["g"] *= 1e-3
    p["beta"] *= 0.3
    p["initial"] *= 10
    p["dF"] *= 10
    _check(dk, p, torch.bfloat16, TOL_BF16, chunk=64)
