"""Which kernels a scalar-gate call runs, by the stages that it reports: the chunk-WY kernels, the
f32 chunk kernels, or, to 16 tokens, the token walk (which reports none).  A call that falls
through to another family reports another family's stages, so the path checks of the other
tests (chunk_util.chunk_stages) cannot pass on it."""
import pytest

torch = pytest.importorskip("torch")

from chunk_util import chunk_stages  # noqa: E402
from gpu_util import dev  # noqa: E402
from test_gpu_chunk_fs import dk  # noqa: E402,F401
from test_gpu_scalar_decode import scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu

F32_STAGES = {"scalar_f32_" + n for n in ("prep", "state_scan", "out", "bprep", "adjoint_scan",
                                          "bgrad")}
BF, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("dtype,T,K,V,chunk,offset,want", [
    (BF, 70, 64, 64, 64, 0, chunk_stages(64)), (BF, 70, 128, 128, 64, 0, chunk_stages(128)),
    (BF, 9, 64, 64, 64, 0, chunk_stages(64)),
    (BF, 70, 64, 64, 16, 0, F32_STAGES), (BF, 70, 64, 64, 64, 1, F32_STAGES),
    (BF, 70, 64, 128, 64, 0, F32_STAGES), (F32, 70, 64, 64, 64, 0, F32_STAGES),
    (F32, 17, 33, 40, 64, 0, F32_STAGES), (F32, 16, 64, 64, 64, 0, set()),
    (BF, 16, 64, 64, 64, 1, set())])
def test_stages_tell_the_kernels(dk, dtype, T, K, V, chunk, offset, want):  # noqa: F811
    p = scalar_problem(T, 2, T, 3, K, V)

    def seq(n):  # offset: bases that are not 16-byte aligned
        t = dev(p[n], dtype)
        buf = torch.empty(t.numel() + offset, dtype=dtype, device="cuda")
        return buf[offset:].view(t.shape).copy_(t)

    a = [seq(n) for n in ("q", "k", "v")] + [dev(p[n]) for n in ("beta", "g", "valid", "reset")]
    dk.stage_timing(True)
    try:
        out, _, _, ck = dk.gdn_scalar_forward(*a, dev(p["initial"]), chunk)
        dk.gdn_scalar_backward(*a, ck, chunk, dev(p["dO"], dtype))
        torch.cuda.synchronize()
        ran = set(dk.stage_times())
    finally:
        dk.stage_timing(False)
    assert ran == want
