"""The HOLA kernels' row forms and schedule merge against the f64 oracle: widths in whole
float4 (vector rows) and not, every padded width, channel-strided operands, odd
slot counts, key walks past the waves of one workgroup and entries that outlive
many chunks.

Gate: 1e-4 (rms-floored), the f32 gate; the products and sums are f32 over at
most 128 channels and 80 slots, so a term adds a few 1e-7.  Positions are exact.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gpu_util import TOL_F32, gate  # noqa: E402
from oracle import hola_oracle as ho  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import delta_kernels
    delta_kernels.lib()
    return delta_kernels


def _dev(x, strided):
    if strided and x.ndim == 4:  # channels four apart
        wide = torch.zeros(*x.shape, 4, device="cuda")
        wide[..., 1] = torch.from_numpy(x).cuda()
        return wide[..., 1].detach()
    return torch.from_numpy(x).cuda()


@pytest.mark.parametrize("K,V,T,cap,chunk,recency,strided", [
    (64, 64, 200, 64, 16, False, False),
    (64, 64, 130, 64, 16, True, True),
    (33, 40, 100, 5, 7, False, False),
    (40, 124, 75, 16, 16, False, False),
    (128, 30, 50, 3, 16, False, True),
    (4, 1, 33, 64, 1, False, False),
    (1, 128, 17, 1, 16, True, False),
])
def test_rows(dk, K, V, T, cap, chunk, recency, strided):
    B, H = 2, 3
    rng = np.random.default_rng(K * 1000 + T)
    r = lambda *s: rng.normal(size=s).astype(np.float32)  # noqa: E731
    p = dict(q=r(B, T, H, K), k=r(B, T, H, K), v=r(B, T, H, V), sink=r(H), up=r(B, T, H, V))
    # Halves: many ties.  Falling on head 0, so that its first tokens stay cached.
    scores = (np.round(2 * rng.exponential(size=(B, T, H))) / 2).astype(np.float32)
    scores[:, :, 0] = -np.arange(T, dtype=np.float32)
    valid = (rng.random((B, T)) < 0.9).astype(np.float32)
    docs = np.zeros((B, T), np.float32)
    docs[1, T // 3:] = 1
    x = {n: _dev(p[n], strided).requires_grad_(n != "up") for n in p}
    sc, va, do = (torch.from_numpy(n).cuda() for n in (scores, valid, docs))
    got = dk.hola_read(x["q"], x["k"], x["v"], sc, va, do, x["sink"], cap, chunk, recency,
                       return_final_positions=True)
    (got.output * x["up"]).sum().backward()
    ref = ho.hola_read(p["q"], p["k"], p["v"], scores[..., None], valid, docs, p["sink"], cap, chunk,
                       recency, upstream=p["up"])
    np.testing.assert_array_equal(got.final_positions.cpu().numpy(), ref["positions"])
    gate("output", got.output, ref["output"], TOL_F32)
    for n in ("q", "k", "v", "sink"):
        gate("d" + n, x[n].grad, ref["d" + n], TOL_F32)
    want = ho.hola_schedule(scores[..., None], valid, docs, cap, chunk, recency)
    plan = dk.hola_schedule(sc, va, do, cap, chunk, recency)
    np.testing.assert_array_equal(plan.cpu().numpy(), want)
