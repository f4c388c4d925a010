"""What the mixer's packed projections keep and compute: each gradient in memory of its own, no
product for a frozen weight, and nothing kept for the backward beyond what its operators read."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from delta_mixers.mixer import GdnMixer, GdnMixerConfig, _Projections  # noqa: E402


def _grads(need):
    x = torch.randn(3, 4, 6, dtype=torch.float64)
    ws = [torch.randn(n, 6, dtype=torch.float64) for n in (5, 2, 3)]
    dz = torch.randn(3, 4, 10, dtype=torch.float64)
    got = _Projections.backward(SimpleNamespace(saved_tensors=(x, *ws), needs_input_grad=need, gates=0,
                                                 extra=0), dz)
    want = [d.flatten(0, 1).t() @ x.flatten(0, 1) for d in dz.split([5, 2, 3], -1)]
    return got, want


def test_gradients_share_no_memory():
    got, want = _grads((True,) * 4)
    for g, w in zip(got[1:], want):
        torch.testing.assert_close(g, w, rtol=1e-12, atol=1e-12)
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()


@pytest.mark.parametrize("frozen", [0, 1, 2])
def test_frozen_weights_cost_nothing(frozen):
    need = [True] * 4
    need[1 + frozen] = False
    got, want = _grads(tuple(need))
    for i, (g, w) in enumerate(zip(got[1:], want)):
        if i == frozen:
            assert g is None
        else:
            torch.testing.assert_close(g, w, rtol=1e-12, atol=1e-12)
    got, _ = _grads((False,) + tuple(need[1:]))
    assert got[0] is None


def _pieces(x, ws, pieces, gates):
    z = list(torch.cat([x @ w.t() for w in ws], -1).split(pieces, -1))
    return [torch.sigmoid(t) if i >= len(pieces) - gates else t for i, t in enumerate(z)]


@pytest.mark.parametrize("pieces,gates", [((7, 3), 1), ((5, 2, 3), 2), ((4, 1, 5), 3), ((10,), 1),
                                          ((6, 4), 0)])
def test_pieces_and_gates(pieces, gates):
    """Bound: float64 products, compared at 1e-12."""
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).requires_grad_()  # noqa: E731
    x, ws = r(3, 4, 6), [r(n, 6) for n in (5, 2, 3)]
    ref = _pieces(x, ws, pieces, gates)
    up = [torch.randn(t.shape, generator=g, dtype=torch.float64) for t in ref]
    kept = [u.clone() for u in up]
    got = _Projections.apply(x, *ws, pieces, gates)
    for a, b in zip(got, ref):
        torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-12)
    for a, b in zip(torch.autograd.grad(got, [x] + ws, up), torch.autograd.grad(ref, [x] + ws, up)):
        torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-12)
    assert all(torch.equal(a, b) for a, b in zip(up, kept))
    # a piece that nothing uses, and the second derivative
    got = _Projections.apply(x, *ws, pieces, gates)
    want = torch.autograd.grad(_pieces(x, ws, pieces, gates)[0].pow(2).sum(), ws, create_graph=True)
    got = torch.autograd.grad(got[0].pow(2).sum(), ws, create_graph=True)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-12)
    second = [torch.autograd.grad(sum(t.pow(2).sum() for t in ts), [x] + ws) for ts in (got, want)]
    for a, b in zip(*second):
        torch.testing.assert_close(a, b, rtol=1e-10, atol=1e-10)


@pytest.mark.gpu
def test_kept_for_the_backward():
    """The buffer of the projections that the operators read (q, k, v, decay, gate), the gates'
    sigmoids and the operators' own results; erase and write are not kept twice."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    B, T, D, H, K, V = 4, 512, 256, 8, 64, 64
    m = GdnMixer(GdnMixerConfig(d_model=D, heads=H, key_dim=K, value_dim=V), device="cuda")
    x = torch.randn(B, T, D, device="cuda", requires_grad=True)
    m(x).sum().backward()  # allocations that stay
    kept, seen = 0, set()

    def pack(t):
        nonlocal kept
        if t.untyped_storage().data_ptr() not in seen:
            seen.add(t.untyped_storage().data_ptr())
            kept += t.untyped_storage().nbytes()
        return t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        y = m(x)
    # The seven projections (erase and write as their sigmoids), the convolution's result, the
    # normed q and k, alpha, the scan's output, its normed rows, the masked x; the weights; and
    # a few values a token (masks, the norms' inverses).
    rows = H * (4 * K + 3 * V) + H * (2 * K + V) + 2 * H * K + H * K + 2 * H * V + D
    weights = sum(p.numel() for p in m.parameters()) + m.q_conv.shape[0] * H * (2 * K + V)
    assert kept <= 4 * (B * T * (rows + 64) + weights)
    assert y.requires_grad
