"""The mixer's packed projections against the same products one by one: columns at ragged
widths (rows that are and are not 16-byte aligned), frozen weights, a weight changed between
the passes (refused, as torch refuses it)."""
import pytest

torch = pytest.importorskip("torch")

from delta_mixers.mixer import GdnMixer, GdnMixerConfig, _Projections  # noqa: E402

F = torch.nn.functional


@pytest.mark.parametrize("widths", [(1,), (8, 8, 16), (33, 33, 40, 7)])
@pytest.mark.parametrize("frozen", [None, 0, 1])
def test_projections(widths, frozen):
    """Bound: float64 products, compared at 1e-12."""
    g = torch.Generator().manual_seed(len(widths))
    x = torch.randn(2, 5, 24, generator=g, dtype=torch.float64, requires_grad=frozen != 0)
    ws = [torch.randn(w, 24, generator=g, dtype=torch.float64,
                      requires_grad=frozen != 1 or i > 0) for i, w in enumerate(widths)]
    up = torch.randn(2, 5, sum(widths), generator=g, dtype=torch.float64)
    ins = [t for t in [x] + ws if t.requires_grad]
    if not ins:
        pytest.skip("nothing to differentiate")
    z = _Projections.apply(x, *ws)
    ref = torch.cat([F.linear(x, w) for w in ws], -1)
    torch.testing.assert_close(z, ref, rtol=1e-12, atol=1e-12)
    for got, want in zip(torch.autograd.grad(z, ins, up), torch.autograd.grad(ref, ins, up)):
        torch.testing.assert_close(got, want, rtol=1e-12, atol=1e-12)


def test_changed_weight_is_refused():
    x = torch.randn(3, 4, requires_grad=True)
    w = torch.randn(5, 4, requires_grad=True)
    z = _Projections.apply(x, w)
    with torch.no_grad():
        w.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        z.sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,keys,values", [(1, 33, 40), (3, 20, 64), (4, 32, 64)])
def test_mixer_reads_its_columns(heads, keys, values):
    """One module, its projections packed and one by one: the same operators on contiguous
    tensors.  Bound: f32 sums of 48 products and a 37-token scan, a few 1e-6; 1e-5."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import delta_kernels as dk
    torch.manual_seed(keys)
    B, T, D, H, K, V = 2, 37, 48, heads, keys, values
    m = GdnMixer(GdnMixerConfig(d_model=D, heads=H, key_dim=K, value_dim=V,
                                cache_policy="none"), device="cuda")
    x = torch.randn(B, T, D, device="cuda", requires_grad=True)
    valid, reset = torch.ones(B, T, device="cuda"), torch.zeros(B, T, device="cuda")
    valid[0, -3:], reset[1, 11] = 0.0, 1.0
    xv = x * valid[..., None]
    docs = torch.cumsum(reset * valid, 1)
    conv = lambda w, c, n: dk.causal_conv(F.linear(xv, w), c, valid, docs,  # noqa: E731
                                          activation="silu").view(B, T, H, n)
    lin = lambda w, n: F.linear(xv, w).view(B, T, H, n)  # noqa: E731
    scan = dk.gdn_training_scan(
        dk.l2_norm(conv(m.q, m.q_conv, K)), dk.l2_norm(conv(m.k, m.k_conv, K)),
        conv(m.v, m.v_conv, V), dk.decay(lin(m.decay, K), m.decay_bias, m.decay_scale),
        torch.sigmoid(lin(m.erase, K)), torch.sigmoid(lin(m.write, V)), valid, reset, None,
        m.cfg.chunk_size)
    y = dk.rms_norm(scan.output, m.norm_weight, lin(m.output_gate, V), m.cfg.norm_epsilon)
    ref = F.linear(y.reshape(B, T, H * V), m.output) * valid[..., None]
    got = m(x, valid, reset)
    up = torch.randn_like(ref)
    ins = [x] + list(m.parameters())
    pairs = [(got, ref)] + list(zip(torch.autograd.grad(got, ins, up),
                                    torch.autograd.grad(ref, ins, up)))
    for a, b in pairs:
        assert float((a - b).norm()) <= 1e-5 * max(float(b.norm()), 1e-30)
