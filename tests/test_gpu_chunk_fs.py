"""The scalar-gate op outside the bf16 chunk-WY shapes: the f32 scalar-gate chunk
kernels (16-token chunks) against the f64 oracle, at the edges of their tiles.

Gates: f32 inputs within 1e-4 (rms-floored) and bf16 inputs within 2e-2, the
gates of the f32 and bf16 paths everywhere in these tests; the kernels'
products and sums are f32, so a chunk of 16 tokens adds a few 1e-7 per term.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gpu_util import TOL_BF16, TOL_F32, dev, gate  # noqa: E402
from test_gpu_scalar_decode import scalar_oracle, scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import delta_kernels
    delta_kernels.lib()
    return delta_kernels


def _check(dk, p, dtype, tol, chunk=64, layout=None):
    if dtype == torch.bfloat16:
        for n in ("q", "k", "v", "dO"):
            p[n] = torch.tensor(p[n]).to(torch.bfloat16).float().numpy()
    x = {n: dev(p[n], dtype if n in ("q", "k", "v", "dO") else torch.float32)
         for n in ("q", "k", "v", "beta", "g", "valid", "reset", "initial", "dO", "dF", "dS")}
    if layout:
        x = {n: layout(n, t) for n, t in x.items()}
    a = [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
    out, fin, sc, ck = dk.gdn_scalar_forward(*a, x["initial"], chunk)
    got = dk.gdn_scalar_backward(*a, ck, chunk, x["dO"], x["dF"], x["dS"])
    o_out, o_fin, o_sc, og, odb, odg = scalar_oracle(p)
    pad = (p["valid"] == 0)[:, :, None]
    gate("output", out, o_out, tol, exact_zero=pad[..., None])
    gate("final_state", fin, o_fin, tol)
    gate("scores", sc, o_sc, tol, exact_zero=pad)
    for n, t, ref in zip(("q", "k", "v"), got, (og["q"], og["k"], og["v"])):
        gate("d" + n, t, ref, tol, exact_zero=pad[..., None])
    gate("dbeta", got[3], odb, tol, exact_zero=pad)
    gate("dg", got[4], odg, tol, exact_zero=pad)
    gate("d_initial", got[5], og["initial"], tol)


# T around the 16-token tiles; widths around the 16-channel tiles, on both sides
# of the 64-wide kernels, with d_k != d_v either way.
@pytest.mark.parametrize("T,K,V", [(1, 16, 16), (15, 1, 3), (16, 17, 64), (17, 64, 15),
                                   (33, 33, 40), (50, 64, 64), (49, 65, 32), (40, 32, 80),
                                   (67, 128, 128), (31, 127, 113)])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, TOL_F32), (torch.bfloat16, TOL_BF16)])
def test_edges_match_oracle(dk, T, K, V, dtype, tol):
    p = scalar_problem(5 + T, 2, T, 3, K, V, masks=False)
    rng = np.random.default_rng(T)
    p["valid"] = (rng.random((2, T)) > 0.15).astype(np.float32)
    p["reset"] = (rng.random((2, T)) < 0.1).astype(np.float32)
    p["valid"][0, 0] = 1
    # chunk 16: no shape here takes the 64-token bf16 kernels
    _check(dk, p, dtype, tol, chunk=16)


def test_extreme_decays_match_oracle(dk):
    """alpha = 1 (g = 0), alpha underflowing to 0 in f32 and g = -inf: dg is the
    full pair products' sum, so a zero decay gives a zero gradient, no NaN."""
    p = scalar_problem(9, 1, 70, 2, 64, 64, masks=False)
    p["g"][0, 5:20] = 0.0
    p["g"][0, 25] = -200.0
    p["g"][0, 40] = -np.inf
    x = {n: dev(p[n]) for n in ("q", "k", "v", "beta", "g", "valid", "reset", "initial", "dO")}
    a = [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
    out, fin, _, ck = dk.gdn_scalar_forward(*a, x["initial"], 64)
    got = dk.gdn_scalar_backward(*a, ck, 64, x["dO"])
    p["dF"][:] = 0
    p["dS"][:] = 0
    o_out, o_fin, _, og, odb, odg = scalar_oracle(p)
    odg[0, 40] = 0.0  # exp(-inf) * dalpha
    for n, t, ref in (("output", out, o_out), ("final", fin, o_fin), ("dq", got[0], og["q"]),
                      ("dk", got[1], og["k"]), ("dv", got[2], og["v"]), ("dbeta", got[3], odb),
                      ("dg", got[4], odg), ("d_initial", got[5], og["initial"])):
        gate(n, t, ref, TOL_F32)


@pytest.mark.parametrize("kind", ["strided", "offset", "expanded"])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, TOL_F32), (torch.bfloat16, TOL_BF16)])
def test_layouts_match_oracle(dk, kind, dtype, tol):
    """Channel strides, misaligned rows and stride-0 heads take the element reads;
    unit-stride aligned rows the four-channel ones."""
    p = scalar_problem(11, 2, 45, 3, 48, 32)
    if kind == "expanded":
        for n in ("q", "k", "v", "dO"):
            p[n][:] = p[n][:, :, :1]

    def layout(n, t):
        if n not in ("q", "k", "v", "dO"):
            return t
        if kind == "strided":
            return t.permute(3, 1, 0, 2).contiguous().permute(2, 1, 3, 0)
        if kind == "offset":  # rows of 50 + 1 elements, from element 1 on
            pad = torch.zeros(t.shape[:3] + (51,), dtype=t.dtype, device=t.device)
            pad[..., 1:1 + t.shape[3]] = t
            return pad[..., 1:1 + t.shape[3]]
        return t[:, :, :1].contiguous().expand(t.shape)

    _check(dk, p, dtype, tol, layout=layout)


def test_backward_windows_are_the_same_bits(dk):
    """A workspace of the queried size holds 4064 chunks of 64 x 64: this shape
    has more, so its backward walks two windows; a workspace that holds them all
    gives the same bits, and so does the library's fixed scratch."""
    from delta_kernels import _ptr, _shape, _stream, _view
    from delta_kernels._lib import check, lib
    L = lib()
    torch.manual_seed(3)
    B, T, H, D = 2, 4200, 8, 64
    r = lambda *s: torch.randn(*s, device="cuda")  # noqa: E731
    q, k, v, dO = (torch.nn.functional.normalize(r(B, T, H, D), dim=-1) for _ in range(4))
    beta, g = torch.sigmoid(r(B, T, H)), -torch.nn.functional.softplus(r(B, T, H))
    valid, reset = torch.ones(B, T, device="cuda"), torch.zeros(B, T, device="cuda")
    dF = r(B, H, D, D)
    out, fin, sc, ck = dk.gdn_scalar_forward(q, k, v, beta, g, valid, reset, None, 64)
    ref = dk.gdn_scalar_backward(q, k, v, beta, g, valid, reset, ck, 64, dO, dF)
    shape = _shape(q, v)
    need = L.gdn_scalar_workspace_bytes(ctypes.byref(shape), 64)
    chunks = B * H * -(-T // 16)
    assert need == 64 << 20 and chunks * (D * D + 32) * 4 > need
    views = [_view(x) for x in (q, k, v, beta, g, valid, reset)]
    dov = _view(dO)
    for noalloc in (False, True):
        got = [torch.empty_like(x) for x in ref]
        args = [ctypes.byref(shape), 64, *[ctypes.byref(x) for x in views], _ptr(ck), ck.numel(),
                ctypes.byref(dov), _ptr(dF), None, *[_ptr(x) for x in got]]
        ws = torch.empty(chunks * (D * D + 32) * 4, dtype=torch.uint8, device="cuda")
        if noalloc:
            check("noalloc", L.gdn_scalar_backward_noalloc(*args, _stream(q)))
        else:
            check("backward", L.gdn_scalar_backward(*args, _ptr(ws), ws.numel(), _stream(q)))
        torch.cuda.synchronize()
        for n, a, b in zip(("dq", "dk", "dv", "dbeta", "dg", "d_initial"), got, ref):
            assert torch.equal(a, b), n
