"""The two read forms of the f32 chunk kernels on one input: whole 16-channel tiles from aligned rows,
and element by element where a base, a row or a channel stride does not allow that.  They read the same
values into the same products, so every result has the same bits; the aligned form is checked against the
oracle by the other tests.  And the scalar-gate backward over several chunk windows.
"""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from test_gpu_chunk_fs import dk  # noqa: E402,F401

pytestmark = pytest.mark.gpu

F32, BF = torch.float32, torch.bfloat16


def _off(t, kind):
    """t with an element before its base, with rows an odd number of elements apart, or with
    channels two apart."""
    if kind == "base":
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        return buf[1:].view(t.shape).copy_(t)
    if kind == "rows":
        buf = torch.empty(*t.shape[:-1], t.shape[-1] + 1, dtype=t.dtype, device="cuda")
        return buf[..., :-1].copy_(t)
    buf = torch.empty(*t.shape, 2, dtype=t.dtype, device="cuda")
    return buf[..., 0].copy_(t)


def _inputs(seed, B, T, H, K, V, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)  # noqa: E731
    x = dict(q=unit(r(B, T, H, K)).to(dtype), k=unit(r(B, T, H, K)).to(dtype), v=r(B, T, H, V).to(dtype),
             alpha=torch.rand(B, T, H, K, generator=g, device="cuda"), erase=torch.sigmoid(r(B, T, H, K)),
             write=torch.sigmoid(r(B, T, H, V)), valid=torch.ones(B, T, device="cuda"),
             reset=torch.zeros(B, T, device="cuda"), initial=r(B, H, K, V), dO=r(B, T, H, V).to(dtype),
             dF=r(B, H, K, V), dS=r(B, T, H, 1))
    x["valid"][0, T // 2] = 0
    x["reset"][0, T // 3] = 1
    return x


def _same(got, want):
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("which", [("q",), ("v",), ("alpha",), ("write",), ("dO",),
                                   ("q", "k", "v", "alpha", "erase", "write", "dO")])
@pytest.mark.parametrize("kind", ["base", "rows", "channels"])
@pytest.mark.parametrize("K,V,dtype", [(32, 64, F32), (64, 48, BF), (128, 16, F32)])
@pytest.mark.parametrize("scores", [False, True])
def test_channel_gates(dk, which, kind, K, V, dtype, scores):  # noqa: F811
    x = _inputs(K + V, 2, 45, 3, K, V, dtype)
    dS = x["dS"] if scores else None

    def call(x):
        a = [x[n] for n in ("q", "k", "v", "alpha", "erase", "write", "valid", "reset")]
        out, fin, sc, ck = dk.gdn_training_forward(*a, x["initial"], 16)
        return [out, fin, sc, *_backward(dk, "gdn2_training", a, ck, x["dO"], x["dF"], dS)]

    _same(call(dict(x, **{n: _off(x[n], kind) for n in which})), call(x))


def _backward(dk, name, a, ck, dO, dF, dS, ws_bytes=0):  # noqa: F811
    """The C call itself: the Python operators hand it dense upstreams."""
    from delta_kernels import _ptr, _shape, _stream, _view
    from delta_kernels._lib import check, lib
    shape, r = _shape(a[0], a[2]), ctypes.byref
    scalar = name == "gdn_scalar"
    views = [_view(t) for t in a]
    outs = [torch.empty(t.shape, dtype=t.dtype, device="cuda") for t in a[:5 if scalar else 6]]
    outs.append(torch.empty(a[0].shape[0], a[0].shape[2], a[0].shape[3], a[2].shape[3], device="cuda"))
    n = getattr(lib(), name + "_workspace_bytes")(r(shape), 16)
    ws = torch.empty(max(n, ws_bytes), dtype=torch.uint8, device="cuda")
    dov = _view(dO)
    check(name, getattr(lib(), name + "_backward")(
        r(shape), 16, *[r(v) for v in views], _ptr(ck), ck.numel(), r(dov), _ptr(dF), _ptr(dS),
        *[_ptr(t) for t in outs], _ptr(ws), ws.numel(), _stream(ck)))
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("which", [("q",), ("v",), ("dO",), ("q", "k", "v", "dO")])
@pytest.mark.parametrize("kind", ["base", "rows", "channels"])
@pytest.mark.parametrize("K,V,dtype", [(32, 64, F32), (64, 64, BF), (128, 16, F32)])
@pytest.mark.parametrize("scores", [False, True])
def test_scalar_gates(dk, which, kind, K, V, dtype, scores):  # noqa: F811
    x = _inputs(K + V, 2, 45, 3, K, V, dtype)
    x.update(beta=x["erase"][..., 0].contiguous(), g=torch.log(x["alpha"][..., 0]).contiguous())
    dS = x["dS"] if scores else None

    def call(x):
        a = [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
        out, fin, sc, ck = dk.gdn_scalar_forward(*a, x["initial"], 16)
        return [out, fin, sc, *_backward(dk, "gdn_scalar", a, ck, x["dO"], x["dF"], dS)]

    _same(call(dict(x, **{n: _off(x[n], kind) for n in which})), call(x))


@pytest.mark.parametrize("which", [("q",), ("alpha",), ("q", "k", "v", "alpha", "erase", "write")])
@pytest.mark.parametrize("kind", ["base", "rows", "channels"])
@pytest.mark.parametrize("K,V,dtype", [(32, 64, F32), (64, 48, BF)])
def test_documents(dk, which, kind, K, V, dtype):  # noqa: F811
    x = _inputs(K + V, 2, 45, 3, K, V, dtype)
    start = torch.zeros(2, 45, dtype=torch.int32, device="cuda")
    start[:, 20:] = 20
    end = torch.full_like(start, 44)
    end[:, :20] = 19
    end[1, 40:] = -1

    def call(x):
        a = [x[n] for n in ("q", "k", "v", "alpha", "erase", "write")]
        out, ck = dk.gdn2_scan_forward(*a, start, end)
        return [out, *dk.gdn2_backward(*a, x["dO"], ck, start, end)]

    _same(call(dict(x, **{n: _off(x[n], kind) for n in which})), call(x))


@pytest.mark.parametrize("T,K,V", [(8000, 33, 40), (4200, 64, 64)])
@pytest.mark.parametrize("scores", [False, True])
def test_windows_are_the_same_bits(dk, T, K, V, scores):  # noqa: F811
    """More chunks than the queried workspace holds at once (64 MiB), the score adjoint's coefficients and
    widths padded to tiles among them, against a workspace that holds them all."""
    B, H = 2, 8
    x = _inputs(T, B, T, H, K, V, F32)
    a = [x["q"], x["k"], x["v"], x["erase"][..., 0].contiguous(),
         torch.log(0.5 + 0.5 * x["alpha"][..., 0]).contiguous(), x["valid"], x["reset"]]
    ck = dk.gdn_scalar_forward(*a, x["initial"], 16)[3]
    chunks, up = B * H * -(-T // 16), lambda n: -(-n // 16) * 16  # noqa: E731
    whole = chunks * (up(K) * up(V) + 32) * 4
    assert whole > 64 << 20
    dS = x["dS"] if scores else None
    two = _backward(dk, "gdn_scalar", a, ck, x["dO"], x["dF"], dS)
    _same(two, _backward(dk, "gdn_scalar", a, ck, x["dO"], x["dF"], dS, whole + (1 << 20)))
