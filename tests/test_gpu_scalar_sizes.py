"""Scalar-gate calls on buffers of exactly the size that the call needs, with the bytes behind them
guarded: the same bits as on larger ones, and nothing written past the end."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from gpu_util import dev  # noqa: E402
from test_gpu_chunk_fs import dk  # noqa: E402,F401
from test_gpu_scalar_decode import scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu

GUARD = 4096


@pytest.mark.parametrize("T,K,V,dtype,bad", [
    (130, 64, 64, torch.bfloat16, False), (130, 128, 128, torch.bfloat16, False),
    (16, 64, 64, torch.float32, False), (9, 33, 40, torch.float32, False),
    (130, 64, 64, torch.float32, False), (50, 33, 40, torch.bfloat16, False),
    (50, 16, 128, torch.float32, True), (130, 128, 17, torch.float32, True)])
def test_exact_buffers(dk, T, K, V, dtype, bad):  # noqa: F811
    from delta_kernels import _code, _ptr, _shape, _stream, _view
    from delta_kernels._lib import check, lib
    L = lib()
    p = scalar_problem(T + K, 2, T, 3, K, V)
    if bad:  # walked by token behind the chunk kernels
        p["k"][1, 20, 2, 0] = float("nan")
    x = {n: dev(p[n], dtype if n in ("q", "k", "v", "dO") else torch.float32) for n in p}
    a = [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
    out, fin, sc, ck0 = dk.gdn_scalar_forward(*a, x["initial"], 64)
    ref = dk.gdn_scalar_backward(*a, ck0, 64, x["dO"], x["dF"], x["dS"])
    shape = _shape(x["q"], x["v"])
    views = [_view(t) for t in a]
    r = ctypes.byref
    qkv = [r(v) for v in views[:3]]
    nck = L.gdn_scalar_call_checkpoint_bytes(r(shape), 64, *qkv)
    nws = L.gdn_scalar_call_workspace_bytes(r(shape), 64, *qkv)
    assert nck == ck0.numel()
    buf = [torch.full((n + GUARD,), 0x5A, dtype=torch.uint8, device="cuda") for n in (nck, nws)]
    got = [torch.empty_like(t) for t in (out, fin, sc)]
    initial, dov = _view(x["initial"]), _view(x["dO"])
    check("scan", L.gdn_scalar_scan(r(shape), 64, *[r(v) for v in views], r(initial), _ptr(got[0]),
                                    _code(out), _ptr(got[1]), _ptr(got[2]), _ptr(buf[0]), nck,
                                    _stream(out)))
    grads = [torch.empty_like(t) for t in ref]
    check("backward", L.gdn_scalar_backward(
        r(shape), 64, *[r(v) for v in views], _ptr(buf[0]), nck, r(dov), _ptr(x["dF"]), _ptr(x["dS"]),
        *[_ptr(t) for t in grads], _ptr(buf[1]), nws, _stream(out)))
    for g, w in zip(got + grads, (out, fin, sc) + tuple(ref)):
        assert torch.allclose(g, w, rtol=0, atol=0, equal_nan=True)
    for b, n in zip(buf, (nck, nws)):
        assert bool((b[n:] == 0x5A).all())
