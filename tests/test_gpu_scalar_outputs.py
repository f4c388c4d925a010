"""The scalar-gate forward for a caller that no backward follows: the outputs of the training forward,
on whichever kernels the forward alone is faster, and the autograd function's choice of it."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from gpu_util import TOL_BF16, TOL_F32, dev, gate  # noqa: E402
from test_gpu_chunk_fs import dk  # noqa: E402,F401
from test_gpu_scalar_decode import scalar_oracle, scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu

F32, BF = torch.float32, torch.bfloat16


def _x(p, dtype):
    return [dev(p[n], dtype if n in ("q", "k", "v") else F32)
            for n in ("q", "k", "v", "beta", "g", "valid", "reset", "initial")]


def _bytes(x, chunk=64):
    from delta_kernels import _shape, _view
    from delta_kernels._lib import lib
    v = [_view(t) for t in x[:3]]
    r = ctypes.byref
    return lib().gdn_scalar_outputs_bytes(r(_shape(x[0], x[2])), chunk, *[r(t) for t in v])


# B, T, H, K, V, dtype, whether the walk takes it (no workspace)
@pytest.mark.parametrize("B,T,H,K,V,dtype,walked", [
    (2, 1, 3, 64, 64, F32, True), (2, 16, 3, 33, 40, F32, True), (2, 17, 3, 64, 64, F32, True),
    (2, 130, 3, 64, 64, F32, False), (2, 90, 3, 128, 17, BF, False), (64, 50, 16, 32, 64, F32, True),
    (32, 70, 16, 48, 33, BF, True), (2, 70, 3, 64, 64, BF, False), (2, 70, 3, 128, 128, BF, False)])
def test_matches_the_oracle(dk, B, T, H, K, V, dtype, walked):  # noqa: F811
    p = scalar_problem(T, min(B, 2), T, H, K, V)
    if dtype == BF:
        for n in ("q", "k", "v"):
            p[n] = torch.tensor(p[n]).to(BF).float().numpy()
    x = _x(p, dtype)
    if B > 2:  # the problem over and over
        x = [t.repeat(B // 2, *[1] * (t.dim() - 1)) for t in x]
    assert (_bytes(x) == 0) == walked
    with torch.no_grad():
        out, fin, sc = dk.gdn_scalar_scan(*x, 64)
    tol = TOL_BF16 if dtype == BF else TOL_F32
    for name, t, ref in zip(("output", "final_state", "scores"), (out, fin, sc), scalar_oracle(p)):
        n = ref.shape[0]
        gate(name, t[:n], ref, tol)
        gate(name, t[-n:], ref, tol)


def test_any_gradient_takes_the_training_forward(dk):  # noqa: F811
    p = scalar_problem(3, 2, 40, 3, 64, 64)
    x = _x(p, F32)
    for i in (0, 1, 2, 3, 4, 7):
        y = [t.clone().requires_grad_(n == i) for n, t in enumerate(x)]
        out = dk.gdn_scalar_scan(*y, 64)[0]
        assert out.requires_grad
        out.sum().backward()
        assert torch.isfinite(y[i].grad).all() and y[i].grad.abs().sum() > 0
        with torch.no_grad():
            assert not dk.gdn_scalar_scan(*y, 64)[0].requires_grad
    assert not dk.gdn_scalar_scan(*x, 64)[0].requires_grad


def test_captured(dk):  # noqa: F811
    for B, T in ((2, 17), (2, 200)):
        x = _x(scalar_problem(T, B, T, 3, 64, 64), F32)
        with torch.no_grad():
            want = dk.gdn_scalar_scan(*x, 64)
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                dk.gdn_scalar_scan(*x, 64)
            torch.cuda.current_stream().wait_stream(s)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                got = dk.gdn_scalar_scan(*x, 64)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(got, want):
                assert torch.equal(a, b)
                a.zero_()


def test_small_workspace_is_refused(dk):  # noqa: F811
    from delta_kernels import _code, _ptr, _shape, _stream, _view
    from delta_kernels._lib import lib
    x = _x(scalar_problem(4, 2, 130, 3, 64, 64), F32)
    n = _bytes(x)
    assert n > 0
    out, fin, sc = (torch.empty(s, device="cuda") for s in ((2, 130, 3, 64), (2, 3, 64, 64), (2, 130, 3)))
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    v = [_view(t) for t in x]
    r = ctypes.byref
    call = lambda p, m: lib().gdn_scalar_outputs(  # noqa: E731
        r(_shape(x[0], x[2])), 64, *[r(t) for t in v], _ptr(out), _code(out), _ptr(fin), _ptr(sc), p, m,
        _stream(out))
    assert call(_ptr(ws), n - 1) == 4
    assert call(None, n) == 1
    assert call(_ptr(ws), n) == 0
    torch.cuda.synchronize()
