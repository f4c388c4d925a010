"""NaN and infinities in the scalar-gate op outside the bf16 chunk-WY shapes reach the tokens that
the recurrence takes them to, and no others: the whole call against the token walk, which is a chain
of 16-token calls (calls that short walk their tokens).

A (batch, head) with a bad input is walked by token, so its results are the chain's bit for bit,
NaN for NaN; with a bad upstream gradient its backward is, from the states of the chunk kernels, so
it has the chain's NaN and infinities and its finite values (1e-4, the f32 gate; 2e-2 in bf16), as
the other heads have.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gpu_util import TOL_BF16, TOL_F32, dev, host  # noqa: E402
from test_gpu_chunk_fs import dk  # noqa: E402,F401
from test_gpu_chunk_fs_error import _walk  # noqa: E402
from test_gpu_scalar_decode import scalar_problem  # noqa: E402

pytestmark = pytest.mark.gpu

NAMES = ("output", "final", "scores", "dq", "dk", "dv", "dbeta", "dg", "dinitial")
INF = float("inf")
# input, channel (None: per-token inputs), value
FORWARD = [("k", 3, np.nan), ("k", 0, INF), ("v", 5, INF), ("v", 0, np.nan), ("q", 2, np.nan),
           ("beta", None, np.nan), ("beta", None, -INF), ("g", None, np.nan), ("g", None, INF),
           ("k", 1, 3e38)]
BACKWARD = [("dO", 4, np.nan), ("dO", 0, -INF), ("dS", None, np.nan), ("dF", 7, np.nan)]


def _x(p, dtype):
    x = {n: dev(p[n], dtype if n in ("q", "k", "v", "dO") else torch.float32)
         for n in ("q", "k", "v", "beta", "g", "valid", "reset", "initial", "dO", "dF", "dS")}
    return x


def _call(dk, x, dO=None):  # noqa: F811
    a = [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
    out, fin, sc, ck = dk.gdn_scalar_forward(*a, x["initial"], 16)
    return [out, fin, sc, *dk.gdn_scalar_backward(*a, ck, 16, x["dO"], x["dF"], x["dS"])]


def _chain(dk, x):  # noqa: F811
    return _walk(dk, [x[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset", "dO", "dS")],
                 x["initial"], x["dF"])


def _head(name, t, b, h):
    return t[b, h] if name in ("final", "dinitial") else t[b, :, h]


def _compare(got, want, b, h, tol, bits):
    for n, g, w in zip(NAMES, got, want):
        if bits:
            assert torch.allclose(_head(n, g, b, h), _head(n, w, b, h), rtol=0, atol=0,
                                  equal_nan=True), n
        g, w = host(g), host(w)
        ok = np.isfinite(w)
        assert np.array_equal(np.isfinite(g), ok), n
        assert np.array_equal(g[~ok], w[~ok], equal_nan=True), n
        g, w = g[ok], w[ok]
        assert np.all(np.abs(g - w) <= tol * (np.abs(w) + np.sqrt(np.mean(w * w)))), n


@pytest.mark.parametrize("name,channel,value", FORWARD + BACKWARD)
@pytest.mark.parametrize("dtype,tol,K,V", [(torch.float32, TOL_F32, 64, 64),
                                           (torch.float32, TOL_F32, 33, 40),
                                           (torch.bfloat16, TOL_BF16, 96, 48)])
@pytest.mark.parametrize("t", [0, 20, 47])
def test_reaches_what_the_recurrence_reaches(dk, name, channel, value, dtype, tol, K, V, t):  # noqa: F811
    b, h = 0, 1
    p = scalar_problem(4, 2, 50, 3, K, V)  # a padded token, a reset and a padded end
    p["valid"][0, t] = 1
    if name == "dF":
        p["dF"][b, h, channel, 3] = value
    elif channel is None:
        p[name][b, t, h] = value
    else:
        p[name][b, t, h, channel] = value
    x = _x(p, dtype)
    got = _call(dk, x)
    forward = name not in ("dO", "dS", "dF")
    if forward:
        assert torch.isfinite(got[0][b, :t, h]).all()
    elif name != "dF":
        assert torch.isfinite(got[5][b, t + 1:, h]).all()
    _compare(got, _chain(dk, x), b, h, tol, forward)


def test_bad_initial_state(dk):  # noqa: F811
    p = scalar_problem(5, 2, 40, 3, 64, 64)
    p["initial"][1, 2, 9, 30] = np.nan
    x = _x(p, torch.float32)
    got = _call(dk, x)
    _compare(got, _chain(dk, x), 1, 2, TOL_F32, True)
    assert torch.isfinite(got[0][1, :, 2, :30]).all()


def test_padding_is_not_read(dk):  # noqa: F811
    """Bad values on a padded token change nothing."""
    p = scalar_problem(6, 2, 40, 3, 64, 64)
    p["valid"][1, 18] = 0
    clean = _call(dk, _x(p, torch.float32))
    for n in ("q", "k", "v", "beta", "g", "dO", "dS"):
        p[n][1, 18] = np.nan
    for n, a, b in zip(NAMES, _call(dk, _x(p, torch.float32)), clean):
        assert torch.equal(a, b), n


def test_bad_upstream_over_two_windows(dk):  # noqa: F811
    """More chunks than the backward's workspace holds at once: the marks of all windows count, and
    the other heads keep their bits."""
    torch.manual_seed(3)
    B, T, H, D = 2, 4200, 8, 64
    r = lambda *s: torch.randn(*s, device="cuda")  # noqa: E731
    x = {n: torch.nn.functional.normalize(r(B, T, H, D), dim=-1) for n in ("q", "k", "v", "dO")}
    x.update(beta=torch.sigmoid(r(B, T, H)), g=-torch.nn.functional.softplus(r(B, T, H)),
             valid=torch.ones(B, T, device="cuda"), reset=torch.zeros(B, T, device="cuda"),
             initial=r(B, H, D, D), dF=r(B, H, D, D), dS=r(B, T, H))
    clean = _call(dk, x)
    for t in (7, 4100):  # of the last window, and of the first
        y = dict(x, dO=x["dO"].clone())
        y["dO"][1, t, 3, 5] = float("nan")
        got, want = _call(dk, y), _chain(dk, y)
        for n, a, c, w in zip(NAMES, got, clean, want):
            if n in ("output", "final", "scores"):
                assert torch.equal(a, c), n
                continue
            assert torch.allclose(_head(n, a, 1, 3), _head(n, w, 1, 3), rtol=1e-3, atol=1e-4,
                                  equal_nan=True), n
            a, c = a.clone(), c.clone()
            _head(n, a, 1, 3).zero_()
            _head(n, c, 1, 3).zero_()
            assert torch.equal(a, c), n


def test_replays(dk):  # noqa: F811
    """A captured call marks afresh on every replay."""
    p = scalar_problem(7, 2, 50, 3, 64, 64)
    x = _x(p, torch.float32)
    good, bad = x["k"].clone(), x["k"].clone()
    bad[0, 20, 1, 3] = float("nan")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        _call(dk, x)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _call(dk, x)
    for k in (good, bad, good, good, bad):
        x["k"].copy_(k)
        graph.replay()
        torch.cuda.synchronize()
        for n, a, w in zip(NAMES, got, _call(dk, x)):
            assert torch.allclose(a, w, rtol=0, atol=0, equal_nan=True), n
