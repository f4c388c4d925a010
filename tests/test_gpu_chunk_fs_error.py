"""The f32 scalar-gate chunk kernels lose no precision against the token walk: both
against the f64 oracle, the walk as a chain of 16-token calls (calls that short walk
their tokens), its backward from the last to the first.

Gate: 1.1 times the walk's normwise error of each result, both as means over the seeds
(the errors of one seed scatter by up to a third with the slowest head's decay).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gpu_util import dev, host  # noqa: E402
from test_gpu_chunk_fs import dk  # noqa: E402,F401
from test_gpu_scalar_decode import scalar_oracle  # noqa: E402

pytestmark = pytest.mark.gpu

NAMES = ("output", "final", "scores", "dq", "dk", "dv", "dbeta", "dg", "dinitial")
STEP = 16


def _problem(seed, B, T, H, K, V):
    rng = np.random.default_rng(seed)
    unit = lambda x: x / np.linalg.norm(x, axis=-1, keepdims=True)  # noqa: E731
    f = lambda x: np.ascontiguousarray(x, np.float32)  # noqa: E731
    bias = rng.random(H) * 6 - 5  # a decay rate a head, from nearly none to a few tokens' memory
    return dict(q=f(unit(rng.normal(size=(B, T, H, K)))), k=f(unit(rng.normal(size=(B, T, H, K)))),
                v=f(rng.normal(size=(B, T, H, V))),
                beta=f(1 / (1 + np.exp(-rng.normal(size=(B, T, H))))),
                g=f(-np.log1p(np.exp(rng.normal(size=(B, T, H)) + bias))),
                valid=np.ones((B, T), np.float32), reset=np.zeros((B, T), np.float32),
                initial=f(0.3 * rng.normal(size=(B, H, K, V))), dO=f(rng.normal(size=(B, T, H, V))),
                dF=f(rng.normal(size=(B, H, K, V))), dS=f(rng.normal(size=(B, T, H))))


def _walk(dk, x, initial, dF):  # noqa: F811
    T = x[0].shape[1]
    cuts = [slice(t, min(t + STEP, T)) for t in range(0, T, STEP)]
    parts = [[t[:, c] for t in x] for c in cuts]
    outs, state = [], initial
    for p in parts:
        out, state, sc, ck = dk.gdn_scalar_forward(*p[:7], state, 64)
        outs.append((out, sc, ck))
    grads, d = [], dF
    for p, o in zip(reversed(parts), reversed(outs)):
        g = dk.gdn_scalar_backward(*p[:7], o[2], 64, p[7].contiguous(), d, p[8].contiguous())
        d = g[5]
        grads.append(g[:5])
    cat = lambda ts: torch.cat(list(ts), 1)  # noqa: E731
    return [cat(o[0] for o in outs), state, cat(o[1] for o in outs),
            *(cat(g[i] for g in reversed(grads)) for i in range(5)), d]


@pytest.mark.parametrize("K,V", [(64, 64), (128, 128), (32, 64)])
def test_no_less_exact_than_the_token_walk(dk, K, V):  # noqa: F811
    chunked, walked = np.zeros(len(NAMES)), np.zeros(len(NAMES))
    for seed in range(4):
        p = _problem(seed, 1, 512, 8, K, V)
        x = [dev(p[n]) for n in ("q", "k", "v", "beta", "g", "valid", "reset", "dO", "dS")]
        initial, dF = dev(p["initial"]), dev(p["dF"])
        out, fin, sc, ck = dk.gdn_scalar_forward(*x[:7], initial, 64)
        got = [out, fin, sc, *dk.gdn_scalar_backward(*x[:7], ck, 64, x[7], dF, x[8])]
        o_out, o_fin, o_sc, og, odb, odg = scalar_oracle(p)
        ref = [o_out, o_fin, o_sc, og["q"], og["k"], og["v"], odb, odg, og["initial"]]
        err = lambda ts: np.array([np.linalg.norm(host(t).reshape(r.shape) - r)  # noqa: E731
                                   / np.linalg.norm(r) for t, r in zip(ts, ref)])
        chunked += err(got)
        walked += err(_walk(dk, x, initial, dF))
    print("\n" + "\n".join(f"{n}: chunked {c / 4:.3e} walk {w / 4:.3e}"
                           for n, c, w in zip(NAMES, chunked, walked)))
    bad = [n for n, c, w in zip(NAMES, chunked, walked) if c > 1.1 * w]
    assert not bad, bad
