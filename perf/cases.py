"""Performance cases: the calls a program makes of this framework, with the sizes, types and
options it makes them with.  listed() holds the named cases, draw() gives more of the same
ranges; prepare() makes what the caller has in hand, run() is one call (with its backward
where the caller trains), exact() the same results in float64 from plain torch.

Kinds:
  scalar    the gated delta rule with one decay and one write strength per token and head (the
            language model's mixer): forward + backward (the two raw calls the model's fused
            block makes, or the autograd function) or the forward alone (prefill, evaluation)
  channel   the GDN-2 training scan with channel-wise gates, padding and resets
  document  the document-limit scan over packed documents
  decode    one token for every carried state
  hola      the exact-memory cache read over the scan's scores, with its gradients
  mixer     the whole GDN-2 mixer module in float32, forward and backward
  lm        the language model: loss and gradients of one training step, or logits
"""
import math
import os
import sys

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "delta-block-lm_amd"))
import delta_kernels as dk  # noqa: E402
from delta_mixers.mixer import GdnMixer, GdnMixerConfig  # noqa: E402
from delta_mixers.model import GdnLM, GdnLMConfig  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _scan(name, kind, dtype, batch, time, heads, keys, values, mode, **more):
    return dict(name=name, kind=kind, dtype=dtype, batch=batch, time=time, heads=heads, keys=keys,
                values=values, mode=mode, **more)


def listed():
    return [
        # One layer's scan of the lm512 language model (16 x 512 tokens, 8 heads of 64).
        _scan("scalar_lm512", "scalar", "bf16", 16, 512, 8, 64, 64, "raw"),
        # Long-context training: 4 x 8192 tokens, 16 heads of 128.
        _scan("scalar_long8k", "scalar", "bf16", 4, 8192, 16, 128, 128, "raw"),
        # The same mixer trained in float32.
        _scan("scalar_f32", "scalar", "f32", 8, 512, 8, 64, 64, "grad"),
        # Prefill of one prompt of ragged length on a carried state, no gradients.
        _scan("scalar_prefill", "scalar", "bf16", 1, 3001, 8, 64, 64, "forward", initial=True),
        # The reference's isolated-scan benchmark, its largest and its smallest shape.
        _scan("channel_ref", "channel", "f32", 8, 512, 4, 32, 64, "grad", initial=True),
        _scan("channel_ref_small", "channel", "f32", 1, 128, 4, 32, 64, "grad", initial=True),
        # Channel-wise gates in bf16, padded and reset sequences of ragged length, chained: an
        # initial state in, a gradient of the final state back.
        _scan("channel_bf16", "channel", "bf16", 16, 509, 8, 64, 64, "grad", initial=True,
              final_grad=True),
        # Packed documents of 16 to 200 tokens.
        _scan("document_packed", "document", "bf16", 16, 512, 8, 64, 64, "grad"),
        # Serving: one token on 256 x 8 carried states.
        dict(name="decode", kind="decode", dtype="f32", batch=256, heads=8, keys=64, values=64),
        # The cache read at the lm512 head shape.
        dict(name="hola_lm512", kind="hola", batch=16, time=512, heads=8, keys=64, values=64,
             capacity=64, chunk=16, recency=False),
        # One mixer layer (d_model 512, 8 heads of 64) on padded, packed sequences.
        dict(name="mixer_layer", kind="mixer", batch=8, time=512, d_model=512, heads=8, keys=64,
             values=64, cache="none"),
        # Loss and gradients of a two-block lm512 model.
        dict(name="lm_step", kind="lm", mode="step", batch=16, time=512, layers=2, d_model=512,
             heads=8, mlp=1408, vocab=32768),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["scalar", "scalar", "scalar", "channel", "channel", "channel", "document",
                       "decode", "hola", "mixer", "lm"])
    if kind == "decode":
        w = rng.choice([32, 64, 64, 128])
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), batch=_log(rng, 1, 512),
                    heads=rng.choice([4, 8, 16]), keys=w, values=rng.choice([w, 64]))
    if kind == "lm":
        d = rng.choice([256, 512])
        return dict(kind=kind, mode=rng.choice(["step", "logits"]), batch=_log(rng, 1, 16),
                    time=_log(rng, 33, 512), layers=rng.choice([1, 2]), d_model=d,
                    heads=rng.choice([4, 8]), mlp=rng.choice([d * 2, 1408]),
                    vocab=rng.choice([4096, 32768]))
    if kind == "mixer":
        return dict(kind=kind, batch=_log(rng, 1, 8), time=_log(rng, 32, 600), d_model=512,
                    heads=rng.choice([4, 8]), keys=rng.choice([32, 64]), values=64,
                    cache=rng.choice(["none", "surprise"]))
    if kind == "hola":
        return dict(kind=kind, batch=_log(rng, 1, 16), time=_log(rng, 64, 1100),
                    heads=rng.choice([4, 8]), keys=rng.choice([32, 64]), values=64,
                    capacity=rng.choice([16, 64]), chunk=16, recency=rng.random() < 0.3)
    heads = rng.choice([4, 8, 16])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    mode = rng.choice(["grad", "grad", "forward"])
    if kind == "scalar":
        if dtype == "bf16":
            keys, values = rng.choice([(64, 64), (64, 64), (128, 128), (96, 96), (64, 128)])
            most = 1 << 17 if (keys, values) in ((64, 64), (128, 128)) else 1 << 13
            mode = rng.choice(["raw", "raw", "forward"])
        else:
            keys, values = rng.choice([(32, 64), (64, 64), (96, 96), (128, 128), (33, 40)])
            most = 1 << 13
    elif dtype == "bf16":
        keys, values = rng.choice([(64, 64), (64, 64), (64, 64), (128, 128), (32, 64)])
        most = 1 << 14 if (keys, values) == (64, 64) else 1 << 13
    else:
        keys, values = rng.choice([(32, 64), (32, 64), (64, 64), (128, 128), (48, 33)])
        most = 1 << 13
    if kind == "document":
        mode = "grad"
    time = _log(rng, 32, 8192 if most > 1 << 13 else 1024)
    batch = _log(rng, 1, max(1, min(32, most // (time * max(1, heads // 4)))))
    case = dict(kind=kind, dtype=dtype, batch=batch, time=time, heads=heads, keys=keys,
                values=values, mode=mode)
    if kind != "document" and rng.random() < 0.5:
        case["initial"] = True
    return case


# ---- inputs ----------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7fffffff)
    return g


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _documents(gen, B, T, lo=16, hi=200):
    """First position of each token's document: documents of lo..hi tokens back to back."""
    n = -(-T // lo)
    ends = torch.randint(lo, hi + 1, (B, n), generator=gen, device="cuda").cumsum(1)
    t = torch.arange(T, device="cuda").expand(B, T).contiguous()
    doc = torch.searchsorted(ends, t, right=True)
    starts = torch.cat([torch.zeros_like(ends[:, :1]), ends], 1)
    first = torch.gather(starts, 1, doc)
    last = torch.clamp(torch.gather(starts, 1, doc + 1) - 1, max=T - 1)
    return doc, first, last


def _lengths(gen, B, T):
    """Valid lengths of a padded batch: the longest fills it."""
    n = torch.randint(max(1, T - T // 4), T + 1, (B,), generator=gen, device="cuda")
    n[0] = T
    return (torch.arange(T, device="cuda")[None] < n[:, None])


def _scan_inputs(case, seed):
    gen = _gen(seed)
    B, T, H, K, V = (case[n] for n in ("batch", "time", "heads", "keys", "values"))
    dt = DTYPES[case["dtype"]]
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x = {"q": _unit(r(B, T, H, K)).to(dt), "k": _unit(r(B, T, H, K)).to(dt),
         "v": r(B, T, H, V).to(dt)}
    if case["kind"] == "scalar":
        # One decay rate per head, from nearly none to a few tokens' memory.
        bias = torch.rand(H, generator=gen, device="cuda") * 6 - 5
        x["beta"] = torch.sigmoid(r(B, T, H))
        x["g"] = -F.softplus(r(B, T, H) + bias)
    else:
        bias = torch.rand(H, K, generator=gen, device="cuda") * 6 - 6
        x["alpha"] = torch.exp(-F.softplus(r(B, T, H, K) + bias))
        x["erase"] = torch.sigmoid(r(B, T, H, K))
        x["write"] = torch.sigmoid(r(B, T, H, V))
    if case["kind"] == "document":
        _, first, last = _documents(gen, B, T)
        live = _lengths(gen, B, T)
        last = torch.minimum(last, live.sum(1, keepdim=True) - 1)
        x["start"] = torch.where(live, first, 1).to(torch.int32)
        x["end"] = torch.where(live, last, 0).to(torch.int32)
    elif case["kind"] == "channel":
        doc, first, _ = _documents(gen, B, T)
        x["valid"] = _lengths(gen, B, T).float()
        x["reset"] = ((first == torch.arange(T, device="cuda")) & (doc > 0)).float()
    else:
        x["valid"] = torch.ones(B, T, device="cuda")
        x["reset"] = torch.zeros(B, T, device="cuda")
    x["initial"] = 0.3 * r(B, H, K, V) if case.get("initial") else None
    x["d_output"] = r(B, T, H, V).to(dt)
    x["d_final"] = r(B, H, K, V) if case.get("final_grad") else None
    return x


def _hola_inputs(case, seed):
    gen = _gen(seed)
    B, T, H, K, V = (case[n] for n in ("batch", "time", "heads", "keys", "values"))
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    doc, _, _ = _documents(gen, B, T)
    return {"q": r(B, T, H, K), "k": r(B, T, H, K), "v": r(B, T, H, V), "sink": 0.5 * r(H),
            "scores": torch.empty(B, T, H, device="cuda").exponential_(generator=gen),
            "valid": _lengths(gen, B, T).float(), "documents": doc.float(),
            "d_output": r(B, T, H, V)}


def _mixer_inputs(case, seed):
    gen = _gen(seed)
    torch.manual_seed(seed & 0x7fffffff)
    B, T = case["batch"], case["time"]
    m = GdnMixer(GdnMixerConfig(d_model=case["d_model"], heads=case["heads"],
                                key_dim=case["keys"], value_dim=case["values"],
                                cache_policy=case["cache"]), device="cuda")
    doc, first, _ = _documents(gen, B, T)
    x = torch.randn(B, T, case["d_model"], generator=gen, device="cuda")
    return {"mixer": m, "x": x, "valid": _lengths(gen, B, T).float(),
            "reset": ((first == torch.arange(T, device="cuda")) & (doc > 0)).float(),
            "dy": torch.randn(x.shape, generator=gen, device="cuda")}


def _lm_inputs(case, seed):
    torch.manual_seed(seed & 0x7fffffff)
    cfg = GdnLMConfig(vocab=case["vocab"], d_model=case["d_model"], layers=case["layers"],
                      heads=case["heads"], mlp_width=case["mlp"])
    model = GdnLM(cfg, device="cuda")
    more = 1 if case["mode"] == "step" else 0
    tokens = torch.randint(0, case["vocab"], (case["batch"], case["time"] + more),
                           generator=_gen(seed), device="cuda")
    return {"model": model, "tokens": tokens}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        one = dict(case, kind="channel", time=1, initial=True)
        s = _scan_inputs(one, seed)
        s["state"] = s["initial"]
        s["valid"], s["reset"] = torch.ones_like(s["valid"]), torch.zeros_like(s["reset"])
    elif kind == "hola":
        s = _hola_inputs(case, seed)
        for n in ("q", "k", "v", "sink"):
            s[n].requires_grad_(True)
    elif kind == "mixer":
        s = _mixer_inputs(case, seed)
        s["x"].requires_grad_(True)
    elif kind == "lm":
        s = _lm_inputs(case, seed)
    else:
        s = _scan_inputs(case, seed)
        if case["mode"] == "grad":
            for n in ("q", "k", "v", "beta", "g", "alpha", "erase", "write", "initial"):
                if s.get(n) is not None:
                    s[n].requires_grad_(True)
    s["case"] = dict(case)
    return s


# ---- one pass ----------------------------------------------------------------------------


def _grads(s, outputs, upstream, names):
    ins = [s[n] for n in names if s.get(n) is not None]
    got = torch.autograd.grad(outputs, ins, upstream)
    return dict(zip(["d" + n for n in names if s.get(n) is not None], got))


def _run_scalar(s, mode):
    a = [s[n] for n in ("q", "k", "v", "beta", "g", "valid", "reset")]
    if mode == "forward":
        with torch.no_grad():
            out, fin, sc = dk.gdn_scalar_scan(*a, s["initial"])
        return {"output": out, "final": fin, "scores": sc}
    if mode == "raw":
        out, fin, sc, ck = dk.gdn_scalar_forward(*a, s["initial"], 64)
        g = dk.gdn_scalar_backward(*a, ck, 64, s["d_output"])
        return {"output": out, "final": fin, "scores": sc, "dq": g[0], "dk": g[1], "dv": g[2],
                "dbeta": g[3], "dg": g[4], "dinitial": g[5]}
    out, fin, sc = dk.gdn_scalar_scan(*a, s["initial"])
    r = _grads(s, [out], [s["d_output"]], ("q", "k", "v", "beta", "g", "initial"))
    return {"output": out, "final": fin, "scores": sc, **r}


def _run_channel(s, mode):
    a = [s[n] for n in ("q", "k", "v", "alpha", "erase", "write", "valid", "reset", "initial")]
    if mode == "forward":
        with torch.no_grad():
            r = dk.gdn_training_scan(*a, chunk_size=16)
        return {"output": r.output, "final": r.final_state, "scores": r.scores}
    r = dk.gdn_training_scan(*a, chunk_size=16)
    outs, ups = [r.output], [s["d_output"]]
    if s["d_final"] is not None:
        outs, ups = outs + [r.final_state], ups + [s["d_final"]]
    g = _grads(s, outs, ups, ("q", "k", "v", "alpha", "erase", "write", "initial"))
    return {"output": r.output, "final": r.final_state, "scores": r.scores, **g}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "scalar":
        return _run_scalar(s, case["mode"])
    if kind == "channel":
        return _run_channel(s, case["mode"])
    if kind == "document":
        names = ("q", "k", "v", "alpha", "erase", "write")
        out = dk.gdn2_scan(*[s[n] for n in names], s["start"], s["end"])
        return {"output": out, **_grads(s, [out], [s["d_output"]], names)}
    if kind == "decode":
        out, sc = dk.gdn_decode_step(s["state"], s["q"], s["k"], s["v"], s["alpha"], s["erase"],
                                     s["write"], s["valid"], s["reset"])
        return {"output": out, "scores": sc, "state": s["state"]}
    if kind == "hola":
        r = dk.hola_read(s["q"], s["k"], s["v"], s["scores"], s["valid"], s["documents"],
                         s["sink"], case["capacity"], case["chunk"], case["recency"], True)
        g = _grads(s, [r.output], [s["d_output"]], ("q", "k", "v", "sink"))
        return {"output": r.output, "positions": r.final_positions, **g}
    if kind == "mixer":
        m, names = s["mixer"], [n for n, _ in s["mixer"].named_parameters()]
        y = m(s["x"], s["valid"], s["reset"])
        g = torch.autograd.grad(y, [s["x"]] + list(m.parameters()), s["dy"])
        return {"y": y, "dx": g[0], **{"d" + n: t for n, t in zip(names, g[1:])}}
    model = s["model"]
    if case["mode"] == "logits":
        with torch.no_grad():
            return {"logits": model(s["tokens"])}
    model.zero_grad(set_to_none=True)
    loss = model.loss(s["tokens"])
    loss.backward()
    return {"loss": loss.detach(), **{"d" + n: p.grad for n, p in model.named_parameters()}}


# ---- what a pass cannot do without ---------------------------------------------------------


def work(case):
    kind, B, H = case["kind"], case["batch"], case["heads"]
    if kind == "lm":
        D, M, L, W, T = (case[n] for n in ("d_model", "mlp", "layers", "vocab", "time"))
        block = D * (4 * H * 64 + 2 * H) + H * 64 * D + 3 * D * M
        weights = L * block + W * D
        rows = B * T
        if case["mode"] == "logits":
            return {"bytes": 4 * weights + 2 * rows * W + 8 * rows,
                    "flops": 2 * rows * weights + L * rows * H * 6 * 64 * 64}
        return {"bytes": 8 * weights + 8 * rows,
                "flops": 6 * rows * weights + L * rows * H * 18 * 64 * 64}
    K, V = case["keys"], case["values"]
    if kind == "mixer":
        T, D = case["time"], case["d_model"]
        weights = D * H * (4 * K + 3 * V) + H * V * D
        return {"bytes": 4 * (4 * B * T * D + 2 * weights),
                "flops": 6 * B * T * weights + 18 * B * T * H * K * V}
    if kind == "hola":
        n, slots = B * case["time"] * H, case["capacity"] + case["chunk"] // 2
        return {"bytes": 4 * n * (4 * K + 4 * V + 1),
                "flops": n * slots * (6 * K + 4 * V)}
    s = 2 if case["dtype"] == "bf16" else 4
    if kind == "decode":
        n = B * H
        return {"bytes": n * (8 * K * V + s * (2 * K + 2 * V) + 4 * (2 * K + V) + 4),
                "flops": 6 * n * K * V}
    n = B * case["time"] * H
    gates = 2 if kind == "scalar" else 2 * K + V
    state = 4 * B * H * K * V
    forward = n * (s * (2 * K + 2 * V) + 4 * gates + 4) + state * (2 if case.get("initial") else 1)
    if case["mode"] == "forward":
        return {"bytes": forward, "flops": 6 * n * K * V}
    backward = n * (s * (2 * K + 2 * V) + 4 * gates) + (state if case.get("initial") else 0)
    return {"bytes": forward + backward, "flops": 18 * n * K * V}


def tolerance(case):
    """About four times what the outputs are off exact(): 1.7e-3 to 1.9e-3 in bf16 (its rounding),
    up to 1.6e-6 in float32, up to 3.4e-2 for the gradients of a bf16 model (two versions of one
    rounding are nearer to each other than that)."""
    kind = case["kind"]
    if kind == "lm":
        return {"rel": 0.03}
    if kind in ("hola", "mixer") or case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 8e-3}


# ---- the same in float64, from plain torch --------------------------------------------------


def _d(t):
    return None if t is None else t.detach().double()


def _steps(S, q, k, v, alpha, erase, write, live, fresh):
    """A run of tokens of the recurrence, token by token."""
    outs, norms = [], []
    for t in range(q.shape[1]):
        lv = live[:, t, None, None, None]
        bar = alpha[:, t, :, :, None] * (S * (1 - lv * fresh[:, t, None, None, None]))
        delta = write[:, t] * v[:, t] - ((erase[:, t] * k[:, t])[..., None] * bar).sum(-2)
        new = bar + k[:, t][..., None] * delta[..., None, :]
        outs.append((new * q[:, t][..., None]).sum(-2) * lv[..., 0])
        norms.append((k[:, t].detach().norm(dim=-1) * delta.detach().norm(dim=-1)) * lv[..., 0, 0])
        S = torch.where(lv > 0, new, S)
    return S, torch.stack(outs, 1), torch.stack(norms, 1)


def _scan64(q, k, v, alpha, erase, write, live, fresh, S):
    outs, norms = [], []
    for t in range(0, q.shape[1], 64):
        part = [x[:, t:t + 64] for x in (q, k, v, alpha, erase, write, live, fresh)]
        if torch.is_grad_enabled():
            S, o, n = checkpoint(_steps, S, *part, use_reentrant=False)
        else:
            S, o, n = _steps(S, *part)
        outs.append(o)
        norms.append(n)
    return torch.cat(outs, 1), S, torch.cat(norms, 1)


def _scan_exact(case, seed):
    x = _scan_inputs(case, seed)
    train = case.get("mode") not in (None, "forward")
    names = [n for n in ("q", "k", "v", "beta", "g", "alpha", "erase", "write") if n in x]
    y = {n: _d(x[n]).requires_grad_(train) for n in names}
    B, T, H, K = x["q"].shape
    V = x["v"].shape[3]
    S0 = _d(x["initial"])
    if S0 is None:
        S0 = torch.zeros(B, H, K, V, dtype=torch.float64, device="cuda")
    S0.requires_grad_(train)
    if case["kind"] == "scalar":
        alpha = torch.exp(y["g"])[..., None].expand(B, T, H, K)
        erase = y["beta"][..., None].expand(B, T, H, K)
        write = y["beta"][..., None].expand(B, T, H, V)
    else:
        alpha, erase, write = y["alpha"], y["erase"], y["write"]
    if case["kind"] == "document":
        live = (x["end"] >= x["start"]).double()
        fresh = (x["start"] == torch.arange(T, device="cuda")).double()
    else:
        live, fresh = _d(x["valid"]), _d(x["reset"])
    with torch.set_grad_enabled(train):
        out, fin, sc = _scan64(y["q"], y["k"], y["v"], alpha, erase, write, live, fresh, S0)
    r = {"output": out.detach()}
    if case["kind"] != "document":
        r.update(final=fin.detach(), scores=sc if case["kind"] == "scalar" else sc[..., None])
    if train:
        total = (out * _d(x["d_output"])).sum()
        if x["d_final"] is not None:
            total = total + (fin * _d(x["d_final"])).sum()
        g = torch.autograd.grad(total, [y[n] for n in names] + [S0])
        r.update({"d" + n: t for n, t in zip(names, g)})
        if case["mode"] == "raw" or case.get("initial"):
            r["dinitial"] = g[-1]
    return r


def _decode_exact(case, seed):
    one = dict(case, kind="channel", time=1, initial=True)
    x = _scan_inputs(one, seed)
    live = torch.ones(case["batch"], 1, dtype=torch.float64, device="cuda")
    a = [_d(x[n]) for n in ("q", "k", "v", "alpha", "erase", "write")]
    S, out, sc = _steps(_d(x["initial"]), *a, live, torch.zeros_like(live))
    return {"output": out, "scores": sc, "state": S}


def _hola64(q, k, v, scores, valid, docs, sink, capacity, chunk, recency):
    B, T, H, K = q.shape
    V = v.shape[3]
    live = valid >= 0.5
    cache = torch.full((B, H, capacity), T, dtype=torch.int64, device=q.device)  # T: empty
    pad = lambda x, fill: torch.cat([x, torch.full_like(x[:, :1], fill)], 1)  # noqa: E731
    kp, vp, sp = (pad(x, 0).transpose(1, 2) for x in (k, v, scores))  # [B, H, T + 1, ...]
    lp, dp = pad(live, False), pad(docs, -1)
    outs = []
    for f in range(0, T, chunk):
        e = min(T, f + chunk)
        own = torch.arange(f, e, device=q.device)
        slots = torch.cat([cache, own.expand(B, H, e - f)], 2)                     # [B, H, n]
        n = slots.shape[2]
        ks = torch.gather(kp, 2, slots[..., None].expand(B, H, n, K))
        vs = torch.gather(vp, 2, slots[..., None].expand(B, H, n, V))
        flat = slots.reshape(B, H * n)
        ls = torch.gather(lp, 1, flat).view(B, H, n)
        ds = torch.gather(dp, 1, flat).view(B, H, n)
        see = (ls[:, :, None] & (ds[:, :, None] == docs[:, None, f:e, None])
               & (slots[:, :, None] <= own[None, None, :, None]))
        logits = torch.matmul(q[:, f:e].transpose(1, 2), ks.transpose(2, 3).contiguous())
        logits = (logits / K ** 0.5).masked_fill(~see, -math.inf)
        logits = torch.cat([logits, sink.view(1, H, 1, 1).expand(B, H, e - f, 1)], 3)
        p = torch.softmax(logits, -1)[..., :-1]
        outs.append((torch.matmul(p, vs) * live[:, None, f:e, None]).transpose(1, 2))
        order = torch.sort(slots, dim=2).values
        flat = order.reshape(B, H * n)
        fit = (torch.gather(lp, 1, flat) & (torch.gather(dp, 1, flat) == docs[:, e - 1:e])).view(
            B, H, n)
        rank = order.double() if recency else torch.gather(sp.detach(), 2, order)
        rank = rank.masked_fill(~fit, -math.inf)
        best = torch.sort(rank, dim=2, descending=True, stable=True).indices[..., :capacity]
        kept = torch.where(torch.gather(fit, 2, best), torch.gather(order, 2, best), T)
        cache = torch.full_like(cache, T)
        cache[..., :kept.shape[2]] = kept
    return torch.cat(outs, 1), torch.where(cache < T, cache, -1).double()


def _hola_exact(case, seed):
    x = {n: _d(t) for n, t in _hola_inputs(case, seed).items()}
    names = ("q", "k", "v", "sink")
    for n in names:
        x[n].requires_grad_(True)
    out, pos = _hola64(x["q"], x["k"], x["v"], x["scores"], x["valid"], x["documents"], x["sink"],
                       case["capacity"], case["chunk"], case["recency"])
    g = torch.autograd.grad((out * x["d_output"]).sum(), [x[n] for n in names])
    return {"output": out.detach(), "positions": pos, **{"d" + n: t for n, t in zip(names, g)}}


def _conv64(x, w, valid, docs):
    y = 0
    T = x.shape[1]
    for lag in range(w.shape[0]):
        if lag >= T:
            break
        m = valid[:, lag:] * valid[:, :T - lag] * (docs[:, lag:] == docs[:, :T - lag])
        y = y + F.pad(x[:, :T - lag] * m[..., None], (0, 0, lag, 0)) * w[lag]
    return F.silu(y)


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _l264(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _mixer_exact(case, seed):
    s = _mixer_inputs(case, seed)
    B, T, H, K, V = (case[n] for n in ("batch", "time", "heads", "keys", "values"))
    names = [n for n, _ in s["mixer"].named_parameters()]
    p = {n: _d(t).requires_grad_(True) for n, t in s["mixer"].named_parameters()}
    x0 = _d(s["x"]).requires_grad_(True)
    valid, reset = _d(s["valid"]), _d(s["reset"])
    x = x0 * valid[..., None]
    docs = torch.cumsum(reset * valid, 1)
    raw_q = _conv64(F.linear(x, p["q"]), p["q_conv"], valid, docs).view(B, T, H, K)
    raw_k = _conv64(F.linear(x, p["k"]), p["k_conv"], valid, docs).view(B, T, H, K)
    v = _conv64(F.linear(x, p["v"]), p["v_conv"], valid, docs).view(B, T, H, V)
    z = (F.linear(x, p["decay"]) + p["decay_bias"]).view(B, T, H, K)
    alpha = torch.exp(-torch.exp(p["decay_scale"])[:, None] * F.softplus(z, threshold=20.0))
    erase = torch.sigmoid(F.linear(x, p["erase"])).view(B, T, H, K)
    write = torch.sigmoid(F.linear(x, p["write"])).view(B, T, H, V)
    S0 = torch.zeros(B, H, K, V, dtype=torch.float64, device="cuda")
    out, _, sc = _scan64(_l264(raw_q), _l264(raw_k), v, alpha, erase, write, valid, reset, S0)
    if case["cache"] != "none":
        read, _ = _hola64(_rms64(raw_q, p["cache_q_norm"], 1e-5),
                          _rms64(raw_k, p["cache_k_norm"], 1e-5), v, sc, valid, docs,
                          p["cache_sink"], 16, 16, False)
        out = out + read * torch.sigmoid(p["cache_gate"]).view(1, 1, H, 1)
    gate = torch.sigmoid(F.linear(x, p["output_gate"])).view(B, T, H, V)
    y = _rms64(out * gate, p["norm_weight"], 1e-5).reshape(B, T, H * V)
    y = F.linear(y, p["output"]) * valid[..., None]
    g = torch.autograd.grad((y * _d(s["dy"])).sum(), [x0] + [p[n] for n in names])
    return {"y": y.detach(), "dx": g[0], **{"d" + n: t for n, t in zip(names, g[1:])}}


def _lm_block64(x, p, n, H, M, eps):
    B, T, _ = x.shape
    W = H * 64
    ones = torch.ones(B, T, dtype=torch.float64, device="cuda")
    z = F.linear(_rms64(x, p[n + "norm1"], eps), p[n + "mixer.in_proj"])
    qkv = _conv64(z[..., :3 * W], p[n + "mixer.qkv_conv"], ones, torch.zeros_like(ones))
    q, k, v = (t.reshape(B, T, H, 64) for t in qkv.split(W, -1))
    gate, beta, dec = z[..., 3 * W:].split([W, H, H], -1)
    g = -torch.exp(p[n + "mixer.decay_scale"]) * F.softplus(dec + p[n + "mixer.decay_bias"])
    wide = lambda t: t[..., None].expand(B, T, H, 64)  # noqa: E731
    beta = wide(torch.sigmoid(beta))
    S0 = torch.zeros(B, H, 64, 64, dtype=torch.float64, device="cuda")
    o, _, _ = _scan64(_l264(q), _l264(k), v, wide(torch.exp(g)), beta, beta, ones,
                      torch.zeros_like(ones), S0)
    o = _rms64(o, p[n + "mixer.norm_weight"], eps).reshape(B, T, W) * F.silu(gate)
    x = x + F.linear(o, p[n + "mixer.out"])
    h = F.linear(_rms64(x, p[n + "norm2"], eps), p[n + "mlp.w13"])
    return x + F.linear(F.silu(h[..., :M]) * h[..., M:], p[n + "mlp.w2"])


def _lm_exact(case, seed):
    s = _lm_inputs(case, seed)
    model, tokens = s["model"], s["tokens"]
    train = case["mode"] == "step"
    p = {n: _d(t).requires_grad_(train) for n, t in model.named_parameters()}
    eps = model.cfg.norm_epsilon
    with torch.set_grad_enabled(train):
        x = F.embedding(tokens[:, :-1] if train else tokens, p["embed"])
        for i in range(case["layers"]):
            x = _lm_block64(x, p, "blocks.%d." % i, case["heads"], case["mlp"], eps)
        logits = F.linear(_rms64(x, p["norm"], eps), p["embed"])
        if not train:
            return {"logits": logits}
        loss = F.cross_entropy(logits.flatten(0, 1), tokens[:, 1:].flatten())
        g = torch.autograd.grad(loss, list(p.values()))
    return {"loss": loss.detach(), **{"d" + n: t for n, t in zip(p, g)}}


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _decode_exact(case, seed)
    if kind == "hola":
        return _hola_exact(case, seed)
    if kind == "mixer":
        return _mixer_exact(case, seed)
    if kind == "lm":
        return _lm_exact(case, seed)
    return _scan_exact(case, seed)
