"""The GDN-2 mixer around the scan (reference crates/mixers/src/lib.rs:205-262
construction, :434-693 forward), on the MI355X operators.

Per block input x [B, T, d_model] with masks valid/reset [B, T]:
  x <- x * valid;  documents = cumsum(reset * valid) over time       (lib.rs:447-455)
  q = l2(silu(conv(x Wq)))   k = l2(silu(conv(x Wk)))   v = silu(conv(x Wv))
  alpha = decay(x Wdecay, decay_bias, decay_scale)                    (lib.rs:460-503)
  erase = sigmoid(x Werase)   write = sigmoid(x Wwrite)              (lib.rs:504-523)
  out = scan(q, k, v, alpha, erase, write; valid, reset)             (lib.rs:524-565)
  y = rms_norm(out, norm_weight, gate = x Wgate, eps 1e-5) Wout * valid (lib.rs:661-693)
With cache_policy "surprise" or "recency" the mixer also reads the HOLA exact
cache (lib.rs:570-660): RMS-normed raw q and k (cache norms, eps 1e-5) attend to
the top-capacity tokens chosen by the scan's scores (or recency), and the read
joins the scan output scaled by sigmoid(cache gate) per head:
  out += hola_read(rms(q_raw), rms(k_raw), v, scores, ...) * sigmoid(gate)
The convolution fuses its SiLU (one pass over the projection), the gated RMSNorm
is one pass, and the recurrence is the HIP scan (channel-wise gates: the
16-token chunk kernels).  Projections are plain GEMMs (torch, hipBLASLt).
The reference's SBD block is not part of this module.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn.functional as F

import delta_kernels as dk


@dataclass
class GdnMixerConfig:
    d_model: int = 512
    heads: int = 8
    key_dim: int = 64
    value_dim: int = 64
    chunk_size: int = 16
    conv_taps: int = 4
    norm_epsilon: float = 1e-5  # burn RmsNormConfig default, the mixer's output norm
    cache_policy: str = "none"  # "none", "surprise" (scan scores) or "recency" (lib.rs:131-158)
    cache_capacity: int = 16


class _Projections(torch.autograd.Function):
    """x W_i^T for every weight [width_i, D], side by side on the last axis.  With a tuple of
    widths and a number behind the weights: the same columns in pieces of these widths, the last
    so many of them through a sigmoid."""

    @staticmethod
    def forward(ctx, x, *args):
        weights, pieces, gates = args, None, 0
        if not torch.is_tensor(args[-1]):
            *weights, pieces, gates = args
        ctx.extra, ctx.gates = len(args) - len(weights), gates
        z = F.linear(x, torch.cat(weights))
        if pieces is None:
            ctx.save_for_backward(x, *weights)
            return z
        out = z.split(pieces, -1)
        if gates:  # the last columns are one strided block
            n = sum(pieces[-gates:])
            z.narrow(-1, z.shape[-1] - n, n).sigmoid_()
        ctx.save_for_backward(x, *weights, *out[len(out) - gates:])
        return out

    @staticmethod
    def backward(ctx, *dz):
        x, *weights = ctx.saved_tensors
        if ctx.gates:
            weights, y = weights[:-ctx.gates], weights[-ctx.gates:]
            dz = dz[:-ctx.gates] + tuple(torch.ops.aten.sigmoid_backward(d, s)
                                         for d, s in zip(dz[-ctx.gates:], y))
        dz = dz[0] if len(dz) == 1 else torch.cat(dz, -1)
        widths = [w.shape[0] for w in weights]
        dz = dz.reshape(-1, dz.shape[-1])
        dx, need = None, ctx.needs_input_grad[1:1 + len(weights)]
        if ctx.needs_input_grad[0]:
            # One projection after another: a single product over all columns is a longer sum
            # in f32 (the pass's error against 64 bits rises from 2.1e-6 to 2.9e-6).
            for d, w in zip(dz.split(widths, 1), weights):
                dx = d @ w if dx is None else dx.addmm_(d, w)
            dx = dx.view(x.shape)
        x = x.reshape(-1, x.shape[-1])
        if not all(need):
            dw = [d.t() @ x if n else None for d, n in zip(dz.split(widths, 1), need)]
        else:
            # One product, then each weight's rows copied to memory of their own: a gradient that
            # is kept keeps no other.
            dw = torch._foreach_mul((dz.t() @ x).split(widths), 1.0)
        return (dx, *dw, *[None] * ctx.extra)


class GdnMixer(torch.nn.Module):
    """Parameters and initialisation follow lib.rs:216-235: bias-free linear
    projections, conv weights U(-0.1, 0.1) [taps, channels], decay_scale 0,
    decay_bias -4, output RMSNorm weight 1."""

    def __init__(self, cfg: GdnMixerConfig, device=None):
        super().__init__()
        self.cfg = cfg
        H, K, V, D = cfg.heads, cfg.key_dim, cfg.value_dim, cfg.d_model
        kw, vw = H * K, H * V

        def linear(i, o):
            w = torch.empty(o, i, device=device)
            torch.nn.init.kaiming_uniform_(w, a=5 ** 0.5)  # burn LinearConfig default init
            return torch.nn.Parameter(w)

        self.q = linear(D, kw)
        self.k = linear(D, kw)
        self.v = linear(D, vw)
        self.decay = linear(D, kw)
        self.erase = linear(D, kw)
        self.write = linear(D, vw)
        self.output_gate = linear(D, vw)
        self.output = linear(vw, D)
        conv = lambda c: torch.nn.Parameter(  # noqa: E731
            torch.empty(cfg.conv_taps, c, device=device).uniform_(-0.1, 0.1))
        self.q_conv, self.k_conv, self.v_conv = conv(kw), conv(kw), conv(vw)
        self.decay_scale = torch.nn.Parameter(torch.zeros(H, device=device))
        self.decay_bias = torch.nn.Parameter(torch.full((kw,), -4.0, device=device))
        self.norm_weight = torch.nn.Parameter(torch.ones(V, device=device))
        if cfg.cache_policy not in ("none", "surprise", "recency"):
            raise ValueError(f"unknown cache policy {cfg.cache_policy!r}")
        if cfg.cache_policy != "none":  # lib.rs:236-243
            self.cache_q_norm = torch.nn.Parameter(torch.ones(K, device=device))
            self.cache_k_norm = torch.nn.Parameter(torch.ones(K, device=device))
            self.cache_gate = torch.nn.Parameter(torch.full((H,), -4.0, device=device))
            self.cache_sink = torch.nn.Parameter(torch.zeros(H, device=device))

    def forward(self, x: torch.Tensor, valid: torch.Tensor = None,
                reset: torch.Tensor = None) -> torch.Tensor:
        cfg = self.cfg
        B, T, _ = x.shape
        H, K, V = cfg.heads, cfg.key_dim, cfg.value_dim
        if valid is None:
            valid = torch.ones(B, T, device=x.device)
        if reset is None:
            reset = torch.zeros(B, T, device=x.device)
        valid, reset = valid.float(), reset.float()
        x = x * valid[..., None]
        docs = torch.cumsum(reset * valid, dim=1)

        # One GEMM for the seven projections (erase and write leave it as sigmoids: the products
        # themselves are not kept), one convolution for q, k and v, one L2 norm for q and k: the
        # host took longer to launch them one by one (66 kernels, 1.6 ms a training pass at
        # 8 x 512 tokens) than they ran.  Every operator reads its columns in place.
        kw, vw = H * K, H * V
        qkv, z_decay, z_gate, erase, write = _Projections.apply(
            x, self.q, self.k, self.v, self.decay, self.output_gate, self.erase, self.write,
            (2 * kw + vw, kw, vw, kw, vw), 2)
        qkv = dk.causal_conv(qkv, torch.cat([self.q_conv, self.k_conv, self.v_conv], 1), valid,
                             docs, activation="silu")
        qk, v = qkv.split([2 * kw, vw], -1)
        raw_q, raw_k = qk.view(B, T, 2, H, K).unbind(2)
        q, k = dk.l2_norm(qk.view(B, T, 2 * H, K)).view(B, T, 2, H, K).unbind(2)
        v = v.view(B, T, H, V)
        alpha = dk.decay(z_decay.view(B, T, H, K), self.decay_bias, self.decay_scale)
        erase, write = erase.view(B, T, H, K), write.view(B, T, H, V)
        scan = dk.gdn_training_scan(q, k, v, alpha, erase, write, valid, reset, None,
                                    cfg.chunk_size)
        out = scan.output
        if cfg.cache_policy != "none":
            exact = dk.hola_read(dk.rms_norm(raw_q, self.cache_q_norm, None, cfg.norm_epsilon),
                                 dk.rms_norm(raw_k, self.cache_k_norm, None, cfg.norm_epsilon),
                                 v, scan.scores, valid, docs, self.cache_sink,
                                 cfg.cache_capacity, cfg.chunk_size,
                                 cfg.cache_policy == "recency").output
            out = out + exact * torch.sigmoid(self.cache_gate).view(1, 1, H, 1)
        mixed = dk.rms_norm(out, self.norm_weight, z_gate.view(B, T, H, V),
                            cfg.norm_epsilon).reshape(B, T, H * V)
        return F.linear(mixed, self.output) * valid[..., None]
