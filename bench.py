#!/usr/bin/env python3
"""GDN scan forward+backward throughput on one MI355X.

Workload: the "lm512" scan shape: B=16, T=512, H=8,
d_k=d_v=64, chunk 64, bf16 q/k/v/dO with f32 gates and state, scalar gates
beta and g generated by SplitMix64 seed 0 (delta_mixers.synthetic).
A step is one forward plus one backward of the scan over the whole batch
(output, final state and scores; gradients of q, k, v, beta, g), with inputs
resident in HBM.  The step is captured once in a HIP graph and replayed.

Prints one JSON line (metric/value/unit/..., roofline, cpu_baseline).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "delta-block-lm_amd"))
sys.path.insert(0, REPO)

PEAK_BF16_TFLOPS = 2500.0   # MI355X dense bf16 MFMA
PEAK_F32_TFLOPS = 157.3     # MI355X dense fp32 MFMA
PEAK_HBM_GBS = 8000.0


def flops_per_token_head(C, K, V):
    """Algorithmic forward FLOPs per token-head of the chunk-WY scan:
    2C^2K x3 (KK^T, QK^T, W) + 2C^2V x2 (U, tril(P) delta) + 2CKV x3 (W S,
    Q S, K^T delta) per chunk + (2/3)C^3 for the triangular inverse, / C."""
    return 6 * C * K + 4 * C * V + 6 * K * V + (2.0 / 3.0) * C * C


def compulsory_bytes_per_token_head(K, V, s_in):
    """Compulsory HBM bytes per token-head that each chunk kernel carries:
    the inputs it must read and the outputs it must write, no intermediates.
    Forward: q, k, v in, beta and g in (f32), o out, score out (f32).
    Backward: q, k, v, dO in, beta and g in, dq, dk, dv out, dbeta and dg out.
    The gradient kernel carries the whole backward's compulsory I/O (beta and
    g reach it through the prep kernel's gate block, equal in size); the
    output kernel carries q, k, v in and o, score out; the prep kernels read
    the operands of their products."""
    return {
        "chunk_prep": (K + V) * s_in + 8,
        "chunk_out": (2 * K + V) * s_in + V * s_in + 4,
        "chunk_bprep": (2 * K + 2 * V) * s_in + 8,
        "chunk_bgrad": (2 * K + 2 * V) * s_in + (2 * K + V) * s_in + 16,
        "state_scan": 0.0,
        "adjoint_scan": 0.0,
    }


def step_bytes(B, T, H, K, V, s_in):
    """Compulsory HBM bytes of one fwd+bwd step (inputs read once per pass,
    outputs written once): fwd = 3 N d s_in + 2 N 4 + N V s_in + B H K V 4 + N 4;
    bwd = 3 N d s_in + 2 N 4 + N V s_in + 3 N d s_in + 2 N 4 (d = K = V here)."""
    N = B * T * H
    fwd = N * ((2 * K + V) * s_in + 8 + V * s_in + 4) + B * H * K * V * 4
    bwd = N * ((2 * K + V) * s_in + 8 + V * s_in + (2 * K + V) * s_in + 8)
    return fwd + bwd


def sources_digest():
    """sha256 (first 16 hex digits) over the kernel sources, file by file in name
    order: the counter profiles record it, and a profile whose digest differs
    from the sources being run is stale (its figures are not reported)."""
    import glob
    import hashlib
    h = hashlib.sha256()
    for path in sorted(glob.glob(os.path.join(REPO, "delta-block-lm_amd", "csrc", "*"))):
        h.update(os.path.basename(path).encode())
        with open(path, "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def load_profile(name):
    """A counter profile under profiles/ and whether it matches the sources:
    (data, "current" | "stale (sources <digest>)" | "absent"); stale data is
    returned as None."""
    path = os.path.join(REPO, "profiles", name)
    if not os.path.exists(path):
        return None, "absent"
    with open(path) as f:
        data = json.load(f)
    if data.get("sources") != sources_digest():
        return None, f"stale (sources {data.get('sources')})"
    return data, "current"


STAGES = ("chunk_prep", "state_scan", "chunk_out", "chunk_bprep", "adjoint_scan", "chunk_bgrad")


def kernel_stage(name):
    """(kernel, stage) of a profiler's kernel name: the library's own name of the
    kernel without its suffix, and the stage that it is (the chunk_, wide_, fc_ and
    fs_ families share the stage names; a scan is state_scan or adjoint_scan by its
    direction argument).  (None, None) for a kernel of another library."""
    import re

    m = re.search(r"gdn2::(?:\(anonymous namespace\)::)?(\w+?)_kernel", name)
    if not m:
        return None, None
    base = m.group(1)
    reverse = {"lr_scan": r"LrCfg<[^<>]*\btrue *>",        # its last argument
               "fc_scan": r"fc_scan_kernel<\d+, true\b",  # its second
               "affine_scan": r"affine_scan_kernel<true>"}.get(base)
    if reverse:
        return base, "adjoint_scan" if re.search(reverse, name) else "state_scan"
    for pre in ("chunk_", "wide_", "fc_", "fs_"):
        if base.startswith(pre) and base[len(pre):] in ("prep", "out", "bprep", "bgrad"):
            return base, "chunk_" + base[len(pre):]
    return base, None


def traffic_from_counters(fetch_dir, write_dir, out_path, probe_bytes):
    """Per-launch HBM bytes of each kernel from two rocprofv3 --pmc runs.
    FETCH_SIZE and WRITE_SIZE are in KiB per dispatch; each is scaled by the
    factor that makes the same counter read the known byte count of the
    plain float32 negation launched by --copy-probe-mb (bytes read = bytes
    written = its size)."""
    import csv
    import glob

    def stage_of(name):
        return "neg" if "neg_kernel" in name else kernel_stage(name)[1]  # the probe

    def read(folder, counter):
        rows = {}
        files = glob.glob(os.path.join(folder, "**", "*counter_collection.csv"), recursive=True)
        if not files:
            raise SystemExit(f"no *counter_collection.csv under {folder}")
        for path in files:
            with open(path) as f:
                for r in csv.DictReader(f):
                    if r["Counter_Name"] != counter:
                        continue
                    key = stage_of(r["Kernel_Name"])
                    if key is None:
                        continue
                    rows.setdefault(key, []).append((float(r["Counter_Value"]),
                                                     int(r["Grid_Size"])))
        return rows

    fetch = read(fetch_dir, "FETCH_SIZE")
    write = read(write_dir, "WRITE_SIZE")
    if "neg" not in fetch or "neg" not in write:
        raise SystemExit("the copy probe (--copy-probe-mb) is missing from the counter runs")
    def probe_kib(rows):  # median over the probe's launches
        vals = sorted(v for v, _ in rows)
        return vals[len(vals) // 2]

    f_scale = probe_bytes / (probe_kib(fetch["neg"]) * 1024.0)
    w_scale = probe_bytes / (probe_kib(write["neg"]) * 1024.0)
    out = {"sources": sources_digest(), "fetch_scale": f_scale, "write_scale": w_scale,
           "probe_bytes": probe_bytes, "bytes_per_launch": {}, "fetch_bytes": {},
           "write_bytes": {}}
    for stage in STAGES:
        if stage in fetch and stage in write:
            fb = sum(v for v, _ in fetch[stage]) / len(fetch[stage]) * 1024.0 * f_scale
            wb = sum(v for v, _ in write[stage]) / len(write[stage]) * 1024.0 * w_scale
            out["fetch_bytes"][stage] = fb
            out["write_bytes"][stage] = wb
            out["bytes_per_launch"][stage] = fb + wb
    text = json.dumps(out, indent=1)
    print(text)
    if out_path:
        with open(out_path, "w") as f:
            f.write(text + "\n")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--config", type=int, default=1, choices=[1, 2, 4],
                    help="1, 2: the scan fwd+bwd; 4: the full lm512 training step")
    ap.add_argument("--hola", action="store_true",
                    help="the HOLA cache read (scores -> cache selection -> attention) fwd+bwd "
                         "at the lm512 head shape")
    ap.add_argument("--doc-scan", action="store_true",
                    help="the document-limit op gdn2_scan (channel-wise gates, packed "
                         "documents) fwd+bwd at the lm512 head shape")
    ap.add_argument("--decode", action="store_true",
                    help="decode steps (one token per sequence) on 256 x 8 "
                         "carried fp32 states, d_k = d_v = 64")
    ap.add_argument("--ref-shape", action="store_true",
                    help="the reference's isolated-scan benchmark (kron_benchmark.rs:73-116): "
                         "gdn2 training scan F and F+B, B8 T512 H4 K32 V64 chunk 16, f32")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--eager", action="store_true", help="no HIP graph")
    ap.add_argument("--copy-probe-mb", type=int, default=0,
                    help="after the timed run, negate a float32 tensor of this many MiB three "
                         "times: the plain-copy kernel that scales the rocprofv3 byte counters")
    ap.add_argument("--traffic", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="no GPU: read two rocprofv3 --pmc output folders (FETCH_SIZE, then "
                         "WRITE_SIZE) of a run with --copy-probe-mb, print the per-launch HBM "
                         "bytes of each chunk kernel and write them to --traffic-out")
    ap.add_argument("--traffic-out", default=None)
    ap.add_argument("--mfma-probe", action="store_true",
                    help="after the timed run, three bf16 8192^3 GEMMs (torch.matmul): the "
                         "calibration kernel of the MFMA-busy counter")
    ap.add_argument("--mfma", metavar="PMC_DIR",
                    help="no GPU: read a rocprofv3 --pmc SQ_VALU_MFMA_BUSY_CYCLES GRBM_GUI_ACTIVE "
                         "output folder of a run with --mfma-probe and print each kernel's MFMA "
                         "utilisation; written to --mfma-out")
    ap.add_argument("--mfma-out", default=None)
    args = ap.parse_args()
    if args.traffic:
        if not args.copy_probe_mb:
            raise SystemExit("--traffic needs --copy-probe-mb (the probe size of the counter runs)")
        traffic_from_counters(args.traffic[0], args.traffic[1], args.traffic_out,
                              args.copy_probe_mb << 20)
        return
    if args.mfma:
        mfma_from_counters(args.mfma, args.mfma_out)
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus {args.gpus}); the scan shards "
              "over batch*heads with no exchange, so per-GPU throughput is the N=1 figure.",
              file=sys.stderr)
        sys.exit(2)

    if args.config == 4:
        bench_train(args)
        return
    if args.doc_scan:
        bench_doc_scan(args)
        return
    if args.ref_shape:
        bench_ref_shape(args)
        return
    if args.hola:
        bench_hola(args)
        return
    if args.decode:
        bench_decode(args)
        return

    import numpy as np
    import torch

    import delta_kernels as dk
    from delta_mixers.synthetic import CONFIGS, generate

    cfg_index = args.config
    cfg = CONFIGS[cfg_index]
    B, T, H, K, V, C = cfg.batch, cfg.time, cfg.heads, cfg.keys, cfg.values, cfg.chunk
    host = generate(cfg, seed=0)
    dtype = torch.bfloat16 if cfg.bf16 else torch.float32
    d = torch.device("cuda:0")
    q = torch.from_numpy(host["q"]).to(d, dtype)
    k = torch.from_numpy(host["k"]).to(d, dtype)
    v = torch.from_numpy(host["v"]).to(d, dtype)
    beta = torch.from_numpy(host["beta"]).to(d)
    g = torch.from_numpy(host["g"]).to(d)
    dO = torch.from_numpy(host["d_output"]).to(d, dtype)
    valid = torch.ones((B, T), device=d)
    reset = torch.zeros((B, T), device=d)
    dk.lib()

    def fwd():
        return dk.gdn_scalar_forward(q, k, v, beta, g, valid, reset, None, C)

    def step():
        out, fin, sc, ck = fwd()
        grads = dk.gdn_scalar_backward(q, k, v, beta, g, valid, reset, ck, C, dO, None, None)
        return (out, fin, sc) + grads

    # Eager reference results, then the captured graph (replays checked against them).
    eager = [t.clone() for t in step()]
    torch.cuda.synchronize()
    graph = None
    if not args.eager:
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(2):
                step()
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            gout = step()
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(gout, eager):
                if not torch.equal(a, b):
                    raise RuntimeError("graph replay differs from the eager step")
    run = graph.replay if graph is not None else step

    for _ in range(args.warmup):
        run()
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    wall0 = time.perf_counter()
    t0.record()
    for _ in range(args.steps):
        run()
    t1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - wall0
    ms = t0.elapsed_time(t1) / args.steps

    # Per-kernel average durations: graphs of back-to-back launches of one kernel.
    def kernel_ms(fn, n=20):
        gr = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            fn()
        torch.cuda.current_stream().wait_stream(s)
        with torch.cuda.graph(gr):
            for _ in range(n):
                fn()
        gr.replay()
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(5):
            gr.replay()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / (5 * n)

    _, _, _, ck = fwd()
    fwd_ms = kernel_ms(fwd)
    bwd_ms = kernel_ms(lambda: dk.gdn_scalar_backward(q, k, v, beta, g, valid, reset, ck, C, dO,
                                                      None, None))

    # Per-kernel durations: HIP events the library records around each of its
    # launches, on the stream the kernels run on (eager calls, averaged).
    dk.stage_timing(True)
    acc, n_timed = {}, 20
    for _ in range(n_timed):
        step()
        torch.cuda.synchronize()
        for name, t in dk.stage_times().items():
            acc[name] = acc.get(name, 0.0) + t
    dk.stage_timing(False)
    stage_ms = {name: t / n_timed for name, t in acc.items()}

    if args.copy_probe_mb:
        src = torch.randn(args.copy_probe_mb << 18, device=d)
        dst = torch.empty_like(src)
        for _ in range(3):
            torch.neg(src, out=dst)
        torch.cuda.synchronize()
    if args.mfma_probe:
        mfma_probe(d)

    N = B * T * H
    f_fwd = flops_per_token_head(C, K, V)
    step_flops = 3 * f_fwd * N
    tokens_per_s = B * T / (ms * 1e-3)
    tflops = step_flops / (ms * 1e-3) / 1e12
    s_in = 2 if cfg.bf16 else 4
    per_th = compulsory_bytes_per_token_head(K, V, s_in)
    kernels = {}
    for name, t in stage_ms.items():
        nbytes = per_th.get(name, 0.0) * N
        kernels[name] = {"ms": t, "compulsory_bytes": nbytes,
                         "GB/s": nbytes / (t * 1e-3) / 1e9 if t > 0 else None}
    if not kernels:
        # Token-sequential path (shapes the chunk kernels do not take): one
        # forward and one backward kernel, whose per-launch durations are the
        # graph-timed fwd_ms / bwd_ms above.
        seq_bytes = {"seq_forward": (2 * K + V) * s_in + V * s_in + 12,
                     "seq_backward": (2 * K + 2 * V) * s_in + (2 * K + V) * s_in + 16}
        for name, t in (("seq_forward", fwd_ms), ("seq_backward", bwd_ms)):
            nbytes = seq_bytes[name] * N
            kernels[name] = {"ms": t, "compulsory_bytes": nbytes, "GB/s": nbytes / (t * 1e-3) / 1e9}
    dom = max(kernels, key=lambda n: kernels[n]["ms"])
    ach = kernels[dom]["GB/s"]
    # Counter profiles of this workload (HBM bytes and MFMA busy per kernel), used
    # only when they were taken of the sources being run.
    tdata, tstate = load_profile(f"{cfg.name}_traffic.json")
    mdata, mstate = load_profile(f"{cfg.name}_mfma.json")
    counter_bytes = (tdata or {}).get("bytes_per_launch", {})
    for name, kv in kernels.items():
        cb = counter_bytes.get(name)
        kv["counter_bytes"] = cb
        kv["counter_GB/s"] = cb / (kv["ms"] * 1e-3) / 1e9 if cb and kv["ms"] > 0 else None
    traffic = counter_bytes.get(dom)
    mfma_util = (mdata or {}).get("mfma_busy")
    sbytes = step_bytes(B, T, H, K, V, s_in)

    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(host, cfg)

    line = {
        "metric": "GDN scan fwd+bwd tokens/s + TFLOP/s (% MFMA peak), lm512 shape, 1 MI355X",
        "value": tokens_per_s,
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16" if cfg.bf16 else "f32",
        "data": f"synthetic (SplitMix64 seed 0, BASELINE configs[{cfg_index}] generator)",
        "config": {"workload": f"{cfg.name}: GDN scan fwd+bwd, scalar gates", "batch": B,
                   "seq_len": T, "heads": H, "d_k": K, "d_v": V, "chunk": C,
                   "parallelism": "none (1 GPU)", "hip_graph": graph is not None},
        "tflops": tflops,
        "pct_peak_bf16": 100 * tflops / PEAK_BF16_TFLOPS,
        "fwd_ms": fwd_ms,
        "bwd_ms": bwd_ms,
        "kernels": kernels,
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": ach, "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": ach / PEAK_HBM_GBS, "traffic": traffic,
                     "step_achieved": sbytes / (ms * 1e-3) / 1e9,
                     "step_frac": sbytes / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS,
                     "mfma_busy": (mfma_util or {}).get(dom),
                     "mfma_busy_per_kernel": mfma_util,
                     "profiles": {"traffic": tstate, "mfma": mstate}},
        "step_roofline": {"compulsory_bytes": sbytes, "GB/s": sbytes / (ms * 1e-3) / 1e9,
                          "frac_hbm": sbytes / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS,
                          "tflops": tflops, "frac_bf16_mfma": tflops / PEAK_BF16_TFLOPS},
        "cpu_baseline": cpu,
        "wall_s_timed": wall,
    }
    print(json.dumps(line))


def train_flops_per_token(cfg, T):
    """Matmul flops of one training token (forward 2 per weight, backward 4):
    every projection, the MLP, the tied head, plus the chunk scan's flops."""
    D, H, K, V, M = cfg.d_model, cfg.heads, cfg.key_dim, cfg.value_dim, cfg.mlp_width
    per_layer = D * (2 * H * K + 2 * H * V + 2 * H) + H * V * D + 3 * D * M
    gemm = 6 * (cfg.layers * per_layer + D * cfg.vocab)
    scan = 3 * cfg.layers * H * flops_per_token_head(cfg.chunk, K, V)
    return gemm + scan


def bench_train(args):
    """One AdamW training step of the 8-block lm512 GDN
    model (random-init weights, uniform random token ids) over B=16 x T=512."""
    import torch

    import delta_kernels as dk
    from delta_mixers.model import GdnLM, GdnLMConfig, make_optimizer, train_step

    cfg = GdnLMConfig()
    B, T = 16, 512
    d = torch.device("cuda:0")
    torch.manual_seed(0)
    model = GdnLM(cfg, device=d)
    opt = make_optimizer(model)
    gen = torch.Generator(device=d).manual_seed(0)
    # T + 1 ids: T positions predict the next id, so every step trains B x T tokens.
    tokens = torch.randint(0, cfg.vocab, (B, T + 1), device=d, generator=gen)
    dk.lib()
    losses = [train_step(model, opt, tokens) for _ in range(max(args.warmup, 1))]
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    wall0 = time.perf_counter()
    t0.record()
    for _ in range(args.steps):
        losses.append(train_step(model, opt, tokens))
    t1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - wall0
    ms = t0.elapsed_time(t1) / args.steps
    loss = [float(x) for x in losses]
    if not all(x == x and abs(x) < 1e4 for x in loss):
        raise RuntimeError(f"non-finite training loss: {loss}")

    # The scan's share: per-kernel events of one eager step.
    dk.stage_timing(True)
    train_step(model, opt, tokens)
    torch.cuda.synchronize()
    stage_ms = dk.stage_times()
    dk.stage_timing(False)

    flops = train_flops_per_token(cfg, T) * B * T
    tflops = flops / (ms * 1e-3) / 1e12
    line = {
        "metric": "lm512 training step (BASELINE configs[4]) tokens/s, 1 MI355X",
        "value": B * T / (ms * 1e-3),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (uniform random token ids, random-init weights)",
        "config": {"workload": "configs[4]: lm512 GDN LM training step (fwd+bwd+AdamW)",
                   "batch": B, "seq_len": T, "d_model": cfg.d_model, "layers": cfg.layers,
                   "heads": cfg.heads, "d_k": cfg.key_dim, "d_v": cfg.value_dim,
                   "mlp": cfg.mlp_width, "vocab": cfg.vocab, "chunk": cfg.chunk,
                   "parallelism": "none (1 GPU)"},
        "roofline": {"bound": "mfma", "achieved": tflops, "peak": PEAK_BF16_TFLOPS,
                     "unit": "TFLOP/s", "frac": tflops / PEAK_BF16_TFLOPS, "traffic": None,
                     "flops_per_step": flops},
        "scan_stage_ms_per_layer": {k: v for k, v in stage_ms.items()},
        "loss_first_last": [loss[0], loss[-1]],
        "cpu_baseline": None,
        "wall_s_timed": wall,
    }
    print(json.dumps(line))


def doc_scan_bytes_per_token_head(K, V):
    """Compulsory HBM bytes of one token-head of gdn2_scan fwd + bwd with bf16
    q/k/v/dO/output and f32 gates: forward reads q, k, v, alpha, erase, write
    and writes the output; backward reads them again plus dO and writes dq, dk,
    dv (bf16) and dalpha, derase, dwrite (f32)."""
    seq = 2 * (2 * K + V)
    gates = 4 * (2 * K + V)
    return (seq + gates + 2 * V) + (seq + gates + 2 * V) + (seq + gates)


def bench_doc_scan(args):
    """gdn2_scan fwd+bwd: B=16, T=512, H=8, d_k=d_v=64 (the lm512 mixer shape),
    bf16 q/k/v, f32 channel-wise gates, packed documents of random lengths."""
    import numpy as np
    import torch

    import delta_kernels as dk
    from oracle import oracle

    B, T, H, K, V = 16, 512, 8, 64, 64
    rng = np.random.default_rng(0)
    d = torch.device("cuda:0")

    def unit(shape):
        x = rng.normal(size=shape).astype(np.float32)
        return x / np.linalg.norm(x, axis=-1, keepdims=True)

    host = {"q": unit((B, T, H, K)), "k": unit((B, T, H, K)),
            "v": rng.normal(size=(B, T, H, V)).astype(np.float32),
            "alpha": rng.uniform(0.9, 1.0, size=(B, T, H, K)).astype(np.float32),
            "erase": rng.uniform(0.0, 1.0, size=(B, T, H, K)).astype(np.float32),
            "write": rng.uniform(0.0, 1.0, size=(B, T, H, V)).astype(np.float32),
            "dO": rng.normal(size=(B, T, H, V)).astype(np.float32)}
    start = np.zeros((B, T), np.int32)
    end = np.zeros((B, T), np.int32)
    for b in range(B):  # documents of 16..200 tokens packed back to back
        s = 0
        while s < T:
            e = min(T - 1, s + int(rng.integers(16, 201)) - 1)
            start[b, s:e + 1], end[b, s:e + 1] = s, e
            s = e + 1
    x = [torch.from_numpy(host[n]).to(d, torch.bfloat16 if n in "qkv" else torch.float32)
         for n in ("q", "k", "v", "alpha", "erase", "write")]
    dO = torch.from_numpy(host["dO"]).to(d, torch.bfloat16)
    ds = torch.from_numpy(start).to(d)
    de = torch.from_numpy(end).to(d)
    dk.lib()

    def step():
        out, ck = dk.gdn2_scan_forward(*x, ds, de)
        return (out,) + dk.gdn2_backward(*x, dO, ck, ds, de)

    for _ in range(max(args.warmup, 1)):
        step()
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    t0.record()
    for _ in range(args.steps):
        step()
    t1.record()
    torch.cuda.synchronize()
    ms = t0.elapsed_time(t1) / args.steps
    nbytes = doc_scan_bytes_per_token_head(K, V) * B * T * H
    ach = nbytes / (ms * 1e-3) / 1e9
    # one more step with the stage timers (outside the timed region)
    dk.stage_timing(True)
    step()
    torch.cuda.synchronize()
    stages = {k: round(v * 1e3, 2) for k, v in dk.stage_times().items()}
    dk.stage_timing(False)

    cpu = None
    if not args.no_cpu_baseline:  # the f64 oracle on 2 of the 16 sequences
        nb = 2
        valid, reset = oracle.doc_limits_to_masks(start[:nb], end[:nb])
        xs = [host[n][:nb].astype(np.float64) for n in ("q", "k", "v", "alpha", "erase", "write")]
        times = []
        t_start = time.perf_counter()
        while len(times) < 3 or time.perf_counter() - t_start < 10:
            c0 = time.perf_counter()
            oracle.scan(*xs, valid, reset)
            oracle.backward(*xs, valid, reset, upstream=host["dO"][:nb].astype(np.float64))
            times.append(time.perf_counter() - c0)
        med = float(np.median(times))
        cpu = {"value": nb * T / med, "unit": "tokens/s", "cores": oracle.threads(),
               "kind": "port",
               "sample": f"f64 oracle fwd+bwd over {nb} of the {B} sequences ({nb}x{T} tokens x "
                         f"{H} heads), OpenMP over the {nb * H} sequences, median of {len(times)}"}
    print(json.dumps({
        "metric": "GDN-2 doc-limit scan (gdn2_scan) fwd+bwd tokens/s, lm512 head shape, 1 MI355X",
        "value": B * T / (ms * 1e-3), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic (seed 0, packed documents of 16-200 tokens)",
        "config": {"workload": "gdn2_scan fwd+bwd, channel-wise gates, doc limits", "batch": B,
                   "seq_len": T, "heads": H, "d_k": K, "d_v": V, "parallelism": "none (1 GPU)"},
        "roofline": {"bound": "hbm", "kernel": "whole fwd+bwd (16-token chunk kernels)",
                     "achieved": ach, "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": ach / PEAK_HBM_GBS, "traffic": None, "compulsory_bytes": nbytes},
        "stage_us": stages,
        "cpu_baseline": cpu}))


def ref_shape_bytes_per_token_head(K, V):
    """Compulsory HBM bytes per token-head of each f32 chunk kernel: the inputs
    it must read and the outputs it must write (4-byte elements), no
    intermediates.  prep reads k, alpha, erase, v, write; out reads q, k,
    alpha, erase, v, write and writes the output and the score; the adjoint scan
    reads dO and forms its additive term from it (no kernel runs in the bprep
    stage); bgrad reads q, k, alpha, erase, v, write, dO and writes dq, dk, dalpha,
    derase, dv, dwrite.  Beyond that the scans move only chunk states."""
    return {"chunk_prep": 4 * (3 * K + 2 * V), "chunk_out": 4 * (4 * K + 3 * V + 1),
            "chunk_bprep": 0.0, "chunk_bgrad": 4 * (8 * K + 5 * V),
            "state_scan": 0.0, "adjoint_scan": 4 * V}


def bench_ref_shape(args):
    """The reference's isolated-scan benchmark (kron_benchmark.rs:1091-1182) at
    its largest shape, B8 T512 H4 K32 V64, chunk 16, f32 q/k/v and channel-wise
    gates (kron_benchmark.rs:73-116 inputs), through gdn2_training_scan /
    gdn2_training_backward.  Protocol as the reference's: first use timed on
    its own, then 2 warm-ups and max(5, --steps) trials of F and of F+B in
    turn, each synchronized before and after on the host clock; value =
    B*T / median(F+B).  Beside it: the HIP-graph replay time of F+B (device
    time, no host overhead) and the per-kernel stage times."""
    import numpy as np
    import torch

    import delta_kernels as dk
    from delta_mixers.synthetic import kron_benchmark_inputs

    B, T, H, K, V, C = 8, 512, 4, 32, 64, 16
    host = kron_benchmark_inputs(B, T)
    d = torch.device("cuda:0")
    x = [torch.from_numpy(host[n]).to(d) for n in ("q", "k", "v", "alpha", "erase", "write")]
    valid = torch.ones((B, T), device=d)
    reset = torch.zeros((B, T), device=d)
    init = torch.from_numpy(host["initial"]).to(d)
    dO = torch.from_numpy(host["d_output"]).to(d)
    dk.lib()

    def fwd():
        return dk.gdn_training_forward(*x, valid, reset, init, C)

    def fwd_bwd():
        out, fin, sc, ck = fwd()
        return (out, fin, sc) + dk.gdn_training_backward(*x, valid, reset, ck, C, dO)

    def timed(fn):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) * 1e3

    first_use = timed(fwd_bwd)
    trials = max(5, args.steps)
    warm = 2
    f_ms, fb_ms = [], []
    for it in range(warm + trials):
        a, b = timed(fwd), timed(fwd_bwd)
        if it >= warm:
            f_ms.append(a)
            fb_ms.append(b)
    f_med, fb_med = float(np.median(f_ms)), float(np.median(fb_ms))

    # device time: F+B captured once in a HIP graph, replays checked and timed
    eager = [t.clone() for t in fwd_bwd()]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            fwd_bwd()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gout = fwd_bwd()
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(gout, eager):
            if not torch.equal(a, b):
                raise RuntimeError("graph replay differs from the eager step")
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    n_rep = max(20, args.steps)
    e0.record()
    for _ in range(n_rep):
        graph.replay()
    e1.record()
    torch.cuda.synchronize()
    graph_ms = e0.elapsed_time(e1) / n_rep

    dk.stage_timing(True)
    acc, n_st = {}, 20
    for _ in range(n_st):
        fwd_bwd()
        torch.cuda.synchronize()
        for name, t in dk.stage_times().items():
            acc[name] = acc.get(name, 0.0) + t
    dk.stage_timing(False)
    stage_ms = {name: t / n_st for name, t in acc.items()}
    if args.copy_probe_mb:
        src = torch.randn(args.copy_probe_mb << 18, device=d)
        dst = torch.empty_like(src)
        for _ in range(3):
            torch.neg(src, out=dst)
        torch.cuda.synchronize()

    N = B * T * H
    per_th = ref_shape_bytes_per_token_head(K, V)
    kernels = {}
    for name, t in stage_ms.items():
        nbytes = per_th.get(name, 0.0) * N
        kernels[name] = {"ms": t, "compulsory_bytes": nbytes,
                         "GB/s": nbytes / (t * 1e-3) / 1e9 if t > 0 else None}
    dom = max(kernels, key=lambda n: kernels[n]["ms"])
    ach = kernels[dom]["GB/s"]
    tdata, tstate = load_profile("refshape_traffic.json")
    counter_bytes = (tdata or {}).get("bytes_per_launch", {})
    for name, kv in kernels.items():
        cb = counter_bytes.get(name)
        kv["counter_bytes"] = cb
        kv["counter_GB/s"] = cb / (kv["ms"] * 1e-3) / 1e9 if cb and kv["ms"] > 0 else None
    traffic = counter_bytes.get(dom)
    step_bytes_fb = sum(per_th[n] for n in per_th) * N
    # fused_gdn2 F+B at B8/T512, Intel Arc MTL, Vulkan: the reference's published
    # figure (docs/optimization/gdn.md:189)
    published_fb_ms = 93.04

    cpu = None
    if not args.no_cpu_baseline:
        from oracle import oracle
        xs = [host[n].astype(np.float64) for n in ("q", "k", "v", "alpha", "erase", "write")]
        ones = np.ones((B, T), np.uint8)
        zeros = np.zeros((B, T), np.uint8)
        up = host["d_output"].astype(np.float64)

        def f64_step():
            oracle.scan(*xs, ones, zeros)
            oracle.backward(*xs, ones, zeros, None, up)

        med, n, wall, first = _median_timed(f64_step, 8.0)
        cpu = {"value": B * T / med, "unit": "tokens/s", "cores": oracle.threads(),
               "kind": "port", "work": "fwd+bwd", "first_use_s": first,
               "sample": f"f64 oracle fwd+bwd over the whole batch ({B}x{T} tokens x {H} heads), "
                         f"2 warm-ups, median of {n} runs ({wall:.1f} s)"}
        cpu.update(cpu_model())

    print(json.dumps({
        "metric": "GDN-2 isolated scan F+B tokens/s, reference benchmark shape (B8 T512 H4 "
                  "K32 V64 C16, f32), 1 MI355X",
        "value": B * T / (fb_med * 1e-3), "unit": "tokens/s", "n_gpus": 1, "steps": trials,
        "warmup": warm, "ms_per_step": fb_med, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": published_fb_ms / fb_med,
        "vs_baseline_note": "published fused_gdn2 F+B 93.04 ms (Intel Arc MTL, Vulkan, f32)",
        "dtype": "f32",
        "data": "synthetic (the reference's SplitMix64 benchmark fixture, seed 1)",
        "config": {"workload": "gdn2_training_scan + gdn2_training_backward, channel-wise "
                               "gates, all-ones upstream", "batch": B, "seq_len": T, "heads": H,
                   "d_k": K, "d_v": V, "chunk": C, "parallelism": "none (1 GPU)"},
        "protocol": "first use separate; 2 warm-ups; trials of F and F+B in turn, host clock, "
                    "synchronized before and after (kron_benchmark.rs:1092-1182)",
        "first_use_ms": first_use, "forward_median_ms": f_med, "forward_ms": f_ms,
        "forward_backward_median_ms": fb_med, "forward_backward_ms": fb_ms,
        "graph_fb_ms": graph_ms, "graph_tokens_per_s": B * T / (graph_ms * 1e-3),
        "kernels": kernels,
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": ach, "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": ach / PEAK_HBM_GBS, "traffic": traffic,
                     "profiles": {"traffic": tstate},
                     "step_compulsory_bytes": step_bytes_fb,
                     "step_achieved": step_bytes_fb / (graph_ms * 1e-3) / 1e9},
        "cpu_baseline": cpu}))


def hola_bytes_per_token_head(K, V, cap, chunk):
    """Compulsory HBM bytes of one token-head of the HOLA read fwd + bwd (f32):
    forward reads q, k, v and the score and writes the output; backward reads
    q, k, v, the output and dO and writes dq, dk, dv."""
    return 4 * ((2 * K + V + 1) + V) + 4 * ((2 * K + V) + 2 * V + (2 * K + V))


def bench_hola(args):
    """HOLA read fwd+bwd: B=16, T=512, H=8, d_k=d_v=64 (the lm512 mixer head
    shape), capacity 64, chunk 16 (the reference's chunk limit), score policy;
    float32 as the reference's operator; packed documents of 16-200 tokens."""
    import numpy as np
    import torch

    import delta_kernels as dk
    from oracle import hola_oracle

    B, T, H, K, V, cap, chunk = 16, 512, 8, 64, 64, 64, 16
    rng = np.random.default_rng(0)
    d = torch.device("cuda:0")
    host = {"q": (rng.normal(size=(B, T, H, K)) / K ** 0.5).astype(np.float32),
            "k": rng.normal(size=(B, T, H, K)).astype(np.float32),
            "v": rng.normal(size=(B, T, H, V)).astype(np.float32),
            "scores": rng.exponential(size=(B, T, H)).astype(np.float32),
            "dO": rng.normal(size=(B, T, H, V)).astype(np.float32)}
    valid = np.ones((B, T), np.float32)
    docs = np.zeros((B, T), np.float32)
    for b in range(B):
        s, doc = 0, 0
        while s < T:
            e = min(T, s + int(rng.integers(16, 201)))
            docs[b, s:e] = doc
            s, doc = e, doc + 1
    sink = np.zeros(H, np.float32)
    x = {n: torch.from_numpy(v).to(d).requires_grad_(n in "qkv") for n, v in host.items()}
    vd, dd = torch.from_numpy(valid).to(d), torch.from_numpy(docs).to(d)
    sk = torch.from_numpy(sink).to(d).requires_grad_(True)
    dk.lib()

    def step():
        r = dk.hola_read(x["q"], x["k"], x["v"], x["scores"], vd, dd, sk, cap, chunk)
        r.output.backward(x["dO"])

    for _ in range(max(args.warmup, 1)):
        step()
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    t0.record()
    for _ in range(args.steps):
        step()
    t1.record()
    torch.cuda.synchronize()
    ms = t0.elapsed_time(t1) / args.steps
    nbytes = hola_bytes_per_token_head(K, V, cap, chunk) * B * T * H
    ach = nbytes / (ms * 1e-3) / 1e9

    cpu = None
    if not args.no_cpu_baseline:  # the f64 oracle on a slice of one sequence's heads
        nb, nt = 1, 256
        xs = {n: host[n][:nb, :nt] for n in host}
        times = []
        t_start = time.perf_counter()
        while len(times) < 2 or time.perf_counter() - t_start < 10:
            c0 = time.perf_counter()
            hola_oracle.hola_read(xs["q"], xs["k"], xs["v"], xs["scores"], valid[:nb, :nt],
                                  docs[:nb, :nt], sink, cap, chunk, False, upstream=xs["dO"])
            times.append(time.perf_counter() - c0)
        med = float(np.median(times))
        cpu = {"value": nb * nt / med, "unit": "tokens/s", "cores": 1, "kind": "port",
               "sample": f"f64 scalar oracle fwd+bwd on {nb}x{nt} tokens x {H} heads, "
                         f"median of {len(times)}"}
    print(json.dumps({
        "metric": "HOLA cache read fwd+bwd tokens/s, lm512 head shape, 1 MI355X",
        "value": B * T / (ms * 1e-3), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32",
        "data": "synthetic (seed 0, exponential scores, documents of 16-200 tokens)",
        "config": {"workload": "hola_read fwd+bwd, score policy", "batch": B, "seq_len": T,
                   "heads": H, "d_k": K, "d_v": V, "capacity": cap, "chunk": chunk,
                   "parallelism": "none (1 GPU)"},
        "roofline": {"bound": "hbm", "kernel": "hola (5 kernels)", "achieved": ach,
                     "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": ach / PEAK_HBM_GBS,
                     "traffic": None, "compulsory_bytes": nbytes},
        "cpu_baseline": cpu}))


def mfma_probe(d):
    """Three bf16 8192^3 GEMMs (hipBLASLt through torch.matmul): a kernel whose
    MFMA pipes are busy for a known share of its time, to calibrate the
    SQ_VALU_MFMA_BUSY_CYCLES reading; prints its achieved TFLOP/s."""
    import torch
    n = 8192
    a = torch.randn(n, n, device=d, dtype=torch.bfloat16)
    b = torch.randn(n, n, device=d, dtype=torch.bfloat16)
    torch.matmul(a, b)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(3):
        torch.matmul(a, b)
    e1.record()
    torch.cuda.synchronize()
    t = e0.elapsed_time(e1) / 3 * 1e-3
    print(json.dumps({"mfma_probe_tflops": 2 * n ** 3 / t / 1e12, "mfma_probe_s": t}),
          file=sys.stderr)


def mfma_from_counters(pmc_dir, out_path):
    """MFMA busy share of each kernel from one rocprofv3 --pmc run collecting
    SQ_VALU_MFMA_BUSY_CYCLES and GRBM_GUI_ACTIVE:
        busy = SQ_VALU_MFMA_BUSY_CYCLES / (GRBM_GUI_ACTIVE / XCDs x CUs x 4 SIMDs)
    (the profiler sums GRBM_GUI_ACTIVE over the 8 XCDs and the MFMA counter over
    every SIMD).  The run must include --mfma-probe: the bf16 GEMM's busy share is
    reported beside its achieved fraction of the bf16 peak as the check."""
    import csv
    import glob

    files = glob.glob(os.path.join(pmc_dir, "**", "*counter_collection.csv"), recursive=True)
    if not files:
        raise SystemExit(f"no *counter_collection.csv under {pmc_dir}")
    per = {}
    for path in files:
        with open(path) as f:
            for r in csv.DictReader(f):
                name = r["Kernel_Name"]
                base, stage = kernel_stage(name)
                key = stage or base or ("gemm" if "Cijk" in name or "gemm" in name.lower()
                                        else None)
                if key is None:
                    continue
                d = per.setdefault(key, {}).setdefault(r.get("Dispatch_Id", r.get("Correlation_Id")),
                                                       {})
                d[r["Counter_Name"]] = d.get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
    XCDS, CUS, SIMDS = 8, 256, 4
    busy = {}
    for key, disp in per.items():
        vals = [v["SQ_VALU_MFMA_BUSY_CYCLES"] / (v["GRBM_GUI_ACTIVE"] / XCDS * CUS * SIMDS)
                for v in disp.values()
                if v.get("GRBM_GUI_ACTIVE") and "SQ_VALU_MFMA_BUSY_CYCLES" in v]
        if vals:
            busy[key] = sorted(vals)[len(vals) // 2]
    out = {"sources": sources_digest(),
           "formula": "SQ_VALU_MFMA_BUSY_CYCLES / (GRBM_GUI_ACTIVE / 8 x 256 CUs x 4 SIMDs)",
           "mfma_busy": {k: busy[k] for k in STAGES if k in busy},
           "calibration_gemm_busy": busy.get("gemm")}
    text = json.dumps(out, indent=1)
    print(text)
    if out_path:
        with open(out_path, "w") as f:
            f.write(text + "\n")


def bench_decode(args):
    """B=256 sequences x H=8 heads, d_k = d_v = 64 fp32
    states drawn N(0, 0.02); one token per sequence per step (q, k, v, beta, g
    from the generator of delta_mixers.synthetic), gdn2_decode_step on the carried state.  A
    step reads and writes every state once: compulsory bytes
    2 B H K V 4 + token I/O, HBM-bound."""
    import numpy as np
    import torch

    import delta_kernels as dk
    from delta_mixers.synthetic import CONFIGS, generate

    cfg = CONFIGS[3]
    B, T, H, K, V = cfg.batch, cfg.time, cfg.heads, cfg.keys, cfg.values
    host = generate(cfg, seed=0)
    d = torch.device("cuda:0")
    q, k, v = (torch.from_numpy(host[n]).to(d) for n in ("q", "k", "v"))
    alpha = torch.exp(torch.from_numpy(host["g"]).to(d))[..., None].expand(B, T, H, K)
    beta = torch.from_numpy(host["beta"]).to(d)[..., None]
    erase, write = beta.expand(B, T, H, K), beta.expand(B, T, H, V)
    state = torch.from_numpy(host["state"]).to(d).contiguous()
    valid = torch.ones((B, 1), device=d)
    reset = torch.zeros((B, 1), device=d)
    dk.lib()
    steps = min(args.steps * 20, T)
    sl = [slice(t, t + 1) for t in range(T)]

    def step(t):
        i = sl[t % T]
        return dk.gdn_decode_step(state, q[:, i], k[:, i], v[:, i], alpha[:, i], erase[:, i],
                                  write[:, i], valid, reset)

    for t in range(max(args.warmup, 1)):
        step(t)
    torch.cuda.synchronize()
    # Per-kernel duration: a graph of back-to-back decode steps (no host gaps).
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step(0)
    torch.cuda.current_stream().wait_stream(s)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        for t in range(steps):
            step(t)
    gr.replay()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    gr.replay()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / steps
    state_bytes = 2 * B * H * K * V * 4
    token_bytes = B * H * (2 * K * 4 + V * 4 + K * 4 + K * 4 + V * 4 + V * 4 + 4)
    nbytes = state_bytes + token_bytes
    ach = nbytes / (ms * 1e-3) / 1e9
    cpu = None
    if not args.no_cpu_baseline:
        from oracle import oracle
        a, e, w = oracle.scalar_gates(host["beta"][:, :1], host["g"][:, :1], K, V)
        xs = [host[n][:, :1].astype(np.float64) for n in ("q", "k", "v")]
        ones = np.ones((B, 1), np.uint8)
        zeros = np.zeros((B, 1), np.uint8)
        st = host["state"].astype(np.float64)
        med, n, wall, first = _median_timed(
            lambda: oracle.scan(*xs, a, e, w, ones, zeros, st), 8.0)
        cpu = {"value": 1.0 / med, "unit": "steps/s", "cores": oracle.threads(), "kind": "port",
               "first_use_s": first,
               "sample": f"f64 oracle one-token scan over all {B}x{H} carried states, 2 "
                         f"warm-ups, median of {n} runs ({wall:.1f} s)"}
        cpu.update(cpu_model())
    print(json.dumps({
        "metric": "GDN decode step (configs[3]) steps/s, 256 x 8 fp32 states, 1 MI355X",
        "value": 1e3 / ms, "unit": "steps/s", "n_gpus": 1, "steps": steps,
        "warmup": args.warmup, "ms_per_step": ms, "us_per_step": ms * 1e3,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic (SplitMix64 seed 0, BASELINE configs[3] generator)",
        "config": {"workload": "decode: gdn2_decode_step on carried states", "batch": B,
                   "heads": H, "d_k": K, "d_v": V, "parallelism": "none (1 GPU)",
                   "hip_graph": True},
        "roofline": {"bound": "hbm", "kernel": "seq_decode", "achieved": ach,
                     "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": ach / PEAK_HBM_GBS,
                     "traffic": None, "compulsory_bytes": nbytes},
        "cpu_baseline": cpu}))


def cpu_model():
    """The host CPU's model name and the cores this process may use."""
    name = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    name = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"cpu_model": name, "nproc": len(os.sched_getaffinity(0))}


def _median_timed(fn, budget_s):
    """The reference's timing protocol (kron_benchmark.rs:1092-1182): the first
    use timed on its own, then 2 warm-ups (the first use is one of them), then
    at least 5 trials and about budget_s seconds; returns (median, trials,
    wall of the trials, first use), seconds."""
    import numpy as np
    t0 = time.perf_counter()
    fn()
    first = time.perf_counter() - t0
    fn()
    times = []
    t_start = time.perf_counter()
    while len(times) < 5 or time.perf_counter() - t_start < budget_s:
        t0 = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t0)
    return float(np.median(times)), len(times), time.perf_counter() - t_start, first


def cpu_baseline(host, cfg, budget_s=8.0):
    """The reference's CPU path restated and timed on this host's cores, on the
    same inputs, in two legs (OpenMP over the B*H sequences):
      * f64 sequential scan + VJP (crates/mixers/src/reference.rs:41-257), the
        oracle: fwd+bwd tokens/s, the headline figure (same unit as the metric);
      * f32 chunked scan (the tensor solver crates/mixers/src/chunk.rs:129-250
        that the gdn-reference-cpu path runs; forward only, the reference has no
        hand-written VJP for it), chunk 64 with forward substitution.
    Protocol: 1 warm-up, >= 3 trials, about budget_s seconds each, median."""
    import numpy as np

    from oracle import oracle

    B, T, H, K, V = cfg.batch, cfg.time, cfg.heads, cfg.keys, cfg.values
    x = {n: host[n].astype(np.float64) for n in ("q", "k", "v", "d_output")}
    a, e, w = oracle.scalar_gates(host["beta"], host["g"], K, V)
    valid = np.ones((B, T), np.uint8)
    reset = np.zeros((B, T), np.uint8)

    def f64_step():
        oracle.scan(x["q"], x["k"], x["v"], a, e, w, valid, reset)
        oracle.backward(x["q"], x["k"], x["v"], a, e, w, valid, reset, None, x["d_output"])

    med, n, wall, first = _median_timed(f64_step, budget_s)
    f64_leg = {"value": B * T / med, "unit": "tokens/s", "cores": oracle.threads(),
               "kind": "port", "work": "fwd+bwd", "first_use_s": first,
               "sample": f"f64 oracle fwd+bwd over the whole {cfg.name} batch ({B}x{T} tokens "
                         f"x {H} heads), 2 warm-ups, median of {n} runs ({wall:.1f} s)"}
    x32 = {n: host[n].astype(np.float32) for n in ("q", "k", "v")}
    a32, e32, w32 = (t.astype(np.float32) for t in (a, e, w))
    v32 = valid.astype(np.float32)
    r32 = reset.astype(np.float32)

    def f32_fwd():
        oracle.chunk_scan_f32(x32["q"], x32["k"], x32["v"], a32, e32, w32, v32, r32, None,
                              cfg.chunk)

    med, n, wall, first = _median_timed(f32_fwd, budget_s)
    f32_leg = {"value": B * T / med, "unit": "tokens/s (forward only)",
               "cores": oracle.chunk_threads(), "kind": "port", "work": "fwd",
               "first_use_s": first,
               "sample": f"f32 chunked scan (chunk {cfg.chunk}) forward over the whole "
                         f"{cfg.name} batch, 2 warm-ups, median of {n} runs ({wall:.1f} s)"}
    out = dict(f64_leg)
    out["legs"] = {"f64_sequential_fwd_bwd": f64_leg, "f32_chunked_fwd": f32_leg}
    out.update(cpu_model())
    return out


if __name__ == "__main__":
    main()
