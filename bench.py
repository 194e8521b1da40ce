#!/usr/bin/env python3
"""Benchmark of the forward (prefill) and greedy decode path on one MI355X.

Headline (the one JSON line): 7B-shape prefill — dim 4096, SwiGLU 11008,
32 layers, 32 heads x 128, vocab 32000, batch 1, seq 512, fp16 weights
~N(0, 0.02) from a fixed seed, uniform random tokens — as tokens/s of whole
forwards (embedding .. per-position cross-entropy), inputs resident in HBM.

Also reported on the same line:
  roofline      the dominant kernel (the FFN up-projection GEMM with the SwiGLU
                epilogue, 2*512*22016*4096 flop per launch) timed alone with HIP
                events on the stream it runs on, against 2.5 PFLOP/s dense fp16;
  decode        7B-shape greedy decode at batch 1 and 16: 2048-token seeded
                prefill into the preallocated KV cache, then 256 steps
                replayed from one HIP graph; tok/s and HBM GB/s;
  prefill_b8    the same forward at batch 8;
  prefill       every other prefill workload: 7B seq 2048 at batch 1 and 8,
                48M (512d/1536h/8L, 8x64) at batch 1, 600M-shape at batch 1
                and 8, 5B-shape at batch 4 (seq 512), each with its device
                time per stage and layer (hb_forward_timed);
  stages_b1     the headline forward's device time per stage (hb_forward_timed,
                the reference's forward_timed split: QKV, attention, Wo,
                residual + norm, FFN up, FFN down, ...), per layer;
  cpu_baseline  the fp32 CPU oracle timed on this host's CPU share the way the
                reference's forward probe times its forward (1 warmup, median
                of 3): whole forwards up to 20 layers; the 5B and 7B shapes as
                1- and 2-layer stacks (per-layer cost = their difference), so
                the scaling to all layers is measured, not assumed; and the
                7B decode step at batch 1 and 16.

  python bench.py [--steps K] [--warmup W] [--gpus 1]
  python bench.py --model 600m --no-decode ...   (one workload alone, for profiling)
"""
import argparse
import dataclasses
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

MFMA_PEAK_F16 = 2.5e15  # dense fp16, MI355X
MODELS = {"7b": "llama_7b", "5b": "llama_5b", "600m": "llama_600m", "48m": "llama_48m"}
HBM_PEAK = 8.0e12

SEED = 1234
STD = 0.02


def fwd_flops(cfg, B, S):
    """2*B*S*[L*(d*q + 2*d*kv + q*d + 3*d*h) + d*V] + B*L*2*q*S*(S+1) (causal attention)."""
    d, q, kv, h, L, V = cfg.dim, cfg.q_dim, cfg.kv_dim, cfg.hidden, cfg.nlayers, cfg.vocab
    return 2 * B * S * (L * (d * q + 2 * d * kv + q * d + 3 * d * h) + d * V) + B * L * 2 * q * S * (S + 1)


def train_flops(cfg, B, S):
    """Algorithmic flops of one training forward + backward: every weight
    product three times (forward, dX, dW: 6*T*params) and causal attention
    3.5 times its forward (scores recomputed, dP, dQ, dK, dV)."""
    d, q, kv, h, L, V = cfg.dim, cfg.q_dim, cfg.kv_dim, cfg.hidden, cfg.nlayers, cfg.vocab
    mats = L * (d * q + 2 * d * kv + q * d + 3 * d * h) + d * V
    return 6 * B * S * mats + 3.5 * B * L * 2 * q * S * (S + 1)


def decode_bytes(cfg, B, p):
    """fp16 bytes one decode step at position p must move: all weights (tied E
    read once for the logits) + K/V read for p+1 positions + K/V write."""
    d, q, kv, h, L, V = cfg.dim, cfg.q_dim, cfg.kv_dim, cfg.hidden, cfg.nlayers, cfg.vocab
    weights = 2 * (L * (d * q + 2 * d * kv + q * d + 3 * d * h) + V * d)
    return weights + B * L * 2 * kv * (p + 1) * 2 + B * L * 2 * kv * 2


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--batch", type=int, default=1)
    ap.add_argument("--seq", type=int, default=512)
    ap.add_argument("--kernel-launches", type=int, default=50)
    ap.add_argument("--decode-steps", type=int, default=256)
    ap.add_argument("--decode-ctx", type=int, default=2048)
    ap.add_argument("--no-decode", action="store_true")
    ap.add_argument("--no-decode-b16", action="store_true")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the 600M / 5B / 7B-seq-2048 prefill workloads")
    ap.add_argument("--no-b8", action="store_true")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-optimizer", action="store_true")
    ap.add_argument("--no-validate", action="store_true")
    ap.add_argument("--no-train", action="store_true")
    ap.add_argument("--train-only", action="store_true",
                    help="only the training forward + backward section (for profiling)")
    ap.add_argument("--kernel-only", action="store_true",
                    help="only the dominant kernel (timed) and a 1 GiB device copy, for counter runs")
    ap.add_argument("--model", choices=sorted(MODELS), default="7b",
                    help="shape of the main forward (default: the benchmark's 7B headline; the others "
                         "are for profiling one workload alone, and skip the other prefill workloads)")
    args = ap.parse_args()

    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on exactly one GPU; --gpus must be 1 "
                                   "(multi-GPU sharding is a design note, not built)"}))
        sys.exit(2)

    import torch  # device memory + streams only; import before the library
    from rustane_amd import hip_bridge as hb
    from rustane_amd.engine import CompiledKernels, ModelConfig

    torch.cuda.init()
    stream = torch.cuda.Stream()  # default priority
    torch.cuda.set_stream(stream)

    cfg = dataclasses.replace(getattr(ModelConfig, MODELS[args.model])(), seq=max(args.seq, 2048))
    name = args.model.upper()
    log(f"[bench] {name}-shape model: {cfg.param_count()/1e9:.3f}B params")
    k = CompiledKernels.compile(cfg)
    k.ctx.set_stream(stream.cuda_stream)
    t0 = time.time()
    k.init_synthetic(SEED, STD)
    torch.cuda.synchronize()
    log(f"[bench] device weights initialised in {time.time()-t0:.1f}s "
        f"({k.model.weight_bytes()/1e9:.2f} GB)")

    B, S = args.batch, args.seq
    tok = hb.synth_tokens(42, 0, cfg.vocab, B * (S + 1)).reshape(B, S + 1)
    d_tok = torch.from_numpy(tok[:, :-1].astype(np.int32).copy()).cuda()
    d_tgt = torch.from_numpy(tok[:, 1:].astype(np.int32).copy()).cuda()
    d_loss = torch.empty(B * S, device="cuda")
    d_mean = torch.empty(1, device="cuda")
    k.model.reserve(B, S)

    def step():
        hb.call("hb_forward_device", k.model.handle, d_tok.data_ptr(), d_tgt.data_ptr(), B, S,
                d_loss.data_ptr(), None, d_mean.data_ptr())

    if args.train_only:
        # the same 1 GiB reference copy as --kernel-only, for scaling counters
        src = torch.empty(1 << 28, dtype=torch.float32, device="cuda").fill_(1.0)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
        print(json.dumps({"train": bench_train(k, cfg, stream, B, S, steps=args.steps)}), flush=True)
        return

    if args.kernel_only:
        # Reference transfer of known size (read 1 GiB + write 1 GiB) for scaling
        # the FETCH_SIZE / WRITE_SIZE counters, then the dominant kernel alone.
        src = torch.empty(1 << 28, dtype=torch.float32, device="cuda").fill_(1.0)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        roofline, _ = time_dominant_kernel(k, cfg, B * S, args.kernel_launches, stream)
        print(json.dumps({"kernel_only": roofline}), flush=True)
        return

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    ev0.record(stream)
    for _ in range(args.steps):
        step()
    ev1.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    k.ctx.synchronize()
    ms_step = ev0.elapsed_time(ev1) / args.steps
    ms_wall = wall * 1e3 / args.steps
    loss = float(d_mean.cpu()[0])
    flops = fwd_flops(cfg, B, S)
    tok_s = B * S / (ms_wall / 1e3)
    log(f"[bench] prefill B={B} S={S}: {ms_wall:.3f} ms/forward (events {ms_step:.3f}), "
        f"{tok_s:,.0f} tok/s, {flops/(ms_wall/1e3)/1e12:.1f} TFLOP/s, loss {loss:.4f} "
        f"(ln V = {math.log(cfg.vocab):.4f})")

    roofline, _ = time_dominant_kernel(k, cfg, B * S, args.kernel_launches, stream)

    extra = {}
    # ---- per-stage device time of the same forward (hb_forward_timed) ----
    extra["stages_b1"] = bench_stages(k, cfg, d_tok, d_tgt, B, S)
    up_in_fwd = extra["stages_b1"]["per_layer_us"]["ffn_up"]
    roofline["us_per_launch_in_forward"] = round(up_in_fwd, 2)
    roofline["frac_in_forward"] = round(roofline["flop_per_launch"] / (up_in_fwd * 1e-6) / MFMA_PEAK_F16, 4)
    # ---- batch 8 prefill ----
    if not args.no_b8 and B == 1:
        B8 = 8
        tok8 = hb.synth_tokens(42, 8, cfg.vocab, B8 * (S + 1)).reshape(B8, S + 1)
        t8 = torch.from_numpy(tok8[:, :-1].astype(np.int32).copy()).cuda()
        g8 = torch.from_numpy(tok8[:, 1:].astype(np.int32).copy()).cuda()
        l8 = torch.empty(B8 * S, device="cuda")
        m8 = torch.empty(1, device="cuda")
        k.model.reserve(B8, S)
        run8 = lambda: hb.call("hb_forward_device", k.model.handle, t8.data_ptr(), g8.data_ptr(), B8,
                               S, l8.data_ptr(), None, m8.data_ptr())
        for _ in range(2):
            run8()
        torch.cuda.synchronize()
        n8 = max(3, args.steps // 2)
        t0 = time.perf_counter()
        for _ in range(n8):
            run8()
        torch.cuda.synchronize()
        ms8 = (time.perf_counter() - t0) * 1e3 / n8
        f8 = fwd_flops(cfg, B8, S)
        extra["prefill_b8"] = {"ms_per_forward": round(ms8, 3), "tok_per_s": round(B8 * S / ms8 * 1e3, 1),
                               "tflop_per_s": round(f8 / ms8 / 1e9, 1),
                               "mfma_frac": round(f8 / (ms8 / 1e3) / MFMA_PEAK_F16, 4),
                               "loss": round(float(m8.cpu()[0]), 5)}
        log(f"[bench] prefill B=8: {ms8:.3f} ms, {extra['prefill_b8']}")

    # ---- the other prefill workloads ----
    if not args.no_configs and B == 1 and S == 512 and args.model == "7b":
        extra["prefill"] = bench_prefill_configs(k, cfg, stream, cpu=not args.no_cpu_baseline)

    # ---- decode ----
    if not args.no_decode:
        from rustane_amd.engine import Decoder
        batches = [1] + ([] if args.no_decode_b16 else [16])
        dec_res = {}
        for DB in batches:
            P, n = args.decode_ctx, args.decode_steps
            dec = Decoder(k, batch=DB, ctx_max=P + n)
            ptok = hb.synth_tokens(42, 100 + DB, cfg.vocab, DB * P).reshape(DB, P)
            t0 = time.perf_counter()
            _, nxt = dec.prefill(ptok)
            pre_ms = (time.perf_counter() - t0) * 1e3
            # warm the captured graph on a throwaway cache of the same shape
            warm = Decoder(k, batch=DB, ctx_max=P + n)
            warm.prefill(ptok)
            warm.greedy(nxt, 4)
            del warm
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            out = dec.greedy(nxt, n)
            dt = time.perf_counter() - t0
            nbytes = sum(decode_bytes(cfg, DB, P + i) for i in range(n))
            gbs = nbytes / dt / 1e9
            dec_res[f"b{DB}"] = {"tok_per_s": round(DB * n / dt, 1), "ms_per_step": round(dt * 1e3 / n, 3),
                                 "GB_per_s": round(gbs, 1), "hbm_frac": round(gbs * 1e9 / HBM_PEAK, 4),
                                 "ctx": f"{P}->{P+n}", "prefill_ms": round(pre_ms, 1),
                                 "first_tokens": out[:4, 0].tolist()}
            log(f"[bench] decode B={DB}: {dec_res[f'b{DB}']}")
            dec.kv.close()
        if not args.no_cpu_baseline:
            dec_res["cpu_baseline_b1"] = cpu_baseline_decode(cfg, args.decode_ctx)
            if "b16" in dec_res:
                dec_res["cpu_baseline_b16"] = cpu_baseline_decode(cfg, args.decode_ctx, batch=16, timed_seqs=2)
        extra["decode"] = dec_res

    # ---- validation loop (windows of a resident token stream) ----
    if not args.no_validate:
        extra["validate"] = bench_validate(k, cfg, stream)

    # ---- optimizer step over the whole model ----
    if not args.no_optimizer:
        extra["optimizer"] = bench_optimizer(k, stream, cpu=not args.no_cpu_baseline)

    # ---- training forward + backward and train_step ----
    if not args.no_train:
        extra["train"] = bench_train(k, cfg, stream, B, S)
        if B == 1 and not args.no_cpu_baseline:
            extra["train"]["cpu_baseline"] = cpu_baseline_train(cfg, S)
        if B == 1 and not args.no_b8:
            # eight sequences per call: the weight-gradient products get K = 4096
            extra["train"]["b8"] = bench_train(k, cfg, stream, 8, S, steps=2)

    # ---- CPU baseline (oracle, bounded sample) ----
    if not args.no_cpu_baseline:
        extra["cpu_baseline"] = cpu_baseline(cfg, S)

    line = {
        "metric": f"prefill tok/s at {name}-shape seq{S} fp16; decode tok/s + % of HBM peak",
        "value": round(tok_s, 1),
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_wall, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp16",
        "data": "synthetic (seeded N(0,0.02) weights, uniform tokens)",
        "config": {"workload": f"{name}-shape prefill forward + CE ({cfg.dim}d/{cfg.hidden}h/{cfg.nlayers}L, "
                               f"{cfg.heads}x{cfg.hd} heads, vocab {cfg.vocab})",
                   "global_batch": B, "seq_len": S, "parallelism": "single-gpu",
                   "tflop_per_forward": round(flops / 1e12, 4),
                   "mfma_frac_whole_forward": round(flops / (ms_wall / 1e3) / MFMA_PEAK_F16, 4),
                   "loss": round(loss, 5)},
        "roofline": roofline,
    }
    line.update({k2: v for k2, v in extra.items() if k2 != "cpu_baseline"})
    if "cpu_baseline" in extra:
        line["cpu_baseline"] = extra["cpu_baseline"]
    print(json.dumps(line), flush=True)


# HBM bytes per launch of the dominant kernel, from two rocprofv3 --pmc runs of
# `bench.py --kernel-only` (FETCH_SIZE, then WRITE_SIZE), each scaled by the
# counter's reading for the 1 GiB reference copy in the same run (FETCH_SIZE
# reads 0.5x the copied bytes, WRITE_SIZE 1.0x): 2 * 106864.5 KiB + 13446.7 KiB.
# Algorithmic bytes of one launch: W1|W3 180.4 MB + X 4.2 MB read, gate 11.3 MB
# written = 195.8 MB.
DOMINANT_TRAFFIC_BYTES = 232_627_904


def time_dominant_kernel(k, cfg, T, launches, stream):
    """The FFN up-projection GEMM (W1|W3 with the SwiGLU epilogue, one launch)
    on layer 0 at T tokens, timed with HIP events on the stream it runs on."""
    import torch
    from rustane_amd import hip_bridge as hb
    xn = (torch.randn(T, cfg.dim, device="cuda") * 0.5).to(torch.float16)
    gate = torch.empty(T, cfg.hidden, dtype=torch.float16, device="cuda")

    def up():
        hb.call("hb_op_ffn_up", k.model.handle, 0, xn.data_ptr(), T, gate.data_ptr(), None)

    for _ in range(5):
        up()
    torch.cuda.synchronize()
    # The launches are captured into one HIP graph on the kernel's own stream and
    # the replay is timed with HIP events on that stream, so host dispatch gaps
    # between launches do not count against the kernel.
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for _ in range(launches):
            up()
    graph.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    graph.replay()
    e1.record(stream)
    torch.cuda.synchronize()
    up_ms = e0.elapsed_time(e1) / launches
    del graph
    up_flops = 2.0 * T * (2 * cfg.hidden) * cfg.dim
    achieved = up_flops / (up_ms / 1e3) / 1e12
    log(f"[bench] ffn-up GEMM {T}x{2*cfg.hidden}x{cfg.dim}: {up_ms*1e3:.1f} us/launch, "
        f"{achieved:.1f} TFLOP/s ({achieved/2500*100:.1f}% of dense fp16 peak)")
    counted = (cfg.dim, cfg.hidden, T) == (4096, 11008, 512)  # the launch the counters were read on
    roofline = {"bound": "mfma", "achieved": round(achieved, 2), "peak": 2500.0, "unit": "TFLOP/s",
                "frac": round(achieved / 2500.0, 4), "traffic": DOMINANT_TRAFFIC_BYTES if counted else None,
                "traffic_source": "rocprofv3 FETCH_SIZE + WRITE_SIZE of this kernel, scaled by a 1 GiB copy "
                                  "(profiles/ffn_up_gemm_7b_b1_counters.md), not measured in this run"
                                  if counted else None,
                "kernel": ("gemm_nt_kernel<192,256,EpiSwiGLU>" if counted else "prefill GEMM, EpiSwiGLU")
                          + " (FFN up, W1|W3 + SwiGLU)",
                "flop_per_launch": up_flops, "us_per_launch": round(up_ms * 1e3, 2),
                "timing": "us_per_launch: launches back to back (HIP events around a graph of them); "
                          "us_per_launch_in_forward: inside the forward, from hb_forward_timed"}
    return roofline, up_ms


def bench_stages(k, cfg, d_tok, d_tgt, B, S, reps=3):
    """hb_forward_timed on the headline forward (the reference's forward_timed,
    layer.rs:821-1015, as device times): each stage's time per layer (layers
    1..L-1; the two-term first layer alone), the median of `reps` timed
    forwards."""
    import torch
    runs = []
    for _ in range(reps + 1):
        runs.append(k.model.forward_timed(d_tok.data_ptr(), d_tgt.data_ptr(), B, S))
    torch.cuda.synchronize()
    runs = runs[1:]
    med = {n: float(np.median([r[n] for r in runs])) for n in runs[0]}
    n = med["layers_summed"]
    per = {"qkv": "sdpa_qkv_ms", "attention": "sdpa_attention_ms", "wo": "wo_ms",
           "residual_rmsnorm2": "residual_rmsnorm2_ms", "ffn_up": "ffn_up_ms", "ffn_down": "ffn_down_ms",
           "ffn_residual_norm": "ffn_residual_norm_ms"}
    res = {"per_layer_us": {a: round(med[b] * 1e3 / n, 2) for a, b in per.items()},
           "layer0_us": round(med["layer0_ms"] * 1e3, 1), "embedding_us": round(med["embedding_ms"] * 1e3, 1),
           "logits_us": round(med["logits_ms"] * 1e3, 1), "cross_entropy_us": round(med["cross_entropy_ms"] * 1e3, 1),
           "total_ms": round(med["total_ms"], 3), "layers_summed": int(n),
           "note": "eager launches with an event after each stage (median of 3 forwards); the graph-replayed "
                   "forward of the headline runs without those events"}
    log(f"[bench] stages B={B}: {res}")
    return res


def bench_validate(k, cfg, stream, steps=32):
    """hb_validate (bin/train.rs:123-163 on the device) over a resident stream of
    2M uniform token ids with a synthetic byte table: windows of seq 512, 8 per
    forward, and one per forward as the reference runs them."""
    import torch
    from rustane_amd import hip_bridge as hb
    toks = hb.synth_tokens(7, 0, cfg.vocab, 2_000_000).astype("<u2")
    tb = (hb.synth_tokens(8, 0, 5, cfg.vocab)).astype("<i4")
    dt = hb.DeviceTokens(k.ctx, tokens=toks)
    res = {"seq": cfg.seq, "windows": steps}
    try:
        for B in (8, 1):
            hb.validate(k.model, dt, tb, B, B)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            avg, bpb, _, _ = hb.validate(k.model, dt, tb, steps, B)
            sec = time.perf_counter() - t0
            res[f"batch{B}"] = {"tok_per_s": round(steps * cfg.seq / sec, 1), "ms": round(sec * 1e3, 2),
                                "avg_loss": round(avg, 5), "bpb": round(bpb, 5)}
    finally:
        dt.close()
    log(f"[bench] validate: {res}")
    return res


class _DeviceArray:
    """A raw device pointer as a CUDA-array-interface object (for torch.as_tensor)."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False),
                                         "version": 2}


def bench_optimizer(k, stream, cpu=True, steps=3):
    """train_step's optimizer half on the whole 7B-shape model (hb_opt_step:
    gradient norm + clip decision + fused AdamW over every weight, refreshing
    the fp16 copy), and the AdamW pass alone (hb_opt_update_weights, the
    dominant kernel: 30 bytes per parameter -- read param/grad/m/v, write
    param/m/v and the fp16 weight). Gradients are N(0, 1e-3) noise written
    into the device arena."""
    import torch
    from rustane_amd import hip_bridge as hb
    from rustane_amd.engine import TrainConfig
    opt = hb.Optimizer(k.model, TrainConfig())
    try:
        ptr, n = opt.grad_arena()
        try:
            torch.as_tensor(_DeviceArray(ptr, n), device="cuda").normal_(0.0, 1e-3)
            grads = "N(0, 1e-3)"
        except Exception as e:  # pragma: no cover - interface not available
            log(f"[bench] optimizer: gradients left at zero ({e})")
            grads = "zero"
        opt.step(0, want_norm=False)
        opt.update_weights(2, 1e-4, 1.0)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for s in range(1, steps + 1):
            opt.step(s, want_norm=False)
        e1.record(stream)
        torch.cuda.synchronize()
        step_ms = e0.elapsed_time(e1) / steps
        e0.record(stream)
        for t in range(1, steps + 1):
            opt.update_weights(t + 3, 1e-4, 1.0)
        e1.record(stream)
        torch.cuda.synchronize()
        upd_ms = e0.elapsed_time(e1) / steps
        norm = opt.grad_norm()
    finally:
        opt.close()
    upd_bytes, step_bytes = 30 * n, 34 * n
    gbs = upd_bytes / (upd_ms / 1e3) / 1e9
    res = {"params": n, "grads": grads, "grad_norm": round(norm, 4),
           "ms_per_optimizer_step": round(step_ms, 3),
           "step_GB_per_s": round(step_bytes / (step_ms / 1e3) / 1e9, 1),
           "adamw_ms": round(upd_ms, 3), "adamw_GB_per_s": round(gbs, 1),
           "roofline": {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK / 1e9,
                        "unit": "GB/s", "frac": round(gbs * 1e9 / HBM_PEAK, 4),
                        "traffic": None, "kernel": "adamw_kernel<true> (fused AdamW, fp16 refresh)",
                        "bytes_per_launch_set": upd_bytes}}
    if cpu:
        res["cpu_baseline"] = cpu_baseline_adam(n)
    log(f"[bench] optimizer: {res}")
    return res


def bench_train(k, cfg, stream, B, S, steps=4):
    """Training on the 7B-shape model: hb_forward_backward_device (forward
    keeping activations + backward accumulating every gradient) alone, and the
    whole train_step (zero grads, forward + backward, hb_opt_step)."""
    import torch
    from rustane_amd import hip_bridge as hb
    from rustane_amd.engine import TrainConfig
    opt = hb.Optimizer(k.model, TrainConfig())
    try:
        tok = hb.synth_tokens(42, 300, cfg.vocab, B * (S + 1)).reshape(B, S + 1)
        d_tok = torch.from_numpy(tok[:, :-1].astype(np.int32).copy()).cuda()
        d_tgt = torch.from_numpy(tok[:, 1:].astype(np.int32).copy()).cuda()
        d_mean = torch.empty(1, device="cuda")
        fb = lambda: opt.forward_backward_device(d_tok.data_ptr(), d_tgt.data_ptr(), B, S, 256.0,
                                                 d_mean=d_mean.data_ptr())
        opt.zero_grads()
        fb()
        torch.cuda.synchronize()
        loss0 = float(d_mean.cpu()[0])
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(steps):
            fb()
        e1.record(stream)
        torch.cuda.synchronize()
        fb_ms = e0.elapsed_time(e1) / steps
        norm = opt.grad_norm()
        t0 = time.perf_counter()
        for s in range(steps):
            opt.zero_grads()
            fb()
            opt.step(s, want_norm=False)
        torch.cuda.synchronize()
        step_ms = (time.perf_counter() - t0) * 1e3 / steps
        loss1 = float(d_mean.cpu()[0])
    finally:
        opt.close()
    fl = train_flops(cfg, B, S)
    tfs = fl / (fb_ms / 1e3) / 1e12
    res = {"batch": B, "seq": S, "ms_per_fwd_bwd": round(fb_ms, 3),
           "tok_per_s_fwd_bwd": round(B * S / fb_ms * 1e3, 1),
           "tflop_per_s": round(fl / fb_ms / 1e9, 1), "mfma_frac": round(fl / (fb_ms / 1e3) / MFMA_PEAK_F16, 4),
           "tflop_per_fwd_bwd": round(fl / 1e12, 3),
           "ms_per_train_step": round(step_ms, 3), "tok_per_s_train_step": round(B * S / step_ms * 1e3, 1),
           "loss_first": round(loss0, 5), "loss_after_steps": round(loss1, 5),
           "grad_norm_x_loss_scale": round(norm, 3),
           "roofline": {"bound": "mfma", "achieved": round(tfs, 1), "peak": MFMA_PEAK_F16 / 1e12,
                        "unit": "TFLOP/s", "frac": round(tfs * 1e12 / MFMA_PEAK_F16, 4), "traffic": None,
                        "kernel": "whole training forward + backward (algorithmic flops)"}}
    log(f"[bench] train: {res}")
    return res


def cpu_baseline_adam(n_params, sample=1 << 26):
    """The oracle's fused AdamW (cpu/adam.rs:95-132 in numpy fp32) on a
    64M-parameter sample; the whole-model time is scaled from it."""
    import oracle.optimizer as OP
    rng = np.random.default_rng(0)
    p = rng.standard_normal(sample, dtype=np.float32)
    g = (rng.standard_normal(sample, dtype=np.float32) * np.float32(1e-3)).astype(np.float32)
    m = np.zeros(sample, np.float32)
    v = np.zeros(sample, np.float32)
    best = 1e9
    for t in (1, 2):
        t0 = time.perf_counter()
        OP.step_fused(p, g, m, v, t, 1e-4, 0.9, 0.95, 1e-8, 0.1, 1.0)
        best = min(best, time.perf_counter() - t0)
    return {"value": round(sample / best / 1e6, 1), "unit": "M params/s", "cores": 1, "kind": "port",
            "sample": f"numpy fp32 step_fused on {sample} parameters (best of 2): {best*1e3:.0f} ms; "
                      f"whole model {n_params * best / sample:.1f} s"}


def cpu_threads():
    """Host threads the CPU baselines use: this process's CPU share. A
    multi-GPU host may allot each GPU a share of its cores (OMP_NUM_THREADS);
    elsewhere every CPU this process may run on."""
    avail = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    share = int(os.environ.get("OMP_NUM_THREADS", "0") or 0)
    return min(share, avail) if share > 0 else avail


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    import platform
    return platform.processor() or "unknown"


def _threads_limited():
    try:
        from threadpoolctl import threadpool_limits
    except ImportError:  # pragma: no cover
        return None
    return threadpool_limits(limits=cpu_threads())


def _oracle_layer(cfg, layer=0):
    """The seeded fp32 weights of one layer (hb_model_init_synthetic's tensor
    ids 16*layer + 0..6), in the oracle's LayerW."""
    import oracle as O
    from rustane_amd import hip_bridge as hb
    d, q, kv, h = cfg.dim, cfg.q_dim, cfg.kv_dim, cfg.hidden
    n = lambda tid, cnt: hb.synth_normal(SEED, 16 * layer + tid, cnt, STD)
    return O.LayerW(wq=n(0, d * q), wk=n(1, d * kv), wv=n(2, d * kv), wo=n(3, q * d), w1=n(4, d * h),
                    w3=n(5, d * h), w2=n(6, d * h), gamma1=np.ones(d, np.float32),
                    gamma2=np.ones(d, np.float32))


_CPU_SAMPLES = {}


def _median_of_3(fn):
    """1 warmup + median of 3 timed calls, the reference's forward probe
    (crates/engine/tests/bench_fwd_only_scale.rs:74-86)."""
    fn()
    ts = []
    for _ in range(3):
        t0 = time.perf_counter()
        fn()
        ts.append(time.perf_counter() - t0)
    return sorted(ts)[1]


def cpu_forward_sample(cfg, B, S, whole_up_to_layers=20):
    """fp32 oracle forward of one sequence of S tokens on the host (embedding ..
    per-position CE), timed as the reference's forward probe times its forward:
    1 warmup + median of 3. Models of up to `whole_up_to_layers` layers run
    whole. Deeper ones run as a 1-layer and a 2-layer stack of the model's
    own first layers: their difference is one layer, the rest the embedding
    and head, and nlayers x layer + head is the forward. The reference has no
    batch dimension: B sequences take B times one. Returns (seconds per
    B-sequence forward, note)."""
    key = (cfg.dim, cfg.hidden, cfg.nlayers, cfg.heads, cfg.vocab, S)
    if key in _CPU_SAMPLES:
        t_seq, note = _CPU_SAMPLES[key]
        return B * t_seq, note
    import dataclasses

    import oracle as O
    from rustane_amd import hip_bridge as hb
    d = cfg.dim
    E = hb.synth_normal(SEED, hb.HB_SYNTH_EMBED_ID, cfg.vocab * d, STD)
    tok = hb.synth_tokens(42, 0, cfg.vocab, S + 1)

    def stack(L):
        oc = dataclasses.replace(O.Config.of(cfg), nlayers=L, seq=max(S, 1))
        w = O.ModelW(embed=E, layers=[_oracle_layer(cfg, l) for l in range(L)], gamma_final=np.ones(d, np.float32))
        return lambda: O.model_forward(oc, w, tok[:-1], tok[1:])

    if cfg.nlayers <= whole_up_to_layers:
        t_seq = _median_of_3(stack(cfg.nlayers))
        note = f"whole {cfg.nlayers}-layer forward {t_seq:.3f} s (1 warmup + median of 3)"
    else:
        t1, t2 = _median_of_3(stack(1)), _median_of_3(stack(2))
        layer = t2 - t1
        head = max(t1 - layer, 0.0)
        t_seq = head + cfg.nlayers * layer
        note = (f"1-layer forward {t1:.3f} s, 2-layer {t2:.3f} s (1 warmup + median of 3 each): "
                f"{layer * 1e3:.0f} ms per layer + {head * 1e3:.0f} ms embedding/head, "
                f"x{cfg.nlayers} layers = {t_seq:.2f} s")
    _CPU_SAMPLES[key] = (t_seq, note)
    return B * t_seq, note


def cpu_baseline(cfg, S):
    """Headline CPU baseline: the fp32 oracle's forward of the main model at
    B=1 on this host's CPU share (cpu_forward_sample: for the 7B shape 1- and
    2-layer stacks, 1 warmup + median of 3 each, scaled to 32 layers)."""
    ctx = _threads_limited()
    try:
        t, note = cpu_forward_sample(cfg, 1, S)
        res = {"value": round(S / t, 2), "unit": "tok/s", "cores": cpu_threads(), "kind": "port",
               "cpu_model": cpu_model(), "host_cpus": os.cpu_count(),
               "sample": f"fp32 numpy oracle, {cfg.nlayers}-layer {cfg.dim}d forward at B=1 S={S}: {note}"}
        log(f"[bench] cpu baseline: {res}")
        return res
    finally:
        if ctx is not None and hasattr(ctx, "unregister"):
            ctx.unregister()


def cpu_baseline_decode(cfg, ctx_len=2048, batch=1, timed_seqs=1):
    """fp32 oracle decode step (DecodeOracle.step) of the 7B shape at position
    ctx_len on the host: one step through a 1-layer and a 2-layer model with a
    filled K/V cache gives the per-layer and the head cost; a 32-layer step
    is head + 32 x layer. Median of 3 steps each. The reference decodes one
    sequence at a time (no batch dimension): a batch of B takes B sequence
    steps, and timed_seqs of them (each its own cache) are timed."""
    import dataclasses

    import oracle as O
    from rustane_amd import hip_bridge as hb
    lim = _threads_limited()
    try:
        lw = _oracle_layer(cfg)
        E = hb.synth_normal(SEED, hb.HB_SYNTH_EMBED_ID, cfg.vocab * cfg.dim, STD)
        steps = []
        for sq in range(timed_seqs):
            times = {}
            for L in (1, 2):
                oc = dataclasses.replace(O.Config.of(cfg), nlayers=L, seq=ctx_len + 8)
                w = O.ModelW(embed=E, layers=[lw] * L, gamma_final=np.ones(cfg.dim, np.float32))
                dec = O.DecodeOracle(oc, w, ctx_max=ctx_len + 8)
                rng = np.random.default_rng(10 * sq + L)
                dec.k[:] = rng.standard_normal(dec.k.shape, dtype=np.float32)
                dec.v[:] = rng.standard_normal(dec.v.shape, dtype=np.float32)
                dec.pos = ctx_len
                ts = []
                for i in range(3):
                    t0 = time.perf_counter()
                    dec.step(int(i + 7 * sq))
                    ts.append(time.perf_counter() - t0)
                times[L] = sorted(ts)[1]
            layer = max(times[2] - times[1], 1e-6)
            head = max(times[1] - layer, 0.0)
            steps.append((head + cfg.nlayers * layer, layer, head))
        seq_step = float(np.mean([t for t, _, _ in steps]))
        layer, head = float(np.mean([l for _, l, _ in steps])), float(np.mean([h for _, _, h in steps]))
        step = batch * seq_step
        who = (f"B={batch}: {timed_seqs} of the {batch} sequences timed, each {seq_step * 1e3:.0f} ms; "
               f"{batch} x one sequence per step" if batch > 1 else "B=1")
        res = {"value": round(batch / step, 3), "unit": "tok/s", "ms_per_step": round(step * 1e3, 1),
               "cores": cpu_threads(), "kind": "port", "cpu_model": cpu_model(),
               "sample": f"fp32 numpy DecodeOracle.step at position {ctx_len}, {who}: {cfg.nlayers} x "
                         f"{layer*1e3:.1f} ms per layer + {head*1e3:.1f} ms embedding/head (median of 3 "
                         f"steps of 1- and 2-layer models with a filled K/V cache)"}
        log(f"[bench] cpu baseline (decode): {res}")
        return res
    finally:
        if lim is not None and hasattr(lim, "unregister"):
            lim.unregister()


def bench_prefill_configs(k7, cfg7, stream, cpu=True):
    """Prefill forwards (embedding .. per-position CE) of the other workloads:
    7B-shape at seq 2048 (batch 1 and 8, on the headline model), the 48M
    workload (512d/1536h/8L, 8x64, vocab 32000) at batch 1, 600M-shape
    (1536d/4096h/20L, 12x128) at batch 1 and 8 and 5B-shape (2560d/6912h/60L,
    20x128) at batch 4, all seq 512 but the first, each on seeded N(0, 0.02)
    device weights; wall time over repeated hb_forward_device calls."""
    import torch
    from rustane_amd import hip_bridge as hb
    from rustane_amd.engine import CompiledKernels, ModelConfig

    def run(k, cfg, B, S, reps):
        tok = hb.synth_tokens(42, 500 + B, cfg.vocab, B * (S + 1)).reshape(B, S + 1)
        dt = torch.from_numpy(tok[:, :-1].astype(np.int32).copy()).cuda()
        dg = torch.from_numpy(tok[:, 1:].astype(np.int32).copy()).cuda()
        dl = torch.empty(B * S, device="cuda")
        dm = torch.empty(1, device="cuda")
        k.model.reserve(B, S)
        f = lambda: hb.call("hb_forward_device", k.model.handle, dt.data_ptr(), dg.data_ptr(), B, S,
                            dl.data_ptr(), None, dm.data_ptr())
        f()
        f()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(reps):
            f()
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) * 1e3 / reps
        k.ctx.synchronize()
        fl = fwd_flops(cfg, B, S)
        r = {"ms_per_forward": round(ms, 3), "tok_per_s": round(B * S / ms * 1e3, 1),
             "tflop_per_s": round(fl / ms / 1e9, 1), "mfma_frac": round(fl / (ms / 1e3) / MFMA_PEAK_F16, 4),
             "tflop_per_forward": round(fl / 1e12, 3), "loss": round(float(dm.cpu()[0]), 5),
             "stages": bench_stages(k, cfg, dt, dg, B, S)}
        if cpu:
            lim = _threads_limited()
            try:
                t, note = cpu_forward_sample(cfg, B, S)
            finally:
                if lim is not None and hasattr(lim, "unregister"):
                    lim.unregister()
            r["cpu_baseline"] = {"value": round(B * S / t, 2), "unit": "tok/s", "cores": cpu_threads(),
                                 "kind": "port", "sample": f"fp32 numpy oracle, one sequence: {note}; x{B}"}
        return r

    out = {}
    for B in (1, 8):
        out[f"7b_s2048_b{B}"] = run(k7, cfg7, B, 2048, 3 if B == 1 else 2)
        log(f"[bench] prefill 7B S=2048 B={B}: {out[f'7b_s2048_b{B}']}")
    for name, mk, batches in (("48m", ModelConfig.llama_48m, (1,)), ("600m", ModelConfig.llama_600m, (1, 8)),
                              ("5b", ModelConfig.llama_5b, (4,))):
        cfg = mk()
        k = CompiledKernels.compile(cfg)
        k.ctx.set_stream(stream.cuda_stream)
        try:
            k.init_synthetic(SEED, STD)
            for B in batches:
                out[f"{name}_s512_b{B}"] = run(k, cfg, B, 512, (40 if name == "48m" else 10) if B == 1 else 5)
                log(f"[bench] prefill {name} S=512 B={B}: {out[f'{name}_s512_b{B}']}")
        finally:
            torch.cuda.synchronize()
            k.model.close()
            k.ctx.close()
    return out


def cpu_baseline_train(cfg, S):
    """fp32 oracle on the host: the forward (with its taps) and the backward of
    one of the 32 layers of the 7B-shape model at one sequence of S tokens,
    the head's forward + backward (final norm, logits, CE, dlogits, dE, dX)
    once; a whole forward + backward is estimated as 32 x layer + head."""
    import oracle as O
    import oracle.backward as OB
    from rustane_amd import hip_bridge as hb
    try:
        from threadpoolctl import threadpool_limits
    except ImportError:  # pragma: no cover
        threadpool_limits = None
    cores = cpu_threads()
    ctx = threadpool_limits(limits=cores) if threadpool_limits else None
    try:
        oc = O.Config.of(cfg)
        d, q, kv, h, V = cfg.dim, cfg.q_dim, cfg.kv_dim, cfg.hidden, cfg.vocab
        n = lambda tid, cnt: hb.synth_normal(SEED, tid, cnt, STD)
        lw = O.LayerW(wq=n(0, d * q), wk=n(1, d * kv), wv=n(2, d * kv), wo=n(3, q * d), w1=n(4, d * h),
                      w3=n(5, d * h), w2=n(6, d * h), gamma1=np.ones(d, np.float32),
                      gamma2=np.ones(d, np.float32))
        E = n(hb.HB_SYNTH_EMBED_ID, V * d)
        tok = hb.synth_tokens(42, 0, V, S + 1)
        x = O.mtrans(O.embedding_forward(E, d, tok[:-1]), S, d)
        rope = O.rope_table(S, cfg.hd)
        gf = np.ones(d, np.float32)
        t0 = time.perf_counter()
        xl, taps = O.layer_forward(oc, lw, x, S, rope)
        t_lf = time.perf_counter() - t0
        t0 = time.perf_counter()
        xf, rinv = O.rmsnorm_channel_first(xl, gf, d, S)
        logits = O.sgemm_at(O.mtrans(xf, d, S), S, d, E, V, np.zeros(S * V, np.float32))
        _, dlog = OB.cross_entropy_fwd_bwd(logits, tok[1:], V, np.float32(1.0 / S))
        dl = (dlog * np.float32(256.0)).reshape(S, V)
        xf2 = np.asarray(xf, np.float32).reshape(d, S)
        _ = (dl.T @ xf2.T).astype(np.float32)
        dxf = (E.reshape(V, d).T @ dl.T).astype(np.float32).reshape(-1)
        dy, _ = OB.rmsnorm_backward_cf(dxf, xl, gf, rinv, d, S)
        t_head = time.perf_counter() - t0
        t0 = time.perf_counter()
        OB.layer_backward(oc, lw, taps, x, dy, S)
        t_lb = time.perf_counter() - t0
        t_full = cfg.nlayers * (t_lf + t_lb) + t_head
        res = {"value": round(S / t_full, 3), "unit": "tok/s", "cores": cores, "kind": "port",
               "sample": f"fp32 numpy oracle: forward + backward of 1 of {cfg.nlayers} layers and the "
                         f"head of the 7B-shape model at one sequence of {S}; full fwd+bwd = "
                         f"{cfg.nlayers} x ({t_lf*1e3:.0f} + {t_lb*1e3:.0f}) ms + {t_head*1e3:.0f} ms "
                         f"= {t_full:.1f} s"}
        log(f"[bench] cpu baseline (train): {res}")
        return res
    finally:
        if ctx is not None:
            ctx.unregister() if hasattr(ctx, "unregister") else None


if __name__ == "__main__":
    main()
