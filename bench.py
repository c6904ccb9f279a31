#!/usr/bin/env python3
"""Headline benchmark: ADKV decode attention, Llama-2-7B shape, one MI355X.

One "step" is one layer's decode-attention for a batch: forward_qk (+append) -> softmax ->
forward_ov (+append) over a resident 4-bit K/V cache, the protocol of the reference's
tools/perf_kernel.py:28-76, issued the way the cache object issues it: one adkv_decode_step call.  Throughput follows its convention (perf_kernel.py:91-104):
tokens/s = B / (32 layers * seconds per layer-step).  Caches are produced by running the encoder
on seeded synthetic K/V (closed loop), and the timed steps rotate over several distinct layer
buffers so no cache level can serve re-reads.

Prints ONE JSON line.  `roofline` prices the dominant kernel (the QK scan) on its algorithmic
bytes, B*H*T*d*bits/8 code bytes per launch, against the 8 TB/s HBM peak; `cpu_baseline` times the
reference's PyTorch CPU path (eager fp32 recurrence + attention, all host cores) on a bounded sample.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
N_LAYERS_MODEL = 32


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=256,
                    help="timed steps; the default covers eight model passes of 32 layer-steps")
    ap.add_argument("--warmup", type=int, default=64,
                    help="untimed steps first; the device clock settles over the first few dozen launches")
    ap.add_argument("--workload", choices=["decode", "encode", "quant_f32"], default="decode",
                    help="decode = headline decode attention (cfg2); encode = streaming quantiser (cfg3: "
                         "B=8 ctx=32768 prefill, then 256 single-token appends)")
    ap.add_argument("--batch", type=int, default=128)
    ap.add_argument("--heads", type=int, default=32)
    ap.add_argument("--kv-heads", type=int, default=0,
                    help="KV heads when fewer than --heads query heads share them (grouped-query "
                         "attention); default: as many as --heads")
    ap.add_argument("--bits", type=int, default=4, choices=[2, 4],
                    help="code width of the decode workload (2 needs --dim 128)")
    ap.add_argument("--dim", type=int, default=128)
    ap.add_argument("--ctx", type=int, default=4096)
    ap.add_argument("--layer-buffers", type=int, default=4,
                    help="distinct K/V caches rotated through (defeats on-die cache reuse)")
    ap.add_argument("--ckpt-interval", type=int, default=256,
                    help="state checkpoint spacing in tokens (0 = none: one sequential replay per head)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also run three 1 GiB device-to-device copies (a known-size kernel to scale "
                         "rocprofv3 FETCH_SIZE/WRITE_SIZE readings by)")
    ap.add_argument("--graph", action="store_true",
                    help="also replay the step from HIP graphs and report that time beside the headline")
    ap.add_argument("--bf16", action="store_true",
                    help="decode workload: q, the new token and the output in bfloat16")
    ap.add_argument("--no-secondary", action="store_true",
                    help="default decode run only: skip the short cfg3 / cfg5 / cfg1 runs reported under `secondary`")
    ap.add_argument("--event-stride", type=int, default=4,
                    help="record the per-stage HIP events on every N-th timed step (1: every step)")
    ap.add_argument("--no-e2e", action="store_true",
                    help="leave the end-to-end generate record (cfg4, about half a minute) out of `secondary`")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-fp16-comparator", action="store_true",
                    help="skip timing the fp16-KV decode kernel beside the ADKV step")
    ap.add_argument("--cpu-sample-batch", type=int, default=128,
                    help="sequences of the batch the host baseline runs (full context, all heads; "
                         "the whole batch of 128 takes about 6 s on 16 cores and 35 GB of host memory)")
    return ap.parse_args()


def cpu_baseline(args, T, D):
    """The reference's PyTorch CPU path timed on this host: for a sample of the batch, the eager
    fp32 per-token recurrence over whole [B, C] tensors for K and for V over the full context
    (src/adkv/train/train_model.py:61-81), then softmax(q.K^T/sqrt(d)).V for the single query
    (src/adkv/train/llama_attention.py:41-44), on all host cores.  That is one decode-attention
    step of one layer, the unit the GPU number is quoted in.  The C oracle of the fp16 recurrence
    (one core) is timed beside it as a secondary figure."""
    import numpy as np
    import torch
    from adkv_amd import synth
    from oracle import oracle as O
    from oracle import torch_cpu

    H = args.heads
    C = H * D
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    Bs = max(1, min(args.batch, args.cpu_sample_batch))
    f32 = lambda p: [t.float().reshape(-1) for t in p.astuple()]
    kp, vp = f32(synth.make_params(H, D, seed=3)), f32(synth.make_params(H, D, seed=4))
    rows = lambda x: x.permute(0, 2, 1, 3).reshape(Bs, T, C).contiguous()          # [B, T, H*d]
    k = rows(synth.make_k(Bs, H, T, D))
    v = rows(synth.make_v(Bs, H, T, D))
    q = synth.make_q(Bs, H, D, dtype=torch.float32).reshape(Bs, C)
    torch_cpu.decode_step(q, k[:, :64], v[:, :64], kp, vp, H, D ** -0.5)            # warm-up
    t0 = time.perf_counter()
    torch_cpu.decode_step(q, k, v, kp, vp, H, D ** -0.5)
    dt = time.perf_counter() - t0
    res = {
        "value": Bs / (N_LAYERS_MODEL * dt),
        "unit": "tokens/s",
        "cores": cores,
        "kind": "port",
        "sample": f"PyTorch CPU eager fp32 (torch {torch.__version__}, {cores} threads): {Bs} of {args.batch} "
                  f"sequences x {H} heads x ctx {T}, one full layer-step (per-token recurrence for K and V, "
                  f"then single-query attention) = {dt:.2f} s; value = {Bs} / (32 layers x that time), "
                  f"i.e. the rate at batch {Bs}, not extrapolated",
    }
    # secondary: the C oracle of the fp16 recurrence (bit-exact), one core
    hs = min(H, 8)
    np16 = lambda t: t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.float16)
    kq = synth.make_params(H, D, seed=3)
    pn = [np16(t)[:hs] for t in kq.astuple()]
    kk = np16(synth.make_k(1, hs, T + 1, D, dtype=torch.float16))
    qq = np16(synth.make_q(1, hs, D))
    kc, vc = O.alloc_cache(1, hs, T + 8, D), O.alloc_cache(1, hs, T + 8, D)
    O.encode_kv_f16(kc, kk[:, :, :T], *pn)
    O.encode_kv_f16(vc, kk[:, :, :T], *pn)
    t0 = time.perf_counter()
    O.decode_step_f16(qq, kc, vc, kk[:, :, T:], kk[:, :, T:], pn, pn, T, D ** -0.5)
    dc = time.perf_counter() - t0
    res["c_oracle_fp16"] = {"value": 1.0 / (N_LAYERS_MODEL * dc * H / hs), "unit": "tokens/s", "cores": 1,
                            "sample": f"C oracle of the fp16 recurrence, 1 sequence x {hs} of {H} heads x ctx {T} "
                                      f"in {dc:.2f} s, scaled linearly to {H} heads"}
    return res


def fp16_comparator(args, dev, adkv_ms):
    """The same decode-attention step over an uncompressed fp16 K/V cache (split-K flash decoding,
    adkv_fp16_decode), timed like the ADKV step.  Reported beside the headline value, never as it."""
    import torch
    from adkv_amd import synth
    from adkv_amd.kernel.fp16_baseline import fp16_decode_attention

    B, H, D, T = args.batch, args.heads, args.dim, args.ctx
    K = synth.make_k(B, H, T, D, layer=0, dtype=torch.float16, device=dev)
    V = synth.make_v(B, H, T, D, layer=0, dtype=torch.float16, device=dev)
    q = synth.make_q(B, H, D, device=dev)
    ws = torch.empty(B * H * (-(-T // 512)) * (D + 2) * 4, dtype=torch.uint8, device=dev)
    for _ in range(max(2, args.warmup)):
        fp16_decode_attention(q, K, V, D ** -0.5, ws)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        fp16_decode_attention(q, K, V, D ** -0.5, ws)
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.steps
    kv_bytes = 2.0 * B * H * T * D * 2
    return {"kernel": "adkv_fp16_decode (fp16 K/V, split-K flash decoding)", "ms_per_step": ms,
            "tokens_per_s": B / (N_LAYERS_MODEL * ms * 1e-3),
            "kv_GBps": kv_bytes / (ms * 1e-3) / 1e9, "hbm_frac": kv_bytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
            "adkv_speedup": ms / adkv_ms}


def encode_record(args, B, T, steps, warmup, cpu=True):
    """cfg3: one step = prefill-quantise B x ctx tokens of K (one launch); afterwards 256 timed
    single-token appends.  tokens quantised / s = B*ctx / t_prefill."""
    import numpy as np
    import torch
    from adkv_amd import synth
    from adkv_amd.kernel import gemv

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    H, D, S = args.heads, args.dim, (args.ckpt_interval or 256)
    n_app = 256
    p = synth.make_params(H, D).to(dev)
    x = synth.make_k(B, H, T + n_app, D, dtype=torch.float16, device=dev)
    xp = x[:, :, :T].contiguous()
    cache = synth.alloc_cache(B, H, T + n_app + 8, D, dev)
    ck = torch.zeros(B, H, (T + n_app) // S + 1, D, 2, dtype=torch.float16, device=dev)
    state = torch.zeros(B, H, D, 2, dtype=torch.float16, device=dev)
    ev = lambda: torch.cuda.Event(enable_timing=True)

    def prefill():
        gemv.append_kv(cache, xp, *p.astuple(), 0, state, ckpt=ck, ckpt_interval=S)

    for _ in range(warmup):
        prefill()
    torch.cuda.synchronize()
    marks = []
    t0 = time.perf_counter()
    for _ in range(steps):
        e0, e1 = ev(), ev()
        e0.record(); prefill(); e1.record()
        marks.append((e0, e1))
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms_step = wall * 1e3 / steps
    k_ms = sum(a.elapsed_time(b) for a, b in marks) / len(marks)

    toks = [x[:, :, T + i:T + i + 1].contiguous() for i in range(n_app)]
    torch.cuda.synchronize()
    a0, a1 = ev(), ev()
    a0.record()
    for i in range(n_app):
        gemv.append_kv(cache, toks[i], *p.astuple(), T + i, state, ckpt=ck, ckpt_interval=S)
    a1.record(); torch.cuda.synchronize()
    append_us = a0.elapsed_time(a1) * 1e3 / n_app

    # K and V rows of the same tokens in one launch (what the cache layer's prefill does)
    pv = synth.make_params(H, D, seed=4).to(dev)
    xv = synth.make_v(B, H, T, D, dtype=torch.float16, device=dev)
    cache_v = synth.alloc_cache(B, H, T + 8, D, dev)
    cache_k2 = synth.alloc_cache(B, H, T + 8, D, dev)
    st_k, st_v = torch.zeros_like(state), torch.zeros_like(state)

    def prefill_pair():
        gemv.append_kv_pair(cache_k2, cache_v, xp, xv, p.astuple(), pv.astuple(), 0, st_k, st_v)

    prefill_pair()
    torch.cuda.synchronize()
    p0, p1 = ev(), ev()
    p0.record()
    for _ in range(steps):
        prefill_pair()
    p1.record(); torch.cuda.synchronize()
    pair_ms = p0.elapsed_time(p1) / steps
    pair_same = bool(torch.equal(cache_k2[:, :, :T // 8], cache[:, :, :T // 8]))

    # bit-exactness of the codes: two sampled heads against the oracle, whole stream
    from oracle import oracle as O
    np16 = lambda t: t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.float16)
    exact = True
    for (b, h) in [(0, 0), (B - 1, H - 1)]:
        want = O.alloc_cache(1, 1, T + n_app + 8, D)
        O.encode_kv_f16(want, np16(x[b:b + 1, h:h + 1]), *[np16(t)[h:h + 1] for t in p.astuple()])
        exact &= bool(np.array_equal(cache[b:b + 1, h:h + 1].cpu().numpy(), want))

    bytes_launch = B * H * T * D * 2.5
    achieved = bytes_launch / (k_ms * 1e-3) / 1e9
    res = {
        "metric": "streaming quantiser tokens quantised/sec (B*ctx / prefill time, one K tensor)",
        "value": B * T / (ms_step * 1e-3), "unit": "tokens/s", "n_gpus": 1,
        "steps": steps, "warmup": warmup, "ms_per_step": ms_step,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f16",
        "data": "synthetic",
        "config": {"workload": f"cfg3 streaming quantise: prefill B={B} H={H} d={D} ctx={T} fp16 -> 4-bit codes, "
                               f"then {n_app} single-token appends with carried state",
                   "batch": B, "heads": H, "head_dim": D, "ctx": T, "bits": 4, "ckpt_interval": S},
        "append_us_per_token_step": append_us,
        "kv_pair": {"ms_per_prefill": pair_ms, "tokens_per_s": B * T / (pair_ms * 1e-3),
                    "k_codes_equal_single_tensor_run": pair_same,
                    "note": "K and V of every token in one launch (adkv_append_kv_pair)"},
        "codes_bit_exact_vs_oracle": exact,
        "roofline": {"kernel": "encode_kernel", "bound": "hbm", "achieved": achieved,
                     "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBPS,
                     # FETCH_SIZE/WRITE_SIZE per prefill launch, scaled by a 1 GiB copy
                     # (profiles/encode_cfg3_and_decode_cfg5_pmc_traffic.md); default workload only
                     "traffic": 2.7015e9 if (B, H, D, T, S) == (8, 32, 128, 32768, 256) else None},
    }
    if cpu:
        hs, Ts = 2, 4096
        xs = np16(x[:1, :hs, :Ts])
        c = O.alloc_cache(1, hs, Ts, D)
        t0 = time.perf_counter()
        O.encode_kv_f16(c, xs, *[np16(t)[:hs] for t in p.astuple()])
        dt = time.perf_counter() - t0
        res["cpu_baseline"] = {"value": Ts / (dt * H / hs), "unit": "tokens/s", "cores": 1, "kind": "port",
                               "sample": f"C oracle encode, 1 sequence x {hs} of {H} heads x {Ts} tokens "
                                         f"in {dt:.2f} s; scaled linearly to {H} heads"}
    return res


def quant_f32_record(args, B, T, steps, warmup):
    """cfg1: the fp32 (train / eval) recurrence over one sequence of 32 heads x 128 channels and
    1024 tokens, K-shaped input with outlier channels.  A step is one pass over the sequence."""
    import numpy as np
    import torch
    from adkv_amd import synth
    from adkv_amd.train import quant_f32

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    H, D = args.heads, args.dim
    C = H * D
    p = synth.make_params(H, D, dtype=torch.float32)
    x = synth.make_k(B, H, T, D, dtype=torch.float32).permute(0, 2, 1, 3).reshape(B, T, C).contiguous()
    pf = [t.float().reshape(-1) for t in p.astuple()]
    xg = x.to(dev)
    zp_i, sc_i, al, be, tg = [t.to(dev) for t in pf]
    smin, smax = math.exp(-4.0), math.exp(4.0)
    zp = torch.empty(B, C, device=dev)
    sc = torch.empty(B, C, device=dev)
    out = torch.empty_like(xg)
    ev = lambda: torch.cuda.Event(enable_timing=True)

    def step():
        return quant_f32(xg, al, be, tg, -8, 7, smin, smax, zp_state=zp, sc_state=sc,
                         zp_init=zp_i, sc_init=sc_i, out=out, want_codes=True)

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    marks = []
    t0 = time.perf_counter()
    for _ in range(steps):
        e0, e1 = ev(), ev()
        e0.record(); _, codes, _, _ = step(); e1.record()
        marks.append((e0, e1))
    torch.cuda.synchronize()
    ms_step = (time.perf_counter() - t0) * 1e3 / steps
    k_ms = sum(a.elapsed_time(b) for a, b in marks) / len(marks)

    from oracle import oracle as O
    t0 = time.perf_counter()
    want = O.quant_f32(x.numpy(), *[t.numpy() for t in pf])
    cpu_s = time.perf_counter() - t0
    exact = bool(np.array_equal(codes.cpu().numpy(), want["codes"])
                 and np.array_equal(out.cpu().numpy().view(np.int32), want["xhat"].view(np.int32))
                 and np.array_equal(sc.cpu().numpy().view(np.int32), want["sc"].view(np.int32)))
    bytes_launch = B * T * C * (4 + 4 + 1)          # fp32 in, fp32 out, int8 codes
    achieved = bytes_launch / (k_ms * 1e-3) / 1e9
    res = {
        "metric": "fp32-recurrence tokens quantised/sec (B*T / pass time, one tensor)",
        "value": B * T / (ms_step * 1e-3), "unit": "tokens/s", "n_gpus": 1,
        "steps": steps, "warmup": warmup, "ms_per_step": ms_step,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": f"cfg1 fp32 recurrence: B={B} T={T} C={C} ({H} heads x {D}), 4-bit range, "
                               f"K-shaped input with outlier channels",
                   "batch": B, "heads": H, "head_dim": D, "ctx": T, "bits": 4},
        "bit_exact_vs_oracle": exact,
        "roofline": {"kernel": "adkv_fp32::quant_kernel", "bound": "hbm", "achieved": achieved,
                     "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBPS,
                     "traffic": None},
        "cpu_baseline": {"value": B * T / cpu_s, "unit": "tokens/s", "cores": 1, "kind": "port",
                         "sample": f"C oracle adkv_o_quant_f32 over the whole workload in {cpu_s:.2f} s"},
    }
    return res


def step_kernels(L, B, Hq, H, T, D, bits, n_ckpt_cap, S):
    """The kernels of one decode_step call: one launch; short segments and their combination; or forward_qk, the
    softmax and forward_ov.  The library's first pair of events brackets the first of them, the last pair the last."""
    sizes = (B, Hq, H, T, D, bits, n_ckpt_cap, S)
    n = L.adkv_decode_step_launches(*sizes, 0)
    if n < 3:                      # few short sequences; short segments
        first = L.adkv_decode_step_kernel_name(*sizes, 0).decode()
        return (first,) if n == 1 else (first, "step_combine_kernel")
    qk, ov = (f(*sizes).decode() for f in (L.adkv_decode_kernel_name, L.adkv_decode_ov_kernel_name))
    return "qk_" + qk, "softmax", "ov_" + ov


def decode_record(args, B, Hq, H, D, T, bits, S, NL, steps, warmup, headline=True, bf16=False):
    """Times `steps` decode_step calls (the product path) over NL rotating layer caches and returns
    the bench record.  headline=False leaves out the comparator, the CPU baseline and the graph
    replay (the secondary records of the default run)."""
    import torch
    from adkv_amd import synth
    from adkv_amd.kernel import gemv

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    act = torch.bfloat16 if bf16 else torch.float16   # q, the new token and the output
    ncap = T // S + 1 if S else 0
    kps, vps, kcs, vcs, kks, vks = [], [], [], [], [], []
    state = torch.zeros(B, H, D, 2, dtype=torch.float16, device=dev)
    for l in range(NL):
        kp = synth.make_params(H, D, bits=bits, seed=3, layer=l).to(dev)
        vp = synth.make_params(H, D, bits=bits, seed=4, layer=l).to(dev)
        kc = synth.alloc_cache(B, H, T + 16, D, dev, bits=bits)
        vc = synth.alloc_cache(B, H, T + 16, D, dev, bits=bits)
        kk = torch.zeros(B, H, ncap, D, 2, dtype=torch.float16, device=dev) if S else None
        vk = torch.zeros(B, H, ncap, D, 2, dtype=torch.float16, device=dev) if S else None
        x = synth.make_k(B, H, T, D, layer=l, dtype=torch.float16, device=dev)
        gemv.append_kv(kc, x, *kp.astuple(), 0, state, ckpt=kk, ckpt_interval=S, bits=bits)
        del x
        x = synth.make_v(B, H, T, D, layer=l, dtype=torch.float16, device=dev)
        gemv.append_kv(vc, x, *vp.astuple(), 0, state, ckpt=vk, ckpt_interval=S, bits=bits)
        del x
        kps.append(kp.astuple()); vps.append(vp.astuple()); kcs.append(kc); vcs.append(vc)
        kks.append(kk); vks.append(vk)
        if NL > 8:
            torch.cuda.empty_cache()   # many resident layer caches: keep the input scratch from fragmenting
    q = synth.make_q(B, Hq, D, device=dev).to(act)
    k_new = synth.make_k(B, H, 1, D, seed=11, dtype=torch.float16, device=dev, t0=T).to(act)
    v_new = synth.make_v(B, H, 1, D, seed=12, dtype=torch.float16, device=dev).to(act)
    scaling = D ** -0.5
    torch.cuda.synchronize()
    torch.cuda.empty_cache()

    if args.calibrate_copy and headline:
        a = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        b = torch.empty_like(a)
        for _ in range(3):
            b.copy_(a)
        torch.cuda.synchronize()
        del a, b

    from adkv_amd import _lib
    L = _lib.lib()
    ncap_arg = ncap if S else 0
    kernels = step_kernels(L, B, Hq, H, T, D, bits, ncap_arg, S)
    ws = torch.empty(gemv.decode_step_workspace_bytes(B, Hq, H, T, D, ncap_arg, S), dtype=torch.uint8, device=dev)

    def fused(l):
        # the product path: what KVCacheLayer_ADKV.decode calls, one library call per layer-step
        return gemv.decode_step(q, kcs[l], vcs[l], k_new, v_new, kps[l], vps[l], T, scaling,
                                 k_ckpt=kks[l], v_ckpt=vks[l], ckpt_interval=S, bits=bits, workspace=ws)

    # four events on every `stride`-th timed step, recorded by the library around the stages of the
    # fused call (an event costs the stream some 2 us, 9 us per step with all four: sampled, they
    # tax the step they are meant to describe four times less)
    stride = max(1, min(args.event_stride, steps))
    marks = []
    for _ in range((steps + stride - 1) // stride):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        for x in e:
            x.record()                     # creates the underlying hipEvent_t
        marks.append(e)
    arr4 = _lib.C.c_void_p * 4

    for i in range(warmup):
        fused(i % NL)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(steps):
        if i % stride == 0:
            L.adkv_set_stage_events(arr4(*[x.cuda_event for x in marks[i // stride]]))
        elif i % stride == 1:
            L.adkv_set_stage_events(None)
        fused(i % NL)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    L.adkv_set_stage_events(None)

    ms_step = wall * 1e3 / steps
    qk_ms = sum(e[0].elapsed_time(e[1]) for e in marks) / len(marks)
    sm_ms = sum(e[1].elapsed_time(e[2]) for e in marks) / len(marks)
    ov_ms = sum(e[2].elapsed_time(e[3]) for e in marks) / len(marks)
    dev_ms = sorted(e[0].elapsed_time(e[3]) for e in marks)[len(marks) // 2]

    # the same step as ONE launch (adkv_set_fused_step), where the plans allow it: timed beside the
    # three launches, never as the headline
    fused_ms = None
    if headline and L.adkv_decode_step_is_fused(B, Hq, H, T, D, bits, ncap_arg, S, 0) == 0:
        L.adkv_set_fused_step(1)
        try:
            if L.adkv_decode_step_is_fused(B, Hq, H, T, D, bits, ncap_arg, S, 0) == 1:
                n_fused = max(8, min(steps, 128))
                for i in range(min(warmup, 16)):
                    fused(i % NL)
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                for i in range(n_fused):
                    fused(i % NL)
                torch.cuda.synchronize()
                fused_ms = (time.perf_counter() - t0) * 1e3 / n_fused
        finally:
            L.adkv_set_fused_step(0)

    # the same step replayed from HIP graphs (one per layer cache): no host work between launches
    graph_ms = None
    if args.graph and headline:
        graphs = []
        side = torch.cuda.Stream()
        for l in range(NL):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.stream(side):
                fused(l)
                torch.cuda.synchronize()
                with torch.cuda.graph(g, stream=side):
                    fused(l)
            graphs.append(g)
        torch.cuda.synchronize()
        for i in range(warmup):
            graphs[i % NL].replay()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i in range(steps):
            graphs[i % NL].replay()
        torch.cuda.synchronize()
        graph_ms = (time.perf_counter() - t0) * 1e3 / steps

    qk_kernel = kernels[0]                              # what the first pair of events brackets
    code_bytes = B * H * T * D * bits / 8.0             # one tensor's codes: bytes per QK launch
    achieved = (1 if len(kernels) == 3 else 2) * code_bytes / (qk_ms * 1e-3) / 1e9
    tokens_s = B / (N_LAYERS_MODEL * ms_step * 1e-3)
    workload_key = f"decode B={B} Hq={Hq} H={H} d={D} ctx={T} bits={bits} ckpt={S}"
    traffic = None
    try:
        with open(os.path.join(ROOT, "profiles", "hbm_traffic.json")) as f:
            rec = json.load(f).get(workload_key)
        if rec and rec.get("kernel") == qk_kernel.split(" ")[0].rstrip(","):
            traffic = rec["bytes_per_launch"]
    except (OSError, ValueError):
        pass

    res = {
        "metric": "decode-attention tokens/sec (B / (32 layers * layer-step time))",
        "value": tokens_s,
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f16",
        "data": "synthetic",
        "config": {
            "workload": f"{'cfg2 Llama-2-7B-shaped' if H == Hq else 'grouped-query'} ADKV decode attention: "
                        f"B={B} H={Hq}{'' if H == Hq else f' (KV heads {H})'} d={D} ctx={T} "
                        f"{bits}-bit K+V codes, step = one decode_step call (forward_qk+softmax+forward_ov, "
                        f"appending the new token), {NL} rotating layer caches, state checkpoints every {S} tokens",
            "batch": B, "heads": Hq, "kv_heads": H, "head_dim": D, "ctx": T, "bits": bits, "ckpt_interval": S,
            "parallelism": "1 GPU",
        },
        "kernel_ms": {"forward_qk": qk_ms, "softmax": sm_ms, "forward_ov": ov_ms,
                      "step_device_median": dev_ms, "steps_with_events": len(marks)},
        "step_code_GBps": 2 * code_bytes / (ms_step * 1e-3) / 1e9,
        "roofline": {
            "kernel": qk_kernel,
            "bound": "hbm",
            "achieved": achieved,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBPS,
            # HBM bytes per QK launch from rocprofv3 FETCH_SIZE / WRITE_SIZE scaled by a copy of
            # known size; kept beside the profile it came from (profiles/hbm_traffic.json)
            "traffic": traffic,
        },
    }
    if len(kernels) == 1:
        res["kernel_ms"] = {"one_launch": qk_ms, "step_device_median": dev_ms, "steps_with_events": len(marks)}
    elif len(kernels) == 2:
        res["kernel_ms"] = {"segments": qk_ms, "combine": ov_ms, "step_device_median": dev_ms, "steps_with_events": len(marks)}
        # units of eight tokens that waves of the values' own hold beside the keys'; 0: a wave takes both
        res["step_values_ahead"] = L.adkv_decode_step_values_ahead(B, Hq, H, T, D, bits, ncap_arg, S)
    else:  # the second big launch of the step, same algorithmic bytes (the V codes)
        res["roofline_ov"] = {"kernel": kernels[2], "bound": "hbm", "achieved": code_bytes / (ov_ms * 1e-3) / 1e9,
                              "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": code_bytes / (ov_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                              "note": "forward_ov stage incl. the partial-sum kernel"}
    # what the memory system itself delivers for these kernels' access pattern with nothing else
    # running (a loads-only probe; result and method in profiles/hbm_pattern_ceiling.json)
    try:
        with open(os.path.join(ROOT, "profiles", "hbm_pattern_ceiling.json")) as f:
            ceil = next(iter(json.load(f).values()))
        res["roofline"]["pattern_ceiling"] = {"GBps": ceil["best_GBps"], "frac_of_peak": ceil["best_GBps"] / HBM_PEAK_GBPS,
                                              "achieved_over_ceiling": achieved / ceil["best_GBps"],
                                              "note": "loads only, same access pattern; method and table in profiles/decode_cfg2_ablation.md"}
    except (OSError, ValueError, StopIteration, KeyError):
        pass
    if fused_ms is not None:
        res["one_launch_step"] = {"ms_per_step": fused_ms, "tokens_per_s": B / (N_LAYERS_MODEL * fused_ms * 1e-3),
                                  "note": "adkv_decode_step with adkv_set_fused_step(1): forward_qk, softmax and forward_ov "
                                          "in one launch (decode_ft_kernel), no stage events, timed after the default three "
                                          "launches, which are the headline, on a device that has come up to its clock "
                                          "since (in turn with them it is the slower one)"}
    if graph_ms is not None:
        res["graph_replay"] = {"ms_per_step": graph_ms, "tokens_per_s": B / (N_LAYERS_MODEL * graph_ms * 1e-3),
                               "note": "the same decode_step step captured once per layer cache and replayed"}
    # The binding roof of these kernels is vector-instruction issue, not HBM: vector instructions
    # per launch (profiles/valu_issue.json, from rocprofv3 SQ_INSTS_VALU) x 4 cycles per wave64
    # instruction / (1024 SIMDs x the kernel's live duration), priced once at the shader clock the
    # device held under this load when the counters were taken and once at the 2.4 GHz it is sold at.
    try:
        with open(os.path.join(ROOT, "profiles", "valu_issue.json")) as f:
            vrec = json.load(f).get(workload_key)
        if vrec and vrec.get("kernel") == qk_kernel.split(" ")[0].rstrip(","):
            slots = vrec["valu_insts_per_launch"] * 4.0 / 1024.0          # issue cycles per SIMD
            res["roofline_valu"] = {
                "kernel": qk_kernel, "bound": "valu",
                "achieved": vrec["valu_insts_per_launch"] / (qk_ms * 1e-3) / 1e12,
                "peak": 1024 * 2.4e9 / 4.0 / 1e12, "unit": "T wave64 instructions/s",
                "frac": slots / (qk_ms * 1e-3 * 2.4e9),
                "frac_at_clock_under_load": slots / (qk_ms * 1e-3 * vrec["shader_clock_hz"]),
                "clock_under_load_GHz": vrec["shader_clock_hz"] / 1e9,
                "valu_busy_measured": vrec["valu_busy"],
                "note": "peak and frac at the 2.4 GHz peak engine clock; frac_at_clock_under_load at the shader clock "
                        "of the counter run (SQ_BUSY_CYCLES / duration: the device holds 1.8-2.15 GHz under this "
                        "kernel, not 2.4); valu_busy_measured = SQ_ACTIVE_INST_VALU x 4 / (busy cycles x 1024 SIMDs) "
                        "in that run; instruction count from profiles/valu_issue.json, duration live"}
            res["roofline"]["binding_roof"] = (
                "vector-instruction issue (see roofline_valu): HBM is the nominal roof of this path, code bytes "
                "against 8 TB/s, but a bit-exact fp16 replay needs six packed instructions per channel pair and token, "
                "and the vector pipe is busy %.0f %% of the cycles at the clock the device sustains"
                % (100 * vrec["valu_busy"]))
    except (OSError, ValueError):
        pass
    if headline and not args.no_fp16_comparator and D == 128 and H == Hq and bits == 4:
        res["fp16_kv_comparator"] = fp16_comparator(args, dev, ms_step)
    if headline and not args.no_cpu_baseline and H == Hq and bits == 4:
        res["cpu_baseline"] = cpu_baseline(args, T, D)
    del kcs, vcs, kks, vks, ws
    torch.cuda.empty_cache()
    return res



def secondary_records(args):
    """Short runs of the other named workloads in the same process, so that one default run shows
    them all: the streaming quantiser (cfg3), the long-context grouped-query 2-bit decode (cfg5), the
    fp32 recurrence (cfg1) and the end-to-end generate of cfg4.  The first three are what
    `--workload ...` prints with fewer steps and without the host baselines; a failure in one is
    reported in its place and does not touch the headline."""
    import torch
    out = {}

    def run(name, fn):
        try:
            out[name] = fn()
        except Exception as e:  # noqa: BLE001 - reported, the headline line must still print
            out[name] = {"error": f"{type(e).__name__}: {e}"}
        torch.cuda.synchronize()
        torch.cuda.empty_cache()

    def cfg3():
        r = encode_record(args, 8, 32768, steps=5, warmup=2, cpu=False)
        return {"workload": r["config"]["workload"], "ms_per_tensor": r["ms_per_step"],
                "tokens_quantised_per_s": r["value"], "append_us_per_token_step": r["append_us_per_token_step"],
                "kv_pair": r["kv_pair"], "codes_bit_exact_vs_oracle": r["codes_bit_exact_vs_oracle"],
                "roofline": r["roofline"]}

    def cfg5():
        r = decode_record(args, 16, 32, 8, 128, 131072, 2, 256, 2, steps=48, warmup=16, headline=False, bf16=True)
        # with 2-bit codes the replay costs what it costs with 4-bit ones on half the bytes: the roof
        # that binds is vector issue, and the record says so; the HBM figure is kept beside it
        out5 = {"workload": r["config"]["workload"], "ms_per_step": r["ms_per_step"], "tokens_per_s": r["value"],
                "kernel_ms": r["kernel_ms"]}
        if "roofline_valu" in r:
            out5["roofline"] = r["roofline_valu"]
            out5["roofline_hbm"] = r["roofline"]
        else:
            out5["roofline"] = r["roofline"]
        return out5

    def cfg1():
        r = quant_f32_record(args, 1, 1024, steps=20, warmup=3)
        return {"workload": r["config"]["workload"], "ms_per_pass": r["ms_per_step"], "tokens_per_s": r["value"],
                "bit_exact_vs_oracle": r["bit_exact_vs_oracle"], "roofline": r["roofline"],
                "cpu_baseline": r["cpu_baseline"]}

    def cfg4():
        # the reference's tools/perf_e2e.py protocol on the configuration's shape: random-init
        # Llama-2-7B geometry in fp16, batch 128, 512 random prompt ids, 256 greedy tokens through
        # transformers' generate with the ADKV cache (one timed repeat after a 4-token warm-up); the
        # largest batch at ctx 4096 by the reference's memory accounting beside it
        from adkv_amd.tools import perf_e2e
        a = perf_e2e.parse_args(["--kv", "adkv", "--batch_size", "128", "--prompt_lenth", "512",
                                 "--output_length", "256", "--num_repeats", "1"])
        r = perf_e2e.generate_run(a)
        m = perf_e2e.max_batch(perf_e2e.parse_args(["--prompt_lenth", "3840", "--output_length", "256"]))
        return {"workload": "end-to-end greedy generate, random-init Llama-2-7B geometry (32 layers, fp16 weights), "
                            "B=128, 512-token prompt, 256 new tokens, ADKV 4-bit cache",
                "generated_tokens_per_s": r["generated_tokens_per_s"], "seconds_per_generate": r["used_time_ms"] / 1e3,
                "peak_mem_GiB": r["peak_mem_GiB"], "adkv_params": r["adkv_params"],
                "max_batch_ctx4096_by_memory_model": {"adkv": m["max_batch_adkv"], "fp16": m["max_batch_fp16"]}}

    run("cfg3_streaming_quantiser", cfg3)
    run("cfg5_long_context_gqa_2bit", cfg5)
    run("cfg1_fp32_recurrence", cfg1)
    if not args.no_e2e:
        run("cfg4_end_to_end_generate", cfg4)
    return out


def main():
    args = parse()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build measures one GPU only (the path shards over batch/heads with no "
              "exchange; nothing multi-GPU is built). Run with --gpus 1.", file=sys.stderr)
        sys.exit(2)

    if args.workload == "encode":
        res = encode_record(args, 8 if args.batch == 128 else args.batch, 32768 if args.ctx == 4096 else args.ctx,
                            args.steps, args.warmup, cpu=not args.no_cpu_baseline)
    elif args.workload == "quant_f32":
        res = quant_f32_record(args, 1 if args.batch == 128 else args.batch,
                               1024 if args.ctx == 4096 else args.ctx, args.steps, args.warmup)
    else:
        Hq = args.heads
        res = decode_record(args, args.batch, Hq, args.kv_heads or Hq, args.dim, args.ctx, args.bits,
                            args.ckpt_interval, args.layer_buffers, args.steps, args.warmup, bf16=args.bf16)
        default_shape = (args.batch, Hq, args.kv_heads or Hq, args.dim, args.ctx, args.bits) == \
            (128, 32, 32, 128, 4096, 4)
        if default_shape and not args.no_secondary:
            res["secondary"] = secondary_records(args)
    print(json.dumps(res))




if __name__ == "__main__":
    main()
