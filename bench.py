"""Prefill / encoder benchmarks on one MI355X.

Default workload (`--workload kev`): the Kev/Qwen3.5 hybrid scoring forward (hidden 1024,
24 layers = 3 Gated DeltaNet : 1 gated GQA attention, attention 16/8 heads x 128, GDN 16 heads x
128, SwiGLU 3584, vocab 151936, decision head over 8 choices) on a batch of 64 sequences x 512
seeded token ids, random-init weights N(0, 0.02) in the model dtype, KV pages of 16 tokens from a
seeded permutation of the pool. One step = one full forward of the 32,768 tokens (every layer,
every token) plus the decision logits; inputs are resident in HBM before timing starts.

`--workload laya`: the ModernBERT-base-shaped encoder (hidden 768, 22 layers, 12 heads x 64,
global attention every third layer with RoPE theta 160000, the rest a +-64 sliding window with
theta 10000, GeGLU 1152, mean-pooled head over 4 labels) on an unpadded varlen batch of 16
sequences with seeded lengths in [256, 4096]. One step = one encoder forward of the whole batch.

Prints one JSON line: whole-job tokens/s, the live-measured roofline of the attention kernel
(MFMA-bound, bf16 dense peak 2.5 PFLOP/s) and, for Kev, of the delta-rule kernel (HBM-bound,
8 TB/s), and the CPU oracle's forward timed on this host's cores as a reported baseline. The
default Kev run also measures the Laya workload (same steps and warmup) and adds its tokens/s and
attention rooflines to the line as `laya` (`--no-laya` skips it).
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

SEED = 20261201
MFMA_PEAK_BF16 = 2.5e15   # dense bf16 / fp16 MFMA, FLOP/s
FP32_PEAK = 157.3e12      # fp32 matrix / vector, FLOP/s
HBM_PEAK = 8.0e12         # bytes/s
# FLOPs of one 64-token chunk of the chunked delta rule for one head (dk = dv = 128): K K^T and
# Q K^T (2 x 64 x 64 x 128 x 2), K S0 and Q S0 (2 x 64 x 128 x 128 x 2), T R
# (64 x 64 x 128 x 2), the triangular inverse (64^3 / 3 x 2), Aqk delta (64 x 64 x 128 x 2) and
# the state update K^T delta (128 x 64 x 128 x 2): 10.66 MFLOP
GDN_CHUNK_FLOPS = 4 * 64 * 64 * 128 * 2 + 3 * 64 * 128 * 128 * 2 + 64 ** 3 / 3 * 2


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--workload", default="kev", choices=["kev", "laya"])
    p.add_argument("--steps", type=int, default=10)
    p.add_argument("--warmup", type=int, default=3)
    p.add_argument("--batch", type=int, default=0, help="sequences (default 64 for kev, 16 for laya)")
    p.add_argument("--seq-len", type=int, default=512, help="kev: tokens per sequence")
    p.add_argument("--dtype", default="bf16", choices=["bf16", "fp16"])
    p.add_argument("--residual", default="bf16", choices=["bf16", "fp32"],
                   help="kev: residual stream dtype of the timed model (bf16 rounds it after every residual add, as "
                        "the reference stores it; fp32 keeps it in fp32); the other mode is timed beside it")
    p.add_argument("--kernel-iters", type=int, default=20)
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--fork-probe", action="store_true",
                   help="time attention on a suffix batch over a shared prefix, and on private prefix copies")
    p.add_argument("--no-laya", action="store_true",
                   help="kev: skip the Laya encoder measurement that the default run adds to its line")
    p.add_argument("--kernels-only", action="store_true",
                   help="time only the roofline kernels (no model; for counter collection)")
    p.add_argument("--copy-probe", type=int, default=0, metavar="BYTES",
                   help="copy BYTES device-to-device 3 times and exit (HBM counter calibration)")
    p.add_argument("--gemm-probe", action="store_true",
                   help="time the own GEMM (hk_linear) at the Kev forward's projection shapes")
    p.add_argument("--attention-probe", action="store_true",
                   help="time paged attention at head widths 256 and 128 (same FLOPs) for both 16-bit types")
    p.add_argument("--cpu-threads", type=int, default=0)
    return p.parse_args()


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def time_launches(fn, iters, stream):
    """Average duration (s) of `fn` launches measured with events on the launch stream."""
    import torch

    fn()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for _ in range(iters):
        fn()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) / 1e3 / iters


def kernel_rooflines(ctx, shape, n_seqs, seq_len, dtype, iters):
    """Times the attention and delta-rule kernels alone on inputs of the forward's shapes and
    layouts (fused-projection q/gate strides, paged pools, token-major GDN inputs)."""
    import numpy as np
    import torch

    from huncho_amd import abi
    from huncho_amd.ops import gated_delta_chunked, gdn_fused, paged_prefill_attention, qk_norm_rope_kv_write

    dev = torch.device("cuda", 0)
    stream = torch.cuda.current_stream(dev)
    n = n_seqs * seq_len
    hq, hkv, d, P = shape.n_heads, shape.n_kv_heads, shape.head_dim, shape.page_size
    rows = 2 * hq * d + 2 * hkv * d
    g = torch.Generator(device=dev).manual_seed(SEED)
    qkv = torch.randn((n, rows), generator=g, device=dev, dtype=torch.float32).to(dtype)
    cu = torch.arange(0, n + 1, seq_len, dtype=torch.int32, device=dev)
    lens = torch.full((n_seqs,), seq_len, dtype=torch.int32, device=dev)
    pages_per = seq_len // P
    perm = abi.synth_permutation(SEED, 5, n_seqs * pages_per)
    bt = torch.from_numpy(perm.reshape(n_seqs, pages_per).copy()).to(dev)
    kp = torch.zeros((n_seqs * pages_per, hkv, P, d), dtype=dtype, device=dev)
    vp = torch.zeros_like(kp)
    cs, sn = abi.rope_table(d, shape.rope_theta, seq_len, True)
    w1 = torch.ones(d, device=dev)
    q = qkv[:, : 2 * hq * d].view(n, hq, 2 * d)[:, :, :d]
    gate = qkv[:, : 2 * hq * d].view(n, hq, 2 * d)[:, :, d:]
    k_in = qkv[:, 2 * hq * d: 2 * hq * d + hkv * d].view(n, hkv, d)
    v_in = qkv[:, 2 * hq * d + hkv * d:].view(n, hkv, d)
    qk_norm_rope_kv_write(ctx, q, k_in, v_in, w1, w1, shape.eps, torch.from_numpy(cs).to(dev),
                          torch.from_numpy(sn).to(dev), d, cu, lens, bt, kp, vp, q)
    out = torch.empty((n, hq, d), dtype=dtype, device=dev)
    t_attn = time_launches(lambda: paged_prefill_attention(ctx, q, kp, vp, bt, cu, lens, seq_len, gate=gate,
                                                           out=out), iters, stream)
    attn_flops = 4.0 * hq * d * seq_len * (seq_len + 1) / 2 * n_seqs
    attn_bytes = n * (3 * hq + 2 * hkv) * d * 2  # Q, K, V, O and the output gate rows

    # the varlen paged GQA prefill batch: 32 sequences with seeded lengths in [64, 2048], pages
    # of 16 from a seeded permutation of a 4096-page pool (the compute-bound attention shape)
    vl = [int(x) for x in abi.synth_uniform_int(20261201, 20, 32, 64, 2048)]
    vn = sum(vl)
    vcu = torch.from_numpy(np.concatenate([[0], np.cumsum(vl)]).astype(np.int32)).to(dev)
    vlens = torch.tensor(vl, dtype=torch.int32, device=dev)
    vperm = abi.synth_permutation(20261201, 11, 4096)
    vneed = [(L + P - 1) // P for L in vl]
    vbt_np = np.full((32, max(vneed)), -1, np.int32)
    k0 = 0
    for s_, m_ in enumerate(vneed):
        vbt_np[s_, :m_] = vperm[k0:k0 + m_]
        k0 += m_
    vbt = torch.from_numpy(vbt_np).to(dev)
    vkp = torch.randn((4096, hkv, P, d), generator=g, device=dev, dtype=torch.float32).to(dtype)
    vvp = torch.randn((4096, hkv, P, d), generator=g, device=dev, dtype=torch.float32).to(dtype)
    vq = torch.randn((vn, hq, d), generator=g, device=dev, dtype=torch.float32).to(dtype)
    vo = torch.empty_like(vq)
    t_var = time_launches(lambda: paged_prefill_attention(ctx, vq, vkp, vvp, vbt, vcu, vlens, max(vl), out=vo),
                          iters, stream)
    var_flops = sum(4.0 * hq * d * L * (L + 1) / 2 for L in vl)
    var_bytes = vn * (2 * hq + 2 * hkv) * d * 2
    del vkp, vvp, vq, vo

    # the fused Gated DeltaNet layer kernel the forward runs: in_proj rows [q | k | v | z]
    # (8192 columns) and [b | a] rows as the GEMMs write them, conv weights, A_log, dt_bias
    H, Hk = shape.lin_n_v_heads, shape.lin_n_k_heads
    conv_dim = shape.conv_dim
    mixed = (torch.randn((n, conv_dim + H * 128), generator=g, device=dev) * 0.5).to(dtype)
    ba = torch.randn((n, 2 * H), generator=g, device=dev).to(dtype)
    conv_w = (torch.randn((conv_dim, 4), generator=g, device=dev) * 0.3).to(dtype).float()
    base_g = -torch.exp(torch.randn(H, generator=g, device=dev) * 0.1)
    dt_bias = torch.randn(H, generator=g, device=dev) * 0.1
    norm_w = 1.0 + torch.randn(128, generator=g, device=dev) * 0.02
    z = mixed[:, conv_dim:]
    fo = torch.empty((n, H, 128), dtype=dtype, device=dev)
    t_fused = time_launches(lambda: gdn_fused(ctx, mixed, conv_w, ba, 0, H, base_g, dt_bias, z, norm_w, shape.eps,
                                              cu, H, Hk, out=fo), iters, stream)
    # per (token, head): q, k, v raw rows 3 x 256 B + z 256 B + b, a 4 B + output 256 B
    fused_bytes = n * H * (3 * 256 + 256 + 4 + 256)

    qg = torch.nn.functional.normalize(torch.randn((n, Hk, 128), generator=g, device=dev), dim=-1)
    kg = torch.nn.functional.normalize(torch.randn((n, Hk, 128), generator=g, device=dev), dim=-1).to(dtype)
    qg = (qg * 128 ** -0.5).to(dtype)
    vg = torch.randn((n, H, 128), generator=g, device=dev).to(dtype)
    gg = -torch.nn.functional.softplus(torch.randn((n, H), generator=g, device=dev)) * 0.5
    bb = torch.sigmoid(torch.randn((n, H), generator=g, device=dev))
    og = torch.empty_like(vg)
    t_gdn = time_launches(lambda: gated_delta_chunked(ctx, qg, kg, vg, gg, bb, cu, out=og), iters, stream)
    gdn_bytes = n * H * (4 * 128 * 2 + 8)
    chunks = math.ceil(seq_len / 64) * n_seqs * H
    gdn_flops = chunks * GDN_CHUNK_FLOPS
    torch.cuda.synchronize()
    return {
        "attention": {"seconds": t_attn, "flops": attn_flops, "bytes": attn_bytes},
        "attention_varlen": {"seconds": t_var, "flops": var_flops, "bytes": var_bytes},
        "delta_rule_fused": {"seconds": t_fused, "flops": gdn_flops, "bytes": fused_bytes},
        "delta_rule": {"seconds": t_gdn, "flops": gdn_flops, "bytes": gdn_bytes},
    }


def fp32_config_kernels(ctx, iters):
    """GPU times of the two fp32 correctness configurations, beside their CPU baselines:
    config 1, GQA causal attention (1 x 256 tokens, 16/8 heads x 128, RoPE theta 1e7, pages of 16
    with an identity table), and config 2, the gated delta rule (1 x 512 tokens, 16 heads x 128,
    chunk 64, fp32 state, final state written). FLOPs and bytes as the survey counts them:
    attention 4 Hq d T(T+1)/2 and Q, K, V, O; the delta rule's recurrence 7 dk dv + 2 dv per
    token and head (the chunked form's own count beside it) and q, k, v, o, g, beta, S_final."""
    import numpy as np
    import torch

    from huncho_amd import abi
    from huncho_amd.ops import gated_delta_chunked, paged_prefill_attention, qk_norm_rope_kv_write

    dev = torch.device("cuda", 0)
    stream = torch.cuda.current_stream(dev)
    T, hq, hkv, d, P = 256, 16, 8, 128, 16
    q = torch.from_numpy(abi.synth_normal(SEED, 31, T * hq * d).reshape(T, hq, d)).to(dev)
    k = torch.from_numpy(abi.synth_normal(SEED, 32, T * hkv * d).reshape(T, hkv, d)).to(dev)
    v = torch.from_numpy(abi.synth_normal(SEED, 33, T * hkv * d).reshape(T, hkv, d)).to(dev)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    lens = torch.tensor([T], dtype=torch.int32, device=dev)
    bt = torch.arange(T // P, dtype=torch.int32, device=dev).view(1, -1)
    kp = torch.zeros((T // P, hkv, P, d), dtype=torch.float32, device=dev)
    vp = torch.zeros_like(kp)
    cs, sn = abi.rope_table(d, 1e7, T, False)
    qk_norm_rope_kv_write(ctx, q, k, v, None, None, 0.0, torch.from_numpy(cs).to(dev), torch.from_numpy(sn).to(dev),
                          d, cu, lens, bt, kp, vp, q)
    o = torch.empty_like(q)
    t_attn = time_launches(lambda: paged_prefill_attention(ctx, q, kp, vp, bt, cu, lens, T, out=o), iters, stream)
    attn_flops = 4.0 * hq * d * T * (T + 1) / 2
    attn_bytes = T * (2 * hq + 2 * hkv) * d * 4

    T2, H = 512, 16
    g = torch.Generator(device=dev).manual_seed(SEED)
    qg = torch.nn.functional.normalize(torch.randn((T2, H, 128), generator=g, device=dev), dim=-1) * 128 ** -0.5
    kg = torch.nn.functional.normalize(torch.randn((T2, H, 128), generator=g, device=dev), dim=-1)
    vg = torch.randn((T2, H, 128), generator=g, device=dev)
    beta = torch.sigmoid(torch.randn((T2, H), generator=g, device=dev))
    gg = -torch.nn.functional.softplus(torch.randn((T2, H), generator=g, device=dev)) * 0.5
    cu2 = torch.tensor([0, T2], dtype=torch.int32, device=dev)
    og = torch.empty_like(vg)
    st = torch.empty((1, H, 128, 128), dtype=torch.float32, device=dev)
    t_gdn = time_launches(lambda: gated_delta_chunked(ctx, qg, kg, vg, gg, beta, cu2, final_state=st, out=og),
                          iters, stream)
    rec_flops = T2 * H * (7 * 128 * 128 + 2 * 128)
    chunk_flops = (T2 // 64) * H * GDN_CHUNK_FLOPS
    gdn_bytes = 4 * T2 * H * 128 * 4 + 2 * T2 * H * 4 + H * 128 * 128 * 4
    torch.cuda.synchronize()

    def entry(kernel, t, flops, nbytes, extra=None):
        e = {"kernel": kernel, "us_per_launch": round(t * 1e6, 2), "tflops": round(flops / t / 1e12, 3),
             "frac_of_fp32_peak": round(flops / t / FP32_PEAK, 4), "gbps": round(nbytes / t / 1e9, 1),
             "frac_of_hbm": round(nbytes / t / HBM_PEAK, 4), "flops_per_launch": flops, "bytes_per_launch": nbytes}
        e.update(extra or {})
        return e

    return {
        "attention_fp32_T256": entry("paged_prefill_attn_f32 (1 x 256, 16q/8kv x 128, P 16 identity table)",
                                     t_attn, attn_flops, attn_bytes),
        "delta_rule_fp32_T512": entry("delta_split_prep, _scan and _out (1 x 512, 16 x 128, chunk 64, final state)", t_gdn, rec_flops,
                                      gdn_bytes, {"chunked_tflops": round(chunk_flops / t_gdn / 1e12, 3)}),
    }


def forward_kernel_times(run_forward, names):
    """Average device durations (us) and launch counts of the kernels whose names contain each
    of `names`, inside one call of run_forward, from the torch profiler's device activity (the
    ROCm tracer records the library's own launches too). None when the profiler yields no
    device events."""
    import torch

    try:
        from torch.profiler import ProfilerActivity, profile

        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            run_forward()
            torch.cuda.synchronize()
        out = {}
        for key, pat in names.items():
            durs = [e.device_time for e in prof.events() if pat in e.name and e.device_time > 0]
            if durs:
                out[key] = {"us_avg": round(sum(durs) / len(durs), 2), "launches": len(durs)}
        return out or None
    except Exception as e:  # the profiler is optional here
        log(f"in-forward kernel times unavailable: {e}")
        return None


def kev_forward_flops(shape, lengths):
    """Algorithmic FLOPs of one Kev forward: the projections (2 per weight per token, unpadded
    widths), causal attention (4 Hq d per visible (query, key) pair) and the chunked delta rule
    (GDN_CHUNK_FLOPS per 64-token chunk and head)."""
    H, I, d = shape.hidden, shape.intermediate, shape.head_dim
    Hv = shape.lin_n_v_heads
    vd = Hv * shape.lin_v_dim
    n = sum(lengths)
    gemm = attn = gdn = 0.0
    for t in shape.layer_types:
        gemm += 2.0 * n * (H * 2 * I + I * H)  # MLP gate|up, down
        if t == 0:
            gemm += 2.0 * n * (H * (shape.conv_dim + vd + 2 * Hv) + vd * H)
            gdn += sum(math.ceil(L / 64) for L in lengths) * Hv * GDN_CHUNK_FLOPS
        else:
            gemm += 2.0 * n * (H * (2 * shape.n_heads * d + 2 * shape.n_kv_heads * d) + shape.n_heads * d * H)
            attn += sum(4.0 * shape.n_heads * d * L * (L + 1) / 2 for L in lengths)
    return {"gemm": gemm, "attention": attn, "delta_rule": gdn, "total": gemm + attn + gdn}


def host_info():
    """This host's CPU as the baseline legs see it: logical CPUs (nproc), the CPUs this process
    may run on (its affinity mask) and the model name from /proc/cpuinfo."""
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        affinity = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        affinity = os.cpu_count() or 1
    return {"nproc": os.cpu_count() or 1, "affinity": affinity, "model": model}


def default_threads(args):
    """All-core leg threads: the affinity mask, capped at 16 (the host CPU share of one GPU)."""
    return args.cpu_threads or max(1, min(16, host_info()["affinity"]))


def timed(fn):
    t0 = time.perf_counter()
    fn()
    return time.perf_counter() - t0


def gemm_probe(iters, tokens):
    """The own GEMM (hk_linear: gemm.hip) at the Kev forward's five projection shapes, each
    timed over `iters` launches with HIP events on torch's stream: GDN q|k|v|z and attention
    q|gate|k|v (store), MLP gate|up with the fused SwiGLU epilogue, out_proj / o_proj and down_proj
    with the fused residual add. Beside each: torch.matmul on the same operands (hipBLASLt with
    torch's own heuristic choice; the forward's pinned solutions are in its kernel trace), and
    for SwiGLU also the separate swiglu pass (hk_swiglu) the forward runs after its GEMM."""
    import torch

    from huncho_amd import abi
    from huncho_amd.kev import KevShape
    from huncho_amd.ops import context_for_torch

    sh = KevShape()
    ctx = context_for_torch(0)
    L = abi.lib()
    g = torch.Generator(device="cuda").manual_seed(SEED)
    M, H, I = tokens, sh.hidden, sh.intermediate
    qkvz = 2 * sh.lin_n_k_heads * sh.lin_key_dim + 2 * sh.lin_n_v_heads * sh.lin_v_dim
    qkv = 2 * sh.n_heads * sh.head_dim + 2 * sh.n_kv_heads * sh.head_dim
    shapes = [("gdn_qkvz", qkvz, H, 0), ("attn_qkv", qkv, H, 0), ("mlp_gate_up_swiglu", 2 * I, H, 2),
              ("out_proj_residual", H, sh.n_heads * sh.head_dim, 1), ("down_proj_residual", H, I, 1)]

    def timed(fn):
        fn()
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(iters):
            fn()
        e.record()
        e.synchronize()
        return s.elapsed_time(e) / iters * 1e3

    out = {}
    for name, n, k, epi in shapes:
        x = (torch.randn((M, k), generator=g, device="cuda") * 0.5).bfloat16()
        w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).bfloat16()
        oc = n // 2 if epi == 2 else n
        y = torch.empty((M, oc), dtype=torch.bfloat16, device="cuda")
        c = torch.randn((M, n), generator=g, device="cuda").bfloat16() if epi == 1 else None

        def own():
            ctx.check(L.hk_linear(ctx.h, abi.HK_BF16, epi, x.data_ptr(), k, w.data_ptr(), k, M, n, k,
                                  c.data_ptr() if c is not None else None, n if c is not None else 0,
                                  y.data_ptr(), oc))

        t_own = timed(own)
        if epi == 1:
            t_blas = timed(lambda: torch.addmm(c, x, w.T))
        else:
            t_blas = timed(lambda: torch.matmul(x, w.T))
        flops = 2.0 * M * n * k
        r = {"own_us": round(t_own, 1), "own_tflops": round(flops / t_own / 1e6), "torch_hipblaslt_us": round(t_blas, 1)}
        if epi == 2:
            gu = torch.empty((M, n), dtype=torch.bfloat16, device="cuda")
            t_sw = timed(lambda: ctx.check(L.hk_swiglu(ctx.h, abi.HK_BF16, gu.data_ptr(), n, I, M, I, y.data_ptr())))
            r["swiglu_pass_us"] = round(t_sw, 1)
        out[name] = r
    print(json.dumps({"gemm_probe": {"tokens": M, "dtype": "bf16", "shapes": out}}), flush=True)


def attention_probe(iters, n_seqs, seq_len):
    """Fresh causal prefill of n_seqs rows of seq_len tokens through pages of 16 (identity block
    tables), bf16 and fp16, at Qwen3.5's default 256-wide heads (q/kv heads 16/4, 8/2, 16/2) and at
    128-wide heads with the FLOPs of the first (32/8). Each shape is timed over `iters` launches with
    HIP events on torch's stream; FLOPs are the causal 4·Hq·d·L(L+1)/2 per row."""
    import torch

    from huncho_amd.ops import context_for_torch, paged_prefill_attention

    ctx = context_for_torch(0)
    g = torch.Generator(device="cuda").manual_seed(SEED)
    P = 16
    pages = n_seqs * ((seq_len + P - 1) // P)
    bt = torch.arange(pages, dtype=torch.int32, device="cuda").reshape(n_seqs, -1)
    cu = torch.arange(0, n_seqs * seq_len + 1, seq_len, dtype=torch.int32, device="cuda")
    cl = torch.full((n_seqs,), seq_len, dtype=torch.int32, device="cuda")
    out = []
    for dt, name in ((torch.bfloat16, "bf16"), (torch.float16, "fp16")):
        for d, hq, hkv in ((256, 16, 4), (256, 8, 2), (256, 16, 2), (128, 32, 8)):
            kp = torch.randn((pages, hkv, P, d), generator=g, device="cuda").to(dt)
            vp = torch.randn((pages, hkv, P, d), generator=g, device="cuda").to(dt)
            q = torch.randn((n_seqs * seq_len, hq, d), generator=g, device="cuda").to(dt)
            o = torch.empty_like(q)

            def run():
                paged_prefill_attention(ctx, q, kp, vp, bt, cu, cl, seq_len, out=o)

            run()
            torch.cuda.synchronize()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            for _ in range(iters):
                run()
            e.record()
            e.synchronize()
            us = s.elapsed_time(e) / iters * 1e3
            flops = 4.0 * hq * d * n_seqs * seq_len * (seq_len + 1) / 2
            out.append({"dtype": name, "head_dim": d, "q_heads": hq, "kv_heads": hkv, "us": round(us, 1),
                        "tflops": round(flops / us / 1e6, 1)})
    if ctx.take_faults():
        raise RuntimeError("attention probe raised a device fault flag")
    print(json.dumps({"attention_probe": {"rows": n_seqs, "seq_len": seq_len, "page_size": P, "shapes": out}}),
          flush=True)


def fork_probe(iters):
    """A suffix batch over one shared prefix (the reference's attention_suffix_batch case,
    kv_pages.rs:180-296): 8 rows whose block tables point at the same 32 prefix pages (512 tokens)
    plus 2 private pages each for a 24-token suffix, against the same batch with a private copy
    of the prefix per row. Times both launches; under `rocprofv3 --pmc FETCH_SIZE` the two
    dispatches give the HBM bytes each reads."""
    import numpy as np
    import torch

    from huncho_amd import abi
    from huncho_amd.kev import KevShape
    from huncho_amd.ops import context_for_torch, paged_prefill_attention

    shape = KevShape()
    hq, hkv, d, P = shape.n_heads, shape.n_kv_heads, shape.head_dim, shape.page_size
    rows, prefix, suffix = 8, 512, 24
    ctx_len = prefix + suffix
    pp, sp = prefix // P, (suffix + P - 1) // P
    dev = torch.device("cuda", 0)
    ctx = context_for_torch(0)
    g = torch.Generator(device=dev).manual_seed(SEED)
    n_pages = rows * (pp + sp)
    perm = abi.synth_permutation(SEED, 17, n_pages)
    kp = torch.randn((n_pages, hkv, P, d), generator=g, device=dev).to(torch.bfloat16)
    vp = torch.randn((n_pages, hkv, P, d), generator=g, device=dev).to(torch.bfloat16)
    shared = np.zeros((rows, pp + sp), np.int32)
    private = np.zeros((rows, pp + sp), np.int32)
    for r in range(rows):
        shared[r, :pp] = perm[:pp]  # every row reads the same prefix pages
        shared[r, pp:] = perm[rows * pp + r * sp: rows * pp + (r + 1) * sp]
        private[r] = perm[r * (pp + sp): (r + 1) * (pp + sp)]
    # the private batch holds the same prefix values in its own pages
    src = torch.from_numpy(shared.reshape(-1).astype(np.int64)).to(dev)
    dst = torch.from_numpy(private.reshape(-1).astype(np.int64)).to(dev)
    kp2, vp2 = kp.clone(), vp.clone()
    kp2[dst] = kp[src]
    vp2[dst] = vp[src]
    n = rows * suffix
    qg = torch.randn((n, hq, 2 * d), generator=g, device=dev).to(torch.bfloat16)
    q, gate = qg[:, :, :d], qg[:, :, d:]
    cu = torch.arange(0, n + 1, suffix, dtype=torch.int32, device=dev)
    lens = torch.full((rows,), ctx_len, dtype=torch.int32, device=dev)
    o1 = torch.empty((n, hq, d), dtype=torch.bfloat16, device=dev)
    o2 = torch.empty_like(o1)
    bt1 = torch.from_numpy(shared).to(dev)
    bt2 = torch.from_numpy(private).to(dev)
    stream = torch.cuda.current_stream(dev)
    t1 = time_launches(lambda: paged_prefill_attention(ctx, q, kp, vp, bt1, cu, lens, suffix, gate=gate, out=o1),
                       iters, stream)
    t2 = time_launches(lambda: paged_prefill_attention(ctx, q, kp2, vp2, bt2, cu, lens, suffix, gate=gate, out=o2),
                       iters, stream)
    torch.cuda.synchronize()
    page_bytes = hkv * P * d * 2 * 2  # K and V of one page, all KV heads
    line = {"probe": "suffix batch over a shared prefix", "rows": rows, "prefix_tokens": prefix,
            "suffix_tokens": suffix, "identical_outputs": bool(torch.equal(o1, o2)),
            "shared_us": round(t1 * 1e6, 2), "private_us": round(t2 * 1e6, 2),
            "kv_bytes_unique_shared": (pp + rows * sp) * page_bytes,
            "kv_bytes_unique_private": rows * (pp + sp) * page_bytes,
            "q_gate_o_bytes": n * hq * d * 2 * 3}
    # forward_fork_batch at its row limit on the Kev model: 63 branches of a 448-token prefix,
    # 64 new tokens each (the cache allocates its state slots up front, so the forks and
    # releases are host bookkeeping plus one state copy per branch)
    from huncho_amd.kev import KevCache, KevModel, synthetic_weights

    model = KevModel(ctx, shape, synthetic_weights(shape, SEED), torch.bfloat16)
    cache = KevCache(model, max_pages=448 // P + 63 * 4 + 8)
    ids = abi.synth_uniform_int(SEED, 901, 64 * 512, 0, shape.vocab - 1)
    parent = cache.prefill(ids[:448].tolist())
    suffixes = [ids[r * 512 + 448:(r + 1) * 512].tolist() for r in range(63)]
    cache.fork_batch(parent, suffixes, 1.3)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    reps = 5
    for _ in range(reps):
        cache.fork_batch(parent, suffixes, 1.3)
    torch.cuda.synchronize()
    t_batch = (time.perf_counter() - t0) / reps
    t0 = time.perf_counter()
    for _ in range(reps):
        branches = [cache.fork(parent) for _ in suffixes]
        for b in branches:
            cache.release(b)
    torch.cuda.synchronize()
    t_forks = (time.perf_counter() - t0) / reps
    line["fork_batch"] = {"suffixes": 63, "prefix_tokens": 448, "suffix_tokens": 64, "dtype": "bf16",
                          "ms_per_batch": round(t_batch * 1e3, 3),
                          "ms_forks_and_releases": round(t_forks * 1e3, 3),
                          "suffix_tokens_per_s": round(63 * 64 / t_batch, 1)}
    cache.close()
    model.close()
    ctx.close()
    print(json.dumps(line), flush=True)


def cpu_baseline(shape, weights, seq_len, threads, n_seqs=12):
    """The CPU oracle's fp32 forward of the same model on this host: an all-core leg over
    n_seqs sequences (OpenMP over rows, heads and (sequence, head) chains) and a single-thread
    leg over one sequence in the reference's scalar order."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from oracle import oracle as O
    from huncho_amd import abi

    cfg = O.QwenConfig(hidden_size=shape.hidden, num_hidden_layers=shape.n_layers,
                       num_attention_heads=shape.n_heads, num_key_value_heads=shape.n_kv_heads,
                       head_dim=shape.head_dim, intermediate_size=shape.intermediate, vocab_size=shape.vocab,
                       rms_norm_eps=shape.eps, layer_types=shape.layer_types, linear_conv_kernel_dim=shape.conv_k,
                       linear_key_head_dim=shape.lin_key_dim, linear_num_key_heads=shape.lin_n_k_heads,
                       linear_num_value_heads=shape.lin_n_v_heads, linear_value_head_dim=shape.lin_v_dim,
                       rope_theta=shape.rope_theta, partial_rotary_factor=shape.rotary_dim / shape.head_dim)
    f = {k: O.bf16_to_f32(v).reshape(v.shape) for k, v in weights.items()}
    model = O.QwenModel(cfg, f, bf16=False)
    seqs = [abi.synth_uniform_int(SEED, 900 + i, seq_len, 0, shape.vocab - 1) for i in range(n_seqs)]
    head_w = f["decision_head.weight"]

    def run(rows):
        for ids in rows:
            _ = model.forward(ids)[-1] @ head_w.T

    O.set_threads(threads)
    dt = timed(lambda: run(seqs))
    O.set_threads(1)
    dt1 = timed(lambda: run(seqs[:1]))
    O.set_threads(threads)
    hi = host_info()
    return {"value": round(n_seqs * seq_len / dt, 2), "unit": "tokens/s", "cores": threads, "kind": "port",
            "sample": f"{n_seqs} sequences x {seq_len} tokens of the same Kev-shaped model (all 24 layers + head), "
                      f"fp32 CPU oracle forward, {threads} OpenMP threads, {dt:.2f} s",
            "host": hi,
            "single_thread": {"value": round(seq_len / dt1, 2), "unit": "tokens/s", "cores": 1,
                              "sample": f"1 sequence x {seq_len} tokens, 1 thread, {dt1:.2f} s"}}


def cpu_kernel_baselines(threads):
    """The oracle's attention and delta-rule kernels on this host, per kernel config: GQA causal
    attention fp32 (T 256, 16/8 heads x 128, pages of 16, identity table), the gated delta rule
    fp32 (T 512, 16 heads, 128 x 128 state) and, as a bounded sample of the varlen bf16 batch,
    its first 4 sequences. Each at `threads` threads and at 1 thread."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    import numpy as np

    from oracle import oracle as O

    out = {}
    rng = np.random.default_rng(SEED)
    # attention, fp32, T = 256
    T, hq, hkv, d, P = 256, 16, 8, 128, 16
    q = rng.standard_normal((T, hq, d), dtype=np.float32)
    kp = rng.standard_normal((T // P, hkv, P, d), dtype=np.float32)
    vp = rng.standard_normal((T // P, hkv, P, d), dtype=np.float32)
    bt = np.arange(T // P, dtype=np.int32)[None]
    cu, lens = np.array([0, T], np.int32), np.array([T], np.int32)
    fl = 4.0 * hq * d * T * (T + 1) / 2
    for nt in (threads, 1):
        O.set_threads(nt)
        reps = 5
        dt = timed(lambda: [O.paged_attention(q, kp, vp, bt, cu, lens, P, d ** -0.5) for _ in range(reps)]) / reps
        out.setdefault("attention_fp32_T256", {})[f"threads_{nt}"] = {"seconds": round(dt, 5),
                                                                       "gflops": round(fl / dt / 1e9, 2)}
    # delta rule, fp32, T = 512
    T, H = 512, 16
    qd = rng.standard_normal((T, H, 128), dtype=np.float32)
    kd = rng.standard_normal((T, H, 128), dtype=np.float32)
    qd /= np.linalg.norm(qd, axis=-1, keepdims=True)
    kd /= np.linalg.norm(kd, axis=-1, keepdims=True)
    vd = rng.standard_normal((T, H, 128), dtype=np.float32)
    beta = (1 / (1 + np.exp(-rng.standard_normal((T, H))))).astype(np.float32)
    gd = (-np.log1p(np.exp(rng.standard_normal((T, H)))) * 0.5).astype(np.float32)
    cu = np.array([0, T], np.int32)
    fl = T * H * (7 * 128 * 128 + 2 * 128)
    for nt in (threads, 1):
        O.set_threads(nt)
        reps = 3
        dt = timed(lambda: [O.gated_delta_rule(qd, kd, vd, gd, beta, cu) for _ in range(reps)]) / reps
        out.setdefault("delta_rule_fp32_T512", {})[f"threads_{nt}"] = {"seconds": round(dt, 5),
                                                                        "gflops": round(fl / dt / 1e9, 2)}
    # varlen paged bf16 attention: the first 4 of 32 sequences (lengths uniform in [64, 2048])
    from huncho_amd import abi

    lengths = [int(x) for x in abi.synth_uniform_int(SEED, 960, 32, 64, 2048)][:4]
    n = sum(lengths)
    pages = [(L + P - 1) // P for L in lengths]
    n_pages = sum(pages)  # a pool of just these sequences' pages, in a seeded permutation
    perm = abi.synth_permutation(SEED, 961, n_pages)
    btv = np.full((4, max(pages)), -1, np.int32)
    k0 = 0
    for s_, np_ in enumerate(pages):
        btv[s_, :np_] = perm[k0:k0 + np_]
        k0 += np_
    qb = O.bf16_bits(rng.standard_normal((n, hq, d), dtype=np.float32))
    kpb = O.bf16_bits(rng.standard_normal((n_pages, hkv, P, d), dtype=np.float32))
    vpb = O.bf16_bits(rng.standard_normal((n_pages, hkv, P, d), dtype=np.float32))
    cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    fl = sum(4.0 * hq * d * L * (L + 1) / 2 for L in lengths)
    O.set_threads(threads)
    dt = timed(lambda: O.paged_attention(qb, kpb, vpb, btv, cu, np.array(lengths, np.int32), P, d ** -0.5))
    out["varlen_attention_bf16_4seqs"] = {"lengths": lengths, f"threads_{threads}": {
        "seconds": round(dt, 5), "gflops": round(fl / dt / 1e9, 2)}}
    return out


def laya_lengths(n_seqs):
    """Seeded varlen batch: lengths uniform in [256, 4096]."""
    from huncho_amd import abi

    return [int(x) for x in abi.synth_uniform_int(SEED, 950, n_seqs, 256, 4096)]


def laya_attention_work(lengths, heads, d, half_window):
    """Algorithmic FLOPs of one bidirectional attention launch: 4*heads*d per visible
    (query, key) pair; all L^2 pairs globally, |i-j| <= half_window locally."""
    import numpy as np

    pairs = 0
    for L in lengths:
        if half_window < 0:
            pairs += L * L
        else:
            i = np.arange(L)
            pairs += int((np.minimum(L - 1, i + half_window) - np.maximum(0, i - half_window) + 1).sum())
    return 4.0 * heads * d * pairs


def laya_kernel_rooflines(ctx, shape, lengths, dtype, iters):
    """Times the global and the windowed attention kernels alone on the encoder's layout (q, k, v
    as token-strided views of fused [tokens][3][heads][64] projection rows)."""
    import numpy as np
    import torch

    from huncho_amd.ops import bidir_attention

    dev = torch.device("cuda", 0)
    stream = torch.cuda.current_stream(dev)
    n = sum(lengths)
    heads, d = shape.n_heads, shape.hidden // shape.n_heads
    g = torch.Generator(device=dev).manual_seed(SEED)
    qkv = torch.randn((n, 3, heads, d), generator=g, device=dev, dtype=torch.float32).to(dtype)
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)).to(dev)
    out = torch.empty((n, heads, d), dtype=dtype, device=dev)
    res = {}
    for name, hw in (("global", -1), ("local", shape.local_window // 2)):
        t = time_launches(lambda: bidir_attention(ctx, qkv[:, 0], qkv[:, 1], qkv[:, 2], cu, max(lengths), hw,
                                                  out=out), iters, stream)
        res[name] = {"seconds": t, "flops": laya_attention_work(lengths, heads, d, hw),
                     "bytes": n * 4 * heads * d * 2}
    torch.cuda.synchronize()
    return res


def laya_cpu_baseline(shape, weights, threads, n_rows=3, n_tokens=2048):
    """The CPU oracle's fp32 encoder forward of a few rows of the same model on this host."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from oracle import oracle as O
    from huncho_amd import abi

    O.set_threads(threads)
    cfg = O.BertConfig(hidden_size=shape.hidden, num_hidden_layers=shape.n_layers,
                       num_attention_heads=shape.n_heads, intermediate_size=shape.intermediate,
                       vocab_size=shape.vocab, global_attn_every_n_layers=shape.global_every,
                       local_attention=shape.local_window, global_rope_theta=shape.global_theta,
                       local_rope_theta=shape.local_theta)
    f = {k: O.bf16_to_f32(v).reshape(v.shape) for k, v in weights.items()}
    model = O.BertModel(cfg, f)
    rows = [abi.synth_uniform_int(SEED, 902 + i, n_tokens, 0, shape.vocab - 1).tolist() for i in range(n_rows)]

    def run(rs):
        for ids in rs:
            h = model.forward([ids])[0]
            _ = f["head.weight"] @ h.mean(0)

    dt = timed(lambda: run(rows))
    O.set_threads(1)
    short = [rows[0][:256]]
    dt1 = timed(lambda: run(short))
    O.set_threads(threads)
    return {"value": round(n_rows * n_tokens / dt, 2), "unit": "tokens/s", "cores": threads, "kind": "port",
            "sample": f"{n_rows} sequences x {n_tokens} tokens of the same ModernBERT-base-shaped encoder (all 22 "
                      f"layers + mean-pooled head), fp32 CPU oracle forward, {threads} OpenMP threads, {dt:.2f} s",
            "host": host_info(),
            "single_thread": {"value": round(256 / dt1, 2), "unit": "tokens/s", "cores": 1,
                              "sample": f"1 sequence x 256 tokens, 1 thread, {dt1:.2f} s"}}


def laya_measure(args, dtype):
    """The Laya encoder workload's bench line (without the CPU baseline)."""
    import numpy as np
    import torch

    from huncho_amd import abi
    from huncho_amd.laya import LayaModel, LayaShape, synthetic_weights
    from huncho_amd.ops import context_for_torch

    shape = LayaShape()
    n_seqs = args.batch or 16
    lengths = laya_lengths(n_seqs)
    n_tokens = sum(lengths)
    t0 = time.perf_counter()
    weights = synthetic_weights(shape, SEED)
    log(f"synthetic weights in {time.perf_counter() - t0:.1f} s; {n_seqs} rows, {n_tokens} tokens")
    ctx = context_for_torch(0)
    info = ctx.device_info()
    model = LayaModel(ctx, shape, weights, dtype)
    batch = model.prepare(lengths)
    ids = torch.from_numpy(abi.synth_uniform_int(SEED, 951, n_tokens, 0, shape.vocab - 1)).to("cuda")
    log(f"model ready on {info.name.decode()} ({info.compute_units} CUs); warmup {args.warmup}")
    for _ in range(args.warmup):
        model.forward_ids(ids, batch)
    torch.cuda.synchronize()
    if ctx.take_faults():
        raise RuntimeError("device faults during warmup")
    log(f"timing {args.steps} steps")
    t0 = time.perf_counter()
    for _ in range(args.steps):
        model.forward_ids(ids, batch)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms = elapsed / args.steps * 1e3
    log(f"{ms:.2f} ms/step; first row logits {np.round(batch['logits'].cpu().numpy()[0], 4).tolist()}")
    kr = laya_kernel_rooflines(ctx, shape, lengths, dtype, args.kernel_iters)
    gl, lo = kr["global"], kr["local"]
    achieved = gl["flops"] / gl["seconds"] / 1e12
    log(f"global attention {gl['seconds'] * 1e6:.1f} us/launch, windowed {lo['seconds'] * 1e6:.1f} us/launch")
    measured = load_traffic("laya") if (n_seqs, args.dtype) == (16, "bf16") else {}
    traffic_of = lambda k: sum(measured[k]) if k in measured else None
    line = {
        "metric": "encoder tokens/s (ModernBERT-base-shaped varlen bf16); attn TFLOP/s as % of MFMA peak",
        "value": round(n_tokens / (elapsed / args.steps), 1),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": args.dtype,
        "data": "synthetic (seeded lengths and token ids, random-init N(0,0.02) weights)",
        "config": {"workload": "laya_modernbert_encoder", "n_seqs": n_seqs, "lengths": "uniform [256, 4096]",
                   "tokens_per_step": n_tokens, "layers": shape.n_layers, "hidden": shape.hidden,
                   "heads": "12 x 64", "global_every": shape.global_every, "local_window": shape.local_window,
                   "mlp": f"GeGLU {shape.intermediate}", "vocab": shape.vocab, "head": f"mean-pool -> {shape.n_out}"},
        "roofline": {"kernel": "bidir_attn_16 (global layer)", "bound": "mfma", "achieved": round(achieved, 2),
                     "peak": MFMA_PEAK_BF16 / 1e12, "unit": "TFLOP/s",
                     "frac": round(achieved * 1e12 / MFMA_PEAK_BF16, 4), "traffic": traffic_of("global"),
                     "us_per_launch": round(gl["seconds"] * 1e6, 2), "flops_per_launch": gl["flops"]},
        "roofline_local_attention": {"kernel": "bidir_attn_16 (window +-64)", "bound": "mfma",
                                     "achieved": round(lo["flops"] / lo["seconds"] / 1e12, 2),
                                     "peak": MFMA_PEAK_BF16 / 1e12, "unit": "TFLOP/s",
                                     "frac": round(lo["flops"] / lo["seconds"] / MFMA_PEAK_BF16, 4),
                                     "us_per_launch": round(lo["seconds"] * 1e6, 2), "flops_per_launch": lo["flops"],
                                     "hbm_frac": round(lo["bytes"] / lo["seconds"] / HBM_PEAK, 4)},
        "device": {"name": info.name.decode(), "cus": info.compute_units, "clock_mhz": info.clock_khz // 1000},
    }
    model.close()
    return line, shape, weights


def run_laya(args, dtype):
    line, shape, weights = laya_measure(args, dtype)
    if not args.no_cpu_baseline:
        threads = default_threads(args)
        log(f"CPU baseline with {threads} threads and 1 thread")
        line["cpu_baseline"] = laya_cpu_baseline(shape, weights, threads)
    print(json.dumps(line), flush=True)


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: every GPU host here has one, and this path shards by "
              f"independent sequences with no collectives (asked for --gpus {args.gpus}).", file=sys.stderr)
        sys.exit(2)
    import torch

    if args.copy_probe:
        src = torch.ones(args.copy_probe // 4, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        log(f"copied {src.numel() * 4} bytes 3 times")
        return
    dtype = torch.bfloat16 if args.dtype == "bf16" else torch.float16
    if args.fork_probe:
        fork_probe(args.kernel_iters)
        return
    if args.gemm_probe:
        gemm_probe(args.kernel_iters, (args.batch or 64) * args.seq_len)
        return
    if args.attention_probe:
        attention_probe(args.kernel_iters, args.batch or 64, args.seq_len)
        return
    if args.kernels_only:
        from huncho_amd.ops import context_for_torch

        ctx = context_for_torch(0)
        if args.workload == "laya":
            from huncho_amd.laya import LayaShape

            kr = laya_kernel_rooflines(ctx, LayaShape(), laya_lengths(args.batch or 16), dtype, args.kernel_iters)
        else:
            from huncho_amd.kev import KevShape

            kr = kernel_rooflines(ctx, KevShape(), args.batch or 64, args.seq_len, dtype, args.kernel_iters)
        print(json.dumps({k: round(v["seconds"] * 1e6, 2) for k, v in kr.items()}), flush=True)
        return
    if args.workload == "laya":
        run_laya(args, dtype)
    else:
        run_kev(args, dtype)


def load_traffic(workload):
    """HBM bytes per launch of the roofline kernels, measured with rocprofv3 FETCH_SIZE and
    WRITE_SIZE passes scaled by a copy of known size (profiles/hbm_traffic.txt, one line per
    `workload kernel fetch_bytes=F write_bytes=W`). Missing file or entry: {}."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", "hbm_traffic.txt")
    out = {}
    if not os.path.exists(path):
        return out
    for line in open(path):
        parts = line.split()
        if len(parts) < 4 or line.startswith("#") or parts[0] != workload:
            continue
        kv = dict(p.split("=", 1) for p in parts[2:] if "=" in p)
        if "fetch_bytes" in kv and "write_bytes" in kv:
            out[parts[1]] = (int(kv["fetch_bytes"]), int(kv["write_bytes"]))
    return out


def run_kev(args, dtype):
    import numpy as np
    import torch

    from huncho_amd import abi
    from huncho_amd.kev import KevModel, KevShape, synthetic_weights
    from huncho_amd.ops import context_for_torch

    shape = KevShape()
    args.batch = args.batch or 64
    t0 = time.perf_counter()
    weights = synthetic_weights(shape, SEED)
    log(f"synthetic weights in {time.perf_counter() - t0:.1f} s")
    ctx = context_for_torch(0)
    info = ctx.device_info()
    res32 = args.residual == "fp32"
    model = KevModel(ctx, shape, weights, dtype, residual_fp32=res32)
    lengths = [args.seq_len] * args.batch
    batch = model.prepare(lengths, seed=SEED)
    ids_np = abi.synth_uniform_int(SEED, 901, sum(lengths), 0, shape.vocab - 1)
    ids = torch.from_numpy(ids_np).to("cuda")
    n_tokens = sum(lengths)
    log(f"model ready on {info.name.decode()} ({info.compute_units} CUs); warmup {args.warmup}")
    for _ in range(args.warmup):
        model.forward_ids(ids, batch)
    torch.cuda.synchronize()
    if ctx.take_faults():
        raise RuntimeError("device faults during warmup")
    log(f"timing {args.steps} steps")
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        model.forward_ids(ids, batch)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms = elapsed / args.steps * 1e3
    logits = batch["logits"].cpu().numpy()
    probs = abi.calibrate(logits[0], 1.3)
    log(f"{ms:.2f} ms/step; first row calibrated probabilities {np.round(probs, 4).tolist()}")
    modes = {args.residual: round(ms, 3)}
    if args.dtype != "fp32":
        # the other residual-stream mode, same batch and steps, for the record
        other = "bf16" if res32 else "fp32"
        model.close()
        alt = KevModel(ctx, shape, weights, dtype, residual_fp32=not res32)
        alt_batch = alt.prepare(lengths, seed=SEED)
        for _ in range(args.warmup):
            alt.forward_ids(ids, alt_batch)
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        for _ in range(args.steps):
            alt.forward_ids(ids, alt_batch)
        torch.cuda.synchronize()
        modes[other] = round((time.perf_counter() - t1) / args.steps * 1e3, 3)
        if ctx.take_faults():
            raise RuntimeError("device faults in the second residual mode")
        alt.close()
        log(f"residual stream {other}: {modes[other]:.2f} ms/step")

    # the roofline kernels as the forward runs them (one forward under the profiler)
    model_b = KevModel(ctx, shape, weights, dtype, residual_fp32=res32)
    batch_b = model_b.prepare(lengths, seed=SEED)
    model_b.forward_ids(ids, batch_b)
    fk = forward_kernel_times(lambda: model_b.forward_ids(ids, batch_b),
                              {"attention": "paged_prefill_attn", "delta_rule_fused": "gdn_chunk16"})
    model_b.close()
    kr = kernel_rooflines(ctx, shape, args.batch, args.seq_len, dtype, args.kernel_iters)
    a, gf, gd = kr["attention"], kr["delta_rule_fused"], kr["delta_rule"]
    # a second tracer in the process (rocprofv3) leaves the torch profiler's device times
    # meaningless (microseconds for these kernels): keep them only when they agree with the
    # standalone timing within 4x
    if fk and any(k in fk and not 0.25 < fk[k]["us_avg"] / (kr[k]["seconds"] * 1e6) < 4.0
                  for k in ("attention", "delta_rule_fused")):
        log(f"in-forward kernel times {fk} disagree with the standalone launches; dropped")
        fk = None
    attn_achieved = a["flops"] / a["seconds"] / 1e12
    log(f"attention {a['seconds'] * 1e6:.1f} us/launch, fused delta rule {gf['seconds'] * 1e6:.1f} us/launch, "
        f"standalone delta rule {gd['seconds'] * 1e6:.1f} us/launch")
    measured = load_traffic("kev") if (args.batch, args.seq_len, args.dtype) == (64, 512, "bf16") else {}
    traffic_of = lambda k: sum(measured[k]) if k in measured else None
    fw = kev_forward_flops(shape, lengths)
    step_s = elapsed / args.steps

    def hbm_line(kernel, r, key):
        return {"kernel": kernel, "bound": "hbm", "achieved": round(r["bytes"] / r["seconds"] / 1e9, 1),
                "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": round(r["bytes"] / r["seconds"] / HBM_PEAK, 4),
                "traffic": traffic_of(key), "us_per_launch": round(r["seconds"] * 1e6, 2),
                "bytes_per_launch": r["bytes"], "tflops": round(r["flops"] / r["seconds"] / 1e12, 2)}

    line = {
        "metric": "prefill tokens/s (Kev-shaped 64x512 bf16); attn TFLOP/s as % of MFMA peak",
        "value": round(n_tokens / step_s, 1),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": args.dtype,
        "data": "synthetic (seeded token ids, random-init N(0,0.02) weights)",
        "config": {"workload": "kev_hybrid_scoring_prefill", "batch": args.batch, "seq_len": args.seq_len,
                   "tokens_per_step": n_tokens, "layers": shape.n_layers, "hidden": shape.hidden,
                   "layer_pattern": "3 gated-delta-rule : 1 gated GQA attention", "attn_heads": "16q/8kv x 128",
                   "gdn_heads": "16 x 128", "mlp": "SwiGLU 3584", "vocab": shape.vocab, "page_size": shape.page_size,
                   "decision_head": shape.n_out, "residual_stream": args.residual},
        # ms per step of both residual-stream modes (the timed one and the other, same batch)
        "ms_per_step_by_residual_stream": modes,
        "forward": {"tflops": round(fw["total"] / step_s / 1e12, 2),
                    "frac_of_mfma_peak": round(fw["total"] / step_s / MFMA_PEAK_BF16, 4),
                    "tflop_per_step": {k: round(v / 1e12, 4) for k, v in fw.items()}},
        "roofline": {"kernel": "paged_prefill_attn", "bound": "mfma", "achieved": round(attn_achieved, 2),
                     "peak": MFMA_PEAK_BF16 / 1e12, "unit": "TFLOP/s",
                     "frac": round(attn_achieved * 1e12 / MFMA_PEAK_BF16, 4), "traffic": traffic_of("attention"),
                     "us_per_launch": round(a["seconds"] * 1e6, 2), "flops_per_launch": a["flops"],
                     "bytes_per_launch": a["bytes"], "hbm_frac": round(a["bytes"] / a["seconds"] / HBM_PEAK, 4),
                     # the roofline ceiling at this launch's arithmetic intensity (FLOP per algorithmic
                     # byte), as a share of the MFMA peak: below 1, HBM bounds the launch first
                     "ceiling_frac": round(min(1.0, a["flops"] / a["bytes"] * HBM_PEAK / MFMA_PEAK_BF16), 4)},
        "roofline_attention_varlen": {
            "kernel": "paged_prefill_attn (32 sequences, lengths 64..2048, no gate)", "bound": "mfma",
            "achieved": round(kr["attention_varlen"]["flops"] / kr["attention_varlen"]["seconds"] / 1e12, 2),
            "peak": MFMA_PEAK_BF16 / 1e12, "unit": "TFLOP/s",
            "frac": round(kr["attention_varlen"]["flops"] / kr["attention_varlen"]["seconds"] / MFMA_PEAK_BF16, 4),
            "us_per_launch": round(kr["attention_varlen"]["seconds"] * 1e6, 2),
            "flops_per_launch": kr["attention_varlen"]["flops"]},
        "roofline_delta_rule": hbm_line("gdn_chunk16<fused> (the forward's Gated DeltaNet layer kernel)", gf,
                                        "delta_rule_fused"),
        "roofline_delta_rule_standalone": hbm_line("gdn_chunk16 (standalone recurrence)", gd, "delta_rule"),
        "device": {"name": info.name.decode(), "cus": info.compute_units, "clock_mhz": info.clock_khz // 1000},
        # the fp32 correctness configurations (1: attention T 256, 2: delta rule T 512) on the GPU
        "fp32_config_kernels": fp32_config_kernels(ctx, args.kernel_iters),
        # average duration of the same kernels inside one forward (profiler device activity),
        # beside the standalone launches the roofline fields time
        "in_forward_kernels": fk,
    }
    if not args.no_cpu_baseline:
        threads = default_threads(args)
        log(f"CPU baseline with {threads} threads and 1 thread")
        line["cpu_baseline"] = cpu_baseline(shape, weights, args.seq_len, threads)
        line["cpu_kernel_baselines"] = cpu_kernel_baselines(threads)
    if not args.no_laya:
        # the second workload (16 varlen ModernBERT-base rows, 256..4096 tokens), same steps
        log("second workload: the Laya encoder")
        sub = argparse.Namespace(**vars(args))
        sub.batch = 0
        laya, _, _ = laya_measure(sub, dtype)
        line["laya"] = {k: laya[k] for k in ("metric", "value", "unit", "steps", "warmup", "ms_per_step", "config",
                                             "roofline", "roofline_local_attention")}
    print(json.dumps(line), flush=True)



if __name__ == "__main__":
    main()
