"""The workloads whose speed is tracked: the scoring forward's layers, each through an entry point
that a program calls, and two whole forwards.

Kinds of case
  attn    QK-norm + RoPE + paged K/V write, then paged causal GQA attention (`ops`): the core of a
          full-attention layer. 16 query and 8 KV heads of 128, pages of 16 from a permuted pool.
  gdn     the fused Gated DeltaNet layer body (`ops.gdn_fused`), 16 heads of 128 x 128, with or
          without a carried recurrent state and conv tail.
  delta   the gated delta rule alone in fp32 (`ops.gated_delta_chunked`) with its final state.
  mlp     RMSNorm, the gate|up projection with its SwiGLU epilogue and the down projection with the
          residual add (`ops.rms_norm`, `hk_linear`): hidden 1024, intermediate 3584.
  bert    ModernBERT attention over the Wqkv rows (`ops.bidir_attention`), 12 heads of 64, global or
          in a window.
  kev     a whole Kev-shaped forward (`KevModel.forward_ids`): decision logits and last hidden rows.
  laya    a whole ModernBERT-base forward (`LayaModel.forward_ids`): logits and hidden rows.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from huncho_amd import abi
from huncho_amd.kev import KevModel, KevShape
from huncho_amd.laya import LayaModel, LayaShape
from huncho_amd.ops import (bidir_attention, context_for_torch, gated_delta_chunked, gdn_fused,
                            paged_prefill_attention, qk_norm_rope_kv_write, rms_norm)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
HK = {"bf16": abi.HK_BF16, "fp16": abi.HK_F16, "fp32": abi.HK_F32}
DEV = "cuda:0"

HQ, HKV, D, PAGE = 16, 8, 128, 16  # Kev full-attention layer
H = 16                             # Gated DeltaNet heads (key and value)
HIDDEN, INTER = 1024, 3584
BERT_HEADS, BERT_D = 12, 64


def listed():
    return [
        # one request of five short questions as independent rows (about 169 positions): the latency
        # of a whole forward. fp16: through 24 layers of random weights bf16 logits are 12 % from
        # the exact ones, fp16 logits 1.5 %, so only the latter tell a fault from a rounding
        {"name": "kev_request", "kind": "kev", "dtype": "fp16", "rows": 5, "lo": 33, "hi": 35},
        # a few short texts through the encoder: the latency of a whole forward
        {"name": "laya_request", "kind": "laya", "dtype": "bf16", "rows": 4, "lo": 64, "hi": 200},
        # the attention layer of a full scoring batch, 64 rows of 512 tokens, with its output gate
        {"name": "attn_batch", "kind": "attn", "dtype": "bf16", "rows": 64, "lo": 512, "hi": 512, "prefix": 0,
         "gate": True},
        # the varlen prefill batch: 32 rows of 64..2048 tokens
        {"name": "attn_varlen", "kind": "attn", "dtype": "bf16", "rows": 32, "lo": 64, "hi": 2048, "prefix": 0,
         "gate": False},
        # five short questions that continue one cached long state, whose pages they share
        {"name": "attn_suffix", "kind": "attn", "dtype": "fp16", "rows": 5, "lo": 20, "hi": 40, "prefix": 2670,
         "gate": True},
        # the Gated DeltaNet layer of a full scoring batch
        {"name": "gdn_batch", "kind": "gdn", "dtype": "bf16", "rows": 64, "lo": 512, "hi": 512, "state": False},
        # the same layer while one long state is prefilled: one row, its state carried on
        {"name": "gdn_long", "kind": "gdn", "dtype": "bf16", "rows": 1, "lo": 2704, "hi": 2704, "state": True},
        # the recurrence of an fp32 model: one row of 512 tokens with its final state
        {"name": "delta_fp32", "kind": "delta", "dtype": "fp32", "rows": 1, "lo": 512, "hi": 512},
        # the MLP block of one request, and of a full scoring batch
        {"name": "mlp_request", "kind": "mlp", "dtype": "bf16", "tokens": 169},
        {"name": "mlp_batch", "kind": "mlp", "dtype": "bf16", "tokens": 32768},
        # the encoder's two attention layers over 16 texts of 256..4096 tokens
        {"name": "bert_global", "kind": "bert", "dtype": "bf16", "rows": 16, "lo": 256, "hi": 4096, "window": -1},
        {"name": "bert_window", "kind": "bert", "dtype": "bf16", "rows": 16, "lo": 256, "hi": 4096, "window": 64},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges: sizes even over their logarithms, rows of unequal
    lengths, both 16-bit types, carried states and prefixes. Token budgets keep a case within the
    largest listed one of its kind."""
    kind = rng.choice(["kev", "laya", "attn", "attn", "attn", "gdn", "gdn", "gdn", "delta", "mlp", "mlp", "bert", "bert"])
    c = {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16"])}

    def rows_of(max_rows, shortest, longest, budget):
        hi = _log_int(rng, shortest, longest)
        c["hi"] = hi
        c["lo"] = rng.choice([hi, max(1, hi // 2), max(1, hi // 8)])
        c["rows"] = min(_log_int(rng, 1, max_rows), max(1, budget // hi))

    if kind == "kev":
        c["dtype"] = "fp16"
        rows_of(64, 8, 512, 2048)
    elif kind == "laya":
        rows_of(16, 16, 512, 2048)
    elif kind == "attn":
        c["prefix"] = rng.choice([0, 0, _log_int(rng, 16, 4096)])
        if c["prefix"]:
            rows_of(63, 1, 128, 4096)
        else:
            rows_of(64, 8, 2048, 32768)
        c["gate"] = rng.random() < 0.75
    elif kind == "gdn":
        c["state"] = rng.random() < 0.5
        rows_of(64, 8, 4096, 32768)
    elif kind == "delta":
        c["dtype"] = "fp32"
        rows_of(16, 8, 2048, 4096)
    elif kind == "mlp":
        c["tokens"] = _log_int(rng, 5, 32768)
    else:
        c["window"] = rng.choice([-1, 64])
        rows_of(16, 16, 4096, 32768)
    return c


# ---- inputs -------------------------------------------------------------------------------------

def _lengths(case, rng):
    """Row lengths in [lo, hi]; the first row has the longest, so max_len is the case's."""
    x = rng.integers(case["lo"], case["hi"] + 1, case["rows"])
    x[0] = case["hi"]
    return [int(v) for v in x]


def _case_lengths(case):
    """The lengths belong to the case, not to the seed: a case's work is the same for every seed."""
    return _lengths(case, np.random.default_rng([case["rows"], case["lo"], case["hi"]]))


def _cu(lengths):
    return torch.tensor(np.concatenate([[0], np.cumsum(lengths)]), dtype=torch.int32, device=DEV)


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def n(self, *shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device=DEV) * std + mean

    def u(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo


def _decay_params(r, heads):
    """A and dt_bias as such layers are initialised: A in [1, 16], softplus(dt_bias) log-even in
    [1e-3, 0.1], so that heads forget within a few tokens or keep hundreds."""
    a = r.u(heads, lo=1.0, hi=16.0)
    dt = torch.exp(r.u(heads, lo=math.log(1e-3), hi=math.log(0.1)))
    return a, torch.log(torch.expm1(dt))


def _prepare_attn(case, seed):
    r = _Rand(seed)
    dt = DTYPES[case["dtype"]]
    lens_new, prefix = _case_lengths(case), case["prefix"]
    n, rows = sum(lens_new), case["rows"]
    cols = 2 * HQ * D + 2 * HKV * D
    qkv = r.n(n, cols).to(dt)  # the fused projection's rows: per head q | gate, then k, then v
    qg = qkv[:, : 2 * HQ * D].view(n, HQ, 2 * D)
    ctx_lens = [prefix + L for L in lens_new]
    shared = prefix // PAGE
    need = [(t + PAGE - 1) // PAGE for t in ctx_lens]
    pages = shared + sum(m - shared for m in need)
    perm = np.random.default_rng(seed).permutation(pages).astype(np.int32)
    bt = np.zeros((rows, max(need)), np.int32)
    at = shared
    for s, m in enumerate(need):
        bt[s, :shared] = perm[:shared]
        bt[s, shared:m] = perm[at:at + m - shared]
        at += m - shared
    kp, vp = r.n(pages, HKV, PAGE, D).to(dt), r.n(pages, HKV, PAGE, D).to(dt)
    cs, sn = abi.rope_table(D, 1e7, max(ctx_lens), HK[case["dtype"]])
    st = {"case": case, "ctx": context_for_torch(0), "qkv": qkv, "q": qg[:, :, :D], "gate": qg[:, :, D:],
          "k": qkv[:, 2 * HQ * D: 2 * HQ * D + HKV * D].view(n, HKV, D),
          "v": qkv[:, 2 * HQ * D + HKV * D:].view(n, HKV, D), "cu": _cu(lens_new), "bt_host": bt,
          "bt": torch.from_numpy(bt).to(DEV), "lens": torch.tensor(ctx_lens, dtype=torch.int32, device=DEV),
          "lens_new": lens_new, "kp": kp, "vp": vp, "cos": torch.from_numpy(cs).to(DEV),
          "sin": torch.from_numpy(sn).to(DEV), "qw": 1.0 + r.n(D, std=0.02), "kw": 1.0 + r.n(D, std=0.02),
          "q_out": torch.empty((n, HQ, D), dtype=dt, device=DEV), "o": torch.empty((n, HQ, D), dtype=dt, device=DEV)}
    return st


def _run_attn(s):
    qk_norm_rope_kv_write(s["ctx"], s["q"], s["k"], s["v"], s["qw"], s["kw"], 1e-6, s["cos"], s["sin"], D, s["cu"],
                          s["lens"], s["bt"], s["kp"], s["vp"], s["q_out"])
    paged_prefill_attention(s["ctx"], s["q_out"], s["kp"], s["vp"], s["bt"], s["cu"], s["lens"], max(s["lens_new"]),
                            gate=s["gate"] if s["case"]["gate"] else None, out=s["o"])
    return {"o": s["o"], "q": s["q_out"], "k_pool": s["kp"], "v_pool": s["vp"]}


def _rms64(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, cos, sin):
    """NeoX rotate-half over the whole last dimension; cos and sin [tokens][d / 2]."""
    a, b = x.chunk(2, -1)
    c, s = cos[:, None], sin[:, None]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_attn(case, seed):
    s = _prepare_attn(case, seed)
    kp, vp = s["kp"].double(), s["vp"].double()
    qs, outs, t0 = [], [], 0
    prefix, P = case["prefix"], PAGE
    new = []
    for i, L in enumerate(s["lens_new"]):
        tok = slice(t0, t0 + L)
        pos = torch.arange(prefix, prefix + L, device=DEV)
        cos, sin = s["cos"][pos].double(), s["sin"][pos].double()
        q = _rope64(_rms64(s["q"][tok].double(), s["qw"].double()), cos, sin)
        k = _rope64(_rms64(s["k"][tok].double(), s["kw"].double()), cos, sin)
        page = s["bt"][i].long()[pos // P]
        kp[page, :, pos % P] = k
        vp[page, :, pos % P] = s["v"][tok].double()
        qs.append(q)
        new.append((tok, pos))
        t0 += L
    for i, (tok, pos) in enumerate(new):
        total = int(pos[-1]) + 1
        pages = s["bt"][i].long()[: (total + P - 1) // P]
        kk = kp[pages].transpose(1, 2).reshape(-1, HKV, D)[:total].permute(1, 2, 0)  # [Hkv][d][keys]
        vv = vp[pages].transpose(1, 2).reshape(-1, HKV, D)[:total].transpose(0, 1)   # [Hkv][keys][d]
        q = qs[i].view(-1, HKV, HQ // HKV, D).permute(1, 2, 0, 3)                    # [Hkv][g][L][d]
        sc = q @ kk[:, None].contiguous() / math.sqrt(D)
        sc.masked_fill_(torch.arange(total, device=DEV)[None] > pos[:, None], -math.inf)
        o = (sc.softmax(-1) @ vv[:, None].contiguous()).permute(2, 0, 1, 3).reshape(-1, HQ, D)
        if case["gate"]:
            o = o * torch.sigmoid(s["gate"][tok].double())
        outs.append(o)
    return {"o": torch.cat(outs), "q": torch.cat(qs), "k_pool": kp, "v_pool": vp}


def _prepare_gdn(case, seed):
    r = _Rand(seed)
    dt = DTYPES[case["dtype"]]
    lens = _case_lengths(case)
    n, rows = sum(lens), case["rows"]
    conv_dim = 3 * H * 128
    mixed = r.n(n, conv_dim + H * 128, std=0.64).to(dt)  # in_proj rows q | k | v | z of normed rows
    a, dt_bias = _decay_params(r, H)
    st = {"case": case, "ctx": context_for_torch(0), "mixed": mixed, "z": mixed[:, conv_dim:], "cu": _cu(lens),
          "lens": lens, "ba": r.n(n, 2 * H, std=0.64).to(dt), "conv_w": r.n(conv_dim, 4, std=0.3).to(dt).float(),
          "base_g": -a, "dt_bias": dt_bias.to(dt).float(), "norm_w": 1.0 + r.n(128, std=0.02),
          "out": torch.empty((n, H, 128), dtype=dt, device=DEV), "hist": None, "init": None, "final": None}
    if case["state"]:
        st["hist"] = r.n(rows, conv_dim, 3, std=0.64).to(dt)
        st["init"] = r.n(rows, H, 128, 128, std=0.1)
        st["final"] = torch.empty_like(st["init"])
    return st


def _run_gdn(s):
    want = s["hist"] is not None
    res = gdn_fused(s["ctx"], s["mixed"], s["conv_w"], s["ba"], 0, H, s["base_g"], s["dt_bias"], s["z"], s["norm_w"],
                    1e-6, s["cu"], H, H, conv_hist=s["hist"], want_tail=want, initial_state=s["init"],
                    final_state=s["final"], out=s["out"])
    return {"o": res[0], "tail": res[1], "state": s["final"]} if want else {"o": res}


def _recurrence64(q, k, v, g, beta, state):
    """The per-token gated delta rule over padded rows: q, k, v [rows][T][heads][128], g and beta
    [rows][T][heads] (0 past a row's end, which leaves its state as it is), state [rows][h][dk][dv]."""
    out = torch.zeros_like(v)
    for t in range(q.shape[1]):
        state = state * torch.exp(g[:, t])[..., None, None]
        kt = k[:, t]
        d = beta[:, t][..., None] * (v[:, t] - (state * kt[..., None]).sum(-2))
        state = state + kt[..., None] * d[..., None, :]
        out[:, t] = (state * q[:, t][..., None]).sum(-2)
    return out, state


def _pad(x, lens):
    """[tokens][...] -> [rows][longest][...], zeros past each row's end"""
    out = x.new_zeros((len(lens), max(lens)) + tuple(x.shape[1:]))
    t0 = 0
    for i, L in enumerate(lens):
        out[i, :L] = x[t0:t0 + L]
        t0 += L
    return out


def _unpad(x, lens):
    return torch.cat([x[i, :L] for i, L in enumerate(lens)])


def _gdn64(mixed, conv_w, hist, ba, base_g, dt_bias, norm_w, lens, init):
    """The layer body in 64 bits: (output rows, conv tails, final state)."""
    conv_dim = 3 * H * 128
    x = _pad(mixed[:, :conv_dim], lens)
    hist = x.new_zeros((len(lens), conv_dim, 3)) if hist is None else hist
    xx = torch.cat([hist.transpose(1, 2), x], 1)  # 3 rows before each row's start
    T = x.shape[1]
    y = F.silu(sum(xx[:, i:i + T] * conv_w[:, i] for i in range(4)))
    tail = torch.stack([xx[i, L:L + 3].T for i, L in enumerate(lens)])
    q, k, v = (t.reshape(len(lens), T, H, 128) for t in y.split(H * 128, -1))
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(128)
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    beta = _pad(torch.sigmoid(ba[:, :H]), lens)
    g = _pad(base_g * F.softplus(ba[:, H:2 * H] + dt_bias), lens)
    o, state = _recurrence64(q, k, v, g, beta, init)
    z = mixed[:, conv_dim:conv_dim + H * 128].reshape(-1, H, 128)
    return _rms64(_unpad(o, lens), norm_w) * F.silu(z), tail, state


def _exact_gdn(case, seed):
    if max(_case_lengths(case)) * case["rows"] > 65536:
        return None
    s = _prepare_gdn(case, seed)
    d = lambda t: None if t is None else t.double()
    init = d(s["init"]) if case["state"] else torch.zeros((case["rows"], H, 128, 128), dtype=torch.float64, device=DEV)
    o, tail, state = _gdn64(d(s["mixed"]), d(s["conv_w"]), d(s["hist"]), d(s["ba"]), d(s["base_g"]), d(s["dt_bias"]),
                            d(s["norm_w"]), s["lens"], init)
    return {"o": o, "tail": tail, "state": state} if case["state"] else {"o": o}


def _prepare_delta(case, seed):
    r = _Rand(seed)
    lens = _case_lengths(case)
    n = sum(lens)
    return {"case": case, "ctx": context_for_torch(0), "cu": _cu(lens), "lens": lens,
            "q": F.normalize(r.n(n, H, 128), dim=-1) * 128 ** -0.5, "k": F.normalize(r.n(n, H, 128), dim=-1),
            "v": r.n(n, H, 128), "g": -F.softplus(r.n(n, H)) * 0.5, "beta": torch.sigmoid(r.n(n, H)),
            "out": torch.empty((n, H, 128), device=DEV), "final": torch.empty((case["rows"], H, 128, 128), device=DEV)}


def _run_delta(s):
    o = gated_delta_chunked(s["ctx"], s["q"], s["k"], s["v"], s["g"], s["beta"], s["cu"], final_state=s["final"],
                            out=s["out"])
    return {"o": o, "state": s["final"]}


def _exact_delta(case, seed):
    s = _prepare_delta(case, seed)
    p = {x: _pad(s[x].double(), s["lens"]) for x in ("q", "k", "v", "g", "beta")}
    zero = torch.zeros((case["rows"], H, 128, 128), dtype=torch.float64, device=DEV)
    o, state = _recurrence64(p["q"], p["k"], p["v"], p["g"], p["beta"], zero)
    return {"o": _unpad(o, s["lens"]), "state": state}


def _prepare_mlp(case, seed):
    r = _Rand(seed)
    dt, n = DTYPES[case["dtype"]], case["tokens"]
    gate, up = r.n(INTER, HIDDEN, std=0.02).to(dt), r.n(INTER, HIDDEN, std=0.02).to(dt)
    # the SwiGLU epilogue's weight rows: blocks of 16 gate rows and the 16 matching up rows
    w_gu = torch.stack([gate.view(-1, 16, HIDDEN), up.view(-1, 16, HIDDEN)], 1).reshape(2 * INTER, HIDDEN).contiguous()
    return {"case": case, "ctx": context_for_torch(0), "x": r.n(n, HIDDEN).to(dt), "norm": 1.0 + r.n(HIDDEN, std=0.02),
            "gate": gate, "up": up, "w_gu": w_gu, "w_down": r.n(HIDDEN, INTER, std=0.02).to(dt),
            "h": torch.empty((n, HIDDEN), dtype=dt, device=DEV), "act": torch.empty((n, INTER), dtype=dt, device=DEV),
            "y": torch.empty((n, HIDDEN), dtype=dt, device=DEV)}


def _linear(s, epilogue, x, w, out, y, c=None):
    s["ctx"].check(abi.lib().hk_linear(
        s["ctx"].h, HK[s["case"]["dtype"]], epilogue, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), x.shape[0],
        out, w.shape[1], c.data_ptr() if c is not None else None, c.stride(0) if c is not None else 0, y.data_ptr(),
        y.stride(0)))


def _run_mlp(s):
    rms_norm(s["ctx"], s["x"], s["norm"], 1e-6, out=s["h"])
    _linear(s, 2, s["h"], s["w_gu"], 2 * INTER, s["act"])
    _linear(s, 1, s["act"], s["w_down"], HIDDEN, s["y"], s["x"])
    return {"y": s["y"], "h": s["h"], "act": s["act"]}


def _exact_mlp(case, seed):
    s = _prepare_mlp(case, seed)
    x = s["x"].double()
    h = _rms64(x, s["norm"].double())
    act = F.silu(h @ s["gate"].double().T) * (h @ s["up"].double().T)
    return {"y": x + act @ s["w_down"].double().T, "h": h, "act": act}


def _prepare_bert(case, seed):
    r = _Rand(seed)
    dt = DTYPES[case["dtype"]]
    lens = _case_lengths(case)
    n, w = sum(lens), BERT_HEADS * BERT_D
    qkv = r.n(n, 3 * w).to(dt)  # Wqkv rows q | k | v
    q, k, v = (qkv[:, i * w:(i + 1) * w].view(n, BERT_HEADS, BERT_D) for i in range(3))
    return {"case": case, "ctx": context_for_torch(0), "qkv": qkv, "q": q, "k": k, "v": v, "cu": _cu(lens),
            "lens": lens, "o": torch.empty((n, BERT_HEADS, BERT_D), dtype=dt, device=DEV)}


def _run_bert(s):
    return bidir_attention(s["ctx"], s["q"], s["k"], s["v"], s["cu"], max(s["lens"]), half_window=s["case"]["window"],
                           out=s["o"])


def _bidir64(q, k, v, lens, window):
    """[tokens][heads][d] -> [tokens][heads][d], one row at a time"""
    outs, t0 = [], 0
    for L in lens:
        qq, kk, vv = (x[t0:t0 + L].transpose(0, 1).contiguous() for x in (q, k, v))
        sc = qq @ kk.transpose(1, 2).contiguous() / math.sqrt(q.shape[-1])
        if window >= 0:
            i = torch.arange(L, device=DEV)
            sc.masked_fill_((i[:, None] - i[None]).abs() > window, -math.inf)
        outs.append((sc.softmax(-1) @ vv).transpose(0, 1))
        t0 += L
    return torch.cat(outs)


def _exact_bert(case, seed):
    s = _prepare_bert(case, seed)
    return _bidir64(s["q"].double(), s["k"].double(), s["v"].double(), s["lens"], case["window"])


def _bf16_bits(t):
    return t.to(torch.bfloat16).cpu().view(torch.int16).numpy().view(np.uint16)


KEV_SHAPE = KevShape(max_context=512)
LAYA_SHAPE = LayaShape(max_context=512)


def _kev_weights(seed):
    """bf16 checkpoint tensors on the GPU: N(0, 0.02) projections and zero-centred norms, the decay
    parameters as such layers are initialised."""
    r = _Rand(seed)
    out = {}
    for name, shape in KEV_SHAPE.weight_shapes().items():
        if name.endswith("A_log"):
            a, dt_bias = _decay_params(r, H)
            out[name] = torch.log(a)
            out[name.replace("A_log", "dt_bias")] = dt_bias
        elif name.endswith("dt_bias"):
            continue
        elif name.endswith("conv1d.weight"):
            out[name] = r.n(*shape, std=0.3)
        elif name.endswith("linear_attn.norm.weight"):
            out[name] = r.n(*shape, std=0.02, mean=1.0)
        else:
            out[name] = r.n(*shape, std=0.02)
        out[name] = out[name].to(torch.bfloat16)
    return {k: v.to(torch.bfloat16) for k, v in out.items()}


def _laya_weights(seed):
    r = _Rand(seed)
    return {k: r.n(*v, std=0.02, mean=1.0 if k.endswith("norm.weight") else 0.0).to(torch.bfloat16)
            for k, v in LAYA_SHAPE.weight_shapes().items()}


def _ids(case, seed, vocab):
    n = sum(_case_lengths(case))
    return torch.from_numpy(np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)).to(DEV)


def _prepare_kev(case, seed):
    ctx = context_for_torch(0)
    w = {k: _bf16_bits(v) for k, v in _kev_weights(seed).items()}
    model = KevModel(ctx, KEV_SHAPE, w, DTYPES[case["dtype"]])
    return {"case": case, "ctx": ctx, "model": model, "batch": model.prepare(_case_lengths(case), seed=seed),
            "ids": _ids(case, seed, KEV_SHAPE.vocab)}


def _run_kev(s):
    logits = s["model"].forward_ids(s["ids"], s["batch"], want_hidden=True)
    return {"logits": logits, "hidden": s["batch"]["hidden"]}


def _rope_rows(lens, d, theta, dtype):
    cs, sn = abi.rope_table(d, theta, max(lens), HK[dtype])
    cs, sn = torch.from_numpy(cs).to(DEV).double(), torch.from_numpy(sn).to(DEV).double()
    return torch.cat([cs[:L] for L in lens]), torch.cat([sn[:L] for L in lens])


def _exact_kev(case, seed):
    lens = _case_lengths(case)
    dt = DTYPES[case["dtype"]]
    w = {k: v.to(dt) for k, v in _kev_weights(seed).items()}
    p = "model.language_model."
    cos, sin = _rope_rows(lens, D, KEV_SHAPE.rope_theta, case["dtype"])
    x = w[p + "embed_tokens.weight"][_ids(case, seed, KEV_SHAPE.vocab).long()].double()
    for i, kind in enumerate(KEV_SHAPE.layer_types):
        W = lambda name: w[f"{p}layers.{i}.{name}"].double()
        h = _rms64(x, 1.0 + W("input_layernorm.weight"))
        if kind == 0:
            la = "linear_attn."
            mixed = h @ torch.cat([W(la + "in_proj_qkv.weight"), W(la + "in_proj_z.weight")]).T
            ba = h @ torch.cat([W(la + "in_proj_b.weight"), W(la + "in_proj_a.weight")]).T
            zero = torch.zeros((len(lens), H, 128, 128), dtype=torch.float64, device=DEV)
            o, _, _ = _gdn64(mixed, W(la + "conv1d.weight")[:, 0], None, ba, -torch.exp(W(la + "A_log")),
                             W(la + "dt_bias"), W(la + "norm.weight"), lens, zero)
            x = x + o.reshape(len(x), -1) @ W(la + "out_proj.weight").T
        else:
            sa = "self_attn."
            qg = (h @ W(sa + "q_proj.weight").T).view(-1, HQ, 2 * D)
            q = _rope64(_rms64(qg[..., :D], 1.0 + W(sa + "q_norm.weight")), cos, sin)
            k = _rope64(_rms64((h @ W(sa + "k_proj.weight").T).view(-1, HKV, D), 1.0 + W(sa + "k_norm.weight")), cos, sin)
            v = (h @ W(sa + "v_proj.weight").T).view(-1, HKV, D)
            k, v = (t.repeat_interleave(HQ // HKV, 1) for t in (k, v))
            o, t0 = [], 0
            for L in lens:
                qq, kk, vv = (t[t0:t0 + L].transpose(0, 1).contiguous() for t in (q, k, v))
                sc = qq @ kk.transpose(1, 2).contiguous() / math.sqrt(D)
                sc.masked_fill_(torch.ones(L, L, dtype=torch.bool, device=DEV).triu(1), -math.inf)
                o.append((sc.softmax(-1) @ vv).transpose(0, 1))
                t0 += L
            o = torch.cat(o) * torch.sigmoid(qg[..., D:])
            x = x + o.reshape(len(x), -1) @ W(sa + "o_proj.weight").T
        h = _rms64(x, 1.0 + W("post_attention_layernorm.weight"))
        x = x + (F.silu(h @ W("mlp.gate_proj.weight").T) * (h @ W("mlp.up_proj.weight").T)) @ W("mlp.down_proj.weight").T
    last = torch.tensor(np.cumsum(lens) - 1, device=DEV)
    hid = _rms64(x[last], 1.0 + w[p + "norm.weight"].double())
    return {"logits": hid @ w["decision_head.weight"].double().T, "hidden": hid}


def _prepare_laya(case, seed):
    ctx = context_for_torch(0)
    w = {k: _bf16_bits(v) for k, v in _laya_weights(seed).items()}
    model = LayaModel(ctx, LAYA_SHAPE, w, DTYPES[case["dtype"]])
    batch = model.prepare(_case_lengths(case))
    return {"case": case, "ctx": ctx, "model": model, "batch": batch, "ids": _ids(case, seed, LAYA_SHAPE.vocab),
            "hidden": torch.empty((batch["n"], LAYA_SHAPE.hidden), dtype=DTYPES[case["dtype"]], device=DEV)}


def _run_laya(s):
    s["model"].forward_ids(s["ids"], s["batch"], s["hidden"])
    return {"logits": s["batch"]["logits"], "hidden": s["hidden"]}


def _exact_laya(case, seed):
    lens = _case_lengths(case)
    dt = DTYPES[case["dtype"]]
    w = {k: v.to(dt).double() for k, v in _laya_weights(seed).items()}
    sh = LAYA_SHAPE
    ln = lambda x, name: F.layer_norm(x, (sh.hidden,), w[name], None, sh.eps)
    x = ln(w["model.embeddings.tok_embeddings.weight"][_ids(case, seed, sh.vocab).long()], "model.embeddings.norm.weight")
    tables = [_rope_rows(lens, BERT_D, t, case["dtype"]) for t in (sh.global_theta, sh.local_theta)]
    for i in range(sh.n_layers):
        p = f"model.layers.{i}."
        local = i % sh.global_every != 0
        h = ln(x, p + "attn_norm.weight")
        q, k, v = (h @ w[p + "attn.Wqkv.weight"].T).view(-1, 3, BERT_HEADS, BERT_D).unbind(1)
        cos, sin = tables[1 if local else 0]
        o = _bidir64(_rope64(q, cos, sin), _rope64(k, cos, sin), v, lens, sh.local_window // 2 if local else -1)
        x = x + o.reshape(len(x), -1) @ w[p + "attn.Wo.weight"].T
        g, u = (ln(x, p + "mlp_norm.weight") @ w[p + "mlp.Wi.weight"].T).chunk(2, -1)
        x = x + (F.gelu(g) * u) @ w[p + "mlp.Wo.weight"].T
    hid = ln(x, "model.final_norm.weight")
    pooled = torch.stack([t.mean(0) for t in hid.split(lens)])
    return {"logits": pooled @ w["head.weight"].T, "hidden": hid}


_KINDS = {"kev": (_prepare_kev, _run_kev, _exact_kev), "laya": (_prepare_laya, _run_laya, _exact_laya),
          "attn": (_prepare_attn, _run_attn, _exact_attn), "gdn": (_prepare_gdn, _run_gdn, _exact_gdn),
          "delta": (_prepare_delta, _run_delta, _exact_delta), "mlp": (_prepare_mlp, _run_mlp, _exact_mlp),
          "bert": (_prepare_bert, _run_bert, _exact_bert)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def exact(case, seed):
    with torch.no_grad():
        return _KINDS[case["kind"]][2](case, seed)


# ---- what a pass cannot do without ----------------------------------------------------------------

def _causal_pairs(lens, prefix=0):
    return sum(L * prefix + L * (L + 1) // 2 for L in lens)


def _window_pairs(lens, window):
    return sum(L * L if window < 0 or window >= L else L * (2 * window + 1) - window * (window + 1) for L in lens)


def work(case):
    kind, e = case["kind"], 4 if case["dtype"] == "fp32" else 2
    if kind == "mlp":
        n = case["tokens"]
        return {"bytes": e * (3 * HIDDEN * INTER + n * (3 * HIDDEN + INTER)), "flops": 2 * n * 3 * HIDDEN * INTER}
    lens = _case_lengths(case)
    n = sum(lens)
    # the recurrence per token and head: decay, S^T k, the rank-one update and S^T q on 128 x 128
    rec = 7 * 128 * 128 + 2 * 128
    if kind == "attn":
        qkv = n * (2 * HQ + 2 * HKV) * D * e  # q, k, v read, q written
        kv_new = n * 2 * HKV * D * e
        o = n * HQ * D * e * (2 if case["gate"] else 1)
        return {"bytes": qkv + kv_new + o + case["prefix"] * 2 * HKV * D * e,
                "flops": 4 * HQ * D * _causal_pairs(lens, case["prefix"])}
    if kind == "gdn":
        state = case["rows"] * H * 128 * 128 * 4 * 2 if case["state"] else 0
        return {"bytes": n * H * (5 * 128 * e + 2 * e) + state, "flops": n * H * rec}
    if kind == "delta":
        return {"bytes": n * H * (4 * 128 * 4 + 8) + case["rows"] * H * 128 * 128 * 4, "flops": n * H * rec}
    if kind == "bert":
        return {"bytes": n * 4 * BERT_HEADS * BERT_D * e,
                "flops": 4 * BERT_HEADS * BERT_D * _window_pairs(lens, case["window"])}
    if kind == "kev":
        sh = KEV_SHAPE
        n_gdn, n_attn = sh.layer_types.count(0), sh.layer_types.count(1)
        w_gdn = HIDDEN * (4 * H * 128 + 2 * H) + H * 128 * HIDDEN
        w_attn = HIDDEN * (2 * HQ + 2 * HKV) * D + HQ * D * HIDDEN
        weights = n_gdn * w_gdn + n_attn * w_attn + sh.n_layers * 3 * HIDDEN * INTER
        return {"bytes": e * (weights + n * HIDDEN),
                "flops": 2 * n * weights + n_gdn * n * H * rec + n_attn * 4 * HQ * D * _causal_pairs(lens)}
    sh = LAYA_SHAPE
    weights = sh.n_layers * (4 * sh.hidden * sh.hidden + 3 * sh.hidden * sh.intermediate)
    pairs = sum(_window_pairs(lens, -1 if i % sh.global_every == 0 else sh.local_window // 2) for i in range(sh.n_layers))
    return {"bytes": e * (weights + 2 * n * sh.hidden), "flops": 2 * n * weights + 4 * sh.hidden * pairs}


def tolerance(case):
    """About four times the distance from `exact` that the roundings of each path's stored values
    cause: the operands and outputs of the 16-bit types, fp16 operands of the recurrence, 24 or 22
    layers of 16-bit storage in the whole forwards, 32-bit sums in the fp32 recurrence."""
    return {"rel": _REL[case["kind"]][case["dtype"]]}


_REL = {
    "attn": {"bf16": 1.6e-2, "fp16": 2.2e-3},
    "gdn": {"bf16": 1.6e-2, "fp16": 3e-3},
    "delta": {"fp32": 4e-6},
    "mlp": {"bf16": 1.6e-2, "fp16": 2.2e-3},
    "bert": {"bf16": 1e-2, "fp16": 1.5e-3},
    "kev": {"fp16": 6e-2},
    "laya": {"bf16": 5e-2, "fp16": 8e-3},
}
