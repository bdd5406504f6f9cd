"""End-to-end parity of the hybrid scoring forward (hk_kev_forward) against the oracle's full
Qwen3.5 forward (ho_qwen_forward) on the same seeded weights and token ids.

Gates: calibrated decision probabilities within 1e-3 absolute of the fp32 oracle for fp16
activations (the qualification external-delta gate, crates/huncho-core/src/conformance.rs:20-48),
within 2e-5 for fp32 (the fp32 probability gate of crates/huncho-backend/tests/kev_reference.rs:79),
and for bf16 no farther from the fp32 oracle than the oracle's own bf16 flow is on the same rows.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from huncho_amd import abi
from huncho_amd.kev import PREFIX, KevModel, KevShape, synthetic_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SEED = 4242


def oracle_model(shape: KevShape, weights: dict, bf16: bool):
    cfg = O.QwenConfig(hidden_size=shape.hidden, num_hidden_layers=shape.n_layers,
                       num_attention_heads=shape.n_heads, num_key_value_heads=shape.n_kv_heads,
                       head_dim=shape.head_dim, intermediate_size=shape.intermediate, vocab_size=shape.vocab,
                       rms_norm_eps=shape.eps, layer_types=shape.layer_types,
                       linear_conv_kernel_dim=shape.conv_k, linear_key_head_dim=shape.lin_key_dim,
                       linear_num_key_heads=shape.lin_n_k_heads, linear_num_value_heads=shape.lin_n_v_heads,
                       linear_value_head_dim=shape.lin_v_dim, rope_theta=shape.rope_theta,
                       partial_rotary_factor=shape.rotary_dim / shape.head_dim)
    f = {k: O.bf16_to_f32(v).reshape(v.shape) for k, v in weights.items()}
    return O.QwenModel(cfg, f, bf16=bf16), f["decision_head.weight"]


def oracle_scores(model, head_w, rows, temperature):
    logits, probs = [], []
    for r in rows:
        h = model.forward(r)
        lg = (h[-1].astype(np.float32) @ head_w.T.astype(np.float32)).astype(np.float32)
        logits.append(lg)
        probs.append(O.calibrate(lg, temperature))
    return np.stack(logits), np.stack(probs)


@pytest.fixture(scope="module")
def ctx():
    from huncho_amd.ops import context_for_torch

    c = context_for_torch(0)
    yield c
    c.close()


KEV_ROW_LENGTHS = [96, 37, 130]


@pytest.fixture(scope="module")
def kev_case():
    """Kev-shaped weights, three seeded rows, and the oracle's calibrated probabilities for
    its bf16 flow (tensors rounded to bf16 where the reference stores them; unlike the
    reference's default bf16 attention, which keeps scores and probabilities in bf16
    (qwen3_5.rs:579, 681-701), the oracle computes them in fp32 as the GPU kernel does) and its
    fp32 flow."""
    shape = KevShape()  # hidden 1024, 24 layers (3 GDN : 1 attention), vocab 151936, 8 choices
    weights = synthetic_weights(shape, SEED)
    rows = [abi.synth_uniform_int(SEED, 500 + i, L, 0, shape.vocab - 1) for i, L in enumerate(KEV_ROW_LENGTHS)]
    ref_model, head_w = oracle_model(shape, weights, bf16=True)
    bf16_logits, bf16_probs = oracle_scores(ref_model, head_w, rows, 1.3)
    del ref_model
    f32_model, _ = oracle_model(shape, weights, bf16=False)
    f32_logits, f32_probs = oracle_scores(f32_model, head_w, rows, 1.3)
    del f32_model
    return dict(shape=shape, weights=weights, rows=rows, bf16_logits=bf16_logits, bf16_probs=bf16_probs,
                f32_logits=f32_logits, f32_probs=f32_probs)


def test_kev_shaped_bf16_probabilities(ctx, kev_case):
    """bf16 activations: with random-init weights this 24-layer residual stack amplifies
    rounding, so any bf16 execution sits ~1e-2 from fp32 in probability. Gate: the GPU is no
    farther from the fp32 oracle than the oracle's own bf16 flow (the reference's bf16 rounding
    points) is, on the same rows."""
    c = kev_case
    model = KevModel(ctx, c["shape"], c["weights"], torch.bfloat16)
    logits, probs = model.forward_batch(c["rows"], temperature=1.3)
    model.close()
    dp = float(np.abs(probs - c["bf16_probs"]).max())
    dp32 = float(np.abs(probs - c["f32_probs"]).max())
    noise = float(np.abs(c["bf16_probs"] - c["f32_probs"]).max())
    dl = float(np.abs(logits - c["bf16_logits"]).max())
    print(f"bf16 Kev-shaped: max |dp| vs oracle bf16 {dp:.3e}, vs oracle fp32 {dp32:.3e} "
          f"(oracle bf16 vs fp32 {noise:.3e}); max |dlogit| {dl:.3e}")
    assert dp32 <= noise, (dp, dp32, noise)


def test_kev_shaped_fp16_probabilities(ctx, kev_case):
    """fp16 activations (same MFMA rate as bf16, 3 more mantissa bits) on the Kev shape:
    calibrated probabilities within 1e-3 absolute of the fp32 forward (the external-delta gate,
    conformance.rs:30-32; the reference's own half-precision gate is 2e-3, kev_reference.rs:71)."""
    c = kev_case
    model = KevModel(ctx, c["shape"], c["weights"], torch.float16)
    logits, probs = model.forward_batch(c["rows"], temperature=1.3)
    model.close()
    assert np.isfinite(logits).all()
    dp = float(np.abs(probs - c["f32_probs"]).max())
    dl = float(np.abs(logits - c["f32_logits"]).max())
    print(f"fp16 Kev-shaped: max |dp| vs oracle fp32 {dp:.3e}; max |dlogit| {dl:.3e}")
    assert dp < 1e-3, dp


def test_kev_shaped_fp32_probabilities(ctx, kev_case):
    """fp32 activations on the Kev shape: probabilities within 2e-5 of the oracle's fp32
    forward (kev_reference.rs:79) and logits within 1e-4 relative."""
    c = kev_case
    model = KevModel(ctx, c["shape"], c["weights"], torch.float32)
    logits, probs = model.forward_batch(c["rows"], temperature=1.3)
    model.close()
    dp = float(np.abs(probs - c["f32_probs"]).max())
    dl = float(np.abs(logits - c["f32_logits"]).max() / np.abs(c["f32_logits"]).max())
    print(f"fp32 Kev-shaped: max |dp| vs oracle fp32 {dp:.3e}; rel dlogit {dl:.3e}")
    assert dp < 2e-5 and dl < 1e-4, (dp, dl)


def test_small_hybrid_fp32_probabilities(ctx):
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, rope_theta=10000.0, n_out=5)
    weights = synthetic_weights(shape, SEED + 1, std=0.05)
    rows = [abi.synth_uniform_int(SEED, 600 + i, L, 0, shape.vocab - 1) for i, L in enumerate([70, 129, 1])]
    model = KevModel(ctx, shape, weights, torch.float32)
    logits, probs = model.forward_batch(rows, temperature=1.3)
    ref_model, head_w = oracle_model(shape, weights, bf16=False)
    ref_logits, ref_probs = oracle_scores(ref_model, head_w, rows, 1.3)
    dp = float(np.abs(probs - ref_probs).max())
    dl = float(np.abs(logits - ref_logits).max() / np.abs(ref_logits).max())
    print(f"fp32 small hybrid: max |dp| = {dp:.3e}, rel dlogit = {dl:.3e}")
    assert dp < 2e-5 and dl < 1e-4, (dp, dl)
    # rows are independent: each row alone gives its batched result (no cross-row leakage
    # through pages, conv windows or chunk boundaries)
    for i, r in enumerate(rows):
        li, _ = model.forward_batch([r], temperature=1.3)
        assert float(np.abs(li[0] - logits[i]).max()) <= 1e-5 * float(np.abs(logits[i]).max()), i
    model.close()


# Qwen3.5-family proportions other than the Kev shape: 256-wide attention heads with partial
# rotary (a quarter of the head, 64 dims) and GQA group 4, which run on the MFMA paged attention
# (two 128-wide halves per K / V tile) and the vectorised QK-norm/RoPE kernel in 16-bit types, on
# the general kernels (general.hip) in fp32; linear-attention value heads twice the key heads
# (q and k repeated per value head, qwen3_5.rs:914-921) on the fused MFMA delta rule
WIDE_SHAPE = dict(hidden=512, n_layers=4, n_heads=4, n_kv_heads=1, head_dim=256, rotary_dim=64, intermediate=1024,
                  vocab=1000, lin_key_dim=128, lin_v_dim=128, lin_n_k_heads=2, lin_n_v_heads=4, n_out=4)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_wide_head_hybrid_against_oracle(ctx, dtype):
    """The whole forward at WIDE_SHAPE against the oracle: fp32 at the fp32 gates (probabilities
    2e-5, logits 1e-4 relative), fp16 at the 1e-3 probability gate, bf16 no farther from the fp32
    flow than the oracle's own bf16 flow is (twice, as two bf16 results that each pass it)."""
    shape = KevShape(**WIDE_SHAPE)
    weights = synthetic_weights(shape, SEED + 7, std=0.05)
    rows = [abi.synth_uniform_int(SEED, 700 + i, L, 0, shape.vocab - 1) for i, L in enumerate([150, 33, 97])]
    model = KevModel(ctx, shape, weights, dtype)
    ident = abi.identity(abi.lib().hk_kev_model_identity, model.h)
    logits, probs = model.forward_batch(rows, temperature=1.3)
    assert ctx.take_faults() == 0
    model.close()
    want = "general" if dtype == torch.float32 else "mfma-16bit"
    assert want in ident["attention_execution"], ident["attention_execution"]
    ref32, head_w = oracle_model(shape, weights, bf16=False)
    f32_logits, f32_probs = oracle_scores(ref32, head_w, rows, 1.3)
    dp = float(np.abs(probs - f32_probs).max())
    dl = float(np.abs(logits - f32_logits).max() / np.abs(f32_logits).max())
    if dtype == torch.float32:
        print(f"wide-head hybrid fp32: max |dp| {dp:.3e}, rel dlogit {dl:.3e}")
        assert dp < 2e-5 and dl < 1e-4, (dp, dl)
    elif dtype == torch.float16:
        print(f"wide-head hybrid fp16: max |dp| {dp:.3e}, rel dlogit {dl:.3e}")
        assert dp < 1e-3, dp
    else:
        ref16, _ = oracle_model(shape, weights, bf16=True)
        _, bf16_probs = oracle_scores(ref16, head_w, rows, 1.3)
        spread = float(np.abs(bf16_probs - f32_probs).max())
        print(f"wide-head hybrid bf16: max |dp| vs fp32 {dp:.3e} (oracle bf16 flow {spread:.3e})")
        assert dp <= 2 * spread, (dp, spread)


def test_max_context_row_fp32(ctx):
    """A row of exactly max_context (8192) tokens beside a 3-token row: 512 pages in its block
    table, 128 key tiles of attention, 128 delta-rule chunks; both rows against the fp32 oracle.
    One token more is rejected before any work."""
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, rope_theta=10000.0, n_out=5, max_context=8192)
    weights = synthetic_weights(shape, SEED + 2, std=0.05)
    rows = [abi.synth_uniform_int(SEED, 900, shape.max_context, 0, shape.vocab - 1),
            abi.synth_uniform_int(SEED, 901, 3, 0, shape.vocab - 1)]
    model = KevModel(ctx, shape, weights, torch.float32)
    logits, probs = model.forward_batch(rows, temperature=1.3)
    ref_model, head_w = oracle_model(shape, weights, bf16=False)
    ref_logits, ref_probs = oracle_scores(ref_model, head_w, rows, 1.3)
    dp = float(np.abs(probs - ref_probs).max())
    dl = float(np.abs(logits - ref_logits).max() / np.abs(ref_logits).max())
    print(f"fp32 max-context row: max |dp| = {dp:.3e}, rel dlogit = {dl:.3e}")
    assert dp < 2e-5 and dl < 1e-4, (dp, dl)
    with pytest.raises(abi.HkError):
        model.forward_batch([np.concatenate([rows[0], rows[1][:1]])])
    assert ctx.take_faults() == 0
    model.close()


def test_forward_rejects_out_of_vocab_before_work(ctx):
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, n_out=3)
    model = KevModel(ctx, shape, synthetic_weights(shape, 3), torch.bfloat16)
    with pytest.raises(ValueError):
        model.forward_batch([[1, 2, 1000]])
    with pytest.raises(ValueError):
        model.forward_batch([[1] * 10] * 65)
    # a device-side out-of-range id (bypassing the host check) raises the token fault bit
    batch = model.prepare([4])
    ids = torch.tensor([1, 2, 5000, 3], dtype=torch.int32, device="cuda")
    model.forward_ids(ids, batch)
    assert ctx.take_faults() & abi.HK_FAULT_TOKEN
    model.close()


def test_forward_rejects_misaligned_workspace(ctx):
    """A workspace that is not 16-byte aligned is refused before any launch (the vector kernels and
    the own GEMM read 16-byte rows carved from it); the same call on the aligned workspace runs."""
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, n_out=3)
    model = KevModel(ctx, shape, synthetic_weights(shape, 3), torch.bfloat16)
    batch = model.prepare([12, 5])
    ids = torch.arange(17, dtype=torch.int32, device="cuda")
    cu_host = batch["cu_host"]
    need = model.workspace_bytes(17, 2)
    ws = torch.empty(need + 64, dtype=torch.uint8, device="cuda")

    def call(offset):
        return abi.lib().hk_kev_forward(
            model.h, ids.data_ptr(), batch["cu"].data_ptr(), cu_host.ctypes.data_as(C.POINTER(C.c_int32)), 2,
            batch["bt"].data_ptr(), batch["bt"].shape[1], batch["num_pages"], ws.data_ptr() + offset, need,
            batch["logits"].data_ptr(), None)

    assert call(8) == abi.HK_ERR_INVALID
    assert "aligned" in abi.lib().hk_ctx_last_error(ctx.h).decode()
    assert call(0) == abi.HK_OK
    torch.cuda.synchronize()
    assert ctx.take_faults() == 0 and np.isfinite(batch["logits"].cpu().numpy()).all()
    model.close()


def test_identity_keys(ctx):
    """The execution-identity keys (Capabilities.extra, qwen3_5.rs:2540-2653) name the device,
    the dtype and the kernels that ran, so a calibration key cannot silently match another path."""
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, n_out=3)
    seen = {}
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        model = KevModel(ctx, shape, synthetic_weights(shape, 3), dt)
        ident = abi.identity(abi.lib().hk_kev_model_identity, model.h)
        model.close()
        for key in ("device", "native_execution", "device_path", "attention_execution", "delta_rule_execution",
                    "activation_dtype", "kv_page_tokens", "recurrent_state_dtype"):
            assert key in ident, key
        assert "gfx950" in ident["device"] and ident["kv_page_tokens"] == "16"
        seen[dt] = ident
    assert seen[torch.bfloat16]["activation_dtype"] == "bf16" and seen[torch.float16]["activation_dtype"] == "fp16"
    assert seen[torch.float32]["delta_rule_execution"] != seen[torch.bfloat16]["delta_rule_execution"]


def test_identity_names_the_split_forms(ctx):
    """Suffix attention and the fp32 delta rule of few rows add in another order than the kernels of large
    batches, so the keys that name them are not those of a library without these forms. The 16-bit delta
    rule's split form has the same bits, and its key stays."""
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000,
                     lin_n_k_heads=2, lin_n_v_heads=2, rotary_dim=64, n_out=3)
    for dt, attn, delta in ((torch.bfloat16, "key-split", "rocm-chunked-c64-mfma-f16-operands-v1"),
                            (torch.float16, "key-split", "rocm-chunked-c64-mfma-f16-operands-v1"),
                            (torch.float32, "rocm-paged-flash-mfma-f32-v1", "few-rows-split")):
        model = KevModel(ctx, shape, synthetic_weights(shape, 3), dt)
        ident = abi.identity(abi.lib().hk_kev_model_identity, model.h)
        model.close()
        assert attn in ident["attention_execution"] and delta in ident["delta_rule_execution"]
