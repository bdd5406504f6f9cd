"""The scratch of the kernels that split few, long rows (fused Gated DeltaNet layer, fp32 delta rule, suffix
attention): no call allocates, which kernel runs follows from the call's sizes alone, the scratch follows its
context from stream to stream without the stream that it left, and a context's block passes to the next one."""
import ctypes as C

import numpy as np
import pytest
import torch

from huncho_amd import abi
from huncho_amd.ops import context_for_torch, gated_delta_chunked, gdn_fused, paged_prefill_attention

pytestmark = pytest.mark.gpu


def randn(*shape, seed=1):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def gdn_call(n, seed=1):
    """A fused layer call over one row of n tokens: f(ctx, out)."""
    mixed = (randn(n, 64 * 128, seed=seed) * 0.6).to(torch.bfloat16)
    z, ba = mixed[:, 48 * 128:], randn(n, 32, seed=seed + 1).to(torch.bfloat16)
    conv_w = (randn(48 * 128, 4, seed=seed + 2) * 0.3).to(torch.bfloat16).float()
    base_g, dt_bias, norm_w = -torch.exp(randn(16, seed=seed + 3)), randn(16, seed=seed + 4) - 3.0, 1.0 + 0.1 * randn(128)
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    return lambda ctx, out: gdn_fused(ctx, mixed, conv_w, ba, 0, 16, base_g, dt_bias, z, norm_w, 1e-6, cu, 16, 16, out=out)


def delta_call(n, seed=1):
    q, k, v = (randn(n, 16, 128, seed=seed + i) for i in range(3))
    q, k = (torch.nn.functional.normalize(x, dim=-1) for x in (q, k))
    g, beta = -torch.nn.functional.softplus(randn(n, 16, seed=seed + 3)), torch.sigmoid(randn(n, 16, seed=seed + 4))
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    return lambda ctx, out: gated_delta_chunked(ctx, q, k, v, g, beta, cu, out=out)


def attn_call(new, context, seed=1):
    pages = (context + 15) // 16
    kp, vp = (randn(pages, 8, 16, 128, seed=seed + i).to(torch.bfloat16) for i in range(2))
    q = randn(new, 16, 128, seed=seed + 2).to(torch.bfloat16)
    bt = torch.arange(pages, dtype=torch.int32, device="cuda").view(1, -1)
    cu = torch.tensor([0, new], dtype=torch.int32, device="cuda")
    lens = torch.tensor([context], dtype=torch.int32, device="cuda")
    return lambda ctx, out: paged_prefill_attention(ctx, q, kp, vp, bt, cu, lens, new, out=out)


def outs():
    bf = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda")
    return bf(3000, 16, 128), torch.empty((1500, 16, 128), device="cuda"), bf(30, 16, 128)


def test_the_first_calls_of_a_context_allocate_nothing():
    calls, o = (gdn_call(3000), delta_call(1500), attn_call(30, 2700)), outs()
    for ctx in (context_for_torch(0), context_for_torch(0)):  # the first also loads the kernels
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for f, x in zip(calls, o):
            f(ctx, x)
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]
        ctx.close()
    assert used == 0, used


def test_a_forward_does_not_depend_on_earlier_calls():
    """An fp32 forward over a long row: the same bits on a context that has only seen this model, and after a
    larger call."""
    from huncho_amd.kev import KevModel, KevShape, synthetic_weights

    ctx = context_for_torch(0)
    n = 8400
    shape = KevShape(hidden=256, n_layers=4, n_heads=2, n_kv_heads=1, intermediate=512, vocab=1000, lin_n_k_heads=16,
                     lin_n_v_heads=16, rotary_dim=64, rope_theta=10000.0, n_out=5, max_context=n)
    model = KevModel(ctx, shape, synthetic_weights(shape, 7, std=0.05), torch.float32)
    ids = torch.from_numpy(np.random.default_rng(1).integers(0, 1000, n).astype(np.int32)).cuda()
    hidden = []
    for _ in range(2):
        batch = model.prepare([n])
        model.forward_ids(ids, batch, want_hidden=True)
        hidden.append(batch["hidden"].clone())
        delta_call(12000)(ctx, torch.empty((12000, 16, 128), device="cuda"))
    torch.cuda.synchronize()
    assert torch.equal(*hidden)
    model.close()
    ctx.close()


def test_the_stream_that_the_context_left_may_be_gone():
    hip = C.CDLL([line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line][0])
    call, out = gdn_call(3000), outs()[0]
    ctx = context_for_torch(0)
    call(ctx, out)
    torch.cuda.synchronize()
    want = out.clone()
    for _ in range(3):
        stream = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
        ctx.set_stream(stream.value)
        out.zero_()
        torch.cuda.synchronize()
        call(ctx, out)
        assert hip.hipStreamSynchronize(stream) == 0 and torch.equal(out, want)
        assert hip.hipStreamDestroy(stream) == 0
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    out.zero_()
    call(ctx, out)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    ctx.close()


def test_blocks_pass_from_context_to_context():
    """Contexts alive at once have blocks of their own; those of destroyed ones are used again, one at most is
    kept, and none is left after the last context."""
    call, x = gdn_call(3000), [outs()[0] for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(3):
        ctxs = [context_for_torch(0) for _ in range(3)]
        for c, o in zip(ctxs, x):
            o.zero_()
            call(c, o)
        torch.cuda.synchronize()
        assert torch.equal(x[0], x[1]) and torch.equal(x[0], x[2])
        before = torch.cuda.mem_get_info()[0]
        ctxs[1].close()
        ctxs[2].close()
        after = torch.cuda.mem_get_info()[0]
        assert 0 <= (after - before) >> 20 <= 600  # one of the two blocks is kept
        ctxs[0].close()


@pytest.mark.parametrize("capturing", [False, True])
def test_captured_calls_do_without(capturing):
    """A captured call replays the kernels without scratch, within the two forms' rounding of each other."""
    ctx = context_for_torch(0)
    for call, like, tol in ((gdn_call(700), (700, 16, 128), 0.0), (delta_call(700), (700, 16, 128), 8e-6),
                            (attn_call(30, 2700), (30, 16, 128), 9.2e-3)):
        want = torch.empty(like, dtype=torch.float32 if tol == 8e-6 else torch.bfloat16, device="cuda")
        got = torch.zeros_like(want)
        call(ctx, want)
        torch.cuda.synchronize()
        if not capturing:
            call(ctx, got)
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            continue
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            call(ctx, got)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            got.zero_()
            graph.replay()
            again = torch.empty_like(want)
            call(ctx, again)
            torch.cuda.synchronize()
            assert torch.equal(again, want)
            assert float((got.double() - want.double()).norm() / want.double().norm()) <= tol
    ctx.close()
