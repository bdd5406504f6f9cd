"""The fused Gated DeltaNet layer for few, long rows (gdn16_split.hip) against gdn_chunk16, which the
same rows take when enough short rows join the batch. Both run the same products in the same order, so
outputs, final states and conv tails are compared bit for bit: rows that end on, before and after a
chunk boundary, an empty row, shared key heads, with and without a carried state."""
import pytest
import torch

from huncho_amd.ops import gdn_fused

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from huncho_amd.ops import context_for_torch

    c = context_for_torch(0)
    yield c
    c.close()


def make(lengths, heads, k_heads, dtype, state, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")
    n, conv_dim = sum(lengths), (2 * k_heads + heads) * 128
    mixed = (r(n, conv_dim + heads * 128) * 0.6).to(dtype)
    d = {"mixed": mixed, "z": mixed[:, conv_dim:], "ba": r(n, 2 * heads).to(dtype),
         "conv_w": (r(conv_dim, 4) * 0.3).to(dtype).float(), "base_g": -torch.exp(r(heads)), "dt_bias": r(heads) - 3.0,
         "norm_w": 1.0 + 0.1 * r(128), "hist": None, "init": None}
    if state:
        d["hist"] = (r(len(lengths), conv_dim, 3) * 0.6).to(dtype)
        d["init"] = r(len(lengths), heads, 128, 128) * 0.1
    return d


def run(ctx, d, lengths, heads, k_heads):
    cu = torch.tensor([0] + lengths, device="cuda").cumsum(0).to(torch.int32)
    final = torch.full((len(lengths), heads, 128, 128), 7.0, device="cuda")
    out, tail = gdn_fused(ctx, d["mixed"], d["conv_w"], d["ba"], 0, heads, d["base_g"], d["dt_bias"], d["z"],
                          d["norm_w"], 1e-6, cu, heads, k_heads, conv_hist=d["hist"], want_tail=True,
                          initial_state=d["init"], final_state=final)
    return out, tail, final


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("state", [False, True])
@pytest.mark.parametrize("lengths,heads,k_heads", [([192], 16, 16), ([2704], 16, 16), ([193, 450], 16, 8),
                                                   ([1000, 0, 257], 8, 8), ([511, 65, 640, 4], 32, 16), ([300], 1, 1), ([128], 16, 16)])
def test_same_bits_as_one_kernel(ctx, dtype, state, lengths, heads, k_heads):
    d = make(lengths, heads, k_heads, dtype, state, 5 + sum(lengths) + heads)
    out, tail, final = run(ctx, d, lengths, heads, k_heads)
    # the same rows with one-token rows behind them: too few chunks per row for the split form
    m = sum(lengths) // 64 + 1
    e = make([1] * m, heads, k_heads, dtype, state, 99)
    both = {k: (torch.cat([d[k], e[k]]) if k in ("mixed", "ba") or (k in ("hist", "init") and state) else d[k]) for k in d}
    both["z"] = both["mixed"][:, (2 * k_heads + heads) * 128:]
    out2, tail2, final2 = run(ctx, both, lengths + [1] * m, heads, k_heads)
    assert ctx.take_faults() == 0
    assert torch.equal(out, out2[: sum(lengths)])
    assert torch.equal(tail, tail2[: len(lengths)])
    assert torch.equal(final, final2[: len(lengths)])


def test_malformed_rows_fault(ctx):
    """A row outside the batch raises the fault bit and leaves the other rows' results as they are."""
    d = make([600], 16, 16, torch.bfloat16, False, 3)
    out, _, _ = run(ctx, d, [600], 16, 16)
    cu = torch.tensor([0, 600, 500], dtype=torch.int32, device="cuda")
    got = torch.zeros_like(out)
    gdn_fused(ctx, d["mixed"], d["conv_w"], d["ba"], 0, 16, d["base_g"], d["dt_bias"], d["z"], d["norm_w"], 1e-6, cu, 16,
              16, out=got)
    assert ctx.take_faults() & 1
    assert torch.equal(got, out)


def test_streams_and_capture(ctx):
    """The scratch follows the context from stream to stream, and a captured call does without it."""
    from huncho_amd.ops import context_for_torch

    d = make([700], 16, 16, torch.bfloat16, False, 8)
    ref, _, _ = run(ctx, d, [700], 16, 16)
    cu = torch.tensor([0, 700], dtype=torch.int32, device="cuda")
    c = context_for_torch(0)
    call = lambda o: gdn_fused(c, d["mixed"], d["conv_w"], d["ba"], 0, 16, d["base_g"], d["dt_bias"], d["z"], d["norm_w"],
                               1e-6, cu, 16, 16, out=o)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [torch.zeros_like(ref) for _ in range(8)]
    for i, o in enumerate(outs):
        c.set_stream(streams[i % 2].cuda_stream)
        call(o)
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
    o = torch.zeros_like(ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.set_stream(torch.cuda.current_stream().cuda_stream)
        call(o)
    for _ in range(3):
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, ref)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.close()
