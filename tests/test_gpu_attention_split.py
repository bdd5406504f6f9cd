"""The key-split paged attention (few rows over long contexts) against float64 attention over the same
16-bit values: contexts that end on, before and after a 64-key tile, one and several q-blocks, rows too
short to be split beside long ones, both head widths, groups of 1 to 8, shared pages, with and without
the gate.

Tolerance (2-norm): a probability, the output, the gate and their product are each rounded once to the
dtype, an rms of 2^-9 / sqrt(3) (bf16) or 2^-12 / sqrt(3) (fp16) per rounding: 2.3e-3 and 2.8e-4 for
four; twice that."""
import math

import numpy as np
import pytest
import torch

from huncho_amd.ops import paged_prefill_attention

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 4.6e-3, torch.float16: 5.6e-4}


@pytest.fixture(scope="module")
def ctx():
    from huncho_amd.ops import context_for_torch

    c = context_for_torch(0)
    yield c
    c.close()


def run(ctx, q_lens, ctx_lens, hq, hkv, d, page, dtype, gate, seed, spare=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)
    n, rows = sum(q_lens), len(q_lens)
    need = [(c + page - 1) // page for c in ctx_lens]
    perm = np.random.default_rng(seed).permutation(sum(need)).astype(np.int32)
    bt = np.zeros((rows, max(need) + spare), np.int32)
    at = 0
    for s, m in enumerate(need):
        bt[s, :m] = perm[at:at + m]
        at += m
    kp, vp = r(sum(need), hkv, page, d), r(sum(need), hkv, page, d)
    qg = r(n, hq, 2 * d)
    q, gt = qg[:, :, :d], qg[:, :, d:]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32, device="cuda")
    lens = torch.tensor(ctx_lens, dtype=torch.int32, device="cuda")
    o = paged_prefill_attention(ctx, q, kp, vp, torch.from_numpy(bt).cuda(), cu, lens, max(q_lens),
                                gate=gt if gate else None)
    assert ctx.take_faults() == 0
    refs, t0 = [], 0
    for s, (L, c) in enumerate(zip(q_lens, ctx_lens)):
        pages = torch.from_numpy(bt[s, :need[s]].astype(np.int64)).cuda()
        kk = kp[pages].transpose(1, 2).reshape(-1, hkv, d)[:c].double().repeat_interleave(hq // hkv, 1)
        vv = vp[pages].transpose(1, 2).reshape(-1, hkv, d)[:c].double().repeat_interleave(hq // hkv, 1)
        qq = q[t0:t0 + L].double().transpose(0, 1).contiguous()
        sc = qq @ kk.permute(1, 2, 0).contiguous() / math.sqrt(d)
        pos = torch.arange(c - L, c, device="cuda")
        sc.masked_fill_(torch.arange(c, device="cuda")[None] > pos[:, None], -math.inf)
        ref = (sc.softmax(-1) @ vv.transpose(0, 1).contiguous()).transpose(0, 1)
        refs.append(ref * torch.sigmoid(gt[t0:t0 + L].double()) if gate else ref)
        t0 += L
    ref = torch.cat(refs)
    return o, float((o.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("q_lens,ctx_lens,hq,hkv,d,page", [
    ([1], [1024], 16, 8, 128, 16), ([30, 20, 40], [2700, 2701, 2751], 16, 8, 128, 16), ([1], [4097], 8, 8, 128, 64),
    ([64, 3], [2048, 10], 16, 8, 128, 16), ([65], [1985], 16, 8, 128, 32), ([300], [1500], 16, 8, 128, 16),
    ([200, 1, 500], [900, 3000, 700], 16, 2, 128, 16), ([33], [3000], 8, 2, 256, 16), ([200], [1300], 16, 4, 256, 16)])
def test_split_matches_float64(ctx, dtype, gate, q_lens, ctx_lens, hq, hkv, d, page):
    _, e = run(ctx, q_lens, ctx_lens, hq, hkv, d, page, dtype, gate, sum(q_lens) + sum(ctx_lens))
    assert e < TOL[dtype], e


def test_short_context_under_a_wide_table(ctx):
    """The ranges follow the context, not the table's width: a short row is not split, and gives the same
    bits as under a table of its own size."""
    a, _ = run(ctx, [20], [150], 16, 8, 128, 16, torch.bfloat16, True, 5)
    b, e = run(ctx, [20], [150], 16, 8, 128, 16, torch.bfloat16, True, 5, spare=500)
    assert torch.equal(a, b) and e < TOL[torch.bfloat16]


def test_a_fresh_row_keeps_its_bits(ctx):
    """A row without cached tokens is not split: alone it gives the bits that it has in a large batch."""
    a, _ = run(ctx, [1100], [1100], 16, 8, 128, 16, torch.bfloat16, True, 7)
    g = torch.Generator(device="cuda").manual_seed(7)  # the same row first among 40
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    need = (1100 + 15) // 16
    kp, vp, qg = r(need, 8, 16, 128), r(need, 8, 16, 128), r(1100, 16, 256)
    bt = torch.from_numpy(np.random.default_rng(7).permutation(need).astype(np.int32)).cuda().view(1, -1).repeat(40, 1)
    cu = torch.arange(0, 40 * 1100 + 1, 1100, dtype=torch.int32, device="cuda")
    q = qg.repeat(40, 1, 1)
    o = paged_prefill_attention(ctx, q[:, :, :128], kp, vp, bt, cu, torch.full((40,), 1100, dtype=torch.int32, device="cuda"),
                                1100, gate=q[:, :, 128:])
    assert torch.equal(a, o[:1100]) and torch.equal(a, o[-1100:])


def rows_of_one_batch(ctx, q_lens, ctx_lens, picks, spares, seed=11):
    """The outputs of each pick of the rows, as batches of their own under tables with spare columns."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    need = [(c + 15) // 16 for c in ctx_lens]
    kp, vp = r(sum(need), 8, 16, 128), r(sum(need), 8, 16, 128)
    first = np.concatenate([[0], np.cumsum(need)])
    qg = [r(L, 16, 256) for L in q_lens]
    out = []
    for pick, spare in zip(picks, spares):
        bt = np.zeros((len(pick), max(need[s] for s in pick) + spare), np.int32)
        for i, s in enumerate(pick):
            bt[i, :need[s]] = np.arange(first[s], first[s] + need[s])
        q = torch.cat([qg[s] for s in pick])
        cu = torch.tensor(np.concatenate([[0], np.cumsum([q_lens[s] for s in pick])]), dtype=torch.int32, device="cuda")
        lens = torch.tensor([ctx_lens[s] for s in pick], dtype=torch.int32, device="cuda")
        o = paged_prefill_attention(ctx, q[:, :, :128], kp, vp, torch.from_numpy(bt).cuda(), cu, lens,
                                    max(q_lens[s] for s in pick), gate=q[:, :, 128:])
        out.append(dict(zip(pick, o.split([q_lens[s] for s in pick]))))
    assert ctx.take_faults() == 0
    return out


@pytest.mark.parametrize("fresh", [65, 600, 1000])
def test_a_fresh_row_keeps_its_bits_beside_suffixes(ctx, fresh):
    """Whether a row is split goes by its own lengths: a row without cached tokens gives the same bits alone,
    under a wide table, and beside a suffix that is split."""
    alone, wide, both = rows_of_one_batch(ctx, [fresh, 30], [fresh, 2700], [[0], [0], [0, 1]], [0, 250, 0])
    assert torch.equal(alone[0], wide[0])
    assert torch.equal(alone[0], both[0])


def test_a_suffix_does_not_depend_on_the_table(ctx):
    """The ranges of a suffix follow its context: the table's width does not change its bits."""
    q_lens, ctx_lens = [30, 20, 33], [2700, 1300, 1100]
    narrow, wide = rows_of_one_batch(ctx, q_lens, ctx_lens, [[0, 1, 2]] * 2, [0, 700])
    assert all(torch.equal(narrow[s], wide[s]) for s in range(3))


def test_many_launches_in_a_row(ctx):
    """The counts of finished ranges are zero again after each launch, whatever the batch before was."""
    a = [run(ctx, *x, 16, 8, 128, 16, torch.bfloat16, True, 9) for x in (([30] * 5, [2700] * 5), ([1], [4097]), ([128], [2048]))]
    for _ in range(3):
        for x, (o, e) in zip((([30] * 5, [2700] * 5), ([1], [4097]), ([128], [2048])), a):
            o2, _ = run(ctx, *x, 16, 8, 128, 16, torch.bfloat16, True, 9)
            assert e < TOL[torch.bfloat16] and torch.equal(o, o2)


def test_nan_and_infinite_scores(ctx):
    """A key whose scores are +inf or NaN makes its rows NaN, as softmax does, in whichever range it lies;
    keys past a row's position do not reach it."""
    g = torch.Generator(device="cuda").manual_seed(2)
    c, L = 2000, 8
    kp = torch.randn((125, 8, 16, 128), generator=g, device="cuda").to(torch.bfloat16)
    vp = torch.randn((125, 8, 16, 128), generator=g, device="cuda").to(torch.bfloat16)
    q = torch.rand((L, 16, 128), generator=g, device="cuda").to(torch.bfloat16) + 0.1
    bt = torch.arange(125, dtype=torch.int32, device="cuda").view(1, -1)
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    lens = torch.tensor([c], dtype=torch.int32, device="cuda")
    for key, val in ((1000, math.inf), (300, math.nan)):
        k2 = kp.clone()
        k2[key // 16, 0, key % 16] = val
        o = paged_prefill_attention(ctx, q, k2, vp, bt, cu, lens, L)
        assert bool(o[:, :2].isnan().all()) and not bool(o[:, 2:].isnan().any())
    k2 = kp.clone()
    k2[124, :, 15] = math.inf  # key 1999: visible to the last row alone
    o = paged_prefill_attention(ctx, q, k2, vp, bt, cu, lens, L)
    assert not bool(o[:-1].isnan().any()) and bool(o[-1].isnan().all())
    ctx.take_faults()
