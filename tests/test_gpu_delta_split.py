"""The fp32 gated delta rule for few rows (delta_rule_split.hip) against the per-token recurrence in
float64: rows that end on, before and after a chunk boundary, an empty row, shared key heads, a carried
state that aliases the final one, and against gdn_chunk_f32, which the same rows take in a larger batch.

Tolerance (2-norm): fp32 sums of 128 products and a few roundings per token, whose errors the state
carries on: 64 x 2^-24 = 4e-6 of the result, as far as gdn_chunk_f32 itself may lie from it."""
import pytest
import torch

from huncho_amd.ops import gated_delta_chunked

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from huncho_amd.ops import context_for_torch

    c = context_for_torch(0)
    yield c
    c.close()


def make(lengths, heads, k_heads, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")
    n = sum(lengths)
    return {"q": torch.nn.functional.normalize(r(n, k_heads, 128), dim=-1) * 128 ** -0.5,
            "k": torch.nn.functional.normalize(r(n, k_heads, 128), dim=-1), "v": r(n, heads, 128),
            "g": -torch.nn.functional.softplus(r(n, heads) - 2.0), "beta": torch.sigmoid(r(n, heads)),
            "s0": r(len(lengths), heads, 128, 128) * 0.1}


def run(ctx, d, lengths, state):
    cu = torch.tensor([0] + lengths, device="cuda").cumsum(0).to(torch.int32)
    st = d["s0"].clone() if state else torch.full_like(d["s0"], 7.0)
    o = gated_delta_chunked(ctx, d["q"], d["k"], d["v"], d["g"], d["beta"], cu, initial_state=st if state else None,
                            final_state=st)
    assert ctx.take_faults() == 0
    return o, st


def recurrence(d, lengths, heads, k_heads, state):
    rep, outs, states, t0 = heads // k_heads, [], [], 0
    q, k = (d[x].double().repeat_interleave(rep, 1) for x in ("q", "k"))
    v, g, b = (d[x].double() for x in ("v", "g", "beta"))
    for s, L in enumerate(lengths):
        S = d["s0"][s].double() if state else torch.zeros(heads, 128, 128, dtype=torch.float64, device="cuda")
        for t in range(t0, t0 + L):
            S = S * torch.exp(g[t])[:, None, None]
            dl = b[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * dl[:, None]
            outs.append((S * q[t][:, :, None]).sum(1))
        states.append(S)
        t0 += L
    return torch.stack(outs), torch.stack(states)


@pytest.mark.parametrize("state", [False, True])
@pytest.mark.parametrize("lengths,heads,k_heads", [([64], 16, 16), ([512], 16, 16), ([65, 191], 16, 8), ([700, 0, 63], 8, 8),
                                                   ([130], 1, 1)])
def test_against_the_recurrence(ctx, state, lengths, heads, k_heads):
    d = make(lengths, heads, k_heads, sum(lengths) + heads)
    o, st = run(ctx, d, lengths, state)
    ro, rs = recurrence(d, lengths, heads, k_heads, state)
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())
    assert rel(o, ro) < 4e-6 and rel(st, rs) < 4e-6, (rel(o, ro), rel(st, rs))
    # the same rows beside enough one-token rows to run on one kernel
    m = 160 // heads + 1 + sum(lengths) // 32
    e = make([1] * m, heads, k_heads, 5)
    both = {x: torch.cat([d[x], e[x]]) for x in d}
    o2, st2 = run(ctx, both, lengths + [1] * m, state)
    assert rel(o, o2[: sum(lengths)].double()) < 8e-6 and rel(st, st2[: len(lengths)].double()) < 8e-6


def test_output_in_place_of_q(ctx):
    """Calls that the split form cannot serve keep their results: o in the place of q."""
    d = make([256], 16, 16, 3)
    o, _ = run(ctx, d, [256], False)
    cu = torch.tensor([0, 256], dtype=torch.int32, device="cuda")
    q = d["q"].clone()
    gated_delta_chunked(ctx, q, d["k"], d["v"], d["g"], d["beta"], cu, out=q)
    assert float((q - o).norm() / o.norm()) < 8e-6
