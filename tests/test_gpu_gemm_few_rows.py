"""The few-row GEMM (gemm_few_rows.hip) against a float64 product of the same 16-bit values: through hk_linear
around the row counts where its tiles begin and K of one to many steps; and each tile, ring and epilogue by
itself, at row counts one more and less than the tile's, column counts that leave a part of a tile, K steps
that do not fill the last barrier's, a second weight, and guard values around every output; and its bits
against those of many rows, which run on gemm.hip.

Gates: 1 unit in the last place of the dtype (2^-7 relative for bf16, 2^-10 for fp16) plus the fp32
accumulation's absolute error over K products; the SwiGLU and GeGLU epilogues 2 units, from the rounded gate
and up products."""
import ctypes as C

import pytest
import torch

from huncho_amd import abi

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


@pytest.fixture(scope="module")
def ctx():
    from huncho_amd.ops import context_for_torch

    c = context_for_torch(0)
    yield c
    c.close()


def linear(ctx, x, w, epi=0, c=None, out_cols=None):
    y = torch.full((x.shape[0] + 1, out_cols or w.shape[0]), 7.0, dtype=x.dtype, device=x.device)
    dt = abi.HK_BF16 if x.dtype == torch.bfloat16 else abi.HK_F16
    ctx.check(abi.lib().hk_linear(ctx.h, dt, epi, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), x.shape[0],
                                  w.shape[0], x.shape[1], c.data_ptr() if c is not None else None,
                                  c.stride(0) if c is not None else 0, y.data_ptr(), y.stride(0)))
    assert bool((y[-1] == 7.0).all())  # nothing is stored past the last row
    return y[:-1]


def within(got, want, dtype, ulps, k):
    g, w = got.double(), want.double()
    return bool(((g - w).abs() <= w.abs() * EPS[dtype] * ulps + 4e-7 * k).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 31, 33, 64, 65, 97, 169, 300, 700])
@pytest.mark.parametrize("n,k", [(256, 64), (1024, 192), (768, 1152), (3584, 320)])
def test_linear_few_rows(ctx, dtype, rows, n, k):
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + n + k)
    pad = torch.randn((rows, k + 8), generator=g, device="cuda").to(dtype) * 0.5
    x = pad[:, :k]  # a row stride wider than the row
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).to(dtype)
    ref = x.double() @ w.double().T
    assert within(linear(ctx, x, w), ref.to(dtype), dtype, 1, k)
    c = torch.randn((rows, n), generator=g, device="cuda").to(dtype)
    assert within(linear(ctx, x, w, 1, c), (ref + c.double()).to(dtype), dtype, 1, k)
    b = ref.view(rows, n // 32, 2, 16).to(dtype).double()
    gate, up = b[:, :, 0].reshape(rows, -1), b[:, :, 1].reshape(rows, -1)
    # a gate or up product next to a rounding boundary may round the other way: one unit of each
    tol = 2 * EPS[dtype] * (gate.abs() * up.abs() + (torch.nn.functional.silu(gate) * up).abs()) + 4e-7 * k
    got = linear(ctx, x, w, 2, out_cols=n // 2).double()
    assert bool(((got - torch.nn.functional.silu(gate) * up).abs() <= tol).all())


class GemmArgs(C.Structure):
    _fields_ = [("x", C.c_void_p), ("w", C.c_void_p), ("c", C.c_void_p), ("y", C.c_void_p), ("ldx", C.c_long),
                ("ldw", C.c_long), ("ldc", C.c_long), ("ldy", C.c_long), ("M", C.c_int), ("N", C.c_int), ("K", C.c_int),
                ("w2", C.c_void_p), ("y2", C.c_void_p), ("ldy2", C.c_long), ("N2", C.c_int)]


STORE, RESIDUAL, SWIGLU, RESIDUAL_F32, GEGLU = range(5)
TILES = [(1, 1), (1, 2), (2, 2), (2, 3), (2, 4), (4, 2)]  # 32-column and 32-row blocks


def guarded(m, n, dtype):
    """[m][n] inside a larger buffer of sevens: (the view, a check that nothing around it was written)."""
    buf = torch.full((m + 2, n + 16), 7.0, dtype=dtype, device="cuda")

    def clean():
        inner = buf[1:m + 1, 8:n + 8].clone()
        buf[1:m + 1, 8:n + 8] = 7.0
        ok = bool((buf == 7.0).all())
        buf[1:m + 1, 8:n + 8] = inner
        return ok

    return buf[1:m + 1, 8:n + 8], clean


def one_tile(dtype, epi, tile, deep, x, w, n_out, c=None, w2=None):
    f = abi.lib().hk_launch_gemm_few_rows_tile
    f.restype, f.argtypes = C.c_int, [C.c_int, C.c_int, C.POINTER(GemmArgs), C.c_int, C.c_int, C.c_void_p]
    y, clean = guarded(x.shape[0], n_out, torch.float32 if epi == RESIDUAL_F32 else dtype)
    a = GemmArgs(x=x.data_ptr(), w=w.data_ptr(), y=y.data_ptr(), ldx=x.stride(0), ldw=w.stride(0), ldy=y.stride(0),
                 M=x.shape[0], N=w.shape[0], K=x.shape[1])
    if c is not None:
        a.c, a.ldc = c.data_ptr(), c.stride(0)
    y2 = clean2 = None
    if w2 is not None:
        y2, clean2 = guarded(x.shape[0], w2.shape[0], dtype)
        a.w2, a.y2, a.ldy2, a.N2 = w2.data_ptr(), y2.data_ptr(), y2.stride(0), w2.shape[0]
    rc = f(1 if dtype == torch.bfloat16 else 2, epi, C.byref(a), tile, deep, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and clean() and (clean2 is None or clean2())
    return (y, y2) if w2 is not None else y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("deep", [0, 1])
@pytest.mark.parametrize("tile", range(6))
def test_every_instance_at_its_edges(dtype, deep, tile):
    nb, mb = TILES[tile]
    g = torch.Generator(device="cuda").manual_seed(10 * tile + deep)
    r = lambda m, n, s=1.0: (torch.randn((m, n), generator=g, device="cuda") * s).to(dtype)
    for m in (1, 32 * mb - 1, 32 * mb + 1):
        for k in (64, 320, 576, 1280):  # 1, 5, 9 and 20 steps
            x = r(m, k + 8, 0.5)[:, :k]
            for n in (8, 40, 264):
                w, w2 = r(n, k, 0.05), r(32 * nb + 8, k, 0.05)
                ref, ref2 = x.double() @ w.double().T, x.double() @ w2.double().T
                assert within(one_tile(dtype, STORE, tile, deep, x, w, n), ref.to(dtype), dtype, 1, k)
                y, y2 = one_tile(dtype, STORE, tile, deep, x, w, n, w2=w2)
                assert within(y, ref.to(dtype), dtype, 1, k) and within(y2, ref2.to(dtype), dtype, 1, k)
                c = r(m, n + 8)[:, :n]
                got = one_tile(dtype, RESIDUAL, tile, deep, x, w, n, c)
                assert within(got, (ref + c.double()).to(dtype), dtype, 1, k)
                c = torch.randn((m, n + 8), generator=g, device="cuda")[:, :n]
                got = one_tile(dtype, RESIDUAL_F32, tile, deep, x, w, n, c).double()
                assert bool(((got - ref - c.double()).abs() <= 4e-7 * k).all())
            if nb % 2 or mb % 2:
                continue
            for n in (32, 96, 288):
                w = r(n, k, 0.05)
                b = (x.double() @ w.double().T).to(dtype).double()
                fused = b.view(m, n // 32, 2, 16)
                for epi, gate, up, act in (
                        (SWIGLU, fused[:, :, 0].reshape(m, -1), fused[:, :, 1].reshape(m, -1), torch.nn.functional.silu),
                        (GEGLU, b[:, :n // 2], b[:, n // 2:], torch.nn.functional.gelu)):
                    tol = 2 * EPS[dtype] * (gate.abs() * up.abs() + (act(gate) * up).abs()) + 4e-7 * k
                    got = one_tile(dtype, epi, tile, deep, x, w, n // 2).double()
                    assert bool(((got - act(gate) * up).abs() <= tol).all()), (epi, m, k, n)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epi,n,k", [(0, 1024, 1024), (1, 1024, 3584), (2, 7168, 1024), (1, 768, 1152)])
def test_rows_do_not_depend_on_the_batch(ctx, dtype, epi, n, k):
    """An output is one chain of sums over K in order on every path, so a row's result is the same bits
    in a batch of any size."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((16384, k), generator=g, device="cuda").to(dtype)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).to(dtype)
    c = torch.randn((16384, n), generator=g, device="cuda").to(dtype) if epi == 1 else None
    cols = n // 2 if epi == 2 else n
    whole = linear(ctx, x, w, epi, c, cols)  # gemm.hip
    for rows in (1, 40, 100, 169, 300, 600, 1200):
        assert torch.equal(linear(ctx, x[:rows], w, epi, c[:rows] if epi == 1 else None, cols), whole[:rows]), rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hidden,heads,inter", [(768, 12, 1152), (256, 4, 176)])
def test_encoder_rows_do_not_depend_on_the_batch(ctx, dtype, hidden, heads, inter):
    """The encoder's few-row path (its GeGLU projection in one launch) gives a row the bits that it has
    in a batch of many rows, which runs the projection and the GeGLU pass on their own. 176 gate columns
    leave a part of a tile."""
    import numpy as np

    from huncho_amd.laya import LayaModel, LayaShape, synthetic_weights

    shape = LayaShape(hidden=hidden, n_layers=3, n_heads=heads, intermediate=inter, vocab=500, max_context=512, n_out=2)
    model = LayaModel(ctx, shape, synthetic_weights(shape, 3, std=0.05), dtype)
    rng = np.random.default_rng(1)
    rows = [rng.integers(0, 500, n).tolist() for n in [70, 1, 200] + [500] * 24]
    many, hm = model.forward_batch(rows, want_hidden=True)
    for n in (1, 2, 3):
        few, hf = model.forward_batch(rows[:n], want_hidden=True)
        assert all(np.array_equal(a, b) for a, b in zip(hf, hm[:n]))
        assert np.array_equal(few, many[:n])
    model.close()
