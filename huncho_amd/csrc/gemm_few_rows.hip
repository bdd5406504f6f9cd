// gemm_few_rows.hip - dense projections of few rows on gfx950 MFMA: Y[m][n] = sum_k X[m][k] W[n][k]
// with the epilogues of gemm.hip, for row counts whose 256 x 256 tiles would leave most of the
// chip's 256 CUs idle (169 rows x 7168 columns are 28 such tiles, x 1024 columns 4).
//
// What bounds such a product is the latency of streaming the weight rows once through too few
// workgroups, not MFMA. So the tile is small, 32 NB columns x 32 MB rows shared by four waves (2 x 2),
// K runs in steps of 64 through a ring of ST stages in LDS, of which ST - U are being loaded (80 to 120 KB per
// CU); where there are tiles enough two workgroups share a CU, and one's loads cover the other's
// reads, barrier and epilogue.
// Each output is one chain of fp32 accumulations over K in order, whatever the tile or the number of
// rows, so a row's result does not change with the batch it comes in: SwiGLU on the 32x32x16 products
// of gemm.hip (the same bits as that kernel), store and residual on 16x16x32 products (the same bits as
// the library's kernels of the large batches, so a prefix computed alone agrees with whole rows in a batch; for the
// smallest batches, few_rows_wins in blas.cpp, the library's choice added in another order).
// (A split of K over the four waves, each with a ring of its own, ran as fast but gave other sums.)
//
// Measured (us, bf16, weights rotated through 600 MB so that they come from HBM; gemm.hip beside it):
//   169 rows, SwiGLU 7168 x 1024       33.9 -> 10.0       600 rows  34.0 -> 21.1
//   169 rows, residual 1024 x 3584      104 -> 11.2      2704 rows  99.4 -> 38.7
//   169 rows, store 8192 x 1024        32.7 -> 9.5        (library 13.6)
//    64 rows, store 2304 x 768         19.2 -> 4.8        (library 7.5)
//   653 rows, GeGLU 2304 x 768: a forward of 22 such layers 1256 -> 1234 against store and the pass over
//                              its rows (the same bits)
// U steps of 64 share a barrier where a wave has few products per step: 32 x 32 tiles over K 3584 took
// 15.7 us with a barrier per step, at any depth of the ring, and 11.2 with one per 4.
//
// Copies, the LDS swizzle and the fragment reads are those of gemm.hip: a K step of an operand row
// is one 128-byte line, copied by buffer_load_dwordx4 ... lds (8 rows per copy; rows past the end
// read as zeros through the resource's bound), its 16-byte chunk c at c ^ ((row >> 1) & 7).
//
// Tiles: workgroup b runs on XCD b % 8. The tiles, all row tiles of a column tile one after
// another, are cut into eight equal ranges, one per XCD, so almost every weight row is fetched into
// one L2, once. (Whole column tiles per XCD left one XCD a sixth of the work of the others at 36
// of them: 2304 x 768, 600 rows, 13.5 us.)
#include <type_traits>

#include "common.hpp"
#include "kernel_args.hpp"

namespace hk {
namespace gemm_few {

constexpr int BK = 64, NTHREADS = 256, ROW_BYTES = BK * 2, BLK_BYTES = 32 * ROW_BYTES;

typedef int i32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4_t buffer_rsrc(const void* base, unsigned bytes) {
    const unsigned long long b = (unsigned long long)base;
    return i32x4_t{__builtin_amdgcn_readfirstlane((int)(b & 0xffffffffu)), __builtin_amdgcn_readfirstlane((int)(b >> 32)),
                   __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}
__device__ __forceinline__ void buf_copy_x4(i32x4_t rsrc, unsigned voff, unsigned soff, unsigned lds) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds) : "memory");
}
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// waits until at most min(steps, STEPS) steps of CPW copies are in flight
template <int STEPS, int CPW> __device__ __forceinline__ void wait_steps(int steps) {
    if constexpr (STEPS == 0) wait_vm<0>();
    else if (steps >= STEPS) wait_vm<STEPS * CPW>();
    else wait_steps<STEPS - 1, CPW>(steps);
}

// as in gemm.hip: bf16 through the hardware reciprocal, fp16 with the IEEE division
template <typename T> __device__ __forceinline__ float silu_f(float x) {
    if constexpr (std::is_same<T, bf16>::value) return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x));
    return x / (1.0f + __expf(-x));
}

template <typename T> __device__ __forceinline__ f32x4 mma16x32(typename Mma16<T>::v8 a, typename Mma16<T>::v8 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mma16x32<bf16>(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x4 mma16x32<f16>(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <typename T, int EPI, int NB, int MB, int ST, int U>
__global__ __launch_bounds__(NTHREADS, 2) void gemm_few_rows(GemmArgs a) {
    typedef typename Mma16<T>::v8 v8;
    constexpr bool GEGLU = EPI == EPI_GEGLU, SWI = EPI == EPI_SWIGLU || GEGLU, RES = EPI == EPI_RESIDUAL || EPI == EPI_RESIDUAL_F32;
    typedef typename std::conditional<EPI == EPI_RESIDUAL_F32, float, T>::type TY;  // rows of c and y
    typedef TY y4 __attribute__((ext_vector_type(4)));
    constexpr int STAGE = (NB + MB) * BLK_BYTES, CPW = NB + MB;  // copies per wave and stage
    static_assert(!SWI || (NB % 2 == 0 && MB % 2 == 0), "a wave's 32 x 32 blocks");
    extern __shared__ __attribute__((aligned(16))) char ssm[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int nt1 = (a.N + 32 * NB - 1) / (32 * NB), nt = nt1 + (a.N2 + 32 * NB - 1) / (32 * NB);
    const int mt = (a.M + 32 * MB - 1) / (32 * MB);
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    int tn = tile / mt;
    const int tm = tile % mt;
    if (tn >= nt) return;
    if (tn >= nt1) {  // the second weight, whose outputs go to rows of their own
        tn -= nt1;
        a.w = a.w2;
        a.y = a.y2;
        a.ldy = a.ldy2;
        a.N = a.N2;
    }
    const int n0 = tn * 32 * NB, m0 = tm * 32 * MB;
    // wave (wn, wm) owns columns n0 + 16 NB wn .. and rows m0 + 16 MB wm ..
    const int wn = wave >> 1, wm = wave & 1;
    const int q4 = lane >> 4, j = lane & 15, g = lane >> 5, lr = lane & 31;

    // the residual rows of this wave's outputs, loaded before the K loop: block (i, jb), 4 columns
    // of row j (clamped, not skipped: rows and columns past the end are not stored)
    y4 cv[RES ? NB : 1][RES ? MB : 1];
    if (RES) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int jb = 0; jb < MB; ++jb) {
                const int n = n0 + 16 * (NB * wn + i) + 4 * q4, m = m0 + 16 * (MB * wm + jb) + j;
                cv[i][jb] = *(const y4*)((const TY*)a.c + (long)min(m, a.M - 1) * a.ldc + min(n, a.N - 4));
            }
    }

    const int crow = lane >> 3, cpc = lane & 7;
    const int lc0 = cpc ^ (crow >> 1), lc1 = cpc ^ (4 + (crow >> 1));
    // GeGLU: the weight holds all gate rows, then all up rows, and the tile's 32-row block c takes gate rows
    // n0 / 2 + 16 c .. + 15 (copies of waves 0 and 1) and their up rows N / 2 further on (waves 2 and 3): the
    // block layout that SwiGLU weights are stored in
    const i32x4_t wrs = GEGLU ? buffer_rsrc(a.w, (unsigned)(a.N * a.ldw * 2))
                              : buffer_rsrc((const T*)a.w + (long)n0 * a.ldw, (unsigned)(min(32 * NB, a.N - n0) * a.ldw * 2));
    const i32x4_t xrs = buffer_rsrc((const T*)a.x + (long)m0 * a.ldx, (unsigned)(min(32 * MB, a.M - m0) * a.ldx * 2));
    // copy c of a stage: 8 rows, odd copies with the swizzle of rows 8 .. 15; wave w issues copies w, w + 4,
    // .. of both operands, all of w's parity
    const int lc = wave & 1 ? lc1 : lc0;
    const unsigned wv = (unsigned)((crow * a.ldw + 8 * lc) * 2), xv = (unsigned)((crow * a.ldx + 8 * lc) * 2);
    const unsigned w8 = (unsigned)(8 * a.ldw * 2), x8 = (unsigned)(8 * a.ldx * 2);
    const unsigned lds0 = lds_address(ssm);
    const int n_steps = a.K / BK;
    auto load_step = [&](int t) {
        const unsigned dst = lds0 + (unsigned)(t % ST) * STAGE, so = (unsigned)t * ROW_BYTES;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const unsigned wo = GEGLU ? (unsigned)(n0 / 16 + 2 * c + (wave & 1) + (wave >> 1) * (a.N / 16)) * w8 : (4 * c + wave) * w8;
            buf_copy_x4(wrs, wv, so + wo, dst + (4 * c + wave) * (8 * ROW_BYTES));
        }
#pragma unroll
        for (int c = 0; c < MB; ++c)
            buf_copy_x4(xrs, xv, so + (4 * c + wave) * x8, dst + (4 * (NB + c) + wave) * (8 * ROW_BYTES));
    };
#pragma unroll
    for (int t = 0; t < ST - U; ++t)
        if (t < n_steps) load_step(t);

    constexpr int WB = SWI ? NB / 2 : NB, XB = SWI ? MB / 2 : MB;  // blocks per wave
    typedef typename std::conditional<SWI, f32x16, f32x4>::type acc_t;
    acc_t acc[WB][XB];
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int jb = 0; jb < XB; ++jb) acc[i][jb] = acc_t{};
    // operand rows: 32x32x16: row lr, chunk 2 s + g of k16-step s; 16x16x32: row j, chunk 4 s + q4 of k32-step s.
    // Blocks start at multiples of 16 rows, so the swizzle is that of the lane's row.
    const int row = SWI ? lr : j, half = SWI ? g : q4, sw = (row >> 1) & 7;
    constexpr int KS = SWI ? 4 : 2, BROWS = SWI ? 32 : 16;
    const int aoff = (16 * NB * wn + row) * ROW_BYTES, boff = (32 * NB + 16 * MB * wm + row) * ROW_BYTES;
    for (int t = 0; t < n_steps; t += U) {
        // this wave's copies of steps t .. t + U - 1 have landed once only those of the steps issued after
        // them are in flight; the barrier makes that all waves', and frees the stages of the U steps before
        wait_steps<ST - 2 * U, CPW>(max(0, n_steps - U - t));
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t + ST - U + u < n_steps) load_step(t + ST - U + u);
        v8 af[U][KS][WB], bf[U][KS][XB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u && t + u >= n_steps) continue;
            const char* st = ssm + ((t + u) % ST) * STAGE;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int co = (((SWI ? 2 : 4) * s + half) ^ sw) << 4;
#pragma unroll
                for (int i = 0; i < WB; ++i) af[u][s][i] = *(const v8*)(st + aoff + co + i * BROWS * ROW_BYTES);
#pragma unroll
                for (int jb = 0; jb < XB; ++jb) bf[u][s][jb] = *(const v8*)(st + boff + co + jb * BROWS * ROW_BYTES);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u && t + u >= n_steps) continue;
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int i = 0; i < WB; ++i)
#pragma unroll
                    for (int jb = 0; jb < XB; ++jb) {
                        if constexpr (SWI) acc[i][jb] = Mma16<T>::mma(af[u][s][i], bf[u][s][jb], acc[i][jb]);
                        else acc[i][jb] = mma16x32<T>(af[u][s][i], bf[u][s][jb], acc[i][jb]);
                    }
        }
    }

#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int jb = 0; jb < XB; ++jb) {
            if constexpr (SWI) {
                // lane (lr, g): row lr, fused rows 32 b + 8 jj + 4 g + r: gate for jj < 2, its up row at jj + 2
                const int nb = n0 + 16 * NB * wn + 32 * i, m = m0 + 16 * MB * wm + 32 * jb + lr;
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    y4 o;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float gv = to_f(from_f<T>(acc[i][jb][4 * jj + r]));
                        o[r] = from_f<TY>((GEGLU ? gelu_erf(gv) : silu_f<T>(gv)) * to_f(from_f<T>(acc[i][jb][4 * (jj + 2) + r])));
                    }
                    if (m < a.M && nb < a.N) *(y4*)((TY*)a.y + (long)m * a.ldy + nb / 2 + 8 * jj + 4 * g) = o;
                }
            } else {
                const int n = n0 + 16 * (NB * wn + i) + 4 * q4, m = m0 + 16 * (MB * wm + jb) + j;
                y4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = from_f<TY>(RES ? acc[i][jb][r] + to_f(cv[i][jb][r]) : acc[i][jb][r]);
                if (m < a.M && n < a.N) *(y4*)((TY*)a.y + (long)m * a.ldy + n) = o;
            }
        }
}

}  // namespace gemm_few
}  // namespace hk

// The tiles and their cost in units of K / 1024 us (beside about 2.2 us of launch and first loads), fitted to the
// times of every tile over ten projections of the models (32 to 8192 columns, K 768 to 3584) at 34 to 32768 rows:
// flat while the tiles fit the chip at once; for more, rising with their number (slope), with a step where the
// third workgroup of a CU begins (past_512), or in rounds of 512 (two workgroups per CU) for the tiles whose
// second workgroup on a CU takes as long as the first. X rows that do not stay in an XCD's L2 are read
// once more for every column tile, at 17 TB/s over the chip: 1024 x 3584 at 4096 rows takes 66.8 us in
// 64-column tiles and 46.1 in 128-column ones, of the same number and size.
namespace {
struct Tile {
    int nb, mb;
    float first, slope, past_512, round;
};
constexpr Tile kTiles[] = {{1, 1, 2.5f, 0.0094f, 0.0f, 0.0f}, {1, 2, 2.9f, 0.0135f, 0.0f, 0.0f}, {2, 2, 5.1f, 0.0153f, 4.2f, 0.0f},
                           {2, 3, 5.3f, 0.0f, 0.0f, 8.2f},    {2, 4, 6.2f, 0.0f, 0.0f, 10.8f},   {4, 2, 6.9f, 0.0f, 0.0f, 10.9f}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

long col_tiles(const hk::GemmArgs* a, const Tile& t) {
    const int w = 32 * t.nb;
    return (a->N + w - 1) / w + (a->N2 + w - 1) / w;
}
long n_tiles(const hk::GemmArgs* a, const Tile& t) { return col_tiles(a, t) * ((a->M + 32 * t.mb - 1) / (32 * t.mb)); }

int best_tile(int epi, const hk::GemmArgs* a, float* cost) {
    const bool x_in_l2 = 2.0f * (float)a->M * (float)a->K < 5e6f;
    int best = -1;
    for (int i = 0; i < kNumTiles; ++i) {
        if ((epi == hk::EPI_SWIGLU || epi == hk::EPI_GEGLU) && (kTiles[i].nb % 2 || kTiles[i].mb % 2)) continue;  // four waves' 32 x 32 blocks
        const Tile& k = kTiles[i];
        const long n = n_tiles(a, k);
        float c = n <= 256 ? k.first
                  : k.round > 0.0f ? k.round * (float)((n + 511) / 512)
                                   : k.first + k.slope * (float)(n - 256) + (n > 512 ? k.past_512 : 0.0f);
        if (!x_in_l2) c += (float)(col_tiles(a, k) * a->M) * (2048.0f / 17e6f);
        if (best < 0 || c < *cost) {
            best = i;
            *cost = c;
        }
    }
    return best;
}
}  // namespace

template <typename T, int EPI, int I, int ST, int U>
static int launch_one(const hk::GemmArgs* a, hipStream_t stream) {
    constexpr int NB = kTiles[I].nb, MB = kTiles[I].mb;
    if constexpr ((EPI == hk::EPI_SWIGLU || EPI == hk::EPI_GEGLU) && (NB % 2 || MB % 2)) {
        return HK_ERR_DEVICE;  // best_tile does not choose it
    } else {
        constexpr int lds = ST * (NB + MB) * hk::gemm_few::BLK_BYTES;
        static_assert(lds <= 160 * 1024, "the ring fits the LDS");
        auto kern = hk::gemm_few::gemm_few_rows<T, EPI, NB, MB, ST, U>;
        // set once, under C++'s thread-safe static initialisation (replicas launch from several threads)
        static const bool configured =
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
        if (!configured) return HK_ERR_DEVICE;
        hipLaunchKernelGGL(kern, dim3((unsigned)((n_tiles(a, kTiles[I]) + 7) / 8 * 8)), dim3(hk::gemm_few::NTHREADS), lds,
                           stream, *a);
        return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
    }
}

template <typename T, int EPI>
static int launch_epi(const hk::GemmArgs* a, int i, int deep, hipStream_t stream) {
    switch (i) {
        case 0: return deep ? launch_one<T, EPI, 0, 18, 4>(a, stream) : launch_one<T, EPI, 0, 9, 4>(a, stream);
        case 1: return deep ? launch_one<T, EPI, 1, 12, 4>(a, stream) : launch_one<T, EPI, 1, 6, 2>(a, stream);
        case 2: return deep ? launch_one<T, EPI, 2, 9, 4>(a, stream) : launch_one<T, EPI, 2, 5, 2>(a, stream);
        case 3: return deep ? launch_one<T, EPI, 3, 8, 2>(a, stream) : launch_one<T, EPI, 3, 4, 1>(a, stream);
        case 4: return deep ? launch_one<T, EPI, 4, 6, 2>(a, stream) : launch_one<T, EPI, 4, 3, 1>(a, stream);
        case 5: return deep ? launch_one<T, EPI, 5, 6, 2>(a, stream) : launch_one<T, EPI, 5, 3, 1>(a, stream);
        default: return HK_ERR_DEVICE;
    }
}

template <typename T>
static int launch_type(int epi, const hk::GemmArgs* a, int i, int deep, hipStream_t stream) {
    switch (epi) {
        case hk::EPI_RESIDUAL: return launch_epi<T, hk::EPI_RESIDUAL>(a, i, deep, stream);
        case hk::EPI_RESIDUAL_F32: return launch_epi<T, hk::EPI_RESIDUAL_F32>(a, i, deep, stream);
        case hk::EPI_SWIGLU: return launch_epi<T, hk::EPI_SWIGLU>(a, i, deep, stream);
        case hk::EPI_GEGLU: return launch_epi<T, hk::EPI_GEGLU>(a, i, deep, stream);
        default: return launch_epi<T, hk::EPI_STORE>(a, i, deep, stream);
    }
}

// Cost of the best tile in units of K / 1024 us (beside about 2.2 us of launch and first loads).
extern "C" float hk_gemm_few_rows_cost(int epi, const hk::GemmArgs* a) {
    float cost = 0.0f;
    best_tile(epi, a, &cost);
    return cost;
}

// dtype16: 1 = bf16, 2 = fp16. The caller has checked: N and N2 % 8 == 0 (SwiGLU, GeGLU: N % 32), K % 64 == 0,
// 16-byte aligned rows (ld % 8 == 0) and row strides below 2^22 elements (32-bit copy offsets).
extern "C" int hk_launch_gemm_few_rows(int dtype16, int epi, const hk::GemmArgs* a, hipStream_t stream) {
    float cost;
    const int i = best_tile(epi, a, &cost);
    // Tiles that fit the chip at once run one workgroup per CU with a ring of up to 160 KB, more tiles two with
    // half of it.
    return hk_launch_gemm_few_rows_tile(dtype16, epi, a, i, n_tiles(a, kTiles[i]) <= 256, stream);
}

// The same with tile i of kTiles and its deep or shallow ring (tests reach every instance through it).
extern "C" int hk_launch_gemm_few_rows_tile(int dtype16, int epi, const hk::GemmArgs* a, int i, int deep, hipStream_t stream) {
    if (a->M == 0) return HK_OK;
    return dtype16 == hk::DT_BF16 ? launch_type<hk::bf16>(epi, a, i, deep, stream)
                                  : launch_type<hk::f16>(epi, a, i, deep, stream);
}
