// gemm_split.hip - dense projections of few rows on gfx950 MFMA: Y[m][n] = sum_k X[m][k] W[n][k]
// with the epilogues of gemm.hip, for row counts whose 256 x 256 tiles would leave most of the
// chip's 256 CUs idle (169 rows x 7168 columns are 28 such tiles, x 1024 columns 4).
//
// What bounds such a product is the latency of streaming the weight rows once through too few
// workgroups, not MFMA. So the tile is small, 32 NB columns x 32 MB rows, and the four waves of a
// workgroup split the K loop instead of the tile: wave w runs the whole tile over K steps
// [w nk / 4, (w + 1) nk / 4) of 64 through a ring of ST stages in LDS of its own. The waves share
// nothing until the end, so the K loop has no barrier, only each wave's own vmcnt waits, and the
// rings of a CU's workgroups keep 96 - 160 KB of loads in flight. The partial sums meet once, in
// fp32, through LDS: every wave adds a quarter of the tile in the order of the waves and runs the
// epilogue on it. The split of K does not depend on the tile shape, so every (NB, MB) gives the
// same sums bit for bit, whatever the number of rows.
//
// Measured (bf16, weights rotated through 600 MB so that they come from HBM; gemm.hip beside it):
//   169 rows, SwiGLU 7168 x 1024       33.9 -> 9.8 us     600 rows  34.0 -> 23.1 us
//   169 rows, residual 1024 x 3584      104 -> 9.0 us    2704 rows  99.4 -> 42.0 us
//   169 rows, store 8192 x 1024        32.7 -> 10.1 us  (library 13.6 us)
//    64 rows, store 2304 x 768         19.2 -> 4.4 us   (library 7.5 us)
// One stage per wave with two or three workgroups per CU beats two or three stages with one
// (64 x 64 tiles, 1200 rows x 7168: 36.5 against 47.5 us): the other workgroup's loads cover a
// wave's reads, its epilogue and the sums. Only the 32 x 32 tile, whose rows are fewest, keeps 4.
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
namespace gemms {

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
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// as in gemm.hip: bf16 through the hardware reciprocal, fp16 with the IEEE division
template <typename T> __device__ __forceinline__ float silu_f(float x) {
    if constexpr (std::is_same<T, bf16>::value) return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x));
    return x / (1.0f + __expf(-x));
}

template <typename T, int EPI, int NB, int MB, int ST>
__global__ __launch_bounds__(NTHREADS, NB * MB < 8 ? 2 : 1) void gemm_ksplit(GemmArgs a) {
    typedef typename Mma16<T>::v8 v8;
    constexpr int STAGE = (NB + MB) * BLK_BYTES, CP = (NB + MB) * 4;
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
    const int g = lane >> 5, lr = lane & 31;

    // this wave's quarter of the epilogue: blocks (i, j), u = wave + 4 t in units of 4 (SwiGLU: 2)
    // runs of 4 columns per block; the residual rows it needs are loaded before the K loop
    constexpr int RUNS = EPI == EPI_SWIGLU ? 2 : 4, UNITS = NB * MB * RUNS / 4;
    static_assert(NB * MB * RUNS % 4 == 0, "the four waves share the epilogue evenly");
    typedef typename std::conditional<EPI == EPI_RESIDUAL_F32, float, T>::type TY;  // rows of c and y
    typedef TY y4 __attribute__((ext_vector_type(4)));
    constexpr bool RES = EPI == EPI_RESIDUAL || EPI == EPI_RESIDUAL_F32;
    y4 cv[UNITS];
    if (RES) {
#pragma unroll
        for (int t = 0; t < UNITS; ++t) {
            const int u = wave + 4 * t, blk = u / RUNS, jj = u % RUNS;
            const int n = n0 + 32 * (blk / MB) + 8 * jj + 4 * g, m = m0 + 32 * (blk % MB) + lr;
            // clamped, not skipped: rows and columns past the end are not stored
            cv[t] = *(const y4*)((const TY*)a.c + (long)min(m, a.M - 1) * a.ldc + min(n, a.N - 4));
        }
    }

    const int crow = lane >> 3, cpc = lane & 7;
    const int lc0 = cpc ^ (crow >> 1), lc1 = cpc ^ (4 + (crow >> 1));
    const i32x4_t wrs = buffer_rsrc((const T*)a.w + (long)n0 * a.ldw, (unsigned)(min(32 * NB, a.N - n0) * a.ldw * 2));
    const i32x4_t xrs = buffer_rsrc((const T*)a.x + (long)m0 * a.ldx, (unsigned)(min(32 * MB, a.M - m0) * a.ldx * 2));
    const unsigned wv[2] = {(unsigned)((crow * a.ldw + 8 * lc0) * 2), (unsigned)((crow * a.ldw + 8 * lc1) * 2)};
    const unsigned xv[2] = {(unsigned)((crow * a.ldx + 8 * lc0) * 2), (unsigned)((crow * a.ldx + 8 * lc1) * 2)};
    const unsigned w8 = (unsigned)(8 * a.ldw * 2), x8 = (unsigned)(8 * a.ldx * 2);
    char* const ring = ssm + wave * (ST * STAGE);
    const unsigned lring = lds_address(ring);
    const int nk = a.K / BK, k0 = wave * nk / 4, k1 = (wave + 1) * nk / 4, n_steps = k1 - k0;
    auto load_step = [&](int t) {
        const unsigned dst = lring + (unsigned)(t % ST) * STAGE, so = (unsigned)(k0 + t) * ROW_BYTES;
#pragma unroll
        for (int c = 0; c < 4 * NB; ++c) buf_copy_x4(wrs, wv[c & 1], so + c * w8, dst + c * (8 * ROW_BYTES));
#pragma unroll
        for (int c = 0; c < 4 * MB; ++c) buf_copy_x4(xrs, xv[c & 1], so + c * x8, dst + (4 * NB + c) * (8 * ROW_BYTES));
    };
#pragma unroll
    for (int t = 0; t < ST; ++t)
        if (t < n_steps) load_step(t);

    f32x16 acc[NB][MB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[i][j] = f32x16{};
    const int sw = (lr >> 1) & 7;
    for (int t = 0; t < n_steps; ++t) {
        // step t has landed once at most the copies of the steps issued after it are in flight
        const int later = min(ST - 1, n_steps - 1 - t);
        if (later == 0) wait_vm<0>();
        else if (later == 1) wait_vm<CP>();
        else if (later == 2) wait_vm<2 * CP>();
        else wait_vm<3 * CP>();
        const char* st = ring + (t % ST) * STAGE + lr * ROW_BYTES;
        v8 af[4][NB], bf[4][MB];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int co = ((2 * s + g) ^ sw) << 4;
#pragma unroll
            for (int i = 0; i < NB; ++i) af[s][i] = *(const v8*)(st + co + i * BLK_BYTES);
#pragma unroll
            for (int j = 0; j < MB; ++j) bf[s][j] = *(const v8*)(st + co + (NB + j) * BLK_BYTES);
        }
        if (t + ST < n_steps) {
            wait_lds();  // the stage has been read before step t + ST is copied over it
            load_step(t + ST);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < MB; ++j) acc[i][j] = Mma16<T>::mma(af[s][i], bf[s][j], acc[i][j]);
    }

    // partial sums in accumulator order, [block][run of 4][lane], over this wave's own (read) ring
    __syncthreads();
    f32x4* const part = (f32x4*)ssm;
    constexpr int WSZ = NB * MB * 4 * 64;  // f32x4 per wave
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
                part[wave * WSZ + ((i * MB + j) * 4 + jj) * 64 + lane] =
                    f32x4{acc[i][j][4 * jj], acc[i][j][4 * jj + 1], acc[i][j][4 * jj + 2], acc[i][j][4 * jj + 3]};
    __syncthreads();
    auto total = [&](int blk, int jj) {
        const f32x4* p = part + (blk * 4 + jj) * 64 + lane;
        return ((p[0] + p[WSZ]) + p[2 * WSZ]) + p[3 * WSZ];
    };
#pragma unroll
    for (int t = 0; t < UNITS; ++t) {
        const int u = wave + 4 * t, blk = u / RUNS, jj = u % RUNS;
        const int nb = n0 + 32 * (blk / MB), m = m0 + 32 * (blk % MB) + lr;
        y4 o;
        int n;
        if (EPI == EPI_SWIGLU) {
            // fused rows 32 b + 8 jj + 4 g + r: gate for jj < 2, its up row at jj + 2
            const f32x4 gs = total(blk, jj), us = total(blk, jj + 2);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                o[r] = from_f<TY>(silu_f<T>(to_f(from_f<T>(gs[r]))) * to_f(from_f<T>(us[r])));
            n = nb / 2 + 8 * jj + 4 * g;
        } else {
            const f32x4 s = total(blk, jj);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = from_f<TY>(RES ? s[r] + to_f(cv[t][r]) : s[r]);
            n = nb + 8 * jj + 4 * g;
        }
        if (m < a.M && nb + 8 * jj + 4 * g < a.N) *(y4*)((TY*)a.y + (long)m * a.ldy + n) = o;
    }
}

}  // namespace gemms
}  // namespace hk

// The tiles and their cost in units of K / 1024 us, fitted to the times of 8 to 8000 rows of the
// projections above: flat while the tiles fit the chip at once, then rising with their number as
// two or three workgroups share a CU, or in rounds (slope 0) where a second workgroup on a CU takes
// as long as a second round (8192 + 32 columns at 169 rows: 258 tiles of 64 x 96 14.7 us, 195 of 128 x
// 64 13.0 us, though 256 of 64 x 96 take 10.1).
// The 128 x 64 tile is the one for the most rows: it reads the fewest operand bytes per product.
namespace {
struct Tile {
    int nb, mb;
    float first, knee, slope;
};
constexpr Tile kTiles[] = {{1, 1, 2.0f, 256, 0.0105f},
                           {1, 2, 3.1f, 256, 0.0105f},
                           {2, 2, 4.0f, 150, 0.0145f},
                           {2, 3, 5.3f, 256, 0.0f},
                           {4, 2, 6.4f, 256, 0.0f}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

long n_tiles(const hk::GemmArgs* a, const Tile& t) {
    const int w = 32 * t.nb;
    return (long)((a->N + w - 1) / w + (a->N2 + w - 1) / w) * ((a->M + 32 * t.mb - 1) / (32 * t.mb));
}

int best_tile(int epi, const hk::GemmArgs* a, float* cost) {
    int best = -1;
    for (int i = epi == hk::EPI_SWIGLU ? 1 : 0; i < kNumTiles; ++i) {  // a 32 x 32 SwiGLU tile has no quarter per wave
        const Tile& k = kTiles[i];
        const long n = n_tiles(a, k);
        const float over = (float)n - k.knee;
        const float c = k.slope == 0.0f ? k.first * (float)((n + 255) / 256) : k.first + k.slope * (over > 0.0f ? over : 0.0f);
        if (best < 0 || c < *cost) {
            best = i;
            *cost = c;
        }
    }
    return best;
}
}  // namespace

template <typename T, int EPI, int I, int ST>
static int launch_one(const hk::GemmArgs* a, hipStream_t stream) {
    constexpr int NB = kTiles[I].nb, MB = kTiles[I].mb;
    constexpr int ring = 4 * ST * (NB + MB) * hk::gemms::BLK_BYTES, sums = 4 * NB * MB * 32 * 32 * 4;
    constexpr int lds = ring > sums ? ring : sums;
    static_assert(lds <= 160 * 1024, "ring and partial sums fit the LDS");
    auto kern = hk::gemms::gemm_ksplit<T, EPI, NB, MB, ST>;
    // set once, under C++'s thread-safe static initialisation (replicas launch from several threads)
    static const bool configured =
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hipLaunchKernelGGL(kern, dim3((unsigned)((n_tiles(a, kTiles[I]) + 7) / 8 * 8)), dim3(hk::gemms::NTHREADS), lds, stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

template <typename T, int EPI>
static int launch_epi(const hk::GemmArgs* a, hipStream_t stream) {
    float cost;
    switch (best_tile(EPI, a, &cost)) {
        case 0:
            if constexpr (EPI != hk::EPI_SWIGLU) return launch_one<T, EPI, 0, 4>(a, stream);
            return HK_ERR_DEVICE;
        case 1: return launch_one<T, EPI, 1, 1>(a, stream);
        case 2: return launch_one<T, EPI, 2, 1>(a, stream);
        case 3: return launch_one<T, EPI, 3, 1>(a, stream);
        default: return launch_one<T, EPI, 4, 1>(a, stream);
    }
}

template <typename T>
static int launch_type(int epi, const hk::GemmArgs* a, hipStream_t stream) {
    switch (epi) {
        case hk::EPI_RESIDUAL: return launch_epi<T, hk::EPI_RESIDUAL>(a, stream);
        case hk::EPI_RESIDUAL_F32: return launch_epi<T, hk::EPI_RESIDUAL_F32>(a, stream);
        case hk::EPI_SWIGLU: return launch_epi<T, hk::EPI_SWIGLU>(a, stream);
        default: return launch_epi<T, hk::EPI_STORE>(a, stream);
    }
}

// Cost of the best tile in units of K / 1024 us (beside about 2 us of launch and first loads).
extern "C" float hk_gemm_split_cost(int epi, const hk::GemmArgs* a) {
    float cost = 0.0f;
    best_tile(epi, a, &cost);
    return cost;
}

// dtype16: 1 = bf16, 2 = fp16. The caller has checked: N and N2 % 8 == 0 (SwiGLU: N % 32), K % 64 == 0,
// 16-byte aligned rows (ld % 8 == 0) and row strides below 2^22 elements (32-bit copy offsets).
extern "C" int hk_launch_gemm_split(int dtype16, int epi, const hk::GemmArgs* a, hipStream_t stream) {
    if (a->M == 0) return HK_OK;
    return dtype16 == hk::DT_BF16 ? launch_type<hk::bf16>(epi, a, stream) : launch_type<hk::f16>(epi, a, stream);
}
