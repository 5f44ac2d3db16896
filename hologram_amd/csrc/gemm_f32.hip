// f32 MatMul (dtype 8; matmul_float, src/cpu/float_kernels.rs:298-399): B
// row-major [k][n] or in the reference's panel-packed layout (src/layout.rs:
// 16-45), [ceil(n/16)][k][16] with zero-padded columns; any m, k, n. All on
// v_mfma_f32_16x16x4_f32 with f32 sums. Three kernels, chosen by launch_matmul_f32:
//   tiles   64 x 64 outputs a workgroup, operands through LDS by DMA
//   split   16 x 16 to 32 x 32 outputs a workgroup, K split over its waves,
//           operands straight into registers: products with few tiles
//   general element-wise loads, for sizes past the others' 32-bit ranges
// None needs scratch, so a product under stream capture needs no call before it.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "holo_kernels.h"

namespace holo {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct F32Args {
    const float *a, *b;
    float *c;
    uint32_t m, n, k, tiles_m, tiles_n;
};

// a row's four columns from col on; vec: 16-byte aligned and col + 4 <= n or col >= n
__device__ __forceinline__ void store4(float *o, f32x4 v, uint32_t col, uint32_t n, bool vec) {
    if (vec) {
        if (col < n) *reinterpret_cast<f32x4 *>(o) = v;
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
            if (col + e < n) o[e] = v[e];
    }
}

// Origin of this workgroup's tile: each XCD (workgroup % 8) takes a run of tiles, walked down columns of 8 tile rows
__device__ __forceinline__ void tile_of(const F32Args &g, uint32_t tm, uint32_t tn, uint32_t *m0, uint32_t *n0) {
    const uint32_t nwg = gridDim.x, wg = blockIdx.x;
    const uint32_t tile = nwg % 8 == 0 ? (wg % 8) * (nwg / 8) + wg / 8 : wg;
    const uint32_t per = 8 * g.tiles_n, first = tile / per * 8, in = tile % per;
    const uint32_t gs = g.tiles_m - first < 8 ? g.tiles_m - first : 8;
    *m0 = (first + in % gs) * tm;
    *n0 = in / gs * tn;
}

// ------------------------------------------------------------ split K ----
// Few tiles: what bounds them is how many loads are in flight, so each of the W
// waves owns the whole 16 MT x 16 NP tile over its own K units of 16 U rows
// (unit w, w + W, ..), fragments loaded from memory into registers one unit
// ahead, no barrier before the sums meet in LDS. Lane (lr, lg) of a 16-row step
// takes k = 4 lg .. 4 lg + 3 of A row lr in one 16-byte load and, of B, column
// lr at the same four rows; MFMA s pairs them at k = 4 lg + s. (With B's rows
// 4 s + lg instead, one 256-byte run a load, and A transposed across lanes by
// permlane swaps: 5% slower; A's 16 rows a load are what it waits for.)
// Rows past M and K read zero through the buffer ranges, columns past N are not
// stored; a 16-byte chunk of A that straddles K goes on with the next row, so
// the last unit clears those elements (zero times that row's infinity would
// be NaN).
// 1 x 2048 x 4096 packed 58 -> 8.7 us, 8 x 4096 x 4096 packed 115 -> 14.6 (64 MiB
// of weights: 11 at the copy rate), 200 x 2048 x 1024 59 -> 19.5, 200 x 2047 x
// 1021 81 -> 20.4, on the 64-tile register-staged kernel before.
template <int MT, int NP, int W, int U, bool kPacked>
__global__ __launch_bounds__(64 * W) void gemm_f32_split_kernel(const F32Args g) {
    constexpr int TM = 16 * MT, TN = 16 * NP, kRow = TN + 4;   // LDS row: 4 rows apart, 16 banks apart
    constexpr uint32_t kUnit = 16 * U;
    static_assert(W * TM * kRow * 4 <= 72 * 1024, "two workgroups a CU by LDS");
    __shared__ __attribute__((aligned(16))) float red[W][TM][kRow];
    const uint32_t M = g.m, N = g.n, K = g.k;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const uint32_t w = __builtin_amdgcn_readfirstlane(uint32_t(tid) >> 6);
    uint32_t m0, n0;
    tile_of(g, TM, TN, &m0, &n0);
    const uint32_t mrows = M - m0 < uint32_t(TM) ? M - m0 : uint32_t(TM);

    const float *__restrict__ A = g.a + uint64_t(m0) * K;
    const uint32_t avo = (lr * K + 4 * lg) * 4u;
    const uint32_t bvo = kPacked ? (4 * lg * 16 + lr) * 4u : (4 * lg * N + lr) * 4u;
    const uint32_t brow = kPacked ? 64u : N * 4u;
    f32x4 a[2][U][MT];
    float b[2][U][NP][4];
    auto load = [&](uint32_t unit, int f) {
        const uint32_t k0 = unit * kUnit;
        const uint32_t left = k0 < K ? K - k0 : 0u;            // k rows from here on
        const uint32_t kb = left ? k0 : 0u;
        const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A + kb), 0,
                                                          left ? int(((mrows - 1) * K + left) * 4u) : 0, 0x00020000);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i)
                a[f][u][i] = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, avo, 64u * K * i + 64u * u, 0));
        if constexpr (kPacked) {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const uint32_t np = (n0 >> 4) + p;
                const bool some = left && np * 16 < N;
                const auto rb = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<float *>(g.b + (uint64_t(some ? np : 0) * K + kb) * 16), 0,
                    some ? int(left * 64u) : 0, 0x00020000);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        b[f][u][p][s] = __uint_as_float(
                            __builtin_amdgcn_raw_buffer_load_b32(rb, bvo, 1024u * u + 64u * s, 0));
            }
        } else {
            const uint64_t rest = (uint64_t(left) * N - (left ? n0 : 0)) * 4u;
            const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.b + uint64_t(kb) * N + n0), 0,
                                                              rest > 0x7fffffffu ? 0x7fffffff : int(rest), 0x00020000);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        b[f][u][p][s] = __uint_as_float(
                            __builtin_amdgcn_raw_buffer_load_b32(rb, bvo + 64u * p, brow * (16 * u + s), 0));
        }
    };
    f32x4 acc[MT][NP];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int p = 0; p < NP; ++p) acc[i][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](uint32_t unit, int f) {
        if ((unit + 1) * kUnit > K) {      // a chunk of A past K goes on with the next row
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        if (unit * kUnit + 16 * u + 4 * lg + s >= K) a[f][u][i][s] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        acc[i][p] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[f][u][i][s], b[f][u][p][s], acc[i][p],
                                                                         0, 0, 0);
    };
    const uint32_t units = (K + kUnit - 1) / kUnit;
    load(w, 0);
    for (uint32_t t = w; t < units; t += 2 * W) {
        load(t + W, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(t, 0);
        __builtin_amdgcn_sched_barrier(0);
        load(t + 2 * W, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(t + W, 1);
        __builtin_amdgcn_sched_barrier(0);
    }

    // the waves' sums, added in wave order
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[w][16 * i + 4 * lg + e][16 * p + lr] = acc[i][p][e];
    __syncthreads();
    const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(g.c) & 15) == 0;
#pragma unroll
    for (int q = tid; q < TM * TN / 4; q += 64 * W) {
        const uint32_t r = q / (TN / 4), c = q % (TN / 4) * 4;
        f32x4 s = *reinterpret_cast<const f32x4 *>(&red[0][r][c]);
#pragma unroll
        for (int v = 1; v < W; ++v) s += *reinterpret_cast<const f32x4 *>(&red[v][r][c]);
        if (r >= mrows) continue;
        store4(g.c + uint64_t(m0 + r) * N + n0 + c, s, n0 + c, N, vec);
    }
}

// ------------------------------------------------- 64 x 64 tiles, LDS DMA ----
// Eight waves a 64 x 64 tile, each 16 x 64 over one half of every 32-deep K slab
// (two waves a SIMD: one's LDS reads under the other's MFMAs), A and B slabs by
// DMA (buffer_load ... lds) into a ring of four stages, a slab's fragments read
// during the slab before. Bound by the matrix cores: a slab is 1024 cycles of
// MFMA a SIMD against 16 KiB of loads a CU. Lane (lr, lg) reads A row lr at k =
// 4 lg .. + 3 and, for MFMA step s, B row 4 lg + s at columns 4 lr .. + 3: one
// 16-byte read each, whose four columns feed four MFMAs (MFMA j computes columns
// 4 lr + j, so a lane's four results of a row are one 16-byte store).
// LDS: an A row's eight 16-byte chunks at chunk ^ (row / 2 % 8); a packed B
// panel's rows at row ^ (panel % 4); a row-major B row as it is: the 16 lanes of
// a quarter wave hit distinct banks.
// Rows past M and K read zero through the buffer ranges (a chunk of A past K is
// sent there), columns past N are not stored. The loads need dword alignment
// only, so any k and n go; an A chunk that straddles K is cleared past it as its
// fragments are read.
// 500 x 1536 x 2000 packed 45.4 -> 27.2 us (20.5 at the MFMA rate), 1000^3 43.7
// -> 20.2, 2048 x 512 x 2048 44 -> 37, 500 x 2000 x 2001 packed 111 -> 37.
// Larger tiles (128 x 64, 64 x 128, 128 x 128): equal where they fill the chip
// (2048 x 512 x 2048 36.7-38.2 us), up to 3.4 times slower where they do not.
constexpr int kStages = 4, kSlab = 32;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

template <int n>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void slab_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <bool kPacked>
__device__ __forceinline__ void gemm_f32_dma(const F32Args &g) {
    constexpr int kLoads = 2;                            // 1 KiB loads a wave a slab: one of A, one of B
    constexpr uint32_t kOffB = 8192, kStage = 16384;     // a stage: A [64][32 k], then B
    // one array per stage: the compiler then knows a DMA into one stage does
    // not feed reads of another, and waits only where a read needs the data
    __shared__ __attribute__((aligned(1024))) uint8_t lds0[kStage], lds1[kStage], lds2[kStage], lds3[kStage];
    auto stage = [&](auto st) -> lds_u8 * {
        constexpr int kS = decltype(st)::value % kStages;
        return kS == 0 ? (lds_u8 *)lds0 : kS == 1 ? (lds_u8 *)lds1 : kS == 2 ? (lds_u8 *)lds2 : (lds_u8 *)lds3;
    };
    const uint32_t M = g.m, N = g.n, K = g.k;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const uint32_t w = __builtin_amdgcn_readfirstlane(uint32_t(tid) >> 6);
    const uint32_t kg = w >> 2, wm = (w & 3) * 16;       // K half, rows
    uint32_t m0, n0;
    tile_of(g, 64, 64, &m0, &n0);
    const uint32_t mrows = M - m0 < 64u ? M - m0 : 64u;

    // DMA addresses of the next slab, walked: A rows 8 w + lane / 8; of B 1 KiB
    // runs: half a panel's 16 rows, or four rows
    const uint32_t arow = 8 * w + lane / 8;
    uint32_t acol = 4u * ((lane & 7) ^ ((arow >> 1) & 7));
    uint32_t avo = (arow * K + acol) * 4u;
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.a + uint64_t(m0) * K), 0,
                                                      int(mrows * K * 4u), 0x00020000);
    const uint32_t panel = (n0 >> 4) + w / 2;
    const bool some = panel * 16 < N;
    const auto rpanel = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(kPacked ? g.b + uint64_t(some ? panel : 0) * K * 16 : g.b), 0,
        kPacked && some ? int(K * 64u) : 0, 0x00020000);
    uint32_t bvo = kPacked ? (((w % 2 * 16 + lane / 4) ^ (w / 2)) * 16 + 4 * (lane & 3)) * 4u
                           : ((4 * w + lane / 16) * N + 4 * (lane & 15)) * 4u;
    const float *bp = g.b + n0;
    int64_t bleft = (int64_t(K) * N - n0) * 4;           // bytes of B from bp on
    auto dma = [&](auto st) {
        lds_u8 *sa = stage(st) + w * 1024u, *sb = stage(st) + kOffB + w * 1024u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, sa, 16, acol < K ? avo : 0x80000000u, 0, 0, 0);
        avo += 4u * kSlab;
        acol += kSlab;
        if constexpr (kPacked) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rpanel, sb, 16, bvo, 0, 0, 0);
            bvo += kSlab * 64u;
        } else {
            const auto rb = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(bp), 0, bleft > 0x7fffffff ? 0x7fffffff : bleft < 0 ? 0 : int(bleft), 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, sb, 16, bvo, 0, 0, 0);
            bp += uint64_t(kSlab) * N;
            bleft -= int64_t(kSlab) * N * 4;
        }
    };

    const uint32_t a_frag = (wm + lr) * 128u + (((4 * kg + lg) ^ ((lr >> 1) & 7)) * 16u);
    uint32_t b_frag[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t R = 16 * kg + 4 * lg + s;
        b_frag[s] = kOffB + (kPacked ? (lr / 4) * 2048u + (R ^ (lr / 4)) * 64u + (lr & 3) * 16u
                                     : R * 256u + lr * 16u);
    }
    f32x4 a[2], b[2][4], acc[4];
    auto fload = [&](auto st, int f, uint32_t s0, auto tail) {   // of slab s0; tail: it may end past K
        const lds_u8 *base = stage(st);
        a[f] = *reinterpret_cast<const lds_f32x4 *>(base + a_frag);
#pragma unroll
        for (int s = 0; s < 4; ++s) b[f][s] = *reinterpret_cast<const lds_f32x4 *>(base + b_frag[s]);
        if (decltype(tail)::value && (s0 + 1) * kSlab > K) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s0 * kSlab + 16 * kg + 4 * lg + s >= K) a[f][s] = 0.f;
        }
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mfmas = [&](int f) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[f][s], b[f][s][j], acc[j], 0, 0, 0);
    };
    // Slab n in stage n % 4, its fragments already read. next: slab n + 1 exists
    // (its DMA is awaited: wait loads issued after it may stay in flight); more:
    // slab n + 3 exists, and its DMA refills the stage of slab n - 1, whose
    // fragments every wave's MFMAs have taken before this barrier.
    auto slab = [&](uint32_t n, auto st, auto wait, auto next, auto more, auto tail) {
        constexpr int kS = decltype(st)::value, kF = kS & 1;
        if constexpr (decltype(next)::value) {
            wait_vm<decltype(wait)::value>();
            slab_barrier();
            if constexpr (decltype(more)::value) dma(std::integral_constant<int, kS + 3>{});
            fload(std::integral_constant<int, kS + 1>{}, kF ^ 1, n + 1, tail);
        }
        mfmas(kF);
        __builtin_amdgcn_sched_barrier(0);
    };
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;
    using s0 = std::integral_constant<int, 0>;
    using s1 = std::integral_constant<int, 1>;
    using s2 = std::integral_constant<int, 2>;
    using s3 = std::integral_constant<int, 3>;
    using w1 = std::integral_constant<int, kLoads>;
    const uint32_t nk = (K + 4 * kSlab - 1) / (4 * kSlab) * 4;   // those past K multiply zeros
    dma(s0{});
    dma(s1{});
    dma(s2{});
    wait_vm<2 * kLoads>();
    slab_barrier();
    fload(s0{}, 0, 0, yes{});
    for (uint32_t s = 0; s + 4 < nk; s += 4) {
        slab(s, s0{}, w1{}, yes{}, yes{}, no{});
        slab(s + 1, s1{}, w1{}, yes{}, yes{}, no{});
        slab(s + 2, s2{}, w1{}, yes{}, yes{}, no{});
        slab(s + 3, s3{}, w1{}, yes{}, yes{}, yes{});
    }
    slab(nk - 4, s0{}, w1{}, yes{}, yes{}, yes{});
    slab(nk - 3, s1{}, w1{}, yes{}, no{}, yes{});
    slab(nk - 2, s2{}, s0{}, yes{}, no{}, yes{});
    slab(nk - 1, s3{}, s0{}, no{}, no{}, no{});

    // the K halves: of a lane's four rows each wave hands two to its partner
    // and adds and stores the other two
    slab_barrier();
    auto row4 = [&](int r) { return f32x4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]}; };
    lds_u8 *mine = stage(s0{}) + w * 2048u + lane * 16u, *theirs = stage(s0{}) + (w ^ 4) * 2048u + lane * 16u;
#pragma unroll
    for (int r = 0; r < 2; ++r) *reinterpret_cast<lds_f32x4 *>(mine + r * 1024u) = kg ? row4(r) : row4(r + 2);
    __syncthreads();
    const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(g.c) & 15) == 0;
    const uint32_t col = n0 + 4 * lr;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const f32x4 y = *reinterpret_cast<const lds_f32x4 *>(theirs + r * 1024u);
        const uint32_t row = wm + 4 * lg + (kg ? r + 2 : r);
        if (row >= mrows) continue;
        store4(g.c + uint64_t(m0 + row) * N + col, (kg ? row4(r + 2) : row4(r)) + y, col, N, vec);
    }
}

template <bool kPacked>
__global__ __launch_bounds__(512) void gemm_f32_dma_kernel(const F32Args g) {
    gemm_f32_dma<kPacked>(g);
}

// ---------------------------------------------------------------- general ----
constexpr int BK32 = 32, APAD32 = 4, BPAD32 = 4;

// Element (k, n) of B; a packed panel's columns are 16 to a k-row.
template <bool kPacked>
__device__ __forceinline__ uint64_t b_index(uint32_t gk, uint32_t gn, uint32_t N, uint32_t K) {
    return kPacked ? (uint64_t(gn >> 4) * K + gk) * 16 + (gn & 15) : uint64_t(gk) * N + gn;
}

// 64-bit element addresses, register-staged 128 x 128 tiles: k or n of 2^22 and more.
template <bool kPacked>
__global__ __launch_bounds__(256) void gemm_f32_general_kernel(const float *__restrict__ A,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C, uint32_t M,
                                                           uint32_t N, uint32_t K) {
    constexpr int WT = 4, BM = 32 * WT, BN = BM, kThreads = 256, kChunks = BM / 32;   // float4 per thread per operand
    __shared__ float As[2][BM][BK32 + APAD32];
    __shared__ float Bs[2][BK32][BN + BPAD32];

    const uint32_t m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int t = threadIdx.x;
    const int wave = t >> 6, lane = t & 63;
    const int wm = (wave >> 1) * 16 * WT, wn = (wave & 1) * 16 * WT;
    const int lr = lane & 15, lg = lane >> 4;

    f32x4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    float4 ra[kChunks], rb[kChunks];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {  // A: BM x 32 floats
            const int c = t + i * kThreads;
            const int r = c / (BK32 / 4), kc = (c % (BK32 / 4)) * 4;
            const uint32_t gm = m0 + r, gk = k0 + kc;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (gm < M && gk + e < K) ? A[uint64_t(gm) * K + gk + e] : 0.0f;
            ra[i] = make_float4(v[0], v[1], v[2], v[3]);
        }
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {  // B: 32 x BN floats
            const int c = t + i * kThreads;
            const int r = c / (BN / 4), nc = (c % (BN / 4)) * 4;
            const uint32_t gk = k0 + r, gn = n0 + nc;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = (gk < K && gn + e < N) ? B[b_index<kPacked>(gk, gn + e, N, K)] : 0.0f;
            rb[i] = make_float4(v[0], v[1], v[2], v[3]);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {
            const int c = t + i * kThreads;
            const int r = c / (BK32 / 4), kc = (c % (BK32 / 4)) * 4;
            *reinterpret_cast<float4 *>(&As[buf][r][kc]) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {
            const int c = t + i * kThreads;
            const int r = c / (BN / 4), nc = (c % (BN / 4)) * 4;
            *reinterpret_cast<float4 *>(&Bs[buf][r][nc]) = rb[i];
        }
    };

    const uint32_t nk = (K + BK32 - 1) / BK32;
    load(0);
    store(0);
    __syncthreads();
    for (uint32_t s = 0; s < nk; ++s) {
        const int cur = s & 1;
        if (s + 1 < nk) load((s + 1) * BK32);
#pragma unroll
        for (int kk = 0; kk < BK32; kk += 4) {
            float af[WT], bfv[WT];
#pragma unroll
            for (int i = 0; i < WT; ++i) af[i] = As[cur][wm + i * 16 + lr][kk + lg];
#pragma unroll
            for (int j = 0; j < WT; ++j) bfv[j] = Bs[cur][kk + lg][wn + j * 16 + lr];
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bfv[j], acc[i][j], 0, 0, 0);
        }
        if (s + 1 < nk) store(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t gm = m0 + wm + i * 16 + lg * 4 + r, gn = n0 + wn + j * 16 + lr;
                if (gm < M && gn < N) C[uint64_t(gm) * N + gn] = acc[i][j][r];
            }
}

}  // namespace

// Which kernel: the least of a model of each one's time, fitted to sweeps (16
// shapes, 1 to 2500 rows, on a 256-CU card): ns per K row and round of 256 workgroups,
// plus 3.4 us, K rounded to what the waves take together. Measured against it:
// 500 x 1536 x 2000 tiles 27.2 us (model 27), split 2 x 2 48.6 (48); 200 x 2048 x
// 1024 34.5 (35) and 19.5 (19.6); 50 x 4096 x 2048 split 2 x 1 22.7 (22.7), 1 x 1
// 25.7 (27), tiles 65; 8 x 4096 x 4096 split 1 x 1 15.4 (15.3), 2 x 1 18.7.
struct F32Form {
    uint32_t tm, tn, kstep, threads;
    float ns;
};
constexpr F32Form kF32Forms[] = {
    {64, 64, 32, 512, 15.3f},      // tiles
    {32, 32, 256, 512, 7.9f},      // split 2 x 2
    {32, 16, 512, 1024, 4.7f},     // split 2 x 1
    {16, 16, 512, 512, 2.9f},      // split 1 x 1
};

hipError_t launch_matmul_f32(const float *a, const float *b, float *c, uint32_t m, uint32_t k, uint32_t n,
                             bool packed, hipStream_t stream) {
    F32Args g{a, b, c, m, n, k, 0, 0};
    int best = -1;
    double least = 0;
    // (k and n within 32-bit offsets of a tile's rows, the grid within 2^32 threads)
    for (int i = 0; i < 4 && k < (1u << 22) && n < (1u << 22); ++i) {
        const F32Form &f = kF32Forms[i];
        const uint64_t tiles = uint64_t((m + f.tm - 1) / f.tm) * ((n + f.tn - 1) / f.tn);
        if (tiles * f.threads >= (1ull << 32)) continue;
        const double t = double(f.ns) * double((k + f.kstep - 1) / f.kstep * f.kstep) * double((tiles + 255) / 256);
        if (best >= 0 && t >= least) continue;
        least = t;
        best = i;
        g.tiles_m = (m + f.tm - 1) / f.tm;
        g.tiles_n = (n + f.tn - 1) / f.tn;
    }
    const dim3 grid(g.tiles_m * g.tiles_n);
#define HOLO_F32(KERNEL, THREADS) hipLaunchKernelGGL(KERNEL, grid, dim3(THREADS), 0, stream, g)
#define HOLO_SPLIT(MT, NP, W, U)                                                  \
    do {                                                                          \
        if (packed) HOLO_F32((gemm_f32_split_kernel<MT, NP, W, U, true>), 64 * W); \
        else HOLO_F32((gemm_f32_split_kernel<MT, NP, W, U, false>), 64 * W);      \
    } while (0)
    if (best == 0 && packed) HOLO_F32(gemm_f32_dma_kernel<true>, 512);
    else if (best == 0) HOLO_F32(gemm_f32_dma_kernel<false>, 512);
    else if (best == 1) HOLO_SPLIT(2, 2, 8, 2);
    else if (best == 2) HOLO_SPLIT(2, 1, 16, 2);
    else if (best == 3) HOLO_SPLIT(1, 1, 8, 4);
    else {
        const dim3 wide((n + 127) / 128, (m + 127) / 128);
        if (packed)
            hipLaunchKernelGGL(gemm_f32_general_kernel<true>, wide, dim3(256), 0, stream, a, b, c, m, n, k);
        else
            hipLaunchKernelGGL(gemm_f32_general_kernel<false>, wide, dim3(256), 0, stream, a, b, c, m, n, k);
    }
#undef HOLO_SPLIT
#undef HOLO_F32
    return hipGetLastError();
}

}  // namespace holo
