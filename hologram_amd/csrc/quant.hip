// quant.hip — the quantized-weight ops: Dequantize (src/cpu/kernels.rs:185-296),
// DequantActivation (:311-388) and MatMulDequant's output-major W8A8 GEMM
// (matmul_i8_pc_omajor / matmul_i4_pc_omajor / matmul_e8cb_omajor,
// src/cpu/simd.rs:5295-5480, 6172-6230, 6867-6950).
//
// The W8A8 GEMM is exact integer arithmetic, so any tiling gives the
// reference's bits: each activation row is quantized once (quantize_row_i8,
// the same operations as the KV quantizer), the dot products accumulate in
// int32 on v_mfma_i32_16x16x64_i8 (four wavefronts split K and add their
// int32 tiles), and the writeback is the reference's expression,
// (acc as f32) * (scale_a * scales[j]).
//
// Layout of the GEMM: a workgroup owns 16 output columns and MT 16-row tiles
// of A. The output-major weight keeps each column's k-vector contiguous, so a
// lane's 16-byte B fragment (k .. k+15 of its column) is one load; lane
// (r, g) of a wavefront holds column r and k-chunk g of each 64-deep step, and
// A row r's chunk g from the quantized rows, so both operands agree on which k
// each byte is. i4 columns unpack 8 bytes to 16 sign-extended levels; e8cb
// columns read two codebook blocks (the 2 KiB codebook staged in LDS).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "holo_device.h"
#include "holo_kernels.h"

namespace holo {
namespace {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// Rust's `f32 as i32`, then clamp(-127, 127) (NaN -> 0), as the KV quantizer.
__device__ __forceinline__ int8_t to_q8(float r) {
    if (r != r) return 0;
    r = r < -127.0f ? -127.0f : (r > 127.0f ? 127.0f : r);
    return static_cast<int8_t>(static_cast<int32_t>(r));
}

// ---------------------------------------------------------- per-token quant --
// One workgroup per row of A (f32): amax with `>` (NaN never wins), then
// q = clamp(round-half-away(x * (127 / amax))), scale amax / 127 (0 for an
// all-zero row, whose q is 0). Row stride kpad >= k; the padding is zeroed so
// the GEMM's whole 64-deep steps read zeros there.
__global__ __launch_bounds__(256) void quant_rows_kernel(const float *__restrict__ a, uint32_t k,
                                                         uint32_t kpad, int8_t *__restrict__ q,
                                                         float *__restrict__ sa) {
    __shared__ float red[4];
    const uint64_t row = blockIdx.x;
    const float *x = a + row * k;
    float amax = 0.0f;
    for (uint32_t c = threadIdx.x; c < k; c += 256) {
        const float v = x[c];
        const float av = v < 0.0f ? -v : v;
        if (av > amax) amax = av;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float o = __shfl_xor(amax, off, 64);
        if (o > amax) amax = o;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = red[0];
    for (int w = 1; w < 4; ++w)
        if (red[w] > amax) amax = red[w];
    int8_t *dst = q + row * kpad;
    if (amax == 0.0f) {
        for (uint32_t c = threadIdx.x; c < kpad; c += 256) dst[c] = 0;
        if (threadIdx.x == 0) sa[row] = 0.0f;
        return;
    }
    const float inv = 127.0f / amax;
    for (uint32_t c = threadIdx.x; c < kpad; c += 256) {
        if (c < k) {
            const float t = x[c] * inv;
            dst[c] = to_q8(t >= 0.0f ? truncf(t + 0.5f) : truncf(t - 0.5f));
        } else {
            dst[c] = 0;
        }
    }
    if (threadIdx.x == 0) sa[row] = amax / 127.0f;
}

// W8A8 needs symmetric weights: a nonzero zero point raises bit 4 of *err
// (reported at the next synchronize as UnsupportedOp). Byte-wise, so the zero
// points need no alignment: an i32 is zero exactly when its four bytes are.
struct ZeroPoints {
    const uint8_t *p;
    uint64_t bytes;
    int *err;
};
constexpr uint32_t kZpBlock = 256 * 16;   // bytes a workgroup checks a round

__device__ __forceinline__ void check_zero_points(const ZeroPoints &z, uint32_t blk, uint32_t nblk) {
    bool bad = false;
    const bool al = (reinterpret_cast<uintptr_t>(z.p) & 15) == 0;
    for (uint64_t b = uint64_t(blk) * kZpBlock; b < z.bytes; b += uint64_t(nblk) * kZpBlock) {
        const uint64_t i = b + threadIdx.x * 16u;
        if (al && i + 16 <= z.bytes) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(z.p + i);
            bad = bad || (v[0] | v[1] | v[2] | v[3]) != 0;
        } else {
            for (uint64_t e = i; e < i + 16 && e < z.bytes; ++e) bad = bad || z.p[e] != 0;
        }
    }
    if (bad) atomicOr(z.err, 4);
}

// The same quantizer over rows of k % 4 == 0 floats, k <= 1024 V, 16-byte
// aligned: a row is read once, V vectors a thread held through the maximum,
// and written four levels a store. The workgroups after the rows check the
// zero points (a launch of their own took as long as an empty kernel). 512 rows
// of 4096: 10 us, and 4.6 us for the check, before; 4.9 us together.
template <int V>
__global__ __launch_bounds__(256) void quant_rows_vec_kernel(const float *__restrict__ a, uint32_t rows,
                                                             uint32_t k, uint32_t kpad,
                                                             int8_t *__restrict__ q,
                                                             float *__restrict__ sa, const ZeroPoints z) {
    __shared__ float red[4];
    if (blockIdx.x >= rows) {
        check_zero_points(z, blockIdx.x - rows, gridDim.x - rows);
        return;
    }
    const uint64_t row = blockIdx.x;
    const float4 *x = reinterpret_cast<const float4 *>(a + row * k);
    float4 v[V];
    float amax = 0.0f;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const uint32_t c = threadIdx.x + 256u * u;
        v[u] = 4 * c < k ? x[c] : float4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float av = e[i] < 0.0f ? -e[i] : e[i];
            if (av > amax) amax = av;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float o = __shfl_xor(amax, off, 64);
        if (o > amax) amax = o;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = red[0];
    for (int w = 1; w < 4; ++w)
        if (red[w] > amax) amax = red[w];
    uint32_t *dst = reinterpret_cast<uint32_t *>(q + row * kpad);
    const float inv = 127.0f / amax;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const uint32_t c = threadIdx.x + 256u * u;
        if (4 * c >= kpad) continue;
        const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        uint32_t w = 0;
        if (amax != 0.0f && 4 * c < k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float t = e[i] * inv;
                w |= uint32_t(uint8_t(to_q8(t >= 0.0f ? truncf(t + 0.5f) : truncf(t - 0.5f)))) << (8 * i);
            }
        dst[c] = w;
    }
    if (threadIdx.x == 0) sa[row] = amax == 0.0f ? 0.0f : amax / 127.0f;
}

// ------------------------------------------------------------- W8A8 GEMM ----
struct QGemm {
    const int8_t *q;          // [m][kpad] quantized activation rows
    const float *sa;          // [m] their scales
    const uint8_t *bq;        // output-major weight (tier layout)
    const int8_t *codebook;   // e8cb: 256 x 8
    const float *scales;      // [n] per-column scales
    const float *residual;    // [m][n] or null
    float *out;               // [m][n]
    uint32_t m, k, n, kpad;
    uint32_t act;             // fused_activation id (0: none)
};

// 16 consecutive k of column j starting at k0 (a multiple of 16) as 16 int8
// levels, zero past k or past the last column.
template <int TIER>
__device__ __forceinline__ i32x4 b_fragment(const QGemm &g, const int8_t *cb, uint32_t j,
                                            uint32_t k0) {
    i32x4 r = {0, 0, 0, 0};
    if (j >= g.n || k0 >= g.k) return r;
    const uint32_t k = g.k;
    if constexpr (TIER == 2) {   // i8: bytes j*k + k0 ..
        const uint8_t *p = g.bq + uint64_t(j) * k + k0;
        if (k0 + 16 <= k && ((reinterpret_cast<uintptr_t>(p) & 15) == 0)) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(p);
            r = i32x4{int32_t(v[0]), int32_t(v[1]), int32_t(v[2]), int32_t(v[3])};
        } else {
            uint32_t w[4] = {0, 0, 0, 0};
            for (int e = 0; e < 16; ++e)
                if (k0 + e < k) w[e >> 2] |= uint32_t(p[e]) << (8 * (e & 3));
            r = i32x4{int32_t(w[0]), int32_t(w[1]), int32_t(w[2]), int32_t(w[3])};
        }
    } else if constexpr (TIER == 10) {   // i4: unit u = j*k + kk, low nibble first
        const uint64_t u0 = uint64_t(j) * k + k0;   // even (k even, k0 % 16 == 0)
        const uint8_t *p = g.bq + (u0 >> 1);
        uint32_t w[4] = {0, 0, 0, 0};
        for (int e = 0; e < 8; ++e) {
            if (k0 + 2 * e >= k) break;
            const uint32_t byte = p[e];
            const int32_t lo = int32_t(byte & 0x0Fu), hi = int32_t(byte >> 4);
            const uint32_t l8 = uint32_t(uint8_t(int8_t(lo >= 8 ? lo - 16 : lo)));
            const uint32_t h8 = uint32_t(uint8_t(int8_t(hi >= 8 ? hi - 16 : hi)));
            w[(2 * e) >> 2] |= l8 << (8 * ((2 * e) & 3));
            w[(2 * e + 1) >> 2] |= h8 << (8 * ((2 * e + 1) & 3));
        }
        r = i32x4{int32_t(w[0]), int32_t(w[1]), int32_t(w[2]), int32_t(w[3])};
    } else {   // e8cb: two 8-row groups, codebook blocks of 8 i8
        const uint8_t *p = g.bq + uint64_t(j) * (k / 8) + k0 / 8;
        uint32_t w[4] = {0, 0, 0, 0};
        for (int h = 0; h < 2; ++h) {
            if (k0 + 8 * h >= k) break;
            const int8_t *blk = cb + uint32_t(p[h]) * 8;
            for (int e = 0; e < 8; ++e) w[2 * h + (e >> 2)] |= uint32_t(uint8_t(blk[e])) << (8 * (e & 3));
        }
        r = i32x4{int32_t(w[0]), int32_t(w[1]), int32_t(w[2]), int32_t(w[3])};
    }
    return r;
}

template <int TIER, int MT>
__global__ __launch_bounds__(256) void gemm_q_omajor_kernel(QGemm g) {
    __shared__ int8_t cb[TIER == 11 ? 256 * 8 : 16];
    __shared__ i32x4 red[3][MT][64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r = lane & 15, gq = lane >> 4;
    if constexpr (TIER == 11) {
        for (int i = tid; i < 256 * 8; i += 256) cb[i] = g.codebook[i];
        __syncthreads();
    }
    const uint32_t n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
    const uint32_t steps = g.kpad / 64;
    const uint32_t per = (steps + 3) / 4;
    const uint32_t s0 = per * wave, s1 = s0 + per < steps ? s0 + per : steps;
    i32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = i32x4{0, 0, 0, 0};
    for (uint32_t s = s0; s < s1; ++s) {
        const uint32_t k0 = s * 64 + 16 * gq;
        const i32x4 bf = b_fragment<TIER>(g, cb, n0 + r, k0);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint32_t row = m0 + 16 * t + r;
            i32x4 af = {0, 0, 0, 0};
            if (row < g.m) {
                const u32x4 v = *reinterpret_cast<const u32x4 *>(g.q + uint64_t(row) * g.kpad + k0);
                af = i32x4{int32_t(v[0]), int32_t(v[1]), int32_t(v[2]), int32_t(v[3])};
            }
            acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, bf, acc[t], 0, 0, 0);
        }
    }
    // the four wavefronts' int32 tiles (exact, so any order)
    if (wave > 0)
#pragma unroll
        for (int t = 0; t < MT; ++t) red[wave - 1][t][lane] = acc[t];
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        i32x4 v = acc[t];
        for (int w = 0; w < 3; ++w) v += red[w][t][lane];
        // C layout of the 16x16 tile: lane holds rows 4*(lane/16) + e, column lane % 16
        const uint32_t j = n0 + r;
        if (j >= g.n) continue;
        const float sj = g.scales[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t i = m0 + 16 * t + 4 * gq + e;
            if (i >= g.m) continue;
            const float si = g.sa[i];
            float o = si == 0.0f ? 0.0f : float(v[e]) * (si * sj);
            if (g.residual) o = o + g.residual[uint64_t(i) * g.n + j];
            if (g.act) o = act_f32_call(g.act, o);
            g.out[uint64_t(i) * g.n + j] = o;
        }
    }
}

// -------------------------------------------------- W8A8, many rows (tiles) --
// BM x BN workgroup tiles, four wavefronts of BM/2 x BN/2 on
// v_mfma_i32_32x32x32_i8, 128-deep K slabs in S LDS stages filled by LDS DMA
// S - 1 slabs ahead. Both operands are k-contiguous, so both fragments are
// plain LDS reads: A [BM][128 bytes] (the quantized rows, zero past k), B
// [BN][128 / 64 / 16 bytes] as the weight is stored: i4 bytes are spread to
// signed levels and e8cb indices looked up (codebook in LDS) as a fragment is
// read, once for the BM/64 products that use it. Chunks of a row sit at chunk ^
// f(row) against bank conflicts. Addresses are walked, one step a slab. Rows
// past m, columns past n and slabs past K read zero through the buffer ranges;
// a slab that reaches past k meets A's zeros. Integer sums are exact, so the
// tile and the order are free.
// Bound by the operand bytes a CU takes in and reads back for its tile. 512 x
// 4096 x 4096, call with the row quantizer: i8 20 us (88 before, on 16-column
// workgroups that re-read A 256 times), i4 31 (185), e8cb 24 (103). Deeper
// rings (96-150 KiB) changed nothing.
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

// vmcnt <= n; reads: lgkmcnt 0 too, else untouched
template <int n, bool reads = false>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (reads ? 0 : 15 << 8));
}

// 8 bytes of i4 (low nibble first) as 16 signed levels.
__device__ __forceinline__ i32x4 spread_i4(uint32_t w0, uint32_t w1) {
    i32x4 r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t b = (h ? w1 : w0) ^ 0x88888888u;   // (u ^ 8) - 8 is the level
        const uint32_t lo = b & 0x0F0F0F0Fu, hi = (b >> 4) & 0x0F0F0F0Fu;
        const uint32_t x = __builtin_amdgcn_perm(hi, lo, 0x05010400u), y = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
        r[2 * h] = int(((x | 0x80808080u) - 0x08080808u) ^ 0x80808080u);
        r[2 * h + 1] = int(((y | 0x80808080u) - 0x08080808u) ^ 0x80808080u);
    }
    return r;
}

template <int BM, int BN, int TIER, int S>
__device__ __forceinline__ void gemm_q_tiled(const QGemm &g) {
    constexpr int MI = BM / 64, NJ = BN / 64;
    constexpr uint32_t PB = TIER == 2 ? 128 : TIER == 10 ? 64 : 16;   // bytes of a column's slab
    constexpr uint32_t kOffB = BM * 128, kStage = kOffB + BN * PB;
    constexpr int LA = BM / 32, LB = TIER == 11 ? 1 : int(BN * PB / 4096);   // 1 KiB loads a wave
    static_assert(kStage >= uint32_t(MI * NJ * 4096), "a stage holds a wave's results");
    static_assert(S == 4 || S == 8, "the rings below");
    __shared__ __attribute__((aligned(1024))) uint8_t l0[kStage], l1[kStage], l2[kStage], l3[kStage],
        l4[S > 4 ? kStage : 16], l5[S > 4 ? kStage : 16], l6[S > 4 ? kStage : 16], l7[S > 4 ? kStage : 16];
    __shared__ __attribute__((aligned(16))) uint8_t cb[TIER == 11 ? 2048 : 16];
    auto stage = [&](auto st) -> lds_u8 * {
        constexpr int k = decltype(st)::value % S;
        return k == 0 ? (lds_u8 *)l0 : k == 1 ? (lds_u8 *)l1 : k == 2 ? (lds_u8 *)l2 : k == 3 ? (lds_u8 *)l3
             : k == 4 ? (lds_u8 *)l4 : k == 5 ? (lds_u8 *)l5 : k == 6 ? (lds_u8 *)l6 : (lds_u8 *)l7;
    };
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(uint32_t(tid) >> 6);
    if constexpr (TIER == 11) {
        for (int i = tid; i < 2048; i += 256) cb[i] = uint8_t(g.codebook[i]);
        __syncthreads();
    }
    // neighbouring workgroups of one XCD share columns of B
    const uint32_t tiles_m = (g.m + BM - 1) / BM;
    uint32_t id = blockIdx.x;
    if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
    const uint32_t m0 = id % tiles_m * BM, n0 = id / tiles_m * BN;
    const uint32_t mrows = g.m - m0 < uint32_t(BM) ? g.m - m0 : uint32_t(BM);
    const uint32_t ncols = g.n - n0 < uint32_t(BN) ? g.n - n0 : uint32_t(BN);
    const uint32_t colb = TIER == 2 ? g.k : TIER == 10 ? g.k / 2 : g.k / 8;   // bytes of a column
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(g.q + uint64_t(m0) * g.kpad), 0,
                                                      int(mrows * g.kpad), 0x00020000);
    const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(g.bq + uint64_t(n0) * colb), 0,
                                                      int(ncols * colb), 0x00020000);
    auto swz8 = [](uint32_t row) { return (row >> 1) & 7u; };                    // 128-byte rows
    auto swz4 = [](uint32_t row) { return ((row >> 1) ^ (row >> 2)) & 3u; };     // 64-byte rows
    uint32_t a_voff[LA], b_voff[LB];
#pragma unroll
    for (int t = 0; t < LA; ++t) {
        const uint32_t row = (wave * LA + t) * 8 + lane / 8;
        a_voff[t] = row * g.kpad + 16u * ((lane & 7) ^ swz8(row));
    }
#pragma unroll
    for (int t = 0; t < LB; ++t) {
        if constexpr (TIER == 2) {
            const uint32_t row = (wave * LB + t) * 8 + lane / 8;
            b_voff[t] = row * colb + 16u * ((lane & 7) ^ swz8(row));
        } else if constexpr (TIER == 10) {
            const uint32_t row = (wave * LB + t) * 16 + lane / 4;
            b_voff[t] = row * colb + 16u * ((lane & 3) ^ swz4(row));
        } else {   // one load holds 64 columns: the waves share the tile's one or two
            b_voff[t] = ((wave % NJ) * 64 + lane) * colb;
        }
    }
    uint32_t todo = g.kpad / 128;
    auto dma = [&](auto st) {
        const bool live = todo != 0;
        lds_u8 *sa = stage(st) + wave * (LA * 1024u);
        lds_u8 *sb = stage(st) + kOffB + (TIER == 11 ? wave % NJ : wave * LB) * 1024u;
#pragma unroll
        for (int t = 0; t < LA; ++t) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, sa + 1024 * t, 16, live ? a_voff[t] : 0x80000000u, 0, 0, 0);
            a_voff[t] += 128;
        }
#pragma unroll
        for (int t = 0; t < LB; ++t) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, sb + 1024 * t, 16, live ? b_voff[t] : 0x80000000u, 0, 0, 0);
            b_voff[t] += PB;
        }
        todo = live ? todo - 1 : 0;
    };
    const uint32_t wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    i32x16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(3))) i32x4 lds_i32x4;
    typedef const __attribute__((address_space(3))) u32x2 lds_u2;
    typedef const __attribute__((address_space(3))) uint16_t lds_u16;
    i32x4 af[2][MI], bf[2][NJ];
    // the fragments of 32 k (step q of a slab) into buffer f
    auto frag = [&](auto st, int q, int f) {
        const lds_u8 *base = stage(st);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const uint32_t row = wm + 32 * i + lr;
            af[f][i] = *reinterpret_cast<lds_i32x4 *>(base + row * 128 + (((2u * q + lg) ^ swz8(lr)) * 16u));
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t row = wn + 32 * j + lr;
            const lds_u8 *b = base + kOffB + row * PB;
            if constexpr (TIER == 2) {
                bf[f][j] = *reinterpret_cast<lds_i32x4 *>(b + (((2u * q + lg) ^ swz8(lr)) * 16u));
            } else if constexpr (TIER == 10) {
                const uint32_t at = ((uint32_t(q) ^ swz4(lr)) * 16u) + 8u * lg;
                const u32x2 w = *reinterpret_cast<lds_u2 *>(b + at);
                bf[f][j] = spread_i4(w.x, w.y);
            } else {
                const uint32_t ix = *reinterpret_cast<lds_u16 *>(b + 4 * q + 2 * lg);
                const uint2 x = *reinterpret_cast<const uint2 *>(cb + (ix & 0xffu) * 8);
                const uint2 y = *reinterpret_cast<const uint2 *>(cb + (ix >> 8) * 8);
                bf[f][j] = i32x4{int(x.x), int(x.y), int(y.x), int(y.y)};
            }
        }
    };
    auto mfmas = [&](int f) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[f][i], bf[f][j], acc[i][j], 0, 0, 0);
    };
    // All of a wave's loads but the newest `n` slabs' have landed, for all waves,
    // and every wave is done reading the stage refilled next: i8 refills the stage
    // of the slab before, so its last reads are waited for here; with a slab's
    // slack (kAhead) they went into products that each step issues before it ends.
    auto landed = [&](auto n) {
        asm volatile("" ::: "memory");
        wait_vm<decltype(n)::value * (LA + LB), TIER == 2>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // i4 / e8cb: a slab's barrier stands before its last products, so that the
    // next slab's first fragments are read and unpacked under them (512 x 4096 x
    // 4096 i4 40 -> 30 us); i8 fragments need no unpacking, and the slab more
    // in flight is worth more (21.0 against 22.2 us).
    constexpr bool kAhead = TIER != 2;
    auto step = [&](auto st) {
        constexpr int kS = decltype(st)::value;
        if constexpr (!kAhead) {
            landed(std::integral_constant<int, S - 2>{});
            dma(std::integral_constant<int, kS + S - 1>{});
            frag(st, 0, 0);
        }
        frag(st, 1, 1);
        mfmas(0);
        frag(st, 2, 0);
        mfmas(1);
        frag(st, 3, 1);
        mfmas(0);
        if constexpr (kAhead) {
            landed(std::integral_constant<int, S - 3>{});
            dma(std::integral_constant<int, kS + S - 1>{});
            frag(std::integral_constant<int, kS + 1>{}, 0, 0);
        }
        mfmas(1);
        if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
    };
    using c0 = std::integral_constant<int, 0>;
    using c1 = std::integral_constant<int, 1>;
    using c2 = std::integral_constant<int, 2>;
    using c3 = std::integral_constant<int, 3>;
    using c4 = std::integral_constant<int, 4>;
    using c5 = std::integral_constant<int, 5>;
    using c6 = std::integral_constant<int, 6>;
    using c7 = std::integral_constant<int, 7>;
    dma(c0{});
    dma(c1{});
    dma(c2{});
    if constexpr (S > 4) {
        dma(c3{});
        dma(c4{});
        dma(c5{});
        dma(c6{});
    }
    if constexpr (kAhead) {
        landed(std::integral_constant<int, S - 2>{});
        frag(c0{}, 0, 0);
    }
    const uint32_t nk = g.kpad / 128;
    for (uint32_t s = 0; s < nk; s += S) {   // slabs past K multiply zeros
        step(c0{});
        step(c1{});
        step(c2{});
        step(c3{});
        if constexpr (S > 4) {
            step(c4{});
            step(c5{});
            step(c6{});
            step(c7{});
        }
    }
    // C layout: acc[r] is row 8 (r / 4) + 4 lg + r % 4, column lr
    const auto rc = __builtin_amdgcn_make_buffer_rsrc(g.out + uint64_t(m0) * g.n, 0, int(mrows * g.n * 4u), 0x00020000);
    const auto rr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(g.residual ? g.residual + uint64_t(m0) * g.n : g.out), 0,
        g.residual ? int(mrows * g.n * 4u) : 0, 0x00020000);
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.sa + m0), 0, int(mrows * 4u), 0x00020000);
    wait_vm<0, true>();   // the last (empty) loads into LDS, the last reads of the stages
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float *mine = reinterpret_cast<float *>(wave == 0 ? l0 : wave == 1 ? l1 : wave == 2 ? l2 : l3);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        float si[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            si[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                  rs, (wm + 32u * i + 8u * (r >> 2) + 4u * lg + (r & 3)) * 4u, 0, 0));
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t col = n0 + wn + 32u * j + lr;
            const float sj = g.scales[col < g.n ? col : g.n - 1];
            const uint32_t off = col < g.n ? ((wm + 32u * i + 4u * lg) * g.n + col) * 4u : 0x80000000u;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t ro = (8u * (r >> 2) + (r & 3)) * g.n * 4u;
                float o = si[r] == 0.0f ? 0.0f : float(acc[i][j][r]) * (si[r] * sj);
                if (g.residual)
                    o = o + __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, off, ro, 0));
                if (g.act) mine[((i * NJ + j) * 16 + r) * 64 + lane] = o;
                else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), rc, off, ro, 0);
            }
        }
    }
    if (g.act) {   // one copy of the activation's code, not one an element
#pragma unroll 1
        for (int e = 0; e < MI * NJ * 16; ++e) {
            const uint32_t i = uint32_t(e) / (16 * NJ), j = uint32_t(e) / 16 % NJ, r = uint32_t(e) % 16;
            const uint32_t col = n0 + wn + 32u * j + lr;
            const uint32_t off = col < g.n ? ((wm + 32u * i + 4u * lg) * g.n + col) * 4u : 0x80000000u;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(act_f32(g.act, mine[e * 64 + lane])), rc, off,
                                                  (8u * (r >> 2) + (r & 3)) * g.n * 4u, 0);
        }
    }
}

template <int BM, int BN, int TIER, int S>
__global__ __launch_bounds__(256, 1) void gemm_q_tiled_kernel(const QGemm g) {
    gemm_q_tiled<BM, BN, TIER, S>(g);
}

// ----------------------------------------------------- W8A8 decode GEMV ----
// Few rows (m <= 4): the dot products on v_dot4c_i32_i8 instead of MFMA, so
// the weight stream is fully coalesced: a wavefront owns kGemvCols columns
// and its 64 lanes sweep each column's k-vector in consecutive chunks (lane
// l takes chunks l, l + 64, ...), one 16-byte (e8cb: 8-byte) load per column
// per chunk; the int32 sums are exact, so the order of the lanes' partial sums
// and of the cross-lane reduction does not matter. Chunks: i8 16 levels
// (16 bytes), i4 32 levels (16 bytes: word t holds levels 8t .. 8t+7, even
// levels in the low nibbles), e8cb 64 levels (8 codebook indices).
constexpr int kGemvCols = 8;
// Workgroups of the GEMV: each loops over column blocks (4 waves x kGemvCols
// columns) with a grid stride, so the e8cb codebook is staged once per
// workgroup and every wavefront streams several blocks.
constexpr uint32_t kGemvGrid = 2048;

// Reduce-scatter of N int32 values (N a power of two, <= 64) over the 64
// lanes: each xor step halves the values a lane holds (it keeps the half its
// lane bit selects and adds its partner's copy of that half), then plain xor
// sums finish the strides left. Lane l ends with the wavefront's total of
// value `index` (the bits the halving steps selected); integer sums are exact,
// so the result is the plain total.
template <int N, int S>
struct Scatter {
    static __device__ __forceinline__ void run(int32_t *v, int lane, int &index) {
        constexpr int H = N / 2;
        const bool up = (lane & S) != 0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int32_t send = up ? v[i] : v[i + H];
            const int32_t recv = __shfl_xor(send, S, 64);
            v[i] = (up ? v[i + H] : v[i]) + recv;
        }
        if (up) index += H;
        Scatter<H, S / 2>::run(v, lane, index);
    }
};
template <int S>
struct Scatter<1, S> {
    static __device__ __forceinline__ void run(int32_t *v, int lane, int &index) {
        v[0] += __shfl_xor(v[0], S, 64);
        Scatter<1, S / 2>::run(v, lane, index);
    }
};
template <>
struct Scatter<1, 0> {
    static __device__ __forceinline__ void run(int32_t *, int, int &) {}
};

template <int TIER>
struct GemvChunk {
    static constexpr uint32_t elems = TIER == 2 ? 16 : (TIER == 10 ? 32 : 64);
    static constexpr uint32_t bytes = TIER == 11 ? 8 : 16;
};

template <int TIER, int M>
__global__ __launch_bounds__(256) void gemv_q_omajor_kernel(QGemm g) {
    using Ch = GemvChunk<TIER>;
    __shared__ __attribute__((aligned(16))) int8_t cbb[TIER == 11 ? 256 * 8 : 16];
    if constexpr (TIER == 11) {
        for (int i = threadIdx.x; i < 256 * 8; i += 256) cbb[i] = g.codebook[i];
        __syncthreads();
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t nchunk = g.k / Ch::elems;
    const uint64_t col_bytes = uint64_t(g.k) * Ch::bytes / Ch::elems;
    const uint32_t nblk = (g.n + 4 * kGemvCols - 1) / (4 * kGemvCols);
    for (uint32_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
    const uint32_t j0 = (blk * 4 + wave) * kGemvCols;
    int32_t acc[M][kGemvCols];
    int32_t corr[M];   // i4: the sum of the activation levels (the nibble bias)
#pragma unroll
    for (int r = 0; r < M; ++r) {
        corr[r] = 0;
#pragma unroll
        for (int c = 0; c < kGemvCols; ++c) acc[r][c] = 0;
    }
    for (uint32_t ch = lane; ch < nchunk; ch += 64) {
        // every column's chunk first, so the loads are in flight together
        u32x4 w[kGemvCols];
        uint64_t wi[kGemvCols];
#pragma unroll
        for (int c = 0; c < kGemvCols; ++c) {
            const uint32_t j = j0 + c < g.n ? j0 + c : g.n - 1;   // a clamped column is never stored
            const uint8_t *p = g.bq + uint64_t(j) * col_bytes + uint64_t(ch) * Ch::bytes;
            if constexpr (TIER == 11) wi[c] = *reinterpret_cast<const uint64_t *>(p);
            else w[c] = ld_stream(reinterpret_cast<const u32x4 *>(p));
        }
#pragma unroll
        for (int r = 0; r < M; ++r) {
            const u32x4 *qa = reinterpret_cast<const u32x4 *>(g.q + uint64_t(r) * g.kpad +
                                                             uint64_t(ch) * Ch::elems);
            if constexpr (TIER == 2) {
                const u32x4 x = qa[0];
#pragma unroll
                for (int c = 0; c < kGemvCols; ++c)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        acc[r][c] = __builtin_amdgcn_sdot4(int(x[t]), int(w[c][t]), acc[r][c], false);
            } else if constexpr (TIER == 10) {
                const u32x4 x0 = qa[0], x1 = qa[1];
                const uint32_t xa[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    // levels 8t .. 8t+7: even ones (low nibbles) and odd ones (high)
                    const uint32_t lo = __builtin_amdgcn_perm(xa[2 * t + 1], xa[2 * t], 0x06040200u);
                    const uint32_t hi = __builtin_amdgcn_perm(xa[2 * t + 1], xa[2 * t], 0x07050301u);
                    corr[r] = __builtin_amdgcn_sdot4(int(xa[2 * t]), 0x01010101, corr[r], false);
                    corr[r] = __builtin_amdgcn_sdot4(int(xa[2 * t + 1]), 0x01010101, corr[r], false);
#pragma unroll
                    for (int c = 0; c < kGemvCols; ++c) {
                        // a nibble u, as (u ^ 8) in 0..15: its signed level is (u ^ 8) - 8
                        const uint32_t b = w[c][t] ^ 0x88888888u;
                        acc[r][c] = __builtin_amdgcn_sdot4(int(lo), int(b & 0x0F0F0F0Fu), acc[r][c], false);
                        acc[r][c] = __builtin_amdgcn_sdot4(int(hi), int((b >> 4) & 0x0F0F0F0Fu), acc[r][c],
                                                           false);
                    }
                }
            } else {
                const u32x4 x0 = qa[0], x1 = qa[1], x2 = qa[2], x3 = qa[3];
                const uint32_t xa[16] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3],
                                         x2[0], x2[1], x2[2], x2[3], x3[0], x3[1], x3[2], x3[3]};
#pragma unroll
                for (int c = 0; c < kGemvCols; ++c)
#pragma unroll
                    for (int h = 0; h < 8; ++h) {
                        const uint32_t half = h < 4 ? uint32_t(wi[c]) : uint32_t(wi[c] >> 32);
                        const uint32_t idx = (half >> (8 * (h & 3))) & 0xffu;
                        const uint64_t v = *reinterpret_cast<const uint64_t *>(cbb + idx * 8);
                        acc[r][c] = __builtin_amdgcn_sdot4(int(xa[2 * h]), int(uint32_t(v)), acc[r][c], false);
                        acc[r][c] = __builtin_amdgcn_sdot4(int(xa[2 * h + 1]), int(uint32_t(v >> 32)),
                                                           acc[r][c], false);
                    }
            }
        }
    }
    // exact int32 totals over the wavefront (the i4 bias folded in first: the
    // totals are linear in the lanes' sums); M = 3 is padded to four rows
    constexpr int MP = M == 3 ? 4 : M;
    int32_t v[MP * kGemvCols];
#pragma unroll
    for (int r = 0; r < MP; ++r)
#pragma unroll
        for (int c = 0; c < kGemvCols; ++c)
            v[r * kGemvCols + c] = r < M ? (TIER == 10 ? acc[r][c] - 8 * corr[r] : acc[r][c]) : 0;
    int index = 0;
    Scatter<MP * kGemvCols, 32>::run(v, lane, index);
    if ((lane & (64 / (MP * kGemvCols) - 1)) == 0) {
        const int r = index / kGemvCols, c = index % kGemvCols;
        const int32_t tot = v[0];
        const uint32_t j = j0 + c;
        if (uint32_t(r) < g.m && j < g.n) {
            const float si = g.sa[r], sj = g.scales[j];
            float o = si == 0.0f ? 0.0f : float(tot) * (si * sj);
            if (g.residual) o = o + g.residual[uint64_t(r) * g.n + j];
            if (g.act) o = act_f32_call(g.act, o);
            g.out[uint64_t(r) * g.n + j] = o;
        }
    }
    }
}

// ------------------------------------------------------------- Dequantize ----
struct DqArgs {
    const uint8_t *in;
    const float *scales;      // per-channel, or null
    const int32_t *zps;       // per-channel, or null
    void *out;
    uint64_t n;
    uint32_t channels, inner;
    uint8_t quant;            // 2 i8, 1 u8, 10 i4
    uint8_t dtype;            // 8 f32, 7 bf16, 6 f16
    float scale;
    int32_t zp;
};

__device__ __forceinline__ int32_t level_at(const DqArgs &d, uint64_t i) {
    if (d.quant == 2) return int32_t(int8_t(d.in[i]));
    if (d.quant == 1) return int32_t(d.in[i]);
    const uint32_t byte = d.in[i >> 1];
    const int32_t v = int32_t((i & 1) ? (byte >> 4) : (byte & 0x0Fu));
    return v >= 8 ? v - 16 : v;
}

__global__ __launch_bounds__(256) void dequant_kernel(DqArgs d) {
    const uint64_t stride = uint64_t(gridDim.x) * 256;
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < d.n; i += stride) {
        float s = d.scale;
        int32_t z = d.zp;
        if (d.scales) {
            const uint32_t ch = uint32_t((i / d.inner) % d.channels);
            s = d.scales[ch];
            z = d.zps[ch];
        }
        // (q - zp) in wrapping i32, then `as f32`, then * scale (kernels.rs:270)
        const int32_t qz = int32_t(uint32_t(level_at(d, i)) - uint32_t(z));
        const float v = float(qz) * s;
        if (d.dtype == 8) static_cast<float *>(d.out)[i] = v;
        else if (d.dtype == 7) static_cast<uint16_t *>(d.out)[i] = uint16_t(__float_as_uint(v) >> 16);
        else static_cast<uint16_t *>(d.out)[i] = f32_to_f16_bits(v);
    }
}

// ------------------------------------------------------- DequantActivation --
struct DqActTable {
    float t[256];
};

__global__ __launch_bounds__(256) void dequant_act_kernel(const uint8_t *__restrict__ in,
                                                          float *__restrict__ out, uint64_t n,
                                                          bool i4, DqActTable tab) {
    const uint64_t stride = uint64_t(gridDim.x) * 256;
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        uint32_t idx;
        if (i4) {
            const uint32_t byte = in[i >> 1];
            idx = (i & 1) ? (byte >> 4) : (byte & 0x0Fu);
        } else {
            idx = in[i];
        }
        out[i] = tab.t[idx];
    }
}

__global__ __launch_bounds__(256) void zp_zero_kernel(const ZeroPoints z) {
    check_zero_points(z, blockIdx.x, gridDim.x);
}

uint32_t grid_for(uint64_t n) {
    const uint64_t b = (n + 255) / 256;
    return uint32_t(b < 4096 ? (b ? b : 1) : 4096);
}

}  // namespace

size_t q_omajor_scratch_bytes(uint32_t m, uint32_t k) {
    const uint64_t kpad = (uint64_t(k) + 127) / 128 * 128;
    return size_t(m) * kpad + size_t(m) * 4 + 256;
}

hipError_t launch_matmul_q_omajor(const QOmajorArgs &a, void *scratch, hipStream_t stream) {
    const uint32_t kpad = (a.k + 127) / 128 * 128;
    int8_t *q = static_cast<int8_t *>(scratch);
    float *sa = reinterpret_cast<float *>(static_cast<uint8_t *>(scratch) +
                                          (uint64_t(a.m) * kpad + 255) / 256 * 256);
    const ZeroPoints z{static_cast<const uint8_t *>(a.zero_points), a.zero_point_bytes, a.err};
    const uint64_t zb = (z.bytes + kZpBlock - 1) / kZpBlock;
    const uint32_t zblocks = uint32_t(zb < 512 ? zb : 512);
    if (a.k % 4 == 0 && kpad <= 8192 && (reinterpret_cast<uintptr_t>(a.a) & 15) == 0 && a.m < (1u << 30)) {
        const dim3 gq(a.m + zblocks);
        if (kpad <= 1024) hipLaunchKernelGGL(quant_rows_vec_kernel<1>, gq, dim3(256), 0, stream, a.a, a.m, a.k, kpad, q, sa, z);
        else if (kpad <= 2048) hipLaunchKernelGGL(quant_rows_vec_kernel<2>, gq, dim3(256), 0, stream, a.a, a.m, a.k, kpad, q, sa, z);
        else if (kpad <= 4096) hipLaunchKernelGGL(quant_rows_vec_kernel<4>, gq, dim3(256), 0, stream, a.a, a.m, a.k, kpad, q, sa, z);
        else hipLaunchKernelGGL(quant_rows_vec_kernel<8>, gq, dim3(256), 0, stream, a.a, a.m, a.k, kpad, q, sa, z);
    } else {
        if (zblocks) hipLaunchKernelGGL(zp_zero_kernel, dim3(zblocks), dim3(256), 0, stream, z);
        hipLaunchKernelGGL(quant_rows_kernel, dim3(a.m), dim3(256), 0, stream, a.a, a.k, kpad, q, sa);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    QGemm g;
    g.q = q;
    g.sa = sa;
    g.bq = static_cast<const uint8_t *>(a.bq);
    g.codebook = a.codebook;
    g.scales = a.scales;
    g.residual = a.residual;
    g.out = a.out;
    g.m = a.m;
    g.k = a.k;
    g.n = a.n;
    g.kpad = kpad;
    g.act = a.act;
    // the decode GEMV when its whole chunks tile k and the loads are aligned
    const uint32_t ce = a.tier == 2 ? 16 : (a.tier == 10 ? 32 : 64);
    const uintptr_t bal = a.tier == 11 ? 7 : 15;
    if (a.m <= 4 && a.k % ce == 0 && (reinterpret_cast<uintptr_t>(a.bq) & bal) == 0) {
        const uint32_t nblk = (a.n + 4 * kGemvCols - 1) / (4 * kGemvCols);
        const dim3 gg(nblk < kGemvGrid ? nblk : kGemvGrid);
#define HOLO_QV(T, M) hipLaunchKernelGGL((gemv_q_omajor_kernel<T, M>), gg, dim3(256), 0, stream, g)
#define HOLO_QVM(T)                         \
    do {                                    \
        switch (a.m) {                      \
            case 1: HOLO_QV(T, 1); break;   \
            case 2: HOLO_QV(T, 2); break;   \
            case 3: HOLO_QV(T, 3); break;   \
            default: HOLO_QV(T, 4); break;  \
        }                                   \
    } while (0)
        switch (a.tier) {
            case 2: HOLO_QVM(2); break;
            case 10: HOLO_QVM(10); break;
            case 11: HOLO_QVM(11); break;
            default: return hipErrorInvalidValue;
        }
#undef HOLO_QVM
#undef HOLO_QV
        return hipGetLastError();
    }
    // Many rows: the tiled kernel where its 16-byte loads fit (whole chunks of
    // the weight's columns) and its ranges hold. Below these rows the kernel
    // that gives 16 columns to a workgroup streams the weight as fast (i8 16
    // rows of 4096 x 4096: 12.1 us against 12.9; e8cb 14.1 against 15.8; i4,
    // whose unpacking it does a row tile at a time, 24.6 against 18.7 at 5 rows).
    const uint32_t kc = a.tier == 2 ? 16 : (a.tier == 10 ? 32 : 128);
    if (a.m > (a.tier == 10 ? 4u : 16u) && a.k % kc == 0 && (reinterpret_cast<uintptr_t>(a.bq) & 15) == 0 &&
        a.n < (1u << 22)) {
        // the smallest tile whose launch is one round of the CUs, else the
        // largest: 512 x 4096 x 4096 i8 takes 27.2 / 21.0 / 25.4 us on 128 x 128
        // / 64 x 128 / 64 x 64, 1024 rows 33.7 / 37.4 / 46.5, 256 rows 25.3 /
        // 17.4 / 15.4
        const uint64_t t64 = uint64_t((a.m + 63) / 64) * ((a.n + 63) / 64);
        const uint64_t t64x128 = uint64_t((a.m + 63) / 64) * ((a.n + 127) / 128);
        const uint32_t bm = t64 > 256 && t64x128 > 256 ? 128 : 64, bn = t64 > 256 ? 128 : 64;
        const uint64_t tiles = uint64_t((a.m + bm - 1) / bm) * ((a.n + bn - 1) / bn);
        if (tiles < (1ull << 31)) {
            const dim3 gt{unsigned(tiles)};
#define HOLO_QTILE(T)                                                                                              \
    do {                                                                                                           \
        if (bm == 128) hipLaunchKernelGGL((gemm_q_tiled_kernel<128, 128, T, 4>), gt, dim3(256), 0, stream, g);     \
        else if (bn == 128) hipLaunchKernelGGL((gemm_q_tiled_kernel<64, 128, T, 4>), gt, dim3(256), 0, stream, g); \
        else hipLaunchKernelGGL((gemm_q_tiled_kernel<64, 64, T, 8>), gt, dim3(256), 0, stream, g);                 \
    } while (0)
            switch (a.tier) {
                case 2: HOLO_QTILE(2); break;
                case 10: HOLO_QTILE(10); break;
                case 11: HOLO_QTILE(11); break;
                default: return hipErrorInvalidValue;
            }
#undef HOLO_QTILE
            return hipGetLastError();
        }
    }
    const bool tall = a.m > 16;
    const dim3 grid((a.n + 15) / 16, tall ? (a.m + 63) / 64 : 1);
#define HOLO_QG(T)                                                                            \
    do {                                                                                      \
        if (tall) hipLaunchKernelGGL((gemm_q_omajor_kernel<T, 4>), grid, dim3(256), 0, stream, g); \
        else hipLaunchKernelGGL((gemm_q_omajor_kernel<T, 1>), grid, dim3(256), 0, stream, g); \
    } while (0)
    switch (a.tier) {
        case 2: HOLO_QG(2); break;
        case 10: HOLO_QG(10); break;
        case 11: HOLO_QG(11); break;
        default: return hipErrorInvalidValue;
    }
#undef HOLO_QG
    return hipGetLastError();
}

hipError_t launch_dequantize(const DequantArgs &a, hipStream_t stream) {
    if (a.n == 0) return hipSuccess;
    DqArgs d;
    d.in = static_cast<const uint8_t *>(a.in);
    d.scales = a.scales;
    d.zps = a.zps;
    d.out = a.out;
    d.n = a.n;
    d.channels = a.channels;
    d.inner = a.inner ? a.inner : 1;
    d.quant = a.quant;
    d.dtype = a.dtype;
    d.scale = a.scale;
    d.zp = a.zp;
    hipLaunchKernelGGL(dequant_kernel, dim3(grid_for(a.n)), dim3(256), 0, stream, d);
    return hipGetLastError();
}

hipError_t launch_dequant_act(const uint8_t *in, float *out, uint64_t n, bool i4,
                              const float table[256], hipStream_t stream) {
    if (n == 0) return hipSuccess;
    DqActTable t;
    for (int i = 0; i < 256; ++i) t.t[i] = table[i];
    hipLaunchKernelGGL(dequant_act_kernel, dim3(grid_for(n)), dim3(256), 0, stream, in, out, n, i4,
                       t);
    return hipGetLastError();
}

}  // namespace holo
