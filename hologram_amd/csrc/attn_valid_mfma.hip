// attn_valid_mfma.hip — DecodeAttentionValid (121) and its mask form (119) on
// the matrix cores, for head_dim up to 128 with 16-byte rows. The semantics
// are attn_valid.hip's: the key list of a plane is its realized past rows, then
// the new rows; a row sees its causal prefix of the list (valid form) or all of
// it with an additive f32 mask (mask form); f32 softmax; a key whose score is
// NaN weighs 0; a row with no visible key is the zero row.
//
// Precision. bf16 / f16 products are exact in f32 and accumulate in f32. The
// softmax weights stay f32: for the PV product each is split into a rounded
// 16-bit part and the 16-bit rounding of what is left (hi + lo, 2^-18 of the
// weight for bf16, 2^-21 for f16), both multiplied with V and summed in f32.
// f16 weights carry a factor 2^15 so neither part meets f16's subnormals.
// f32 operands use the f32 matrix instructions throughout.
//
// Non-finite values. A weight of 0 (a key past its row's limit) times a
// non-finite V is NaN on the matrix cores, and so is an infinite V under a
// split weight, where the reference skips the key or keeps the infinity. A
// non-finite V in a share always leaves a non-finite accumulator, so a
// workgroup that ends with one redoes its share with the scalar walk
// (walk_row); a share that ends finite held no such value.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "holo_device.h"
#include "holo_kernels.h"

namespace holo {
namespace {

constexpr int kThreads = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr float kLog2e = 1.4426950408889634f;
constexpr uint32_t kOob = 0x80000000u;   // an offset past every buffer range: loads nothing
constexpr float kPScale = 15.0f;         // f16 weights: p * 2^15

__device__ __forceinline__ __amdgpu_buffer_rsrc_t range(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, int(bytes), 0x00020000);
}
__device__ __forceinline__ uint32_t read_u32_le(const uint8_t *p) {   // any alignment
    return uint32_t(p[0]) | (uint32_t(p[1]) << 8) | (uint32_t(p[2]) << 16) | (uint32_t(p[3]) << 24);
}
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ float max_half(float v) {      // with the lane 32 apart
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
}
__device__ __forceinline__ float max_quarter(float v) {   // with the lanes 16, 32, 48 apart
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max_half(fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1])));
}

// 2^x of an online softmax step: NaN (a NaN score, or an infinite score less
// an infinite maximum) and anything below f32's range give 0.
__device__ __forceinline__ float weight(float x) { return __builtin_amdgcn_exp2f(fmaxf(x, -200.0f)); }

// Two weights as 16-bit hi parts and the 16-bit rounding of the remainders.
template <int DT>
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
    if constexpr (DT == 7) {
        hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
        const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xFFFF0000u);
        lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{ra, rb}, bf16x2));
    } else {
        const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
        hi = __builtin_bit_cast(uint32_t, h);
        lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a - float(h[0]), b - float(h[1])));
    }
}
template <int DT>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (DT == 7)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == 7)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ float ld_elem(const void *p, uint64_t i) {
    if constexpr (DT == 8) return static_cast<const float *>(p)[i];
    else if constexpr (DT == 7) return __uint_as_float(uint32_t(static_cast<const uint16_t *>(p)[i]) << 16);
    else return f16_bits_to_f32(static_cast<const uint16_t *>(p)[i]);
}
template <int DT>
__device__ __forceinline__ void st_elem(void *p, uint64_t i, float v) {
    if constexpr (DT == 8) static_cast<float *>(p)[i] = v;
    else if constexpr (DT == 7) static_cast<uint16_t *>(p)[i] = uint16_t(__float_as_uint(v) >> 16);
    else static_cast<uint16_t *>(p)[i] = f32_to_f16_bits(v);
}

// One query row over list entries [j0, j1) by one wavefront, in the
// reference's scalar steps: a key per lane for the scores, then a column (or
// two) per lane for PV, key by key, entries past the row's limit left out.
// Kept small (no unrolling): it only runs for a share that holds a non-finite
// V. `single`: writes the output row; else (m, l, acc) at pp, m times munit.
template <int DT>
__device__ __forceinline__ void walk_row(const AttnValidArgs &a, uint32_t plane, uint32_t r, uint32_t vis,
                                         uint32_t j0, uint32_t j1, bool single, float munit, float *pp) {
    const uint32_t lane = threadIdx.x & 63, D = a.D, R = a.H / a.Hkv * a.M, qi = r % a.M;
    const uint32_t total = vis + a.nnew;
    const uint32_t lim = a.mask ? total : vis + (qi + 1 < a.nnew ? qi + 1 : a.nnew);
    const uint64_t q0 = (uint64_t(plane) * R + r) * D;
    const uint64_t p0 = uint64_t(plane) * a.past, n0 = uint64_t(plane) * a.nnew;
    const uint32_t end = j1 < lim ? j1 : lim;
    float m = -INFINITY, l = 0.0f, acc[2] = {0.0f, 0.0f};
#pragma unroll 1
    for (uint32_t jb = j0; jb < end; jb += 64) {
        const uint32_t j = jb + lane;
        float s = -INFINITY;
        if (j < end) {
            const bool past = j < vis;
            const void *k = past ? a.kp : a.kn;
            const uint64_t k0 = (past ? p0 + j : n0 + j - vis) * D;
            float d = 0.0f;
#pragma unroll 1
            for (uint32_t c = 0; c < D; ++c) d = fmaf(ld_elem<DT>(a.q, q0 + c), ld_elem<DT>(k, k0 + c), d);
            s = d / a.scale;
            if (a.mask) s = s + a.mask[uint64_t(qi) * total + j];
        }
        float mb = s;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) mb = fmaxf(mb, __shfl_xor(mb, o, 64));
        const float mn = fmaxf(m, mb);
        float p = 0.0f, al = 1.0f;
        if (mn != -INFINITY) {
            p = s == -INFINITY ? 0.0f : exp_det(s - mn);
            al = m == -INFINITY ? 0.0f : exp_det(m - mn);
        }
        float ps = p;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) ps += __shfl_xor(ps, o, 64);
        l = l * al + ps;
        m = mn;
        acc[0] *= al;
        acc[1] *= al;
        const uint32_t n = end - jb < 64 ? end - jb : 64;
#pragma unroll 1
        for (uint32_t i = 0; i < n; ++i) {
            const bool past = jb + i < vis;
            const void *v = past ? a.vp : a.vn;
            const uint64_t v0 = (past ? p0 + jb + i : n0 + jb + i - vis) * D;
            const float w = __shfl(p, int(i), 64);
            if (lane < D) acc[0] = fmaf(w, ld_elem<DT>(v, v0 + lane), acc[0]);
            if (lane + 64 < D) acc[1] = fmaf(w, ld_elem<DT>(v, v0 + lane + 64), acc[1]);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t c = lane + 64u * h;
        if (c >= D) continue;
        if (single) st_elem<DT>(a.out, q0 + c, m == -INFINITY ? 0.0f : acc[h] / (l > 1e-30f ? l : 1e-30f));
        else pp[2 + c] = acc[h];
    }
    if (!single && lane == 0) {
        pp[0] = m * munit;
        pp[1] = l;
    }
}

// ------------------------------------------------- many rows (a prompt) ----
// A workgroup takes 128 of a plane's G*M query rows (contiguous in q: heads
// kvh*G .. kvh*G+G-1), 32 a wave, over a share of the list in 64-key tiles.
// K and V tiles go from memory into LDS by DMA (lane l of a load writes its 16
// bytes at LDS base + 16 l), the next tile's while this one is computed; each
// 16-byte chunk of a row sits at chunk ^ f(row), so the K reads (32 rows, one
// chunk) and the transposing V reads (4 rows x 64 bytes a half) meet distinct
// banks. Per tile and wave:
//     S^T[64 keys x 32 rows] = K . Q^T     32x32x16
//     online softmax, a row per lane column (its keys in the lane and the
//     lane 32 apart)
//     O^T[D x 32 rows] += V^T . (hi + lo)^T  32x32x16; a lane's 8 scores of a
//     16-key step are its operand when V^T's keys are read in the order the
//     S^T layout holds them (4 lg + 0..3, 8 + 4 lg + 0..3).
// Bound by the matrix and vector work of a wave (the softmax is about as long
// as the products; one wave a SIMD at the size below). 509 rows x 32 heads over
// 8 kv heads of 128 dims, 2 sequences, after 1537 cached keys, bf16: 63 us (470
// TFLOP/s) against 3.88 ms for the scalar walk's kernel. A tile holds 64
// consecutive list entries wherever the past ends, so past || new gives the
// bits of the same keys precatenated.
constexpr uint32_t kRowsWg = 128, kTile = 64;

template <int RB>
__device__ __forceinline__ uint32_t swz_k(uint32_t row) {
    return RB == 256 ? (row & 15u) : ((row >> 1) & 7u);
}
template <int RB>
__device__ __forceinline__ uint32_t swz_v(uint32_t row) {
    return RB == 256 ? 4u * (row & 3u) : 4u * ((row >> 1) & 1u);
}

template <int DT, int DB, bool kMask>
__device__ __forceinline__ void attn_valid_rows(const AttnValidArgs &a, const uint32_t tiles,
                                                const uint32_t nsplit, float *__restrict__ part) {
    constexpr int RB = DB <= 2 ? 128 : 256;          // LDS bytes of a key row
    constexpr int NK = 2 * DB;                       // 16-dim steps of the scores
    constexpr int LPW = int(kTile) * RB / 4096;      // 1 KiB loads a wave, each of K and V
    constexpr uint32_t CPR = RB / 16, RPL = 1024 / RB;   // chunks a row, rows a load
    __shared__ __attribute__((aligned(1024))) uint8_t k0s[kTile * RB], v0s[kTile * RB],
        k1s[kTile * RB], v1s[kTile * RB];
    const uint32_t D = a.D, R = a.H / a.Hkv * a.M;
    // neighbouring workgroups of one XCD share a plane's K and V; later tiles
    // (more visible keys) first
    uint32_t id = blockIdx.x;
    const uint32_t nwg = gridDim.x;
    if (nwg % 8 == 0) id = (id % 8) * (nwg / 8) + id / 8;
    const uint32_t split = id % nsplit, rest = id / nsplit;
    const uint32_t tile = tiles - 1 - rest % tiles, plane = rest / tiles;
    const uint32_t r0 = tile * kRowsWg;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const uint32_t wave = uniform(uint32_t(tid) >> 6);

    uint32_t vis = kMask ? a.past : read_u32_le(a.valid_len);   // realized past rows
    vis = uniform(vis < a.past ? vis : a.past);
    const uint32_t total = vis + a.nnew;
    // list entries row r sees, those any row of the workgroup sees
    auto limit = [&](uint32_t r) -> uint32_t {
        const uint32_t qi = r % a.M;
        return kMask ? total : vis + (qi + 1 < a.nnew ? qi + 1 : a.nnew);
    };
    const uint32_t rl = (r0 + kRowsWg < R ? r0 + kRowsWg : R) - 1;
    const uint32_t most = r0 / a.M == rl / a.M ? limit(rl) : total;
    const uint32_t ntl = (most + kTile - 1) / kTile;
    const uint32_t per = (ntl + nsplit - 1) / nsplit;
    const uint32_t t0 = split * per < ntl ? split * per : ntl;
    const uint32_t t1 = t0 + per < ntl ? t0 + per : ntl;

    // this lane's row (a copy of the last one past R), its limit, and the
    // least and the most of the wave
    const uint32_t wr0 = r0 + 32u * wave;
    const uint32_t row = wr0 + lr < R ? wr0 + lr : R - 1;
    const uint32_t lim = limit(row);
    const uint32_t wl = wr0 + 31 < R ? wr0 + 31 : R - 1, wf = wr0 < R ? wr0 : R - 1;
    const bool one_head = wf / a.M == wl / a.M;
    const uint32_t wmin = one_head ? limit(wf) : limit(0), wmax = one_head ? limit(wl) : total;
    const uint32_t qi = row % a.M;

    const uint32_t rowb = D * 2u;
    u32x4 qf[NK];
    {
        const uint16_t *qp = static_cast<const uint16_t *>(a.q) + (uint64_t(plane) * R + row) * D + 8 * lg;
#pragma unroll
        for (int k = 0; k < NK; ++k)
            qf[k] = uint32_t(16 * k + 8 * lg) < D ? *reinterpret_cast<const u32x4 *>(qp + 16 * k)
                                                  : u32x4{0, 0, 0, 0};
    }

    uint32_t koff[LPW], voff[LPW];
#pragma unroll
    for (int t = 0; t < LPW; ++t) {
        const uint32_t r = (wave * LPW + t) * RPL + lane / CPR, c = lane % CPR;
        const uint32_t ck = c ^ swz_k<RB>(r), cv = c ^ swz_v<RB>(r);
        koff[t] = 8u * ck < D ? r * rowb + ck * 16u : kOob;
        voff[t] = 8u * cv < D ? r * rowb + cv * 16u : kOob;
    }
    const uint64_t pbase = uint64_t(plane) * a.past * rowb, nbase = uint64_t(plane) * a.nnew * rowb;
    auto dma = [&](uint32_t t, uint8_t *ks, uint8_t *vs) {
        const bool live = t < t1;
        const uint32_t key0 = t * kTile;
        lds_u8 *kd = (lds_u8 *)ks + wave * (LPW * 1024u), *vd = (lds_u8 *)vs + wave * (LPW * 1024u);
        const bool past = key0 < vis;
        const uint8_t *kb = static_cast<const uint8_t *>(past ? a.kp : a.kn) + (past ? pbase : nbase);
        const uint8_t *vb = static_cast<const uint8_t *>(past ? a.vp : a.vn) + (past ? pbase : nbase);
        const uint32_t bytes = live ? (past ? vis : a.nnew) * rowb : 0u;   // past the range: zeros
        const uint32_t so = live ? (past ? key0 : key0 - vis) * rowb : 0u;
        const auto rk = range(kb, bytes), rv = range(vb, bytes);
#pragma unroll
        for (int i = 0; i < LPW; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, kd + 1024 * i, 16, koff[i], so, 0, 0);
#pragma unroll
        for (int i = 0; i < LPW; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, vd + 1024 * i, 16, voff[i], so, 0, 0);
    };

    // The tile in which the past ends comes from the past's rows (zeros beyond
    // them); before it is used, each wave loads the new rows over the zeros it
    // wrote itself.
    const uint32_t tmid = vis % kTile != 0 && a.nnew != 0 ? vis / kTile : 0xffffffffu;
    auto patch = [&](uint8_t *ks, uint8_t *vs) {
        __builtin_amdgcn_s_waitcnt((15 << 8) | (7 << 4));   // vmcnt(0)
        lds_u8 *kd = (lds_u8 *)ks + wave * (LPW * 1024u), *vd = (lds_u8 *)vs + wave * (LPW * 1024u);
        const uint32_t np = vis % kTile, back = np * rowb;
        const auto rk = range(static_cast<const uint8_t *>(a.kn) + nbase, a.nnew * rowb);
        const auto rv = range(static_cast<const uint8_t *>(a.vn) + nbase, a.nnew * rowb);
#pragma unroll
        for (int i = 0; i < LPW; ++i)
            if ((wave * LPW + i) * RPL + lane / CPR >= np) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rk, kd + 1024 * i, 16, koff[i] == kOob ? kOob : koff[i] - back, 0, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rv, vd + 1024 * i, 16, voff[i] == kOob ? kOob : voff[i] - back, 0, 0, 0);
            }
    };

    f32x16 o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    // scores in log2 units; the mask form keeps natural units (a mask of the
    // type's lowest value stays finite) and scales the difference
    float m = -INFINITY, l = 0.0f;
    const float mul = kMask ? 1.0f / a.scale : kLog2e / a.scale;

    // fragment offsets within a tile
    const uint32_t krow = uint32_t(lr) * RB;
    uint32_t vfrag;
    const uint32_t g16 = uint32_t(lane) >> 4, r16 = uint32_t(lane) & 15u;
    const uint32_t vrow = 4u * (g16 >> 1) + (r16 >> 2);
    vfrag = vrow * RB + (r16 & 1u) * 8u;
    const uint32_t vchunk = 2u * (g16 & 1u) + ((r16 & 3u) >> 1);   // of 32-dim block 0

    auto step = [&](uint32_t t, uint8_t *ks, uint8_t *vs, uint8_t *kn, uint8_t *vn) {
        __builtin_amdgcn_s_waitcnt((15 << 8) | (7 << 4));   // vmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint32_t key0 = t * kTile;
        float mk[kMask ? 32 : 1];
        if constexpr (kMask) {
            const uint32_t j = key0 + 4u * lg;
            const float *mrow = a.mask + uint64_t(qi) * total;
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                const uint32_t jj = j + 32u * (r >> 4) + 8u * ((r & 15) >> 2) + (r & 3);
                mk[r] = mrow[jj < total ? jj : total - 1];
            }
        }
        dma(t + 1, kn, vn);
        if (key0 >= wmax) return;
        f32x16 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const lds_u8 *p = (const lds_u8 *)ks + 32u * kb * RB + krow +
                                  ((uint32_t(2 * k + lg) ^ swz_k<RB>(lr)) * 16u);
                const u32x4 kf = *reinterpret_cast<const __attribute__((address_space(3))) u32x4 *>(p);
                s[kb] = mfma32<DT>(kf, qf[k], s[kb]);
            }
        }
        const bool full = key0 + kTile <= wmin;
        float mt = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float x = s[kb][r] * mul;
                if constexpr (kMask) x = x + mk[16 * kb + r];
                if (!full) x = key0 + 32u * kb + 8u * (r >> 2) + 4u * lg + (r & 3) < lim ? x : -INFINITY;
                s[kb][r] = x;
                mt = fmaxf(mt, x);
            }
        mt = max_half(mt);
        const float mn = fmaxf(m, mt);
        if (__any(mn > m)) {
            const float al = weight(kMask ? (m - mn) * kLog2e : m - mn);
            l *= al;
#pragma unroll
            for (int d = 0; d < DB; ++d) o[d] *= al;
            m = mn;
        }
        const float ms = DT == 6 && !kMask ? m - kPScale : m;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float x = s[kb][r] - ms;
                if constexpr (kMask) {
                    x *= kLog2e;
                    if constexpr (DT == 6) x += kPScale;
                }
                const float p = weight(x);
                l += p;
                s[kb][r] = p;
            }
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const int kb = st >> 1, hh = st & 1;
            u32x4 ph, pl;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t h, w;
                split2<DT>(s[kb][8 * hh + 2 * i], s[kb][8 * hh + 2 * i + 1], h, w);
                ph[i] = h;
                pl[i] = w;
            }
#pragma unroll
            for (int d = 0; d < DB; ++d) {
                const uint32_t c = (vchunk + 4u * d) ^ swz_v<RB>(vrow);
                const lds_u8 *p = (const lds_u8 *)vs + (32u * kb + 16u * hh) * RB + vfrag + c * 16u;
                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    reinterpret_cast<lds_i16x4 *>(const_cast<lds_u8 *>(p)));
                const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    reinterpret_cast<lds_i16x4 *>(const_cast<lds_u8 *>(p + 8u * RB)));
                const u32x4 vf = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                o[d] = mfma32<DT>(vf, ph, o[d]);
                o[d] = mfma32<DT>(vf, pl, o[d]);
            }
        }
    };
    if (t0 < t1) {
        dma(t0, k0s, v0s);
        for (uint32_t t = t0; t < t1; t += 2) {
            if (t == tmid) patch(k0s, v0s);
            step(t, k0s, v0s, k1s, v1s);
            if (t + 1 < t1) {
                if (t + 1 == tmid) patch(k1s, v1s);
                step(t + 1, k1s, v1s, k0s, v0s);
            }
        }
    }

    bool bad = false;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) bad = bad || !(fabsf(o[d][r]) <= 3.4028235e38f);
    const float lsum = l + __shfl_xor(l, 32, 64);
    const uint32_t planes = a.B * a.Hkv;
    __builtin_amdgcn_s_waitcnt((15 << 8) | (7 << 4));   // the last (empty) loads into LDS
    if (__syncthreads_or(bad)) {
        const uint32_t j0 = t0 * kTile, j1 = t1 * kTile < total ? t1 * kTile : total;
        for (uint32_t rr = r0 + wave; rr <= rl; rr += kThreads / 64)
            walk_row<DT>(a, plane, rr, vis, j0, j1, nsplit == 1, kMask ? 1.0f : kLog2e,
                         part + ((uint64_t(split) * planes + plane) * R + rr) * uint64_t(D + 2));
        return;
    }
    // O^T: lane holds dims 32 d + 8 (r/4) + 4 lg + r%4 of its row
    if (wr0 + lr >= R) return;
    if (nsplit == 1) {
        const float den = DT == 6 ? lsum * 0x1p-15f : lsum;
        const float inv = m == -INFINITY ? 0.0f : 1.0f / (den > 1e-30f ? den : 1e-30f);
        uint16_t *orow = static_cast<uint16_t *>(a.out) + (uint64_t(plane) * R + row) * D;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const uint32_t dim = 32 * d + 2 * r + 4 * lg;
                if (dim >= D) continue;
                uint16_t e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = (DT == 6 ? o[d][r + i] * 0x1p-15f : o[d][r + i]) * inv;
                    e[i] = DT == 7 ? uint16_t(__float_as_uint(v) >> 16) : f32_to_f16_bits(v);
                }
                *reinterpret_cast<uint2 *>(orow + dim) =
                    make_uint2(e[0] | (uint32_t(e[1]) << 16), e[2] | (uint32_t(e[3]) << 16));
            }
        return;
    }
    float *pp = part + ((uint64_t(split) * planes + plane) * R + row) * uint64_t(D + 2);
    const float un = DT == 6 ? 0x1p-15f : 1.0f;
    if (lg == 0) *reinterpret_cast<f32x2 *>(pp) = f32x2{m, lsum * un};
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const uint32_t dim = 32 * d + 8 * (r >> 2) + 4 * lg + (r & 3);
            if (dim < D) *reinterpret_cast<f32x2 *>(pp + 2 + dim) = f32x2{o[d][r] * un, o[d][r + 1] * un};
        }
}

template <int DT, int DB, bool kMask>
__global__ __launch_bounds__(kThreads, 2) void attn_valid_rows_kernel(const AttnValidArgs a,
                                                                      const uint32_t tiles,
                                                                      const uint32_t nsplit,
                                                                      float *__restrict__ part) {
    attn_valid_rows<DT, DB, kMask>(a, tiles, nsplit, part);
}

// -------------------------------------------------------- merged shares ----
// One thread per output value: every share's m and l of its row and its own
// accumulator, weighted in share order. kNat: m in natural units, else log2.
template <int DT, bool kNat>
__global__ __launch_bounds__(kThreads) void attn_valid_combine_kernel(const AttnValidArgs a,
                                                                      const uint32_t nsplit,
                                                                      const uint64_t values,
                                                                      const float *__restrict__ part) {
    const uint64_t i = uint64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= values) return;
    const uint32_t D = a.D;
    const uint64_t row = i / D, rows = values / D;
    const uint32_t c = uint32_t(i % D);
    const float *p0 = part + row * (D + 2);
    const uint64_t step = rows * (D + 2);
    constexpr uint32_t N = 8;
    float mc[N], lc[N], oc[N];
#pragma unroll
    for (uint32_t u = 0; u < N; ++u) {
        const float *p = p0 + (u < nsplit ? u : nsplit - 1) * step;
        mc[u] = p[0];
        lc[u] = p[1];
        oc[u] = p[2 + c];
    }
    float m = -INFINITY;
#pragma unroll
    for (uint32_t u = 0; u < N; ++u) m = fmaxf(m, mc[u]);
    for (uint32_t s = N; s < nsplit; ++s) m = fmaxf(m, p0[s * step]);
    auto w = [&](float x) { return weight(kNat ? (x - m) * kLog2e : x - m); };
    float x = 0.0f, l = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < N; ++u)
        if (u < nsplit) {
            const float ws = w(mc[u]);
            l = l + ws * lc[u];
            x = fmaf(ws, oc[u], x);
        }
    for (uint32_t s = N; s < nsplit; ++s) {
        const float ws = w(p0[s * step]);
        l = l + ws * p0[s * step + 1];
        x = fmaf(ws, p0[s * step + 2 + c], x);
    }
    st_elem<DT>(a.out, i, m == -INFINITY ? 0.0f : x / (l > 1e-30f ? l : 1e-30f));
}

int cus() {
    static const int n = [] {
        int dev = 0, c = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0)
            c = 256;
        return c;
    }();
    return n;
}

struct RowsPlan {
    uint32_t tiles, nsplit;
};

// Prompt rows: one workgroup a 128-row tile; fewer tiles than CUs share a
// tile's list among workgroups (at least 4 key tiles each).
RowsPlan rows_plan(uint32_t B, uint32_t H, uint32_t Hkv, uint32_t M, uint32_t past, uint32_t nnew) {
    RowsPlan p;
    const uint64_t R = uint64_t(H / Hkv) * M;
    p.tiles = uint32_t((R + kRowsWg - 1) / kRowsWg);
    const uint64_t wgs = uint64_t(B) * Hkv * p.tiles;
    const uint64_t kt = (uint64_t(past) + nnew + kTile - 1) / kTile;
    uint64_t ns = uint64_t(cus()) / wgs;
    if (ns > kt / 4) ns = kt / 4;
    if (ns > 64) ns = 64;
    p.nsplit = uint32_t(ns < 1 ? 1 : ns);
    return p;
}

template <int DT, bool kMask>
hipError_t run_rows(const AttnValidArgs &a, float *part, hipStream_t stream) {
    const RowsPlan p = rows_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew);
    const dim3 grid(p.tiles * a.B * a.Hkv * p.nsplit);
    const uint32_t db = a.D <= 64 ? 2 : (a.D + 31) / 32;
    if (db == 2)
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 2, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, part);
    else if (db == 3)
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 3, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, part);
    else
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 4, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, part);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.nsplit == 1) return e;
    const uint64_t values = uint64_t(a.B) * a.H * a.M * a.D;
    hipLaunchKernelGGL((attn_valid_combine_kernel<DT, kMask>), dim3(unsigned((values + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, stream, a, p.nsplit, values, part);
    return hipGetLastError();
}

}  // namespace

// More than 16 query rows a plane (a prompt), 16-bit operands with 16-byte
// rows, head_dim <= 128 (the accumulators of a wider head do not fit a wave's
// registers), every buffer within a 32-bit range. Up to 16 rows the loads of K
// and V bound the call, not the products.
bool attn_valid_rows_applies(const AttnValidArgs &a) {
    if ((a.dtype != 7 && a.dtype != 6) || a.D % 8 != 0 || a.D > 128) return false;
    const uint64_t R = uint64_t(a.H / a.Hkv) * a.M;
    if (R <= 16 || R > (1u << 30)) return false;
    uintptr_t al = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.out);
    if (a.past) al |= reinterpret_cast<uintptr_t>(a.kp) | reinterpret_cast<uintptr_t>(a.vp);
    if (a.nnew) al |= reinterpret_cast<uintptr_t>(a.kn) | reinterpret_cast<uintptr_t>(a.vn);
    if ((al & 15) != 0) return false;
    const uint64_t lim = 1ull << 31;
    if (uint64_t(a.past) * a.D * 2 >= lim || uint64_t(a.nnew) * a.D * 2 >= lim) return false;
    const RowsPlan p = rows_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew);
    return uint64_t(p.tiles) * a.B * a.Hkv * p.nsplit < lim &&
           uint64_t(a.B) * a.H * a.M * a.D / kThreads < lim;
}

size_t attn_valid_rows_scratch_bytes(uint32_t B, uint32_t H, uint32_t Hkv, uint32_t M, uint32_t past,
                                     uint32_t nnew, uint32_t D) {
    if (uint64_t(H / Hkv) * M <= 16 || D > 128) return 0;
    const RowsPlan p = rows_plan(B, H, Hkv, M, past, nnew);
    return p.nsplit == 1 ? 0 : size_t(p.nsplit) * B * H * M * (size_t(D) + 2) * sizeof(float);
}

hipError_t launch_attn_valid_rows(const AttnValidArgs &a, void *scratch, hipStream_t stream) {
    if (!attn_valid_rows_applies(a)) return hipErrorInvalidValue;
    float *part = static_cast<float *>(scratch);
    if (a.dtype == 7)
        return a.mask ? run_rows<7, true>(a, part, stream) : run_rows<7, false>(a, part, stream);
    return a.mask ? run_rows<6, true>(a, part, stream) : run_rows<6, false>(a, part, stream);
}

}  // namespace holo
