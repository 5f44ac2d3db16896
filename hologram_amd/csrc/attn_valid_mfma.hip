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
// (walk_rows); a share that ends finite held no such value.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

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

// Over the wavefront, in every lane: rotations within rows of 16, then max_quarter's
// exchanges.
template <int n>
__device__ __forceinline__ float row_ror(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + n, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, row_ror<8>(v));
    v = fmaxf(v, row_ror<4>(v));
    v = fmaxf(v, row_ror<2>(v));
    return max_quarter(fmaxf(v, row_ror<1>(v)));
}
__device__ __forceinline__ float wave_sum(float v) {
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(y[0]) + __uint_as_float(y[1]);
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

// n <= RN query rows from r on over list entries [j0, j1) by one wavefront, in the
// reference's scalar steps (the scores in the four sums of attn_valid.hip's walk):
// 64 keys at a time, a key per lane for the scores, then a column (or two) per
// lane for PV, key by key, entries past a row's limit left out. It runs for a
// share that holds a non-finite V. q and the weights pass through lds (RN (D + 64)
// floats of the wavefront's own), so that each K and V byte is read once for RN
// rows: a 509-row chunk after 1537 keys, 2 sequences of 32 heads over 8 of 128
// dims, takes 2.8 ms with an infinity in V (32 a row at a time, 3.9 on the general
// form, 0.06 without the infinity), 8 decode rows over 7002 keys 185 us (1276;
// 295), 64 rows after 200 keys 65 us (4.0 ms; 57). Bound by the issue of its few
// waves: four or eight K loads in flight instead of two are 5-15% slower.
// `single`: writes the output rows; else (m, l, acc) at pp, D + 2 floats a row, m
// times munit.
template <int DT, int RN>
__device__ __forceinline__ void walk_rows(const AttnValidArgs &a, const uint32_t plane, const uint32_t r,
                                          const uint32_t n, const uint32_t vis, const uint32_t j0,
                                          const uint32_t j1, const bool single, const float munit, float *pp,
                                          float *lds) {
    constexpr uint32_t kEs = DT == 8 ? 4 : 2, E = 16 / kEs;   // elements of 16 bytes
    const uint32_t lane = threadIdx.x & 63, D = a.D, R = a.H / a.Hkv * a.M, total = vis + a.nnew;
    const uint64_t q0 = (uint64_t(plane) * R + r) * D;
    const uint64_t p0 = uint64_t(plane) * a.past, n0 = uint64_t(plane) * a.nnew;
    float *const qs = lds, *const ps = lds + RN * D;
    auto row = [&](int i) { return uint32_t(i) < n ? uint32_t(i) : n - 1; };   // past n: the last one again
    for (uint32_t x = lane; x < RN * D; x += 64) qs[x] = ld_elem<DT>(a.q, q0 + uint64_t(row(int(x / D))) * D + x % D);
    uint32_t lim[RN], mrow[RN], most = 0, least = total;
    float m[RN], l[RN], acc[RN][2];
#pragma unroll
    for (int i = 0; i < RN; ++i) {
        const uint32_t qi = uniform((r + row(i)) % a.M);
        mrow[i] = qi;
        lim[i] = uniform(a.mask ? total : vis + (qi + 1 < a.nnew ? qi + 1 : a.nnew));
        most = lim[i] > most ? lim[i] : most;
        least = lim[i] < least ? lim[i] : least;
        m[i] = -INFINITY;
        l[i] = acc[i][0] = acc[i][1] = 0.0f;
    }
    const uint32_t end = j1 < most ? j1 : most;
    const uint32_t c0 = lane < D ? lane : 0, c1 = lane + 64 < D ? lane + 64 : 0;   // (columns past D: not stored)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
    for (uint32_t jb = j0; jb < end; jb += 64) {
        const uint32_t j = jb + lane < end ? jb + lane : end - 1;
        const uint8_t *k = static_cast<const uint8_t *>(j < vis ? a.kp : a.kn) + (j < vis ? p0 + j : n0 + j - vis) * D * kEs;
        float d[RN][4] = {}, mk[RN];
        if (a.mask)
#pragma unroll
            for (int i = 0; i < RN; ++i) mk[i] = a.mask[uint64_t(mrow[i]) * total + j];
        auto dims = [&](u32x4 w, uint32_t c) {
            float kv[E];
#pragma unroll
            for (uint32_t e = 0; e < E; ++e) {
                if constexpr (DT == 8) kv[e] = __uint_as_float(w[e]);
                else if constexpr (DT == 7) kv[e] = __uint_as_float(e & 1 ? w[e / 2] & 0xFFFF0000u : w[e / 2] << 16);
                else kv[e] = float(__builtin_bit_cast(_Float16, uint16_t(w[e / 2] >> (16 * (e & 1)))));
            }
#pragma unroll
            for (int i = 0; i < RN; ++i)
#pragma unroll
                for (uint32_t e = 0; e < E; e += 4) {
                    const f32x4 qv = *reinterpret_cast<const f32x4 *>(qs + i * D + c + e);
#pragma unroll
                    for (int t = 0; t < 4; ++t) d[i][t] = fmaf(qv[t], kv[e + t], d[i][t]);
                }
        };
        uint32_t c = 0;
#pragma unroll 1
        for (; c + 2 * E <= D; c += 2 * E) {   // two loads in flight
            u32x4 w[2];
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) w[u] = *reinterpret_cast<const u32x4 *>(k + (c + u * E) * kEs);
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) dims(w[u], c + u * E);
        }
#pragma unroll 1
        for (; c < D; c += E) dims(*reinterpret_cast<const u32x4 *>(k + c * kEs), c);
#pragma unroll
        for (int i = 0; i < RN; ++i) {
            float s = ((d[i][0] + d[i][1]) + (d[i][2] + d[i][3])) / a.scale;
            if (a.mask) s = s + mk[i];
            if (jb + lane >= end || j >= lim[i]) s = -INFINITY;
            const float mn = fmaxf(m[i], wave_max(s));
            float p = 0.0f, al = 1.0f;
            if (mn != -INFINITY) {
                p = s == -INFINITY ? 0.0f : exp_det(s - mn);
                al = m[i] == -INFINITY ? 0.0f : exp_det(m[i] - mn);
            }
            l[i] = l[i] * al + wave_sum(p);
            m[i] = mn;
            acc[i][0] *= al;
            acc[i][1] *= al;
            ps[i * 64 + lane] = p;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        auto pv = [&](auto whole) {   // every row sees the whole block, or key by key
#pragma unroll 1
            for (uint32_t t0 = 0; t0 < 64 && jb + t0 < end; t0 += 16) {
                float v[16][2];
#pragma unroll
                for (uint32_t t = 0; t < 16; ++t) {
                    const uint32_t y = jb + t0 + t < end ? jb + t0 + t : end - 1;
                    const void *vb = y < vis ? a.vp : a.vn;
                    const uint64_t v0 = (y < vis ? p0 + y : n0 + y - vis) * D;
                    v[t][0] = ld_elem<DT>(vb, v0 + c0);
                    v[t][1] = ld_elem<DT>(vb, v0 + c1);
                }
#pragma unroll
                for (int i = 0; i < RN; ++i)
#pragma unroll
                    for (uint32_t u = 0; u < 16; u += 4) {
                        const f32x4 w = *reinterpret_cast<const f32x4 *>(ps + i * 64 + t0 + u);
#pragma unroll
                        for (uint32_t t = 0; t < 4; ++t) {
                            const uint32_t y = jb + t0 + u + t;
                            const bool in = decltype(whole)::value || (y < end && y < lim[i]);
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const float x = fmaf(w[t], v[u + t][h], acc[i][h]);
                                acc[i][h] = in ? x : acc[i][h];
                            }
                        }
                    }
            }
        };
        if (jb + 64 <= least && jb + 64 <= end) pv(std::true_type{});
        else pv(std::false_type{});
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
#pragma unroll
    for (int i = 0; i < RN; ++i) {
        if (uint32_t(i) >= n) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t c = lane + 64u * h;
            if (c >= D) continue;
            const float den = l[i] > 1e-30f ? l[i] : 1e-30f;
            if (single) st_elem<DT>(a.out, q0 + uint64_t(i) * D + c, m[i] == -INFINITY ? 0.0f : acc[i][h] / den);
            else pp[i * (D + 2) + 2 + c] = acc[i][h];
        }
        if (!single && lane == 0) {
            pp[i * (D + 2)] = m[i] * munit;
            pp[i * (D + 2) + 1] = l[i];
        }
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
// 8 kv heads of 128 dims, 2 sequences, after 1537 cached keys, bf16: 59 us (505
// TFLOP/s) against 3.88 ms for the scalar walk's kernel. A tile holds 64
// consecutive list entries wherever the past ends, so past || new gives the
// bits of the same keys precatenated.
// A launch that would leave most CUs idle gives a tile's rows to 2, 4 or 8
// workgroups (srows rows each): all load K and V, but only the waves that hold a
// workgroup's rows compute, and it walks and stores its rows only, with the same bits.
// 64 rows x 32 heads over 8 after 200 keys, 128 dims: 14.1 -> 12.9 us, 395 -> 65
// with an infinity in V (56 and 57 on the general form); 100 f16 rows with a mask
// after 412 keys 31.4 -> 22.4 (1230 -> 317); 8 rows after 64 keys 7.7 -> 7.9 (48 -> 28).
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
                                                const uint32_t nsplit, const uint32_t slices,
                                                const uint32_t srows, float *__restrict__ part) {
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
    const uint32_t split = id % nsplit, rest = id / nsplit / slices;
    const uint32_t slice = id / nsplit % slices;   // its waves' rows are this workgroup's
    const uint32_t tile = tiles - 1 - rest % tiles, plane = rest / tiles;
    const uint32_t r0 = tile * kRowsWg;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const uint32_t wave = uniform(uint32_t(tid) >> 6);
    const uint32_t rs = slice * srows, re = rs + srows;
    const bool mine = 32 * wave < re && 32 * wave + 32 > rs;

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
        asm volatile("" ::: "memory");
        // this tile's loads, and this wave's reads of the buffers loaded into next
        __builtin_amdgcn_s_waitcnt(7 << 4);   // vmcnt(0) lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint32_t key0 = t * kTile;
        float mk[kMask ? 32 : 1];
        if (kMask && mine) {
            const uint32_t j = key0 + 4u * lg;
            const float *mrow = a.mask + uint64_t(qi) * total;
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                const uint32_t jj = j + 32u * (r >> 4) + 8u * ((r & 15) >> 2) + (r & 3);
                mk[r] = mrow[jj < total ? jj : total - 1];
            }
        }
        dma(t + 1, kn, vn);
        if (key0 >= wmax || !mine) return;
        f32x16 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const lds_u8 *p = (const lds_u8 *)ks + 32u * kb * RB + krow +
                                  ((uint32_t(2 * k + lg) ^ swz_k<RB>(lr)) * 16u);
                const u32x4 kf = *reinterpret_cast<const __attribute__((address_space(3))) u32x4 *>(p);
                s[kb] = mfma32<DT>(kf, qf[k], s[kb]);
            }
        float mt = -INFINITY;
        auto scores = [&](auto full) {   // every row of the wave sees the whole tile, or masked
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float x = s[kb][r] * mul;
                    if constexpr (kMask) x = x + mk[16 * kb + r];
                    if constexpr (!decltype(full)::value)
                        x = key0 + 32u * kb + 8u * (r >> 2) + 4u * lg + (r & 3) < lim ? x : -INFINITY;
                    s[kb][r] = x;
                    mt = fmaxf(mt, x);
                }
        };
        if (key0 + kTile <= wmin) scores(std::true_type{});
        else scores(std::false_type{});
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
        float *const own = reinterpret_cast<float *>(wave == 0 ? k0s : wave == 1 ? v0s : wave == 2 ? k1s : v1s);
#pragma unroll 1
        for (uint32_t rr = r0 + rs + 4 * wave; rr < r0 + re && rr <= rl; rr += 4 * (kThreads / 64))
            walk_rows<DT, 4>(a, plane, rr, rl - rr < 4 ? rl - rr + 1 : 4, vis, j0, j1, nsplit == 1,
                             kMask ? 1.0f : kLog2e,
                             part + ((uint64_t(split) * planes + plane) * R + rr) * uint64_t(D + 2), own);
        return;
    }
    // O^T: lane holds dims 32 d + 8 (r/4) + 4 lg + r%4 of its row
    if (wr0 + lr >= R || 32 * wave + lr < rs || 32 * wave + lr >= re) return;
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
                                                                      const uint32_t slices, const uint32_t srows,
                                                                      float *__restrict__ part) {
    attn_valid_rows<DT, DB, kMask>(a, tiles, nsplit, slices, srows, part);
}

// --------------------------------------------- few rows (a decode step) ----
// A workgroup takes 16 of a plane's query rows over a share of the list; its
// four wavefronts take the share's KB-key blocks in turn (KB 32, f32 16) and
// merge in LDS. Each byte of K and V comes from memory once, straight into
// registers, the next block's while this one is computed:
//     S^T[KB keys x 16 rows] = K . Q^T   16x16x32 (f32 16x16x4); a lane holds
//         16 bytes of key row lane % 16, chunk 4 s + lane / 16
//     O^T[D x 16 rows] += V^T . P^T      a lane holds CW columns of the keys
//         its scores belong to; 16-bit columns are turned into k-vectors with
//         byte permutes, f32 ones need no turning
// Loads are never behind a branch: a key past the list reads the list's last
// row (its score is masked).
// Bound by HBM: 32 heads over 8 kv heads of 128 dims, 8 sequences, 7002 keys,
// bf16 (229 MB, 289 read: up to two blocks past a wave's share): 52 us (4.4 TB/s;
// the kernel alone 47.5 us, 6.1 TB/s of what it reads) against
// 339 us for the scalar walk's kernels; 3500 f32 keys (235 MB): 51 against 192.
template <int DT, int DMAX>
struct FewShape {
    static constexpr int kEs = DT == 8 ? 4 : 2;
    static constexpr int MB = DT == 8 ? 1 : 2;           // 16-key groups a block
    static constexpr int KB = 16 * MB;
    static constexpr int NS = DMAX * kEs / 64;           // 64-byte steps of a K row
    static constexpr int NH = DT == 8 ? DMAX / 64 : 1;   // 16-byte column groups of V, f32
    static constexpr int CW = DT == 8 ? 4 : DMAX / 16;   // V columns a lane holds of a group
    static constexpr int VR = 4 * MB;                    // V rows a lane holds
    static constexpr int NC = DT == 8 ? 4 * NH : CW;     // accumulator tiles
};

template <int DT, int DMAX, bool kMask>
__device__ __forceinline__ void attn_valid_few(const AttnValidArgs &a, const uint32_t tiles,
                                               const uint32_t nsplit, float *__restrict__ part) {
    using S = FewShape<DT, DMAX>;
    constexpr int KB = S::KB, MB = S::MB, NS = S::NS, NH = S::NH, CW = S::CW, VR = S::VR, NC = S::NC;
    constexpr uint32_t kEs = S::kEs;
    typedef uint32_t vvec __attribute__((ext_vector_type(CW * S::kEs / 4)));
    __shared__ float red_m[4][16], red_l[4][16];
    __shared__ __attribute__((aligned(16))) float red_o[4][16][DMAX];
    const uint32_t D = a.D, R = a.H / a.Hkv * a.M, planes = a.B * a.Hkv;
    const uint32_t split = blockIdx.x % nsplit, rest = blockIdx.x / nsplit;
    const uint32_t tile = rest % tiles, plane = rest / tiles;
    const uint32_t r0 = tile * 16, nr = R - r0 < 16 ? R - r0 : 16;
    const int tid = threadIdx.x, lane = tid & 63, q16 = lane & 15, g = lane >> 4;
    const uint32_t wave = uniform(uint32_t(tid) >> 6);

    uint32_t vis = kMask ? a.past : read_u32_le(a.valid_len);
    vis = uniform(vis < a.past ? vis : a.past);
    const uint32_t total = vis + a.nnew;
    auto limit = [&](uint32_t r) -> uint32_t {
        const uint32_t qi = r % a.M;
        return kMask ? total : vis + (qi + 1 < a.nnew ? qi + 1 : a.nnew);
    };
    const uint32_t rl = r0 + nr - 1;
    const uint32_t most = r0 / a.M == rl / a.M ? limit(rl) : total;
    const uint32_t least = r0 / a.M == rl / a.M ? limit(r0) : limit(0);
    const uint32_t nb = (most + KB - 1) / KB, per = (nb + nsplit - 1) / nsplit;
    const uint32_t b0 = split * per < nb ? split * per : nb, b1 = b0 + per < nb ? b0 + per : nb;
    const uint32_t row = uint32_t(q16) < nr ? r0 + q16 : rl;   // this lane column's query row
    const uint32_t lim = limit(row), qi = row % a.M;

    const uint32_t rowb = D * kEs;
    const uint8_t *kp = static_cast<const uint8_t *>(a.kp) + uint64_t(plane) * a.past * rowb;
    const uint8_t *vp = static_cast<const uint8_t *>(a.vp) + uint64_t(plane) * a.past * rowb;
    const uint8_t *kn = static_cast<const uint8_t *>(a.kn) + uint64_t(plane) * a.nnew * rowb;
    const uint8_t *vn = static_cast<const uint8_t *>(a.vn) + uint64_t(plane) * a.nnew * rowb;
    const bool whole = D == DMAX;      // else chunks and columns past D read the row's first, as zeros

    struct Blk {
        u32x4 k[MB][NS];
        vvec v[VR][NH];
        float m[kMask ? 4 * MB : 1];
    };
    auto load = [&](uint32_t b, Blk &o) {
        const uint32_t key0 = b * KB;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            uint32_t j = key0 + 16 * mb + q16;
            j = j < total ? j : total - 1;
            const uint8_t *p = j < vis ? kp + uint64_t(j) * rowb : kn + uint64_t(j - vis) * rowb;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint32_t off = 64u * s + 16u * g;
                const u32x4 *src = reinterpret_cast<const u32x4 *>(p + (whole || off < rowb ? off : 0u));
                o.k[mb][s] = DT == 8 ? *src : __builtin_nontemporal_load(src);
            }
        }
#pragma unroll
        for (int i = 0; i < VR; ++i) {
            uint32_t j = key0 + 16 * (i >> 2) + 4 * g + (i & 3);
            j = j < total ? j : total - 1;
            const uint8_t *p = j < vis ? vp + uint64_t(j) * rowb : vn + uint64_t(j - vis) * rowb;
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const uint32_t off = (64u * h + uint32_t(CW * q16)) * kEs;
                const vvec *src = reinterpret_cast<const vvec *>(p + (whole || off < rowb ? off : 0u));
                o.v[i][h] = DT == 8 ? *src : __builtin_nontemporal_load(src);
            }
        }
        if constexpr (kMask) {
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) {
                const uint32_t j = key0 + 16 * (r >> 2) + 4 * g + (r & 3);
                o.m[r] = a.mask[uint64_t(qi) * total + (j < total ? j : total - 1)];
            }
        }
    };

    u32x4 qf[NS];
    {
        const uint8_t *p = static_cast<const uint8_t *>(a.q) + (uint64_t(plane) * R + row) * rowb;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint32_t off = 64u * s + 16u * g;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(p + (whole || off < rowb ? off : 0u));
            qf[s] = whole || off < rowb ? v : u32x4{0, 0, 0, 0};
        }
    }
    f32x4 o[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.0f;
    const float mul = kMask ? 1.0f / a.scale : kLog2e / a.scale;

    auto compute = [&](uint32_t b, Blk &x) {
        const uint32_t key0 = b * KB;
        if (!whole) {   // keys' chunks past D: zeros (they multiply zeros of Q, and must be finite)
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (64u * s + 16u * g >= rowb)
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) x.k[mb][s] = u32x4{0, 0, 0, 0};
        }
        f32x4 sc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            sc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (DT == 8) {
                // 32 dims at a time, in four sums of 8 products: the roundings of one
                // chain made the f32 result's error 1.3-1.8 times the element-wise
                // walk's, of four chains up to 1.035 over few keys; 0.75-0.97 so
#pragma unroll
                for (int s0 = 0; s0 < NS; s0 += 2) {
                    f32x4 part[4] = {};
#pragma unroll
                    for (int s = s0; s < s0 + 2; ++s)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                __uint_as_float(x.k[mb][s][i]), __uint_as_float(qf[s][i]), part[i], 0, 0, 0);
                    sc[mb] += (part[0] + part[1]) + (part[2] + part[3]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < NS; ++s) sc[mb] = mfma16<DT>(x.k[mb][s], qf[s], sc[mb]);
            }
        }
        const bool full = key0 + KB <= least;
        float p[4 * MB], mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4 * MB; ++r) {
            float v = sc[r >> 2][r & 3] * mul;
            if constexpr (kMask) v = v + x.m[r];
            if (!full) v = key0 + 16 * (r >> 2) + 4 * g + (r & 3) < lim ? v : -INFINITY;
            p[r] = v;
            mt = fmaxf(mt, v);
        }
        mt = max_quarter(mt);
        const float mn = fmaxf(m, mt);
        if (__any(mn > m)) {
            const float al = weight(kMask ? (m - mn) * kLog2e : m - mn);
            l *= al;
#pragma unroll
            for (int c = 0; c < NC; ++c) o[c] *= al;
            m = mn;
        }
#pragma unroll
        for (int r = 0; r < 4 * MB; ++r) {
            float v = p[r] - m;
            if constexpr (kMask) v *= kLog2e;
            // f32: the score times mul without a rounding of its own (a masked or
            // non-finite one as it stands)
            else if constexpr (DT == 8) v = p[r] > -INFINITY && p[r] < INFINITY ? fmaf(sc[r >> 2][r & 3], mul, -m) : v;
            if constexpr (DT == 6) v += kPScale;
            p[r] = weight(v);
            l += p[r];
        }
        if constexpr (DT == 8) {
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[4 * h + c] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            __uint_as_float(x.v[e][h][c]), p[e], o[4 * h + c], 0, 0, 0);
        } else {
            u32x4 ph, pl;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t hi, lo;
                split2<DT>(p[(2 * i) % (4 * MB)], p[(2 * i + 1) % (4 * MB)], hi, lo);
                ph[i] = hi;
                pl[i] = lo;
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                // column c of the lane's eight rows
                const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
                u32x4 vf;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    vf[i] = __builtin_amdgcn_perm(x.v[(2 * i + 1) % VR][0][c >> 1], x.v[(2 * i) % VR][0][c >> 1], sel);
                o[c] = mfma16<DT>(vf, ph, o[c]);
                o[c] = mfma16<DT>(vf, pl, o[c]);
            }
        }
    };

    {   // two blocks in registers: one computed while the other loads
        Blk x, y;
        uint32_t b = b0 + wave;
        if (b < b1) {
            load(b, x);
            for (; b < b1; b += 8) {
                load(b + 4, y);
                compute(b, x);
                load(b + 8, x);
                if (b + 4 < b1) compute(b + 4, y);
            }
        }
    }

    // the four wavefronts' states; O^T: o[c] holds row lane % 16, dims
    // CW (4 g + e) + c (+ 64 h)
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) {
        red_m[wave][q16] = m;
        red_l[wave][q16] = l;
    }
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < CW; ++c) red_o[wave][q16][64 * h + CW * (4 * g + e) + c] = o[CW * h + c][e];
    __syncthreads();
    constexpr int kOut = 16 * DMAX / kThreads;
    float res[kOut], ms[kOut], ls[kOut];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
        const uint32_t idx = uint32_t(tid) + kThreads * i, rr = idx / DMAX, c = idx % DMAX;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) mx = fmaxf(mx, red_m[w][rr]);
        float x = 0.0f, lt = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float d = red_m[w][rr] - mx;
            const float wt = weight(kMask ? d * kLog2e : d);
            lt = lt + wt * red_l[w][rr];
            x = fmaf(wt, red_o[w][rr][c], x);
        }
        bad = bad || (rr < nr && c < D && !(fabsf(x) <= 3.4028235e38f));
        const float un = DT == 6 ? 0x1p-15f : 1.0f;
        res[i] = x * un;
        ms[i] = mx;
        ls[i] = lt * un;
    }
    if (__syncthreads_or(bad)) {
        const uint32_t j0 = b0 * KB, j1 = b1 * KB < total ? b1 * KB : total;
        const uint32_t rr = r0 + 4 * wave;
        if (rr <= rl)
            walk_rows<DT, 4>(a, plane, rr, rl - rr < 4 ? rl - rr + 1 : 4, vis, j0, j1, nsplit == 1,
                             kMask ? 1.0f : kLog2e,
                             part + ((uint64_t(split) * planes + plane) * R + rr) * uint64_t(D + 2), &red_o[wave][0][0]);
        return;
    }
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
        const uint32_t idx = uint32_t(tid) + kThreads * i, rr = idx / DMAX, c = idx % DMAX;
        if (rr >= nr || c >= D) continue;
        if (nsplit == 1) {
            const float v = ms[i] == -INFINITY ? 0.0f : res[i] / (ls[i] > 1e-30f ? ls[i] : 1e-30f);
            st_elem<DT>(a.out, (uint64_t(plane) * R + r0 + rr) * D + c, v);
        } else {
            float *pp = part + ((uint64_t(split) * planes + plane) * R + r0 + rr) * uint64_t(D + 2);
            pp[2 + c] = res[i];
            if (c == 0) *reinterpret_cast<f32x2 *>(pp) = f32x2{ms[i], ls[i]};
        }
    }
}

template <int DT, int DMAX, bool kMask>
__global__ __launch_bounds__(kThreads, 2) void attn_valid_few_kernel(const AttnValidArgs a,
                                                                     const uint32_t tiles,
                                                                     const uint32_t nsplit,
                                                                     float *__restrict__ part) {
    attn_valid_few<DT, DMAX, kMask>(a, tiles, nsplit, part);
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
#pragma unroll 8
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
#pragma unroll 8
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

struct Shares {
    uint32_t tiles, nsplit;
};

// The list of a tile of rows is cut so that every CU holds `per_cu` workgroups,
// in shares of at least `keys` keys.
Shares shares(uint32_t B, uint32_t H, uint32_t Hkv, uint32_t M, uint32_t past, uint32_t nnew, uint32_t rows,
              uint32_t keys, uint32_t per_cu) {
    Shares p;
    const uint64_t R = uint64_t(H / Hkv) * M;
    p.tiles = uint32_t((R + rows - 1) / rows);
    const uint64_t wgs = uint64_t(B) * Hkv * p.tiles;
    uint64_t ns = uint64_t(per_cu) * cus() / wgs;
    const uint64_t most = (uint64_t(past) + nnew) / keys;
    if (ns > most) ns = most;
    if (ns > 128) ns = 128;
    p.nsplit = uint32_t(ns < 1 ? 1 : ns);
    return p;
}

// The plan within the general form's scratch: a call asks for what its sizes ask
// for, so neither its bits nor what it may grow depend on what ran before it or
// on a capture. Few rows always fit; of 60 drawn prompts five would gain from
// more shares, 1.1 times as fast and one 1.8.
Shares within(Shares p, const AttnValidArgs &a) {
    const uint64_t one = uint64_t(a.B) * a.H * a.M * (uint64_t(a.D) + 2) * sizeof(float);
    const uint64_t most = attn_valid_scratch_bytes(a.B, a.H, a.Hkv, a.M, a.past, a.nnew, a.D) / one;
    if (p.nsplit > most) p.nsplit = uint32_t(most < 1 ? 1 : most);
    return p;
}

// Prompt rows: one workgroup a 128-row tile, at least 4 key tiles a share.
Shares rows_plan(uint32_t B, uint32_t H, uint32_t Hkv, uint32_t M, uint32_t past, uint32_t nnew) {
    return shares(B, H, Hkv, M, past, nnew, kRowsWg, 4 * kTile, 1);
}
// Few rows: a share is at least a block for each of the four wavefronts.
Shares few_plan(uint32_t B, uint32_t H, uint32_t Hkv, uint32_t M, uint32_t past, uint32_t nnew) {
    return shares(B, H, Hkv, M, past, nnew, 16, 128, 2);
}

template <int DT, bool kMask>
hipError_t combine(const AttnValidArgs &a, uint32_t nsplit, const float *part, hipStream_t stream) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || nsplit == 1) return e;
    const uint64_t values = uint64_t(a.B) * a.H * a.M * a.D;
    hipLaunchKernelGGL((attn_valid_combine_kernel<DT, kMask>), dim3(unsigned((values + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, stream, a, nsplit, values, part);
    return hipGetLastError();
}

template <int DT, bool kMask>
hipError_t run_few(const AttnValidArgs &a, float *part, hipStream_t stream) {
    const Shares p = within(few_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew), a);
    const dim3 grid(p.tiles * a.B * a.Hkv * p.nsplit);
    if (a.D <= 64)
        hipLaunchKernelGGL((attn_valid_few_kernel<DT, 64, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, part);
    else
        hipLaunchKernelGGL((attn_valid_few_kernel<DT, 128, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, part);
    return combine<DT, kMask>(a, p.nsplit, part, stream);
}

template <int DT, bool kMask>
hipError_t run_rows(const AttnValidArgs &a, float *part, hipStream_t stream) {
    const Shares p = within(rows_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew), a);
    // rows a workgroup: halved while the workgroups still fit the CUs one to one;
    // 16 keep the walk's four waves busy (four rows each)
    const uint32_t wgs = p.tiles * a.B * a.Hkv * p.nsplit, n = uint32_t(cus());
    uint32_t srows = kRowsWg;
    while (srows > 16 && 2 * (kRowsWg / srows) * wgs <= n) srows /= 2;
    const uint64_t R = uint64_t(a.H / a.Hkv) * a.M;
    const uint32_t slices = uint32_t(((R < kRowsWg ? R : kRowsWg) + srows - 1) / srows);
    const dim3 grid(wgs * slices);
    const uint32_t db = a.D <= 64 ? 2 : (a.D + 31) / 32;
    if (db == 2)
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 2, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, slices, srows, part);
    else if (db == 3)
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 3, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, slices, srows, part);
    else
        hipLaunchKernelGGL((attn_valid_rows_kernel<DT, 4, kMask>), grid, dim3(kThreads), 0, stream, a,
                           p.tiles, p.nsplit, slices, srows, part);
    return combine<DT, kMask>(a, p.nsplit, part, stream);
}

}  // namespace

// Which form takes a call. Both: head_dim <= 128 (the accumulators of a wider
// head do not fit a wave's registers) with 16-byte rows and operands. 16-bit
// operands of more than 16 rows a plane take the prompt form: there the
// products bound the call, up to 16 rows the loads of K and V do. f32 operands
// take the few-row form at any count, 16 rows a workgroup: the f32 matrix
// instructions bound it (300 rows x 32 heads over 8 kv heads of 128 dims, 2
// sequences, 700 cached keys: 116 us, 1363 with the scalar walk).
enum class Form { none, few, rows };

static Form form_of(const AttnValidArgs &a) {
    const bool f32 = a.dtype == 8;
    if ((!f32 && a.dtype != 7 && a.dtype != 6) || a.D % (f32 ? 4 : 8) != 0 || a.D > 128) return Form::none;
    if (!(kLog2e / a.scale <= 3.4e38f)) return Form::none;   // scores are multiplied by it
    const uint64_t R = uint64_t(a.H / a.Hkv) * a.M, lim = 1ull << 31;
    uintptr_t al = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.out);
    if (a.past) al |= reinterpret_cast<uintptr_t>(a.kp) | reinterpret_cast<uintptr_t>(a.vp);
    if (a.nnew) al |= reinterpret_cast<uintptr_t>(a.kn) | reinterpret_cast<uintptr_t>(a.vn);
    if ((al & 15) != 0 || uint64_t(a.past) + a.nnew > (1u << 30)) return Form::none;
    const bool rows = !f32 && R > 16;
    // the prompt form reads through 32-bit buffer ranges
    if (rows && (R > (1u << 30) || uint64_t(a.past) * a.D * 2 >= lim || uint64_t(a.nnew) * a.D * 2 >= lim))
        return Form::none;
    const Shares p = rows ? rows_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew)
                          : few_plan(a.B, a.H, a.Hkv, a.M, a.past, a.nnew);
    if (uint64_t(p.tiles) * a.B * a.Hkv * p.nsplit >= lim || uint64_t(a.B) * a.H * a.M * a.D / kThreads >= lim)
        return Form::none;
    return rows ? Form::rows : Form::few;
}

bool attn_valid_mfma_applies(const AttnValidArgs &a) { return form_of(a) != Form::none; }

template <int DT>
static hipError_t run_form(const AttnValidArgs &a, Form f, float *part, hipStream_t stream) {
    if constexpr (DT != 8)
        if (f == Form::rows)
            return a.mask ? run_rows<DT, true>(a, part, stream) : run_rows<DT, false>(a, part, stream);
    return a.mask ? run_few<DT, true>(a, part, stream) : run_few<DT, false>(a, part, stream);
}

hipError_t launch_attn_valid_mfma(const AttnValidArgs &a, void *scratch, hipStream_t stream) {
    const Form f = form_of(a);
    if (f == Form::none) return hipErrorInvalidValue;
    float *part = static_cast<float *>(scratch);
    switch (a.dtype) {
        case 7: return run_form<7>(a, f, part, stream);
        case 6: return run_form<6>(a, f, part, stream);
        default: return run_form<8>(a, f, part, stream);
    }
}

}  // namespace holo
