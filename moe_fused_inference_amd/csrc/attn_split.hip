// attn_split.hip -- decode attention over the FP8 cache, split along the
// context: the path of attn.hip's entries for several tokens over a long cache
// (their contract, position rule, byte codec and dispatch are there).
//
//   attn_split_kernel  workgroup (split s, kv head g, row group): the split's
//                      positions against up to 48 query rows (tokens x heads
//                      of the kv head), a wave taking every fourth unit of 32
//                      positions with its own running softmax; the four
//                      waves' sums meet in LDS -> one record (reference, sum,
//                      128 column sums) per query row and split.
//   attn_split_merge_kernel  workgroup (query head, token): merges the row's
//                      records (am::merge_head) to o and / or its MXFP4 rows.
//
// The number of splits is fixed by the host from max_pos (about one round of
// workgroups), but a split's positions are an equal share of the context that
// dpos gives, so a short context in a large cache fills the chip as well.
//
// What bounds it is VALU work (the codec, the softmax) and, at short contexts,
// one memory latency; what the layout does about it:
//  * Both products are computed transposed, S^T = K Q^T and O^T = V^T P^T: the
//    MFMA leaves a lane with four positions of each of two 16-position tiles
//    of one query, which is the lane's B operand of the second product as it
//    stands, so P passes through no LDS and no barrier; a query's softmax
//    state is one lane's.  (Any assignment of positions or head dimensions to
//    the reduction index will do as long as both operands use it.)
//  * K rows load as 16 bytes a lane, V rows as 8 (whole 128-byte rows per
//    instruction): lane l holds columns 8 l .. 8 l + 7 of V, and column tile c
//    of the product is the columns 8 l + c.
//  * Codec: a byte of exponent 0 (m * 2^-6) has a normal E4M3 code of the same
//    value, found for four bytes at once with one byte permute as the table;
//    then the hardware's OCP conversion gives two values per instruction, about
//    3 instructions a byte and no LDS table.  Bytes of exponent 15, which the
//    codec reads as 56 (8 + m) and a cache holds only for |v| >= 240, send the
//    wave's unit through a longer path.
//  * In the second product V is bf16 (every codec value is) and P is three bf16
//    parts, whose sum is the fp32 probability at any size: one score far above
//    the others leaves the others' sum.  (Two fp16 parts, a third of the MFMAs
//    and a few conversions less, took 134 us of the 136 below, but cut a
//    probability off at 2^-31 of its row's largest: 65520 scores e^17.5 below
//    one, of values 448 and 2^-6, were wrong by 1e-4, and are by 7e-7.)  exp is
//    the hardware's exp2 of fma(s, log2(e) / sqrt(D), -m), with m kept in that
//    base so that a row's terms and the merge agree on it.
//  * At most three row tiles a workgroup: their accumulators, a unit's operands
//    and the next unit's bytes fit 256 registers, two waves per SIMD.  (Five
//    tiles decode each byte once for 72 rows, but past 256 registers the
//    accumulators move between register files at every step: 37 us against 25
//    at 9 tokens and 23001 positions.)
// Measured on MI355X (32 / 4 heads, the raw scores kept, four layers, each with
// its KV write, in a graph): 9 tokens over 23001 positions 243 us by chunks, 136
// here; relative error against 64 bits 1.9e-6 and 2.1e-7.
#include "attn_merge.h"
#include "attn_split.h"
#include "kv_codec.h"
#include "mx_device.h"
#include "mx_host.h"

namespace {

using am::kD;
using am::kPart;

constexpr int kUnit = 32;      // positions per wave and step
constexpr float kSlack = 8.0f;         // a term is at most 2^8
constexpr float kWide = 262144.0f;     // a reference past it: an exponent's rounding is up to 2^-6 and more
constexpr float kNone = -3e38f;        // the reference of a row that has seen nothing: exp2(-inf - kNone) = 0
constexpr int kMaxRT = 3;      // 16-row tiles per workgroup
constexpr int kLdsRow = kD + 8;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mx::v4f mfma_bf16(uint4 a, uint4 b, mx::v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
}

// Units per split for a context of n positions: equal shares in whole rounds of the four waves.
__device__ __forceinline__ int units_per_split(int n, int nsplit) {
    const int nu = (n + kUnit - 1) / kUnit;
    const int per = (nu + nsplit - 1) / nsplit;
    return max(4, (per + 3) & ~3);
}

// A unit's bytes as a lane loads them, by buffer loads relative to the
// workgroup's first position (rows past the cache read zeros; the V cache may
// start at any dword).
struct RawK {
    v4u k[2][2];   // [tile][half]: row 16 tile + l16, bytes 64 half + 16 lq ..
};
struct RawV {
    v2u v[8];          // position 4 lq + t (t < 4), 16 + 4 lq + t - 4: columns 8 l16 ..
};

__device__ __forceinline__ void load_k(RawK& r, __amdgpu_buffer_rsrc_t rk, uint32_t vo, uint32_t rs) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) r.k[t][j] = __builtin_amdgcn_raw_buffer_load_b128(rk, vo + 16 * t * rs + 64 * j, 0, 0);
}
__device__ __forceinline__ void load_v(RawV& r, __amdgpu_buffer_rsrc_t rv, uint32_t vo, uint32_t rs) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
        r.v[t] = __builtin_amdgcn_raw_buffer_load_b64(rv, vo + (16 * (t >> 2) + (t & 3)) * rs, 0, 0);
}

// The unit's MFMA operands: kd[tile][kt] (positions x 8 of the 32 dimensions
// of step kt), vd[c] (columns 8 l16 + c x 8 positions).
template <bool EXP15>
__device__ __forceinline__ void decode_k(const RawK& r, uint4 (&kd)[2][4], uint32_t& e15) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t w[4], f[4], o[8];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                w[d] = kv::ready<EXP15>(r.k[t][j][d], f[d], e15);
                o[2 * d] = kv::pair_of<false, EXP15>(w[d], f[d]);
                o[2 * d + 1] = kv::pair_of<true, EXP15>(w[d], f[d]);
            }
            kd[t][2 * j] = make_uint4(o[0], o[1], o[2], o[3]);
            kd[t][2 * j + 1] = make_uint4(o[4], o[5], o[6], o[7]);
        }
}
__device__ __forceinline__ void decode_k(const RawK& r, uint4 (&kd)[2][4]) {
    uint32_t e15 = 0;
    decode_k<false>(r, kd, e15);
    if (__ballot((e15 & 0x80808080u) != 0u)) {
        uint32_t none = 0;
        decode_k<true>(r, kd, none);
    }
}
template <bool EXP15>
__device__ __forceinline__ void decode_v(const RawV& r, uint4 (&vd)[8], uint32_t& e15) {
    uint32_t o[8][4];
#pragma unroll
    for (int t2 = 0; t2 < 4; ++t2) {   // positions 2 t2, 2 t2 + 1 of the lane's eight
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            uint32_t fa, fb;
            const uint32_t a = kv::ready<EXP15>(r.v[2 * t2][d], fa, e15), b = kv::ready<EXP15>(r.v[2 * t2 + 1][d], fb, e15);
            const uint32_t c01 = __builtin_amdgcn_perm(b, a, 0x05010400u), c23 = __builtin_amdgcn_perm(b, a, 0x07030602u);
            uint32_t f01 = 0, f23 = 0;
            if constexpr (EXP15) {
                f01 = __builtin_amdgcn_perm(fb, fa, 0x05010400u);
                f23 = __builtin_amdgcn_perm(fb, fa, 0x07030602u);
            }
            o[4 * d][t2] = kv::pair_of<false, EXP15>(c01, f01);
            o[4 * d + 1][t2] = kv::pair_of<true, EXP15>(c01, f01);
            o[4 * d + 2][t2] = kv::pair_of<false, EXP15>(c23, f23);
            o[4 * d + 3][t2] = kv::pair_of<true, EXP15>(c23, f23);
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) vd[c] = make_uint4(o[c][0], o[c][1], o[c][2], o[c][3]);
}
__device__ __forceinline__ void decode_v(const RawV& r, uint4 (&vd)[8]) {
    uint32_t e15 = 0;
    decode_v<false>(r, vd, e15);
    if (__ballot((e15 & 0x80808080u) != 0u)) {
        uint32_t none = 0;
        decode_v<true>(r, vd, none);
    }
}

// Eight fp32 terms as three bf16 parts each, whose sum each is (8 bits a part,
// rounded to nearest, the rest exact).
__device__ __forceinline__ void parts(float (&t)[8], uint4 (&p)[3]) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{t[2 * i], t[2 * i + 1]}), bf16x2_t));
            t[2 * i] -= __uint_as_float(o[i] << 16);
            t[2 * i + 1] -= __uint_as_float(o[i] & 0xFFFF0000u);
        }
        p[j] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// a * b rounded, minus c: not one fma.
__device__ __forceinline__ float mul_then_sub(float a, float b, float c) {
#pragma clang fp contract(off)
    const float ab = a * b;
    return ab - c;
}

// The maximum over the four lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ __forceinline__ float max_over_lq(float v) {
    {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_over_lq(float v) {
    {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

struct SplitArgs {
    const uint16_t* q;
    const uint8_t* kvk;
    const uint8_t* kvv;
    float* sc;
    float* part;
    const int32_t* dpos;
    int M, Hq, Hkv, lg, max_pos, nsplit;   // lg = log2(Hq / Hkv)
    int sc_vec;                            // sc rows are 16-byte aligned
    int fixed;                             // a split is 4 units whatever the context: max_pos has no more
    float c;                               // log2(e) / sqrt(D)
};

template <int RT>
__global__ __launch_bounds__(256, 2) void attn_split_kernel(SplitArgs a) {
    constexpr int R = 16 * RT;
    __shared__ __align__(16) uint16_t qs[RT > 1 ? R : 1][kLdsRow];
    __shared__ __align__(16) float mo[4][16][kD + 4];
    __shared__ float mm[4][16], ml[4][16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int g = blockIdx.y, r0 = blockIdx.z * R, G = 1 << a.lg;
    const int rows = a.M << a.lg;
    const uint32_t rs = (uint32_t)a.Hkv * kD;
    // the K / V rows from position 32 u on: lane offsets of unit u, unit stride 32 rs
    auto rows_from = [&](const uint8_t* c, int u) {
        const int64_t skip = (int64_t)u * kUnit * rs + g * kD, left = (int64_t)a.max_pos * rs - skip;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(c + skip), (short)0,
                                                 (uint32_t)(left < 0 ? 0 : left < 0x7FFFFFFF ? left : 0x7FFFFFFF), 0x00020000);
    };
    uint32_t ko = (wave * kUnit + l16) * rs + 16 * lq, vo = (wave * kUnit + 4 * lq) * rs + 8 * l16;
    RawK rk;
    RawV rv;
    // (the rows of a fixed split are loaded before the context is known: one memory latency less)
    int u0 = 4 * blockIdx.x, upw = 4;
    __amdgpu_buffer_rsrc_t bk, bv;
    if (a.fixed) {
        bk = rows_from(a.kvk, u0);
        bv = rows_from(a.kvv, u0);
        load_k(rk, bk, ko, rs);
        load_v(rv, bv, vo, rs);
    }
    const int base = *a.dpos;
    const int n = min(base + a.M, a.max_pos);          // positions 0 .. n - 1 are seen by some token
    if (!a.fixed) {
        upw = units_per_split(n, a.nsplit);
        u0 = blockIdx.x * upw;
    }
    if (u0 * kUnit >= n) return;                       // uniform
    const int u1 = min(u0 + upw, (n + kUnit - 1) / kUnit);
    if (!a.fixed) {
        bk = rows_from(a.kvk, u0);
        bv = rows_from(a.kvv, u0);
        load_k(rk, bk, ko, rs);
        load_v(rv, bv, vo, rs);
    }
    // q: one tile's operands straight into registers, more through LDS
    auto q_row = [&](int r) { return a.q + ((int64_t)(r >> a.lg) * a.Hq + g * G + (r & (G - 1))) * kD; };
    uint4 q1[RT > 1 ? 1 : 4];
    if constexpr (RT == 1) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            q1[kt] = *reinterpret_cast<const uint4*>(q_row(min(r0 + l16, rows - 1)) + 64 * (kt >> 1) + 16 * lq + 8 * (kt & 1));
            if (r0 + l16 >= rows) q1[kt] = make_uint4(0, 0, 0, 0);
        }
    } else {
        for (int i = tid; i < R * 16; i += 256) {
            const int r = i >> 4, ch = i & 15;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (r0 + r < rows) v = *reinterpret_cast<const uint4*>(q_row(r0 + r) + 8 * ch);
            *reinterpret_cast<uint4*>(&qs[r][8 * ch]) = v;
        }
    }
    // the lane's query of tile rt: row r0 + 16 rt + l16, its token a whole number
    // of tokens past tile 0's (G divides 16); rows that are none, and tokens
    // outside the cache, see everything and write nothing
    const int pos0 = base + ((r0 + l16) >> a.lg), tok = 16 >> a.lg;
    bool out[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) out[rt] = r0 + 16 * rt + l16 < rows && pos0 + rt * tok >= 0 && pos0 + rt * tok < a.max_pos;
    // the query's row of sc, position 4 lq
    float* const sc0 = a.sc + ((int64_t)((r0 + l16) >> a.lg) * a.Hq + g * G + (l16 & (G - 1))) * a.max_pos + 4 * lq;
    const int64_t sc_tile = (int64_t)tok * a.Hq * a.max_pos;
    const int lim_min = base + (r0 >> a.lg);
    float m[RT], l[RT];
    bool wide[RT];   // uniform: a row's reference is past kWide
    mx::v4f acc[RT][8];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = kNone;
        l[rt] = 0.0f;
        wide[rt] = false;
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[rt][c] = mx::v4f{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (RT > 1) __syncthreads();
    for (int u = u0 + wave; u < u1; u += 4) {
        const int p0 = u * kUnit;
        const bool more = u + 4 < u1;
        uint4 kd[2][4];
        decode_k(rk, kd);
        ko += 4 * kUnit * rs;
        if (more) load_k(rk, bk, ko, rs);
        uint4 p[RT][3];   // P of each row tile in three parts
        const bool masked = p0 + kUnit - 1 > lim_min;   // uniform
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (rt > 0 && r0 + 16 * rt >= rows) break;
            mx::v4f s[2] = {mx::v4f{0.f, 0.f, 0.f, 0.f}, mx::v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                uint4 qf;
                if constexpr (RT == 1) qf = q1[kt];
                else qf = *reinterpret_cast<const uint4*>(&qs[16 * rt + l16][64 * (kt >> 1) + 16 * lq + 8 * (kt & 1)]);
                s[0] = mfma_bf16(kd[0][kt], qf, s[0]);
                s[1] = mfma_bf16(kd[1][kt], qf, s[1]);
            }
            // s[t][i]: position p0 + 16 t + 4 lq + i
            if (a.sc) {
                float* row = sc0 + (rt * sc_tile + p0);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int pp = p0 + 16 * t + 4 * lq;
                    if (a.sc_vec && !masked) {
                        if (out[rt]) __builtin_nontemporal_store(s[t], reinterpret_cast<mx::v4f*>(row + 16 * t));
                    } else if (out[rt]) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (pp + i <= pos0 + rt * tok) row[16 * t + i] = s[t][i];
                    }
                }
            }
            if (masked) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (out[rt] && p0 + 16 * t + 4 * lq + i > pos0 + rt * tok) s[t][i] = -INFINITY;
            }
            // m is the reference of the row's terms, not their maximum: it follows
            // the maximum only past a factor of 2^kSlack (any reference gives the
            // same quotient; the sums of a first unit need no rescaling at all), so
            // that the row's lanes need not agree on a maximum at every unit
            const float top = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                                    fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
            if (__ballot(top * a.c > m[rt] + kSlack)) {
                const float mn = fmaxf(m[rt], max_over_lq(top) * a.c);
                if (u != u0 + wave) {
                    const float al = __builtin_amdgcn_exp2f(m[rt] - mn);
                    l[rt] *= al;
#pragma unroll
                    for (int c = 0; c < 8; ++c)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[rt][c][i] *= al;
                }
                m[rt] = mn;
                wide[rt] = __ballot(fabsf(mn) > kWide && mn != kNone) != 0ull;
            }
            float t[8];
            if (!wide[rt]) {
#pragma unroll
                for (int i = 0; i < 8; ++i) t[i] = fmaf(s[i >> 2][i & 3], a.c, -m[rt]);
            } else {   // the rounded product, as in m: the fma's would differ from it by more than a term
#pragma unroll
                for (int i = 0; i < 8; ++i) t[i] = mul_then_sub(s[i >> 2][i & 3], a.c, m[rt]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) t[i] = __builtin_amdgcn_exp2f(t[i]);
            l[rt] += ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
            parts(t, p[rt]);
        }
        vo += 4 * kUnit * rs;
        uint4 vd[8];
        decode_v(rv, vd);
        if (more) load_v(rv, bv, vo, rs);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (rt > 0 && r0 + 16 * rt >= rows) break;
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int j = 2; j >= 0; --j) acc[rt][c] = mfma_bf16(vd[c], p[rt][j], acc[rt][c]);
        }
    }
    // the four waves' sums of each tile in LDS, then one record per row: acc[rt][c][i]
    // is column 8 (4 lq + i) + c of query l16
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt > 0) __syncthreads();
        const float ls = sum_over_lq(l[rt]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float* d = &mo[wave][l16][8 * (4 * lq + i)];
            *reinterpret_cast<float4*>(d) = make_float4(acc[rt][0][i], acc[rt][1][i], acc[rt][2][i], acc[rt][3][i]);
            *reinterpret_cast<float4*>(d + 4) = make_float4(acc[rt][4][i], acc[rt][5][i], acc[rt][6][i], acc[rt][7][i]);
        }
        if (lq == 0) {
            mm[wave][l16] = m[rt];
            ml[wave][l16] = ls;
        }
        __syncthreads();
        const int qr = tid >> 4, c0 = 8 * (tid & 15);
        const int rr = r0 + 16 * rt + qr, pos = base + (rr >> a.lg);
        if (rr >= rows || pos < 0 || pos >= a.max_pos || u0 * kUnit > pos) continue;   // no record: the merge reads none
        const float gm = fmaxf(fmaxf(mm[0][qr], mm[1][qr]), fmaxf(mm[2][qr], mm[3][qr]));
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, den = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float wt = __builtin_amdgcn_exp2f(mm[w][qr] - gm);
            den = fmaf(wt, ml[w][qr], den);
            const float4 x = *reinterpret_cast<const float4*>(&mo[w][qr][c0]), y = *reinterpret_cast<const float4*>(&mo[w][qr][c0 + 4]);
            o[0] = fmaf(wt, x.x, o[0]); o[1] = fmaf(wt, x.y, o[1]); o[2] = fmaf(wt, x.z, o[2]); o[3] = fmaf(wt, x.w, o[3]);
            o[4] = fmaf(wt, y.x, o[4]); o[5] = fmaf(wt, y.y, o[5]); o[6] = fmaf(wt, y.z, o[6]); o[7] = fmaf(wt, y.w, o[7]);
        }
        float* rec = a.part + (((int64_t)(rr >> a.lg) * a.Hq + g * G + (rr & (G - 1))) * a.nsplit + blockIdx.x) * kPart;
        *reinterpret_cast<float4*>(rec + 4 + c0) = make_float4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<float4*>(rec + 8 + c0) = make_float4(o[4], o[5], o[6], o[7]);
        if (c0 == 0) {
            rec[0] = gm;
            rec[1] = den;
        }
    }
}

// Up to 4 NF splits: every record is loaded at once, before the context is
// known, and the ones past the token's position are left out after (one
// memory latency instead of two); NF = 0: more, am::merge_head.
template <int NF>
__global__ __launch_bounds__(256) void attn_split_merge_kernel(const float* __restrict__ part, float* __restrict__ o,
                                                               uint8_t* __restrict__ oq, uint8_t* __restrict__ os,
                                                               const int32_t* __restrict__ dpos, int M, int Hq,
                                                               int max_pos, int nsplit, int fixed) {
    __shared__ am::MergeLds lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x, mt = blockIdx.y;
    const float* rec = part + ((int64_t)mt * Hq + h) * nsplit * kPart;
    const int base = *dpos;
    float2 st[NF > 0 ? NF : 1], cs[NF > 0 ? NF : 1];
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        const float* r = rec + (int64_t)min(wave + 4 * i, nsplit - 1) * kPart;
        st[i] = *reinterpret_cast<const float2*>(r);
        cs[i] = *reinterpret_cast<const float2*>(r + 4 + 2 * lane);
    }
    const int pos = base + mt;
    if (pos < 0 || pos >= max_pos) return;
    const int upw = fixed ? 4 : units_per_split(min(base + M, max_pos), nsplit);
    const int n = pos / (upw * kUnit) + 1;   // splits that hold positions 0..pos
    float r0, r1;
    if constexpr (NF == 0) {
        if (!am::merge_head<true>(rec, n, lds, r0, r1)) return;
    } else {
        float gm = -INFINITY;
#pragma unroll
        for (int i = 0; i < NF; ++i) gm = wave + 4 * i < n ? fmaxf(gm, st[i].x) : gm;
        if (lane == 0) lds.red[wave] = gm;
        __syncthreads();
        gm = fmaxf(fmaxf(lds.red[0], lds.red[1]), fmaxf(lds.red[2], lds.red[3]));
        float den = 0.0f;
        float2 num = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            if (wave + 4 * i < n) {
                const float w = __builtin_amdgcn_exp2f(st[i].x - gm);
                den = fmaf(w, st[i].y, den);
                num.x = fmaf(w, cs[i].x, num.x);
                num.y = fmaf(w, cs[i].y, num.y);
            }
        }
        lds.nred[wave][lane] = num;
        if (lane == 0) lds.dred[wave] = den;
        __syncthreads();
        if (wave != 0) return;
        den = (lds.dred[0] + lds.dred[1]) + (lds.dred[2] + lds.dred[3]);
        r0 = ((lds.nred[0][lane].x + lds.nred[1][lane].x) + (lds.nred[2][lane].x + lds.nred[3][lane].x)) / den;
        r1 = ((lds.nred[0][lane].y + lds.nred[1][lane].y) + (lds.nred[2][lane].y + lds.nred[3][lane].y)) / den;
    }
    am::write_head(o, oq, os, mt, h, Hq, r0, r1);
}

}  // namespace

namespace mxh {

namespace {
struct Plan {
    int RT, groups, nsplit, most;
};
Plan plan(int M, int Hq, int Hkv, int max_pos) {
    Plan p;
    const int tiles = (int)(((int64_t)M * (Hq / Hkv) + 15) / 16);
    p.groups = (tiles + kMaxRT - 1) / kMaxRT;
    p.RT = (tiles + p.groups - 1) / p.groups;
    // one round of workgroups (two per CU), no split below the 128 positions of
    // a round of its waves: a split more is a record more per row to merge
    const int64_t want = 512 / ((int64_t)Hkv * p.groups);
    p.most = (max_pos + 4 * kUnit - 1) / (4 * kUnit);
    p.nsplit = want < 1 ? 1 : (want < p.most ? (int)want : p.most);
    return p;
}
}  // namespace

size_t attn_split_record_bytes(int M, int Hq, int Hkv, int max_pos) {
    return (size_t)M * Hq * plan(M, Hq, Hkv, max_pos).nsplit * kPart * sizeof(float);
}

int attn_split(const void* q, const uint8_t* kvk, const uint8_t* kvv, const int32_t* dpos, float* sc, float* o,
               uint8_t* oq, uint8_t* os, int M, int Hq, int Hkv, int max_pos, void* workspace, hipStream_t st) {
    const int G = Hq / Hkv;
    const Plan pl = plan(M, Hq, Hkv, max_pos);
    SplitArgs a{static_cast<const uint16_t*>(q), kvk, kvv, sc, static_cast<float*>(workspace), dpos, M, Hq, Hkv, 0, max_pos,
                pl.nsplit, 0, pl.nsplit == pl.most, (float)(1.4426950408889634 / sqrt((double)kD))};
    while ((1 << a.lg) < G) ++a.lg;
    a.sc_vec = ((uintptr_t)sc & 15) == 0 && max_pos % 4 == 0;
    const dim3 grid(a.nsplit, Hkv, pl.groups);
    switch (pl.RT) {
        case 1: hipLaunchKernelGGL(attn_split_kernel<1>, grid, dim3(256), 0, st, a); break;
        case 2: hipLaunchKernelGGL(attn_split_kernel<2>, grid, dim3(256), 0, st, a); break;
        default: hipLaunchKernelGGL(attn_split_kernel<3>, grid, dim3(256), 0, st, a); break;
    }
    const int rc = launch_status("attn_decode (splits)");
    if (rc != MXFP4_OK) return rc;
    auto* merge = a.nsplit <= 32 ? attn_split_merge_kernel<8> : a.nsplit <= 64 ? attn_split_merge_kernel<16> : attn_split_merge_kernel<0>;
    hipLaunchKernelGGL(merge, dim3(Hq, M), dim3(256), 0, st, a.part, o, oq, os, dpos, M, Hq, max_pos, a.nsplit, a.fixed);
    return launch_status("attn_decode (merge)");
}

}  // namespace mxh
