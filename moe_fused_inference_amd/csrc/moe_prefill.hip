// moe_prefill.hip -- grouped MoE for prefill / batched tokens on gfx950.
//
// Replaces the per-expert Python loop of ModelRunnerV2.moe_compute
// (runtime/model_runner_v2.py:108-122):
//     for e in experts:
//         idx, slots = torch.where(topi == e)
//         g = forward(h[idx], gate_e); u = forward(h[idx], up_e)    # x -> half -> MXFP4
//         y = forward(silu(g) * u, down_e).to(bf16)                 # fp32 h -> half -> MXFP4
//         out.index_add_(0, idx, y * scores[idx, slots])
// which issues 3 launches per active expert and syncs on torch.where, with
// four or five stream-ordered launches and no host synchronisation:
//
//   1. routing            a stable counting sort of the (token, slot) pairs by
//                         expert, row-major within one -- exactly torch.where's
//                         order: one launch, or two from kR1Max pairs on.
//   2. quantization       h (T, H) bf16 -> fp16-rounded -> MXFP4, once per
//                         token (the per-row quantization does not depend on
//                         which expert gathers the row), as further workgroups
//                         of the (first) routing launch.
//   3. grouped GEMM, gate/up   tiles of (expert, up to 192 of its tokens, 128
//                         features): A = gathered token rows, W = the gate
//                         rows of the features + their up rows; the
//                         epilogue computes h = silu(g)*u in fp32, rounds it
//                         to fp16 (the x.to(half) of the `forward` binding)
//                         and quantizes it to MXFP4 in registers.
//   4. grouped GEMM, down      tiles of 256 output columns: A = the
//                         expert's quantized h rows; the epilogue writes
//                         bf16(bf16(y) * score) per (token, slot) pair.
//   5. combine_kernel     out[t] = bf16(sum over the token's slots, fp32,
//                         slot order).  Ids outside [0, n_experts) contribute
//                         nothing, as an id missing from `experts` does in
//                         the reference.
//
// The grouped GEMMs use v_mfma_scale_f32_32x32x64_f8f6f4 with the operands
// swapped: the weight tile is the MFMA's A operand, so each lane ends with
// one token and 16 features of a 32-feature block.  The 32-block amax of h is
// then one exchange with lane l^32, and the nibbles pack into 8-byte stores.
#include <algorithm>

#include "lds_dma.h"
#include "mx_device.h"
#include "mx_host.h"
#include "quant_rows.h"

namespace {

constexpr int kMaxExperts = 1024;
constexpr int kMaxTopk = 32;

enum { MODE_GATEUP = 0, MODE_DOWN = 1 };

// ------------------------------------------------------------------ routing
// Workgroup b lists the pairs routed to experts 2b and 2b+1 (each id is
// read once per pass for two experts: half the traffic of one expert per
// workgroup, at twice the compare-and-ballot work per id, which is what
// bounds a workgroup here).  Each of the 8 waves owns a contiguous eighth of
// the row-major (token, slot) pairs: a first coalesced pass counts, per expert,
// its matches (ballot) and its valid ids below the first expert; the waves
// exchange the counts once through LDS; a second pass writes each expert's
// matches in order (ballot rank), so the result is a stable sort by expert
// id.  With `sscore`, the pair's routing weight is written beside it in
// sorted order (fp32 of the bf16 score), so the down epilogue needs no
// dependent load.
constexpr int kRouteEpw = 2;        // experts per workgroup
constexpr int kRouteWaves = 8;
__global__ __launch_bounds__(64 * kRouteWaves) void route_kernel(const int64_t* __restrict__ topi, int P, int n_exp,
                                                                 int* __restrict__ counts, int* __restrict__ offs,
                                                                 int* __restrict__ pairs,
                                                                 const uint16_t* __restrict__ scores,
                                                                 float* __restrict__ sscore) {
    __shared__ int s_eq[kRouteWaves][kRouteEpw], s_lt[kRouteWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int E0 = blockIdx.x * kRouteEpw;
    const int per_wave = ((P + 64 * kRouteWaves - 1) / (64 * kRouteWaves)) * 64;
    const int w0 = min(wave * per_wave, P);
    const int w1 = min(w0 + per_wave, P);
    constexpr int U = 16;  // chunks of 64 ids in flight per pass step (all of a wave's at P = 16384)
    int n_eq[kRouteEpw];
#pragma unroll
    for (int k = 0; k < kRouteEpw; ++k) n_eq[k] = 0;
    int n_lt = 0;
    for (int b = w0; b < w1; b += 64 * U) {
        int64_t id[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {   // clamped, unconditional loads: all U in flight at once
            const int p = b + 64 * u + lane;
            const int64_t v = topi[min(p, P - 1)];
            id[u] = p < w1 ? v : -1;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int k = 0; k < kRouteEpw; ++k)   // (ids >= n_exp match no expert)
                n_eq[k] += E0 + k < n_exp ? __popcll(__ballot(id[u] == (int64_t)(E0 + k))) : 0;
            n_lt += (id[u] >= 0 && id[u] < (int64_t)E0) ? 1 : 0;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n_lt += __shfl_xor(n_lt, o);
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < kRouteEpw; ++k) s_eq[wave][k] = n_eq[k];
        s_lt[wave] = n_lt;
    }
    __syncthreads();
    // expert E0+k starts after the valid ids below E0 and the matches of
    // E0 .. E0+k-1; this wave's matches of it after those of earlier waves
    int base = 0;
    for (int w = 0; w < kRouteWaves; ++w) base += s_lt[w];
    int pos[kRouteEpw];
#pragma unroll
    for (int k = 0; k < kRouteEpw; ++k) {
        int tot = 0, before = 0;
        for (int w = 0; w < kRouteWaves; ++w) {
            tot += s_eq[w][k];
            before += w < wave ? s_eq[w][k] : 0;
        }
        pos[k] = base + before;
        if (threadIdx.x == 0 && E0 + k < n_exp) {
            counts[E0 + k] = tot;
            offs[E0 + k] = base;
        }
        base += tot;
    }
    // second pass, in segments of 64*U ids: the wave's matches of the
    // segment, in order and grouped by expert, into its own LDS list, then
    // out with coalesced stores (one store per match would cost a memory
    // instruction per ballot)
    __shared__ int2 s_list[kRouteWaves][64 * U];
    int2* list = s_list[wave];
    for (int b = w0; b < w1; b += 64 * U) {
        int64_t id[U];
        uint16_t sc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = b + 64 * u + lane;
            const int64_t v = topi[min(p, P - 1)];
            id[u] = p < w1 ? v : -1;
            sc[u] = sscore ? scores[min(p, P - 1)] : (uint16_t)0;
        }
        int cnt[kRouteEpw], kb[kRouteEpw], rank[kRouteEpw];
        int kacc = 0;
#pragma unroll
        for (int k = 0; k < kRouteEpw; ++k) {
            cnt[k] = 0;
#pragma unroll
            for (int u = 0; u < U; ++u)
                cnt[k] += E0 + k < n_exp ? __popcll(__ballot(id[u] == (int64_t)(E0 + k))) : 0;
            kb[k] = kacc;
            kacc += cnt[k];
            rank[k] = 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int k = 0; k < kRouteEpw; ++k) {
                const bool m = E0 + k < n_exp && id[u] == (int64_t)(E0 + k);
                const unsigned long long bal = __ballot(m);
                if (m) list[kb[k] + rank[k] + __popcll(bal & ((1ull << lane) - 1ull))] = make_int2(b + 64 * u + lane, (int)sc[u]);
                rank[k] += __popcll(bal);
            }
        }
#pragma unroll
        for (int k = 0; k < kRouteEpw; ++k) {
            for (int q = lane; q < cnt[k]; q += 64) {
                const int2 v = list[kb[k] + q];
                pairs[pos[k] + q] = v.x;
                if (sscore) sscore[pos[k] + q] = mx::bf16_to_f32((uint16_t)v.y);
            }
            pos[k] += cnt[k];
        }
    }
}

// ------------------------------------------------------------------ routing, counting sort
// The same grouping (a stable sort of the row-major pairs by expert id) as a
// counting sort in two launches, whose work per id does not grow with the
// number of experts.  Chunks of kRtChunk ids; a wave takes 64 consecutive
// ids at a time and finds, for each lane, the lanes holding the same id with
// one ballot per id bit (the id's bits agree), so its rank among the equal
// ids of the 64 is a popcount.
//   route_count_kernel    chunk c: per-expert counts of its valid ids ->
//                         hist (nchunk, n_exp).
//   route_scatter_kernel  chunk c: expert e's pairs start at offs[e] (sum of
//                         the counts of ids below e) + the counts of e in
//                         chunks below c + in earlier waves of c + the
//                         earlier 64-id groups of the wave + the rank;
//                         writes pairs (and the sorted routing weights), and
//                         chunk 0 writes counts / offs.
constexpr int kRtWaves = 4;
constexpr int kRtGroups = 4;                          // 64-id groups per wave
constexpr int kRtChunk = 64 * kRtWaves * kRtGroups;   // 1024 ids per workgroup

__device__ __forceinline__ uint64_t same_id_lanes(int id, bool valid, int bits) {
    uint64_t m = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
        const uint64_t s = __ballot((id >> b) & 1);
        m &= ((id >> b) & 1) ? s : ~s;
    }
    return m;
}

__device__ __forceinline__ int id_bits(int n_exp) { return 32 - __clz(max(n_exp - 1, 1)); }

// The token rows' quantization (x -> fp16 -> MXFP4) rides in the route
// count launch as the workgroups past its chunks: it does not depend on the
// routing, and the count's few latency-bound workgroups leave the CUs free.
struct XQuant {
    const void* x;      // (T, H) bf16
    int T, H, Kp;       // Kp: H padded to whole K steps
    int lt, gx;         // quantize_rows_kernel's layout: 2^lt threads per row, gx row groups
    uint8_t* q;         // (T, Kp/2)
    uint8_t* s;         // (T, Kp/32)
};

// Quantizer workgroup `local` of 256 threads (tid < 256).
__device__ __forceinline__ void xquant_block(const XQuant& xq, int local, int tid) {
    const int bx = local % xq.gx, by = local / xq.gx;
    const int64_t row = (int64_t)bx * (256 >> xq.lt) + (tid >> xq.lt);
    const int u = by * (1 << xq.lt) + (tid & ((1 << xq.lt) - 1));
    mxq::quantize_unit<MXFP4_DT_BF16, 1>(xq.x, xq.H, xq.T, xq.H, xq.Kp, true, row, u, xq.q, xq.s);
}

__global__ __launch_bounds__(64 * kRtWaves) void route_count_kernel(const int64_t* __restrict__ topi, int P, int n_exp,
                                                                   int* __restrict__ hist, int* __restrict__ qctr,
                                                                   int nchunk, XQuant xq) {
    __shared__ int h[kMaxExperts];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if ((int)blockIdx.x >= nchunk) {
        xquant_block(xq, (int)blockIdx.x - nchunk, tid);
        return;
    }
    if (qctr && blockIdx.x == 0 && tid < 16) qctr[tid] = 0;   // the grouped GEMMs' tile queues (8 each)
    for (int e = tid; e < n_exp; e += 64 * kRtWaves) h[e] = 0;
    const int bits = id_bits(n_exp);
    int id[kRtGroups];
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) {   // unconditional (clamped) loads: all in flight at once
        const int p = blockIdx.x * kRtChunk + (wave * kRtGroups + k) * 64 + lane;
        const int64_t v = topi[min(p, P - 1)];
        id[k] = (p < P && v >= 0 && v < n_exp) ? (int)v : -1;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) {
        const bool valid = id[k] >= 0;
        const uint64_t m = same_id_lanes(id[k], valid, bits);
        if (valid && (m & ((1ull << lane) - 1ull)) == 0) atomicAdd(&h[id[k]], __popcll(m));   // group leader
    }
    __syncthreads();
    for (int e = tid; e < n_exp; e += 64 * kRtWaves) hist[(int64_t)blockIdx.x * n_exp + e] = h[e];
}

__global__ __launch_bounds__(64 * kRtWaves) void route_scatter_kernel(const int64_t* __restrict__ topi, int P,
                                                                     int n_exp, const int* __restrict__ hist,
                                                                     int* __restrict__ counts, int* __restrict__ offs,
                                                                     int* __restrict__ pairs,
                                                                     const uint16_t* __restrict__ scores,
                                                                     float* __restrict__ sscore) {
    __shared__ int base[kMaxExperts];              // where expert e's pairs of this chunk start
    __shared__ int wh[kRtWaves][kMaxExperts];      // per-wave counts, then exclusive prefix over waves
    __shared__ int wsum[kRtWaves];
    __shared__ int carry;                          // running total of the scan over earlier slices
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nchunk = gridDim.x, c = blockIdx.x;
    if (tid == 0) carry = 0;
    const int bits = id_bits(n_exp);
    int id[kRtGroups];
    int64_t raw[kRtGroups];
    uint16_t sc[kRtGroups] = {};
    // all loads first (no use of a loaded value in between: one round trip)
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) raw[k] = topi[min(c * kRtChunk + (wave * kRtGroups + k) * 64 + lane, P - 1)];
    if (sscore) {
#pragma unroll
        for (int k = 0; k < kRtGroups; ++k) sc[k] = scores[min(c * kRtChunk + (wave * kRtGroups + k) * 64 + lane, P - 1)];
    }
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) {
        const int p = c * kRtChunk + (wave * kRtGroups + k) * 64 + lane;
        id[k] = (p < P && raw[k] >= 0 && raw[k] < n_exp) ? (int)raw[k] : -1;
    }
    // per expert: the total over all chunks and the count in chunks below c
    for (int e0 = 0; e0 < n_exp; e0 += 64 * kRtWaves) {
        const int e = e0 + tid;
        const int ec = min(e, n_exp - 1);
        int tot = 0, bef = 0;
        for (int cb = 0; cb < nchunk; cb += 16) {
            int v[16];   // 16 unconditional (clamped) loads in flight, then the sums
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = hist[(int64_t)min(cb + i, nchunk - 1) * n_exp + ec];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int x = (cb + i < nchunk && e < n_exp) ? v[i] : 0;
                tot += x;
                bef += cb + i < c ? x : 0;
            }
        }
        // exclusive scan of tot over e: waves, then the waves' sums
        int incl = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();   // wsum, and carry from the previous slice
        int run = carry;
        for (int w = 0; w < wave; ++w) run += wsum[w];
        const int ex = run + incl - tot;
        if (e < n_exp) {
            base[e] = ex + bef;
            if (c == 0) {
                counts[e] = tot;
                offs[e] = ex;
            }
#pragma unroll
            for (int w = 0; w < kRtWaves; ++w) wh[w][e] = 0;
        }
        __syncthreads();   // every read of carry and wsum is done
        if (tid == 64 * kRtWaves - 1) carry = run + incl;   // read after the next slice's first barrier
    }
    __syncthreads();
    // this wave's counts per expert (group leaders; one writer per expert and group)
    uint64_t mk[kRtGroups];
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) {
        const bool valid = id[k] >= 0;
        mk[k] = same_id_lanes(id[k], valid, bits);
        if (valid && (mk[k] & ((1ull << lane) - 1ull)) == 0) wh[wave][id[k]] += __popcll(mk[k]);
    }
    __syncthreads();
    // exclusive prefix over the waves, per expert
    for (int e = tid; e < n_exp; e += 64 * kRtWaves) {
        int run = 0;
        for (int w = 0; w < kRtWaves; ++w) {
            const int v = wh[w][e];
            wh[w][e] = run;
            run += v;
        }
    }
    __syncthreads();
    // positions: the wave's earlier groups are counted in wh as it goes
#pragma unroll
    for (int k = 0; k < kRtGroups; ++k) {
        if (id[k] < 0) continue;
        const int at = base[id[k]] + wh[wave][id[k]] + __popcll(mk[k] & ((1ull << lane) - 1ull));
        const int p = c * kRtChunk + (wave * kRtGroups + k) * 64 + lane;
        pairs[at] = p;
        if (sscore) sscore[at] = mx::bf16_to_f32(sc[k]);
        // after every lane has its position, the group leader moves the
        // wave's offset of this expert past the group
        if ((mk[k] & ((1ull << lane) - 1ull)) == 0) wh[wave][id[k]] += __popcll(mk[k]);
    }
}

// Both launches in one for up to kR1Max pairs: workgroup 0 alone sorts, wave w
// taking the w-th sixteenth of the pairs in 64-id groups; the workgroups past
// it quantize x (four of the quantizer's blocks each).  What bounds it at these
// sizes is latency, so a launch and the histograms' trip through memory saved
// are worth a single workgroup's ballots (measured on MI355X, 100 tokens x 8:
// count + scatter 4.3 + 5.4 us, 4.3 us here).  kR1Max is what the kR1Groups ids
// that a lane holds come to; the gain goes down to 2 us there (500 tokens: the
// call 92.0 and 90.1 us), so there is no longer version.
constexpr int kR1Waves = 16, kR1Groups = 4;
constexpr int kR1Max = 64 * kR1Waves * kR1Groups;

__global__ __launch_bounds__(64 * kR1Waves) void route_one_kernel(const int64_t* __restrict__ topi, int P, int n_exp,
                                                                  int* __restrict__ qctr, int* __restrict__ counts,
                                                                  int* __restrict__ offs, int* __restrict__ pairs,
                                                                  const uint16_t* __restrict__ scores,
                                                                  float* __restrict__ sscore, XQuant xq) {
    __shared__ uint16_t wh[kR1Waves][kMaxExperts];   // per-wave counts, then exclusive prefix over waves
    __shared__ int base[kMaxExperts];
    __shared__ int wsum[kR1Waves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x > 0) {
        xquant_block(xq, 4 * ((int)blockIdx.x - 1) + (tid >> 8), tid & 255);
        return;
    }
    if (tid < 16) qctr[tid] = 0;   // the grouped GEMMs' tile queues (8 each)
    const int groups = (P + 64 * kR1Waves - 1) / (64 * kR1Waves);   // of 64 ids per wave, <= kR1Groups
    const int p0 = wave * groups * 64 + lane;
    int id[kR1Groups];
    int64_t raw[kR1Groups];
    uint16_t sc[kR1Groups];
#pragma unroll
    for (int k = 0; k < kR1Groups; ++k) {   // unconditional (clamped) loads: all in flight at once
        const int p = min(p0 + 64 * k, P - 1);
        raw[k] = topi[p];
        sc[k] = scores[p];
    }
    for (int i = tid; i < kR1Waves * kMaxExperts / 2; i += 64 * kR1Waves) reinterpret_cast<uint32_t*>(wh)[i] = 0;
    const int bits = id_bits(n_exp);
    __syncthreads();
    uint64_t mk[kR1Groups];
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int k = 0; k < kR1Groups; ++k) {
        id[k] = k < groups && p0 + 64 * k < P && raw[k] >= 0 && raw[k] < n_exp ? (int)raw[k] : -1;
        mk[k] = 0;
        if (k >= groups) continue;   // uniform
        const bool valid = id[k] >= 0;
        mk[k] = same_id_lanes(id[k], valid, bits);
        if (valid && (mk[k] & below) == 0) wh[wave][id[k]] += (uint16_t)__popcll(mk[k]);   // one writer per expert and group
    }
    __syncthreads();
    // thread e: expert e's prefix over the waves, then the scan over experts
    int tot = 0;
    if (tid < n_exp) {
#pragma unroll
        for (int w = 0; w < kR1Waves; ++w) {
            const int v = wh[w][tid];
            wh[w][tid] = (uint16_t)tot;
            tot += v;
        }
    }
    int incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = 0;
    for (int w = 0; w < wave; ++w) run += wsum[w];
    if (tid < n_exp) {
        base[tid] = run + incl - tot;
        counts[tid] = tot;
        offs[tid] = run + incl - tot;
    }
    __syncthreads();
    for (int k = 0; k < groups; ++k) {
        int e = -1, p = p0 + 64 * k;
        uint64_t m = 0;
        uint16_t s = 0;
#pragma unroll
        for (int q = 0; q < kR1Groups; ++q)
            if (q == k) {
                e = id[q];
                m = mk[q];
                s = sc[q];
            }
        if (e < 0) continue;
        const int at = base[e] + wh[wave][e] + __popcll(m & below);
        pairs[at] = p;
        sscore[at] = mx::bf16_to_f32(s);
        // after every lane has its position, the group leader moves the wave's offset past the group
        if ((m & below) == 0) wh[wave][e] += (uint16_t)__popcll(m);
    }
}

// ------------------------------------------------------------------ weights
struct StackedW {                // expert e of projection j at base[j] + e * stride
    const uint8_t* wp[3];
    const uint8_t* ws[3];
    int64_t wp_stride[3], ws_stride[3];
    __device__ const uint8_t* p(int e, int j) const { return wp[j] + (int64_t)e * wp_stride[j]; }
    __device__ const uint8_t* s(int e, int j) const { return ws[j] + (int64_t)e * ws_stride[j]; }
};
struct TableW {                  // device table (n_experts, 6) int64: gate wp/ws, up wp/ws, down wp/ws
    const int64_t* tab;
    __device__ const uint8_t* p(int e, int j) const { return reinterpret_cast<const uint8_t*>(tab[e * 6 + 2 * j]); }
    __device__ const uint8_t* s(int e, int j) const { return reinterpret_cast<const uint8_t*>(tab[e * 6 + 2 * j + 1]); }
};

struct GArgs {
    const uint8_t* aq;       // GATEUP: token rows (T); DOWN: sorted h rows (P)
    const uint8_t* as;       // matching scale rows
    int ald, asld;           // bytes from row to row of aq / as (whole K steps)
    const int* counts;
    const int* offs;
    const int* pairs;
    int topk;
    int Kp;                  // K of this GEMM: H (gate/up) or Mi (down)
    int Nw;                  // weight rows per projection: Mi (gate/up) or H (down)
    uint8_t* hq;             // GATEUP out: MXFP4 h in sorted order, rows hld bytes apart
    uint8_t* hs;             //             and its scales, hsld apart
    int hld, hsld;
    uint16_t* yd;            // DOWN out: (P, H) bf16 at the pair's own index
    const float* sscore;     // DOWN: (P) routing weights in sorted pair order
    int a_rows;              // rows of aq / as (T for gate/up, P for down)
};

// Scale word of a lane: byte ks = block 2*ks + h of the step's eight bytes lo,
// hi; RG: the bytes outside `keep` (blocks past the row) become 127.
template <bool RG>
__device__ __forceinline__ uint32_t scale_word(uint32_t lo, uint32_t hi, int h, uint32_t keep) {
    const uint32_t w = __builtin_amdgcn_perm(hi, lo, h ? 0x07050301u : 0x06040200u);
    return RG ? (w & keep) | (0x7F7F7F7Fu & ~keep) : w;
}

template <int OP>
__device__ __forceinline__ mx::v16f mfma32(uint4 a, uint4 b, mx::v16f c, uint32_t sa, uint32_t sb) {
    mx::v8i av = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
    mx::v8i bv = {(int)b.x, (int)b.y, (int)b.z, (int)b.w, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, c, 4, 4, OP, (int)sa, OP, (int)sb);
}

// Weight row of tile row rho (0..127).  Gate/up: rows [32b, 32b+32) hold
// projection b&1 (0 gate, 1 up) of features f0 + 32*(b>>1) + 0..31, so a
// wave's two 32-row blocks are the gate and up rows of the same features.
template <int MODE>
__device__ __forceinline__ int weight_row(int rho, int n0, int& proj) {
    if (MODE == MODE_GATEUP) {
        const int b = rho >> 5;
        proj = b & 1;
        return n0 + 32 * (b >> 1) + (rho & 31);
    }
    proj = 2;
    return n0 + rho;
}

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    typedef uint16_t v2s __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2s, a), __builtin_bit_cast(v2s, b)));
}

// Gate/up epilogue of NI 32-token blocks of a wave, 64 tile rows apart: h =
// silu(g)*u, fp16, MXFP4 rows in sorted pair order.  Bound by its vector
// instructions (a tile's 16384 features, 4 us of a 21 us tile with 23
// instruction slots each, 8 of them exp2 and rcp): from the fp16 on it works
// on pairs, the amax as integers, which also shows a NaN, and one mixed fma a
// feature for scale, tie and sign of zero.  MI355X, 2048 tokens x 8 of 128
// experts, H = 2048, Mi = 768: the launch 63.1 -> 60.6 us.
// (silu(g)*u is rounded to fp32 and then to fp16, as stated above; a lone
// value's product and conversion had become one instruction that rounds the
// product once, which is another fp16 value where the fp32 one is a midpoint:
// 0 to 2 of the 12.6 million features then have another code or block scale.)
template <int NI>
__device__ __forceinline__ void gateup_epilogue(mx::v16f (&acc)[2][2], const GArgs& g, int n0, int off, int mt,
                                                int mrows, int rbase, int wn, int lr, int h) {
    // acc[i][j] element q of lane l: token rbase + 64*i + l%32, weight row
    // wn*64 + 32j + 8(q/4) + 4h + q%4 of the tile
    {
        const int fb = n0 + 32 * wn;           // first feature of this wave's 32-block
        const int Mi = g.Nw;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int rloc = rbase + 64 * i + lr;
            // v in fp16, two a register; the sign-less halves compare as integers
            v2h v[8];
            uint32_t top = 0;
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const v2f f = {mx::silu_mul_fast(acc[i][0][2 * p], acc[i][1][2 * p]),
                               mx::silu_mul_fast(acc[i][0][2 * p + 1], acc[i][1][2 * p + 1])};
                v[p] = __builtin_convertvector(f, v2h);
                top = max_u16x2(top, __builtin_bit_cast(uint32_t, v[p]) & 0x7FFF7FFFu);
            }
            uint32_t amax = max(top & 0xFFFFu, top >> 16);
            if (__builtin_expect(amax > 0x7C00u, 0)) {   // a NaN counts as 0
                amax = 0;
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    uint32_t b = __builtin_bit_cast(uint32_t, v[p]);
                    if ((b & 0x7FFFu) > 0x7C00u) b &= 0xFFFF0000u;
                    if (((b >> 16) & 0x7FFFu) > 0x7C00u) b &= 0xFFFFu;
                    v[p] = __builtin_bit_cast(v2h, b);
                    amax = max(amax, max(b & 0x7FFFu, (b >> 16) & 0x7FFFu));
                }
            }
            amax = max(amax, (uint32_t)__shfl_xor((int)amax, 32));
            const uint32_t code = mx::e8m0_code((float)__builtin_bit_cast(_Float16, (uint16_t)amax));
            // one ulp up, so that v / scale at a midpoint (v has 11 bits) rounds
            // up as the hardware rounds to even; the + 0 makes -0 code 0
            const float inv = __uint_as_float(__float_as_uint(mx::e8m0_inv_scale(code)) + 1u);
            uint32_t piece[4];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                auto arg = [&](_Float16 x) { return __builtin_fmaf((float)x, inv, 0.0f); };
                const v2h a = v[2 * q4], b = v[2 * q4 + 1];
                piece[q4] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, arg(a.x), arg(a.y), 1.0f, 0);
                piece[q4] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(piece[q4], arg(b.x), arg(b.y), 1.0f, 1);
            }
            // lane h holds features 8*q4 + 4h + 0..3 -> bytes 4*q4 + 2h, +1
            const uint32_t send = h ? (piece[0] | (piece[1] << 16)) : (piece[2] | (piece[3] << 16));
            const uint32_t recv = __shfl_xor(send, 32);
            uint2 d;
            if (h == 0) {
                d.x = piece[0] | ((recv & 0xFFFFu) << 16);
                d.y = piece[1] | ((recv >> 16) << 16);
            } else {
                d.x = (recv & 0xFFFFu) | (piece[2] << 16);
                d.y = (recv >> 16) | (piece[3] << 16);
            }
            if (rloc < mrows && fb < Mi) {
                const int64_t srow_i = off + mt + rloc;
                *reinterpret_cast<uint2*>(g.hq + srow_i * g.hld + (fb >> 1) + 8 * h) = d;
                if (h == 0) g.hs[srow_i * g.hsld + (fb >> 5)] = (uint8_t)code;
            }
        }
    }
}

// ------------------------------------------------------------------ 192 x 256 tiles, 8 waves
// Tiles of up to 192 tokens x 256 weight rows (gate/up: the gate and up rows
// of 128 features; down: 256 output columns), 8 waves in 2 (tokens) x 4
// (weight rows), a wave owning up to 3 x 2 MFMA accumulators.  K step 256,
// so every copied row piece is a whole 128-byte line (global -> LDS by
// buffer_load ... lds, XOR swizzle of the 16-byte chunks).  The weight rows,
// which stream from HBM, sit in a 3-stage ring and the token rows, which
// mostly hit L2, in a 2-stage ring: during step k the copies of the token
// rows of step k+1 and of the weight rows of step k+2 are in flight, in that
// order, so the wait at the top of step k+1 leaves the last five copies (the
// weights of step k+2) outstanding.  One workgroup per CU (156 KB of LDS).
//  * The token tile is sized to the expert's count in 64-row steps (only
//    ceil(rows / 64) * 64 token rows are copied), and a wave issues the MFMAs
//    of only those of its 32-token blocks that hold routed tokens, so an
//    expert with ~130 tokens costs what ~130 tokens need.  Token block i of
//    wave (wm, wn) is tile block 2i + wm: the two waves of a SIMD share the
//    routed rows, so each one's MFMAs run while the other waits on its
//    operand reads, which are issued one MFMA substep ahead.
//  * All tiles of one expert run on workgroups of one residue mod 8, i.e.
//    on one XCD (workgroups are dealt to the 8 XCDs round-robin), so the
//    expert's gathered token rows are fetched into one L2.
//  * Kp not a multiple of 256 (RG): the token and h rows are the launch's own,
//    so they sit whole K steps apart; of the weights, which the caller laid
//    out, the lanes whose chunk lies past a row's end copy zeros, and a row's
//    scale bytes, which then start at any byte, come as the three aligned dwords
//    that hold a step's eight and are shifted into place by the reader.  The
//    blocks past the end read as zeros with scale 127 on both sides.  Measured on
//    MI355X, 2000 tokens, 60 experts, H = 2016, Mi = 992: 302 us on the
//    register-staged 128 x 128 tiles these sizes had, 154 us here; 20 tokens, 100
//    experts, H = 1984, Mi = 736: 104 and 70 us.
constexpr int X_BM = 192, X_BN = 256;
constexpr int X_ROWB = 128;                           // bytes per row per K step
constexpr int X_A = X_BM * X_ROWB;                    // 24 KB of token rows
constexpr int X_W = X_BN * X_ROWB;                    // 32 KB of weight rows
constexpr int X_AST = X_A + X_BM * 8;                 // token stage: rows + 8 scale bytes per row
constexpr int X_THREADS = 512;
constexpr int XP_MAXJ = kMaxExperts / 8;              // experts per group
constexpr int XP_TROW = 136;                          // down transpose: 128 B + 8 per row

// LDS layout: the 3-stage weight ring, the token ring, the down tile's pair
// indices and weights, the group's units, expert counts and offsets, the
// queue's unit.
template <bool RG>
struct XL {
    static constexpr int WST = X_W + X_BN * (RG ? 12 : 8);   // weight stage: rows + scale bytes per row
    static constexpr int ARING = 3 * WST;
    static constexpr int PP = ARING + 2 * X_AST;
    static constexpr int UCUM = PP + 8 * X_BM;               // int[XP_MAXJ + 1]: units of the experts below j
    static constexpr int ECNT = UCUM + 4 * (XP_MAXJ + 1);    // int[XP_MAXJ]: expert counts
    static constexpr int EOFF = ECNT + 4 * XP_MAXJ;          // int[XP_MAXJ]: expert offsets
    static constexpr int SLOT = EOFF + 4 * XP_MAXJ;          // int: the unit the queue handed out
    static constexpr int BYTES = SLOT + 16;
    static constexpr int WCP = RG ? 6 : 5;                   // weight copies per wave and step
    static_assert(BYTES <= 160 * 1024 && XP_MAXJ <= 128, "xp LDS layout (two experts per lane in the prefix)");
    static_assert(8 * 32 * XP_TROW <= WST, "the down transposes fit weight stage 0");
};

// Per-tile copy plan of one wave: na token-row blocks (8 rows of 128 bytes
// each), 4 weight-row blocks, one weight-scale copy (32 rows x 8 bytes) and,
// for waves < 2 na, one token-scale copy.
struct XCopiesAll {
    mx::v4u ars, wrs, sars, swrs;
    uint32_t avo[3], wvo[4], savo, swvo;
    int na;
};
template <bool RG>
struct XCopies : XCopiesAll {};
template <>
struct XCopies<true> : XCopiesAll {
    uint32_t swvo2;   // the third scale dword's offset, lanes 0 .. 31: row 32 * wave + lane
    uint32_t shw;     // the shifts of the lane's two operand rows' scales (bits 0-1, 8-9)
};

// Source rows of a wave's copies of one token tile: the rows of its three
// token-row blocks (64j + 8*wave + lane/8) and of its token-scale copy
// (32*wave + lane/2), clamped to the tile.  Gate/up: the sorted pair index
// (the token is it / topk, taken by x8_plan_rows); down: the sorted h row.
template <int MODE>
__device__ __forceinline__ void x8_rows(int (&rw)[4], const GArgs& g, int off, int mt, int mrows, int wave, int lane) {
    auto src = [&](int r) {
        const int rc = min(r, mrows - 1);
        return MODE == MODE_GATEUP ? g.pairs[off + mt + rc] : off + mt + rc;
    };
#pragma unroll
    for (int j = 0; j < 3; ++j) rw[j] = src(64 * j + 8 * wave + (lane >> 3));
    rw[3] = src(32 * wave + (lane >> 1));
}

template <int MODE, bool RG, class W>
__device__ __forceinline__ void x8_plan_rows(XCopies<RG>& c, const GArgs& g, const W& w, int e, int n0, int mrows,
                                             const int (&rw)[4], int wave, int lane) {
    const uint32_t cbytes = (uint32_t)g.Kp >> 1, nch = (uint32_t)g.Kp >> 5;
    const int slot = lane & 7;
    c.na = (mrows + 63) >> 6;
    auto row_of = [&](int v) { return MODE == MODE_GATEUP ? v / g.topk : v; };
    const uint32_t ald = RG ? (uint32_t)g.ald : cbytes, asld = RG ? (uint32_t)g.asld : nch;
    c.ars = mx::buf_rsrc(g.aq, (int64_t)g.a_rows * ald);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int r = 64 * j + 8 * wave + (lane >> 3);   // block 8j + wave
        c.avo[j] = (uint32_t)row_of(rw[j]) * ald + ((slot ^ mx::swz_key128(r)) << 4);
    }
    // weight blocks 4*wave + j: rows 32*wave .. +31, one projection (RG: relative to row n0)
    int proj;
    weight_row<MODE>(32 * wave, n0, proj);
    const int nbase = RG ? n0 : 0;
    const int64_t wrows = RG ? min(g.Nw - n0, X_BN) : g.Nw;
    c.wrs = mx::buf_rsrc(w.p(e, proj) + (int64_t)nbase * cbytes, wrows * cbytes);
    auto rel_row = [&](int rho) {
        int pj;
        return (uint32_t)(min(weight_row<MODE>(rho, n0, pj), g.Nw - 1) - nbase);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int rho = 32 * wave + 8 * j + (lane >> 3);
        c.wvo[j] = rel_row(rho) * cbytes + ((slot ^ mx::swz_key128(rho)) << 4);
    }
    // scale copies: lane -> row 32 * wave + lane / 2, 4 of its 8 bytes
    c.sars = mx::buf_rsrc(g.as, (int64_t)g.a_rows * asld);
    c.savo = (uint32_t)row_of(rw[3]) * asld + 4 * (lane & 1);
    const uint8_t* sw = w.s(e, proj) + (int64_t)nbase * nch;
    if constexpr (RG) {
        const uint32_t d = (uint32_t)(uintptr_t)sw & 3u;
        c.swrs = mx::buf_rsrc(sw - d, (wrows * nch + d + 3) & ~3ll);
        c.swvo = ((rel_row(32 * wave + (lane >> 1)) * nch + d) & ~3u) + 4 * (lane & 1);
        // the rows this lane's operand reads will take: 64 * (wave % 4) + 32 j + lane % 32
        auto shift = [&](int j) {
            const uint32_t rr = rel_row(64 * (wave & 3) + 32 * j + (lane & 31));
            return (rr * nch + (uint32_t)(uintptr_t)w.s(e, MODE == MODE_GATEUP ? j : 2)) & 3u;
        };
        c.swvo2 = ((rel_row(32 * wave + (lane & 31)) * nch + d) & ~3u) + 8;
        c.shw = shift(0) | (shift(1) << 8);
    } else {
        c.swrs = mx::buf_rsrc(sw, wrows * nch);
        c.swvo = rel_row(32 * wave + (lane >> 1)) * nch + 4 * (lane & 1);
    }
}

// The token-row copies of K step s into the token stage at `abuf`, part
// `part` (parts 0-1), and the weight-row copies of step s into the weight
// stage at `wbuf`, part `part` (parts 2-3): within a step all token copies
// come first and the last XL::WCP are the weight copies.  `left` (RG): the
// row's 32-blocks from this step on.
// Bit 31 set for a lane whose chunk of a row (r mod 16 of them) lies past the
// row's end: an offset out of every range, the copy writes zeros.
template <bool RG>
__device__ __forceinline__ uint32_t past_end(int r, int left) {
    if (!RG || left >= 8) return 0u;   // uniform
    const int slot = threadIdx.x & 7;
    return (slot ^ mx::swz_key128(r)) >= left ? 0x80000000u : 0u;
}

template <bool RG>
__device__ __forceinline__ void x8_issue_a(const XCopies<RG>& c, uint32_t abuf, int s, int part, int wave, int left) {
    const uint32_t kofs = (uint32_t)s * X_ROWB;
    const uint32_t past = past_end<RG>(8 * wave + ((threadIdx.x & 63) >> 3), left);
    if (part == 0) {
        if (c.na > 0) mx::dma16(c.avo[0] | past, c.ars, kofs, abuf + wave * 1024);
        if (c.na > 1) mx::dma16(c.avo[1] | past, c.ars, kofs, abuf + (8 + wave) * 1024);
        if (wave < 2 * c.na) mx::dma4(c.savo, c.sars, (uint32_t)s * 8, abuf + X_A + 256 * wave);
    } else if (c.na > 2) {
        mx::dma16(c.avo[2] | past, c.ars, kofs, abuf + (16 + wave) * 1024);
    }
}
template <bool RG>
__device__ __forceinline__ void x8_issue_w(const XCopies<RG>& c, uint32_t wbuf, int s, int part, int wave, int left) {
    const uint32_t kofs = (uint32_t)s * X_ROWB;
    const int j0 = 2 * (part - 2);
#pragma unroll
    for (int p = 0; p < 2; ++p)
        mx::dma16(c.wvo[j0 + p] | past_end<RG>(8 * p + ((threadIdx.x & 63) >> 3), left), c.wrs, kofs,
                  wbuf + (4 * wave + j0 + p) * 1024);
    if (part == 2) mx::dma4(c.swvo, c.swrs, (uint32_t)s * 8, wbuf + X_W + 256 * wave);
    if constexpr (RG) {
        if (part == 3 && (threadIdx.x & 63) < 32)
            mx::dma4(c.swvo2, c.swrs, (uint32_t)s * 8, wbuf + X_W + 8 * X_BN + 128 * wave);
    }
}

// ------------------------------------------------------------------ persistent 192 x 256 tiles
// grouped_gemm_xp_kernel<MODE>: the tiles above, with one workgroup per CU
// that takes tiles from its group's queue until the queue is empty.  A
// tile's plan and first copies (weights of steps 0 and 1, tokens of step 0)
// are issued during the previous tile's epilogue, so they land while that
// epilogue runs instead of after one workgroup has exited and the next has
// started (a workgroup per tile, one per CU: 140 us per config-3b call
// against 133 us).
//  * Groups: workgroup b is in group b % 8, i.e. on XCD b % 8 (workgroups
//    are dealt to the XCDs round-robin), and group x computes the experts
//    e = x, x+8, ..., so an expert's token rows are fetched into one L2.
//  * Units: a group's tiles are (expert j, token tile, weight-row tile),
//    expert-major, then token tile, then weight-row tile, so the weight-row
//    tiles of an expert run at about the same time and share its token rows.
//    At the start every workgroup counts its group's units from the expert
//    counts (a prefix over the group's experts, in LDS); a unit index names
//    its tile by a ballot over the prefix.  Workgroup k of a group (of P)
//    takes units k and k + P first; the group's queue (an atomic counter the
//    route kernel zeroes) hands out the rest from 2P on, one per tile and a
//    tile ahead, so the next tile is known when a tile starts and its source
//    rows load during the K loop.
//  * The weight ring is used from stage 1 on (K step s in stage (s+1) % 3):
//    the down epilogue transposes its blocks in stage 0, which the next tile
//    first refills during its step 0, after the barrier every wave reaches
//    only past its epilogue.  The next tile's copies go to stages 1 and 2
//    and token stage 0, read by no wave once all are past the last K step.
//  * Waits: the copies are invisible to the compiler (inline asm), so a load
//    whose value is used while copies are in flight would make it wait for
//    all of them.  The loads of a tile (the next tile's source rows, the
//    queue atomic, the down tile's pair indices and weights) are issued at
//    its start and used only after its K loop, where no copy is in flight.
struct XpTile {
    int e, n0, off, mt, mrows;
};

// The tile of unit u (uniform): the expert j of the group with
// ucum[j] <= u < ucum[j+1], found by a ballot over the group's experts.
template <int MODE, bool RG>
__device__ __forceinline__ XpTile xp_tile_of(const uint8_t* smem, int grp, int nj, int ntiles, int u, int lane) {
    const int* ucum = reinterpret_cast<const int*>(smem + XL<RG>::UCUM);
    int j = 0;
    for (int b = 0; b < nj; b += 64) {
        const int jj = b + lane;
        const bool hit = jj < nj && ucum[jj] <= u && u < ucum[jj + 1];
        const uint64_t m = __ballot(hit);
        if (m) {
            j = b + __ffsll((unsigned long long)m) - 1;
            break;
        }
    }
    j = __builtin_amdgcn_readfirstlane(j);
    const int local = u - ucum[j];
    const int mti = local / ntiles;
    const int nt = local - mti * ntiles;
    XpTile t;
    t.e = grp + 8 * j;
    t.off = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(smem + XL<RG>::EOFF)[j]);
    const int cnt = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(smem + XL<RG>::ECNT)[j]);
    t.mt = __builtin_amdgcn_readfirstlane(mti * X_BM);
    t.mrows = min(X_BM, cnt - t.mt);
    t.n0 = __builtin_amdgcn_readfirstlane(nt * (MODE == MODE_GATEUP ? X_BN / 2 : X_BN));
    return t;
}

// A tile's first copies in three parts, in the order the K loop's waits
// count on: 0, the weights of step 0 (stage 1); 1, the tokens of step 0;
// 2, the weights of step 1 (stage 2).  Before part 0 the plan's offsets and
// descriptors pass through an empty asm, so that they (and the compiler's
// waits for the plan's loads) are complete before the first copy is
// issued: a wait placed after a copy would also wait for the copy, which
// the compiler does not count.
template <bool RG>
__device__ __forceinline__ void xp_prologue_part(XCopies<RG>& c, uint32_t ring, int nch, int wave, int part) {
    using L = XL<RG>;
    if (part == 0) {
        asm volatile("" : "+v"(c.avo[0]), "+v"(c.avo[1]), "+v"(c.avo[2]), "+v"(c.savo), "+v"(c.wvo[0]),
                     "+v"(c.wvo[1]), "+v"(c.wvo[2]), "+v"(c.wvo[3]), "+v"(c.swvo), "+s"(c.ars), "+s"(c.wrs),
                     "+s"(c.sars), "+s"(c.swrs) :: "memory");
        if constexpr (RG) asm volatile("" : "+v"(c.swvo2), "+v"(c.shw) :: "memory");
        x8_issue_w<RG>(c, ring + L::WST, 0, 2, wave, nch);
        x8_issue_w<RG>(c, ring + L::WST, 0, 3, wave, nch);
    } else if (part == 1) {
        x8_issue_a<RG>(c, ring + L::ARING, 0, 0, wave, nch);
        x8_issue_a<RG>(c, ring + L::ARING, 0, 1, wave, nch);
    } else if (nch > 8) {
        x8_issue_w<RG>(c, ring + 2 * L::WST, 1, 2, wave, nch - 8);
        x8_issue_w<RG>(c, ring + 2 * L::WST, 1, 3, wave, nch - 8);
    }
}

template <int MODE, bool RG, int NB, class Issue>
__device__ __forceinline__ void xp_epilogue(mx::v16f (&acc)[3][2], const GArgs& g, uint8_t* smem, const XpTile& t,
                                            int wave, int lane, Issue&& issue);

// K loop of one wave on tile t (its prologue already issued), then
// `sync()` (every wave past the K loop, the tile's pair rows in LDS), then
// the epilogue with the next tile's plan and first copies (`issue(part)`)
// issued before it and between its blocks: the copies' latency hides under
// the epilogue, and the epilogue's VALU work fills the time a wave waits
// for the memory pipeline to accept them.  (All copies after the epilogue
// measured slower: their latency is then exposed.)
// NB = the wave's 32-token blocks holding routed tokens (0..3).
template <int MODE, bool RG, int NB, class Sync, class Issue>
__device__ __forceinline__ void xp_tile(const XCopies<RG>& c, const GArgs& g, uint8_t* smem, uint32_t ring,
                                        const XpTile& t, int wave, int lane, Sync&& sync, Issue&& issue) {
    const int wm = wave >> 2, wn = wave & 3;
    const int lr = lane & 31, h = lane >> 5;
    const int key = mx::swz_key128(lr);
    using L = XL<RG>;
    const int nch = g.Kp >> 5;
    const int nsteps = (nch + 7) >> 3;
    mx::v16f acc[3][2];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

    for (int it = 0; it < nsteps; ++it) {
        // this wave's copies of step it have landed (the weights of step
        // it+1, issued last, may still be in flight) and its reads of step
        // it-1 are done; after the barrier every wave's
        if (it + 1 < nsteps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(L::WCP) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const bool more_a = it + 1 < nsteps, more_w = it + 2 < nsteps;
        const uint8_t* wst = smem + ((it + 1) % 3) * L::WST;
        const uint8_t* ast = smem + L::ARING + (it & 1) * X_AST;
        const uint32_t anxt = ring + L::ARING + ((it + 1) & 1) * X_AST;
        const uint32_t wnxt = ring + (it % 3) * L::WST;   // step it+2: stage (it+3) % 3, step it-1's
        const uint8_t* la = ast + (32 * wm + lr) * X_ROWB;
        const uint8_t* lw = wst + (wn * 64 + lr) * X_ROWB;
        const uint8_t* lsa = ast + X_A + (32 * wm + lr) * 8;
        const uint8_t* lsw = wst + X_W + (wn * 64 + lr) * 8;
        uint32_t sa[3], sb[2];
        const int left = nch - 8 * it;   // 32-blocks of the row from this step on
        uint32_t keep = 0xFFFFFFFFu;     // RG: the blocks 2 ks + h < left
        if (RG && left < 8) keep = left + 1 - h >= 8 ? 0xFFFFFFFFu : (1u << (4 * ((left + 1 - h) & ~1))) - 1u;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const uint2 v = *reinterpret_cast<const uint2*>(lsa + i * 64 * 8);
            sa[i] = scale_word<RG>(v.x, v.y, h, keep);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint2 v = *reinterpret_cast<const uint2*>(lsw + j * 32 * 8);
            if constexpr (RG) {
                const uint32_t v2 = *reinterpret_cast<const uint32_t*>(wst + X_W + 8 * X_BN + (wn * 64 + j * 32 + lr) * 4);
                const uint32_t sh = j ? c.shw >> 8 : c.shw;   // alignbyte takes bits 0-1
                v = make_uint2(__builtin_amdgcn_alignbyte(v.y, v.x, sh), __builtin_amdgcn_alignbyte(v2, v.y, sh));
            }
            sb[j] = scale_word<RG>(v.x, v.y, h, keep);
        }
        uint4 af[2][3], bf[2][2];
        auto load = [&](int ks, int r) {
            const int koff = ((2 * ks + h) ^ key) << 4;
#pragma unroll
            for (int i = 0; i < NB; ++i) af[r][i] = *reinterpret_cast<const uint4*>(la + koff + i * 64 * X_ROWB);
#pragma unroll
            for (int j = 0; j < 2; ++j) bf[r][j] = *reinterpret_cast<const uint4*>(lw + koff + j * 32 * X_ROWB);
        };
        if (NB > 0) load(0, 0);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            __builtin_amdgcn_sched_barrier(0);
            if (ks < 2) {
                if (more_a) x8_issue_a<RG>(c, anxt, it + 1, ks, wave, left - 8);
            } else if (more_w) {
                x8_issue_w<RG>(c, wnxt, it + 2, ks, wave, left - 16);
            }
            if (NB > 0) {
                if (ks + 1 < 4) load(ks + 1, (ks + 1) & 1);
                const int r = ks & 1;
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        if (ks == 0) acc[i][j] = mfma32<0>(bf[r][j], af[r][i], acc[i][j], sb[j], sa[i]);
                        if (ks == 1) acc[i][j] = mfma32<1>(bf[r][j], af[r][i], acc[i][j], sb[j], sa[i]);
                        if (ks == 2) acc[i][j] = mfma32<2>(bf[r][j], af[r][i], acc[i][j], sb[j], sa[i]);
                        if (ks == 3) acc[i][j] = mfma32<3>(bf[r][j], af[r][i], acc[i][j], sb[j], sa[i]);
                    }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) mx::pin(acc[i][j]);
    sync();
    issue(0);
    xp_epilogue<MODE, RG, NB>(acc, g, smem, t, wave, lane, issue);
}

// Epilogue of one wave's token blocks (NB of them) of tile t; issues parts 1
// and 2 of the next tile's first copies between its blocks.
template <int MODE, bool RG, int NB, class Issue>
__device__ __forceinline__ void xp_epilogue(mx::v16f (&acc)[3][2], const GArgs& g, uint8_t* smem, const XpTile& t,
                                            int wave, int lane, Issue&& issue) {
    const int wm = wave >> 2, wn = wave & 3;
    const int lr = lane & 31, h = lane >> 5;
    if (NB == 0) {
        issue(1);
        issue(2);
        return;
    }
    if (MODE == MODE_DOWN) {
        // bf16(bf16(y) * score) through LDS, one 32-token block at a time in
        // the wave's own 32-row buffer of weight stage 0, so that a store
        // writes 8 whole 128-byte row segments; rows 136 bytes apart make
        // the 8-byte writes of 32 lanes (one row each) hit distinct banks
        uint8_t* tb = smem + wave * 32 * XP_TROW;
        const int* lp = reinterpret_cast<const int*>(smem + XL<RG>::PP);
        const float* ls = reinterpret_cast<const float*>(smem + XL<RG>::PP + 4 * X_BM);
        // lane: buffer row 8*st + lane/8 (tile row 64*i + 32*wm + 8*st +
        // lane/8), 16 bytes at column chunk lane%8
        const int ch = lane & 7;
        const int col = t.n0 + wn * 64 + 8 * ch;
        const int lim = col < g.Nw ? t.mrows - 32 * wm - (lane >> 3) : 0;   // tile rows < lim + 32*wm + lane/8 are routed
        const uint8_t* tr = tb + (lane >> 3) * XP_TROW + 16 * ch;
        const int* pr = lp + 32 * wm + (lane >> 3);
        uint16_t* yc = g.yd + col;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const float sc = ls[64 * i + 32 * wm + lr];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    uint32_t b[2];
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const uint32_t y2 = mx::f32x2_to_bf16x2(acc[i][j][4 * q4 + 2 * r], acc[i][j][4 * q4 + 2 * r + 1]);
                        b[r] = mx::f32x2_to_bf16x2(__uint_as_float(y2 << 16) * sc, __uint_as_float(y2 & 0xFFFF0000u) * sc);
                    }
                    // element q of block j: column 32j + 8(q/4) + 4h + q%4
                    *reinterpret_cast<uint2*>(tb + lr * XP_TROW + (32 * j + 8 * q4 + 4 * h) * 2) = make_uint2(b[0], b[1]);
                }
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const int toff = 64 * i + 8 * st;   // tile row - (32*wm + lane/8)
                if (toff < lim) {
                    const uint4 v = *reinterpret_cast<const uint4*>(tr + 8 * st * XP_TROW);
                    *reinterpret_cast<uint4*>(yc + (int64_t)pr[toff] * g.Nw) = v;
                }
            }
            if (i < 2) issue(i + 1);
        }
        if (NB == 1) issue(2);
        return;
    }
    if (NB >= 2) {
        mx::v16f sub[2][2] = {{acc[0][0], acc[0][1]}, {acc[1][0], acc[1][1]}};
        gateup_epilogue<2>(sub, g, t.n0, t.off, t.mt, t.mrows, 32 * wm, wn, lr, h);
        issue(1);
    }
    if (NB == 1 || NB == 3) {
        mx::v16f sub[2][2] = {{acc[NB - 1][0], acc[NB - 1][1]}, {acc[NB - 1][0], acc[NB - 1][1]}};
        gateup_epilogue<1>(sub, g, t.n0, t.off, t.mt, t.mrows, 64 * (NB - 1) + 32 * wm, wn, lr, h);
        if (NB == 1) issue(1);
    }
    issue(2);
}

template <int MODE, bool RG, class W>
__global__ __launch_bounds__(X_THREADS, 1) void grouped_gemm_xp_kernel(GArgs g, W w, int ntiles, int n_exp,
                                                                       int* __restrict__ qctr) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int grp = blockIdx.x & 7;
    const int kw = blockIdx.x >> 3;              // workgroup of the group
    const int per = gridDim.x >> 3;              // workgroups per group
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ring = __builtin_amdgcn_readfirstlane(mx::lds_addr(smem));
    int* ucum = reinterpret_cast<int*>(smem + XL<RG>::UCUM);
    int* ecnt = reinterpret_cast<int*>(smem + XL<RG>::ECNT);
    int* eoff = reinterpret_cast<int*>(smem + XL<RG>::EOFF);
    int* slot = reinterpret_cast<int*>(smem + XL<RG>::SLOT);
    const int nj = n_exp > grp ? (n_exp - grp + 7) / 8 : 0;
    if (nj == 0) return;
    for (int j = tid; j < nj; j += X_THREADS) {
        ecnt[j] = g.counts[grp + 8 * j];
        eoff[j] = g.offs[grp + 8 * j];
    }
    __syncthreads();
    if (wave == 0) {   // units below expert j: exclusive prefix, two experts per lane
        const int j0 = 2 * lane;
        const int u0 = j0 < nj ? (ecnt[j0] + X_BM - 1) / X_BM * ntiles : 0;
        const int u1 = j0 + 1 < nj ? (ecnt[j0 + 1] + X_BM - 1) / X_BM * ntiles : 0;
        int v = u0 + u1;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(v, d);
            if (lane >= d) v += o;
        }
        const int ex = v - u0 - u1;
        ucum[j0] = ex;
        ucum[j0 + 1] = ex + u0;
        if (lane == 63) ucum[128] = v;
    }
    __syncthreads();
    const int nunits = __builtin_amdgcn_readfirstlane(ucum[nj]);
    // units kw and kw + per are this workgroup's first two; the queue hands
    // out the rest, from 2 * per on
    if (kw >= nunits) return;
    const int nch = g.Kp >> 5;
    XpTile t = xp_tile_of<MODE, RG>(smem, grp, nj, ntiles, kw, lane);
    XCopies<RG> c;
    {
        int rw[4];
        x8_rows<MODE>(rw, g, t.off, t.mt, t.mrows, wave, lane);
        x8_plan_rows<MODE, RG>(c, g, w, t.e, t.n0, t.mrows, rw, wave, lane);
    }
    for (int part = 0; part < 3; ++part) xp_prologue_part<RG>(c, ring, nch, wave, part);
    int un1 = kw + per;                          // the next tile's unit (uniform)
    const int trow = wave * 64 + lane;
    for (;;) {
        // Issued now, used only after the K loop: the next tile's source
        // rows, the queue's unit for the tile after it, and the down tile's
        // pair indices and weights.  No loaded value is merged with a
        // default (a merge is a use, and the compiler's wait for it would
        // also wait for the copies in flight, which it does not count): the
        // atomic's result is read only by the lane that issued it, every
        // load is unconditional (clamped rows).  atomicInc, because the
        // compiler's wave aggregation of atomic adds uses the result at once.
        const bool more = un1 < nunits;
        XpTile tn = t;
        int rwn[4];
        if (more) {
            tn = xp_tile_of<MODE, RG>(smem, grp, nj, ntiles, un1, lane);
            x8_rows<MODE>(rwn, g, tn.off, tn.mt, tn.mrows, wave, lane);
        }
        int uq;
        if (tid == 0) uq = (int)atomicInc(reinterpret_cast<unsigned*>(qctr + grp), 0xFFFFFFFFu);
        int rp = 0;
        float rs = 0.0f;
        if (MODE == MODE_DOWN) {
            const int r = t.off + t.mt + min(trow, t.mrows - 1);
            rp = g.pairs[r];
            rs = g.sscore[r];
        }
        XCopies<RG> cn = c;
        auto sync = [&]() {
            if (MODE == MODE_DOWN && trow < t.mrows) {
                reinterpret_cast<int*>(smem + XL<RG>::PP)[trow] = rp;
                reinterpret_cast<float*>(smem + XL<RG>::PP + 4 * X_BM)[trow] = rs;
            }
            if (tid == 0) *slot = uq;
            // every wave is past its last operand read of this tile (the
            // next tile's copies may overwrite the stages), the pair rows
            // and the queue's unit are in LDS
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto issue = [&](int part) {
            if (more) {
                if (part == 0) x8_plan_rows<MODE, RG>(cn, g, w, tn.e, tn.n0, tn.mrows, rwn, wave, lane);
                xp_prologue_part<RG>(cn, ring, nch, wave, part);
            }
        };
        // the wave's token blocks 2i + wm (i < nb) holding routed rows
        const int nb = min(((t.mrows + 31) / 32 - (wave >> 2) + 1) >> 1, 3);
        switch (nb) {
            case 3: xp_tile<MODE, RG, 3>(c, g, smem, ring, t, wave, lane, sync, issue); break;
            case 2: xp_tile<MODE, RG, 2>(c, g, smem, ring, t, wave, lane, sync, issue); break;
            case 1: xp_tile<MODE, RG, 1>(c, g, smem, ring, t, wave, lane, sync, issue); break;
            default: xp_tile<MODE, RG, 0>(c, g, smem, ring, t, wave, lane, sync, issue); break;
        }
        if (!more) break;
        un1 = 2 * per + __builtin_amdgcn_readfirstlane(*slot);
        t = tn;
        c = cn;
    }
}

// out[t, c] = bf16(sum_{k < topk, id valid} yd[t*topk + k, c]); 8 columns per
// thread.  K8 (topk <= 8): a token's ids and then its rows are all loaded
// before any is used, two memory latencies instead of one per slot; from
// kCombineFew workgroups on others cover them and the plain loop is as fast
// (MI355X, 100 tokens x 8 of 2048: 6.4 us and 4.7; 2048 tokens 12.2 and
// 12.6).
constexpr int kCombineFew = 1024;

template <bool K8>
__global__ __launch_bounds__(256) void prefill_combine_kernel(const uint16_t* __restrict__ yd,
                                                              const int64_t* __restrict__ topi, int T, int topk,
                                                              int H, int n_exp, uint16_t* __restrict__ out) {
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int per_row = H >> 3;
    if (gid >= (int64_t)T * per_row) return;
    const int t = (int)(gid / per_row);
    const int c = (int)(gid - (int64_t)t * per_row) * 8;
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = 0.0f;
    auto add = [&](const uint4& v) {
        const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[2 * i] += mx::bf16_to_f32((uint16_t)(wv[i] & 0xFFFFu));
            s[2 * i + 1] += mx::bf16_to_f32((uint16_t)(wv[i] >> 16));
        }
    };
    const uint16_t* row = yd + (int64_t)t * topk * H + c;
    if constexpr (K8) {
        int64_t id[8];
        uint4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) id[k] = topi[(int64_t)t * topk + min(k, topk - 1)];
        // (rows of invalid ids are loaded, never written, and left out)
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const uint4*>(row + (int64_t)min(k, topk - 1) * H);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k < topk && id[k] >= 0 && id[k] < n_exp) add(v[k]);
    } else {
        for (int k = 0; k < topk; ++k) {
            const int64_t id = topi[(int64_t)t * topk + k];
            if (id < 0 || id >= n_exp) continue;
            add(*reinterpret_cast<const uint4*>(row + (int64_t)k * H));
        }
    }
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        o[i] = (uint32_t)mx::f32_to_bf16_rne(s[2 * i]) | ((uint32_t)mx::f32_to_bf16_rne(s[2 * i + 1]) << 16);
    *reinterpret_cast<uint4*>(out + (int64_t)t * H + c) = make_uint4(o[0], o[1], o[2], o[3]);
}

// ------------------------------------------------------------------ host
struct WsLayout {
    size_t counts, offs, pairs, sscore, hist, qctr, xq, xs, hq, hs, yd, total;
};

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
inline int64_t pad256(int v) { return ((int64_t)v + 255) & ~(int64_t)255; }

// CUs per XCD of the current device (its CU count / 8), cached per device:
// the persistent grouped GEMMs launch one workgroup per CU.
int cus_per_xcd() {
    static int cache[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 32;
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) n = 256;
        cache[dev] = n / 8;
    }
    return cache[dev];
}

WsLayout ws_layout(int T, int topk, int n_exp, int H, int Mi) {
    const size_t P = (size_t)T * topk;
    const size_t Hp = pad256(H), Mp = pad256(Mi);   // the launch's own rows: whole K steps
    WsLayout L;
    size_t o = 0;
    L.counts = o; o = align256(o + sizeof(int) * n_exp);
    L.offs = o;   o = align256(o + sizeof(int) * n_exp);
    L.pairs = o;  o = align256(o + sizeof(int) * P);
    L.sscore = o; o = align256(o + sizeof(float) * P);
    L.hist = o;   o = align256(o + sizeof(int) * ((P + kRtChunk - 1) / kRtChunk) * n_exp);
    L.qctr = o;   o = align256(o + sizeof(int) * 16);
    L.xq = o;     o = align256(o + (size_t)T * (Hp / 2));
    L.xs = o;     o = align256(o + (size_t)T * (Hp / 32));
    L.hq = o;     o = align256(o + P * (Mp / 2));
    L.hs = o;     o = align256(o + P * (Mp / 32));
    L.yd = o;     o = align256(o + P * H * sizeof(uint16_t));
    L.total = o;
    return L;
}

// One kernel's LDS reservation, once per kernel and process.
template <int MODE, bool RG, class W>
int reserve_xp() {
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(grouped_gemm_xp_kernel<MODE, RG, W>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, XL<RG>::BYTES);
    MXH_REQUIRE(e == hipSuccess, "moe_prefill: cannot reserve %d B of LDS: %s", XL<RG>::BYTES, hipGetErrorString(e));
    return MXFP4_OK;
}

// A grouped GEMM over every expert's rows, one persistent workgroup per CU.
template <int MODE, class W>
int launch_xp(const GArgs& g, const W& w, int n_exp, int* qctr, hipStream_t st) {
    const int per_tile = MODE == MODE_GATEUP ? X_BN / 2 : X_BN;
    const int ntiles = (g.Nw + per_tile - 1) / per_tile;
    const dim3 grid(8 * cus_per_xcd());
    int rc;
    // (without RG the weights are addressed with 32-bit offsets from the expert's first row)
    if (g.Kp % 256 == 0 && (int64_t)g.Nw * (g.Kp / 2) < (1ll << 32)) {
        if ((rc = reserve_xp<MODE, false, W>()) != MXFP4_OK) return rc;
        hipLaunchKernelGGL((grouped_gemm_xp_kernel<MODE, false, W>), grid, dim3(X_THREADS), XL<false>::BYTES, st, g, w, ntiles,
                           n_exp, qctr);
    } else {
        if ((rc = reserve_xp<MODE, true, W>()) != MXFP4_OK) return rc;
        hipLaunchKernelGGL((grouped_gemm_xp_kernel<MODE, true, W>), grid, dim3(X_THREADS), XL<true>::BYTES, st, g, w, ntiles,
                           n_exp, qctr);
    }
    return mxh::launch_status(MODE == MODE_GATEUP ? "moe_prefill gate/up" : "moe_prefill down");
}

template <class W>
int run_prefill_pass(const void* x, const int64_t* topi, const uint16_t* scores, W w, int n_exp, int T, int topk,
                     int H, int Mi, void* out, void* workspace, hipStream_t st) {
    const WsLayout L = ws_layout(T, topk, n_exp, H, Mi);
    const int Hp = (int)pad256(H), Mp = (int)pad256(Mi);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    int* counts = reinterpret_cast<int*>(ws + L.counts);
    int* offs = reinterpret_cast<int*>(ws + L.offs);
    int* pairs = reinterpret_cast<int*>(ws + L.pairs);
    const int P = T * topk;

    float* sscore = reinterpret_cast<float*>(ws + L.sscore);
    int* hist = reinterpret_cast<int*>(ws + L.hist);
    const int nchunk = (P + kRtChunk - 1) / kRtChunk;
    int* qctr = reinterpret_cast<int*>(ws + L.qctr);
    // x -> fp16 -> MXFP4 once per token (the reference quantizes each gathered
    // copy; the bytes are identical), in the same launch: quantize_rows_kernel's
    // layout (x is 16-byte aligned and H a multiple of 32, so the vector path)
    XQuant xqa{x, T, H, Hp, 2, 0, ws + L.xq, ws + L.xs};
    while ((1 << xqa.lt) < Hp / 8 && xqa.lt < 8) ++xqa.lt;
    xqa.gx = (T + (256 >> xqa.lt) - 1) / (256 >> xqa.lt);
    const int xq_gy = (Hp / 8 + (1 << xqa.lt) - 1) >> xqa.lt;
    if (P <= kR1Max) {
        hipLaunchKernelGGL(route_one_kernel, dim3(1 + (xqa.gx * xq_gy + 3) / 4), dim3(64 * kR1Waves), 0, st, topi, P, n_exp,
                           qctr, counts, offs, pairs, scores, sscore, xqa);
    } else {
        hipLaunchKernelGGL(route_count_kernel, dim3(nchunk + xqa.gx * xq_gy), dim3(64 * kRtWaves), 0, st, topi, P, n_exp,
                           hist, qctr, nchunk, xqa);
        hipLaunchKernelGGL(route_scatter_kernel, dim3(nchunk), dim3(64 * kRtWaves), 0, st, topi, P, n_exp, hist, counts,
                           offs, pairs, scores, sscore);
    }
    int rc = mxh::launch_status("moe_prefill route");
    if (rc != MXFP4_OK) return rc;

    GArgs g{};
    g.counts = counts;
    g.offs = offs;
    g.pairs = pairs;
    g.topk = topk;
    g.hq = ws + L.hq;
    g.hs = ws + L.hs;
    g.hld = Mp / 2;
    g.hsld = Mp / 32;
    g.yd = reinterpret_cast<uint16_t*>(ws + L.yd);
    g.sscore = sscore;

    g.aq = ws + L.xq;
    g.as = ws + L.xs;
    g.ald = Hp / 2;
    g.asld = Hp / 32;
    g.Kp = H;
    g.Nw = Mi;
    g.a_rows = T;
    rc = launch_xp<MODE_GATEUP>(g, w, n_exp, qctr, st);
    if (rc != MXFP4_OK) return rc;

    g.aq = ws + L.hq;
    g.as = ws + L.hs;
    g.ald = Mp / 2;
    g.asld = Mp / 32;
    g.Kp = Mi;
    g.Nw = H;
    g.a_rows = P;
    rc = launch_xp<MODE_DOWN>(g, w, n_exp, qctr + 8, st);
    if (rc != MXFP4_OK) return rc;

    const int64_t threads = (int64_t)T * (H / 8);
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    auto* combine = topk <= 8 && blocks < kCombineFew ? prefill_combine_kernel<true> : prefill_combine_kernel<false>;
    hipLaunchKernelGGL(combine, dim3(blocks), dim3(256), 0, st, reinterpret_cast<const uint16_t*>(ws + L.yd), topi, T, topk, H,
                       n_exp, static_cast<uint16_t*>(out));
    return mxh::launch_status("moe_prefill combine");
}

template <class W>
int run_prefill(const void* x, const int64_t* topi, const uint16_t* scores, W w, int n_exp, int T, int topk,
                int H, int Mi, void* out, void* workspace, size_t ws_bytes, hipStream_t st) {
    MXH_REQUIRE(x && topi && scores && out && workspace, "moe_prefill: null pointer");
    MXH_REQUIRE(T > 0 && topk > 0 && topk <= kMaxTopk, "moe_prefill: T=%d topk=%d (need T > 0, 0 < topk <= %d)",
                T, topk, kMaxTopk);
    MXH_REQUIRE(n_exp > 0 && n_exp <= kMaxExperts, "moe_prefill: n_experts=%d (1..%d)", n_exp, kMaxExperts);
    MXH_REQUIRE(H > 0 && H % 32 == 0 && Mi > 0 && Mi % 32 == 0,
                "moe_prefill: H=%d and Mi=%d must be positive multiples of 32", H, Mi);
    MXH_REQUIRE((int64_t)T * topk < (1ll << 31) / 2, "moe_prefill: T*topk too large");
    MXH_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)workspace & 255) == 0,
                "moe_prefill: x/out must be 16-byte and workspace 256-byte aligned");
    MXH_REQUIRE(ws_bytes >= ws_layout(T, topk, n_exp, H, Mi).total, "moe_prefill: workspace of %zu bytes < required %zu",
                ws_bytes, ws_layout(T, topk, n_exp, H, Mi).total);
    // the copies address the token and h rows with 31-bit byte offsets: more
    // tokens than that go in several passes, one after the other
    const int64_t row = std::max(pad256(H) / 2, topk * (pad256(Mi) / 2));
    MXH_REQUIRE(row < (1ll << 31), "moe_prefill: H=%d, topk=%d x Mi=%d too large", H, topk, Mi);
    const int per = (int)std::min<int64_t>(T, ((1ll << 31) - 1) / row);
    for (int t0 = 0; t0 < T; t0 += per) {
        const int rc = run_prefill_pass<W>(static_cast<const uint8_t*>(x) + (int64_t)t0 * H * 2, topi + (int64_t)t0 * topk,
                                           scores + (int64_t)t0 * topk, w, n_exp, std::min(per, T - t0), topk, H, Mi,
                                           static_cast<uint8_t*>(out) + (int64_t)t0 * H * 2, workspace, st);
        if (rc != MXFP4_OK) return rc;
    }
    return MXFP4_OK;
}

}  // namespace

extern "C" int mxfp4_moe_group(const int64_t* topi, int T, int topk, int n_experts, int* counts, int* offsets,
                               int* pairs, void* stream) {
    MXH_REQUIRE(topi && counts && offsets && pairs, "moe_group: null pointer");
    MXH_REQUIRE(T > 0 && topk > 0 && (int64_t)T * topk < (1ll << 30), "moe_group: T=%d topk=%d", T, topk);
    MXH_REQUIRE(n_experts > 0 && n_experts <= kMaxExperts, "moe_group: n_experts=%d (1..%d)", n_experts, kMaxExperts);
    hipLaunchKernelGGL(route_kernel, dim3((n_experts + kRouteEpw - 1) / kRouteEpw), dim3(64 * kRouteWaves), 0,
                       mxh::as_stream(stream), topi, T * topk, n_experts,
                       counts, offsets, pairs, nullptr, nullptr);
    return mxh::launch_status("moe_group");
}

extern "C" size_t mxfp4_moe_prefill_workspace_size(int T, int topk, int n_experts, int H, int Mi) {
    if (T <= 0 || topk <= 0 || n_experts <= 0 || H <= 0 || Mi <= 0) return 0;
    return ws_layout(T, topk, n_experts, H, Mi).total;
}

extern "C" int mxfp4_moe_prefill(const void* x, const int64_t* topi, const uint16_t* scores,
                                 const uint8_t* gate_wp, const uint8_t* gate_ws, const uint8_t* up_wp,
                                 const uint8_t* up_ws, const uint8_t* down_wp, const uint8_t* down_ws,
                                 int n_experts, int T, int topk, int H, int Mi, void* out, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    MXH_REQUIRE(gate_wp && gate_ws && up_wp && up_ws && down_wp && down_ws, "moe_prefill: null weight pointer");
    MXH_REQUIRE(((uintptr_t)gate_wp & 15) == 0 && ((uintptr_t)up_wp & 15) == 0 && ((uintptr_t)down_wp & 15) == 0,
                "moe_prefill: packed weights must be 16-byte aligned");
    StackedW w;
    w.wp[0] = gate_wp; w.ws[0] = gate_ws;
    w.wp[1] = up_wp;   w.ws[1] = up_ws;
    w.wp[2] = down_wp; w.ws[2] = down_ws;
    w.wp_stride[0] = w.wp_stride[1] = (int64_t)Mi * (H / 2);
    w.ws_stride[0] = w.ws_stride[1] = (int64_t)Mi * (H / 32);
    w.wp_stride[2] = (int64_t)H * (Mi / 2);
    w.ws_stride[2] = (int64_t)H * (Mi / 32);
    return run_prefill(x, topi, scores, w, n_experts, T, topk, H, Mi, out, workspace, workspace_bytes,
                       mxh::as_stream(stream));
}

extern "C" int mxfp4_moe_prefill_tab(const void* x, const int64_t* topi, const uint16_t* scores,
                                     const int64_t* expert_tab, int n_experts, int T, int topk, int H, int Mi,
                                     void* out, void* workspace, size_t workspace_bytes, void* stream) {
    MXH_REQUIRE(expert_tab, "moe_prefill_tab: null expert table");
    TableW w{expert_tab};
    return run_prefill(x, topi, scores, w, n_experts, T, topk, H, Mi, out, workspace, workspace_bytes,
                       mxh::as_stream(stream));
}
