// Span attention of one query and head by one wavefront, touching only the rows the query attends.
//
// Lanes first act as "one lane per attention slot" (window slots 0..2R, then the L tree slots): each lane
// fetches its key row and forms the full dot product, so the softmax statistics need only wave-wide
// max / sum reductions.  For the value pass the lanes switch to "one lane per output channel": the slot
// weights and rows are broadcast lane by lane and V rows are read coalesced.
#pragma once
#include "hsa_common.h"

namespace hsa {

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Tables: idx / mask [N, L], or the canonical ones with `causal` (idx null).  CHUNKS: 2R+1+L <= 64 * CHUNKS.
struct GatherTables {
    const int32_t *idx;
    const uint8_t *mask;
    int N, L, R, causal;
};

// q, o: the query's rows of this head; k, v: the first key / value row of this batch element and head, row_stride
// elements apart; w: the query's weights [2R+1+L] or null; lse: its log-sum-exp (log2 domain) or null.
// zero_if_dead: a query whose scores are all -inf gets zeros instead of NaN.
template <typename T, int CHUNKS>
__device__ __forceinline__ void gather_query(const GatherTables &t, int n, const typename T::storage *q,
                                             const typename T::storage *k, const typename T::storage *v,
                                             size_t row_stride, int D, float scale, bool zero_if_dead,
                                             typename T::storage *o, float *w, float *lse) {
    const int lane = threadIdx.x & 63;
    const int Wn = 2 * t.R + 1, S = Wn + t.L;
    int row[CHUNKS];
    float sc[CHUNKS];
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int s = c * 64 + lane;
        int r = -1;
        if (s < Wn) {
            int j = n + s - t.R;
            if (j >= 0 && j < t.N && (!t.causal || j <= n)) r = j;
        } else if (s < S) {
            int l = s - Wn;
            int m;
            bool dead;
            if (t.idx) {
                m = t.idx[(size_t)n * t.L + l];
                dead = (m == -1) || (t.mask && t.mask[(size_t)n * t.L + l] != 0);
            } else {
                m = level_offset(t.N, l) + ((n >> l) ^ 1);
                dead = t.causal && (((n >> l) & 1) == 0);
            }
            if (!dead) r = m;
        }
        row[c] = r;
        float x = -INFINITY;
        if (r >= 0) {
            const typename T::storage *kr = k + (size_t)r * row_stride;
            float acc = 0.f;
            for (int d = 0; d < D; ++d) acc = fmaf(to_float<T>(q[d]), to_float<T>(kr[d]), acc);
            x = acc * scale;
        }
        sc[c] = x;
        mx = fmaxf(mx, x);
    }
    mx = wave_max(mx);
    if (zero_if_dead && mx == -INFINITY) mx = 0.f;
    float den = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        float e = (row[c] >= 0) ? expf(sc[c] - mx) : 0.f;
        sc[c] = e;
        den += e;
    }
    den = wave_sum(den);
    den = fmaxf(den, 1.0e-5f);
    if (lse && lane == 0) *lse = (mx + logf(den)) * 1.4426950408889634f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) sc[c] = sc[c] / den;
    if (w) {
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            const int s = c * 64 + lane;
            if (s < S) w[s] = sc[c];
        }
    }
    for (int d0 = 0; d0 < D; d0 += 64) {
        const int d = d0 + lane;
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            const int lim = S - c * 64 < 64 ? S - c * 64 : 64;
            for (int s = 0; s < lim; ++s) {
                int r = __shfl(row[c], s, 64);
                float p = __shfl(sc[c], s, 64);
                if (r >= 0 && d < D) acc = fmaf(p, to_float<T>(v[(size_t)r * row_stride + d]), acc);
            }
        }
        if (d < D) o[d] = from_float<T>(acc);
    }
}

}  // namespace hsa
