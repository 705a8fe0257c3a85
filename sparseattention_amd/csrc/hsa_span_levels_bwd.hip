// Backward of the small levels of the span-node update, one launch per level.
//
// The levels of HierarchicalAttention.cross_update_Y (reference
// hierarchical_attention/modules/attention.py:119-157) depend on one another: the gradient of a
// level's rows is what the projections of the level above send down, d = [dK | dV] [Wk; Wv], plus the
// rows' own.  With a matrix product and a parent backward per level that is two dependent launches of
// 6 to 10 us each while a level has a few hundred rows, whatever it computes.
//
// Here a workgroup of four wavefronts owns 16 rows of a level and one head.  The product for these
// rows and this head's channels is split over the wavefronts along the contraction (2 H Dh long),
// operands streamed from L2 in MFMA order (rows as they lie, weights put in that order once by the caller); the
// four partial tiles meet in LDS, and the same workgroup runs the parent backward on them: d never
// reaches memory and is not rounded.  The parents' rows are requested before the product.
//
// Bound: latency of one dependent launch (a head's weights, 4 H Dh^2 bytes, from L2 per workgroup) up to
// about 256 rows over the batch, beyond that the weights read again by every 16 rows.  us per level,
// fp16, 12 heads of 64 channels: 7.0 to 7.6 up to 256 rows, 13.5 at 512, 30 at 2048 (8 heads: 5.6 to 5.9,
// 6.6, 16.6) against 14 to 17 for the product and the parent backward.  Weights as plain transposed rows (64
// bytes a row and step) took 11.1 instead of 7.2; eight wavefronts with the whole contraction in flight 13.6.
#include "hsa_mma.h"

namespace hsa {

namespace {

constexpr int SB_WAVES = 4, SB_THREADS = 64 * SB_WAVES;

struct SpanBwdArgs {
    const uint16_t *dy, *qkv, *kv, *w_kv;  // first level's first row of each
    uint16_t *dqkv, *dkv;
    int B, P, H;              // parents of this level per batch element
    int lgP;
    long dy_bs, dy_rs, qkv_bs, qkv_rs, dqkv_bs, dqkv_rs, kv_bs;
    long par_row, child_row;  // this level's first parent row (dy, qkv) and first child row (kv)
    long up_row;              // the rows' own row as children of the level above, -1: the root level
    float scale;
};

template <typename T> __device__ __forceinline__ void sb_unpack(u32x2_t v, float (&f)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = to_float<T>((uint16_t)(v[e >> 1] >> (16 * (e & 1))));
}
template <typename T> __device__ __forceinline__ u32x2_t sb_pack(float a, float b, float c, float d) {
    return u32x2_t{Mma<T>::pack(a, b), Mma<T>::pack(c, d)};
}

template <typename T, int DH>
__global__ void __launch_bounds__(SB_THREADS) span_level_bwd_kernel(SpanBwdArgs p) {
    constexpr int NT = DH / 16, LPR = DH / 4;  // 16-column tiles; lanes per (row, head), four channels each
    constexpr int NK = 4;                      // contraction steps in flight per wavefront
    constexpr int PASSES = LPR > 16 ? 2 : 1;   // the workgroup holds 16 rows of up to 64 channels at a time
    __shared__ __align__(16) float part[SB_WAVES][16][DH];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r = lane & 15;
    const int h = blockIdx.y, Dm = p.H * DH, rows = p.B * p.P;
    const int m0 = blockIdx.x * 16;

    // the parents' and children's pieces of this thread's (row, four channels), requested first
    u32x2_t rq[PASSES], rk[PASSES], rv[PASSES], k0[PASSES], k1[PASSES], v0[PASSES], v1[PASSES], rg[PASSES];
    long o_dqkv[PASSES], o_dkv[PASSES];
    bool live[PASSES];
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
        const int u = s * SB_THREADS + (int)threadIdx.x;
        const int rr = (u / LPR) & 15, c = h * DH + 4 * (u % LPR);
        const int m = m0 + rr;
        live[s] = u < 16 * LPR && m < rows;
        const int mm = m < rows ? m : rows - 1;
        const int b = mm >> p.lgP, i = mm & (p.P - 1);
        const uint16_t *par = p.qkv + b * p.qkv_bs + (p.par_row + i) * p.qkv_rs + c;
        const uint16_t *chl = p.kv + b * p.kv_bs + (p.child_row + 2 * i) * (2 * Dm) + c;
        rg[s] = *reinterpret_cast<const u32x2_t *>(p.dy + b * p.dy_bs + (p.par_row + i) * p.dy_rs + c);
        rq[s] = *reinterpret_cast<const u32x2_t *>(par);
        rk[s] = *reinterpret_cast<const u32x2_t *>(par + Dm);
        rv[s] = *reinterpret_cast<const u32x2_t *>(par + 2 * Dm);
        k0[s] = *reinterpret_cast<const u32x2_t *>(chl);
        v0[s] = *reinterpret_cast<const u32x2_t *>(chl + Dm);
        k1[s] = *reinterpret_cast<const u32x2_t *>(chl + 2 * Dm);
        v1[s] = *reinterpret_cast<const u32x2_t *>(chl + 3 * Dm);
        o_dqkv[s] = b * p.dqkv_bs + (p.par_row + i) * p.dqkv_rs + c;
        o_dkv[s] = b * p.kv_bs + (p.child_row + 2 * i) * (2 * Dm) + c;
    }

    const bool inner = p.up_row >= 0;
    if (inner) {
        // d[row, channel] over this wavefront's share of the contraction steps
        const int m = m0 + r < rows ? m0 + r : rows - 1;
        const uint16_t *a = p.dkv + (m >> p.lgP) * p.kv_bs + (p.up_row + (m & (p.P - 1))) * (2 * Dm) + 8 * g;
        const int nsteps = 2 * Dm / 32;
        const uint16_t *b = p.w_kv + (long)h * NT * nsteps * 512 + 8 * lane;
        f32x4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int first = w; first < nsteps; first += NK * SB_WAVES) {
            u32x4_t x[NK], y[NK][NT];
#pragma unroll
            for (int s = 0; s < NK; ++s) {  // steps behind the end fetch the first one again and count as zero
                const int k = first + s * SB_WAVES, at = k < nsteps ? k : first;
                x[s] = *reinterpret_cast<const u32x4_t *>(a + 32 * at);
#pragma unroll
                for (int t = 0; t < NT; ++t) y[s][t] = *reinterpret_cast<const u32x4_t *>(b + ((long)t * nsteps + at) * 512);
            }
            __builtin_amdgcn_sched_barrier(0);  // every request before the first product
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                if (first + s * SB_WAVES >= nsteps) {
                    x[s] = u32x4_t{0, 0, 0, 0};
#pragma unroll
                    for (int t = 0; t < NT; ++t) y[s][t] = u32x4_t{0, 0, 0, 0};
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = Mma<T>::k32(x[s], y[s][t], acc[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[w][4 * g + e][16 * t + r] = acc[t][e];
    }
    __syncthreads();

#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
        const int u = s * SB_THREADS + (int)threadIdx.x;
        const int rr = (u / LPR) & 15, c = 4 * (u % LPR);
        float q[4], kp[4], vp[4], a0[4], a1[4], b0[4], b1[4], d[4];
        sb_unpack<T>(rg[s], d);
        sb_unpack<T>(rq[s], q);
        sb_unpack<T>(rk[s], kp);
        sb_unpack<T>(rv[s], vp);
        sb_unpack<T>(k0[s], a0);
        sb_unpack<T>(k1[s], a1);
        sb_unpack<T>(v0[s], b0);
        sb_unpack<T>(v1[s], b1);
        if (inner) {
            f32x4 t0 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < SB_WAVES; ++i) t0 += *reinterpret_cast<const f32x4 *>(&part[i][rr][c]);
#pragma unroll
            for (int e = 0; e < 4; ++e) d[e] += t0[e];
        }
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, p0 = 0.f, p1 = 0.f, p2 = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s0 = fmaf(q[e], kp[e], s0);
            s1 = fmaf(q[e], a0[e], s1);
            s2 = fmaf(q[e], a1[e], s2);
            p0 = fmaf(d[e], vp[e], p0);
            p1 = fmaf(d[e], b0[e], p1);
            p2 = fmaf(d[e], b1[e], p2);
        }
        s0 = group_sum(s0, LPR) * p.scale; s1 = group_sum(s1, LPR) * p.scale; s2 = group_sum(s2, LPR) * p.scale;
        p0 = group_sum(p0, LPR); p1 = group_sum(p1, LPR); p2 = group_sum(p2, LPR);
        const float mx = fmaxf(s0, fmaxf(s1, s2));
        const float e0 = expf(s0 - mx), e1 = expf(s1 - mx), e2 = expf(s2 - mx);
        const float den = e0 + e1 + e2 + 1e-9f;
        const float w0 = e0 / den, w1 = e1 / den, w2 = e2 / den;
        const float dot = w0 * p0 + w1 * p1 + w2 * p2;
        const float ds0 = w0 * (p0 - dot) * p.scale, ds1 = w1 * (p1 - dot) * p.scale, ds2 = w2 * (p2 - dot) * p.scale;
        if (!live[s]) continue;
        float dq[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) dq[e] = ds0 * kp[e] + ds1 * a0[e] + ds2 * a1[e];
        auto put = [&](uint16_t *o, float f, const float (&x)[4]) {
            *reinterpret_cast<u32x2_t *>(o) = sb_pack<T>(f * x[0], f * x[1], f * x[2], f * x[3]);
        };
        uint16_t *par = p.dqkv + o_dqkv[s], *chl = p.dkv + o_dkv[s];
        put(par, 1.0f, dq);
        put(par + Dm, ds0, q);
        put(par + 2 * Dm, w0, d);
        put(chl, ds1, q);
        put(chl + Dm, w1, d);
        put(chl + 2 * Dm, ds2, q);
        put(chl + 3 * Dm, w2, d);
    }
}

}  // namespace

}  // namespace hsa

extern "C" {

int hsa_span_levels_bwd(const void *dy, const void *qkv, const void *kv, const void *w_kv, void *dqkv, void *dkv, int B,
                        int C, int H, int Dh, int64_t dy_bs, int64_t dy_rs, int64_t qkv_bs, int64_t qkv_rs,
                        int64_t dqkv_bs, int64_t dqkv_rs, int dtype, void *stream) {
    using namespace hsa;
    HSA_REQUIRE(dy && qkv && kv && w_kv && dqkv && dkv, "null pointer");
    HSA_REQUIRE(B >= 1 && C >= 2 && H >= 1 && ilog2_exact(C) >= 1, "bad shape B=%d C=%d H=%d", B, C, H);
    if ((dtype != HSA_F16 && dtype != HSA_BF16) || (Dh != 32 && Dh != 64 && Dh != 128) || H > 65535 ||
        (long)B * C > (1l << 30))
        return fail(HSA_ERR_UNSUPPORTED, "span levels backward: H=%d Dh=%d dtype=%d not handled", H, Dh, dtype);
    const int64_t Dm = (int64_t)H * Dh;
    HSA_REQUIRE(dy_rs >= Dm && qkv_rs >= 3 * Dm && dqkv_rs >= 3 * Dm, "row stride below the row's length");
    // rows are moved in pieces of four elements, dkv rows and weights in pieces of eight
    HSA_REQUIRE((((uintptr_t)dy | (uintptr_t)qkv | (uintptr_t)dqkv | (uintptr_t)(2 * (dy_bs | dy_rs | qkv_bs | qkv_rs | dqkv_bs | dqkv_rs))) & 7) == 0 &&
                    (((uintptr_t)kv | (uintptr_t)dkv | (uintptr_t)w_kv) & 15) == 0,
                "span levels backward needs 8-byte aligned rows (kv, dkv and the weights 16)");
    SpanBwdArgs p = {};
    p.dy = (const uint16_t *)dy; p.qkv = (const uint16_t *)qkv; p.kv = (const uint16_t *)kv; p.w_kv = (const uint16_t *)w_kv;
    p.dqkv = (uint16_t *)dqkv; p.dkv = (uint16_t *)dkv;
    p.B = B; p.H = H;
    p.dy_bs = dy_bs; p.dy_rs = dy_rs; p.qkv_bs = qkv_bs; p.qkv_rs = qkv_rs; p.dqkv_bs = dqkv_bs; p.dqkv_rs = dqkv_rs;
    p.kv_bs = (long)(2 * C - 2) * 2 * Dm;
    p.scale = 1.0f / sqrtf((float)Dh);
    hipStream_t st = (hipStream_t)stream;
    // from the root down: level t has C >> (t + 1) parents
    for (int t = ilog2_exact(C) - 1; t >= 0; --t) {
        p.P = C >> (t + 1);
        p.lgP = ilog2_exact(p.P);
        p.par_row = C - (C >> t);
        p.child_row = 2 * (long)C - ((2 * (long)C) >> t);
        p.up_row = p.P == 1 ? -1 : 2 * (long)C - ((2 * (long)C) >> (t + 1));
        const dim3 grid((unsigned)(((long)B * p.P + 15) / 16), (unsigned)H);
#define HSA_SPAN_BWD(TT)                                                          \
    if (Dh == 32) span_level_bwd_kernel<TT, 32><<<grid, SB_THREADS, 0, st>>>(p);         \
    else if (Dh == 64) span_level_bwd_kernel<TT, 64><<<grid, SB_THREADS, 0, st>>>(p);    \
    else span_level_bwd_kernel<TT, 128><<<grid, SB_THREADS, 0, st>>>(p)
        if (dtype == HSA_F16) { HSA_SPAN_BWD(F16); } else { HSA_SPAN_BWD(BF16); }
#undef HSA_SPAN_BWD
        const int rc = check_launch("span_level_bwd_kernel");
        if (rc != HSA_OK) return rc;
    }
    return HSA_OK;
}

}  // extern "C"
