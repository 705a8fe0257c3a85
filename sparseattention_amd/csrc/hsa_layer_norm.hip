// Residual sum and layer norm in one pass over the rows, forward and backward.
//
// The decoder layer of the reference's model (hierarchical_attention_project/
// Hierarchical_Transformer_Pretrain.py:375-428) adds a branch to its residual stream and hands the
// sum to a layer norm three times per layer.  Done as separate kernels that is six row-sized
// passes over memory (read a, b, write s; read s, write n; and the norm's own launch), and torch's
// layer norm kernel moves 67 MB in 45 us at B8 N4096 d512 bf16 (1.5 TB/s).
//
// Bound: HBM.  A row of C channels is held by a group of LPR lanes, 16 bytes per lane and piece, for
// as long as it is needed: every input is read once, the sum and the norm are written once.  Mean
// and variance are taken in two passes over the registers, in fp32, on the sum as rounded to the
// element type (what a separate norm would read).  A wavefront walks rows with the next row's
// pieces requested before the current one is reduced; weight and bias stay in registers.
// B8 N4096 d512 bf16 (134 MB): 25 us (5.4 TB/s) against 66 us for the two kernels it replaces; backward at
// B4 N1024 d512: 7.5 + 7.2 us against 13.4 + 11.6 us and the addition of the two gradients.
#include "hsa_common.h"

namespace hsa {

namespace {

constexpr int LN_THREADS = 256;

template <typename T> constexpr int ln_vec() { return 16 / (int)sizeof(typename T::storage); }

template <typename T> struct alignas(16) LnPiece { typename T::storage e[ln_vec<T>()]; };

template <typename T>
__device__ __forceinline__ void ln_unpack(const LnPiece<T> &p, float (&f)[ln_vec<T>()]) {
#pragma unroll
    for (int e = 0; e < ln_vec<T>(); ++e) f[e] = to_float<T>(p.e[e]);
}
template <typename T>
__device__ __forceinline__ LnPiece<T> ln_pack(const float (&f)[ln_vec<T>()]) {
    LnPiece<T> p;
#pragma unroll
    for (int e = 0; e < ln_vec<T>(); ++e) p.e[e] = from_float<T>(f[e]);
    return p;
}

struct LnArgs {
    const void *a, *b, *gamma, *beta;
    void *sum, *norm;
    float *stats;  // [rows, 2]: mean, reciprocal standard deviation (or null)
    long rows;
    int pieces;    // 16-byte pieces per row
    float inv_c, eps;
};

// LPR lanes hold a row, NP pieces each; ADD: the row is a + b, and the sum is written
template <typename T, int LPR, int NP, bool ADD>
__global__ void __launch_bounds__(LN_THREADS) add_layer_norm_kernel(LnArgs p) {
    constexpr int VEC = ln_vec<T>();
    using P = LnPiece<T>;
    const int sub = threadIdx.x % LPR;
    const long step = (long)gridDim.x * (LN_THREADS / LPR);
    long row = (long)blockIdx.x * (LN_THREADS / LPR) + threadIdx.x / LPR;
    if (row >= p.rows) return;
    bool has[NP];
    float ga[NP][VEC], be[NP][VEC];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int pc = i * LPR + sub;
        has[i] = pc < p.pieces;
        const int at = has[i] ? pc : 0;
        ln_unpack<T>(reinterpret_cast<const P *>(p.gamma)[at], ga[i]);
        ln_unpack<T>(reinterpret_cast<const P *>(p.beta)[at], be[i]);
    }
    P ra[NP], rb[NP];
    auto request = [&](long r) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const size_t at = (size_t)r * p.pieces + (has[i] ? i * LPR + sub : 0);
            ra[i] = reinterpret_cast<const P *>(p.a)[at];
            if constexpr (ADD) rb[i] = reinterpret_cast<const P *>(p.b)[at];
        }
    };
    request(row);
    while (true) {
        float v[NP][VEC];
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            ln_unpack<T>(ra[i], v[i]);
            if constexpr (ADD) {
                float w[VEC];
                ln_unpack<T>(rb[i], w);
                const size_t at = (size_t)row * p.pieces + i * LPR + sub;
                float t[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) t[e] = v[i][e] + w[e];
                const P o = ln_pack<T>(t);
                if (has[i]) reinterpret_cast<P *>(p.sum)[at] = o;
                ln_unpack<T>(o, v[i]);
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) s += has[i] ? v[i][e] : 0.f;
        }
        const long next = row + step;
        if (next < p.rows) request(next);
        const float mean = group_sum(s, LPR) * p.inv_c;
        float q = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                v[i][e] -= mean;
                q += has[i] ? v[i][e] * v[i][e] : 0.f;
            }
        const float rstd = 1.0f / sqrtf(group_sum(q, LPR) * p.inv_c + p.eps);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            float o[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) o[e] = fmaf(v[i][e] * rstd, ga[i][e], be[i][e]);
            if (has[i]) reinterpret_cast<P *>(p.norm)[(size_t)row * p.pieces + i * LPR + sub] = ln_pack<T>(o);
        }
        if (p.stats && sub == 0) {
            p.stats[2 * row] = mean;
            p.stats[2 * row + 1] = rstd;
        }
        if (next >= p.rows) break;
        row = next;
    }
}

struct LnBwdArgs {
    const void *dnorm, *dsum, *s, *gamma;
    const float *stats;
    void *dx;
    float *partial;  // [workgroups, 2, C]: sums of dnorm * xhat and of dnorm
    long rows;
    int pieces;
    float inv_c;
};

// dx = dsum + rstd * (g - mean(g) - xhat * mean(g * xhat)),  g = dnorm * gamma;  the weight's and the
// bias's gradients are summed over a workgroup's rows and written as one partial row
template <typename T, int LPR, int NP>
__global__ void __launch_bounds__(LN_THREADS) add_layer_norm_bwd_kernel(LnBwdArgs p) {
    constexpr int VEC = ln_vec<T>();
    constexpr int RPW = LN_THREADS / LPR;  // rows a workgroup works on at a time
    using P = LnPiece<T>;
    extern __shared__ float red[];         // [RPW - 1][LPR * NP * VEC] per gradient, one after the other
    const int sub = threadIdx.x % LPR, grp = threadIdx.x / LPR;
    const long step = (long)gridDim.x * RPW;
    bool has[NP];
    float ga[NP][VEC], dg[NP][VEC], db[NP][VEC];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int pc = i * LPR + sub;
        has[i] = pc < p.pieces;
        ln_unpack<T>(reinterpret_cast<const P *>(p.gamma)[has[i] ? pc : 0], ga[i]);
#pragma unroll
        for (int e = 0; e < VEC; ++e) { dg[i][e] = 0.f; db[i][e] = 0.f; }
    }
    P rn[NP], rs[NP], rd[NP];
    float mean = 0.f, rstd = 0.f;
    auto request = [&](long r) {
        mean = p.stats[2 * r];
        rstd = p.stats[2 * r + 1];
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const size_t at = (size_t)r * p.pieces + (has[i] ? i * LPR + sub : 0);
            rn[i] = reinterpret_cast<const P *>(p.dnorm)[at];
            rs[i] = reinterpret_cast<const P *>(p.s)[at];
            if (p.dsum) rd[i] = reinterpret_cast<const P *>(p.dsum)[at];
        }
    };
    long row = (long)blockIdx.x * RPW + grp;
    if (row < p.rows) request(row);
    for (; row < p.rows; row += step) {
        float x[NP][VEC], g[NP][VEC], d[NP][VEC];
        const float rstd_now = rstd;
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            ln_unpack<T>(rs[i], x[i]);
            ln_unpack<T>(rn[i], g[i]);
            if (p.dsum) ln_unpack<T>(rd[i], d[i]);
            else
#pragma unroll
                for (int e = 0; e < VEC; ++e) d[i][e] = 0.f;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                x[i][e] = (x[i][e] - mean) * rstd;
                dg[i][e] = fmaf(g[i][e], x[i][e], dg[i][e]);
                db[i][e] += g[i][e];
                g[i][e] *= ga[i][e];
                s1 += has[i] ? g[i][e] : 0.f;
                s2 += has[i] ? g[i][e] * x[i][e] : 0.f;
            }
        }
        if (row + step < p.rows) request(row + step);
        const float m1 = group_sum(s1, LPR) * p.inv_c, m2 = group_sum(s2, LPR) * p.inv_c;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            float o[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) o[e] = fmaf(rstd_now, g[i][e] - m1 - x[i][e] * m2, d[i][e]);
            if (has[i]) reinterpret_cast<P *>(p.dx)[(size_t)row * p.pieces + i * LPR + sub] = ln_pack<T>(o);
        }
    }
    // the workgroup's row groups meet in LDS, one gradient after the other
    constexpr int W = LPR * NP * VEC;
    const int C = p.pieces * VEC;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        float(&acc)[NP][VEC] = which == 0 ? dg : db;
        if (grp > 0)
#pragma unroll
            for (int i = 0; i < NP; ++i)
#pragma unroll
                for (int e = 0; e < VEC; ++e) red[(grp - 1) * W + (i * LPR + sub) * VEC + e] = acc[i][e];
        __syncthreads();
        if (grp == 0)
#pragma unroll
            for (int i = 0; i < NP; ++i)
                if (has[i]) {
                    float *o = p.partial + ((size_t)blockIdx.x * 2 + which) * C + (i * LPR + sub) * VEC;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        float t = acc[i][e];
                        for (int r = 0; r < RPW - 1; ++r) t += red[r * W + (i * LPR + sub) * VEC + e];
                        o[e] = t;
                    }
                }
        __syncthreads();
    }
}

// column sums of the partial rows: 64 columns and four row groups per workgroup
template <typename T>
__global__ void __launch_bounds__(256) layer_norm_grads_kernel(const float *partial, typename T::storage *dgamma,
                                                               typename T::storage *dbeta, int wgs, int C) {
    __shared__ float red[4][64];
    const int col = blockIdx.x * 64 + (threadIdx.x & 63), part = threadIdx.x >> 6;
    float t = 0.f;
    if (col < 2 * C) {
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        int i = part;
        for (; i + 12 < wgs; i += 16)
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] += partial[(size_t)(i + 4 * u) * 2 * C + col];
        for (; i < wgs; i += 4) a[0] += partial[(size_t)i * 2 * C + col];
        t = (a[0] + a[1]) + (a[2] + a[3]);
    }
    red[part][threadIdx.x & 63] = t;
    __syncthreads();
    if (part == 0 && col < 2 * C) {
        t = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
        if (col < C) dgamma[col] = from_float<T>(t);
        else dbeta[col - C] = from_float<T>(t);
    }
}

// workgroups of the backward: enough to fill the chip twice, at least four rows for every row group
int ln_bwd_wgs(long rows) {
    const long w = (rows + 15) / 16;
    return (int)(w < 1 ? 1 : w > 512 ? 512 : w);
}

template <typename T, int LPR, int NP>
int ln_launch(const LnArgs &p, hipStream_t st) {
    constexpr int RPW = LN_THREADS / LPR;
    long wgs = (p.rows + RPW - 1) / RPW;
    if (wgs > 2048) wgs = 2048;  // eight workgroups on each of the 256 CUs
    if (p.b) add_layer_norm_kernel<T, LPR, NP, true><<<(unsigned)wgs, LN_THREADS, 0, st>>>(p);
    else add_layer_norm_kernel<T, LPR, NP, false><<<(unsigned)wgs, LN_THREADS, 0, st>>>(p);
    return check_launch("add_layer_norm_kernel");
}

template <typename T, int LPR, int NP>
int ln_bwd_launch(const LnBwdArgs &p, void *dgamma, void *dbeta, hipStream_t st) {
    using S = typename T::storage;
    constexpr int VEC = ln_vec<T>(), RPW = LN_THREADS / LPR;
    const int wgs = ln_bwd_wgs(p.rows), C = p.pieces * VEC;
    const size_t lds = (size_t)(RPW - 1) * LPR * NP * VEC * sizeof(float);
    add_layer_norm_bwd_kernel<T, LPR, NP><<<wgs, LN_THREADS, lds, st>>>(p);
    int rc = check_launch("add_layer_norm_bwd_kernel");
    if (rc != HSA_OK) return rc;
    layer_norm_grads_kernel<T><<<(2 * C + 63) / 64, 256, 0, st>>>(p.partial, (S *)dgamma, (S *)dbeta, wgs, C);
    return check_launch("layer_norm_grads_kernel");
}

// lanes per row and pieces per lane: a row of up to 32 pieces takes half a wavefront, wider ones a
// wavefront with as few pieces per lane as hold the row
#define HSA_LN_SWITCH(T, pieces, CALL)                                              \
    if ((pieces) <= 32) return CALL(T, 32, 1);                                      \
    if ((pieces) <= 64) return CALL(T, 64, 1);                                      \
    if ((pieces) <= 128) return CALL(T, 64, 2);                                     \
    if ((pieces) <= 192) return CALL(T, 64, 3);                                     \
    if ((pieces) <= 256) return CALL(T, 64, 4);                                     \
    return fail(HSA_ERR_UNSUPPORTED, "layer norm rows of %d 16-byte pieces", (pieces));
constexpr int LN_MAX_PIECES = 256;

template <typename T> int ln_typed(const LnArgs &p, hipStream_t st) {
#define HSA_LN_CALL(T, LPR, NP) ln_launch<T, LPR, NP>(p, st)
    HSA_LN_SWITCH(T, p.pieces, HSA_LN_CALL)
#undef HSA_LN_CALL
}
template <typename T> int ln_bwd_typed(const LnBwdArgs &p, void *dgamma, void *dbeta, hipStream_t st) {
#define HSA_LN_CALL(T, LPR, NP) ln_bwd_launch<T, LPR, NP>(p, dgamma, dbeta, st)
    HSA_LN_SWITCH(T, p.pieces, HSA_LN_CALL)
#undef HSA_LN_CALL
}

}  // namespace

}  // namespace hsa

extern "C" {

int hsa_add_layer_norm_ok(int C, int dtype) {
    if (dtype != HSA_F32 && dtype != HSA_F16 && dtype != HSA_BF16) return 0;
    const int vec = 16 / hsa::elem_size(dtype);
    return C >= vec && C % vec == 0 && C / vec <= hsa::LN_MAX_PIECES;
}

int hsa_add_layer_norm_fwd(const void *a, const void *b, const void *gamma, const void *beta, void *sum, void *norm,
                           float *stats, long rows, int C, float eps, int dtype, void *stream) {
    HSA_REQUIRE(a && gamma && beta && norm, "null pointer");
    HSA_REQUIRE((b == nullptr) == (sum == nullptr), "the sum is written exactly when there is something to add");
    HSA_REQUIRE(rows >= 1, "bad row count %ld", rows);
    if (!hsa_add_layer_norm_ok(C, dtype)) return hsa::fail(HSA_ERR_UNSUPPORTED, "layer norm of %d channels, dtype %d", C, dtype);
    HSA_REQUIRE((((uintptr_t)a | (uintptr_t)b | (uintptr_t)gamma | (uintptr_t)beta | (uintptr_t)sum | (uintptr_t)norm) & 15) == 0,
                "layer norm needs 16-byte aligned tensors");
    const hsa::LnArgs p = {a, b, gamma, beta, sum, norm, stats, rows, C / (16 / hsa::elem_size(dtype)), 1.0f / C, eps};
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case HSA_F32: return hsa::ln_typed<hsa::F32>(p, st);
        case HSA_F16: return hsa::ln_typed<hsa::F16>(p, st);
        default: return hsa::ln_typed<hsa::BF16>(p, st);
    }
}

size_t hsa_add_layer_norm_bwd_workspace_bytes(long rows, int C) {
    return (size_t)hsa::ln_bwd_wgs(rows) * 2 * C * sizeof(float);
}

int hsa_add_layer_norm_bwd(const void *dnorm, const void *dsum, const void *s, const float *stats, const void *gamma,
                           void *dx, void *dgamma, void *dbeta, void *workspace, size_t workspace_bytes, long rows,
                           int C, int dtype, void *stream) {
    HSA_REQUIRE(dnorm && s && stats && gamma && dx && dgamma && dbeta && workspace, "null pointer");
    HSA_REQUIRE(rows >= 1, "bad row count %ld", rows);
    if (!hsa_add_layer_norm_ok(C, dtype)) return hsa::fail(HSA_ERR_UNSUPPORTED, "layer norm of %d channels, dtype %d", C, dtype);
    HSA_REQUIRE((((uintptr_t)dnorm | (uintptr_t)dsum | (uintptr_t)s | (uintptr_t)gamma | (uintptr_t)dx) & 15) == 0,
                "layer norm needs 16-byte aligned tensors");
    HSA_REQUIRE(workspace_bytes >= hsa_add_layer_norm_bwd_workspace_bytes(rows, C), "workspace too small (%zu bytes)", workspace_bytes);
    const hsa::LnBwdArgs p = {dnorm, dsum, s, gamma, stats, dx, (float *)workspace, rows, C / (16 / hsa::elem_size(dtype)), 1.0f / C};
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case HSA_F32: return hsa::ln_bwd_typed<hsa::F32>(p, dgamma, dbeta, st);
        case HSA_F16: return hsa::ln_bwd_typed<hsa::F16>(p, dgamma, dbeta, st);
        default: return hsa::ln_bwd_typed<hsa::BF16>(p, dgamma, dbeta, st);
    }
}

}  // extern "C"
