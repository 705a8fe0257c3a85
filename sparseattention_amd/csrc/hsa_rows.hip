// Leaf rows and span-node rows as one 16-bit matrix, and the way back for their gradients.
//
// HierarchicalAttention.update_X_from_Y (reference hierarchical_attention/modules/attention.py:178-195)
// projects cat([x, y]) to keys and values.  Under autocast x and y come in fp32 and 16 bits: the
// concatenation is made in fp32, converted once per projection, and in the backward two fp32 copies of the
// gradients are added, cut apart, converted again and added to the query projection's.  Here the rows are
// converted on the way into one [B, N + M, C] matrix (x's also by themselves, for the queries); the
// backward adds the projections' input gradients in fp32 and writes each part in its own type.
//
// Bound: HBM; eight elements per thread, every row read and written once.  B8 N2048 C768, x fp32, y fp16:
// 27 us forward (151 MB, 5.6 TB/s), 34 us backward (201 MB, 5.9 TB/s); with them the module's training step
// takes 1744 us instead of 1961.
#include "hsa_common.h"

namespace hsa {

namespace {

struct alignas(16) Rows8 { uint16_t e[8]; };
struct alignas(16) Rows8F { float e[8]; };

template <typename T> __device__ __forceinline__ void rows_load(const void *p, long at, float (&f)[8]) {
    if constexpr (sizeof(typename T::storage) == 4) {
        const Rows8F v = *reinterpret_cast<const Rows8F *>((const float *)p + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = v.e[e];
    } else {
        const Rows8 v = *reinterpret_cast<const Rows8 *>((const uint16_t *)p + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = to_float<T>(v.e[e]);
    }
}
template <typename T> __device__ __forceinline__ void rows_store(void *p, long at, const float (&f)[8]) {
    if constexpr (sizeof(typename T::storage) == 4) {
        Rows8F v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v.e[e] = f[e];
        *reinterpret_cast<Rows8F *>((float *)p + at) = v;
    } else {
        Rows8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v.e[e] = from_float<T>(f[e]);
        *reinterpret_cast<Rows8 *>((uint16_t *)p + at) = v;
    }
}

struct RowsArgs {
    const void *a, *b;  // pack: x, y; unpack: the two gradients
    const void *c;      // unpack: a third gradient, of the rows of x alone (or null)
    void *o, *o2;       // pack: the matrix, x's rows once more by themselves (or null); unpack: dx, dy (either may be null)
    int N, M, C;
    long pieces;        // of the whole matrix
};

// piece i of the matrix -> element offset in the matrix and in x (from_x) or y
__device__ __forceinline__ bool rows_at(const RowsArgs &p, long i, long &at, long &part) {
    at = i * 8;
    const long row = at / p.C;
    const int c = (int)(at - row * p.C);
    const long b = row / (p.N + p.M);
    const int r = (int)(row - b * (p.N + p.M));
    const bool from_x = r < p.N;
    part = (from_x ? b * p.N + r : b * p.M + (r - p.N)) * p.C + c;
    return from_x;
}

template <typename T, typename X, typename Y>
__global__ void __launch_bounds__(256) pack_rows_kernel(RowsArgs p) {
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < p.pieces; i += (long)gridDim.x * 256) {
        long at, part;
        float f[8];
        const bool from_x = rows_at(p, i, at, part);
        if (from_x) rows_load<X>(p.a, part, f);
        else rows_load<Y>(p.b, part, f);
        rows_store<T>(p.o, at, f);
        if (from_x && p.o2) rows_store<T>(p.o2, part, f);
    }
}

template <typename T, typename X, typename Y>
__global__ void __launch_bounds__(256) add_split_rows_kernel(RowsArgs p) {
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < p.pieces; i += (long)gridDim.x * 256) {
        long at, part;
        const bool from_x = rows_at(p, i, at, part);
        if (!(from_x ? p.o : p.o2)) continue;
        float f[8], g[8];
        rows_load<T>(p.a, at, f);
        rows_load<T>(p.b, at, g);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] += g[e];
        if (from_x && p.c) {
            rows_load<T>(p.c, part, g);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] += g[e];
        }
        if (from_x) rows_store<X>(p.o, part, f);
        else rows_store<Y>(p.o2, part, f);
    }
}

template <typename T> int rows_launch(const RowsArgs &p, bool pack, bool x32, bool y32, hipStream_t st) {
    long wgs = (p.pieces + 255) / 256;
    if (wgs > 4096) wgs = 4096;  // sixteen workgroups on each of the 256 CUs
    const unsigned n = (unsigned)wgs;
#define HSA_ROWS(X, Y)                                               \
    if (pack) pack_rows_kernel<T, X, Y><<<n, 256, 0, st>>>(p);       \
    else add_split_rows_kernel<T, X, Y><<<n, 256, 0, st>>>(p)
    if (x32 && y32) { HSA_ROWS(F32, F32); }
    else if (x32) { HSA_ROWS(F32, T); }
    else if (y32) { HSA_ROWS(T, F32); }
    else { HSA_ROWS(T, T); }
#undef HSA_ROWS
    return check_launch(pack ? "pack_rows_kernel" : "add_split_rows_kernel");
}

int rows_checked(RowsArgs &p, bool pack, int B, int N, int M, int C, int x_dtype, int y_dtype, int dtype, hipStream_t st) {
    HSA_REQUIRE(B >= 1 && N >= 1 && M >= 1 && C >= 8 && C % 8 == 0, "bad shape B=%d N=%d M=%d C=%d", B, N, M, C);
    HSA_REQUIRE(dtype == HSA_F16 || dtype == HSA_BF16, "rows of a 16-bit type only (dtype %d)", dtype);
    HSA_REQUIRE((x_dtype == HSA_F32 || x_dtype == dtype) && (y_dtype == HSA_F32 || y_dtype == dtype), "bad part types %d, %d",
                x_dtype, y_dtype);
    HSA_REQUIRE((((uintptr_t)p.a | (uintptr_t)p.b | (uintptr_t)p.c | (uintptr_t)p.o | (uintptr_t)p.o2) & 15) == 0, "rows need 16-byte aligned tensors");
    p.N = N; p.M = M; p.C = C;
    p.pieces = (long)B * (N + M) * C / 8;
    return dtype == HSA_F16 ? rows_launch<F16>(p, pack, x_dtype == HSA_F32, y_dtype == HSA_F32, st)
                            : rows_launch<BF16>(p, pack, x_dtype == HSA_F32, y_dtype == HSA_F32, st);
}

}  // namespace

}  // namespace hsa

extern "C" {

int hsa_pack_rows(const void *x, const void *y, void *out, void *out_x, int B, int N, int M, int C, int x_dtype, int y_dtype,
                  int dtype, void *stream) {
    HSA_REQUIRE(x && y && out, "null pointer");
    hsa::RowsArgs p = {x, y, nullptr, out, out_x, 0, 0, 0, 0};
    return hsa::rows_checked(p, true, B, N, M, C, x_dtype, y_dtype, dtype, (hipStream_t)stream);
}

int hsa_add_split_rows(const void *a, const void *b, const void *c, void *dx, void *dy, int B, int N, int M, int C, int x_dtype,
                       int y_dtype, int dtype, void *stream) {
    HSA_REQUIRE(a && b && (dx || dy), "null pointer");
    hsa::RowsArgs p = {a, b, c, dx, dy, 0, 0, 0, 0};
    return hsa::rows_checked(p, false, B, N, M, C, x_dtype, y_dtype, dtype, (hipStream_t)stream);
}

}  // extern "C"
