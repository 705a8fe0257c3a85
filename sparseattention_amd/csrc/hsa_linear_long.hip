// Product with a long contraction: out[r, n] = sum over k of X[r, k] * W[k, n], 16-bit operands, fp32 sums: the input
// gradient of a vocabulary projection, where K is the vocabulary (tens of thousands, of any number: the rows
// of X begin at any element) and the result small.
//
// 4096 x 512 with K = 50257 are 32 tiles of 256 x 256 for 256 CUs; the library's product takes 543 us.  Here the
// contraction is split as well (every workgroup one tile over one part of it, one part per XCD, whose rows
// of W its L2 then holds once) and a second launch adds the fp32 partial tiles in a fixed order: 247 us.
// Tile, stages and operand order as in hsa_linear.hip; the rows of X come through registers (16 bytes a lane
// from any address, which the direct transfer does not promise) and are written to the LDS a step later.
//
// Bound: the matrix cores, 211 GFLOP at 1.2 PFLOP/s; the partial tiles, 67 MB there and back, add 20 us.
#include "hsa_lds_dma.h"

namespace hsa {

namespace {

constexpr int LL_TILE = 256, LL_STEP = 64, LL_THREADS = 512;
constexpr int LL_XB = LL_TILE * LL_STEP * 2, LL_STAGE = 2 * LL_XB, LL_PITCH = 2 * LL_TILE;

typedef u32x4_t LlPiece __attribute__((aligned(2)));
typedef short ll_s16x4 __attribute__((ext_vector_type(4)));

struct LlArgs {
    const char *x, *w;
    float *partial;    // [splits, M, N]
    long ld_x, ld_w;   // bytes
    int M, N, K, chunk, col_tiles, tiles;
};

__device__ const uint4 ll_zero_piece = {0, 0, 0, 0};

__device__ __forceinline__ u32x2_t ll_read_tr(const char *p) {
    return __builtin_bit_cast(
        u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ll_s16x4 *)p));
}

template <typename T>
__global__ void __launch_bounds__(LL_THREADS, 2) linear_long_kernel(LlArgs p) {
    __shared__ __attribute__((aligned(1024))) char lds[2 * LL_STAGE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r = lane & 15, wm = w >> 1, wn = w & 1;
    const uint32_t lds0 = lds_address(lds);
    // consecutive items on one XCD: the tiles of one part of the contraction
    const int per = gridDim.x >> 3, rest = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int item = xcd * per + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
    const int split = item / p.tiles, tile = item - split * p.tiles, rt = tile / p.col_tiles;
    int m0 = rt * LL_TILE, n0 = (tile - rt * p.col_tiles) * LL_TILE;
    m0 = m0 < p.M - LL_TILE ? m0 : p.M - LL_TILE;  // (the last ones flush with the end)
    n0 = n0 < p.N - LL_TILE ? n0 : p.N - LL_TILE;
    const int k0 = split * p.chunk, k1 = k0 + p.chunk < p.K ? k0 + p.chunk : p.K;
    const int steps = (k1 - k0 + LL_STEP - 1) / LL_STEP;

    // ---- transfers.  X: rows 32 w + 8 q + lane / 8, piece lane & 7, permuted; W: rows of the contraction 8 w + 2 q +
    // lane / 32, piece lane & 31, permuted in pairs.
    const int lrow = lane >> 3, lslot = lane & 7;
    const char *load_x = p.x + (long)(m0 + 32 * w + lrow) * p.ld_x + 2l * k0;
    const char *load_w = p.w + (long)(k0 + 8 * w) * p.ld_w + 2l * n0;
    u32x4_t xr[4];
    auto piece_of = [&](int q) { return lslot ^ ((lrow >> 1) | ((q & 1) << 2)); };
    uint32_t off_w[4];
    const int wrow = lane >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = 8 * w + 2 * q + wrow, key = (row & 3) | ((row & 8) >> 1), piece = lane & 31;
        off_w[q] = (uint32_t)(2 * q + wrow) * (uint32_t)p.ld_w + 16 * (((piece >> 1) ^ key) << 1 | (piece & 1));
    }
    auto load = [&](int s) {
        if (s >= steps) return;
        const int left = k1 - k0 - s * LL_STEP;  // contraction elements from this stage on
        const char *x = load_x + s * (2l * LL_STEP), *wb = load_w + (long)s * LL_STEP * p.ld_w;
        const uint32_t to = lds0 + (s & 1) * LL_STAGE + LL_XB + w * 4096;
        if (left >= LL_STEP) {
#pragma unroll
            for (int q = 0; q < 4; ++q) xr[q] = *(const LlPiece *)(x + 8 * q * p.ld_x + 16 * piece_of(q));
#pragma unroll
            for (int q = 0; q < 4; ++q) lds_dma16(wb + off_w[q], to + q * 1024);
        } else {  // the end of the contraction: zeros behind it on both sides
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int at = 8 * piece_of(q);
                const uint16_t *e = (const uint16_t *)(x + 8 * q * p.ld_x) + at;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t lo = at + 2 * i < left ? e[2 * i] : 0, hi = at + 2 * i + 1 < left ? e[2 * i + 1] : 0;
                    xr[q][i] = lo | hi << 16;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const void *a = 8 * w + 2 * q + wrow < left ? (const void *)(wb + off_w[q]) : (const void *)&ll_zero_piece;
                lds_dma16(a, to + q * 1024);
            }
        }
    };
    auto keep = [&](int s) {  // a stage's rows of X from the registers to their place
        if (s >= steps) return;
        char *to = lds + (s & 1) * LL_STAGE + w * 4096 + 16 * lane;
#pragma unroll
        for (int q = 0; q < 4; ++q) *(u32x4_t *)(to + q * 1024) = xr[q];
    };

    // ---- operands, as in hsa_linear.hip
    int rd_x[2], rd_w[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd_x[h] = (wm * 64 + r) * 128 + 16 * ((4 * h + g) ^ (r >> 1));
#pragma unroll
    for (int j = 0; j < 8; ++j)
        rd_w[j] = LL_XB + (8 * g + (r >> 2)) * LL_PITCH + 32 * ((wn * 8 + j) ^ ((r >> 2) | ((g & 1) << 2))) + 8 * (r & 3);
    u32x4_t ox[2][4], ow[8];
    auto fetch_x = [&](int buf, int h, u32x4_t (&o)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = *(const u32x4_t *)(lds + buf * LL_STAGE + rd_x[h] + i * 2048);
    };
    auto fetch_w = [&](int buf, int h, int j) {
        const char *q = lds + buf * LL_STAGE + rd_w[j] + h * 32 * LL_PITCH;
        const u32x2_t a = ll_read_tr(q), b = ll_read_tr(q + 4 * LL_PITCH);
        ow[j] = u32x4_t{a[0], a[1], b[0], b[1]};
    };
    f32x4 acc[4][8];  // [16 rows][16 columns]: lane (g, r) holds row r, columns 4 g ..
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](const u32x4_t (&x)[4], int buf, int h, u32x4_t (&next)[4]) {
        fetch_x(buf, h, next);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][j] = Mma<T>::k32(ow[j], x[i], acc[i][j]);
            fetch_w(buf, h, j);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    load(0);
    keep(0);
    wait_vmem_all_but<0>();
    lds_only_barrier();
    load(1);
    fetch_x(0, 0, ox[0]);
#pragma unroll
    for (int j = 0; j < 8; ++j) fetch_w(0, 0, j);
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        products(ox[0], buf, 1, ox[1]);
        // the next stage is there; its rows of X go to where the stage before this one lay, which everybody has
        // read; behind the barrier this one's place takes the stage after next
        wait_vmem_all_but<0>();
        keep(s + 1);
        lds_only_barrier();
        load(s + 2);
        __builtin_amdgcn_sched_barrier(0);
        products(ox[1], buf ^ 1, 0, ox[0]);  // (behind the last stage: operands that nothing uses)
    }
    float *out = p.partial + ((long)split * p.M + m0 + wm * 64 + r) * p.N + n0 + wn * 128 + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) *(f32x4 *)(out + (long)(16 * i) * p.N + 16 * j) = acc[i][j];
}

// the parts added up in a fixed order, eight elements per thread
template <typename T>
__global__ void __launch_bounds__(256) linear_long_sum_kernel(const float *partial, int splits, long slab, int N, long ld_out, char *out) {
    const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (at >= slab) return;
    f32x4 t[2] = {};
#pragma unroll 4
    for (int s = 0; s < splits; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) t[h] += *(const f32x4 *)(partial + s * slab + at + 4 * h);
    const long row = at / N, col = at - row * N;
    *(u32x4_t *)(out + row * ld_out + 2 * col) =
        u32x4_t{Mma<T>::pack(t[0][0], t[0][1]), Mma<T>::pack(t[0][2], t[0][3]), Mma<T>::pack(t[1][0], t[1][1]), Mma<T>::pack(t[1][2], t[1][3])};
}

struct LlPlan {
    int row_tiles, col_tiles, chunk, splits;
};

// about one workgroup per CU; the parts of the contraction are whole steps
LlPlan plan(int M, int N, int K) {
    LlPlan q;
    q.row_tiles = (M + LL_TILE - 1) / LL_TILE;
    q.col_tiles = (N + LL_TILE - 1) / LL_TILE;
    const int tiles = q.row_tiles * q.col_tiles, want = tiles >= 256 ? 1 : 256 / tiles, steps = (K + LL_STEP - 1) / LL_STEP;
    q.chunk = (steps + want - 1) / want * LL_STEP;
    q.splits = (K + q.chunk - 1) / q.chunk;
    return q;
}

bool handled(int M, int N, int K, int dtype) {
    return (dtype == HSA_F16 || dtype == HSA_BF16) && M >= LL_TILE && N >= LL_TILE && N % 8 == 0 && K >= 2 * LL_STEP &&
           M <= (1 << 20) && N <= (1 << 16) && K <= (1 << 24) && (long)M * N <= (1l << 31);
}

}  // namespace

}  // namespace hsa

extern "C" {

size_t hsa_linear_long_workspace_bytes(int M, int N, int K, int dtype) {
    if (!hsa::handled(M, N, K, dtype)) return 0;
    const hsa::LlPlan q = hsa::plan(M, N, K);
    return (size_t)q.splits * M * N * sizeof(float);
}

int hsa_linear_long_pays(int M, int N, int K, int dtype) {
    if (!hsa::handled(M, N, K, dtype)) return 0;
    // us, library / here (M x N, K): 1024 x 512, 50257 270 / 76; 4096 x 512, 50257 525 / 247; 8192 x 512, 50257 585 / 484; 4096 x
    // 768, 50257 550 / 375; 4096 x 512, 10001 93 / 66; 2048 x 768, 5003 49 / 41.  Not: 8192 x 768, 50257 662 / 827 (192 workgroups),
    // 4096 x 256, 4001 32 / 35, 1024 x 256, 2001 13 / 30.
    const hsa::LlPlan q = hsa::plan(M, N, K);
    const int blocks = q.row_tiles * q.col_tiles * q.splits;
    return K >= 5000 && M >= 512 && q.splits > 1 && blocks >= 230 && blocks <= 256;
}

int hsa_linear_long(const void *x, int64_t ld_x, const void *w, int64_t ld_w, void *out, int64_t ld_out, int M, int N, int K,
                    void *workspace, size_t workspace_bytes, int dtype, void *stream) {
    using namespace hsa;
    HSA_REQUIRE(x && w && out && workspace, "null pointer");
    if (!handled(M, N, K, dtype)) return fail(HSA_ERR_UNSUPPORTED, "long contraction: sizes not handled (M=%d N=%d K=%d)", M, N, K);
    HSA_REQUIRE(ld_x >= K && ld_w >= N && ld_out >= N && ld_x <= (1l << 25) && ld_w <= (1l << 25), "bad row strides");
    HSA_REQUIRE(ld_w % 8 == 0 && ld_out % 8 == 0 && (((uintptr_t)w | (uintptr_t)out | (uintptr_t)workspace) & 15) == 0 && ((uintptr_t)x & 1) == 0,
                "long contraction needs 16-byte aligned rows of the weight and the result");
    HSA_REQUIRE(workspace_bytes >= hsa_linear_long_workspace_bytes(M, N, K, dtype), "workspace too small (%zu bytes)", workspace_bytes);
    const LlPlan q = plan(M, N, K);
    LlArgs p = {(const char *)x, (const char *)w, (float *)workspace, 2 * (long)ld_x, 2 * (long)ld_w, M, N, K, q.chunk, q.col_tiles,
                q.row_tiles * q.col_tiles};
    const unsigned grid = (unsigned)(p.tiles * q.splits), sums = (unsigned)(((long)M * N / 8 + 255) / 256);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == HSA_F16) linear_long_kernel<F16><<<grid, LL_THREADS, 0, st>>>(p);
    else linear_long_kernel<BF16><<<grid, LL_THREADS, 0, st>>>(p);
    const int rc = check_launch("linear_long_kernel");
    if (rc != HSA_OK) return rc;
    if (dtype == HSA_F16) linear_long_sum_kernel<F16><<<sums, 256, 0, st>>>(p.partial, q.splits, (long)M * N, N, 2 * (long)ld_out, (char *)out);
    else linear_long_sum_kernel<BF16><<<sums, 256, 0, st>>>(p.partial, q.splits, (long)M * N, N, 2 * (long)ld_out, (char *)out);
    return check_launch("linear_long_sum_kernel");
}

}  // extern "C"
