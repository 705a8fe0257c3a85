// Weight and bias gradient of a linear projection: dW[o, i] = sum over rows of dY[r, o] * X[r, i], db[o] =
// sum over rows of dY[r, o].  16-bit operands, fp32 sums.
//
// The contraction runs over the tokens (thousands) while the result has the size of a weight (a few
// hundred squared), so tiling the result alone leaves the chip idle: 768 x 768 over 16384 rows are 36
// tiles of 128 x 128 for 256 CUs, and the library's product takes 90 us (0.2 PFLOP/s).  Here the rows are
// split as well: a workgroup owns one 128 x 128 tile over one chunk of rows, and a second launch adds
// the chunks' fp32 partial tiles in a fixed order.  Several pairs (dY, X) whose products add up to one
// result (the levels of the span-node update) go into the same two launches.
//
// Both operands lie with the contraction as their slow dimension.  Rows go from global memory straight
// into LDS as they are (16 bytes a lane, four stages of 32 rows) and are transposed on the way out by
// ds_read_b64_tr_b16 (a group of 16 lanes reads a 4 x 16 block, each lane receives one column).  The
// 32-byte pieces of row r are permuted by (r & 3) | (r & 8) >> 1, applied on the global side of the
// transfer, so that the rows of two such blocks lie in different banks (no conflicts counted).  A
// stage's operands are read one step before they are multiplied (without that: 92 against 75 us for
// the launch at 32760 x 1536 x 768).
//
// Bound: the CU's LDS pipe together with the barrier per step: 0.28 us per 32 rows with one workgroup
// on a CU, 0.5 us for two, where the matrix cores alone would need 0.11 and 0.21.  Slower: operands
// transposed in registers with byte permutes on the way into LDS (102 us), tiles of 256 x 128 with
// a wavefront share of 128 x 64 (110 us: the accumulators spill into moves between register files).
//
// Both launches, us, against the library's product (bf16): rows x O x I
//   4096 x 512 x 512    16.6 / 27    16384 x 768 x 768    33 / 90     32767 x 768 x 768    50 / 191
//   4096 x 2048 x 512   22.6 / 29    16384 x 2304 x 768   67 / 127    32760 x 1536 x 768   81 / 208
// and the bias gradient, a reduction of 17 to 38 us of its own, adds 1 to 5 us here.
#include "hsa_lds_dma.h"

namespace hsa {

namespace {

constexpr int WG_ROWS = 32, WG_STAGES = 4, WG_THREADS = 256, WG_TILE = 128;
constexpr int WG_ROW_BYTES = 2 * WG_TILE;
constexpr int WG_ARRAY = WG_ROWS * WG_ROW_BYTES;  // one operand's rows of a stage
constexpr int WG_STAGE = 2 * WG_ARRAY;            // four of them: 64 KiB, two workgroups per CU
constexpr int WG_ROUND = WG_ROWS * WG_STAGES;  // rows per round through the stages; a chunk is a multiple

struct WgSeg {
    const char *dy, *x;
    long ld_dy, ld_x;  // bytes
    long rows, chunk;
    int O, o_first, tiles, first_block, splits;
    float *partial;    // [splits, O, I]
};
struct WgArgs {
    WgSeg seg[HSA_WEIGHT_GRAD_MAX_SEGMENTS];
    int nseg, I, i_tiles;
    float *bias_partial;  // [splits of the first segment, O] or null
};

__device__ const uint4 wg_zero_piece = {0, 0, 0, 0};

typedef short wg_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2_t lds_read_tr(const char *p) {
    return __builtin_bit_cast(
        u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) wg_s16x4 *)p));
}

template <typename T>
__global__ void __launch_bounds__(WG_THREADS, 2) weight_grad_kernel(WgArgs p) {
    __shared__ __attribute__((aligned(1024))) char lds[WG_STAGES * WG_STAGE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r = lane & 15;
    // consecutive work items run on one XCD: the tiles of a chunk read the same rows, from its L2
    const int nb = gridDim.x, xcd = blockIdx.x & 7, per = nb >> 3, rest = nb & 7;
    int item = xcd * per + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
    int s = 0;
    while (s + 1 < p.nseg && item >= p.seg[s + 1].first_block) ++s;
    const WgSeg sg = p.seg[s];
    const int I = p.I;
    item -= sg.first_block;
    const int tile = item % sg.tiles, split = item / sg.tiles;
    const int o0 = tile / p.i_tiles * WG_TILE, i0 = tile % p.i_tiles * WG_TILE;
    const long row0 = (long)split * sg.chunk;
    const long row1 = row0 + sg.chunk < sg.rows ? row0 + sg.chunk : sg.rows;
    const int steps = (int)((row1 - row0 + WG_ROWS - 1) / WG_ROWS);

    // this lane's pieces of the rows it transfers: rows 8 w + 4 j + g of a stage, slot r; columns behind the
    // matrix (last tile): any piece of the row, the products are not stored
    const int piece = 8 * ((((r >> 1) ^ (g | ((w & 1) << 2))) << 1) | (r & 1));
    const int cx = i0 + piece < I ? i0 + piece : 0, cd = o0 + piece < sg.O ? o0 + piece : 0;
    const uint32_t lds0 = lds_address(lds);
    const uintptr_t zero = (uintptr_t)&wg_zero_piece, base_x = (uintptr_t)sg.x + 2 * cx, base_dy = (uintptr_t)sg.dy + 2 * cd;
    auto request = [&](int step, int buf) {
        const uint32_t base = lds0 + buf * WG_STAGE + w * (WG_ARRAY / 4);
        const long row = row0 + (long)step * WG_ROWS + 8 * w + g;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool in = row + 4 * j < row1;  // rows behind the chunk: zeros on both sides
            uintptr_t px = base_x + (row + 4 * j) * sg.ld_x, pd = base_dy + (row + 4 * j) * sg.ld_dy;
            px = in ? px : zero;
            pd = in ? pd : zero;
            lds_dma16_pair((const void *)px, (const void *)pd, base + 1024 * j, base + WG_ARRAY + 1024 * j);
        }
    };

    // wavefront (w >> 1, w & 1) of the tile: 64 columns of X by 64 of dY
    const int wm = w >> 1, wn = w & 1;
    const int rd_swz = (r >> 2) | ((g & 1) << 2), rd_row = 8 * g + (r >> 2), rd_in = 16 * ((r >> 1) & 1) + 8 * (r & 1);
    int rd_x[4], rd_dy[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        rd_x[t] = rd_row * WG_ROW_BYTES + rd_in + 32 * ((wm * 4 + t) ^ rd_swz);
        rd_dy[t] = WG_ARRAY + rd_row * WG_ROW_BYTES + rd_in + 32 * ((wn * 4 + t) ^ rd_swz);
    }
    f32x4 acc[4][4], bias[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        bias[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    constexpr uint32_t one2 = Mma<T>::kOne | ((uint32_t)Mma<T>::kOne << 16);
    const u32x4_t ones = {one2, one2, one2, one2};
    const bool with_bias = p.bias_partial && i0 == 0 && wm == 0 && s == 0;

    struct Operands { u32x4_t x[4], dy[4]; };
    auto fetch = [&](const char *stage, Operands &v) {
        auto column = [](const char *q) {
            const u32x2_t a = lds_read_tr(q), b = lds_read_tr(q + 4 * WG_ROW_BYTES);
            return u32x4_t{a[0], a[1], b[0], b[1]};
        };
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v.x[t] = column(stage + rd_x[t]);
            v.dy[t] = column(stage + rd_dy[t]);
        }
    };
    auto products = [&](const Operands &v) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = Mma<T>::k32(v.x[i], v.dy[j], acc[i][j]);
        if (with_bias)
#pragma unroll
            for (int j = 0; j < 4; ++j) bias[j] = Mma<T>::k32(ones, v.dy[j], bias[j]);
    };

    // When step t begins, stage t is in registers and stages t + 1 .. t + 3 are in flight or there; behind
    // the barrier stage t + 1 is there for everyone and nobody reads stage t's buffer any more, which takes
    // stage t + 4.  Stages behind the last fetch zeros, so the number of transfers in flight is always
    // the same.
#pragma unroll
    for (int t = 0; t < WG_STAGES; ++t) request(t, t);
    Operands v[2];
    wait_vmem_all_but<4 * (WG_STAGES - 1)>();  // four transfers per stage
    lds_only_barrier();
    fetch(lds, v[0]);
    for (int step = 0; step < steps; step += WG_STAGES) {
#pragma unroll
        for (int u = 0; u < WG_STAGES; ++u) {
            wait_vmem_all_but<4 * (WG_STAGES - 2)>();
            lds_only_barrier();
            request(step + u + WG_STAGES, u);
            fetch(lds + (u + 1) % WG_STAGES * WG_STAGE, v[(u + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
            products(v[u & 1]);
        }
    }
    wait_vmem_all_but<0>();  // no transfer outlives the workgroup's LDS

    float *out = sg.partial + (size_t)split * sg.O * I;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int o = o0 + wn * 64 + j * 16 + r;
        if (o >= sg.O) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = i0 + (wm * 4 + i) * 16 + 4 * g;
            if (c < I) *reinterpret_cast<f32x4 *>(out + (size_t)o * I + c) = acc[i][j];
        }
        if (with_bias && g == 0) p.bias_partial[(size_t)split * sg.O + o] = bias[j][0];
    }
}

struct WgReduce {
    const float *partial[HSA_WEIGHT_GRAD_MAX_SEGMENTS];
    int o_first[HSA_WEIGHT_GRAD_MAX_SEGMENTS], O[HSA_WEIGHT_GRAD_MAX_SEGMENTS], splits[HSA_WEIGHT_GRAD_MAX_SEGMENTS];
    int nseg, rows, I;
    void *dw;
    const float *bias_partial;
    void *dbias;
};

// the chunks' partial results added up in a fixed order, four elements per thread; the threads behind
// them do the bias
template <typename T>
__global__ void __launch_bounds__(256) weight_grad_reduce_kernel(WgReduce p) {
    using S = typename T::storage;
    const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 4, n = (long)p.rows * p.I;
    if (at < n) {
        const int o = (int)(at / p.I), i = (int)(at % p.I);
        f32x4 t[4] = {};
        for (int s = 0; s < p.nseg; ++s) {
            const int so = o - p.o_first[s];
            if (so < 0 || so >= p.O[s]) continue;
            const float *src = p.partial[s] + (size_t)so * p.I + i;
            const size_t slab = (size_t)p.O[s] * p.I;
            int k = 0;
            for (; k + 4 <= p.splits[s]; k += 4)
#pragma unroll
                for (int u = 0; u < 4; ++u) t[u] += *reinterpret_cast<const f32x4 *>(src + (k + u) * slab);
            for (; k < p.splits[s]; ++k) t[0] += *reinterpret_cast<const f32x4 *>(src + k * slab);
        }
        const f32x4 sum = (t[0] + t[1]) + (t[2] + t[3]);
        S *dst = (S *)p.dw + at;
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = from_float<T>(sum[e]);
        return;
    }
    const long o = (at - n) / 4;
    if (!p.dbias || o >= p.O[0]) return;
    float t = 0.f;
    for (int k = 0; k < p.splits[0]; ++k) t += p.bias_partial[(size_t)k * p.O[0] + o];
    ((S *)p.dbias)[o] = from_float<T>(t);
}

int tiles_of(int n) { return (n + WG_TILE - 1) / WG_TILE; }

// Rows per chunk: the least of (steps of a workgroup) x (time of a step, which grows with the
// workgroups a CU holds) + (partial results written and read back), with the measured times of a step and
// 5 TB/s for the partial results.  Within 4 % of the best chunk in a sweep of 1 to 64 chunks over 14
// sizes from 256 x 512 x 512 to 32760 x 1536 x 768.
long chunk_rows(int nseg, const hsa_weight_grad_segment *seg, int I) {
    long most = 0;
    for (int s = 0; s < nseg; ++s) most = seg[s].rows > most ? seg[s].rows : most;
    long best = 0, before = 0;
    double least = 0;
    for (long n = 1; n <= 128; ++n) {
        const long chunk = ((most + n - 1) / n + WG_ROUND - 1) / WG_ROUND * WG_ROUND;
        if (chunk == before) continue;
        before = chunk;
        double blocks = 0, bytes = 0;
        for (int s = 0; s < nseg; ++s) {
            const double splits = (double)((seg[s].rows + chunk - 1) / chunk);
            blocks += splits * tiles_of(seg[s].O) * tiles_of(I);
            bytes += 8.0 * splits * seg[s].O * I;
        }
        const double step = blocks <= 256 ? 0.285 : 0.5 * (double)(((long)blocks + 511) / 512);  // us per 32 rows
        const double us = step * (double)(chunk / WG_ROWS) + bytes * 2e-7;
        if (best == 0 || us < least) {
            best = chunk;
            least = us;
        }
        if (chunk == WG_ROUND) break;
    }
    return best;
}

bool segments_ok(int nseg, const hsa_weight_grad_segment *seg, int I) {
    if (nseg < 1 || nseg > HSA_WEIGHT_GRAD_MAX_SEGMENTS || !seg || I < 8 || I % 8) return false;
    for (int s = 0; s < nseg; ++s)
        if (seg[s].rows < 1 || seg[s].O < 8 || seg[s].O % 8 || seg[s].o_first < 0 || seg[s].o_first % 4 ||
            (long)tiles_of(seg[s].O) * tiles_of(I) > (1 << 20))
            return false;
    return true;
}

}  // namespace

}  // namespace hsa

extern "C" {

size_t hsa_weight_grad_workspace_bytes(int nseg, const hsa_weight_grad_segment *seg, int I, int with_bias) {
    if (!hsa::segments_ok(nseg, seg, I)) return 0;
    const long chunk = hsa::chunk_rows(nseg, seg, I);
    size_t fl = 0;
    for (int s = 0; s < nseg; ++s) fl += (size_t)((seg[s].rows + chunk - 1) / chunk) * seg[s].O * I;
    if (with_bias) fl += (size_t)((seg[0].rows + chunk - 1) / chunk) * seg[0].O;
    return fl * sizeof(float);
}

int hsa_weight_grad(int nseg, const hsa_weight_grad_segment *seg, int O, int I, void *dw, void *dbias, int out_dtype,
                    void *workspace, size_t workspace_bytes, int dtype, void *stream) {
    using namespace hsa;
    HSA_REQUIRE(dw && workspace && seg, "null pointer");
    HSA_REQUIRE(dtype == HSA_F16 || dtype == HSA_BF16, "weight gradient of 16-bit operands only (dtype %d)", dtype);
    HSA_REQUIRE(out_dtype == HSA_F32 || out_dtype == dtype, "bad result type %d", out_dtype);
    if (!segments_ok(nseg, seg, I)) return fail(HSA_ERR_UNSUPPORTED, "weight gradient: sizes not handled (I=%d)", I);
    HSA_REQUIRE(!dbias || (nseg == 1 && seg[0].o_first == 0 && seg[0].O == O), "a bias gradient goes with one segment");
    uintptr_t bits = (uintptr_t)dw | (uintptr_t)workspace;
    for (int s = 0; s < nseg; ++s) {
        HSA_REQUIRE(seg[s].dy && seg[s].x, "null pointer");
        HSA_REQUIRE(seg[s].o_first + seg[s].O <= O, "segment %d writes rows %d..%d of %d", s, seg[s].o_first,
                    seg[s].o_first + seg[s].O, O);
        HSA_REQUIRE(seg[s].ld_dy >= seg[s].O && seg[s].ld_x >= I, "segment %d: row stride below the row's length", s);
        bits |= (uintptr_t)seg[s].dy | (uintptr_t)seg[s].x | (uintptr_t)(2 * seg[s].ld_dy) | (uintptr_t)(2 * seg[s].ld_x);
    }
    HSA_REQUIRE((bits & 15) == 0, "weight gradient needs 16-byte aligned rows");
    HSA_REQUIRE(workspace_bytes >= hsa_weight_grad_workspace_bytes(nseg, seg, I, dbias != nullptr),
                "workspace too small (%zu bytes)", workspace_bytes);
    const long chunk = chunk_rows(nseg, seg, I);
    WgArgs p = {};
    WgReduce q = {};
    float *ws = (float *)workspace;
    long blocks = 0;
    p.nseg = q.nseg = nseg;
    p.I = q.I = I;
    p.i_tiles = tiles_of(I);
    for (int s = 0; s < nseg; ++s) {
        WgSeg &t = p.seg[s];
        t.dy = (const char *)seg[s].dy;
        t.x = (const char *)seg[s].x;
        t.ld_dy = 2 * seg[s].ld_dy;
        t.ld_x = 2 * seg[s].ld_x;
        t.rows = seg[s].rows;
        t.chunk = chunk;
        t.O = seg[s].O;
        t.o_first = seg[s].o_first;
        t.tiles = tiles_of(t.O) * p.i_tiles;
        t.first_block = (int)blocks;
        t.splits = (int)((t.rows + chunk - 1) / chunk);
        t.partial = ws;
        ws += (size_t)t.splits * t.O * I;
        blocks += (long)t.tiles * t.splits;
        q.partial[s] = t.partial;
        q.o_first[s] = t.o_first;
        q.O[s] = t.O;
        q.splits[s] = t.splits;
    }
    HSA_REQUIRE(blocks < (1l << 31), "too many tiles");
    if (dbias) p.bias_partial = ws;
    q.rows = O;
    q.dw = dw;
    q.bias_partial = p.bias_partial;
    q.dbias = dbias;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == HSA_F16) weight_grad_kernel<F16><<<(unsigned)blocks, WG_THREADS, 0, st>>>(p);
    else weight_grad_kernel<BF16><<<(unsigned)blocks, WG_THREADS, 0, st>>>(p);
    int rc = check_launch("weight_grad_kernel");
    if (rc != HSA_OK) return rc;
    const long threads = (long)O * I / 4 + (dbias ? O : 0);
    const unsigned grid = (unsigned)((threads + 255) / 256);
    if (out_dtype == HSA_F32) weight_grad_reduce_kernel<F32><<<grid, 256, 0, st>>>(q);
    else if (dtype == HSA_F16) weight_grad_reduce_kernel<F16><<<grid, 256, 0, st>>>(q);
    else weight_grad_reduce_kernel<BF16><<<grid, 256, 0, st>>>(q);
    return check_launch("weight_grad_reduce_kernel");
}

}  // extern "C"
