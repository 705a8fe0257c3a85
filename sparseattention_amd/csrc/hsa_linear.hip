// Linear projections: out[r, n] = sum over k of X[r, k] * W[n, k] (+ bias[n]), and with the weight read the other
// way round, sum over k of X[r, k] * W[k, n] (the input gradient of a projection).  16-bit operands, fp32 sums.
// Several projections of one contraction length (the queries, keys and values of leaves and nodes) go into one
// launch, each with row blocks that lie apart in memory on either side (the leaves' and the nodes' rows of
// the joined key buffer).
//
// Why not the library's product: the contraction is short (up to 768; read the other way round up to 2304), so at
// 512 a tile is 8 steps of 64 and then 128 KB of results; the library starts a workgroup per tile, which pays for
// its first rows and its last stores each time.  Here a workgroup stays on its CU and walks tiles: the rows of the
// next tile's first two steps are requested before the results of the last one are stored.
//
// Tile 256 x 256 (or 256 x 192 where that leaves fewer CUs idle in the last round), eight wavefronts of 64 rows by
// 128 (96) columns.  Two stages of 64 contraction steps, both operands straight into LDS; a row's 16-byte pieces are
// permuted by its number, on the global side of the transfer, so that operand reads meet no bank twice.  Each step is
// two halves of 32: while one is multiplied, the operands of the next are read (the X side into a second set
// of registers, the W side in place, a fragment after its last use).  The last tiles of a row or column
// range lie flush with its end and compute what they share with their neighbour twice, to the same bits:
// no partial tiles.  The products are taken as (columns of the result) x (rows), so that a lane holds four
// consecutive columns; two exchanges between lanes make 128-byte lines of eight rows out of them
// (16 x 64 bytes: 1930 us at 32768 x 50304 x 512, lines 1890, lines stored past the caches 1550).
//
// Results whose rows begin at any element (a vocabulary of odd size): a line that two tiles share costs more
// than the line.  With rows enough, a tile takes every 64th row: their results lie alike in their lines, so the
// tiles' columns can begin where the lines do (32768 x 50257 x 512: 1710 us; the library 2160).  Else the rows go
// through the LDS and are stored as 16-byte pieces where they lie (4096 x 50257 x 512: 230 to 250 us, the library 330 to
// 350; stored as they come 330, before the XCDs' walks began apart).
//
// The transfers of a stage are requested one by one between the products of a half step: together, behind the
// barrier, they hold up all wavefronts at once (32768 x 2048 x 512: 73.3 -> 70.2 us, 16376 x 768 x 2304 55.7 -> 50.0).
//
// Bound: the matrix cores (1.4 PFLOP/s in the steps) and, not overlapped with them, the stores of the results
// at the rate of the memory (a third of the time at 32768 x 2048 x 512; the matrix cores are busy for 46 % of it, and
// for 63 % at 16384 x 768 x 2304).  Not faster (66 us on the same card): two workgroups of 128 x 256 on a CU, whose
// stores would overlap (82); four wavefronts for the transfers alone, so that none waits for its stores (72); starts
// spread over a tile's time (66).
#include "hsa_lds_dma.h"

#include <cmath>
#include <type_traits>

namespace hsa {

namespace {

constexpr int LN_STEP = 64;

struct LnSeg {
    const char *x, *w;
    const uint16_t *bias;
    char *out;
    long ld_x, ld_w, ld_out, batch_x, batch_out;  // bytes
    int rows, cols;                                // per batch element
    int row_tiles, col_tiles;                      // row_tiles: per batch element
    int all_row_tiles, first;                      // over the batch; first tile
    int period;                                    // ANY: tiles hold every period-th row, whose results lie alike in lines
};
struct LnArgs {
    LnSeg seg[HSA_LINEAR_MAX_SEGMENTS];
    int nseg, K, tiles, group;
};

// Where tile t lies: rows m0, m0 + period .. of batch element b of a segment, columns from n0.  `group` row tiles, column
// by column, then the next.
struct LnPlace {
    int seg, b, m0, n0;
};
template <int BM, int BN, int ANY>
__host__ __device__ __forceinline__ LnPlace place_of(const LnArgs &p, int t) {
    LnPlace c;
    c.seg = 0;
    while (c.seg + 1 < p.nseg && t >= p.seg[c.seg + 1].first) ++c.seg;
    const LnSeg &s = p.seg[c.seg];
    t -= s.first;
    const int per_group = p.group * s.col_tiles, grp = t / per_group, in = t - grp * per_group;
    const int left = s.all_row_tiles - grp * p.group, rows = left < p.group ? left : p.group;
    const int ct = in / rows, rt = grp * p.group + in - ct * rows;
    c.b = rt / s.row_tiles;
    c.m0 = (rt - c.b * s.row_tiles) * BM;
    c.n0 = ct * BN;
    if constexpr (ANY == 2) {
        const int each = s.row_tiles / s.period, in_batch = rt - c.b * s.row_tiles, rho = in_batch / each;
        const int rows = (s.rows - rho + s.period - 1) / s.period - BM, at = (in_batch - rho * each) * BM;
        c.m0 = rho + s.period * (at < rows ? at : rows);
        // whole lines: all but the first and the last columns' tiles begin where a line does
        if (ct) c.n0 -= (int)(((uintptr_t)s.out + c.b * s.batch_out + c.m0 * s.ld_out) & 127) / 2;
    } else {
        c.m0 = c.m0 < s.rows - BM ? c.m0 : s.rows - BM;
    }
    c.n0 = c.n0 < s.cols - BN ? c.n0 : s.cols - BN;
    return c;
}

// The tiles of an XCD: consecutive ones, since they share rows of X and W in its L2.  Where rows go through the LDS
// (ANY == 1) the walks begin in the middle, an eighth of the columns apart: with the same number of row tiles each, all
// eight XCDs would ask for the same columns' weights at the same time from beginning to end (us, library / together /
// apart, 48305 columns: 14336 x 256 645 / 804 / 565, 10240 x 256 463 / 578 / 391, 14336 x 512 908 / 1037 / 798).
struct LnWalk {
    int first, count, shift;
    __host__ __device__ __forceinline__ int tile(int t) const {
        t += shift;
        return first + (t < count ? t : t - count);
    }
};
template <int ANY> __host__ __device__ __forceinline__ LnWalk walk_of(const LnArgs &p, int xcd) {
    const int per = p.tiles >> 3, rest = p.tiles & 7;
    LnWalk w = {xcd * per + (xcd < rest ? xcd : rest), per + (xcd < rest), 0};
    if (ANY == 1 && w.count) {
        const int per_group = p.group * p.seg[0].col_tiles, ahead = (xcd * per_group / 8 - w.first) % per_group;
        w.shift = w.count < per_group ? (int)((long)xcd * w.count / 8) : ahead < 0 ? ahead + per_group : ahead;
    }
    return w;
}

// one transfer of 1 KiB: a scalar base and 32-bit offsets per lane
__device__ __forceinline__ void lds_dma16_from(const char *base, uint32_t off, uint32_t lds) {
    uint32_t keep;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(off), "s"(base), "s"(lds)
        : "memory");
}

// lane l's 2 bytes, as the low half of LDS[lds_base + 4 l]
__device__ __forceinline__ void lds_dma2(const void *g, uint32_t lds_base) {
    uint32_t keep;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_ushort %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(g), "s"(lds_base)
        : "memory");
}

__device__ const uint16_t ln_no_bias[256] = {};

typedef u32x4_t LnLoosePiece __attribute__((aligned(2)));

typedef short ln_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2_t ln_read_tr(const char *p) {
    return __builtin_bit_cast(
        u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ln_s16x4 *)p));
}

// BM, BN: rows and columns of a tile; TW: W is [K, N] instead of [N, K]; PAST: results stored past the caches;
// ANY: rows of the result begin at any element (2: tiles of rows that lie alike in lines)
template <typename T, int BM, int BN, bool TW, bool PAST, int ANY = 0>
__global__ void __launch_bounds__(2 * BM, 2) linear_kernel(LnArgs p) {
    constexpr int XB = BM * LN_STEP * 2, STAGE = XB + BN * LN_STEP * 2;  // bytes of a stage
    constexpr int NJ = BN / 32, NP = NJ / 2, QW = BN * 4 / BM;
    constexpr int PITCH = 2 * BN;  // of a row of W in the LDS, TW
    __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
    __shared__ __attribute__((aligned(16))) uint32_t lds_bias[2][BN];
    constexpr int OUT_PITCH = BN + 16;  // bytes: a wavefront's columns of a row, and 16 so that rows lie in other banks
    __shared__ __attribute__((aligned(16))) char lds_out[ANY == 1 ? BM / 32 * 8 * OUT_PITCH : 16];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r = lane & 15, wm = w >> 1, wn = w & 1;
    const uint32_t lds0 = lds_address(lds);
    const LnWalk walk = walk_of<ANY>(p, blockIdx.x & 7);
    const int count = walk.count, slots = gridDim.x >> 3, slot = blockIdx.x >> 3;
    if (slot >= count) return;
    auto tile_of = [&](int t) { return place_of<BM, BN, ANY>(p, walk.tile(t)); };

    // ---- transfers.  X: rows 32 w + 8 q + lane / 8, piece lane & 7 of 8.  W likewise (8 QW w + ..), or, TW,
    // rows of the contraction: pieces (w QW + q) 64 + lane of rows of BN / 8.
    // (offsets per lane that differ otherwise than by whole rows: X and W two each; at TW and 192 columns all three)
    constexpr int W_OFFSETS = TW && BN == 192 ? 3 : 2;
    constexpr auto w_kind = [](int q) { return TW && BN == 192 ? q : TW && BN == 128 ? q >> 1 : q & 1; };
    constexpr auto w_rows = [](int q) { return !TW ? (q & ~1) * 8 : BN == 192 ? 0 : BN == 128 ? (q & 1) * 4 : (q >> 1) * 4; };
    const int lrow = lane >> 3, lslot = lane & 7;
    uint32_t off_x[2], off_w[W_OFFSETS];
    long ld_x = 0, ld_w = 0;
    const char *load_x = nullptr, *load_w = nullptr;
    int lt = slot, lk = 0, lbuf = 0;
    auto aim = [&]() {
        const LnPlace c = tile_of(lt);
        const LnSeg &s = p.seg[c.seg];
        ld_x = ANY == 2 ? s.period * s.ld_x : s.ld_x;
        ld_w = s.ld_w;
        load_x = s.x + c.b * s.batch_x + c.m0 * s.ld_x + w * 32 * ld_x;
        load_w = TW ? s.w + 2l * c.n0 : s.w + (long)(c.n0 + w * 8 * QW) * ld_w;
#pragma unroll
        for (int q = 0; q < 2; ++q) off_x[q] = (uint32_t)(8 * q + lrow) * (uint32_t)ld_x + 16 * (lslot ^ ((lrow >> 1) | (q << 2)));
#pragma unroll
        for (int o = 0; o < W_OFFSETS; ++o) {
            if constexpr (TW) {
                const int q = BN == 128 ? 2 * o : o, at = (w * QW + q) * 64 + lane, row = at / (BN / 8), piece = at - row * (BN / 8);
                const int key = BN != 192 ? (row & 3) | ((row & 8) >> 1) : ((row >> 1) & 1) | ((row >> 2) & 2);
                off_w[o] = (uint32_t)row * (uint32_t)ld_w + 16 * (((piece >> 1) ^ key) << 1 | (piece & 1));
            } else {
                off_w[o] = (uint32_t)(8 * o + lrow) * (uint32_t)ld_w + 16 * (lslot ^ ((lrow >> 1) | (((w * QW + o) & 1) << 2)));
            }
        }
    };
    // transfer q of the stage that the cursor is at (4 of X's rows, QW of W's)
    auto load_one = [&](int q) {
        const uint32_t to = lds0 + lbuf * STAGE;
        if (q < 4) {
            lds_dma16_from(load_x + 2l * lk + (q & 2) * 8 * ld_x, off_x[q & 1], to + w * 4096 + q * 1024);
        } else {
            const int v = q - 4;
            lds_dma16_from((TW ? load_w + lk * ld_w : load_w + 2l * lk) + w_rows(v) * ld_w, off_w[w_kind(v)],
                           to + XB + w * (QW * 1024) + v * 1024);
        }
    };
    auto advance = [&]() {  // (behind the last stage: the last one once more, which nothing reads)
        lbuf ^= 1;
        if (lk + LN_STEP < p.K) {
            lk += LN_STEP;
        } else if (lt + slots < count) {
            lk = 0;
            lt += slots;
            aim();
        }
    };
    auto load = [&]() {
#pragma unroll
        for (int q = 0; q < 4 + QW; ++q) load_one(q);
        advance();
    };

    // ---- operands: lane (g, r) holds row r of X's 16, column r of W's, contraction 8 g .. of 32
    int rd_x[2], rd_w[TW ? NJ : 2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd_x[h] = (wm * 64 + r) * 128 + 16 * ((4 * h + g) ^ (r >> 1));
    if constexpr (TW) {
        // a group of 16 lanes reads 4 rows by 16 columns, lane i the i & 3-th four columns of row i >> 2
        const int key = BN != 192 ? (r >> 2) | ((g & 1) << 2) : ((r >> 3) & 1) | ((g & 1) << 1);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            rd_w[j] = XB + (8 * g + (r >> 2)) * PITCH + 32 * ((wn * NJ + j) ^ key) + 8 * (r & 3);
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) rd_w[h] = XB + (wn * (BN / 2) + r) * 128 + 16 * ((4 * h + g) ^ (r >> 1));
    }
    u32x4_t ox[2][4], ow[NJ];
    auto fetch_x = [&](int buf, int h, u32x4_t (&o)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = *(const u32x4_t *)(lds + buf * STAGE + rd_x[h] + i * 2048);
    };
    auto fetch_w = [&](int buf, int h, int j) {
        if constexpr (TW) {
            const char *q = lds + buf * STAGE + rd_w[j] + h * 32 * PITCH;
            const u32x2_t a = ln_read_tr(q), b = ln_read_tr(q + 4 * PITCH);
            ow[j] = u32x4_t{a[0], a[1], b[0], b[1]};
        } else {
            ow[j] = *(const u32x4_t *)(lds + buf * STAGE + rd_w[h] + j * 2048);
        }
    };
    f32x4 acc[4][NJ];  // [16 rows][16 columns]: lane (g, r) holds row r, columns 4 g ..
    // The products of 32 contraction steps while the next operands (half h of `buf`) take the places of those used up
    // and, LOAD, the transfers of a stage are requested.
    auto products = [&](auto LOAD, const u32x4_t (&x)[4], int buf, int h, u32x4_t (&next)[4]) {
        fetch_x(buf, h, next);
        if constexpr (!LOAD) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i][j] = Mma<T>::k32(ow[j], x[i], acc[i][j]);
                fetch_w(buf, h, j);
            }
            // (the order written here is the order issued)
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, TW ? 2 : 1, 0);
            }
        } else {
            // a transfer between products: requested together they would hold up all wavefronts at once
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i][j] = Mma<T>::k32(ow[j], x[i], acc[i][j]);
                fetch_w(buf, h, j);
#pragma unroll
                for (int q = j * (4 + QW) / NJ; q < (j + 1) * (4 + QW) / NJ; ++q) load_one(q);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<bool, true> with_loads;
    const std::integral_constant<bool, false> without;

    // the bias of a tile's columns, one per thread
    auto load_bias = [&](const LnPlace &c, int to) {
        const uint16_t *b = p.seg[c.seg].bias;
        const int at = (int)threadIdx.x;
        if (at < BN) lds_dma2(b ? b + c.n0 + at : ln_no_bias + at, lds_address(lds_bias[to]) + 256 * w);
    };
    LnPlace c = tile_of(slot);
    int which = 0;
    load_bias(c, 0);
    aim();
    load();
    load();
    int buf = 0;
    wait_vmem_all_but<4 + QW>();  // (K >= 2 stages)
    lds_only_barrier();
    fetch_x(0, 0, ox[0]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) fetch_w(0, 0, j);
    bool stored = false;
    for (int t = slot; t < count; t += slots) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < p.K; k += LN_STEP) {
            products(without, ox[0], buf, 1, ox[1]);
            // The next stage and the bias are there (the results of the last tile, stored after they were
            // requested, need not be), and, behind the barrier, everybody has read this stage: its place
            // takes the one after next.
            if (stored) wait_vmem_all_but<4 * NP>();
            else wait_vmem_all_but<0>();
            stored = false;
            lds_only_barrier();
            __builtin_amdgcn_sched_barrier(0);
            buf ^= 1;
            products(with_loads, ox[1], buf, 0, ox[0]);  // (behind the last stage: operands that nothing uses)
            advance();
        }
        // ---- results
        const LnSeg &s = p.seg[c.seg];
        const int col = 16 * (g & 1) + 8 * (g >> 1);  // of a lane's eight columns in 32, after the exchange
        const long ld_out = ANY == 2 ? s.period * s.ld_out : s.ld_out;
        char *out = s.out + c.b * s.batch_out + c.m0 * s.ld_out + wm * 64 * ld_out + 2 * (c.n0 + wn * (BN / 2) + col);
        if (t + slots < count) {
            c = tile_of(t + slots);
            load_bias(c, which ^ 1);
        }
        auto store = [&](char *q, u32x4_t v) {
            // (2: the first and last columns' tiles begin at any element)
            using piece_t = std::conditional_t<ANY == 2, LnLoosePiece, u32x4_t>;
            if constexpr (PAST) __builtin_nontemporal_store(v, (piece_t *)q);
            else *(piece_t *)q = v;
        };
        auto eight = [&](int i, int jp) {
            u32x2_t d[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = 2 * jp + h;
                const u32x4_t b = *(const u32x4_t *)(lds_bias[which] + wn * (BN / 2) + 16 * j + 4 * g);
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + to_float<T>((uint16_t)b[e]);
                d[h] = u32x2_t{Mma<T>::pack(v[0], v[1]), Mma<T>::pack(v[2], v[3])};
            }
            // groups 1 and 3 of the first 16 columns against groups 0 and 2 of the second
            const auto lo = __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false);
            const auto hi = __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false);
            return u32x4_t{lo[0], hi[0], lo[1], hi[1]};
        };
        // the sixteen columns of jp and jp + 1, lanes of rows r and r + 8 exchanging halves: lane (g, r) then holds, in
        // a of row r & 7 and in b of row 8 + (r & 7), eight columns at 32 (r / 8) + col
        auto lines = [&](int i, int jp, u32x4_t &a, u32x4_t &b) {
            const u32x4_t v0 = eight(i, jp), v1 = eight(i, jp + 1);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t give = r < 8 ? v1[e] : v0[e];
                const uint32_t got = __builtin_amdgcn_update_dpp(0, give, 0x128, 0xF, 0xF, true);  // row_ror:8
                a[e] = r < 8 ? v0[e] : got;
                b[e] = r < 8 ? got : v1[e];
            }
        };
        if constexpr (ANY == 1) {
            // Eight rows at a time through the LDS, from where they are read 16 bytes at a time as they lie in
            // memory; the elements before the first and behind the last such piece, eight a row, one by one.
            char *mine = lds_out + w * 8 * OUT_PITCH;
            char *rows = out - 2 * col;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                u32x4_t v[2][2];  // [rows 0 .. 7, 8 .. 15][columns 0 .. 63, 64 .. 127]
                lines(i, 0, v[0][0], v[1][0]);
                lines(i, 2, v[0][1], v[1][1]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        *(u32x4_t *)(mine + (r & 7) * OUT_PITCH + 128 * q + (r & 8) * 8 + 2 * col) = v[h][q];
                    char *eight_rows = rows + (long)(16 * i + 8 * h) * ld_out;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int row = 4 * u + (lane >> 4), piece = lane & 15;
                        char *to = eight_rows + row * ld_out;
                        const int before = (int)(-(intptr_t)to & 15);  // bytes up to the first whole piece
                        u32x4_t d;
                        __builtin_memcpy(&d, __builtin_assume_aligned(mine + row * OUT_PITCH + before + 16 * piece, 2), 16);
                        if (piece < 15 || before == 0) store(to + before + 16 * piece, d);
                    }
                    const int row = lane >> 3, e = lane & 7;
                    char *to = eight_rows + row * ld_out;
                    const int before = (int)(-(intptr_t)to & 15) / 2, at = e < before ? e : 120 + e;
                    const uint16_t one = *(const uint16_t *)(mine + row * OUT_PITCH + 2 * at);
                    if (before != 0) *(uint16_t *)(to + 2 * at) = one;
                }
            }
        } else {
#pragma unroll
            for (int jp = 0; jp + 1 < NP; jp += 2)
#pragma unroll
                for (int i = 0; i < 4; ++i) {  // a store covers eight rows by 128 bytes
                    u32x4_t a, b;
                    lines(i, jp, a, b);
                    char *q = out + (long)(16 * i + (r & 7)) * ld_out + 64 * jp + (r & 8) * 8;
                    store(q, a);
                    store(q + 8 * ld_out, b);
                }
            if constexpr (NP & 1)
#pragma unroll
                for (int i = 0; i < 4; ++i) store(out + (long)(16 * i + r) * ld_out + 64 * (NP - 1), eight(i, NP - 1));
        }
        stored = true;
        which ^= 1;
    }
    wait_vmem_all_but<0>();  // no transfer outlives the workgroup's LDS
}

// ---- few rows.  256 x 512 x 512 is a prompt's projection: 0.13 GFLOP, nothing but latency.  A workgroup owns 32 x 32
// results and its wavefronts a quarter of the contraction each, taken in groups of 128 whose operands are all
// requested before the first is multiplied, straight into registers in operand order; the partial tiles meet
// in the LDS.  One trip to memory, four products deep, one exchange.
constexpr int LS_TILE = 32, LS_WAVES = 4, LS_DEPTH = 4;  // LS_DEPTH: steps of 32 requested together

template <typename T>
__global__ void __launch_bounds__(64 * LS_WAVES) linear_few_rows_kernel(LnArgs p) {
    __shared__ float part[LS_WAVES][LS_TILE][LS_TILE + 4];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r = lane & 15;
    int t = blockIdx.x, seg = 0;
    while (seg + 1 < p.nseg && t >= p.seg[seg + 1].first) ++seg;
    const LnSeg &q = p.seg[seg];
    t -= q.first;
    const int rt = t / q.col_tiles, n0 = (t - rt * q.col_tiles) * LS_TILE, batch = rt / q.row_tiles;
    const int m0 = (rt - batch * q.row_tiles) * LS_TILE;
    const int steps = p.K / 32;
    const bool whole = steps < 2 * LS_WAVES;  // a short contraction: each wavefront all of it for a quarter of the results
    const int s0 = whole ? 0 : steps * w / LS_WAVES, n = whole ? steps : steps * (w + 1) / LS_WAVES - s0;
    const char *px[2], *pw[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // rows and columns behind the end: the last one's, not stored
        const int m = m0 + 16 * i + r < q.rows ? m0 + 16 * i + r : q.rows - 1;
        const int col = n0 + 16 * i + r < q.cols ? n0 + 16 * i + r : q.cols - 1;
        px[i] = q.x + batch * q.batch_x + m * q.ld_x + 64 * s0 + 16 * g;
        pw[i] = q.w + col * q.ld_w + 64 * s0 + 16 * g;
    }
    if (whole) {
        const char *x = w & 2 ? px[1] : px[0], *wt = w & 1 ? pw[1] : pw[0];
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < n; ++s)
            acc = Mma<T>::k32(*(const u32x4_t *)(wt + 64 * s), *(const u32x4_t *)(x + 64 * s), acc);
        *(f32x4 *)&part[0][8 * (w & 2) + r][16 * (w & 1) + 4 * g] = acc;
    } else {
        f32x4 acc[2][2];  // [rows][columns]: lane (g, r) holds row r, columns 4 g ..
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        struct Ops {
            u32x4_t x[2], w[2];
        };
        auto request = [&](int s, Ops &o) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                o.x[i] = *(const u32x4_t *)(px[i] + 64 * s);
                o.w[i] = *(const u32x4_t *)(pw[i] + 64 * s);
            }
        };
        auto products = [&](const Ops &o) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = Mma<T>::k32(o.w[j], o.x[i], acc[i][j]);
        };
        Ops o[LS_DEPTH];
        int s = 0;
        if (n >= LS_DEPTH) {
#pragma unroll
            for (int u = 0; u < LS_DEPTH; ++u) request(u, o[u]);
            for (s = LS_DEPTH; s + LS_DEPTH <= n; s += LS_DEPTH)
#pragma unroll
                for (int u = 0; u < LS_DEPTH; ++u) {
                    products(o[u]);
                    request(s + u, o[u]);
                }
#pragma unroll
            for (int u = 0; u < LS_DEPTH; ++u) products(o[u]);
        }
        for (; s < n; ++s) {
            request(s, o[0]);
            products(o[0]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) *(f32x4 *)&part[w][16 * i + r][16 * j + 4 * g] = acc[i][j];
    }
    __syncthreads();
    const int row = threadIdx.x >> 3, c = (threadIdx.x & 7) * 4;
    if (m0 + row >= q.rows || n0 + c >= q.cols) return;  // (cols is a multiple of 4)
    f32x4 sum = *(const f32x4 *)&part[0][row][c];
    if (!whole)
#pragma unroll
        for (int u = 1; u < LS_WAVES; ++u) sum += *(const f32x4 *)&part[u][row][c];
    if (q.bias)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += to_float<T>(q.bias[n0 + c + e]);
    *(u32x2_t *)(q.out + batch * q.batch_out + (m0 + row) * q.ld_out + 2 * (n0 + c)) =
        u32x2_t{Mma<T>::pack(sum[0], sum[1]), Mma<T>::pack(sum[2], sum[3])};
}

// tiles, rows by columns; the fourth is the few-row kernel's, the last for results whose rows begin at any element
struct LnTile {
    int rows, cols;
};
constexpr LnTile LN_TILES[5] = {{256, 256}, {256, 192}, {128, 128}, {LS_TILE, LS_TILE}, {256, 256}};

template <typename T, bool TW>
void launch(int tile, bool past, const LnArgs &p, hipStream_t st) {
    auto go = [&](auto kernel, int bm) { kernel<<<256 * 256 / bm, 2 * bm, 0, st>>>(p); };
    if (tile == 0) past ? go(linear_kernel<T, 256, 256, TW, true>, 256) : go(linear_kernel<T, 256, 256, TW, false>, 256);
    else if (tile == 1) past ? go(linear_kernel<T, 256, 192, TW, true>, 256) : go(linear_kernel<T, 256, 192, TW, false>, 256);
    else if (tile == 2) go(linear_kernel<T, 128, 128, TW, false>, 128);
    else if constexpr (!TW) {
        // (rows through the LDS: through the caches as well; past them 1024 x 50257 x 512 74 -> 85 us, 8192 x 30001 x 512 298 ->
        // 326, before the walks began apart)
        if (p.seg[0].period > 1) past ? go(linear_kernel<T, 256, 256, false, true, 2>, 256) : go(linear_kernel<T, 256, 256, false, false, 2>, 256);
        else go(linear_kernel<T, 256, 256, false, false, 1>, 256);
    }
}

long tiles_of(const hsa_linear_segment &s, LnTile t) {
    return (long)s.batches * ((s.rows + t.rows - 1) / t.rows) * ((s.cols + t.cols - 1) / t.cols);
}

// what the kernel of a tile takes
bool takes(int tile, int nseg, const hsa_linear_segment *seg, int K, bool w_rows_contract) {
    if (nseg < 1 || nseg > HSA_LINEAR_MAX_SEGMENTS || !seg || K > (1 << 20)) return false;
    const bool few = tile == 3, any = tile == 4;
    if (any && w_rows_contract) return false;
    if (few ? K < 32 || K % 32 || w_rows_contract : K < 2 * LN_STEP || K % LN_STEP) return false;
    for (int i = 0; i < nseg; ++i) {
        const hsa_linear_segment &s = seg[i];
        if (s.batches < 1 || s.rows < (few ? 1 : LN_TILES[tile].rows) || s.cols < (few ? 4 : LN_TILES[tile].cols) ||
            s.cols % (any ? 1 : few ? 4 : 8) || s.batches > (1 << 24) || s.rows > (1 << 28) || s.cols > (1 << 24) || s.ld_x < K ||
            s.ld_w < (w_rows_contract ? s.cols : K) || s.ld_out < s.cols || s.ld_x > (1 << 21) || s.ld_w > (1 << 21))
            return false;
        const int64_t strides = s.ld_x | s.ld_w | (any ? 0 : s.ld_out) | (s.batches > 1 ? s.batch_x | (any ? 0 : s.batch_out) : 0);
        const uintptr_t bits = (uintptr_t)s.x | (uintptr_t)s.w | (any ? 8 : 1) * (uintptr_t)s.out | 8 * (uintptr_t)s.bias;
        if (strides % 8 || bits % 16) return false;
    }
    return true;
}

double all_tiles(int tile, int nseg, const hsa_linear_segment *seg) {
    double n = 0;
    for (int i = 0; i < nseg; ++i) n += (double)tiles_of(seg[i], LN_TILES[tile]);
    return n;
}

// rows after which results of a row stride lie in their lines of 64 elements as before
int line_period(int64_t ld_out) {
    int64_t a = ld_out & 63, line = 64;
    while (a) {
        const int64_t rest = line % a;
        line = a;
        a = rest;
    }
    return (int)(64 / line);
}

// the tiles of a launch; false: too many
bool plan(int tile, int nseg, const hsa_linear_segment *seg, int K, LnArgs &p) {
    const LnTile size = LN_TILES[tile];
    p.nseg = nseg;
    p.K = K;
    p.group = 2048 / size.rows;
    long tiles = 0;
    for (int i = 0; i < nseg; ++i) {
        const hsa_linear_segment &s = seg[i];
        LnSeg &t = p.seg[i];
        t.x = (const char *)s.x;
        t.w = (const char *)s.w;
        t.bias = (const uint16_t *)s.bias;
        t.out = (char *)s.out;
        t.ld_x = 2 * s.ld_x;
        t.ld_w = 2 * s.ld_w;
        t.ld_out = 2 * s.ld_out;
        t.batch_x = 2 * s.batch_x;
        t.batch_out = 2 * s.batch_out;
        t.rows = s.rows;
        t.cols = s.cols;
        t.period = 1;
        t.row_tiles = (s.rows + size.rows - 1) / size.rows;
        t.col_tiles = (s.cols + size.cols - 1) / size.cols;
        // Tiles of rows that lie alike where whole lines pay for it.  They take 0.9 of the time of consecutive rows
        // through the LDS for the same number of tiles, but a row class that does not fill its tiles makes for more of
        // them (us, library / alike / through the LDS, in brackets their tiles by the others': 50257 columns, 32768
        // rows 2180 / 1693 / 1897 (1), 16384 1108 / 866 / 951 (1), 28672 1899 / 1688 / 1668 (1.14), 24576 1635 / 1705 / 1405 (1.33),
        // 20480 1357 / 1730 / 1169 (1.6); 50260, 4096 rows 342 / 224 / 247 (1), 7168 462 / 426 / 414 (1.14), 5120 415 / 430 /
        // 296 (1.6)), and the first and the last columns' tiles begin at any element all the same (16384 rows of 3001 75 / 70
        // / 61, 32768 138 / 137 / 114, of 5001 227 / 210 / 201, of 8001 380 / 298 / 332, of 10001 435 / 364 / 406).
        const int period = tile == 4 && nseg == 1 ? line_period(s.ld_out) : 1;
        if (period > 1 && s.rows / period >= size.rows && t.col_tiles >= 32) {
            const int row_tiles = period * (((s.rows + period - 1) / period + size.rows - 1) / size.rows);
            if (row_tiles * 20l <= t.row_tiles * 23l) {
                t.period = period;
                t.row_tiles = row_tiles;
                // (a tile begins up to 63 columns before its place: the last one has to reach the end)
                t.col_tiles = (s.cols + 63 + size.cols - 1) / size.cols;
            }
        }
        const double n = (double)s.batches * t.row_tiles * t.col_tiles;
        if (n + tiles >= (double)(1 << 30)) return false;
        t.all_row_tiles = s.batches * t.row_tiles;
        t.first = (int)tiles;
        tiles += (long)n;
    }
    p.tiles = (int)tiles;
    // rows that begin anywhere: neighbours in a row side by side, their common lines meet in one L2 (2 / 4 / 8: 1669 / 2061
    // / 2138 us at 28672 x 50257 x 512, 428 / 443 / 537 at 7168; 10001 columns 351 / 357 / 345 and 93 / 92 / 91)
    if (tile == 4 && p.seg[0].period == 1) p.group = 2;
    return true;
}

}  // namespace

}  // namespace hsa

extern "C" {

int hsa_linear_tile(int nseg, const hsa_linear_segment *seg, int K, int w_rows_contract, int dtype) {
    using namespace hsa;
    if (dtype != HSA_F16 && dtype != HSA_BF16) return -1;
    double results = 0;
    if (nseg < 1 || nseg > HSA_LINEAR_MAX_SEGMENTS || !seg) return -1;
    for (int i = 0; i < nseg; ++i) results += (double)seg[i].batches * seg[i].rows * seg[i].cols;
    // Few rows (us on the GPU, library / here; the call takes 20 / 5 us of host time, and sizes like these wait for the
    // host): 64 x 512 x 512 5.2 / 4.3, 256 x 512 x 512 5.2 / 4.4, 512 x 512 x 256 4.4 / 3.8, 256 x 2048 x 512 6.0 / 6.2, 256 x
    // 1024 x 1024 5.6 / 6.2, 512 x 672 x 672 7.2 / 5.6.  Replayed from a graph the library is the faster one by up to 2 us
    // where more than two workgroups meet on a CU or, from contractions of 768 on, more than one: 768 x 768 x 384 5.6 / 6.9,
    // 512 x 2048 x 256 5.2 / 6.7, 384 x 768 x 768 5.7 / 7.9.  Beyond: 512 x 2048 x 512 6.4 / 9.7, 256 x 512 x 2048 6.3 / 9.3.
    // Several projections are several library calls.
    if (K <= 1024 && results * K <= (double)(1 << 27) * (nseg + 1) && takes(3, nseg, seg, K, w_rows_contract)) return 3;
    // Tiles: rounds of the chip times the time of a tile, 256 x 256 as 1 (256 x 192 0.8, two of 128 x 128 on one CU 0.74).
    // The library has the better inner loop from contractions of about 1000 on and with its widest tiles at
    // 768; at 512 and below this kernel is the faster one unless it leaves a good part of the chip idle
    // (rows x cols x K, us, library / here): 8192 x 1536 x 512 27.9 / 18.9, 16384 x 1536 x 512 40.7 / 32, 32768 x 2048
    // x 512 78 / 70, 4096 x 2048 x 512 15.6 / 15.1, 16384 x 768 x 768 24.2 / 22.8, 32752 x 768 x 768 46.5 / 38; not taken:
    // 4096 x 512 x 512 8.0 / 8.9, 8192 x 768 x 768 15.2 / 17.5, 16384 x 3072 x 768 69 / 72, 16384 x 1024 x 1024 30.5 / 34,
    // 32768 x 512 x 2048 50 / 56.  With the weight's rows along the contraction the library is slower: 16384 x 768 x 768
    // 26.3 / 23.2, x 1536 41.1 / 36.6, x 2304 57.7 / 50.0; not taken although it gains where the tiles fill the chip: 32768 x 768 x
    // 3072 146 / 125, 16384 x 1024 x 3072 84 / 81, 32768 x 512 x 4096 119 / 113 (but 8192 x 1024 x 3072 53 / 59).  Rows that begin
    // anywhere (a vocabulary of 50257): 256 x 50257 x 512 34 / 25, 1024 98 / 74, 4096 340 / 240, 8192 576 / 474, 32768 2140 /
    // 1710; not taken: 4096 x 50257 x 768 346 / 314, 8192 593 / 630, 32768 2321 / 2309.
    int best = -1;
    double least = 0;
    for (int t = 0; t < 3; ++t) {
        if (!takes(t, nseg, seg, K, w_rows_contract)) continue;
        const double n = all_tiles(t, nseg, seg);
        const double us = t == 0 ? ceil(n / 256) : t == 1 ? 0.8 * ceil(n / 256) : n <= 256 ? 0.42 : 0.74 * ceil(n / 512);
        if (best < 0 || us <= least) {
            best = t;
            least = us;
        }
    }
    if (best < 0 && takes(4, nseg, seg, K, w_rows_contract)) {
        best = 4;
        least = ceil(all_tiles(4, nseg, seg) / 256);
    }
    if (best < 0) return -1;
    const double used = results / (65536.0 * 256.0) / least;
    if (K > (w_rows_contract ? 2304 : 768) || used < (K > 512 ? 0.9 : 0.6) || (K > 512 && best != 1 && !w_rows_contract)) return -1;
    return best;
}

int hsa_linear_rectangles(int nseg, const hsa_linear_segment *seg, int K, int w_rows_contract, int tile, int (*rects)[8], int capacity) {
    using namespace hsa;
    HSA_REQUIRE(tile >= 0 && tile < 5 && tile != 3 && capacity >= 0 && (rects || !capacity), "bad tile %d or no room", tile);
    LnArgs p = {};
    if (!takes(tile, nseg, seg, K, w_rows_contract != 0) || !plan(tile, nseg, seg, K, p))
        return fail(HSA_ERR_UNSUPPORTED, "projection: sizes or alignment not handled by tile %d (K=%d)", tile, K);
    const bool alike = p.seg[0].period > 1;
    int at = 0;
    for (int xcd = 0; xcd < 8; ++xcd) {
        const LnWalk walk = tile == 4 && !alike ? walk_of<1>(p, xcd) : walk_of<0>(p, xcd);
        for (int i = 0; i < walk.count && at < capacity; ++i, ++at) {
            const int t = walk.tile(i);
            const LnPlace c = tile == 1 ? place_of<256, 192, 0>(p, t) : tile == 2 ? place_of<128, 128, 0>(p, t)
                              : tile == 4 && alike ? place_of<256, 256, 2>(p, t) : place_of<256, 256, 0>(p, t);
            const int rect[8] = {c.seg, c.b, c.m0, p.seg[c.seg].period, LN_TILES[tile].rows, c.n0, LN_TILES[tile].cols, xcd};
            for (int e = 0; e < 8; ++e) rects[at][e] = rect[e];
        }
    }
    return p.tiles;
}

int hsa_linear(int nseg, const hsa_linear_segment *seg, int K, int w_rows_contract, int tile, int dtype, void *stream) {
    using namespace hsa;
    HSA_REQUIRE(dtype == HSA_F16 || dtype == HSA_BF16, "projections of 16-bit operands only (dtype %d)", dtype);
    HSA_REQUIRE(tile >= 0 && tile < 5, "bad tile %d", tile);
    if (!takes(tile, nseg, seg, K, w_rows_contract != 0))
        return fail(HSA_ERR_UNSUPPORTED, "projection: sizes or alignment not handled by tile %d (K=%d)", tile, K);
    LnArgs p = {};
    if (!plan(tile, nseg, seg, K, p)) return fail(HSA_ERR_UNSUPPORTED, "projection: too many tiles");
    double bytes = 0;
    for (int i = 0; i < nseg; ++i) {
        HSA_REQUIRE(seg[i].x && seg[i].w && seg[i].out, "null pointer");
        bytes += 2.0 * seg[i].batches * seg[i].rows * seg[i].cols;
    }
    // large results go past the caches: they would push the operands' rows out of the L2s (4 MiB each) before the
    // next kernel could find them there (everything above 16 MiB against 256 MiB: a six-layer forward of 32768 tokens
    // 5727 -> 5678 us, a module in training 1650 -> 1628)
    const bool past = bytes > (double)(1 << 24);
    const hipStream_t st = (hipStream_t)stream;
    if (tile == 3) {
        if (dtype == HSA_F16) linear_few_rows_kernel<F16><<<p.tiles, 64 * LS_WAVES, 0, st>>>(p);
        else linear_few_rows_kernel<BF16><<<p.tiles, 64 * LS_WAVES, 0, st>>>(p);
        return check_launch("linear_few_rows_kernel");
    }
    if (dtype == HSA_F16) w_rows_contract ? launch<F16, true>(tile, past, p, st) : launch<F16, false>(tile, past, p, st);
    else w_rows_contract ? launch<BF16, true>(tile, past, p, st) : launch<BF16, false>(tile, past, p, st);
    return check_launch("linear_kernel");
}

}  // extern "C"
