// Span attention backward, MFMA tile kernels (16-bit element types, canonical tree tables).
//
// Two launches, the flash-attention split adapted to the window + tree structure:
//
//  (A) query-stationary, one wavefront per (batch, head, 16-query block): recomputes the score
//      tiles S^T[key, query] exactly like the forward, then
//          dP^T = V_blk . dO_blk^T          delta[q] = sum_key P dP
//          dS^T = P (dP - delta) / sqrt(D)   dQ^T[ch, q] = K_blk^T . dS^T
//      and stores dQ plus two numbers per (query, head): the log2-domain log-sum-exp and delta.
//      The tree key blocks are also evaluated in the other orientation (S[query, slot]), which
//      puts the queries into the MFMA contraction: dK^T[ch, slot] = Q^T . dS, dV^T = dO^T . P.
//      Nodes of levels 1..4 are attended only from inside the block: their rows are final and
//      written directly.  A node of level l >= 5 collects from the 2^(l-4) blocks under its
//      sibling: a wavefront that walks a strip of four blocks finishes level 5 itself and sums
//      the levels above over its strip; what is left is stored as fp32 partial rows (per strip
//      and level >= 6, or per block and level >= 5 for strips of one block), and pass (B)'s
//      trailing workgroups sum each node's contiguous run (deterministic, no atomics).
//  (B) key-stationary, one wavefront per (batch, head, 16-leaf key block): loops over the query
//      blocks whose window reaches the key block, rebuilds P and dS from the saved statistics
//      and accumulates dK^T = Q^T . dS, dV^T = dO^T . P in registers.  Every leaf row of dK / dV
//      is written once; no atomics.
//
// Operand plumbing is the forward kernel's: row-contiguous 16-byte global accesses, per-wavefront
// LDS re-layout into MFMA operand order, transposed operands through an MFMA with a 0/1
// selection matrix.
#pragma once

#include "hsa_attn_tile.h"

namespace hsa {

struct BwdTileParams {
    const uint16_t *q, *k, *v, *dout;
    uint16_t *dq, *dk, *dv;
    float *stats;   // [B, N, H, 2]: log2-domain lse, delta
    float *partial; // [2, B, N/16, H, L-4, D] fp32 per-block partial rows of dK, dV for levels >= 4
    int B, N, M, H, L, R;
    int dh;         // channels per head (kernels built for part heads; else the template's D)
    int n_units;
    float scale_log2e, scale;
    // rows the key pass's trailing workgroups finish from the partial rows (none: red_wgs == 0)
    int causal, red_first_row, red_wgs, red_lg_sb;  // red_lg_sb: log2 of the query pass's blocks per strip
};

// the one-pass variant (hsa_attn_bwd_fused.h) also takes what the forward left behind
struct BwdFusedParams {
    BwdTileParams t;
    const uint16_t *out;  // forward output [B, N, H, D]
    const float *lse;     // forward log-sum-exp [B, N, H], log2 domain
};

constexpr int BWD_WPB = 4;  // wavefronts per workgroup
// threads that share one output row piece in the one-pass variant's second launch
constexpr int BWD_FUSED_RED_SPLIT = 8;

// Hardware hands consecutive workgroup ids to the 8 XCDs in turn; with this remap workgroups that
// are consecutive in the returned index run on the same XCD, so neighbouring strips (which share
// halo rows and upper tree nodes) share an L2.
__device__ __forceinline__ int bwd_xcd_remap(int wg, int nwg) {
    return (nwg & 7) == 0 ? (wg & 7) * (nwg >> 3) + (wg >> 3) : wg;
}

// Blocks one wavefront of either pass walks (1 only for sequences whose block count is no multiple
// of it): leaf blocks (query pass) or query blocks (key pass) slide along the strip in operand
// form, NBW+1 of them when causal, 2 NBW+1 otherwise.
constexpr int BWD_STRIP = 4;  // the reduction and the level-5 pairing assume four: a strip is the 64 leaves under a level-6 node
// Wavefronts per SIMD the query pass is compiled for: two (256 registers) where that holds its
// operands without spilling, which a strip with five sliding leaf blocks at D = 64 and every
// variant at D = 128 do not.
constexpr int bwd_query_waves(int D, int nkl, int sb) {
    return (nkl <= 5 && (D <= 32 || (D <= 64 && (nkl <= 3 || sb == 1)))) ? 2 : 1;
}

// DC > 0: part heads (hsa_attn_tile.h), DC channels of the layout's D in the contractions.  B3 H8 N2048 D96 R16
// causal, both passes: 48.1 us in bf16 and 61.4 in fp16 (1640 on the gather kernels; 42.2 with weights and
// score gradients rounded to 16 bits; the one pass 49; with rows looked at one by one instead of a second
// form of the code 53.4 in bf16)
template <typename T, int D, int DC = 0>
struct BwdTile {
    using M_ = Mma<T>;
    static constexpr int KS = (DC ? DC : D) / 32, NJ = (DC ? DC : D) / 16, CPR = D / 8, RPI = 64 / CPR, NLD = TILE_Q / RPI;
    // a block in LDS: rows back to back, the 16-byte pieces of row r at piece index p ^ swz(r)
    // (conflict-free from both sides, see hsa_attn_tile.h); slots keep the size of a padded block
    static constexpr int RB = D * 2, RPB = RB >= 256 ? 1 : 256 / RB, BLK_BYTES = TILE_Q * (RB + 16);
    __device__ static __forceinline__ int swz(int row) { return (row / RPB) % CPR; }

    int lane, r16, g, lrow, lchk, op_swz;
    unsigned char *lds;
    u32x4_t Pi[2];

    __device__ __forceinline__ void init(unsigned char *wave_lds, int lane_) {
        lane = lane_;
        r16 = lane & 15;
        g = lane >> 4;
        lrow = lane / CPR;
        lchk = lane % CPR;
        op_swz = swz(r16);
        lds = wave_lds;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int e = 4 * jj + (r16 & 3);
            const uint32_t one = (g == (r16 >> 2)) ? (uint32_t)M_::kOne << (16 * (e & 1)) : 0u;
            const int wi = e >> 1;
            Pi[jj] = u32x4_t{wi == 0 ? one : 0u, wi == 1 ? one : 0u, wi == 2 ? one : 0u, wi == 3 ? one : 0u};
        }
    }
    // rows -> LDS -> operand pieces
    __device__ __forceinline__ void put(int slot, const u32x4_t (&raw)[NLD]) const {
        unsigned char *reg = lds + slot * BLK_BYTES;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int row = i * RPI + lrow;
            *reinterpret_cast<u32x4_t *>(reg + row * RB + 16 * (lchk ^ swz(row))) = raw[i];
        }
    }
    __device__ __forceinline__ void get(int slot, u32x4_t (&dst)[KS]) const {
        const unsigned char *reg = lds + slot * BLK_BYTES + r16 * RB;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) dst[ks] = *reinterpret_cast<const u32x4_t *>(reg + 16 * ((4 * ks + g) ^ op_swz));
    }
    // weights and score gradients in the second products: rounded to the element type once; for part heads (see
    // hsa_attn_tile.h) all their bits.  The fp16 gradients have no range that a sum of two fp16 numbers could
    // be sure to hold, so those products run on the fp32 matrix instruction.
    using W = typename std::conditional<DC == 0, RoundedWeights<T>,
                                        typename std::conditional<std::is_same<T, BF16>::value, SplitWeights<BF16>, Fp32Weights<T>>::type>::type;
    // sets the channels behind a part head to zero: of the operands on both sides, since 0 times a repeated
    // infinity is NaN
    __device__ __forceinline__ void clear_behind(u32x4_t (&x)[KS], int dh) const {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (8 * (4 * ks + g) >= dh) x[ks] = u32x4_t{0u, 0u, 0u, 0u};
    }
    // rows of a block with an infinity or a NaN, one bit each (the same value in every lane)
    __device__ __forceinline__ uint32_t odd_rows(const u32x4_t (&x)[KS]) const {
        LargestBits m;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) m.add(x[ks]);
        const uint64_t lanes = __ballot(!m.template finite<T>());
        const uint32_t two = (uint32_t)(lanes | (lanes >> 32));
        return (two | (two >> 16)) & 0xffffu;
    }
    // a key / value block on entry: nothing behind the head; returns odd_rows of the keys
    __device__ __forceinline__ uint32_t odd_keys(u32x4_t (&k)[KS], u32x4_t (&v)[KS], int dh) const {
        clear_behind(k, dh);
        clear_behind(v, dh);
        return odd_rows(k);
    }
    // the same rows set to zero in a block in transposed form
    __device__ __forceinline__ void clear_rows(u32x2_t (&x)[NJ], uint32_t rows) const {
        const uint32_t mine = rows >> (4 * g);
        u32x2_t keep;
#pragma unroll
        for (int p = 0; p < 2; ++p)
            keep[p] = ((mine >> (2 * p)) & 1 ? 0u : 0xffffu) | ((mine >> (2 * p + 1)) & 1 ? 0u : 0xffff0000u);
#pragma unroll
        for (int j = 0; j < NJ; ++j) x[j] &= keep;
    }
    // weight and score gradient of query 4g + i: nothing for a dead slot whatever the operands hold; where the
    // query's dO row has been cleared, NaN instead of the weight
    __device__ __forceinline__ void settle(bool dead, uint32_t odd_g, int i, float &weight, float &grad) const {
        if (dead) weight = grad = 0.f;
        if ((odd_g >> (4 * g + i)) & 1)
            if (weight != 0.f) weight = __builtin_nanf("");
    }
    // operand rows -> "lane = channel, regs = rows" form
    __device__ __forceinline__ void transpose(const u32x4_t (&op)[KS], u32x2_t (&dst)[NJ]) const {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            f32x4 z = {0.f, 0.f, 0.f, 0.f};
            f32x4 r = M_::k32(op[j >> 1], Pi[j & 1], z);
            dst[j] = u32x2_t{M_::pack_exact(r[0], r[1]), M_::pack_exact(r[2], r[3])};
        }
    }
    // result tiles [channel, column] (this lane: column r16, channels 32ks+8g+4jj+i) -> packed
    // 16-bit pieces in LDS slot `slot`, one row per column
    __device__ __forceinline__ void put_result(int slot, const f32x4 (&t)[NJ], float mul) const {
        unsigned char *reg = lds + slot * BLK_BYTES + r16 * RB;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const f32x4 a = t[2 * ks], b = t[2 * ks + 1];
            *reinterpret_cast<u32x4_t *>(reg + 16 * ((4 * ks + g) ^ op_swz)) =
                u32x4_t{M_::pack(a[0] * mul, a[1] * mul), M_::pack(a[2] * mul, a[3] * mul),
                        M_::pack(b[0] * mul, b[1] * mul), M_::pack(b[2] * mul, b[3] * mul)};
        }
    }
    __device__ __forceinline__ u32x4_t get_row_piece(int slot, int i) const {
        const int row = i * RPI + lrow;
        return *reinterpret_cast<const u32x4_t *>(lds + slot * BLK_BYTES + row * RB + 16 * (lchk ^ swz(row)));
    }
};

// ---------------------------------------------------------------------------------------------
// (A) query-stationary pass
// ---------------------------------------------------------------------------------------------
// A wavefront walks a strip of SB consecutive query blocks (SB * 16 <= 64 queries, aligned): the
// leaf key / value operands slide along the strip in registers (each leaf row is fetched once per
// strip), the far tree block (levels >= 6, the same nodes for the whole strip) is fetched once,
// and the partial rows it collects are summed over the strip's blocks before they are written.
// A block's rows are requested when its turn comes: holding the next block's rows in registers
// as well would cost the second wavefront per SIMD (more than 256 registers at D = 64), and two
// wavefronts that cover each other's waits are worth more than the prefetch.
//
// Part heads do with infinities and NaN what the gather kernels do: they reach the rows that have to do with
// theirs and no others.  A strip that meets one walks again in a second form of the code, in which dead
// slots are selected away instead of biased away, the channels behind the head are zero on both sides, and
// a row with such an element counts as zero in the products that carry it to other rows (a query that
// attends to it has its NaN through the weights).  The same in the key pass.
//
// Partial rows (fp32): level 5 per query block when SB == 1, entry 1 of [2][B][N/16][H][2][D]
// (dK then dV; entry 0 and, for longer strips, the whole area stay unused); levels >= 6 per
// strip, [2][B][N/16/SB][H][L-6][D], right behind.

// The second walk of a strip that has met an infinity or a NaN (part heads).
template <typename T, int D, int NBW, bool CAUSAL, int SB, int DC>
__device__ __forceinline__ void bwd_query_again(const BwdTileParams &p, int unit, unsigned char *lds, float *carry) {
    constexpr bool ODD = true;
    int lane = threadIdx.x & 63;
    // the first walk's rows are written before they are again, and none of its values are kept for the second
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(lane), "+s"(unit)::"memory");
#include "hsa_attn_bwd_query_walk.inl"
}

template <typename T, int D, int NBW, bool CAUSAL, int SB, int DC = 0>
__global__ void __launch_bounds__(BWD_WPB * 64)
__attribute__((amdgpu_waves_per_eu(bwd_query_waves(D, CAUSAL ? NBW + 1 : 2 * NBW + 1, SB))))
attn_bwd_tile_query_kernel(BwdTileParams p) {
    constexpr int LDS_SLOTS = 4, BLK_BYTES = BwdTile<T, D, DC>::BLK_BYTES;
    __shared__ __align__(16) unsigned char smem[BWD_WPB * LDS_SLOTS * BLK_BYTES];
    // level-5 rows (dK, dV) of an even block, kept until the odd block of the pair adds its own
    __shared__ __align__(16) float carry_mem[SB > 1 ? BWD_WPB * 2 * D : 4];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = bwd_xcd_remap((int)blockIdx.x, (int)gridDim.x) * BWD_WPB + wave;
    if (unit >= p.n_units) return;
    unsigned char *lds = smem + wave * LDS_SLOTS * BLK_BYTES;
    float *carry = carry_mem + (SB > 1 ? wave * 2 * D : 0);
    constexpr bool ODD = false;
    const int lane = threadIdx.x & 63;
#include "hsa_attn_bwd_query_walk.inl"
    if constexpr (PART)
        if (__any(odd_scores != 0.f)) bwd_query_again<T, D, NBW, CAUSAL, SB, DC>(p, unit, lds, carry);
}

template <typename T, int SPLIT = 1>
__device__ __forceinline__ void bwd_reduce_rows(const float *__restrict__ partial, typename T::storage *__restrict__ dk,
                                                typename T::storage *__restrict__ dv, int B, int N, int M, int H, int D,
                                                int L, int causal, int first_row, int lg_sb, size_t t);

// ---------------------------------------------------------------------------------------------
// (B) key-stationary pass over the leaf key blocks
// ---------------------------------------------------------------------------------------------
// A wavefront walks SB consecutive key blocks; the query blocks whose window reaches a key block
// (NQB of them) slide along in registers in operand form, so each query / dO row is fetched once
// per strip instead of once per key block it touches.

template <typename T, int D, int NBW, bool CAUSAL, int SB, int DC>
__device__ __forceinline__ void bwd_key_again(const BwdTileParams &p, int unit, unsigned char *lds) {
    constexpr bool ODD = true;
    int lane = threadIdx.x & 63;
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(lane), "+s"(unit)::"memory");  // as in bwd_query_again
#include "hsa_attn_bwd_key_walk.inl"
}

// The last red_wgs workgroups of the grid do not take key blocks: they sum the query pass's
// partial rows into the upper tree levels' dK / dV rows (independent of the leaf rows this pass
// writes), which fills the chip while the key blocks' last loads and stores drain.
template <typename T, int D, int NBW, bool CAUSAL, int SB, int DC = 0>
__global__ void __launch_bounds__(BWD_WPB * 64)
attn_bwd_tile_key_kernel(BwdTileParams p) {
    constexpr int LDS_SLOTS = 4, BLK_BYTES = BwdTile<T, D, DC>::BLK_BYTES;
    __shared__ __align__(16) unsigned char smem[BWD_WPB * LDS_SLOTS * BLK_BYTES];

    const int key_wgs = (int)gridDim.x - p.red_wgs;
    if ((int)blockIdx.x >= key_wgs) {
        using S = typename T::storage;
        bwd_reduce_rows<T>(p.partial, reinterpret_cast<S *>(p.dk), reinterpret_cast<S *>(p.dv), p.B, p.N, p.M, p.H,
                           DC > 0 ? p.dh : D, p.L, p.causal, p.red_first_row, p.red_lg_sb,
                           (size_t)((int)blockIdx.x - key_wgs) * (BWD_WPB * 64) + threadIdx.x);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = bwd_xcd_remap((int)blockIdx.x, key_wgs) * BWD_WPB + wave;
    if (unit >= p.n_units) return;
    unsigned char *lds = smem + wave * LDS_SLOTS * BLK_BYTES;
    constexpr bool ODD = false;
    const int lane = threadIdx.x & 63;
#include "hsa_attn_bwd_key_walk.inl"
    if constexpr (PART)
        if (__any(odd_scores != 0.f)) bwd_key_again<T, D, NBW, CAUSAL, SB, DC>(p, unit, lds);
}

// Rows from first_row on (a level the query pass left unfinished, up to anything above row 2N-2):
// node (l, p) sums the partial rows of the query blocks (levels 4, 5) or strips (levels >= 6)
// under its sibling; nodes nobody attends (the root, right-hand nodes when causal, rows past
// 2N-1) get zeros.  SPLIT consecutive threads per (batch, row, head, four channels) share the
// partial rows of one output (the top levels have the most: one per strip of the sequence),
// index t.  lg_sb = log2 of the blocks per strip of the query pass.
template <typename T, int SPLIT>
__device__ __forceinline__ void bwd_reduce_rows(const float *__restrict__ partial, typename T::storage *__restrict__ dk,
                                                typename T::storage *__restrict__ dv, int B, int N, int M, int H, int D,
                                                int L, int causal, int first_row, int lg_sb, size_t t) {
    using S = typename T::storage;
    struct alignas(4 * sizeof(S)) Pack { S e[4]; };
    static_assert(SPLIT == 1 || SPLIT == 2 || SPLIT == 4 || SPLIT == 8, "lanes that share an output");
    const int sub = (int)(t % SPLIT);
    t /= SPLIT;
    const int D4 = D / 4;
    const size_t per_b = (size_t)(M - first_row) * H * D4;
    if (t >= (size_t)B * per_b) return;
    const int b = (int)(t / per_b);
    const size_t r = t % per_b;
    const int row = first_row + (int)(r / ((size_t)H * D4));
    const int h = (int)((r / D4) % H);
    const int d = 4 * (int)(r % D4);
    f32x4 vk = {0.f, 0.f, 0.f, 0.f}, vv = {0.f, 0.f, 0.f, 0.f};
    if (row < 2 * N - 2) {
        int lvl = 4;
        while (row >= level_offset(N, lvl + 1)) ++lvl;
        const int pidx = row - level_offset(N, lvl);
        if (!causal || (pidx & 1) == 0) {
            const int NB = N / TILE_Q;
            const int blk0 = (pidx ^ 1) << (lvl - 4);  // first query block under the sibling
            const float *pk, *pv;
            size_t stride;
            int n;
            if (lvl < 6) {
                n = 1 << (lvl - 4);
                stride = (size_t)H * 2 * D;
                pk = partial + (((size_t)b * NB + blk0) * H + h) * 2 * D + (size_t)(lvl - 4) * D + d;
                pv = pk + (size_t)B * NB * H * 2 * D;
            } else {
                // lg_sb >= 3 (the one-pass variant's strips of eight or more blocks): the area is laid out per
                // run of four blocks; level 6 has a row per run, the levels above one per strip, in
                // the strip's first run
                const int LF = L - 6;
                const int lgl = lg_sb >= 3 ? 2 : lg_sb;             // layout granularity
                const int lg = (lg_sb >= 3 && lvl == 6) ? 2 : lg_sb;  // blocks summed into one row
                const int NR = NB >> lgl;
                n = (1 << (lvl - 4)) >> lg;
                stride = ((size_t)H * LF * D) << (lg - lgl);
                const float *far = partial + 2 * (size_t)B * NB * H * 2 * D;
                pk = far + (((size_t)b * NR + (blk0 >> lgl)) * H + h) * LF * D + (size_t)(lvl - 6) * D + d;
                pv = pk + (size_t)B * NR * H * LF * D;
            }
            // eight independent 16-byte loads per tensor in flight per round trip
            int i = 0;
            if constexpr (SPLIT > 1) {
                for (i = sub; i + 3 * SPLIT < n; i += 4 * SPLIT) {
                    f32x4 a[4], c[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        a[u] = *reinterpret_cast<const f32x4 *>(pk + (size_t)(i + u * SPLIT) * stride);
                        c[u] = *reinterpret_cast<const f32x4 *>(pv + (size_t)(i + u * SPLIT) * stride);
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) { vk += a[u]; vv += c[u]; }
                }
                for (; i < n; i += SPLIT) {
                    vk += *reinterpret_cast<const f32x4 *>(pk + (size_t)i * stride);
                    vv += *reinterpret_cast<const f32x4 *>(pv + (size_t)i * stride);
                }
                i = n;
            }
            for (; i + 8 <= n; i += 8) {
                f32x4 a[8], c[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    a[u] = *reinterpret_cast<const f32x4 *>(pk + (size_t)(i + u) * stride);
                    c[u] = *reinterpret_cast<const f32x4 *>(pv + (size_t)(i + u) * stride);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) { vk += a[u]; vv += c[u]; }
            }
            for (; i < n; ++i) {
                vk += *reinterpret_cast<const f32x4 *>(pk + (size_t)i * stride);
                vv += *reinterpret_cast<const f32x4 *>(pv + (size_t)i * stride);
            }
        }
    }
    if constexpr (SPLIT > 1) {
        // the lanes of a group are neighbours in the wavefront and all of them get here
#pragma unroll
        for (int m = 1; m < SPLIT; m <<= 1)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                vk[u] += __shfl_xor(vk[u], m, 64);
                vv[u] += __shfl_xor(vv[u], m, 64);
            }
        if (sub != 0) return;
    }
    const size_t o = ((size_t)b * M + row) * H * D + (size_t)h * D + d;
    Pack ok, ov;
#pragma unroll
    for (int u = 0; u < 4; ++u) { ok.e[u] = from_float<T>(vk[u]); ov.e[u] = from_float<T>(vv[u]); }
    *reinterpret_cast<Pack *>(dk + o) = ok;
    *reinterpret_cast<Pack *>(dv + o) = ov;
}

template <typename T, int D>
int attn_bwd_tile_launch_td(const BwdTileParams &p, int nbw, bool causal, int sb, hipStream_t st);
// part heads: layout of D channels, DC of them in the contractions
template <typename T, int D, int DC>
int attn_bwd_tile_part_launch_td(const BwdTileParams &p, int nbw, bool causal, int sb, hipStream_t st);

}  // namespace hsa
