// Eligibility test and launch parameters of the MFMA tile kernel.
#include "hsa_attn_tile.h"

#include <stdlib.h>

#include <atomic>

namespace hsa {

// window radius in 16-row leaf blocks: up to 4 (R <= 64) when causal, where a query block sees
// NBW + 1 leaf blocks; up to 2 (R <= 32) otherwise, where it sees 2 NBW + 1
constexpr int TILE_MAX_NBW_CAUSAL = 4;
constexpr int TILE_MAX_NBW = 2;
constexpr int TILE_MAX_NBW_WIDE = 4;

// Experiment knobs of the tile launch: strip length in query blocks (0 = by problem size),
// wavefronts per workgroup (0 = by head count), XCD remap on/off, alternating strip direction on/off.  Initialised
// once per process from HSA_ATTN_TILE_SB / _WPB / _SWZ / _ALT, changed afterwards only through
// hsa_attn_tile_tune; a launch reads four atomics, never the environment.
struct TileKnobs {
    std::atomic<int> sb{0}, wpb{0}, swizzle{1}, alternate{1};
    TileKnobs() {
        if (const char *e = getenv("HSA_ATTN_TILE_SB")) { int x = atoi(e); if (x == 1 || x == 2 || x == 4 || x == 8) sb = x; }
        if (const char *e = getenv("HSA_ATTN_TILE_SWZ")) swizzle = atoi(e) != 0;
        if (const char *e = getenv("HSA_ATTN_TILE_ALT")) alternate = atoi(e) != 0;
        if (const char *e = getenv("HSA_ATTN_TILE_WPB")) { int x = atoi(e); if (x >= 1 && x <= 8) wpb = x; }
    }
};
static TileKnobs &tile_knobs() {
    static TileKnobs k;
    return k;
}

// the two knobs the fp32 tile launch shares
void attn_tile_knobs_sb_swizzle(int *sb, int *swizzle) {
    *sb = tile_knobs().sb > 4 ? 4 : (int)tile_knobs().sb;  // strips of more than four blocks: 16-bit kernels only
    *swizzle = tile_knobs().swizzle;
}

int attn_tile_tune(int sb, int wpb, int swizzle, int alternate) {
    if (!(sb == -1 || sb == 0 || sb == 1 || sb == 2 || sb == 4 || sb == 8))
        return fail(HSA_ERR_INVALID, "strip length %d", sb);
    if (!(wpb == -1 || (wpb >= 0 && wpb <= 8))) return fail(HSA_ERR_INVALID, "wavefronts per workgroup %d", wpb);
    TileKnobs &k = tile_knobs();
    if (sb >= 0) k.sb = sb;
    if (wpb >= 0) k.wpb = wpb;
    if (swizzle >= 0) k.swizzle = swizzle != 0;
    if (alternate >= 0) k.alternate = alternate != 0;
    return HSA_OK;
}

bool attn_tile_eligible(int N, int M, int H, int D, int L, int R, int dtype, bool canonical,
                        bool want_weights, bool causal) {
    (void)H;
    if (!canonical) return false;
    // the weights of a query block are assembled in the wavefront's LDS region: a row of
    // 2R+1+L floats has to fit the operand pitch
    if (want_weights && 2 * R + 1 + L > D * 2 + 16) return false;
    if (dtype != HSA_F16 && dtype != HSA_BF16) return false;
    if (!tile_head_ok(D) || (tile_head_is_part(D) && (want_weights || R > TILE_PART_MAX_R))) return false;
    if (N < TILE_Q || ilog2_exact(N) != L || L > TILE_MAX_LEVELS) return false;
    if (M < 2 * N - 1) return false;
    const int nbw = (R + TILE_Q - 1) / TILE_Q;
    if (causal) return nbw <= TILE_MAX_NBW_CAUSAL;
    // without the causal mask: up to five leaf blocks everywhere, seven or nine with one query
    // block per wavefront
    return nbw <= TILE_MAX_NBW || nbw <= TILE_MAX_NBW_WIDE;
}

// Strip length (query blocks per wavefront) and wavefronts per workgroup.
//
// A CU takes one workgroup of up to eight wavefronts at a time (four at 128 channels: one wavefront per
// SIMD), so what counts is how many query blocks the busiest CU walks, sb * wpb * ceil(workgroups /
// 256), and whether they fit one resident round: every further round repeats the first loads' latency,
// which a longer strip spreads over more blocks (measured per block against one round of strips of four:
// 1.7 for single blocks, 1.2 to 1.45 for two, 1.15 for four, 1.1 for eight).  Among equals more
// wavefronts win in one round (more loads in flight), longer strips in several.  Without the causal mask
// strips of eight lose (three leaf blocks per query block in 256 registers: B8 H8 N8192 D64 84.3 -> 89.8
// us).
//
// Against the longest strip that filled every wavefront slot (us, bf16, causal unless noted): B5 N1024
// H12 D64 16.0 -> 10.5, not causal 18.1 -> 10.7; B12 N512 H8 D64 11.7 -> 9.1; B4 N2048 H6 D64 11.5 ->
// 9.2; B3 N2048 H12 D64 15.6 -> 13.1; B12 N1024 H8 D64 17.9 -> 15.3, B6 N2048 H8 not causal 20.1 -> 16.4;
// B2 N8192 H10 D64 24.9 -> 22.7; B3 N4096 H6 D128 26.1 -> 22.9; B3 N2048 H8 D96 19.8 -> 17.0.  B8 N2048
// H8 D64 (strips of four), B16 N512 H8 D64 (two) and the long sequences (eight) stay as they were.
//
// Wavefronts per workgroup: all the variant allows, or a divisor of the head count at least half as
// large, so that a workgroup's wavefronts are heads of one strip and read whole contiguous token rows;
// four in one round where that leaves fewer blocks to the busiest CU.
struct StripChoice {
    int sb, wpb;
};
StripChoice choose_strip(long blocks, int H, int max_wpb, int most, bool eight, int forced_sb, int forced_wpb) {
    int full = max_wpb;
    if (H % max_wpb != 0)
        for (int d = max_wpb - 1; d >= max_wpb / 2; --d)
            if (H % d == 0) { full = d; break; }
    const int first = forced_wpb ? forced_wpb : full;
    StripChoice best = {1, first};
    long least = -1;
    const int longest = forced_sb ? forced_sb : (eight ? 8 : most);
    for (int wpb : {first, 4}) {
        if (wpb != first && (forced_wpb || wpb > max_wpb || (H % wpb != 0 && H % full == 0))) continue;
        for (int sb = forced_sb ? forced_sb : 1; sb <= longest; sb *= 2) {
            const long wgs = (blocks / sb + wpb - 1) / wpb, rounds = (wgs + 255) / 256;
            if (wpb != first && rounds > 1) continue;
            const long one[] = {120, 100, 100, 100}, several[] = {170, 145, 115, 110};
            const int lg = sb == 1 ? 0 : sb == 2 ? 1 : sb == 4 ? 2 : 3;
            // in units of 1/1600 block; ties: more wavefronts in one round, longer strips in several
            const long cost = rounds * sb * wpb * (rounds > 1 ? several : one)[lg] * 16 + (rounds > 1 ? 8 / sb : sb);
            if (least < 0 || cost < least) {
                least = cost;
                best = {sb, wpb};
            }
        }
    }
    return best;
}

int attn_tile_dispatch(const void *q, const void *k, const void *v, void *out, float *weights, float *lse, int B,
                       int N, int M, int H, int D, int L, int R, int causal, int dtype, hipStream_t st) {
    if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0)
        return fail(HSA_ERR_INVALID, "tile kernel needs 16-byte aligned tensors");
    TileParams p;
    p.q = (const uint16_t *)q; p.k = (const uint16_t *)k; p.v = (const uint16_t *)v;
    p.out = (uint16_t *)out;
    p.weights = weights;
    p.lse = lse;
    p.B = B; p.N = N; p.M = M; p.H = H; p.L = L; p.R = R;
    const int NB = N / TILE_Q;
    TileKnobs &knobs = tile_knobs();
    const int nbw = (R + TILE_Q - 1) / TILE_Q;
    const bool part = tile_head_is_part(D);
    // longest strip the variant takes: four blocks, with four or five leaf blocks per query block two
    // (shorter strips keep the operands in registers), with more one
    int most = 4;
    if (nbw >= (causal ? 3 : 2)) most = 2;
    if (nbw >= 4 && !knobs.sb) most = 1;        // longer strips spill at five leaf blocks + halo
    if (!causal && nbw > TILE_MAX_NBW) most = 1;  // seven or nine leaf blocks: one block per wavefront
    if (weights) most = 1;
    while (most > NB) most >>= 1;               // NB is a power of two
    // two runs of four blocks: the window's neighbouring leaf blocks are fetched once per eight blocks
    const bool runs_built = most == 4 && !weights && !part && nbw >= 1 && nbw <= (causal ? 2 : 1) && NB >= 8;
    const StripChoice c = choose_strip((long)B * H * NB, H, D > 64 ? 4 : 8, most, runs_built && causal, knobs.sb, knobs.wpb);
    int sb = c.sb > 4 ? 4 : c.sb, runs = c.sb > 4 && runs_built ? 2 : 1;
    if (sb > most) sb = most;
    p.runs = runs;
    p.NS = NB / (sb * runs);
    sb *= runs;  // the launchers switch on the strip length
    const long units = (long)B * p.NS * H;
    if (units > 0x3fffffffL) return fail(HSA_ERR_UNSUPPORTED, "problem too large for one launch");
    p.n_units = (int)units;
    p.xcd_swizzle = knobs.swizzle;
    p.alternate = knobs.alternate;
    p.dh = D;
    p.scale_log2e = 1.4426950408889634f / sqrtf((float)D);
    const int wpb = c.wpb;
    if (weights) {
        // one query block per wavefront
        p.NS = NB;
        const long wunits = (long)B * NB * H;
        if (wunits > 0x3fffffffL) return fail(HSA_ERR_UNSUPPORTED, "problem too large for one launch");
        p.n_units = (int)wunits;
        if (dtype == HSA_BF16) {
            if (D == 32) return attn_tile_weights_launch_td<BF16, 32>(p, nbw, causal != 0, wpb, st);
            if (D == 64) return attn_tile_weights_launch_td<BF16, 64>(p, nbw, causal != 0, wpb, st);
            return attn_tile_weights_launch_td<BF16, 128>(p, nbw, causal != 0, wpb, st);
        }
        if (D == 32) return attn_tile_weights_launch_td<F16, 32>(p, nbw, causal != 0, wpb, st);
        if (D == 64) return attn_tile_weights_launch_td<F16, 64>(p, nbw, causal != 0, wpb, st);
        return attn_tile_weights_launch_td<F16, 128>(p, nbw, causal != 0, wpb, st);
    }
    if (lse && weights) return fail(HSA_ERR_UNSUPPORTED, "weights and log-sum-exp outputs together are not built");
    if (part) {
        const bool bf = dtype == HSA_BF16, c = causal != 0;
        if (D < 32) return bf ? attn_tile_part_launch_td<BF16, 32, 32>(p, nbw, c, sb, wpb, st)
                              : attn_tile_part_launch_td<F16, 32, 32>(p, nbw, c, sb, wpb, st);
        if (D < 64) return bf ? attn_tile_part_launch_td<BF16, 64, 64>(p, nbw, c, sb, wpb, st)
                              : attn_tile_part_launch_td<F16, 64, 64>(p, nbw, c, sb, wpb, st);
        if (D <= 96) return bf ? attn_tile_part_launch_td<BF16, 128, 96>(p, nbw, c, sb, wpb, st)
                               : attn_tile_part_launch_td<F16, 128, 96>(p, nbw, c, sb, wpb, st);
        return bf ? attn_tile_part_launch_td<BF16, 128, 128>(p, nbw, c, sb, wpb, st)
                  : attn_tile_part_launch_td<F16, 128, 128>(p, nbw, c, sb, wpb, st);
    }
    if (lse) {
        if (dtype == HSA_BF16) {
            if (D == 32) return attn_tile_lse_launch_td<BF16, 32>(p, nbw, causal != 0, sb, wpb, st);
            if (D == 64) return attn_tile_lse_launch_td<BF16, 64>(p, nbw, causal != 0, sb, wpb, st);
            return attn_tile_lse_launch_td<BF16, 128>(p, nbw, causal != 0, sb, wpb, st);
        }
        if (D == 32) return attn_tile_lse_launch_td<F16, 32>(p, nbw, causal != 0, sb, wpb, st);
        if (D == 64) return attn_tile_lse_launch_td<F16, 64>(p, nbw, causal != 0, sb, wpb, st);
        return attn_tile_lse_launch_td<F16, 128>(p, nbw, causal != 0, sb, wpb, st);
    }
    if (dtype == HSA_BF16) {
        if (D == 32) return attn_tile_launch_td<BF16, 32>(p, nbw, causal != 0, sb, wpb, st);
        if (D == 64) return attn_tile_launch_td<BF16, 64>(p, nbw, causal != 0, sb, wpb, st);
        return attn_tile_launch_td<BF16, 128>(p, nbw, causal != 0, sb, wpb, st);
    }
    if (D == 32) return attn_tile_launch_td<F16, 32>(p, nbw, causal != 0, sb, wpb, st);
    if (D == 64) return attn_tile_launch_td<F16, 64>(p, nbw, causal != 0, sb, wpb, st);
    return attn_tile_launch_td<F16, 128>(p, nbw, causal != 0, sb, wpb, st);
}

}  // namespace hsa
