// Instantiates the 16-bit tile kernels for part heads (head sizes other than 32 / 64 / 128, see
// hsa_attn_tile.h): forward and two-pass backward of one (element type, layout, contraction) triple,
// and the one-pass backward of one (element type, layout) pair.
//
// Built for window radius 1..32 (radius 0 runs on the radius-16 variants), strips of one, two and
// four blocks.
#pragma once
#include "hsa_attn_bwd_fused.h"

namespace hsa {

template <typename T, int D, int NBW, bool CAUSAL, int DC, bool LSE>
static int tile_part_launch_sb(const TileParams &p, int sb, int wpb, hipStream_t st) {
    constexpr int MAXW = tile_max_wpb<D, (CAUSAL ? NBW + 1 : 2 * NBW + 1)>();
    if (wpb > MAXW) wpb = MAXW;
    const int nwg = (p.n_units + wpb - 1) / wpb;
    const LaunchEvents ev = take_launch_events();
    if (ev.start && ev.stop) (void)hipEventRecord(ev.start, st);
    switch (sb) {
        case 1: attn_tile_kernel<T, D, NBW, CAUSAL, 1, false, LSE, 1, DC><<<nwg, wpb * 64, 0, st>>>(p); break;
        case 2: attn_tile_kernel<T, D, NBW, CAUSAL, 2, false, LSE, 1, DC><<<nwg, wpb * 64, 0, st>>>(p); break;
        case 4: attn_tile_kernel<T, D, NBW, CAUSAL, 4, false, LSE, 1, DC><<<nwg, wpb * 64, 0, st>>>(p); break;
        default: return fail(HSA_ERR_UNSUPPORTED, "strip length %d not built for part heads", sb);
    }
    const int rc = check_launch("attn_tile_kernel (part head)");
    if (ev.start && ev.stop) (void)hipEventRecord(ev.stop, st);
    return rc;
}

template <typename T, int D, int NBW, bool CAUSAL, int DC>
static int tile_part_launch(const TileParams &p, int sb, int wpb, hipStream_t st) {
    if (!p.lse) return tile_part_launch_sb<T, D, NBW, CAUSAL, DC, false>(p, sb, wpb, st);
    // the one-pass backward's range
    if constexpr (NBW == 1 || CAUSAL) return tile_part_launch_sb<T, D, NBW, CAUSAL, DC, true>(p, sb, wpb, st);
    return fail(HSA_ERR_UNSUPPORTED, "the log-sum-exp output is built for window radius up to 16, or 32 with the causal mask");
}

template <typename T, int D, int NBW, bool CAUSAL, int DC>
static int bwd_part_launch(const BwdTileParams &p, int sb, hipStream_t st) {
    BwdTileParams q = p;
    q.n_units = p.n_units / sb;
    q.red_lg_sb = sb == BWD_STRIP ? 2 : 0;
    const int nwg = (q.n_units + BWD_WPB - 1) / BWD_WPB;
    if (sb == BWD_STRIP) attn_bwd_tile_query_kernel<T, D, NBW, CAUSAL, BWD_STRIP, DC><<<nwg, BWD_WPB * 64, 0, st>>>(q);
    else if (sb == 1) attn_bwd_tile_query_kernel<T, D, NBW, CAUSAL, 1, DC><<<nwg, BWD_WPB * 64, 0, st>>>(q);
    else return fail(HSA_ERR_INVALID, "internal: strip length %d not built", sb);
    const int rc = check_launch("attn_bwd_tile_query_kernel (part head)");
    if (rc != HSA_OK) return rc;
    if (sb == BWD_STRIP)
        attn_bwd_tile_key_kernel<T, D, NBW, CAUSAL, BWD_STRIP, DC><<<nwg + q.red_wgs, BWD_WPB * 64, 0, st>>>(q);
    else attn_bwd_tile_key_kernel<T, D, NBW, CAUSAL, 1, DC><<<nwg + q.red_wgs, BWD_WPB * 64, 0, st>>>(q);
    return check_launch("attn_bwd_tile_key_kernel (part head)");
}

#define HSA_PART_INSTANTIATE(T, D, DC)                                                                       \
    template <>                                                                                              \
    int attn_tile_part_launch_td<T, D, DC>(const TileParams &p, int nbw, bool causal, int sb, int wpb,       \
                                           hipStream_t st) {                                                 \
        if (nbw > 2) return fail(HSA_ERR_UNSUPPORTED, "window radius too large for a part head");            \
        if (nbw == 2) return causal ? tile_part_launch<T, D, 2, true, DC>(p, sb, wpb, st)                    \
                                    : tile_part_launch<T, D, 2, false, DC>(p, sb, wpb, st);                  \
        return causal ? tile_part_launch<T, D, 1, true, DC>(p, sb, wpb, st)                                  \
                      : tile_part_launch<T, D, 1, false, DC>(p, sb, wpb, st);                                \
    }                                                                                                        \
    template <>                                                                                              \
    int attn_bwd_tile_part_launch_td<T, D, DC>(const BwdTileParams &p, int nbw, bool causal, int sb,         \
                                               hipStream_t st) {                                             \
        if (nbw > 2) return fail(HSA_ERR_UNSUPPORTED, "window radius too large for a part head");            \
        if (nbw == 2) return causal ? bwd_part_launch<T, D, 2, true, DC>(p, sb, st)                          \
                                    : bwd_part_launch<T, D, 2, false, DC>(p, sb, st);                        \
        return causal ? bwd_part_launch<T, D, 1, true, DC>(p, sb, st)                                        \
                      : bwd_part_launch<T, D, 1, false, DC>(p, sb, st);                                      \
    }

#define HSA_PART_FUSED_INSTANTIATE(T, D)                                                                     \
    template <>                                                                                              \
    int attn_bwd_fused_part_launch_td<T, D>(const BwdFusedParams &fp, bool causal, hipStream_t st) {         \
        return bwd_fused_launch<T, D, true>(fp, causal, st);                                                 \
    }

}  // namespace hsa
