// The K'-side backward kernel for wide K windows (sa2_mfma_bwd_kp_lone.h): its layout in LDS, when it is taken, and what a
// launch of it is made of.
#pragma once

#include "sa2_mfma_common.h"

namespace sa2 {

// A launch of a main kernel of the K' side
struct KpLaunch {
    KpPlan plan;
    int nkb, total, left;
    float *dq_part, *kpart;
};
int launch_mfma_bwd_kp_lone_bf16(const Problem& p, const KpLaunch& l, hipStream_t st);
int launch_mfma_bwd_kp_lone_fp16(const Problem& p, const KpLaunch& l, hipStream_t st);

namespace {

template <int D>
struct KpLoneCfg {
    static constexpr int W = 4, T = W * 64;    // wavefronts, threads per workgroup
    static constexpr int U = D == 64 ? 2 : 1;  // units (consecutive deltas) a wavefront holds per round
    static constexpr int DK = D / 16, DT = D / 32;
    using Tile = QuadTile<D>;                  // K and V tiles in LDS
    static constexpr int NREQ = Tile::NGROUP / W;                    // groups of a tile a wavefront requests
    static constexpr int TILE_BYTES = Tile::BYTES;
    static constexpr int STAGE_BYTES = 2 * TILE_BYTES;               // K tile, then V tile
    static constexpr int NSTAGE = 4;
    static constexpr int AS = D + 4;           // fp32 accumulator row stride
    static constexpr size_t LDS_LIMIT = 160 * 1024;
    static constexpr size_t row_bytes(int rows) { return (size_t)((rows + Tile::RPW - 1) / Tile::RPW) * Tile::GROUP; }     // rows laid out as in a tile
    // raw = true: the q and dO rows the workgroup touches are copied to LDS; otherwise the
    // wavefronts read them from global memory once per unit.  wide = true: the K' rows lie there as (k2 + bias) * scale * log2(e) in
    // fp32, rather than as they are
    static size_t main_bytes(int w2, bool raw, bool wide = false) {
        const int rq = BQ + w2;
        return (size_t)NSTAGE * STAGE_BYTES + row_bytes(BQ) + (wide ? (size_t)BQ * AS * 4 : row_bytes(BQ)) + (raw ? 2 * row_bytes(rq) : 0) +
               2 * ((rq + 3) / 4 * 4) * 4 + (size_t)rq * AS * 4;
    }
    static size_t final_bytes() { return (size_t)W * 2 * BQ * AS * 4; }
    static size_t lds_bytes(int w2, bool raw, bool wide = false) { return main_bytes(w2, raw, wide) > final_bytes() ? main_bytes(w2, raw, wide) : final_bytes(); }
    static bool raw_fits(int w2) { return lds_bytes(w2, true) <= LDS_LIMIT; }
    static bool wide_fits(int w2) { return lds_bytes(w2, raw_fits(w2), true) <= LDS_LIMIT; }
    static bool fits(int w2) { return lds_bytes(w2, false) <= LDS_LIMIT; }
    // Whether the kernel is taken, by the keys a K' row's queries see on average (the window, less where the sequence begins): a tile of
    // the sweep takes it less than the two-wavefront kernel, but what lies between two sweeps and around them is not overlapped, and a
    // wavefront without a unit in a round is idle: `busy` is the keys per unit that a round has room for.  `units`: deltas of a
    // workgroup, `mean`: with the shorter last segment.  Fitted to both kernels at 150 shapes; time of the other one over this one's, K' side with its pre- and post-pass:
    // head_dim 64: N3000 BH8 w 150/9 0.98, /20 0.99, /31 1.02, w 250/4 1.01, /9 1.06, /31 1.08; N1500 BH8 w 250/20 1.06; N1000 BH30 w 250/31 1.10;
    //   BH16 N4096 w 256/64 1.15; one to three deltas 0.80 - 0.99 with up to 240 keys; N2600 BH4 w 150/40 (segments of 24 and 17) 0.96.  Many deltas on less than one and a half workgroups a CU:
    //   N6950 BH1 w 226/40 0.93, N2743 BH2 w 243/40 0.97, N1411 BH5 w 171/64 0.97, N1492 BH5 w 310/40 1.00, N649 BH11 w 420/23 1.06;
    //   fewer: N492 BH11 w 362/20 1.04, N969 BH7 w 272/20 1.02, N469 BH13 w 267/12 1.03, N886 BH9 w 359/8 0.93.
    // head_dim 128: N16384 BH8 w 260/4 1.02, /9 1.05, /31 1.08; N8192 BH3 w 300/4 0.96, /9 1.02, /31 1.04; N1000 BH30 w 300/31 1.06; N1200 BH6 w 260/31 0.90.
    //   Between one and three workgroups a CU both signs occur (0.96 - 1.10) and the older, later line stays.
    static bool wanted(int N, int w1, int units, double mean, int64_t workgroups) {
        const int64_t w = w1 < N ? w1 : N;
        const double keys = w - w * w / (2.0 * N), waves = (double)workgroups / CUS;
        const int rounds = (units + U * W - 1) / (U * W);
        const double busy = keys * mean / (rounds * U * W);
        if (D == 64) return (units >= 6 && busy >= 136 && (waves >= 1.5 || units < 24)) || (keys >= 300 && keys >= 250 + 1000.0 / units);
        return (units >= 8 && busy >= 210 && waves >= 3) || (keys >= 420 && keys >= 320 + (160 + 3000.0 / rounds) / waves);
    }
};

}  // namespace
}  // namespace sa2
