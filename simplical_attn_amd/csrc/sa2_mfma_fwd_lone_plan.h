// The 16-bit forward kernel with two units per wavefront (sa2_mfma_fwd_lone.h): its layout in LDS, when it is taken, and its arguments.
#pragma once

#include "sa2_mfma_common.h"

namespace sa2 {

struct FwdLoneArgs {
    Problem p;
    int nqb, total, left;                      // query blocks per head, workgroups, whether the pre-pass ran
};
int launch_mfma_fwd_lone_bf16(const FwdLoneArgs& args, hipStream_t st);
int launch_mfma_fwd_lone_fp16(const FwdLoneArgs& args, hipStream_t st);

namespace {

template <int D>
struct FwdLoneCfg {
    static constexpr int W = 4, T = W * 64;    // wavefronts, threads per workgroup
    static constexpr int U = 2, UPR = U * W;   // units (consecutive deltas) a wavefront holds per round, units of a round
    static constexpr int DK = D / 16, DT = D / 32;
    static constexpr int OWNED = U * (DT * 16 + DK * 4);             // accumulation registers
    static constexpr int PER_SIMD = D == 64 ? 2 : 1;                 // wavefronts per SIMD (two workgroups per CU at head_dim 64)
    static constexpr bool UNROLL = D == 128;   // tiles of a sweep in fours: 1080 against 1095 us at B1 H16 N8192 w 512/31; at head_dim 64 +3 %
    static constexpr bool MAXIMA_FIRST = D == 128;                   // in the second pass: a sweep for the reference points (sa2_mfma_fwd_lone.h)
    using Tile = QuadTile<D>;                  // K and V tiles in LDS
    static constexpr int NREQ = Tile::NGROUP / W;                    // groups of a tile a wavefront requests
    static constexpr int TILE_BYTES = Tile::BYTES;
    static constexpr int STAGE_BYTES = 2 * TILE_BYTES;               // K tile, then V tile
    static constexpr int NSTAGE = 4;
    static constexpr int SLOTS = 64;           // rows of the K' and V' rings
    static constexpr int QS = D + 4, AS = D + 4;                     // row strides of q and of the merged sums (fp32)
    static constexpr int K2_AT = NSTAGE * STAGE_BYTES, V2_AT = K2_AT + SLOTS / Tile::RPW * Tile::GROUP;
    static constexpr int Q_AT = V2_AT + SLOTS / Tile::RPW * Tile::GROUP, X_AT = Q_AT + BQ * QS * 4;
    static constexpr int UP_AT = X_AT + (2 * W + 1) * BQ * 4, LDS_BYTES = UP_AT + 16;
    static_assert(W * BQ * AS * 4 <= Q_AT, "the merged sums lie over the rings");
    static_assert(LDS_BYTES <= 160 * 1024, "");
    // Gradients of the first queries, whose weights are few, follow the rounding of their outputs closely.  At head_dim 128 the
    // eight-wavefront kernel rounds to 16 bits between rounds and this one does not: it leaves the first block of every head to that
    // one, in a launch of its own (about 20 us), so that gradients do not depend on which kernel a problem is given to.
    static constexpr bool FIRST_ELSEWHERE = D == 128;
    // Whether the kernel is taken rather than the one with eight wavefronts of one unit.  head_dim 64: where two workgroups share a
    // CU, from more workgroups than CUs on.  Time of the other kernel over this one's, bf16: B1 H16 N4096 w 16 .. 1024/31 1.51 - 1.22,
    // w2 0 .. 8 1.40 - 1.63; B1 H8 w 256/31 N1056 (264 blocks) 1.32, N1024 (256; w 128/16) 0.89, 64 blocks 0.98, 128 in two shares 0.95.
    // head_dim 128, without the further launch: where a wavefront's two units are mostly there, since a round takes the same with
    // one (B1 H16 N4096 w 512: w2 1 0.81, 3 0.84, 4 .. 6 0.96 - 0.99, 7 1.05, 11 0.97, 12 1.01, 19 1.03, 31 1.10), and with it, where
    // the sweeps are long enough: a round gains about 0.1 us per tile and CU.
    static bool wanted(int64_t workgroups, int units, int N, int w1) {
        if (D == 64) return workgroups > CUS;
        const int rounds = (units + UPR - 1) / UPR;
        const int64_t w = w1 < N ? w1 : N;
        return 4 * units > 3 * UPR * rounds && workgroups * rounds * ((w - w * w / (2 * (int64_t)N)) / TJ + 1) >= FIRST_PAYS;
    }
    static constexpr int64_t FIRST_PAYS = 120000;
};

}  // namespace
}  // namespace sa2
