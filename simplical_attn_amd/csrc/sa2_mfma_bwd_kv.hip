// MFMA backward for gfx950, the K-side kernel (dK and dV): how a launch divides its work.  The kernel is in
// sa2_mfma_bwd_kv.h, compiled once per element type.
#include "sa2_mfma_common.h"

namespace sa2 {
int launch_mfma_bwd_kv_bf16(const Problem& p, int kb, int nsplit, hipStream_t st, BwdSums* sums);
int launch_mfma_bwd_kv_fp16(const Problem& p, int kb, int nsplit, hipStream_t st, BwdSums* sums);
namespace {

constexpr int KV_MAX_SPLIT = 16;       // workgroups a key block's stream of units is split over, at most
constexpr int KV_MIN_SHARE = 4, KV_MIN_SHARE_ONE = 2;      // units a share holds at least; where all are of one query block

// Geometry of a launch: 32-row K blocks per wavefront, and the number of shares a key block's stream of units is split into:
// the cut that ends first by a model in microseconds: a unit's time by head_dim and blocks, what a change of the query block
// costs beside it, prologue and epilogue, the partial sums' bytes and their summation launch.  Workgroups that all start at once
// take as long as the longest; more of them fill the chip one behind the other, which ends behind the mean load by 0.6 of the
// longest, or in whole waves if that is sooner (workgroups of one length).  The launch that adds the partial sums takes 4 us where
// there are few, 6.5 from 64 Ki elements on.  Against every cut at 59 sizes (profiles/plan_cuts.md): within 3 % of the best at 46,
// 3 - 18 % off at 12 (most of one head or up to 64 queries, 1 to 3 us), and 43 % where the bytes bind.  The partial sums
// stay under what SA2_STATIC_WORKSPACE_BYTES leaves beside the K'-side kernel's, or 128 MiB where those alone exceed it.
// Measured with the row term and the sums (us, the kernel with two wavefronts per SIMD -> now): B2 H4 N512 D64 w 256/256
// 256 -> 185, B3 H6 N777 D64 w 100/20 102 -> 68, B2 H8 N2048 D64 w 512/32 458 -> 323, B5 H29 N448 D32 w 816/96 1183 -> 1130 (two
// shares, all that the bytes allow; the best eight take 790), B1 H4 N2048 D128 w 512/32 199 -> 160, B2 H4 N17 D64 w 16/16 14.2 -> 13.8.
// At head_dim 128 and up to 130 queries the present kernel is 1 to 2 us slower than that one (B2 H4 w 128/24, N 33 18.4 -> 20.3, N 130
// 30.8 -> 31.6): its own time, 12.8 -> 14.7 us for shares of five units.
struct KvPlan {
    int kb, nsplit;
};
double kv_time(int64_t workgroups, double longest, double mean) {
    if (workgroups <= CUS) return longest;
    const double waves = (double)((workgroups + CUS - 1) / CUS) * longest, filled = (double)workgroups / CUS * mean + 0.6 * longest;
    return waves < filled ? waves : filled;
}
KvPlan kv_plan(int B, int N, int H, int D, int w1, int w2, size_t room) {
    KvPlan best{1, 1};
    const int64_t bh = (int64_t)B * H;
    const int per = (w2 < N - 1 ? w2 : N - 1) + 1;                                   // units of a query block, at most
    const double kp = (double)kp_side_scratch_bytes(B, N, H, D, w1, w2, room), other = kp + (double)bh * N * 4 + 1024;
    double cap = other < (double)SA2_STATIC_WORKSPACE_BYTES ? (double)SA2_STATIC_WORKSPACE_BYTES - other : 134217728.0;
    if (cap > (double)room - kp) cap = (double)room - kp;
    const double elements = (double)bh * N * D, sum_launch = 4 + 2.5 * (elements < 65536 ? elements / 65536 : 1);
    double least = 0;
    for (int kb = 1; kb <= (D <= 64 ? 2 : 1); ++kb) {
        const int vj = 128 * kb, njb = (N + vj - 1) / vj;
        const int64_t base = bh * njb;
        // query blocks a key block streams: at most, and on average (fewer at the end of the sequence)
        const int nqb = (N + BQ - 1) / BQ;
        int blocks = (vj + (w1 < N ? w1 : N) + BQ - 1) / BQ + 1;
        blocks = blocks < nqb ? blocks : nqb;
        double mean_blocks = 0;
        const int sampled = njb < 64 ? njb : 64;
        for (int x = 0; x < sampled; ++x) {
            const int64_t jb = (int64_t)x * njb / sampled, last = jb * vj + vj - 1 + w1;
            mean_blocks += (double)((last < N - 1 ? last : N - 1) / BQ - jb * vj / BQ + 1) / sampled;
        }
        const double unit = D == 128 ? 0.77 : D == 64 ? (kb == 2 ? 0.69 : 0.433) : kb == 2 ? 0.558 : 0.417, change = 0.56;
        const double longest = blocks * (per * unit + change), mean = mean_blocks * (per * window_fill(w2, N) * unit + change);
        for (int ns = 1; ns <= KV_MAX_SPLIT; ++ns) {
            const double part = ns > 1 ? 2.0 * ns * bh * N * D * 4 : 0;
            if (ns > 1 && (base * ns > 16 * CUS || (int64_t)blocks * per / ns < (blocks == 1 ? KV_MIN_SHARE_ONE : KV_MIN_SHARE) || part > cap)) break;
            // (an XCD hands its workgroups to its four shader engines in turn: where key blocks and shares repeat as often, one engine
            // has all the longest)
            const double each = longest / ns + 3.8, most = (double)((base * ns + CUS - 1) / CUS) * each;
            const double run = base * ns > CUS && njb > 1 && 4 % (njb * ns) == 0 ? most : kv_time(base * ns, each, mean / ns + 3.8);
            const double cost = run + (ns > 1 ? sum_launch + part / 3.3e6 : 0);
            if (least == 0 || cost < least) {
                least = cost;
                best = KvPlan{kb, ns};
            }
        }
    }
    return best;
}

}  // namespace

size_t kv_split_scratch_bytes(int B, int N, int H, int head_dim, int w1, int w2, size_t room) {
    const int D = mfma_width(head_dim);
    const KvPlan pl = kv_plan(B, N, H, D, w1, w2, room);
    return pl.nsplit > 1 ? (size_t)2 * pl.nsplit * B * H * (size_t)N * D * sizeof(float) : 0;
}

int mfma_kv_route(int B, int N, int H, int head_dim, int w1, int w2) {
    const KvPlan pl = kv_plan(B, N, H, mfma_width(head_dim), w1, w2, ROOM_ANY);
    return pl.kb | pl.nsplit << 8;
}

int launch_mfma_bwd_kv(const Problem& p, int dtype, hipStream_t st, BwdSums* sums) {
    const KvPlan pl = kv_plan(p.B, p.N, p.H, mfma_width(p.D), p.w1, p.w2, p.room);
    return dtype == SA2_F16 ? launch_mfma_bwd_kv_fp16(p, pl.kb, pl.nsplit, st, sums) : launch_mfma_bwd_kv_bf16(p, pl.kb, pl.nsplit, st, sums);
}

}  // namespace sa2
