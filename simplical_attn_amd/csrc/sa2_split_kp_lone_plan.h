// The K'-side backward kernel of the plane-split kernels with one wavefront per SIMD (sa2_split_kp_lone.h): its layout in LDS, and what a
// launch of it is made of.
#pragma once

#include "sa2_mfma_common.h"

namespace sa2 {

struct SplitKpLaunch {
    KpPlan plan;
    int nkb, per_seg;
    float *dq_part, *kpart;
};
// `width`: of the kernel; `two_planes`: products of a unit have 16 bits
int launch_split_kp_lone_bf16(const Problem& p, int width, bool two_planes, const SplitKpLaunch& l, hipStream_t st);
int launch_split_kp_lone_fp16(const Problem& p, int width, bool two_planes, const SplitKpLaunch& l, hipStream_t st);
int launch_split_kp_lone_fp32(const Problem& p, int width, bool two_planes, const SplitKpLaunch& l, hipStream_t st);

namespace {

// PLANES: of a K or V tile
template <int D, int PLANES>
struct SplitKpLoneCfg {
    static constexpr int W = 4, THREADS = W * 64;
    static constexpr int NK = PLANES, DK = D / 16, DT = D / 32;
    static constexpr bool DMA = NK == 1;       // tiles straight from global memory
    static constexpr int BLOCK = 2048, PLANE = DT * BLOCK, TILE = NK * PLANE, STAGE = 2 * TILE, NSTAGE = DMA ? 4 : 3;      // bytes
    static constexpr int AS = D + 4;           // fp32 accumulator row stride
    static constexpr size_t LDS_LIMIT = 160 * 1024;
    static constexpr size_t row_bytes(int rows) { return (size_t)((rows + 3) / 4) * QuadTile<128>::GROUP; }
    // raw = true: the q and dO rows the workgroup touches are copied to LDS; otherwise they are read from global memory once per unit
    static size_t main_bytes(int segw, bool raw) {
        const int rq = BQ + segw - 1;
        return (size_t)NSTAGE * STAGE + 2 * row_bytes(BQ) + (raw ? 2 * row_bytes(rq) : 0) + 2 * ((rq + 3) / 4 * 4) * 4 + (size_t)rq * AS * 4;
    }
    static size_t final_bytes() { return (size_t)W * 2 * BQ * AS * 4; }
    static size_t lds_bytes(int segw, bool raw) { return main_bytes(segw, raw) > final_bytes() ? main_bytes(segw, raw) : final_bytes(); }
    static bool raw_fits(int segw) { return lds_bytes(segw, true) <= LDS_LIMIT; }
    static bool fits(int segw) { return lds_bytes(segw, false) <= LDS_LIMIT; }
};

}  // namespace
}  // namespace sa2
