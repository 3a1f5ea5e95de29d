// fp32 arithmetic on the 16-bit matrix pipes of gfx950: fp32 tensors of head dims up to 128, and 16-bit tensors of
// the head dims the 16-bit kernels do not have, in kernels 32, 64, 96 and 128 columns wide.
//
// Every operand is carried as a sum of bf16 planes: x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m),
// which holds all 24 bits of an fp32 value (under 2^-110 those down to 2^-133; blocks of such values, and infinities, are
// computed by rows, see the end of split_fwd_kernel and split_guard_kernel).  A product of two such sums is taken as the MFMAs h*h, h*m, m*h, h*l, l*h, m*m
// (v_mfma_f32_32x32x16_bf16: exact 16-bit products, a sum rounded to nearest once per eight of them); what is left out,
// m*l + l*m + l*l, is below 2^-25 of |x*y| and below 2^-27 in the mean.  bf16 tensors are one plane and fp16 tensors two,
// exactly, so that with a three-plane partner they take three and five MFMAs.
//
// Errors against fp64 (relative 2-norm, N(0,1) inputs; dq, dk1, dv1, dv2 in units of 1e-7), here and before:
//   B1 H2 N128 D64 w 32/16     4.1 4.7 3.7 2.4   v_mfma_f32_32x32x2_f32 5.1 5.8 4.5 2.7, fp32 FMA kernels 3.3 3.6 2.3 2.1
//   B1 H1 N2048 D64 w 512/32   5.5 7.5 6.3 3.2   v_mfma_f32_32x32x2_f32 6.6 9.2 7.4 4.0, fp32 FMA kernels 5.0 7.7 7.3 3.3
//   B1 H1 N1024 D96 w 512/32   4.6 4.9 3.4 2.6   fp32 FMA kernels 4.7 8.0 7.3 3.0
// (the outputs of 32, 64 and 128 columns stood on the fp32 MFMA before, the others on the FMA kernels).
//
// Why: v_mfma_f32_32x32x2_f32 runs at a sixteenth of the bf16 rate; six bf16 MFMAs do the same work in 6/16 of its
// time.  The price is vector work (about 5.5 instructions to split a value), which runs beside the MFMAs.
//
// Same expanded-row view as the 16-bit kernels: rows r = (i, delta), Q~[r] = q[i] * (k2[i-delta] + k2_bias) *
// scale*log2(e), dO~[r] = dO[i] * (v2[i-delta] + v2_bias), formed in fp32 and then split.  With the logits computed
// transposed (S^T = K1 . Q~^T) a lane's accumulator registers are, once split, the B operand of R^T += V1^T . P^T.
//
// K/V (or unit) tiles go through LDS as planes, row-major with a row stride of D + 16 elements: row operands are 16-byte
// reads of a row, transposed operands ds_read_b64_tr_b16 reads of the same tile.  (Neither is free of bank conflicts in every width: at
// head_dim 64 in fp32 38 to 43 % of the cycles of LDS are lost to them, see profiles/pmc_counters_c2f32.md.)  A tile
// is read from global memory into registers a step ahead, split on its way into LDS, one barrier per tile.
//
//   split_fwd_kernel    32 queries per workgroup; wavefront w takes delta = w, w+W, ... and keeps one
//                       online softmax and one output accumulator across its units; the W are
//                       merged once at the end.
//                       At 64 columns (fp32 but for the finer sums) and in 16 bits at 96 mostly sa2_split_fwd_lone.h (lone_forward
//                       below).  Backward: fp32 at 64 columns and less (but for the finer sums) and 16 bits at 64 and 96 mostly
//                       sa2_split_kp_lone.h (lone_kp) and sa2_split_kv_lone.h (lone_kv).
//   split_kp_kernel     32 K' rows per workgroup and every delta (or a segment of them).  After a unit's
//                       sweep its three reductions go to fp32 accumulators in LDS in column-rotated
//                       phases: dK' and dV' rows are aligned with the unit's rows, dQ rows are shifted by
//                       delta; the dQ accumulator is written once per workgroup as a partial.
//   split_kv_kernel     128 K/V rows per workgroup (32 per wavefront pair, resident in registers as B
//                       operands), streaming every unit (query block, delta) that can see them.
// The backward kernels pair their eight wavefronts as the 16-bit kernels do (one P and one dS wavefront per SIMD, so that
// each holds the planes of one operand and one accumulator in 256 registers: four wavefronts that did both needed 350 and
// moved 136 of them between the two register files per tile; at 128 columns in fp32 they do not fit all the same, and 470
// bytes per lane of the K'-side kernel and 300 of the K-side one go through scratch memory).  A step has two halves.  In the first the P wavefront
// computes S and, beside the other's dP MFMAs, the exponentials and the split of P; in the second it adds P's product
// while the dS wavefront multiplies and splits dS, whose product follows.
// Every output element has one writer and a fixed summation order: no atomics, bitwise reproducible.
#include "sa2_fma_rows.h"
#include "sa2_split_kp_lone_plan.h"
#include "sa2_split_common.h"

namespace sa2 {
namespace {

constexpr int NPAIR = 4;               // wavefront pairs per workgroup of the backward kernels
constexpr int XT = NPAIR * 2 * 64;     // threads per workgroup
constexpr int XJ = NPAIR * 32;         // K rows per workgroup of the K-side kernel

template <class T, int D>
struct SplitCfg {
    static constexpr int NK = T::PLANES;       // planes of a K or V tile
    static constexpr bool LIMIT = T::DTYPE == SA2_F32;
    static constexpr int DK = D / 16;          // k-steps of a contraction over head_dim
    static constexpr int DT = D / 32;          // 32-column blocks of an output contraction
    static constexpr int RS = D + 16;          // row stride of a plane (elements)
    static constexpr int RSB = RS * 2;         // ... in bytes
    static constexpr int PLANE = 32 * RS;      // elements
    static constexpr int AS = D + 4;           // row stride of fp32 accumulators in LDS
    static constexpr size_t LDS_LIMIT = 160 * 1024;
    // Forward: eight wavefronts (two per SIMD) where operands and accumulators fit 256 registers, else four.
    static constexpr int FW = D <= 64 ? 8 : 4;
    static constexpr int KV_TILE = NK * PLANE;             // a K or V tile
    static constexpr int KV_STAGE = 2 * KV_TILE;           // K tile, then V tile
    static constexpr size_t FWD_TILES = (size_t)2 * KV_STAGE * 2;
    static constexpr size_t FWD_MERGE = (size_t)FW * 32 * AS * 4;
    static constexpr size_t FWD_FMA = smem_bytes(D, FW);
    static constexpr size_t larger(size_t a, size_t b) { return a > b ? a : b; }
    static constexpr size_t FWD_LDS = larger(FWD_FMA, larger(FWD_TILES, FWD_MERGE)) + 2 * FW * 32 * 4;
    // K'-side: two stages, or one (a barrier more per tile) where two would leave no room for the dQ accumulator
    static constexpr int KP_STAGES = D == 128 && NK == 3 ? 1 : 2;
    static constexpr size_t KP_TILES = (size_t)KP_STAGES * KV_STAGE * 2;
    static constexpr size_t PX_BYTES = (size_t)NPAIR * 4096;           // P on its way to the dS wavefront: fp32, a tile per pair
    // the stages, P, the dQ accumulator (32 + w2 rows) and the dK' and dV' accumulators (32 rows each)
    static size_t kp_lds(int w2) { return KP_TILES + PX_BYTES + (size_t)(32 + w2 + 64) * AS * 4; }
    static bool kp_fits(int w2) { return kp_lds(w2) <= LDS_LIMIT; }
    // K-side: a unit is the Q~ and dO~ tiles of three planes
    static constexpr int UNIT_TILE = 3 * PLANE;
    static constexpr int UNIT_STAGE = 2 * UNIT_TILE;
    static constexpr size_t KV_LDS = (size_t)2 * UNIT_STAGE * 2 + PX_BYTES + 2 * 2 * 32 * 16;
};

// c += a * b over the plane products m*m, h*l, l*h (sum 2), h*m, m*h (1) and h*h (0) with LO <= sum <= HI, the small ones
// first
template <int LO, int HI, int NA, int NB>
__device__ __forceinline__ floatx16 mma_sums(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], floatx16 c) {
#pragma unroll
    for (int sum = HI; sum >= LO; --sum)
#pragma unroll
        for (int x = 0; x < NA; ++x)
            if (sum - x >= 0 && sum - x < NB) c = ElemBF16::mfma(a[x], b[sum - x], c, 0, 0, 0);
    return c;
}
template <int NA, int NB>
__device__ __forceinline__ floatx16 mma(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], floatx16 c) {
    return mma_sums<0, 2>(a, b, c);
}
// A contraction over head_dim.  An MFMA rounds its sum once per eight products, so a chain of all plane products rounds
// 0.75 D times at the size of the result.  FINE: the small products have a chain of their own, which leaves D / 8.  With
// accumulate() below it costs B1 H8 N1024 D96 w 256/32 fp32 1.14 -> 1.32 ms a step and takes its errors from 1.3 times the
// FMA kernels' to theirs.
template <bool FINE>
struct Chain {
    floatx16 main, small;
    __device__ __forceinline__ void clear() {
        main = zero16();
        if constexpr (FINE) small = zero16();
    }
    template <int NA, int NB>
    __device__ __forceinline__ void add(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB]) {
        if constexpr (FINE) {
            small = mma_sums<1, 2>(a, b, small);
            main = mma_sums<0, 0>(a, b, main);
        } else {
            main = mma(a, b, main);
        }
    }
    __device__ __forceinline__ floatx16 sum() const {
        if constexpr (FINE) return main + small;
        else return main;
    }
};
// acc += the product of a 32-row tile; `operand(ks, dt, a)` reads its transposed operand.  FINE: the tile is summed by
// itself, so that the accumulator over all tiles is rounded once per tile instead of 24 times.
template <bool FINE, int NA, int DT, class Read>
__device__ __forceinline__ void accumulate(floatx16 (&acc)[DT], const bf16x8 (&b)[2][3], Read&& operand) {
    if constexpr (FINE) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            bf16x8 a[2][NA];
            floatx16 t = zero16();
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                operand(ks, dt, a[ks]);
                t = mma_sums<1, 2>(a[ks], b[ks], t);
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) t = mma_sums<0, 0>(a[ks], b[ks], t);
            acc[dt] += t;
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                bf16x8 a[NA];
                operand(ks, dt, a);
                acc[dt] = mma(a, b[ks], acc[dt]);
            }
    }
}
constexpr int mma_count(int na, int nb = 3) {
    int n = 0;
    for (int x = 0; x < na; ++x)
        for (int y = 0; y < nb; ++y) n += x + y <= 2;
    return n;
}
// Spreads VALU instructions over the MFMAs of the block it closes
template <int MFMAS, int VALUS>
__device__ __forceinline__ void interleave() {
    constexpr int PER = (VALUS + MFMAS - 1) / MFMAS;
#pragma unroll
    for (int x = 0; x < MFMAS; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x402, PER, 0);
    }
}
// Row operand (rows of the tile as MFMA rows) of k-step kk and transposed operand (rows as the contraction index) of
// k-step ks and 32-column block dt, all planes.  `addr`: LDS byte address of plane 0 plus the lane part.
template <int N, int RSB>
__device__ __forceinline__ void row_operand(uint32_t addr, int kk, bf16x8 (&o)[N]) {
#pragma unroll
    for (int n = 0; n < N; ++n) o[n] = lds_read_x8(addr + (uint32_t)(n * 32 * RSB + kk * 32));
}
// Lane part of a transposed read: within 16 lanes, lane s supplies the address of row s/4, columns 4*(s%4)..+3, and lane
// i receives column i of those four rows; the four 16-lane groups take the rows 0-3 / 4-7 (by half) of the 16-column
// halves of a 32-column block, so that the eight values are the k-slots of a 32x32 accumulator handed on.
template <int RSB>
__device__ __forceinline__ uint32_t column_lane(int lane) {
    const int grp = lane >> 4, s = lane & 15;
    return (uint32_t)((4 * (grp >> 1) + (s >> 2)) * RSB + (16 * (grp & 1) + 4 * (s & 3)) * 2);
}
template <int N, int RSB>
__device__ __forceinline__ void column_operand(uint32_t addr, int ks, int dt, bf16x8 (&o)[N]) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef v4s __attribute__((address_space(3)))* lds_v4s;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        union { v4s h[2]; bf16x8 v; } u;
        const uint32_t a = addr + (uint32_t)(n * 32 * RSB + 16 * ks * RSB + dt * 64);
        u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)a);
        u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(a + 8 * RSB));
        o[n] = u.v;
    }
}

// Rows [j0, j0+32) of two tensors (clamped to the sequence) from global memory to registers, and
// from there, split, to the two tiles of a stage.  NT threads.
template <class T, int D, int NT>
struct TileRegs {
    static constexpr int ALL = 32 * D / 4, KR = (ALL + NT - 1) / NT;       // groups of four columns: of a tile, per thread
    typename T::Raw a[KR], b[KR];
    template <bool PAD>
    __device__ __forceinline__ void load(const typename T::T* ap, int64_t as, const typename T::T* bp, int64_t bs, int j0, int N, int tid, int width) {
#pragma unroll
        for (int u = 0; u < KR; ++u) {
            const int c = tid + NT * u;
            if (ALL % NT != 0 && c >= ALL) break;
            const int row = c / (D / 4), col = c - row * (D / 4);
            int j = j0 + row;
            j = j < N ? j : N - 1;
            a[u] = raw4<T, PAD>(ap + (int64_t)j * as, col * 4, width);
            b[u] = raw4<T, PAD>(bp + (int64_t)j * bs, col * 4, width);
        }
    }
    __device__ __forceinline__ void store(uint16_t* stage, int tid) const {
        using C = SplitCfg<T, D>;
#pragma unroll
        for (int u = 0; u < KR; ++u) {
            const int c = tid + NT * u;
            if (ALL % NT != 0 && c >= ALL) break;
            const int row = c / (D / 4), col = c - row * (D / 4);
            store_planes<C::NK, C::LIMIT>(T::widen(a[u]), stage + row * C::RS + col * 4, C::PLANE);
            store_planes<C::NK, C::LIMIT>(T::widen(b[u]), stage + C::KV_TILE + row * C::RS + col * 4, C::PLANE);
        }
    }
};
// The product row x * (y + bias) * mul of eight columns from `col` on, split into three planes; N = 2: x * y, which of two bf16 values
// has 16 bits and two planes hold exactly
template <class T, bool PAD, int N = 3>
__device__ __forceinline__ void product_planes(const typename T::T* xrow, const typename T::T* yrow, int col, int width, float bias, float mul,
                                               bf16x8 (&o)[N]) {
    const float4 x0 = cols4<T, PAD>(xrow, col, width), x1 = cols4<T, PAD>(xrow, col + 4, width);
    const float4 y0 = cols4<T, PAD>(yrow, col, width), y1 = cols4<T, PAD>(yrow, col + 4, width);
    if constexpr (N == 2) {
        const float r[8] = {x0.x * y0.x, x0.y * y0.y, x0.z * y0.z, x0.w * y0.w, x1.x * y1.x, x1.y * y1.y, x1.z * y1.z, x1.w * y1.w};
        split8<2>(r, o);
        return;
    }
    const float r[8] = {x0.x * mul * (y0.x + bias), x0.y * mul * (y0.y + bias), x0.z * mul * (y0.z + bias), x0.w * mul * (y0.w + bias),
                        x1.x * mul * (y1.x + bias), x1.y * mul * (y1.y + bias), x1.z * mul * (y1.z + bias), x1.w * mul * (y1.w + bias)};
    split8<N>(r, o);
}

// ================================================================== forward =====
// SPLIT: one of nsplit shares of the rounds, unnormalised sums to the workspace (see launch_fwd_merge).
// NQ: planes of Q~; two where q*k2 has 16 bits (exact_products below): the scale is multiplied onto the logits instead, which take
// two MFMAs per k-step rather than three.
template <class T, int D, int MODE, bool SPLIT, int NQ>
__global__ __launch_bounds__((SplitCfg<T, D>::FW * 64)) __attribute__((amdgpu_waves_per_eu(SplitCfg<T, D>::FW / 4, SplitCfg<T, D>::FW / 4)))
void split_fwd_kernel(Problem p, int nqb, int total) {
    using C = SplitCfg<T, D>;
    constexpr int W = C::FW, NT = W * 64;
    constexpr bool PAD = MODE != EXACT, FINE = MODE == PADDED_FINE;
    typedef typename T::T EL;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_f[];
    uint16_t* tiles = (uint16_t*)smem_f;                                             // two stages
    float* mrg_m = (float*)(smem_f + (C::FWD_LDS - (size_t)2 * W * 32 * 4));         // [W][32]
    float* mrg_l = mrg_m + W * 32;                                                   // [W][32]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    int pid = xcd_order(blockIdx.x, total), share = 0;
    if constexpr (SPLIT) {
        share = pid % p.nsplit;
        pid /= p.nsplit;
    }
    const int bh = pid / nqb, qb = pid - bh * nqb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int i0 = qb * BQ, i = i0 + ln, ic = i < N ? i : N - 1;
    const int i_last = i0 + BQ - 1 < N ? i0 + BQ - 1 : N - 1;

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k1p = (const EL*)p.k1.p + p.k1.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v1p = (const EL*)p.v1.p + p.v1.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);

    const int jt_lo = (i0 - w1 > 0 ? i0 - w1 : 0) / TJ, jt_hi = i_last / TJ;
    const int nt = jt_hi - jt_lo + 1;
    const int n_units = (w2 < i_last ? w2 : i_last) + 1;
    const int all_rounds = (n_units + W - 1) / W;
    const int per_share = SPLIT ? ((w2 + W) / W + p.nsplit - 1) / p.nsplit : all_rounds;
    const int round0 = SPLIT ? share * per_share : 0;
    const int round1 = round0 + per_share < all_rounds ? round0 + per_share : all_rounds;
    if (SPLIT && round0 >= round1) {             // a block near the start of the sequence has fewer rounds
        if (tid < 32 && i0 + tid < N)
            ((float2*)p.scratch)[(int64_t)share * p.B * p.H * N + (int64_t)bh * N + i0 + tid] = make_float2(-INFINITY, 0.f);
        return;
    }
    const float qscale = p.scale * LOG2E;

    const uint32_t tiles_addr = lds_address(tiles);
    const uint32_t row_lane = (uint32_t)(ln * C::RSB + hf * 16), col_lane = column_lane<C::RSB>(lane);

    TileRegs<T, D, NT> next;                     // the tile on its way from global memory to LDS
    auto request = [&](int s) { next.template load<PAD>(k1p, p.k1.sn, v1p, p.v1.sn, (jt_lo + s) * TJ, N, tid, p.D); };
    request(0);
    next.store(tiles, tid);
    request(1 % nt);
    __syncthreads();

    // the wavefront's running softmax over its units: reference exponent, sum, weighted output
    float M = -INFINITY, L = 0.f;
    floatx16 oacc[C::DT];
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) oacc[dt] = zero16();

    int g = 0;
    for (int round = round0; round < round1; ++round) {
        const int delta = round * W + wave;
        const bool ok = delta < n_units;
        const int kr = ic - delta > 0 ? ic - delta : 0;
        const bool row_ok = ok && i < N && i >= delta;
        const bool rows_full = i0 >= delta && i0 + BQ - 1 < N;

        bf16x8 qf[C::DK][NQ];
        if (ok) {
#pragma unroll
            for (int kk = 0; kk < C::DK; ++kk)
                product_planes<T, PAD, NQ>(qp + (int64_t)ic * p.q.sn, k2p + (int64_t)kr * p.k2.sn, kk * 16 + hf * 8, p.D, p.k2_bias, qscale, qf[kk]);
        }
        float m = -INFINITY, l = 0.f;
        floatx16 racc[C::DT];
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) racc[dt] = zero16();

        for (int s = 0; s < nt; ++s, ++g) {
            if (ok) {
                const int j0 = (jt_lo + s) * TJ;
                const uint32_t Ks = tiles_addr + (uint32_t)((g & 1) * C::KV_STAGE * 2);
                const uint32_t Vt = Ks + (uint32_t)(C::KV_TILE * 2) + col_lane;
                Chain<FINE> logits;
                logits.clear();
#pragma unroll
                for (int kk = 0; kk < C::DK; ++kk) {
                    bf16x8 ka[C::NK];
                    row_operand<C::NK, C::RSB>(Ks + row_lane, kk, ka);
                    logits.add(ka, qf[kk]);
                }
                floatx16 sacc = logits.sum();
                if constexpr (NQ == 2) sacc *= qscale;
                // register v of this lane: key j0 + 8*(v/4) + 4*hf + v%4
                const bool interior = rows_full && (j0 + TJ - 1 <= i0) && (j0 >= i0 + BQ - 1 - w1);
                if (!interior) {
                    const int hi = i - j0 - 4 * hf, lo = hi - w1;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int c = 8 * (v >> 2) + (v & 3);
                        sacc[v] = (row_ok && c <= hi && c >= lo) ? sacc[v] : -INFINITY;
                    }
                }
                float mx = sacc[0];
#pragma unroll
                for (int v = 1; v < 16; ++v) mx = fmaxf(mx, sacc[v]);
                mx = fmaxf(mx, other_half(mx));
                const float m_new = fmaxf(m, mx);
                const float m_use = m_new == -INFINITY ? 0.f : m_new;
                const float alpha = fast_exp2(m - m_use);
                m = m_new;
                if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
                    l *= alpha;
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                        for (int v = 0; v < 16; ++v) racc[dt][v] *= alpha;
                }
                bf16x8 pb[2][3];
                float rs = 0.f;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    float pv[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        pv[t] = fast_exp2(sacc[8 * ks + t] - m_use);
                        rs += pv[t];
                    }
                    split8<3>(pv, pb[ks]);
                }
                l += rs;
                accumulate<FINE, C::NK>(racc, pb, [&](int ks, int dt, bf16x8 (&va)[C::NK]) { column_operand<C::NK, C::RSB>(Vt, ks, dt, va); });
            }
            // (unconditional: past the last step this moves a tile nobody reads, which is cheaper than a branch
            // around register arrays)
            next.store(tiles + ((g + 1) & 1) * C::KV_STAGE, tid);
            request((s + 2) % nt);
            __syncthreads();
        }

        if (ok) {
            // fold the unit into the wavefront's running result: O += e^(m-M) * (v2 + bias) * R
            const float lt = l + other_half(l);
            const float M_new = fmaxf(M, m);
            const float Mu = M_new == -INFINITY ? 0.f : M_new;
            const float a = fast_exp2(M - Mu), c = fast_exp2(m - Mu);
            L = L * a + lt * c;
            M = M_new;
            const EL* vrow = v2p + (int64_t)kr * p.v2.sn;
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const float4 x = cols4<T, PAD>(vrow, dt * 32 + 8 * g4 + 4 * hf, p.D);
                    oacc[dt][4 * g4 + 0] = oacc[dt][4 * g4 + 0] * a + c * racc[dt][4 * g4 + 0] * (x.x + p.v2_bias);
                    oacc[dt][4 * g4 + 1] = oacc[dt][4 * g4 + 1] * a + c * racc[dt][4 * g4 + 1] * (x.y + p.v2_bias);
                    oacc[dt][4 * g4 + 2] = oacc[dt][4 * g4 + 2] * a + c * racc[dt][4 * g4 + 2] * (x.z + p.v2_bias);
                    oacc[dt][4 * g4 + 3] = oacc[dt][4 * g4 + 3] * a + c * racc[dt][4 * g4 + 3] * (x.w + p.v2_bias);
                }
        }
    }

    // ---- merge the wavefronts (the tile stages are free: the sweep's last barrier is behind us) ----
    float* mrg = (float*)smem_f;                           // [W][32][AS]
    {
        float* row = mrg + (wave * 32 + ln) * C::AS + 4 * hf;
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
                *(float4*)(row + dt * 32 + 8 * g4) = make_float4(oacc[dt][4 * g4], oacc[dt][4 * g4 + 1], oacc[dt][4 * g4 + 2],
                                                                 oacc[dt][4 * g4 + 3]);
        if (hf == 0) {
            mrg_m[wave * 32 + ln] = M;
            mrg_l[wave * 32 + ln] = L;
        }
    }
    __syncthreads();
    constexpr int TPR = NT / 32;                           // threads per row
    const int row = tid / TPR, io = i0 + row;
    bool nan = false, tiny = false, usual = T::DTYPE != SA2_F32;      // of the results (see below)
    if (io < N) {
        float Mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) Mx = fmaxf(Mx, mrg_m[w * 32 + row]);
        const float Mu = Mx == -INFINITY ? 0.f : Mx;
        float wgt[W], Ls = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            wgt[w] = fast_exp2(mrg_m[w * 32 + row] - Mu);
            Ls += mrg_l[w * 32 + row] * wgt[w];
        }
        const int64_t rows = (int64_t)p.B * p.H * N, prow = share * rows + (int64_t)bh * N + io;
        if (SPLIT && tid % TPR == 0) ((float2*)p.scratch)[prow] = make_float2(Mx, Ls);
        // sum_w + 1e-8 in units of 2^Mu (reference.py:74); for a tiny Mu the epsilon dominates
        const bool big = Mu > LOG2_EPS;
        const float denom = big ? Ls + 1e-8f * fast_exp2(-Mu) : Ls * fast_exp2(Mu - LOG2_EPS) + 1.f;
        const float inv = big ? 1.f / denom : fast_exp2(Mu - LOG2_EPS) / denom;
        EL* orow = (EL*)p.out.p + p.out.off(b, io, h);
#pragma unroll
        for (int col = 4 * (tid % TPR); col < D; col += 4 * TPR) {
            if (PAD && !SPLIT && col >= p.D) continue;
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const float4 y = *(const float4*)(mrg + (w * 32 + row) * C::AS + col);
                acc.x += wgt[w] * y.x; acc.y += wgt[w] * y.y; acc.z += wgt[w] * y.z; acc.w += wgt[w] * y.w;
            }
            const float r[4] = {acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                nan |= r[t] != r[t];
                if (T::DTYPE == SA2_F32) {
                    usual |= fabsf(r[t]) >= TINY;
                    tiny |= r[t] != 0.f && fabsf(r[t]) < TINY;
                }
            }
            if constexpr (SPLIT) *(float4*)((float*)p.scratch + 2 * rows * p.nsplit + prow * D + col) = acc;
            else T::store(orow + col, r[0], r[1], r[2], r[3]);
        }
        if (!SPLIT && tid % TPR == 0)
            p.lse[(int64_t)bh * N + io] = big ? LN2 * Mu + logf(denom) : LN_EPS + logf(denom);
        nan |= Ls != Ls;
    }

    // ---- what the planes do not cover: the block again, by rows, in fp32 FMA arithmetic ----
    // Infinite operands (their lower planes are NaN) and NaN in rows that the windows leave out (a weight of zero times
    // NaN) both show as NaN in the results.  fp32 values under 2^-110 have lost their last plane; a block whose results
    // all lie under TINY may come from such.
    if (!__syncthreads_or(nan || tiny)) return;
    const bool any_nan = __syncthreads_or(nan), any_usual = __syncthreads_or(usual);
    if (!any_nan && any_usual) return;
    {
        // (a row whose q holds a NaN is NaN as it stands: a block of such rows, as a run that has diverged sends them, is done)
        bool q_nan = false;
        for (int col = 4 * (tid % TPR); io < N && col < p.D; col += 4 * TPR) {
            const float4 x = cols4<T, PAD>((const EL*)p.q.p + p.q.off(b, io, h), col, p.D);
            q_nan |= x.x != x.x || x.y != x.y || x.z != x.z || x.w != x.w;
        }
        const uint64_t row_lanes = (((uint64_t)1 << TPR) - 1) << (lane / TPR * TPR);
        const bool row_nan = (__builtin_amdgcn_ballot_w64(q_nan) & row_lanes) != 0;
        if (!__syncthreads_or(io < N && !row_nan)) return;
    }
    const int d_lo = round0 * W, d_hi = round1 * W - 1 < w2 ? round1 * W - 1 : w2;
    for (int r0 = 0; r0 < BQ && i0 + r0 < N; r0 += W)
        fma_fwd_rows<typename T::Fma>(p, bh, i0 + r0, d_lo, d_hi, (float*)smem_f, [&](int ir, int ln_r, float m, float l, const float (&acc)[MAXC]) {
            if constexpr (SPLIT) {
                const int64_t rows = (int64_t)p.B * p.H * N, prow = share * rows + (int64_t)bh * N + ir;
                if (ln_r == 0) ((float2*)p.scratch)[prow] = make_float2(m * LOG2E, l);
#pragma unroll
                for (int c = 0; c < MAXC; ++c)
                    if (ln_r + 64 * c < p.D) ((float*)p.scratch)[2 * rows * p.nsplit + prow * D + ln_r + 64 * c] = acc[c];
            } else {
                fma_store_row<typename T::Fma>(p, bh, ir, ln_r, m, l, acc);
            }
        });
}


// ============================================== backward: which arithmetic =====
// The row term, and whether the planes cover the operands: they do not where one is infinite or NaN, where products of q
// and K' or of dO and V' may overflow, or (bf16) LSE / scale, and (fp32) where all of a tensor's values in a workgroup's rows are so small, and
// not zero, that products of them come under 2^-110.  Each workgroup takes a run of consecutive rows and leaves its
// verdict in guard[blockIdx.x]: 0 covered, 1 not, 2 not but every row has a NaN in q or nothing else in dO, which makes
// everything that such rows reach NaN as it stands.  The two kernels below run whatever it says; where it is 1, or 2 for some
// rows only, split_fma_bwd_kernel computes all gradients again by rows (not where a run that has diverged sends nothing but NaN).  Bound by reading the seven tensors once: fp32 B2 H8 N2048 D64 (59 MB) 16 us, the row term alone
// 9; the launch that looks at the verdicts 5.
constexpr int GUARD_MOST = 1024, GUARD_ROWS = 64;      // workgroups at most, rows per workgroup at least
inline int guard_blocks(int64_t rows) {
    const int64_t n = (rows + GUARD_ROWS - 1) / GUARD_ROWS;
    return (int)(n < GUARD_MOST ? n : GUARD_MOST);
}
size_t guard_bytes(int B, int N, int H) { return ((size_t)guard_blocks((int64_t)B * H * N) * sizeof(int) + 255) / 256 * 256; }
constexpr float GUARD_HIGH = 1.152921504606847e18f;    // 2^60: twice that is an exponent short of fp32's largest
constexpr float GUARD_LOW = 8.881784197001252e-16f;    // 2^-50; dO: 2^-60
constexpr float GUARD_LOW_DO = 8.673617379884035e-19f;
template <class T>
__global__ __launch_bounds__(256) void split_guard_kernel(Problem p, int lpr_log2, int64_t rows, int64_t per_block, int* __restrict__ guard) {
    constexpr int PER = 16 / sizeof(typename T::T), SETS = 7;
    constexpr bool F32 = T::DTYPE == SA2_F32;
    const int lane = threadIdx.x & 63, lpr = 1 << lpr_log2, sub = lane & (lpr - 1);       // lanes per row
    const int step = 4 << (6 - lpr_log2);
    const int64_t first = (int64_t)blockIdx.x * per_block, last = first + per_block < rows ? first + per_block : rows;
    const Tensor* const set[SETS] = {&p.dout, &p.q, &p.k2, &p.v2, &p.k1, &p.v1, &p.out};  // the first four enter products
    bool bad = false, all_nan = true;
    unsigned seen = 0;                       // bit t: tensor t has a usual value here, bit 8 + t: one that is small but not zero
    for (int64_t r0 = first; r0 < last; r0 += step) {
        const int64_t row = r0 + ((int)(threadIdx.x >> 6) << (6 - lpr_log2)) + (lane >> lpr_log2);
        float s = 0.f;
        bool q_nan = false, do_some = false;
        if (row < last && sub * PER < p.D) {
            const int i = (int)(row % p.N), bh = (int)(row / p.N), b = bh / p.H, h = bh - b * p.H;
            union { uint4 v; typename T::Fma e[PER]; } x[SETS];
#pragma unroll
            for (int t = 0; t < SETS; ++t) x[t].v = *(const uint4*)((const typename T::T*)set[t]->p + set[t]->off(b, i, h) + sub * PER);
            float y[PER / 2];
#pragma unroll
            for (int e = 0; e < PER / 2; ++e)
                y[e] = fmaf(to_float(x[6].e[e + PER / 2]), to_float(x[0].e[e + PER / 2]), to_float(x[6].e[e]) * to_float(x[0].e[e]));
#pragma unroll
            for (int half = PER / 4; half > 0; half >>= 1)
#pragma unroll
                for (int e = 0; e < half; ++e) y[e] += y[e + half];
            s = y[0];
#pragma unroll
            for (int t = 0; t < SETS; ++t) {
                float most = 0.f;
#pragma unroll
                for (int e = 0; e < PER; ++e) {
                    const float a = fabsf(to_float(x[t].e[e]));
                    bad |= !(a < INFINITY);
                    if (t == 0) do_some |= a == a;
                    if (t == 1) q_nan |= a != a;
                    most = fmaxf(most, a);
                }
                if (t < 4) bad |= most >= GUARD_HIGH;
                if (F32 && t < 6) {
                    const bool usual = most >= (t == 0 ? GUARD_LOW_DO : GUARD_LOW);
                    seen |= (usual ? 1u : most > 0.f ? 256u : 0u) << t;
                }
            }
            if (sub == 0) {
                const float lse = p.lse[row];
                bad |= !(fabsf(lse) < (T::PLANES == 1 ? GUARD_HIGH : INFINITY));
            }
        }
        for (int off = lpr >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        bad |= s != s;
        if (row < last && sub == 0) p.dsum[row] = s;
        const uint64_t row_lanes = (lpr < 64 ? ((uint64_t)1 << lpr) - 1 : ~(uint64_t)0) << (lane & ~(lpr - 1));
        const bool row_nan = (__builtin_amdgcn_ballot_w64(q_nan) & row_lanes) != 0 || (__builtin_amdgcn_ballot_w64(do_some) & row_lanes) == 0;
        all_nan &= row >= last || row_nan;
    }
    if constexpr (F32) {
        for (int t = 0; t < 6; ++t) {
            const bool usual = __syncthreads_or(seen >> t & 1), small = __syncthreads_or(seen >> (8 + t) & 1);
            bad |= small && !usual;
        }
    }
    const bool verdict = __syncthreads_or(bad), some = __syncthreads_or(!all_nan);
    if (threadIdx.x == 0) guard[blockIdx.x] = first >= last ? 3 : verdict ? (some ? 1 : 2) : 0;      // (3: no rows, no say)
}
__device__ __forceinline__ bool guarded(const int* __restrict__ guard, int n) {
    int seen = 0;
    for (int c = threadIdx.x; c < n; c += blockDim.x) seen |= 1 << guard[c];
    if (!__syncthreads_or(seen & 6)) return false;
    return __syncthreads_or(seen & 3);                       // (verdicts of 2 throughout: nothing to do)
}
// All gradients by rows, where the guard says so (launched last: it overwrites what the sums left)
constexpr int FMA_ROWS = 4, FMA_BLOCKS = 512;
template <class E>
__global__ __launch_bounds__(FMA_ROWS * 64) void split_fma_bwd_kernel(Problem p, const int* __restrict__ guard, int nguard, int nblk, int64_t blocks) {
    extern __shared__ float smem[];
    if (!guarded(guard, nguard)) return;
    const OwnerArgs k = owner_k(p), k2 = owner_k2(p);
    for (int64_t x = blockIdx.x; x < blocks; x += gridDim.x) {
        const int bh = (int)(x / nblk), first = (int)(x - (int64_t)bh * nblk) * FMA_ROWS;
        if (p.dq.p) fma_dq_rows<E>(p, bh, first, smem);
        if (p.dk1.p || p.dv1.p) fma_owner_rows<E>(p, k, bh, first, smem);
        if (p.dk2.p || p.dv2.p) fma_owner_rows<E>(p, k2, bh, first, smem);
    }
}

// ============================================== backward, K' side: dQ, dK', dV' =====
// P between the wavefronts of a pair: 16 values per lane as four 16-byte chunks, chunk-major (no bank conflicts)
__device__ __forceinline__ void px_put(float* px, int lane, const float (&p)[16]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) *(fx4*)(px + c * 256 + lane * 4) = fx4{p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
}
__device__ __forceinline__ void px_get(const float* px, int lane, float (&p)[16]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const fx4 x = *(const fx4*)(px + c * 256 + lane * 4);
        p[4 * c] = x[0]; p[4 * c + 1] = x[1]; p[4 * c + 2] = x[2]; p[4 * c + 3] = x[3];
    }
}
template <int N>
__device__ __forceinline__ void split16(const float (&x)[16], bf16x8 (&o)[2][N]) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        float h[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) h[t] = x[8 * ks + t];
        split8<N>(h, o[ks]);
    }
}

// The K' window in nseg segments of segw deltas, one workgroup per (segment, K' block): segment-major launch order.
// nseg > 1: fp32 partial dK', dV' to `kpart` ([dV' | dK'][nseg][B*H][N][D]).
template <class T, int D, int MODE>
__global__ __launch_bounds__(XT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void split_kp_kernel(Problem p, int nkb, int per_seg, float* __restrict__ dq_part, int nseg, int segw, float* __restrict__ kpart) {
    using C = SplitCfg<T, D>;
    constexpr bool PAD = MODE != EXACT, FINE = MODE == PADDED_FINE;
    typedef typename T::T EL;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_f[];
    uint16_t* tiles = (uint16_t*)smem_f;
    float* px_all = (float*)(smem_f + C::KP_TILES);
    float* dk_s = px_all + NPAIR * 1024;         // [32][AS]: dK' rows k0 .. k0+31 (before the scale)
    float* dv_s = dk_s + 32 * C::AS;             // [32][AS]: dV' rows
    float* dq_s = dv_s + 32 * C::AS;             // [32 + segw - 1][AS]: dQ rows k0 + first delta .. (before the scale)

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int role = wave >> 2, pr = wave & 3;   // role 0: P wavefront, 1: dS wavefront
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    const int seg = (int)blockIdx.x / per_seg;
    const int pid = xcd_order((int)blockIdx.x - seg * per_seg, per_seg);
    const int bh = pid / nkb, kb = pid - bh * nkb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int k0 = kb * BQ, k = k0 + ln, kc = k < N ? k : N - 1;
    const int dlo = seg * segw;                  // first delta of the segment
    const int RQ = 32 + segw - 1;                // rows of the dQ accumulator

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k1p = (const EL*)p.k1.p + p.k1.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v1p = (const EL*)p.v1.p + p.v1.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);
    const EL* dop = (const EL*)p.dout.p + p.dout.off(b, 0, h);
    const bool want_dq = p.dq.p != nullptr;

    const int nu_all = (w2 < N - 1 - k0 ? w2 : N - 1 - k0) + 1;        // deltas with k0 + delta < N
    const int n_units = nu_all - dlo < segw ? nu_all - dlo : segw;     // of this segment (may be <= 0)
    const int nrounds = (n_units + NPAIR - 1) / NPAIR;
    const float qscale = p.scale * LOG2E;
    const uint32_t tiles_addr = lds_address(tiles);
    const uint32_t row_lane = (uint32_t)(ln * C::RSB + hf * 16), col_lane = column_lane<C::RSB>(lane);
    float* px = px_all + pr * 1024;

    for (int c = tid; c < (RQ + 64) * C::AS; c += XT) dk_s[c] = 0.f;       // all three accumulators

    TileRegs<T, D, XT> next;                     // the tile on its way from global memory to LDS
    auto rounds = [&](auto ROLE_TAG) {
        constexpr int ROLE = decltype(ROLE_TAG)::value;
        const int d_end = dlo + n_units - 1;
        auto first_tile = [&](int round) {                    // of the round's smallest delta
            const int i_min = k0 + dlo + round * NPAIR;
            return (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
        };
        auto request = [&](int jt) { next.template load<PAD>(k1p, p.k1.sn, v1p, p.v1.sn, jt * TJ, N, tid, p.D); };
        if (nrounds > 0) request(first_tile(0));
        for (int round = 0; round < nrounds; ++round) {
            // tiles of the round's units (within the sequence)
            const int d_first = dlo + round * NPAIR;
            const int d_last = d_first + NPAIR - 1 < d_end ? d_first + NPAIR - 1 : d_end;
            const int i_max = k0 + 31 + d_last < N - 1 ? k0 + 31 + d_last : N - 1;
            const int jt_lo = first_tile(round), jt_hi = i_max / TJ;
            const int nt = jt_hi - jt_lo + 1;

            const int delta = d_first + pr;
            const bool ok = delta <= d_end;
            const int i = k + delta, ic = i < N ? i : N - 1;
            const bool row_ok = ok && i < N;                  // (k <= i < N)
            const int iw_lo = k0 + delta, iw_hi = k0 + 31 + delta < N - 1 ? k0 + 31 + delta : N - 1;   // this unit's queries
            const bool rows_full = k0 + 31 + delta < N;

            bf16x8 xf[C::DK][3];                              // Q~ (P wavefront) or dO~ (dS wavefront)
            float lead = 0.f;                                 // LSE or D, to be taken off the first chain
            if (ok) {
#pragma unroll
                for (int kk = 0; kk < C::DK; ++kk) {
                    const int col = kk * 16 + hf * 8;
                    if constexpr (ROLE == 0)
                        product_planes<T, PAD>(qp + (int64_t)ic * p.q.sn, k2p + (int64_t)kc * p.k2.sn, col, p.D, p.k2_bias, qscale, xf[kk]);
                    else
                        product_planes<T, PAD>(dop + (int64_t)ic * p.dout.sn, v2p + (int64_t)kc * p.v2.sn, col, p.D, p.v2_bias, 1.f, xf[kk]);
                }
                lead = (ROLE == 0 ? p.lse : p.dsum)[(int64_t)bh * N + ic];
            }
            floatx16 acc[C::DT];                              // R or G
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt) acc[dt] = zero16();

            // (the previous round's last barrier has passed: the stages are free)
            auto put_next = [&](int s) {                      // tile s + 1 to its stage, tile s + 2 requested
                if (s + 1 < nt) next.store(tiles + (C::KP_STAGES == 2 ? (s + 1) & 1 : 0) * C::KV_STAGE, tid);
                if (s + 2 < nt) request(jt_lo + s + 2);
            };
            next.store(tiles, tid);
            if (nt > 1) request(jt_lo + 1);
            __syncthreads();
            for (int s = 0; s < nt; ++s) {
                const int j0 = (jt_lo + s) * TJ;
                // tiles that hold no key of this unit's windows are skipped by the pair
                const bool in = ok && j0 <= iw_hi && j0 + TJ - 1 >= iw_lo - w1;
                const uint32_t Ks = tiles_addr + (uint32_t)((C::KP_STAGES == 2 ? s & 1 : 0) * C::KV_STAGE * 2);
                const uint32_t Vs = Ks + (uint32_t)(C::KV_TILE * 2);
                bf16x8 pb[2][3];
                floatx16 first;                               // logits less LSE, or dP less D
                if (ROLE == 1 && C::KP_STAGES == 2) put_next(s);
                if (in) {
                    Chain<FINE> chain;
                    chain.clear();
                    if (ROLE == 0) __builtin_amdgcn_s_setprio(1);
#pragma unroll
                    for (int kk = 0; kk < C::DK; ++kk) {
                        bf16x8 a[C::NK];
                        row_operand<C::NK, C::RSB>((ROLE == 0 ? Ks : Vs) + row_lane, kk, a);
                        chain.add(a, xf[kk]);
                    }
                    float x = lead;
                    asm volatile("" : "+v"(x));               // (planes made where they are used: one register to keep)
                    first = ElemBF16::mfma(lead_ones(hf), ROLE == 0 ? lse_planes(x) : lead_planes(x, 0.f), chain.sum(), 0, 0, 0);
                    if (ROLE == 0) {
                        __builtin_amdgcn_s_setprio(0);
                        float pv[16];
#pragma unroll
                        for (int v = 0; v < 16; ++v) pv[v] = fast_exp2(first[v]);
                        if (!(rows_full && (j0 + TJ - 1 <= iw_lo) && (j0 >= iw_lo + 31 - w1))) {
                            const int hi = i - j0 - 4 * hf, lo = hi - w1;
#pragma unroll
                            for (int v = 0; v < 16; ++v) {
                                const int c = 8 * (v >> 2) + (v & 3);
                                pv[v] = row_ok && c <= hi && c >= lo ? pv[v] : 0.f;
                            }
                        }
                        px_put(px, lane, pv);
                        split16<3>(pv, pb);
                    }
                }
                __syncthreads();
                if (in) {
                    if (ROLE == 1) {
                        float pv[16];
                        px_get(px, lane, pv);
#pragma unroll
                        for (int v = 0; v < 16; ++v) pv[v] *= first[v];
                        split16<3>(pv, pb);
                    }
                    accumulate<FINE, C::NK>(acc, pb, [&](int ks, int dt, bf16x8 (&a)[C::NK]) {
                        column_operand<C::NK, C::RSB>((ROLE == 0 ? Vs : Ks) + col_lane, ks, dt, a);
                    });
                }
                if (C::KP_STAGES == 1) __syncthreads();       // everyone is done with the only stage
                if (ROLE == 0 || C::KP_STAGES == 1) put_next(s);
                __syncthreads();
            }

            // ---- the unit's reductions into the workgroup's LDS accumulators: dV'[k] += R*dO[i] (P wavefronts),
            //      dK'[k] += G*q[i] (rows ln) and dQ[i] += G*k2~[k] (rows ln + delta; dS wavefronts).  Four phases; in phase
            //      ph pair pr owns column group (pr + ph) % 4 of every row, so no two wavefronts touch an element at
            //      once and every element sums in a fixed order.  The rows are read once, before the phases. ----
            typename T::Raw x[4 * C::DT], y[ROLE == 1 ? 4 * C::DT : 1];
            {
                const EL* xrow = ROLE == 0 ? dop + (int64_t)ic * p.dout.sn : qp + (int64_t)ic * p.q.sn;
                const EL* krow = k2p + (int64_t)kc * p.k2.sn;
#pragma unroll
                for (int e = 0; e < 4 * C::DT; ++e) {
                    const int col = (e >> 2) * 32 + 8 * (e & 3) + 4 * hf;
                    x[e] = raw4<T, PAD>(xrow, col, p.D);
                    if (ROLE == 1) y[ROLE == 1 ? e : 0] = raw4<T, PAD>(krow, col, p.D);
                }
            }
            if (round + 1 < nrounds) request(first_tile(round + 1));
            auto reduce = [&](auto PR_TAG) {
                constexpr int PR = decltype(PR_TAG)::value;
                float* arow = (ROLE == 0 ? dv_s : dk_s) + ln * C::AS + 4 * hf;
                float* dqrow = dq_s + (ln + delta - dlo) * C::AS + 4 * hf;
#pragma unroll
                for (int ph = 0; ph < 4; ++ph) {
                    constexpr int G4S[4] = {PR, (PR + 1) & 3, (PR + 2) & 3, (PR + 3) & 3};
                    const int g4 = G4S[ph];
                    if (row_ok) {
#pragma unroll
                        for (int dt = 0; dt < C::DT; ++dt) {
                            const int col = dt * 32 + 8 * g4;
                            const fx4 xv = T::widen(x[4 * dt + g4]);
                            fx4 a = *(fx4*)(arow + col);
#pragma unroll
                            for (int t = 0; t < 4; ++t) a[t] += acc[dt][4 * g4 + t] * xv[t];
                            *(fx4*)(arow + col) = a;
                            if (ROLE == 1 && want_dq) {
                                const fx4 yv = T::widen(y[ROLE == 1 ? 4 * dt + g4 : 0]);
                                fx4 o = *(fx4*)(dqrow + col);
#pragma unroll
                                for (int t = 0; t < 4; ++t) o[t] += acc[dt][4 * g4 + t] * (yv[t] + p.k2_bias);
                                *(fx4*)(dqrow + col) = o;
                            }
                        }
                    }
                    __syncthreads();
                }
            };
            switch (pr) {
                case 0: reduce(std::integral_constant<int, 0>{}); break;
                case 1: reduce(std::integral_constant<int, 1>{}); break;
                case 2: reduce(std::integral_constant<int, 2>{}); break;
                default: reduce(std::integral_constant<int, 3>{}); break;
            }
        }
    };
    if (role == 0) rounds(std::integral_constant<int, 0>{});
    else rounds(std::integral_constant<int, 1>{});
    __syncthreads();

    // ---- dK' and dV' rows of the block ----
    for (int c = tid; c < 2 * 32 * (D / 4); c += XT) {
        const int which = c / (32 * (D / 4)), rem = c - which * 32 * (D / 4);     // 0: dV', 1: dK'
        const int row = rem / (D / 4), col = (rem - row * (D / 4)) * 4, ko = k0 + row;
        const Tensor& t = which ? p.dk2 : p.dv2;
        if (ko >= N || !t.p) continue;
        const float sc = which ? p.scale : 1.f;
        const fx4 a = *(const fx4*)((which ? dk_s : dv_s) + row * C::AS + col) * sc;
        if (nseg > 1) *(fx4*)(kpart + ((((int64_t)which * nseg + seg) * p.B * p.H + bh) * N + ko) * D + col) = a;
        else if (!PAD || col < p.D) T::store((EL*)t.p + t.off(b, ko, h) + col, a[0], a[1], a[2], a[3]);
    }
    // ---- dQ partial: rows k0 + dlo .. (rows of deltas beyond the end of the sequence hold zeros) ----
    if (want_dq) {
        float* part = dq_part + (((int64_t)bh * nkb + kb) * nseg + seg) * (int64_t)RQ * D;
        for (int c = tid; c < RQ * (D / 4); c += XT) {
            const int r = c / (D / 4), col = (c - r * (D / 4)) * 4;
            *(fx4*)(part + (int64_t)r * D + col) = *(const fx4*)(dq_s + r * C::AS + col) * p.scale;
        }
    }
}

// =================================================== backward, K side: dK, dV =====
// nsplit > 1 (grids smaller than the chip): the workgroup takes the sp-th share of the key block's stream
// of units and writes fp32 partial sums to `part` ([dK | dV][nsplit][B*H][N][D]) for bwd_sum_kernel.
template <class T, int D, bool SPLIT, int MODE>
__global__ __launch_bounds__(XT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void split_kv_kernel(Problem p, int njb, int total, int nsplit_arg, float* __restrict__ part) {
    const int nsplit = SPLIT ? nsplit_arg : 1;
    using C = SplitCfg<T, D>;
    constexpr bool PAD = MODE != EXACT, FINE = MODE == PADDED_FINE;
    typedef typename T::T EL;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_f[];
    uint16_t* tiles = (uint16_t*)smem_f;
    float* px_all = (float*)(tiles + 2 * C::UNIT_STAGE);
    unsigned char* lead_s = (unsigned char*)(px_all + NPAIR * 1024);     // [2][LSE, D][32 queries] lead_planes

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int role = wave >> 2, pr = wave & 3;   // role 0: P wavefront (K rows, dV), 1: dS wavefront (V rows, dK)
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    const int pid = xcd_order(blockIdx.x, total);
    const int sp = pid % nsplit, pj = pid / nsplit;
    const int bh = pj / njb, jb = pj - bh * njb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int j0 = jb * XJ, jw = j0 + 32 * pr, j = jw + ln, jc = j < N ? j : N - 1;

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k1p = (const EL*)p.k1.p + p.k1.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v1p = (const EL*)p.v1.p + p.v1.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);
    const EL* dop = (const EL*)p.dout.p + p.dout.off(b, 0, h);
    const float qscale = p.scale * LOG2E;

    const uint32_t tiles_addr = lds_address(tiles);
    const uint32_t row_lane = (uint32_t)(ln * C::RSB + hf * 16), col_lane = column_lane<C::RSB>(lane);

    float* px = px_all + pr * 1024;

    // the pair's K rows (P wavefront) or V rows (dS wavefront) as resident B operands (column = key j)
    bf16x8 kf[C::DK][C::NK];
    {
        const EL* row = role ? v1p + (int64_t)jc * p.v1.sn : k1p + (int64_t)jc * p.k1.sn;
#pragma unroll
        for (int kk = 0; kk < C::DK; ++kk) {
            const int col = kk * 16 + hf * 8;
            const float4 x0 = cols4<T, PAD>(row, col, p.D), x1 = cols4<T, PAD>(row, col + 4, p.D);
            const float r[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            split8<C::NK, C::LIMIT>(r, kf[kk]);
        }
    }
    floatx16 acc[C::DT];                         // dV^T or dK^T
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) acc[dt] = zero16();

    const int j_last = j0 + XJ - 1 < N ? j0 + XJ - 1 : N - 1;
    const int i_max = (int)((int64_t)j_last + w1 < N - 1 ? j_last + w1 : N - 1);
    auto units_of = [&](int ib) {
        const int il = ib * BQ + BQ - 1 < N ? ib * BQ + BQ - 1 : N - 1;
        return (w2 < il ? w2 : il) + 1;
    };
    // The units (query block, delta) that see the key block, in stream order, and this workgroup's share of
    // them: from delta d_first of block ib_lo to delta d_last of block ib_hi.  The shares cut the stream
    // counted with w2 + 1 slots per block (a block near the start of the sequence has fewer units: the slots
    // beyond are skipped).
    int ib_lo = j0 / BQ, ib_hi = i_max / BQ, d_first = 0, d_last = w2;
    bool empty_share = ib_lo > ib_hi;
    if constexpr (SPLIT) {
        const int per = w2 + 1, ib0 = ib_lo;
        const int slots = (ib_hi - ib_lo + 1) * per;
        const int chunk = (slots + nsplit - 1) / nsplit;
        const int v_lo = sp * chunk, v_hi = (v_lo + chunk < slots ? v_lo + chunk : slots) - 1;
        empty_share = v_lo > v_hi;
        if (!empty_share) {
            ib_lo = ib0 + v_lo / per;
            d_first = v_lo - (ib_lo - ib0) * per;
            ib_hi = ib0 + v_hi / per;
            d_last = v_hi - (ib_hi - ib0) * per;
            if (d_first >= units_of(ib_lo)) {        // the share starts in the slots a short block does not have
                ++ib_lo;
                d_first = 0;
            }
            empty_share = !(ib_lo < ib_hi || (ib_lo == ib_hi && d_first <= d_last));
        }
    }
    // (a share of a split launch may be empty: it walks one unit without touching it and writes zeros)
    if (empty_share) {
        ib_lo = ib_hi = j0 / BQ;
        d_first = d_last = 0;
    }

    // ---- forming a unit: Q~ and dO~ tiles (32 rows), LSE and D of its queries ----
    constexpr int ALL = 32 * D / 4, KR = (ALL + XT - 1) / XT;      // groups of four columns: of a tile, per thread
    typename T::Raw fq[KR], fk[KR], fd[KR], fv[KR];
    float f_lead = 0.f;                       // LSE (threads 0-31) or D (32-63) of a query
    // (LSE and D of a unit by the two halves of wavefront 0: by one half, one after the other, the kernel took 4 % longer at
    // 128 columns, where that wavefront is on the step's critical path)
    auto fetch_unit = [&](int ib, int delta) {
#pragma unroll
        for (int u = 0; u < KR; ++u) {
            const int c = tid + XT * u;
            if (ALL % XT != 0 && c >= ALL) break;
            const int row = c / (D / 4), col = c - row * (D / 4);
            int i = ib * BQ + row;
            i = i < N ? i : N - 1;
            const int k = i - delta > 0 ? i - delta : 0;
            fq[u] = raw4<T, PAD>(qp + (int64_t)i * p.q.sn, col * 4, p.D);
            fk[u] = raw4<T, PAD>(k2p + (int64_t)k * p.k2.sn, col * 4, p.D);
            fd[u] = raw4<T, PAD>(dop + (int64_t)i * p.dout.sn, col * 4, p.D);
            fv[u] = raw4<T, PAD>(v2p + (int64_t)k * p.v2.sn, col * 4, p.D);
        }
        if (tid < 64) {
            int i = ib * BQ + ln;
            i = i < N ? i : N - 1;
            f_lead = (hf ? p.dsum : p.lse)[(int64_t)bh * N + i];
        }
    };
    auto store_unit = [&](int buf) {
        uint16_t* Qs = tiles + buf * C::UNIT_STAGE;
        uint16_t* Ds = Qs + C::UNIT_TILE;
#pragma unroll
        for (int u = 0; u < KR; ++u) {
            const int c = tid + XT * u;
            if (ALL % XT != 0 && c >= ALL) break;
            const int row = c / (D / 4), col = c - row * (D / 4);
            const float kb = p.k2_bias, vb = p.v2_bias;
            const fx4 q4 = T::widen(fq[u]), k4 = T::widen(fk[u]), d4 = T::widen(fd[u]), v4 = T::widen(fv[u]);
            const fx4 qt = {q4[0] * qscale * (k4[0] + kb), q4[1] * qscale * (k4[1] + kb), q4[2] * qscale * (k4[2] + kb), q4[3] * qscale * (k4[3] + kb)};
            const fx4 dt = {d4[0] * (v4[0] + vb), d4[1] * (v4[1] + vb), d4[2] * (v4[2] + vb), d4[3] * (v4[3] + vb)};
            store_planes<3, false>(qt, Qs + row * C::RS + col * 4, C::PLANE);
            store_planes<3, false>(dt, Ds + row * C::RS + col * 4, C::PLANE);
        }
        if (tid < 64) {
            const float x = hf ? f_lead : f_lead * LOG2E;
            *(bf16x8*)(lead_s + (buf * 64 + tid) * 16) = lead_planes(x, hf ? 0.f : lse_rest(f_lead, x));
        }
    };

    fetch_unit(ib_lo, d_first);
    store_unit(0);
    __syncthreads();
    auto stream = [&](auto ROLE_TAG) {
        constexpr int ROLE = decltype(ROLE_TAG)::value;
        int ib = ib_lo, delta = d_first, nu = units_of(ib_lo), buf = 0;
        while (true) {
            int nib = ib, ndelta = delta + 1;
            if (ndelta >= nu) {
                nib = ib + 1;
                ndelta = 0;
            }
            const bool more = SPLIT ? (nib < ib_hi || (nib == ib_hi && ndelta <= d_last)) : nib <= ib_hi;
            if (more) fetch_unit(nib, ndelta);

            const int i0 = ib * BQ;
            const bool touches = (i0 + BQ - 1 >= jw) && ((int64_t)i0 <= (int64_t)jw + 31 + w1) && jw < N && !empty_share;
            const uint32_t Qs = tiles_addr + (uint32_t)(buf * C::UNIT_STAGE * 2);
            const uint32_t Ds = Qs + (uint32_t)(C::UNIT_TILE * 2);
            bf16x8 pb[2][3];
            floatx16 first;                   // logits less LSE, or dP less D: register v is query i0 + 8*(v/4) + 4*hf + v%4
            if (touches) {
                Chain<FINE> chain;
                chain.clear();
                if (ROLE == 0) __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int kk = 0; kk < C::DK; ++kk) {
                    bf16x8 a[3];
                    row_operand<3, C::RSB>((ROLE == 0 ? Qs : Ds) + row_lane, kk, a);
                    chain.add(a, kf[kk]);
                }
                const bf16x8 lead = *(const bf16x8*)(lead_s + (buf * 64 + ROLE * 32 + ln) * 16);
                first = ElemBF16::mfma(lead, lead_ones(hf), chain.sum(), 0, 0, 0);
                if (ROLE == 0) {
                    __builtin_amdgcn_s_setprio(0);
                    float pv[16];
#pragma unroll
                    for (int v = 0; v < 16; ++v) pv[v] = fast_exp2(first[v]);
                    if (!((i0 >= jw + 31) && ((int64_t)i0 + 31 <= (int64_t)jw + w1) && (i0 + BQ - 1 < N) && (i0 >= delta))) {
                        const int lo = j - i0 - 4 * hf;                                    // c >= lo  <=>  j <= i
                        const int hi = (int)((int64_t)j + w1 - i0 < (1 << 20) ? j + w1 - i0 : (1 << 20)) - 4 * hf;   // i <= j + w1
                        const int dlo = delta - i0 - 4 * hf, nhi = N - 1 - i0 - 4 * hf;
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int c = 8 * (v >> 2) + (v & 3);
                            pv[v] = (j < N) && (c >= lo) && (c <= hi) && (c >= dlo) && (c <= nhi) ? pv[v] : 0.f;
                        }
                    }
                    px_put(px, lane, pv);
                    split16<3>(pv, pb);
                }
            }
            __syncthreads();
            if (touches) {
                if (ROLE == 1) {
                    float pv[16];
                    px_get(px, lane, pv);
#pragma unroll
                    for (int v = 0; v < 16; ++v) pv[v] *= first[v];
                    split16<3>(pv, pb);
                }
                accumulate<FINE, 3>(acc, pb, [&](int ks, int dt, bf16x8 (&a)[3]) {
                    column_operand<3, C::RSB>((ROLE == 0 ? Ds : Qs) + col_lane, ks, dt, a);
                });
            }
            if (!more) break;
            store_unit(buf ^ 1);          // (the other buffer was last read one step ago, before that step's barrier)
            __syncthreads();
            if (nib != ib) nu = units_of(nib);
            ib = nib;
            delta = ndelta;
            buf ^= 1;
        }
    };
    if (role == 0) stream(std::integral_constant<int, 0>{});
    else stream(std::integral_constant<int, 1>{});

    if (j < N) {
        // Q~ carries scale*log2(e): dK = ln2 * sum dS * Q~
        const int which = role ? 0 : 1;
        const Tensor& t = which ? p.dv1 : p.dk1;
        if (t.p) {
            const float sc = which ? 1.f : LN2;
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int col = dt * 32 + 8 * g4 + 4 * hf;
                    const float x0 = acc[dt][4 * g4] * sc, x1 = acc[dt][4 * g4 + 1] * sc, x2 = acc[dt][4 * g4 + 2] * sc, x3 = acc[dt][4 * g4 + 3] * sc;
                    if constexpr (SPLIT)
                        *(float4*)(part + (((which * (int64_t)nsplit + sp) * p.B * p.H + bh) * N + j) * D + col) = make_float4(x0, x1, x2, x3);
                    else if (!PAD || col < p.D)
                        T::store((EL*)t.p + t.off(b, j, h) + col, x0, x1, x2, x3);
                }
        }
    }
}

// Shares a key block's query blocks are split into when the K-side grid is smaller than the chip: doubled until the grid
// holds two waves.  Against every number of shares (profiles/plan_cuts.md): within 11 % of the best at seven of ten sizes,
// 22 - 37 % off at small ones whose best is no power of two (bf16 B2 H3 N777 D40 w 100/20: 140 us in eight, 102 in six).
int split_kv_nsplit(int B, int N, int H, int D, int w1, int w2, size_t room) {
    const int64_t bh = (int64_t)B * H, base = bh * ((N + XJ - 1) / XJ);
    const int blocks = (XJ + (w1 < N ? w1 : N) + BQ - 1) / BQ + 1;
    const int64_t units = (int64_t)blocks * ((w2 < N - 1 ? w2 : N - 1) + 1);     // of a key block's stream, at most
    int ns = 1;                                                                  // shares of at least 8 units
    while (ns < 16 && base * ns * 2 <= 512 && (int64_t)ns * 2 * 8 <= units && (int64_t)2 * ns * 2 * bh * N * D * 4 <= ((int64_t)32 << 20) &&
           (size_t)2 * ns * 2 * bh * N * D * 4 <= room)
        ns *= 2;
    return ns;
}
size_t split_kv_bytes(int B, int N, int H, int D, int nsplit) { return nsplit > 1 ? (size_t)2 * nsplit * B * H * (size_t)N * D * sizeof(float) : 0; }
size_t split_dq_part_bytes(int B, int N, int H, int D, const KpPlan& pl) {
    return ((size_t)B * H * ((N + BQ - 1) / BQ) * pl.nseg * (size_t)(31 + pl.segw) * D * sizeof(float) + 255) / 256 * 256;
}
size_t split_kp_bytes(int B, int N, int H, int D, const KpPlan& pl) {
    return split_dq_part_bytes(B, N, H, D, pl) + (pl.nseg > 1 ? (size_t)2 * pl.nseg * B * H * (size_t)N * D * sizeof(float) : 0);
}
// Whether products of a unit have 16 bits, so that two planes hold them and the scale may wait until they are summed (a scale with which such
// products and sums stay as far from the ends of fp32 as scaled ones; the backward's LSE / scale: see split_guard_kernel)
template <class T>
bool exact_products(const Problem& p, bool backward) {
    return T::DTYPE == SA2_BF16 && p.k2_bias == 0.f && (!backward || p.v2_bias == 0.f) && p.scale >= 8.6736174e-19f && p.scale <= 1024.f;     // 2^-60 .. 2^10
}
// Whether the kernels with one wavefront per SIMD are taken (sa2_split_fwd_lone.h, sa2_split_kv_lone.h, sa2_split_kp_lone.h)
template <class T, int D, int MODE>
constexpr bool lone() { return T::DTYPE == SA2_F32 ? MODE != PADDED_FINE && D <= 64 : D == 64 || D == 96; }
// Units of a forward's round.  At 96 columns grids that are at once on the chip in rounds of four are shared so, by split_fwd_kernel: a round
// is all of such a launch, and two units per wavefront take it longer.  Rounds of eight against rounds of four, us: fp16 D80 B2 H8 N33 w 65/15
// 20.5 / 16.6, B1 H4 N128 w 16/16 20.9 / 19.7, B1 H2 N300 w 200/12 33.2 / 31.1, w 40/24 23.5 / 22.9, B1 H4 N46 w 45/46 22.7 / 20.2, H1 N95 w 29/30 22.1 /
// 20.6, B1 H2 N128 w 128/100 30.0 / 38.7.  Where logits have two planes (bf16) only for the shortest sequences: N33 16.9 / 15.0, B1 H1 N64 w 16/8
// 16.1 / 14.4, B1 H1 N35 w 34/19 17.5 / 16.1, but B1 H4 N512 w 40/15 19.5 / 20.4.
template <class T, int D, int MODE>
int forward_round(int B, int N, int H, int w2) {
    if constexpr (lone<T, D, MODE>() && D == 96) {
        const int units = (w2 < N - 1 ? w2 : N - 1) + 1;
        const bool few = T::PLANES == 1 ? units <= 24 && N <= 64 : units <= 20 || N <= 96;
        return few && units > 8 && (int64_t)B * H * ((N + BQ - 1) / BQ) * ((units + 3) / 4) <= CUS ? 4 : 8;
    }
    return SplitCfg<T, D>::FW;
}
// ... by the forward: at 32 columns not.  (Two units of a wavefront share an accumulator, whose longer chain of sums shows there: 1 - 4 % more error
// in an fp32 output at head_dim 32 - 0.99 to 1.0 at 64 - for 5 - 10 % less time at most sizes, and 5 - 19 % more with few deltas or at head_dim 16.)
// Nor where two units of a wavefront have little to lie beside: few deltas in short sweeps, and sequences of up to three tiles whose rounds are all at
// once on the chip.  Two units per wavefront against one, us:
//   fp32 D64: B1 H2 N119 w 23/1 12.9 / 10.0, H1 N826 w 31/2 13.0 / 10.7, B1 H64 N1173 w 17/2 90 / 75, B1 H8 N2054 w 761/2 119 / 109, H2 N756 w 86/4 18.4 /
//     17.7, H46 N131 w 90/4 19.7 / 18.7, but H7 N388 w 405/4 33.9 / 37.7 and six deltas N1052 w 49 44.4 / 46.2, N388 w 387 34.3 / 38.1
//   fp16 D48: N119 w 23/1 12.8 / 9.9, N1173 w 17/2 88.6 / 72.9, N274 w 27/5 13.8 / 11.5, N378 w 64/6 33.6 / 28.3, N1698 w 28/7 87 / 78, but w 387/5 31.6 / 35.6,
//     N4221 w 766/2 126 / 129      D80: N119 w 23/1 15.5 / 12.8, N709 w 12/3 18.5 / 14.5, but N467 w 192/1 24.2 / 25.2, N5041 w 256/3 80 / 87
//   bf16 D40: N119 w 23/1 10.8 / 9.2, N1173 w 17/2 72 / 66, w 86/4 16.7 / 14.6, N274 w 27/5 11.8 / 10.6, but N467 w 192/1 15.7 / 16.6, N1052 w 49/5 35.1 / 35.4
//     D96: N45 w 16/1 12.8 / 11.7, w 78/1 14.1 / 13.6, but N826 w 31/2 12.8 / 13.6
//   N33 - 96, D64 fp32: B1 H25 N33 w 32/13 20.8 / 17.6, H8 N67 w 52/9 23.5 / 20.0, H2 N76 w 76/37 20.9 / 19.3, H1 N46 w 45/46 19.4 / 17.8, but (not at once) H53 N67
//     w 23/23 29.0 / 35.9
template <class T, int D, int MODE>
bool lone_forward(int B, int N, int H, int w1, int w2, int nsplit) {
    if constexpr (!lone<T, D, MODE>() || D == 32) return false;
    const int units = (w2 < N - 1 ? w2 : N - 1) + 1, keys = w1 < N ? w1 : N;
    if constexpr (D == 96) {
        if (nsplit > 1) return forward_round<T, D, MODE>(B, N, H, w2) == 8;
        return T::PLANES == 1 ? units > 2 || keys > 96 : units > 4 || keys > 192;
    }
    if (N <= 96 && (int64_t)B * H * ((N + BQ - 1) / BQ) * ((units + 7) / 8) <= CUS) return false;
    if (T::DTYPE == SA2_F32) return units > (keys <= 128 ? 5 : 4);
    if (T::DTYPE == SA2_F16) return units > 8 || keys > (units <= 4 ? 320 : 192);
    return units > 8 || keys > (units <= 2 ? 128 : units <= 5 ? 96 : 32);
}
// Deltas per segment: what the dQ accumulator in LDS holds, or fewer where the grid asks for it
template <class T, int D, int MODE>
KpPlan split_kp_plan(int B, int N, int H, int w1, int w2, size_t room) {
    using C = SplitCfg<T, D>;
    int most = NPAIR;
    auto fits = [](int segw) {
        if constexpr (lone<T, D, MODE>()) return SplitKpLoneCfg<D, T::PLANES>::fits(segw);
        else return C::kp_fits(segw - 1);
    };
    while (most < w2 + 1 && fits(most + NPAIR)) most += NPAIR;
    return plan_segments(B, N, H, w1, w2, NPAIR, most, room, [](int) { return false; }, [&](const KpPlan& pl) { return split_kp_bytes(B, N, H, D, pl); });
}

// Whether the K' side takes its kernel with one wavefront per SIMD: not where all rounds of four deltas are at once on the chip, so that each is
// all of a workgroup, and the sweeps are short.  One wavefront per SIMD against pairs there, K' side with guard and sums, us: fp32 D16 B1 H1 N58 w 35/12 23.7 /
// 21.6, H2 N225 w 89/10 28.0 / 27.2, H1 N1314 w 17/10 26.0 / 24.3, D32 H2 N119 w 23/1 24.4 / 23.2, fp16 D48 H2 N119 w 23/1 26.4 / 24.7, N1314 w 17/10 29.8 /
// 27.8, D80 34.9 / 31.9 (N58), 42.0 / 39.9 (N225), bf16 D40 24.8 / 22.9 and 28.7 / 28.0; wide windows: fp32 D16 H1 N599 w 465/1 1.05, D32 1.07, bf16 D40 1.06 the
// other way, fp16 0.98.  fp32 D64 and bf16 at 96 columns are faster with one everywhere (1.04 and 1.13 at the median of such grids).
template <class T, int D, int MODE>
bool lone_kp(int B, int N, int H, int w1, int w2, const KpPlan& pl) {
    if constexpr (!lone<T, D, MODE>()) return false;
    if constexpr (T::DTYPE == SA2_F32 ? D == 64 : T::PLANES == 1 && D == 96) return true;
    const int units = (w2 < N - 1 ? w2 : N - 1) + 1, keys = w1 < N ? w1 : N;
    const int64_t rounds = (int64_t)B * H * ((N + BQ - 1) / BQ) * ((units + NPAIR - 1) / NPAIR);
    return rounds > CUS || keys > (T::DTYPE == SA2_F16 ? 256 : 128) || !SplitCfg<T, D>::kp_fits(pl.segw - 1);
}
// ... and the K side: in fp16 not for few deltas of sequences that leave its blocks of 128 keys half empty.  us, one wavefront per SIMD against pairs: D48
// B1 H1 N58 w 35/12 27.3 / 26.5, H17 N79 w 125/1 26.8 / 24.5, D80 35.8 / 33.9 and 35.2 / 31.9, but H2 N76 w 76/37 36.2 / 39.2, H50 N74 w 73/55 117 / 145.
template <class T, int D, int MODE>
bool lone_kv(int N, int w2) { return lone<T, D, MODE>() && (T::DTYPE != SA2_F16 || N > 80 || w2 >= 20); }

// ------------------------------------------------------------------ launchers ----
template <class T, int D, int MODE>
int launch_split_fwd(const Problem& p, hipStream_t st) {
    if (lone_forward<T, D, MODE>(p.B, p.N, p.H, p.w1, p.w2, p.nsplit)) {
        const int rc = (T::DTYPE == SA2_F32 ? launch_split_fwd_lone_fp32 : T::DTYPE == SA2_F16 ? launch_split_fwd_lone_fp16 : launch_split_fwd_lone_bf16)(
            p, D, exact_products<T>(p, false), st);
        return rc != SA2_OK || p.nsplit <= 1 ? rc : launch_fwd_merge(p, D, T::DTYPE, st);
    }
    using C = SplitCfg<T, D>;
    const int nqb = (p.N + BQ - 1) / BQ;
    const int64_t total = (int64_t)nqb * p.B * p.H, grid = total * (p.nsplit > 1 ? p.nsplit : 1);
    if (grid > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return false;
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(C::FW * 64), C::FWD_LDS, st, p, nqb, (int)grid);
        return hipGetLastError() == hipSuccess;
    };
    auto go_split = [&](auto nq) {
        constexpr int NQ = decltype(nq)::value;
        return p.nsplit > 1 ? go(split_fwd_kernel<T, D, MODE, true, NQ>) : go(split_fwd_kernel<T, D, MODE, false, NQ>);
    };
    bool ok;
    if constexpr (T::PLANES == 1) ok = exact_products<T>(p, false) ? go_split(std::integral_constant<int, 2>{}) : go_split(std::integral_constant<int, 3>{});
    else ok = go_split(std::integral_constant<int, 3>{});
    if (!ok) return SA2_ERR_LAUNCH_FAILED;
    return p.nsplit > 1 ? launch_fwd_merge(p, D, T::DTYPE, st) : SA2_OK;
}

template <class T, int D, int MODE>
int launch_split_bwd(const Problem& p, hipStream_t st) {
    using C = SplitCfg<T, D>;
    BwdSums sums = {};
    const size_t room = room_left(p.room, guard_bytes(p.B, p.N, p.H));
    const KpPlan pl = split_kp_plan<T, D, MODE>(p.B, p.N, p.H, p.w1, p.w2, room);
    const size_t kp_bytes = (split_kp_bytes(p.B, p.N, p.H, D, pl) + 255) / 256 * 256;
    const int nsplit = split_kv_nsplit(p.B, p.N, p.H, D, p.w1, p.w2, room_left(room, kp_bytes));
    const size_t part_bytes = kp_bytes + split_kv_bytes(p.B, p.N, p.H, D, nsplit);
    if (p.scratch_bytes < part_bytes + guard_bytes(p.B, p.N, p.H)) return SA2_ERR_WORKSPACE_TOO_SMALL;
    int* guard = (int*)((char*)p.scratch + part_bytes);
    const int64_t rows = (int64_t)p.B * p.H * p.N;
    const int nguard = guard_blocks(rows);
    {
        int lpr_log2 = 0;
        while ((int)(16 / sizeof(typename T::T)) << lpr_log2 < p.D) ++lpr_log2;
        hipLaunchKernelGGL(split_guard_kernel<T>, dim3((unsigned)nguard), dim3(256), 0, st, p, lpr_log2, rows, (rows + nguard - 1) / nguard, guard);
        if (hipGetLastError() != hipSuccess) return SA2_ERR_LAUNCH_FAILED;
    }
    if (p.dq.p || p.dk2.p || p.dv2.p) {
        const int nkb = (p.N + BQ - 1) / BQ;
        const int64_t per_seg = (int64_t)nkb * p.B * p.H, total = per_seg * pl.nseg;
        if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
        float* part = (float*)p.scratch;
        float* kpart = (float*)((char*)p.scratch + split_dq_part_bytes(p.B, p.N, p.H, D, pl));
        if (lone_kp<T, D, MODE>(p.B, p.N, p.H, p.w1, p.w2, pl)) {
            const SplitKpLaunch l = {pl, nkb, (int)per_seg, part, kpart};
            const int rc = (T::DTYPE == SA2_F32 ? launch_split_kp_lone_fp32 : T::DTYPE == SA2_F16 ? launch_split_kp_lone_fp16 : launch_split_kp_lone_bf16)(
                p, D, exact_products<T>(p, true), l, st);
            if (rc != SA2_OK) return rc;
        } else if constexpr (!(lone<T, D, MODE>() && (T::DTYPE == SA2_F32 ? D == 64 : T::PLANES == 1 && D == 96))) {
            if (!allow_full_lds((const void*)split_kp_kernel<T, D, MODE>)) return SA2_ERR_LAUNCH_FAILED;
            hipLaunchKernelGGL((split_kp_kernel<T, D, MODE>), dim3((unsigned)total), dim3(XT), C::kp_lds(pl.segw - 1), st, p, nkb, (int)per_seg, part,
                               pl.nseg, pl.segw, kpart);
            if (hipGetLastError() != hipSuccess) return SA2_ERR_LAUNCH_FAILED;
        }
        sums.dq = p.dq.p ? part : nullptr;
        sums.nkb = nkb;
        sums.nseg = sums.kp_n = pl.nseg;
        sums.segw = pl.segw;
        sums.kp = pl.nseg > 1 ? kpart : nullptr;
    }
    if (p.dk1.p || p.dv1.p) {
        const int njb = (p.N + XJ - 1) / XJ;
        const int64_t total = (int64_t)njb * p.B * p.H * nsplit;
        if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
        float* part = nsplit > 1 ? (float*)((char*)p.scratch + kp_bytes) : nullptr;
        if (lone_kv<T, D, MODE>(p.N, p.w2)) {
            const int rc = (T::DTYPE == SA2_F32 ? launch_split_kv_lone_fp32 : T::DTYPE == SA2_F16 ? launch_split_kv_lone_fp16 : launch_split_kv_lone_bf16)(
                p, D, exact_products<T>(p, true), nsplit, part, st);
            if (rc != SA2_OK) return rc;
        } else if constexpr (!lone<T, D, MODE>() || T::DTYPE == SA2_F16) {
            auto go = [&](auto kernel) {
                if (!allow_full_lds((const void*)kernel)) return false;
                hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(XT), C::KV_LDS, st, p, njb, (int)total, nsplit, part);
                return hipGetLastError() == hipSuccess;
            };
            if (!(nsplit > 1 ? go(split_kv_kernel<T, D, true, MODE>) : go(split_kv_kernel<T, D, false, MODE>))) return SA2_ERR_LAUNCH_FAILED;
        }
        sums.kv = part;
        sums.kv_n = nsplit;
    }
    const int rc = launch_bwd_sums(p, sums, D, T::DTYPE, st);
    if (rc != SA2_OK) return rc;
    const int nblk = (p.N + FMA_ROWS - 1) / FMA_ROWS;
    const int64_t blocks = (int64_t)nblk * p.B * p.H;
    if (!allow_full_lds((const void*)split_fma_bwd_kernel<typename T::Fma>)) return SA2_ERR_LAUNCH_FAILED;
    hipLaunchKernelGGL(split_fma_bwd_kernel<typename T::Fma>, dim3((unsigned)(blocks < FMA_BLOCKS ? blocks : FMA_BLOCKS)), dim3(FMA_ROWS * 64),
                       smem_bytes(p.D, FMA_ROWS), st, p, guard, nguard, nblk, blocks);
    return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
}

// rows on a 16-byte grid
template <int PER_CHUNK>
bool rows16(const Tensor& t, int B, int N, int H) {
    constexpr int M = PER_CHUNK - 1;
    if (!t.p) return true;
    if ((uintptr_t)t.p & 15u) return false;
    return !((B > 1 && (t.sb & M)) || (N > 1 && (t.sn & M)) || (H > 1 && (t.sh & M)));
}

// Kernel width of a head_dim, and the call f(memory type, width, MODE) for it.  16-bit tensors come here only with head
// dims that the 16-bit kernels do not have, always padded or 96 columns wide.
int split_width(int D) { return D <= 32 ? 32 : D <= 64 ? 64 : D <= 96 ? 96 : 128; }
template <class F>
int for_split_width(int D, int dtype, F&& f) {
    auto of_width = [&](auto m, auto width) {
        constexpr int W = decltype(width)::value;
        if constexpr (decltype(m)::DTYPE == SA2_F32) {
            if constexpr (W != 96) {
                if (D == W) return f(m, width, std::integral_constant<int, EXACT>{});
            }
            if constexpr (W == 32) {
                if (D == 16) return f(m, width, std::integral_constant<int, PADDED>{});
            }
            return f(m, width, std::integral_constant<int, PADDED_FINE>{});
        } else {
            return f(m, width, std::integral_constant<int, PADDED>{});
        }
    };
    auto of_type = [&](auto m) {
        switch (split_width(D)) {
            case 32: return of_width(m, std::integral_constant<int, 32>{});
            case 64: return of_width(m, std::integral_constant<int, 64>{});
            case 96: return of_width(m, std::integral_constant<int, 96>{});
            default: return of_width(m, std::integral_constant<int, 128>{});
        }
    };
    return dtype == SA2_F32 ? of_type(MemF32{}) : dtype == SA2_F16 ? of_type(Mem16<ElemF16>{}) : of_type(Mem16<ElemBF16>{});
}

}  // namespace

// fp32: any multiple of four columns.  16 bits: multiples of eight that the 16-bit kernels do not take.
bool f32_mfma_supported(int D, int dtype) {
    if (D < 4 || D > 128) return false;
    return dtype == SA2_F32 ? D % 4 == 0 : D % 8 == 0 && D != 16 && D != 32 && D != 64 && D != 128;
}

bool f32_mfma_bwd_supported(int D, int w2, int dtype) {
    (void)w2;                // any K' window: wide ones are walked in segments
    return f32_mfma_supported(D, dtype);
}

bool f32_mfma_layout_ok(const Problem& p, int dtype, bool backward) {
    auto ok = [&](const Tensor& t) { return dtype == SA2_F32 ? rows16<4>(t, p.B, p.N, p.H) : rows16<8>(t, p.B, p.N, p.H); };
    const Tensor* fwd[] = {&p.q, &p.k1, &p.k2, &p.v1, &p.v2, &p.out};
    for (const Tensor* t : fwd)
        if (!ok(*t)) return false;
    if (backward) {
        const Tensor* bwd[] = {&p.dout, &p.dq, &p.dk1, &p.dk2, &p.dv1, &p.dv2};
        for (const Tensor* t : bwd)
            if (!ok(*t)) return false;
    }
    return true;
}

size_t f32_mfma_bwd_scratch_bytes(int B, int N, int H, int head_dim, int w1, int w2, int dtype, size_t room) {
    const size_t guard = guard_bytes(B, N, H);
    size_t bytes = 0;
    room = room_left(room, guard);
    for_split_width(head_dim, dtype, [&](auto m, auto width, auto mode) {
        constexpr int D = decltype(width)::value;
        const size_t kp = (split_kp_bytes(B, N, H, D, split_kp_plan<decltype(m), D, decltype(mode)::value>(B, N, H, w1, w2, room)) + 255) / 256 * 256;
        bytes = kp + split_kv_bytes(B, N, H, D, split_kv_nsplit(B, N, H, D, w1, w2, room_left(room, kp))) + guard;
        return 0;
    });
    return bytes;
}

int f32_mfma_fwd_nsplit(int B, int N, int H, int head_dim, int w1, int w2, int dtype, size_t room) {
    return for_split_width(head_dim, dtype, [&](auto m, auto width, auto mode) {
        constexpr int D = decltype(width)::value;
        const int round = forward_round<decltype(m), D, decltype(mode)::value>(B, N, H, w2);
        // (fp32 up to 64 columns: two short rounds stay one launch, though two shares take B1 H1 N1314 D64 w 17/10 17.8 us for 19.8, H3 N253 w 20/11
        // 17.6 for 19.8: there a forward without a workspace, which captured callers of the static workspace make, gives the bits of one with it.)
        return plan_forward(B, N, H, D, w1, w2, round, dtype == SA2_F32 && D <= 64 ? 4 : 0, room);
    });
}
// (of tests) whether its forward has two units per wavefront, and 256 * shares; whether its K' and K side have one wavefront per SIMD, and 256 *
// segments or shares
int split_kp_route(int B, int N, int H, int head_dim, int w1, int w2, int dtype) {
    return for_split_width(head_dim, dtype, [&](auto m, auto width, auto mode) {
        const KpPlan pl = split_kp_plan<decltype(m), decltype(width)::value, decltype(mode)::value>(B, N, H, w1, w2, ROOM_ANY);
        return pl.nseg << 8 | (int)lone_kp<decltype(m), decltype(width)::value, decltype(mode)::value>(B, N, H, w1, w2, pl);
    });
}
int split_kv_route(int B, int N, int H, int head_dim, int w1, int w2, int dtype) {
    return for_split_width(head_dim, dtype, [&](auto m, auto width, auto mode) {
        return split_kv_nsplit(B, N, H, decltype(width)::value, w1, w2, ROOM_ANY) << 8 | (int)lone_kv<decltype(m), decltype(width)::value, decltype(mode)::value>(N, w2);
    });
}
int split_fwd_route(int B, int N, int H, int head_dim, int w1, int w2, int dtype) {
    const int ns = f32_mfma_fwd_nsplit(B, N, H, head_dim, w1, w2, dtype, ROOM_ANY);
    return ns << 8 | for_split_width(head_dim, dtype, [&](auto m, auto width, auto mode) {
        return (int)lone_forward<decltype(m), decltype(width)::value, decltype(mode)::value>(B, N, H, w1, w2, ns);
    });
}
size_t f32_mfma_fwd_part_bytes(int B, int N, int H, int head_dim, int nsplit) { return fwd_part_bytes(B, N, H, split_width(head_dim), nsplit); }

int launch_f32_mfma_fwd(const Problem& p, int dtype, hipStream_t st) {
    return for_split_width(p.D, dtype, [&](auto m, auto width, auto mode) {
        return launch_split_fwd<decltype(m), decltype(width)::value, decltype(mode)::value>(p, st);
    });
}

int launch_f32_mfma_bwd(const Problem& p, int dtype, hipStream_t st) {
    return for_split_width(p.D, dtype, [&](auto m, auto width, auto mode) {
        return launch_split_bwd<decltype(m), decltype(width)::value, decltype(mode)::value>(p, st);
    });
}

}  // namespace sa2
