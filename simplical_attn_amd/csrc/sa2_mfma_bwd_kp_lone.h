// The K'-side backward kernel (dQ, dK' and dV') of the tuned 16-bit kernels for wide K windows, head_dim 64 and 128; included
// once per element type.  Sums, partials and segments are those of sa2_mfma_bwd_kp.hip, which also says what a unit is.
//
// Four wavefronts, one per SIMD with all 512 registers (sa2_mfma_lone.h), hold one unit each per round, or two consecutive
// deltas at head_dim 64, and sweep the K1/V1 window in 32-key tiles that go straight from global memory into a ring in LDS,
// three tiles ahead.  Per tile and unit a wavefront computes
//   A: S^T = K1.Q~^T - LSE and dP^T = V1.dO~^T,  B: P = exp2(S) and dS = P * (dP - D),  C: R^T += V1^T.P^T and G^T += K1^T.dS^T,
// B between the MFMAs of A and C of the other unit (of the next tile at head_dim 128), operand reads eight MFMAs ahead of their
// use: nothing is handed from one wavefront to another, and every operand read serves all units of the wavefront.
// Within a sweep the next tile's address is one addition per tensor; only the last three tiles, which ask for the next round's
// first ones, work it out (some fifty scalar instructions, which cost a lone wavefront as much as vector ones).
// Where LDS has the room the K' rows lie there in fp32 as (k2 + bias) * scale * log2(e): a word of Q~ takes five vector instructions
// instead of eleven, an element of dQ's sums three instead of five (K' side 2433 -> 2400 us and 394 -> 374 at the first two sizes below).
// What bounds it: the instructions beside the MFMAs, at head_dim 128 also power.  Time stamps of a workgroup's rounds, us: B1 H16 N8192
// D128 w 512/32 forming 1.8, sweep of 18 tiles 13.3, sums 1.8, dQ 1.5; B2 H8 N2048 D64 w 512/32 1.6, 17.2, 2.1, 1.8.  K' side with row term,
// pre-pass and sums against the two-wavefront kernel, in turn on one machine (bf16): B2 H8 N2048 D64 w 512/32 428 -> 375 us,
// B1 H16 N8192 D128 w 512/32 2831 -> 2570.
#pragma once

#include "sa2_mfma_bwd_kp_plan.h"
#include "sa2_mfma_lone.h"

namespace sa2 {
namespace {

// RAW, WIDE: see KpLoneCfg::main_bytes.  The K' window is cut into nseg runs of segw deltas, one workgroup per (K' block, segment).
// Each writes its own dQ partial (rows k0 + seg*segw ..) and, when nseg > 1, fp32 partial dK' and dV' to `kpart`
// ([dV' | dK'][nseg][B*H][N][D]) for bwd_sum_kernel.  left = 1: the pre-pass took the unit delta = w2 of every block and left
// its results in the output tensors and in rows w2 .. of the dQ partials.
template <class E, int D, bool RAW, bool WIDE>
__global__ __launch_bounds__(KpLoneCfg<D>::T) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mfma_bwd_kp_lone_kernel(Problem p, int nkb, int total, float* __restrict__ dq_part, int left, int nseg, int segw, float* __restrict__ kpart) {
    typedef typename E::scalar EL;
    typedef typename E::x8 X8;
    using C = KpLoneCfg<D>;
    constexpr int U = C::U, KW = C::W, KT = C::T;
    using L = Lone<256>;
    constexpr int UPR = KW * U;                               // units per round
    constexpr int DK = C::DK, DT = C::DT;
    constexpr bool DVV = D == 128;
    using T = typename C::Tile;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int w2s = segw - 1;                                 // deltas of a segment, minus one (w2 when there is one segment)
    const int RQ = BQ + w2s;                                  // query rows this workgroup touches
    unsigned char* k2_s = smem_raw + (size_t)C::NSTAGE * C::STAGE_BYTES;               // K' rows k0 .. k0+31, as in a tile, or
    float* kt_s = (float*)k2_s;                               // (WIDE) [BQ][AS] times scale * log2(e)
    unsigned char* v2_s = k2_s + (WIDE ? (size_t)BQ * C::AS * 4 : C::row_bytes(BQ));   // V' rows
    unsigned char* q_s = v2_s + C::row_bytes(BQ);             // q rows kq .. kq+RQ-1  (when RAW)
    unsigned char* do_s = q_s + C::row_bytes(RQ);             // dO rows               (when RAW)
    const int RQ4 = (RQ + 3) & ~3;
    float* lse_s = (float*)(RAW ? do_s + C::row_bytes(RQ) : q_s);          // [RQ] LSE * log2(e)
    float* dsum_s = lse_s + RQ4;                              // [RQ] D_i
    float* dqacc = dsum_s + RQ4;                              // [RQ][AS]

    // lane parts of what happens once per round are computed where they are used
    auto here = [&]() __attribute__((always_inline)) {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;

    // Launch order: all (K' block, head) pairs of segment 0, then those of segment 1, ...: the last segment
    // is the short one, and workgroups that alternate between long and short in launch order end up with
    // the long ones on half of the CUs (measured: twice the time).  Within a segment consecutive blocks go
    // to the same XCD.
    const int per_seg = total / nseg, seg = (int)blockIdx.x / per_seg;
    const int pb = xcd_order((int)blockIdx.x - seg * per_seg, per_seg);
    const int bh = pb / nkb, kb = pb - bh * nkb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int k0 = kb * BQ;
    const int dlo = seg * segw;                               // first delta of the segment
    const int dhi = dlo + w2s < w2 ? dlo + w2s : w2;          // last one
    const int kq = k0 + dlo;                                  // query of K' row k0 at the segment's first delta
    const int i_hi = (int)((int64_t)k0 + BQ - 1 + dhi < N - 1 ? k0 + BQ - 1 + dhi : N - 1);

    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* k1p = (const uint16_t*)p.k1.p + p.k1.off(b, 0, h);
    const uint16_t* k2p = (const uint16_t*)p.k2.p + p.k2.off(b, 0, h);
    const uint16_t* v1p = (const uint16_t*)p.v1.p + p.v1.off(b, 0, h);
    const uint16_t* v2p = (const uint16_t*)p.v2.p + p.v2.off(b, 0, h);
    const uint16_t* dop = (const uint16_t*)p.dout.p + p.dout.off(b, 0, h);

    // the unit delta = w2 exists for this block and the pre-pass took it
    const bool has_left = left && k0 + w2 <= N - 1;
    const int nu_all = (w2 < N - 1 - k0 ? w2 : N - 1 - k0) + 1 - (has_left ? 1 : 0);      // units of the K' block
    const int n_units = nu_all - dlo < segw ? nu_all - dlo : segw;                        // of this segment (may be <= 0)
    const int nrounds = n_units > 0 ? (n_units + UPR - 1) / UPR : 0;
    // Tiles a round sweeps: from the first tile of its smallest delta to the last tile of its largest one
    auto round_first = [&](int round) __attribute__((always_inline)) {
        const int i_min = kq + round * UPR;
        return (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
    };
    auto round_last = [&](int round) __attribute__((always_inline)) {
        const int dl = (round + 1) * UPR - 1 < n_units - 1 ? (round + 1) * UPR - 1 : n_units - 1;
        const int i_max = kq + dl + BQ - 1 < N - 1 ? kq + dl + BQ - 1 : N - 1;
        return i_max / TJ;
    };
    const bool want_dq = p.dq.p != nullptr;

    // ---- tiles: wavefront w requests groups w, w + 4 of both, straight into LDS, in the order of the sweeps ----
    const uint32_t lds0 = lds_address(smem_raw);
    const int jt_end = (N - 1) / TJ;
    const bool near_end = N % TJ != 0 && i_hi / TJ == jt_end;          // (a tile whose rows past the end read the last one)
    uint32_t k_off[C::NREQ], v_off[C::NREQ];                  // byte offset of the lane's chunk from a tile's first row
    int next_round = 0, next_tile = round_first(0), next_last = round_last(0);
    const char *k_next = (const char*)k1p, *v_next = (const char*)v1p;      // first rows of the next tile
    const int64_t k_step = (int64_t)TJ * 2 * p.k1.sn, v_step = (int64_t)TJ * 2 * p.v1.sn;
    auto aim = [&](int jt) __attribute__((always_inline)) {   // lane offsets for tile jt: where the rows end, the last tile's differ
        const int l = here() & 63, col = T::dma_chunk(l) * 8;
        const int last = jt == jt_end ? N - 1 - jt_end * TJ : TJ - 1;
#pragma unroll
        for (int x = 0; x < C::NREQ; ++x) {
            const int t_row = (wave + KW * x) * T::RPW + T::dma_row(l), r = t_row < last ? t_row : last;
            k_off[x] = ((uint32_t)r * (uint32_t)p.k1.sn + col) * 2u;
            v_off[x] = ((uint32_t)r * (uint32_t)p.v1.sn + col) * 2u;
        }
    };
    auto request_part = [&](auto X, uint32_t stage) __attribute__((always_inline)) {        // K's groups, then V's
        constexpr int x = decltype(X)::value % C::NREQ;
        const uint32_t to = stage + (uint32_t)((wave + KW * x) * T::GROUP);
        if constexpr (decltype(X)::value < C::NREQ) lds_request(k_next, k_off[x], to);
        else lds_request(v_next, v_off[x], to + C::TILE_BYTES);
    };
    auto request_tile = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<2 * C::NREQ>([&](auto X) __attribute__((always_inline)) { request_part(X, stage); });
    };
    // The tile after the one requested last (behind the last round: that one again, which nothing reads).  In pieces without
    // branches, which ride on MFMAs: scalar instructions cost a lone wavefront as much as vector ones.  ON: within a sweep
    // (the caller counts next_tile up).
    int wrap = 0, nr = 0, more = 0, first = 0, last = 0;
    auto next_piece = [&](auto I, auto ON) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        if constexpr (decltype(ON)::value) {
            if constexpr (i == 0) k_next += k_step;
            if constexpr (i == 1) v_next += v_step;
            return;
        }
        auto here_on = [](int& x) __attribute__((always_inline)) {       // (no piece moves up to another)
            x = __builtin_amdgcn_readfirstlane(x);
            asm volatile("" : "+s"(x));
        };
        if constexpr (i == 0) {
            here_on(next_tile);
            wrap = next_tile == next_last;
            nr = next_round + wrap;
            more = nr < nrounds;
        } else if constexpr (i == 1) {
            here_on(nr);
            const int lo = kq + nr * UPR - w1;
            first = (int)((unsigned)(lo > 0 ? lo : 0) / TJ);
        } else if constexpr (i == 2) {
            here_on(nr);
            const int d = (nr + 1) * UPR < n_units ? (nr + 1) * UPR : n_units, hi = kq + d + BQ - 2;
            last = (int)((unsigned)(hi < N - 1 ? hi : N - 1) / TJ);
        } else if constexpr (i == 3) {
            here_on(first);
            here_on(last);
            first = more ? first : next_tile;
            next_tile = wrap ? first : next_tile + 1;
            next_round = more ? nr : next_round;
            next_last = more ? last : next_last;
        } else if constexpr (i == 4) {
            here_on(next_tile);
            k_next = (const char*)k1p + next_tile * k_step;
        } else if constexpr (i == 5) {
            here_on(next_tile);
            v_next = (const char*)v1p + next_tile * v_step;
        }
    };
    auto next_request = [&]() __attribute__((always_inline)) {
        static_for<6>([&](auto I) __attribute__((always_inline)) { next_piece(I, std::false_type{}); });
        if (near_end) aim(next_tile);
    };
    constexpr int INFLIGHT = 2 * C::NREQ;                     // requests of one tile (two are under way)
    auto step_barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(INFLIGHT) : "memory");
    };

    // ---- rows, LSE, D and the dQ accumulator.  What goes through registers is loaded first and stored last. ----
    auto request_rows = [&](const uint16_t* base, int64_t sn, int first, int rows, const unsigned char* to) __attribute__((always_inline)) {
        const int l = here() & 63, col = T::dma_chunk(l) * 8;
        for (int g = wave; g * T::RPW < rows; g += KW) {
            const int r = first + g * T::RPW + T::dma_row(l), rc = r < N ? r : N - 1;
            lds_request(base + (int64_t)rc * sn + col, lds0 + (uint32_t)(to - smem_raw) + (uint32_t)(g * T::GROUP));
        }
    };
    auto row_value = [&](const float* of, int c) __attribute__((always_inline)) { return of[(int64_t)bh * N + (kq + c < N ? kq + c : N - 1)]; };
    {
        const float lse0 = row_value(p.lse, tid), dsum0 = row_value(p.dsum, tid);
        u4 from_left[D / 32] = {};                            // rows w2 .. w2+31 of the accumulator start from the pre-pass contribution
        const bool take = has_left && want_dq;
        if (take) {
#pragma unroll
            for (int x = 0; x < D / 32; ++x)
                from_left[x] = *(const u4*)(dq_part + (((int64_t)bh * nkb + kb) * RQ + w2) * D + (tid + x * KT) * 4);
        }
        constexpr int NK2 = BQ * (D / 8) / KT;                // 16-byte chunks of the K' rows per thread
        uint4 kraw[NK2];
        if constexpr (WIDE) {
#pragma unroll
            for (int x = 0; x < NK2; ++x) {
                const int c = tid + x * KT, r = k0 + c / (D / 8);
                kraw[x] = *(const uint4*)(k2p + (int64_t)(r < N ? r : N - 1) * p.k2.sn + c % (D / 8) * 8);
            }
        } else {
            request_rows(k2p, p.k2.sn, k0, BQ, k2_s);
        }
        request_rows(v2p, p.v2.sn, k0, BQ, v2_s);
        if constexpr (RAW) {
            request_rows(qp, p.q.sn, kq, RQ, q_s);
            request_rows(dop, p.dout.sn, kq, RQ, do_s);
        }
        if (nrounds > 0) {
            aim(next_tile);
            static_for<2>([&](auto I) __attribute__((always_inline)) { next_piece(LONE_C(4 + decltype(I)::value), std::false_type{}); });
            request_tile(lds0);
#pragma unroll 1
            for (int x = 1; x < C::NSTAGE - 1; ++x) {
                next_request();
                request_tile(lds0 + x * C::STAGE_BYTES);
            }
        }
        if constexpr (WIDE) {
            const float qscale = p.scale * LOG2E;
#pragma unroll
            for (int x = 0; x < NK2; ++x) {
                const int c = tid + x * KT;
                const uint32_t w[4] = {kraw[x].x, kraw[x].y, kraw[x].z, kraw[x].w};
                float* to = kt_s + c / (D / 8) * C::AS + c % (D / 8) * 8;
#pragma unroll
                for (int t = 0; t < 4; t += 2)
                    *(float4*)(to + 2 * t) = make_float4((E::lo(w[t]) + p.k2_bias) * qscale, (E::hi(w[t]) + p.k2_bias) * qscale,
                                                         (E::lo(w[t + 1]) + p.k2_bias) * qscale, (E::hi(w[t + 1]) + p.k2_bias) * qscale);
            }
        }
        for (int c = tid; c < RQ * (C::AS / 4); c += KT) ((float4*)dqacc)[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (tid < RQ) {
            lse_s[tid] = lse0 * LOG2E;
            dsum_s[tid] = dsum0;
        }
        for (int c = tid + KT; c < RQ; c += KT) {
            lse_s[c] = row_value(p.lse, c) * LOG2E;
            dsum_s[c] = row_value(p.dsum, c);
        }
        if (take) {
            __syncthreads();
#pragma unroll
            for (int x = 0; x < D / 32; ++x) {
                const int it = tid + x * KT;
                float4 y = __builtin_bit_cast(float4, from_left[x]);
                if constexpr (WIDE) {
                    const float qscale = p.scale * LOG2E;
                    y.x *= qscale; y.y *= qscale; y.z *= qscale; y.w *= qscale;
                }
                *(float4*)(dqacc + (w2 + it / (D / 4)) * C::AS + it % (D / 4) * 4) = y;
            }
        }
    }
    // 16 bytes of row `rel` as the row operand of k-step kk holds them, and 4 elements from column 8*e + 4*hf on: q or dO row kq + rel
    // (the copy in LDS, or global memory), K' or V' row k0 + rel
    auto lds_row8 = [&](const unsigned char* rows, int rel, int hf_, int kk) __attribute__((always_inline)) {
        return *(const uint4*)(rows + T::row_at(0, (uint32_t)(T::row_off(rel) + (hf_ ^ T::flip(rel)) * 16), kk));
    };
    auto lds_row4 = [&](const unsigned char* rows, int rel, int hf_, int e) __attribute__((always_inline)) {
        return *(const uint2*)(rows + T::row_off(rel) + e / 4 * T::BLOCK + (e % 4 ^ T::flip(rel)) * 16 + hf_ * 8);
    };
    auto far_row = [&](const uint16_t* base, int64_t sn, int rel) __attribute__((always_inline)) { return base + (int64_t)(kq + rel < N ? kq + rel : N - 1) * sn; };
    const float qscale = p.scale * LOG2E;
    const uint32_t row_lane = T::row_lane(lane), col_lane = T::column_lane(lane);            // row, transposed operand

    // ---- a wavefront's sweep (the phases A, B and C of an element: one unit's share of a tile) ----
    // accumulation registers: R tiles, G tiles, Q~ and dO~ as B operands, dK' and (head_dim 64) dV'
    constexpr int R0 = 0, G0 = U * DT * 16, Q0 = 2 * U * DT * 16, O0 = Q0 + U * DK * 4, DK0 = 192, DV0 = DK0 + DT * 16;
    static_assert(O0 + U * DK * 4 <= 192 && (DVV ? DV0 : DV0 + DT * 16) <= 256, "");
    floatx16 dvv[DVV ? DT : 1];                               // dV' at head_dim 128
#pragma unroll
    for (int dt = 0; dt < (DVV ? DT : 1); ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) dvv[dt][v] = 0.f;
    X8 ka[DK], va[DK];                                        // row operands of the K and V tile
    X8 vt[DT][2], kt[DT][2];                                  // transposed operands
    floatx16 s[U], dp[U];
    u4 pw[U][2], dw[U][2];                                    // P, dS in 16 bits
    floatx16 nl[U];                                           // -LSE*log2e of the lane's row, -inf where the pair is outside the windows
    float drow_sum[U];                                        // D of the lane's row
    uint32_t sc = lds0 + (C::NSTAGE - 1) * C::STAGE_BYTES, sa = lds0, sb = lds0 + C::STAGE_BYTES, sd = lds0 + 2 * C::STAGE_BYTES;      // stages of tiles t-1, t, t+1, t+2
    constexpr bool LONG = DK == 8;                            // operands of head_dim 128 are read one kind at a time
    constexpr int NE = 2 * DK;                                // MFMAs of a phase
    static_assert(NE == 4 * DT, "");

    auto read_row = [&](auto WHICH, auto KK, uint32_t stage) __attribute__((always_inline)) {
        constexpr int kk = decltype(KK)::value;
        const X8 x = lds_read_x8<X8>(T::row_at(stage + decltype(WHICH)::value * C::TILE_BYTES, row_lane, kk));
        if constexpr (decltype(WHICH)::value) va[kk] = x;
        else ka[kk] = x;
    };
    auto read_first_rows = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<DK>([&](auto KK) __attribute__((always_inline)) {
            read_row(LONE_C(0), KK, stage);
            if constexpr (!LONG) read_row(LONE_C(1), KK, stage);
        });
    };
    // in the order of the R and G products
    auto read_column = [&](auto X, uint32_t stage) __attribute__((always_inline)) {
        constexpr int which = decltype(X)::value / (2 * DT), ks = decltype(X)::value / DT % 2, dt = decltype(X)::value % DT;
        const X8 x = quad_tile_column<D, X8>(stage + (which ? 0 : C::TILE_BYTES), col_lane, dt, ks);
        if constexpr (which) kt[dt][ks] = x;
        else vt[dt][ks] = x;
    };
    auto a_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, kk = i % DK, at = (u * DK + kk) * 4;
        if constexpr (i == 0) L::tile_start<Q0 + at>(s[u], ka[0], nl[u]);
        else if constexpr (i < DK) L::tile_more<Q0 + at>(s[u], ka[kk]);
        else if constexpr (i == DK) L::tile_start<O0 + at>(dp[u], va[0]);
        else L::tile_more<O0 + at>(dp[u], va[kk]);
    };
    auto c_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value;
        constexpr int which = i / (2 * DT), ks = i / DT % 2, dt = i % DT;
        if constexpr (which == 0) L::sum_more<R0 + (u * DT + dt) * 16>(vt[dt][ks], __builtin_bit_cast(X8, pw[u][ks]));
        else L::sum_more<G0 + (u * DT + dt) * 16>(kt[dt][ks], __builtin_bit_cast(X8, dw[u][ks]));
    };
    // (an exponential's result may not be read by the next instruction: a pair is rounded behind the next pair's exponentials)
    auto round_p = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value;
        pw[u][i / 4][i % 4] = pack2<E>(s[u][2 * i], s[u][2 * i + 1]);
    };
    auto p_item = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, e = 2 * i;
        float x = fast_exp2(s[u][e]), y = fast_exp2(s[u][e + 1]);
        stays(x);
        stays(y);
        s[u][e] = x;
        s[u][e + 1] = y;
        if constexpr (i > 0) round_p(UN, LONE_C(i - 1));
    };
    // dS from the unrounded weights but for a sweep's first tile: nothing but dS itself is rounded to 16 bits.  (From the rounded ones, as
    // the two-wavefront kernel forms it, whose weights cross LDS in 16 bits, it is two instructions a pair more and the 2-norm errors of dQ
    // and dK' against fp32 are 4 - 9 % larger.)  The first tile's weights are rounded before they meet dP: it holds all keys of the first queries,
    // which have few weights, all large, so that single gradients there follow the rounding of each, and a gradient does not depend on which of
    // the two kernels a problem is given to (up to 0.5 of its root mean square elsewhere with unrounded ones, B1 H8 N32768 D128 w 1024/64).
    auto first_tile = [&](auto UN) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value;
        static_for<8>([&](auto X) __attribute__((always_inline)) {
            constexpr int e = 2 * decltype(X)::value;
            const uint32_t w = pack2<E>(s[u][e], s[u][e + 1]);
            s[u][e] = E::lo(w);
            s[u][e + 1] = E::hi(w);
        });
    };
    auto ds_item = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, ks = i / 4, t = i % 4, e = 2 * i;
        if constexpr (i == 0) round_p(UN, LONE_C(7));
        uint32_t w = pack2<E>(s[u][e] * (dp[u][e] - drow_sum[u]), s[u][e + 1] * (dp[u][e + 1] - drow_sum[u]));
        stays(w);
        dw[u][ks][t] = w;
    };
    auto b_all = [&](auto UN) __attribute__((always_inline)) {
        static_for<8>([&](auto X) __attribute__((always_inline)) { p_item(UN, X); });
        static_for<8>([&](auto X) __attribute__((always_inline)) { ds_item(UN, X); });
    };
    // One unit: A(t), then C(t-1), whose four groups of MFMAs (R^T and G^T, each from the keys' first and second half) free the
    // halves of P and dS one after the other for B(t).  B(t) starts beside the second half of A(t), where the logits are done,
    // forms dS in fp32 in the place of dP, and rounds its second half beside the first MFMAs of A(t+1): nothing is left to do between two tiles.
    constexpr int BAR = 2 * DT;                               // MFMA of phase C that the tile's barrier stands before
    auto exp_item = [&](auto I) __attribute__((always_inline)) {
        float x = fast_exp2(s[0][decltype(I)::value]);
        stays(x);
        s[0][decltype(I)::value] = x;
    };
    auto p_word = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        uint32_t w = pack2<E>(s[0][2 * i], s[0][2 * i + 1]);
        stays(w);
        pw[0][i / 4][i % 4] = w;
    };
    auto ds_value = [&](auto I) __attribute__((always_inline)) {
        constexpr int e = decltype(I)::value;
        float x = s[0][e] * (dp[0][e] - drow_sum[0]);
        stays(x);
        dp[0][e] = x;
    };
    auto ds_word = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        uint32_t w = pack2<E>(dp[0][2 * i], dp[0][2 * i + 1]);
        stays(w);
        dw[0][i / 4][i % 4] = w;
    };
    // items LO .. HI-1 of a kind
    auto items = [&](auto LO, auto HI, auto&& f) __attribute__((always_inline)) {
        static_for<decltype(HI)::value - decltype(LO)::value>([&](auto X) __attribute__((always_inline)) { f(LONE_C(decltype(LO)::value + decltype(X)::value)); });
    };
    auto single = [&](auto DO_C, auto ON) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        static_assert(LONG && sizeof(DO_C) > 0, "one unit per wavefront: head_dim 128");
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(0), I);
            if constexpr (i < DK) read_row(LONE_C(1), I, sa);
            next_piece(LONE_C(i - 1), ON);
            if constexpr (CC) deal<12, i - 4, 12>([&](auto X) __attribute__((always_inline)) { read_column(X, sc); });
            if constexpr (CC && i < 4) ds_word(LONE_C(4 + i));
            if constexpr (i >= DK + 2) items(LONE_C(2 * (i - DK - 2)), LONE_C(2 * (i - DK - 2) + 2), exp_item);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) finished(s[0], dp[0]);
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            if constexpr (i == BAR) step_barrier();
            if constexpr (CC) {
                c_mfma(LONE_C(0), I);
                if constexpr (i < 4) read_column(LONE_C(12 + i), sc);
            }
            if constexpr (i >= BAR) read_row(LONE_C(0), LONE_C(i - BAR), sb);
            constexpr int EXPS[17] = {12, 14, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16, 16};
            constexpr int PW[17] = {0, 0, 0, 0, 0, 2, 4, 4, 4, 6, 8, 8, 8, 8, 8, 8, 8};
            constexpr int DSV[17] = {0, 0, 0, 2, 4, 5, 6, 8, 10, 10, 11, 12, 14, 15, 16, 16, 16};
            constexpr int DSW[17] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 2, 3, 4};
            items(LONE_C(EXPS[i]), LONE_C(EXPS[i + 1]), exp_item);
            if constexpr (!CC && i == 2) first_tile(LONE_C(0));           // (all weights are formed, none is used yet)
            items(LONE_C(PW[i]), LONE_C(PW[i + 1]), p_word);
            items(LONE_C(DSV[i]), LONE_C(DSV[i + 1]), ds_value);
            items(LONE_C(DSW[i]), LONE_C(DSW[i + 1]), ds_word);
            if constexpr (i >= BAR) deal<2 * C::NREQ, (i - BAR) / 2, NE - BAR - DT>([&](auto X) __attribute__((always_inline)) { if constexpr (i % 2 == 0) request_part(X, sc); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto single_last = [&]() __attribute__((always_inline)) {                       // C of tile t-1 alone
        items(LONE_C(4), LONE_C(8), ds_word);
        static_for<4 * DT>([&](auto X) __attribute__((always_inline)) { read_column(X, sc); });
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(0), I); });
    };
    // Two units: A(t, 0), C(t-1, 1), A(t, 1), C(t, 0); the transposed operands of tile t serve C(t, 0) and C(t, 1).
    // The weights and dS of a unit are formed from the end of its phase A to the beginning of its phase C.
    auto pair = [&](auto DO_C, auto ON) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        auto later = [&](auto UN, auto I) __attribute__((always_inline)) {
            deal<8, decltype(I)::value, NE>([&](auto X) __attribute__((always_inline)) { ds_item(UN, X); });
        };
        auto early = [&](auto UN, auto I) __attribute__((always_inline)) {
            deal<8, decltype(I)::value, NE>([&](auto X) __attribute__((always_inline)) { p_item(UN, X); });
        };
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            a_mfma(LONE_C(0), I);
            if constexpr (decltype(I)::value % 2 == 0) next_piece(LONE_C(decltype(I)::value / 2 - 1), ON);
            if constexpr (CC) later(LONE_C(U - 1), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            if constexpr (CC) c_mfma(LONE_C(U - 1), I);
            if constexpr (i % 2 == 0 && i / 2 < 3) next_piece(LONE_C(3 + i / 2), ON);
            early(LONE_C(0), I);
            if constexpr (i >= 2) read_column(LONE_C(i - 2), sa);                   // (the MFMA that read its register is past)
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) first_tile(LONE_C(0));
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            a_mfma(LONE_C(U - 1), I);
            if constexpr (decltype(I)::value < 2) read_column(LONE_C(NE - 2 + decltype(I)::value), sa);
            later(LONE_C(0), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        // (no wait for reads of LDS: what is requested into, the stage of tile t-1, was last read by MFMAs that have been issued)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(INFLIGHT) : "memory");
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            c_mfma(LONE_C(0), I);
            read_row(LONE_C(i / DK), LONE_C(i % DK), sb);
            early(LONE_C(U - 1), I);
            if constexpr (i == 1) static_for<C::NREQ>([&](auto X) __attribute__((always_inline)) { request_part(X, sc); });
            if constexpr (i == NE - 2) static_for<C::NREQ>([&](auto X) __attribute__((always_inline)) { request_part(LONE_C(C::NREQ + decltype(X)::value), sc); });
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) first_tile(LONE_C(U - 1));
        stays(s[U - 1]);
    };
    auto pair_last = [&]() __attribute__((always_inline)) {                         // C(t-1, 1) alone
        static_for<8>([&](auto X) __attribute__((always_inline)) { ds_item(LONE_C(U - 1), X); });
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(U - 1), I); });
    };
    // One of two units has keys in the tile: it alone, nothing pending before or behind
    auto half = [&](auto UN) __attribute__((always_inline)) {
        static_for<NE>([&](auto I) __attribute__((always_inline)) { a_mfma(UN, I); });
        static_for<4 * DT>([&](auto X) __attribute__((always_inline)) { read_column(X, sa); });
        finished(s[decltype(UN)::value], dp[decltype(UN)::value]);
        b_all(UN);
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(UN, I); });
        step_barrier();
        next_request();
        request_tile(sc);
        read_first_rows(sb);
    };
    auto rotate = [&]() __attribute__((always_inline)) {
        L::keep_out();
        const uint32_t x = sc;
        sc = sa;
        sa = sb;
        sb = sd;
        sd = x;
    };

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    X8 zero;
#pragma unroll
    for (int t = 0; t < 8; ++t) zero[t] = (EL)0.f;
    static_for<(DVV ? 1 : 2) * DT * 4>([&](auto X) __attribute__((always_inline)) { L::set_regs<DK0 + 4 * decltype(X)::value>(0u, 0u, 0u, 0u); });
    if (nrounds > 0) read_first_rows(sa);

    for (int round = 0; round < nrounds; ++round) {
        // ---- operands, sums and row values of the round's units (one that does not exist: its neighbour's, and left out of all sums) ----
        const int d0 = round * UPR + wave * U;                // first delta of this wavefront
        const bool any = d0 < n_units;
        float lse2[U];
        asm volatile("s_nop 3" : "+v"(zero));
        static_for<2 * U * DT>([&](auto X) __attribute__((always_inline)) { L::sum_zero<16 * decltype(X)::value>(zero); });
        auto form = [&](auto BIASED) __attribute__((always_inline)) {
            const float kb = decltype(BIASED)::value ? p.k2_bias : 0.f, vb = decltype(BIASED)::value ? p.v2_bias : 0.f;
            const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
            uint4 qx[U][DK], ox[U][DK];                       // all reads of the rows first
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int delta = d0 + u < n_units ? d0 + u : n_units - 1;
#pragma unroll
                for (int kk = 0; kk < DK; ++kk) {
                    if constexpr (RAW) {
                        qx[u][kk] = lds_row8(q_s, ln_ + delta, hf_, kk);
                        ox[u][kk] = lds_row8(do_s, ln_ + delta, hf_, kk);
                    } else {
                        qx[u][kk] = load_cols8<false>(far_row(qp, p.q.sn, ln_ + delta), kk * 16 + hf_ * 8, p.D);
                        ox[u][kk] = load_cols8<false>(far_row(dop, p.dout.sn, ln_ + delta), kk * 16 + hf_ * 8, p.D);
                    }
                }
                lse2[u] = lse_s[ln_ + delta];
                drow_sum[u] = dsum_s[ln_ + delta];
            }
            static_for<DK>([&](auto KK) __attribute__((always_inline)) {
                constexpr int kk = decltype(KK)::value;
                float kt[8], vt_[8];                          // K'~ (scaled) and V'~ of the lane's row: the same for all units
                if constexpr (WIDE) {
                    const float* src = kt_s + ln_ * C::AS + kk * 16 + hf_ * 8;
                    const float4 k0_ = *(const float4*)src, k1_ = *(const float4*)(src + 4);
                    kt[0] = k0_.x; kt[1] = k0_.y; kt[2] = k0_.z; kt[3] = k0_.w;
                    kt[4] = k1_.x; kt[5] = k1_.y; kt[6] = k1_.z; kt[7] = k1_.w;
                } else {
                    const uint4 kx = lds_row8(k2_s, ln_, hf_, kk);
                    const uint32_t kw[4] = {kx.x, kx.y, kx.z, kx.w};
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        kt[2 * t] = (E::lo(kw[t]) + kb) * qscale;
                        kt[2 * t + 1] = (E::hi(kw[t]) + kb) * qscale;
                    }
                }
                const uint4 vx = lds_row8(v2_s, ln_, hf_, kk);
                const uint32_t vw[4] = {vx.x, vx.y, vx.z, vx.w};
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    vt_[2 * t] = E::lo(vw[t]) + vb;
                    vt_[2 * t + 1] = E::hi(vw[t]) + vb;
                }
                static_for<U>([&](auto UN) __attribute__((always_inline)) {
                    constexpr int u = decltype(UN)::value, at = (u * DK + kk) * 4;
                    const uint32_t qw[4] = {qx[u][kk].x, qx[u][kk].y, qx[u][kk].z, qx[u][kk].w}, ow[4] = {ox[u][kk].x, ox[u][kk].y, ox[u][kk].z, ox[u][kk].w};
                    uint32_t qt[4], ot[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        qt[t] = pack2<E>(E::lo(qw[t]) * kt[2 * t], E::hi(qw[t]) * kt[2 * t + 1]);
                        ot[t] = pack2<E>(E::lo(ow[t]) * vt_[2 * t], E::hi(ow[t]) * vt_[2 * t + 1]);
                    }
                    L::set_regs<Q0 + at>(qt[0], qt[1], qt[2], qt[3]);
                    L::set_regs<O0 + at>(ot[0], ot[1], ot[2], ot[3]);
                });
            });
        };
        if ((WIDE ? 0.f : p.k2_bias) != 0.f || p.v2_bias != 0.f) form(std::true_type{});
        else form(std::false_type{});
        L::keep_out();

        // ---- the sweep: tiles [t0, t1] hold keys of the first unit, [t2, t3] of the last one; [p0, p1] need no mask ----
        const int s0 = round_first(round), s1 = round_last(round);
        int t0 = 1, t1 = 0, t2 = 1, t3 = 0, p0 = 1, p1 = 0;
        if (any) {
            auto range = [&](int delta, int& a, int& z, int& pa, int& pz) __attribute__((always_inline)) {
                const int i_min = kq + delta, i_max = i_min + BQ - 1 < N - 1 ? i_min + BQ - 1 : N - 1;
                a = (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
                z = i_max / TJ;
                pa = i_max - w1 > 0 ? (i_max - w1 + TJ - 1) / TJ : 0;
                pz = i_min + BQ - 1 < N ? (i_min + 1) / TJ - 1 : -1;
            };
            int q0, q1;
            range(d0, t0, t1, p0, p1);
            const bool both = U > 1 && d0 + 1 < n_units;
            range(both ? d0 + 1 : d0, t2, t3, q0, q1);
            p0 = q0 > p0 ? q0 : p0;
            p1 = q1 < p1 ? q1 : p1;
        }
        const int a0 = t0 > t2 ? t0 : t2, a1 = t1 < t3 ? t1 : t3;         // tiles of all units
        bool unmasked = false;
        // the start of the S tiles for tile jt
        auto enter_tile = [&](int jt) __attribute__((always_inline)) {
            const bool plain = jt >= p0 && jt <= p1;
            if (plain && unmasked) return;
            unmasked = plain;
            const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
            static_for<U>([&](auto UN) __attribute__((always_inline)) {
                constexpr int u = decltype(UN)::value;
                const int i = kq + ln_ + d0 + u;
                const bool row_ok = i < N && d0 + u < n_units;
                // element v of this lane is key 32 * jt + 8*(v/4) + 4*hf + v%4
                const int hi = i - jt * TJ - 4 * hf_, lo = hi - w1;
                uint32_t seen = 0;                            // bit c: key 32 * jt + 4*hf + c
                if (row_ok && hi >= 0 && lo < TJ) seen = (hi >= TJ - 1 ? ~0u : (2u << hi) - 1) & (lo > 0 ? ~0u << lo : ~0u);
                if (plain) seen = ~0u;
                const int v0 = __float_as_int(-lse2[u]), v1 = __float_as_int(-INFINITY);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    int m = (int)(seen << (31 - 8 * (v >> 2) - (v & 3))) >> 31;
                    asm("" : "+v"(m));                  // (two instructions; as a comparison it is three and a wait)
                    nl[u][v] = __int_as_float((v0 & m) | (v1 & ~m));
                }
                asm volatile("s_nop 3" : "+v"(nl[u]));
            });
        };
        // tiles (from jt on) that need nothing done between them
        auto until = [&](int jt) __attribute__((always_inline)) {
            if (jt < p0 || jt > p1 || near_end) return 1;
            return (p1 < a1 ? p1 : a1) - jt + 1;
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        auto aim_ahead = [&]() __attribute__((always_inline)) {        // (for the request of the step that follows)
            if (near_end) {
                const int t = next_tile, n = next_round, z = next_last;
                static_for<4>([&](auto I) __attribute__((always_inline)) { next_piece(I, std::false_type{}); });
                aim(next_tile);
                next_tile = t;
                next_round = n;
                next_last = z;
            }
        };
        for (int jt = s0; jt <= s1;) {
            if (jt >= a0 && jt <= a1) {
                enter_tile(jt);
                aim_ahead();
                if constexpr (U == 1) single(no, no);
                else pair(no, no);
                rotate();
                ++jt;
                while (jt <= a1) {
                    enter_tile(jt);
                    aim_ahead();
                    // those of them that request within the sweep, then the others
                    const int n = until(jt), on = near_end ? 0 : n < next_last - next_tile ? n : next_last - next_tile;
                    for (int k = on; k > 0; --k) {
                        if constexpr (U == 1) single(yes, yes);
                        else pair(yes, yes);
                        rotate();
                    }
                    next_tile += on;
                    for (int k = n - on; k > 0; --k) {
                        if constexpr (U == 1) single(yes, no);
                        else pair(yes, no);
                        rotate();
                    }
                    jt += n;
                }
                if constexpr (U == 1) single_last();
                else pair_last();
                continue;
            }
            bool done = false;
            if constexpr (U > 1) {
                if (jt >= t0 && jt <= t1) {
                    enter_tile(jt);
                    half(LONE_C(0));
                    done = true;
                } else if (jt >= t2 && jt <= t3) {
                    enter_tile(jt);
                    half(LONE_C(U - 1));
                    done = true;
                }
            }
            if (!done) {
                step_barrier();
                next_request();
                request_tile(sc);
                read_first_rows(sb);
            }
            rotate();
            ++jt;
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

        // ---- sums over the units: dV'[k] += R * dO[k+delta], dK'[k] += G * q[k+delta] (scale applied at the end) ----
        static_for<U>([&](auto UN) __attribute__((always_inline)) {
            constexpr int u = decltype(UN)::value;
            if (d0 + u >= n_units) return;
            const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
            uint2 qx[4 * DT], ox[4 * DT];
#pragma unroll
            for (int e = 0; e < 4 * DT; ++e) {
                if constexpr (RAW) {
                    qx[e] = lds_row4(q_s, ln_ + d0 + u, hf_, e);
                    ox[e] = lds_row4(do_s, ln_ + d0 + u, hf_, e);
                } else {
                    qx[e] = load_cols4<false>(far_row(qp, p.q.sn, ln_ + d0 + u), e * 8 + 4 * hf_, p.D);
                    ox[e] = load_cols4<false>(far_row(dop, p.dout.sn, ln_ + d0 + u), e * 8 + 4 * hf_, p.D);
                }
            }
            auto add = [&](auto TO, auto FROM, uint2 x) __attribute__((always_inline)) {
                constexpr int to = decltype(TO)::value, from = decltype(FROM)::value;
                const float4 a = L::get_regs<to>(), g = L::get_regs<from>();
                L::set_regs<to>(__float_as_uint(a.x + g.x * E::lo(x.x)), __float_as_uint(a.y + g.y * E::hi(x.x)),
                                __float_as_uint(a.z + g.z * E::lo(x.y)), __float_as_uint(a.w + g.w * E::hi(x.y)));
            };
            static_for<4 * DT>([&](auto X) __attribute__((always_inline)) {
                constexpr int e = decltype(X)::value;
                add(LONE_C(DK0 + 4 * e), LONE_C(G0 + u * DT * 16 + 4 * e), qx[e]);
                if constexpr (DVV) {
                    constexpr int v = 4 * (e % 4), from = R0 + 4 * e;
                    const float4 g = L::get_regs<from>();
                    floatx16& to = dvv[e / 4];
                    to[v] += g.x * E::lo(ox[e].x);
                    to[v + 1] += g.y * E::hi(ox[e].x);
                    to[v + 2] += g.z * E::lo(ox[e].y);
                    to[v + 3] += g.w * E::hi(ox[e].y);
                } else {
                    add(LONE_C(DV0 + 4 * e), LONE_C(R0 + u * DT * 16 + 4 * e), ox[e]);
                }
            });
        });
        // ---- dQ[k + delta] += G * k2~[k]   The four wavefronts add into the shared fp32
        // accumulator (scale is applied when the partial is written out) in four phases; in phase t wavefront w owns the
        // 16-column blocks (w + t) % 4 (and that + 4 when D = 128), so no two wavefronts touch an element at the same time and
        // every element receives its contributions in a fixed order (a wavefront's units one after the other). ----
        if (want_dq) {
            auto add_block = [&](auto B) __attribute__((always_inline)) {
                constexpr int blk = decltype(B)::value;
                constexpr int NV = DK / 2;                    // float4 slots of a block
                const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
                float4 kt[NV];                                // (WIDE: scaled)
                // slot e of the block -> 8-column group
                static_for<NV>([&](auto SL) __attribute__((always_inline)) {
                    constexpr int e = decltype(SL)::value, g8 = 2 * (blk + 4 * (e >> 1)) + (e & 1);
                    if constexpr (WIDE) {
                        kt[e] = *(const float4*)(kt_s + ln_ * C::AS + g8 * 8 + 4 * hf_);
                    } else {
                        const uint2 x = lds_row4(k2_s, ln_, hf_, g8);
                        kt[e] = make_float4(E::lo(x.x) + p.k2_bias, E::hi(x.x) + p.k2_bias, E::lo(x.y) + p.k2_bias, E::hi(x.y) + p.k2_bias);
                    }
                });
                static_for<U>([&](auto UN) __attribute__((always_inline)) {
                    constexpr int u = decltype(UN)::value;
                    if (d0 + u >= n_units) return;
                    float* arow = dqacc + (ln_ + d0 + u) * C::AS + 4 * hf_;
                    float4 a[NV];
                    static_for<NV>([&](auto SL) __attribute__((always_inline)) {
                        constexpr int e = decltype(SL)::value, g8 = 2 * (blk + 4 * (e >> 1)) + (e & 1);
                        a[e] = *(float4*)(arow + g8 * 8);
                    });
                    static_for<NV>([&](auto SL) __attribute__((always_inline)) {
                        constexpr int e = decltype(SL)::value, g8 = 2 * (blk + 4 * (e >> 1)) + (e & 1);
                        constexpr int gr = G0 + u * DT * 16 + 4 * g8;
                        const float4 g = L::get_regs<gr>();
                        a[e].x += g.x * kt[e].x;
                        a[e].y += g.y * kt[e].y;
                        a[e].z += g.z * kt[e].z;
                        a[e].w += g.w * kt[e].w;
                        *(float4*)(arow + g8 * 8) = a[e];
                    });
                    // (the second unit's rows overlap the first one's, shifted by one: its reads must see the first
                    // unit's writes, which the same lanes' program order does not give across lanes)
                    if constexpr (U > 1) __builtin_amdgcn_wave_barrier();
                });
            };
#pragma unroll 1
            for (int t = 0; t < 4; ++t) {
                switch ((wave + t) & 3) {
                    case 0: add_block(LONE_C(0)); break;
                    case 1: add_block(LONE_C(1)); break;
                    case 2: add_block(LONE_C(2)); break;
                    default: add_block(LONE_C(3)); break;
                }
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
        }
        L::keep_out();
    }

    // ---- dQ partial of this workgroup ------------------------------------------------
    const int tid_f = here();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the last requests: LDS is reused below)
    __syncthreads();
    if (want_dq) {
        constexpr int CH = D / 4;
        float* dst = dq_part + (((int64_t)bh * nkb + kb) * nseg + seg) * RQ * D;
        for (int it = tid_f; it < RQ * CH; it += KT) {
            const int row = it / CH, c0 = (it - row * CH) * 4;
            float4 a = *(const float4*)(dqacc + row * C::AS + c0);
            const float sc_ = WIDE ? LN2 : p.scale;           // (WIDE: the sums carry scale * log2(e))
            a.x *= sc_; a.y *= sc_; a.z *= sc_; a.w *= sc_;
            *(float4*)(dst + (int64_t)row * D + c0) = a;
        }
    }
    // ---- dK' and dV': the four wavefronts' sums added through LDS ----------------
    // item -> (tensor, K' row, 8 columns); a thread's items are it = tid, tid + KT, ...
    constexpr int CHF = D / 8;
    constexpr int ITEMS = (2 * BQ * CHF + KT - 1) / KT;
    // what the pre-pass left in the output rows (the contribution of the unit delta = w2),
    // requested now so that it arrives while the wavefronts' sums go through LDS
    uint4 pre[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        pre[j] = make_uint4(0, 0, 0, 0);
        const int it = tid_f + j * KT;
        if (it >= 2 * BQ * CHF) break;
        const int which = it / (BQ * CHF);
        const int rem = it - which * BQ * CHF;
        const int row = rem / CHF, c0 = (rem - row * CHF) * 8;
        if (has_left) {
            const Tensor& t = which ? p.dk2 : p.dv2;
            if (k0 + row < N && t.p) pre[j] = *(const uint4*)((const uint16_t*)t.p + t.off(b, k0 + row, h) + c0);
        }
    }
    __syncthreads();
    {
        const int ln_f = tid_f & 31, hf_f = (tid_f >> 5) & 1;
        static_for<2 * 4 * DT>([&](auto X) __attribute__((always_inline)) {
            constexpr int x = decltype(X)::value, which = x / (4 * DT), e = x % (4 * DT), r = (which ? DV0 : DK0) + 4 * e;
            float* row = (float*)smem_raw + ((size_t)which * KW + wave) * BQ * C::AS + ln_f * C::AS + 4 * hf_f;
            if constexpr (which && DVV) *(float4*)(row + e * 8) = make_float4(dvv[e / 4][4 * (e % 4)], dvv[e / 4][4 * (e % 4) + 1], dvv[e / 4][4 * (e % 4) + 2], dvv[e / 4][4 * (e % 4) + 3]);
            else *(float4*)(row + e * 8) = L::get_regs<r>();
        });
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int it = tid_f + j * KT;
        if (it >= 2 * BQ * CHF) break;
        const int which = it / (BQ * CHF);                          // 0: dV', 1: dK'
        const int rem = it - which * BQ * CHF;
        const int row = rem / CHF, c0 = (rem - row * CHF) * 8;
        const int k = k0 + row;
        const Tensor& t = which ? p.dk2 : p.dv2;
        if (k >= N || !t.p) continue;
        float acc[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] = 0.f;
        const float* base = (const float*)smem_raw + (size_t)(which ? 0 : KW) * BQ * C::AS;
#pragma unroll
        for (int w = 0; w < KW; ++w) {
            const float* rp = base + (size_t)w * BQ * C::AS + row * C::AS + c0;
            const float4 a = *(const float4*)rp, c4 = *(const float4*)(rp + 4);
            acc[0] += a.x; acc[1] += a.y; acc[2] += a.z; acc[3] += a.w;
            acc[4] += c4.x; acc[5] += c4.y; acc[6] += c4.z; acc[7] += c4.w;
        }
        const float sc_ = which ? p.scale : 1.f;
        if (nseg > 1) {
            float* dst = kpart + ((((int64_t)which * nseg + seg) * p.B * p.H + bh) * N + k) * D + c0;
            *(float4*)dst = make_float4(acc[0] * sc_, acc[1] * sc_, acc[2] * sc_, acc[3] * sc_);
            *(float4*)(dst + 4) = make_float4(acc[4] * sc_, acc[5] * sc_, acc[6] * sc_, acc[7] * sc_);
            continue;
        }
        uint16_t* dst = (uint16_t*)t.p + t.off(b, k, h) + c0;
        const uint4 x = pre[j];                                     // zeros where the pre-pass did not run
        const float part[8] = {E::lo(x.x), E::hi(x.x), E::lo(x.y), E::hi(x.y),
                               E::lo(x.z), E::hi(x.z), E::lo(x.w), E::hi(x.w)};
        union { EL hh[8]; uint4 u; } o;
#pragma unroll
        for (int c = 0; c < 8; ++c) o.hh[c] = (EL)(acc[c] * sc_ + part[c]);
        *(uint4*)dst = o.u;
    }
}

template <class E, int D>
int launch_kp_lone_width(const Problem& p, const KpLaunch& l, hipStream_t st) {
    using C = KpLoneCfg<D>;
    const bool raw = C::raw_fits(l.plan.segw - 1), wide = C::wide_fits(l.plan.segw - 1);
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return SA2_ERR_LAUNCH_FAILED;
        hipLaunchKernelGGL(kernel, dim3((unsigned)l.total), dim3(C::T), C::lds_bytes(l.plan.segw - 1, raw, wide), st, p, l.nkb, l.total, l.dq_part, l.left,
                           l.plan.nseg, l.plan.segw, l.kpart);
        return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
    };
    if (wide) return raw ? go(mfma_bwd_kp_lone_kernel<E, D, true, true>) : go(mfma_bwd_kp_lone_kernel<E, D, false, true>);
    return raw ? go(mfma_bwd_kp_lone_kernel<E, D, true, false>) : go(mfma_bwd_kp_lone_kernel<E, D, false, false>);
}
template <class E>
int launch_kp_lone(const Problem& p, const KpLaunch& l, hipStream_t st) {
    return p.D == 128 ? launch_kp_lone_width<E, 128>(p, l, st) : launch_kp_lone_width<E, 64>(p, l, st);
}

}  // namespace
}  // namespace sa2
