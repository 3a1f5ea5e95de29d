// The 16-bit forward kernel with two units per wavefront, head_dim 64 and 128; included once per element type.  What a unit, a
// share and the pre-pass are is said in sa2_mfma_fwd.hip, whose results, launches and workspace these are.
//
// Four wavefronts hold two units (consecutive deltas) each per round and sweep the K window from the queries' own tile down, in
// 32-key tiles that go straight from global memory into a ring in LDS, three tiles ahead.  Sums and Q~ live in accumulation
// registers and the MFMAs are placed by hand (sa2_mfma_lone.h).  Per tile a wavefront computes
//   A(0), C'(1), A(1), C(0):  A: S^T = K1.Q~^T - m,  C: R^T += V1^T.exp2(S^T)  (C' of the tile before)
// with a unit's exponentials between the MFMAs of the other one: every K and V operand is read once for two units, half of the
// LDS traffic per MFMA that eight wavefronts of one unit had, and no result waits for another wavefront.  Running sums of
// R * (v2 + bias) stay in registers for all rounds and the four wavefronts are merged once, in fp32.  The K' and V' rows are
// a ring of 64 rows in LDS, of which a round needs 39 and eight new ones: any K' window.
//
// At head_dim 128 a wavefront has a SIMD to itself (504 registers).  At head_dim 64 it needs 256 and two workgroups share a CU: one
// computes under the prologue, the forming of Q~ and the merge of the other, and scalar, LDS and vector instructions of one issue
// beside those of the other (one workgroup per CU: 176 us where two take 146, B2 H8 N2048 w 512/31).
// What bounds it: the instructions beside the MFMAs (sa2_mfma_lone.h: four of them are free under each).  A tile has 32 (head_dim
// 128) or 16 MFMAs and 145 or 110 others.  Forward, bf16: B1 H16 N8192 D128 w 512/32 1274 -> 1174 us, B2 H8 N2048 D64 w 512/31
// 180 -> 146, B1 H16 N4096 D64 w 64/31 153 -> 98, B2 H4 N512 D64 w 256/256 128 -> 100.  (A(0) taken in turn
// with C'(0), A(1) with C'(1), so that no MFMA follows the one it adds to: 2 % slower at head_dim 128.)
#pragma once

#include "sa2_mfma_fwd_lone_plan.h"
#include "sa2_mfma_lone.h"

namespace sa2 {
namespace {

// The first pass keeps one reference point per row and wavefront: the largest logit of its first two units in the queries' own
// tile, which holds a key of every row (fp16: and in the tile before, since a weight must stay below 65504).  A row whose sum
// is not finite afterwards sends the workgroup through the SAFE pass.  At head_dim 64 every unit has a reference point of its own there,
// which follows the maxima; the first 32 queries, whose windows are a single tile, take that pass at once: their few weights are
// rounded less often so (a unit's largest one is 1).  At head_dim 128, where the eight-wavefront kernel takes the first queries
// (FwdLoneCfg::FIRST_ELSEWHERE), a sweep of the logit MFMAs alone finds the largest logit of a row in both units, and the sweep of
// the first pass follows from that point, with explicit masks where a tile needs them.  (Following the maxima there, a wavefront
// alone on its SIMD ran MFMAs, exponentials and the rescaling of sums one after the other, and the second pass cost more than that of
// the eight-wavefront kernel.)  A block that has found a sum that is not finite gives the first pass up two rounds later.
// Forward, us, eight wavefronts / maxima followed / this; fp16 B1 H16 N8192 D128 w 512/32, q, k1 and k2 N(0, std^2): std 1 (no second
// pass) 1324 / 1249 / 1259, 1.25 2206 / 1644 / 1463, 1.5 3287 / 4368 / 2836, 2 and more 3274 / 4608 / 2942; bf16, std 2 1268 / 1196 / 1192,
// 3 3167 / 4563 / 2886.  fp16 B2 H8 N2048 D64 w 512/32, std 2 582 / 559 / 492 (maxima followed: rescaling costs two wavefronts per SIMD less).
template <class E, int D, bool SAFE, bool SPLIT>
__device__ __forceinline__ bool fwd_lone_block(const Problem& p, int nqb, int total, int left) {
    typedef typename E::scalar EL;
    typedef typename E::x8 X8;
    typedef typename E::x2 X2;
    using C = FwdLoneCfg<D>;
    using L = Lone<C::OWNED>;
    using T = typename C::Tile;
    constexpr int U = C::U, KW = C::W, KT = C::T, UPR = KW * U, DK = C::DK, DT = C::DT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    unsigned char* k2_s = smem_raw + C::K2_AT;                // K' rows, ring
    unsigned char* v2_s = smem_raw + C::V2_AT;                // V' rows, ring
    float* q_s = (float*)(smem_raw + C::Q_AT);                // q rows * scale * log2(e), fp32
    float* xch_m = (float*)(smem_raw + C::X_AT);              // [KW][BQ] reference points
    float* xch_l = xch_m + KW * BQ;                           // [KW][BQ] sums
    float* lam_s = xch_l + KW * BQ;                           // [BQ] reference point of the pre-pass partial
    int* given_up = (int*)(smem_raw + C::UP_AT);              // [round % 2] a sum of the block is not finite

    auto here = [&]() __attribute__((always_inline)) {        // (lane parts of what happens once per round are computed there)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    const int tid = here();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;

    int pid = xcd_order(blockIdx.x, total), share = 0;
    if constexpr (SPLIT) {
        share = pid % p.nsplit;
        pid /= p.nsplit;
    }
    const int bh = pid / nqb, qb = pid - bh * nqb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    if (qb == 0 && C::FIRST_ELSEWHERE) return false;
    if (qb == 0 && !SAFE) return true;
    const int i0 = qb * BQ, i_last = i0 + BQ - 1 < N - 1 ? i0 + BQ - 1 : N - 1;

    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* k1p = (const uint16_t*)p.k1.p + p.k1.off(b, 0, h);
    const uint16_t* k2p = (const uint16_t*)p.k2.p + p.k2.off(b, 0, h);
    const uint16_t* v1p = (const uint16_t*)p.v1.p + p.v1.off(b, 0, h);
    const uint16_t* v2p = (const uint16_t*)p.v2.p + p.v2.off(b, 0, h);

    const bool has_left = left && i_last >= w2;               // the pre-pass took the unit delta = w2
    const int n_units = (w2 < i_last ? w2 : i_last) + 1 - (has_left ? 1 : 0);
    const int all_rounds = (n_units + UPR - 1) / UPR;
    const int per_share = SPLIT ? ((w2 + UPR) / UPR + p.nsplit - 1) / p.nsplit : all_rounds;
    const int round0 = SPLIT ? share * per_share : 0;
    const int round1 = round0 + per_share < all_rounds ? round0 + per_share : all_rounds;
    if constexpr (SPLIT) {
        if (round0 >= round1) {                               // a block near the start of the sequence has fewer rounds
            if (tid < BQ && i0 + tid < N) {
                const int64_t rows = (int64_t)p.B * p.H * N;
                ((float2*)p.scratch)[share * rows + (int64_t)bh * N + i0 + tid] = make_float2(-INFINITY, 0.f);
            }
            return false;
        }
    }
    // tiles of every sweep, from jt_hi down to jt_lo; [p_lo, jt_hi - 1] need no mask
    const int jt_hi = qb, jt_lo = (i0 - w1 > 0 ? i0 - w1 : 0) / TJ;
    const int p_lo = i0 + BQ - 1 - w1 > 0 ? (i0 + BQ - 1 - w1 + TJ - 1) / TJ : 0;

    // ---- tiles: wavefront w requests groups w, w + 4 of both, straight into LDS, in the order of the sweeps ----
    const uint32_t lds0 = lds_address(smem_raw);
    const bool near_end = i0 + BQ > N;                        // (the first tile's rows past the end read the last one)
    uint32_t k_off[C::NREQ], v_off[C::NREQ];                  // byte offset of the lane's chunk from a tile's first row
    int next_tile = jt_hi, wrap = 0;
    const int64_t k_step = (int64_t)TJ * 2 * p.k1.sn, v_step = (int64_t)TJ * 2 * p.v1.sn;
    const char *const k_top = (const char*)k1p + jt_hi * k_step, *const v_top = (const char*)v1p + jt_hi * v_step;
    const char *k_next = k_top, *v_next = v_top;              // first rows of the next tile
    auto aim = [&](int jt) __attribute__((always_inline)) {
        const int l = here() & 63, col = T::dma_chunk(l) * 8;
        const int last = jt == jt_hi && near_end ? N - 1 - i0 : TJ - 1;
#pragma unroll
        for (int x = 0; x < C::NREQ; ++x) {
            const int t_row = (wave + KW * x) * T::RPW + T::dma_row(l), r = t_row < last ? t_row : last;
            k_off[x] = ((uint32_t)r * (uint32_t)p.k1.sn + col) * 2u;
            v_off[x] = ((uint32_t)r * (uint32_t)p.v1.sn + col) * 2u;
        }
    };
    auto request_k = [&](auto X, uint32_t stage) __attribute__((always_inline)) {
        lds_request(k_next, k_off[decltype(X)::value], stage + (uint32_t)((wave + KW * decltype(X)::value) * T::GROUP));
    };
    auto request_v = [&](auto X, uint32_t stage) __attribute__((always_inline)) {
        lds_request(v_next, v_off[decltype(X)::value], stage + (uint32_t)((wave + KW * decltype(X)::value) * T::GROUP) + C::TILE_BYTES);
    };
    auto request_tile = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<C::NREQ>([&](auto X) __attribute__((always_inline)) { request_k(X, stage); });
        static_for<C::NREQ>([&](auto X) __attribute__((always_inline)) { request_v(X, stage); });
    };
    // The tile after the one requested last (the sweeps follow each other; what is requested behind the last one nothing
    // reads).  In pieces that ride on MFMAs: scalar instructions cost a wavefront as much as vector ones.  ON: within a sweep
    // (the caller counts next_tile down).
    auto next_piece = [&](auto I, auto ON) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        if constexpr (decltype(ON)::value) {
            if constexpr (i == 1) k_next -= k_step;
            if constexpr (i == 2) v_next -= v_step;
        } else {
            if constexpr (i >= 0 && i < 3) {                  // (no piece moves up to another)
                next_tile = __builtin_amdgcn_readfirstlane(next_tile);
                asm volatile("" : "+s"(next_tile));
            }
            if constexpr (i == 0) {
                wrap = next_tile == jt_lo;
                next_tile = wrap ? jt_hi : next_tile - 1;
            } else if constexpr (i == 1) {
                k_next = wrap ? k_top : k_next - k_step;
            } else if constexpr (i == 2) {
                v_next = wrap ? v_top : v_next - v_step;
            }
        }
    };
    auto next_request = [&]() __attribute__((always_inline)) {
        static_for<3>([&](auto I) __attribute__((always_inline)) { next_piece(I, std::false_type{}); });
        if (near_end) aim(next_tile);
    };
    auto aim_ahead = [&]() __attribute__((always_inline)) {   // (for the request of the step that follows)
        if (near_end) aim(next_tile == jt_lo ? jt_hi : next_tile - 1);
    };
    constexpr int INFLIGHT = 2 * C::NREQ;                     // requests of one tile (two tiles are under way)
    auto step_barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(INFLIGHT) : "memory");
    };

    // ---- K' and V' rows: row k at slot (k - i0 + 7) % 64, so that a round's eight new rows are whole groups ----
    constexpr int SLOTS = C::SLOTS;
    auto request_octet = [&](int rel) __attribute__((always_inline)) {              // rel = k - i0 + 7 of the first, a multiple of 8
        constexpr int GP = 8 / T::RPW;                        // groups of eight rows
        if (wave < 2 * GP) {
            const int l = here() & 63, g = wave % GP;
            const bool vs = wave >= GP;
            const int k = i0 - 7 + rel + g * T::RPW + T::dma_row(l), kc = k < 0 ? 0 : (k < N ? k : N - 1);
            const uint16_t* src = (vs ? v2p + (int64_t)kc * p.v2.sn : k2p + (int64_t)kc * p.k2.sn) + T::dma_chunk(l) * 8;
            const int group = (rel & (SLOTS - 1)) / T::RPW + g;
            lds_request(src, lds0 + (uint32_t)((vs ? C::V2_AT : C::K2_AT) + group * T::GROUP));
        }
    };
    auto slot_of = [&](int ln_, int delta) __attribute__((always_inline)) { return (ln_ + 7 - delta) & (SLOTS - 1); };
    auto lds_row8 = [&](const unsigned char* rows, int r, int hf_, int kk) __attribute__((always_inline)) {
        return *(const uint4*)(rows + T::row_at(0, (uint32_t)(T::row_off(r) + (hf_ ^ T::flip(r)) * 16), kk));
    };
    auto lds_row4 = [&](const unsigned char* rows, int r, int hf_, int e) __attribute__((always_inline)) {
        return *(const uint2*)(rows + T::row_off(r) + e / 4 * T::BLOCK + (e % 4 ^ T::flip(r)) * 16 + hf_ * 8);
    };

    bool bad = false;
    {
        constexpr int CPR = D / 8, NQ = BQ * CPR / KT;        // 16-byte chunks of a row; of q per thread
        uint4 qx[NQ];
#pragma unroll
        for (int x = 0; x < NQ; ++x) {
            const int c = tid + x * KT, row = c / CPR, r = i0 + row < N ? i0 + row : N - 1;
            qx[x] = *(const uint4*)(qp + (int64_t)r * p.q.sn + c % CPR * 8);
        }
        float lam = 0.f;
        if (has_left) lam = p.lse[(int64_t)bh * N + (i0 + (tid & 31) < N ? i0 + (tid & 31) : N - 1)];
        aim(next_tile);
        for (int x = 4; x >= -1; --x) request_octet(8 * (x - round0));
        request_tile(lds0);
#pragma unroll 1
        for (int x = 1; x < C::NSTAGE - 1; ++x) {
            next_request();
            request_tile(lds0 + x * C::STAGE_BYTES);
        }
        if (tid < 2) given_up[tid] = 0;
        const float qscale = p.scale * LOG2E;
#pragma unroll
        for (int x = 0; x < NQ; ++x) {
            const int c = tid + x * KT;
            float* to = q_s + c / CPR * C::QS + c % CPR * 8;
            *(float4*)to = make_float4(E::lo(qx[x].x) * qscale, E::hi(qx[x].x) * qscale, E::lo(qx[x].y) * qscale, E::hi(qx[x].y) * qscale);
            *(float4*)(to + 4) = make_float4(E::lo(qx[x].z) * qscale, E::hi(qx[x].z) * qscale, E::lo(qx[x].w) * qscale, E::hi(qx[x].w) * qscale);
        }
        if (has_left && tid < BQ) {
            bad = !(lam == lam);                              // the pre-pass overflowed: the block takes its second pass
            lam_s[tid] = lam;
        }
    }
    const uint32_t row_lane = T::row_lane(lane), col_lane = T::column_lane(lane);            // row, transposed operand

    // ---- a wavefront's sweep.  Accumulation registers: R tiles of the units, then Q~ as B operands ----
    constexpr int R0 = 0, Q0 = U * DT * 16;
    static_assert(Q0 + U * DK * 4 <= C::OWNED, "");
    constexpr int NE = DK;                                    // MFMAs of a phase
    static_assert(NE == 2 * DT, "");
    X8 ka[DK], vt[DT][2];                                     // row operands of the K tile, transposed ones of the V tile
    floatx16 s[U], nl;                                        // logits; -m of the lane's row, -inf where the key is outside the window
    u4 pw[U][2];                                              // weights in 16 bits
    float l[U], rs[U];                                        // sums of the weights: of the sweep, of the tile
    floatx16 wacc[DT];                                        // sum of R * (v2 + bias) over the wavefront's units
    float Mw = -INFINITY, Lw = 0.f;                           // its reference point and sum of weights
    uint32_t sc = lds0 + (C::NSTAGE - 1) * C::STAGE_BYTES, sa = lds0, sb = lds0 + C::STAGE_BYTES, sd = lds0 + 2 * C::STAGE_BYTES;      // stages of tiles t-1, t, t+1, t+2
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) wacc[dt][v] = 0.f;
    const X2 one = {(EL)1.f, (EL)1.f};

    auto read_row = [&](auto KK, uint32_t stage) __attribute__((always_inline)) {
        ka[decltype(KK)::value] = lds_read_x8<X8>(T::row_at(stage, row_lane, decltype(KK)::value));
    };
    auto read_column = [&](auto X, uint32_t stage) __attribute__((always_inline)) {          // in the order of the C phase
        constexpr int ks = decltype(X)::value / DT, dt = decltype(X)::value % DT;
        vt[dt][ks] = quad_tile_column<D, X8>(stage + C::TILE_BYTES, col_lane, dt, ks);
    };
    auto a_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, at = Q0 + (u * DK + i) * 4;
        if constexpr (i == 0) L::template tile_start<at>(s[u], ka[0], nl);
        else L::template tile_more<at>(s[u], ka[i]);
    };
    auto logit_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {         // (from zero)
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, at = Q0 + (u * DK + i) * 4;
        if constexpr (i == 0) L::template tile_start<at>(s[u], ka[0]);
        else L::template tile_more<at>(s[u], ka[i]);
    };
    auto c_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, ks = decltype(I)::value / DT, dt = decltype(I)::value % DT;
        L::template sum_more<R0 + (u * DT + dt) * 16>(vt[dt][ks], __builtin_bit_cast(X8, pw[u][ks]));
    };
    // Softmax items of a unit: item i forms one exponential, and of the pair before it a rounded pair or its share of the sum (an
    // exponential's result may not be read by the next instruction); the last two end both.
    constexpr int ITEMS = 18;
    auto item = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value;
        if constexpr (i < 16) {
            float x = fast_exp2(s[u][i]);
            stays(x);
            s[u][i] = x;
        }
        constexpr int pair = i / 2 - 1;
        if constexpr (pair >= 0 && i % 2 == 0) {
            uint32_t w = pack2<E>(s[u][2 * pair], s[u][2 * pair + 1]);
            stays(w);
            pw[u][pair / 4][pair % 4] = w;
        } else if constexpr (pair >= 0) {
            float r = E::dot2(__builtin_bit_cast(X2, (uint32_t)pw[u][pair / 4][pair % 4]), one, pair == 0 ? 0.f : rs[u], false);
            stays(r);
            rs[u] = r;
        }
        if constexpr (i == ITEMS - 1) {
            l[u] += rs[u];
            stays(l[u]);
        }
    };
    // A tile in four phases, A(t, 0), C(t-1, 1), A(t, 1), C(t, 0).  A unit's softmax lies behind MFMAs 2 .. of the phase after its
    // A, all of the next phase, and MFMAs 0 and 1 of its C (whose second half needs the second half of the weights).
    constexpr int NS = 2 * NE;
    auto softmax = [&](auto UN, auto SLOT) __attribute__((always_inline)) {
        deal<ITEMS, decltype(SLOT)::value, NS>([&](auto X) __attribute__((always_inline)) { item(UN, X); });
    };
    auto step = [&](auto DO_C, auto ON) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;            // (the first tile of a sweep has no tile before it)
        static_for<NE>([&](auto I) __attribute__((always_inline)) {                 // A(t, 0)
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(0), I);
            next_piece(LONE_C(i - 1), ON);
            if constexpr (CC) softmax(LONE_C(1), LONE_C(NE - 2 + i));
            else read_column(I, sa);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (CC) {
            static_for<NE>([&](auto I) __attribute__((always_inline)) {             // C(t-1, 1)
                constexpr int i = decltype(I)::value;
                c_mfma(LONE_C(1), I);
                if constexpr (i >= 2) read_column(LONE_C(i - 2), sa);               // (the MFMA that read its register is past)
                if constexpr (i < 2) softmax(LONE_C(1), LONE_C(2 * NE - 2 + i));
                if constexpr (i >= 2) softmax(LONE_C(0), LONE_C(i - 2));
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        static_for<NE>([&](auto I) __attribute__((always_inline)) {                 // A(t, 1)
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(1), I);
            if constexpr (CC && i < 2) read_column(LONE_C(NE - 2 + i), sa);
            if constexpr (CC) softmax(LONE_C(0), LONE_C(NE - 2 + i));
            else deal<ITEMS, i - 2, NE - 2>([&](auto X) __attribute__((always_inline)) { item(LONE_C(0), X); });
            __builtin_amdgcn_sched_barrier(0);
        });
        // (no wait for reads of LDS: what is requested into, the stage of tile t-1, was last read by MFMAs that have been issued)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(INFLIGHT) : "memory");
        static_for<NE>([&](auto I) __attribute__((always_inline)) {                 // C(t, 0)
            constexpr int i = decltype(I)::value;
            c_mfma(LONE_C(0), I);
            read_row(I, sb);
            if constexpr (CC && i < 2) softmax(LONE_C(0), LONE_C(2 * NE - 2 + i));
            if constexpr (i >= 2) softmax(LONE_C(1), LONE_C(i - 2));
            if constexpr (i % 2 == 1) {
                deal<2 * C::NREQ, i / 2, NE / 2>([&](auto X) __attribute__((always_inline)) {
                    constexpr int x = decltype(X)::value;
                    if constexpr (x < C::NREQ) request_k(LONE_C(x), sc);
                    else request_v(LONE_C(x - C::NREQ), sc);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        stays(s[1]);
    };
    auto last_step = [&]() __attribute__((always_inline)) {                         // C(t, 1) of the last tile
        static_for<NE + 2>([&](auto I) __attribute__((always_inline)) { softmax(LONE_C(1), LONE_C(NE - 2 + decltype(I)::value)); });
        stays(l[1]);
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(1), I); });
    };
    auto rotate = [&]() __attribute__((always_inline)) {
        L::keep_out();
        const uint32_t x = sc;
        sc = sa;
        sa = sb;
        sb = sd;
        sd = x;
    };
    // keys of tile jt inside the window of the lane's row: bit c is key 32 * jt + 4*hf + c, element v of a tile is key 8*(v/4) + v%4 + 4*hf
    auto keys_seen = [&](int jt) __attribute__((always_inline)) {
        const int t = here(), ln_ = t & 31, hf_ = t >> 5 & 1;
        const int hi = i0 + ln_ - jt * TJ - 4 * hf_, lo = hi - w1;
        uint32_t seen = 0;
        if (hi >= 0 && lo < TJ) seen = (hi >= TJ - 1 ? ~0u : (2u << hi) - 1) & (lo > 0 ? ~0u << lo : ~0u);
        return seen;
    };
    bool unmasked = false;
    float round_max = -INFINITY;                              // (second pass at head_dim 128) reference point of the round's units
    auto enter_tile = [&](int jt) __attribute__((always_inline)) {                  // the start of the S tiles of tile jt
        const bool plain = jt >= p_lo && jt < jt_hi;
        if (plain && unmasked) return;
        unmasked = plain;
        const uint32_t seen = plain ? ~0u : keys_seen(jt);
        const float ref = SAFE ? round_max : Mw;
        const int v0 = ref == -INFINITY ? 0 : __float_as_int(-ref), v1 = __float_as_int(-INFINITY);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            int m = (int)(seen << (31 - 8 * (v >> 2) - (v & 3))) >> 31;
            asm("" : "+v"(m));                                // (two instructions; as a comparison it is three and a wait)
            nl[v] = __int_as_float((v0 & m) | (v1 & ~m));
        }
        asm volatile("s_nop 3" : "+v"(nl));
    };
    // the units' logits in the tile whose row operands are in `ka` and their largest ones, where the lane's row has a key; the others
    // become -inf
    auto tile_logits = [&](int jt, int d0, float (&mx)[U]) __attribute__((always_inline)) {
        const int t = here(), i = i0 + (t & 31);
        const uint32_t seen = keys_seen(jt);
#pragma unroll
        for (int v = 0; v < 16; ++v) nl[v] = 0.f;
        asm volatile("s_nop 3" : "+v"(nl));
        static_for<U * NE>([&](auto I) __attribute__((always_inline)) { a_mfma(LONE_C(decltype(I)::value / NE), LONE_C(decltype(I)::value % NE)); });
        finished(s[0], s[1]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool row = i < N && i >= d0 + u && d0 + u < n_units;
            float m = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[u][v] = row && (seen >> (8 * (v >> 2) + (v & 3)) & 1) ? s[u][v] : -INFINITY;
                m = fmaxf(m, s[u][v]);
            }
            mx[u] = fmaxf(m, other_half(m));
        }
    };

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    X8 zero;
#pragma unroll
    for (int t = 0; t < 8; ++t) zero[t] = (EL)0.f;
    static_for<DK>([&](auto KK) __attribute__((always_inline)) { read_row(KK, sa); });

    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    for (int round = round0; round < round1; ++round) {
        // A block that takes the second pass gives up the first one: what was written at the end of the round before the last
        // one all wavefronts see alike, since every round has a barrier.
        if (!SAFE && __builtin_amdgcn_readfirstlane(given_up[round & 1])) break;
        const int d0 = round * UPR + wave * U;                // first delta of this wavefront
        const bool any = d0 < n_units;
        request_octet(-8 * (round + 2));                      // (landed two tiles from now; their slots hold rows of no round from the last one on)
        // ---- Q~ of the round's units (one that does not exist: its neighbour's, and left out of the sums) ----
        asm volatile("s_nop 3" : "+v"(zero));
        static_for<U * DT>([&](auto X) __attribute__((always_inline)) { L::template sum_zero<R0 + 16 * decltype(X)::value>(zero); });
        {
            const int t = here(), ln_ = t & 31, hf_ = t >> 5 & 1;
            const float* qrow = q_s + ln_ * C::QS + hf_ * 8;
            int slot[U];
#pragma unroll
            for (int u = 0; u < U; ++u) slot[u] = slot_of(ln_, d0 + u < n_units ? d0 + u : n_units - 1);
            auto form = [&](auto BIASED) __attribute__((always_inline)) {
                const float kb = decltype(BIASED)::value ? p.k2_bias : 0.f;
                static_for<DK>([&](auto KK) __attribute__((always_inline)) {
                    constexpr int kk = decltype(KK)::value;
                    const float4 qa = *(const float4*)(qrow + kk * 16), qc = *(const float4*)(qrow + kk * 16 + 4);
                    static_for<U>([&](auto UN) __attribute__((always_inline)) {
                        constexpr int u = decltype(UN)::value, at = Q0 + (u * DK + kk) * 4;
                        const uint4 k = lds_row8(k2_s, slot[u], hf_, kk);
                        L::template set_regs<at>(pack2<E>(qa.x * (E::lo(k.x) + kb), qa.y * (E::hi(k.x) + kb)),
                                                 pack2<E>(qa.z * (E::lo(k.y) + kb), qa.w * (E::hi(k.y) + kb)),
                                                 pack2<E>(qc.x * (E::lo(k.z) + kb), qc.y * (E::hi(k.z) + kb)),
                                                 pack2<E>(qc.z * (E::lo(k.w) + kb), qc.w * (E::hi(k.w) + kb)));
                    });
                });
            };
            if (p.k2_bias != 0.f) form(std::true_type{});
            else form(std::false_type{});
        }
#pragma unroll
        for (int u = 0; u < U; ++u) l[u] = 0.f;
        L::keep_out();
        asm volatile("s_nop 3" ::: "memory");

        if (!any) {
            // no unit for this wavefront in this round: keep the requests moving
            for (int jt = (SAFE && C::MAXIMA_FIRST ? 2 : 1) * (jt_hi - jt_lo + 1); jt > 0; --jt) {
                step_barrier();
                next_request();
                request_tile(sc);
                rotate();
            }
            continue;
        }
        float mu[U];                                          // (SAFE) reference points of the units
        // (SAFE) the tile whose logits `tile_logits` left: weights of a unit from its reference point, sums of both, the next tile's rows
        auto weigh = [&](auto UN, float m0) __attribute__((always_inline)) {
#pragma unroll
            for (int v = 0; v < 16; ++v) s[decltype(UN)::value][v] -= m0;
            static_for<ITEMS>([&](auto X) __attribute__((always_inline)) { item(UN, X); });
        };
        auto tile_sums = [&]() __attribute__((always_inline)) {
            static_for<NE>([&](auto X) __attribute__((always_inline)) { read_column(X, sa); });
            asm volatile("s_nop 7" ::: "memory");
            static_for<U * NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(decltype(I)::value / NE), LONE_C(decltype(I)::value % NE)); });
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        };
        auto next_rows = [&]() __attribute__((always_inline)) {
            step_barrier();
            next_request();
            request_tile(sc);
            static_for<DK>([&](auto KK) __attribute__((always_inline)) { read_row(KK, sb); });
            rotate();
        };
        if constexpr (SAFE && C::MAXIMA_FIRST) {
            // a sweep for the largest logit of the row in both units, then the sweep of the first pass where no tile needs a mask
            float top[U], mx[U];
#pragma unroll
            for (int u = 0; u < U; ++u) top[u] = -INFINITY;
            for (int jt = jt_hi; jt >= jt_lo; --jt) {
                if (jt == jt_hi || jt < p_lo) {
                    tile_logits(jt, d0, mx);
#pragma unroll
                    for (int u = 0; u < U; ++u) top[u] = fmaxf(top[u], mx[u]);
                    next_rows();
                    continue;
                }
                static_for<NE>([&](auto I) __attribute__((always_inline)) {
                    logit_mfma(LONE_C(0), I);
                    __builtin_amdgcn_sched_barrier(0);
                });
                step_barrier();
                next_request();
                request_tile(sc);
                static_for<NE>([&](auto I) __attribute__((always_inline)) {
                    constexpr int i = decltype(I)::value;
                    logit_mfma(LONE_C(1), I);
                    if constexpr (i >= 2) read_row(LONE_C(i - 2), sb);              // (the MFMA that read its register is past)
                    deal<16, i - 2, NE - 2>([&](auto X) __attribute__((always_inline)) { top[0] = fmaxf(top[0], s[0][decltype(X)::value]); });
                    __builtin_amdgcn_sched_barrier(0);
                });
                finished(s[0], s[1]);
                static_for<2>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(NE - 2 + decltype(X)::value), sb); });
#pragma unroll
                for (int v = 0; v < 16; ++v) top[1] = fmaxf(top[1], s[1][v]);
                rotate();
            }
            const int row = i0 + (here() & 31);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float m = fmaxf(top[u], other_half(top[u]));
                top[u] = row < N && row >= d0 + u && d0 + u < n_units ? m : -INFINITY;
            }
            round_max = fmaxf(top[0], top[1]);
            const float ref = round_max == -INFINITY ? 0.f : round_max;
#pragma unroll
            for (int u = 0; u < U; ++u) mu[u] = round_max;
            unmasked = false;
            for (int jt = jt_hi; jt >= jt_lo;) {
                if (jt == jt_hi || jt < p_lo) {
                    tile_logits(jt, d0, mx);
                    static_for<U>([&](auto UN) __attribute__((always_inline)) { weigh(UN, ref); });
                    tile_sums();
                    next_rows();
                    --jt;
                    continue;
                }
                enter_tile(jt);
                aim_ahead();
                step(no, no);
                rotate();
                for (--jt; jt >= p_lo && jt >= jt_lo; --jt) {
                    aim_ahead();
                    step(yes, no);
                    rotate();
                }
                last_step();
                asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
            }
        } else if constexpr (SAFE) {
#pragma unroll
            for (int u = 0; u < U; ++u) mu[u] = -INFINITY;
            for (int jt = jt_hi; jt >= jt_lo; --jt) {
                float mx[U];
                tile_logits(jt, d0, mx);
                static_for<U>([&](auto UN) __attribute__((always_inline)) {
                    constexpr int u = decltype(UN)::value;
                    const float mn = fmaxf(mu[u], mx[u]), m0 = mn == -INFINITY ? 0.f : mn, alpha = fast_exp2(mu[u] - m0);
                    mu[u] = mn;
                    l[u] *= alpha;
                    static_for<DT * 4>([&](auto X) __attribute__((always_inline)) {
                        constexpr int r = R0 + u * DT * 16 + 4 * decltype(X)::value;
                        const float4 x = L::template get_regs<r>();
                        L::template set_regs<r>(__float_as_uint(x.x * alpha), __float_as_uint(x.y * alpha), __float_as_uint(x.z * alpha), __float_as_uint(x.w * alpha));
                    });
                    weigh(UN, m0);
                });
                tile_sums();
                next_rows();
            }
        } else {
            if (round == round0) {
                float mx[U];
                tile_logits(jt_hi, d0, mx);
                Mw = fmaxf(mx[0], mx[1]);
                if constexpr (E::DTYPE == SA2_F16) {
                    if (jt_lo < jt_hi) {
                        static_for<DK>([&](auto KK) __attribute__((always_inline)) { read_row(KK, sb); });
                        tile_logits(jt_hi - 1, d0, mx);
                        Mw = fmaxf(Mw, fmaxf(mx[0], mx[1]));
                        static_for<DK>([&](auto KK) __attribute__((always_inline)) { read_row(KK, sa); });
                    }
                }
            }
            unmasked = false;
            enter_tile(jt_hi);
            aim_ahead();
            step(no, no);
            rotate();
            for (int jt = jt_hi - 1; jt >= jt_lo;) {
                enter_tile(jt);
                aim_ahead();
                // tiles that need nothing done between them, and those of them that request within the sweep
                const int n = jt < p_lo || near_end ? 1 : jt - p_lo + 1, on = near_end ? 0 : (n < next_tile - jt_lo ? n : next_tile - jt_lo);
                int k = on;
                for (; C::UNROLL && k >= 4; k -= 4) {                      // (after four the stages are where they were)
                    static_for<4>([&](auto) __attribute__((always_inline)) {
                        step(yes, yes);
                        rotate();
                    });
                }
                for (; k > 0; --k) {
                    step(yes, yes);
                    rotate();
                }
                next_tile -= on;
                for (k = n - on; k > 0; --k) {
                    step(yes, no);
                    rotate();
                }
                jt -= n;
            }
            last_step();
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        }

        // ---- the units join the wavefront's running result: sum += weight * (v2 + bias) * R ----
        {
            const int t = here(), ln_ = t & 31, hf_ = t >> 5 & 1, i = i0 + ln_;
            auto join = [&](auto UN, auto ALL, auto WEIGHED, float c) __attribute__((always_inline)) {
                constexpr int u = decltype(UN)::value;
                const bool row = decltype(ALL)::value || (i < N && i >= d0 + u && d0 + u < n_units);
                const float lt = l[u] + other_half(l[u]);
                Lw += row ? (decltype(WEIGHED)::value ? c * lt : lt) : 0.f;
                bad |= row && !(lt < 1e30f);
                const int slot = slot_of(ln_, d0 + u < n_units ? d0 + u : n_units - 1);
                uint2 x[4 * DT];
#pragma unroll
                for (int e = 0; e < 4 * DT; ++e) x[e] = lds_row4(v2_s, slot, hf_, e);
                static_for<4 * DT>([&](auto X) __attribute__((always_inline)) {
                    constexpr int e = decltype(X)::value, v = 4 * (e % 4);
                    float4 r = L::template get_regs<R0 + u * DT * 16 + 4 * e>();
                    const uint2 w = x[e];
                    if constexpr (!decltype(ALL)::value) r = row ? r : make_float4(0.f, 0.f, 0.f, 0.f);
                    if constexpr (decltype(WEIGHED)::value) r = make_float4(c * r.x, c * r.y, c * r.z, c * r.w);
                    floatx16& to = wacc[e / 4];
                    to[v] += r.x * (E::lo(w.x) + p.v2_bias);
                    to[v + 1] += r.y * (E::hi(w.x) + p.v2_bias);
                    to[v + 2] += r.z * (E::lo(w.y) + p.v2_bias);
                    to[v + 3] += r.w * (E::hi(w.y) + p.v2_bias);
                });
            };
            if constexpr (SAFE) {
                const float mn = fmaxf(Mw, fmaxf(mu[0], mu[1])), m0 = mn == -INFINITY ? 0.f : mn, a = fast_exp2(Mw - m0);
                Mw = mn;
                Lw *= a;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int v = 0; v < 16; ++v) wacc[dt][v] *= a;
                static_for<U>([&](auto UN) __attribute__((always_inline)) { join(UN, no, yes, fast_exp2(mu[decltype(UN)::value] - m0)); });
            } else if (i0 >= d0 + U - 1 && i0 + BQ <= N && d0 + U <= n_units) {
                static_for<U>([&](auto UN) __attribute__((always_inline)) { join(UN, yes, no, 1.f); });
            } else {
                static_for<U>([&](auto UN) __attribute__((always_inline)) { join(UN, no, no, 1.f); });
            }
            if (!SAFE && __builtin_amdgcn_ballot_w64(bad)) {
                if ((t & 63) == 0) given_up[round & 1] = 1;
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // (a sweep's barriers do not wait for it)
            }
        }
        L::keep_out();
    }

    // ---- merge the four wavefronts and the pre-pass partial, whose sum is 1 at its reference point ----
    const int tid_m = here(), ln_m = tid_m & 31, hf_m = tid_m >> 5 & 1;
    constexpr int TPR = KT / BQ, ACN = D / TPR;               // threads per row, columns per thread
    const int aq = tid_m / TPR, ac = tid_m % TPR * ACN, io = i0 + aq;
    uint4 part[ACN / 8];
#pragma unroll
    for (int c = 0; c < ACN / 8; ++c) {
        part[c] = make_uint4(0, 0, 0, 0);
        if (has_left) part[c] = *(const uint4*)((const uint16_t*)p.out.p + p.out.off(b, io < N ? io : N - 1, h) + ac + 8 * c);
    }
    if (hf_m == 0) {
        xch_m[wave * BQ + ln_m] = Mw;
        xch_l[wave * BQ + ln_m] = Lw;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the last requests: the sums go over the rings)
    __syncthreads();
    auto reference = [&](int row) __attribute__((always_inline)) {
        float mx = has_left ? lam_s[row] : -INFINITY;
#pragma unroll
        for (int w = 0; w < KW; ++w) mx = fmaxf(mx, xch_m[w * BQ + row]);
        return mx;
    };
    float* sums = (float*)smem_raw;                           // [KW][BQ][AS]
    {
        const float cw = Mw == -INFINITY ? 0.f : fast_exp2(Mw - reference(ln_m));
        float* row = sums + (wave * BQ + ln_m) * C::AS + 4 * hf_m;
#pragma unroll
        for (int e = 0; e < 4 * DT; ++e) {
            const floatx16& a = wacc[e / 4];
            const int v = 4 * (e % 4);
            *(float4*)(row + 8 * e) = make_float4(cw * a[v], cw * a[v + 1], cw * a[v + 2], cw * a[v + 3]);
        }
    }
    const float Ms = reference(aq), Mu = Ms == -INFINITY ? 0.f : Ms;
    const float al = has_left && lam_s[aq] > -INFINITY ? fast_exp2(lam_s[aq] - Mu) : 0.f;
    float Ls = al;
#pragma unroll
    for (int w = 0; w < KW; ++w) {
        const float mw = xch_m[w * BQ + aq];
        Ls += xch_l[w * BQ + aq] * (mw == -INFINITY ? 0.f : fast_exp2(mw - Mu));             // (NaN logits: Mw -inf, Lw NaN)
    }
    const bool again = __syncthreads_or(bad ? 1 : 0) && !SAFE;
    float acc[ACN];
#pragma unroll
    for (int c = 0; c < ACN / 8; ++c) {
        const uint4 x = part[c];
        const float y[8] = {E::lo(x.x), E::hi(x.x), E::lo(x.y), E::hi(x.y), E::lo(x.z), E::hi(x.z), E::lo(x.w), E::hi(x.w)};
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[8 * c + t] = has_left ? al * y[t] : 0.f;
    }
#pragma unroll
    for (int w = 0; w < KW; ++w)
#pragma unroll
        for (int c = 0; c < ACN; c += 4) {
            const float4 a = *(const float4*)(sums + (w * BQ + aq) * C::AS + ac + c);
            acc[c] += a.x; acc[c + 1] += a.y; acc[c + 2] += a.z; acc[c + 3] += a.w;
        }
    if (again) return true;                                   // (uniform over the workgroup; the pre-pass left nothing that is read again)
    if (io < N) {
        if constexpr (SPLIT) {
            const int64_t rows = (int64_t)p.B * p.H * N, row = share * rows + (int64_t)bh * N + io;
            float* to = (float*)p.scratch + 2 * rows * p.nsplit + row * D + ac;
#pragma unroll
            for (int c = 0; c < ACN; c += 2) *(float2*)(to + c) = make_float2(acc[c], acc[c + 1]);
            if (tid_m % TPR == 0) ((float2*)p.scratch)[row] = make_float2(Ms, Ls);
            return false;
        }
        const float inv = 1.f / (Ls + 1e-8f * fast_exp2(-Ms));
        uint16_t* to = (uint16_t*)p.out.p + p.out.off(b, io, h) + ac;
#pragma unroll
        for (int c = 0; c < ACN; c += 8) {
            union { EL e[8]; uint4 u; } o;
#pragma unroll
            for (int t = 0; t < 8; ++t) o.e[t] = (EL)(acc[c + t] * inv);
            *(uint4*)(to + c) = o.u;
        }
        if (tid_m % TPR == 0) {
            float lse;
            if (Ms > LOG2_EPS) lse = LN2 * (Ms + __log2f(Ls + 1e-8f * fast_exp2(-Ms)));
            else lse = LN_EPS + log1pf(Ls * fast_exp2(Ms - LOG2_EPS));
            p.lse[(int64_t)bh * N + io] = lse;
        }
    }
    return false;
}

// (one argument: it starts the kernel argument segment, from which the second pass reads it again)
template <class E, int D, bool SPLIT>
__global__ __launch_bounds__(FwdLoneCfg<D>::T) __attribute__((amdgpu_waves_per_eu(FwdLoneCfg<D>::PER_SIMD, FwdLoneCfg<D>::PER_SIMD)))
void mfma_fwd_lone_kernel(FwdLoneArgs args) {
    if (fwd_lone_block<E, D, false, SPLIT>(args.p, args.nqb, args.total, args.left)) {        // (uniform over the workgroup)
        __syncthreads();
        typedef const __attribute__((address_space(4))) FwdLoneArgs* arg_ptr;
        arg_ptr segment = (arg_ptr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(segment));
        const FwdLoneArgs* again = (const FwdLoneArgs*)segment;
        fwd_lone_block<E, D, true, SPLIT>(again->p, again->nqb, again->total, 0);
    }
}

template <class E, int D>
int launch_fwd_lone_width(const FwdLoneArgs& args, hipStream_t st) {
    using C = FwdLoneCfg<D>;
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return SA2_ERR_LAUNCH_FAILED;
        hipLaunchKernelGGL(kernel, dim3((unsigned)args.total), dim3(C::T), C::LDS_BYTES, st, args);
        return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
    };
    if constexpr (C::FIRST_ELSEWHERE) return args.p.nsplit > 1 ? SA2_ERR_UNSUPPORTED : go(mfma_fwd_lone_kernel<E, D, false>);
    else return args.p.nsplit > 1 ? go(mfma_fwd_lone_kernel<E, D, true>) : go(mfma_fwd_lone_kernel<E, D, false>);
}
template <class E>
int launch_fwd_lone(const FwdLoneArgs& args, hipStream_t st) {
    return args.p.D == 128 ? launch_fwd_lone_width<E, 128>(args, st) : launch_fwd_lone_width<E, 64>(args, st);
}

}  // namespace
}  // namespace sa2
