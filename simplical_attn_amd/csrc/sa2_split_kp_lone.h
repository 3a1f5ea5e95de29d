// The K'-side backward kernel (dQ, dK' and dV') of the plane-split kernels with one wavefront per SIMD; included once per element
// type.  Arithmetic, partials and segments are those of split_kp_kernel (sa2_split_mfma.hip), which says what a unit and a plane are.
//
// A workgroup owns 32 K' rows k0 .. and a run of deltas.  Four wavefronts hold one unit each per round, as planes in accumulation
// registers (sa2_mfma_lone.h), and sweep the K/V window in 32-key tiles.  Per tile and unit a wavefront computes
//   A: S^T = K1.Q~^T - LSE and dP^T = V1.dO~^T - D,   B: P = exp2(S), dS = P * dP, both split into planes,   C: R^T += V1^T.P^T and G^T += K1^T.dS^T
// with C of the tile before and B between the MFMAs, in the order of the K-side kernel (sa2_split_kv_lone.h, which also says how a tile
// of planes lies in LDS and what NU is).  Tiles of one plane come straight from global memory, three ahead, into a ring of four;
// others are split by all threads between the MFMAs, one tile ahead, from registers that were requested a tile before, into a ring of three.
#pragma once

#include "sa2_split_kp_lone_plan.h"
#include "sa2_split_lone.h"

namespace sa2 {
namespace {

// RAW: the q and dO rows lie in LDS (SplitKpLoneCfg::main_bytes)
template <class T, int D, int NU, int MODE, bool RAW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void split_kp_lone_kernel(Problem p, int nkb, int per_seg, float* __restrict__ dq_part, int nseg, int segw, float* __restrict__ kpart) {
    using C = SplitKpLoneCfg<D, T::PLANES>;
    using L = Lone<256>;
    typedef typename T::T EL;
    typedef typename T::Raw Raw;
    typedef bf16x8 X8;
    constexpr bool PAD = MODE != EXACT;
    constexpr int DK = C::DK, DT = C::DT, NK = C::NK, KW = C::W, KT = C::THREADS;
    constexpr int CHUNK = 16 / (int)sizeof(EL);               // elements of a 16-byte chunk
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int RQ = BQ + segw - 1, RQ4 = (RQ + 3) & ~3;        // query rows this workgroup touches
    unsigned char* k2_s = smem_raw + C::NSTAGE * C::STAGE;    // K' rows k0 .. k0+31
    unsigned char* v2_s = k2_s + C::row_bytes(BQ);            // V' rows
    unsigned char* q_s = v2_s + C::row_bytes(BQ);             // q rows kq ..  (RAW)
    unsigned char* do_s = q_s + C::row_bytes(RQ);             // dO rows       (RAW)
    float* lse_s = (float*)(RAW ? do_s + C::row_bytes(RQ) : q_s);
    float* dsum_s = lse_s + RQ4;
    float* dqacc = dsum_s + RQ4;                              // [RQ][AS]

    auto here = [&]() __attribute__((always_inline)) {        // (lane parts of what happens once per round are computed there)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    const int seg = (int)blockIdx.x / per_seg;                // (segment-major launch order: see split_kp_kernel)
    const int pid = xcd_order((int)blockIdx.x - seg * per_seg, per_seg);
    const int bh = pid / nkb, kb = pid - bh * nkb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int k0 = kb * BQ, dlo = seg * segw, kq = k0 + dlo;  // kq: query of K' row k0 at the segment's first delta
    const bool want_dq = p.dq.p != nullptr;

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k1p = (const EL*)p.k1.p + p.k1.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v1p = (const EL*)p.v1.p + p.v1.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);
    const EL* dop = (const EL*)p.dout.p + p.dout.off(b, 0, h);
    const float qscale = p.scale * LOG2E;

    const int nu_all = (w2 < N - 1 - k0 ? w2 : N - 1 - k0) + 1;            // deltas with k0 + delta < N
    const int n_units = nu_all - dlo < segw ? nu_all - dlo : segw;         // of this segment (may be <= 0)
    const int nrounds = n_units > 0 ? (n_units + KW - 1) / KW : 0;
    // tiles a round sweeps: from the first tile of its smallest delta to the last tile of its largest one
    auto round_first = [&](int round) __attribute__((always_inline)) {
        const int i_min = kq + round * KW;
        return (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
    };
    auto round_last = [&](int round) __attribute__((always_inline)) {
        const int dl = (round + 1) * KW - 1 < n_units - 1 ? (round + 1) * KW - 1 : n_units - 1;
        const int i_max = kq + dl + BQ - 1 < N - 1 ? kq + dl + BQ - 1 : N - 1;
        return i_max / TJ;
    };

    // ---- tiles, in the order of the sweeps (behind the last one: that one again, which nothing reads) ----
    const uint32_t lds0 = lds_address(smem_raw);
    int next_round = 0, next_tile = round_first(0), next_last = round_last(0);
    auto next = [&]() __attribute__((always_inline)) {
        if (next_tile < next_last) {
            ++next_tile;
        } else if (next_round + 1 < nrounds) {
            ++next_round;
            next_tile = round_first(next_round);
            next_last = round_last(next_round);
        }
    };
    // one plane: straight to LDS.  A wavefront instruction brings 16 rows of 64 bytes; the tile's are dealt over the wavefronts.
    constexpr int PIECES = 2 * DT, NREQ = C::DMA ? 2 * PIECES / KW : 0;    // pieces of a tile; requests of a wavefront for both tiles
    static_assert(!C::DMA || 2 * PIECES % KW == 0, "");
    const bool near_end = N % TJ != 0;                        // (a tile whose rows past the end read the last one)
    int64_t piece_off[C::DMA ? NREQ : 1];                     // bytes from the tile's first row to the lane's chunk
    auto aim = [&](int jt) __attribute__((always_inline)) {
        const int l = here() & 63;
#pragma unroll
        for (int n = 0; n < NREQ; ++n) {
            const int piece = wave + KW * n, vs = piece >= PIECES, x = piece - vs * PIECES;        // (uniform)
            const int row = 16 * (x & 1) + (l >> 2), col = (x >> 1) * 32 + ((l & 3) ^ (l >> 4 & 3)) * 8, most = N - 1 - jt * TJ;
            // (columns from p.D on meet zeros of the unit, or are not written)
            piece_off[n] = ((row < most ? row : most) * (vs ? p.v1.sn : p.k1.sn) + (PAD && col >= p.D ? 0 : col)) * (int64_t)sizeof(EL);
        }
    };
    auto request_piece = [&](auto X, uint32_t stage) __attribute__((always_inline)) {
        constexpr int n = decltype(X)::value;
        const int piece = wave + KW * n, vs = piece >= PIECES, x = piece - vs * PIECES;
        const char* base = (const char*)(vs ? v1p + (int64_t)next_tile * TJ * p.v1.sn : k1p + (int64_t)next_tile * TJ * p.k1.sn);
        lds_request(base + piece_off[n], stage + (uint32_t)(vs * C::TILE + (x >> 1) * C::BLOCK + (x & 1) * 1024));
    };
    auto request_tile = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<NREQ>([&](auto X) __attribute__((always_inline)) { request_piece(X, stage); });
    };
    // more planes: through registers.  Thread t brings the columns 32*dt + 4*(t % 8) .. of row t / 8.
    const int s_row = tid >> 3, s_col = (tid & 7) * 4;
    const uint32_t s_lane = (uint32_t)(s_row * 64 + (((tid & 7) >> 1) ^ (s_row >> 2 & 3)) * 16 + (tid & 1) * 8);
    Raw tk[DT], tv[DT];
    auto load_tile = [&]() __attribute__((always_inline)) {
        const int j = next_tile * TJ + s_row < N ? next_tile * TJ + s_row : N - 1;
        const EL *ks = k1p + (int64_t)j * p.k1.sn, *vs = v1p + (int64_t)j * p.v1.sn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            tk[dt] = raw4<T, PAD>(ks, dt * 32 + s_col, p.D);
            tv[dt] = raw4<T, PAD>(vs, dt * 32 + s_col, p.D);
        }
    };
    // item f: two columns of the K or V tile, in steps of up to five instructions
    constexpr int NF = C::DMA ? 0 : 4 * DT, STEPS = 2 * NK - 1;
    uint32_t fw[NK][2];
    float fa[2], fh[2];
    auto stage_step = [&](auto X, uint32_t to) __attribute__((always_inline)) {
        constexpr int f = decltype(X)::value / STEPS, m = decltype(X)::value % STEPS, dt = f / 4, which = f / 2 % 2, e = f % 2 * 2;
        if constexpr (m == 0) {
            const fx4 y = T::widen(which ? tv[dt] : tk[dt]);
            fa[0] = y[e];
            fa[1] = y[e + 1];
            constexpr float MOST = 3.3895313892515355e38f;    // (see split2)
            const uint32_t w = T::DTYPE == SA2_F32 ? pack2(__builtin_amdgcn_fmed3f(fa[0], -MOST, MOST), __builtin_amdgcn_fmed3f(fa[1], -MOST, MOST)) : pack2(fa[0], fa[1]);
            fw[0][e / 2] = w;
            stays(fw[0][e / 2]);
        } else if constexpr (m % 2 == 1) {
            fh[0] = bf16_lo(fw[m / 2][e / 2]);
            fh[1] = bf16_hi(fw[m / 2][e / 2]);
            stays(fh[0]);
            stays(fh[1]);
        } else {
            fa[0] -= fh[0];
            fa[1] -= fh[1];
            fw[m / 2][e / 2] = pack2(fa[0], fa[1]);
            stays(fw[m / 2][e / 2]);
        }
        if constexpr (m == STEPS - 1 && e == 2) {
#pragma unroll
            for (int n = 0; n < NK; ++n)
                *(ux2 __attribute__((address_space(3)))*)(uintptr_t)(to + (uint32_t)(which * C::TILE + n * C::PLANE + dt * C::BLOCK)) = ux2{fw[n][0], fw[n][1]};
        }
    };
    auto stage_all = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<NF * STEPS>([&](auto X) __attribute__((always_inline)) { stage_step(X, stage + s_lane); });
    };

    // ---- rows: 16-byte chunk c of row r of a copy in LDS (laid out as a tile of 256-byte rows, sa2_mfma_common.h) ----
    using Q4 = QuadTile<128>;
    auto chunk = [&](const unsigned char* rows, int r, int c) __attribute__((always_inline)) {
        return rows + Q4::row_off(r) + c / 4 * Q4::BLOCK + c % 4 * 16;
    };
    auto request_rows = [&](const EL* base, int64_t sn, int first, int rows, const unsigned char* to) __attribute__((always_inline)) {
        const int l = here() & 63, col = Q4::dma_chunk(l) * CHUNK;
        for (int g = wave; g * Q4::RPW < rows; g += KW) {
            const int r = first + g * Q4::RPW + Q4::dma_row(l), rc = r < N ? r : N - 1;
            const void* src = col < p.D ? (const void*)(base + (int64_t)rc * sn + col) : (const void*)zero_chunk;
            lds_request(src, lds0 + (uint32_t)(to - smem_raw) + (uint32_t)(g * Q4::GROUP));
        }
    };
    // four columns from 8*e + 4*hf on of a row of a copy; of the q (0) or dO (1) row kq + rel
    auto copy4 = [&](const unsigned char* rows, int r, int hf_, int e) __attribute__((always_inline)) {
        if constexpr (sizeof(EL) == 4) return *(const Raw*)chunk(rows, r, 2 * e + hf_);
        else return *(const Raw*)(chunk(rows, r, e) + hf_ * 8);
    };
    auto unit4 = [&](int which, int rel, int hf_, int e) __attribute__((always_inline)) {
        if constexpr (RAW) return copy4(which ? do_s : q_s, rel, hf_, e);
        else {
            const int64_t i = kq + rel < N ? kq + rel : N - 1;
            return raw4<T, PAD>(which ? dop + i * p.dout.sn : qp + i * p.q.sn, 8 * e + 4 * hf_, p.D);
        }
    };
    // eight columns from 16*kk + 8*hf on, as two groups of four
    struct Eight { Raw a, c; };
    auto copy8 = [&](const unsigned char* rows, int r, int hf_, int kk) __attribute__((always_inline)) {
        if constexpr (sizeof(EL) == 4) {
            const unsigned char* at = chunk(rows, r, 4 * kk + 2 * hf_);
            return Eight{*(const Raw*)at, *(const Raw*)(at + 16)};
        } else {
            const uint4 x = *(const uint4*)chunk(rows, r, 2 * kk + hf_);
            return Eight{__builtin_bit_cast(Raw, make_uint2(x.x, x.y)), __builtin_bit_cast(Raw, make_uint2(x.z, x.w))};
        }
    };
    auto unit8 = [&](int which, int rel, int hf_, int kk) __attribute__((always_inline)) {
        if constexpr (RAW) return copy8(which ? do_s : q_s, rel, hf_, kk);
        else {
            const int64_t i = kq + rel < N ? kq + rel : N - 1;
            const EL* row = which ? dop + i * p.dout.sn : qp + i * p.q.sn;
            return Eight{raw4<T, PAD>(row, 16 * kk + 8 * hf_, p.D), raw4<T, PAD>(row, 16 * kk + 8 * hf_ + 4, p.D)};
        }
    };
    auto row_value = [&](const float* of, int c) __attribute__((always_inline)) { return of[(int64_t)bh * N + (kq + c < N ? kq + c : N - 1)]; };
    {
        request_rows(k2p, p.k2.sn, k0, BQ, k2_s);
        request_rows(v2p, p.v2.sn, k0, BQ, v2_s);
        if constexpr (RAW) {
            request_rows(qp, p.q.sn, kq, RQ, q_s);
            request_rows(dop, p.dout.sn, kq, RQ, do_s);
        }
        if (nrounds > 0) {
            if constexpr (C::DMA) {
                aim(next_tile);
                request_tile(lds0);
                for (int x = 1; x < C::NSTAGE - 1; ++x) {
                    next();
                    if (near_end) aim(next_tile);
                    request_tile(lds0 + x * C::STAGE);
                }
            } else {
                load_tile();
                stage_all(lds0);
                next();
                load_tile();
            }
        }
        for (int c = tid; c < RQ * (C::AS / 4); c += KT) ((float4*)dqacc)[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int c = tid; c < RQ; c += KT) {
            lse_s[c] = row_value(p.lse, c);
            dsum_s[c] = row_value(p.dsum, c);
        }
    }

    // ---- a wavefront's sweep ----
    // accumulation registers: R and G tiles, Q~ and dO~ as planes of B operands, LSE and D as one each, dK' and dV' where there is room
    constexpr int R0 = 0, G0 = DT * 16, Q0 = 2 * DT * 16, O0 = Q0 + NU * DK * 4, LS0 = O0 + NU * DK * 4, LD0 = LS0 + 4, DK0 = LD0 + 4, DV0 = DK0 + DT * 16;
    constexpr bool DKA = DK0 + DT * 16 <= 256, DVA = DV0 + DT * 16 <= 256;
    static_assert(DK0 <= 256, "");
    floatx16 dkv[DKA ? 1 : DT], dvv[DVA ? 1 : DT];
#pragma unroll
    for (int dt = 0; dt < (DKA ? 1 : DT); ++dt) dkv[dt] = zero16();
#pragma unroll
    for (int dt = 0; dt < (DVA ? 1 : DT); ++dt) dvv[dt] = zero16();
    constexpr Products<NK, NU> PA;                            // plane of the tile, of the unit
    constexpr Products<NK, 3> PC;                             // plane of the tile, of P or dS
    constexpr int NP = PA.n, NC = PC.n;
    constexpr int CH = NP * DK + 1;                           // MFMAs of a chain of phase A (the last one takes LSE or D off)
    constexpr int NG = DT * NC;                               // MFMAs of a quarter of phase C: one half of the keys, R or G
    constexpr int NA = 2 * CH, NS = NA + 4 * NG;
    constexpr int AHEAD = NP >= 5 ? 1 : NP == 3 ? 2 : 3;      // k-steps that row operands are read ahead
    constexpr int BEHIND = NC >= 5 ? 1 : 3;                   // column blocks that transposed operands are read ahead
    X8 ro[AHEAD + 1][NK], co[BEHIND + 1][NK];
    floatx16 s, dp, nl;                                       // nl: what a chain of S starts from, -inf where the pair is outside the windows
    u4 pw[2][3], dw[2][3];
    const X8 ones = lead_ones(hf);
    uint32_t sa = lds0, sb = lds0 + C::STAGE, sc = lds0 + (C::NSTAGE - 1) * C::STAGE, sd = lds0 + 2 * C::STAGE;      // stages of tiles t, t+1, t-1 and (four) t+2
    const uint32_t row_lane = (uint32_t)(ln * 64 + (hf ^ (ln >> 2 & 3)) * 16);
    const uint32_t col_lane = [&]() {
        const int grp = lane >> 4, x = lane & 15, r = 4 * (grp >> 1) + (x >> 2), c = 2 * (grp & 1) + ((x & 3) >> 1);
        return (uint32_t)(r * 64 + (c ^ (r >> 2)) * 16 + (x & 1) * 8);
    }();
    static_assert(C::STAGE % 64 == 0, "");
    uint32_t r0 = 0, r1 = 0, c0 = 0, c1 = 0;                  // the lane's addresses in a stage, for even and odd k-steps and slices of eight rows
    auto at_stage = [&](uint32_t stage, uint32_t part, uint32_t& even, uint32_t& odd) __attribute__((always_inline)) {
        even = stage + part;
        odd = even ^ 32u;
        stays(even);
        stays(odd);
    };
    // entry e of phase A: k-step e % DK of S (K tile) or dP (V tile)
    auto read_row = [&](auto EN, auto X) __attribute__((always_inline)) {
        constexpr int e = decltype(EN)::value, x = decltype(X)::value, which = e / DK, kk = e % DK;
        ro[e % (AHEAD + 1)][x] = lds_read_x8<X8>((kk & 1 ? r1 : r0) + (uint32_t)(which * C::TILE + x * C::PLANE + kk / 2 * C::BLOCK));
    };
    auto read_first_rows = [&](uint32_t stage) __attribute__((always_inline)) {
        at_stage(stage, row_lane, r0, r1);
        static_for<AHEAD * NK>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(decltype(X)::value / NK), LONE_C(decltype(X)::value % NK)); });
    };
    // entry e of phase C: quarter e / DT (R's halves, from the V tile, then G's), column block e % DT
    auto read_column = [&](auto EN, auto X) __attribute__((always_inline)) {
        constexpr int e = decltype(EN)::value, x = decltype(X)::value, which = e / (2 * DT), ks = e / DT % 2, dt = e % DT;
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef v4s __attribute__((address_space(3)))* lds_v4s;
        constexpr uint32_t at = (which ? 0 : C::TILE) + x * C::PLANE + dt * C::BLOCK + ks * 1024;
        union { v4s half[2]; X8 v; } u;
        u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c0 + at));
        u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c1 + at + 512));
        co[e % (BEHIND + 1)][x] = u.v;
    };
    auto a_mfma = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value, which = i / CH, m = i % CH;
        if constexpr (m == CH - 1) {
            if constexpr (which) L::template tile_more<LD0>(dp, ones);
            else L::template tile_more<LS0>(s, ones);
        } else {
            constexpr int kk = m / NP, x = PA.x[m % NP], y = PA.y[m % NP], e = which * DK + kk, at = (which ? O0 : Q0) + (y * DK + kk) * 4;
            const X8& a = ro[e % (AHEAD + 1)][x];
            if constexpr (which) {
                if constexpr (m == 0) L::template tile_start<at>(dp, a);
                else L::template tile_more<at>(dp, a);
            } else {
                if constexpr (m == 0) L::template tile_start<at>(s, a, nl);
                else L::template tile_more<at>(s, a);
            }
        }
    };
    auto c_mfma = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value, e = i / NC, which = e / (2 * DT), ks = e / DT % 2, dt = e % DT, x = PC.x[i % NC], y = PC.y[i % NC];
        if constexpr (which) L::template sum_more<G0 + dt * 16>(co[e % (BEHIND + 1)][x], __builtin_bit_cast(X8, dw[ks][y]));
        else L::template sum_more<R0 + dt * 16>(co[e % (BEHIND + 1)][x], __builtin_bit_cast(X8, pw[ks][y]));
    };
    auto exp_item = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        float x = fast_exp2(NU == 2 ? s[i] * qscale : s[i]);
        stays(x);
        s[i] = x;
    };
    auto ds_item = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        float x = s[i] * dp[i];
        stays(x);
        dp[i] = x;
    };
    float sh[2];
    auto split_step = [&](floatx16& of, u4 (&to)[3], auto KS, auto I) __attribute__((always_inline)) { split_word_step<decltype(KS)::value, decltype(I)::value>(of, to, sh); };
    // The barrier of a tile: tile t+1 is in LDS for all, and tile t-1, whose stage is used again, was read to the end.
    constexpr int BAR = NS - 6, STAGED = NK == 1 ? 0 : BAR - 8 - 2 * NG;      // its slot; the slot by which tile t+1 is staged
    static_assert((BEHIND + 1) * NC - NK + 1 > 6, "the last transposed operands are requested before the barrier");
    auto tile_barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::DMA ? NREQ : 63) : "memory"); };
    auto beside = [&](auto SLOT, auto DO_C, uint32_t stage_at) __attribute__((always_inline)) {
        constexpr int slot = decltype(SLOT)::value;
        if constexpr (decltype(DO_C)::value) within<16, slot, 1, CH - 1>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[1], LONE_C(1), X); });
        within<16, slot, CH + 2, NA + 1>(exp_item);
        within<16, slot, NA + 2, NA + NG>(ds_item);
        within<16, slot, NA + NG, NA + 2 * NG>([&](auto X) __attribute__((always_inline)) { split_step(s, pw[0], LONE_C(0), X); });
        within<16, slot, NA + 2 * NG, NA + 3 * NG>([&](auto X) __attribute__((always_inline)) { split_step(s, pw[1], LONE_C(1), X); });
        within<16, slot, NA + 3 * NG, NS>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[0], LONE_C(0), X); });
        if constexpr (!C::DMA) {
            within<NF * STEPS, slot, 0, STAGED>([&](auto X) __attribute__((always_inline)) { stage_step(X, stage_at); });
            if constexpr (slot == STAGED) {
                next();
                load_tile();
            }
        }
    };
    // the tile at sa, and C of the one before it
    auto tile = [&](auto DO_C) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        uint32_t stage_at = sb + s_lane;
        if constexpr (!C::DMA) stays(stage_at);
        if constexpr (CC) at_stage(sc, col_lane, c0, c1);
        static_for<NA>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / CH * DK + i % CH / NP, m = i % CH % NP;
            a_mfma(I);
            if constexpr (i % CH < CH - 1 && e + AHEAD < 2 * DK) deal<NK, m, NP>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(e + AHEAD), X); });
            constexpr int first = NA - BEHIND * NK;
            if constexpr (CC && i >= first) read_column(LONE_C((i - first) / NK), LONE_C((i - first) % NK));
            beside(I, DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) finished(s, dp);
        static_for<4 * NG>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / NC, m = i % NC, slot = NA + i;
            if constexpr (slot == BAR) {
                tile_barrier();
                at_stage(sb, row_lane, r0, r1);
            }
            if constexpr (CC) {
                c_mfma(I);
                if constexpr (e + BEHIND < 4 * DT && m < NK) read_column(LONE_C(e + BEHIND), LONE_C(m));
            }
            if constexpr (slot >= BAR && slot < BAR + AHEAD * NK) read_row(LONE_C((slot - BAR) / NK), LONE_C((slot - BAR) % NK));
            if constexpr (C::DMA) {
                if constexpr (slot == BAR) {
                    next();
                    if (near_end) aim(next_tile);
                }
                if constexpr (slot > BAR) deal<NREQ, slot - BAR - 1, NS - BAR - 1>([&](auto X) __attribute__((always_inline)) { request_piece(X, sc); });
            }
            beside(LONE_C(NA + i), DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto last_sums = [&]() __attribute__((always_inline)) {                         // C of tile t-1 alone
        static_for<16>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[1], LONE_C(1), X); });
        at_stage(sc, col_lane, c0, c1);
        static_for<BEHIND * NK>([&](auto X) __attribute__((always_inline)) { read_column(LONE_C(decltype(X)::value / NK), LONE_C(decltype(X)::value % NK)); });
        static_for<4 * NG>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / NC, m = i % NC;
            c_mfma(I);
            if constexpr (e + BEHIND < 4 * DT && m < NK) read_column(LONE_C(e + BEHIND), LONE_C(m));
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto idle = [&]() __attribute__((always_inline)) {                              // a tile that holds no key of this wavefront's unit
        if constexpr (!C::DMA) {
            stage_all(sb);
            next();
            load_tile();
        }
        tile_barrier();
        if constexpr (C::DMA) {
            next();
            if (near_end) aim(next_tile);
            request_tile(sc);
        }
    };
    auto rotate = [&]() __attribute__((always_inline)) {
        L::keep_out();
        const uint32_t x = sc;
        sc = sa;
        sa = sb;
        if constexpr (C::NSTAGE == 4) {
            sb = sd;
            sd = x;
        } else {
            sb = x;
        }
    };

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    X8 zero;
#pragma unroll
    for (int t = 0; t < 8; ++t) zero[t] = (__bf16)0.f;
    if constexpr (DKA) static_for<DT * 4>([&](auto X) __attribute__((always_inline)) { L::template set_regs<DK0 + 4 * decltype(X)::value>(0u, 0u, 0u, 0u); });
    if constexpr (DVA) static_for<DT * 4>([&](auto X) __attribute__((always_inline)) { L::template set_regs<DV0 + 4 * decltype(X)::value>(0u, 0u, 0u, 0u); });

    for (int round = 0; round < nrounds; ++round) {
        const int d0 = round * KW + wave;                     // this wavefront's delta, relative to the segment
        const bool any = d0 < n_units;
        const int delta = any ? d0 : n_units - 1;             // (one that does not exist: its neighbour's, and left out of all sums)
        asm volatile("s_nop 3" : "+v"(zero));
        static_for<2 * DT>([&](auto X) __attribute__((always_inline)) { L::template sum_zero<16 * decltype(X)::value>(zero); });
        {
            const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1, u = ln_ + delta;
            // the product row x * mul * (y + bias) of eight columns as NU planes (two: x * y), as in product_planes
            auto form = [&](auto KK, auto AT, const Eight& x, const Eight& y, float bias, float mul) __attribute__((always_inline)) {
                const fx4 xa = T::widen(x.a), xc = T::widen(x.c), ya = T::widen(y.a), yc = T::widen(y.c);
                float r[8];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    r[t] = NU == 2 ? xa[t] * ya[t] : xa[t] * mul * (ya[t] + bias);
                    r[4 + t] = NU == 2 ? xc[t] * yc[t] : xc[t] * mul * (yc[t] + bias);
                }
                X8 o[NU];
                split8<NU>(r, o);
                static_for<NU>([&](auto Y) __attribute__((always_inline)) {
                    const u4 w = __builtin_bit_cast(u4, o[decltype(Y)::value]);
                    L::template set_regs<decltype(AT)::value + (decltype(Y)::value * DK + decltype(KK)::value) * 4>(w[0], w[1], w[2], w[3]);
                });
            };
            Eight qx[DK], ox[DK];                             // all reads of the two rows first
#pragma unroll
            for (int kk = 0; kk < DK; ++kk) {
                qx[kk] = unit8(0, u, hf_, kk);
                ox[kk] = unit8(1, u, hf_, kk);
            }
            static_for<DK>([&](auto KK) __attribute__((always_inline)) {
                form(KK, LONE_C(Q0), qx[decltype(KK)::value], copy8(k2_s, ln_, hf_, decltype(KK)::value), p.k2_bias, qscale);
                form(KK, LONE_C(O0), ox[decltype(KK)::value], copy8(v2_s, ln_, hf_, decltype(KK)::value), p.v2_bias, 1.f);
            });
            float lse = lse_s[u], x = NU == 2 ? lse / p.scale : lse * LOG2E;
            stays(x);                                         // (rounded: taken together with the split, the rest would count twice)
            const u4 a = __builtin_bit_cast(u4, lead_planes(x, NU == 2 ? fmaf(-x, p.scale, lse) / p.scale : lse_rest(lse, x)));
            const u4 c = __builtin_bit_cast(u4, lead_planes(dsum_s[u], 0.f));
            L::template set_regs<LS0>(a[0], a[1], a[2], a[3]);
            L::template set_regs<LD0>(c[0], c[1], c[2], c[3]);
        }
        L::keep_out();

        // ---- the sweep: tiles [t0, t1] hold keys of the unit, [p0, p1] need no mask ----
        const int s0 = round_first(round), s1 = round_last(round);
        int t0 = 1, t1 = 0, p0 = 1, p1 = 0;
        if (any) {
            const int i_min = kq + delta, i_max = i_min + BQ - 1 < N - 1 ? i_min + BQ - 1 : N - 1;
            t0 = (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
            t1 = i_max / TJ;
            p0 = i_max - w1 > 0 ? (i_max - w1 + TJ - 1) / TJ : 0;
            p1 = i_min + BQ - 1 < N ? (i_min + 1) / TJ - 1 : -1;
        }
        bool unmasked = false;
        auto enter_tile = [&](int jt) __attribute__((always_inline)) {              // the start of the S tile for tile jt
            const bool plain = jt >= p0 && jt <= p1;
            if (plain && unmasked) return;
            unmasked = plain;
            const int l = here(), i = kq + (l & 31) + d0;
            // element v of this lane is key 32 * jt + 8*(v/4) + 4*hf + v%4
            const int hi = i - jt * TJ - 4 * (l >> 5 & 1), lo = hi - w1;
            uint32_t seen = 0;                                // bit c: key 32 * jt + 4*hf + c
            if (i < N && hi >= 0 && lo < TJ) seen = (hi >= TJ - 1 ? ~0u : (2u << hi) - 1) & (lo > 0 ? ~0u << lo : ~0u);
            if (plain) seen = ~0u;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                int m = (int)(seen << (31 - 8 * (v >> 2) - (v & 3))) >> 31;
                asm("" : "+v"(m));
                nl[v] = __int_as_float(__float_as_int(-INFINITY) & ~m);
            }
            asm volatile("s_nop 3" : "+v"(nl));
        };
        for (int jt = s0; jt <= s1;) {
            if (jt < t0 || jt > t1) {
                idle();
                rotate();
                ++jt;
                continue;
            }
            read_first_rows(sa);
            enter_tile(jt);
            tile(std::false_type{});
            rotate();
            for (++jt; jt <= t1;) {
                enter_tile(jt);
                const int n = jt < p0 || jt > p1 ? 1 : (p1 < t1 ? p1 : t1) - jt + 1;           // tiles that need nothing done between them
                for (int k = n; k > 0; --k) {
                    tile(std::true_type{});
                    rotate();
                }
                jt += n;
            }
            last_sums();
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

        // ---- sums over the units: dV'[k] += R * dO[k+delta], dK'[k] += G * q[k+delta] (scale applied at the end) ----
        if (any) {
            const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
            Raw qx[4 * DT], ox[4 * DT];
#pragma unroll
            for (int e = 0; e < 4 * DT; ++e) {
                qx[e] = unit4(0, ln_ + d0, hf_, e);
                ox[e] = unit4(1, ln_ + d0, hf_, e);
            }
            auto add = [&](auto E_, auto FROM, auto TO, auto IN_ACC, floatx16* v, const Raw& x) __attribute__((always_inline)) {
                constexpr int e = decltype(E_)::value;
                const float4 g = L::template get_regs<decltype(FROM)::value + 4 * e>();
                const fx4 y = T::widen(x);
                if constexpr (decltype(IN_ACC)::value) {
                    const float4 a = L::template get_regs<decltype(TO)::value + 4 * e>();
                    L::template set_regs<decltype(TO)::value + 4 * e>(__float_as_uint(a.x + g.x * y[0]), __float_as_uint(a.y + g.y * y[1]),
                                                                      __float_as_uint(a.z + g.z * y[2]), __float_as_uint(a.w + g.w * y[3]));
                } else {
                    floatx16& to = v[e / 4];
                    to[4 * (e % 4)] += g.x * y[0];
                    to[4 * (e % 4) + 1] += g.y * y[1];
                    to[4 * (e % 4) + 2] += g.z * y[2];
                    to[4 * (e % 4) + 3] += g.w * y[3];
                }
            };
            static_for<4 * DT>([&](auto X) __attribute__((always_inline)) {
                add(X, LONE_C(G0), LONE_C(DK0), std::integral_constant<bool, DKA>{}, dkv, qx[decltype(X)::value]);
                add(X, LONE_C(R0), LONE_C(DV0), std::integral_constant<bool, DVA>{}, dvv, ox[decltype(X)::value]);
            });
        }
        // ---- dQ[k + delta] += G * k2~[k], in four phases: in phase t wavefront w owns the columns 8*((w + t) % 4) .. of every 32-column
        // block, so no two wavefronts touch an element at the same time and every element sums in a fixed order ----
        if (want_dq) {
            auto add_block = [&](auto B) __attribute__((always_inline)) {
                if (!any) return;
                const int l = here(), ln_ = l & 31, hf_ = l >> 5 & 1;
                float* arow = dqacc + (ln_ + d0) * C::AS + 4 * hf_;
                float4 a[DT];
                fx4 k[DT];
                static_for<DT>([&](auto X) __attribute__((always_inline)) {
                    constexpr int dt = decltype(X)::value, e = 4 * dt + decltype(B)::value;
                    k[dt] = T::widen(copy4(k2_s, ln_, hf_, e));
                    a[dt] = *(float4*)(arow + 8 * e);
                });
                static_for<DT>([&](auto X) __attribute__((always_inline)) {
                    constexpr int dt = decltype(X)::value, e = 4 * dt + decltype(B)::value;
                    const float4 g = L::template get_regs<G0 + 4 * e>();
                    a[dt].x += g.x * (k[dt][0] + p.k2_bias);
                    a[dt].y += g.y * (k[dt][1] + p.k2_bias);
                    a[dt].z += g.z * (k[dt][2] + p.k2_bias);
                    a[dt].w += g.w * (k[dt][3] + p.k2_bias);
                    *(float4*)(arow + 8 * e) = a[dt];
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

    // ---- dQ partial of this workgroup (rows of deltas beyond the end of the sequence hold zeros) ----
    const int tid_f = here();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the last requests: LDS is reused below)
    __syncthreads();
    if (want_dq) {
        float* dst = dq_part + (((int64_t)bh * nkb + kb) * nseg + seg) * (int64_t)RQ * D;
        for (int it = tid_f; it < RQ * (D / 4); it += KT) {
            const int row = it / (D / 4), col = it % (D / 4) * 4;
            float4 a = *(const float4*)(dqacc + row * C::AS + col);
            a.x *= p.scale; a.y *= p.scale; a.z *= p.scale; a.w *= p.scale;
            *(float4*)(dst + (int64_t)row * D + col) = a;
        }
    }
    __syncthreads();
    // ---- dK' and dV': the four wavefronts' sums added through LDS ----
    {
        const int ln_ = tid_f & 31, hf_ = tid_f >> 5 & 1;
        static_for<2 * 4 * DT>([&](auto X) __attribute__((always_inline)) {
            constexpr int x = decltype(X)::value, which = x / (4 * DT), e = x % (4 * DT);                // 0: dV', 1: dK'
            float* row = (float*)smem_raw + ((size_t)(which * KW + wave) * BQ + ln_) * C::AS + 8 * e + 4 * hf_;
            if constexpr (which ? DKA : DVA) {
                constexpr int at = (which ? DK0 : DV0) + 4 * e;
                *(float4*)row = L::template get_regs<at>();
            } else {
                const floatx16& v = (which ? dkv : dvv)[e / 4];
                *(float4*)row = make_float4(v[4 * (e % 4)], v[4 * (e % 4) + 1], v[4 * (e % 4) + 2], v[4 * (e % 4) + 3]);
            }
        });
    }
    __syncthreads();
    for (int it = tid_f; it < 2 * BQ * (D / 4); it += KT) {
        const int which = it / (BQ * (D / 4)), rem = it - which * (BQ * (D / 4)), row = rem / (D / 4), col = rem % (D / 4) * 4, k = k0 + row;
        const Tensor& t = which ? p.dk2 : p.dv2;
        if (k >= N || !t.p) continue;
        fx4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < KW; ++w) a += *(const fx4*)((float*)smem_raw + ((size_t)(which * KW + w) * BQ + row) * C::AS + col);
        if (which) a *= p.scale;
        if (nseg > 1) *(fx4*)(kpart + ((((int64_t)which * nseg + seg) * p.B * p.H + bh) * N + k) * D + col) = a;
        else if (!PAD || col < p.D) T::store((EL*)t.p + t.off(b, k, h) + col, a[0], a[1], a[2], a[3]);
    }
}

template <class T, int D, int NU, int MODE>
int launch_split_kp_lone(const Problem& p, const SplitKpLaunch& l, hipStream_t st) {
    using C = SplitKpLoneCfg<D, T::PLANES>;
    const bool raw = C::raw_fits(l.plan.segw);
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return SA2_ERR_LAUNCH_FAILED;
        hipLaunchKernelGGL(kernel, dim3((unsigned)((int64_t)l.per_seg * l.plan.nseg)), dim3(C::THREADS), C::lds_bytes(l.plan.segw, raw), st, p, l.nkb, l.per_seg,
                           l.dq_part, l.plan.nseg, l.plan.segw, l.kpart);
        return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
    };
    return raw ? go(split_kp_lone_kernel<T, D, NU, MODE, true>) : go(split_kp_lone_kernel<T, D, NU, MODE, false>);
}

}  // namespace
}  // namespace sa2
