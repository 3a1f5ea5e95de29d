// The K-side backward kernel (dK and dV) of the plane-split kernels with one wavefront per SIMD; included once per element type.
// Arithmetic, shares and partial sums are those of split_kv_kernel (sa2_split_mfma.hip), which says what a unit and a plane are.
//
// A workgroup owns 128 consecutive K/V rows, 32 per wavefront, resident as planes in accumulation registers beside the sums of
// dK and dV (sa2_mfma_lone.h), and streams every unit (query block, delta) that sees them; the units' Q~ and dO~ tiles are formed by
// all threads, two units ahead, into a ring of four in LDS.  Per unit a wavefront computes
//   A: S = Q~.K^T - LSE and dP = dO~.V^T - D,   B: P = exp2(S), dS = P * dP, both split into planes,   C: dV^T += dO~^T.P and dK^T += Q~^T.dS
// with C of the unit before, B and the forming between the MFMAs: a product of planes takes the matrix pipe as long as eleven
// instructions take to split two weights, and neither waits for the other.  A thread forms four columns of a row per 32-column
// block; its part of q and dO stays in registers for a query block, K' and V' rows come from global memory one unit ahead.
//
// What bounds it: the matrix pipe (fp32 head_dim 64: 98 MFMAs of 33 cycles in a unit's 4200; bf16 at 96 columns 86 in 4350) and the
// instructions beside it, 4.5 to 5.5 per MFMA of which four are free.  K side, us, wavefronts in pairs / this: fp32 B2 H8 N2048 D64
// w 512/32 1670 / 1320, bf16 B1 H8 N2048 D96 w 255/31 725 / 415.  (Splits of eleven instructions behind one MFMA and none behind the next:
// 1430 and 440.)
//
// NU: planes of a unit.  Two where the products q*k2 and dO*v2 have 16 bits (bf16 tensors without biases): the scale is then multiplied onto
// the logits, and LSE / scale is what comes off the chain.
//
// A tile of a plane lies in 32-column blocks of 32 rows of 64 bytes, whose four 16-byte chunks are exchanged by (row / 4) % 4: row
// operands (16 rows of one chunk), transposed ones (four rows of 64 bytes) and the stores of the forming (eight rows of 64 bytes) are all
// free of bank conflicts.
#pragma once

#include "sa2_split_lone.h"
#include "sa2_units.h"

namespace sa2 {
namespace {

template <class T, int D, int NU>
struct SplitKvLoneCfg {
    static constexpr int W = 4, THREADS = W * 64, ROWS = W * 32;     // wavefronts, threads, K rows per workgroup
    static constexpr int NK = T::PLANES, DK = D / 16, DT = D / 32;
    static constexpr int BLOCK = 2048, PLANE = DT * BLOCK, TILE = NU * PLANE, UNIT = 2 * TILE, NUNIT = 4;      // bytes
    static constexpr int LEAD_AT = NUNIT * UNIT;                     // [block % 4][LSE, D][32 queries] lead_planes
    static constexpr size_t LDS_BYTES = (size_t)LEAD_AT + 4 * 2 * BQ * 16;
    // accumulation registers
    static constexpr int DV0 = 0, DK0 = DT * 16, K0 = 2 * DT * 16, V0 = K0 + NK * DK * 4, ONE0 = V0 + NK * DK * 4;
    static constexpr int USED = ONE0 + 4, OWNED = USED <= 192 ? 192 : 256;
    static_assert(USED <= 256 && LDS_BYTES <= 160 * 1024, "");
};
template <class T, int D, int NU, int MODE>
__global__ __launch_bounds__((SplitKvLoneCfg<T, D, NU>::THREADS)) __attribute__((amdgpu_waves_per_eu(1, 1)))
void split_kv_lone_kernel(Problem p, int njb, int total, int nsplit, float* __restrict__ part) {
    using C = SplitKvLoneCfg<T, D, NU>;
    using L = Lone<C::OWNED>;
    typedef typename T::T EL;
    typedef typename T::Raw Raw;
    typedef bf16x8 X8;
    constexpr bool PAD = MODE != EXACT;
    constexpr int DK = C::DK, DT = C::DT, NK = C::NK;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int N = p.N, w1 = p.w1, w2 = p.w2;

    auto here = [&]() __attribute__((always_inline)) {        // (lane parts of what happens once per query block are computed there)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    const int pid = xcd_order(blockIdx.x, total);
    const int sp = pid % nsplit, pj = pid / nsplit;
    const int bh = pj / njb, jb = pj - bh * njb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int j0 = jb * C::ROWS, jw = j0 + 32 * wave;         // this wavefront's K rows: jw .. jw + 31

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);
    const EL* dop = (const EL*)p.dout.p + p.dout.off(b, 0, h);
    const float qscale = p.scale * LOG2E;

    // ---- the stream of units (query block, delta) and this workgroup's share of it: see split_kv_kernel ----
    const int j_last = j0 + C::ROWS - 1 < N ? j0 + C::ROWS - 1 : N - 1;
    const int i_max = (int)((int64_t)j_last + w1 < N - 1 ? j_last + w1 : N - 1);
    int ib_lo = j0 / BQ, ib_hi = i_max / BQ, d_first = 0, d_last = w2;
    auto last_unit_of = [&](int ib) __attribute__((always_inline)) {            // the last delta of a block
        const int il = ib * BQ + BQ - 1 < N ? ib * BQ + BQ - 1 : N - 1;
        int d = w2 < il ? w2 : il;
        if (ib == ib_hi && d_last < d) d = d_last;
        return d;
    };
    bool has_work = ib_lo <= ib_hi;
    if (nsplit > 1) {
        const int per = w2 + 1, ib0 = ib_lo;
        const int slots = (ib_hi - ib_lo + 1) * per;
        const int chunk = (slots + nsplit - 1) / nsplit;
        const int v_lo = sp * chunk, v_hi = (v_lo + chunk < slots ? v_lo + chunk : slots) - 1;
        has_work = v_lo <= v_hi;
        if (has_work) {
            ib_lo = ib0 + v_lo / per;
            d_first = v_lo - (ib_lo - ib0) * per;
            ib_hi = ib0 + v_hi / per;
            d_last = v_hi - (ib_hi - ib0) * per;
            const int il = ib_lo * BQ + BQ - 1 < N ? ib_lo * BQ + BQ - 1 : N - 1;
            if (d_first > (w2 < il ? w2 : il)) {              // the share starts in the slots a short block does not have
                ++ib_lo;
                d_first = 0;
            }
            has_work = ib_lo < ib_hi || (ib_lo == ib_hi && d_first <= d_last);
        }
    }

    // ---- forming: thread t the columns 32*dt + 4*(t % 8) .. of row t / 8 ----
    const uint32_t lds0 = lds_address(smem_raw);
    const int f_row = tid >> 3, f_col = (tid & 7) * 4;
    const uint32_t f_lane = (uint32_t)(f_row * 64 + (((tid & 7) >> 1) ^ (f_row >> 2 & 3)) * 16 + (tid & 1) * 8);
    fx4 qv[DT], dv[DT];                                       // of the block that is formed: q (times scale * log2(e)) and dO
    Raw fq[DT], fd[DT], fk[DT], fv[DT];                       // on their way: q and dO of the block after it, K' and V' of the next unit
    float row_raw = 0.f;                                      // LSE (threads 0-31) or D (32-63) of that block's queries
    auto request_block = [&](int ib) __attribute__((always_inline)) {
        const int i = ib * BQ + f_row < N ? ib * BQ + f_row : N - 1;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            fq[dt] = raw4<T, PAD>(qp + (int64_t)i * p.q.sn, dt * 32 + f_col, p.D);
            fd[dt] = raw4<T, PAD>(dop + (int64_t)i * p.dout.sn, dt * 32 + f_col, p.D);
        }
        const int t = here();
        if (t < 2 * BQ) {
            const int r = ib * BQ + (t & 31) < N ? ib * BQ + (t & 31) : N - 1;
            row_raw = (t < BQ ? p.lse : p.dsum)[(int64_t)bh * N + r];
        }
    };
    auto take_block = [&](int ib) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            qv[dt] = T::widen(fq[dt]);
            if constexpr (NU == 3) qv[dt] *= qscale;
            dv[dt] = T::widen(fd[dt]);
        }
        const int t = here();
        if (t < 2 * BQ) {
            X8 lead;
            if (t >= BQ) {
                lead = lead_planes(row_raw, 0.f);
            } else if (NU == 3) {
                float x = row_raw * LOG2E;
                stays(x);                                     // (rounded: taken together with the split, lse_rest would count twice)
                lead = lead_planes(x, lse_rest(row_raw, x));
            } else {
                float x = row_raw / p.scale;
                stays(x);
                lead = lead_planes(x, fmaf(-x, p.scale, row_raw) / p.scale);
            }
            *(X8*)(smem_raw + C::LEAD_AT + ((ib & 3) * 2 * BQ + t) * 16) = lead;
        }
    };
    // cursors: the unit that is formed next (two ahead of the one in work), and the one whose K' and V' rows are requested next
    int f_ib = ib_lo, f_delta = d_first, f_stop = 0, l_ib = ib_lo, l_delta = d_first, l_stop = 0;
    auto stop_of = [&](int ib) __attribute__((always_inline)) { return ib <= ib_hi ? last_unit_of(ib) : NEVER; };
    auto request_unit = [&]() __attribute__((always_inline)) {
        const int i = l_ib * BQ + f_row < N ? l_ib * BQ + f_row : N - 1, k = i - l_delta > 0 ? i - l_delta : 0;
        const EL *ks = k2p + (int64_t)k * p.k2.sn, *vs = v2p + (int64_t)k * p.v2.sn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            fk[dt] = raw4<T, PAD>(ks, dt * 32 + f_col, p.D);
            fv[dt] = raw4<T, PAD>(vs, dt * 32 + f_col, p.D);
        }
        ++l_delta;
    };
    auto request_turn = [&]() __attribute__((always_inline)) {
        if (l_delta <= l_stop) return;
        ++l_ib;
        l_delta = 0;
        l_stop = stop_of(l_ib);
    };
    auto form_turn = [&](int n) __attribute__((always_inline)) {
        f_delta += n;
        if (f_delta <= f_stop) return;
        ++f_ib;
        f_delta = 0;
        f_stop = stop_of(f_ib);
        take_block(f_ib);
        request_block(f_ib + 1);
    };
    // Item f: two columns of Q~ or dO~, in STEPS steps of three or four instructions; the second of a row's two items per block
    // sends its words off.
    constexpr int NF = 4 * DT, STEPS = 2 * NU - 1;
    uint32_t fw[NU][2];
    float fy[2], fa[2], fh[2];
    auto form_step = [&](auto X, uint32_t to) __attribute__((always_inline)) {
        constexpr int f = decltype(X)::value / STEPS, m = decltype(X)::value % STEPS, dt = f / 4, which = f / 2 % 2, e = f % 2 * 2;
        const fx4& x = which ? dv[dt] : qv[dt];
        if constexpr (m == 0) {
            const fx4 y = T::widen(which ? fv[dt] : fk[dt]);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                fy[t] = NU == 2 ? y[e + t] : y[e + t] + (which ? p.v2_bias : p.k2_bias);
                fa[t] = x[e + t] * fy[t];
            }
        } else if constexpr (m % 2 == 1) {
            const uint32_t w = pack2(fa[0], fa[1]);
            fw[m / 2][e / 2] = w;
            fh[0] = bf16_lo(w);
            fh[1] = bf16_hi(w);
        } else {
#pragma unroll
            for (int t = 0; t < 2; ++t) fa[t] = m == 2 ? fmaf(x[e + t], fy[t], -fh[t]) : fa[t] - fh[t];
            if constexpr (m == STEPS - 1) fw[NU - 1][e / 2] = pack2(fa[0], fa[1]);
        }
        if constexpr (m == STEPS - 1) stays(fw[NU - 1][e / 2]);
        else stays(fa[0]), stays(fa[1]);
        if constexpr (m == STEPS - 1 && e == 2) {
#pragma unroll
            for (int n = 0; n < NU; ++n)
                *(ux2 __attribute__((address_space(3)))*)(uintptr_t)(to + (uint32_t)(which * C::TILE + n * C::PLANE + dt * C::BLOCK)) = ux2{fw[n][0], fw[n][1]};
        }
    };
    auto form_all = [&](uint32_t unit) __attribute__((always_inline)) {
        static_for<NF * STEPS>([&](auto X) __attribute__((always_inline)) { form_step(X, unit + f_lane); });
    };

    // ---- the work of a wavefront ----
    constexpr Products<NU, NK> PA;                            // unit plane, K or V plane
    constexpr Products<NU, 3> PC;                             // unit plane, plane of P or dS
    constexpr int NP = PA.n, NC = PC.n;
    constexpr int CH = NP * DK + 1;                           // MFMAs of a chain of phase A (the last one takes LSE or D off)
    constexpr int NG = DT * NC;                               // MFMAs of a quarter of phase C: one half of the queries, dV or dK
    constexpr int NA = 2 * CH, NS = NA + 4 * NG;              // of phase A, of a unit
    constexpr int AHEAD = NP >= 5 ? 1 : NP == 3 ? 2 : 3;      // k-steps that row operands are read ahead
    X8 ro[AHEAD + 1][NU], co[2][NU];                          // row operands by k-step, transposed ones by column block
    X8 lead_s, lead_d;
    floatx16 s, dp, nl;                                       // nl: what a chain of S starts from, -inf where the pair is outside the windows
    u4 pw[2][3], dw[2][3];                                    // planes of P and dS of each half of the queries
    uint32_t ua = lds0, ub = lds0 + C::UNIT, uc = lds0 + 2 * C::UNIT, ud = lds0 + 3 * C::UNIT;         // units t, t+1, t+2, t-1
    const uint32_t row_lane = (uint32_t)(ln * 64 + (hf ^ (ln >> 2 & 3)) * 16);
    const uint32_t col_lane = [&]() {
        const int grp = lane >> 4, x = lane & 15, r = 4 * (grp >> 1) + (x >> 2), c = 2 * (grp & 1) + ((x & 3) >> 1);
        return (uint32_t)(r * 64 + (c ^ (r >> 2)) * 16 + (x & 1) * 8);
    }();
    // The lane's addresses in a unit, for even and odd k-steps and slices of eight rows (UNIT and all blocks are multiples of 64, so that the
    // odd ones differ in one bit); opaque, so that what is added to them goes into the instructions' offsets.
    static_assert(C::UNIT % 64 == 0, "");
    uint32_t r0 = 0, r1 = 0, c0 = 0, c1 = 0;
    auto at_unit = [&](uint32_t unit, uint32_t part, uint32_t& even, uint32_t& odd) __attribute__((always_inline)) {
        even = unit + part;
        odd = even ^ 32u;
        stays(even);
        stays(odd);
    };

    // entry e of phase A: k-step e % DK of S (from the Q~ tile) or dP (dO~)
    auto read_row = [&](auto EN, auto X) __attribute__((always_inline)) {
        constexpr int e = decltype(EN)::value, x = decltype(X)::value, which = e / DK, kk = e % DK;
        ro[e % (AHEAD + 1)][x] = lds_read_x8<X8>((kk & 1 ? r1 : r0) + (uint32_t)(which * C::TILE + x * C::PLANE + kk / 2 * C::BLOCK));
    };
    // entry e of phase C: quarter e / DT (dV's halves, from the dO~ tile, then dK's), column block e % DT
    auto read_column = [&](auto EN, auto X) __attribute__((always_inline)) {
        constexpr int e = decltype(EN)::value, x = decltype(X)::value, which = e / (2 * DT), ks = e / DT % 2, dt = e % DT;
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef v4s __attribute__((address_space(3)))* lds_v4s;
        constexpr uint32_t at = (which ? 0 : C::TILE) + x * C::PLANE + dt * C::BLOCK + ks * 1024;
        union { v4s half[2]; X8 v; } u;
        u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c0 + at));
        u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c1 + at + 512));
        co[e % 2][x] = u.v;
    };
    auto read_first_rows = [&]() __attribute__((always_inline)) {
        at_unit(ua, row_lane, r0, r1);
        static_for<AHEAD * NU>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(decltype(X)::value / NU), LONE_C(decltype(X)::value % NU)); });
    };
    auto a_mfma = [&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value, which = i / CH, m = i % CH;
        if constexpr (m == CH - 1) {
            if constexpr (which) L::template tile_more<C::ONE0>(dp, lead_d);
            else L::template tile_more<C::ONE0>(s, lead_s);
        } else {
            constexpr int kk = m / NP, x = PA.x[m % NP], y = PA.y[m % NP], e = which * DK + kk;
            constexpr int at = (which ? C::V0 : C::K0) + (y * DK + kk) * 4;
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
        if constexpr (which) L::template sum_more<C::DK0 + dt * 16>(co[e % 2][x], __builtin_bit_cast(X8, dw[ks][y]));
        else L::template sum_more<C::DV0 + dt * 16>(co[e % 2][x], __builtin_bit_cast(X8, pw[ks][y]));
    };
    // Vector work on a unit: 16 exponentials; 16 products dS = P * dP, in the place of dP; eight words of each plane of P and of dS
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
    // the slots of the forming, where the splits leave room beside the MFMAs; behind them the next unit's rows are requested
    constexpr int FORM = NP >= 5 ? 2 : CH, FORMED = NP >= 5 ? NA + NG : NA + 3 * NG;
    auto beside = [&](auto SLOT, auto DO_C, uint32_t form_at) __attribute__((always_inline)) {
        constexpr int slot = decltype(SLOT)::value;
        if constexpr (decltype(DO_C)::value) within<16, slot, 1, CH - 1>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[1], LONE_C(1), X); });
        within<16, slot, CH + 2, NA + 1>(exp_item);
        within<16, slot, NA + 2, NA + NG>(ds_item);
        within<16, slot, NA + NG, NA + 2 * NG>([&](auto X) __attribute__((always_inline)) { split_step(s, pw[0], LONE_C(0), X); });
        within<16, slot, NA + 2 * NG, NA + 3 * NG>([&](auto X) __attribute__((always_inline)) { split_step(s, pw[1], LONE_C(1), X); });
        within<16, slot, NA + 3 * NG, NS>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[0], LONE_C(0), X); });
        within<NF * STEPS, slot, FORM, FORMED>([&](auto X) __attribute__((always_inline)) { form_step(X, form_at); });
        if constexpr (slot == FORMED) request_unit();
    };
    auto unit = [&](auto DO_C) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        uint32_t form_at = uc + f_lane;
        stays(form_at);
        if constexpr (CC) at_unit(ud, col_lane, c0, c1);
        static_for<NA>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / CH * DK + i % CH / NP, m = i % CH % NP;
            a_mfma(I);
            // One barrier per unit, which says two things: unit t+1 is formed (what a wavefront has stored is in LDS, since reads
            // that it issued later have returned), and unit t-2, over which t+2 is formed, was read to the end.
            if constexpr (i == 1) asm volatile("s_barrier" ::: "memory");
            if constexpr (i % CH < CH - 1 && e + AHEAD < 2 * DK) deal<NU, m, NP>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(e + AHEAD), X); });
            if constexpr (CC && i >= NA - NU) read_column(LONE_C(0), LONE_C(i - (NA - NU)));
            beside(I, DO_C, form_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) finished(s, dp);
        static_for<4 * NG>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / NC, m = i % NC;
            if constexpr (CC) {
                c_mfma(I);
                if constexpr (e + 1 < 4 * DT && m < NU) read_column(LONE_C(e + 1), LONE_C(m));
            }
            if constexpr (i == 4 * NG - AHEAD * NU) at_unit(ub, row_lane, r0, r1);
            if constexpr (i >= 4 * NG - AHEAD * NU) read_row(LONE_C((i - (4 * NG - AHEAD * NU)) / NU), LONE_C((i - (4 * NG - AHEAD * NU)) % NU));
            beside(LONE_C(NA + i), DO_C, form_at);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto last_sums = [&]() __attribute__((always_inline)) {                         // C of unit t-1 alone
        at_unit(ud, col_lane, c0, c1);
        static_for<16>([&](auto X) __attribute__((always_inline)) { split_step(dp, dw[1], LONE_C(1), X); });
        static_for<NU>([&](auto X) __attribute__((always_inline)) { read_column(LONE_C(0), X); });
        static_for<4 * NG>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, e = i / NC, m = i % NC;
            c_mfma(I);
            if constexpr (e + 1 < 4 * DT && m < NU) read_column(LONE_C(e + 1), LONE_C(m));
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto rotate = [&]() __attribute__((always_inline)) {
        L::keep_out();
        const uint32_t x = ua;
        ua = ub;
        ub = uc;
        uc = ud;
        ud = x;
    };

    {
        X8 z;
#pragma unroll
        for (int t = 0; t < 8; ++t) z[t] = (__bf16)0.f;
        asm volatile("s_nop 3" : "+v"(z));
        static_for<2 * DT>([&](auto X) __attribute__((always_inline)) { L::template sum_zero<16 * decltype(X)::value>(z); });
    }
    if (has_work) {
        // ---- prologue: K and V rows as resident planes, units 0 and 1 ----
        request_block(ib_lo);
        l_stop = stop_of(ib_lo);
        f_stop = l_stop;
        request_unit();
        request_turn();
        {
            const int jc = jw + ln < N ? jw + ln : N - 1;
            const EL* rows[2] = {(const EL*)p.k1.p + p.k1.off(b, jc, h), (const EL*)p.v1.p + p.v1.off(b, jc, h)};
            static_for<2 * DK>([&](auto X) __attribute__((always_inline)) {
                constexpr int which = decltype(X)::value / DK, kk = decltype(X)::value % DK;
                const int col = kk * 16 + hf * 8;
                const float4 x0 = cols4<T, PAD>(rows[which], col, p.D), x1 = cols4<T, PAD>(rows[which], col + 4, p.D);
                const float r[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
                X8 o[NK];
                split8<NK, T::DTYPE == SA2_F32>(r, o);
                static_for<NK>([&](auto Y) __attribute__((always_inline)) {
                    constexpr int y = decltype(Y)::value;
                    const u4 w = __builtin_bit_cast(u4, o[y]);
                    L::template set_regs<(which ? C::V0 : C::K0) + (y * DK + kk) * 4>(w[0], w[1], w[2], w[3]);
                });
            });
            const u4 ones = __builtin_bit_cast(u4, lead_ones(hf));
            L::template set_regs<C::ONE0>(ones[0], ones[1], ones[2], ones[3]);
        }
        take_block(ib_lo);
        request_block(ib_lo + 1);
        form_all(ua);
        form_turn(1);
        request_unit();
        request_turn();
        form_all(ub);
        form_turn(1);
        request_unit();
        request_turn();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

        int ib = ib_lo, delta = d_first, stop = last_unit_of(ib_lo);
        bool more = true, mine = false;                       // mine: this wavefront's keys see one of the block's queries
        // the block's row values and masks
        auto enter_block = [&]() __attribute__((always_inline)) {
            const int i0 = ib * BQ, t = here(), ln = t & 31, hf = t >> 5 & 1;
            mine = (i0 + BQ - 1 >= jw) && ((int64_t)i0 <= (int64_t)jw + 31 + w1) && jw < N;
            if (!mine) return;
            const unsigned char* lead = smem_raw + C::LEAD_AT + ((ib & 3) * 2 * BQ + ln) * 16;
            lead_s = *(const X8*)lead;
            lead_d = *(const X8*)(lead + BQ * 16);
#pragma unroll
            for (int v = 0; v < 16; ++v) nl[v] = 0.f;
            if ((i0 >= jw + 31) && ((int64_t)i0 + 31 <= (int64_t)jw + w1) && (i0 + BQ - 1 < N)) return;
            // element v of this lane is query i0 + 8*(v/4) + 4*hf + v%4, column j
            const int j = jw + ln, lo = j - i0 - 4 * hf, nhi = N - 1 - i0 - 4 * hf;
            const int hi = (int)((int64_t)j + w1 - i0 < 1 << 20 ? j + w1 - i0 : 1 << 20) - 4 * hf;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int c = 8 * (v >> 2) + (v & 3);
                nl[v] = ((j < N) & (c >= lo) & (c <= hi) & (c <= nhi)) ? 0.f : -INFINITY;
            }
        };
        // rows whose K' row lies before the sequence leave for good: delta only grows within a block
        auto enter_unit = [&]() __attribute__((always_inline)) {
            if (delta > ib * BQ) {
                const int dlo = delta - ib * BQ - 4 * (here() >> 5 & 1);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int c = 8 * (v >> 2) + (v & 3);
                    nl[v] = c >= dlo ? nl[v] : -INFINITY;
                }
            }
            asm volatile("s_nop 3" : "+v"(nl), "+v"(lead_s), "+v"(lead_d));
        };
        // units (the present one included) until something changes: the block or its masks, or a cursor's block
        auto until = [&]() __attribute__((always_inline)) {
            int n = units_left(units_left(stop - delta + 1, f_delta, f_stop), l_delta, l_stop);
            if (stop > ib * BQ) {
                const int whole = ib * BQ - delta + 1;
                if (whole < n) n = whole > 1 ? whole : 1;
            }
            return n;
        };
        auto advance = [&](int n) __attribute__((always_inline)) {                  // behind n units
            request_turn();
            form_turn(n);
            L::keep_out();
            delta += n;
            if (delta > stop) {
                ++ib;
                delta = 0;
                more = ib <= ib_hi;
                if (!more) {
                    mine = false;
                    return;
                }
                stop = last_unit_of(ib);
                enter_block();
                L::keep_out();
            }
            enter_unit();
            L::keep_out();
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        enter_block();
        enter_unit();
        while (more) {
            if (!mine) {
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                form_all(uc);
                request_unit();
                rotate();
                advance(1);
                continue;
            }
            read_first_rows();
            unit(no);
            rotate();
            advance(1);
            while (mine) {
                const int n = until();
                for (int k = n; k > 0; --k) {
                    unit(yes);
                    rotate();
                }
                advance(n);
            }
            last_sums();
        }
    }

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    const int j = jw + ln;
    static_for<2>([&](auto W_) __attribute__((always_inline)) {
        constexpr int role = decltype(W_)::value;            // 0: dV, 1: dK
        const Tensor& t = role ? p.dk1 : p.dv1;
        const float sc = role ? (NU == 3 ? LN2 : p.scale) : 1.f;         // (NU 3: Q~ carries scale * log2(e))
        if (!t.p) return;
        EL* dst = (EL*)t.p + t.off(b, j < N ? j : N - 1, h) + 4 * hf;
        const int64_t BH = (int64_t)p.B * p.H;
        float* pdst = nsplit > 1 ? part + ((((role ? 0 : 1) * (int64_t)nsplit + sp) * BH + bh) * N + (j < N ? j : N - 1)) * D + 4 * hf : nullptr;
        static_for<4 * DT>([&](auto Y) __attribute__((always_inline)) {
            constexpr int at = (role ? C::DK0 : C::DV0) + 4 * decltype(Y)::value, col = 8 * decltype(Y)::value;
            const float4 x = L::template get_regs<at>();
            if (j >= N) return;
            if (nsplit > 1) *(float4*)(pdst + col) = make_float4(x.x * sc, x.y * sc, x.z * sc, x.w * sc);
            else if (!PAD || col + 4 * hf < p.D) T::store(dst + col, x.x * sc, x.y * sc, x.z * sc, x.w * sc);
        });
    });
}

template <class T, int D, int NU, int MODE>
int launch_split_kv_lone(const Problem& p, int nsplit, float* part, hipStream_t st) {
    using C = SplitKvLoneCfg<T, D, NU>;
    const int njb = (p.N + C::ROWS - 1) / C::ROWS;
    const int64_t total = (int64_t)njb * p.B * p.H * nsplit;
    if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    if (!allow_full_lds((const void*)split_kv_lone_kernel<T, D, NU, MODE>)) return SA2_ERR_LAUNCH_FAILED;
    hipLaunchKernelGGL((split_kv_lone_kernel<T, D, NU, MODE>), dim3((unsigned)total), dim3(C::THREADS), C::LDS_BYTES, st, p, njb, (int)total, nsplit, part);
    return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
}

}  // namespace
}  // namespace sa2
