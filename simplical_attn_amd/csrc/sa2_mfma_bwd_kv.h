// The K-side backward kernel (dK and dV) of the tuned 16-bit kernels, head_dim 16 .. 128; included once per element type.
//
// A workgroup owns 128 consecutive K/V rows, or 256 (head_dim up to 64, unless the grid is too small for that): 32 or two
// times 32 per wavefront, resident as MFMA B operands.  It streams every unit of expanded rows that can see them: unit
// (query block ib, delta) is the 32 rows r = (i0 + r, k = i - delta) with
// Q~[r] = q[i] * k2~[k] * scale*log2(e) and dO~[r] = dO[i] * v2~[k], formed by the whole workgroup into a ring of three
// units in LDS, two units ahead.  Per unit and 32 rows of K, one wavefront computes
//   A: S = Q~.K^T - LSE and dP = dO~.V^T - D,   B: P = exp2(S) and dS = P * dP,   C: dV^T += dO~^T.P and dK^T += Q~^T.dS.
// Transposed operands come from the same unit tiles through ds_read_b64_tr_b16; the tiles are laid out in row groups so
// that both kinds of read are free of bank conflicts.  Every output element has one writer and a fixed summation order.
//
// One wavefront per SIMD with all 512 registers does A, B and C itself (sa2_mfma_lone.h): B(t) and the forming of unit t+2
// stand between the MFMAs of A(t+1) and C(t), operand reads eight MFMAs ahead of their use.
// The arrangement before it (two wavefronts per SIMD, one with S, P and dV, one with dP, dS and dK, P handed over in LDS, a
// barrier per unit) ran matrix pipe, vector ALU and LDS one after the other, 2500 cycles per unit of 1024 MFMA cycles; here
// it is 1700 to 1800.  With the row-term kernel, us: B2 H8 N2048 D64 w 512/32 458 -> 323, B1 H16 N8192 D128 w 512/32
// 2715 -> 2300; at D128 the board's power is the next limit.
//
// Small grids (fewer workgroups than the chip holds) split a key block's stream of units over up to sixteen workgroups
// (shares of whole units, at least four each); each writes its fp32 partial dK and dV to the workspace and bwd_sum_kernel
// adds the partials in split order.
#pragma once

#include "sa2_mfma_lone.h"

namespace sa2 {
namespace {

constexpr int VW = 4;                  // wavefronts per workgroup, one per SIMD
constexpr int VT = VW * 64;            // threads per workgroup

// KB: 32-row blocks of K/V rows per wavefront
template <int D, int KB>
struct KvCfg {
    static constexpr int VJ = VW * 32 * KB;        // K rows per workgroup
    static constexpr int DK = D / 16;
    static constexpr int DT = D / 32;
    // A unit tile (32 rows) in LDS keeps groups of RPW rows together: within a group the 16-byte
    // chunk c of row q sits at byte (c * RPW + q) * 16, groups lie GROUP bytes apart.  Row operand
    // reads (16 bytes per lane) and transposed operand reads are both bank-conflict free in it.
    static constexpr int RPW = 512 / D;        // rows per group: 4 (D = 128), 8 (D = 64), 16 (D = 32)
    static constexpr int GROUP = 1024 + 16 * RPW;
    static constexpr int NGROUP = BQ / RPW;
    static constexpr int TILE_BYTES = NGROUP * GROUP;
    static constexpr int UNIT_BYTES = 2 * TILE_BYTES;      // Q~ tile, then dO~ tile
    static constexpr int row_off(int r) { return (r / RPW) * GROUP + (r % RPW) * 16; }    // chunk 0 of row r
    static constexpr int NUNIT = 3;
    static constexpr int NCH = NGROUP > VW ? NGROUP / VW : 1;      // row groups a forming wavefront forms
    static constexpr size_t LDS_LIMIT = 160 * 1024;
    // K'/V' rows kept: a window of ws + 1 deltas over a query block and (unless it is walked in segments) the next 32 rows
    static constexpr int ring_rows(int ws, bool seg) { return (ws + RPW - 1) / RPW * RPW + (seg ? BQ + RPW : 2 * BQ); }
    static constexpr size_t BASE_BYTES = (size_t)NUNIT * UNIT_BYTES + 8 * BQ * 4 + 2 * NGROUP * 1024;
    static constexpr size_t lds_bytes(int ws, bool seg) { return BASE_BYTES + 2 * (size_t)ring_rows(ws, seg) * D * 2; }
    static bool fits(int w2) { return lds_bytes(w2, false) <= LDS_LIMIT; }
    // widest run of deltas (minus one) whose K'/V' rows LDS holds at once
    static constexpr int max_segment() { return (int)((LDS_LIMIT - BASE_BYTES) / (2 * D * 2)) / RPW * RPW - BQ - RPW; }
};

// BIAS = false: k2_bias and v2_bias are both zero (the reference's default), the adds drop out.
// nsplit > 1: the workgroup takes the sp-th share of the key block's units and writes fp32 partial sums to `part`
// ([2][nsplit][B*H][N][D]: dK before its scale, then dV).
// SEG = true: a K' window too wide for LDS is walked in segments of ws_arg + 1 deltas; LDS holds the K'/V' rows of one
// segment of a query block and they are reloaded at every segment.
// PAD: the tensors have p.D <= D columns (see load_cols8).
template <class E, int D, bool BIAS, int KB, bool SEG, bool PAD>
__global__ __launch_bounds__(VT) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mfma_bwd_kv_kernel(Problem p, int njb, int total, int nsplit, float* __restrict__ part, int ws_arg) {
    typedef typename E::x8 X8;
    using C = KvCfg<D, KB>;
    using L = Lone<192>;
    constexpr int VJ = C::VJ, DK = C::DK, DT = C::DT, NCH = C::NCH, RPW = C::RPW;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int ws = SEG ? ws_arg : w2;
    const int R = C::ring_rows(ws, SEG);                      // K'/V' rows kept: a ring, row k at (k - k_base) % R
    float* rows_s = (float*)(smem_raw + (size_t)C::NUNIT * C::UNIT_BYTES);      // [4][-LSE*log2(e) | -D_i][BQ], by ib % 4
    unsigned char* qd_s = (unsigned char*)(rows_s + 8 * BQ);  // q and dO rows of the next block, in row groups
                                                              // (behind them: K' rows in row groups, then V' rows)
    const uint32_t side = (uint32_t)(R * D * 2);              // bytes from a K' row to the V' row

    // lane parts of what happens once per query block are computed where they are used: hoisted out of the sweep they would
    // cost it its registers
    auto here = [&]() __attribute__((always_inline)) {
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
    const int j0 = jb * VJ;
    const int jw = j0 + 32 * KB * wave;          // this wavefront's K rows: jw .. jw + 32*KB - 1

    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* k2p = (const uint16_t*)p.k2.p + p.k2.off(b, 0, h);
    const uint16_t* v2p = (const uint16_t*)p.v2.p + p.v2.off(b, 0, h);
    const uint16_t* dop = (const uint16_t*)p.dout.p + p.dout.off(b, 0, h);

    // registers (see above) of the sums and of the resident operands
    constexpr int DV0 = 0, DK0 = KB * DT * 16, K0 = 2 * KB * DT * 16, V0 = K0 + KB * DK * 4;
    static_assert(V0 + KB * DK * 4 <= 192, "");
    const float qscale = p.scale * LOG2E;
    const int j_last = (j0 + VJ - 1 < N ? j0 + VJ - 1 : N - 1);
    const int i_max = (int)((int64_t)j_last + w1 < N - 1 ? j_last + w1 : N - 1);
    // The units (query block, delta) that see the key block, in stream order, and this workgroup's share of
    // them: from delta d_first of block ib_lo to delta d_last of block ib_hi.  The shares cut the stream
    // counted with w2 + 1 slots per block (a block near the start of the sequence has fewer units: the slots
    // beyond are skipped).
    int ib_lo = j0 / BQ, ib_hi = i_max / BQ, d_first = 0, d_last = w2;
    auto last_unit_of = [&](int ib) __attribute__((always_inline)) {            // the last delta of a block
        const int il = (ib * BQ + BQ - 1 < N ? ib * BQ + BQ - 1 : N - 1);
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
            const int il = (ib_lo * BQ + BQ - 1 < N ? ib_lo * BQ + BQ - 1 : N - 1);
            if (d_first > (w2 < il ? w2 : il)) {     // the share starts in the slots a short block does not have
                ++ib_lo;
                d_first = 0;
            }
            has_work = ib_lo < ib_hi || (ib_lo == ib_hi && d_first <= d_last);
        }
    }

    // ---- forming: wavefront g forms row groups g, g + 4, ..: lane L the 16-byte chunk L / RPW of row L % RPW, so that its
    // stores fill a group's 1 KB contiguously.  The thread's chunks of the block's q and dO rows stay in registers. ----
    const bool former = C::NGROUP >= VW || wave < C::NGROUP;
    const int f_col = lane / RPW;
    auto f_row = [&](int c) __attribute__((always_inline)) { return (wave + VW * c) * RPW + (here() & 63) % RPW; };
    float qv[NCH][8], dv[NCH][8];
    uint32_t f_at[NCH];                            // ring row of the K' and V' chunks of the next unit to be formed
    const uint32_t qd_addr = lds_address(smem_raw) + (uint32_t)(C::NUNIT * C::UNIT_BYTES + 8 * BQ * 4), k2_addr = qd_addr + 2 * C::NGROUP * 1024;
    const uint32_t f_lane = k2_addr + (uint32_t)(f_col * RPW * 16);
    int k_base = 0;                              // a multiple of RPW
    float row_raw = 0.f;
    // one row group (RPW rows from row0 on) of a tensor straight to LDS at `to`, in the order that the forming lanes read
    auto request_group = [&](const uint16_t* base, int64_t sn, int row0, uint32_t to) __attribute__((always_inline)) {
        const int l = here() & 63, col = l / RPW * 8;
        int r = row0 + l % RPW;
        r = r < 0 ? 0 : (r < N ? r : N - 1);
        const void* src = base + (int64_t)r * sn + col;
        if constexpr (PAD) src = col < p.D ? src : (const void*)zero_chunk;
        lds_request(src, to);
    };
    // q, dO, LSE and D rows of a block: every wavefront the groups it forms
    auto request_block = [&](int ib) __attribute__((always_inline)) {
        if (former) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int g = wave + VW * c;
                request_group(qp, p.q.sn, ib * BQ + g * RPW, qd_addr + (uint32_t)(g * 1024));
                request_group(dop, p.dout.sn, ib * BQ + g * RPW, qd_addr + (uint32_t)((C::NGROUP + g) * 1024));
            }
        }
        const int t = here();
        if (t < 2 * BQ) {
            const int i = ib * BQ + (t & 31) < N ? ib * BQ + (t & 31) : N - 1;
            row_raw = (t < BQ ? p.lse : p.dsum)[(int64_t)bh * N + i];
        }
    };
    auto take_block = [&](int ib) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const unsigned char* src = qd_s + (wave + VW * c) % C::NGROUP * 1024 + (here() & 63) * 16;
            const uint4 qa_ = *(const uint4*)src, da_ = *(const uint4*)(src + C::NGROUP * 1024);
            const uint32_t qw[4] = {qa_.x, qa_.y, qa_.z, qa_.w}, dw_[4] = {da_.x, da_.y, da_.z, da_.w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                qv[c][2 * t] = E::lo(qw[t]) * qscale;
                qv[c][2 * t + 1] = E::hi(qw[t]) * qscale;
                dv[c][2 * t] = E::lo(dw_[t]);
                dv[c][2 * t + 1] = E::hi(dw_[t]);
            }
        }
        const int u = here();
        if (u < 2 * BQ) rows_s[(ib & 3) * 2 * BQ + u] = u < BQ ? -row_raw * LOG2E : -row_raw;
    };
    auto request_side = [&](int k0, int groups) __attribute__((always_inline)) {            // row groups of K' and V' from row k0 on (a multiple of RPW off k_base)
        for (int g = wave; g < groups; g += VW) {
            const uint32_t to = (uint32_t)((k0 + g * RPW - k_base) % R * (D * 2));
            request_group(k2p, p.k2.sn, k0 + g * RPW, k2_addr + to);
            request_group(v2p, p.v2.sn, k0 + g * RPW, k2_addr + side + to);
        }
    };
    auto load_side = [&](int k0) __attribute__((always_inline)) {                            // a window from row k0 on
        k_base = k0 >= 0 ? k0 / RPW * RPW : -((-k0 + RPW - 1) / RPW * RPW);
        request_side(k_base, (k0 + ws + BQ - k_base + RPW - 1) / RPW);
    };
    auto aim = [&](int ib, int delta) __attribute__((always_inline)) {          // the next unit to be formed
        const int at0 = (ib * BQ - delta - k_base) % R;
#pragma unroll
        for (int c = 0; c < NCH; ++c) f_at[c] = (uint32_t)(at0 + f_row(c) < R ? at0 + f_row(c) : at0 + f_row(c) - R);
    };
    auto aim_next = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) f_at[c] = f_at[c] == 0 ? (uint32_t)R - 1 : f_at[c] - 1;
    };
    // cursor of the unit to be formed next, and the last delta before something has to change
    int f_ib = ib_lo, f_delta = d_first, f_stop = 0;
    auto run_end = [&](int ib, int delta) __attribute__((always_inline)) {
        const int d = last_unit_of(ib);
        return SEG && delta + ws < d ? delta + ws : d;
    };

    const uint32_t units_addr = lds_address(smem_raw);
    // this lane's part of a row operand read (row ln, the k-slots of its half; k-step kk adds
    // kk * KKB) and of a transposed operand read (32-column block dt adds dt * DTB)
    const uint32_t row_lane = (uint32_t)((ln / RPW) * C::GROUP + (hf * RPW + ln % RPW) * 16);
    const uint32_t col_lane = lds_group_column_lane_offset<RPW, C::GROUP>(lane);
    const uint32_t form_lane = (uint32_t)(wave * C::GROUP + lane * 16);
    constexpr uint32_t KKB = 32 * RPW, DTB = 64 * RPW;

    u4 kx[NCH], vx[NCH];
    u4 fw[NCH][2];                               // Q~ and dO~ chunks of the unit in work
    auto form_read = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const uint32_t a = f_lane + f_at[c] / RPW * 1024 + f_at[c] % RPW * 16;
            kx[c] = *(lds_u4)(uintptr_t)a;
            vx[c] = *(lds_u4)(uintptr_t)(a + side);
        }
    };
    // item f: word f % 8 / 2 of Q~ or dO~ (in turn) of chunk f / 8
    auto form_item = [&](auto F) __attribute__((always_inline)) {
        constexpr int f = decltype(F)::value, c = f / 8, which = f % 2, t = f % 8 / 2;
        const uint32_t w = which ? vx[c][t] : kx[c][t];
        const float bias = BIAS ? (which ? p.v2_bias : p.k2_bias) : 0.f;
        const float* a = which ? dv[c] : qv[c];
        fw[c][which][t] = BIAS ? pack2<E>(a[2 * t] * (E::lo(w) + bias), a[2 * t + 1] * (E::hi(w) + bias))
                               : pack2<E>(a[2 * t] * E::lo(w), a[2 * t + 1] * E::hi(w));
    };
    auto form_store = [&](auto X, uint32_t unit) __attribute__((always_inline)) {
        constexpr int c = decltype(X)::value / 2, which = decltype(X)::value % 2;
        if (!former) return;
        *(u4 __attribute__((address_space(3)))*)(uintptr_t)(unit + form_lane + which * C::TILE_BYTES + c * (VW * C::GROUP)) = fw[c][which];
    };
    auto form_all = [&](uint32_t unit) __attribute__((always_inline)) {
        form_read();
        static_for<8 * NCH>([&](auto F) __attribute__((always_inline)) { form_item(F); });
        static_for<2 * NCH>([&](auto X) __attribute__((always_inline)) { form_store(X, unit); });
        aim_next();
    };
    // behind a unit's forming: the cursor moves on; where the block (or the run of deltas) ends, what was requested for the
    // next one is taken and the one after it requested
    auto form_advance = [&](int n) __attribute__((always_inline)) {
        f_delta += n;
        if (f_ib > ib_hi || f_delta <= f_stop) return;
        if (SEG && f_stop < last_unit_of(f_ib)) {
            f_stop = run_end(f_ib, f_delta);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                 // nobody still forms from the old rows
            load_side(f_ib * BQ - f_delta - ws);
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
            ++f_ib;
            f_delta = 0;
            if (f_ib > ib_hi) return;
            f_stop = run_end(f_ib, 0);
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(row_raw) :: "memory");
            take_block(f_ib);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                 // the rows that are here now, for all
            if constexpr (SEG) {
                load_side(f_ib * BQ - ws);
                asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (f_ib < ib_hi) {
                request_block(f_ib + 1);
                if constexpr (!SEG) request_side(f_ib * BQ + BQ, C::NGROUP);
            }
        }
        aim(f_ib, f_delta);
    };

    // ---- the work of a wavefront.  An element is one K block's share of a unit: the tiles S and dP (phase A), the weights
    // P = exp2(S) and dS = P * dP (phase B, vector arithmetic), the sums dV^T += dO~^T.P and dK^T += Q~^T.dS (phase C).  While
    // the MFMAs of A(e) and C(e-1) run one after the other, the vector ALU works on B(e-1), B(e) and the unit to be formed.
    X8 qa[DK], da[DK];                                        // row operands of Q~ and dO~
    X8 dot[DT][2], qt[DT][2];                                 // transposed operands
    floatx16 s[2], dp[2];                                     // by parity of the element
    u4 pw[2][2], dw[2][2];                                    // P, dS in 16 bits
    floatx16 nl[KB], nd;                                      // -LSE*log2e (-inf where the pair is outside the windows) and -D of the block's rows
    uint32_t ua = units_addr, ub = units_addr + C::UNIT_BYTES, uc = units_addr + 2 * C::UNIT_BYTES;      // units t, t+1, t-1 / t+2
    constexpr bool LONG = DK == 8;                            // operands of head_dim 128 are read one kind at a time
    constexpr int NE = 2 * DK, NF = 8 * NCH;                  // MFMAs of a phase, items of a unit's forming
    static_assert(NE == 4 * DT, "");

    auto read_row = [&](auto WHICH, auto KK, uint32_t unit) __attribute__((always_inline)) {
        constexpr int kk = decltype(KK)::value;
        const X8 x = lds_read_x8<X8>(unit + decltype(WHICH)::value * C::TILE_BYTES + row_lane + kk * KKB);
        if constexpr (decltype(WHICH)::value) da[kk] = x;
        else qa[kk] = x;
    };
    auto read_first_rows = [&](uint32_t unit) __attribute__((always_inline)) {
        static_for<DK>([&](auto KK) __attribute__((always_inline)) {
            read_row(std::integral_constant<int, 0>{}, KK, unit);
            if constexpr (!LONG) read_row(std::integral_constant<int, 1>{}, KK, unit);
        });
    };
    // in the order of the dV and dK products
    auto read_column = [&](auto X, uint32_t unit) __attribute__((always_inline)) {
        constexpr int which = decltype(X)::value / (2 * DT), ks = decltype(X)::value / DT % 2, dt = decltype(X)::value % DT;
        const uint32_t a = unit + col_lane + (which ? 0 : C::TILE_BYTES) + dt * DTB;
        if constexpr (which) qt[dt][ks] = lds_group_column_operand_at<C, X8>(a, ks);
        else dot[dt][ks] = lds_group_column_operand_at<C, X8>(a, ks);
    };
    auto read_columns = [&](auto LO, auto HI, uint32_t unit) __attribute__((always_inline)) {
        static_for<decltype(HI)::value - decltype(LO)::value>([&](auto X) __attribute__((always_inline)) {
            read_column(std::integral_constant<int, decltype(LO)::value + decltype(X)::value>{}, unit);
        });
    };
    auto a_mfma = [&](auto XP, auto SB, auto I) __attribute__((always_inline)) {
        constexpr int x = decltype(XP)::value, sb = decltype(SB)::value, i = decltype(I)::value, kk = i % DK;
        constexpr int at = (sb * DK + kk) * 4;
        if constexpr (i == 0) L::tile_start<K0 + at>(s[x], qa[0], nl[sb]);
        else if constexpr (i < DK) L::tile_more<K0 + at>(s[x], qa[kk]);
        else if constexpr (i == DK) L::tile_start<V0 + at>(dp[x], da[0], nd);
        else L::tile_more<V0 + at>(dp[x], da[kk]);
    };
    auto c_mfma = [&](auto XP, auto SB, auto I) __attribute__((always_inline)) {
        constexpr int x = decltype(XP)::value, sb = decltype(SB)::value, i = decltype(I)::value;
        constexpr int which = i / (2 * DT), ks = i / DT % 2, dt = i % DT;
        if constexpr (which == 0) L::sum_more<DV0 + (sb * DT + dt) * 16>(dot[dt][ks], __builtin_bit_cast(X8, pw[x][ks]));
        else L::sum_more<DK0 + (sb * DT + dt) * 16>(qt[dt][ks], __builtin_bit_cast(X8, dw[x][ks]));
    };
    // (an exponential's result may not be read by the next instruction: a pair is rounded behind the next pair's exponentials)
    auto round_p = [&](auto XP, auto I) __attribute__((always_inline)) {
        constexpr int x = decltype(XP)::value, i = decltype(I)::value;
        pw[x][i / 4][i % 4] = pack2<E>(s[x][2 * i], s[x][2 * i + 1]);
    };
    auto p_item = [&](auto XP, auto I) __attribute__((always_inline)) {
        constexpr int x = decltype(XP)::value, i = decltype(I)::value, e = 2 * i;
        s[x][e] = fast_exp2(s[x][e]);
        s[x][e + 1] = fast_exp2(s[x][e + 1]);
        if constexpr (i > 0) round_p(XP, std::integral_constant<int, i - 1>{});
    };
    // (from the rounded weights, for the first queries: see the K'-side kernel, sa2_mfma_bwd_kp_lone.h.  Their units, the first of a stream,
    // go through the same code as all others; the unrounded ones would be two instructions a pair less, 323 -> 312 us at D64, and dK 4 % closer.)
    auto ds_item = [&](auto XP, auto I) __attribute__((always_inline)) {
        constexpr int x = decltype(XP)::value, i = decltype(I)::value, ks = i / 4, t = i % 4, e = 2 * i;
        if constexpr (i == 0) round_p(XP, std::integral_constant<int, 7>{});
        const uint32_t pp = pw[x][ks][t];
        dw[x][ks][t] = pack2<E>(E::lo(pp) * dp[x][e], E::hi(pp) * dp[x][e + 1]);
    };
    auto unit_barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // One K block per unit.  A(t), under the forming of unit t+2; then C(t-1), whose four groups of MFMAs (dV^T and dK^T, each
    // from the rows' first and second half) free the halves of P and dS one after the other for B(t).
    constexpr int BAR = LONG ? 2 * DT : 0;                    // MFMA of phase C that the unit's barrier stands before
    auto single = [&](auto DO_C) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        form_read();
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(0), LONE_C(0), I);
            if constexpr (LONG && i < DK) read_row(LONE_C(1), I, ua);
            if constexpr (CC) {
                if constexpr (LONG) deal<12, i - 4, 12>([&](auto X) __attribute__((always_inline)) { read_column(X, uc); });
                else deal<4 * DT, decltype(I)::value, NE - 2>([&](auto X) __attribute__((always_inline)) { read_column(X, uc); });
            }
            deal<NF, decltype(I)::value, NE + DT>(form_item);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, group = i / DT;
            if constexpr (i == BAR) unit_barrier();
            if constexpr (CC) {
                c_mfma(LONE_C(0), LONE_C(0), I);
                if constexpr (LONG && i < 4) read_column(LONE_C(12 + i), uc);
            }
            if constexpr (LONG && i >= BAR) read_row(LONE_C(0), LONE_C(i - BAR), ub);
            if constexpr (!LONG) read_row(LONE_C(i / DK), LONE_C(i % DK), ub);
            if constexpr (group == 0) deal<NF, NE + i, NE + DT>(form_item);
            deal<2 * NCH, i - 2 * DT, DT>([&](auto X) __attribute__((always_inline)) { form_store(X, uc); });
            if constexpr (group == 1 || group == 2) deal<8, i - DT, 2 * DT>([&](auto X) __attribute__((always_inline)) { p_item(LONE_C(0), X); });
            if constexpr (group == 3) deal<4, i - 3 * DT, DT>([&](auto X) __attribute__((always_inline)) { ds_item(LONE_C(0), X); });
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<4>([&](auto X) __attribute__((always_inline)) { ds_item(LONE_C(0), LONE_C(4 + decltype(X)::value)); });
        aim_next();
    };
    auto single_last = [&]() __attribute__((always_inline)) {                       // C of unit t-1 alone
        static_for<4 * DT>([&](auto X) __attribute__((always_inline)) { read_column(X, uc); });
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(0), LONE_C(0), I); });
    };
    // Two K blocks per unit: A(t, 0), C(t-1, 1), A(t, 1), C(t, 0); the transposed operands of unit t serve C(t, 0) and C(t, 1).
    // The weights and dS of a block are formed from the end of its phase A to the beginning of its phase C, the unit t+2 throughout.
    auto pair = [&](auto DO_C) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;
        constexpr int EARLY = 6;                              // weights (of eight pairs) formed before the other block's phase A
        auto later = [&](auto XP, auto I) __attribute__((always_inline)) {
            deal<16 - EARLY, decltype(I)::value, NE>([&](auto X) __attribute__((always_inline)) {
                constexpr int x = decltype(X)::value;
                if constexpr (x < 8 - EARLY) p_item(XP, LONE_C(EARLY + x));
                else ds_item(XP, LONE_C(x - (8 - EARLY)));
            });
        };
        auto early = [&](auto XP, auto I) __attribute__((always_inline)) {
            deal<EARLY, decltype(I)::value, NE>([&](auto X) __attribute__((always_inline)) { p_item(XP, X); });
        };
        auto form = [&](auto PHASE, auto I) __attribute__((always_inline)) { deal<NF, decltype(PHASE)::value * NE + decltype(I)::value, 4 * NE - 2>(form_item); };
        form_read();
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            a_mfma(LONE_C(0), LONE_C(0), I);
            if constexpr (CC) later(LONE_C(1), I);
            form(LONE_C(0), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            if constexpr (CC) c_mfma(LONE_C(1), LONE_C(KB - 1), I);
            early(LONE_C(0), I);
            form(LONE_C(1), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            a_mfma(LONE_C(1), LONE_C(KB - 1), I);
            deal<4 * DT, decltype(I)::value, NE - 2>([&](auto X) __attribute__((always_inline)) { read_column(X, ua); });
            later(LONE_C(0), I);
            form(LONE_C(2), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        unit_barrier();
        static_for<NE>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            c_mfma(LONE_C(0), LONE_C(0), I);
            read_row(LONE_C(i / DK), LONE_C(i % DK), ub);
            early(LONE_C(1), I);
            form(LONE_C(3), I);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<2 * NCH>([&](auto X) __attribute__((always_inline)) { form_store(X, uc); });
        aim_next();
    };
    auto pair_last = [&]() __attribute__((always_inline)) {                         // C(t-1, 1) alone
        static_for<2>([&](auto X) __attribute__((always_inline)) { p_item(LONE_C(1), LONE_C(6 + decltype(X)::value)); });
        static_for<8>([&](auto X) __attribute__((always_inline)) { ds_item(LONE_C(1), X); });
        static_for<NE>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(1), LONE_C(KB - 1), I); });
    };

    {
        X8 z;
#pragma unroll
        for (int t = 0; t < 8; ++t) z[t] = (typename E::scalar)0.f;
        asm volatile("s_nop 3" : "+v"(z));
        static_for<2 * KB * DT>([&](auto X) __attribute__((always_inline)) { L::sum_zero<16 * decltype(X)::value>(z); });
    }
    if (has_work) {
        // ---- prologue: rows of the first block, units 0 and 1 ----
        request_block(ib_lo);
        load_side(ib_lo * BQ - (SEG ? d_first : 0) - ws);
        static_for<KB * DK>([&](auto X) __attribute__((always_inline)) {       // K and V rows as resident B operands
            constexpr int x = decltype(X)::value, sb = x / DK, col = x % DK * 16;
            const int j = jw + 32 * sb + ln, jc = j < N ? j : N - 1, c = col + hf * 8;
            const uint16_t* ks = (const uint16_t*)p.k1.p + p.k1.off(b, jc, h) + c;
            const uint16_t* vs = (const uint16_t*)p.v1.p + p.v1.off(b, jc, h) + c;
            L::load_regs<K0 + 4 * x>(PAD && c >= p.D ? (const void*)zero_chunk : (const void*)ks);
            L::load_regs<V0 + 4 * x>(PAD && c >= p.D ? (const void*)zero_chunk : (const void*)vs);
        });
        f_stop = run_end(f_ib, f_delta);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(row_raw) :: "memory");
        take_block(ib_lo);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (ib_lo < ib_hi) {
            request_block(ib_lo + 1);
            if constexpr (!SEG) request_side(ib_lo * BQ + BQ, C::NGROUP);
        }
        aim(f_ib, f_delta);
        form_all(ua);
        form_advance(1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        form_all(ub);
        form_advance(1);
        read_first_rows(ua);

        int ib = ib_lo, delta = d_first, stop = last_unit_of(ib_lo), mask = 0;
        bool more = true;
        // the block's row values and masks, this wavefront's K blocks that see one of its queries
        auto enter_block = [&]() __attribute__((always_inline)) {
            const int i0 = ib * BQ, ln = here() & 31, hf = here() >> 5 & 1;
            mask = 0;
#pragma unroll
            for (int sb = 0; sb < KB; ++sb) {
                const int jb0 = jw + 32 * sb;
                if ((i0 + BQ - 1 >= jb0) && ((int64_t)i0 <= (int64_t)jb0 + 31 + w1) && jb0 < N) mask |= 1 << sb;
            }
            if (!mask) return;
            const float* src = rows_s + (ib & 3) * 2 * BQ + 4 * hf;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const float4 a = *(const float4*)(src + 8 * g4);
                nl[0][4 * g4] = a.x; nl[0][4 * g4 + 1] = a.y; nl[0][4 * g4 + 2] = a.z; nl[0][4 * g4 + 3] = a.w;
                const float4 c = *(const float4*)(src + BQ + 8 * g4);
                nd[4 * g4] = c.x; nd[4 * g4 + 1] = c.y; nd[4 * g4 + 2] = c.z; nd[4 * g4 + 3] = c.w;
            }
            if constexpr (KB == 2) nl[1] = nl[0];
#pragma unroll
            for (int sb = 0; sb < KB; ++sb) {
                const int jb0 = jw + 32 * sb, j = jb0 + ln;
                const bool interior = (i0 >= jb0 + 31) && ((int64_t)i0 + 31 <= (int64_t)jb0 + w1) && (i0 + BQ - 1 < N);
                if (interior) continue;
                // element v of this lane is query i0 + 8*(v/4) + 4*hf + v%4, column j
                const int lo = j - i0 - 4 * hf;
                const int hi = (int)((int64_t)j + w1 - i0 < 1 << 20 ? j + w1 - i0 : 1 << 20) - 4 * hf;
                const int nhi = N - 1 - i0 - 4 * hf;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int c = 8 * (v >> 2) + (v & 3);
                    nl[sb][v] = ((j < N) & (c >= lo) & (c <= hi) & (c <= nhi)) ? nl[sb][v] : -INFINITY;
                }
            }
        };
        // rows whose K' row lies before the sequence leave for good: delta only grows within a block
        auto enter_unit = [&]() __attribute__((always_inline)) {
            if (delta > ib * BQ) {
                const int hf = here() >> 5 & 1, dlo = delta - ib * BQ - 4 * hf;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int c = 8 * (v >> 2) + (v & 3);
#pragma unroll
                    for (int sb = 0; sb < KB; ++sb) nl[sb][v] = c >= dlo ? nl[sb][v] : -INFINITY;
                }
            }
        };
        auto rotate = [&]() __attribute__((always_inline)) {
            L::keep_out();
            const uint32_t u = uc;
            uc = ua;
            ua = ub;
            ub = u;
        };
        // units (the present one included) until something changes: the block or its masks, or what is formed from
        auto until = [&]() __attribute__((always_inline)) {
            int n = stop - delta + 1;
            if (f_ib <= ib_hi && f_stop - f_delta + 1 < n) n = f_stop - f_delta + 1;
            if (stop > ib * BQ) {
                const int whole = ib * BQ - delta + 1;
                if (whole < n) n = whole > 1 ? whole : 1;
            }
            return n;
        };
        // behind n units
        auto advance = [&](int n) __attribute__((always_inline)) {
            form_advance(n);
            L::keep_out();
            delta += n;
            if (delta > stop) {
                ++ib;
                delta = 0;
                more = ib <= ib_hi;
                if (!more) {
                    mask = 0;
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
        // units with K blocks of this wavefront
        auto run_single = [&]() __attribute__((always_inline)) {
            single(no);
            rotate();
            advance(1);
            while (mask) {
                const int n = until();
                for (int k = n; k > 0; --k) {
                    single(yes);
                    rotate();
                }
                advance(n);
            }
            single_last();
        };
        auto run_pair = [&]() __attribute__((always_inline)) {
            pair(no);
            rotate();
            advance(1);
            while (mask) {
                const int n = until();
                for (int k = n; k > 0; --k) {
                    pair(yes);
                    rotate();
                }
                advance(n);
            }
            pair_last();
        };
        enter_block();
        enter_unit();
        while (more) {
            if (mask == 0) {
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                read_first_rows(ub);
                form_all(uc);
                rotate();
                advance(1);
            } else if constexpr (KB == 1) {
                run_single();
            } else {
                run_pair();
            }
        }
    }

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    static_for<2 * KB>([&](auto X) __attribute__((always_inline)) {
        constexpr int role = decltype(X)::value / KB, sb = decltype(X)::value % KB;
        const Tensor& t = role ? p.dk1 : p.dv1;
        const float sc = role ? LN2 : 1.f;               // Q~ carries scale*log2(e)
        const int j = jw + 32 * sb + ln;
        if (!t.p) return;
        uint16_t* dst = (uint16_t*)t.p + t.off(b, j < N ? j : N - 1, h) + 4 * hf;
        // (split: fp32 partial of this share: [dK | dV][split][batch*head][position][column])
        const int64_t BH = (int64_t)p.B * p.H;
        float* pdst = nsplit > 1 ? part + ((((role ? 0 : 1) * (int64_t)nsplit + sp) * BH + bh) * N + (j < N ? j : N - 1)) * D + 4 * hf : nullptr;
        static_for<4 * DT>([&](auto Y) __attribute__((always_inline)) {
            constexpr int dt = decltype(Y)::value / 4, g4 = decltype(Y)::value % 4, at = (role ? DK0 : DV0) + (sb * DT + dt) * 16 + 4 * g4;
            const float4 x = L::get_regs<at>();
            const float x0 = x.x * sc, x1 = x.y * sc, x2 = x.z * sc, x3 = x.w * sc;
            if (j >= N) return;
            if (nsplit > 1) {
                *(float4*)(pdst + dt * 32 + 8 * g4) = make_float4(x0, x1, x2, x3);
            } else {
                if (PAD && dt * 32 + 8 * g4 >= p.D) return;
                *(uint2*)(dst + dt * 32 + 8 * g4) = make_uint2(pack2<E>(x0, x1), pack2<E>(x2, x3));
            }
        });
    });
}

template <class E, int D, int KB, bool PAD>
int launch_kv_geometry(const Problem& p, int nsplit, hipStream_t st, BwdSums* sums) {
    using C = KvCfg<D, KB>;
    const int njb = (p.N + C::VJ - 1) / C::VJ;
    const int64_t total = (int64_t)njb * p.B * p.H * nsplit;
    if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    const bool seg = !C::fits(p.w2), bias = p.k2_bias != 0.f || p.v2_bias != 0.f;
    const int ws = p.w2 < C::max_segment() ? p.w2 : C::max_segment();
    const size_t lds = C::lds_bytes(ws, seg);
    // the partial sums of a split launch lie behind the K'-side kernel's part of the workspace
    float* part = nullptr;
    if (nsplit > 1) {
        const size_t off = kp_side_scratch_bytes(p.B, p.N, p.H, D, p.w1, p.w2, p.room);
        if (p.scratch_bytes < off + kv_split_scratch_bytes(p.B, p.N, p.H, D, p.w1, p.w2, p.room)) return SA2_ERR_WORKSPACE_TOO_SMALL;
        part = (float*)((char*)p.scratch + off);
    }
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return false;
        hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(VT), lds, st, p, njb, (int)total, nsplit, part, ws);
        return true;
    };
    // (the segmented kernel exists with the bias adds only)
    const bool ok = seg    ? go(mfma_bwd_kv_kernel<E, D, true, KB, true, PAD>)
                    : bias ? go(mfma_bwd_kv_kernel<E, D, true, KB, false, PAD>)
                           : go(mfma_bwd_kv_kernel<E, D, false, KB, false, PAD>);
    if (!ok) return SA2_ERR_LAUNCH_FAILED;
    if (hipGetLastError() != hipSuccess) return SA2_ERR_LAUNCH_FAILED;
    sums->kv = part;
    sums->kv_n = nsplit;
    return SA2_OK;
}

// kb: 32-row blocks of K/V rows per wavefront
template <class E>
int launch_kv(const Problem& p, int kb, int nsplit, hipStream_t st, BwdSums* sums) {
    if (p.D == 128) return launch_kv_geometry<E, 128, 1, false>(p, nsplit, st, sums);
    if (p.D == 64)
        return kb == 2 ? launch_kv_geometry<E, 64, 2, false>(p, nsplit, st, sums) : launch_kv_geometry<E, 64, 1, false>(p, nsplit, st, sums);
    return kb == 2 ? launch_kv_geometry<E, 32, 2, true>(p, nsplit, st, sums) : launch_kv_geometry<E, 32, 1, true>(p, nsplit, st, sums);
}

}  // namespace
}  // namespace sa2
