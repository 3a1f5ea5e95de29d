// The forward kernel of the plane-split kernels with two units per wavefront and one wavefront per SIMD; included once per element type.
// Arithmetic, shares and the cases that are computed by rows are those of split_fwd_kernel (sa2_split_mfma.hip), which says what a unit and a
// plane are; how a tile of planes lies in LDS and what NQ is (there NU) stands in sa2_split_kv_lone.h.
//
// A workgroup owns 32 queries.  Four wavefronts hold two units (consecutive deltas) each per round, Q~ and the R tiles in accumulation
// registers (sa2_mfma_lone.h), and sweep the K window from the queries' own tile down, in 32-key tiles.  Per tile a wavefront computes
//   A(0), C'(1), A(1), C(0):  A: S^T = K1.Q~^T - m,  C: R^T += V1^T.P^T  with P = exp2(S^T) split into planes  (C' of the tile before)
// with a unit's exponentials, sums and splits between the MFMAs of the other one.  Tiles of one plane come straight from global memory into a
// ring of three; others are split by all threads between the MFMAs, one tile ahead, into a ring of two.  K' and V' rows lie in a ring of 64,
// eight new ones a round.  Running sums of R * (v2 + bias) stay in registers for all rounds and the wavefronts are merged once.
//
// What bounds it: the instructions beside the MFMAs (fp32 head_dim 64: 98 MFMAs, 520 others in a tile's 4500 cycles; bf16 at 96 columns 62 and
// 380).  Forward, us, one unit per wavefront (eight of them at 64 columns, four at 96) / this: bf16 B1 H8 N2048 D96 w 255/31 330 / 141, fp16 D80 393 / 219,
// fp32 B2 H8 N2048 D64 w 512/32 795 / 737, bf16 B2 H4 N2048 D40 w 255/31 143 / 113.
//
// The reference point m of a row is the largest logit of the wavefront's first two units in the queries' own tile, which holds a key of every
// row.  A logit less m is rounded at the size of the difference.  So the largest logit S of each further tile is looked at before the
// exponentials, and a unit's sums are brought to a reference point there where S - m is more than 8 octaves and more than twice |S|, at whose size S is
// rounded in any case, or more than 40 octaves (weights and their sums stay far from overflow until then; a block whose sums of values do not
// is computed by rows).  The tile's logits are then formed again without m, by a branch that usual logits hardly take (with eight times their
// spread the first two sizes above take 165 and 245).  With keys of the own tile 15, 30, 1e3 and 1e5 octaves below the row's others
// and only a step at 64 octaves, taken off the rounded difference, fp32 outputs were 1.6, 2.4, 39 and 4800 times as far from fp64 as with a
// maximum taken per tile; now they are as far (0.97).
#pragma once

#include "sa2_fma_rows.h"
#include "sa2_split_lone.h"

namespace sa2 {
namespace {

template <class T, int D, int NQ>
struct SplitFwdLoneCfg {
    static constexpr int W = 4, THREADS = W * 64, U = 2, UPR = U * W;          // units of a wavefront and of a round
    static constexpr int NK = T::PLANES, DK = D / 16, DT = D / 32;
    static constexpr bool DMA = NK == 1;       // tiles straight from global memory
    static constexpr int BLOCK = 2048, PLANE = DT * BLOCK, TILE = NK * PLANE, STAGE = 2 * TILE, NSTAGE = DMA ? 3 : 2;      // bytes
    static constexpr int AS = D + 4, SLOTS = 64;                               // fp32 row stride of the merged sums; rows of the K' and V' rings
    static constexpr size_t row_bytes(int rows) { return (size_t)(rows / 4) * QuadTile<128>::GROUP; }
    static constexpr size_t TILES = (size_t)NSTAGE * STAGE, ROWS = row_bytes(BQ) + 2 * row_bytes(SLOTS);       // q, K', V'
    static constexpr size_t larger(size_t a, size_t b) { return a > b ? a : b; }
    static constexpr size_t X_AT = larger(larger(TILES + ROWS, (size_t)W * BQ * AS * 4), smem_bytes(D, W));
    static constexpr size_t LDS_BYTES = X_AT + 2 * W * BQ * 4;
    // accumulation registers: R tiles, planes of Q~, the reference point's.  (It comes off the logits last, by an MFMA of its planes, which costs
    // one rounding at the size of the result.  A chain that starts from it rounds every step at its size.)
    static constexpr int R0 = 0, Q0 = U * DT * 16, M0 = Q0 + U * NQ * DK * 4, USED = M0 + U * 4, OWNED = USED <= 96 ? 96 : USED <= 192 ? 192 : 256;
    static_assert(USED <= 256 && LDS_BYTES <= 160 * 1024, "");
};

template <class T, int D, int NQ, int MODE, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void split_fwd_lone_kernel(Problem p, int nqb, int total) {
    using C = SplitFwdLoneCfg<T, D, NQ>;
    using L = Lone<C::OWNED>;
    typedef typename T::T EL;
    typedef typename T::Raw Raw;
    typedef bf16x8 X8;
    constexpr bool PAD = MODE != EXACT;
    constexpr int DK = C::DK, DT = C::DT, NK = C::NK, KW = C::W, KT = C::THREADS, UPR = C::UPR;
    constexpr int CHUNK = 16 / (int)sizeof(EL);               // elements of a 16-byte chunk
    constexpr int R0 = C::R0, Q0 = C::Q0;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    unsigned char* q_s = smem_raw + C::TILES;                 // q rows of the block
    unsigned char* k2_s = q_s + C::row_bytes(BQ);             // K' rows, ring
    unsigned char* v2_s = k2_s + C::row_bytes(C::SLOTS);      // V' rows, ring
    float* mrg_m = (float*)(smem_raw + C::X_AT);              // [KW][BQ] reference points
    float* mrg_l = mrg_m + KW * BQ;                           // [KW][BQ] sums

    auto here = [&]() __attribute__((always_inline)) {        // (lane parts of what happens once per round are computed there)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    const int tid = here();
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
    const int i0 = qb * BQ, i_last = i0 + BQ - 1 < N - 1 ? i0 + BQ - 1 : N - 1;

    const EL* qp = (const EL*)p.q.p + p.q.off(b, 0, h);
    const EL* k1p = (const EL*)p.k1.p + p.k1.off(b, 0, h);
    const EL* k2p = (const EL*)p.k2.p + p.k2.off(b, 0, h);
    const EL* v1p = (const EL*)p.v1.p + p.v1.off(b, 0, h);
    const EL* v2p = (const EL*)p.v2.p + p.v2.off(b, 0, h);
    const float qscale = p.scale * LOG2E;

    const int n_units = (w2 < i_last ? w2 : i_last) + 1;
    const int all_rounds = (n_units + UPR - 1) / UPR;
    const int per_share = SPLIT ? ((w2 + UPR) / UPR + p.nsplit - 1) / p.nsplit : all_rounds;
    const int round0 = SPLIT ? share * per_share : 0;
    const int round1 = round0 + per_share < all_rounds ? round0 + per_share : all_rounds;
    if (SPLIT && round0 >= round1) {                          // a block near the start of the sequence has fewer rounds
        if (tid < BQ && i0 + tid < N)
            ((float2*)p.scratch)[(int64_t)share * p.B * p.H * N + (int64_t)bh * N + i0 + tid] = make_float2(-INFINITY, 0.f);
        return;
    }
    // tiles of every sweep, from jt_hi down to jt_lo; [p_lo, jt_hi - 1] need no mask
    const int jt_hi = qb, jt_lo = (i0 - w1 > 0 ? i0 - w1 : 0) / TJ;
    const int p_lo = i0 + BQ - 1 - w1 > 0 ? (i0 + BQ - 1 - w1 + TJ - 1) / TJ : 0;

    // ---- tiles, in the order of the sweeps (what is requested behind the last one nothing reads) ----
    const uint32_t lds0 = lds_address(smem_raw);
    const int64_t k_step = (int64_t)TJ * p.k1.sn, v_step = (int64_t)TJ * p.v1.sn;
    const EL *const k_top = k1p + jt_hi * k_step, *const v_top = v1p + jt_hi * v_step;
    const EL *k_next = k_top, *v_next = v_top;                // first rows of the next tile
    int next_tile = jt_hi;
    auto next = [&]() __attribute__((always_inline)) {
        const bool wrap = next_tile == jt_lo;
        next_tile = wrap ? jt_hi : next_tile - 1;
        k_next = wrap ? k_top : k_next - k_step;
        v_next = wrap ? v_top : v_next - v_step;
    };
    const int most_hi = N - 1 - i0;                           // rows past the end of the sequence in tile jt_hi read the last one
    // one plane: straight to LDS, in pieces of 16 rows by 64 bytes (a wavefront instruction), dealt over the wavefronts
    constexpr int PIECES = 2 * DT, NREQ = C::DMA ? 2 * PIECES / KW : 0;
    static_assert(!C::DMA || 2 * PIECES % KW == 0, "");
    const bool near_end = most_hi < TJ - 1;
    int64_t piece_off[C::DMA ? NREQ : 1];                     // bytes from the tile's first row to the lane's chunk
    auto aim = [&](int jt) __attribute__((always_inline)) {
        const int l = here() & 63, most = jt == jt_hi ? most_hi : TJ - 1;
#pragma unroll
        for (int n = 0; n < NREQ; ++n) {
            const int piece = wave + KW * n, vs = piece >= PIECES, x = piece - vs * PIECES;        // (uniform)
            const int row = 16 * (x & 1) + (l >> 2), col = (x >> 1) * 32 + ((l & 3) ^ (l >> 4 & 3)) * 8;
            // (columns from p.D on meet zeros of the unit, or are not written)
            piece_off[n] = ((row < most ? row : most) * (vs ? p.v1.sn : p.k1.sn) + (PAD && col >= p.D ? 0 : col)) * (int64_t)sizeof(EL);
        }
    };
    auto request_piece = [&](auto X, uint32_t stage) __attribute__((always_inline)) {
        constexpr int n = decltype(X)::value;
        const int piece = wave + KW * n, vs = piece >= PIECES, x = piece - vs * PIECES;
        const char* base = (const char*)(vs ? v_next : k_next);
        lds_request(base + piece_off[n], stage + (uint32_t)(vs * C::TILE + (x >> 1) * C::BLOCK + (x & 1) * 1024));
    };
    auto request_tile = [&](uint32_t stage) __attribute__((always_inline)) {
        static_for<NREQ>([&](auto X) __attribute__((always_inline)) { request_piece(X, stage); });
    };
    // more planes: through registers.  Thread t brings the columns 32*dt + 4*(t % 8) .. of row t / 8.
    const int s_row = tid >> 3, s_col = (tid & 7) * 4;
    const uint32_t s_lane = (uint32_t)(s_row * 64 + (((tid & 7) >> 1) ^ (s_row >> 2 & 3)) * 16 + (tid & 1) * 8);
    Raw tk[DT], tv[DT];
    int64_t k_off = s_row * p.k1.sn, v_off = s_row * p.v1.sn; // elements from the tile's first row to the thread's
    auto load_tile = [&]() __attribute__((always_inline)) {
        if (near_end) {
            const int most = next_tile == jt_hi ? most_hi : TJ - 1, j = s_row < most ? s_row : most;
            k_off = j * p.k1.sn;
            v_off = j * p.v1.sn;
        }
        const EL *ks = k_next + k_off, *vs = v_next + v_off;
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

    // ---- rows, laid out as a tile of 256-byte rows (sa2_mfma_common.h); K' and V' row k at slot (k - i0 + 7) % 64, so that a round's
    // eight new rows are whole groups ----
    using Q4 = QuadTile<128>;
    auto chunk = [&](const unsigned char* rows, int r, int c) __attribute__((always_inline)) { return rows + Q4::row_off(r) + c / 4 * Q4::BLOCK + c % 4 * 16; };
    auto request_group = [&](const EL* base, int64_t sn, int row0, const unsigned char* to) __attribute__((always_inline)) {          // four rows
        const int l = here() & 63, col = Q4::dma_chunk(l) * CHUNK, r = row0 + Q4::dma_row(l), rc = r < 0 ? 0 : (r < N ? r : N - 1);
        const void* src = col < p.D ? (const void*)(base + (int64_t)rc * sn + col) : (const void*)zero_chunk;
        lds_request(src, lds0 + (uint32_t)(to - smem_raw));
    };
    auto request_octet = [&](int rel) __attribute__((always_inline)) {              // rel = k - i0 + 7 of the first, a multiple of 8
        const int g = wave & 1, vs = wave >> 1, at = ((rel & (C::SLOTS - 1)) / 4 + g) * Q4::GROUP;
        request_group(vs ? v2p : k2p, vs ? p.v2.sn : p.k2.sn, i0 - 7 + rel + 4 * g, (vs ? v2_s : k2_s) + at);
    };
    auto slot_of = [&](int ln_, int delta) __attribute__((always_inline)) { return (ln_ + 7 - delta) & (C::SLOTS - 1); };
    auto copy4 = [&](const unsigned char* rows, int r, int hf_, int e) __attribute__((always_inline)) {       // four columns from 8*e + 4*hf on
        if constexpr (sizeof(EL) == 4) return *(const Raw*)chunk(rows, r, 2 * e + hf_);
        else return *(const Raw*)(chunk(rows, r, e) + hf_ * 8);
    };
    struct Eight { Raw a, c; };
    auto copy8 = [&](const unsigned char* rows, int r, int hf_, int kk) __attribute__((always_inline)) {      // eight from 16*kk + 8*hf on
        if constexpr (sizeof(EL) == 4) {
            const unsigned char* at = chunk(rows, r, 4 * kk + 2 * hf_);
            return Eight{*(const Raw*)at, *(const Raw*)(at + 16)};
        } else {
            const uint4 x = *(const uint4*)chunk(rows, r, 2 * kk + hf_);
            return Eight{__builtin_bit_cast(Raw, make_uint2(x.x, x.y)), __builtin_bit_cast(Raw, make_uint2(x.z, x.w))};
        }
    };
    {
        for (int g = wave; g < BQ / 4; g += KW) request_group(qp, p.q.sn, i0 + 4 * g, q_s + g * Q4::GROUP);
        for (int x = 4; x >= -1; --x) request_octet(8 * (x - round0));
        if constexpr (C::DMA) {
            aim(next_tile);
            request_tile(lds0);
            for (int x = 1; x < C::NSTAGE; ++x) {
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

    // ---- a wavefront's sweep ----
    constexpr Products<NK, NQ> PA;                            // plane of the tile, of Q~
    constexpr Products<NK, 3> PC;                             // plane of the tile, of P
    constexpr int NP = PA.n, NC = PC.n;
    constexpr int NA = NP * DK + 1, NE = 2 * DT, NV = NE * NC;           // MFMAs of a phase A; V operands; MFMAs of a phase C
    constexpr int P2 = NA, P3 = NA + NV, P4 = 2 * NA + NV, NS = 2 * (NA + NV);         // slots of a tile: A(0), C'(1), A(1), C(0)
    constexpr int AHEAD = NP >= 5 ? 1 : NP == 3 ? 2 : 3;      // k-steps that row operands are read ahead
    static_assert(AHEAD <= DK, "");
    X8 ro[AHEAD + 1][NK], vt[NE][NK];
    floatx16 s[2], nl;                                        // logits; what their chains start from: 0, -inf where the key is outside the window
    float m[2];                                               // reference points of the units (of the logits as the chains give them)
    const float octaves = NQ == 2 ? qscale : 1.f, near = 8.f / octaves, far = 40.f / octaves;
    const X8 ones = lead_ones(hf);
    u4 pw[2][2][3];                                           // planes of the weights: unit, half of the keys
    float l[2], rs[2];                                        // sums of the weights: of the sweep, of the tile
    floatx16 wacc[DT];                                        // sum of R * (v2 + bias) over the wavefront's units
    float Mw = 0.f, Lw = 0.f;                                 // its reference point and sum of weights
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) wacc[dt] = zero16();
    uint32_t sa = lds0, sb = lds0 + C::STAGE, sc = lds0 + (C::NSTAGE - 1) * C::STAGE;         // stages of tiles t, t+1 and (three) t+2
    const uint32_t row_lane = (uint32_t)(ln * 64 + (hf ^ (ln >> 2 & 3)) * 16);
    const uint32_t col_lane = [&]() {
        const int grp = lane >> 4, x = lane & 15, r = 4 * (grp >> 1) + (x >> 2), c = 2 * (grp & 1) + ((x & 3) >> 1);
        return (uint32_t)(r * 64 + (c ^ (r >> 2)) * 16 + (x & 1) * 8);
    }();
    uint32_t r0 = 0, r1 = 0, c0 = 0, c1 = 0;                  // the lane's addresses in a stage, for even and odd k-steps and slices of eight rows
    static_assert(C::STAGE % 64 == 0, "");
    auto at_stage = [&](uint32_t stage, uint32_t part, uint32_t& even, uint32_t& odd) __attribute__((always_inline)) {
        even = stage + part;
        odd = even ^ 32u;
        stays(even);
        stays(odd);
    };
    auto read_row = [&](auto KK, auto X) __attribute__((always_inline)) {
        constexpr int kk = decltype(KK)::value, x = decltype(X)::value;
        ro[kk % (AHEAD + 1)][x] = lds_read_x8<X8>((kk & 1 ? r1 : r0) + (uint32_t)(x * C::PLANE + kk / 2 * C::BLOCK));
    };
    auto read_first_rows = [&]() __attribute__((always_inline)) {
        static_for<AHEAD * NK>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(decltype(X)::value / NK), LONE_C(decltype(X)::value % NK)); });
    };
    auto read_column = [&](auto EN, auto X) __attribute__((always_inline)) {        // entry e: half e / DT of the keys, column block e % DT
        constexpr int e = decltype(EN)::value, x = decltype(X)::value, ks = e / DT, dt = e % DT;
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef v4s __attribute__((address_space(3)))* lds_v4s;
        constexpr uint32_t at = C::TILE + x * C::PLANE + dt * C::BLOCK + ks * 1024;
        union { v4s half[2]; X8 v; } u;
        u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c0 + at));
        u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(c1 + at + 512));
        vt[e][x] = u.v;
    };
    auto a_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value;
        if constexpr (i == NP * DK) {
            L::template tile_more<C::M0 + 4 * u>(s[u], ones);
        } else {
            constexpr int kk = i / NP, x = PA.x[i % NP], y = PA.y[i % NP], at = Q0 + ((u * NQ + y) * DK + kk) * 4;
            if constexpr (i == 0) L::template tile_start<at>(s[u], ro[0][x], nl);
            else L::template tile_more<at>(s[u], ro[kk % (AHEAD + 1)][x]);
        }
    };
    auto a_reads = [&](auto I) __attribute__((always_inline)) {                     // the rows read beside MFMA i of a phase A
        constexpr int kk = decltype(I)::value / NP, m = decltype(I)::value % NP;
        if constexpr (kk + AHEAD < DK) deal<NK, m, NP>([&](auto X) __attribute__((always_inline)) { read_row(LONE_C(kk + AHEAD), X); });
    };
    auto c_mfma = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, i = decltype(I)::value, e = i / NC, ks = e / DT, dt = e % DT, x = PC.x[i % NC], y = PC.y[i % NC];
        L::template sum_more<R0 + (u * DT + dt) * 16>(vt[e][x], __builtin_bit_cast(X8, pw[u][ks][y]));
    };
    // Softmax items of a unit, 24 for each half of the keys: an exponential and the share of the element before it in the sum, then the
    // split of a word's planes in four steps.  (An exponential's result may not be read by the next instruction.)
    float sh[2][2];
    constexpr int ITEMS = 48;
    auto item = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, ks = decltype(I)::value / 24, j = decltype(I)::value % 24;
        if constexpr (j < 8) {
            constexpr int e = 8 * ks + j;
            float x = fast_exp2(NQ == 2 ? s[u][e] * qscale : s[u][e]);
            stays(x);
            s[u][e] = x;
        } else {
            split_word_step<decltype(LONE_C(ks))::value, j - 8>(s[u], pw[u][ks], sh[u]);
        }
    };
    // (the sums: beside the exponentials they would wait for them)
    auto sum_item = [&](auto UN, auto I) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value, e = decltype(I)::value;
        if constexpr (e == 0) rs[u] = s[u][0];
        else rs[u] += s[u][e];
        if constexpr (e == 15) {
            l[u] += rs[u];
            stays(l[u]);
        } else if constexpr (e > 0) {
            stays(rs[u]);
        }
    };
    // The items of a unit take half of the slots of a tile, from the fifth MFMA behind its phase A on.  Element e joins the sum after
    // its exponential and before its word is split.
    constexpr int HALF = NA + NV - 2;
    auto softmax = [&](auto UN, auto SLOT) __attribute__((always_inline)) {
        deal<ITEMS, decltype(SLOT)::value, HALF>([&](auto X) __attribute__((always_inline)) {
            constexpr int x = decltype(X)::value, ks = x / 24, j = x % 24;
            if constexpr (j >= 1 && j < 8) sum_item(UN, LONE_C(8 * ks + j - 1));
            if constexpr (j == 8) sum_item(UN, LONE_C(8 * ks + 7));
            item(UN, X);
        });
    };
    auto set_reference = [&](auto UN) __attribute__((always_inline)) {              // the planes of m
        constexpr int u = decltype(UN)::value;
        const u4 w = __builtin_bit_cast(u4, lead_planes(m[u], 0.f));
        L::template set_regs<C::M0 + 4 * u>(w[0], w[1], w[2], w[3]);
        asm volatile("s_nop 3" ::: "memory");
    };
    // In two parts, behind the third and fourth MFMA after the unit's phase A: the largest of its logits (relative to m), and what is to be
    // done where it is too large.  The unit's R tiles and sum are complete then but for this tile.
    float top = 0.f;
    auto max3 = [](float a, float b, float c) __attribute__((always_inline)) {
        float r;
        asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
        return r;
    };
    // Tile jt_now's logits of a unit, without the reference point, from K rows in global memory: their stage may be written again by now.
    int jt_now = jt_hi;
    auto form_logits = [&](auto UN) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value;
        const int t = here(), j = jt_now * TJ + (t & 31);
        const EL* row = k1p + (int64_t)(j < N ? j : N - 1) * p.k1.sn;
        constexpr int GROUP = NK == 1 ? DK : NK == 2 && D == 64 ? 2 : 1;      // k-steps whose loads are under way together: what registers there are
        static_assert(DK % GROUP == 0, "");
        static_for<DK / GROUP>([&](auto GR) __attribute__((always_inline)) {
            Raw x[GROUP][2];
#pragma unroll
            for (int g = 0; g < GROUP; ++g) {
                const int col = (decltype(GR)::value * GROUP + g) * 16 + (t >> 5 & 1) * 8;
                x[g][0] = raw4<T, PAD>(row, col, p.D);
                x[g][1] = raw4<T, PAD>(row, col + 4, p.D);
            }
            __builtin_amdgcn_sched_barrier(0);
            static_for<GROUP>([&](auto KK) __attribute__((always_inline)) {
                constexpr int kk = decltype(GR)::value * GROUP + decltype(KK)::value;
                const fx4 a = T::widen(x[decltype(KK)::value][0]), c = T::widen(x[decltype(KK)::value][1]);
                const float y[8] = {a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
                X8 k[NK];
                split8<NK, T::DTYPE == SA2_F32>(y, k);
#pragma unroll
                for (int n = 0; n < NK; ++n) asm volatile("s_nop 3" : "+v"(k[n]));
                static_for<NP>([&](auto I) __attribute__((always_inline)) {
                    constexpr int i = decltype(I)::value, at = Q0 + ((u * NQ + PA.y[i]) * DK + kk) * 4;
                    if constexpr (kk == 0 && i == 0) L::template tile_start<at>(s[u], k[PA.x[i]], nl);
                    else L::template tile_more<at>(s[u], k[PA.x[i]]);
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        finished(s[u], nl);
    };
    auto watch = [&](auto UN, auto PART) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value;
        if constexpr (decltype(PART)::value == 0) {
            top = max3(max3(max3(max3(s[u][0], s[u][1], s[u][2]), s[u][3], s[u][4]), s[u][5], s[u][6]), s[u][7], s[u][8]);
            stays(top);
        } else {
            top = max3(max3(max3(max3(top, s[u][9], s[u][10]), s[u][11], s[u][12]), s[u][13], s[u][14]), s[u][15], s[u][15]);
            auto too_large = [&](float x) __attribute__((always_inline)) { return x > __builtin_amdgcn_fmed3f(near, far, 2.f * fabsf(m[u] + x)); };
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(too_large(top)) != 0, 0)) {
                const bool move = too_large(fmaxf(top, other_half(top)));
                form_logits(UN);
                float best = s[u][0];
#pragma unroll
                for (int v = 1; v < 16; ++v) best = fmaxf(best, s[u][v]);
                best = fmaxf(best, other_half(best));
                const float alpha = move ? fast_exp2((m[u] - best) * octaves) : 1.f;
                m[u] = move ? best : m[u];
                l[u] *= alpha;
                set_reference(UN);
                L::template tile_more<C::M0 + 4 * u>(s[u], ones);
                finished(s[u], nl);
                static_for<DT * 4>([&](auto X) __attribute__((always_inline)) {
                    constexpr int r = R0 + u * DT * 16 + 4 * decltype(X)::value;
                    const float4 x = L::template get_regs<r>();
                    L::template set_regs<r>(__float_as_uint(x.x * alpha), __float_as_uint(x.y * alpha), __float_as_uint(x.z * alpha), __float_as_uint(x.w * alpha));
                });
            }
        }
    };
    constexpr int STAGED = P4 - 8;                            // the slot by which tile t+1 is staged
    auto beside = [&](auto SLOT, auto CC0, uint32_t stage_at) __attribute__((always_inline)) {
        constexpr int slot = decltype(SLOT)::value;
        // unit 0: from P2 + 4 on; unit 1: from P4 + 4 on, into the next tile
        if constexpr (slot == P2 + 2 || slot == P2 + 3) watch(LONE_C(0), LONE_C(slot - (P2 + 2)));
        if constexpr (slot == P4 + 2 || slot == P4 + 3) watch(LONE_C(1), LONE_C(slot - (P4 + 2)));
        softmax(LONE_C(0), LONE_C(slot - (P2 + 4)));
        if constexpr (slot >= P4 + 4) softmax(LONE_C(1), LONE_C(slot - (P4 + 4)));
        else if constexpr (decltype(CC0)::value) softmax(LONE_C(1), LONE_C(slot + NS - (P4 + 4)));
        if constexpr (!C::DMA) {
            deal<NF * STEPS, slot - NA / 2, STAGED - NA / 2>([&](auto X) __attribute__((always_inline)) { stage_step(X, stage_at); });
            if constexpr (slot == STAGED) {
                next();
                load_tile();
            }
        }
    };
    // tile t+1 is in LDS for all, tile t was read to the end
    auto tile_barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::DMA ? NREQ : 63) : "memory"); };
    auto tile = [&](auto DO_C) __attribute__((always_inline)) {
        constexpr bool CC = decltype(DO_C)::value;            // (the first tile of a sweep has no tile before it)
        uint32_t stage_at = sb + s_lane;
        if constexpr (!C::DMA) stays(stage_at);
        at_stage(sa, col_lane, c0, c1);
        static_for<NA>([&](auto I) __attribute__((always_inline)) {                 // A(t, 0)
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(0), I);
            a_reads(I);
            if constexpr (!CC) deal<NE * NK, i, NA>([&](auto X) __attribute__((always_inline)) { read_column(LONE_C(decltype(X)::value / NK), LONE_C(decltype(X)::value % NK)); });
            beside(I, DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!CC) finished(s[0], nl);
        // V operand e is read again behind its last MFMA
        auto columns_behind = [&](auto J) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value - 1, e = j / NC - 1, x = j % NC;
            if constexpr (CC && e >= 0 && e < NE && x < NK) read_column(LONE_C(e), LONE_C(x));
        };
        static_for<NV>([&](auto I) __attribute__((always_inline)) {                 // C(t-1, 1)
            constexpr int i = decltype(I)::value;
            if constexpr (CC) c_mfma(LONE_C(1), I);
            columns_behind(I);
            constexpr int first = NV - AHEAD * NK - 2;
            if constexpr (i >= first && i < first + AHEAD * NK) read_row(LONE_C((i - first) / NK), LONE_C((i - first) % NK));
            beside(LONE_C(P2 + i), DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NA>([&](auto I) __attribute__((always_inline)) {                 // A(t, 1)
            a_mfma(LONE_C(1), I);
            a_reads(I);
            columns_behind(LONE_C(NV + decltype(I)::value));
            beside(LONE_C(P3 + decltype(I)::value), DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        tile_barrier();
        at_stage(sb, row_lane, r0, r1);
        if constexpr (C::DMA) {
            next();
            if (near_end) aim(next_tile);
        }
        static_for<NV>([&](auto I) __attribute__((always_inline)) {                 // C(t, 0)
            constexpr int i = decltype(I)::value, first = NV - AHEAD * NK - 2;
            c_mfma(LONE_C(0), I);
            if constexpr (i >= first && i < first + AHEAD * NK) read_row(LONE_C((i - first) / NK), LONE_C((i - first) % NK));
            if constexpr (C::DMA) deal<NREQ, i - 2, NV - 4>([&](auto X) __attribute__((always_inline)) { request_piece(X, sa); });
            beside(LONE_C(P4 + i), DO_C, stage_at);
            __builtin_amdgcn_sched_barrier(0);
        });
        stays(s[1]);
    };
    auto last_sums = [&]() __attribute__((always_inline)) {                         // C(t, 1) of the last tile
        static_for<P2 + 2>([&](auto I) __attribute__((always_inline)) { softmax(LONE_C(1), LONE_C(decltype(I)::value + NS - (P4 + 4))); });
        static_for<NV>([&](auto I) __attribute__((always_inline)) {
            // (the last items, which a tile has beside the first MFMAs here)
            c_mfma(LONE_C(1), I);
        });
    };
    // One unit per wavefront (the last round of a share, where four units or less are left): half the MFMAs, one after the other
    auto solo = [&]() __attribute__((always_inline)) {
        at_stage(sa, row_lane, r0, r1);
        at_stage(sa, col_lane, c0, c1);
        read_first_rows();
        static_for<NA>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            a_mfma(LONE_C(0), I);
            a_reads(I);
            deal<NE * NK, i, NA>([&](auto X) __attribute__((always_inline)) { read_column(LONE_C(decltype(X)::value / NK), LONE_C(decltype(X)::value % NK)); });
            __builtin_amdgcn_sched_barrier(0);
        });
        finished(s[0], nl);
        watch(LONE_C(0), LONE_C(0));
        watch(LONE_C(0), LONE_C(1));
        static_for<HALF>([&](auto SLOT) __attribute__((always_inline)) { softmax(LONE_C(0), SLOT); });
        asm volatile("s_nop 3" ::: "memory");
        static_for<NV>([&](auto I) __attribute__((always_inline)) { c_mfma(LONE_C(0), I); });
    };
    auto advance_tile = [&]() __attribute__((always_inline)) {                      // a tile without MFMAs, or behind them
        if constexpr (!C::DMA) {
            stage_all(sb);
            next();
            load_tile();
        }
        tile_barrier();
        if constexpr (C::DMA) {
            next();
            if (near_end) aim(next_tile);
            request_tile(sa);
        }
    };
    auto rotate = [&]() __attribute__((always_inline)) {
        L::keep_out();
        const uint32_t x = sa;
        sa = sb;
        if constexpr (C::NSTAGE == 3) {
            sb = sc;
            sc = x;
        } else {
            sb = x;
        }
    };
    // keys of tile jt inside the window of the lane's row: bit c is key 32 * jt + 4*hf + c, element v of a tile is key 8*(v/4) + v%4 + 4*hf
    auto keys_seen = [&](int jt) __attribute__((always_inline)) {
        const int t = here(), hi = i0 + (t & 31) - jt * TJ - 4 * (t >> 5 & 1), lo = hi - w1;
        uint32_t seen = 0;
        if (hi >= 0 && lo < TJ) seen = (hi >= TJ - 1 ? ~0u : (2u << hi) - 1) & (lo > 0 ? ~0u << lo : ~0u);
        return seen;
    };
    bool unmasked = false;
    auto enter_tile = [&](int jt) __attribute__((always_inline)) {                  // the start of the S tiles of tile jt
        const bool plain = jt >= p_lo && jt < jt_hi;
        if (plain && unmasked) return;
        unmasked = plain;
        const uint32_t seen = plain ? ~0u : keys_seen(jt);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            int x = (int)(seen << (31 - 8 * (v >> 2) - (v & 3))) >> 31;
            asm("" : "+v"(x));
            nl[v] = __int_as_float(__float_as_int(-INFINITY) & ~x);
        }
        asm volatile("s_nop 3" : "+v"(nl));
    };
    // the units' logits in the tile at sa and their largest ones, where the lane's row has a key; the others become -inf
    auto tile_logits = [&](int jt, int d0, float (&mx)[2]) __attribute__((always_inline)) {
        const int t = here(), i = i0 + (t & 31);
        const uint32_t seen = keys_seen(jt);
        nl = zero16();
        asm volatile("s_nop 3" : "+v"(nl));
        at_stage(sa, row_lane, r0, r1);
        static_for<2>([&](auto UN) __attribute__((always_inline)) {
            static_for<DK>([&](auto KK) __attribute__((always_inline)) {
                static_for<NK>([&](auto X) __attribute__((always_inline)) { read_row(KK, X); });
                static_for<NP>([&](auto M) __attribute__((always_inline)) { a_mfma(UN, LONE_C(decltype(KK)::value * NP + decltype(M)::value)); });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        finished(s[0], s[1]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
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
    for (int t = 0; t < 8; ++t) zero[t] = (__bf16)0.f;
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    for (int round = round0; round < round1; ++round) {
        const bool alone = n_units - round * UPR <= KW;                     // one unit per wavefront
        const int d0 = round * UPR + wave * (alone ? 1 : 2);  // first delta of this wavefront
        const bool any = d0 < n_units;
        request_octet(-8 * (round + 2));
        // ---- Q~ of the round's units (one that does not exist: its neighbour's, and left out of the sums) ----
        asm volatile("s_nop 3" : "+v"(zero));
        static_for<2 * DT>([&](auto X) __attribute__((always_inline)) { L::template sum_zero<R0 + 16 * decltype(X)::value>(zero); });
        {
            const int t = here(), ln_ = t & 31, hf_ = t >> 5 & 1;
            static_for<2 * DK>([&](auto X) __attribute__((always_inline)) {
                constexpr int u = decltype(X)::value % 2, kk = decltype(X)::value / 2;
                const Eight q = copy8(q_s, ln_, hf_, kk), k = copy8(k2_s, slot_of(ln_, d0 + u < n_units ? d0 + u : n_units - 1), hf_, kk);
                const fx4 xa = T::widen(q.a), xc = T::widen(q.c), ya = T::widen(k.a), yc = T::widen(k.c);
                float r[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    r[e] = NQ == 2 ? xa[e] * ya[e] : xa[e] * qscale * (ya[e] + p.k2_bias);
                    r[4 + e] = NQ == 2 ? xc[e] * yc[e] : xc[e] * qscale * (yc[e] + p.k2_bias);
                }
                X8 o[NQ];
                split8<NQ>(r, o);
                static_for<NQ>([&](auto Y) __attribute__((always_inline)) {
                    const u4 w = __builtin_bit_cast(u4, o[decltype(Y)::value]);
                    L::template set_regs<Q0 + ((u * NQ + decltype(Y)::value) * DK + kk) * 4>(w[0], w[1], w[2], w[3]);
                });
            });
        }
        l[0] = l[1] = 0.f;
        L::keep_out();
        asm volatile("s_nop 3" ::: "memory");
        if (!any) {                                           // no unit for this wavefront in this round: keep the tiles moving
            for (int jt = jt_hi; jt >= jt_lo; --jt) {
                advance_tile();
                rotate();
            }
            continue;
        }
        if (round == round0) {
            float mx[2];
            tile_logits(jt_hi, d0, mx);
            Mw = fmaxf(mx[0], mx[1]);
            // (No key here: none of the row's sums are taken.  Logits that are all -inf: far below any other.)
            const int i = i0 + (here() & 31);
            Mw = Mw != -INFINITY ? Mw : i < N && i >= d0 ? -8.507059173023462e37f : 0.f;
        }
        static_for<2>([&](auto UN) __attribute__((always_inline)) {
            m[decltype(UN)::value] = Mw;
            set_reference(UN);
        });
        {
            unmasked = false;
            if (alone) {
                for (jt_now = jt_hi; jt_now >= jt_lo; --jt_now) {
                    enter_tile(jt_now);
                    solo();
                    advance_tile();
                    rotate();
                }
            } else {
                at_stage(sa, row_lane, r0, r1);
                read_first_rows();
                jt_now = jt_hi;
                enter_tile(jt_now);
                tile(no);
                rotate();
                for (--jt_now; jt_now >= jt_lo;) {
                    enter_tile(jt_now);
                    const int stop = jt_now < p_lo ? jt_now : p_lo;        // tiles down to there need nothing done between them
                    for (; jt_now >= stop; --jt_now) {
                        tile(yes);
                        rotate();
                    }
                }
                last_sums();
            }
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        }

        // ---- the units join the wavefront's running result: sum += weight * (v2 + bias) * R ----
        {
            const int t = here(), ln_ = t & 31, hf_ = t >> 5 & 1, i = i0 + ln_;
            bool row[2];
            float M = Mw;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                row[u] = i < N && i >= d0 + u && d0 + u < n_units && !(u && alone);
                M = row[u] ? fmaxf(M, m[u]) : M;
            }
            auto join = [&](auto WEIGHED) __attribute__((always_inline)) {
                float w[2] = {1.f, 1.f};
                if constexpr (decltype(WEIGHED)::value) {
                    const float a = fast_exp2((Mw - M) * octaves);
#pragma unroll
                    for (int u = 0; u < 2; ++u) w[u] = row[u] ? fast_exp2((m[u] - M) * octaves) : 0.f;
                    Lw *= a;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) wacc[dt] *= a;
                }
                static_for<2>([&](auto UN) __attribute__((always_inline)) {
                    constexpr int u = decltype(UN)::value;
                    if (u && alone) return;
                    const float lt = l[u] + other_half(l[u]);
                    Lw += row[u] ? w[u] * lt : 0.f;
                    const int slot = slot_of(ln_, d0 + u < n_units ? d0 + u : n_units - 1);
                    Raw x[4 * DT];
#pragma unroll
                    for (int e = 0; e < 4 * DT; ++e) x[e] = copy4(v2_s, slot, hf_, e);
                    static_for<4 * DT>([&](auto X) __attribute__((always_inline)) {
                        constexpr int e = decltype(X)::value, v = 4 * (e % 4);
                        float4 r = L::template get_regs<R0 + u * DT * 16 + 4 * e>();
                        r = row[u] ? r : make_float4(0.f, 0.f, 0.f, 0.f);
                        if constexpr (decltype(WEIGHED)::value) r = make_float4(w[u] * r.x, w[u] * r.y, w[u] * r.z, w[u] * r.w);
                        const fx4 y = T::widen(x[e]);
                        floatx16& to = wacc[e / 4];
                        to[v] += r.x * (y[0] + p.v2_bias);
                        to[v + 1] += r.y * (y[1] + p.v2_bias);
                        to[v + 2] += r.z * (y[2] + p.v2_bias);
                        to[v + 3] += r.w * (y[3] + p.v2_bias);
                    });
                });
            };
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(m[0] != Mw || m[1] != Mw) != 0, 0)) join(yes);
            else join(no);
            Mw = M;
        }
        L::keep_out();
    }

    // ---- merge the wavefronts ----
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the last requests: the sums go over the tiles)
    __syncthreads();
    const int tid_m = here(), ln_m = tid_m & 31, hf_m = tid_m >> 5 & 1;
    float* mrg = (float*)smem_raw;                            // [KW][BQ][AS]
    {
        float* row = mrg + (wave * BQ + ln_m) * C::AS + 4 * hf_m;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
                *(float4*)(row + dt * 32 + 8 * g4) = make_float4(wacc[dt][4 * g4], wacc[dt][4 * g4 + 1], wacc[dt][4 * g4 + 2], wacc[dt][4 * g4 + 3]);
        if (hf_m == 0) {
            mrg_m[wave * BQ + ln_m] = Lw > 0.f || Lw != Lw ? Mw * octaves : -INFINITY;      // (a row without a key has no say in the reference)
            mrg_l[wave * BQ + ln_m] = Lw;
        }
    }
    __syncthreads();
    constexpr int TPR = KT / BQ;                              // threads per row
    const int row = tid_m / TPR, io = i0 + row;
    // of the results (see split_fwd_kernel); weights of up to 2^40 may make an infinite sum of values whose mean is finite
    constexpr float MOST = 3.4028234663852886e38f;
    bool bad = false, tiny = false, usual = T::DTYPE != SA2_F32;
    if (io < N) {
        float Mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < KW; ++w) Mx = fmaxf(Mx, mrg_m[w * BQ + row]);
        const float Mu = Mx == -INFINITY ? 0.f : Mx;
        float wgt[KW], Ls = 0.f;
#pragma unroll
        for (int w = 0; w < KW; ++w) {
            wgt[w] = fast_exp2(mrg_m[w * BQ + row] - Mu);
            Ls += mrg_l[w * BQ + row] * wgt[w];
        }
        const int64_t rows = (int64_t)p.B * p.H * N, prow = share * rows + (int64_t)bh * N + io;
        if (SPLIT && tid_m % TPR == 0) ((float2*)p.scratch)[prow] = make_float2(Mx, Ls);
        // The reference points need not be maxima: results in units of 2^e.  sum_w + 1e-8 in units of 2^Me (reference.py:74); for a tiny Me the
        // epsilon dominates
        const int e = __builtin_amdgcn_frexp_expf(Ls);
        const float Me = Mu + (float)e, Le = ldexpf(Ls, -e);
        const bool big = Me > LOG2_EPS;
        const float denom = big ? Le + 1e-8f * fast_exp2(-Me) : Le * fast_exp2(Me - LOG2_EPS) + 1.f;
        const float inv = big ? 1.f / denom : fast_exp2(Me - LOG2_EPS) / denom;
        EL* orow = (EL*)p.out.p + p.out.off(b, io, h);
#pragma unroll
        for (int col = 4 * (tid_m % TPR); col < D; col += 4 * TPR) {
            if (PAD && !SPLIT && col >= p.D) continue;
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < KW; ++w) {
                const float4 y = *(const float4*)(mrg + (w * BQ + row) * C::AS + col);
                acc.x += wgt[w] * y.x; acc.y += wgt[w] * y.y; acc.z += wgt[w] * y.z; acc.w += wgt[w] * y.w;
            }
            const float r[4] = {ldexpf(acc.x, -e) * inv, ldexpf(acc.y, -e) * inv, ldexpf(acc.z, -e) * inv, ldexpf(acc.w, -e) * inv};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bad |= !(fabsf(r[t]) <= MOST);
                if (T::DTYPE == SA2_F32) {
                    usual |= fabsf(r[t]) >= TINY;
                    tiny |= r[t] != 0.f && fabsf(r[t]) < TINY;
                }
            }
            if constexpr (SPLIT) *(float4*)((float*)p.scratch + 2 * rows * p.nsplit + prow * D + col) = acc;
            else T::store(orow + col, r[0], r[1], r[2], r[3]);
        }
        if (!SPLIT && tid_m % TPR == 0) p.lse[(int64_t)bh * N + io] = exact_lse(Mu, denom, big, e);
        bad |= !(Ls <= MOST);
    }

    // ---- what the planes do not cover: the block again, by rows (see split_fwd_kernel) ----
    if (!__syncthreads_or(bad || tiny)) return;
    const bool any_bad = __syncthreads_or(bad), any_usual = __syncthreads_or(usual);
    if (!any_bad && any_usual) return;
    {
        // (a row whose q holds a NaN is NaN as it stands: a block of such rows is done)
        bool q_nan = false;
        for (int col = 4 * (tid_m % TPR); io < N && col < p.D; col += 4 * TPR) {
            const float4 x = cols4<T, PAD>((const EL*)p.q.p + p.q.off(b, io, h), col, p.D);
            q_nan |= x.x != x.x || x.y != x.y || x.z != x.z || x.w != x.w;
        }
        const uint64_t row_lanes = (((uint64_t)1 << TPR) - 1) << ((tid_m & 63) / TPR * TPR);
        const bool row_nan = (__builtin_amdgcn_ballot_w64(q_nan) & row_lanes) != 0;
        if (!__syncthreads_or(io < N && !row_nan)) return;
    }
    const int d_lo = round0 * UPR, d_hi = round1 * UPR - 1 < w2 ? round1 * UPR - 1 : w2;
    for (int x = 0; x < BQ && i0 + x < N; x += KW)
        fma_fwd_rows<typename T::Fma>(p, bh, i0 + x, d_lo, d_hi, (float*)smem_raw, [&](int ir, int ln_r, float m, float l_r, const float (&acc)[MAXC]) {
            if constexpr (SPLIT) {
                const int64_t rows = (int64_t)p.B * p.H * N, prow = share * rows + (int64_t)bh * N + ir;
                if (ln_r == 0) ((float2*)p.scratch)[prow] = make_float2(m * LOG2E, l_r);
#pragma unroll
                for (int c = 0; c < MAXC; ++c)
                    if (ln_r + 64 * c < p.D) ((float*)p.scratch)[2 * rows * p.nsplit + prow * D + ln_r + 64 * c] = acc[c];
            } else {
                fma_store_row<typename T::Fma>(p, bh, ir, ln_r, m, l_r, acc);
            }
        });
}

template <class T, int D, int NQ, int MODE>
int launch_split_fwd_lone(const Problem& p, hipStream_t st) {
    using C = SplitFwdLoneCfg<T, D, NQ>;
    const int nqb = (p.N + BQ - 1) / BQ;
    const int64_t total = (int64_t)nqb * p.B * p.H * (p.nsplit > 1 ? p.nsplit : 1);
    if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return SA2_ERR_LAUNCH_FAILED;
        hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(C::THREADS), C::LDS_BYTES, st, p, nqb, (int)total);
        return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
    };
    return p.nsplit > 1 ? go(split_fwd_lone_kernel<T, D, NQ, MODE, true>) : go(split_fwd_lone_kernel<T, D, NQ, MODE, false>);
}

}  // namespace
}  // namespace sa2
