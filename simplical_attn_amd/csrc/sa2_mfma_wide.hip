// MFMA kernels for 16-bit tensors whose head_dim the tuned kernels do not take: head_dim 256
// (bf16 or fp16), forward and backward, on v_mfma_f32_32x32x16_bf16 / _f16.
//
// Same expanded-row view as the tuned kernels (rows r = (i, delta), Q~[r] = q[i] * k2~[i-delta] *
// scale*log2(e), dO~[r] = dO[i] * v2~[i-delta], both rounded to the element type).  Four wavefronts per
// workgroup, one per SIMD with all 512 registers: that is room for a row operand of 256 columns and for
// the accumulators of all 256 output columns of two contractions, so that nothing is computed twice.
// (The arrangement before took the output columns in two passes of 128, each with the logits over the
// whole head_dim: 1.5x the forward's and 1.33x the backward's MFMA work, and left the matrix pipe idle
// under every wait and every piece of vector arithmetic.)  A lone wavefront hides its latencies itself:
// operand reads are opaque instructions issued one or two blocks of MFMAs ahead of their use, waits count
// outstanding LDS operations, vector arithmetic stands between the MFMAs, and accumulators that live
// through a sweep are pinned to accumulation registers.
//
//   wide_fwd_kernel   32 queries per workgroup; wavefront w takes delta = w, w+4, ... with one online
//                     softmax and one output accumulator across its units, merged once at the end.
//   wide_kp_kernel    32 K' rows per workgroup and a run of deltas, two pairs of wavefronts.
//   wide_kv_kernel    128 K/V rows per workgroup (32 per wavefront, resident in registers as B
//                     operands), streaming every unit (query block, delta) that can see them.
// Measured at B1 H8 N4096 w 512/32, bf16 (us, two column passes -> now): 2215 -> 890, 3860 -> 2170, 4900 -> 1530; the MFMAs'
// rate inside the sweeps is 0.9 to 1.0 PFLOP/s, where a large matrix product reaches 1.2 on this card.
// Every output element has one writer and a fixed summation order: no atomics, bitwise reproducible.
#include "sa2_mfma_common.h"

namespace sa2 {
namespace {

constexpr int WW = 4;                  // wavefronts per workgroup
constexpr int WT = WW * 64;            // threads per workgroup
constexpr int WJ = WW * 32;            // K rows per workgroup of the K-side kernel
constexpr int WKV_SIDE = 40;           // K' and V' rows the K-side kernel keeps in LDS: the 32 of a unit, and eight to come or past
constexpr int WKP_DQ = 34;             // dQ rows the K'-side kernel keeps in LDS: the 33 of a round, and one to make pairs
constexpr int WSIDE = 36;              // K' and V' rows the forward keeps in LDS: the 35 of a round, and one to make pairs

typedef float fx4 __attribute__((ext_vector_type(4)));
typedef unsigned ux4 __attribute__((ext_vector_type(4)));     // 16 bytes in flight (a plain vector: stays in registers)

__device__ __forceinline__ floatx16 zeros16() {
    floatx16 z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.f;
    return z;
}
template <class E>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    union { typename E::x2 h; uint32_t u; } v;
    v.h = __builtin_convertvector((f2){a, b}, typename E::x2);
    return v.u;
}
// a[r] * mul * (b[r] + bias) of two 16-byte chunks (8 elements), rounded to the element type
template <class E, bool BIASED = true>
__device__ __forceinline__ typename E::x8 product8(const ux4& a, const ux4& b, float bias, float mul) {
    union { uint32_t w[4]; typename E::x8 v; } r;
#pragma unroll
    for (int t = 0; t < 4; ++t)
        r.w[t] = BIASED ? pack2<E>(E::lo(a[t]) * mul * (E::lo(b[t]) + bias), E::hi(a[t]) * mul * (E::hi(b[t]) + bias))
                        : pack2<E>(E::lo(a[t]) * mul * E::lo(b[t]), E::hi(a[t]) * mul * E::hi(b[t]));
    return r.v;
}

// ---- tiles -----------------------------------------------------------------------
// A 32-row tile of a 256-column tensor in LDS: sixteen groups of two rows, each written by one direct
// global->LDS load of a wavefront (1 KB; lane L puts the 16-byte chunk L / 2 of row L % 2 at byte 16 * L)
// and GROUP bytes apart.  Row operand reads are free of bank conflicts, transposed ones take two passes.  (A swizzle of the
// chunks that frees both measured the same or slower, forward 889 -> 915 us and K-side 1526 -> 1537 us at B1 H8 N4096
// w 512/32: LDS is not what the kernels wait for, and its addresses cost vector instructions.)
struct WT256 {
    static constexpr int RPW = 2, GROUP = 1024 + 32, NGROUP = 16;
    static constexpr int BYTES = NGROUP * GROUP;
    static constexpr int row_off(int r) { return (r / RPW) * GROUP + (r % RPW) * 16; }
};
constexpr size_t WIDE_KP_LDS = (size_t)4 * WT256::BYTES + 2 * 6144 + 2 * (WSIDE / 2) * WT256::GROUP + (size_t)WKP_DQ * 260 * 4;
static_assert(WIDE_KP_LDS >= (size_t)WW * 32 * 260 * 4 && WIDE_KP_LDS <= 160 * 1024, "the last sums lie over everything");
constexpr size_t WIDE_KV_LDS = (size_t)6 * WT256::BYTES + 2 * (WKV_SIDE / 2) * WT256::GROUP + 2 * 2 * 32 * 4;
constexpr size_t WIDE_FWD_LDS = (size_t)7 * WT256::BYTES + 2 * (WSIDE / 2) * WT256::GROUP;
static_assert(WIDE_FWD_LDS >= (size_t)WW * 32 * 260 * 4 + 2 * WW * 32 * 4 && WIDE_FWD_LDS <= 160 * 1024, "the merge lies over the tiles");
typedef __attribute__((address_space(3))) void* wide_lds_ptr;
typedef const __attribute__((address_space(1))) void* wide_glb_ptr;

// The four groups of wavefront `wave` of the tile of rows j0 .. j0+31 (rows past the end of the sequence read the
// last one): `lane_off` is the byte offset of the lane's chunk in the wavefront's first group.
__device__ __forceinline__ void wide_request(const uint16_t* base, int64_t sn, int j0, int N, int wave, int lane, uint32_t lane_off,
                                             unsigned char* dst) {
    const char* g = (const char*)(base + (int64_t)j0 * sn);
    if (__builtin_expect(j0 + 32 <= N, 1)) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
            __builtin_amdgcn_global_load_lds((wide_glb_ptr)(g + (lane_off + (uint32_t)x * ((uint32_t)sn * 4u))), (wide_lds_ptr)(dst + (4 * wave + x) * WT256::GROUP), 16, 0, 0);
    } else {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int row = 8 * wave + 2 * x + (lane & 1), r = row < N - 1 - j0 ? row : N - 1 - j0;
            __builtin_amdgcn_global_load_lds((wide_glb_ptr)(g + ((uint32_t)r * (uint32_t)sn + (uint32_t)(lane >> 1) * 8) * 2u),
                                             (wide_lds_ptr)(dst + (4 * wave + x) * WT256::GROUP), 16, 0, 0);
        }
    }
}
// Transposed operands of k-step KS (rows 16*KS .. +15) of the column blocks DT0 .. DT0+N-1, as opaque reads
template <int KS, int DT0, int N, int I = 0, int M>
__device__ __forceinline__ void wide_tr_issue(uint32_t addr, lds_half_operand (&h)[M]) {
    if constexpr (I < N) {
        constexpr int o = (DT0 + I) * 64 * WT256::RPW + WT256::row_off(16 * KS);
        lds_tr_issue<o, o + WT256::row_off(8)>(addr, h[2 * I], h[2 * I + 1]);
        wide_tr_issue<KS, DT0, N, I + 1>(addr, h);
    }
}
// acc += a * b with the accumulator in accumulation registers.  Opaque: beside 256 registers of accumulators that live
// through a whole sweep the compiler's own placement moves some of them to scratch memory in every step.  Operands that
// the vector ALU writes pass through settle_operand first; results are read behind settle_acc.
template <class X8>
__device__ __forceinline__ void mfma_acc(floatx16& acc, const X8& a, const X8& b) {
    if constexpr (std::is_same<X8, bf16x8>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// The same into vector registers, for results that the vector ALU reads: at least four more MFMAs are issued before it
// does (see wait_acc), which outlasts the matrix pipe's latency.
template <class X8>
__device__ __forceinline__ void mfma_vec(floatx16& acc, const X8& a, const X8& b) {
    if constexpr (std::is_same<X8, bf16x8>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
template <class X8>
__device__ __forceinline__ void mfma_vec_zero(floatx16& acc, const X8& a, const X8& b) {          // acc = a * b
    if constexpr (std::is_same<X8, bf16x8>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
}
// Accumulators start from here rather than from a constant, and every loop over MFMAs keeps them out of its branches:
// a value that meets another one of vector registers is copied between the two files in every step.
template <int N>
__device__ __forceinline__ void zero_acc(floatx16 (&acc)[N]) {
    bf16x8 z;
#pragma unroll
    for (int t = 0; t < 8; ++t) z[t] = (__bf16)0.f;
    asm volatile("s_nop 3" : "+v"(z));
#pragma unroll
    for (int x = 0; x < N; ++x) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %1, 0" : "=a"(acc[x]) : "v"(z));
}
__device__ __forceinline__ void settle_c(floatx16& acc) { asm volatile("s_nop 3" : "+v"(acc)); }
__device__ __forceinline__ void wait_acc(floatx16& acc) { asm volatile("s_nop 7" : "+v"(acc)); }
template <class X8>
__device__ __forceinline__ void settle_operand(X8 (&x)[2]) { asm volatile("s_nop 3" : "+v"(x[0]), "+v"(x[1])); }
__device__ __forceinline__ void settle_halves(lds_half_operand (&x)[8]) {
    asm volatile("s_nop 3" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]));
}
template <int N>
__device__ __forceinline__ void settle_acc(floatx16 (&acc)[N]) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int x = 0; x < N; ++x) asm volatile("" : "+a"(acc[x]));
}
// 16 bytes from / to LDS as opaque operations, in the order of the program
template <int OFF, class V>
__device__ __forceinline__ void lds_read16(uint32_t addr, V& v) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF)); }
template <int OFF, class V>
__device__ __forceinline__ void lds_write16(uint32_t addr, const V& v) { asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory"); }
__device__ __forceinline__ void opaque(int& x) { asm volatile("" : "+v"(x)); }
template <class V>
__device__ __forceinline__ void arrived(V& a, V& b) { asm volatile("" : "+v"(a), "+v"(b)); }          // (behind the wait for them)
// keeps values that the vector ALU updates between two sweeps in accumulation registers during them
template <int N>
__device__ __forceinline__ void stay_acc(floatx16 (&acc)[N]) {
#pragma unroll
    for (int x = 0; x < N; ++x) asm volatile("" : "+a"(acc[x]));
}
// Row operands of the k-steps K0 .. K0+3
template <int K0, int I = 0, class X8>
__device__ __forceinline__ void wide_rows4(uint32_t addr, X8 (&r)[4]) {
    if constexpr (I < 4) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(r[I]) : "v"(addr), "n"((K0 + I) * 32 * WT256::RPW));
        wide_rows4<K0, I + 1>(addr, r);
    }
}
// at most PENDING LDS operations issued so far are outstanding; the halves named here may be used from here on
template <int PENDING>
__device__ __forceinline__ void lds_wait_halves(lds_half_operand (&x)[8]) {
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7])
                 : "n"(PENDING));
}
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}
// Row operands of the k-steps K0 .. K0+7
template <int K0, int I = 0, class X8>
__device__ __forceinline__ void wide_row_issue(uint32_t addr, X8 (&r)[8]) {
    if constexpr (I < 8) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(r[I]) : "v"(addr), "n"((K0 + I) * 32 * WT256::RPW));
        wide_row_issue<K0, I + 1>(addr, r);
    }
}

// ================================================================== forward =====
// What bounds it: in the sweep the matrix pipe at the rate that power allows (1.09 us per step of 32 MFMAs per wavefront,
// 1.0 PFLOP/s), and between two sweeps the forming of Q~ and the sum over the unit, 6 us per round.  The logits of tile t
// run under the softmax arithmetic of tile t-1, operand reads are one block of eight MFMAs ahead of their use, and the
// last eight value MFMAs of a tile run behind the step's barrier, under the next tile's operand reads.
// B1 H8 N4096 w 512/32 bf16: 2215 us in two column passes, 890 now; B1 H3 N700 w 500/100 949 -> 233 (shares of the rounds).
// SAFE: the second pass of a block in which a weight overflowed (logits growing by tens of octaves along the window after
// the reference point was fixed): the reference point follows the maxima on every tile, nothing is pipelined.
// Returns whether that pass is needed.
template <class E, bool SPLIT, bool SAFE>
__device__ __forceinline__ bool wide_fwd_block(const Problem& p, int nqb, int total, unsigned char* smem_w) {
    typedef typename E::scalar EL;
    typedef typename E::x8 X8;
    typedef typename E::x2 X2;
    constexpr int D = 256, DK = 16, DT = 8, TB = WT256::BYTES;
    const int tid = threadIdx.x;
    unsigned char* q_s = smem_w + 6 * TB;                    // q rows of the block
    unsigned char* k2_s = q_s + TB;                          // ring of WSIDE K' rows
    unsigned char* v2_s = k2_s + WSIDE / 2 * WT256::GROUP;   // ... and V' rows

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
    const int i0 = qb * BQ, i = i0 + ln;
    const int i_last = i0 + BQ - 1 < N ? i0 + BQ - 1 : N - 1;

    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* k1p = (const uint16_t*)p.k1.p + p.k1.off(b, 0, h);
    const uint16_t* k2p = (const uint16_t*)p.k2.p + p.k2.off(b, 0, h);
    const uint16_t* v1p = (const uint16_t*)p.v1.p + p.v1.off(b, 0, h);
    const uint16_t* v2p = (const uint16_t*)p.v2.p + p.v2.off(b, 0, h);

    // The sweep goes from the diagonal tile down: every row has a key in its first tile, which fixes its reference point.
    const int jt_lo = (i0 - w1 > 0 ? i0 - w1 : 0) / TJ, jt_hi = i0 / TJ;
    const int nt = jt_hi - jt_lo + 1;
    const int n_units = (w2 < i_last ? w2 : i_last) + 1;
    const int all_rounds = (n_units + WW - 1) / WW;
    const int per_share = SPLIT ? ((w2 + WW) / WW + p.nsplit - 1) / p.nsplit : all_rounds;
    const int round0 = SPLIT ? share * per_share : 0;
    const int round1 = round0 + per_share < all_rounds ? round0 + per_share : all_rounds;
    if constexpr (SPLIT) {
        if (round0 >= round1) {                  // a block near the start of the sequence has fewer rounds
            if (tid < BQ && i0 + tid < N)
                ((float2*)p.scratch)[share * (int64_t)p.B * p.H * N + (int64_t)bh * N + i0 + tid] = make_float2(-INFINITY, 0.f);
            return false;
        }
    }
    const int total_steps = (round1 - round0) * nt;
    const float qscale = p.scale * LOG2E;

    // ---- requests: step g asks for the K tile of step g+2 and the V tile of step g+1, in rings of three ----
    const uint32_t k_off = ((uint32_t)(8 * wave + (lane & 1)) * (uint32_t)p.k1.sn + (uint32_t)(lane >> 1) * 8) * 2u;
    const uint32_t v_off = ((uint32_t)(8 * wave + (lane & 1)) * (uint32_t)p.v1.sn + (uint32_t)(lane >> 1) * 8) * 2u;
    int kt = 0, kstage = 0, kleft = total_steps, vt = 0, vstage = 0, vleft = total_steps;
    auto request_k = [&]() {
        wide_request(k1p, p.k1.sn, (jt_hi - kt) * TJ, N, wave, lane, k_off, smem_w + kstage * TB);
        kt = kt + 1 == nt ? 0 : kt + 1;
        kstage = kstage == 2 ? 0 : kstage + 1;
        --kleft;
    };
    auto request_v = [&]() {
        wide_request(v1p, p.v1.sn, (jt_hi - vt) * TJ, N, wave, lane, v_off, smem_w + (3 + vstage) * TB);
        vt = vt + 1 == nt ? 0 : vt + 1;
        vstage = vstage == 2 ? 0 : vstage + 1;
        --vleft;
    };
    // K'/V' row u counts back from row i0 + 31 of share's first round; it sits at place u % WSIDE of its ring.  A round
    // needs rows 4r .. 4r+34; `pair` is a pair of rows (u = 2 * pair, 2 * pair + 1).
    auto request_side = [&](const uint16_t* base, int64_t sn, int pair, unsigned char* ring) {
        int k = i0 + BQ - 1 - round0 * WW - 2 * pair - (lane & 1);
        k = k < 0 ? 0 : (k < N ? k : N - 1);
        __builtin_amdgcn_global_load_lds((wide_glb_ptr)(base + (int64_t)k * sn + (lane >> 1) * 8),
                                         (wide_lds_ptr)(ring + (pair % (WSIDE / 2)) * WT256::GROUP), 16, 0, 0);
    };
    request_k();
    request_v();
    wide_request(qp, p.q.sn, i0, N, wave, lane, ((uint32_t)(8 * wave + (lane & 1)) * (uint32_t)p.q.sn + (uint32_t)(lane >> 1) * 8) * 2u, q_s);
    for (int x = wave; x < WSIDE / 2; x += WW) {
        request_side(k2p, p.k2.sn, x, k2_s);
        request_side(v2p, p.v2.sn, x, v2_s);
    }
    if (kleft > 0) request_k();
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    const uint32_t smem_addr = lds_address(smem_w);
    const uint32_t row_lane = (uint32_t)((ln / 2) * WT256::GROUP + (hf * 2 + (ln & 1)) * 16);
    const uint32_t col_lane = lds_group_column_lane_offset<WT256::RPW, WT256::GROUP>(lane);

    // the wavefront's running softmax over its units: reference exponent (one per row for all units), sum, weighted output
    float m = -INFINITY, L = 0.f;
    floatx16 wacc[DT], racc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) wacc[dt][v] = 0.f;

    bool bad = false;
    int buf = 0;                                             // ring stage of the current step's K tile
    for (int round = round0; round < round1; ++round) {
        const int rr = round - round0;
        const int delta = round * WW + wave;
        const bool ok = delta < n_units;
        const bool row_ok = i < N && i >= delta;
        const bool rows_full = ok && i0 >= delta && i0 + BQ - 1 < N;
        const int place = (BQ - 1 - ln + rr * WW + wave) % WSIDE;
        const uint32_t side = (uint32_t)((place / 2) * WT256::GROUP + (place & 1) * 16);
        X8 qf[DK];
#pragma unroll
        for (int kk = 0; kk < DK; ++kk) {
            const ux4 qa = *(const ux4*)(q_s + row_lane + kk * 64);
            const ux4 kb = *(const ux4*)(k2_s + side + hf * 32 + kk * 64);
            qf[kk] = product8<E>(qa, kb, p.k2_bias, qscale);
        }
        float l = 0.f, mu = -INFINITY;            // (mu: the unit's own reference point in the second pass)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) racc[dt] = zeros16();
        // -inf where the key lies outside the window of the row.  Element v of this lane is key j0 + 8*(v/4) + 4*hf + v%4.
        auto mask = [&](floatx16& s, int j0) {
            int hi = i - j0 - 4 * hf;
            asm volatile("" : "+v"(hi));          // (compared here, not kept from one round to the next)
            const int lo = hi - w1;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int c = 8 * (v >> 2) + (v & 3);
                s[v] = (row_ok && c <= hi && c >= lo) ? s[v] : -INFINITY;
            }
        };
        auto tile_plain = [&](int j0) { return rows_full && j0 + TJ - 1 <= i0 && j0 >= i0 + BQ - 1 - w1; };
        if (!SAFE && ok && __builtin_amdgcn_ballot_w64(m == -INFINITY) != 0) {
            // the reference point of the wavefront's rows: the maximum of the first tile (0 for a row that has no key at all)
            floatx16 t = zeros16();
#pragma unroll
            for (int kk = 0; kk < DK; ++kk) t = E::mfma(lds_read_x8<X8>(smem_addr + buf * TB + row_lane + kk * 64), qf[kk], t, 0, 0, 0);
            mask(t, jt_hi * TJ);
            float mx = t[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) mx = fmaxf(mx, t[v]);
            mx = fmaxf(mx, other_half(mx));
            if (m == -INFINITY) m = mx == -INFINITY ? 0.f : mx;
        }

        floatx16 cur, prev;
        X8 pb[2], pb1;                            // weights of the tile before; of the one before that, second k-step
        lds_half_operand va[16], vb[16];
        // weights of the logits `s` and their row sum (this lane's half of the keys)
        auto weights = [&](const floatx16& s, float ref) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int t = 0; t < 8; ++t) pb[ks][t] = (EL)fast_exp2(s[ks * 8 + t] - ref);
            const X2 ones = {(EL)1.f, (EL)1.f};
            float r = 0.f;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                r = E::dot2(__builtin_shufflevector(pb[ks], pb[ks], 0, 1), ones, r, false);
                r = E::dot2(__builtin_shufflevector(pb[ks], pb[ks], 2, 3), ones, r, false);
                r = E::dot2(__builtin_shufflevector(pb[ks], pb[ks], 4, 5), ones, r, false);
                r = E::dot2(__builtin_shufflevector(pb[ks], pb[ks], 6, 7), ones, r, false);
            }
            return r;
        };
        auto value_mfmas = [&](const lds_half_operand (&x)[16], const X8& w) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) racc[dt] = E::mfma(lds_join<X8>(x[2 * dt], x[2 * dt + 1]), w, racc[dt], 0, 0, 0);
        };
        auto logit_mfmas = [&](const X8 (&k)[8], int k0, floatx16 c) {
#pragma unroll
            for (int x = 0; x < 8; ++x) c = E::mfma(k[x], qf[k0 + x], c, 0, 0, 0);
            return c;
        };
        auto end_step = [&](bool both) {
            if (both) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            buf = buf == 2 ? 0 : buf + 1;
        };
        auto begin_step = [&]() {
            const bool both = kleft > 0;
            if (vleft > 0) request_v();
            if (both) request_k();
            return both;
        };

        auto side_rows = [&]() {
            // (every wavefront has formed its Q~ and is done with the round before)
            if (wave < 2) request_side(k2p, p.k2.sn, 2 * rr + WSIDE / 2 + wave, k2_s);
            else if (rr > 0) request_side(v2p, p.v2.sn, 2 * rr + WSIDE / 2 - 4 + wave, v2_s);
            if (nt == 1) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        };
        if constexpr (SAFE) {
            for (int s = 0; s < nt; ++s) {
                const bool both = begin_step();
                if (ok) {
                    const int j0 = (jt_hi - s) * TJ;
                    cur = zeros16();
#pragma unroll
                    for (int kk = 0; kk < DK; ++kk) cur = E::mfma(lds_read_x8<X8>(smem_addr + buf * TB + row_lane + kk * 64), qf[kk], cur, 0, 0, 0);
                    if (!tile_plain(j0)) mask(cur, j0);
                    float mx = cur[0];
#pragma unroll
                    for (int v = 1; v < 16; ++v) mx = fmaxf(mx, cur[v]);
                    const float m_new = fmaxf(mu, fmaxf(mx, other_half(mx))), m_use = m_new == -INFINITY ? 0.f : m_new;
                    const float alpha = fast_exp2(mu - m_use);
                    mu = m_new;
                    l *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int v = 0; v < 16; ++v) racc[dt][v] *= alpha;
                    l += weights(cur, m_use);
                }
                end_step(both);                  // (the V tile of a step is complete behind its barrier)
                if (s == 0) side_rows();
                if (ok) {
                    const uint32_t vt_addr = smem_addr + (3 + (buf == 0 ? 2 : buf - 1)) * TB + col_lane;
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt)
                            racc[dt] = E::mfma(lds_group_column_operand_at<WT256, X8>(vt_addr + dt * 64 * WT256::RPW, ks), pb[ks], racc[dt], 0, 0, 0);
                }
            }
        } else {
        // ---- first step: logits only ----
        {
            const bool both = begin_step();
            if (ok) {
                X8 k0[8], k1[8];
                const uint32_t a = smem_addr + buf * TB + row_lane;
                wide_row_issue<0>(a, k0);
                wide_row_issue<8>(a, k1);
                lds_wait<8>(k0);
                prev = logit_mfmas(k0, 0, zeros16());
                lds_wait<0>(k1);
                prev = logit_mfmas(k1, 8, prev);
                mask(prev, jt_hi * TJ);          // (the diagonal tile)
            }
            end_step(both);
        }
        side_rows();
        for (int s = 1; s < nt; ++s) {
            const bool both = begin_step();
            if (ok) {
                const int j0 = (jt_hi - s) * TJ;
                X8 k0[8], k1[8];
                const uint32_t a = smem_addr + buf * TB + row_lane;
                const uint32_t vt_addr = smem_addr + (3 + (buf == 0 ? 2 : buf - 1)) * TB + col_lane;
                wide_row_issue<0>(a, k0);
                wide_row_issue<8>(a, k1);
                __builtin_amdgcn_sched_barrier(0);
                if (s > 1) value_mfmas(vb, pb1);
                lds_wait<8>(k0);
                cur = logit_mfmas(k0, 0, zeros16());
                lds_wait<0>(k1);
                wide_tr_issue<0, 0, 8>(vt_addr, va);
                cur = logit_mfmas(k1, 8, cur);
                const float rs = weights(prev, m);
                l += rs;
                bad |= !(rs < E::WEIGHT_LIMIT);
                pb1 = pb[1];
                lds_settle(va);
                wide_tr_issue<1, 0, 8>(vt_addr, vb);
                value_mfmas(va, pb[0]);
                lds_settle(vb);
                prev = cur;
                if (!tile_plain(j0)) mask(prev, j0);
            }
            end_step(both);
        }
        // ---- last tile's values ----
        if (ok) {
            const uint32_t vt_addr = smem_addr + (3 + (buf == 0 ? 2 : buf - 1)) * TB + col_lane;
            wide_tr_issue<0, 0, 8>(vt_addr, va);
            if (nt > 1) value_mfmas(vb, pb1);
            const float rs = weights(prev, m);
            l += rs;
            bad |= !(rs < E::WEIGHT_LIMIT);
            lds_settle(va);
            wide_tr_issue<1, 0, 8>(vt_addr, vb);
            value_mfmas(va, pb[0]);
            lds_settle(vb);
            value_mfmas(vb, pb[1]);
        }
        }
        // ---- the unit joins the running result: O += (v2 + bias) * R ----
        if (ok) {
            const float lt = l + other_half(l);
            float a = 1.f, c = 1.f;
            if constexpr (SAFE) {
                const float M_new = fmaxf(m, mu), Mu = M_new == -INFINITY ? 0.f : M_new;
                a = fast_exp2(m - Mu);
                c = fast_exp2(mu - Mu);
                m = M_new;
                L *= a;
            }
            L += c * lt;
            const unsigned char* vrow = v2_s + side + hf * 8;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const uint2 x = *(const uint2*)(vrow + (4 * dt + g4) * 32);
                    const float y[4] = {E::lo(x.x), E::hi(x.x), E::lo(x.y), E::hi(x.y)};
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int v = 4 * g4 + t;
                        if constexpr (SAFE) wacc[dt][v] = wacc[dt][v] * a + c * racc[dt][v] * (y[t] + p.v2_bias);
                        else wacc[dt][v] += racc[dt][v] * (y[t] + p.v2_bias);
                    }
                }
        }
    }

    // ---- merge the four wavefronts ----
    if constexpr (!SAFE) {
        if (__syncthreads_or(bad ? 1 : 0)) return true;
    }
    else __syncthreads();
    constexpr int AS = D + 4;
    float* mrg = (float*)smem_w;                           // [WW][32][AS]
    float* mrg_m = mrg + WW * 32 * AS;                     // [WW][32]
    float* mrg_l = mrg_m + WW * 32;
    {
        float* row = mrg + (wave * 32 + ln) * AS + 4 * hf;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
                *(float4*)(row + dt * 32 + 8 * g4) = make_float4(wacc[dt][4 * g4], wacc[dt][4 * g4 + 1], wacc[dt][4 * g4 + 2],
                                                                 wacc[dt][4 * g4 + 3]);
        if (hf == 0) {
            mrg_m[wave * 32 + ln] = L > 0.f || L != L ? m : -INFINITY;         // (a row without a key has no say in the reference)
            mrg_l[wave * 32 + ln] = L;
        }
    }
    __syncthreads();
    const int row = tid >> 3, io = i0 + row;
    if (io < N) {
        float Mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < WW; ++w) Mx = fmaxf(Mx, mrg_m[w * 32 + row]);
        const float Mu = Mx == -INFINITY ? 0.f : Mx;
        float wgt[WW], Ls = 0.f;
#pragma unroll
        for (int w = 0; w < WW; ++w) {
            wgt[w] = fast_exp2(mrg_m[w * 32 + row] - Mu);
            Ls += mrg_l[w * 32 + row] * wgt[w];
        }
        const int64_t rows = (int64_t)p.B * p.H * N, prow = share * rows + (int64_t)bh * N + io;
        float* part = (float*)p.scratch + 2 * rows * p.nsplit + prow * D;      // (SPLIT)
        // sum_w + 1e-8 in units of 2^Mu; for a tiny Mu the epsilon dominates
        const bool big = Mu > LOG2_EPS;
        const float denom = big ? Ls + 1e-8f * fast_exp2(-Mu) : Ls * fast_exp2(Mu - LOG2_EPS) + 1.f;
        const float inv = big ? 1.f / denom : fast_exp2(Mu - LOG2_EPS) / denom;
        uint16_t* orow = (uint16_t*)p.out.p + p.out.off(b, io, h);
#pragma unroll
        for (int x = 0; x < DT; ++x) {
            const int col = 32 * x + 4 * (tid & 7);
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < WW; ++w) {
                const float4 y = *(const float4*)(mrg + (w * 32 + row) * AS + col);
                acc.x += wgt[w] * y.x; acc.y += wgt[w] * y.y; acc.z += wgt[w] * y.z; acc.w += wgt[w] * y.w;
            }
            if constexpr (SPLIT) *(float4*)(part + col) = acc;
            else *(uint2*)(orow + col) = make_uint2(E::pack(acc.x * inv, acc.y * inv), E::pack(acc.z * inv, acc.w * inv));
        }
        if ((tid & 7) == 0) {
            if constexpr (SPLIT) ((float2*)p.scratch)[prow] = make_float2(Mx, Ls);
            else p.lse[(int64_t)bh * N + io] = big ? LN2 * Mu + logf(denom) : LN_EPS + logf(denom);
        }
    }
    return false;
}

// (A function of its own, so that its registers do not count where the first pass allocates its: inlined, it pushed the
// output accumulator of the first pass to scratch memory.)
template <class E, bool SPLIT>
__device__ __attribute__((noinline))
void wide_fwd_again(const Problem __attribute__((address_space(4))) * p, int nqb, int total, uint32_t lds) {
    wide_fwd_block<E, SPLIT, true>(*(const Problem*)p, nqb, total, (unsigned char*)(__attribute__((address_space(3))) unsigned char*)(uintptr_t)lds);
}
template <class E, bool SPLIT>
__global__ __launch_bounds__(WT) __attribute__((amdgpu_waves_per_eu(1, 1)))
void wide_fwd_kernel(Problem p, int nqb, int total) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_w[];
    if (wide_fwd_block<E, SPLIT, false>(p, nqb, total, smem_w))              // (uniform over the workgroup)
        wide_fwd_again<E, SPLIT>((const Problem __attribute__((address_space(4)))*)__builtin_amdgcn_kernarg_segment_ptr(), nqb, total, lds_address(smem_w));
}

// ============================================== backward, K' side: dQ, dK', dV' =====
// A workgroup owns 32 consecutive K' rows k0 .. k0+31 and a run of deltas (all of them, or a segment where the K' blocks
// alone leave the chip idle); unit delta is the 32 expanded rows (i = k + delta, k).  Two pairs of wavefronts hold one
// unit each per round and sweep the K/V window in 32-key tiles, two tiles of each in LDS.  In a pair one wavefront works
// on the K tile only, S^T = K1.Q~^T and G^T += K1^T.dS^T, the other on the V tile only, dP^T = V1.dO~^T and
// R^T += V1^T.P^T; half way through a step they exchange P (16 bit, as the MFMA takes it) and dP - D (fp32).  So each holds
// one row operand and one output of all 256 columns, and beside them the sum over its deltas of G*q (dK') or R*dO (dV'),
// which are aligned with the K' rows.  dQ rows are shifted by delta: a ring of fp32 rows in LDS, whose two oldest rows
// leave for the workgroup's partial after every round.
// What bounds it: in the sweep the matrix pipe (1.25 us per step of 32 MFMAs per wavefront), and between two sweeps the sums
// over the unit (9 us per round, 30 % of the time at a K window of 512).  The second half of a step's last contraction runs
// in the next step, from registers: it covers that step's first LDS reads and the exponentials.  The K' row stays in
// registers although some of it is pushed to scratch memory in the sweep: reading it from the tensor again in every round
// measured 2340 against 2200 us.  B1 H8 N4096 w 512/32 bf16: 3860 us in two column passes, 2170 now.
template <class E, bool BIASED>
__global__ __launch_bounds__(WT) __attribute__((amdgpu_waves_per_eu(1, 1)))
void wide_kp_kernel(Problem p, int nkb, int total, float* __restrict__ dq_part, int nseg, int segw, float* __restrict__ kpart) {
    typedef typename E::scalar EL;
    typedef typename E::x8 X8;
    constexpr int D = 256, DK = 16, DT = 8, TB = WT256::BYTES, AS = D + 4;
    constexpr int RING = WSIDE / 2;                          // pairs of rows in the rings of q and dO rows
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_w[];
    unsigned char* px = smem_w + 4 * TB;                     // (K tiles, then V tiles)  [pair][P: 2 KB, dP: 4 KB]
    unsigned char* q_s = px + 2 * 6144;
    unsigned char* do_s = q_s + RING * WT256::GROUP;
    float* dq_s = (float*)(do_s + RING * WT256::GROUP);      // [WKP_DQ][AS]

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = wave >> 1, pair = wave & 1;             // role 0: K tile, 1: V tile
    // (segments one after the other in launch order: the last one is the short one)
    const int per_seg = total / nseg, seg = (int)blockIdx.x / per_seg;
    const int pid = xcd_order((int)blockIdx.x - seg * per_seg, per_seg);
    const int bh = pid / nkb, kb = pid - bh * nkb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int k0 = kb * BQ, kq = k0 + seg * segw;            // query of K' row k0 at the first delta
    const int nu_all = (w2 < N - 1 - k0 ? w2 : N - 1 - k0) + 1 - seg * segw;
    const int n_units = nu_all < segw ? nu_all : segw;       // (may be <= 0)
    const int nrounds = n_units > 0 ? (n_units + 1) / 2 : 0;
    const int RQ = BQ + segw - 1;                            // rows of the dQ partial
    const bool want_dq = p.dq.p != nullptr;

    const uint16_t* k1p = (const uint16_t*)p.k1.p + p.k1.off(b, 0, h);
    const uint16_t* v1p = (const uint16_t*)p.v1.p + p.v1.off(b, 0, h);
    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* dop = (const uint16_t*)p.dout.p + p.dout.off(b, 0, h);

    auto here = [&]() {                                      // (lane parts are computed where they are used)
        int t = threadIdx.x;
        opaque(t);
        return t & 63;
    };
    // ---- tiles: step g works on slot g & 1 and asks for the tile of step g + 1 (of this round or the next) ----
    auto round_first = [&](int r) {
        const int i_min = kq + 2 * r;
        return (i_min - w1 > 0 ? i_min - w1 : 0) / TJ;
    };
    auto round_last = [&](int r) {
        const int d = 2 * r + 1 < n_units - 1 ? 2 * r + 1 : n_units - 1;
        const int i_max = kq + d + BQ - 1 < N - 1 ? kq + d + BQ - 1 : N - 1;
        return i_max / TJ;
    };
    int slot = 0, next_round = 0, next_tile = round_first(0), next_last = round_last(0);
    auto request_tile = [&](int to) {
        if (next_round < nrounds) {
            const int lane = here();
            const uint32_t r2 = 8 * wave + (lane & 1), c2 = (lane >> 1) * 8;
            wide_request(k1p, p.k1.sn, next_tile * TJ, N, wave, lane, (r2 * (uint32_t)p.k1.sn + c2) * 2u, smem_w + to * TB);
            wide_request(v1p, p.v1.sn, next_tile * TJ, N, wave, lane, (r2 * (uint32_t)p.v1.sn + c2) * 2u, smem_w + (2 + to) * TB);
        }
        if (next_tile == next_last) {
            ++next_round;
            next_tile = round_first(next_round);
            next_last = round_last(next_round);
        } else {
            ++next_tile;
        }
    };
    // ---- q and dO rows kq + u, u in [2r, 2r+32] in round r: pair u / 2 at place (u / 2) % RING ----
    auto request_rows = [&](const uint16_t* base, int64_t sn, int at, unsigned char* ring) {
        const int lane = here();
        const int i = kq + 2 * at + (lane & 1) < N ? kq + 2 * at + (lane & 1) : N - 1;
        __builtin_amdgcn_global_load_lds((wide_glb_ptr)(base + (int64_t)i * sn + (lane >> 1) * 8),
                                         (wide_lds_ptr)(ring + (at % RING) * WT256::GROUP), 16, 0, 0);
    };
    request_tile(0);
    for (int x = wave; x < RING; x += WW) {
        request_rows(qp, p.q.sn, x, q_s);
        request_rows(dop, p.dout.sn, x, do_s);
    }
    for (int c = threadIdx.x; c < WKP_DQ * AS; c += WT) dq_s[c] = 0.f;

    const Tensor& rt = role ? p.v2 : p.k2;                   // the wavefront's K' or V' row, as a row operand holds it
    ux4 raw[DK];
    {
        const int lane = here(), k = k0 + (lane & 31) < N ? k0 + (lane & 31) : N - 1;
        const uint16_t* src = (const uint16_t*)rt.p + rt.off(b, k, h) + (lane >> 5) * 8;
#pragma unroll
        for (int kk = 0; kk < DK; ++kk) raw[kk] = *(const ux4*)(src + kk * 16);
    }
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) asm volatile("" : "+v"(raw[kk]));
    // The pair's unit in a round.  A last round of one unit: the second pair takes the same one with weights of zero, so that
    // a NaN it meets belongs to rows inside the windows (behind them it would reach rows that have no part in it).
    const int last_unit = n_units > 0 ? n_units - 1 : 0;
    auto unit_of = [&](int r) { return 2 * r + pair < last_unit ? 2 * r + pair : last_unit; };
    // LSE * log2(e) (role 0) or D (role 1) of the lane's row, one round ahead
    auto row_value = [&](int r) {
        const int i = kq + (here() & 31) + unit_of(r), ic = i < N ? i : N - 1;
        return role ? p.dsum[(int64_t)bh * N + ic] : p.lse[(int64_t)bh * N + ic] * LOG2E;
    };
    float value_next = row_value(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const uint32_t lds0 = lds_address(smem_w);
    auto k2_of = [&](float x) { return BIASED ? x + p.k2_bias : x; };
    floatx16 pacc[DT];                                       // dK' before the scale (role 0), dV' (role 1)
    zero_acc(pacc);

    // dQ rows [u0, u1) of the ring to the partial, their places to zero
    auto flush = [&](int u0, int u1, int t, int threads) {
        float* part = dq_part + (((int64_t)bh * nkb + kb) * nseg + seg) * (int64_t)RQ * D;
        for (int c = t; c < (u1 - u0) * (D / 4); c += threads) {
            const int u = u0 + c / (D / 4), col = (c % (D / 4)) * 4;
            float4* src = (float4*)(dq_s + (u % WKP_DQ) * AS + col);
            float4 a = u < 2 * nrounds + 32 ? *src : make_float4(0.f, 0.f, 0.f, 0.f);
            *(float4*)(part + (int64_t)u * D + col) = make_float4(a.x * p.scale, a.y * p.scale, a.z * p.scale, a.w * p.scale);
            if (u < 2 * nrounds + 32) *src = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto sweep = [&](auto ROLE) {
        constexpr int R = decltype(ROLE)::value;
        unsigned char* rows_s = R ? do_s : q_s;
        for (int round = 0; round < nrounds; ++round) {
            const int delta = unit_of(round);                // relative to the segment
            const bool has_unit = 2 * round + pair < n_units;
            float value = value_next;
            asm volatile("" : "+v"(value));
            if (round + 1 < nrounds) value_next = row_value(round + 1);
            X8 rf[DK];                                       // Q~ or dO~
            {
#pragma unroll
                for (int kk = 0; kk < DK; ++kk) asm volatile("" : "+v"(raw[kk]));     // (unpacked here, not once for all rounds)
                const int lane = here(), u = (lane & 31) + delta;
                const unsigned char* src = rows_s + ((u >> 1) % RING) * WT256::GROUP + (u & 1) * 16 + (lane >> 5) * 32;
#pragma unroll
                for (int kk = 0; kk < DK; ++kk)
                    rf[kk] = product8<E, BIASED>(*(const ux4*)(src + kk * 64), raw[kk], R ? p.v2_bias : p.k2_bias, R ? 1.f : p.scale * LOG2E);
            }
#pragma unroll
            for (int kk = 0; kk < DK; ++kk) asm volatile("s_nop 1" : "+v"(rf[kk]));
            floatx16 acc[DT];                                // G or R
            zero_acc(acc);
            stay_acc(pacc);
            X8 ro[4][4];                                     // row operands of a chunk of four MFMAs
            lds_half_operand ta[8], tb[8], pa[8], pc[8];     // transposed operands; pa, pc: of the half that runs in the next step
            X8 wb[2];                                        // dS or P
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                pa[t] = pc[t] = lds_half_operand{0, 0, 0, 0};
                wb[0][t] = wb[1][t] = (EL)0.f;
            }
            settle_operand(wb);
            settle_halves(pa);
            settle_halves(pc);
            auto second = [&](lds_half_operand (&x)[8], int dt0, int ks, int y) { mfma_acc(acc[dt0 + y], lds_join<X8>(x[2 * y], x[2 * y + 1]), wb[ks]); };

            const int tile_first = round_first(round), tile_last = round_last(round);
            for (int jt = tile_first; jt <= tile_last; ++jt) {
                const int lane = here(), ln = lane & 31, hf = lane >> 5;
                const uint32_t tile = lds0 + (uint32_t)((2 * R + slot) * TB);
                const uint32_t row_a = tile + (uint32_t)((ln / 2) * WT256::GROUP + (hf * 2 + (ln & 1)) * 16);
                const uint32_t col_a = tile + lds_group_column_lane_offset<WT256::RPW, WT256::GROUP>(lane);
                const uint32_t px_a = lds0 + (uint32_t)(4 * TB + pair * 6144 + lane * 16);
                request_tile(slot ^ 1);
                // ---- S or dP ----
                wide_rows4<0>(row_a, ro[0]);
                wide_rows4<4>(row_a, ro[1]);
#pragma unroll
                for (int y = 0; y < 4; ++y) second(pa, 0, 1, y);
                wide_rows4<8>(row_a, ro[2]);
                floatx16 s;
                lds_wait<8>(ro[0]);
                mfma_vec_zero(s, ro[0][0], rf[0]);
#pragma unroll
                for (int y = 1; y < 4; ++y) mfma_vec(s, ro[0][y], rf[y]);
                wide_rows4<12>(row_a, ro[3]);
                lds_wait<8>(ro[1]);
#pragma unroll
                for (int y = 0; y < 4; ++y) mfma_vec(s, ro[1][y], rf[4 + y]);
                lds_wait<4>(ro[2]);
#pragma unroll
                for (int y = 0; y < 4; ++y) mfma_vec(s, ro[2][y], rf[8 + y]);
                lds_wait<0>(ro[3]);
#pragma unroll
                for (int y = 0; y < 4; ++y) mfma_vec(s, ro[3][y], rf[12 + y]);
                second(pc, 4, 1, 0);
                second(pc, 4, 1, 1);
                wait_acc(s);
                if constexpr (R == 0) {
                    // element v of this lane is key 32 * jt + 8*(v/4) + 4*hf + v%4, the row's query is kq + ln + delta
                    const int j0 = jt * TJ, i_min = kq + delta;
                    if (!(i_min + BQ - 1 < N && has_unit && j0 + TJ - 1 <= i_min && j0 >= i_min + BQ - 1 - w1)) {
                        int hi = i_min + ln - j0 - 4 * hf;
                        opaque(hi);
                        const int lo = hi - w1;
                        const bool row_ok = i_min + ln < N && has_unit;
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int c = 8 * (v >> 2) + (v & 3);
                            s[v] = row_ok && c <= hi && c >= lo ? s[v] : -INFINITY;
                        }
                    }
                    X8 pw[2];
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
#pragma unroll
                        for (int t = 0; t < 8; ++t) {
                            s[8 * g + t] = fast_exp2(s[8 * g + t] - value);
                            pw[g][t] = (EL)s[8 * g + t];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        second(pc, 4, 1, 2 + g);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    lds_write16<0>(px_a, pw[0]);
                    lds_write16<1024>(px_a, pw[1]);
                } else {
                    fx4 d[4];
#pragma unroll
                    for (int v = 0; v < 16; ++v) d[v >> 2][v & 3] = s[v] - value;
                    second(pc, 4, 1, 2);
                    second(pc, 4, 1, 3);
                    lds_write16<2048>(px_a, d[0]);
                    lds_write16<3072>(px_a, d[1]);
                    lds_write16<4096>(px_a, d[2]);
                    lds_write16<5120>(px_a, d[3]);
                }
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                // (both pairs are past the rows of the round before: the places of its first two take the next ones)
                if (round > 0 && jt == tile_first && pair == 0) {
                    if constexpr (R == 0) request_rows(qp, p.q.sn, round + RING - 1, q_s);
                    else request_rows(dop, p.dout.sn, round + RING - 1, do_s);
                }
                // ---- G or R: first half here, second half in the next step ----
                if constexpr (R == 0) {
                    fx4 d[4];
                    lds_read16<2048>(px_a, d[0]);
                    lds_read16<3072>(px_a, d[1]);
                    lds_read16<4096>(px_a, d[2]);
                    lds_read16<5120>(px_a, d[3]);
                    wide_tr_issue<0, 0, 4>(col_a, ta);
                    asm volatile("s_waitcnt lgkmcnt(8)" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]));
                    wide_tr_issue<0, 4, 4>(col_a, tb);
#pragma unroll
                    for (int v = 0; v < 16; ++v) wb[v >> 3][v & 7] = (EL)(s[v] * d[v >> 2][v & 3]);
                    settle_operand(wb);
                } else {
                    lds_read16<0>(px_a, wb[0]);
                    lds_read16<1024>(px_a, wb[1]);
                    wide_tr_issue<0, 0, 4>(col_a, ta);
                    asm volatile("s_waitcnt lgkmcnt(8)" : "+v"(wb[0]), "+v"(wb[1]));
                    wide_tr_issue<0, 4, 4>(col_a, tb);
                }
                lds_wait_halves<8>(ta);
#pragma unroll
                for (int y = 0; y < 4; ++y) second(ta, 0, 0, y);
                wide_tr_issue<1, 0, 4>(col_a, pa);
                lds_wait_halves<8>(tb);
#pragma unroll
                for (int y = 0; y < 4; ++y) second(tb, 4, 0, y);
                wide_tr_issue<1, 4, 4>(col_a, pc);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                lds_wait_halves<0>(pa);
                lds_wait_halves<0>(pc);
                asm volatile("s_barrier" ::: "memory");
                slot ^= 1;
            }
#pragma unroll
            for (int y = 0; y < 4; ++y) second(pa, 0, 1, y);
#pragma unroll
            for (int y = 0; y < 4; ++y) second(pc, 4, 1, y);
            settle_acc(acc);
            // ---- sums over the unit's rows: dK'[k] += G * q[i] or dV'[k] += R * dO[i] ... ----
            {
                const int lane = here(), hf = lane >> 5, u = (lane & 31) + delta;
                const unsigned char* src = rows_s + ((u >> 1) % RING) * WT256::GROUP + (u & 1) * 16 + hf * 8;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const uint2 x = *(const uint2*)(src + (4 * dt + g4) * 32);
                        pacc[dt][4 * g4 + 0] += acc[dt][4 * g4 + 0] * E::lo(x.x);
                        pacc[dt][4 * g4 + 1] += acc[dt][4 * g4 + 1] * E::hi(x.x);
                        pacc[dt][4 * g4 + 2] += acc[dt][4 * g4 + 2] * E::lo(x.y);
                        pacc[dt][4 * g4 + 3] += acc[dt][4 * g4 + 3] * E::hi(x.y);
                    }
                stay_acc(pacc);
            }
            // ... and dQ[k + delta] += G * k2~[k]: the two pairs' rows overlap, so each takes one half of the columns at a time ----
            if (want_dq) {
                if constexpr (R == 0) {
                    auto add_dq = [&](auto HALF) {
                        constexpr int dt0 = decltype(HALF)::value * 4;
                        const int lane = here();
                        float* row = dq_s + (((lane & 31) + delta) % WKP_DQ) * AS + (lane >> 5) * 4;
#pragma unroll
                        for (int kk = 2 * dt0; kk < 2 * dt0 + 8; ++kk) {
                            // the row operand's 16-byte chunks as the accumulators' columns: 16*kk + 4*hf .. and 16*kk + 8 + 4*hf ..
                            const auto e0 = __builtin_amdgcn_permlane32_swap(raw[kk][0], raw[kk][2], false, false);
                            const auto e1 = __builtin_amdgcn_permlane32_swap(raw[kk][1], raw[kk][3], false, false);
#pragma unroll
                            for (int g = 0; g < 2; ++g) {
                                const int dt = kk / 2, g4 = 2 * (kk & 1) + g;
                                float4 a = *(float4*)(row + dt * 32 + 8 * g4);
                                a.x += acc[dt][4 * g4 + 0] * k2_of(E::lo(e0[g]));
                                a.y += acc[dt][4 * g4 + 1] * k2_of(E::hi(e0[g]));
                                a.z += acc[dt][4 * g4 + 2] * k2_of(E::lo(e1[g]));
                                a.w += acc[dt][4 * g4 + 3] * k2_of(E::hi(e1[g]));
                                *(float4*)(row + dt * 32 + 8 * g4) = a;
                            }
                        }
                    };
                    if (pair) add_dq(std::integral_constant<int, 1>{});
                    else add_dq(std::integral_constant<int, 0>{});
                    __syncthreads();
                    if (pair) add_dq(std::integral_constant<int, 0>{});
                    else add_dq(std::integral_constant<int, 1>{});
                    __syncthreads();
                } else {
                    __syncthreads();
                    __syncthreads();
                    flush(2 * round, 2 * round + 2, here() + pair * 64, 128);
                }
            }
        }
    };
    if (role == 0) sweep(std::integral_constant<int, 0>{});
    else sweep(std::integral_constant<int, 1>{});

    // ---- what is left of the dQ partial, then dK' and dV' (two wavefronts each) through LDS ----
    __syncthreads();
    if (want_dq) {
        flush(2 * nrounds, RQ, threadIdx.x, WT);
        __syncthreads();
    }
    float* sums = (float*)smem_w;                            // [WW][32][AS]
    {
        const int lane = here();
        float* row = sums + (wave * 32 + (lane & 31)) * AS + 4 * (lane >> 5);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
                *(float4*)(row + dt * 32 + 8 * g4) = make_float4(pacc[dt][4 * g4], pacc[dt][4 * g4 + 1], pacc[dt][4 * g4 + 2], pacc[dt][4 * g4 + 3]);
    }
    __syncthreads();
    for (int it = threadIdx.x; it < 2 * BQ * (D / 4); it += WT) {
        const int which = it / (BQ * (D / 4));               // 0: dV', 1: dK'
        const int r = it / (D / 4) % BQ, col = it % (D / 4) * 4, k = k0 + r;
        const Tensor& t = which ? p.dk2 : p.dv2;
        if (k >= N || !t.p) continue;
        const float* src = sums + ((which ? 0 : 2) * 32 + r) * AS + col;
        const float4 x = *(const float4*)src, y = *(const float4*)(src + 32 * AS);
        const float sc = which ? p.scale : 1.f;
        const float4 o = make_float4((x.x + y.x) * sc, (x.y + y.y) * sc, (x.z + y.z) * sc, (x.w + y.w) * sc);
        if (nseg > 1) *(float4*)(kpart + ((((int64_t)which * nseg + seg) * p.B * p.H + bh) * N + k) * D + col) = o;
        else *(uint2*)((uint16_t*)t.p + t.off(b, k, h) + col) = make_uint2(pack2<E>(o.x, o.y), pack2<E>(o.z, o.w));
    }
}

// =================================================== backward, K side: dK, dV =====
// A workgroup owns 128 K/V rows, 32 per wavefront, resident in registers as B operands beside the accumulators of all
// 256 columns of dK and dV (384 of the 512 registers of the one wavefront per SIMD), and streams every unit (query
// block, delta) that sees them.  The unit's Q~ and dO~ tiles are formed by all wavefronts from the block's q and dO rows
// and a ring of K' and V' rows in LDS, one unit ahead.
// What bounds it: power; without the forming the units run at the 1.2 PFLOP/s of a large matrix product, and the forming's
// LDS traffic and arithmetic add a quarter.  B1 H8 N4096 w 512/32 bf16: 4900 us in two column passes, 1530 now.  A unit is
// sixteen chunks of four MFMAs; the operands of a chunk are requested two chunks before, an eighth of the forming rides
// on every second one, and the last two chunks run behind the unit's barrier, under the first operand reads of the next.
// nsplit > 1 (grids smaller than the chip): the workgroup takes the sp-th share of the key block's stream of units and
// writes fp32 partial sums to `part` ([dK | dV][nsplit][B*H][N][D]).
template <class E, bool SPLIT, bool BIASED>
__global__ __launch_bounds__(WT) __attribute__((amdgpu_waves_per_eu(1, 1)))
void wide_kv_kernel(Problem p, int njb, int total, int nsplit_arg, float* __restrict__ part) {
    const int nsplit = SPLIT ? nsplit_arg : 1;
    typedef typename E::scalar EL;
    typedef typename E::x8 X8;
    constexpr int D = 256, DK = 16, DT = 8, TB = WT256::BYTES;
    constexpr int RING = WKV_SIDE / 2;                       // pairs of rows in a K'/V' ring
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_w[];
    unsigned char* q_s = smem_w + 4 * TB;                    // (0 .. 3: the Q~ and dO~ tiles of two units)
    unsigned char* do_s = q_s + TB;
    unsigned char* k2_s = do_s + TB;
    unsigned char* v2_s = k2_s + RING * WT256::GROUP;
    float* lse_s = (float*)(v2_s + RING * WT256::GROUP);     // [2][32]  -LSE*log2(e) of the block's queries
    float* dsum_s = lse_s + 2 * 32;                          // [2][32]  -D_i

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pid = xcd_order(blockIdx.x, total);
    const int sp = pid % nsplit, pj = pid / nsplit;
    const int bh = pj / njb, jb = pj - bh * njb;
    const int b = bh / p.H, h = bh - b * p.H;
    const int N = p.N, w1 = p.w1, w2 = p.w2;
    const int j0 = jb * WJ, jw = j0 + 32 * wave;

    const uint16_t* qp = (const uint16_t*)p.q.p + p.q.off(b, 0, h);
    const uint16_t* k1p = (const uint16_t*)p.k1.p + p.k1.off(b, 0, h);
    const uint16_t* k2p = (const uint16_t*)p.k2.p + p.k2.off(b, 0, h);
    const uint16_t* v1p = (const uint16_t*)p.v1.p + p.v1.off(b, 0, h);
    const uint16_t* v2p = (const uint16_t*)p.v2.p + p.v2.off(b, 0, h);
    const uint16_t* dop = (const uint16_t*)p.dout.p + p.dout.off(b, 0, h);
    const float qscale = p.scale * LOG2E;

    // this wavefront's K and V rows as resident B operands (column = key j)
    X8 kf[DK], vf[DK];
    const int ln = threadIdx.x & 31, hf = (threadIdx.x >> 5) & 1, jc = jw + ln < N ? jw + ln : N - 1;
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
        kf[kk] = *(const X8*)(k1p + (int64_t)jc * p.k1.sn + kk * 16 + hf * 8);
        vf[kk] = *(const X8*)(v1p + (int64_t)jc * p.v1.sn + kk * 16 + hf * 8);
    }
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) asm volatile("" : "+v"(kf[kk]), "+v"(vf[kk]));     // (here, so that nothing waits for them in the stream)
    const int j_last = j0 + WJ - 1 < N ? j0 + WJ - 1 : N - 1;
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

    // ---- rows of a query block: q and dO, and the first rows of the K'/V' rings.  Row u of a ring counts back from row
    //      i0 + 31 - d0 (d0: the first delta of the block's run); unit delta takes the rows delta - d0 .. delta - d0 + 31 ----
    // (what derives from the lane is computed where it is used: kept in registers through the stream it costs the operands theirs)
    auto here = [&]() {
        int t = threadIdx.x;
        opaque(t);
        return t & 63;
    };
    auto request_side = [&](const uint16_t* base, int64_t sn, int top, int pair, unsigned char* ring) {
        const int lane = here();
        int k = top - 2 * pair - (lane & 1);
        k = k < 0 ? 0 : (k < N ? k : N - 1);
        __builtin_amdgcn_global_load_lds((wide_glb_ptr)(base + (int64_t)k * sn + (lane >> 1) * 8),
                                         (wide_lds_ptr)(ring + (pair % RING) * WT256::GROUP), 16, 0, 0);
    };
    auto request_block = [&](int ib, int d0, int par) {
        const int lane = here();
        int i = ib * BQ + (lane & 31);
        i = i < N ? i : N - 1;
        const float lse = p.lse[(int64_t)bh * N + i], dsum = p.dsum[(int64_t)bh * N + i];
        const uint32_t r2 = 8 * wave + (lane & 1), c2 = (lane >> 1) * 8;
        wide_request(qp, p.q.sn, ib * BQ, N, wave, lane, (r2 * (uint32_t)p.q.sn + c2) * 2u, q_s);
        wide_request(dop, p.dout.sn, ib * BQ, N, wave, lane, (r2 * (uint32_t)p.dout.sn + c2) * 2u, do_s);
        for (int x = wave; x < RING; x += WW) {
            request_side(k2p, p.k2.sn, ib * BQ + BQ - 1 - d0, x, k2_s);
            request_side(v2p, p.v2.sn, ib * BQ + BQ - 1 - d0, x, v2_s);
        }
        if (wave == 0 && lane < 32) {
            lse_s[par * 32 + lane] = -lse * LOG2E;
            dsum_s[par * 32 + lane] = -dsum;
        }
    };

    // ---- forming: this wavefront's groups wave + 4x of the tiles, one 16-byte chunk per lane, tensor and x ----
    const uint32_t lds0 = lds_address(smem_w);
    constexpr uint32_t XG = 4 * WT256::GROUP;
    int du = 0;                                              // unit to form: delta - d0
    auto place_of = [&](int lane) { return (BQ - 1 - 2 * wave - (lane & 1) + du) % WKV_SIDE; };      // of the row that goes with group `wave`
    auto ring_at = [&](int lane, int place, int x) {         // byte offset of the row that goes with group wave + 4x
        int g = (place >> 1) - 4 * x;
        g = g < 0 ? g + RING : g;
        return (uint32_t)(g * WT256::GROUP + (place & 1) * 16 + (lane >> 1) * 32);
    };
    auto form_plain = [&](int buf) {
        const int lane = here(), place = place_of(lane);
        const uint32_t form_lane = (uint32_t)(wave * WT256::GROUP + lane * 16);
#pragma unroll 1
        for (int x = 0; x < 4; ++x) {
            const uint32_t r = ring_at(lane, place, x);
            const ux4 qa = *(const ux4*)(q_s + form_lane + x * XG), ka = *(const ux4*)(k2_s + r);
            const ux4 da = *(const ux4*)(do_s + form_lane + x * XG), va = *(const ux4*)(v2_s + r);
            *(X8*)(smem_w + (2 * buf) * TB + form_lane + x * XG) = product8<E>(qa, ka, p.k2_bias, qscale);
            *(X8*)(smem_w + (2 * buf + 1) * TB + form_lane + x * XG) = product8<E>(da, va, p.v2_bias, 1.f);
        }
    };

    int ib = ib_lo, delta = d_first, d0 = d_first, nu = units_of(ib_lo), buf = 0, par = 0;
    request_block(ib, d0, par);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    form_plain(0);
    __syncthreads();

    X8 ro[4][4];                                             // row operands and (halves of) transposed operands of
    lds_half_operand to[4][8];                               // the chunks c, by c % 4
    X8 pb[2], dsb[2];
    floatx16 dkacc[DT], dvacc[DT];
    // (the last two chunks of a unit run at the start of the wavefront's next one: none outstanding yet)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            dsb[x][t] = (EL)0.f;
            to[2 + x][t] = lds_half_operand{0, 0, 0, 0};
        }
    settle_operand(dsb);
    settle_halves(to[2]);
    settle_halves(to[3]);
    // chunk c of a unit: 0-3 S, 4-7 dP, 8-11 dV, 12-15 dK
    auto issue = [&](auto C, uint32_t row_a, uint32_t col_a) {
        constexpr int c = decltype(C)::value;
        if constexpr (c < 8) wide_rows4<(c & 3) * 4>(row_a + (c < 4 ? 0u : (uint32_t)TB), ro[c & 3]);
        else wide_tr_issue<(c >> 1) & 1, (c & 1) * 4, 4>(col_a + (c < 12 ? (uint32_t)TB : 0u), to[c & 3]);
    };
    auto tail_mfma = [&](auto C, int x) {                    // dV and dK
        constexpr int c = decltype(C)::value;
        const X8 a = lds_join<X8>(to[c & 3][2 * x], to[c & 3][2 * x + 1]);
        constexpr int dt0 = (c & 1) * 4, ks = (c >> 1) & 1;
        if constexpr (c < 12) mfma_acc(dvacc[dt0 + x], a, pb[ks]);
        else mfma_acc(dkacc[dt0 + x], a, dsb[ks]);
    };
    auto tail_chunk = [&](auto C) {
#pragma unroll
        for (int x = 0; x < 4; ++x) tail_mfma(C, x);
    };
    // One unit, and beside it the forming of the next one of the query block (after the last one: of nothing that is used).
    // LDS operations return in order: a wait for n outstanding ones is a wait for everything issued before the last n.
    // The vector ALU's work sits between the MFMAs one by one: a wavefront issues in order, and alone on its SIMD it
    // would leave the matrix pipe idle for as long as a longer piece takes.
    auto unit = [&]() {
        const int lane = here(), ln = lane & 31, hf = lane >> 5, j = jw + ln;
        const uint32_t form_lane = (uint32_t)(wave * WT256::GROUP + lane * 16);
        const uint32_t row_lane = (uint32_t)((ln / 2) * WT256::GROUP + (hf * 2 + (ln & 1)) * 16);
        const uint32_t col_lane = lds_group_column_lane_offset<WT256::RPW, WT256::GROUP>(lane);
        const int place = place_of(lane);
        const uint32_t tile = lds0 + (uint32_t)(buf * 2 * TB), row_a = tile + row_lane, col_a = tile + col_lane;
        const uint32_t next = lds0 + (uint32_t)((buf ^ 1) * 2 * TB) + form_lane;
        const uint32_t raw_a = lds0 + 4 * TB + form_lane, ring_a = lds0 + 6 * TB;
        const uint32_t per_query = lds0 + (uint32_t)(6 * TB + 2 * RING * WT256::GROUP + par * 128 + hf * 16);
        const int i0 = ib * BQ;
        // register v of this lane: query i0 + 8*(v/4) + 4*hf + v%4, key j
        const bool interior = (i0 >= jw + 31) && ((int64_t)i0 + 31 <= (int64_t)jw + w1) && (i0 + BQ - 1 < N) && (i0 >= delta);
        // The forming in eight slices of one 16-byte chunk each (group wave + 4 * (k / 2), Q~ for even k and dO~ for odd):
        // slice 0 beside the tail of the unit before, slice k beside the chunks 2k-2 and 2k-1, a pair of elements after
        // every second MFMA.
        ux4 fa[2], fb[2];
        auto form_read = [&](auto K) {
            constexpr int k = decltype(K)::value, x = k >> 1, which = k & 1;
            lds_read16<which * TB + x * (int)XG>(raw_a, fa[which]);
            lds_read16<which * RING * WT256::GROUP>(ring_a + ring_at(lane, place, x), fb[which]);
        };
        auto form_pair = [&](auto K, int y) {
            constexpr int which = decltype(K)::value & 1;
            const float bias = which ? p.v2_bias : p.k2_bias, mul = which ? 1.f : qscale;
            const uint32_t u = fa[which][y], v = fb[which][y];
            if constexpr (BIASED) fa[which][y] = pack2<E>(E::lo(u) * mul * (E::lo(v) + bias), E::hi(u) * mul * (E::hi(v) + bias));
            else fa[which][y] = pack2<E>(E::lo(u) * mul * E::lo(v), E::hi(u) * mul * E::hi(v));
        };
        auto form_write = [&](auto K) {
            constexpr int k = decltype(K)::value;
            lds_write16<(k & 1) * TB + (k >> 1) * (int)XG>(next, fa[k & 1]);
        };
        fx4 lp[4], dp[4];
        lds_read16<0>(per_query, lp[0]);
        lds_read16<32>(per_query, lp[1]);
        lds_read16<64>(per_query, lp[2]);
        lds_read16<96>(per_query, lp[3]);
        form_read(std::integral_constant<int, 0>{});
        issue(std::integral_constant<int, 0>{}, row_a, col_a);
        tail_chunk(std::integral_constant<int, 14>{});
        form_read(std::integral_constant<int, 1>{});
        issue(std::integral_constant<int, 1>{}, row_a, col_a);
        asm volatile("s_waitcnt lgkmcnt(10)" : "+v"(fa[0]), "+v"(fb[0]));
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            tail_mfma(std::integral_constant<int, 15>{}, y);
            __builtin_amdgcn_sched_barrier(0);
            form_pair(std::integral_constant<int, 0>{}, y);
            __builtin_amdgcn_sched_barrier(0);
        }
        form_write(std::integral_constant<int, 0>{});
        floatx16 sacc, dpacc;
        static_for<16>([&](auto CC) {
            constexpr int c = decltype(CC)::value;
            if constexpr ((c & 1) == 1 && c < 13) form_read(std::integral_constant<int, (c + 3) / 2>{});
            if constexpr (c == 3) {
                lds_read16<256>(per_query, dp[0]);
                lds_read16<288>(per_query, dp[1]);
                lds_read16<320>(per_query, dp[2]);
                lds_read16<352>(per_query, dp[3]);
            }
            if constexpr (c < 14) issue(std::integral_constant<int, c + 2>{}, row_a, col_a);
            // what may be outstanding: the operands of the next two chunks, and the forming's accesses beside them
            constexpr int len1 = c + 1 > 15 ? 0 : c + 1 < 8 ? 4 : 8, len2 = c + 2 > 15 ? 0 : c + 2 < 8 ? 4 : 8;
            constexpr int want = len1 + len2 + ((c & 1) ? (c < 13 ? 2 : 0) + (c == 3 ? 4 : 0) : c < 14 ? 1 : 0);
            constexpr int n = want > 15 ? 15 : want;
            if constexpr (c < 8) lds_wait<n>(ro[c & 3]);
            else lds_wait_halves<n>(to[c & 3]);
            if constexpr (c == 0) {
                arrived(lp[0], lp[1]);
                arrived(lp[2], lp[3]);
#pragma unroll
                for (int v = 0; v < 16; ++v) sacc[v] = lp[v >> 2][v & 3];
                settle_c(sacc);
            }
            if constexpr (c == 4) {
                arrived(dp[0], dp[1]);
                arrived(dp[2], dp[3]);
#pragma unroll
                for (int v = 0; v < 16; ++v) dpacc[v] = dp[v >> 2][v & 3];
                settle_c(dpacc);
            }
            if constexpr ((c & 1) == 0 && c < 14) arrived(fa[(c / 2 + 1) & 1], fb[(c / 2 + 1) & 1]);
            if constexpr (c == 6) {
                wait_acc(sacc);
                if (!interior) {
                    int lo = j - i0 - 4 * hf;                                          // c >= lo  <=>  j <= i
                    opaque(lo);                           // (a branch: few units need the mask)
                    const int hi = lo < (1 << 20) - w1 ? lo + w1 : (1 << 20);          // i <= j + w1
                    const int dlo = delta - j + lo, nhi = N - 1 - j + lo;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int y = 8 * (v >> 2) + (v & 3);
                        sacc[v] = (j < N) && (y >= lo) && (y <= hi) && (y >= dlo) && (y <= nhi) ? sacc[v] : -INFINITY;
                    }
                }
            }
            if constexpr (c == 10) wait_acc(dpacc);
            if constexpr (c < 14) {
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    if constexpr (c < 4) mfma_vec(sacc, ro[c & 3][y], kf[4 * c + y]);
                    else if constexpr (c < 8) mfma_vec(dpacc, ro[c & 3][y], vf[4 * (c - 4) + y]);
                    else tail_mfma(CC, y);
                    __builtin_amdgcn_sched_barrier(0);
                    if ((y & 1) == 0) form_pair(std::integral_constant<int, c / 2 + 1>{}, 2 * (c & 1) + y / 2);
                    if constexpr (c == 6 || c == 7) {                    // the weights P
#pragma unroll
                        for (int v = 8 * (c - 6) + 2 * y; v < 8 * (c - 6) + 2 * y + 2; ++v) {
                            sacc[v] = fast_exp2(sacc[v]);
                            pb[v >> 3][v & 7] = (EL)sacc[v];
                        }
                    }
                    if constexpr (c == 10 || c == 11) {                  // dS
#pragma unroll
                        for (int v = 8 * (c - 10) + 2 * y; v < 8 * (c - 10) + 2 * y + 2; ++v) dsb[v >> 3][v & 7] = (EL)(sacc[v] * dpacc[v]);
                    }
                    if ((c & 1) == 1 && y == 2) form_write(std::integral_constant<int, c / 2 + 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (c == 7) settle_operand(pb);
                if constexpr (c == 11) settle_operand(dsb);
            }
        });
    };

    bool more = true;
    // one unit of the stream: requests and forming of what comes next, with the wavefront's own work on it or without
    auto step = [&](auto WORK) {
        int nib = ib, ndelta = delta + 1;
        if (ndelta >= nu) {
            nib = ib + 1;
            ndelta = 0;
        }
        more = SPLIT ? (nib < ib_hi || (nib == ib_hi && ndelta <= d_last)) : nib <= ib_hi;
        const bool form = more && nib == ib;                 // the next unit belongs to the same query block
        du = form ? ndelta - d0 : 0;
        if (form) {
            if ((du & 3) == 0) {                             // four more rows for each ring, where four are no longer needed
                const int pair = (du + WKV_SIDE - 4) / 2 + (wave & 1), top = ib * BQ + BQ - 1 - d0;
                if (wave < 2) request_side(k2p, p.k2.sn, top, pair, k2_s);
                else request_side(v2p, p.v2.sn, top, pair, v2_s);
            }
        } else if (more) {
            request_block(nib, 0, par ^ 1);
        }
        if constexpr (decltype(WORK)::value) unit();
        else if (form) form_plain(buf ^ 1);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (more && nib != ib) {
            nu = units_of(nib);
            d0 = 0;
            par ^= 1;
            form_plain(buf ^ 1);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        ib = nib;
        delta = ndelta;
        buf ^= 1;
    };
    // the wavefront's keys are seen by a run of query blocks (none: keys past the end of the sequence, or an empty share)
    const int t_lo = jw / BQ, t_hi = jw < N && !empty_share ? (int)(((int64_t)jw + 31 + w1) / BQ < (1 << 26) ? ((int64_t)jw + 31 + w1) / BQ : (1 << 26)) : -1;
    zero_acc(dkacc);
    zero_acc(dvacc);
    while (more && (ib < t_lo || t_hi < 0)) step(std::false_type{});
    while (more && ib <= t_hi) step(std::true_type{});
    tail_chunk(std::integral_constant<int, 14>{});
    tail_chunk(std::integral_constant<int, 15>{});
    while (more) step(std::false_type{});
    settle_acc(dkacc);
    settle_acc(dvacc);

    const int lane_f = here(), hf_f = lane_f >> 5, j = jw + (lane_f & 31);
    if (j < N && SPLIT) {
        const int64_t BH = (int64_t)p.B * p.H;
        float* dkp = p.dk1.p ? part + (((0 * (int64_t)nsplit + sp) * BH + bh) * N + j) * D + 4 * hf_f : nullptr;
        float* dvp = p.dv1.p ? part + (((1 * (int64_t)nsplit + sp) * BH + bh) * N + j) * D + 4 * hf_f : nullptr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                if (dkp) *(float4*)(dkp + dt * 32 + 8 * g4) = make_float4(dkacc[dt][4 * g4] * LN2, dkacc[dt][4 * g4 + 1] * LN2,
                                                                           dkacc[dt][4 * g4 + 2] * LN2, dkacc[dt][4 * g4 + 3] * LN2);
                if (dvp) *(float4*)(dvp + dt * 32 + 8 * g4) = make_float4(dvacc[dt][4 * g4], dvacc[dt][4 * g4 + 1], dvacc[dt][4 * g4 + 2],
                                                                           dvacc[dt][4 * g4 + 3]);
            }
    } else if (j < N) {
        uint16_t* dkp = p.dk1.p ? (uint16_t*)p.dk1.p + p.dk1.off(b, j, h) + 4 * hf_f : nullptr;
        uint16_t* dvp = p.dv1.p ? (uint16_t*)p.dv1.p + p.dv1.off(b, j, h) + 4 * hf_f : nullptr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                // Q~ carries scale*log2(e): dK = ln2 * sum dS * Q~
                if (dkp) *(uint2*)(dkp + dt * 32 + 8 * g4) = make_uint2(E::pack(dkacc[dt][4 * g4] * LN2, dkacc[dt][4 * g4 + 1] * LN2),
                                                                         E::pack(dkacc[dt][4 * g4 + 2] * LN2, dkacc[dt][4 * g4 + 3] * LN2));
                if (dvp) *(uint2*)(dvp + dt * 32 + 8 * g4) = make_uint2(E::pack(dvacc[dt][4 * g4], dvacc[dt][4 * g4 + 1]),
                                                                         E::pack(dvacc[dt][4 * g4 + 2], dvacc[dt][4 * g4 + 3]));
            }
    }
}

// Shares of a key block's stream of units: the least time by grid_time with about 2.3 us per unit and the time of a dozen
// units around them: within 6 % of the best of sixteen at eight sizes.  Partial sums may take 64 MiB, or `room`.
int wide_kv_nsplit(int B, int N, int H, int D, int w1, int w2, size_t room) {
    constexpr double UNIT = 2.3, AROUND = 12;
    const int64_t bh = (int64_t)B * H, base = bh * ((N + WJ - 1) / WJ);
    const int64_t units = (int64_t)((WJ + (w1 < N ? w1 : N)) / BQ + 1) * ((w2 < N - 1 ? w2 : N - 1) + 1);      // of a key block's stream, at most
    const double fill = window_fill(w1, N) * window_fill(w2, N);
    int best = 1;
    double least = 0;
    for (int ns = 1; ns <= 16 && units / ns >= 4; ++ns) {
        const double part = ns > 1 ? 2.0 * ns * bh * N * D * 4 : 0, per = (double)((units + ns - 1) / ns);
        if (part > 67108864.0 || part > (double)room) break;
        const double cost = UNIT * grid_time(base * ns, per + AROUND, per * fill + AROUND) + (ns > 1 ? SUM_LAUNCH_STEPS + part / PART_BYTES_PER_STEP : 0);
        if (least == 0 || cost < 0.97 * least) {
            least = cost;
            best = ns;
        }
    }
    return best;
}
size_t wide_dq_part_bytes(int B, int N, int H, const KpPlan& pl) {
    return ((size_t)B * H * ((N + BQ - 1) / BQ) * pl.nseg * (size_t)(BQ + pl.segw - 1) * 256 * sizeof(float) + 255) / 256 * 256;
}
size_t wide_kp_part_bytes(int B, int N, int H, const KpPlan& pl) { return pl.nseg > 1 ? (size_t)2 * pl.nseg * B * H * (size_t)N * 256 * sizeof(float) : 0; }
KpPlan wide_kp_plan(int B, int N, int H, int w1, int w2, size_t room) {
    return plan_segments(B, N, H, w1, w2, 2, w2 + 1, room, [](int) { return false; },      // (the work between two sweeps takes long here)
                         [&](const KpPlan& pl) { return wide_dq_part_bytes(B, N, H, pl) + wide_kp_part_bytes(B, N, H, pl); });
}
size_t wide_kp_bytes(int B, int N, int H, int w1, int w2, size_t room) {
    const KpPlan pl = wide_kp_plan(B, N, H, w1, w2, room);
    return (wide_dq_part_bytes(B, N, H, pl) + wide_kp_part_bytes(B, N, H, pl) + 255) / 256 * 256;
}

// ------------------------------------------------------------------ launchers ----
template <class E>
int launch_wide_fwd_of(const Problem& p, hipStream_t st) {
    const int nqb = (p.N + BQ - 1) / BQ, nsplit = p.nsplit > 1 ? p.nsplit : 1;
    const int64_t total = (int64_t)nqb * p.B * p.H * nsplit;
    if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    auto go = [&](auto kernel) {
        if (!allow_full_lds((const void*)kernel)) return false;
        hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(WT), WIDE_FWD_LDS, st, p, nqb, (int)total);
        return hipGetLastError() == hipSuccess;
    };
    if (!(nsplit > 1 ? go(wide_fwd_kernel<E, true>) : go(wide_fwd_kernel<E, false>))) return SA2_ERR_LAUNCH_FAILED;
    return nsplit > 1 ? launch_fwd_merge(p, 256, E::DTYPE, st) : SA2_OK;
}

template <class E>
int launch_wide_bwd_of(const Problem& p, hipStream_t st) {
    constexpr int D = 256;
    int rc = launch_rowdot(p.out, p.dout, p.dsum, p.B, p.N, p.H, p.D, E::DTYPE, st);
    if (rc != SA2_OK) return rc;
    const bool biased = p.k2_bias != 0.f || p.v2_bias != 0.f;           // (the common case pays for none of it)
    BwdSums sums = {};
    const KpPlan pl = wide_kp_plan(p.B, p.N, p.H, p.w1, p.w2, p.room);
    const size_t kp_bytes = wide_kp_bytes(p.B, p.N, p.H, p.w1, p.w2, p.room);
    const int nsplit = wide_kv_nsplit(p.B, p.N, p.H, D, p.w1, p.w2, room_left(p.room, kp_bytes));
    if (((p.dq.p || pl.nseg > 1) || nsplit > 1) && p.scratch_bytes < wide_bwd_scratch_bytes(p.B, p.N, p.H, D, p.w1, p.w2, p.room)) return SA2_ERR_WORKSPACE_TOO_SMALL;
    if (p.dq.p || p.dk2.p || p.dv2.p) {
        const int nkb = (p.N + BQ - 1) / BQ;
        const int64_t total = (int64_t)nkb * p.B * p.H * pl.nseg;
        if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
        float* part = (float*)p.scratch;
        float* kpart = (float*)((char*)p.scratch + wide_dq_part_bytes(p.B, p.N, p.H, pl));
        auto go = [&](auto kernel) {
            if (!allow_full_lds((const void*)kernel)) return false;
            hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(WT), WIDE_KP_LDS, st, p, nkb, (int)total, part, pl.nseg, pl.segw, kpart);
            return hipGetLastError() == hipSuccess;
        };
        if (!(biased ? go(wide_kp_kernel<E, true>) : go(wide_kp_kernel<E, false>))) return SA2_ERR_LAUNCH_FAILED;
        sums.dq = p.dq.p ? part : nullptr;
        sums.nkb = nkb;
        sums.nseg = pl.nseg;
        sums.segw = pl.segw;
        sums.kp = pl.nseg > 1 ? kpart : nullptr;
        sums.kp_n = pl.nseg;
    }
    if (p.dk1.p || p.dv1.p) {
        const int njb = (p.N + WJ - 1) / WJ;
        const int64_t total = (int64_t)njb * p.B * p.H * nsplit;
        if (total > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
        float* part = (float*)((char*)p.scratch + kp_bytes);
        auto go = [&](auto kernel) {
            if (!allow_full_lds((const void*)kernel)) return false;
            hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(WT), WIDE_KV_LDS, st, p, njb, (int)total, nsplit, part);
            return hipGetLastError() == hipSuccess;
        };
        if (!(nsplit > 1 ? (biased ? go(wide_kv_kernel<E, true, true>) : go(wide_kv_kernel<E, true, false>))
                         : (biased ? go(wide_kv_kernel<E, false, true>) : go(wide_kv_kernel<E, false, false>)))) return SA2_ERR_LAUNCH_FAILED;
        sums.kv = nsplit > 1 ? part : nullptr;
        sums.kv_n = nsplit;
    }
    return launch_bwd_sums(p, sums, D, E::DTYPE, st);
}

}  // namespace

bool wide_supported(int D, int dtype) { return (dtype == SA2_BF16 || dtype == SA2_F16) && D == 256; }

bool wide_bwd_supported(int D, int w2, int dtype) {
    (void)w2;                // any K' window: wide ones are walked in segments
    return wide_supported(D, dtype);
}

size_t wide_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room) {
    const size_t kp_bytes = wide_kp_bytes(B, N, H, w1, w2, room);
    const int ns = wide_kv_nsplit(B, N, H, D, w1, w2, room_left(room, kp_bytes));
    return kp_bytes + (ns > 1 ? (size_t)2 * ns * B * H * (size_t)N * D * sizeof(float) : 0);
}

int wide_fwd_nsplit(int B, int N, int H, int w1, int w2, size_t room) { return plan_forward(B, N, H, 256, w1, w2, WW, 0, room); }

int launch_wide_fwd(const Problem& p, int dtype, hipStream_t st) {
    return dtype == SA2_F16 ? launch_wide_fwd_of<ElemF16>(p, st) : launch_wide_fwd_of<ElemBF16>(p, st);
}

int launch_wide_bwd(const Problem& p, int dtype, hipStream_t st) {
    return dtype == SA2_F16 ? launch_wide_bwd_of<ElemF16>(p, st) : launch_wide_bwd_of<ElemBF16>(p, st);
}

}  // namespace sa2
