// MFMA backward for gfx950 (bf16 or fp16, head_dim 32, 64 or 128): dispatch to the two kernels,
// sa2_mfma_bwd_kp.hip for dQ, dK', dV' and sa2_mfma_bwd_kv.hip for dK, dV, after the row-dot kernel.
//
// Same expanded-row view as the forward: rows r = (i, delta), Q~[r] = q[i] *
// k2~[i-delta] * scale*log2(e) and dO~[r] = dO[i] * v2~[i-delta], both in the element type, with
// P = exp2(S - LSE*log2e) recomputed from the saved log-sum-exp and dS = P * (dO~.v1 - D_i).
// Both kernels take any K' window: one too wide for their LDS buffers is walked in segments of deltas.
//
// Every output element has one writer and a fixed summation order: no atomics,
// bitwise reproducible.
#include "sa2_mfma_common.h"

namespace sa2 {
namespace {

// E: the gradients' element type (float or a 16-bit one).
// The gradients that the two kernels left as fp32 partial sums, one launch for all of them (grid dimension y).
// Four columns of one row per thread; what bounds it is reading the partials once.  (A kernel per kind, as before, cost
// three launches of 5-10 us each at small sizes, most of it latency: the partials of a row were read one after the
// other.  Here four reads are in flight.)
constexpr int SUM_DQ = 0, SUM_DK1 = 1, SUM_DV1 = 2, SUM_DV2 = 3, SUM_DK2 = 4;
template <class E>
__global__ __launch_bounds__(256) void bwd_sum_kernel(Problem p, BwdSums s, int D, unsigned kinds, int64_t items) {
    const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (it >= items) return;
    const int kind = (kinds >> (4 * blockIdx.y)) & 15;
    const int col = (int)(it % (D / 4)) * 4;
    if (col >= p.D) return;
    const int64_t rowid = it / (D / 4);
    const int i = (int)(rowid % p.N), bh = (int)(rowid / p.N);
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](const float* src) {
        const float4 y = *(const float4*)src;
        acc.x += y.x; acc.y += y.y; acc.z += y.z; acc.w += y.w;
    };
    if (kind == SUM_DQ) {
        // the partials of the K' blocks and segments that reach query i, in block and segment order
        const int reach = BQ + p.w2, rows = BQ + s.segw - 1;         // queries a block reaches; rows of one partial
        const int kb_lo = i - reach + 1 <= 0 ? 0 : (i - reach + BQ) / BQ, kb_hi = i / BQ;
        const float* base = s.dq + (int64_t)bh * s.nkb * s.nseg * rows * D + col;
        if (s.nseg == 1) {
#pragma unroll 4
            for (int kb = kb_lo; kb <= kb_hi; ++kb) add(base + ((int64_t)kb * rows + (i - kb * BQ)) * D);
        } else {
            for (int kb = kb_lo; kb <= kb_hi; ++kb) {
                const int rel = i - kb * BQ;                         // segment g holds rel - g * segw in [0, rows)
                const int hi = rel / s.segw < s.nseg - 1 ? rel / s.segw : s.nseg - 1;
                const int lo = rel - rows + 1 <= 0 ? 0 : (rel - rows + s.segw) / s.segw;
#pragma unroll 4
                for (int g = lo; g <= hi; ++g) add(base + (((int64_t)kb * s.nseg + g) * rows + (rel - g * s.segw)) * D);
            }
        }
    } else {
        const bool k_side = kind <= SUM_DV1;
        const int which = k_side ? kind - SUM_DK1 : kind - SUM_DV2, n = k_side ? s.kv_n : s.kp_n;
        const int64_t step = (int64_t)p.B * p.H * p.N * D;           // one share or segment
        const float* src = (k_side ? s.kv : s.kp) + (int64_t)which * n * step + rowid * D + col;
#pragma unroll 4
        for (int x = 0; x < n; ++x) add(src + x * step);
    }
    const Tensor& t = kind == SUM_DQ ? p.dq : kind == SUM_DK1 ? p.dk1 : kind == SUM_DV1 ? p.dv1 : kind == SUM_DV2 ? p.dv2 : p.dk2;
    const int b = bh / p.H, h = bh - b * p.H;
    if constexpr (std::is_same<E, float>::value) *(float4*)((float*)t.p + t.off(b, i, h) + col) = acc;
    else *(uint2*)((uint16_t*)t.p + t.off(b, i, h) + col) = make_uint2(E::pack(acc.x, acc.y), E::pack(acc.z, acc.w));
}

// out and LSE of a split forward: the shares' sums brought to a common reference exponent, in share order.  One
// thread per four columns, four shares' reads in flight; bound by reading the partial outputs once.
template <class E>
__global__ __launch_bounds__(256) void fwd_merge_kernel(Problem p, int D, int64_t items) {
    const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (it >= items) return;
    const int col = (int)(it % (D / 4)) * 4;
    if (col >= p.D) return;
    const int64_t row = it / (D / 4), rows = (int64_t)p.B * p.H * p.N;
    const float2* ml = (const float2*)p.scratch;                       // (M, L) of [share][row]
    const float* part = (const float*)p.scratch + 2 * rows * p.nsplit;
    float M = -INFINITY;
    int e = -126;
#pragma unroll 4
    for (int x = 0; x < p.nsplit; ++x) {
        const float2 s = ml[x * rows + row];
        M = fmaxf(M, s.x);
        const int es = __builtin_amdgcn_frexp_expf(s.y);
        e = es > e ? es : e;
    }
    const float Mu = M == -INFINITY ? 0.f : M;
    // M need not be the row's maximum: all sums in units of 2^e, so that those of up to sixteen shares add up without overflow
    e += 4;
    const float Me = Mu + (float)e;
    float L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int x = 0; x < p.nsplit; ++x) {
        const float2 s = ml[x * rows + row];
        if (s.x == -INFINITY && s.y == 0.f) continue;                  // (an empty share left no sums; NaN logits leave L NaN)
        const float w = ldexpf(fast_exp2(s.x - Mu), -e);
        const float4 y = *(const float4*)(part + (x * rows + row) * D + col);
        L += w * s.y;
        acc.x += w * y.x; acc.y += w * y.y; acc.z += w * y.z; acc.w += w * y.w;
    }
    // sum + 1e-8 in units of 2^Me; for a tiny Me the epsilon dominates
    const bool big = Me > LOG2_EPS;
    const float denom = big ? L + 1e-8f * fast_exp2(-Me) : L * fast_exp2(Me - LOG2_EPS) + 1.f;
    const float inv = big ? 1.f / denom : fast_exp2(Me - LOG2_EPS) / denom;
    const int i = (int)(row % p.N), bh = (int)(row / p.N), b = bh / p.H, h = bh - b * p.H;
    if constexpr (std::is_same<E, float>::value)
        *(float4*)((float*)p.out.p + p.out.off(b, i, h) + col) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
    else
        *(uint2*)((uint16_t*)p.out.p + p.out.off(b, i, h) + col) = make_uint2(E::pack(acc.x * inv, acc.y * inv), E::pack(acc.z * inv, acc.w * inv));
    if (col == 0) p.lse[row] = exact_lse(Mu, denom, big, e);
}

}  // namespace

int launch_fwd_merge(const Problem& p, int width, int dtype, hipStream_t st) {
    const int64_t items = (int64_t)p.B * p.H * p.N * (width / 4);
    const dim3 grid((unsigned)((items + 255) / 256));
    if (dtype == SA2_F32) hipLaunchKernelGGL((fwd_merge_kernel<float>), grid, dim3(256), 0, st, p, width, items);
    else if (dtype == SA2_F16) hipLaunchKernelGGL((fwd_merge_kernel<ElemF16>), grid, dim3(256), 0, st, p, width, items);
    else hipLaunchKernelGGL((fwd_merge_kernel<ElemBF16>), grid, dim3(256), 0, st, p, width, items);
    return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
}

bool mfma_bwd_supported(int B, int N, int H, int D, int w1, int w2, int dtype) {
    return mfma_supported(B, N, H, D, w1, w2, dtype);
}

// Workspace of the K'-side kernel (dQ partials, and the dK', dV' partials of a segmented launch),
// rounded up so that what follows it stays 256-byte aligned
size_t kp_side_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room) {
    return (kp_scratch_bytes(B, N, H, D, w1, w2, room) + 255) / 256 * 256;
}

size_t mfma_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room) {
    return kp_side_scratch_bytes(B, N, H, D, w1, w2, room) + kv_split_scratch_bytes(B, N, H, D, w1, w2, room);
}

int launch_bwd_sums(const Problem& p, const BwdSums& sums, int width, int dtype, hipStream_t st) {
    unsigned kinds = 0;
    int n = 0;
    auto want = [&](int kind, const float* part, const Tensor& t) {
        if (part && t.p) kinds |= (unsigned)kind << (4 * n++);
    };
    want(SUM_DQ, sums.dq, p.dq);
    want(SUM_DK1, sums.kv, p.dk1);
    want(SUM_DV1, sums.kv, p.dv1);
    want(SUM_DV2, sums.kp, p.dv2);
    want(SUM_DK2, sums.kp, p.dk2);
    if (n == 0) return SA2_OK;
    const int64_t items = (int64_t)p.B * p.H * p.N * (width / 4);
    const dim3 grid((unsigned)((items + 255) / 256), (unsigned)n);
    if (dtype == SA2_F32) hipLaunchKernelGGL((bwd_sum_kernel<float>), grid, dim3(256), 0, st, p, sums, width, kinds, items);
    else if (dtype == SA2_F16) hipLaunchKernelGGL((bwd_sum_kernel<ElemF16>), grid, dim3(256), 0, st, p, sums, width, kinds, items);
    else hipLaunchKernelGGL((bwd_sum_kernel<ElemBF16>), grid, dim3(256), 0, st, p, sums, width, kinds, items);
    return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED;
}

int launch_mfma_bwd(const Problem& p, int dtype, hipStream_t st) {
    int rc = launch_rowdot(p.out, p.dout, p.dsum, p.B, p.N, p.H, p.D, dtype, st);
    if (rc != SA2_OK) return rc;
    BwdSums sums = {};
    if (p.dq.p || p.dk2.p || p.dv2.p) {
        rc = launch_mfma_bwd_kp(p, dtype, st, &sums);
        if (rc != SA2_OK) return rc;
    }
    if (p.dk1.p || p.dv1.p) rc = launch_mfma_bwd_kv(p, dtype, st, &sums);
    if (rc != SA2_OK) return rc;
    return launch_bwd_sums(p, sums, mfma_width(p.D), dtype, st);
}

}  // namespace sa2
