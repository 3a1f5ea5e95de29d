// Generic fp32-FMA kernels: any element type (fp32 / bf16 / fp16 I/O), any
// D <= 256, any window.  All arithmetic is fp32 with accurate expf/logf, so
// this path carries the 1e-5 parity bar of the fp32 configuration and serves
// every shape the MFMA kernels do not take.  The rows themselves: sa2_fma_rows.h.
#include <type_traits>

#include "sa2_fma_rows.h"

namespace sa2 {
namespace {

constexpr int ROWS_PER_BLOCK = 4;   // wavefronts per workgroup, one owned row each
template <typename T>
__global__ __launch_bounds__(ROWS_PER_BLOCK * 64) void generic_fwd_kernel(Problem p, int nblk) {
    extern __shared__ float smem[];
    const int bh = blockIdx.x / nblk, blk = blockIdx.x - bh * nblk;
    fma_fwd_rows<T>(p, bh, blk * ROWS_PER_BLOCK, 0, p.w2, smem,
                    [&](int i, int lane, float m, float l, const float (&acc)[MAXC]) { fma_store_row<T>(p, bh, i, lane, m, l, acc); });
}
template <typename T>
__global__ __launch_bounds__(ROWS_PER_BLOCK * 64) void generic_bwd_dq_kernel(Problem p, int nblk) {
    extern __shared__ float smem[];
    const int bh = blockIdx.x / nblk, blk = blockIdx.x - bh * nblk;
    fma_dq_rows<T>(p, bh, blk * ROWS_PER_BLOCK, smem);
}
template <typename T>
__global__ __launch_bounds__(ROWS_PER_BLOCK * 64) void generic_bwd_owner_kernel(Problem p, OwnerArgs a, int nblk) {
    extern __shared__ float smem[];
    const int bh = blockIdx.x / nblk, blk = blockIdx.x - bh * nblk;
    fma_owner_rows<T>(p, a, bh, blk * ROWS_PER_BLOCK, smem);
}

// dsum[b,h,i] = sum_d dout*out, one wavefront per row.
template <typename T>
__global__ __launch_bounds__(256) void rowdot_kernel(Tensor out, Tensor dout, float* dsum, int N, int H, int D,
                                                     int64_t rows) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    const int i = (int)(row % N);
    const int bh = (int)(row / N);
    const int b = bh / H, h = bh - b * H;
    const T* op = (const T*)out.p + out.off(b, i, h);
    const T* gp = (const T*)dout.p + dout.off(b, i, h);
    float s = 0.f;
    for (int d = lane; d < D; d += 64) s = fmaf(to_float(op[d]), to_float(gp[d]), s);
    s = wave_sum(s);
    if (lane == 0) dsum[row] = s;
}

// The same for rows on a 16-byte grid: a lane takes the 16-byte chunk of a row (8 or 4 elements) in one load per tensor,
// the next power of two of the chunks of a row share it (at head_dim 96 in 16 bits: 12 of 16 lanes work).  Bound by
// reading both tensors: fp32 B4 N7559 H8 D64 (124 MB) 53 us with a wavefront per row, 27 us so.  A lane adds its products
// in pairs, which makes the sum as deep as the kernel above makes it, with the same error (a chain of the eight products
// of 16-bit rows: 6 % more at head_dim 96).
template <typename T>
__global__ __launch_bounds__(256) void rowdot_vec_kernel(Tensor out, Tensor dout, float* dsum, int N, int H, int D, int lpr_log2,
                                                         int64_t rows) {
    constexpr int PER = 16 / sizeof(T);
    const int lane = threadIdx.x & 63;
    const int lpr = 1 << lpr_log2;                        // lanes per row
    const int64_t row = (((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) << (6 - lpr_log2)) + (lane >> lpr_log2);
    const int sub = lane & (lpr - 1);
    float s = 0.f;
    if (row < rows && sub * PER < D) {
        const int i = (int)(row % N);
        const int bh = (int)(row / N);
        const int b = bh / H, h = bh - b * H;
        union { uint4 v; T e[PER]; } o, g;
        o.v = *(const uint4*)((const T*)out.p + out.off(b, i, h) + sub * PER);
        g.v = *(const uint4*)((const T*)dout.p + dout.off(b, i, h) + sub * PER);
        float x[PER / 2];
#pragma unroll
        for (int t = 0; t < PER / 2; ++t)
            x[t] = fmaf(to_float(o.e[t + PER / 2]), to_float(g.e[t + PER / 2]), to_float(o.e[t]) * to_float(g.e[t]));
#pragma unroll
        for (int half = PER / 4; half > 0; half >>= 1)
#pragma unroll
            for (int t = 0; t < half; ++t) x[t] += x[t + half];
        s = x[0];
    }
    for (int off = lpr >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (row < rows && sub == 0) dsum[row] = s;
}

template <typename F>
int dispatch_dtype(int dtype, F&& f) {
    switch (dtype) {
        case SA2_F32: return f((float*)nullptr);
        case SA2_BF16: return f((bf16_t*)nullptr);
        case SA2_F16: return f((f16_t*)nullptr);
    }
    return SA2_ERR_BAD_DTYPE;
}

int check_launch() { return hipGetLastError() == hipSuccess ? SA2_OK : SA2_ERR_LAUNCH_FAILED; }

template <typename K>
bool allow_big_lds(K kernel, size_t bytes) {
    return bytes <= 64 * 1024 || allow_full_lds((const void*)kernel);
}

}  // namespace

int launch_rowdot(const Tensor& out, const Tensor& dout, float* dsum, int B, int N, int H, int D, int dtype,
                  hipStream_t st) {
    const int64_t rows = (int64_t)B * H * N;
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    // rows on a 16-byte grid: the vector kernel
    const int per = dtype == SA2_F32 ? 4 : 8;
    auto aligned = [&](const Tensor& t) {
        return ((uintptr_t)t.p & 15u) == 0 && (B == 1 || t.sb % per == 0) && (N == 1 || t.sn % per == 0) && (H == 1 || t.sh % per == 0);
    };
    int lpr_log2 = 0;
    while ((per << lpr_log2) < D) ++lpr_log2;
    const bool vec = D % per == 0 && aligned(out) && aligned(dout);
    return dispatch_dtype(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (vec) {
            const int64_t per_block = (int64_t)4 << (6 - lpr_log2);           // rows per workgroup
            const int64_t vblocks = (rows + per_block - 1) / per_block;
            hipLaunchKernelGGL(rowdot_vec_kernel<T>, dim3((unsigned)vblocks), dim3(256), 0, st, out, dout, dsum, N, H, D, lpr_log2, rows);
        } else {
            hipLaunchKernelGGL(rowdot_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st, out, dout, dsum, N, H, D, rows);
        }
        return check_launch();
    });
}

int launch_generic_fwd(const Problem& p, int dtype, hipStream_t st) {
    const int nblk = (p.N + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    const int64_t blocks = (int64_t)nblk * p.B * p.H;
    if (blocks > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    const size_t lds = smem_bytes(p.D, ROWS_PER_BLOCK);
    return dispatch_dtype(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (!allow_big_lds(generic_fwd_kernel<T>, lds)) return (int)SA2_ERR_LAUNCH_FAILED;
        hipLaunchKernelGGL(generic_fwd_kernel<T>, dim3((unsigned)blocks), dim3(ROWS_PER_BLOCK * 64), lds, st, p, nblk);
        return check_launch();
    });
}

size_t generic_bwd_scratch_bytes(int, int, int, int, int, int) { return 0; }

int launch_generic_bwd(const Problem& p, int dtype, hipStream_t st) {
    const int nblk = (p.N + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    const int64_t blocks = (int64_t)nblk * p.B * p.H;
    if (blocks > 0x7fffffffLL) return SA2_ERR_TOO_LARGE;
    const size_t lds = smem_bytes(p.D, ROWS_PER_BLOCK);
    int rc = launch_rowdot(p.out, p.dout, p.dsum, p.B, p.N, p.H, p.D, dtype, st);
    if (rc != SA2_OK) return rc;
    return dispatch_dtype(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        const dim3 grid((unsigned)blocks), block(ROWS_PER_BLOCK * 64);
        if (p.dq.p) {
            if (!allow_big_lds(generic_bwd_dq_kernel<T>, lds)) return (int)SA2_ERR_LAUNCH_FAILED;
            hipLaunchKernelGGL(generic_bwd_dq_kernel<T>, grid, block, lds, st, p, nblk);
            if (check_launch() != SA2_OK) return (int)SA2_ERR_LAUNCH_FAILED;
        }
        if (!allow_big_lds(generic_bwd_owner_kernel<T>, lds)) return (int)SA2_ERR_LAUNCH_FAILED;
        if (p.dk1.p || p.dv1.p) {
            const OwnerArgs a = owner_k(p);
            hipLaunchKernelGGL(generic_bwd_owner_kernel<T>, grid, block, lds, st, p, a, nblk);
            if (check_launch() != SA2_OK) return (int)SA2_ERR_LAUNCH_FAILED;
        }
        if (p.dk2.p || p.dv2.p) {
            const OwnerArgs a = owner_k2(p);
            hipLaunchKernelGGL(generic_bwd_owner_kernel<T>, grid, block, lds, st, p, a, nblk);
            if (check_launch() != SA2_OK) return (int)SA2_ERR_LAUNCH_FAILED;
        }
        return (int)SA2_OK;
    });
}

}  // namespace sa2
