// What the plane-split kernels share (see sa2_split_mfma.hip): element types, columns, and values as sums of bf16 planes.
#pragma once

#include "sa2_mfma_common.h"

namespace sa2 {
namespace {

__device__ __forceinline__ floatx16 zero16() {
    floatx16 z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.f;
    return z;
}
constexpr float TINY = 7.888609052210118e-31f;     // 2^-100
typedef float fx4 __attribute__((ext_vector_type(4)));      // 16 bytes in flight (plain vectors: stay in registers)
typedef unsigned ux2 __attribute__((ext_vector_type(2)));

// The element type of the tensors: four columns as they lie in memory (Raw), their fp32 values, and fp32 values rounded
// to the type.  Everything between the loads and the stores is fp32.
struct MemF32 {
    typedef float T;
    typedef fx4 Raw;
    typedef float Fma;                             // the type's name in sa2_fma_rows.h
    static constexpr int DTYPE = SA2_F32;
    static constexpr int PLANES = 3;
    static __device__ __forceinline__ fx4 widen(Raw x) { return x; }
    static __device__ __forceinline__ void store(T* p, float a, float b, float c, float d) { *(float4*)p = make_float4(a, b, c, d); }
};
template <class E>
struct Mem16 {
    typedef uint16_t T;
    typedef ux2 Raw;
    typedef typename std::conditional<E::DTYPE == SA2_BF16, bf16_t, f16_t>::type Fma;
    static constexpr int DTYPE = E::DTYPE;
    static constexpr int PLANES = E::DTYPE == SA2_BF16 ? 1 : 2;      // bf16 planes that hold a value exactly
    static __device__ __forceinline__ fx4 widen(Raw x) { return fx4{E::lo(x[0]), E::hi(x[0]), E::lo(x[1]), E::hi(x[1])}; }
    static __device__ __forceinline__ void store(T* p, float a, float b, float c, float d) {
        *(uint2*)p = make_uint2(E::pack(a, b), E::pack(c, d));
    }
};

// MODE of a kernel: tensors as wide as the kernel, or narrower (PAD below); PADDED_FINE: with finer sums (Chain and
// accumulate) for the fp32 head dims that ran on the FMA kernels before (16, which was padded onto the fp32 MFMA, did not)
constexpr int EXACT = 0, PADDED = 1, PADDED_FINE = 2;

// Four columns of a row.  PAD: the tensors have width <= D columns; the kernel's columns from there on read as zeros
// and are not written (rows are multiples of four elements, so four columns are inside or outside together).
template <class T, bool PAD>
__device__ __forceinline__ typename T::Raw raw4(const typename T::T* row, int col, int width) {
    if constexpr (PAD) {
        if (col >= width) return (typename T::Raw)(0);
    }
    return *(const typename T::Raw*)(row + col);
}
template <class T, bool PAD>
__device__ __forceinline__ float4 cols4(const typename T::T* row, int col, int width) {
    const fx4 x = T::widen(raw4<T, PAD>(row, col, width));
    return make_float4(x[0], x[1], x[2], x[3]);
}

// ---- planes ----
__device__ __forceinline__ uint32_t pack2(float a, float b) {          // one v_cvt_pk_bf16_f32
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    union { bf16x2 v; uint32_t u; } r;
    r.v = __builtin_convertvector((f32x2{a, b}), bf16x2);
    return r.u;
}
// The first N planes of two values (packed pairs).  LIMIT: values above the largest bf16 (fp32's lowest values, which mask
// keys, among them) are split from there on; without it their first plane would be infinite.
template <int N, bool LIMIT = false>
__device__ __forceinline__ void split2(float a, float b, uint32_t (&o)[N]) {
    constexpr float MOST = 3.3895313892515355e38f;
    o[0] = LIMIT ? pack2(__builtin_amdgcn_fmed3f(a, -MOST, MOST), __builtin_amdgcn_fmed3f(b, -MOST, MOST)) : pack2(a, b);
#pragma unroll
    for (int n = 1; n < N; ++n) {
        a -= bf16_lo(o[n - 1]);
        b -= bf16_hi(o[n - 1]);
        o[n] = pack2(a, b);
    }
}
// Eight values (two groups of four) as an MFMA operand per plane
template <int N, bool LIMIT = false>
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&o)[N]) {
    union { uint32_t u[4]; bf16x8 v; } r[N];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        uint32_t w[N];
        split2<N, LIMIT>(x[2 * t], x[2 * t + 1], w);
#pragma unroll
        for (int n = 0; n < N; ++n) r[n].u[t] = w[n];
    }
#pragma unroll
    for (int n = 0; n < N; ++n) o[n] = r[n].v;
}
// Four columns to the planes of a tile (`dst`: plane 0; planes lie `plane` elements apart)
template <int N, bool LIMIT>
__device__ __forceinline__ void store_planes(const fx4& x, uint16_t* dst, int plane) {
    uint32_t a[N], b[N];
    split2<N, LIMIT>(x[0], x[1], a);
    split2<N, LIMIT>(x[2], x[3], b);
#pragma unroll
    for (int n = 0; n < N; ++n) *(uint2*)(dst + n * plane) = make_uint2(a[n], b[n]);
}
// LSE*log2(e) or D is taken off a finished chain by one more MFMA: an operand of its planes against ones (in the lanes of
// the first eight slots).  Subtracted last and exactly, it costs one rounding; a chain that starts from it rounds every
// step at its size, which doubled the error of the gradients.
__device__ __forceinline__ bf16x8 lead_planes(float x, float rest) {
    union { uint32_t u[4]; bf16x8 v; } r;
    uint32_t w[3];
    split2<3>(-x, -rest, w);
    r.u[0] = w[0]; r.u[1] = w[1]; r.u[2] = w[2]; r.u[3] = 0;
    return r.v;
}
__device__ __forceinline__ float lse_rest(float lse, float x) {        // what x = LSE*log2(e) lost when it was rounded
    constexpr float LOG2E_REST = 1.9259629911e-8f;       // log2(e) - LOG2E
    return fmaf(lse, LOG2E, -x) + lse * LOG2E_REST;
}
__device__ __forceinline__ bf16x8 lse_planes(float lse) { return lead_planes(lse * LOG2E, lse_rest(lse, lse * LOG2E)); }
__device__ __forceinline__ bf16x8 lead_ones(int hf) {
    uint32_t w = hf ? 0u : 0x3f803f80u;
    asm volatile("" : "+v"(w));                          // (made where it is used: four registers less to keep)
    union { uint32_t u[4]; bf16x8 v; } r;
    r.u[0] = r.u[1] = r.u[2] = r.u[3] = w;
    return r.v;
}
}  // namespace
}  // namespace sa2
