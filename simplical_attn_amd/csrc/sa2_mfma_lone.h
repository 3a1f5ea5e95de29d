// Building blocks of the 16-bit kernels that place their MFMAs by hand, head_dim up to 128: one wavefront per SIMD with up to
// 512 registers (forward at head_dim 128, both backward kernels) or two with 256 each (forward at head_dim 64).
//
// A lone wavefront hides its latencies itself, so the order of instructions is fixed in the source (a sched_barrier behind
// every MFMA).  What costs what was measured on the instructions alone: an MFMA takes 33 cycles, under which four more vector
// instructions are free (with six it takes 45, with eight 48); a read of LDS takes 4 to 7 of its own right behind an MFMA and 14 behind vector instructions; an
// s_nop up to 9, which is why no instruction there reads the result of an exponential or the operand of an MFMA just written.
//
// The MFMAs are opaque to the compiler, which neither guards nor schedules them: listing_check.py looks over what it makes
// around them whenever they are built.
#pragma once

#include <type_traits>

#include "sa2_mfma_common.h"

namespace sa2 {
namespace {

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}
#define LONE_C(n) std::integral_constant<int, (n)>{}
// f for those of N items that fall to slot SLOT of SLOTS
template <int N, int SLOT, int SLOTS, class F>
__device__ __forceinline__ void deal(F&& f) {
    constexpr int a = SLOT < 0 ? 0 : SLOT < SLOTS ? SLOT : SLOTS, z = SLOT + 1 < 0 ? 0 : SLOT + 1 < SLOTS ? SLOT + 1 : SLOTS;
    constexpr int lo = N * a / SLOTS, hi = N * z / SLOTS;
    static_for<hi - lo>([&](auto Y) __attribute__((always_inline)) { f(std::integral_constant<int, lo + decltype(Y)::value>{}); });
}

template <class E>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    union { typename E::x2 h; uint32_t u; } v;
    v.h = __builtin_convertvector((f2){a, b}, typename E::x2);
    return v.u;
}
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef const u4 __attribute__((address_space(3)))* lds_u4;

// Accumulation registers 0 .. OWNED-1 (96, 192 or 256) belong to the kernel, not to the compiler: the sums that live through a
// sweep and the resident operands are named by number in the instructions below, and each of these says that it destroys
// them all, so that nothing else is ever kept there.  (Left to the compiler, beside 300 other registers of the sweep, sums and
// operands move between the two files or to scratch memory in every step.)
#define LONE_REGS_96 \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
    "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
    "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
    "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
    "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
    "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95"
#define LONE_REGS LONE_REGS_96, \
    "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
    "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", \
    "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
    "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
    "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
    "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191"
#define LONE_REGS_ALL LONE_REGS, \
    "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
    "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", \
    "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
    "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
template <int OWNED>
struct Lone {
#define LONE_MFMA(text, out, ...) \
    if constexpr (std::is_same<X8, bf16x8>::value) { \
        if constexpr (OWNED == 256) asm volatile("v_mfma_f32_32x32x16_bf16 " text : out : __VA_ARGS__ : LONE_REGS_ALL); \
        else if constexpr (OWNED == 96) asm volatile("v_mfma_f32_32x32x16_bf16 " text : out : __VA_ARGS__ : LONE_REGS_96); \
        else asm volatile("v_mfma_f32_32x32x16_bf16 " text : out : __VA_ARGS__ : LONE_REGS); \
    } else { \
        if constexpr (OWNED == 256) asm volatile("v_mfma_f32_32x32x16_f16 " text : out : __VA_ARGS__ : LONE_REGS_ALL); \
        else if constexpr (OWNED == 96) asm volatile("v_mfma_f32_32x32x16_f16 " text : out : __VA_ARGS__ : LONE_REGS_96); \
        else asm volatile("v_mfma_f32_32x32x16_f16 " text : out : __VA_ARGS__ : LONE_REGS); \
    }
    // d = a * operand B + c, d += a * operand B: tiles in vector registers, whose first reader comes at least two MFMAs later
    template <int B, class X8>
    static __device__ __forceinline__ void tile_start(floatx16& d, const X8& a, const floatx16& c) {
        LONE_MFMA("%0, %1, a[%3:%4], %2", "=&v"(d), "v"(a), "v"(c), "n"(B), "n"(B + 3))
    }
    template <int B, class X8>
    static __device__ __forceinline__ void tile_start(floatx16& d, const X8& a) {            // (c = 0)
        LONE_MFMA("%0, %1, a[%2:%3], 0", "=&v"(d), "v"(a), "n"(B), "n"(B + 3))
    }
    template <int B, class X8>
    static __device__ __forceinline__ void tile_more(floatx16& d, const X8& a) {
        LONE_MFMA("%0, %1, a[%2:%3], %0", "+v"(d), "v"(a), "n"(B), "n"(B + 3))
    }
    // sum S += a * b
    template <int S, class X8>
    static __device__ __forceinline__ void sum_more(const X8& a, const X8& b) {
        LONE_MFMA("a[%2:%3], %0, %1, a[%2:%3]", , "v"(a), "v"(b), "n"(S), "n"(S + 15))
    }
    // sum S = 0 (z: an operand of zeros)
    template <int S, class X8>
    static __device__ __forceinline__ void sum_zero(const X8& z) {
        LONE_MFMA("a[%1:%2], %0, %0, 0", , "v"(z), "n"(S), "n"(S + 15))
    }
#undef LONE_MFMA
    // (a value that is read between two of these instructions only could still be given one of the registers)
    static __device__ __forceinline__ void keep_out() {
        if constexpr (OWNED == 256) asm volatile("" ::: LONE_REGS_ALL);
        else if constexpr (OWNED == 96) asm volatile("" ::: LONE_REGS_96);
        else asm volatile("" ::: LONE_REGS);
    }
    // registers R .. R+3, R a multiple of four (one by one the compiler would put a wait between them)
    template <int R>
    static __device__ __forceinline__ void set_regs(uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3) {
#define LONE_SET "v_accvgpr_write_b32 a[%4:%4], %0\n\tv_accvgpr_write_b32 a[%5:%5], %1\n\tv_accvgpr_write_b32 a[%6:%6], %2\n\tv_accvgpr_write_b32 a[%7:%7], %3"
        if constexpr (OWNED == 256) asm volatile(LONE_SET ::"v"(x0), "v"(x1), "v"(x2), "v"(x3), "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS_ALL);
        else if constexpr (OWNED == 96) asm volatile(LONE_SET ::"v"(x0), "v"(x1), "v"(x2), "v"(x3), "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS_96);
        else asm volatile(LONE_SET ::"v"(x0), "v"(x1), "v"(x2), "v"(x3), "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS);
#undef LONE_SET
    }
    template <int R>
    static __device__ __forceinline__ float4 get_regs() {
        float4 x;
#define LONE_GET "v_accvgpr_read_b32 %0, a[%4:%4]\n\tv_accvgpr_read_b32 %1, a[%5:%5]\n\tv_accvgpr_read_b32 %2, a[%6:%6]\n\tv_accvgpr_read_b32 %3, a[%7:%7]"
        if constexpr (OWNED == 256) asm volatile(LONE_GET : "=v"(x.x), "=v"(x.y), "=v"(x.z), "=v"(x.w) : "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS_ALL);
        else if constexpr (OWNED == 96) asm volatile(LONE_GET : "=v"(x.x), "=v"(x.y), "=v"(x.z), "=v"(x.w) : "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS_96);
        else asm volatile(LONE_GET : "=v"(x.x), "=v"(x.y), "=v"(x.z), "=v"(x.w) : "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3) : LONE_REGS);
#undef LONE_GET
        return x;
    }
    // registers R .. R+3 from global memory (a vector-memory operation that the compiler does not count)
    template <int R>
    static __device__ __forceinline__ void load_regs(const void* src) {
        if constexpr (OWNED == 256) asm volatile("global_load_dwordx4 a[%1:%2], %0, off" ::"v"(src), "n"(R), "n"(R + 3) : "memory", LONE_REGS_ALL);
        else if constexpr (OWNED == 96) asm volatile("global_load_dwordx4 a[%1:%2], %0, off" ::"v"(src), "n"(R), "n"(R + 3) : "memory", LONE_REGS_96);
        else asm volatile("global_load_dwordx4 a[%1:%2], %0, off" ::"v"(src), "n"(R), "n"(R + 3) : "memory", LONE_REGS);
    }
};

// what the vector ALU has made of x by here is not put off behind a branch
template <class T>
__device__ __forceinline__ void stays(T& x) { asm volatile("" : "+v"(x)); }
// the MFMAs that write the two tiles have ended
__device__ __forceinline__ void finished(floatx16& a, floatx16& b) { asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a), "+v"(b)); }

// 16 bytes per lane from global memory straight to LDS, lane L to `to` + 16 * L.  Opaque: the compiler would wait for it
// before every read of LDS.
__device__ __forceinline__ void lds_request(const void* src, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(src) : "memory");
}
// the same from a base that all lanes share and a byte offset of the lane's own
__device__ __forceinline__ void lds_request(const void* base, uint32_t off, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(off), "s"(base) : "memory");
}

}  // namespace
}  // namespace sa2
