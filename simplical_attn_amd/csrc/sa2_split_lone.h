// What the plane-split kernels with one wavefront per SIMD share: the order of plane products, and the vector work on a tile of weights.
#pragma once

#include "sa2_mfma_lone.h"
#include "sa2_split_common.h"

namespace sa2 {
namespace {

// plane products with a sum of planes up to two, the small ones first
template <int NA, int NB>
struct Products {
    int x[NA * NB] = {}, y[NA * NB] = {}, n = 0;
    constexpr Products() {
        for (int sum = 2; sum >= 0; --sum)
            for (int a = 0; a < NA; ++a)
                if (sum - a >= 0 && sum - a < NB) {
                    x[n] = a;
                    y[n] = sum - a;
                    ++n;
                }
    }
};

// The three planes of elements 8*KS + 2*t and the next one of a tile as word t of its half KS, in four steps of two or three
// instructions (I = 4*t + step); the elements are used up, `h` is kept from one step to the next.
template <int KS, int I>
__device__ __forceinline__ void split_word_step(floatx16& of, u4 (&to)[3], float (&h)[2]) {
    constexpr int t = I / 4, m = I % 4, e = 8 * KS + 2 * t;
    if constexpr (m == 0 || m == 2) {
        const uint32_t w = pack2(of[e], of[e + 1]);
        to[m / 2][t] = w;
        h[0] = bf16_lo(w);
        if constexpr (m == 2) h[1] = bf16_hi(w);
        stays(h[0]);
    } else if constexpr (m == 1) {
        float x = of[e] - h[0], y = of[e + 1] - bf16_hi(to[0][t]);
        stays(y);
        of[e] = x;
        of[e + 1] = y;
    } else {
        uint32_t w = pack2(of[e] - h[0], of[e + 1] - h[1]);
        stays(w);
        to[2][t] = w;
    }
}
// f for those of N items that fall to slot SLOT of the slots [FROM, TO)
template <int N, int SLOT, int FROM, int TO, class F>
__device__ __forceinline__ void within(F&& f) { deal<N, SLOT - FROM, TO - FROM>(f); }

}  // namespace
}  // namespace sa2
