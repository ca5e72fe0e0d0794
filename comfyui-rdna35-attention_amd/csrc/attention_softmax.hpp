// The online softmax of the attention kernels on 32-key half chunks: shared by
// attention.hip (padded head dims above 64) and attention_d64.hip.
//
// Scores are held transposed (a query is a lane column): s[nt][v] is the score
// of key 8(v/4) + 4half + v%4 of the half for query tile nt, column col.
#pragma once

#include "kernels.hpp"

namespace pisa {

constexpr float kLazyRescale = 8.0f;  // log2 headroom before the running max is moved

// Sum of the 8 elements of a packed operand, fp32 accumulation (v_dot2 with ones).
__device__ __forceinline__ float sum8(bf16x8 x, float acc) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(x, x, 0, 1), one, acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(x, x, 2, 3), one, acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(x, x, 4, 5), one, acc, false);
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(x, x, 6, 7), one, acc, false);
}
__device__ __forceinline__ float sum8(f16x8 x, float acc) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(x, x, 0, 1), one, acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(x, x, 2, 3), one, acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(x, x, 4, 5), one, acc, false);
    return __builtin_amdgcn_fdot2(__builtin_shufflevector(x, x, 6, 7), one, acc, false);
}

// The chunk loop works on 32-key half chunks.  One straight-line region per
// half h issues the 16 score MFMAs of half h+1 interleaved with the
// exponentials of half h, then the 16 PV MFMAs of half h interleaved with the
// operand loads of the next chunk and with the masking and column maxima of
// half h+1 (whose scores are ready by then); only the rare running-max move
// branches, after the region.  VALU, memory and MFMA work of the one wave on
// the SIMD thus overlap.

// Column maxima of half-chunk scores s[nt] (s[nt][v] = score of key
// 8(v/4) + 4half + v%4 of the half, query tile nt, column col) in log2 units
// (`c` converts the scores to them).  IEEE `maximum` (NaN-propagating) is
// v_maximum3_f32, two scores per instruction with no canonicalising of the
// MFMA results that fmaxf needs first (12 fewer VALU instructions per half
// chunk at NT = 2).  A NaN score makes its column's output NaN either way: its
// probability is NaN whatever the running max is.
// With two tiles, one swap of the lanes' partial maxima leaves lanes 0-31 with
// both halves' values of tile 0 and lanes 32-63 with those of tile 1; their
// maximum, swapped with itself, gives every lane both column maxima.
template <int NT>
__device__ __forceinline__ void half_max(const f32x16 (&s)[NT], float c, float (&mx)[NT]) {
    float x[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        x[nt] = s[nt][0];
#pragma unroll
        for (int v = 1; v < 16; ++v) x[nt] = __builtin_elementwise_maximum(x[nt], s[nt][v]);
    }
    if constexpr (NT == 2) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
        const float both = __builtin_elementwise_maximum(__uint_as_float(r[0]), __uint_as_float(r[1]));
        const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(both), __float_as_uint(both), false, false);
        mx[0] = __uint_as_float(b[0]) * c;
        mx[1] = __uint_as_float(b[1]) * c;
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const float2 p = pair_xor32(x[nt]);
            mx[nt] = __builtin_elementwise_maximum(p.x, p.y) * c;
        }
    }
}

// Running-max update from the column maxima mx of the next half.  The running
// max only moves when a column's max exceeds it by kLazyRescale, so the O
// rescale runs on the first half chunk and rarely after; probabilities stay
// below 2^kLazyRescale.  `enable` false (scores past the last chunk) leaves
// the state unchanged.  The running max m of a column is held as the two
// values the per-half code uses, both set only when m moves: nm = -m (0 while
// m = -inf: the exponent offset of the probabilities) and mth = m +
// kLazyRescale (the threshold, -inf while m = -inf).  -nm is m exactly, so
// every decision is the one m itself would give, and so is the factor
// 2^(m - mx) < 2^-kLazyRescale of a finite m; while m = -inf, l and O are
// still zero, and min(., 0) keeps the factor finite (no 0 * inf).
template <int NT, int MD>
__device__ __forceinline__ void rescale_to(const float (&mx)[NT], bool enable, float (&nm)[NT], float (&mth)[NT],
                                          float (&l)[NT], float (&lt)[NT], f32x16 (&o)[MD][NT]) {
    bool need[NT];
    bool any_need = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        need[nt] = enable && mx[nt] > mth[nt];
        any_need = any_need || need[nt];
    }
    if (__any(any_need)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const float alpha = need[nt] ? __builtin_amdgcn_exp2f(fminf(-nm[nt] - mx[nt], 0.0f)) : 1.0f;
            nm[nt] = need[nt] ? -mx[nt] : nm[nt];
            mth[nt] = need[nt] ? mx[nt] + kLazyRescale : mth[nt];
            l[nt] *= alpha;
            lt[nt] *= alpha;
#pragma unroll
            for (int md = 0; md < MD; ++md)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[md][nt][v] *= alpha;
        }
    }
}

// Probabilities of a half chunk as packed PV operands pf[nt][ss] (keys
// 16ss .. 16ss+15 of the half in swap23 order, which is the accumulator row
// order), and their masses: l (and lt for tail chunks) sum the rounded
// probabilities the PV product uses, so every output row's weights sum to 1.
// Exact chunks accumulate straight into l; tail chunks form the half's sum
// first, which goes to both l and lt.
template <typename T, int NT>
__device__ __forceinline__ void probs_half(const f32x16 (&s)[NT], float c, const float (&nm)[NT], float (&l)[NT],
                                           float (&lt)[NT], bool tail, typename Elem<T>::vec8 (&pf)[NT][2]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float neg_m = nm[nt];
        float rs = tail ? 0.0f : l[nt];
#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
            typename Elem<T>::vec8 p;
#pragma unroll
            for (int e = 0; e < 8; ++e) p[e] = from_f32<T>(__builtin_amdgcn_exp2f(fmaf(s[nt][ss * 8 + e], c, neg_m)));
            pf[nt][ss] = p;
            rs = sum8(p, rs);
        }
        l[nt] = tail ? l[nt] + rs : rs;
        lt[nt] = tail ? lt[nt] + rs : lt[nt];
    }
}

}  // namespace pisa
