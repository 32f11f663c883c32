// What the chunked forms of the recurrences share: chunks of 16 tokens, and 16 x 16 products in double on the matrix cores.
#pragma once
#include "common.h"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int CT = 16;                                       // tokens of a chunk
constexpr int MLD = CT + 1;                                  // doubles a row of a 16 x 16 matrix takes in LDS (its columns then lie in different banks)

// First chunk slot of a sequence whose tokens start at row `lo`: sequences never overlap, and all fit num_tokens / 16 + batch slots.
__device__ __forceinline__ int chunk_base(int lo, int seq) { return lo / CT + seq; }

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    const u32x2 v = __builtin_bit_cast(u32x2, x);
    const u32x2 r = {(uint32_t)__builtin_amdgcn_mov_dpp((int)v[0], CTRL, 0xf, 0xf, true), (uint32_t)__builtin_amdgcn_mov_dpp((int)v[1], CTRL, 0xf, 0xf, true)};
    return __builtin_bit_cast(double, r);
}
// The sums of four values over the 16 lanes of a row; lane g is left with that of value g & 3.
__device__ __forceinline__ double row16_sum4(double v0, double v1, double v2, double v3, int g) {
    const bool odd = g & 1, high = g & 2;
    const double lo = (odd ? v1 : v0) + dpp_f64<0xB1>(odd ? v0 : v1), hi = (odd ? v3 : v2) + dpp_f64<0xB1>(odd ? v2 : v3);     // neighbours
    double x = (high ? hi : lo) + dpp_f64<0x4E>(high ? lo : hi);         // pairs
    x += dpp_f64<0x124>(x);                                              // rotations by 4 and 8 within the row
    return x + dpp_f64<0x128>(x);
}

// Lower triangular 16 x 16 matrices in double on the matrix cores.  Index i of an operand or of a result's column (lane & 15) stands for token
// chunk_tok(i): element e of a lane in quarter q of the wave is then token 4 q + e, in a result's rows as in the contraction's steps.  So a result is
// the next product's right operand as it stands, and its transpose's left operand; what is needed as a left operand is carried transposed too.
__device__ __forceinline__ int chunk_tok(int i) { return 4 * (i & 3) + (i >> 2); }

__device__ __forceinline__ f64x4 mfma_f64(const f64x4& l, const f64x4& r, f64x4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f64_16x16x4f64(l[e], r[e], c, 0, 0, 0);
    return c;
}
// c + l r where only l's tokens up to a result's own row (T: column) enter, and nothing above the diagonal: what is not finite in a token then
// leaves the tokens before it alone.  W: r's columns are channels and not tokens.
template <bool T, bool W>
__device__ __forceinline__ f64x4 mfma_f64_below(const f64x4& l, const f64x4& r, const f64x4& c, int q, int own) {
    f64x4 res = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int t = 0; t < CT; ++t) {
        f64x4 lm, rm;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = 4 * q + e <= t;
            lm[e] = in ? l[e] : 0.0;
            rm[e] = in ? r[e] : 0.0;
        }
        const f64x4 x = mfma_f64(lm, rm, c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (T ? own == t && (W || 4 * q + e <= t) : 4 * q + e == t && (W || own <= t)) res[e] = x[e];
    }
    return res;
}
}  // namespace
