// Row-wise operators around an fp32 residual stream, for designs whose residual sum, norms and softcap must stay in
// 32-bit while projections run in the activation type A (bf16, or fp32 for a model served in full precision):
//   embedding rows -> fp32 stream (+ a copy in A), Dynamic-Tanh norm fused with the residual add that precedes it,
//   tanh-GELU gate, [stream | first embedding] concatenation for a looped stack, row gather, logit softcap.
// Every kernel is one workgroup per row (or a flat element grid) with 16-byte accesses where the row allows.
#include "common.h"
#include <algorithm>
#include <type_traits>
#include "gemm_any.h"

namespace {

template <typename A>
__device__ __forceinline__ float ldf(const A* p, int64_t i) {
    return (float)p[i];
}

struct DytNorm {            // tanh(alpha * x) * w + b; all three in the activation type
    const void* alpha;
    const void* w;
    const void* b;
};

// tanh for the norm: the library's where everything is fp32; for bf16 results 1 - 2 / (e^2z + 1) on the hardware's 2^x and
// reciprocal (about 1e-6 absolute; the result is rounded to 8 bits of mantissa).
template <typename A>
__device__ __forceinline__ float dyt_tanh(float z) {
    if constexpr (sizeof(A) == 4) {
        return tanhf(z);
    } else {
        const float e = __builtin_amdgcn_exp2f(fminf(z, 20.f) * 2.8853900817779268f);        // e^(2z)
        return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
    }
}

// x[row] = (accumulate ? x[row] : 0) + post(y[row]) + bias;  h[row] = next(x[row]).
// y null: the stream is only normalised.  post / next with a null weight are skipped (next: no h written).
// VEC: dim % 4 == 0 and every row 16-byte (A: 8-byte) aligned: four consecutive elements per lane, one access each.
template <typename A, bool VEC>
__global__ __launch_bounds__(256) void residual_dyt_kernel(const A* __restrict__ y, int64_t y_stride, DytNorm post, const A* __restrict__ bias,
                                                           float* __restrict__ x, int accumulate, DytNorm next, A* __restrict__ h,
                                                           int64_t h_stride, int dim) {
    typedef A A4 __attribute__((ext_vector_type(4)));
    const int64_t row = blockIdx.x;
    const float pa = post.w ? ldf((const A*)post.alpha, 0) : 0.f;
    const float na = next.w ? ldf((const A*)next.alpha, 0) : 0.f;
    float* xr = x + row * dim;
    constexpr int W = VEC ? 4 : 1;
    for (int c = threadIdx.x * W; c < dim; c += 256 * W) {
        float s[W], t[W], bv[W], pw[W], pb[W], nw[W], nb[W];
        if constexpr (VEC) {
            const f32x4 xv = accumulate ? *reinterpret_cast<const f32x4*>(xr + c) : f32x4{0.f, 0.f, 0.f, 0.f};
            const A4 zero = {(A)0.f, (A)0.f, (A)0.f, (A)0.f};
            const A4 yv = y ? *reinterpret_cast<const A4*>(y + row * y_stride + c) : zero;
            const A4 b4 = bias ? *reinterpret_cast<const A4*>(bias + c) : zero;
            const A4 pw4 = post.w ? *reinterpret_cast<const A4*>((const A*)post.w + c) : zero, pb4 = post.w ? *reinterpret_cast<const A4*>((const A*)post.b + c) : zero;
            const A4 nw4 = next.w ? *reinterpret_cast<const A4*>((const A*)next.w + c) : zero, nb4 = next.w ? *reinterpret_cast<const A4*>((const A*)next.b + c) : zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[e] = xv[e];
                t[e] = (float)yv[e];
                bv[e] = (float)b4[e];
                pw[e] = (float)pw4[e];
                pb[e] = (float)pb4[e];
                nw[e] = (float)nw4[e];
                nb[e] = (float)nb4[e];
            }
        } else {
            s[0] = accumulate ? xr[c] : 0.f;
            t[0] = y ? ldf(y, row * y_stride + c) : 0.f;
            bv[0] = bias ? ldf(bias, c) : 0.f;
            pw[0] = post.w ? ldf((const A*)post.w, c) : 0.f;
            pb[0] = post.w ? ldf((const A*)post.b, c) : 0.f;
            nw[0] = next.w ? ldf((const A*)next.w, c) : 0.f;
            nb[0] = next.w ? ldf((const A*)next.b, c) : 0.f;
        }
        float hv[W];
#pragma unroll
        for (int e = 0; e < W; ++e) {
            if (y) s[e] += post.w ? dyt_tanh<A>(pa * t[e]) * pw[e] + pb[e] : t[e];
            s[e] += bv[e];
            hv[e] = next.w ? dyt_tanh<A>(na * s[e]) * nw[e] + nb[e] : 0.f;
        }
        if constexpr (VEC) {
            if (y || bias) *reinterpret_cast<f32x4*>(xr + c) = f32x4{s[0], s[1], s[2], s[3]};
            if (next.w) *reinterpret_cast<A4*>(h + row * h_stride + c) = A4{(A)hv[0], (A)hv[1], (A)hv[2], (A)hv[3]};
        } else {
            if (y || bias) xr[c] = s[0];
            if (next.w) h[row * h_stride + c] = (A)hv[0];
        }
    }
}

template <typename A>
__global__ __launch_bounds__(256) void embedding_stream_kernel(const int64_t* __restrict__ ids, const A* __restrict__ table, float* __restrict__ x,
                                                               A* __restrict__ x0, int64_t x0_stride, int dim, int64_t vocab) {
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row];
    const bool ok = id >= 0 && id < vocab;
    for (int c = threadIdx.x; c < dim; c += 256) {
        const A v = ok ? table[id * dim + c] : (A)0.f;
        x[row * dim + c] = (float)v;
        if (x0) x0[row * x0_stride + c] = v;
    }
}

// out[row, :dim] = A(x[row]); the second half of the row (the first embedding) is already there.
template <typename A>
__global__ __launch_bounds__(256) void stream_cast_kernel(const float* __restrict__ x, A* __restrict__ out, int64_t out_stride, int dim) {
    const int64_t row = blockIdx.x;
    for (int c = threadIdx.x; c < dim; c += 256) out[row * out_stride + c] = (A)x[row * dim + c];
}

__global__ __launch_bounds__(256) void gather_rows_f32_kernel(const float* __restrict__ x, const int32_t* __restrict__ index, float* __restrict__ out, int dim) {
    const int64_t row = blockIdx.x;
    const int64_t src = index[row];
    for (int c = threadIdx.x; c < dim; c += 256) out[row * dim + c] = x[src * dim + c];
}

// out = cap tanh(z scale / cap), or z scale without a cap.  E: elements a lane, 8 where rows and strides allow 16-byte accesses.
// us, 256 x 32768 with a cap: 19.5 and 13.5 (67 MB), 64 x 32768 6.2 and 5.3.
template <typename A, int E>
__global__ __launch_bounds__(256) void logits_scale_kernel(const A* __restrict__ z, int64_t z_stride, float* __restrict__ out, int64_t rows, int vocab, float scale,
                                                           float cap) {
    int64_t row;
    int c;
    if (!nvh_piece<E>(rows, vocab, row, c)) return;
    float v[E];
    nvh_load_piece<A, E>(z + row * z_stride + c, v);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const float x = v[e] * scale;
        v[e] = cap > 0.f ? cap * tanhf(x / cap) : x;
    }
    nvh_store_piece<float, E>(out + row * vocab + c, v);
}
static void launch_logits_scale(const void* z, int64_t z_stride, float* out, int64_t rows, int64_t vocab, float scale, float cap, bool act_f32, hipStream_t st) {
    const bool vec = rows * vocab >= NVH_PIECES && vocab % 8 == 0 && z_stride % 8 == 0 && nvh_aligned16(z) && nvh_aligned16(out);
    const dim3 grid((unsigned)nvh_cdiv(rows * vocab, vec ? 2048 : 256));
    auto launch = [&](auto kernel, auto type) { kernel<<<grid, 256, 0, st>>>((const decltype(type)*)z, z_stride, out, rows, (int)vocab, scale, cap); };
    if (act_f32) launch(vec ? &logits_scale_kernel<float, 8> : &logits_scale_kernel<float, 1>, 0.f);
    else launch(vec ? &logits_scale_kernel<bf16, 8> : &logits_scale_kernel<bf16, 1>, (bf16)0.f);
}

// x[row] = table[id] * scale + pos_table[position] (fp32); ids or positions outside their tables give zeros for that term.
template <typename A>
__global__ __launch_bounds__(256) void embedding_pos_stream_kernel(const int64_t* __restrict__ ids, const int64_t* __restrict__ positions,
                                                                   const A* __restrict__ table, const A* __restrict__ pos_table, float scale,
                                                                   float* __restrict__ x, int dim, int64_t vocab, int64_t max_pos) {
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row], p = pos_table ? positions[row] : -1;
    const bool ok = id >= 0 && id < vocab, pok = p >= 0 && p < max_pos;
    for (int c = threadIdx.x; c < dim; c += 256) {
        const float e = ok ? (float)table[id * dim + c] * scale : 0.f;
        x[row * dim + c] = e + (pok ? (float)pos_table[p * dim + c] : 0.f);
    }
}

__device__ __forceinline__ float block_sum4(float v, float* scratch) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    return scratch[0] + scratch[1] + scratch[2] + scratch[3];
}

// The close of a layer whose sublayers all read one norm of the stream, and the norm that opens the next layer, per row:
//   s = branch_scale * (unit(a) wa + unit(b) wb) + c + c32;   x <- x + s;   h <- norm(x)
// unit(v) = v / sqrt(mean(v^2) + branch_eps) where the branch has a weight (wa / wb), v itself where it has none; absent
// terms are skipped.  norm: 1 = layer norm ((x - mean) / sqrt(var + eps) w + b, var the mean squared deviation),
// 2 = RMS norm (x rsqrt(mean of squares + eps) w), 0 = none (no h).  Everything is fp32; the row sits in LDS meanwhile.
struct CloseArgs {
    const void *a, *wa, *b, *wb, *c;
    const float* c32;
    int64_t a_stride, b_stride, c_stride, c32_stride;
    float branch_scale, branch_eps;
    float* x;
    int norm;
    const void *nw, *nb;
    float eps;
    void* h;
    int64_t h_stride;
    int dim;
};

template <typename A>
__device__ __forceinline__ f32x4 load4(const A* p) {
    if constexpr (sizeof(A) == 4) {
        return *reinterpret_cast<const f32x4*>(p);
    } else {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
        return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    }
}
template <typename A>
__device__ __forceinline__ void store4(A* p, const f32x4& v) {
    if constexpr (sizeof(A) == 4) *reinterpret_cast<f32x4*>(p) = v;
    else *reinterpret_cast<bf16x4*>(p) = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
}

// A mixture of experts' result as terms of a close: sum over a token's `top` choices, in choice order, of weight * y[position] (positions < 0 are
// skipped, null weights are 1), plus the shared expert's row, times sigmoid of the token's gate logit where there is one - what nvh_moe_combine writes.
struct MoeTerms {
    const void* y;             // rows of the chosen experts by position (null: no such terms)
    int64_t ldy;
    const int32_t* pos;        // [T, top]
    const float* weights;      // [T, top] or null
    int top;
    const void* shared;        // [T, ld] or null
    int64_t shared_stride;
    const float* gate;
    int64_t gate_stride;
};
// ... of row t at N consecutive columns from c on: the positions and rows of four choices are on their way together.
template <typename A, int N>
__device__ __forceinline__ void moe_sum(const MoeTerms& m, int64_t t, int c, float (&s)[N]) {
    auto load = [](const A* p, float (&v)[N]) {
        if constexpr (N == 4) {
            const f32x4 x = load4(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = x[e];
        } else {
            v[0] = (float)p[0];
        }
    };
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = 0.f;
    const float sg = m.gate ? 1.0f / (1.0f + expf(-m.gate[t * m.gate_stride])) : 1.0f;
    float sh[N];
    if (m.shared) load((const A*)m.shared + t * m.shared_stride + c, sh);
    for (int r0 = 0; r0 < m.top; r0 += 4) {
        int pos[4];
        float w[4], v[4][N];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t at = t * m.top + min(r0 + u, m.top - 1);
            pos[u] = m.pos[at];
            w[u] = m.weights ? m.weights[at] : 1.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) load((const A*)m.y + (int64_t)max(pos[u], 0) * m.ldy + c, v[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (r0 + u < m.top && pos[u] >= 0)
#pragma unroll
                for (int e = 0; e < N; ++e) s[e] = __builtin_fmaf(w[u], v[u][e], s[e]);
    }
    if (m.shared)
#pragma unroll
        for (int e = 0; e < N; ++e) s[e] += sg * sh[e];
}

// The closes with four columns a lane and access: the row stays in registers, and everything is on its way before the first sum needs it.  A row is
// a chain of a load, one or two sums across the workgroup and a store, whose latencies are the launch at any number of rows that a step brings
// (column by column through LDS every pass over the row waits for its own loads).  R: pieces of 1024 columns.  MOE: with a mixture's terms.
// us for 64 rows of 1024, column by column and this: residual norm with two terms 9.1 and 4.4; a mixture's launch and a close after it 7.8 + 5.0 and 4.5.
// FORM: what a call can have; terms that it has not cost registers and branches all the same.  us, bf16, one form for everything and so: one branch, 64 x 1024
// 3.4 and 2.9, 64 x 4096 6.0 and 4.3, 1000 x 5120 35.9 and 14.8; the norm alone, fp32, 1000 x 5120 30.0 and 11.6 (with five pieces instead of eight, and the
// norm's weights requested when the sums have begun: they come from L2, and what long rows need is more rows a CU).  THREADS: rows of at most 256 columns are
// one wave's, without a barrier (4000 x 64, two branches 10.6 and 5.3).  None of it changes a sum.
enum CloseForm { CLOSE_ANY, CLOSE_ONE, CLOSE_BRANCH, CLOSE_SUMS };        // everything; no second branch; a branch alone, no mean and no bias; no branch
template <typename A, int R, bool MOE, int FORM, int THREADS>
__global__ __launch_bounds__(THREADS) void residual_norm_vec_kernel(CloseArgs p, MoeTerms m) {
    constexpr bool HAS_A = FORM != CLOSE_SUMS, HAS_B = FORM == CLOSE_ANY, HAS_C = FORM != CLOSE_BRANCH, CENTRED = FORM != CLOSE_BRANCH;
    static_assert(!MOE || HAS_C, "a mixture's sum is a term");
    constexpr bool LATE = R > 4 && FORM != CLOSE_BRANCH;      // the norm's weights after the first sums
    __shared__ float red[16];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    const bool has_a = FORM == CLOSE_BRANCH || (HAS_A && p.a);
    const A* a = (const A*)p.a + (HAS_A ? row * p.a_stride : 0);
    const A* b = HAS_B && p.b ? (const A*)p.b + row * p.b_stride : nullptr;
    const A* c = HAS_C && p.c ? (const A*)p.c + row * p.c_stride : nullptr;
    const float* c32 = HAS_C && p.c32 ? p.c32 + row * p.c32_stride : nullptr;
    const A *pa = HAS_A ? (const A*)p.wa : nullptr, *pb = HAS_B ? (const A*)p.wb : nullptr, *bias = CENTRED && p.norm ? (const A*)p.nb : nullptr;
    float* xr = p.x + row * dim;
    auto sum = [](float v, float* at) { return THREADS == 64 ? wave_sum(v) : block_sum4(v, at); };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 va[R], vb[R], x[R], wa[R], wb[R], vc[R], vc32[R], nw[R], nb[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + THREADS * j) * 4;
        va[j] = vb[j] = x[j] = wa[j] = wb[j] = vc[j] = vc32[j] = nw[j] = nb[j] = zero;
        if (col < dim) {
            if (has_a) va[j] = load4(a + col);
            if (b) vb[j] = load4(b + col);
            if (c) vc[j] = load4(c + col);
            if (c32) vc32[j] = load4(c32 + col);
            x[j] = load4(xr + col);
            if (pa) wa[j] = load4(pa + col);
            if (pb) wb[j] = load4(pb + col);
            if (!LATE && p.norm) nw[j] = load4((const A*)p.nw + col);
            if (!LATE && bias) nb[j] = load4(bias + col);
            if constexpr (MOE) {
                float s[4];
                moe_sum<A, 4>(m, row, col, s);
                vc32[j] = f32x4{s[0], s[1], s[2], s[3]};
            }
        }
    }
    float ia = 1.f, ib = 1.f, sa = 0.f, sb = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sa += va[j][e] * va[j][e];
            if (HAS_B) sb += vb[j][e] * vb[j][e];
        }
    if (pa) ia = 1.0f / sqrtf(sum(sa, red) / (float)dim + p.branch_eps);
    if (pb) ib = 1.0f / sqrtf(sum(sb, red + 4) / (float)dim + p.branch_eps);
    float total = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + THREADS * j) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = 0.f;
            if (has_a) s += pa ? va[j][e] * ia * wa[j][e] : va[j][e];
            if (b) s += pb ? vb[j][e] * ib * wb[j][e] : vb[j][e];
            if (HAS_A) s *= p.branch_scale;
            if (c) s += vc[j][e];
            if (MOE || c32) s += vc32[j][e];
            x[j][e] += s;
            if (CENTRED) total += x[j][e];
        }
        if (col < dim && (MOE || has_a || b || c || c32)) *reinterpret_cast<f32x4*>(xr + col) = x[j];
    }
    if (p.norm == 0) return;
    if constexpr (LATE) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int col = (threadIdx.x + THREADS * j) * 4;
            if (col < dim) {
                nw[j] = load4((const A*)p.nw + col);
                if (bias) nb[j] = load4(bias + col);
            }
        }
    }
    const float mean = CENTRED && p.norm == 1 ? sum(total, red + 8) / (float)dim : 0.f;
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const bool in = (threadIdx.x + THREADS * j) * 4 < dim;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (CENTRED) x[j][e] = in ? x[j][e] - mean : 0.f;        // (columns past the end are 0 as they are)
            sq += x[j][e] * x[j][e];
        }
    }
    const float inv = 1.0f / sqrtf(sum(sq, red + 12) / (float)dim + p.eps);
    A* h = (A*)p.h + row * p.h_stride;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + THREADS * j) * 4;
        if (col < dim) store4(h + col, bias ? x[j] * inv * nw[j] + nb[j] : x[j] * inv * nw[j]);
    }
}

// R for rows of `dim` columns, or 0 where the vector form does not serve them.
static int close_pieces(int dim) { return dim % 4 || dim > 8192 ? 0 : dim <= 1024 ? 1 : dim <= 2048 ? 2 : dim <= 4096 ? 4 : 8; }
template <typename A>
static bool rows_of_fours(const void* p, int64_t stride) {   // (absent rows do)
    return !p || (stride % 4 == 0 && ((uintptr_t)p % (4 * sizeof(A))) == 0);
}
template <typename A>
static bool moe_of_fours(const MoeTerms& m) {
    return rows_of_fours<A>(m.y, m.ldy) && rows_of_fours<A>(m.shared, m.shared_stride);
}
#define NVH_CLOSE_CASES(KERNEL, ...)                                                             \
    switch (pieces * (m.y ? -1 : 1)) {                                                           \
        case 1: KERNEL<A, 1, false><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case 2: KERNEL<A, 2, false><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case 4: KERNEL<A, 4, false><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case 8: KERNEL<A, 8, false><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case -1: KERNEL<A, 1, true><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case -2: KERNEL<A, 2, true><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        case -4: KERNEL<A, 4, true><<<grid, 256, 0, st>>>(__VA_ARGS__); break;                   \
        default: KERNEL<A, 8, true><<<grid, 256, 0, st>>>(__VA_ARGS__);                          \
    }

template <typename A>
static bool launch_residual_norm_vec(const CloseArgs& p, const MoeTerms& m, int64_t rows, hipStream_t st) {
    const int pieces = close_pieces(p.dim);
    if (!pieces || !rows_of_fours<A>(p.a, p.a_stride) || !rows_of_fours<A>(p.b, p.b_stride) || !rows_of_fours<A>(p.c, p.c_stride) ||
        !rows_of_fours<float>(p.c32, p.c32_stride) || !rows_of_fours<A>(p.wa, 0) || !rows_of_fours<A>(p.wb, 0) || !rows_of_fours<A>(p.nw, 0) ||
        !rows_of_fours<A>(p.nb, 0) || (p.norm && !rows_of_fours<A>(p.h, p.h_stride)) || !nvh_aligned16(p.x) || !moe_of_fours<A>(m))
        return false;
    const dim3 grid((unsigned)rows);
    const bool branch = p.a && !p.b && !p.c && !p.c32 && !m.y && p.norm != 1 && !p.nb;
    auto launch = [&](auto r, auto threads) {
        constexpr int R = decltype(r)::value, T = decltype(threads)::value;
        auto form = [&](auto f, auto moe) { residual_norm_vec_kernel<A, R, decltype(moe)::value, decltype(f)::value, T><<<grid, T, 0, st>>>(p, m); };
        const std::true_type with{};
        const std::false_type without{};
        if (branch) return form(std::integral_constant<int, CLOSE_BRANCH>{}, without);
        if (!p.a && !p.b) return m.y ? form(std::integral_constant<int, CLOSE_SUMS>{}, with) : form(std::integral_constant<int, CLOSE_SUMS>{}, without);
        if (!p.b) return m.y ? form(std::integral_constant<int, CLOSE_ONE>{}, with) : form(std::integral_constant<int, CLOSE_ONE>{}, without);
        return m.y ? form(std::integral_constant<int, CLOSE_ANY>{}, with) : form(std::integral_constant<int, CLOSE_ANY>{}, without);
    };
    const std::integral_constant<int, 256> four_waves{};
    if (p.dim <= 256) launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 64>{});
    else if (pieces == 1) launch(std::integral_constant<int, 1>{}, four_waves);
    else if (pieces == 2) launch(std::integral_constant<int, 2>{}, four_waves);
    else if (pieces == 4) launch(std::integral_constant<int, 4>{}, four_waves);
    else if (p.dim <= 5120 && !branch) launch(std::integral_constant<int, 5>{}, four_waves);
    else if (p.dim <= 6144 && !branch) launch(std::integral_constant<int, 6>{}, four_waves);
    else launch(std::integral_constant<int, 8>{}, four_waves);
    return true;
}

template <typename A, bool MOE>
__global__ __launch_bounds__(256) void residual_norm_kernel(CloseArgs p, MoeTerms m) {
    extern __shared__ float rowbuf[];
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    const A* a = p.a ? (const A*)p.a + row * p.a_stride : nullptr;
    const A* b = p.b ? (const A*)p.b + row * p.b_stride : nullptr;
    const A* c = p.c ? (const A*)p.c + row * p.c_stride : nullptr;
    const float* c32 = p.c32 ? p.c32 + row * p.c32_stride : nullptr;
    float ia = 1.f, ib = 1.f;
    if (a && p.wa) {
        float s = 0.f;
        for (int i = threadIdx.x; i < dim; i += 256) {
            const float v = (float)a[i];
            s += v * v;
        }
        ia = 1.0f / sqrtf(block_sum4(s, red) / (float)dim + p.branch_eps);
    }
    if (b && p.wb) {
        float s = 0.f;
        for (int i = threadIdx.x; i < dim; i += 256) {
            const float v = (float)b[i];
            s += v * v;
        }
        ib = 1.0f / sqrtf(block_sum4(s, red) / (float)dim + p.branch_eps);
    }
    float* xr = p.x + row * dim;
    float sum = 0.f;
    for (int i = threadIdx.x; i < dim; i += 256) {
        float s = 0.f;
        if (a) s += p.wa ? (float)a[i] * ia * (float)((const A*)p.wa)[i] : (float)a[i];
        if (b) s += p.wb ? (float)b[i] * ib * (float)((const A*)p.wb)[i] : (float)b[i];
        s *= p.branch_scale;
        if (c) s += (float)c[i];
        if (c32) s += c32[i];
        if constexpr (MOE) {
            float e[1];
            moe_sum<A, 1>(m, row, i, e);
            s += e[0];
        }
        const float v = xr[i] + s;
        if (MOE || a || b || c || c32) xr[i] = v;
        rowbuf[i] = v;
        sum += v;
    }
    if (p.norm == 0) return;
    float mean = 0.f;
    if (p.norm == 1) mean = block_sum4(sum, red) / (float)dim;
    float sq = 0.f;
    for (int i = threadIdx.x; i < dim; i += 256) {
        const float d = rowbuf[i] - mean;
        sq += d * d;
    }
    const float inv = 1.0f / sqrtf(block_sum4(sq, red) / (float)dim + p.eps);
    A* h = (A*)p.h + row * p.h_stride;
    for (int i = threadIdx.x; i < dim; i += 256) {
        float v = (rowbuf[i] - mean) * inv * (float)((const A*)p.nw)[i];
        if (p.nb) v += (float)((const A*)p.nb)[i];
        h[i] = (A)v;
    }
}

// The close of a sublayer in a stack that norms AFTER the sum, per row:
//   v = alpha x + ls (y + y32);   x <- v rsqrt(mean(v^2) + eps) (offset + w);   h <- x in the activation type
// alpha: the weight of the old stream in the sum; ls: a per-column scale of the sublayer's result (null: 1); y (type A) and
// y32 (fp32) are the sublayer's result, either or both may be absent (none: the norm alone, with alpha; write_x 0 then leaves
// the stream as it is and gives h only).  offset 1 serves
// a weight that is stored around zero.  The stream stays fp32; the sum, the statistics and the product are fp32.
struct PostNormArgs {
    const void* y;
    int64_t y_stride;
    const float* y32;
    int64_t y32_stride;
    const void* ls;
    float alpha;
    float* x;
    const void* nw;
    float offset, eps;
    void* h;
    int64_t h_stride;
    int dim, write_x;
};

template <typename A, bool MOE>
__global__ __launch_bounds__(256) void residual_postnorm_kernel(PostNormArgs p, MoeTerms m) {
    extern __shared__ float rowbuf[];
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    const A* y = p.y ? (const A*)p.y + row * p.y_stride : nullptr;
    const float* y32 = p.y32 ? p.y32 + row * p.y32_stride : nullptr;
    const A* ls = (const A*)p.ls;
    float* xr = p.x + row * dim;
    float sq = 0.f;
    for (int i = threadIdx.x; i < dim; i += 256) {
        float v = p.alpha * xr[i];
        if (MOE || y || y32) {
            float s = y ? (float)y[i] : 0.f;
            if (y32) s += y32[i];
            if constexpr (MOE) {
                float e[1];
                moe_sum<A, 1>(m, row, i, e);
                s += e[0];
            }
            if (ls) s *= (float)ls[i];
            v += s;
        }
        rowbuf[i] = v;
        sq += v * v;
    }
    const float inv = 1.0f / sqrtf(block_sum4(sq, red) / (float)dim + p.eps);
    A* h = p.h ? (A*)p.h + row * p.h_stride : nullptr;
    for (int i = threadIdx.x; i < dim; i += 256) {
        const float v = rowbuf[i] * inv * (p.offset + (float)((const A*)p.nw)[i]);
        if (p.write_x) xr[i] = v;
        if (h) h[i] = (A)v;
    }
}

template <typename A, int R, bool MOE>
__global__ __launch_bounds__(256) void residual_postnorm_vec_kernel(PostNormArgs p, MoeTerms m) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    float* xr = p.x + row * dim;
    const bool any = MOE || p.y || p.y32;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};
    f32x4 x[R], y[R], y32[R], ls[R], nw[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + 256 * j) * 4;
        x[j] = y[j] = y32[j] = nw[j] = zero;
        ls[j] = one;
        if (col < dim) {
            x[j] = load4(xr + col);
            if (p.y) y[j] = load4((const A*)p.y + row * p.y_stride + col);
            if (p.y32) y32[j] = load4(p.y32 + row * p.y32_stride + col);
            if (p.ls) ls[j] = load4((const A*)p.ls + col);
            nw[j] = load4((const A*)p.nw + col);
            if constexpr (MOE) {
                float s[4];
                moe_sum<A, 4>(m, row, col, s);
                y32[j] = f32x4{s[0], s[1], s[2], s[3]};
            }
        }
    }
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = p.alpha * x[j][e];
            if (any) {
                float s = y[j][e];
                if (MOE || p.y32) s += y32[j][e];
                if (p.ls) s *= ls[j][e];
                v += s;
            }
            x[j][e] = v;
            sq += v * v;
        }
    const float inv = 1.0f / sqrtf(block_sum4(sq, red) / (float)dim + p.eps);
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + 256 * j) * 4;
        if (col >= dim) continue;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[j][e] * inv * (p.offset + nw[j][e]);
        if (p.write_x) *reinterpret_cast<f32x4*>(xr + col) = v;
        if (p.h) store4((A*)p.h + row * p.h_stride + col, v);
    }
}

template <typename A>
static bool launch_residual_postnorm_vec(const PostNormArgs& p, const MoeTerms& m, int64_t rows, hipStream_t st) {
    const int pieces = close_pieces(p.dim);
    if (!pieces || !rows_of_fours<A>(p.y, p.y_stride) || !rows_of_fours<float>(p.y32, p.y32_stride) || !rows_of_fours<A>(p.ls, 0) || !rows_of_fours<A>(p.nw, 0) ||
        !rows_of_fours<A>(p.h, p.h_stride) || !nvh_aligned16(p.x) || !moe_of_fours<A>(m))
        return false;
    const dim3 grid((unsigned)rows);
    NVH_CLOSE_CASES(residual_postnorm_vec_kernel, p, m)
    return true;
}

// The close of a sublayer whose RESULT is normed before it joins the stream (the sublayer itself read the stream as it is), per row:
//   y = sa a + sb b + c32;   x <- x + mult * w * y / sqrt(mean(y^2) + eps);   h <- x in the activation type (when asked for)
// a, b (type A) and c32 (fp32) are the sublayer's terms, any of them absent; w: one number for all columns (w_elems 1) or one a
// column.  Sums, statistics and the stream are fp32; the row sits in LDS between the two passes.
struct SubNormArgs {
    const void *a, *b;
    const float* c32;
    int64_t a_stride, b_stride, c32_stride;
    float sa, sb, mult, eps;
    const void* w;
    int w_elems;
    float* x;
    void* h;
    int64_t h_stride;
    int dim;
};

template <typename A, bool MOE>
__global__ __launch_bounds__(256) void residual_subnorm_kernel(SubNormArgs p, MoeTerms m) {
    extern __shared__ float rowbuf[];
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    const A* a = p.a ? (const A*)p.a + row * p.a_stride : nullptr;
    const A* b = p.b ? (const A*)p.b + row * p.b_stride : nullptr;
    const float* c32 = p.c32 ? p.c32 + row * p.c32_stride : nullptr;
    float sq = 0.f;
    for (int i = threadIdx.x; i < dim; i += 256) {
        float y = 0.f;
        if (a) y = p.sa * (float)a[i];
        if (b) y = __builtin_fmaf(p.sb, (float)b[i], y);
        if (c32) y += c32[i];
        if constexpr (MOE) {
            float e[1];
            moe_sum<A, 1>(m, row, i, e);
            y += e[0];
        }
        rowbuf[i] = y;
        sq += y * y;
    }
    const float inv = p.mult / sqrtf(block_sum4(sq, red) / (float)dim + p.eps);
    float* xr = p.x + row * dim;
    A* h = p.h ? (A*)p.h + row * p.h_stride : nullptr;
    const A* w = (const A*)p.w;
    for (int i = threadIdx.x; i < dim; i += 256) {
        const float v = xr[i] + rowbuf[i] * inv * (float)w[p.w_elems == 1 ? 0 : i];
        xr[i] = v;
        if (h) h[i] = (A)v;
    }
}

template <typename A, int R, bool MOE>
__global__ __launch_bounds__(256) void residual_subnorm_vec_kernel(SubNormArgs p, MoeTerms m) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int dim = p.dim;
    float* xr = p.x + row * dim;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const float w1 = p.w_elems == 1 ? (float)((const A*)p.w)[0] : 0.f;
    f32x4 x[R], y[R], b[R], c[R], w[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + 256 * j) * 4;
        x[j] = y[j] = b[j] = c[j] = zero;
        w[j] = f32x4{w1, w1, w1, w1};
        if (col < dim) {
            if (p.a) y[j] = load4((const A*)p.a + row * p.a_stride + col);
            if (p.b) b[j] = load4((const A*)p.b + row * p.b_stride + col);
            if (p.c32) c[j] = load4(p.c32 + row * p.c32_stride + col);
            x[j] = load4(xr + col);
            if (p.w_elems != 1) w[j] = load4((const A*)p.w + col);
            if constexpr (MOE) {
                float s[4];
                moe_sum<A, 4>(m, row, col, s);
                c[j] = f32x4{s[0], s[1], s[2], s[3]};
            }
        }
    }
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = p.a ? p.sa * y[j][e] : 0.f;
            if (p.b) v = __builtin_fmaf(p.sb, b[j][e], v);
            if (MOE || p.c32) v += c[j][e];
            y[j][e] = v;
            sq += v * v;
        }
    const float inv = p.mult / sqrtf(block_sum4(sq, red) / (float)dim + p.eps);
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int col = (threadIdx.x + 256 * j) * 4;
        if (col >= dim) continue;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[j][e] + y[j][e] * inv * w[j][e];
        *reinterpret_cast<f32x4*>(xr + col) = v;
        if (p.h) store4((A*)p.h + row * p.h_stride + col, v);
    }
}

template <typename A>
static bool launch_residual_subnorm_vec(const SubNormArgs& p, const MoeTerms& m, int64_t rows, hipStream_t st) {
    const int pieces = close_pieces(p.dim);
    if (!pieces || !rows_of_fours<A>(p.a, p.a_stride) || !rows_of_fours<A>(p.b, p.b_stride) || !rows_of_fours<float>(p.c32, p.c32_stride) ||
        (p.w_elems != 1 && !rows_of_fours<A>(p.w, 0)) || !rows_of_fours<A>(p.h, p.h_stride) || !nvh_aligned16(p.x) || !moe_of_fours<A>(m))
        return false;
    const dim3 grid((unsigned)rows);
    NVH_CLOSE_CASES(residual_subnorm_vec_kernel, p, m)
    return true;
}

// y = act(g) (* u when gated): g = columns [0, inter) and u = columns [inter, 2 inter) of the row.
// act: 0 silu, 1 gelu (tanh form), 2 squared relu.
// E: elements a lane, 8 where rows and strides allow 16-byte accesses.
// us, one element a lane behind a division in 64 bits and so: silu 1024 x 3072 10.0 and 6.0 (19 MB), gelu 8.5 and 6.6; 4000 x 768 10.0 and 6.1.
template <typename A, int E>
__global__ __launch_bounds__(256) void act_mul_kernel(const A* __restrict__ gu, int64_t gu_stride, A* __restrict__ y, int64_t y_stride, int64_t rows, int inter,
                                                      int act, int gated) {
    int64_t row;
    int c;
    if (!nvh_piece<E>(rows, inter, row, c)) return;
    const A* src = gu + row * gu_stride + c;
    float v[E], u[E];
    nvh_load_piece<A, E>(src, v);
    if (gated) nvh_load_piece<A, E>(src + inter, u);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        v[e] = nvh_activation(v[e], act);
        if (gated) v[e] *= u[e];
    }
    nvh_store_piece<A, E>(y + row * y_stride + c, v);
}
static void launch_act_mul(const void* x, int64_t row_stride, void* y, int64_t y_stride, int64_t rows, int64_t inter, int act, int gated, bool act_f32, hipStream_t st) {
    const bool vec = rows * inter >= NVH_PIECES && inter % 8 == 0 && row_stride % 8 == 0 && y_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(y);
    const dim3 grid((unsigned)nvh_cdiv(rows * inter, vec ? 2048 : 256));
    auto launch = [&](auto kernel, auto type) {
        typedef decltype(type) A;
        kernel<<<grid, 256, 0, st>>>((const A*)x, row_stride, (A*)y, y_stride, rows, (int)inter, act, gated);
    };
    if (act_f32) launch(vec ? &act_mul_kernel<float, 8> : &act_mul_kernel<float, 1>, 0.f);
    else launch(vec ? &act_mul_kernel<bf16, 8> : &act_mul_kernel<bf16, 1>, (bf16)0.f);
}

// xIELU with the two numbers (p, q) of `params`, in fp32:  z > 0: softplus(p) z^2 + z / 2;  else (1/2 + softplus(q)) (e^z - 1 - z) + z / 2.
// VEC: eight consecutive elements a lane (row and row strides multiples of eight elements, 16-byte aligned).
template <typename A, bool VEC>
__global__ __launch_bounds__(256) void xielu_kernel(const A* __restrict__ x, int64_t x_stride, A* __restrict__ y, int64_t y_stride, int64_t rows, int inter,
                                                    const A* __restrict__ params) {
    constexpr int E = VEC ? 8 : 1;
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * E;
    if (i >= rows * inter) return;
    const int64_t row = i / inter;
    const int c = (int)(i - row * inter);
    auto softplus = [](float t) {
        if constexpr (sizeof(A) == 4) return fmaxf(t, 0.f) + log1pf(expf(-fabsf(t)));
        else return nvh_softplus_hw(t);
    };
    const float pos = softplus((float)params[0]), neg = 0.5f + softplus((float)params[1]);
    const A* src = x + row * x_stride + c;
    A* dst = y + row * y_stride + c;
    A in[E], out[E];
    if constexpr (VEC) __builtin_memcpy(in, __builtin_assume_aligned(src, 16), sizeof(in));
    else in[0] = src[0];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const float z = (float)in[e];
        if constexpr (sizeof(A) == 4) out[e] = (A)((z > 0.f ? pos * z * z : neg * (expm1f(fminf(z, 0.f)) - z)) + 0.5f * z);
        else out[e] = (A)nvh_xielu_hw(z, pos, neg);
    }
    if constexpr (VEC) __builtin_memcpy(__builtin_assume_aligned(dst, 16), out, sizeof(out));
    else dst[0] = out[0];
}


// ---------------------------------------------------------------------------------------------------------------
// The any-shape product (gemm_any.h) over one weight matrix: tile (blockIdx.x, blockIdx.y) covers 64 columns and the 64
// rows that start at 64 blockIdx.y.
template <bool OUT_F32>
__global__ __launch_bounds__(256) void gemm_any_bf16_kernel(const bf16* __restrict__ x, int64_t ldx, const bf16* __restrict__ w, int64_t ldw,
                                                            const bf16* __restrict__ bias, void* __restrict__ yv, int64_t ldy, int M, int N, int K,
                                                            int vec_ok) {
    const int m0 = blockIdx.y * nvh_any::GT;
    nvh_any::gemm_any_bf16_tile<OUT_F32>(x, ldx, w, ldw, bias, yv, ldy, nvh_any::RowMap{nullptr, m0, min(nvh_any::GT, M - m0)}, blockIdx.x * nvh_any::GT, N, K, vec_ok);
}

template <int MR, int NC>
__global__ __launch_bounds__(256) void gemm_any_f32_kernel(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw,
                                                           const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, int M, int N, int K, int vec_ok) {
    for (int64_t m0 = blockIdx.y * 16 * MR; m0 < M; m0 += (int64_t)gridDim.y * 16 * MR)      // (once, but for more rows than a grid has tiles)
        nvh_any::gemm_any_f32_tile<MR, NC>(x, ldx, w, ldw, bias, y, ldy, nvh_any::RowMap{nullptr, (int)m0, (int)min((int64_t)16 * MR, M - m0)}, 0, blockIdx.x * 16 * NC, N, K, vec_ok);
}

template <int MR, int NC, int STAGES>
__global__ __launch_bounds__(256) void gemm_any_f32_ring_kernel(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, const float* __restrict__ bias,
                                                                float* __restrict__ y, int64_t ldy, int M, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) char ring_lds[];
    for (int64_t m0 = blockIdx.y * 16 * MR; m0 < M; m0 += (int64_t)gridDim.y * 16 * MR) {    // (once, but for more rows than a grid has tiles)
        nvh_any::gemm_any_f32_ring<MR, NC, STAGES>(x, ldx, w, K, bias, y, ldy, nvh_any::RowMap{nullptr, (int)m0, (int)min((int64_t)16 * MR, M - m0)}, 0,
                                                   blockIdx.x * 16 * NC, N, K, nullptr, 0, 0, ring_lds);
        __syncthreads();
    }
}

template <int MR, int NC, int STAGES>
bool launch_f32_ring(const float* x, int64_t ldx, const float* w, const float* bias, float* y, int64_t ldy, int64_t M, int64_t N, int64_t K, hipStream_t st) {
    constexpr int lds = nvh_any::f32_ring_bytes<MR, NC, STAGES>();
    static std::atomic<uint64_t> granted{0};
    if (lds > 64 * 1024 && !nvh_grant_lds(granted, reinterpret_cast<const void*>(&gemm_any_f32_ring_kernel<MR, NC, STAGES>), lds)) return false;
    gemm_any_f32_ring_kernel<MR, NC, STAGES><<<dim3((unsigned)nvh_cdiv(N, 16 * NC), (unsigned)std::min<int64_t>(nvh_cdiv(M, 16 * MR), 65535)), 256, lds, st>>>(
        x, ldx, w, bias, y, ldy, (int)M, (int)N, (int)K);
    return true;
}

}  // namespace

#define NVH_STREAM_ARGS_OK(name, cond) NVH_REQUIRE(cond, NVH_EINVAL, name ": bad argument")

extern "C" int32_t nvh_embedding_stream(const int64_t* ids, const void* table, float* x, void* x0, int64_t x0_stride,
                                        int64_t num_tokens, int64_t dim, int64_t vocab, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_embedding_stream", ids && table && x && num_tokens >= 0 && dim > 0 && vocab > 0);
    if (num_tokens == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) embedding_stream_kernel<float><<<dim3((unsigned)num_tokens), 256, 0, st>>>(ids, (const float*)table, x, (float*)x0, x0_stride, (int)dim, vocab);
    else embedding_stream_kernel<bf16><<<dim3((unsigned)num_tokens), 256, 0, st>>>(ids, (const bf16*)table, x, (bf16*)x0, x0_stride, (int)dim, vocab);
    NVH_CHECK_LAUNCH("nvh_embedding_stream");
    return NVH_OK;
}

extern "C" int32_t nvh_residual_dyt(const void* y, int64_t y_stride, const void* post_alpha, const void* post_w, const void* post_b,
                                    const void* bias, float* x, int32_t accumulate, const void* next_alpha, const void* next_w,
                                    const void* next_b, void* h, int64_t h_stride, int64_t rows, int64_t dim, int32_t act_f32,
                                    nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_residual_dyt", x && rows >= 0 && dim > 0 && (!post_w || (post_alpha && post_b && y)) &&
                                               (!next_w || (next_alpha && next_b && h)) && (accumulate || y || bias));
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    const DytNorm post{post_alpha, post_w, post_b}, next{next_alpha, next_w, next_b};
    const int esz = act_f32 ? 4 : 2;
    auto al = [&](const void* p, int bytes) { return p == nullptr || ((uintptr_t)p % bytes) == 0; };
    const bool vec = dim % 4 == 0 && al(x, 16) && al(y, 4 * esz) && y_stride % 4 == 0 && al(h, 4 * esz) && h_stride % 4 == 0 && al(bias, 4 * esz) &&
                     al(post_w, 4 * esz) && al(post_b, 4 * esz) && al(next_w, 4 * esz) && al(next_b, 4 * esz);
    const dim3 grid((unsigned)rows);
    if (act_f32) {
        if (vec) residual_dyt_kernel<float, true><<<grid, 256, 0, st>>>((const float*)y, y_stride, post, (const float*)bias, x, accumulate, next, (float*)h, h_stride, (int)dim);
        else residual_dyt_kernel<float, false><<<grid, 256, 0, st>>>((const float*)y, y_stride, post, (const float*)bias, x, accumulate, next, (float*)h, h_stride, (int)dim);
    } else {
        if (vec) residual_dyt_kernel<bf16, true><<<grid, 256, 0, st>>>((const bf16*)y, y_stride, post, (const bf16*)bias, x, accumulate, next, (bf16*)h, h_stride, (int)dim);
        else residual_dyt_kernel<bf16, false><<<grid, 256, 0, st>>>((const bf16*)y, y_stride, post, (const bf16*)bias, x, accumulate, next, (bf16*)h, h_stride, (int)dim);
    }
    NVH_CHECK_LAUNCH("nvh_residual_dyt");
    return NVH_OK;
}

extern "C" int32_t nvh_stream_cast(const float* x, void* out, int64_t out_stride, int64_t rows, int64_t dim, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_stream_cast", x && out && rows >= 0 && dim > 0 && out_stride >= dim);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) stream_cast_kernel<float><<<dim3((unsigned)rows), 256, 0, st>>>(x, (float*)out, out_stride, (int)dim);
    else stream_cast_kernel<bf16><<<dim3((unsigned)rows), 256, 0, st>>>(x, (bf16*)out, out_stride, (int)dim);
    NVH_CHECK_LAUNCH("nvh_stream_cast");
    return NVH_OK;
}

extern "C" int32_t nvh_gelu_tanh_mul(const void* gate_up, int64_t row_stride, void* y, int64_t rows, int64_t inter, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_gelu_tanh_mul", gate_up && y && rows >= 0 && inter > 0 && row_stride >= 2 * inter);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    launch_act_mul(gate_up, row_stride, y, inter, rows, inter, 1, 1, act_f32, st);
    NVH_CHECK_LAUNCH("nvh_gelu_tanh_mul");
    return NVH_OK;
}

extern "C" int32_t nvh_gather_rows_f32(const float* x, const int32_t* index, float* out, int64_t rows, int64_t dim, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_gather_rows_f32", x && index && out && rows >= 0 && dim > 0);
    if (rows == 0) return NVH_OK;
    gather_rows_f32_kernel<<<dim3((unsigned)rows), 256, 0, (hipStream_t)stream>>>(x, index, out, (int)dim);
    NVH_CHECK_LAUNCH("nvh_gather_rows_f32");
    return NVH_OK;
}

extern "C" int32_t nvh_logit_softcap(const void* logits, int64_t row_stride, float* out, int64_t rows, int64_t vocab, float cap, int32_t act_f32,
                                     nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_logit_softcap", logits && out && rows >= 0 && vocab > 0 && row_stride >= vocab);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    launch_logits_scale(logits, row_stride, out, rows, vocab, 1.0f, cap, act_f32, st);
    NVH_CHECK_LAUNCH("nvh_logit_softcap");
    return NVH_OK;
}

extern "C" int32_t nvh_gemm_any_nt(const void* x, int64_t x_row_stride, const void* w, const void* bias, void* y, int64_t y_row_stride,
                                   int64_t M, int64_t N, int64_t K, int32_t in_f32, int32_t out_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_gemm_any_nt", x && w && y && M >= 0 && N > 0 && K > 0 && M < (1 << 30) && N < (1 << 30) && K < (1 << 30) &&
                                              x_row_stride >= K && y_row_stride >= N);
    NVH_REQUIRE(!in_f32 || out_f32, NVH_ENOSYS, "nvh_gemm_any_nt: fp32 operands give an fp32 product");
    if (M == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)nvh_cdiv(N, nvh_any::GT), (unsigned)nvh_cdiv(M, nvh_any::GT));
    if (in_f32) {
        // (16 rows or fewer: small tiles, so that more workgroups share the weights' stream; the same sums either way)
        const int vec_ok = nvh_any::f32_vec_ok(x, x_row_stride, w, K);
        if (vec_ok && K % nvh_any::F32_CHUNK == 0) {
            // The tile whose rounds over the CUs take least.  16 x 16 (two workgroups a CU) and 32 x 32 tiles while they fill at most a round;
            // then 32 x 64 or 64 x 64 ones, a workgroup a CU, a round of which takes 13 and 22 us for K = 1024.
            // 16 rows or fewer are one row tile, whose time is the weights' way: 16 x 16 at any width, beyond a round with three stages, three workgroups
            // a CU.  us, without a ring, 32 x 64 and this: 1 x 32000 x 1024 32.1, 33.8, 27.5; 1 x 32000 x 256 12.3, 14.1, 10.8; 1 x 12288 x 5120 49.5,
            // 56.8, 46.0; 16 x 32000 x 1024 50.4, 34.9, 30.2; 16 x 12288 x 5120 84.5, 58.5, 53.3; two columns blocks a tile 27.5 at one row of
            // 32000 x 1024, but 51.3 of 12288 x 5120.
            auto tiles = [&](int rows, int cols) { return nvh_cdiv(M, rows) * nvh_cdiv(N, cols); };
#define NVH_F32_RING(MR, NC, STAGES) launch_f32_ring<MR, NC, STAGES>((const float*)x, x_row_stride, (const float*)w, (const float*)bias, (float*)y, y_row_stride, M, N, K, st)
            bool ok;
            if (tiles(16, 16) <= 512) ok = NVH_F32_RING(1, 1, 4);
            else if (M <= 16) ok = NVH_F32_RING(1, 1, 3);
            else if (tiles(32, 32) <= 256) ok = NVH_F32_RING(2, 2, 2);
            else if (nvh_cdiv(tiles(64, 64), 256) * 22 < nvh_cdiv(tiles(32, 64), 256) * 13) ok = NVH_F32_RING(4, 4, 2);
            else ok = NVH_F32_RING(2, 4, 2);
#undef NVH_F32_RING
            NVH_REQUIRE(ok, NVH_ENOSYS, "nvh_gemm_any_nt: more than 64 KB of LDS for a workgroup refused");
            NVH_CHECK_LAUNCH("nvh_gemm_any_nt");
            return NVH_OK;
        }
        if (M <= 16) gemm_any_f32_kernel<1, 1><<<dim3((unsigned)nvh_cdiv(N, 16), 1), 256, 0, st>>>((const float*)x, x_row_stride, (const float*)w, K, (const float*)bias, (float*)y, y_row_stride, (int)M, (int)N, (int)K, vec_ok);
        else gemm_any_f32_kernel<2, 2><<<dim3((unsigned)nvh_cdiv(N, 32), (unsigned)std::min<int64_t>(nvh_cdiv(M, 32), 65535)), 256, 0, st>>>((const float*)x, x_row_stride, (const float*)w, K, (const float*)bias, (float*)y, y_row_stride, (int)M, (int)N, (int)K, vec_ok);
    } else {
        const int vec_ok = K % 8 == 0 && x_row_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(w);
        // (the same bits: this form's rows of columns through LDS, whole k-tiles ahead; the other takes any shape, stride and bias)
        if (!bias && nvh_any::launch_short_product(x, x_row_stride, w, y, y_row_stride, M, N, K, out_f32 != 0, st)) {
            NVH_CHECK_LAUNCH("nvh_gemm_any_nt");
            return NVH_OK;
        }
        if (out_f32) gemm_any_bf16_kernel<true><<<grid, 256, 0, st>>>((const bf16*)x, x_row_stride, (const bf16*)w, K, (const bf16*)bias, y, y_row_stride, (int)M, (int)N, (int)K, vec_ok);
        else gemm_any_bf16_kernel<false><<<grid, 256, 0, st>>>((const bf16*)x, x_row_stride, (const bf16*)w, K, (const bf16*)bias, y, y_row_stride, (int)M, (int)N, (int)K, vec_ok);
    }
    NVH_CHECK_LAUNCH("nvh_gemm_any_nt");
    return NVH_OK;
}

extern "C" int32_t nvh_embedding_pos_stream(const int64_t* ids, const int64_t* positions, const void* table, const void* pos_table, float scale,
                                            float* x, int64_t num_tokens, int64_t dim, int64_t vocab, int64_t max_positions, int32_t act_f32,
                                            nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_embedding_pos_stream", ids && table && x && num_tokens >= 0 && dim > 0 && vocab > 0 && (!pos_table || (positions && max_positions > 0)));
    if (num_tokens == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) embedding_pos_stream_kernel<float><<<dim3((unsigned)num_tokens), 256, 0, st>>>(ids, positions, (const float*)table, (const float*)pos_table, scale, x, (int)dim, vocab, max_positions);
    else embedding_pos_stream_kernel<bf16><<<dim3((unsigned)num_tokens), 256, 0, st>>>(ids, positions, (const bf16*)table, (const bf16*)pos_table, scale, x, (int)dim, vocab, max_positions);
    NVH_CHECK_LAUNCH("nvh_embedding_pos_stream");
    return NVH_OK;
}

// The closes column by column, a row in LDS: any size and alignment.
template <typename Args>
static int32_t launch_close_columns(void (*kernel)(Args, MoeTerms), const Args& p, const MoeTerms& m, int64_t rows, int64_t dim, hipStream_t st) {
    const size_t lds = sizeof(float) * (size_t)dim;
    if (lds > 48 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        NVH_REQUIRE(e == hipSuccess, NVH_ENOSYS, "close of a residual row: %zu bytes of LDS refused", lds);
    }
    kernel<<<dim3((unsigned)rows), 256, lds, st>>>(p, m);
    return NVH_OK;
}

static int32_t residual_norm(const void* a, int64_t a_stride, const void* a_weight, const void* b, int64_t b_stride, const void* b_weight,
                             float branch_scale, float branch_eps, const void* c, int64_t c_stride, const float* c32, int64_t c32_stride, float* x,
                             int32_t norm_kind, const void* norm_weight, const void* norm_bias, float eps, void* h, int64_t h_stride, int64_t rows,
                             int64_t dim, const MoeTerms& m, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_residual_norm", x && rows >= 0 && dim > 0 && dim <= 32768 && norm_kind >= 0 && norm_kind <= 2 && (norm_kind == 0 || (norm_weight && h)) &&
                                                (!a_weight || a) && (!b_weight || b));
    if (rows == 0) return NVH_OK;
    const CloseArgs p{a, a_weight, b, b_weight, c, c32, a_stride, b_stride, c_stride, c32_stride, branch_scale, branch_eps, x, norm_kind,
                      norm_weight, norm_bias, eps, h, h_stride, (int)dim};
    hipStream_t st = (hipStream_t)stream;
    if (act_f32 ? launch_residual_norm_vec<float>(p, m, rows, st) : launch_residual_norm_vec<bf16>(p, m, rows, st)) {
        NVH_CHECK_LAUNCH("nvh_residual_norm");
        return NVH_OK;
    }
    const int32_t rc = act_f32 ? (m.y ? launch_close_columns(&residual_norm_kernel<float, true>, p, m, rows, dim, st) : launch_close_columns(&residual_norm_kernel<float, false>, p, m, rows, dim, st))
                               : (m.y ? launch_close_columns(&residual_norm_kernel<bf16, true>, p, m, rows, dim, st) : launch_close_columns(&residual_norm_kernel<bf16, false>, p, m, rows, dim, st));
    if (rc != NVH_OK) return rc;
    NVH_CHECK_LAUNCH("nvh_residual_norm");
    return NVH_OK;
}

extern "C" int32_t nvh_residual_norm(const void* a, int64_t a_stride, const void* a_weight, const void* b, int64_t b_stride, const void* b_weight,
                                     float branch_scale, float branch_eps, const void* c, int64_t c_stride, const float* c32, int64_t c32_stride,
                                     float* x, int32_t norm_kind, const void* norm_weight, const void* norm_bias, float eps, void* h,
                                     int64_t h_stride, int64_t rows, int64_t dim, int32_t act_f32, nvh_stream_t stream) {
    return residual_norm(a, a_stride, a_weight, b, b_stride, b_weight, branch_scale, branch_eps, c, c_stride, c32, c32_stride, x, norm_kind, norm_weight, norm_bias, eps, h, h_stride, rows, dim,
                        MoeTerms{}, act_f32, stream);
}

extern "C" int32_t nvh_residual_norm_moe(const void* a, int64_t a_stride, const void* a_weight, const void* b, int64_t b_stride,
                                         const void* b_weight, float branch_scale, float branch_eps, const void* c, int64_t c_stride,
                                         const float* c32, int64_t c32_stride, float* x, int32_t norm_kind, const void* norm_weight,
                                         const void* norm_bias, float eps, void* h, int64_t h_stride, int64_t rows, int64_t dim, const void* moe_y,
                                         int64_t moe_y_stride, const int32_t* pos_of_pair, const float* moe_weights, int64_t top, const void* shared,
                                         int64_t shared_stride, const float* shared_gate, int64_t shared_gate_stride, int32_t act_f32,
                                         nvh_stream_t stream) {
    NVH_REQUIRE(moe_y && pos_of_pair && top > 0 && top <= 4096 && moe_y_stride >= dim && (!shared || shared_stride >= dim) && (shared || !shared_gate) &&
                    !c32, NVH_EINVAL, "nvh_residual_norm_moe: bad argument");
    const MoeTerms m{moe_y, moe_y_stride, pos_of_pair, moe_weights, (int)top, shared, shared_stride, shared_gate, shared_gate_stride};
    return residual_norm(a, a_stride, a_weight, b, b_stride, b_weight, branch_scale, branch_eps, c, c_stride, c32, c32_stride, x, norm_kind, norm_weight, norm_bias, eps, h, h_stride, rows, dim, m, act_f32, stream);
}

static int32_t residual_postnorm(const void* y, int64_t y_stride, const float* y32, int64_t y32_stride, const void* layer_scale, float alpha,
                                 float* x, int32_t write_x, const void* norm_weight, float weight_offset, float eps, void* h, int64_t h_stride,
                                 int64_t rows, int64_t dim, const MoeTerms& m, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_residual_postnorm", x && norm_weight && rows >= 0 && dim > 0 && dim <= 32768 && (!y || y_stride >= dim) && (!y32 || y32_stride >= dim) &&
                                                    (!h || h_stride >= dim));
    if (rows == 0) return NVH_OK;
    const PostNormArgs p{y, y_stride, y32, y32_stride, layer_scale, alpha, x, norm_weight, weight_offset, eps, h, h_stride, (int)dim, write_x};
    hipStream_t st = (hipStream_t)stream;
    if (act_f32 ? launch_residual_postnorm_vec<float>(p, m, rows, st) : launch_residual_postnorm_vec<bf16>(p, m, rows, st)) {
        NVH_CHECK_LAUNCH("nvh_residual_postnorm");
        return NVH_OK;
    }
    const int32_t rc = act_f32 ? (m.y ? launch_close_columns(&residual_postnorm_kernel<float, true>, p, m, rows, dim, st) : launch_close_columns(&residual_postnorm_kernel<float, false>, p, m, rows, dim, st))
                               : (m.y ? launch_close_columns(&residual_postnorm_kernel<bf16, true>, p, m, rows, dim, st) : launch_close_columns(&residual_postnorm_kernel<bf16, false>, p, m, rows, dim, st));
    if (rc != NVH_OK) return rc;
    NVH_CHECK_LAUNCH("nvh_residual_postnorm");
    return NVH_OK;
}

extern "C" int32_t nvh_residual_postnorm(const void* y, int64_t y_stride, const float* y32, int64_t y32_stride, const void* layer_scale, float alpha,
                                         float* x, int32_t write_x, const void* norm_weight, float weight_offset, float eps, void* h,
                                         int64_t h_stride, int64_t rows, int64_t dim, int32_t act_f32, nvh_stream_t stream) {
    return residual_postnorm(y, y_stride, y32, y32_stride, layer_scale, alpha, x, write_x, norm_weight, weight_offset, eps, h, h_stride, rows, dim,
                            MoeTerms{}, act_f32, stream);
}

extern "C" int32_t nvh_residual_postnorm_moe(const void* y, int64_t y_stride, const float* y32, int64_t y32_stride, const void* layer_scale,
                                             float alpha, float* x, int32_t write_x, const void* norm_weight, float weight_offset, float eps,
                                             void* h, int64_t h_stride, int64_t rows, int64_t dim, const void* moe_y, int64_t moe_y_stride,
                                             const int32_t* pos_of_pair, const float* moe_weights, int64_t top, const void* shared,
                                             int64_t shared_stride, const float* shared_gate, int64_t shared_gate_stride, int32_t act_f32,
                                             nvh_stream_t stream) {
    NVH_REQUIRE(moe_y && pos_of_pair && top > 0 && top <= 4096 && moe_y_stride >= dim && (!shared || shared_stride >= dim) && (shared || !shared_gate) &&
                    !y32, NVH_EINVAL, "nvh_residual_postnorm_moe: bad argument");
    const MoeTerms m{moe_y, moe_y_stride, pos_of_pair, moe_weights, (int)top, shared, shared_stride, shared_gate, shared_gate_stride};
    return residual_postnorm(y, y_stride, y32, y32_stride, layer_scale, alpha, x, write_x, norm_weight, weight_offset, eps, h, h_stride, rows, dim, m, act_f32, stream);
}

static int32_t residual_subnorm(const void* a, int64_t a_stride, float a_scale, const void* b, int64_t b_stride, float b_scale, const float* c32,
                                int64_t c32_stride, float mult, const void* weight, int64_t weight_elems, float eps, float* x, void* h,
                                int64_t h_stride, int64_t rows, int64_t dim, const MoeTerms& m, int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_residual_subnorm", x && weight && (a || b || c32 || m.y) && rows >= 0 && dim > 0 && dim <= 32768 && (weight_elems == 1 || weight_elems == dim));
    if (rows == 0) return NVH_OK;
    const SubNormArgs p{a, b, c32, a_stride, b_stride, c32_stride, a_scale, b_scale, mult, eps, weight, (int)weight_elems, x, h, h_stride, (int)dim};
    hipStream_t st = (hipStream_t)stream;
    if (act_f32 ? launch_residual_subnorm_vec<float>(p, m, rows, st) : launch_residual_subnorm_vec<bf16>(p, m, rows, st)) {
        NVH_CHECK_LAUNCH("nvh_residual_subnorm");
        return NVH_OK;
    }
    const int32_t rc = act_f32 ? (m.y ? launch_close_columns(&residual_subnorm_kernel<float, true>, p, m, rows, dim, st) : launch_close_columns(&residual_subnorm_kernel<float, false>, p, m, rows, dim, st))
                               : (m.y ? launch_close_columns(&residual_subnorm_kernel<bf16, true>, p, m, rows, dim, st) : launch_close_columns(&residual_subnorm_kernel<bf16, false>, p, m, rows, dim, st));
    if (rc != NVH_OK) return rc;
    NVH_CHECK_LAUNCH("nvh_residual_subnorm");
    return NVH_OK;
}

extern "C" int32_t nvh_residual_subnorm(const void* a, int64_t a_stride, float a_scale, const void* b, int64_t b_stride, float b_scale,
                                        const float* c32, int64_t c32_stride, float mult, const void* weight, int64_t weight_elems, float eps,
                                        float* x, void* h, int64_t h_stride, int64_t rows, int64_t dim, int32_t act_f32, nvh_stream_t stream) {
    return residual_subnorm(a, a_stride, a_scale, b, b_stride, b_scale, c32, c32_stride, mult, weight, weight_elems, eps, x, h, h_stride, rows, dim,
                           MoeTerms{}, act_f32, stream);
}

extern "C" int32_t nvh_residual_subnorm_moe(const void* a, int64_t a_stride, float a_scale, const void* b, int64_t b_stride, float b_scale,
                                            const float* c32, int64_t c32_stride, float mult, const void* weight, int64_t weight_elems, float eps,
                                            float* x, void* h, int64_t h_stride, int64_t rows, int64_t dim, const void* moe_y, int64_t moe_y_stride,
                                            const int32_t* pos_of_pair, const float* moe_weights, int64_t top, const void* shared,
                                            int64_t shared_stride, const float* shared_gate, int64_t shared_gate_stride, int32_t act_f32,
                                            nvh_stream_t stream) {
    NVH_REQUIRE(moe_y && pos_of_pair && top > 0 && top <= 4096 && moe_y_stride >= dim && (!shared || shared_stride >= dim) && (shared || !shared_gate) &&
                    !c32, NVH_EINVAL, "nvh_residual_subnorm_moe: bad argument");
    const MoeTerms m{moe_y, moe_y_stride, pos_of_pair, moe_weights, (int)top, shared, shared_stride, shared_gate, shared_gate_stride};
    return residual_subnorm(a, a_stride, a_scale, b, b_stride, b_scale, c32, c32_stride, mult, weight, weight_elems, eps, x, h, h_stride, rows, dim, m, act_f32, stream);
}

extern "C" int32_t nvh_act_mul(const void* x, int64_t row_stride, void* y, int64_t y_stride, int64_t rows, int64_t inter, int32_t act, int32_t gated,
                               int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_act_mul", x && y && rows >= 0 && inter > 0 && act >= 0 && act <= 2 && row_stride >= (gated ? 2 : 1) * inter && y_stride >= inter);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    launch_act_mul(x, row_stride, y, y_stride, rows, inter, act, gated, act_f32, st);
    NVH_CHECK_LAUNCH("nvh_act_mul");
    return NVH_OK;
}

extern "C" int32_t nvh_xielu(const void* x, int64_t row_stride, void* y, int64_t y_stride, int64_t rows, int64_t inter, const void* params, int32_t act_f32,
                             nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_xielu", x && y && params && rows >= 0 && inter > 0 && row_stride >= inter && y_stride >= inter);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    const bool vec = inter % 8 == 0 && row_stride % 8 == 0 && y_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(y);
    const dim3 grid((unsigned)nvh_cdiv(rows * inter, vec ? 2048 : 256));
    if (act_f32) {
        if (vec) xielu_kernel<float, true><<<grid, 256, 0, st>>>((const float*)x, row_stride, (float*)y, y_stride, rows, (int)inter, (const float*)params);
        else xielu_kernel<float, false><<<grid, 256, 0, st>>>((const float*)x, row_stride, (float*)y, y_stride, rows, (int)inter, (const float*)params);
    } else {
        if (vec) xielu_kernel<bf16, true><<<grid, 256, 0, st>>>((const bf16*)x, row_stride, (bf16*)y, y_stride, rows, (int)inter, (const bf16*)params);
        else xielu_kernel<bf16, false><<<grid, 256, 0, st>>>((const bf16*)x, row_stride, (bf16*)y, y_stride, rows, (int)inter, (const bf16*)params);
    }
    NVH_CHECK_LAUNCH("nvh_xielu");
    return NVH_OK;
}

extern "C" int32_t nvh_logits_scale(const void* logits, int64_t row_stride, float* out, int64_t rows, int64_t vocab, float scale, float cap,
                                    int32_t act_f32, nvh_stream_t stream) {
    NVH_STREAM_ARGS_OK("nvh_logits_scale", logits && out && rows >= 0 && vocab > 0 && row_stride >= vocab);
    if (rows == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    launch_logits_scale(logits, row_stride, out, rows, vocab, scale, cap, act_f32, st);
    NVH_CHECK_LAUNCH("nvh_logits_scale");
    return NVH_OK;
}
