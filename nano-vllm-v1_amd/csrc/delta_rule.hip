// Generalized delta rule: a per-head matrix state S [dk, dv] in fp32 that every token updates,
//   S <- diag(w) S - (a * u) (u^T S) + k v^T     (both terms read the old S),   o = S^T r,
// with a decay w in (0, 1) and a removal rate a per key channel and u the unit-length key.
//   nvh_delta_prep   per token and channel, all in fp32: the decay from its low-rank logit
//                    w = exp(-c * sigmoid(w0 + W2 tanh(l))) (c = e^-1/2 by default), a = sigmoid(a_raw + a_bias),
//                    u = k / sqrt(sum k^2 + 1e-6); leaves, per token and head, the contiguous fp32 row
//                    [r | k | w | u | a*u | v] that the scan reads.
//   nvh_delta_scan   walks a sequence's tokens in order from the state its slot holds (or from zero when the sequence
//                    starts) and leaves the state there.  Columns of S are independent of each other, so the work is
//                    spread over (sequence, head, column); each column is held by 16 lanes (4 when dk is no multiple
//                    of 16), each with every 16th (4th) row, which meet twice per token in a cross-lane sum.  The order of
//                    every sum is fixed by the sizes alone: decoding token by token, or cut into other portions, gives the
//                    same bits.
//   nvh_delta_scan_chunked   the same, portions of many tokens in chunks of 16 (see there).
//   nvh_delta_post   per head: o / rms(o), times the norm weight and the sigmoid output gate, to the activation type.
//   nvh_gated_delta_prep   the gated delta rule, S <- g S; d = beta (v - S^T k); S <- S + k d^T; o = S^T q, with one decay g per head
//                    and a write strength beta per head, is the recurrence above with w = g on every channel, u = k (a unit
//                    vector), a u = beta g k and the written key beta k: g S - beta g k (k^T S) + beta k v^T.  The prep runs the
//                    short causal convolution (continued from the sequence's carried inputs) and silu over the q | k | v
//                    channels, makes q and k unit vectors per head (q also times dk^-1/2), forms beta = sigmoid(b) and
//                    g = exp(-exp(A_log) softplus(a + dt_bias)), all in fp32, and leaves the scan's rows; q and k heads
//                    may be shared by groups of value heads, and the value size is free.
#include "common.h"
#include "scan_chunk.h"

namespace {

template <typename A>
__device__ __forceinline__ float ldf(const A* p, int64_t i) {
    return (float)p[i];
}
__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }

struct DeltaPrepArgs {
    const void *r, *k, *v;     // [T, ld] rows of H*dk
    int64_t r_stride, k_stride, v_stride;
    const void* a_raw;         // [T, ld]
    int64_t a_stride;
    const void* lowrank;       // [T, ld] rows of `rank` (the first decay projection, before its tanh)
    int64_t l_stride;
    const void *w2, *w0, *a_bias;   // [H*dk, rank], [H*dk], [H*dk]
    float* out;                // [T, H, 6, dk]: r | k | w | u | a*u | v per head, contiguous
    int H, dk, rank;
    float decay_scale;
};

struct GatedDeltaPrepArgs {
    const void* qkv;           // [T, ld]: the convolved channels q (G dk) | k (G dk) | v (H dv) of the projection row
    int64_t qkv_stride;
    const void *b, *a;         // [T, ld]: H columns each (write strength and decay logits)
    int64_t b_stride, a_stride;
    const void* conv_w;        // [C, taps], last column on the current token
    const void *dt_bias, *a_log;    // [H]
    const float* conv_state;   // [slots, taps - 1, C]
    const int32_t *slots, *cu_seqlens_q, *context_lens;
    float* out;                // [T, H, 5 dk + dv]: q | beta k | g | k | beta g k | v
    int batch, taps, H, G, dk, dv;
};

__device__ __forceinline__ float softplusf_(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// One workgroup per (token, value head): the convolved, activated channels of the head's q / k group and of its own v meet in LDS,
// two waves sum the squares of q and k, then the head's row is written.  (Heads that share a q / k group convolve it again each: a
// few hundred channels, against a launch that would otherwise have as many workgroups as tokens only.)
template <typename A>
__global__ __launch_bounds__(256) void gated_delta_prep_kernel(GatedDeltaPrepArgs p) {
    extern __shared__ float sh[];                            // [dk] q, [dk] k, [dv] v of this head, then the two inverse lengths
    const int64_t t = blockIdx.x;
    const int h = blockIdx.y, dk = p.dk, dv = p.dv, g = h / (p.H / p.G);
    const int nqk = p.G * dk, C = 2 * nqk + p.H * dv, taps = p.taps, n = 2 * dk + dv;
    float* inv = sh + n;
    int seq = (int)t;
    if (p.cu_seqlens_q) {
        int lo_b = 0, hi_b = p.batch;                        // the sequence whose rows hold token t
        while (hi_b - lo_b > 1) {
            const int mid = (lo_b + hi_b) >> 1;
            if (p.cu_seqlens_q[mid] <= t) lo_b = mid;
            else hi_b = mid;
        }
        seq = lo_b;
    }
    const int lo = p.cu_seqlens_q ? p.cu_seqlens_q[seq] : seq, hi = p.cu_seqlens_q ? p.cu_seqlens_q[seq + 1] : seq + 1;
    const int j = (int)t - lo;
    const int slot = p.slots[seq];
    const bool carried = slot >= 0 && p.context_lens[seq] != hi - lo;
    const float* st = carried ? p.conv_state + (int64_t)slot * (taps - 1) * C : nullptr;
    for (int e = threadIdx.x; e < n; e += 256) {
        const int c = e < dk ? g * dk + e : (e < 2 * dk ? nqk + g * dk + (e - dk) : 2 * nqk + h * dv + (e - 2 * dk));      // the channel of the row
        float acc = 0.f;
        for (int k = 0; k < taps; ++k) {                     // tap k multiplies the input taps - 1 - k tokens back
            const int back = taps - 1 - k, src = j - back;
            float in = 0.f;
            if (src >= 0) in = ldf((const A*)p.qkv, (t - back) * p.qkv_stride + c);
            else if (st) in = st[(int64_t)(taps - 1 + src) * C + c];
            acc = __builtin_fmaf(ldf((const A*)p.conv_w, (int64_t)c * taps + k), in, acc);
        }
        sh[e] = acc / (1.0f + expf(-acc));
    }
    const float beta = sigmoidf_(ldf((const A*)p.b, t * p.b_stride + h));
    const float dec = expf(-expf(ldf((const A*)p.a_log, h)) * softplusf_(ldf((const A*)p.a, t * p.a_stride + h) + ldf((const A*)p.dt_bias, h)));
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wave < 2) {                                          // q, k
        float ss = 0.f;
        for (int i = lane; i < dk; i += 64) ss += sh[wave * dk + i] * sh[wave * dk + i];
        ss = wave_sum(ss);
        if (lane == 0) inv[wave] = 1.0f / sqrtf(ss + 1e-6f);
    }
    __syncthreads();
    const int row = 5 * dk + dv;
    const float qs = inv[0] / sqrtf((float)dk), ks = inv[1];
    float* out = p.out + (t * p.H + h) * (int64_t)row;
    for (int i = threadIdx.x; i < dk; i += 256) {
        const float ku = sh[dk + i] * ks;
        out[i] = sh[i] * qs;
        out[dk + i] = beta * ku;
        out[2 * dk + i] = dec;
        out[3 * dk + i] = ku;
        out[4 * dk + i] = beta * dec * ku;
    }
    for (int i = threadIdx.x; i < dv; i += 256) out[5 * dk + i] = sh[2 * dk + i];
}

// The same for TT consecutive tokens a workgroup: a lane has a channel's weights and its inputs of all of them on the way at once and reads an input
// once instead of once per tap.  Same sums in the same order.
// us, one token a workgroup and two or four, heads of 128 x 128: 1000 tokens of 8 heads 33.5 and 17.4 (25 MB written), of 4 15.7 and 11.2, 2000 of 8 61.6 and
// 28.8, 300 of 8 11.4 and 8.3; eight tokens a workgroup 19.2, 15.7, 30.2, 11.5.
// carried_out: every sequence starts in this step, so no lane reads a slot and the last TAPS - 1 tokens of each leave their inputs there (a launch of 3.9 us less);
// a q or k channel that several heads share is the first one's.
template <typename A, int TT, int TAPS>
__global__ __launch_bounds__(256) void gated_delta_prep_run_kernel(GatedDeltaPrepArgs p, int64_t num_tokens, int vec, float* carried_out) {
    extern __shared__ __attribute__((aligned(16))) float sh[];                            // [TT][n] q (dk) | k (dk) | v (dv) of this head, then the numbers of the tokens
    __shared__ int slot_of[TT], end_of[TT];
    __shared__ int first_of[TT], state_of[TT];               // the first row of the token's sequence in this step; its slot, or -1: nothing carried
    const int64_t t0 = (int64_t)blockIdx.x * TT;
    const int nt = (int)min((int64_t)TT, num_tokens - t0), tid = threadIdx.x;
    const int h = blockIdx.y, dk = p.dk, dv = p.dv, g = h / (p.H / p.G);
    const int nqk = p.G * dk, C = 2 * nqk + p.H * dv, n = 2 * dk + dv;
    float *inv = sh + TT * n, *beta = inv + 2 * TT, *dec = beta + TT;
    if (tid < TT) {
        const int64_t t = t0 + min(tid, nt - 1);
        int seq = (int)t, lo = (int)t, hi = (int)t + 1;
        if (p.cu_seqlens_q) {
            int lo_b = 0, hi_b = p.batch;                    // the sequence whose rows hold token t
            while (hi_b - lo_b > 1) {
                const int mid = (lo_b + hi_b) >> 1;
                if (p.cu_seqlens_q[mid] <= t) lo_b = mid;
                else hi_b = mid;
            }
            seq = lo_b;
            lo = p.cu_seqlens_q[seq];
            hi = p.cu_seqlens_q[seq + 1];
        }
        const int slot = p.slots[seq];
        first_of[tid] = lo;
        slot_of[tid] = slot;
        end_of[tid] = hi;
        state_of[tid] = slot >= 0 && p.context_lens[seq] != hi - lo ? slot : -1;
        beta[tid] = sigmoidf_(ldf((const A*)p.b, t * p.b_stride + h));
        dec[tid] = expf(-expf(ldf((const A*)p.a_log, h)) * softplusf_(ldf((const A*)p.a, t * p.a_stride + h) + ldf((const A*)p.dt_bias, h)));
    }
    __syncthreads();
    for (int e = tid; e < n; e += 256) {
        const int c = e < dk ? g * dk + e : (e < 2 * dk ? nqk + g * dk + (e - dk) : 2 * nqk + h * dv + (e - 2 * dk));      // the channel of the row
        float w[TAPS], in[TT + TAPS - 1];                    // in[u]: the input of token t0 - (TAPS - 1) + u (rows outside the step: any, not used)
#pragma unroll
        for (int k = 0; k < TAPS; ++k) w[k] = ldf((const A*)p.conv_w, (int64_t)c * TAPS + k);
#pragma unroll
        for (int u = 0; u < TT + TAPS - 1; ++u) in[u] = ldf((const A*)p.qkv, min(max(t0 - (TAPS - 1) + u, (int64_t)0), num_tokens - 1) * p.qkv_stride + c);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            const int j = (int)(t0 + tt) - first_of[tt];     // tokens of the sequence before this one in the step
            const float* st = state_of[tt] >= 0 ? p.conv_state + (int64_t)state_of[tt] * (TAPS - 1) * C + c : nullptr;
            float acc = 0.f;
#pragma unroll
            for (int k = 0; k < TAPS; ++k) {                 // tap k multiplies the input TAPS - 1 - k tokens back
                const int src = j - (TAPS - 1 - k);
                float x = in[tt + k];
                if (src < 0) x = st ? st[(int64_t)(TAPS - 1 + src) * C] : 0.f;
                acc = __builtin_fmaf(w[k], x, acc);
            }
            if (tt < nt) sh[tt * n + e] = acc / (1.0f + expf(-acc));
            if (carried_out && tt < nt && slot_of[tt] >= 0 && (e >= 2 * dk || h % (p.H / p.G) == 0)) {
                const int len = end_of[tt] - first_of[tt], s = j - (len - (TAPS - 1));
                float* to = carried_out + (int64_t)slot_of[tt] * (TAPS - 1) * C + c;
                if (s >= 0) to[(int64_t)s * C] = in[tt + TAPS - 1];
                if (j == 0)
                    for (int k = 0; k < TAPS - 1 - len; ++k) to[(int64_t)k * C] = 0.f;
            }
        }
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63;
    for (int i = wave; i < 2 * nt; i += 4) {                 // q, k of every token
        const float* x = sh + (i >> 1) * n + (i & 1) * dk;
        float ss = 0.f;
        for (int c = lane; c < dk; c += 64) ss += x[c] * x[c];
        ss = wave_sum(ss);
        if (lane == 0) inv[i] = 1.0f / sqrtf(ss + 1e-6f);
    }
    __syncthreads();
    const int row = 5 * dk + dv;
    float* out = p.out + (t0 * p.H + h) * (int64_t)row;
    const float scale = sqrtf((float)dk);
    auto rows_out = [&](auto piece) {                        // (a piece: one number, or four where every part of a row is a multiple of four)
        using V = decltype(piece);
        constexpr int W = sizeof(V) / sizeof(float);
        for (int i = tid; i < nt * dk / W; i += 256) {
            const int tt = i * W / dk, c = i * W - tt * dk;
            float* o = out + (int64_t)tt * p.H * row + c;
            const float* x = sh + tt * n + c;
            const float qs = inv[2 * tt] / scale, ks = inv[2 * tt + 1], b = beta[tt], d = dec[tt];
            V q = *reinterpret_cast<const V*>(x), k = *reinterpret_cast<const V*>(x + dk), bk, bdk, dd;
#pragma unroll
            for (int e = 0; e < W; ++e) {
                float *qe = reinterpret_cast<float*>(&q) + e, *ke = reinterpret_cast<float*>(&k) + e;
                *qe *= qs;
                *ke *= ks;
                reinterpret_cast<float*>(&bk)[e] = b * *ke;
                reinterpret_cast<float*>(&bdk)[e] = b * d * *ke;
                reinterpret_cast<float*>(&dd)[e] = d;
            }
            *reinterpret_cast<V*>(o) = q;
            *reinterpret_cast<V*>(o + dk) = bk;
            *reinterpret_cast<V*>(o + 2 * dk) = dd;
            *reinterpret_cast<V*>(o + 3 * dk) = k;
            *reinterpret_cast<V*>(o + 4 * dk) = bdk;
        }
        for (int i = tid; i < nt * dv / W; i += 256) {
            const int tt = i * W / dv, c = i * W - tt * dv;
            *reinterpret_cast<V*>(out + (int64_t)tt * p.H * row + 5 * dk + c) = *reinterpret_cast<const V*>(sh + tt * n + 2 * dk + c);
        }
    };
    if (vec) rows_out(f32x4{});                              // (uniform)
    else rows_out(0.f);
}

template <int TT>
void launch_gated_delta_prep_run(const GatedDeltaPrepArgs& p, int64_t num_tokens, bool act_f32, float* carried_out, hipStream_t st) {
    const dim3 grid((unsigned)nvh_cdiv(num_tokens, TT), (unsigned)p.H);
    const size_t lds = sizeof(float) * (size_t)(TT * (2 * p.dk + p.dv) + 4 * TT);
    const int vec = p.dk % 4 == 0 && p.dv % 4 == 0 && nvh_aligned16(p.out);
    auto launch = [&](auto kernel) { kernel<<<grid, 256, lds, st>>>(p, num_tokens, vec, carried_out); };
    if (act_f32) launch(p.taps == 2 ? &gated_delta_prep_run_kernel<float, TT, 2> : p.taps == 3 ? &gated_delta_prep_run_kernel<float, TT, 3> : &gated_delta_prep_run_kernel<float, TT, 4>);
    else launch(p.taps == 2 ? &gated_delta_prep_run_kernel<bf16, TT, 2> : p.taps == 3 ? &gated_delta_prep_run_kernel<bf16, TT, 3> : &gated_delta_prep_run_kernel<bf16, TT, 4>);
}

// TT tokens a workgroup share every row of W2, which a lane reads for its channel (VEC: 16 bytes at a time); the order of a logit's sum is the same
// for any TT.  Read once per token, two bytes at a time, those rows bound the launch: 1024 tokens, 16 heads of 64, rank 64, 36.7 us; four tokens a
// workgroup 13.0 us, of which the 25 MB that it writes cannot do without 5.
template <typename A, int TT, bool VEC>
__global__ __launch_bounds__(256) void delta_prep_kernel(DeltaPrepArgs p, int num_tokens) {
    extern __shared__ __attribute__((aligned(16))) float tl[];       // [TT][rank] tanh of the low-rank rows
    const int64_t t0 = (int64_t)blockIdx.x * TT;
    const int nt = (int)min((int64_t)TT, num_tokens - t0), rank = p.rank;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
        for (int r = threadIdx.x; r < rank; r += 256) tl[tt * rank + r] = tanhf(ldf((const A*)p.lowrank, (t0 + min(tt, nt - 1)) * p.l_stride + r));
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, dk = p.dk;
    for (int h = blockIdx.y * 4 + wave; h < p.H; h += 4 * gridDim.y) {      // one head per wave; grid.y covers the heads four at a time
        float inv[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            float ss = 0.f;
            for (int i = lane; i < dk; i += 64) {
                const float kv = ldf((const A*)p.k, (t0 + min(tt, nt - 1)) * p.k_stride + h * dk + i);
                ss += kv * kv;
            }
            inv[tt] = 1.0f / sqrtf(wave_sum(ss) + 1e-6f);
        }
        for (int i = lane; i < dk; i += 64) {
            const int c = h * dk + i;
            float z[TT];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) z[tt] = ldf((const A*)p.w0, c);
            const A* w2r = (const A*)p.w2 + (int64_t)c * rank;
            if constexpr (VEC) {
                for (int r = 0; r < rank; r += 8) {
                    float w[8];
                    nvh_load8(w2r, r, 8, 1, w);
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) z[tt] = __builtin_fmaf(w[e], tl[tt * rank + r + e], z[tt]);
                    }
                }
            } else {
                for (int r = 0; r < rank; ++r) {
                    const float w = ldf(w2r, r);
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt) z[tt] = __builtin_fmaf(w, tl[tt * rank + r], z[tt]);
                }
            }
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                if (tt >= nt) break;
                const int64_t t = t0 + tt;
                float* out = p.out + (t * p.H + h) * 6 * dk;
                const float kv = ldf((const A*)p.k, t * p.k_stride + c);
                const float u = kv * inv[tt];
                const float a = sigmoidf_(ldf((const A*)p.a_raw, t * p.a_stride + c) + ldf((const A*)p.a_bias, c));
                out[i] = ldf((const A*)p.r, t * p.r_stride + c);
                out[dk + i] = kv;
                out[2 * dk + i] = expf(-p.decay_scale * sigmoidf_(z[tt]));
                out[3 * dk + i] = u;
                out[4 * dk + i] = a * u;
                out[5 * dk + i] = ldf((const A*)p.v, t * p.v_stride + c);
            }
        }
    }
}

struct DeltaScanArgs {
    const float* pack;         // [T, H, 5 dk + dv]: r | k | w | u | a*u (dk each) | v (dv) per head, from a prep kernel
    float* state;              // [slots, H, dk, dv]
    const int32_t* slots;      // [B]
    const int32_t* cu_seqlens_q;    // [B+1] or null (one token per sequence)
    const int32_t* context_lens;    // [B]: tokens of the sequence including this step's (a step that holds them all starts from zero)
    float* out;                // [T, H*dv]
    int H, dk, dv;
    int skip_from;             // portions of this many tokens and more are left to the chunked form (1 << 30: none)
};

// Lanes per state column (SUBS: 16 when dk is a multiple of 16, else 4), rows i = SUBS * ii + sub held by lane `sub`; a
// workgroup of 256 lanes owns 256 / SUBS columns of one (sequence, head).  Tokens are staged TOK at a time: the loads
// of the next TOK tokens are in flight (in registers) while the current ones are walked from LDS.
// EXACT: dk == DKQ * SUBS, so the loops over a lane's rows carry no run-time bound (see attention_any.hip).
template <int DKQ, int SUBS, bool EXACT>
__global__ __launch_bounds__(256) void delta_scan_kernel(DeltaScanArgs p) {
    constexpr int COLS = 256 / SUBS;
    constexpr int CH = (5 * DKQ * SUBS + COLS + 255) / 256;  // loads per lane and token
    constexpr int TOK = (32 / CH) < 2 ? 2 : (32 / CH);
    extern __shared__ float sm[];                            // [TOK][5 dk + COLS]: r | k | w | u | au | v (this workgroup's columns)
    const int seq = blockIdx.x, head = blockIdx.y;
    const int dk = p.dk, dv = p.dv, dkq = (dk + SUBS - 1) / SUBS;      // rows i = SUBS * ii + sub >= dk (ragged dk) are held as zeros
    const int col0 = blockIdx.z * COLS, lcol = threadIdx.x / SUBS, col = col0 + lcol, sub = threadIdx.x % SUBS;
    const bool live = col < dv;
    const int lo = p.cu_seqlens_q ? p.cu_seqlens_q[seq] : seq, hi = p.cu_seqlens_q ? p.cu_seqlens_q[seq + 1] : seq + 1;
    const int slot = p.slots[seq];
    // a padded row, or left to the chunked form (uniform over the workgroup; in one test)
    if (slot < 0 || (unsigned)(hi - lo - 1) >= (unsigned)(p.skip_from - 1)) return;
    const bool fresh = p.context_lens[seq] == hi - lo;
    float* sp = p.state + (((int64_t)slot * p.H + head) * dk) * dv;
    float S[DKQ];
    // rows of a lane: DKQ consecutive ones when the sizes are exact (one 16-byte LDS read per operand and four rows), every
    // SUBS-th one otherwise
    auto row_of = [&](int ii) { return EXACT ? DKQ * sub + ii : SUBS * ii + sub; };
#pragma unroll
    for (int ii = 0; ii < DKQ; ++ii) S[ii] = (live && !fresh && (EXACT || row_of(ii) < dk)) ? sp[(int64_t)row_of(ii) * dv + col] : 0.f;
    const int rowf = 5 * dk + COLS;
    // Row of a token as this workgroup needs it: the five dk-vectors, then its COLS columns of v.  Every load is
    // unconditional (indices clamped into the row and into the sequence), so all of a stage's loads are in flight together.
    float pre[TOK][CH];
    const int prow = 5 * dk + dv;                            // a head's row of the pack
    const float* base = p.pack + (int64_t)head * prow;
    const int64_t tok_stride = (int64_t)p.H * prow;
    auto fetch = [&](int t0) {
#pragma unroll
        for (int tt = 0; tt < TOK; ++tt) {
            const int64_t tok = min(t0 + tt, hi - 1);
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int e = threadIdx.x + 256 * c;
                const int src = min(e < 5 * dk ? e : e + col0, prow - 1);
                pre[tt][c] = base[tok * tok_stride + src];
            }
        }
    };
    fetch(lo);
    for (int t0 = lo; t0 < hi; t0 += TOK) {
        const int nt = min(TOK, hi - t0);
        __syncthreads();                                     // the previous stage's readers are done
#pragma unroll
        for (int tt = 0; tt < TOK; ++tt)
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int e = threadIdx.x + 256 * c;
                if (e < rowf) sm[tt * rowf + e] = pre[tt][c];
            }
        __syncthreads();
        if (t0 + TOK < hi) fetch(t0 + TOK);
        // A token's operands are read from LDS one token ahead, so the reads' latency is off the chain S -> dot -> S.
        float cr[DKQ], ck[DKQ], cw[DKQ], cu[DKQ], ca[DKQ], cv;
        auto read_token = [&](int tt, float (&xr)[DKQ], float (&xk)[DKQ], float (&xw)[DKQ], float (&xu)[DKQ], float (&xa)[DKQ], float& xv) {
            const float* row = sm + tt * rowf;
            if constexpr (EXACT && DKQ % 4 == 0) {
#pragma unroll
                for (int c4 = 0; c4 < DKQ / 4; ++c4) {
                    const int i = DKQ * sub + 4 * c4;
                    const f32x4 vr = *reinterpret_cast<const f32x4*>(row + i), vk = *reinterpret_cast<const f32x4*>(row + dk + i),
                                vw = *reinterpret_cast<const f32x4*>(row + 2 * dk + i), vu = *reinterpret_cast<const f32x4*>(row + 3 * dk + i),
                                va = *reinterpret_cast<const f32x4*>(row + 4 * dk + i);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        xr[4 * c4 + e] = vr[e];
                        xk[4 * c4 + e] = vk[e];
                        xw[4 * c4 + e] = vw[e];
                        xu[4 * c4 + e] = vu[e];
                        xa[4 * c4 + e] = va[e];
                    }
                }
                xv = row[5 * dk + lcol];
                return;
            }
#pragma unroll
            for (int ii = 0; ii < DKQ; ++ii)
                if (EXACT || ii < dkq) {
                    const int i = row_of(ii);
                    const bool in = EXACT || i < dk;         // (a row beyond dk: all operands zero, its state stays zero)
                    xr[ii] = in ? row[i] : 0.f;
                    xk[ii] = in ? row[dk + i] : 0.f;
                    xw[ii] = in ? row[2 * dk + i] : 0.f;
                    xu[ii] = in ? row[3 * dk + i] : 0.f;
                    xa[ii] = in ? row[4 * dk + i] : 0.f;
                }
            xv = row[5 * dk + lcol];
        };
        // one token: reads S, leaves the new S and the output (the operands were read one token ahead)
        auto token = [&](int tt, const float (&xr)[DKQ], const float (&xk)[DKQ], const float (&xw)[DKQ], const float (&xu)[DKQ],
                         const float (&xa)[DKQ], float xv) {
            float dot = 0.f;
#pragma unroll
            for (int ii = 0; ii < DKQ; ++ii)
                if (EXACT || ii < dkq) dot = __builtin_fmaf(xu[ii], S[ii], dot);
            if constexpr (SUBS == 16) {
                dot = row16_sum(dot);
            } else {
                dot += NVH_DPP(dot, 0xB1);
                dot += NVH_DPP(dot, 0x4E);
            }
            float o = 0.f;
#pragma unroll
            for (int ii = 0; ii < DKQ; ++ii)
                if (EXACT || ii < dkq) {
                    const float sn = __builtin_fmaf(xw[ii], S[ii], __builtin_fmaf(xk[ii], xv, -(xa[ii] * dot)));
                    S[ii] = sn;
                    o = __builtin_fmaf(sn, xr[ii], o);
                }
            if constexpr (SUBS == 16) {
                o = row16_sum(o);
            } else {
                o += NVH_DPP(o, 0xB1);
                o += NVH_DPP(o, 0x4E);
            }
            if (live && sub == 0) p.out[(int64_t)(t0 + tt) * p.H * dv + head * dv + col] = o;
        };
        // two register sets take turns (no copies): while one token is worked on, the next one's operands arrive
        float nr[DKQ], nk[DKQ], nw[DKQ], nu[DKQ], na[DKQ], nv;
        read_token(0, cr, ck, cw, cu, ca, cv);
        int tt = 0;
        for (; tt + 1 < nt; tt += 2) {
            read_token(tt + 1, nr, nk, nw, nu, na, nv);
            token(tt, cr, ck, cw, cu, ca, cv);
            read_token(min(tt + 2, TOK - 1), cr, ck, cw, cu, ca, cv);
            token(tt + 1, nr, nk, nw, nu, na, nv);
        }
        if (tt < nt) token(tt, cr, ck, cw, cu, ca, cv);
    }
    if (live) {
#pragma unroll
        for (int ii = 0; ii < DKQ; ++ii)
            if (EXACT || row_of(ii) < dk) sp[(int64_t)row_of(ii) * dv + col] = S[ii];
    }
}

// One token per sequence (a decode step), dk = 16 DKQ: a workgroup holds 4 NC4 columns of a head's state, a lane R consecutive rows of four of them,
// so that a row's columns are read and written as they lie - the form above reads 16 bytes of a row at a time.  The rows' sums are formed in its
// order: DKQ rows one after the other, then pairs, fours, eights and the sixteen (row16_sum), the pairs in a lane and the rest through LDS, so
// every bit is the same.  Bound by the state's way from and to memory.
// us, the form above and this one: 64 sequences with 8 heads of 128 x 128 40.8 and 17.7 (3.8 TB/s both ways), 16 heads of 64 x 64 23.0 and 8.3; 16 with
// 8 heads of 128 x 128 11.7 and 5.5; one 4.5 and 3.5.
template <int DKQ, int NC4>
__global__ __launch_bounds__(256) void delta_token_kernel(DeltaScanArgs p) {
    constexpr int dk = 16 * DKQ, GROUPS = 256 / NC4, SUBS = 16 / GROUPS, R = SUBS * DKQ;      // row groups; runs of DKQ rows and rows of a lane
    static_assert(GROUPS * SUBS == 16 && GROUPS >= 4, "the sixteen runs of rows, at least four to be summed through LDS");
    __shared__ __attribute__((aligned(16))) float ops[5 * dk];        // r | k | w | u | au
    __shared__ f32x4 part[2][GROUPS][NC4];
    const int seq = blockIdx.x, head = blockIdx.y, dv = p.dv, tid = threadIdx.x;
    const int slot = p.slots[seq];
    if (slot < 0) return;                                    // a padded row (uniform)
    const bool fresh = p.context_lens[seq] == 1;
    const int c4 = tid % NC4, grp = tid / NC4, col = (blockIdx.z * NC4 + c4) * 4, row0 = grp * R;
    const bool live = col < dv;                              // (dv a multiple of 4)
    float* sp = p.state + (((int64_t)slot * p.H + head) * dk + row0) * dv + min(col, dv - 4);
    const float* pack = p.pack + ((int64_t)seq * p.H + head) * (5 * dk + dv);
    f32x4 S[R];
#pragma unroll
    for (int i = 0; i < R; ++i) S[i] = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(sp + (int64_t)i * dv);
    for (int i = tid; i < 5 * dk; i += 256) ops[i] = pack[i];
    const f32x4 v = *reinterpret_cast<const f32x4*>(pack + 5 * dk + min(col, dv - 4));
    __syncthreads();
    const float *r = ops + row0, *k = r + dk, *w = k + dk, *u = w + dk, *au = u + dk;
    // the sum over all rows of four columns, of which a lane brings its runs' sums
    auto total = [&](const f32x4 (&run)[SUBS], int which) {
        f32x4 mine = run[0];
        if constexpr (SUBS == 2) mine = run[0] + run[1];
        if constexpr (SUBS == 4) mine = (run[0] + run[1]) + (run[2] + run[3]);
        part[which][grp][c4] = mine;
        __syncthreads();
        f32x4 x[GROUPS];
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) x[g] = part[which][g][c4];
#pragma unroll
        for (int n = GROUPS / 2; n >= 1; n /= 2)
#pragma unroll
            for (int g = 0; g < n; ++g) x[g] = x[2 * g] + x[2 * g + 1];
        return x[0];
    };
    f32x4 run[SUBS];
#pragma unroll
    for (int s = 0; s < SUBS; ++s) {
        run[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DKQ; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) run[s][e] = __builtin_fmaf(u[s * DKQ + i], S[s * DKQ + i][e], run[s][e]);
    }
    const f32x4 dot = total(run, 0);
#pragma unroll
    for (int s = 0; s < SUBS; ++s) {
        run[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DKQ; ++i) {
            const int at = s * DKQ + i;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[at][e] = __builtin_fmaf(w[at], S[at][e], __builtin_fmaf(k[at], v[e], -(au[at] * dot[e])));
                run[s][e] = __builtin_fmaf(S[at][e], r[at], run[s][e]);
            }
        }
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < R; ++i) *reinterpret_cast<f32x4*>(sp + (int64_t)i * dv) = S[i];
    }
    const f32x4 o = total(run, 1);
    if (live && grp == 0) *reinterpret_cast<f32x4*>(p.out + ((int64_t)seq * p.H + head) * dv + col) = o;
}

// Whether a step of one token per sequence takes delta_token_kernel: rows of whole aligned groups of four columns.
static bool delta_token_ok(const DeltaScanArgs& p) {
    return !p.cu_seqlens_q && p.dv % 4 == 0 && nvh_aligned16(p.pack) && nvh_aligned16(p.state) && nvh_aligned16(p.out);
}

template <int DKQ>
static void launch_delta_token(const DeltaScanArgs& p, int64_t batch, hipStream_t st) {
    // 128 columns a workgroup as long as every CU gets two, else 64 (the results are the same)
    if (DKQ <= 8 && batch * p.H * nvh_cdiv(p.dv, 128) >= 512 && p.dv > 64)
        delta_token_kernel<DKQ, DKQ <= 8 ? 32 : 16><<<dim3((unsigned)batch, (unsigned)p.H, (unsigned)nvh_cdiv(p.dv, 128)), 256, 0, st>>>(p);
    else
        delta_token_kernel<DKQ, 16><<<dim3((unsigned)batch, (unsigned)p.H, (unsigned)nvh_cdiv(p.dv, 64)), 256, 0, st>>>(p);
}

// ---------------------------------------------------------------------------------------------------------------
// The chunked form, for portions of many tokens (token by token every token costs the chain S -> u^T S -> S, 0.25 - 0.33 us, whatever the chip
// has idle).  Within a chunk of 16 tokens the recurrence is linear in the chunk's first state S0.  With P_t the product of the decays of tokens
// 0 .. t, the removals d_t = u_t^T S_(t-1) satisfy
//   d_t + sum_(s<t) A_ts d_s = (u_t P_(t-1)) S0 + sum_(s<t) K_ts v_s,    A_ts = u_t . (w_(s+1) .. w_(t-1) a_s),  K_ts the same with k_s,
// a unit lower triangular system, so D = W S0 + Y and, with the outputs' own pair products, O = Q S0 + Z, and the state behind the chunk is
//   S = P_15 S0 + K'^T V - A'^T D,      K'_s = w_(s+1) .. w_15 k_s,  A' likewise.
// W, Q, Y, Z, K', A' and P need no state: one launch forms them for all chunks at once.  The second launch walks the chunks: per chunk products of
// 16 x 16 a wave on the matrix cores and one meeting of the waves.  Results differ from the token-by-token form within rounding.  What is summed over
// a chunk's pairs of tokens, the triangular inverse and P_15 S0 + K'^T V are held in double (against float64, in the 2-norm over 1024 tokens: outputs
// 4.6e-8, states 3.4e-8; token by token 8.3e-8 and 4.9e-8; with K'^T V alone in double 5.0e-8 for the states, with nothing there 7.2e-8).
// us at one sequence of 1024 tokens, token by token and in chunks (both launches): 16 heads of 64 x 64: 271, 27 + 47; 8 heads of 128 x 128: 331,
// 28 + 78.  The first launch is bound by its chain when the chip is not full (11 us at 256 tokens), and else by the double products (172 us at 8448
// records of 64 x 64); the second by the chain of a chunk, 0.74 us.
// What the first launch keeps in LDS: r | k | w | u | au, 16 rows of dk + 4 floats each, and in doubles the decays and their reciprocals (16 rows of
// dk + 2 each), which later give their place to four matrices.
__host__ __device__ constexpr int chunk_rows_floats(int dk) { return 5 * CT * (dk + 4); }
__host__ __device__ constexpr int chunk_doubles(int dk) { return 2 * CT * (dk + 2) > 4 * CT * MLD ? 2 * CT * (dk + 2) : 4 * CT * MLD; }

struct DeltaChunkArgs {
    DeltaScanArgs s;
    float* ws;                 // a record per (chunk slot, head), see chunk_record
    int batch;
};

// Floats of a record: W | Q | A'^T | K'^T (16 dk each, as the lanes of the second launch read them) | P (dk) | Y | Z | V (16 dv each, likewise).
__host__ __device__ __forceinline__ int64_t chunk_record(int dk, int dv) { return 65 * (int64_t)dk + 48 * (int64_t)dv; }
struct Tri {
    f64x4 n, t;                // X and its transpose
};

template <bool SAFE>
__device__ __forceinline__ f64x4 tri_mul_n(const f64x4& l, const f64x4& r, const f64x4& c, int q, int own) {      // l: the left matrix transposed
    if constexpr (SAFE) return mfma_f64_below<false, false>(l, r, c, q, own);
    else return mfma_f64(l, r, c);
}
template <bool SAFE>
__device__ __forceinline__ f64x4 tri_mul_t(const f64x4& l, const f64x4& r, const f64x4& c, int q, int own) {      // the transposed product
    if constexpr (SAFE) return mfma_f64_below<true, false>(l, r, c, q, own);
    else return mfma_f64(l, r, c);
}

// From a chunk's pair products A, K, Rk, Ra to what its columns are multiplied with, as left operands (that is, transposed):
//   T = (I + A)^-1 = (I - A)(I + A^2)(I + A^4)(I + A^8)   (A^16 = 0; in double, since powers may be large),
//   G = Ra T,   M = T K,   N = Rk - Ra M,      so that   W = T U',  Q = R' - G U',  Y = M V,  Z = N V.
struct ChunkFactors {
    f64x4 T, G, M, N;
};
template <bool SAFE>
__device__ __forceinline__ ChunkFactors chunk_factors(const double* mats, int q, int own) {
    const f64x4 zero = {0.0, 0.0, 0.0, 0.0};
    auto load = [&](int which, bool strict) {
        Tri x;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * q + e;
            x.n[e] = mats[(which * CT + t) * MLD + own];
            x.t[e] = mats[(which * CT + own) * MLD + t];
            if (SAFE && (strict ? own >= t : own > t)) x.n[e] = 0.0;
            if (SAFE && (strict ? t >= own : t > own)) x.t[e] = 0.0;
        }
        return x;
    };
    const Tri A = load(0, true), K = load(1, true), Rk = load(2, false), Ra = load(3, false);
    auto square = [&](const Tri& x) { return Tri{tri_mul_n<SAFE>(x.t, x.n, zero, q, own), tri_mul_t<SAFE>(x.n, x.t, zero, q, own)}; };
    auto grow = [&](const Tri& x, const f64x4& pn) { return Tri{tri_mul_n<SAFE>(x.t, pn, x.n, q, own), tri_mul_t<SAFE>(pn, x.t, x.t, q, own)}; };
    const Tri P2 = square(A), P4 = square(P2);
    const f64x4 P8 = tri_mul_n<SAFE>(P4.t, P4.n, zero, q, own);
    Tri T;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const double one = 4 * q + e == own ? 1.0 : 0.0;
        T.n[e] = one - A.n[e];
        T.t[e] = one - A.t[e];
    }
    T = grow(T, P2.n);
    T = grow(T, P4.n);
    T = grow(T, P8);
    ChunkFactors f;
    f.T = T.t;
    f.G = tri_mul_t<SAFE>(T.n, Ra.t, zero, q, own);
    const f64x4 Mn = tri_mul_n<SAFE>(T.t, K.n, zero, q, own);
    f.M = tri_mul_t<SAFE>(K.n, T.t, zero, q, own);
    f.N = Rk.t - tri_mul_t<SAFE>(Mn, Ra.t, zero, q, own);
    return f;
}

// CPL: key channels a lane of the pair products holds (dk = 16 CPL).
template <int CPL>
__global__ __launch_bounds__(256, CPL <= 4 ? 4 : 2) void delta_chunk_prep_kernel(DeltaChunkArgs a) {
    extern __shared__ __attribute__((aligned(16))) float sm[];       // (chunk_rows_floats, chunk_doubles)
    const DeltaScanArgs& p = a.s;
    constexpr int dk = 16 * CPL, LD = dk + 4, DLD = dk + 2;
    const int dv = p.dv, head = blockIdx.x, cslot = blockIdx.y, tid = threadIdx.x;
    int first = 0, end = a.batch;                            // the last sequence whose chunk slots begin at or before this one
    while (end - first > 1) {
        const int mid = (first + end) >> 1;
        if (chunk_base(p.cu_seqlens_q[mid], mid) <= cslot) first = mid;
        else end = mid;
    }
    const int lo = p.cu_seqlens_q[first], hi = p.cu_seqlens_q[first + 1];
    const int t0 = lo + CT * (cslot - chunk_base(lo, first)), nt = min(CT, hi - t0);
    if (hi - lo < p.skip_from || nt <= 0 || p.slots[first] < 0) return;      // (uniform)
    const int64_t prow = 5 * dk + dv, tok_stride = (int64_t)p.H * prow;
    const float* base = p.pack + (int64_t)t0 * tok_stride + (int64_t)head * prow;
    float* rec = a.ws + ((int64_t)cslot * p.H + head) * chunk_record(dk, dv);
    auto row = [&](int which, int t) { return sm + (which * CT + t) * LD; };
    double *mats = reinterpret_cast<double*>(sm + chunk_rows_floats(dk)), *cums = mats, *rcums = mats + CT * DLD;
    // Everything the workgroup reads is requested at once, on every path (a load under a condition would be waited for on its own).  Tokens beyond
    // the portion's end change nothing: decay 1, everything else 0.
    constexpr int PIECES = CT * 5 * dk / 4, ROUNDS = (PIECES + 255) / 256;
    f32x4 piece[ROUNDS];
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int e = min(tid + 256 * i, PIECES - 1), t = e / (5 * dk / 4), c4 = (e - t * (5 * dk / 4)) * 4;
        piece[i] = *reinterpret_cast<const f32x4*>(base + min(t, nt - 1) * tok_stride + c4);
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, q = lane >> 4, vtiles = dv >> 4;
    constexpr int VAHEAD = 2;                                // tiles of v that a wave requests up front
    f32x4 vt[VAHEAD];
    auto load_v = [&](int tile) {                            // (this lane's four tokens of a column)
        const float* vp = base + 5 * dk + 16 * min(tile, vtiles - 1) + col;
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = vp[min(4 * q + e, nt - 1) * tok_stride];
        return x;
    };
#pragma unroll
    for (int i = 0; i < VAHEAD; ++i) vt[i] = load_v(wave + 4 * i);
    bool odd = false;                                        // does r, k, w, u or au hold a value that is not finite
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int e = tid + 256 * i, t = e / (5 * dk / 4), c4 = (e - t * (5 * dk / 4)) * 4, which = c4 / dk;
        const float fill = which == 2 ? 1.f : 0.f;
        if (PIECES % 256 == 0 || e < PIECES) *reinterpret_cast<f32x4*>(row(which, t) + (c4 - which * dk)) = t < nt ? piece[i] : f32x4{fill, fill, fill, fill};
#pragma unroll
        for (int c = 0; c < 4; ++c) odd |= !(fabsf(piece[i][c]) <= 3.402823466e+38f);
    }
    odd = __syncthreads_or(odd);
    const int s = tid >> 4, g = tid & 15, ch = g * CPL, own = chunk_tok(col);
    const f64x4 zero = {0.0, 0.0, 0.0, 0.0};
    double cum[CPL], before[CPL];                            // the decay up to token s, with and without its own
    bool far = odd;
#pragma unroll
    for (int i = 0; i < CPL; ++i) before[i] = 1.0;
#pragma unroll 4
    for (int t = 0; t < CT - 1; ++t) {
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            const double w = row(2, t)[ch + i];
            before[i] *= t < s ? w : 1.0;
        }
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
        cum[i] = before[i] * row(2, s)[ch + i];
        far |= !(cum[i] >= 1e-80 && cum[i] <= 1e80);
        cums[s * DLD + ch + i] = cum[i];
        rcums[s * DLD + ch + i] = 1.0 / cum[i];
    }
    far = __syncthreads_or(far);
    float ap[CPL], kp[CPL];                                  // a and k of token s, decayed to the chunk's end
    f64x4 pairs = zero;
    if (!far) {
        // A, K, Rk, Ra = U' (a / cum)^T, U' (k / cum)^T, R' (k / cum)^T, R' (a / cum)^T, a matrix a wave; a lane's channels of a step are those
        // of quarter q.  All in double, where the quotients neither over- nor underflow within the limits checked above.
        const bool r_left = wave >= 2, k_right = wave == 1 || wave == 2;
        const float *lrow = row(r_left ? 0 : 3, own) + q * (dk / 4), *rrow = row(k_right ? 1 : 4, own) + q * (dk / 4);
        const double *lcum = cums + (r_left ? own : max(own - 1, 0)) * DLD + q * (dk / 4), *rcum = rcums + own * DLD + q * (dk / 4);
        const bool first_u = !r_left && own == 0;
        f64x4 other = zero;
#pragma unroll
        for (int j = 0; j < dk / 4; j += 2) {
            const double l0 = lrow[j] * (first_u ? 1.0 : lcum[j]), l1 = lrow[j + 1] * (first_u ? 1.0 : lcum[j + 1]);
            pairs = __builtin_amdgcn_mfma_f64_16x16x4f64(l0, rrow[j] * rcum[j], pairs, 0, 0, 0);
            other = __builtin_amdgcn_mfma_f64_16x16x4f64(l1, rrow[j + 1] * rcum[j + 1], other, 0, 0, 0);
        }
        pairs += other;
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            const double rest = cums[(CT - 1) * DLD + ch + i] * rcums[s * DLD + ch + i];
            ap[i] = (float)(row(4, s)[ch + i] * rest);
            kp[i] = (float)(row(1, s)[ch + i] * rest);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * q + e;
            mats[(wave * CT + t) * MLD + own] = (r_left ? own <= t : own < t) ? pairs[e] : 0.0;
        }
    } else {                                                 // 16 lanes share token s, each with CPL channels, and walk t = 0 .. 15
        double xa[CPL], xk[CPL];
#pragma unroll
        for (int i = 0; i < CPL; ++i) xa[i] = xk[i] = 0.0;
#pragma unroll 1
        for (int t = 0; t < CT; ++t) {
            double dA = 0.0, dK = 0.0, dRk = 0.0, dRa = 0.0;
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const double u = row(3, t)[ch + i], w = row(2, t)[ch + i], r = row(0, t)[ch + i];
                dA = __builtin_fma(u, xa[i], dA);
                dK = __builtin_fma(u, xk[i], dK);
                xa[i] = t == s ? row(4, t)[ch + i] : xa[i] * w;
                xk[i] = t == s ? row(1, t)[ch + i] : xk[i] * w;
                dRk = __builtin_fma(r, xk[i], dRk);
                dRa = __builtin_fma(r, xa[i], dRa);
            }
            const double sum = row16_sum4(dA, dK, dRk, dRa, g);
            if (g < 4) mats[(g * CT + t) * MLD + s] = sum;
        }
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            ap[i] = (float)xa[i];
            kp[i] = (float)xk[i];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i) {                          // A', K', U', R' in place
        row(4, s)[ch + i] = ap[i];
        row(1, s)[ch + i] = kp[i];
        row(3, s)[ch + i] = (float)(row(3, s)[ch + i] * before[i]);
        row(0, s)[ch + i] = (float)(row(0, s)[ch + i] * cum[i]);
        if (s == CT - 1) rec[64 * dk + ch + i] = (float)cum[i];
    }
    __syncthreads();
    ChunkFactors f;                                          // computed by one wave, not always on the same SIMD
    const bool elected = wave == (int)((blockIdx.x / 8 + blockIdx.y) & 3);
    if (elected) {
        f = odd ? chunk_factors<true>(mats, q, own) : chunk_factors<false>(mats, q, own);
        f64x4* out = reinterpret_cast<f64x4*>(mats) + lane;
        out[0] = f.T;
        out[64] = f.G;
        out[128] = f.M;
        out[192] = f.N;
    }
    __syncthreads();
    {
        const f64x4* in = reinterpret_cast<const f64x4*>(mats) + lane;
        f.T = in[0];
        f.G = in[64];
        f.M = in[128];
        f.N = in[192];
    }
#pragma unroll
    for (int i = 0; i < (CPL + 3) / 4; ++i) {                // 16 key channels a wave: W and Q with the channels as rows, as the second launch reads them
        const int tile = wave + 4 * i;
        if (CPL % 4 && tile >= CPL) break;
        const int c0 = 16 * tile;
        f64x4 u, Q;
        const f32x4 rp = *reinterpret_cast<const f32x4*>(row(0, own) + c0 + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            u[e] = row(3, 4 * q + e)[c0 + own];
            Q[e] = rp[e];
        }
        f64x4 W;
        if (odd) {
            W = mfma_f64_below<true, true>(u, f.T, zero, q, own);
            Q -= mfma_f64_below<true, true>(u, f.G, zero, q, own);
        } else {
            W = mfma_f64(u, f.T, zero);
            Q -= mfma_f64(u, f.G, zero);
        }
        float* out = rec + (tile * 64 + q * 16 + own) * 4;
        *reinterpret_cast<f32x4*>(out) = f32x4{(float)W[0], (float)W[1], (float)W[2], (float)W[3]};
        *reinterpret_cast<f32x4*>(out + 16 * dk) = f32x4{(float)Q[0], (float)Q[1], (float)Q[2], (float)Q[3]};
        f32x4 A, K;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            A[e] = row(4, 4 * q + e)[c0 + col];
            K[e] = row(1, 4 * q + e)[c0 + own];              // (for a product in double, whose rows lie otherwise)
        }
        float* at = rec + 32 * dk + (tile * 64 + lane) * 4;
        *reinterpret_cast<f32x4*>(at) = A;
        *reinterpret_cast<f32x4*>(at + 16 * dk) = K;
    }
    auto values = [&](int tile, f32x4 v) {                   // 16 columns of v: Y and Z
        f64x4 x;
        bool vodd = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (4 * q + e >= nt) v[e] = 0.f;
            vodd |= !(fabsf(v[e]) <= 3.402823466e+38f);
            x[e] = v[e];
        }
        f64x4 Y, Z;
        if (odd || __any(vodd)) {
            Y = mfma_f64_below<false, true>(f.M, x, zero, q, own);
            Z = mfma_f64_below<false, true>(f.N, x, zero, q, own);
        } else {
            Y = mfma_f64(f.M, x, zero);
            Z = mfma_f64(f.N, x, zero);
        }
        float* out = rec + 65 * dk + (tile * 64 + lane) * 4;
        *reinterpret_cast<f32x4*>(out) = f32x4{(float)Y[0], (float)Y[1], (float)Y[2], (float)Y[3]};
        *reinterpret_cast<f32x4*>(out + 16 * dv) = f32x4{(float)Z[0], (float)Z[1], (float)Z[2], (float)Z[3]};
        *reinterpret_cast<f32x4*>(out + 32 * dv) = v;
    };
#pragma unroll
    for (int i = 0; i < VAHEAD; ++i)
        if (wave + 4 * i < vtiles) values(wave + 4 * i, vt[i]);
    for (int tile = wave + 4 * VAHEAD; tile < vtiles; tile += 4) values(tile, load_v(tile));
}

// NW waves of 16 TPW key channels each hold 16 columns of a head's state, in the layout in which a product leaves its result (row 4 q + e of lane
// (q, column) in element e) - which is also the layout in which it takes its right operand, so a state never moves between lanes.  What bounds the
// launch is the chain of a chunk in these waves: D's product, the meeting, A's product, the new state.  So as much as can be is done beside them: NW
// helpers form K'^T V in double a chunk ahead, and one wave more sums the waves' parts of
// the outputs, a chunk behind, and writes them; it loads nothing, since a load's turn to be waited for lies behind the stores of the chunk before.
// us of both launches, eight waves (four for 64 channels) with all of it in them and so: 1024 tokens of 16 heads of 64 x 64 73.6 and 66.0, 1000 of 8 heads of
// 128 x 128 105 and 97, of 4 heads 97 and 89; errors against float64 5.4e-8 and 5.4e-8, 5.7e-8 and 5.6e-8.  At 128 channels eight parts in place of the four
// sums of two: 114.
typedef double f64x2 __attribute__((ext_vector_type(2)));
template <int NW, int TPW>
struct ScanMeet {                                            // by chunk parity; a lane's own place
    f32x4 d[2][NW][64], o[2][NW][64], z[2][64];
    f64x2 kv[2][NW * TPW][2][64];
};
template <int NW, int TPW>
__global__ __launch_bounds__(64 * (2 * NW + 1)) void delta_chunk_scan_kernel(DeltaChunkArgs a) {
    constexpr int dk = 16 * NW * TPW;
    __shared__ ScanMeet<NW, TPW> meet;
    const DeltaScanArgs& p = a.s;
    const int seq = blockIdx.x, head = blockIdx.y, dv = p.dv, cb = blockIdx.z;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63, col = lane & 15, q = lane >> 4;
    const int lo = p.cu_seqlens_q[seq], hi = p.cu_seqlens_q[seq + 1], slot = p.slots[seq];
    if (slot < 0 || hi <= lo || hi - lo < p.skip_from) return;       // (uniform)
    const int64_t record = chunk_record(dk, dv), step = (int64_t)p.H * record;
    const float* rec = a.ws + ((int64_t)chunk_base(lo, seq) * p.H + head) * record;
    const int chunks = (hi - lo + CT - 1) / CT;
    // Every wave comes to chunks + 1 barriers: one per chunk, and one behind the last.
    if (wave == 2 * NW) {                                    // the outputs: the parts of chunk j are written before the barrier of chunk j + 1
        float* out = p.out + (int64_t)lo * p.H * dv + head * dv + 16 * cb + col;
        __syncthreads();
        for (int j = 0; j < chunks; ++j) {
            __syncthreads();
            f32x4 res = meet.o[j & 1][0][lane];
#pragma unroll
            for (int w = 1; w < NW; ++w) res += meet.o[j & 1][w][lane];
            res += meet.z[j & 1][lane];
            const int t = CT * j + 4 * q;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (lo + t + e < hi) out[(int64_t)(t + e) * p.H * dv] = res[e];
        }
        return;
    }
    constexpr int AHEAD = TPW == 1 ? 4 : 3;                  // records in flight
    // body(j, x): chunk j with its operands; fetch(record, x) requests a chunk's
    auto walk = [&](auto& x, auto fetch, auto body) {
        auto request = [&](int j, auto& to) { fetch(rec + (int64_t)min(j, chunks - 1) * step, to); };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) request(i, x[i]);
        int j = 0;
        for (; j + AHEAD <= chunks; j += AHEAD) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                body(j + i, x[i]);
                request(j + i + AHEAD, x[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int i = 0; i < AHEAD - 1; ++i)
            if (j + i < chunks) body(j + i, x[i]);
        __syncthreads();                                     // (the last chunk's outputs)
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    if (wave >= NW) {
        const int w = wave - NW;
        struct Operands {
            f32x4 K[TPW], V, Z;
        } x[AHEAD];
        walk(
            x,
            [&](const float* r, Operands& to) {
#pragma unroll
                for (int i = 0; i < TPW; ++i) to.K[i] = *reinterpret_cast<const f32x4*>(r + 48 * dk + (TPW * w + i) * 256 + 4 * lane);
                to.Z = *reinterpret_cast<const f32x4*>(r + 65 * dk + 16 * dv + cb * 256 + 4 * lane);
                to.V = *reinterpret_cast<const f32x4*>(r + 65 * dk + 32 * dv + cb * 256 + 4 * lane);
            },
            [&](int j, const Operands& y) {
                f64x4 kv[TPW];
#pragma unroll
                for (int i = 0; i < TPW; ++i) kv[i] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < TPW; ++i) kv[i] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)y.K[i][e], (double)y.V[e], kv[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < TPW; ++i) {
                    meet.kv[j & 1][TPW * w + i][0][lane] = f64x2{kv[i][0], kv[i][1]};
                    meet.kv[j & 1][TPW * w + i][1][lane] = f64x2{kv[i][2], kv[i][3]};
                }
                __syncthreads();                             // (of the other parity: the state's waves have read it before they came to this barrier)
                if (w == 0) meet.z[j & 1][lane] = y.Z;
            });
        return;
    }
    __builtin_amdgcn_s_setprio(3);                           // (ahead of the helpers at the matrix pipe)
    const bool fresh = p.context_lens[seq] == hi - lo;
    float* sp = p.state + (((int64_t)slot * p.H + head) * dk + 16 * TPW * wave + 4 * q) * dv + 16 * cb + col;
    f32x4 S[TPW];
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
        S[i] = zero;
        if (!fresh) {
#pragma unroll
            for (int e = 0; e < 4; ++e) S[i][e] = sp[(int64_t)(16 * i + e) * dv];
        }
    }
    struct Operands {
        f32x4 W[TPW], Q[TPW], A[TPW], P[TPW], Y;
    } x[AHEAD];
    walk(
        x,
        [&](const float* r, Operands& to) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                const float* m = r + (TPW * wave + i) * 256 + 4 * lane;
                to.W[i] = *reinterpret_cast<const f32x4*>(m);
                to.Q[i] = *reinterpret_cast<const f32x4*>(m + 16 * dk);
                to.A[i] = *reinterpret_cast<const f32x4*>(m + 32 * dk);
                to.P[i] = *reinterpret_cast<const f32x4*>(r + 64 * dk + 16 * (TPW * wave + i) + 4 * q);
            }
            to.Y = *reinterpret_cast<const f32x4*>(r + 65 * dk + cb * 256 + 4 * lane);
        },
        [&](int j, const Operands& y) {
            f32x4 d[TPW], o[TPW], ad[TPW];
#pragma unroll
            for (int i = 0; i < TPW; ++i) d[i] = o[i] = ad[i] = zero;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TPW; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(y.W[i][e], S[i][e], d[i], 0, 0, 0);
            if constexpr (TPW == 2) d[0] += d[1];             // (two short chains and their sum: a chain over both tiles rounds more)
            meet.d[j & 1][wave][lane] = d[0];
            __syncthreads();                                 // (the buffers of the other parity: every wave has left them before it came here)
            f32x4 part[NW];
            f64x4 kv[TPW];
#pragma unroll
            for (int w = 0; w < NW; ++w) part[w] = meet.d[j & 1][w][lane];
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                const f64x2 a01 = meet.kv[j & 1][TPW * wave + i][0][lane], a23 = meet.kv[j & 1][TPW * wave + i][1][lane];
                kv[i] = f64x4{a01[0], a01[1], a23[0], a23[1]};
            }
            __builtin_amdgcn_sched_barrier(0);
            // (while the parts come)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TPW; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(y.Q[i][e], S[i][e], o[i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            f32x4 sum = y.Y;
#pragma unroll
            for (int w = 0; w < NW; ++w) sum += part[w];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TPW; ++i) ad[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(y.A[i][e], sum[e], ad[i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (TPW == 2) o[0] += o[1];
            meet.o[j & 1][wave][lane] = o[0];
            // (with the decayed state on it in double too, a state is rounded once a chunk: 3.4e-8 off instead of 5.0e-8)
#pragma unroll
            for (int i = 0; i < TPW; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) kv[i][e] = __builtin_fma((double)y.P[i][e], (double)S[i][e], kv[i][e]);
#pragma unroll
            for (int i = 0; i < TPW; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) S[i][e] = (float)(kv[i][e] - ad[i][e]);
        });
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sp[(int64_t)(16 * i + e) * dv] = S[i][e];
}

template <typename A>
__global__ __launch_bounds__(256) void delta_post_kernel(const float* __restrict__ o, const A* __restrict__ norm_w, const A* __restrict__ gate,
                                                         int64_t gate_stride, A* __restrict__ y, int64_t y_stride, int64_t rows, int H, int dv, float eps) {
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);     // (token, head) per wave
    if (item >= rows * H) return;
    const int64_t t = item / H;
    const int h = (int)(item - t * H), lane = threadIdx.x & 63;
    const float* orow = o + (t * H + h) * dv;
    float ss = 0.f;
    for (int i = lane; i < dv; i += 64) ss += orow[i] * orow[i];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)dv + eps);
    for (int i = lane; i < dv; i += 64) {
        const int c = h * dv + i;
        const float g = gate ? sigmoidf_(ldf(gate, t * gate_stride + c)) : 1.0f;
        y[t * y_stride + c] = (A)(orow[i] * inv * ldf(norm_w, c) * g);
    }
}

}  // namespace

extern "C" int32_t nvh_delta_prep(const void* r, int64_t r_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                  const void* a_raw, int64_t a_stride, const void* lowrank, int64_t lowrank_stride,
                                  const void* w2, const void* w0, const void* a_bias, float* out, int64_t num_tokens, int64_t heads, int64_t dk,
                                  int64_t rank, float decay_scale, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(r && k && v && a_raw && lowrank && w2 && w0 && a_bias && out, NVH_EINVAL, "nvh_delta_prep: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && heads > 0 && dk > 0 && rank > 0 && rank <= 8192, NVH_EINVAL, "nvh_delta_prep: bad sizes");
    if (num_tokens == 0) return NVH_OK;
    DeltaPrepArgs p{r, k, v, r_stride, k_stride, v_stride, a_raw, a_stride, lowrank, lowrank_stride, w2, w0, a_bias, out, (int)heads, (int)dk, (int)rank, decay_scale};
    hipStream_t st = (hipStream_t)stream;
    // several tokens a workgroup where that still leaves every CU some (and the rows of W2 can be read in whole pieces)
    constexpr int TT = 4;
    const size_t lds = sizeof(float) * (size_t)rank;
    const unsigned hblocks = (unsigned)nvh_cdiv(heads, 4);
    const bool tiled = nvh_cdiv(num_tokens, TT) * hblocks >= 512 && rank % 8 == 0 && rank <= 1024 && nvh_aligned16(w2);
    const dim3 grid((unsigned)(tiled ? nvh_cdiv(num_tokens, TT) : num_tokens), hblocks);
    if (tiled) {
        if (act_f32) delta_prep_kernel<float, TT, true><<<grid, 256, lds * TT, st>>>(p, (int)num_tokens);
        else delta_prep_kernel<bf16, TT, true><<<grid, 256, lds * TT, st>>>(p, (int)num_tokens);
    } else {
        if (act_f32) delta_prep_kernel<float, 1, false><<<grid, 256, lds, st>>>(p, (int)num_tokens);
        else delta_prep_kernel<bf16, 1, false><<<grid, 256, lds, st>>>(p, (int)num_tokens);
    }
    NVH_CHECK_LAUNCH("nvh_delta_prep");
    return NVH_OK;
}

template <int DKQ, int SUBS, bool EXACT>
static void launch_delta_scan_as(const DeltaScanArgs& p, int64_t batch, hipStream_t st) {
    constexpr int COLS = 256 / SUBS;
    constexpr int CH = (5 * DKQ * SUBS + COLS + 255) / 256;
    constexpr int TOK = (32 / CH) < 2 ? 2 : (32 / CH);
    const dim3 grid((unsigned)batch, (unsigned)p.H, (unsigned)nvh_cdiv(p.dv, COLS));
    const size_t lds = sizeof(float) * (size_t)TOK * (5 * p.dk + COLS);
    delta_scan_kernel<DKQ, SUBS, EXACT><<<grid, 256, lds, st>>>(p);
}

static int32_t launch_delta_scan(const DeltaScanArgs& p, int64_t batch, hipStream_t st) {
    // (the choice depends on dk alone, so a sequence sees one summation order whatever the batch or the cut)
    if (delta_token_ok(p)) {                                 // (the bits of the form below)
        switch (p.dk) {
            case 64: launch_delta_token<4>(p, batch, st); NVH_CHECK_LAUNCH("nvh_delta_scan"); return NVH_OK;
            case 128: launch_delta_token<8>(p, batch, st); NVH_CHECK_LAUNCH("nvh_delta_scan"); return NVH_OK;
            case 256: launch_delta_token<16>(p, batch, st); NVH_CHECK_LAUNCH("nvh_delta_scan"); return NVH_OK;
        }
    }
    if (p.dk % 16 == 0) {
        switch (p.dk / 16) {
            case 1: launch_delta_scan_as<1, 16, true>(p, batch, st); break;
            case 2: launch_delta_scan_as<2, 16, true>(p, batch, st); break;
            case 3: launch_delta_scan_as<3, 16, true>(p, batch, st); break;
            case 4: launch_delta_scan_as<4, 16, true>(p, batch, st); break;
            case 6: launch_delta_scan_as<6, 16, true>(p, batch, st); break;
            case 8: launch_delta_scan_as<8, 16, true>(p, batch, st); break;
            case 16: launch_delta_scan_as<16, 16, true>(p, batch, st); break;
            default:
                if (p.dk / 16 <= 8) launch_delta_scan_as<8, 16, false>(p, batch, st);
                else launch_delta_scan_as<16, 16, false>(p, batch, st);
        }
    } else {
        const int dkq = (p.dk + 3) / 4;
        if (dkq <= 8) launch_delta_scan_as<8, 4, false>(p, batch, st);
        else if (dkq <= 16) launch_delta_scan_as<16, 4, false>(p, batch, st);
        else if (dkq <= 32) launch_delta_scan_as<32, 4, false>(p, batch, st);
        else launch_delta_scan_as<64, 4, false>(p, batch, st);
    }
    NVH_CHECK_LAUNCH("nvh_delta_scan");
    return NVH_OK;
}

static int32_t gated_delta_prep(const void* qkv, int64_t qkv_stride, const void* b, int64_t b_stride, const void* a, int64_t a_stride,
                                const void* conv_w, const void* dt_bias, const void* a_log, const float* conv_state, float* carried_out, const int32_t* slots,
                                const int32_t* cu_seqlens_q, const int32_t* context_lens, float* out, int64_t batch, int64_t num_tokens,
                                int64_t taps, int64_t heads, int64_t qk_heads, int64_t dk, int64_t dv, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(qkv && b && a && conv_w && dt_bias && a_log && slots && context_lens && out, NVH_EINVAL, "nvh_gated_delta_prep: null pointer");
    NVH_REQUIRE(batch >= 0 && num_tokens >= 0 && taps >= 1 && heads > 0 && qk_heads > 0 && heads % qk_heads == 0 && dk > 0 && dv > 0, NVH_EINVAL,
                "nvh_gated_delta_prep: bad sizes");
    NVH_REQUIRE(taps == 1 || conv_state, NVH_EINVAL, "nvh_gated_delta_prep: null state");
    NVH_REQUIRE(cu_seqlens_q || num_tokens == batch, NVH_EINVAL, "nvh_gated_delta_prep: one token per sequence without cu_seqlens_q");
    const int64_t channels = 2 * qk_heads * dk + heads * dv;
    NVH_REQUIRE(qkv_stride >= channels, NVH_EINVAL, "nvh_gated_delta_prep: projection row too short");
    const size_t lds = sizeof(float) * (size_t)(2 * dk + dv + 2);
    NVH_REQUIRE(lds <= 64 * 1024 && heads <= 65535, NVH_ENOSYS, "nvh_gated_delta_prep: head sizes %ld + %ld above the kernel's limit", (long)dk, (long)dv);
    if (num_tokens == 0 || batch == 0) return NVH_OK;
    GatedDeltaPrepArgs p{qkv, qkv_stride, b, a, b_stride, a_stride, conv_w, dt_bias, a_log, conv_state, slots, cu_seqlens_q, context_lens, out,
                         (int)batch, (int)taps, (int)heads, (int)qk_heads, (int)dk, (int)dv};
    hipStream_t st = (hipStream_t)stream;
    // Tokens a workgroup: four, or two where four leave the chip fewer than four workgroups a CU; below two and a half a CU (long rows of a sequence's tokens, which
    // share their inputs: two) one token each, as ever.  us, one and two, 64 tokens of 16 heads of 64 x 64: single tokens 5.8 and 6.3, of a prompt 5.2 and 5.4; 100
    // of a prompt 6.7 and 6.1; 128 of 8 heads of 128 x 128 6.7 and 6.2.
    const bool run = taps >= 2 && taps <= 4 && (2 * dk + dv + 4) * 4 * (int64_t)sizeof(float) <= 32 * 1024;
    if (run && num_tokens * heads >= 4096) launch_gated_delta_prep_run<4>(p, num_tokens, act_f32, carried_out, st);
    else if (run && num_tokens * heads >= (2 * dk + dv >= 256 && batch < num_tokens ? 1024 : 1280)) launch_gated_delta_prep_run<2>(p, num_tokens, act_f32, carried_out, st);
    else {
        const dim3 grid((unsigned)num_tokens, (unsigned)heads);
        if (act_f32) gated_delta_prep_kernel<float><<<grid, 256, lds, st>>>(p);
        else gated_delta_prep_kernel<bf16><<<grid, 256, lds, st>>>(p);
        if (carried_out) {
            NVH_CHECK_LAUNCH("nvh_gated_delta_prep");
            return nvh_conv_state_update(qkv, qkv_stride, carried_out, slots, cu_seqlens_q, context_lens, batch, taps, channels, act_f32, stream);
        }
    }
    NVH_CHECK_LAUNCH("nvh_gated_delta_prep");
    return NVH_OK;
}

extern "C" int32_t nvh_gated_delta_prep(const void* qkv, int64_t qkv_stride, const void* b, int64_t b_stride, const void* a, int64_t a_stride,
                                        const void* conv_w, const void* dt_bias, const void* a_log, const float* conv_state, const int32_t* slots,
                                        const int32_t* cu_seqlens_q, const int32_t* context_lens, float* out, int64_t batch, int64_t num_tokens,
                                        int64_t taps, int64_t heads, int64_t qk_heads, int64_t dk, int64_t dv, int32_t act_f32, nvh_stream_t stream) {
    return gated_delta_prep(qkv, qkv_stride, b, b_stride, a, a_stride, conv_w, dt_bias, a_log, conv_state, nullptr, slots, cu_seqlens_q, context_lens, out, batch,
                            num_tokens, taps, heads, qk_heads, dk, dv, act_f32, stream);
}

extern "C" int32_t nvh_gated_delta_prep_starting(const void* qkv, int64_t qkv_stride, const void* b, int64_t b_stride, const void* a, int64_t a_stride,
                                                 const void* conv_w, const void* dt_bias, const void* a_log, float* conv_state, const int32_t* slots,
                                                 const int32_t* cu_seqlens_q, const int32_t* context_lens, float* out, int64_t batch, int64_t num_tokens,
                                                 int64_t taps, int64_t heads, int64_t qk_heads, int64_t dk, int64_t dv, int32_t act_f32, nvh_stream_t stream) {
    return gated_delta_prep(qkv, qkv_stride, b, b_stride, a, a_stride, conv_w, dt_bias, a_log, conv_state, taps > 1 ? conv_state : nullptr, slots, cu_seqlens_q,
                            context_lens, out, batch, num_tokens, taps, heads, qk_heads, dk, dv, act_f32, stream);
}

extern "C" int32_t nvh_delta_scan(const float* pack, float* state, const int32_t* slots, const int32_t* cu_seqlens_q,
                                  const int32_t* context_lens, float* out, int64_t batch, int64_t heads, int64_t dk, int64_t dv, nvh_stream_t stream) {
    NVH_REQUIRE(pack && state && slots && context_lens && out, NVH_EINVAL, "nvh_delta_scan: null pointer");
    NVH_REQUIRE(batch >= 0 && heads > 0 && dk > 0 && dv > 0, NVH_EINVAL, "nvh_delta_scan: bad sizes");
    NVH_REQUIRE(dk <= 256, NVH_ENOSYS, "nvh_delta_scan: key size %ld above 256", (long)dk);
    if (batch == 0) return NVH_OK;
    DeltaScanArgs p{pack, state, slots, cu_seqlens_q, context_lens, out, (int)heads, (int)dk, (int)dv, 1 << 30};
    return launch_delta_scan(p, batch, (hipStream_t)stream);
}

// Head sizes that the chunked form is built for: whole 16-wide tiles, at most eight waves of key channels.
static bool delta_chunkable(int64_t dk, int64_t dv) {
    return dv % 16 == 0 && dv <= 16 * 65535 && (dk == 16 || dk == 32 || dk == 48 || dk == 64 || dk == 96 || dk == 128);
}

extern "C" int64_t nvh_delta_chunk_workspace_bytes(int64_t num_tokens, int64_t batch, int64_t heads, int64_t dk, int64_t dv) {
    if (!delta_chunkable(dk, dv) || num_tokens < 0 || batch < 0 || heads <= 0 || heads > 65535 || num_tokens / CT + batch > 65535) return 0;
    return (num_tokens / CT + batch) * heads * chunk_record((int)dk, (int)dv) * (int64_t)sizeof(float);
}

template <int CPL>
static void launch_delta_chunks(const DeltaChunkArgs& a, int64_t slots, int64_t batch, hipStream_t st) {
    const size_t lds = sizeof(float) * (size_t)chunk_rows_floats(16 * CPL) + sizeof(double) * (size_t)chunk_doubles(16 * CPL);
    if (lds > 60 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_prep_kernel<CPL>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    // (heads fastest: with a multiple of eight heads a head's records are written and read by the same XCD, through its L2)
    delta_chunk_prep_kernel<CPL><<<dim3((unsigned)a.s.H, (unsigned)slots), 256, lds, st>>>(a);
    // (at most four waves of key channels, one a SIMD: more of them would share a SIMD's matrix pipe and have more parts to exchange)
    constexpr int TPW = CPL > 4 ? 2 : 1, NW = CPL / TPW;
    delta_chunk_scan_kernel<NW, TPW><<<dim3((unsigned)batch, (unsigned)a.s.H, (unsigned)(a.s.dv / 16)), 64 * (2 * NW + 1), 0, st>>>(a);
}

extern "C" int32_t nvh_delta_scan_chunked(const float* pack, float* state, const int32_t* slots, const int32_t* cu_seqlens_q,
                                          const int32_t* context_lens, float* out, int64_t batch, int64_t num_tokens, int64_t heads, int64_t dk,
                                          int64_t dv, int64_t min_tokens, float* workspace, nvh_stream_t stream) {
    NVH_REQUIRE(pack && state && slots && cu_seqlens_q && context_lens && out && workspace, NVH_EINVAL, "nvh_delta_scan_chunked: null pointer");
    NVH_REQUIRE(batch >= 0 && num_tokens >= 0 && num_tokens < (1 << 30) && heads > 0 && heads <= 65535 && num_tokens / CT + batch <= 65535 && min_tokens >= 1 && min_tokens < (1 << 30), NVH_EINVAL,
                "nvh_delta_scan_chunked: bad sizes");
    NVH_REQUIRE(delta_chunkable(dk, dv), NVH_ENOSYS, "nvh_delta_scan_chunked: head size %ld x %ld", (long)dk, (long)dv);
    NVH_REQUIRE(nvh_aligned16(pack) && nvh_aligned16(workspace), NVH_EINVAL, "nvh_delta_scan_chunked: 16-byte alignment required");
    if (batch == 0 || num_tokens == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    const DeltaScanArgs p{pack, state, slots, cu_seqlens_q, context_lens, out, (int)heads, (int)dk, (int)dv, (int)min_tokens};
    const DeltaChunkArgs a{p, workspace, (int)batch};
    const int64_t cslots = num_tokens / CT + batch;
    switch (dk / 16) {
        case 1: launch_delta_chunks<1>(a, cslots, batch, st); break;
        case 2: launch_delta_chunks<2>(a, cslots, batch, st); break;
        case 3: launch_delta_chunks<3>(a, cslots, batch, st); break;
        case 4: launch_delta_chunks<4>(a, cslots, batch, st); break;
        case 6: launch_delta_chunks<6>(a, cslots, batch, st); break;
        default: launch_delta_chunks<8>(a, cslots, batch, st);
    }
    NVH_CHECK_LAUNCH("nvh_delta_scan_chunked");
    if (batch == 1 && num_tokens >= min_tokens) return NVH_OK;
    return launch_delta_scan(p, batch, st);                  // the portions below min_tokens
}

extern "C" int32_t nvh_delta_post(const float* o, const void* norm_weight, const void* gate, int64_t gate_stride, void* y, int64_t y_stride,
                                  int64_t rows, int64_t heads, int64_t dv, float eps, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(o && norm_weight && y && rows >= 0 && heads > 0 && dv > 0, NVH_EINVAL, "nvh_delta_post: bad argument");
    if (rows == 0) return NVH_OK;
    const unsigned blocks = (unsigned)nvh_cdiv(rows * heads, 4);
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) delta_post_kernel<float><<<dim3(blocks), 256, 0, st>>>(o, (const float*)norm_weight, (const float*)gate, gate_stride, (float*)y, y_stride, rows, (int)heads, (int)dv, eps);
    else delta_post_kernel<bf16><<<dim3(blocks), 256, 0, st>>>(o, (const bf16*)norm_weight, (const bf16*)gate, gate_stride, (bf16*)y, y_stride, rows, (int)heads, (int)dv, eps);
    NVH_CHECK_LAUNCH("nvh_delta_post");
    return NVH_OK;
}
