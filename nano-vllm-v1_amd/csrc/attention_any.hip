// Paged causal attention for any head sizes (query/key size `dim`, value size `vdim`, any page size), with the pieces a
// gated, value-rotating attention needs around it:
//   nvh_attn_rotary_prep  per token, over the fused projection row [q | k | v | gate]: RMS norm over the WHOLE q and the
//                         whole k projection, or over every head by itself with one weight row shared by the heads
//                         (norm_per_head), partial rotary on q and k (frequency table given by the
//                         caller, so any scaling rule fits), rotation of the value by its own position over all of
//                         vdim, sigmoid of the per-head gate; q goes to a packed buffer, k and v to their cache slots.
//                         Keys are cached [pages, page, G, dim]; values TRANSPOSED within a page, [pages, G, vdim, page],
//                         so the attention reads a value column over consecutive keys in one piece (its matrix
//                         product wants V^T) and never transposes on the fly.
//   nvh_attn_kv_store     keys and values that need neither norm nor rotation, from the projection row to those cache slots, with an
//                         optional mixture of the value with another layer's value of the same token; in one-token steps also
//                         the block means that the tokens complete (below).  The query is read from the projection row in place.
//   nvh_attn_paged_any    softmax attention of var-len queries over the paged cache, scores / weights in fp32; the
//                         epilogue turns each head's output back by the query's position and multiplies the gate.
//                         Optional: a distance bias, score -= slope[head] * (query position - key position), and a
//                         sliding window that keeps the first tokens: query i sees key j <= i when i - j < window or
//                         j < keep_first; key tiles that no query of a workgroup can see are never loaded.
//                         Optional: chunks, query i sees key j <= i only when both lie in the same block of `chunk`
//                         positions counted from the sequence's start; and a sink per head, a learned logit that joins the
//                         softmax's denominator as one more term, as it is, standing for no token (it is the state a row starts from:
//                         maximum = sink, sum = 1, output = 0).
//                         Optional: pooled blocks in front of a window, one key and value (the means of the cached rows, see
//                         nvh_attn_pool_blocks) for each block of `pool` positions that lies wholly before the query's window,
//                         under the same softmax; a softcap, score <- cap tanh(score / cap); and a query temperature, q times
//                         1 + coef ln(floor((p + 1) / every) + 1) at position p.
//                         Optional: a learned bias per head and distance, score += bias[head][min(distance, len - 1)], and a gate per
//                         output element (a row of logits per token, beside the gate per head) in the epilogue.
//                         Steps in which every sequence brings one query: the heads that share a KV head share a workgroup
//                         (groups of more than 16 heads in parts); when that leaves most of the chip idle, a sequence's key
//                         tiles are dealt out to several workgroups whose rows a second launch merges.
//   nvh_attn_pool_blocks  the means of the blocks that a step has filled: keys and values read back from the cache as it holds
//                         them (so a block's mean does not depend on the steps that brought its tokens), fp32 sums, written to the
//                         page of the block's last token, rows [pages, pool_rows, G, dim] and [pages, pool_rows, G, vdim].
// Activations and caches are of type A (bf16 or fp32).  Key tiles always start at key 0 of a sequence and every query
// row keeps its own running maximum and sum, so a query's result does not depend on how the prompt was cut into steps
// or on what else is in the batch.
#include <type_traits>

#include "common.h"

namespace {

template <typename A>
__device__ __forceinline__ float ldf(const A* p, int64_t i) {
    return (float)p[i];
}

__device__ __forceinline__ float block_sum_256(float v, float* scratch) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    return scratch[0] + scratch[1] + scratch[2] + scratch[3];
}

struct PrepArgs {
    const void* proj;          // [T, ld] : q (H*dim) | k (G*dim) | v (G*vdim) | gate (H)
    int64_t ld;
    const void *q_norm, *k_norm;   // [H*dim], [G*dim]; norm_per_head: [dim] each, shared by the heads
    int norm_per_head;
    float eps;
    const int64_t* positions;
    const float* qk_freq;      // [rot_dims / 2]
    float qk_mag;
    int rot_dims, qk_interleaved;
    const float* v_freq;       // [vdim / 2], or null: values are stored as they are
    int v_interleaved;
    void* q_out;               // [T, H*dim]
    float* gate_out;           // [T, H], or null (no gate columns in proj)
    void *k_cache, *v_cache;   // [pages, page, G, dim], [pages, G, vdim, page] (values transposed within a page)
    const int32_t* slot_mapping;
    int H, G, dim, vdim, page;
};

template <typename A>
__global__ __launch_bounds__(256) void attn_rotary_prep_kernel(PrepArgs a) {
    __shared__ float red[4];
    extern __shared__ float head_inv[];                      // norm_per_head: 1 / rms of every q head, then of every k head
    const int64_t t = blockIdx.x;
    const A* row = (const A*)a.proj + t * a.ld;
    const int nq = a.H * a.dim, nk = a.G * a.dim, nv = a.G * a.vdim;
    const A* qr = row;
    const A* kr = row + nq;
    const A* vr = kr + nk;
    float inv_q = 1.f, inv_k = 1.f;
    if (a.q_norm && a.norm_per_head) {                       // a wave per head in turn (q heads, then k heads: they lie one after the other)
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        for (int h = wave; h < a.H + a.G; h += 4) {
            const A* hr = qr + (int64_t)h * a.dim;
            float ss = 0.f;
            for (int i = lane; i < a.dim; i += 64) {
                const float v = ldf(hr, i);
                ss += v * v;
            }
            ss = wave_sum(ss);
            if (lane == 0) head_inv[h] = 1.0f / sqrtf(ss / (float)a.dim + a.eps);
        }
        __syncthreads();
    } else if (a.q_norm) {                                   // (null norm weights: q and k pass as they are)
        float sq = 0.f, sk = 0.f;
        for (int i = threadIdx.x; i < nq; i += 256) {
            const float v = ldf(qr, i);
            sq += v * v;
        }
        for (int i = threadIdx.x; i < nk; i += 256) {
            const float v = ldf(kr, i);
            sk += v * v;
        }
        sq = block_sum_256(sq, red);
        sk = block_sum_256(sk, red);
        inv_q = 1.0f / sqrtf(sq / (float)nq + a.eps), inv_k = 1.0f / sqrtf(sk / (float)nk + a.eps);
    }
    const float pos = (float)a.positions[t];
    const int64_t slot = a.slot_mapping ? a.slot_mapping[t] : -1;
    // q and k: norm, then rotary on the first rot_dims dimensions of every head
    for (int which = 0; which < 2; ++which) {
        const int n = which ? nk : nq;
        const A* src = which ? kr : qr;
        const A* wn = (const A*)(which ? a.k_norm : a.q_norm);
        const float inv = which ? inv_k : inv_q;
        const int hbase = which ? a.H : 0;
        A* dst = which ? (slot >= 0 && a.k_cache ? (A*)a.k_cache + slot * nk : nullptr) : (A*)a.q_out + t * nq;
        if (!dst) continue;
        for (int i = threadIdx.x; i < n; i += 256) {
            const int d = i % a.dim;
            const float rinv = a.norm_per_head && wn ? head_inv[hbase + i / a.dim] : inv;
            float v = wn ? ldf(src, i) * rinv * ldf(wn, a.norm_per_head ? d : i) : ldf(src, i);
            if (d < a.rot_dims) {
                int partner, pair;
                bool first;
                pair_of(d, a.rot_dims, a.qk_interleaved, partner, pair, first);
                const int j = i - d + partner;
                const float o = wn ? ldf(src, j) * rinv * ldf(wn, a.norm_per_head ? partner : j) : ldf(src, j);
                float sn, cs;
                rot_sincos<A>(pos * a.qk_freq[pair], sn, cs);
                const float c = cs * a.qk_mag, s = sn * a.qk_mag;
                v = first ? v * c - o * s : v * c + o * s;
            }
            dst[i] = (A)v;
        }
    }
    if (slot >= 0 && a.v_cache) {
        A* dst = (A*)a.v_cache + (slot / a.page) * a.page * nv + slot % a.page;      // element i of the row goes to dst[i * page]
        for (int i = threadIdx.x; i < nv; i += 256) {
            float v = ldf(vr, i);
            if (a.v_freq) {
                const int d = i % a.vdim;
                int partner, pair;
                bool first;
                pair_of(d, a.vdim, a.v_interleaved, partner, pair, first);
                const float o = ldf(vr, i - d + partner);
                float s, c;
                rot_sincos<A>(pos * a.v_freq[pair], s, c);
                v = first ? v * c - o * s : v * c + o * s;
            }
            dst[(int64_t)i * a.page] = (A)v;
        }
    }
    if (a.gate_out)
        for (int h = threadIdx.x; h < a.H; h += 256) a.gate_out[t * a.H + h] = 1.0f / (1.0f + expf(-ldf(vr + nv, h)));
}

// The same with eight consecutive elements per lane and 16-byte accesses (head sizes and rotated dimensions that keep a piece of eight on one side
// of a rotation, aligned rows).  A token's workgroup requests everything it reads at once - its pieces, their rotation partners, the weights of
// both - and the sines and cosines of a position are formed once for all heads.  Values: piece by piece beside q and k (`v_tiles` 0), or, for many
// tokens, by workgroups of their own behind the tokens' (64 tokens by 64 columns, turned in LDS, so that tokens that lie side by side in a page leave
// as one cache line).
// us, the form above and this one, 16 + 8 heads of 128 x 128: 1000 tokens 24.6 and 9.3, 64 tokens 17.1 and 8.1.
constexpr int PREP_PAIRS = 128;                              // rotation pairs of a head at most
constexpr int PREP_TILE_TOKENS = 128;                       // tokens from which values go by tiles
constexpr int VT = 64;                                       // tokens and columns of a value tile
template <typename A, int J>
__global__ __launch_bounds__(256) void attn_rotary_prep_vec_kernel(PrepArgs a, int64_t tokens, int v_tiles) {
    __shared__ float smem[VT * (VT + 1)];                    // a value tile, or: sums per piece (256 J), cosines, sines, partial sums of the rows
    const int nq = a.H * a.dim, nk = a.G * a.dim, nv = a.G * a.vdim, tid = threadIdx.x;
    // v: eight values of a row from column c on, turned by the token's position
    auto turned = [&](const A* vr, int c, float pos, float (&x)[8]) {
        nvh_load8(vr, c, 8, 1, x);
        if (!a.v_freq) return;
        const int d = c % a.vdim, half = a.vdim >> 1;
        float o[8];
        if (!a.v_interleaved) nvh_load8(vr, d < half ? c + half : c - half, 8, 1, o);
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            int partner, pair;
            bool first;
            pair_of(d + e, a.vdim, a.v_interleaved, partner, pair, first);
            const float other = a.v_interleaved ? x[e ^ 1] : o[e];
            float sn, cs;
            rot_sincos<A>(pos * a.v_freq[pair], sn, cs);
            y[e] = first ? x[e] * cs - other * sn : x[e] * cs + other * sn;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = y[e];
    };
    if ((int64_t)blockIdx.x >= tokens) {                     // (uniform) a value tile
        const int tile = (int)(blockIdx.x - tokens), c0 = tile % v_tiles * VT;
        const int64_t t0 = (int64_t)(tile / v_tiles) * VT;
#pragma unroll
        for (int j = 0; j < VT * VT / 8 / 256; ++j) {
            const int i = tid + 256 * j, r = i >> 3, c = c0 + ((i & 7) << 3);
            const int64_t t = min(t0 + r, tokens - 1);
            if (c < nv) {
                float x[8];
                turned((const A*)a.proj + t * a.ld + nq + nk, c, (float)a.positions[t], x);
#pragma unroll
                for (int e = 0; e < 8; ++e) smem[r * (VT + 1) + c - c0 + e] = x[e];
            }
        }
        __syncthreads();
        const int r = tid & (VT - 1);
        const int64_t slot = t0 + r < tokens ? a.slot_mapping[t0 + r] : -1;
        if (slot < 0) return;
        A* dst = (A*)a.v_cache + (slot / a.page) * a.page * nv + slot % a.page;
#pragma unroll
        for (int j = 0; j < VT / 4; ++j) {
            const int c = (tid >> 6) + 4 * j;
            if (c0 + c < nv) dst[(int64_t)(c0 + c) * a.page] = (A)smem[r * (VT + 1) + c];
        }
        return;
    }
    const int64_t t = blockIdx.x;
    const A* row = (const A*)a.proj + t * a.ld;
    const int64_t slot = a.slot_mapping ? a.slot_mapping[t] : -1;
    const float pos = (float)a.positions[t];
    const int pieces = (nq + nk) >> 3, half = a.rot_dims >> 1, per_head = a.dim >> 3;
    float *sums = smem, *cosines = smem + 256 * J, *sines = cosines + PREP_PAIRS, *red = sines + PREP_PAIRS;
    const bool normed = a.q_norm != nullptr;
    float x[J][8], o[J][8], w[J][8], wo[J][8];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = min(tid + 256 * j, pieces - 1) << 3, d = c % a.dim;          // (q and k adjoin; pieces past the last repeat it)
        const int to = d >= a.rot_dims || a.qk_interleaved ? 0 : (d < half ? half : -half);
        nvh_load8(row, c, 8, 1, x[j]);
        if (!a.qk_interleaved) nvh_load8(row, c + to, 8, 1, o[j]);
        if (normed) {
            const A* wn = (const A*)(c < nq ? a.q_norm : a.k_norm);
            const int at = a.norm_per_head ? d : (c < nq ? c : c - nq);
            nvh_load8(wn, at, 8, 1, w[j]);
            if (!a.qk_interleaved) nvh_load8(wn, at + to, 8, 1, wo[j]);
        }
    }
    for (int i = tid; i < half; i += 256) {
        float sn, cs;
        rot_sincos<A>(pos * a.qk_freq[i], sn, cs);
        cosines[i] = cs * a.qk_mag;
        sines[i] = sn * a.qk_mag;
    }
    // a head's pieces side by side in a wave: their sum there, and in `sums`; else `sums` has the pieces'.
    // (us, chains through `sums` and so, 16 + 8 heads of 128, 64 tokens: 5.7 and 5.4; 1000 9.1 and 8.9)
    const bool in_lanes = a.norm_per_head && (per_head == 8 || per_head == 16 || per_head == 32);
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int i = tid + 256 * j;
        float ss[4];                                         // (in pairs, as a wave's lanes add: chains leave 1 / rms of 128 elements 4.9e-8 off, of 256 5.6e-8, these 4.3e-8)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss[e] = __builtin_fmaf(x[j][2 * e + 1], x[j][2 * e + 1], x[j][2 * e] * x[j][2 * e]);
        ss[0] = (ss[0] + ss[1]) + (ss[2] + ss[3]);
        float head = ss[0];
        if (in_lanes) {                                      // (uniform)
            head += NVH_DPP(head, 0xB1);
            head += NVH_DPP(head, 0x4E);
            head += NVH_DPP(head, 0x141);
            if (per_head >= 16) head += NVH_DPP(head, 0x140);
            if (per_head >= 32) head = pair16_sum(head);
        }
        sums[i] = head;
        if (i < pieces) (i << 3 < nq ? sq : sk) += ss[0];
    }
    if (normed && !a.norm_per_head) {                        // (uniform)
        sq = wave_sum(sq);
        sk = wave_sum(sk);
        if ((tid & 63) == 0) {
            red[tid >> 6] = sq;
            red[4 + (tid >> 6)] = sk;
        }
    }
    __syncthreads();
    const float inv_q = normed && !a.norm_per_head ? 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)nq + a.eps) : 1.f;
    const float inv_k = normed && !a.norm_per_head ? 1.0f / sqrtf(((red[4] + red[5]) + (red[6] + red[7])) / (float)nk + a.eps) : 1.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int i = tid + 256 * j, c = i << 3, d = c % a.dim;
        if (i >= pieces) break;
        const bool is_k = c >= nq;
        if (normed) {
            float rinv = is_k ? inv_k : inv_q;
            if (a.norm_per_head) {
                const float* hs = sums + i / per_head * per_head;
                float ss = in_lanes ? sums[i] : 0.f;
                if (!in_lanes)
                    for (int p = 0; p < per_head; p += 2) ss += hs[p] + (p + 1 < per_head ? hs[p + 1] : 0.f);
                rinv = 1.0f / sqrtf(ss / (float)a.dim + a.eps);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[j][e] = x[j][e] * rinv * w[j][e];
                if (!a.qk_interleaved) o[j][e] = o[j][e] * rinv * wo[j][e];
            }
        }
        A out[8];
        if (d < a.rot_dims) {
            const bool first = d < half;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int pair = a.qk_interleaved ? (d + e) >> 1 : (first ? d + e : d + e - half);
                const float cs = cosines[pair], sn = sines[pair];
                if (a.qk_interleaved) out[e] = (A)(e & 1 ? x[j][e] * cs + x[j][e ^ 1] * sn : x[j][e] * cs - x[j][e ^ 1] * sn);
                else out[e] = (A)(first ? x[j][e] * cs - o[j][e] * sn : x[j][e] * cs + o[j][e] * sn);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) out[e] = (A)x[j][e];
        }
        if (!is_k) __builtin_memcpy(__builtin_assume_aligned((A*)a.q_out + t * nq + c, 16), out, sizeof(out));
        else if (slot >= 0 && a.k_cache) __builtin_memcpy(__builtin_assume_aligned((A*)a.k_cache + slot * nk + (c - nq), 16), out, sizeof(out));
    }
    const A* vr = row + nq + nk;
    if (v_tiles == 0 && slot >= 0 && a.v_cache) {
        A* dst = (A*)a.v_cache + (slot / a.page) * a.page * nv + slot % a.page;      // element i of the row goes to dst[i * page]
        for (int i = 255 - tid; i < nv >> 3; i += 256) {     // (from the last lane down: the first ones have more pieces of q and k)
            float v[8];
            turned(vr, i << 3, pos, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) dst[(int64_t)((i << 3) + e) * a.page] = (A)v[e];
        }
    }
    if (a.gate_out)
        for (int h = tid; h < a.H; h += 256) a.gate_out[t * a.H + h] = 1.0f / (1.0f + expf(-ldf(vr + nv, h)));
}

// Whether attn_rotary_prep_vec_kernel takes the call: pieces of eight that lie on one side of every rotation, and aligned.
template <typename A>
static bool prep_vec_ok(const PrepArgs& a) {
    const int per16 = 16 / (int)sizeof(A);
    const auto rotates = [](int n, int interleaved) { return n % (interleaved ? 8 : 16) == 0; };
    return a.dim % 8 == 0 && a.vdim % 8 == 0 && rotates(a.rot_dims, a.qk_interleaved) && a.rot_dims <= 2 * PREP_PAIRS &&
           (!a.v_freq || rotates(a.vdim, a.v_interleaved)) && (a.H + a.G) * a.dim <= 8 * 256 * 4 && a.ld % per16 == 0 && nvh_aligned16(a.proj) &&
           nvh_aligned16(a.q_out) && (!a.k_cache || nvh_aligned16(a.k_cache)) && (!a.q_norm || (nvh_aligned16(a.q_norm) && nvh_aligned16(a.k_norm)));
}

template <typename A>
static void launch_rotary_prep(const PrepArgs& a, int64_t tokens, size_t lds, hipStream_t st) {
    if (!prep_vec_ok<A>(a)) {
        attn_rotary_prep_kernel<A><<<dim3((unsigned)tokens), 256, lds, st>>>(a);
        return;
    }
    const int nv = a.G * a.vdim, pieces = (a.H + a.G) * a.dim / 8;
    const int v_tiles = tokens >= PREP_TILE_TOKENS && a.v_cache && a.slot_mapping ? (int)nvh_cdiv(nv, VT) : 0;
    const dim3 grid((unsigned)(tokens + nvh_cdiv(tokens, VT) * v_tiles));
    if (pieces <= 256) attn_rotary_prep_vec_kernel<A, 1><<<grid, 256, 0, st>>>(a, tokens, v_tiles);
    else if (pieces <= 512) attn_rotary_prep_vec_kernel<A, 2><<<grid, 256, 0, st>>>(a, tokens, v_tiles);
    else attn_rotary_prep_vec_kernel<A, 4><<<grid, 256, 0, st>>>(a, tokens, v_tiles);
}

// ---------------------------------------------------------------------------------------------------------------
constexpr int AQ = 16;        // queries per workgroup (one 16-lane row of a wave per query)
constexpr int AK = 32;        // keys per tile
constexpr int AVC_MAX = 32;   // value columns per lane (the kernel's AVC: 16, or 32 for wide values): vdim <= 16 * AVC_MAX

struct AttnArgs {
    const void* q;             // [T, ldq]: H*dim columns
    int64_t ldq;
    const void *k_cache, *v_cache;
    const int32_t* cu_seqlens_q;    // [B+1], or null: one query per sequence (row b is sequence b)
    const int32_t* context_lens;    // [B]: keys of the sequence including this step's tokens
    const int32_t* block_tables;
    int64_t table_stride;
    int batch, page;
    int H, G, dim, vdim;
    float scale;
    const float* gate;         // [T, H] or null
    const float* v_freq;       // [vdim/2] or null: no turning back
    int v_interleaved;
    void* out;                 // [T, H*vdim]
    const void* gate_elems;    // [T, ld_elems]: H*vdim logits whose sigmoids multiply the output's elements, or null
    int64_t ld_elems;
    const float* slopes;       // [H] or null: score -= slopes[head] * (query position - key position)
    const float* bias;         // [H, bias_len] or null: score += bias[head][min(query position - key position, bias_len - 1)]
    int bias_len;
    int window, keep_first;    // window > 0: key j is visible to query i only when i - j < window or j < keep_first
    int chunk;                 // chunk > 0: ... and only when j >= (i / chunk) * chunk
    const float* sinks;        // [H] or null: a logit per head that joins the denominator of every row of that head
    float softcap;             // > 0: score <- softcap tanh(score / softcap)
    float temp_coef;           // temp_every > 0: scores of the query at position p times 1 + temp_coef ln(floor((p + 1) / temp_every) + 1)
    int temp_every;
    int pool, pool_rows;       // pool > 0 (with a window): blocks of `pool` positions before the window are seen through their means ...
    const void *pk, *pv;       // ... [pages, pool_rows, G, dim], [pages, pool_rows, G, vdim], in the page of the block's last position
    int pages_offset;          // byte offset in LDS of the sequence's page ids (matrix-core kernel)
    int ml_offset;             // ... of the waves' (max, sum) pairs in the one-query form
    int bias_offset, bias_ld;  // ... and of the heads' bias rows, bias_ld floats apart
    int kv_split;              // one-query form: workgroups per (sequence, KV head), each with H / (G kv_split) of the group's heads
    int key_parts;             // one-query form: workgroups that share a sequence's key tiles (tile j goes to part j % key_parts); > 1: the
    float* parts;              // parts leave [batch, G kv_split, key_parts, 16, vdim + 2] (unnormalised rows, then max and sum) here
    int balance;               // one-query form: sequences are dealt out by their length where one sees more keys than this (balanced_place; 0: never)
};

// The key tiles (of `tile` keys, starting at multiples of it) that a workgroup whose first query sits at position qlo has to
// walk: all of them without a window; with one, the tiles that hold kept first tokens and then those from the window of
// the first query on.  next(k0) is the start of the tile after k0.
struct TileWalk {
    int first_end, win_start, tile;
    __device__ __forceinline__ TileWalk(int window, int keep_first, int chunk, int qlo, int tile_) : tile(tile_) {
        first_end = window > 0 ? ((keep_first + tile_ - 1) / tile_) * tile_ : 0;
        win_start = window > 0 ? (max(qlo - window + 1, 0) / tile_) * tile_ : 0;
        // (the chunk of the first query starts no later than any other query's: earlier tiles are seen by none)
        if (chunk > 0) win_start = max(win_start, ((qlo / chunk) * chunk / tile_) * tile_);
    }
    __device__ __forceinline__ int next(int k0) const {
        const int n = k0 + tile;
        return (n >= first_end && n < win_start) ? win_start : n;
    }
};

// Pooled blocks that the query at qpos sees: those whose last position is <= qpos - window.
__device__ __forceinline__ int blocks_seen(int qpos, int window, int pool) { return qpos >= window ? (qpos - window + 1) / pool : 0; }

// Where the mean of block b lies: the page of the block's last position (as an index into the sequence's pages) and the row
// within that page (blocks whose last position is in page n are numbered from floor(n page / pool) on).
__device__ __forceinline__ void block_place(int b, int pool, int page, int& page_index, int& row) {
    page_index = (b * pool + pool - 1) / page;
    row = b - page_index * page / pool;
}

__device__ __forceinline__ float query_temperature(int qpos, float coef, int every) {
    return every > 0 ? 1.0f + coef * logf((float)((qpos + 1) / every + 1)) : 1.0f;
}

// The tiles in order: with pooled blocks, ceil(blocks / tile) tiles of them first - their start is counted up to 0 from below,
// tile v of n starts at (v - n) tile - and then the token tiles of the walk.
struct TileOrder {
    TileWalk walk;
    int pooled_span;           // pooled tiles times tile
    __device__ __forceinline__ TileOrder(const TileWalk& w, int blocks) : walk(w), pooled_span((blocks + w.tile - 1) / w.tile * w.tile) {}
    __device__ __forceinline__ int first_token_tile() const { return walk.first_end > 0 || walk.win_start == 0 ? 0 : walk.win_start; }
    __device__ __forceinline__ int first() const { return pooled_span > 0 ? -pooled_span : first_token_tile(); }
    __device__ __forceinline__ int next(int k0) const {
        if (k0 >= 0) return walk.next(k0);
        return k0 + walk.tile < 0 ? k0 + walk.tile : first_token_tile();
    }
    __device__ __forceinline__ int block_of(int k0) const { return k0 + pooled_span; }       // (k0 < 0) the tile's first block
};

__device__ __forceinline__ bool key_visible(int key, int qpos, int window, int keep_first, int chunk) {
    return key <= qpos && (window <= 0 || qpos - key < window || key < keep_first) && (chunk <= 0 || key >= (qpos / chunk) * chunk);
}

// The sigmoid of an element gate: the library's exponential where everything is fp32, the hardware's 2^x and reciprocal for bf16 results.
template <typename A>
__device__ __forceinline__ float elem_gate(float z) {
    if constexpr (sizeof(A) == 4) return 1.0f / (1.0f + expf(-z));
    else return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * 1.4426950408889634f));
}

template <typename A, int AVC>
__global__ __launch_bounds__(256) void attn_paged_any_kernel(AttnArgs a) {
    extern __shared__ float smem[];
    // which (sequence, query tile) is this workgroup's
    int seq = -1, q0 = 0, qlen = 0, qbase = 0;
    {
        int tile = blockIdx.x;
        for (int b = 0; b < a.batch; ++b) {
            const int lo = a.cu_seqlens_q ? a.cu_seqlens_q[b] : b, hi = a.cu_seqlens_q ? a.cu_seqlens_q[b + 1] : b + 1;
            const int tiles = (hi - lo + AQ - 1) / AQ;
            if (tile < tiles) {
                seq = b;
                q0 = tile * AQ;
                qlen = hi - lo;
                qbase = lo;
                break;
            }
            tile -= tiles;
        }
    }
    if (seq < 0) return;                                     // (uniform over the workgroup)
    const int head = blockIdx.y, kvh = head / (a.H / a.G);
    const int dim = a.dim, vdim = a.vdim;
    const int klen = a.context_lens[seq];
    const int past = klen - qlen;                            // keys before this step's first query
    const int nq = min(AQ, qlen - q0);
    const int kd = dim + 1, vd = vdim + 1;
    float* qs = smem;                                        // [AQ][dim]
    float* ks = qs + AQ * dim;                               // [AK][dim + 1]
    float* vs = ks + AK * kd;                                // [AK][vdim + 1]
    float* ps = vs + AK * vd;                                // [AQ][AK]
    const int tid = threadIdx.x, qi = tid >> 4, sub = tid & 15;
    for (int i = tid; i < AQ * dim; i += 256) {
        const int r = i / dim, d = i - r * dim;
        const float sc = a.scale * query_temperature(past + q0 + r, a.temp_coef, a.temp_every);
        qs[i] = r < nq ? ldf((const A*)a.q, (int64_t)(qbase + q0 + r) * a.ldq + head * dim + d) * sc : 0.f;
    }
    float acc[AVC];
#pragma unroll
    for (int c = 0; c < AVC; ++c) acc[c] = 0.f;
    // (a sink is what the row starts from: it has been seen with score sink, weight 1 and no value)
    float m_run = a.sinks ? a.sinks[head] : -INFINITY, l_run = a.sinks ? 1.f : 0.f;
    const int qpos = past + q0 + qi;                         // this lane's query position (valid for qi < nq)
    const int last_key = past + q0 + nq - 1;                 // the tile's last query sees keys 0..last_key
    const int32_t* table = a.block_tables + (int64_t)seq * a.table_stride;
    const float slope = a.slopes ? a.slopes[head] : 0.f;
    const float* bias = a.bias ? a.bias + (int64_t)head * a.bias_len : nullptr;
    const int nblocks = a.pool > 0 ? blocks_seen(last_key, a.window, a.pool) : 0, my_blocks = a.pool > 0 ? blocks_seen(qpos, a.window, a.pool) : 0;
    const TileOrder order(TileWalk(a.window, a.keep_first, a.chunk, past + q0, AK), nblocks);
    for (int k0 = order.first(); k0 <= last_key; k0 = order.next(k0)) {
        const bool pooled = k0 < 0;                          // (uniform) a tile of block means; bk0: its first block
        const int bk0 = order.block_of(k0);
        __syncthreads();                                     // the previous tile's readers are done
        if (pooled) {
            for (int i = tid; i < AK * (dim + vdim); i += 256) {
                const int r = i / (dim + vdim), d = i - r * (dim + vdim), b = bk0 + r;
                float v = 0.f;
                if (b < nblocks) {
                    int pi, row;
                    block_place(b, a.pool, a.page, pi, row);
                    const int64_t at = ((int64_t)table[pi] * a.pool_rows + row) * a.G + kvh;
                    v = d < dim ? ldf((const A*)a.pk, at * dim + d) : ldf((const A*)a.pv, at * vdim + d - dim);
                }
                (d < dim ? ks[r * kd + d] : vs[r * vd + d - dim]) = v;
            }
        } else {
        for (int i = tid; i < AK * dim; i += 256) {
            const int r = i / dim, d = i - r * dim, key = k0 + r;
            float v = 0.f;
            if (key <= last_key) {
                const int64_t slot = (int64_t)table[key / a.page] * a.page + key % a.page;
                v = ldf((const A*)a.k_cache, (slot * a.G + kvh) * dim + d);
            }
            ks[r * kd + d] = v;
        }
        for (int i = tid; i < AK * vdim; i += 256) {
            const int r = i / vdim, d = i - r * vdim, key = k0 + r;
            float v = 0.f;
            if (key <= last_key) {
                v = ldf((const A*)a.v_cache, (((int64_t)table[key / a.page] * a.G + kvh) * vdim + d) * a.page + key % a.page);
            }
            vs[r * vd + d] = v;
        }
        }
        __syncthreads();
        // scores of query qi against keys sub and sub + 16 of the tile
        float s0 = 0.f, s1 = 0.f;
        const float* qrow = qs + qi * dim;
        const float *kr0 = ks + sub * kd, *kr1 = ks + (sub + 16) * kd;
        for (int d = 0; d < dim; ++d) {
            const float qv = qrow[d];
            s0 = __builtin_fmaf(qv, kr0[d], s0);
            s1 = __builtin_fmaf(qv, kr1[d], s1);
        }
        if (a.softcap > 0.f) {
            s0 = a.softcap * tanhf(s0 / a.softcap);
            s1 = a.softcap * tanhf(s1 / a.softcap);
        }
        const bool ok0 = qi < nq && (pooled ? bk0 + sub < my_blocks : key_visible(k0 + sub, qpos, a.window, a.keep_first, a.chunk));
        const bool ok1 = qi < nq && (pooled ? bk0 + sub + 16 < my_blocks : key_visible(k0 + sub + 16, qpos, a.window, a.keep_first, a.chunk));
        s0 = ok0 ? s0 - slope * (float)(qpos - (k0 + sub)) : -INFINITY;
        s1 = ok1 ? s1 - slope * (float)(qpos - (k0 + sub + 16)) : -INFINITY;
        if (bias) {
            if (ok0) s0 += bias[min(qpos - (k0 + sub), a.bias_len - 1)];
            if (ok1) s1 += bias[min(qpos - (k0 + sub + 16), a.bias_len - 1)];
        }
        const float m_new = fmaxf(m_run, row16_max(fmaxf(s0, s1)));
        // (unseen keys and those that a bias masks weigh nothing; a row that has seen nothing else yet keeps m = -inf)
        const float p0 = s0 == -INFINITY ? 0.f : expf(s0 - m_new), p1 = s1 == -INFINITY ? 0.f : expf(s1 - m_new);
        const float alpha = m_new == -INFINITY ? 1.f : expf(m_run - m_new);
        l_run = l_run * alpha + row16_sum(p0 + p1);
        m_run = m_new;
        ps[qi * AK + sub] = p0;
        ps[qi * AK + sub + 16] = p1;
        __syncthreads();
        const float* prow = ps + qi * AK;
#pragma unroll
        for (int c = 0; c < AVC; ++c) {
            const int col = sub + 16 * c;
            if (col < vdim) {
                float s = acc[c] * alpha;
                for (int r = 0; r < AK; ++r) s = __builtin_fmaf(prow[r], vs[r * vd + col], s);
                acc[c] = s;
            }
        }
    }
    // epilogue: normalise, turn back by the query's position, gate
    __syncthreads();
    float* os = ks;                                          // [AQ][vdim] (fits: AK >= AQ)
#pragma unroll
    for (int c = 0; c < AVC; ++c) {
        const int col = sub + 16 * c;
        if (col < vdim) os[qi * vdim + col] = l_run > 0.f ? acc[c] / l_run : 0.f;
    }
    __syncthreads();
    if (qi < nq) {
        const int64_t tok = qbase + q0 + qi;
        const float g = a.gate ? a.gate[tok * a.H + head] : 1.0f;
        const float pos = (float)qpos;
#pragma unroll
        for (int c = 0; c < AVC; ++c) {
            const int col = sub + 16 * c;
            if (col < vdim) {
                float v = os[qi * vdim + col];
                if (a.v_freq) {
                    int partner, pair;
                    bool first;
                    pair_of(col, vdim, a.v_interleaved, partner, pair, first);
                    const float o = os[qi * vdim + partner];
                    float sn, cs;
                    rot_sincos<A>(pos * a.v_freq[pair], sn, cs);
                    v = first ? v * cs + o * sn : v * cs - o * sn;        // the rotation by -pos
                }
                if (a.gate_elems) v *= elem_gate<A>(ldf((const A*)a.gate_elems, tok * a.ld_elems + head * vdim + col));
                ((A*)a.out)[(tok * a.H + head) * vdim + col] = (A)(v * g);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// The same attention for fp32 caches on the matrix cores (16x16x4, fp32 in and out), dim = 16 NKS and vdim = 16 NVT, pages of whole 16-key blocks.
// A workgroup is 16 rows - consecutive queries of one head or, where every sequence brings one query (`grouped`), the heads of a KV group - and its
// four waves take every fourth block of 16 keys: S^T = K Q^T leaves a lane the scores of query lane % 16 and keys 4 (lane / 16) + e, which is how
// O^T = V^T P^T takes them, so nothing is exchanged but a maximum.  A value is used once per workgroup: keys and values go from the cache to the
// registers, the next block's while this one's products run, and LDS holds only the waves' results for the merge.  Which wave a key falls to depends
// on its position alone and a row's results on no other row, so neither the cut nor the batch changes a bit.
// us, the form above (two scalar LDS reads for two multiply-adds) and this one, 16 heads of 128 x 128 over 8: 301 queries 168 and 26, 1024 queries 897
// and 127, 1024 at the end of 4096 keys 4468 and 464, one query over 1500 keys 778 and 58, 64 x one over 700 keys 1134 and 72; 16 heads of 256 x 192
// over one, 1024 queries: 1673 and 210.  A short prompt is bound by the chain of its longest tile (load, product, exponentials, product per 64 keys),
// a long one by the fp32 products (124 TFLOP/s at most).
template <int NKS, int NVT>
__global__ __launch_bounds__(256) void attn_paged_f32_kernel(AttnArgs a, int grouped) {
    extern __shared__ __attribute__((aligned(16))) float smem[];     // [4 waves][16 rows][vdim + 4] outputs, then [4][16] maxima and sums
    constexpr int dim = 16 * NKS, vdim = 16 * NVT, OLD = vdim + 4, BLOCK = 16, TILE = 64;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, row = lane & 15, quarter = lane >> 4;
    const int group = a.H / a.G;
    int seq = -1, q0 = 0, qlen = 1, qbase = 0, head0, nq;
    if (grouped) {
        const int parts = (group + 15) / 16, part = blockIdx.y % parts;
        if ((int)blockIdx.x < a.batch) seq = qbase = blockIdx.x;
        head0 = (blockIdx.y / parts) * group + 16 * part;
        nq = min(16, group - 16 * part);
    } else {
        int tile = blockIdx.x;
        for (int b = 0; b < a.batch; ++b) {
            const int lo = a.cu_seqlens_q ? a.cu_seqlens_q[b] : b, hi = a.cu_seqlens_q ? a.cu_seqlens_q[b + 1] : b + 1;
            const int tiles = (hi - lo + AQ - 1) / AQ;
            if (tile < tiles) {
                seq = b;
                q0 = tile * AQ;
                qlen = hi - lo;
                qbase = lo;
                break;
            }
            tile -= tiles;
        }
        head0 = blockIdx.y;
        nq = min(AQ, qlen - q0);
    }
    if (seq < 0) return;                                     // (uniform over the workgroup)
    const int kvh = head0 / group;
    const int past = a.context_lens[seq] - qlen;             // keys before this step's first query
    const int myrow = min(row, nq - 1), head = grouped ? head0 + myrow : head0, qtok = grouped ? 0 : q0 + myrow;      // (rows past nq repeat the last)
    const int qpos = past + qtok, last_key = past + q0 + (grouped ? 0 : nq - 1);
    const int32_t* table = a.block_tables + (int64_t)seq * a.table_stride;
    const int nblocks = a.pool > 0 ? blocks_seen(last_key, a.window, a.pool) : 0, my_blocks = a.pool > 0 ? blocks_seen(qpos, a.window, a.pool) : 0;
    const TileOrder order(TileWalk(a.window, a.keep_first, a.chunk, past + q0, TILE), nblocks);
    const float *kc = (const float*)a.k_cache, *vc = (const float*)a.v_cache;
    f32x4 k[NKS], v[NVT], acc[NVT], qr[NKS];
    // The block of the tile at k0 that is this wave's.  Blocks past the last key repeat the one that holds it: nobody sees them.
    auto fetch_k = [&](int k0) {
        const float* src;
        if (k0 < 0) {
            int pi, at;
            block_place(min(order.block_of(k0) + BLOCK * wave + row, nblocks - 1), a.pool, a.page, pi, at);
            src = (const float*)a.pk + (((int64_t)table[pi] * a.pool_rows + at) * a.G + kvh) * dim;
        } else {
            const int kb = min(k0 + BLOCK * wave, last_key / BLOCK * BLOCK), page = kb / a.page;
            src = kc + (((int64_t)table[page] * a.page + (min(kb + row, last_key) - page * a.page)) * a.G + kvh) * dim;
        }
#pragma unroll
        for (int j = 0; j < NKS; ++j) k[j] = *reinterpret_cast<const f32x4*>(src + 16 * j + 4 * quarter);
    };
    auto fetch_v = [&](int k0) {
        if (k0 < 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int pi, at;
                block_place(min(order.block_of(k0) + BLOCK * wave + 4 * quarter + e, nblocks - 1), a.pool, a.page, pi, at);
                const float* src = (const float*)a.pv + (((int64_t)table[pi] * a.pool_rows + at) * a.G + kvh) * vdim + row;
#pragma unroll
                for (int c = 0; c < NVT; ++c) v[c][e] = src[16 * c];
            }
        } else {
            const int kb = min(k0 + BLOCK * wave, last_key / BLOCK * BLOCK), page = kb / a.page;
            const float* src = vc + (((int64_t)table[page] * a.G + kvh) * vdim + row) * a.page + (kb - page * a.page) + 4 * quarter;
#pragma unroll
            for (int c = 0; c < NVT; ++c) v[c] = *reinterpret_cast<const f32x4*>(src + (int64_t)16 * c * a.page);
        }
    };
    int k0 = order.first();
    if (k0 <= last_key) {                                    // (a sequence without keys has no pages)
        fetch_k(k0);
        fetch_v(k0);
    }
    {
        const float* src = (const float*)a.q + (int64_t)(qbase + qtok) * a.ldq + head * dim + 4 * quarter;
        const float sc = a.scale * query_temperature(qpos, a.temp_coef, a.temp_every);
#pragma unroll
        for (int j = 0; j < NKS; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) qr[j][e] = src[16 * j + e] * sc;
        }
    }
#pragma unroll
    for (int c = 0; c < NVT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (a sink is what the row starts from: it has been seen with score sink, weight 1 and no value - by the first wave)
    const bool sunk = a.sinks && wave == 0;
    float m_run = sunk ? a.sinks[head] : -INFINITY, l_run = sunk && quarter == 0 ? 1.f : 0.f;     // (a lane sums its own keys' weights)
    const float slope = a.slopes ? a.slopes[head] : 0.f;
    const float* bias = a.bias ? a.bias + (int64_t)head * a.bias_len : nullptr;
    while (k0 <= last_key) {
        const bool pooled = k0 < 0;                          // (uniform) a tile of block means
        const int next = order.next(k0), kb = k0 + BLOCK * wave, key0 = kb + 4 * quarter, block0 = pooled ? order.block_of(k0) + BLOCK * wave + 4 * quarter : 0;
        float biases[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) biases[e] = bias[min(max(qpos - (key0 + e), 0), a.bias_len - 1)];
        }
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int j = 0; j < NKS; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (j & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][e], qr[j][e], s1, 0, 0, 0);
                else s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][e], qr[j][e], s0, 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_k(next);                                       // (past the end: a block that was read before)
        __builtin_amdgcn_sched_barrier(0);
        f32x4 s = s0 + s1;
        float top = m_run;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (a.softcap > 0.f) s[e] = a.softcap * tanhf(s[e] / a.softcap);
            const bool ok = pooled ? block0 + e < my_blocks : key_visible(key0 + e, qpos, a.window, a.keep_first, a.chunk);
            s[e] = ok ? s[e] - slope * (float)(qpos - (key0 + e)) + biases[e] : -INFINITY;
            top = fmaxf(top, s[e]);
        }
        top = rows_max(top);
        // (a row that sees nothing yet keeps m = -inf)
        const float alpha = top == -INFINITY ? 1.f : expf(m_run - top);
        f32x4 p;
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = s[e] == -INFINITY ? 0.f : expf(s[e] - top);       // (unseen, or a bias that masks)
        l_run = l_run * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
        m_run = top;
        if (!pooled && kb + BLOCK - 1 > last_key) {          // what the page holds past the last key may be anything
#pragma unroll
            for (int c = 0; c < NVT; ++c) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[c][e] = key0 + e <= last_key ? v[c][e] : 0.f;
            }
        }
#pragma unroll
        for (int c = 0; c < NVT; ++c) acc[c] *= alpha;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int c = 0; c < NVT; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c][e], p[e], acc[c], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_v(next);
        __builtin_amdgcn_sched_barrier(0);
        k0 = next;
    }
    l_run = rows_sum(l_run);
    float* ml = smem + 4 * 16 * OLD;                         // [4][16][2]
    {
        float* out = smem + (wave * 16 + row) * OLD + 4 * quarter;
#pragma unroll
        for (int c = 0; c < NVT; ++c) *reinterpret_cast<f32x4*>(out + 16 * c) = acc[c];
        if (quarter == 0) {
            ml[(wave * 16 + row) * 2] = m_run;
            ml[(wave * 16 + row) * 2 + 1] = l_run;
        }
    }
    __syncthreads();
    // epilogue, 16 lanes a row: merge the waves, normalise, turn back by the query's position, gate
    const int qi = tid >> 4, sub = tid & 15;
    float weight[4], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, ml[(w * 16 + qi) * 2]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float mw = ml[(w * 16 + qi) * 2];
        weight[w] = mw == -INFINITY ? 0.f : expf(mw - m);
        l += weight[w] * ml[(w * 16 + qi) * 2 + 1];
    }
    float* os = smem + qi * OLD;                             // (the first wave's rows: every lane replaces the elements that it has read)
#pragma unroll
    for (int c = 0; c < NVT; ++c) {
        const int col = sub + 16 * c;
        float o = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) o += weight[w] * smem[(w * 16 + qi) * OLD + col];
        os[col] = l > 0.f ? o / l : 0.f;
    }
    __syncthreads();
    if (qi < nq) {
        const int64_t tok = qbase + (grouped ? 0 : q0 + qi);
        const int h = grouped ? head0 + qi : head0;
        const float g = a.gate ? a.gate[tok * a.H + h] : 1.0f, pos = (float)(past + (grouped ? 0 : q0 + qi));
#pragma unroll
        for (int c = 0; c < NVT; ++c) {
            const int col = sub + 16 * c;
            float x = os[col];
            if (a.v_freq) {
                int partner, pair;
                bool first;
                pair_of(col, vdim, a.v_interleaved, partner, pair, first);
                float sn, cs;
                rot_sincos<float>(pos * a.v_freq[pair], sn, cs);
                x = first ? x * cs + os[partner] * sn : x * cs - os[partner] * sn;      // the rotation by -pos
            }
            if (a.gate_elems) x *= elem_gate<float>(((const float*)a.gate_elems)[tok * a.ld_elems + h * vdim + col]);
            ((float*)a.out)[(tok * a.H + h) * vdim + col] = x * g;
        }
    }
}

template <int NKS, int NVT>
static void launch_attn_f32(const AttnArgs& a, int64_t total_q, hipStream_t st) {
    const size_t lds = sizeof(float) * (size_t)(4 * 16 * (16 * NVT + 4) + 4 * 16 * 2);
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_paged_f32_kernel<NKS, NVT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const bool grouped = !a.cu_seqlens_q;
    const dim3 grid(grouped ? (unsigned)a.batch : (unsigned)(total_q / AQ + a.batch), (unsigned)(grouped ? a.G * ((a.H / a.G + 15) / 16) : a.H));
    attn_paged_f32_kernel<NKS, NVT><<<grid, 256, lds, st>>>(a, grouped);
}

// Head sizes (dim / 16, vdim / 16) that the fp32 matrix-core form is built for; false: another one.
static bool dispatch_attn_f32(const AttnArgs& a, int64_t total_q, hipStream_t st) {
    if (a.dim % 16 || a.vdim % 16) return false;
#define NVH_ATTN_F32(K, V)                       \
    if (a.dim == 16 * K && a.vdim == 16 * V) {   \
        launch_attn_f32<K, V>(a, total_q, st);   \
        return true;                             \
    }
    NVH_ATTN_F32(1, 1) NVH_ATTN_F32(2, 2) NVH_ATTN_F32(4, 4) NVH_ATTN_F32(6, 6) NVH_ATTN_F32(8, 8) NVH_ATTN_F32(4, 8) NVH_ATTN_F32(8, 4) NVH_ATTN_F32(16, 12) NVH_ATTN_F32(16, 16)
#undef NVH_ATTN_F32
    return false;
}

// ---------------------------------------------------------------------------------------------------------------
// The same attention on the matrix cores, for bf16 caches with dim and vdim multiples of 16.  A workgroup is 64
// consecutive queries of one (sequence, head): four waves of 16 queries, all walking the same 64-key tiles (K rows and
// V transposed in LDS).  Per tile a wave forms S^T = K Q^T (lane: query lane%16, keys 4 (lane/16) + r of each 16-key
// block), keeps max / sum / weights in fp32, and accumulates O^T = V^T P^T with the weights as the B operand - as two
// bf16 terms, p = hi + lo, so a weight enters the product with 16 bits of mantissa and the sums stay fp32.  Tiles start
// at key 0 and every query has its own running maximum, so the result of a query does not depend on the cut or the batch.
typedef short s16x4 __attribute__((ext_vector_type(4)));
constexpr int MQ = 64, MK = 64;

// EXACT: dim == 16 NKS and vdim == 16 NVT, so no loop below carries a run-time bound (a guarded loop body is a branch, and the
// scheduler then cannot issue the LDS reads of several matrix instructions ahead of them).
// GROUPED (steps in which every sequence brings one query): a workgroup is one (sequence, KV head) and the 16 rows of a
// wave are the query heads that share this KV head, so its keys and values are read once for all of them; the four
// waves split every tile's keys and their partial results are merged at the end (the sums of a row are then formed in
// another order than in the other form: equal within fp32 rounding, not bit for bit).
// (The same split with 16 consecutive queries of one head as the rows was measured for prompts: no faster for one
// 1024-token chunk, 1.7-1.9 x slower from two chunks on, because it stages K/V four times as often.  Not kept.)
// VAR: the plain variant, the one with pooled blocks, softcap and query temperature, or the one with a learned distance bias (none
// carries code of the others).
enum AttnVariant { VAR_PLAIN, VAR_EXT, VAR_BIAS };
// One query per sequence: which sequence and group of heads a workgroup takes.  All workgroups of a step fit the chip a few to a CU, the ones numbered
// L and L + 256 beside each other, and as they lie that gives a CU the same long sequence twice.  So the work is dealt out by length: the
// longest sequences to the first 256 workgroups, the next ones to the next 256 in the opposite order, and so on.  Every workgroup ranks the
// sequences for itself; a result does not depend on where it is computed.
// us, as they lay and dealt out, 64 sequences of 512 .. 1535 keys, 8 KV heads: 128 x 128 51.2 and 46.3 in one model, 75.3 and 67.7 in another, with a
// query temperature or pooled blocks 54.5 and 49.2; 128 x 64 58.0 and 52.2; 64 x 128 72.8 and 69.7.
// The ranking costs each workgroup 0.7 us and more as the batch grows, and gives nothing where the sequences are short or alike (dealt out by as they
// lay, means over five forms of heads: 5 .. 60 keys 1.12 at 64 sequences, 1.24 at 100, 1.48 at 200; 300 keys each 1.05, 1.11, 1.21; 20 .. 275
// keys 0.97, 1.06, 1.23).  So there are at most 128 sequences, and the longest has to see a quarter more keys than the shortest and more than 192 of them,
// beyond 64 sequences more than 512 (a.balance; to find out that it does not costs 0.2 us: 6.4 us for 5 .. 60 keys were 6.2).
constexpr int BALANCE_MAX = 128;
constexpr int balance_from(int batch) { return batch <= 64 ? 192 : 512; }
__device__ __forceinline__ int balance_keys(const AttnArgs& a, int b) {      // keys that the sequence's query sees (roughly: what counts is the order)
    if (b >= a.batch) return -1;
    int len = a.context_lens[b];
    if (a.chunk > 0) len = len > 0 ? (len - 1) % a.chunk + 1 : 0;
    if (a.window > 0) len = min(len, a.window + a.keep_first);
    return len;
}
__device__ __forceinline__ int wave_max_of(int v) {                          // (0 .. 2^23: exact as floats, and in their order as integers)
    const int m = __float_as_int(row16_max((float)v));
    return (int)__int_as_float(max(max(__builtin_amdgcn_readlane(m, 0), __builtin_amdgcn_readlane(m, 16)), max(__builtin_amdgcn_readlane(m, 32), __builtin_amdgcn_readlane(m, 48))));
}
__device__ __forceinline__ bool balanced_place(const AttnArgs& a, int* keys, int& seq, int& by) {
    const int tid = threadIdx.x, lane = tid & 63, total = gridDim.x * gridDim.y, L = blockIdx.x + gridDim.x * blockIdx.y;
    const int len0 = balance_keys(a, lane), len1 = balance_keys(a, lane + 64);
    if (!__any(max(len0, len1) > a.balance)) return false;     // (every wave holds the same lengths: uniform, also over the workgroup)
    const int longest = wave_max_of(max(max(len0, len1), 0));
    const int spread = wave_max_of(max(len0 < 0 ? 0 : max(longest - len0, 0), len1 < 0 ? 0 : max(longest - len1, 0)));
    if (4 * spread < longest) return false;
    const int round = L >> 8, in_round = min(256, total - 256 * round), at = L & 255;
    const int item = 256 * round + (round & 1 ? in_round - 1 - at : at), want = item / (int)gridDim.y;
    const int len = tid < 64 ? len0 : len1;
    const int key = tid < a.batch ? (len << 8 | (255 - tid)) : -1;
    if (tid < BALANCE_MAX) keys[tid] = key;
    __syncthreads();
    int rank = 0;
    for (int j = 0; j < a.batch; j += 4) {                   // (four at a time: behind the batch lie the -1 of the lanes without a sequence)
        const int4 other = *reinterpret_cast<const int4*>(keys + j);
        rank += (other.x > key) + (other.y > key) + (other.z > key) + (other.w > key);
    }
    __syncthreads();
    if (tid < a.batch && rank == want) keys[0] = tid;
    __syncthreads();
    seq = __builtin_amdgcn_readfirstlane(keys[0]);
    by = item - want * (int)gridDim.y;
    __syncthreads();                                         // (the place is used for other things from here on)
    return true;
}

constexpr float LOG2E_F = 1.4426950408889634f;
// (two forms of the loop's arithmetic must not cost a wave per SIMD: as many as one form alone leaves room for)
// (32 x 32 would fit five in 96 registers: us, four and five, 32 heads over 8, 32 prompts of 1000 tokens 376 and 349, but 1024 behind 2000 77 and 80, 4 heads with
// slopes 64.9 and 68.5; learned bias, 1024 behind 2000, 48 and 56)
constexpr int attn_waves(int nks, int nvt, int mode, int var) { return nks + nvt <= 4 ? 4 : nks + nvt <= (mode == 1 && nvt <= 4 && var != VAR_EXT ? 12 : 8) ? 3 : nks + nvt <= 16 ? 2 : 1; }
// Wide heads leave one wave per SIMD and use its whole register file: there a second form of the loop's arithmetic costs more in registers than the
// masking that it leaves out, but for prompts without a window, chunk or slope, of which most tiles are seen whole.  FORMS: whether there are two.
// us, one form and two: 192 x 192, one query over each of 200 sequences, softcap 1.00 and 1.22 of one form's time; 160 x 128 in the bounded kernel, 64
// queries 0.99 and 1.11; 192 x 128, windows of 128 keys 0.99 and 1.06; whole prompts 256 x 256 0.99 and 0.92, 192 x 192 1.00 and 0.97, 128 x 256 0.99
// and 0.96 (all of the time that the masked form took before there were two).
constexpr bool attn_wide(int nks, int nvt) { return nks + nvt > 16; }
template <int NKS, int NVT, bool EXACT, int MODE, int VAR, bool FORMS>
__global__ __launch_bounds__(256, attn_waves(NKS, NVT, MODE, VAR)) void attn_paged_mfma_kernel(AttnArgs a) {
    constexpr bool GROUPED = MODE == 1;                      // rows are the heads of a KV group (one query per sequence)
    constexpr bool EXT = VAR == VAR_EXT, BIAS = VAR == VAR_BIAS;
    constexpr bool SPLIT = MODE != 0;                        // the waves share 16 rows and split the keys
    // LEAN: a row's maximum and its sum cross their four lanes on the vector ALU, and the values' rows lie in LDS as the products read them; the same bits as
    // the other form's.  us without and with it: 16 heads of 128 x 128 over 8, prompts of 1000 tokens 36.1 and 34.1, 1024 behind 2000 119.8 and 110.3, 32 of
    // 1000 575 and 536; 32 x 32, 1024 behind 2000 50.4 and 43.1; 64 single tokens behind 1024 (32 x 32) 16.2 and 14.5.  Wide heads, one wave a SIMD, are bound
    // by how their loop is laid out (with the scores' units of the next lines): 192 x 128 without a window 214 and 171, but with slopes 218 and 236; 256 x 256
    // 306 and 312.
    // (Scores kept times log2 e, which saves an instruction a weight, and a lane's sums left to the end, were 1 % faster still.  But such a score is rounded at its
    // own size instead of a weight at its distance from the maximum, and a bias or sink at the end of fp32's range leaves it.)
    constexpr bool LEAN = !attn_wide(NKS, NVT);
    constexpr int ROWS_Q = MQ;                               // queries per workgroup
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    int seq = -1, q0 = 0, qlen = 0, qbase = 0, by = blockIdx.y;
    if (GROUPED && a.balance && balanced_place(a, reinterpret_cast<int*>(smem_raw), seq, by)) {      // (uniform)
        qbase = seq;
        qlen = 1;
    } else if (!a.cu_seqlens_q) {                            // one query per sequence
        if ((int)blockIdx.x < a.batch) {
            seq = qbase = blockIdx.x;
            qlen = 1;
        }
    } else {
        int tile = blockIdx.x;
        for (int b = 0; b < a.batch; ++b) {
            const int lo = a.cu_seqlens_q[b], hi = a.cu_seqlens_q[b + 1];
            const int tiles = (hi - lo + ROWS_Q - 1) / ROWS_Q;
            if (tile < tiles) {
                seq = b;
                q0 = tile * ROWS_Q;
                qlen = hi - lo;
                qbase = lo;
                break;
            }
            tile -= tiles;
        }
    }
    if (seq < 0) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
    // GROUPED: `by` counts (KV head, part of its group of heads); the parts of one KV head read the same keys and values
    const int group = GROUPED ? a.H / (a.G * a.kv_split) : a.H / a.G;
    const int kvh = GROUPED ? by / a.kv_split : by / group;
    const int head = GROUPED ? by * group + min(fr, group - 1) : by;       // (GROUPED: this lane's row is a head)
    const int dim = EXACT ? 16 * NKS : a.dim, vdim = EXACT ? 16 * NVT : a.vdim, nks = dim >> 4, nvt = vdim >> 4;
    const int klen = a.context_lens[seq], past = klen - qlen;
    const int nq = GROUPED ? 1 : min(ROWS_Q, qlen - q0);
    const int nrows = GROUPED ? group : nq;                  // real rows of the workgroup's 64
    const int kld = dim + 8, vld = MK + 8;                   // LDS row strides in elements (16-byte aligned rows)
    // Place of key k in a column's row of V: of every 32 keys a lane's eight (four of either 16-key block) lie side by side, a 16-byte read that meets no
    // bank twice.
    auto vplace = [](int k) { return !LEAN ? k : (k & ~31) | (k >> 2 & 3) << 3 | (k >> 4 & 1) << 2 | (k & 3); };
    bf16* ks = reinterpret_cast<bf16*>(smem_raw);            // [MK][dim + 8]
    bf16* vt = ks + MK * kld;                                // [vdim][MK + 8]: V transposed
    // GROUPED: every wave holds the same 16 rows (heads) and takes the 16 keys kt = wave of every 64-key tile, with its own
    // running maximum, sum and output; the four partial results are merged at the end.
    const int qrow = SPLIT ? fr : wave * 16 + fr;            // this lane's row within the workgroup
    const bool qok = qrow < nrows;
    constexpr int NKT = SPLIT ? 1 : 4;                       // 16-key blocks of a tile per wave
    const int qpos = GROUPED ? past : past + q0 + qrow;
    const int last_key = past + q0 + nq - 1;
    const int part = GROUPED ? (int)blockIdx.z : 0, nparts = GROUPED ? a.key_parts : 1;
    float* prow = nullptr;                                   // this workgroup's record among the parts
    if (GROUPED && nparts > 1) prow = a.parts + (((int64_t)seq * gridDim.y + by) * nparts + part) * 16 * (vdim + 2);
    if (last_key < 0 && prow) {                              // a padded row: every part records "no keys", the merge then writes zeros
        if (tid < 16) {
            prow[tid * (vdim + 2) + vdim] = -INFINITY;
            prow[tid * (vdim + 2) + vdim + 1] = 0.f;
        }
        return;
    }
    if (last_key < 0) {                                      // a padded row of a captured step (no keys): zeros, and no address is formed
        for (int i = tid; i < nrows * vdim; i += 256) {
            const int r = i / vdim;
            const int64_t tok = GROUPED ? qbase : qbase + q0 + r;
            const int hd = GROUPED ? by * group + r : by;
            ((bf16*)a.out)[(tok * a.H + hd) * vdim + (i - r * vdim)] = (bf16)0.f;
        }
        return;
    }
    const bf16* qg = (const bf16*)a.q + (int64_t)(qbase + q0 + (qok && !GROUPED ? qrow : 0)) * a.ldq + head * dim;
    // A lane's part of the query row: eight columns of every 32 (K32 products of 32; of a last 16 columns the lanes of the product's first
    // half hold eight each and the others zeros) or, where the size is not a constant, four columns of every 16.  A chain of dependent
    // products keeps to one shape: a product of 16 right behind a product of 32 that it adds to has given wrong sums.  The empty statements make
    // the loads complete here: a load still under way at its first use in the tile loop would put a wait for ALL loads, those of the
    // tile after next included, into every turn.
    constexpr int K32 = EXACT ? (NKS + 1) / 2 : 0, K16 = EXACT ? 0 : NKS;
    constexpr bool HALF = EXACT && NKS % 2 == 1;             // the last product of 32 has 16 columns
    auto kcol = [&](int i) { return i * 32 + (HALF && i == K32 - 1 ? (fq & 1) * 8 : fq * 8); };
    bf16x8 qf32[K32 > 0 ? K32 : 1];
    s16x4 qf16[K16 > 0 ? K16 : 1];
#pragma unroll
    for (int i = 0; i < K32; ++i) {
        qf32[i] = *reinterpret_cast<const bf16x8*>(qg + kcol(i));
        if (HALF && i == K32 - 1 && fq >= 2) qf32[i] = bf16x8{};
    }
#pragma unroll
    for (int i = 0; i < K16; ++i)
        if (i < nks) qf16[i] = *reinterpret_cast<const s16x4*>(qg + i * 16 + fq * 4);
        else qf16[i] = s16x4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < K32; ++i) asm volatile("" : "+v"(qf32[i]));
#pragma unroll
    for (int i = 0; i < K16; ++i) asm volatile("" : "+v"(qf16[i]));
    f32x4 o[NVT];
#pragma unroll
    for (int i = 0; i < NVT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    if (a.sinks && (!SPLIT || (wave == 0 && part == 0))) {   // the sink is what a row starts from; where waves or parts share a row, one of them holds it
        m_run = a.sinks[head];
        l_run = 1.f;
    }
    const int32_t* table = a.block_tables + (int64_t)seq * a.table_stride;
    const bool wave_idle = !SPLIT && wave * 16 >= nrows;     // no row of this wave is real
    const int wave_last = SPLIT ? last_key : past + q0 + min(wave * 16 + 15, nq - 1);   // keys beyond it are masked for the whole wave
    // A tile's global loads (16 bytes each; K rows as they lie, V rows = value columns over 64 consecutive keys of one page)
    // are issued two tiles ahead into registers, without a condition (past the end: the last tile once more), so that the number of
    // loads under way is the same on every path; what lies beyond the last key is zeroed on the way into LDS.
    constexpr int KCH = (NKS + 1) / 2, VCH = (NVT + 1) / 2;  // 16-byte pieces per lane: MK * dim / 8 / 256
    const int kcols = dim >> 3;
    // The sequence's page ids go to LDS once: a tile's addresses then hang on no other load.  A tile lies within one page
    // (page % MK == 0).
    int* pages_s = reinterpret_cast<int*>(smem_raw + a.pages_offset);
    for (int i = tid; i <= last_key / a.page; i += 256) pages_s[i] = table[i];
    // The heads' bias rows too, each with three entries in front of distance 0 (never seen) and behind the last: a lane's four scores
    // of consecutive keys then read four consecutive entries wherever they start.
    const float* bias_row = nullptr;
    if constexpr (BIAS) {
        float* bias_s = reinterpret_cast<float*>(smem_raw + a.bias_offset);
        const int heads_here = GROUPED ? group : 1;
        const float* src = a.bias + (int64_t)(GROUPED ? by * group : head) * a.bias_len;
        for (int i = tid; i < heads_here * a.bias_ld; i += 256) {
            const int r = i / a.bias_ld, d = i - r * a.bias_ld - 3;
            bias_s[i] = src[(int64_t)r * a.bias_len + min(max(d, 0), a.bias_len - 1)];
        }
        bias_row = bias_s + (GROUPED ? min(fr, group - 1) : 0) * a.bias_ld + 3;
    }
    __syncthreads();
    auto fetch = [&](int k0, bf16x8 (&kpre)[KCH], bf16x8 (&vpre)[VCH]) {
        const int64_t pg = __builtin_amdgcn_readfirstlane(pages_s[k0 / a.page]);     // (uniform)
        const int in_page = k0 % a.page, krow = a.G * dim;
        const bf16* kbase = (const bf16*)a.k_cache + ((pg * a.page + in_page) * a.G + kvh) * dim;
        const bf16* vbase = (const bf16*)a.v_cache + (pg * a.G + kvh) * vdim * a.page + in_page;
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            const int i = tid + 256 * j;
            kpre[j] = *reinterpret_cast<const bf16x8*>(kbase + (uint32_t)(min(i / kcols, MK - 1) * krow + ((i % kcols) << 3)));
        }
#pragma unroll
        for (int j = 0; j < VCH; ++j) {
            const int i = tid + 256 * j;
            vpre[j] = *reinterpret_cast<const bf16x8*>(vbase + (uint32_t)(min(i >> 3, vdim - 1) * a.page + ((i & 7) << 3)));
        }
    };
    auto store_keys = [&](int rows, bf16x8 (&kpre)[KCH]) {   // rows: those of the tile that hold anything
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            const int i = tid + 256 * j;
            if ((EXACT && 256 * (j + 1) <= MK * kcols) || i < MK * kcols) {
                const int r = i / kcols, c = (i % kcols) << 3;
                *reinterpret_cast<bf16x8*>(ks + r * kld + c) = r < rows ? kpre[j] : bf16x8{};
            }
        }
    };
    const float slope = a.slopes ? a.slopes[head] : 0.f;
    const float row_scale = EXT ? a.scale * query_temperature(qpos, a.temp_coef, a.temp_every) : a.scale;
    const float cap_in = EXT && a.softcap > 0.f ? 2.0f * LOG2E_F / a.softcap : 0.f;          // tanh(s / cap) = 1 - 2 / (2^(cap_in s) + 1)
    const int nblocks = EXT && a.pool > 0 ? blocks_seen(last_key, a.window, a.pool) : 0, my_blocks = EXT && a.pool > 0 ? blocks_seen(qpos, a.window, a.pool) : 0;
    // keys a row sees: lo_window (or one of the first keep_first) and lo_chunk at least, qpos at most
    const int lo_window = a.window > 0 ? qpos - a.window + 1 : 0, lo_chunk = a.chunk > 0 ? qpos / a.chunk * a.chunk : 0;
    // A tile between these two is seen whole by every row of the wave (uniform): nothing to mask.  Most of a long context is, and the work per
    // score bounds the loop.
    // us, every tile masked and so: 16 heads of 128 x 128 over 8, prompts of 1024 tokens 57.3 and 45.6, 32 of 1000 727 and 577, 1024 behind 3072 204 and 156, 8 of
    // 100 14.6 and 13.4; 64 single tokens behind 1024 57.8 and 55.2.
    const int wave_first = __builtin_amdgcn_readfirstlane(SPLIT ? qpos : past + q0 + wave * 16), wave_lastq = __builtin_amdgcn_readfirstlane(wave_last);
    const int whole_from = max(a.window > 0 ? wave_lastq - a.window + 1 : 0, a.chunk > 0 ? wave_lastq / a.chunk * a.chunk : 0);
    const int whole_to = a.slopes ? -1 : wave_first - MK + 1;                // (first keys from .. to, both included)
    // The tile in LDS, its first key k0 (pooled_tile: its first block) against this wave's queries.
    auto compute = [&](auto pooled_tile, auto whole_tile, int k0) {
        constexpr bool POOLED = decltype(pooled_tile)::value, WHOLE = decltype(whole_tile)::value;
        // (wave-uniform; no barrier below)
        if (wave_idle || (POOLED ? k0 >= blocks_seen(wave_last, a.window, a.pool) : k0 > wave_last)) return;
        f32x4 sc[NKT];
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            const int kt = SPLIT ? wave : t;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < K32; ++i) {
                const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + (kt * 16 + fr) * kld + kcol(i));
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf32[i], acc, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < K16; ++i)
                if (i < nks) {
                    const s16x4 kf = *reinterpret_cast<const s16x4*>(ks + (kt * 16 + fr) * kld + i * 16 + fq * 4);
                    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(kf, qf16[i], acc, 0, 0, 0);
                }
            sc[t] = acc;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            // (distances beyond the row's last entry take its value; negative ones belong to keys that are not seen)
            const float* brow = nullptr;
            if constexpr (BIAS) brow = bias_row + min(max(qpos - (k0 + (SPLIT ? wave : t) * 16 + fq * 4) - 3, -3), a.bias_len - 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = k0 + (SPLIT ? wave : t) * 16 + fq * 4 + r;
                float v;
                if constexpr (BIAS) {
                    v = __builtin_fmaf(sc[t][r], row_scale, brow[3 - r]);
                } else {
#pragma clang fp contract(off)                               // (one rounding in either form: a row's bits do not depend on where its wave begins)
                    v = sc[t][r] * row_scale;
                }
                if (EXT && cap_in > 0.f) v = a.softcap - 2.0f * a.softcap * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * cap_in) + 1.0f);
                if constexpr (!WHOLE) {
                    const bool seen = POOLED ? key < my_blocks : (key <= qpos) & ((key >= lo_window) | (key < a.keep_first)) & (key >= lo_chunk);
                    if (!BIAS && !POOLED) v = __builtin_fmaf(-slope, (float)(qpos - key), v);
                    v = (qok & seen) ? v : -INFINITY;
                }
                sc[t][r] = v;
                mx = fmaxf(mx, sc[t][r]);
            }
        }
        if constexpr (LEAN) {
            mx = rows_max(mx);
        } else {
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        }
        const float m_new = fmaxf(m_run, mx);
        // e^x as the hardware's 2^(x log2 e): fp32 throughout, about 1 ulp of the distance from the maximum, wherever the scores lie
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E_F);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;                // (a row that has seen nothing: its scores are -inf, their weights 0)
        float sum = 0.f;
        // The weights as the B operand of products over 32 rows: of two 16-key blocks, once with hi and once with lo - or, where a wave
        // has one block only, of that block's keys twice, with hi and with lo
        constexpr int NP = SPLIT ? 1 : NKT / 2;
        bf16x8 pf[NP], pg[NP];
#pragma unroll
        for (int t = 0; t < NKT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (the test: the same value, but without it the form that is not LEAN is laid out so that it takes up to a tenth longer)
                const float pv = !LEAN && !WHOLE && sc[t][r] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((sc[t][r] - m_ref) * LOG2E_F);
                sum += pv;
                const bf16 hi = (bf16)pv;
                const bf16 lo = (bf16)(pv - (float)hi);
                if constexpr (SPLIT) {
                    pf[0][r] = hi;
                    pf[0][4 + r] = lo;
                } else {
                    pf[t / 2][t % 2 * 4 + r] = hi;
                    pg[t / 2][t % 2 * 4 + r] = lo;
                }
            }
        if constexpr (LEAN) {
            sum = rows_sum(sum);
        } else {
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
        }
        l_run = l_run * alpha + sum;
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < NVT; ++i)
            if (EXACT || i < nvt) {
                f32x4 acc = o[i] * alpha;
                const bf16* vrow = vt + (i * 16 + fr) * vld + fq * (LEAN ? 8 : 4);
#pragma unroll
                for (int t = 0; t < NP; ++t) {
                    bf16x8 vf;
                    if constexpr (SPLIT) {
                        const bf16x4 v0 = *reinterpret_cast<const bf16x4*>(vrow + (LEAN ? (wave >> 1) * 32 + (wave & 1) * 4 : wave * 16));
                        vf = __builtin_shufflevector(v0, v0, 0, 1, 2, 3, 4, 5, 6, 7);
                    } else if constexpr (LEAN) {
                        vf = *reinterpret_cast<const bf16x8*>(vrow + t * 32);
                    } else {
                        const bf16x4 v0 = *reinterpret_cast<const bf16x4*>(vrow + 2 * t * 16), v1 = *reinterpret_cast<const bf16x4*>(vrow + (2 * t + 1) * 16);
                        vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
                    }
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[t], acc, 0, 0, 0);
                    if constexpr (!SPLIT) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pg[t], acc, 0, 0, 0);
                }
                o[i] = acc;
            }
    };
    auto tile = [&](int k0, int k_after, bf16x8 (&kpre)[KCH], bf16x8 (&vpre)[VCH]) {
        __syncthreads();
        store_keys(last_key - k0 + 1, kpre);
#pragma unroll
        for (int j = 0; j < VCH; ++j) {
            const int i = tid + 256 * j;
            if ((EXACT && 256 * (j + 1) <= vdim * 8) || i < vdim * 8) {
                const int c = i >> 3, piece = (i & 7) << 3;
                bf16x8 v = vpre[j];
                if (k0 + MK - 1 > last_key) {                // (uniform: only the sequence's last tile)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (k0 + piece + e > last_key) v[e] = (bf16)0.f;
                }
                bf16* dst = vt + c * vld + vplace(piece);
                if constexpr (LEAN) {
                    *reinterpret_cast<bf16x4*>(dst) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
                    *reinterpret_cast<bf16x4*>(dst + 8) = __builtin_shufflevector(v, v, 4, 5, 6, 7);
                } else {
                    *reinterpret_cast<bf16x8*>(dst) = v;
                }
            }
        }
        __syncthreads();
        fetch(k_after, kpre, vpre);
        if (FORMS && k0 >= whole_from && k0 <= whole_to) compute(std::false_type{}, std::true_type{}, k0);
        else compute(std::false_type{}, std::false_type{}, k0);
    };
    // Two register sets, two tiles ahead: the loads of the tile after next are issued when a tile has been handed to LDS.
    bf16x8 kA[KCH], vA[VCH], kB[KCH], vB[VCH];
    const TileWalk walk(a.window, a.keep_first, a.chunk, GROUPED ? past : past + q0, MK);
    // (with key parts a workgroup walks the tiles whose number is its own modulo the number of parts)
    auto mine = [&](int k0) { return nparts == 1 || (k0 / MK) % nparts == part; };
    auto next_tile = [&](int k0) {
        int n = walk.next(k0);
        while (n <= last_key && !mine(n)) n = walk.next(n);
        return n;
    };
    int ka = walk.first_end > 0 || walk.win_start == 0 ? 0 : walk.win_start;
    if (!mine(ka)) ka = next_tile(ka);
    int kb = next_tile(ka);
    if (ka > last_key) kb = ka;
    const int k_last = last_key / MK * MK;                   // the tile that holds the last key
    fetch(min(ka, k_last), kA, vA);
    __builtin_amdgcn_sched_barrier(0);                       // (the loads of the first tile stay ahead of the second's)
    if constexpr (EXT) {
        // The tiles of block means come first, one ahead: rows as they lie in their pages, keys in the pieces of a token tile, values in
        // pieces of eight columns of one row (a wave takes 64 rows of the same columns, so its transposed writes into LDS fall side by side).
        auto fetch_pooled = [&](int b0) {
            auto row_of = [&](int r) {
                int pi, row;
                block_place(min(b0 + r, nblocks - 1), a.pool, a.page, pi, row);
                return ((int64_t)pages_s[pi] * a.pool_rows + row) * a.G + kvh;
            };
#pragma unroll
            for (int j = 0; j < KCH; ++j) {
                const int i = tid + 256 * j;
                kB[j] = *reinterpret_cast<const bf16x8*>((const bf16*)a.pk + row_of(min(i / kcols, MK - 1)) * dim + ((i % kcols) << 3));
            }
            const int64_t vrow = row_of(tid & (MK - 1)) * vdim;
#pragma unroll
            for (int j = 0; j < VCH; ++j)
                vB[j] = *reinterpret_cast<const bf16x8*>((const bf16*)a.pv + vrow + min(((tid + 256 * j) / MK) << 3, vdim - 8));
        };
        const int bstep = MK * nparts;
        int b0 = MK * part;
        if (b0 < nblocks) fetch_pooled(b0);
        for (; b0 < nblocks; b0 += bstep) {
            __syncthreads();
            store_keys(nblocks - b0, kB);
#pragma unroll
            for (int j = 0; j < VCH; ++j) {
                const int i = tid + 256 * j, r = i & (MK - 1), c = (i / MK) << 3;
                if (c < vdim) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) vt[(c + e) * vld + vplace(r)] = r < nblocks - b0 ? vB[j][e] : (bf16)0.f;
                }
            }
            __syncthreads();
            fetch_pooled(b0 + bstep);                        // (past the end: the last block's row once more)
            compute(std::true_type{}, std::false_type{}, b0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    fetch(min(kb, k_last), kB, vB);
    __builtin_amdgcn_sched_barrier(0);
    while (kb <= last_key) {                                 // (one way out: with a second one the waits would count for the shorter path)
        const int ka2 = next_tile(kb), kb2 = next_tile(ka2);
        tile(ka, min(ka2, k_last), kA, vA);
        tile(kb, min(kb2, k_last), kB, vB);
        ka = ka2;
        kb = kb2;
    }
    if (ka <= last_key) tile(ka, ka, kA, vA);
    // epilogue through LDS: [MQ][vdim] fp32, then turn back by the query's position, gate, store
    __syncthreads();
    float* os = reinterpret_cast<float*>(smem_raw);
    if constexpr (SPLIT) {
        // the four waves' partial results [wave][16 rows][vdim] and their (max, sum), merged into the first wave's rows
        float* ml = reinterpret_cast<float*>(smem_raw + a.ml_offset);
#pragma unroll
        for (int i = 0; i < NVT; ++i)
            if (EXACT || i < nvt)
#pragma unroll
                for (int r = 0; r < 4; ++r) os[(wave * 16 + fr) * vdim + i * 16 + fq * 4 + r] = o[i][r];
        if (fq == 0) {
            ml[(wave * 16 + fr) * 2] = m_run;
            ml[(wave * 16 + fr) * 2 + 1] = l_run;
        }
        __syncthreads();
        for (int i = tid; i < nrows * vdim; i += 256) {
            const int r = i / vdim, col = i - r * vdim;
            float big = -INFINITY;
#pragma unroll
            for (int w = 0; w < 4; ++w) big = fmaxf(big, ml[(w * 16 + r) * 2]);
            float num = 0.f, den = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float mw = ml[(w * 16 + r) * 2];
                const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((mw - big) * LOG2E_F);
                num += os[(w * 16 + r) * vdim + col] * f;
                den += ml[(w * 16 + r) * 2 + 1] * f;
            }
            if (prow) {                                      // a part's record: the row relative to its maximum, then maximum and sum
                prow[r * (vdim + 2) + col] = num;
                if (col == 0) {
                    prow[r * (vdim + 2) + vdim] = big;
                    prow[r * (vdim + 2) + vdim + 1] = den;
                }
            } else {
                os[i] = den > 0.f ? num / den : 0.f;         // (element i of the first wave's rows: read above by this lane only)
            }
        }
        if (prow) return;                                    // (uniform) the merge launch finishes the rows
    } else {
        const float inv_l = l_run > 0.f ? 1.0f / l_run : 0.f;
#pragma unroll
        for (int i = 0; i < NVT; ++i)
            if (EXACT || i < nvt)
#pragma unroll
                for (int r = 0; r < 4; ++r) os[qrow * vdim + i * 16 + fq * 4 + r] = o[i][r] * inv_l;
    }
    __syncthreads();
    if (!a.v_freq) {                                         // nothing to turn back: eight elements a lane (vdim is a multiple of 16)
        const int pieces = vdim >> 3;
        for (int i = tid; i < nrows * pieces; i += 256) {
            const int r = i / pieces, c = (i - r * pieces) << 3;
            const int64_t tok = GROUPED ? qbase : qbase + q0 + r;
            const int hd = GROUPED ? by * group + r : by;
            const float g = a.gate ? a.gate[tok * a.H + hd] : 1.0f;
            bf16x8 ge, out;
            if (a.gate_elems) ge = *reinterpret_cast<const bf16x8*>((const bf16*)a.gate_elems + tok * a.ld_elems + hd * vdim + c);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = os[r * vdim + c + e] * g;
                if (a.gate_elems) v *= elem_gate<bf16>((float)ge[e]);
                out[e] = (bf16)v;
            }
            *reinterpret_cast<bf16x8*>((bf16*)a.out + (tok * a.H + hd) * vdim + c) = out;
        }
        return;
    }
    // one lane per rotation pair: both elements, one sine and cosine
    const int half = vdim >> 1;
    for (int i = tid; i < nrows * half; i += 256) {
        const int r = i / half, pair = i - r * half;
        const int c1 = a.v_interleaved ? 2 * pair : pair, c2 = a.v_interleaved ? 2 * pair + 1 : pair + half;
        const int64_t tok = GROUPED ? qbase : qbase + q0 + r;
        const int hd = GROUPED ? by * group + r : by;
        float u = os[r * vdim + c1], v = os[r * vdim + c2];
        if (a.v_freq) {
            float sn, cs;
            sincos_turns((float)(GROUPED ? past : past + q0 + r) * a.v_freq[pair], sn, cs);
            const float u2 = u * cs + v * sn;                // the rotation by -position
            v = v * cs - u * sn;
            u = u2;
        }
        const float g = a.gate ? a.gate[tok * a.H + hd] : 1.0f;
        bf16* dst = (bf16*)a.out + (tok * a.H + hd) * vdim;
        dst[c1] = (bf16)(u * g);
        dst[c2] = (bf16)(v * g);
    }
}

// The rows of the key parts of a (sequence, group of heads) merged: out = gate * sum_p num_p e^(m_p - m) / sum_p den_p e^(m_p - m).
__global__ __launch_bounds__(256) void attn_merge_parts_kernel(const float* __restrict__ parts, int nparts, int rows, int vdim, int H, const float* __restrict__ gate,
                                                               const bf16* __restrict__ gate_elems, int64_t ld_elems, bf16* __restrict__ out) {
    // one workgroup per (sequence, group of heads, row): a lane per value column
    const int seq = blockIdx.x, hg = blockIdx.y, r = blockIdx.z;
    const float* base = parts + (((int64_t)seq * gridDim.y + hg) * nparts * 16 + r) * (vdim + 2);
    const int64_t pstride = (int64_t)16 * (vdim + 2);
    float big = -INFINITY;
    for (int p = 0; p < nparts; ++p) big = fmaxf(big, base[p * pstride + vdim]);
    const int hd = hg * rows + r;
    const float g = gate ? gate[(int64_t)seq * H + hd] : 1.0f;
    for (int col = threadIdx.x; col < vdim; col += 256) {
        float num = 0.f, den = 0.f;
        for (int p = 0; p < nparts; ++p) {
            const float* pr = base + p * pstride;
            if (pr[vdim] == -INFINITY) continue;             // a part without keys (its row is not written)
            const float f = __builtin_amdgcn_exp2f((pr[vdim] - big) * LOG2E_F);
            num += pr[col] * f;
            den += pr[vdim + 1] * f;
        }
        float v = den > 0.f ? num / den * g : 0.f;
        if (gate_elems) v *= elem_gate<bf16>((float)gate_elems[seq * ld_elems + (int64_t)hd * vdim + col]);
        out[((int64_t)seq * H + hd) * vdim + col] = (bf16)v;
    }
}

// One query per sequence: the heads of a KV group share a workgroup - up to 16 of them; a larger group is cut into parts.  A launch
// that would leave most of the chip idle is widened: where nothing turns the values back (no v_freq) by giving a sequence's key
// tiles to several workgroups in turn, whose rows a second launch merges (the keys and values are still read once); otherwise by
// cutting the group of heads further (its parts then read the same keys and values at about the same time).  Which workgroup a
// head or a tile falls to enters the result within fp32 rounding only (the order of the merge).
struct OneQueryPlan {
    int split, key_parts;
};
static OneQueryPlan one_query_plan(int64_t batch, int H, int G, bool turned_back) {
    const int group = H / G;
    int split = 1;
    while (group / split > 16 && group % (2 * split) == 0) split *= 2;
    int parts = 1;
    if (!turned_back) {
        while (batch * G * split * parts * 2 <= 256 && parts < 16) parts *= 2;       // (two workgroups a CU measured slower: 53 against 37 us)
    } else {
        while (batch * G * split < 256 && group % (2 * split) == 0 && group / split > 2) split *= 2;
    }
    return OneQueryPlan{split, parts};
}
static size_t one_query_parts_bytes(int64_t batch, int H, int G, int vdim, bool turned_back) {
    const OneQueryPlan pl = one_query_plan(batch, H, G, turned_back);
    return pl.key_parts > 1 ? sizeof(float) * (size_t)batch * G * pl.split * pl.key_parts * 16 * (vdim + 2) : 0;
}

// The bias rows in LDS: at most BIAS_LDS bytes (the caller makes sure that one row fits; a group of heads whose rows do not takes the
// form with one head per workgroup).
constexpr size_t BIAS_LDS = 64 * 1024;
static int bias_row_floats(int bias_len) { return (bias_len + 6) | 1; }      // (odd: the rows of a group start in different banks)

template <int NKS, int NVT, bool EXACT, int VAR>
static void launch_attn_mfma(const AttnArgs& a, int64_t total_q, hipStream_t st) {
    const size_t tiles = sizeof(bf16) * ((size_t)MK * (a.dim + 8) + (size_t)a.vdim * (MK + 8));
    const size_t outs = sizeof(float) * (size_t)MQ * a.vdim;
    AttnArgs b = a;
    b.pages_offset = (int)(((tiles > outs ? tiles : outs) + 15) & ~(size_t)15);
    b.ml_offset = (int)((b.pages_offset + sizeof(int) * (size_t)a.table_stride + 15) & ~(size_t)15);
    b.bias_offset = (int)(b.ml_offset + sizeof(float) * 4 * 16 * 2);
    const int group = a.H / a.G;
    OneQueryPlan pl = one_query_plan(a.batch, a.H, a.G, a.v_freq != nullptr);
    if (!a.parts) pl.key_parts = 1;
    size_t bias_bytes = 0, bias_group_bytes = 0;             // of one head, of the heads of a one-query workgroup
    if (VAR == VAR_BIAS) {
        b.bias_ld = bias_row_floats(a.bias_len);
        bias_bytes = sizeof(float) * (size_t)b.bias_ld;
        bias_group_bytes = bias_bytes * (group / pl.split);
    }
    const bool grouped = total_q == a.batch && group / pl.split <= 16 && bias_group_bytes <= BIAS_LDS && !nvh_switch_on(SW_EXP_A);
    const size_t lds = b.bias_offset + (grouped ? bias_group_bytes : bias_bytes);
    constexpr bool WIDE = attn_wide(NKS, NVT);
    const auto one_query = &attn_paged_mfma_kernel<NKS, NVT, EXACT, 1, VAR, !WIDE>, prompt = &attn_paged_mfma_kernel<NKS, NVT, EXACT, 0, VAR, !WIDE>;
    const auto prompt_two = &attn_paged_mfma_kernel<NKS, NVT, EXACT, 0, VAR, !WIDE || (EXACT && VAR == VAR_PLAIN)>;
    const bool two_forms = !a.window && !a.chunk && !a.slopes;
    if (lds > 64 * 1024)                                     // (wide heads or long page tables; a refusal shows as a failed launch)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(grouped ? one_query : two_forms ? prompt_two : prompt), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (grouped) {
        b.kv_split = pl.split;
        b.key_parts = pl.key_parts;
        // (one workgroup a CU or less: nothing to pair; lengths of 2^23 and more do not fit the keys; a query that cannot see many keys: balanced_place)
        int64_t most = (int64_t)a.table_stride * a.page;
        b.balance = pl.key_parts == 1 && a.batch <= BALANCE_MAX && (int64_t)a.batch * a.G * pl.split > 256 && most < (1 << 23) ? balance_from(a.batch) : 0;
        if (a.chunk > 0) most = std::min(most, (int64_t)a.chunk);
        if (a.window > 0) most = std::min(most, (int64_t)a.window + a.keep_first);
        if (most <= b.balance) b.balance = 0;
        one_query<<<dim3((unsigned)a.batch, (unsigned)(a.G * pl.split), (unsigned)pl.key_parts), 256, lds, st>>>(b);
        if (pl.key_parts > 1)
            attn_merge_parts_kernel<<<dim3((unsigned)a.batch, (unsigned)(a.G * pl.split), (unsigned)(group / pl.split)), 256, 0, st>>>(a.parts, pl.key_parts, group / pl.split, a.vdim, a.H, a.gate,
                                                                                                        (const bf16*)a.gate_elems, a.ld_elems, (bf16*)a.out);
    } else {
        const dim3 grid((unsigned)(total_q / MQ + a.batch), (unsigned)a.H);
        (two_forms ? prompt_two : prompt)<<<grid, 256, lds, st>>>(b);
    }
}

// Exact instantiations for the head sizes in use (dim/16, vdim/16); any other 16-aligned pair takes a bounded one.
#define NVH_ATTN_EXACT(X) X(1, 1) X(2, 2) X(3, 3) X(4, 4) X(5, 5) X(6, 6) X(8, 8) X(12, 12) X(16, 16) X(2, 4) X(4, 2) X(4, 8) X(8, 4) X(8, 16) X(16, 8) X(12, 8) X(16, 12)
// The variant with pooled blocks, softcap or query temperature: fewer exact pairs.
#define NVH_ATTN_EXACT_EXT(X) X(2, 2) X(4, 4) X(6, 6) X(8, 8) X(16, 16) X(4, 8) X(8, 4) X(8, 16) X(16, 8)
// ... and the one with a learned distance bias.
#define NVH_ATTN_EXACT_BIAS(X) X(2, 2) X(3, 3) X(4, 4) X(5, 5) X(6, 6) X(8, 8) X(12, 12) X(16, 16) X(4, 8) X(8, 4) X(8, 16) X(16, 8)
template <int VAR>
static void dispatch_attn_mfma(const AttnArgs& a, int64_t total_q, hipStream_t st) {
    const int nks = a.dim / 16, nvt = a.vdim / 16;
#define NVH_ATTN_CASE(K, V)                              \
    if (nks == K && nvt == V) {                          \
        launch_attn_mfma<K, V, true, VAR>(a, total_q, st); \
        return;                                          \
    }
    if constexpr (VAR == VAR_EXT) {
        NVH_ATTN_EXACT_EXT(NVH_ATTN_CASE)
    } else if constexpr (VAR == VAR_BIAS) {
        NVH_ATTN_EXACT_BIAS(NVH_ATTN_CASE)
    } else {
        NVH_ATTN_EXACT(NVH_ATTN_CASE)
    }
#undef NVH_ATTN_CASE
    if (nks <= 4 && nvt <= 4) launch_attn_mfma<4, 4, false, VAR>(a, total_q, st);
    else if (nks <= 8 && nvt <= 8) launch_attn_mfma<8, 8, false, VAR>(a, total_q, st);
    else launch_attn_mfma<16, 16, false, VAR>(a, total_q, st);
}

// The means of the blocks that were filled by this step, one block per workgroup (blockIdx.x; several workgroups, blockIdx.y, share its
// columns): block b of a sequence is due when its last position is among the step's.  Rows are read from the cache as it holds them.
struct PoolArgs {
    const void *k_cache, *v_cache;
    const int32_t *cu_seqlens_q, *context_lens, *block_tables;
    int64_t table_stride;
    int batch, page, G, dim, vdim, pool, pool_rows;
    void *pk, *pv;
};

// The mean of column i (of n) over block b of a sequence, from the rows that the cache holds (values: transposed within a page).
template <typename A>
__device__ __forceinline__ void block_mean_column(const A* cache, A* pooled, int i, int n, bool transposed, int b, int pool, int page, int pool_rows, const int32_t* table) {
    const int p0 = b * pool;
    int pi = p0 / page;
    const int off0 = p0 - pi * page;
    float sum = 0.f;
    // (a block may lie across pages: page by page, each a plain run of rows)
    for (int done = 0, off = off0; done < pool; off = 0, ++pi) {
        const int n_here = min(pool - done, page - off);
        const int64_t pg = table[pi];
        const A* src = transposed ? cache + (pg * n + i) * page + off : cache + (pg * page + off) * n + i;
        const int64_t step = transposed ? 1 : n;
#pragma unroll 8
        for (int j = 0; j < n_here; ++j) sum += ldf(src, j * step);
        done += n_here;
    }
    int pi_out, row;
    block_place(b, pool, page, pi_out, row);
    pooled[((int64_t)table[pi_out] * pool_rows + row) * n + i] = (A)(sum / (float)pool);
}

template <typename A>
__global__ __launch_bounds__(256) void attn_pool_blocks_kernel(PoolArgs a) {
    int seq = -1, b = 0;
    if (!a.cu_seqlens_q) {                                   // one token per sequence: its block is due when it is the block's last
        const int len = a.context_lens[blockIdx.x];
        if (len > 0 && len % a.pool == 0) {
            seq = blockIdx.x;
            b = len / a.pool - 1;
        }
    } else {
        int at = blockIdx.x;
        for (int i = 0; i < a.batch; ++i) {
            const int len = a.context_lens[i], past = len - (a.cu_seqlens_q[i + 1] - a.cu_seqlens_q[i]);
            const int first = past / a.pool, due = len / a.pool - first;
            if (at < due) {
                seq = i;
                b = first + at;
                break;
            }
            at -= due;
        }
    }
    if (seq < 0) return;                                     // (uniform over the workgroup)
    const int i = blockIdx.y * 256 + threadIdx.x, nk = a.G * a.dim, nv = a.G * a.vdim;
    if (i >= nk + nv) return;
    const int32_t* table = a.block_tables + (int64_t)seq * a.table_stride;
    if (i < nk) block_mean_column((const A*)a.k_cache, (A*)a.pk, i, nk, false, b, a.pool, a.page, a.pool_rows, table);
    else block_mean_column((const A*)a.v_cache, (A*)a.pv, i - nk, nv, true, b, a.pool, a.page, a.pool_rows, table);
}

// Keys and values to their cache slots: a workgroup takes KT tokens of the step and KC columns of both rows.  Keys pass as they lie;
// values turn in LDS, so that tokens which lie side by side in a page leave in one piece (64 of them: a whole cache line, which no
// other workgroup then touches).  With `pool` (one token per sequence: row t of the tables is token t's) the columns' means of the
// blocks that these tokens complete follow in the same launch.
constexpr int KT = 64;
struct KvStoreArgs {
    const void *k, *v;         // [T, ld]: nk and nv columns
    int64_t ld;
    const void* v_mix;         // one number l, or null: the value is (1 - l) v + l v_first
    const void* v_first;       // [T, ld_first]
    int64_t ld_first;
    void *k_cache, *v_cache;
    const int32_t* slot_mapping;
    int T, page, nk, nv, vec_k, vec_v, vec_first;
    int pool, pool_rows;
    const int64_t* positions;
    const int32_t* block_tables;
    int64_t table_stride;
    void *pk, *pv;
};

template <typename A, int KC>
__global__ __launch_bounds__(256) void attn_kv_store_kernel(KvStoreArgs a) {
    __shared__ float tile[KT][KC + 1];
    __shared__ int slots[KT], due_tok[KT], due_block[KT], due_count;             // due: the tokens that complete a block, and the block
    const int tid = threadIdx.x, t0 = blockIdx.x * KT, c0 = blockIdx.y * KC;
    if (tid < KT) {
        const int t = t0 + tid;
        const int slot = t < a.T ? a.slot_mapping[t] : -1;
        slots[tid] = slot;
        if (a.pool) {                                        // (the first KT = 64 lanes are one wave)
            const int len = slot >= 0 ? (int)a.positions[t] + 1 : 0;
            const bool due = slot >= 0 && len % a.pool == 0;
            const unsigned long long mask = __ballot(due);
            if (due) {
                const int at = __popcll(mask & ((1ull << tid) - 1));
                due_tok[at] = t;
                due_block[at] = len / a.pool - 1;
            }
            if (tid == 0) due_count = __popcll(mask);
        }
    }
    __syncthreads();
    const float lam = a.v_mix ? ldf((const A*)a.v_mix, 0) : 0.f;
    constexpr int CP = KC / 8;                               // pieces of eight columns per token
#pragma unroll
    for (int i = tid; i < KT * CP; i += 256) {
        const int r = i / CP, c = c0 + (i % CP) * 8, slot = slots[r];
        const int64_t t = t0 + r;
        if (slot < 0) continue;
        float x[8];
        if (c < a.nk) {
            nvh_load8((const A*)a.k + t * a.ld, c, a.nk - c, a.vec_k, x);
            A* dst = (A*)a.k_cache + (int64_t)slot * a.nk + c;
            A out[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) out[e] = (A)x[e];
            if (a.vec_k) {
                __builtin_memcpy(__builtin_assume_aligned(dst, 16), out, sizeof(out));
            } else {
                for (int e = 0; e < min(8, a.nk - c); ++e) dst[e] = out[e];
            }
        }
        if (c < a.nv) {
            nvh_load8((const A*)a.v + t * a.ld, c, a.nv - c, a.vec_v, x);
            if (a.v_mix) {
                float f[8];
                nvh_load8((const A*)a.v_first + t * a.ld_first, c, a.nv - c, a.vec_first, f);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = (1.0f - lam) * x[e] + lam * f[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) tile[r][c - c0 + e] = x[e];
        }
    }
    __syncthreads();
    {
        const int r = tid % KT, slot = slots[r];             // (256 is a multiple of KT)
        if (slot >= 0) {
            A* dst = (A*)a.v_cache + (int64_t)(slot / a.page) * a.page * a.nv + slot % a.page;
#pragma unroll
            for (int c = tid / KT; c < KC; c += 256 / KT)
                if (c0 + c < a.nv) dst[(int64_t)(c0 + c) * a.page] = (A)tile[r][c];
        }
    }
    if (a.pool == 0) return;
    __syncthreads();                                         // (the workgroup's own stores are among what the means read)
    for (int i = tid; i < due_count * 2 * KC; i += 256) {
        const int at = i / (2 * KC), c = c0 + i % KC;
        const int32_t* table = a.block_tables + (int64_t)due_tok[at] * a.table_stride;
        if (i % (2 * KC) < KC) {
            if (c < a.nk) block_mean_column((const A*)a.k_cache, (A*)a.pk, c, a.nk, false, due_block[at], a.pool, a.page, a.pool_rows, table);
        } else {
            if (c < a.nv) block_mean_column((const A*)a.v_cache, (A*)a.pv, c, a.nv, true, due_block[at], a.pool, a.page, a.pool_rows, table);
        }
    }
}

template <typename A, int KC>
static void launch_kv_store(const KvStoreArgs& a, hipStream_t st) {
    attn_kv_store_kernel<A, KC><<<dim3((unsigned)nvh_cdiv(a.T, KT), (unsigned)nvh_cdiv(a.nk > a.nv ? a.nk : a.nv, KC)), 256, 0, st>>>(a);
}

}  // namespace

extern "C" int32_t nvh_attn_rotary_prep(const void* proj, int64_t proj_row_stride, const void* q_norm_weight, const void* k_norm_weight,
                                        float eps, const int64_t* positions, const float* qk_freq, float qk_mag, int64_t rot_dims,
                                        int32_t qk_interleaved, const float* v_freq, int32_t v_interleaved, void* q_out, float* gate_out,
                                        void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t page, int64_t num_tokens,
                                        int64_t num_q_heads, int64_t num_kv_heads, int64_t dim, int64_t vdim, int32_t norm_per_head, int32_t act_f32,
                                        nvh_stream_t stream) {
    NVH_REQUIRE(proj && positions && q_out && !q_norm_weight == !k_norm_weight, NVH_EINVAL, "nvh_attn_rotary_prep: null pointer");
    NVH_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && dim > 0 && vdim > 0 && num_tokens >= 0 && page > 0, NVH_EINVAL, "nvh_attn_rotary_prep: bad sizes");
    NVH_REQUIRE(rot_dims >= 0 && rot_dims <= dim && rot_dims % 2 == 0 && (rot_dims == 0 || qk_freq), NVH_EINVAL,
                "nvh_attn_rotary_prep: rot_dims %ld does not fit dim %ld", (long)rot_dims, (long)dim);
    NVH_REQUIRE(!v_freq || vdim % 2 == 0, NVH_EINVAL, "nvh_attn_rotary_prep: rotated values need an even vdim");
    NVH_REQUIRE(proj_row_stride >= (num_q_heads + num_kv_heads) * dim + num_kv_heads * vdim + (gate_out ? num_q_heads : 0), NVH_EINVAL,
                "nvh_attn_rotary_prep: projection row too short");
    if (num_tokens == 0) return NVH_OK;
    PrepArgs a{proj, proj_row_stride, q_norm_weight, k_norm_weight, norm_per_head, eps, positions, qk_freq, qk_mag, (int)rot_dims, qk_interleaved,
               v_freq, v_interleaved, q_out, gate_out, k_cache, v_cache, slot_mapping, (int)num_q_heads, (int)num_kv_heads, (int)dim, (int)vdim, (int)page};
    hipStream_t st = (hipStream_t)stream;
    const size_t lds = norm_per_head ? sizeof(float) * (size_t)(num_q_heads + num_kv_heads) : 0;
    NVH_REQUIRE(lds <= 32 * 1024, NVH_ENOSYS, "nvh_attn_rotary_prep: %ld heads above the per-head norm's limit", (long)(num_q_heads + num_kv_heads));
    if (act_f32) launch_rotary_prep<float>(a, num_tokens, lds, st);
    else launch_rotary_prep<bf16>(a, num_tokens, lds, st);
    NVH_CHECK_LAUNCH("nvh_attn_rotary_prep");
    return NVH_OK;
}

extern "C" int32_t nvh_attn_paged_any(const void* q, int64_t q_row_stride, const void* k_cache, const void* v_cache, const int32_t* cu_seqlens_q,
                                      const int32_t* context_lens, const int32_t* block_tables, int64_t table_stride, int64_t batch,
                                      int64_t total_q, int64_t page, int64_t num_q_heads, int64_t num_kv_heads, int64_t dim, int64_t vdim,
                                      float scale, const float* gate, const void* gate_elems, int64_t gate_elems_stride, const float* v_freq, int32_t v_interleaved,
                                      const float* slopes, const float* bias, int64_t bias_len, int64_t window, int64_t keep_first, int64_t chunk, const float* sinks, float softcap, float temp_coef,
                                      int64_t temp_every, int64_t pool, int64_t pool_rows, const void* pooled_k, const void* pooled_v, void* out,
                                      float* parts_ws, int64_t parts_ws_bytes, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(!bias || (bias_len > 0 && bias_len < (1 << 20) && pool == 0), NVH_EINVAL, "nvh_attn_paged_any: a distance bias has a row per head and no pooled blocks beside it");
    NVH_REQUIRE(!gate_elems || gate_elems_stride >= num_q_heads * vdim, NVH_EINVAL, "nvh_attn_paged_any: gate row too short");
    NVH_REQUIRE(softcap >= 0.f && temp_every >= 0 && temp_every < (1 << 30), NVH_EINVAL, "nvh_attn_paged_any: bad softcap or query temperature");
    NVH_REQUIRE(pool >= 0 && pool < (1 << 30) && (pool == 0 || (pooled_k && pooled_v && pool_rows >= nvh_cdiv(page, pool) && window > 0 && keep_first == 0 && chunk == 0 && !slopes)),
                NVH_EINVAL, "nvh_attn_paged_any: pooled blocks go with a plain window and caches of their means");
    NVH_REQUIRE(window >= 0 && keep_first >= 0 && window < (1 << 30) && keep_first < (1 << 30), NVH_EINVAL, "nvh_attn_paged_any: bad window");
    NVH_REQUIRE(chunk >= 0 && chunk < (1 << 30), NVH_EINVAL, "nvh_attn_paged_any: bad chunk");
    NVH_REQUIRE(q && k_cache && v_cache && context_lens && block_tables && out, NVH_EINVAL, "nvh_attn_paged_any: null pointer");
    NVH_REQUIRE(batch >= 0 && total_q >= 0 && page > 0 && num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0 && dim > 0 && vdim > 0,
                NVH_EINVAL, "nvh_attn_paged_any: bad sizes");
    NVH_REQUIRE(vdim <= 16 * AVC_MAX, NVH_ENOSYS, "nvh_attn_paged_any: vdim %ld above %d", (long)vdim, 16 * AVC_MAX);
    NVH_REQUIRE(!v_freq || vdim % 2 == 0, NVH_EINVAL, "nvh_attn_paged_any: rotated values need an even vdim");
    const size_t lds = sizeof(float) * (size_t)(AQ * dim + AK * (dim + 1) + AK * (vdim + 1) + AQ * AK);
    NVH_REQUIRE(lds <= 160 * 1024, NVH_ENOSYS, "nvh_attn_paged_any: dim %ld + vdim %ld need %zu bytes of LDS", (long)dim, (long)vdim, lds);
    if (lds > 64 * 1024) {                                   // beyond the default limit of dynamic LDS: raise it for both forms (gfx950: 160 KB per workgroup)
        const hipError_t e1 = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_paged_any_kernel<float, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        const hipError_t e2 = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_paged_any_kernel<bf16, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        const hipError_t e3 = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_paged_any_kernel<float, 32>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        const hipError_t e4 = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_paged_any_kernel<bf16, 32>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        NVH_REQUIRE(e1 == hipSuccess && e2 == hipSuccess && e3 == hipSuccess && e4 == hipSuccess, NVH_ENOSYS, "nvh_attn_paged_any: %zu bytes of LDS refused", lds);
    }
    if (batch == 0 || total_q == 0) return NVH_OK;
    NVH_REQUIRE(q_row_stride >= num_q_heads * dim, NVH_EINVAL, "nvh_attn_paged_any: query row too short");
    AttnArgs a{q, q_row_stride, k_cache, v_cache, cu_seqlens_q, context_lens, block_tables, table_stride, (int)batch, (int)page, (int)num_q_heads,
               (int)num_kv_heads, (int)dim, (int)vdim, scale, gate, v_freq, v_interleaved, out, gate_elems, gate_elems_stride, slopes, bias, (int)bias_len, (int)window, (int)keep_first, (int)chunk, sinks, softcap, temp_coef, (int)temp_every, (int)pool, (int)pool_rows,
               pooled_k, pooled_v, 0, 0, 0, 0, 1, 1, nullptr, 0};
    // at most ceil(len / AQ) tiles per sequence: total_q / AQ + batch bounds their number (surplus workgroups exit)
    const dim3 grid((unsigned)(total_q / AQ + batch), (unsigned)num_q_heads);
    hipStream_t st = (hipStream_t)stream;
    // bf16 with 16-aligned head sizes: the matrix-core kernel (the choice depends on the sizes and the type only)
    const bool mfma = !act_f32 && dim % 16 == 0 && vdim % 16 == 0 && dim <= 256 && vdim <= 256 && page % MK == 0 && q_row_stride % 8 == 0 && nvh_aligned16(q) && nvh_aligned16(k_cache) &&
                      nvh_aligned16(v_cache) && (pool == 0 || (nvh_aligned16(pooled_k) && nvh_aligned16(pooled_v))) && nvh_aligned16(out) &&
                      (!gate_elems || (gate_elems_stride % 8 == 0 && nvh_aligned16(gate_elems) && !v_freq)) &&
                      (!bias || (sizeof(float) * (size_t)bias_row_floats((int)bias_len) <= BIAS_LDS && softcap == 0.f && temp_every == 0 && !slopes)) && !nvh_switch_on(SW_ATTN_ANY_NO_MFMA);
    if (mfma) {
        // (scratch for the key parts of the one-query form: used when it is given and large enough, see nvh_attn_paged_any_parts_bytes)
        const size_t need = total_q == batch ? one_query_parts_bytes(batch, (int)num_q_heads, (int)num_kv_heads, (int)vdim, v_freq != nullptr) : 0;
        if (parts_ws && need && (size_t)parts_ws_bytes >= need) a.parts = parts_ws;
        if (bias) dispatch_attn_mfma<VAR_BIAS>(a, total_q, st);
        else if (pool > 0 || softcap > 0.f || temp_every > 0) dispatch_attn_mfma<VAR_EXT>(a, total_q, st);
        else dispatch_attn_mfma<VAR_PLAIN>(a, total_q, st);
    } else if (act_f32 && page % 16 == 0 && nvh_aligned16(k_cache) && nvh_aligned16(v_cache) && (pool == 0 || nvh_aligned16(pooled_k)) &&
               !nvh_switch_on(SW_ATTN_ANY_NO_MFMA) && dispatch_attn_f32(a, total_q, st)) {      // (launched)
    } else if (vdim <= 256) {                                // (16 value columns a lane; the choice depends on the size alone)
        if (act_f32) attn_paged_any_kernel<float, 16><<<grid, 256, lds, st>>>(a);
        else attn_paged_any_kernel<bf16, 16><<<grid, 256, lds, st>>>(a);
    } else {
        if (act_f32) attn_paged_any_kernel<float, 32><<<grid, 256, lds, st>>>(a);
        else attn_paged_any_kernel<bf16, 32><<<grid, 256, lds, st>>>(a);
    }
    NVH_CHECK_LAUNCH("nvh_attn_paged_any");
    return NVH_OK;
}

extern "C" int64_t nvh_attn_paged_any_parts_bytes(int64_t batch, int64_t total_q, int64_t num_q_heads, int64_t num_kv_heads, int64_t dim, int64_t vdim,
                                                  int64_t page, int32_t turned_back, int32_t act_f32) {
    if (batch <= 0 || total_q != batch || act_f32 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
    if (dim % 16 || vdim % 16 || dim > 256 || vdim > 256 || page % MK) return 0;           // (the matrix-core kernel's sizes)
    return (int64_t)one_query_parts_bytes(batch, (int)num_q_heads, (int)num_kv_heads, (int)vdim, turned_back != 0);
}

extern "C" int32_t nvh_attn_pool_blocks(const void* k_cache, const void* v_cache, const int32_t* cu_seqlens_q, const int32_t* context_lens,
                                        const int32_t* block_tables, int64_t table_stride, int64_t batch, int64_t total_q, int64_t page, int64_t num_kv_heads,
                                        int64_t dim, int64_t vdim, int64_t pool, int64_t pool_rows, void* pooled_k, void* pooled_v, int32_t act_f32,
                                        nvh_stream_t stream) {
    NVH_REQUIRE(k_cache && v_cache && context_lens && block_tables && pooled_k && pooled_v, NVH_EINVAL, "nvh_attn_pool_blocks: null pointer");
    NVH_REQUIRE(batch >= 0 && total_q >= 0 && page > 0 && num_kv_heads > 0 && dim > 0 && vdim > 0 && pool > 0 && pool < (1 << 30) && pool_rows >= nvh_cdiv(page, pool) &&
                    (cu_seqlens_q || total_q == batch),
                NVH_EINVAL, "nvh_attn_pool_blocks: bad sizes");
    if (batch == 0 || total_q == 0) return NVH_OK;
    const PoolArgs a{k_cache, v_cache, cu_seqlens_q, context_lens, block_tables, table_stride, (int)batch, (int)page, (int)num_kv_heads, (int)dim, (int)vdim, (int)pool,
                     (int)pool_rows, pooled_k, pooled_v};
    // a sequence's n tokens fill at most n / pool + 1 blocks (surplus workgroups exit)
    const dim3 grid((unsigned)(cu_seqlens_q ? total_q / pool + batch : batch), (unsigned)nvh_cdiv(num_kv_heads * (dim + vdim), 256));
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) attn_pool_blocks_kernel<float><<<grid, 256, 0, st>>>(a);
    else attn_pool_blocks_kernel<bf16><<<grid, 256, 0, st>>>(a);
    NVH_CHECK_LAUNCH("nvh_attn_pool_blocks");
    return NVH_OK;
}

extern "C" int32_t nvh_attn_kv_store(const void* k, const void* v, int64_t row_stride, const void* v_mix, const void* v_first, int64_t v_first_stride, void* k_cache,
                                     void* v_cache, const int32_t* slot_mapping, int64_t page, int64_t num_tokens, int64_t num_kv_heads, int64_t dim, int64_t vdim,
                                     int64_t pool, int64_t pool_rows, const int64_t* positions, const int32_t* block_tables, int64_t table_stride, void* pooled_k,
                                     void* pooled_v, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(k && v && k_cache && v_cache && slot_mapping, NVH_EINVAL, "nvh_attn_kv_store: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && num_tokens < (1 << 30) && page > 0 && num_kv_heads > 0 && dim > 0 && vdim > 0 && row_stride >= num_kv_heads * dim &&
                    row_stride >= num_kv_heads * vdim && num_kv_heads * (dim + vdim) < (1 << 30),
                NVH_EINVAL, "nvh_attn_kv_store: bad sizes");
    NVH_REQUIRE(!v_mix || (v_first && v_first_stride >= num_kv_heads * vdim), NVH_EINVAL, "nvh_attn_kv_store: values to mix in are missing or too short");
    NVH_REQUIRE(pool >= 0 && pool < (1 << 30) && (pool == 0 || (positions && block_tables && pooled_k && pooled_v && pool_rows >= nvh_cdiv(page, pool))), NVH_EINVAL,
                "nvh_attn_kv_store: bad pooled blocks");
    if (num_tokens == 0) return NVH_OK;
    const int64_t nk = num_kv_heads * dim, nv = num_kv_heads * vdim;
    const bool rows8 = row_stride % 8 == 0;
    const KvStoreArgs a{k, v, row_stride, v_mix, v_first, v_first_stride, k_cache, v_cache, slot_mapping, (int)num_tokens, (int)page, (int)nk, (int)nv,
                        rows8 && nk % 8 == 0 && nvh_aligned16(k) && nvh_aligned16(k_cache), rows8 && nvh_aligned16(v), v_first_stride % 8 == 0 && nvh_aligned16(v_first),
                        (int)pool, (int)pool_rows, positions, block_tables, table_stride, pooled_k, pooled_v};
    hipStream_t st = (hipStream_t)stream;
    // Narrower column tiles where the tokens alone do not fill the chip.  (64 sequences of one token, 1024 columns, us: 64 tokens x 32
    // columns 7.7, 16 x 32 12.2, 4 x 128 12.8, 4 x 64 17.1, 1 x 256 18.7: a wave that writes one column of many pages beats many that
    // write many columns of few.)
    if (num_tokens >= 512) {
        if (act_f32) launch_kv_store<float, 64>(a, st);
        else launch_kv_store<bf16, 64>(a, st);
    } else {
        if (act_f32) launch_kv_store<float, 32>(a, st);
        else launch_kv_store<bf16, 32>(a, st);
    }
    NVH_CHECK_LAUNCH("nvh_attn_kv_store");
    return NVH_OK;
}
