// Mixture of experts: a token goes to the `top` experts whose router logits are largest, mixed with the weights that a
// softmax over just these `top` logits gives.
//   nvh_moe_route     fp32 router logits [T, E] -> expert ids and weights [T, top] (ties go to the lower expert id);
//                     nvh_moe_route_linear forms the logits itself (x W^T + b in fp32) in the same launch
//   nvh_moe_align     the (token, choice) pairs ordered by expert: for every position in that order the token it comes
//                     from, for every pair its position, and a list of 64-row tiles (expert, first position, rows) that
//                     covers every expert's block - all on the device, so a step never waits for the host and the whole
//                     layer can sit in a captured graph (the tile list has a fixed upper bound: pairs / 64 + experts)
//   nvh_gemm_grouped_any_nt   y[pos] = x[src(pos)] W[expert of pos]^T over that tile list: the any-shape product
//                     (gemm_any.h) with a weight matrix per tile and rows gathered through an index, bf16 on the matrix
//                     cores or true fp32.  A row's result does not depend on where in its expert's block it lies.
//   nvh_moe_combine   out fp32 [T, dim] = sum over a token's choices, in choice order, of weight * y[pos] (+ shared[t])
#include <algorithm>
#include "common.h"
#include "gemm_any.h"

namespace {

// One wave per token: lane l holds logits l, l + 64, ...; `top` rounds of a wave-wide argmax.
constexpr int ROUTE_MAX_PER_LANE = 16;      // experts <= 1024

__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ logits, int64_t stride, int32_t* __restrict__ ids, float* __restrict__ weights,
                                                        int64_t tokens, int experts, int top) {
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tokens) return;
    const int lane = threadIdx.x & 63;
    float z[ROUTE_MAX_PER_LANE];
#pragma unroll
    for (int j = 0; j < ROUTE_MAX_PER_LANE; ++j) {
        const int e = lane + 64 * j;
        z[j] = e < experts ? logits[t * stride + e] : -INFINITY;
    }
    float first = 0.f, denom = 0.f;
    for (int r = 0; r < top; ++r) {
        float bv = -INFINITY;
        int be = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < ROUTE_MAX_PER_LANE; ++j) {
            const int e = lane + 64 * j;
            if (z[j] > bv || (z[j] == bv && e < be && z[j] != -INFINITY)) {
                bv = z[j];
                be = e;
            }
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float ov = __shfl_xor(bv, off, 64);
            const int oe = __shfl_xor(be, off, 64);
            if (ov > bv || (ov == bv && oe < be)) {
                bv = ov;
                be = oe;
            }
        }
        if (r == 0) first = bv;
        const float w = expf(bv - first);                    // the first choice is the largest: exponents <= 0
        denom += w;
        if (lane == 0) {
            ids[t * top + r] = be;
            weights[t * top + r] = w;
        }
#pragma unroll
        for (int j = 0; j < ROUTE_MAX_PER_LANE; ++j)
            if (lane + 64 * j == be) z[j] = -INFINITY;       // taken
    }
    if (lane == 0)
        for (int r = 0; r < top; ++r) weights[t * top + r] = weights[t * top + r] / denom;
}

// (Routing over 16 experts of 1024 columns, us a launch, 64 and 1000 tokens: 12.3 and 12.7 with a piece of 512 at a time, a chain of lane exchanges for
// every comparison of the argmax and the weights read back to be divided; now 4.8 and 6.3.)
// Dot products of a token's row with EG rows of K, row(g) for g < EG, in fp32: a lane takes 8 consecutive elements of every 512, in order.
// Whole pieces of 512 go PIECES at a time, all their loads ahead of the sums: the rows come from L2, and its latency is what a token waits for.
// (The order of a sum does not depend on EG and PIECES.)
template <int EG, int PIECES, typename A, typename Row>
__device__ __forceinline__ void route_dots(const A* __restrict__ xr, Row row, int K, int vec, int lane, float (&acc)[EG]) {
#pragma unroll
    for (int g = 0; g < EG; ++g) acc[g] = 0.f;
    int k0 = lane * 8;
    if (vec) {                                               // (uniform)
        for (int left = K; left >= 512 * PIECES; left -= 512 * PIECES, k0 += 512 * PIECES) {
            float xv[PIECES][8], wv[PIECES][EG][8];
#pragma unroll
            for (int u = 0; u < PIECES; ++u) {
                nvh_load8(xr, k0 + 512 * u, 8, true, xv[u]);
#pragma unroll
                for (int g = 0; g < EG; ++g) nvh_load8(row(g), k0 + 512 * u, 8, true, wv[u][g]);
            }
#pragma unroll
            for (int u = 0; u < PIECES; ++u)
#pragma unroll
                for (int g = 0; g < EG; ++g)
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc[g] = __builtin_fmaf(xv[u][i], wv[u][g][i], acc[g]);
        }
    }
    for (; k0 < K; k0 += 512) {
        float xv[8];
        nvh_load8(xr, k0, K - k0, vec, xv);
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            float wv[8];
            nvh_load8(row(g), k0, K - k0, vec, wv);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[g] = __builtin_fmaf(xv[i], wv[i], acc[g]);
        }
    }
}

// The largest of a wave's values z[j] of lane l, number l + 64 j (ties: the lowest number); 0x7fffffff and -inf where none is above -inf.
template <int PL>
__device__ __forceinline__ int pick_largest(const float (&z)[PL], float& best) {
    float m = z[0];
#pragma unroll
    for (int j = 1; j < PL; ++j) m = fmaxf(m, z[j]);
    m = wave_max(m);
    best = m;
    if (m > -INFINITY) {
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const unsigned long long at = __ballot(z[j] == m);
            if (at) return 64 * j + __builtin_ctzll(at);
        }
    }
    best = -INFINITY;
    return 0x7fffffff;
}

// The same with the router's product inside: z[e] = x . w[e] + bias[e] in fp32.  One workgroup per token: its four waves take the experts four at
// a time in turn, every dot product spread over a wave's lanes and summed across it; the logits meet in LDS and the first wave picks.
// PL: experts a lane of the picking wave holds: experts <= 64 PL.
template <typename A, int PL, int PIECES>
__global__ __launch_bounds__(256) void moe_route_linear_kernel(const A* __restrict__ x, int64_t ldx, const A* __restrict__ w, const A* __restrict__ bias,
                                                               int32_t* __restrict__ ids, float* __restrict__ weights, float* __restrict__ logits_out,
                                                               int experts, int K, int top, int vec, int sigmoid_scores) {
    __shared__ float zs[64 * PL];
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const A* xr = x + t * ldx;
    constexpr int EG = 4;
    for (int e0 = wave * EG; e0 < experts; e0 += 4 * EG) {
        float acc[EG];
        route_dots<EG, PIECES>(xr, [&](int g) { return w + (int64_t)min(e0 + g, experts - 1) * K; }, K, vec, lane, acc);
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            const int e = e0 + g;
            const float s = wave_sum(acc[g]) + (bias && e < experts ? (float)bias[e] : 0.f);
            if (lane == 0 && e < experts) {
                zs[e] = s;
                if (logits_out) logits_out[t * experts + e] = s;
            }
        }
    }
    __syncthreads();
    if (wave != 0) return;
    float z[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) z[j] = lane + 64 * j < experts ? zs[lane + 64 * j] : -INFINITY;
    float first = 0.f, denom = 0.f, mine = 0.f;
    for (int r = 0; r < top; ++r) {
        float bv;
        const int be = pick_largest<PL>(z, bv);
        if (r == 0) first = bv;
        // (sigmoid scores: an expert's weight is its own score, whatever the others'; the order by logit is the order by score)
        const float wgt = sigmoid_scores ? 1.0f / (1.0f + expf(-bv)) : expf(bv - first);
        denom += wgt;
        if (lane == (r & 63)) mine = wgt;                    // (kept until the sum is known; 64 of them at most)
        if (lane == 0) {
            ids[t * top + r] = be;
            if (top > 64) weights[t * top + r] = wgt;
        }
#pragma unroll
        for (int j = 0; j < PL; ++j)
            if (lane + 64 * j == be) z[j] = -INFINITY;
    }
    if (top <= 64) {
        if (lane < top) weights[t * top + lane] = sigmoid_scores ? mine : mine / denom;
    } else if (lane == 0 && !sigmoid_scores) {
        for (int r = 0; r < top; ++r) weights[t * top + r] = weights[t * top + r] / denom;
    }
}

// Routing by scores: s = softmax(x W^T) over ALL experts; the choice goes by s + correction (a per-expert offset that
// does not enter the weights), optionally restricted to groups of neighbouring experts - a group's score is its largest
// choice score and only the `keep` best groups stay eligible (the others count as minus infinity); the `top` best eligible
// experts are taken (ties: lower id) and weighted by their s times `scale`, not renormalised - or (`renorm`) divided by their sum.  `aux` [n_aux, K]: further
// rows that read the same input; their fp32 products go to aux_out [T, n_aux] (a gate of the layer, say).
// One workgroup per token, products as in moe_route_linear_kernel; the first wave picks.
// PL: experts (and groups) a lane of the picking wave holds: experts <= 64 PL.
// us, one wave's rows a piece at a time (eight at once) and now, 16 experts and one more row of 1024, bf16: 64 tokens 6.8 and 4.7, 1008 tokens 7.8 and
// 5.8; 64 + 1 16.6 and 8.2, 18.8 and 11.9; fp32, 16 + 1: 6.2 and 4.8, 8.0 and 7.2.
template <typename A, int PL, int EG, int PIECES>
__global__ __launch_bounds__(256) void moe_route_scored_kernel(const A* __restrict__ x, int64_t ldx, const A* __restrict__ w, const A* __restrict__ correction,
                                                               const A* __restrict__ aux, float* __restrict__ aux_out, int n_aux, int32_t* __restrict__ ids,
                                                               float* __restrict__ weights, float* __restrict__ scores_out, int experts, int K, int top,
                                                               int groups, int keep, float scale, int renorm, int vec) {
    __shared__ float zs[64 * PL];            // logits, then scores
    __shared__ float cs[64 * PL];            // choice scores
    __shared__ float gsc[64 * PL];           // 1 for a kept group
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const A* xr = x + t * ldx;
    // every wave takes EG rows at a time; past the last row: that one again
    const int rows = experts + n_aux;
    for (int e0 = wave * EG; e0 < rows; e0 += 4 * EG) {
        float acc[EG];
        route_dots<EG, PIECES>(xr, [&](int g) {
            const int e = min(e0 + g, rows - 1);
            return e < experts ? w + (int64_t)e * K : aux + (int64_t)(e - experts) * K;
        }, K, vec, lane, acc);
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            const int e = e0 + g;
            const float sum = wave_sum(acc[g]);
            if (lane == 0 && e < experts) zs[e] = sum;
            else if (lane == 0 && e < rows) aux_out[t * n_aux + (e - experts)] = sum;
        }
    }
    __syncthreads();
    const bool picker = wave == 0;                           // the first wave picks; the others only keep the barriers company
    // softmax over all experts
    float z[PL];
    if (picker) {
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            z[j] = lane + 64 * j < experts ? zs[lane + 64 * j] : -INFINITY;
            mx = fmaxf(mx, z[j]);
        }
        mx = wave_max(mx);
        float den = 0.f;
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            z[j] = lane + 64 * j < experts ? expf(z[j] - mx) : 0.f;
            den += z[j];
        }
        den = wave_sum(den);
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const int e = lane + 64 * j;
            if (e < experts) {
                const float sc = z[j] / den;
                zs[e] = sc;
                if (scores_out) scores_out[t * experts + e] = sc;
                z[j] = sc + (correction ? (float)correction[e] : 0.f);
                cs[e] = z[j];
            } else {
                z[j] = -INFINITY;
            }
        }
    }
    __syncthreads();
    if (groups > 1 && keep < groups) {                       // (uniform)
        const int gsz = experts / groups;
        float gv[PL];
        bool gone[PL];
        if (picker) {
#pragma unroll
            for (int j = 0; j < PL; ++j) {
                const int g = lane + 64 * j;
                gone[j] = g >= groups;
                gv[j] = -INFINITY;
                if (g < groups) {
                    for (int i = 0; i < gsz; ++i) gv[j] = fmaxf(gv[j], cs[g * gsz + i]);
                    gsc[g] = 0.f;                            // becomes 1 for a kept group
                }
            }
        }
        __syncthreads();
        if (picker) {
            for (int r = 0; r < keep; ++r) {
                float bv = -INFINITY;
                int bg = 0x7fffffff;
#pragma unroll
                for (int j = 0; j < PL; ++j)
                    if (!gone[j] && (bg == 0x7fffffff || gv[j] > bv)) {
                        bv = gv[j];
                        bg = lane + 64 * j;
                    }
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const float ov = __shfl_xor(bv, off, 64);
                    const int og = __shfl_xor(bg, off, 64);
                    if (og != 0x7fffffff && (bg == 0x7fffffff || ov > bv || (ov == bv && og < bg))) {
                        bv = ov;
                        bg = og;
                    }
                }
                if (lane == 0) gsc[bg] = 1.f;
#pragma unroll
                for (int j = 0; j < PL; ++j)
                    if (lane + 64 * j == bg) gone[j] = true;
            }
        }
        __syncthreads();
        if (picker) {
#pragma unroll
            for (int j = 0; j < PL; ++j) {
                const int e = lane + 64 * j;
                if (e < experts && gsc[e / gsz] == 0.f) z[j] = -INFINITY;
            }
        }
    }
    if (!picker) return;
    bool taken[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) taken[j] = lane + 64 * j >= experts;
    float total = 0.f, mine = 0.f;
    for (int r = 0; r < top; ++r) {
        // the largest that is left, the lowest number among equals (nothing above -inf left, or nothing that compares: the lowest number left)
        float bv, open[PL];
#pragma unroll
        for (int j = 0; j < PL; ++j) open[j] = taken[j] ? -INFINITY : z[j];
        int be = pick_largest<PL>(open, bv);
        if (be == 0x7fffffff) {
#pragma unroll
            for (int j = PL - 1; j >= 0; --j) {
                const unsigned long long at = __ballot(!taken[j]);
                if (at) be = 64 * j + __builtin_ctzll(at);
            }
        }
        const float wgt = zs[be] * scale;
        if (lane == (r & 63)) mine = wgt;                    // (kept until the sum is known; 64 of them at most)
        if (lane == 0) {
            ids[t * top + r] = be;
            if (top > 64) weights[t * top + r] = wgt;
        }
        total += zs[be];
#pragma unroll
        for (int j = 0; j < PL; ++j)
            if (lane + 64 * j == be) taken[j] = true;
    }
    if (top <= 64) {
        if (lane < top) weights[t * top + lane] = renorm ? mine / (total + 1e-20f) : mine;
    } else if (renorm && lane == 0) {
        for (int r = 0; r < top; ++r) weights[t * top + r] = weights[t * top + r] / (total + 1e-20f);
    }
}

// One workgroup: every pair counts itself with its expert, which is its rank there; the sums over the experts before are a scan by one wave; a pair's position is
// the two together.  What bounds it is the chain of launch, load, barriers and stores.  us, before (counts, starts by one lane, a second count for the
// positions; 1024 threads always) and so, tokens x choices of experts: 64 x 2 of 16 2.8 and 2.6, 1000 x 4 of 16 4.9 and 3.9, 1000 x 4 of 64 7.4 and 4.0,
// 301 x 8 of 128 9.6 and 3.8, 1000 x 8 of 256 20.1 and 8.3, 4000 x 8 of 64 23.6 and 20.0, 8000 x 8 of 64 42.3 and 39.4 (four kept pairs a thread instead of
// sixteen, and the ranks of the others left in memory meanwhile: 26.7 and 53.4).
// (Which position a pair gets within its block depends on the order the lanes arrive in; nothing downstream depends on it.)
// KEPT: pairs whose expert and place a thread keeps in registers; those beyond are counted first and take their places from their run's end.
template <int KEPT>
__global__ __launch_bounds__(1024) void moe_align_kernel(const int32_t* __restrict__ ids, int64_t pairs, int experts, int top, int32_t* __restrict__ src_token,
                                                         int32_t* __restrict__ pos_of_pair, int32_t* __restrict__ tile_expert, int32_t* __restrict__ tile_row0,
                                                         int32_t* __restrict__ tile_rows, int max_tiles) {
    extern __shared__ int sh[];                              // [experts] counts, [experts] starts, [experts + 1] first tiles
    int* count = sh;
    int* start = sh + experts;
    int* tile0 = sh + 2 * experts;
    const int tid = threadIdx.x, threads = blockDim.x;
    int kept_e[KEPT], kept_rank[KEPT];
#pragma unroll
    for (int u = 0; u < KEPT; ++u) {
        const int64_t i = tid + (int64_t)u * threads;
        kept_e[u] = i < pairs ? ids[i] : -1;
    }
    for (int e = tid; e < experts; e += threads) count[e] = 0;
    __syncthreads();
    // a pair's rank among its expert's is what the count was when it came
#pragma unroll
    for (int u = 0; u < KEPT; ++u)
        if (kept_e[u] >= 0 && kept_e[u] < experts) kept_rank[u] = atomicAdd(&count[kept_e[u]], 1);
    const bool more = pairs > (int64_t)KEPT * threads;             // (uniform)
    if (more) __syncthreads();                               // every rank is taken before a pair without one is counted: the ranks are a run's first places
    for (int64_t i = tid + (int64_t)KEPT * threads; i < pairs; i += threads) {
        const int e = ids[i];
        if (e >= 0 && e < experts) atomicAdd(&count[e], 1);  // (no rank: it would have to wait in memory; these places are taken from the run's end, below)
    }
    __syncthreads();
    if (tid < 64) {                                          // sums over the experts before, 64 of them at a time
        int rows = 0, tiles = 0;
        for (int e0 = 0; e0 < experts; e0 += 64) {
            const int e = e0 + tid, n = e < experts ? count[e] : 0, nt = (n + nvh_any::GT - 1) / nvh_any::GT;
            int r = n, t = nt;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int ro = __shfl_up(r, d, 64), to = __shfl_up(t, d, 64);
                r += tid >= d ? ro : 0;
                t += tid >= d ? to : 0;
            }
            if (e < experts) {
                start[e] = rows + r - n;
                tile0[e] = tiles + t - nt;
            }
            rows += __shfl(r, 63, 64);
            tiles += __shfl(t, 63, 64);
        }
        if (tid == 0) tile0[experts] = tiles;
    }
    __syncthreads();
    for (int i = tile0[experts] + tid; i < max_tiles; i += threads) tile_rows[i] = 0;
    for (int e = tid; e < experts; e += threads) {
        const int n = count[e];
        for (int k = 0, t = tile0[e]; k < n && t < max_tiles; k += nvh_any::GT, ++t) {
            tile_expert[t] = e;
            tile_row0[t] = start[e] + k;
            tile_rows[t] = min(nvh_any::GT, n - k);
        }
    }
#pragma unroll
    for (int u = 0; u < KEPT; ++u) {
        const int64_t i = tid + (int64_t)u * threads;
        if (i >= pairs) continue;
        const bool ok = kept_e[u] >= 0 && kept_e[u] < experts;
        const int pos = ok ? start[kept_e[u]] + kept_rank[u] : -1;
        if (ok) src_token[pos] = (int32_t)((uint32_t)i / (uint32_t)top);
        pos_of_pair[i] = pos;
    }
    if (more) __syncthreads();                               // the counts have been read; now they go down to what was counted with a rank
    for (int64_t i = tid + (int64_t)KEPT * threads; i < pairs; i += threads) {
        const int e = ids[i];
        const bool ok = e >= 0 && e < experts;
        const int pos = ok ? start[e] + atomicAdd(&count[e], -1) - 1 : -1;
        if (ok) src_token[pos] = (int32_t)((uint32_t)i / (uint32_t)top);
        pos_of_pair[i] = pos;
    }
}

struct GroupedArgs {
    const void* x;             // rows of K
    int64_t ldx;
    const int32_t* gather;     // [pairs]: source row of x for every output row (null: the output row's own index)
    const void* w;             // [experts, N, K]
    void* y;                   // [pairs, N]
    int64_t ldy;
    const int32_t *tile_expert, *tile_row0, *tile_rows;
    int N, K, vec_ok, relu2;
    // gated products (w's rows are [gate | up] of N / 2 each, y the activation's N / 2 columns): what gated_pair() needs beside the sums
    int act;                   // 0 .. 2: activation() of the gate times the other half; 3: glu_clamp()
    const int32_t* pos_of_pair;       // with `weights` (a choice's weight times the expert's input): the row of a token's choice, [tokens, top]
    const float* weights;
    int top;
    float limit, alpha;
};

// What glu_clamp_pairs_kernel does to a pair of sums.
__device__ __forceinline__ float glu_clamp(float gate, float up, float w, float limit, float alpha) {
    const float g = fminf(gate * w, limit), u = fminf(fmaxf(up * w, -limit), limit);
    return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
}

// The weight row at place r of a gated tile that starts at place n0: of every sixteen places 4 q + {0, 1} are gate rows and 4 q + {2, 3} the up rows
// of the same two columns, so the four sums of a lane are two finished pairs.  BLOCKS: sixteens that a wave multiplies; a lane's pairs in them are neighbours.
template <int BLOCKS>
__device__ __forceinline__ int gated_row(int n0, int r, int inter) {
    const int block = (r >> 4) % BLOCKS, q = (r >> 2) & 3;
    return min(n0 / 2 + r / (16 * BLOCKS) * 8 * BLOCKS + q * 2 * BLOCKS + block * 2 + (r & 1), inter - 1) + (r & 2 ? inter : 0);
}

// The weight of the choice of token `tok` whose row is m.
__device__ __forceinline__ float choice_weight(const GroupedArgs& a, int tok, int m) {
    const int64_t first = (int64_t)tok * a.top;
    float w = 1.0f;
    for (int j0 = 0; j0 < a.top; j0 += 4) {
        int pos[4];
        float wj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = min(j0 + u, a.top - 1);
            pos[u] = a.pos_of_pair[first + j];
            wj[u] = a.weights[first + j];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) w = pos[u] == m ? wj[u] : w;
    }
    return w;
}

template <bool OUT_F32>
__global__ __launch_bounds__(256) void gemm_grouped_bf16_kernel(GroupedArgs a) {
    const int rows = a.tile_rows[blockIdx.y];
    if (rows <= 0) return;                                   // (uniform: a tile beyond the list's end)
    const bf16* w = (const bf16*)a.w + (int64_t)a.tile_expert[blockIdx.y] * a.N * a.K;
    const nvh_any::RowMap rm{a.gather, a.tile_row0[blockIdx.y], rows};
    const int n0 = blockIdx.x * nvh_any::GT;
    if (a.vec_ok && a.K % 32 == 0 && rows <= 32) {           // (uniform; the results are the same bit for bit)
        const nvh_any::Epilogue epi{nullptr, nullptr, 0, a.relu2};
        if (rows <= 16) nvh_any::gemm_any_bf16_few_rows<OUT_F32, 1>((const bf16*)a.x, a.ldx, w, a.K, a.y, a.ldy, rm, n0, a.N, a.K, epi);
        else nvh_any::gemm_any_bf16_few_rows<OUT_F32, 2>((const bf16*)a.x, a.ldx, w, a.K, a.y, a.ldy, rm, n0, a.N, a.K, epi);
        return;
    }
    nvh_any::gemm_any_bf16_tile<OUT_F32>((const bf16*)a.x, a.ldx, w, a.K, nullptr, a.y, a.ldy, rm, n0, a.N, a.K, a.vec_ok, nullptr, 0, a.relu2);
}

// Wait until at most `ahead` steps (PW loads of this wave each) are still on their way.
template <int PW, int MOST>
__device__ __forceinline__ void wait_steps_in_flight(int ahead) {
    if constexpr (MOST == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        static_assert(PW * MOST < 64, "vmcnt is six bits");
        if (ahead >= MOST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PW * MOST) : "memory");
        else wait_steps_in_flight<PW, MOST - 1>(ahead);
    }
}

// The same product where experts have many rows (bf16, K a multiple of 64): tiles of 128 rows - two neighbouring tiles of the list - by 128 columns,
// four waves of 64 x 64, two workgroups a CU, operands brought to LDS by 16-byte LDS-DMA a k-step ahead.  What bounds both forms is the operands' way from L2 to LDS, and a 128 x 128 tile needs half of what four 64 x 64 tiles take; sums in the
// same order, bit for bit the same results.
// us at 16 experts, the general 64 x 64 tiles, the tiles for few rows below and this one, rows an expert x N x K: 126 x 1536 x 1024 35.0, 24.2,
// 25.3; 250 x 1536 x 1024 51.5, 38.4, 35.1 (360 TFLOP/s); 250 x 1024 x 768 32.9, 21.5, 19.0; 500 x 1536 x 1024 85, 65, 49; 126 x 1024 x 384
// 17.2, 9.4, 12.3.  Tried and slower at these sizes: eight waves and three stages with one workgroup a CU (a grid is seldom whole rounds;
// with four barriers a k-tile, as the dense products' eight waves were then: their loop of one barrier has not been tried here), stages of 32 k four ahead.
constexpr int TALL = 128;

// Whether tile `t` of the list goes on where tile t - 1, a full one, of the same expert ends.
__device__ __forceinline__ bool tile_goes_on(const GroupedArgs& a, int t) {
    return a.tile_expert[t] == a.tile_expert[t - 1] && a.tile_rows[t - 1] == nvh_any::GT && a.tile_row0[t] == a.tile_row0[t - 1] + nvh_any::GT;
}

// Two pairs of sums, rounded as the product alone leaves them, and what becomes of them.
__device__ __forceinline__ bf16x2 gated_pair(const GroupedArgs& a, f32x4 v, float weight) {
    bf16x2 o;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float g = (float)(bf16)v[e], u = (float)(bf16)v[2 + e];
        o[e] = (bf16)(a.act == 3 ? glu_clamp(g, u, weight, a.limit, a.alpha) : nvh_activation(g, a.act) * u);
    }
    return o;
}

// Four consecutive columns of an output row, finished.
template <bool OUT_F32>
__device__ __forceinline__ void store_grouped(const GroupedArgs& a, int64_t m, int n, f32x4 v) {
    if (a.relu2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = fmaxf(v[e], 0.f);
            v[e] *= v[e];
        }
    }
    if constexpr (OUT_F32) {
        *reinterpret_cast<f32x4*>((float*)a.y + m * a.ldy + n) = v;
    } else {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (bf16)v[e];
        *reinterpret_cast<bf16x4*>((bf16*)a.y + m * a.ldy + n) = o;
    }
}

template <bool OUT_F32, bool GATED = false>
__global__ __launch_bounds__(256, 2) void gemm_grouped_tall_bf16_kernel(GroupedArgs a, int max_tiles, int tiles_n) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    // Workgroup ids go round the XCDs: two neighbouring list tiles with all their columns fall to one, so a row is fetched into one L2.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int t = 2 * ((slot / (2 * tiles_n)) * 8 + xcd) + (slot / tiles_n & 1), n0 = slot % tiles_n * TALL;
    if (t >= max_tiles) return;
    int rows = a.tile_rows[t];
    if (rows <= 0) return;                                   // (uniform: a tile beyond the list's end)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // How many tiles before this one belong to the same run of rows: an odd one was taken by its predecessor.
    int before = 0;
    for (int base = t; base > 0; base -= 64) {
        const int at = base - lane;
        const unsigned long long run = __ballot(at > 0 && tile_goes_on(a, max(at, 1)));
        const int n = run == ~0ull ? 64 : __builtin_ctzll(~run);
        before += n;
        if (n < 64) break;
    }
    if (before & 1) return;
    const int expert = a.tile_expert[t], row0 = a.tile_row0[t];
    if (t + 1 < max_tiles && a.tile_rows[t + 1] > 0 && tile_goes_on(a, t + 1)) rows += a.tile_rows[t + 1];
    const int N = a.N, K = a.K;
    const bf16 *x = (const bf16*)a.x, *w = (const bf16*)a.w + (int64_t)expert * N * K;
    // LDS per stage: 128 rows of w, then 128 of x, 64 k (128 bytes) each; 16-byte piece c of row r lies at place c ^ ((r >> 1) & 7), which spreads a
    // fragment read over all banks.  A DMA instruction brings 8 rows: a wave's are pieces wave, wave + 4, ...
    constexpr int STAGE = 2 * TALL * 128, PW = 2 * TALL / 8 / 4;
    const bf16* src[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int p = wave + 4 * i, r = (p & 15) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
        if (p < 16) {
            src[i] = w + (int64_t)(GATED ? gated_row<4>(n0, r, N / 2) : min(n0 + r, N - 1)) * K + chunk * 8;
        } else {                                             // (rows beyond the tile's repeat its last: not written)
            const int at = row0 + min(r, rows - 1);
            src[i] = x + (int64_t)(a.gather ? a.gather[at] : at) * a.ldx + chunk * 8;
        }
    }
    const int steps = K / 64;
    auto stage = [&](int step) {
        char* base = smem + (step & 1) * STAGE;
#pragma unroll
        for (int i = 0; i < PW; ++i)
            __builtin_amdgcn_global_load_lds((const GLOBAL_AS void*)(src[i] + step * 64), (LDS_AS void*)(base + (wave + 4 * i) * 1024), 16, 0, 0);
    };
    const int wn = (wave & 1) * 64, wm = (wave >> 1) * 64, fr = lane & 15, fq = lane >> 4;
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    __shared__ float row_weight[GATED ? TALL : 1];           // (looked up by a thread a row while the first step is on its way)
    const bool weighs = GATED && a.weights && tid < rows;
    const int tok = weighs ? a.gather[row0 + tid] : 0;
    stage(0);
    if (weighs) row_weight[tid] = choice_weight(a, tok, row0 + tid);
    if constexpr (GATED) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // (before the barriers below)
    for (int step = 0; step < steps; ++step) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this wave's pieces of the step
        __builtin_amdgcn_s_barrier();                        // everybody's; and everybody has left the stage that is filled next
        asm volatile("" ::: "memory");
        if (step + 1 < steps) stage(step + 1);
        const char *ws = smem + (step & 1) * STAGE, *xs = ws + TALL * 128;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 wf[4], xf[4];
            const int kc = ks * 4 + fq;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = wn + 16 * i + fr;
                wf[i] = *reinterpret_cast<const bf16x8*>(ws + r * 128 + ((kc ^ ((r >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = wm + 16 * j + fr;
                xf[j] = *reinterpret_cast<const bf16x8*>(xs + r * 128 + ((kc ^ ((r >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
        }
    }
    // a lane holds, for weight tile i and row tile j: row wm + 16 j + fr, columns wn + 16 i + 4 fq + e (N a multiple of 4)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = wm + 16 * j + fr;
        if (r >= rows) continue;
        if constexpr (GATED) {                               // eight neighbouring columns
            const float weight = a.weights ? row_weight[r] : 1.0f;
            const int c = (n0 + wn) / 2 + 8 * fq, inter = N / 2;
            bf16* out = (bf16*)a.y + (int64_t)(row0 + r) * a.ldy + c;
            bf16x8 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bf16x2 pair = gated_pair(a, acc[i][j], weight);
                o[2 * i] = pair[0];
                o[2 * i + 1] = pair[1];
            }
            if (inter % 8 == 0 && a.ldy % 8 == 0) {
                if (c < inter) *reinterpret_cast<bf16x8*>(out) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (c + e < inter) out[e] = o[e];
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + wn + 16 * i + 4 * fq;
            if (n < N) store_grouped<OUT_F32>(a, row0 + r, n, acc[i][j]);
        }
    }
}

template <bool OUT_F32, bool GATED = false>
static bool launch_grouped_tall(const GroupedArgs& a, int64_t max_tiles, hipStream_t st) {
    const int64_t tiles_n = nvh_cdiv(a.N, TALL), slots = nvh_cdiv(max_tiles, 16) * 16 * tiles_n;
    constexpr int lds = 2 * 2 * TALL * 128;
    if (slots >= (1ll << 31)) return false;
    gemm_grouped_tall_bf16_kernel<OUT_F32, GATED><<<dim3((unsigned)slots), 256, lds, st>>>(a, (int)max_tiles, (int)tiles_n);
    return true;
}

// A list tile of at most 16 MT rows by 64 columns (K a multiple of 64, N of 4): a wave's 16 columns and all rows, operands through a ring of LDS
// stages of 64 k each, filled by 16-byte LDS-DMA all stages but one ahead.  What it waits for is the weights' stream.  us at 16 experts, the general
// tiles (operands through registers, or straight from memory for few rows) and this one, rows an expert x N x K: 1 x 1536 x 1024 10.2 and 7.4,
// 16 x 1536 x 1024 23.8 and 13.6 (3.7 TB/s), 8 x 768 x 1024 11.2 and 7.1, 16 x 1024 x 768 11.7 and 6.7, 64 x 1536 x 1024 26.4 and 18.2.
constexpr int SHORT_N = 64, SHORT_LDS = 64 * 1024;
template <bool OUT_F32, int MT, bool GATE = false, bool GATED = false>
__device__ __forceinline__ void gemm_grouped_short_tile(const GroupedArgs& a, int expert, int row0, int rows, int n0, char* smem, const bf16* gate = nullptr, int64_t ldg = 0) {
    constexpr int STAGE = (SHORT_N + 16 * MT) * 128, STAGES = SHORT_LDS / STAGE, AHEAD = STAGES - 1;
    constexpr int PIECES = SHORT_N / 8 + 2 * MT, PW = (PIECES + 3) / 4;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int N = a.N, K = a.K;
    const bf16 *x = (const bf16*)a.x, *w = (const bf16*)a.w + (int64_t)expert * N * K;
    // (LDS rows and places as in the tall form; pieces 0 .. 7 are w's, then x's; a wave without a last piece of its own brings the first ones once more)
    const bf16* src[PW];
    int off[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int p = (wave + 4 * i) % PIECES, r = (p < 8 ? p : p - 8) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
        if (p < 8) {
            src[i] = w + (int64_t)(GATED ? gated_row<1>(n0, r, N / 2) : min(n0 + r, N - 1)) * K + chunk * 8;
        } else {
            const int at = row0 + min(r, rows - 1);
            src[i] = x + (int64_t)(a.gather ? a.gather[at] : at) * a.ldx + chunk * 8;
        }
        off[i] = p * 1024;
    }
    const int steps = K / 64, fr = lane & 15, fq = lane >> 4;
    auto stage = [&](int step) {
        char* base = smem + step % STAGES * STAGE;
#pragma unroll
        for (int i = 0; i < PW; ++i)
            __builtin_amdgcn_global_load_lds((const GLOBAL_AS void*)(src[i] + step * 64), (LDS_AS void*)(base + off[i]), 16, 0, 0);
    };
    f32x4 acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int n = n0 + wave * 16 + 4 * fq;
    bf16x4 gates[MT];
    if constexpr (GATE) {                                    // (older than the stages: the counted waits below only get stricter)
#pragma unroll
        for (int j = 0; j < MT; ++j) gates[j] = *reinterpret_cast<const bf16x4*>(gate + (int64_t)(row0 + min(16 * j + fr, rows - 1)) * ldg + min(n, N - 4));
    }
    __shared__ float row_weight[GATED ? nvh_any::GT : 1];    // (as in the tall form)
    const bool weighs = GATED && a.weights && tid < rows;
    const int tok = weighs ? a.gather[row0 + tid] : 0;
    for (int step = 0; step < AHEAD && step < steps; ++step) stage(step);
    if (weighs) row_weight[tid] = choice_weight(a, tok, row0 + tid);
    if constexpr (GATED) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (int step = 0; step < steps; ++step) {
        wait_steps_in_flight<PW, AHEAD - 1>(min(AHEAD - 1, steps - 1 - step));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (step + AHEAD < steps) stage(step + AHEAD);       // (into the stage that everybody left before this barrier)
        const char *ws = smem + step % STAGES * STAGE, *xs = ws + SHORT_N * 128;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int kc = ks * 4 + fq, rw = wave * 16 + fr;
            const bf16x8 wf = *reinterpret_cast<const bf16x8*>(ws + rw * 128 + ((kc ^ ((rw >> 1) & 7)) << 4));
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const int r = 16 * j + fr;
                const bf16x8 xf = *reinterpret_cast<const bf16x8*>(xs + r * 128 + ((kc ^ ((r >> 1) & 7)) << 4));
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, acc[j], 0, 0, 0);
            }
        }
    }
    if (n >= N) return;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        if (16 * j + fr >= rows) continue;
        if constexpr (GATE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][e] *= nvh_any::sigmoid((float)gates[j][e]);
        }
        if constexpr (GATED)
            *reinterpret_cast<bf16x2*>((bf16*)a.y + (int64_t)(row0 + 16 * j + fr) * a.ldy + n / 2) = gated_pair(a, acc[j], a.weights ? row_weight[16 * j + fr] : 1.0f);
        else
            store_grouped<OUT_F32>(a, row0 + 16 * j + fr, n, acc[j]);
    }
}

template <bool OUT_F32, bool GATED = false>
__global__ __launch_bounds__(256) void gemm_grouped_short_bf16_kernel(GroupedArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int rows = a.tile_rows[blockIdx.y];
    if (rows <= 0) return;                                   // (uniform: a tile beyond the list's end)
    const int expert = a.tile_expert[blockIdx.y], row0 = a.tile_row0[blockIdx.y], n0 = blockIdx.x * SHORT_N;
    if (rows <= 16) gemm_grouped_short_tile<OUT_F32, 1, false, GATED>(a, expert, row0, rows, n0, smem);
    else if (rows <= 32) gemm_grouped_short_tile<OUT_F32, 2, false, GATED>(a, expert, row0, rows, n0, smem);
    else gemm_grouped_short_tile<OUT_F32, 4, false, GATED>(a, expert, row0, rows, n0, smem);
}

// One weight matrix, 64 rows a tile.  us, the general form and this, fp32 results: 1 x 32768 x 1024 14.6 and 13.0 (5.2 TB/s), 64 x 32768 x 1024 20.2 and 16.8,
// 64 x 152064 x 1024 94 and 76, 256 x 32768 x 1024 62 and 51, 1 x 512 x 1024 8.4 and 5.3, 16 x 1024 x 4096 29.1 and 14.9.
template <bool OUT_F32>
__global__ __launch_bounds__(256) void gemm_short_bf16_kernel(GroupedArgs a, int M) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int row0 = blockIdx.y * nvh_any::GT, rows = min(nvh_any::GT, M - row0), n0 = blockIdx.x * SHORT_N;
    if (rows <= 16) gemm_grouped_short_tile<OUT_F32, 1>(a, 0, row0, rows, n0, smem);
    else if (rows <= 32) gemm_grouped_short_tile<OUT_F32, 2>(a, 0, row0, rows, n0, smem);
    else gemm_grouped_short_tile<OUT_F32, 4>(a, 0, row0, rows, n0, smem);
}

// One weight matrix a head, x and y by columns: head blockIdx.z's operands start x_head and y_head elements after the one before it.  With K of one or two
// hundred a tile is one trip to memory, so what counts is that all of it, the gate too, is asked for at once and that sums leave four columns at a time.
// Bit for bit the general form's results.  us, that form and this, 16 heads, rows x N x K: 64 x 192 x 128 4.7 and 3.4, 64 x 128 x 192 with a gate 7.8
// and 4.5, 1 x 128 x 192 with a gate 4.9 and 3.5, 64 x 128 x 512 6.3 and 4.9, 1000 x 192 x 128 10.9 and 6.3, 1000 x 512 x 128 24.0 and 13.0.
template <bool GATE>
__global__ __launch_bounds__(256) void gemm_heads_short_bf16_kernel(GroupedArgs a, int M, int64_t x_head, int64_t y_head, const bf16* gate, int64_t ldg) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int h = blockIdx.z, row0 = blockIdx.y * nvh_any::GT, rows = min(nvh_any::GT, M - row0), n0 = blockIdx.x * SHORT_N;
    a.x = (const bf16*)a.x + h * x_head;
    a.y = (bf16*)a.y + h * y_head;
    if constexpr (GATE) gate += (int64_t)h * a.N;
    if (rows <= 16) gemm_grouped_short_tile<false, 1, GATE>(a, h, row0, rows, n0, smem, gate, ldg);
    else if (rows <= 32) gemm_grouped_short_tile<false, 2, GATE>(a, h, row0, rows, n0, smem, gate, ldg);
    else gemm_grouped_short_tile<false, 4, GATE>(a, h, row0, rows, n0, smem, gate, ldg);
}

// fp32 (K a multiple of 32) through the waves' LDS rings: a list tile by 64 columns, a workgroup a CU, for callers whose experts have many rows, or by 32
// columns, two workgroups a CU, 49 rows and more in two halves.  Bit for bit the results of the form below.
// us, the form below, by 32 and by 64 columns, rows an expert x N x K over 16 experts: 8 x 576 x 1024 19.2, 14.5, 13.8; 38 x 576 x 1024 31.8, 27.8, 21.0;
// 38 x 1536 x 1024 58.6, 48.1, 40.8; 125 x 1536 x 1024 126, 102, 91; 19 x 576 x 1024 (64 experts) 53.7, 43.0, 45.9; 2.5 x 1536 x 1024 25.9, 22.0, 25.6.
// By 32 columns, a grid of at most 256 workgroups has two of them share a tile's rows: one of 128 rows x 1024 x 384 7.4 (the form below), 9.2, so 6.9.
template <int NC>
__global__ __launch_bounds__(256, NC == 2 ? 2 : 1) void gemm_grouped_f32_ring_kernel(GroupedArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int rows = a.tile_rows[blockIdx.y];
    if (rows <= 0) return;                                   // (uniform: a tile beyond the list's end)
    const float *x = (const float*)a.x, *w = (const float*)a.w + (int64_t)a.tile_expert[blockIdx.y] * a.N * a.K;
    const nvh_any::RowMap rm{a.gather, a.tile_row0[blockIdx.y], rows};
    const int n0 = blockIdx.x * 16 * NC;
#define NVH_RING(MR, STAGES, R0) nvh_any::gemm_any_f32_ring<MR, NC, STAGES>(x, a.ldx, w, a.K, nullptr, (float*)a.y, a.ldy, rm, R0, n0, a.N, a.K, nullptr, 0, a.relu2, smem)
    if (NC == 2 && gridDim.z == 2) {                         // (uniform) a half of the tile each
        const int r0 = blockIdx.z * 32;
        if (rows <= r0) return;
        if (rows - r0 <= 16) {
            NVH_RING(1, 3, r0);
        } else {
            NVH_RING(2, 2, r0);
        }
    } else if (rows <= 16) {
        NVH_RING(1, 3, 0);
    } else if (NC == 4 && rows <= 32) {
        NVH_RING(2, 3, 0);
    } else if (rows > 32 && rows <= 48) {
        NVH_RING(3, 2, 0);
    } else if constexpr (NC == 4) {
        NVH_RING(4, 2, 0);
    } else {
        for (int r0 = 0; r0 < rows; r0 += 32) {
            if (r0) __syncthreads();                         // (the first half's sums have been read)
            NVH_RING(2, 2, r0);
        }
    }
#undef NVH_RING
}
template <int NC>
bool launch_grouped_f32(const GroupedArgs& a, int64_t max_tiles, hipStream_t st) {
    constexpr int lds = std::max({nvh_any::f32_ring_bytes<1, NC, 3>(), nvh_any::f32_ring_bytes<2, NC, NC == 4 ? 3 : 2>(), nvh_any::f32_ring_bytes<3, NC, 2>(), NC == 4 ? nvh_any::f32_ring_bytes<4, NC, 2>() : 0});
    static_assert(lds <= (NC == 4 ? 160 : 80) * 1024);
    static std::atomic<uint64_t> granted{0};
    if (!nvh_grant_lds(granted, reinterpret_cast<const void*>(&gemm_grouped_f32_ring_kernel<NC>), lds)) return false;
    const int64_t grid = nvh_cdiv(a.N, 16 * NC) * max_tiles;
    gemm_grouped_f32_ring_kernel<NC><<<dim3((unsigned)nvh_cdiv(a.N, 16 * NC), (unsigned)max_tiles, NC == 2 && grid <= 256 ? 2 : 1), 256, lds, st>>>(a);
    return true;
}

// (a tile of the list is 64 rows: blockIdx.z is its upper or lower half)
__global__ __launch_bounds__(256) void gemm_grouped_f32_kernel(GroupedArgs a) {
    const int rows = a.tile_rows[blockIdx.y], r0 = blockIdx.z * 32;
    if (rows <= r0) return;                                  // (uniform)
    const float* w = (const float*)a.w + (int64_t)a.tile_expert[blockIdx.y] * a.N * a.K;
    const nvh_any::RowMap rm{a.gather, a.tile_row0[blockIdx.y], rows};
    if (rows - r0 <= 16)
        nvh_any::gemm_any_f32_tile<1, 2>((const float*)a.x, a.ldx, w, a.K, nullptr, (float*)a.y, a.ldy, rm, r0, blockIdx.x * 32, a.N, a.K, a.vec_ok, nullptr, 0, a.relu2);
    else
        nvh_any::gemm_any_f32_tile<2, 2>((const float*)a.x, a.ldx, w, a.K, nullptr, (float*)a.y, a.ldy, rm, r0, blockIdx.x * 32, a.N, a.K, a.vec_ok, nullptr, 0, a.relu2);
}

template <typename A>
__global__ __launch_bounds__(256) void moe_combine_kernel(const A* __restrict__ y, int64_t ldy, const int32_t* __restrict__ pos_of_pair, const float* __restrict__ weights,
                                                          const A* __restrict__ shared, int64_t shared_stride, const float* __restrict__ shared_gate,
                                                          int64_t gate_stride, float* __restrict__ out, int dim, int top) {
    const int64_t t = blockIdx.x;
    const float sg = shared_gate ? 1.0f / (1.0f + expf(-shared_gate[t * gate_stride])) : 1.0f;
    for (int c = threadIdx.x; c < dim; c += 256) {
        float s = 0.f;
        for (int r = 0; r < top; ++r) {
            const int pos = pos_of_pair[t * top + r];
            if (pos >= 0) s = __builtin_fmaf(weights ? weights[t * top + r] : 1.0f, (float)y[(int64_t)pos * ldy + c], s);
        }
        if (shared) s += sg * (float)shared[t * shared_stride + c];
        out[t * dim + c] = s;
    }
}

// The experts' activation where a pair's routing weight multiplies the expert's INPUT: the rows of the first grouped product were
// formed from the unweighted token, and since that product is linear, row * weight is the product of the weighted token.  Then, with
// the gate's value capped above and the other half's value clamped to +-limit,
//   g = min(w G, limit);  u = clamp(w U, -limit, limit);  y = g sigmoid(alpha g) (u + 1).
// A pair's row is pos_of_pair[pair] (< 0: the pair has no row).  E: elements a lane, 8 where rows and strides allow 16-byte accesses.
template <typename A, int E>
__global__ __launch_bounds__(256) void glu_clamp_pairs_kernel(const A* __restrict__ gu, int64_t gu_stride, const int32_t* __restrict__ pos_of_pair,
                                                              const float* __restrict__ weights, A* __restrict__ y, int64_t y_stride, int64_t pairs, int inter, float limit,
                                                              float alpha) {
    int64_t pair;
    int c;
    if (!nvh_piece<E>(pairs, inter, pair, c)) return;
    const int pos = pos_of_pair[pair];
    if (pos < 0) return;
    const float w = weights ? weights[pair] : 1.0f;
    const A* row = gu + (int64_t)pos * gu_stride + c;
    float v[E], up[E];
    nvh_load_piece<A, E>(row, v);
    nvh_load_piece<A, E>(row + inter, up);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = glu_clamp(v[e], up[e], w, limit, alpha);
    nvh_store_piece<A, E>(y + (int64_t)pos * y_stride + c, v);
}
// The same with a workgroup a pair.
template <typename A>
__global__ __launch_bounds__(256) void glu_clamp_rows_kernel(const A* __restrict__ gu, int64_t gu_stride, const int32_t* __restrict__ pos_of_pair,
                                                             const float* __restrict__ weights, A* __restrict__ y, int64_t y_stride, int inter, float limit, float alpha) {
    const int64_t pair = blockIdx.x;
    const int pos = pos_of_pair[pair];
    if (pos < 0) return;
    const float w = weights ? weights[pair] : 1.0f;
    const A* row = gu + (int64_t)pos * gu_stride;
    for (int c = threadIdx.x; c < inter; c += 256) y[(int64_t)pos * y_stride + c] = (A)glu_clamp((float)row[c], (float)row[inter + c], w, limit, alpha);
}

}  // namespace

extern "C" int32_t nvh_moe_route(const float* logits, int64_t row_stride, int32_t* ids, float* weights, int64_t num_tokens, int64_t experts,
                                 int64_t top, nvh_stream_t stream) {
    NVH_REQUIRE(logits && ids && weights, NVH_EINVAL, "nvh_moe_route: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && experts > 0 && top > 0 && top <= experts && row_stride >= experts, NVH_EINVAL, "nvh_moe_route: bad sizes");
    NVH_REQUIRE(experts <= 64 * ROUTE_MAX_PER_LANE, NVH_ENOSYS, "nvh_moe_route: %ld experts above %d", (long)experts, 64 * ROUTE_MAX_PER_LANE);
    if (num_tokens == 0) return NVH_OK;
    moe_route_kernel<<<dim3((unsigned)nvh_cdiv(num_tokens, 4)), 256, 0, (hipStream_t)stream>>>(logits, row_stride, ids, weights, num_tokens, (int)experts, (int)top);
    NVH_CHECK_LAUNCH("nvh_moe_route");
    return NVH_OK;
}

extern "C" int32_t nvh_moe_route_linear(const void* x, int64_t x_row_stride, const void* w, const void* bias, int32_t* ids, float* weights,
                                        float* logits_out, int64_t num_tokens, int64_t experts, int64_t K, int64_t top, int32_t sigmoid_scores,
                                        int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(x && w && ids && weights, NVH_EINVAL, "nvh_moe_route_linear: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && experts > 0 && top > 0 && top <= experts && K > 0 && K < (1 << 30) && x_row_stride >= K, NVH_EINVAL, "nvh_moe_route_linear: bad sizes");
    NVH_REQUIRE(experts <= 64 * ROUTE_MAX_PER_LANE, NVH_ENOSYS, "nvh_moe_route_linear: %ld experts above %d", (long)experts, 64 * ROUTE_MAX_PER_LANE);
    if (num_tokens == 0) return NVH_OK;
    const dim3 grid((unsigned)num_tokens);
    hipStream_t st = (hipStream_t)stream;
    const int vec = K % 8 == 0 && x_row_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(w);
#define NVH_ROUTE_LINEAR(A, PL, PIECES) moe_route_linear_kernel<A, PL, PIECES><<<grid, 256, 0, st>>>((const A*)x, x_row_stride, (const A*)w, (const A*)bias, ids, weights, logits_out, (int)experts, (int)K, (int)top, vec, sigmoid_scores)
    // Many experts: the rows come at L2's rate, and one piece at a time leaves room for more waves a CU, in fp32 always, in bf16 where a row has not two whole
    // ones (256 rows of 1000, 1100 tokens 72.9 and 44.5 us, 4000 169 and 132).
    const bool two = K >= 1024;
    if (experts <= 64) {
        if (act_f32) NVH_ROUTE_LINEAR(float, 1, 2);
        else NVH_ROUTE_LINEAR(bf16, 1, 2);
    } else if (experts <= 256) {
        if (act_f32) NVH_ROUTE_LINEAR(float, 4, 1);
        else if (two) NVH_ROUTE_LINEAR(bf16, 4, 2);
        else NVH_ROUTE_LINEAR(bf16, 4, 1);
    } else {
        if (act_f32) NVH_ROUTE_LINEAR(float, ROUTE_MAX_PER_LANE, 1);
        else if (two) NVH_ROUTE_LINEAR(bf16, ROUTE_MAX_PER_LANE, 2);
        else NVH_ROUTE_LINEAR(bf16, ROUTE_MAX_PER_LANE, 1);
    }
#undef NVH_ROUTE_LINEAR
    NVH_CHECK_LAUNCH("nvh_moe_route_linear");
    return NVH_OK;
}

extern "C" int32_t nvh_moe_route_scored(const void* x, int64_t x_row_stride, const void* w, const void* correction, const void* aux, float* aux_out,
                                        int64_t num_aux, int32_t* ids, float* weights, float* scores_out, int64_t num_tokens, int64_t experts, int64_t K,
                                        int64_t top, int64_t groups, int64_t keep, float scale, int32_t renorm, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(x && w && ids && weights && (num_aux == 0 || (aux && aux_out)), NVH_EINVAL, "nvh_moe_route_scored: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && experts > 0 && top > 0 && top <= experts && K > 0 && K < (1 << 30) && x_row_stride >= K && num_aux >= 0 && num_aux <= 64, NVH_EINVAL,
                "nvh_moe_route_scored: bad sizes");
    NVH_REQUIRE(groups >= 1 && experts % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (experts / groups), NVH_EINVAL,
                "nvh_moe_route_scored: %ld groups (keep %ld) do not fit %ld experts, top %ld", (long)groups, (long)keep, (long)experts, (long)top);
    NVH_REQUIRE(experts <= 64 * ROUTE_MAX_PER_LANE, NVH_ENOSYS, "nvh_moe_route_scored: %ld experts above %d", (long)experts, 64 * ROUTE_MAX_PER_LANE);
    if (num_tokens == 0) return NVH_OK;
    const dim3 grid((unsigned)num_tokens);
    hipStream_t st = (hipStream_t)stream;
    const int vec = K % 8 == 0 && x_row_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(w) && (!aux || nvh_aligned16(aux));
#define NVH_ROUTE_SCORED(A, PL, EG, PIECES) moe_route_scored_kernel<A, PL, EG, PIECES><<<grid, 256, 0, st>>>((const A*)x, x_row_stride, (const A*)w, (const A*)correction, (const A*)aux, aux_out, (int)num_aux, ids, weights, scores_out, (int)experts, (int)K, (int)top, (int)groups, (int)keep, scale, renorm, vec)
    const int64_t rows = experts + num_aux;
    // Rows a wave: four, or three where that is as many passes (17 .. 24 rows), or in fp32; the fp32 rows of many experts come at L2's rate, and more
    // waves a CU are worth more than two pieces at once (128 experts, 1008 tokens: 28.7 us as it was, 31.4 with two rows of two pieces, 26.7 so).
    // Two pieces at once where a row has two and the tokens are few: they cost registers, which more than four workgroups a CU need more, and without two
    // whole pieces they are never used.  us, bf16, as it was before either, two at once and one: 17 rows of 1024, 64 tokens 7.4, 4.9, 5.0, 4000 19.0, 14.3, 12.0;
    // of 1000, 4000 tokens 19.2, 20.8, 14.9; 6 rows of 96, 4000 tokens 12.1, 13.6, 9.6.
    // More experts than a wave picks from at once: two pieces at any number of tokens (128 experts of 2048, 2000 tokens 55.7 and 58.1).
    const bool two = K >= 1024 && (num_tokens <= 1024 || experts > 64);
#define NVH_ROUTE_PIECES(A, PL, EG)                \
    if (two) NVH_ROUTE_SCORED(A, PL, EG, 2);      \
    else NVH_ROUTE_SCORED(A, PL, EG, 1)
    if (experts <= 64) {
        if (act_f32) { NVH_ROUTE_PIECES(float, 1, 3); }
        else if (rows > 16 && rows <= 24) { NVH_ROUTE_PIECES(bf16, 1, 3); }
        else { NVH_ROUTE_PIECES(bf16, 1, 4); }
    } else if (experts <= 256) {
        if (act_f32) NVH_ROUTE_SCORED(float, 4, 4, 1);
        else { NVH_ROUTE_PIECES(bf16, 4, 4); }
    } else {
        if (act_f32) NVH_ROUTE_SCORED(float, ROUTE_MAX_PER_LANE, 4, 1);
        else { NVH_ROUTE_PIECES(bf16, ROUTE_MAX_PER_LANE, 4); }
    }
#undef NVH_ROUTE_PIECES
#undef NVH_ROUTE_SCORED
    NVH_CHECK_LAUNCH("nvh_moe_route_scored");
    return NVH_OK;
}

extern "C" int64_t nvh_moe_max_tiles(int64_t pairs, int64_t experts) { return pairs / nvh_any::GT + experts; }

extern "C" int32_t nvh_moe_align(const int32_t* ids, int64_t num_tokens, int64_t experts, int64_t top, int32_t* src_token, int32_t* pos_of_pair,
                                 int32_t* tile_expert, int32_t* tile_row0, int32_t* tile_rows, int64_t max_tiles, nvh_stream_t stream) {
    NVH_REQUIRE(ids && src_token && pos_of_pair && tile_expert && tile_row0 && tile_rows, NVH_EINVAL, "nvh_moe_align: null pointer");
    NVH_REQUIRE(num_tokens >= 0 && experts > 0 && experts <= 4096 && top > 0 && max_tiles >= nvh_moe_max_tiles(num_tokens * top, experts) && num_tokens * top < (1 << 30),
                NVH_EINVAL, "nvh_moe_align: bad sizes");
    if (num_tokens == 0) return NVH_OK;
    const size_t lds = sizeof(int) * (size_t)(3 * experts + 1);
    const int64_t pairs = num_tokens * top;
    auto launch = [&](auto kernel, int threads) { kernel<<<dim3(1), threads, lds, (hipStream_t)stream>>>(ids, pairs, (int)experts, (int)top, src_token, pos_of_pair, tile_expert, tile_row0, tile_rows, (int)max_tiles); };
    if (pairs <= 1024) launch(&moe_align_kernel<4>, 256);
    else if (pairs <= 4096) launch(&moe_align_kernel<4>, 1024);
    else launch(&moe_align_kernel<16>, 1024);
    NVH_CHECK_LAUNCH("nvh_moe_align");
    return NVH_OK;
}

static int32_t grouped_product(const void* x, int64_t x_row_stride, const int32_t* gather, const void* w, void* y, int64_t y_row_stride,
                               const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* tile_rows, int64_t max_tiles,
                               int64_t N, int64_t K, int32_t relu2, int32_t in_f32, int32_t out_f32, int32_t tall, nvh_stream_t stream) {
    NVH_REQUIRE(x && w && y && tile_expert && tile_row0 && tile_rows, NVH_EINVAL, "nvh_gemm_grouped_any_nt: null pointer");
    NVH_REQUIRE(max_tiles >= 0 && max_tiles < 65536 && N > 0 && K > 0 && N < (1 << 30) && K < (1 << 30) && x_row_stride >= K && y_row_stride >= N, NVH_EINVAL,
                "nvh_gemm_grouped_any_nt: bad sizes");
    NVH_REQUIRE(!in_f32 || out_f32, NVH_ENOSYS, "nvh_gemm_grouped_any_nt: fp32 operands give an fp32 product");
    if (max_tiles == 0) return NVH_OK;
    const int vec_ok = in_f32 ? nvh_any::f32_vec_ok(x, x_row_stride, w, K) : K % 8 == 0 && x_row_stride % 8 == 0 && nvh_aligned16(x) && nvh_aligned16(w);
    const GroupedArgs a{x, x_row_stride, gather, w, y, y_row_stride, tile_expert, tile_row0, tile_rows, (int)N, (int)K, vec_ok, relu2};
    const dim3 grid((unsigned)nvh_cdiv(N, nvh_any::GT), (unsigned)max_tiles);
    hipStream_t st = (hipStream_t)stream;
    if (!in_f32 && vec_ok && K % 64 == 0 && N % 4 == 0 && y_row_stride % 4 == 0 && nvh_aligned16(y)) {
        if (!(tall && (out_f32 ? launch_grouped_tall<true>(a, max_tiles, st) : launch_grouped_tall<false>(a, max_tiles, st)))) {
            if (out_f32) gemm_grouped_short_bf16_kernel<true><<<grid, 256, SHORT_LDS, st>>>(a);
            else gemm_grouped_short_bf16_kernel<false><<<grid, 256, SHORT_LDS, st>>>(a);
        }
        NVH_CHECK_LAUNCH("nvh_gemm_grouped_any_nt");
        return NVH_OK;
    }
    if (in_f32 && vec_ok && K % nvh_any::F32_CHUNK == 0) {
        const bool ok = tall ? launch_grouped_f32<4>(a, max_tiles, st) : launch_grouped_f32<2>(a, max_tiles, st);
        NVH_REQUIRE(ok, NVH_ENOSYS, "nvh_gemm_grouped_any_nt: more than 64 KB of LDS for a workgroup refused");
    } else if (in_f32) gemm_grouped_f32_kernel<<<dim3((unsigned)nvh_cdiv(N, 32), (unsigned)max_tiles, 2), 256, 0, st>>>(a);
    else if (out_f32) gemm_grouped_bf16_kernel<true><<<grid, 256, 0, st>>>(a);
    else gemm_grouped_bf16_kernel<false><<<grid, 256, 0, st>>>(a);
    NVH_CHECK_LAUNCH("nvh_gemm_grouped_any_nt");
    return NVH_OK;
}

// The experts' gated first half in one launch: the activation has its gate and up sums side by side in a lane, so rows of 2 inter are neither written nor read.
// Sums, their rounding and the activation's formulas are those of two launches.  us, two launches and one, 16 experts, K 1024, tokens x choices, inter:
// 1 x 2, 768 7.5 and 6.4; 64 x 2, 384 8.3 and 6.3; 64 x 2, 768 12.3 and 10.1; 1000 x 2, 768 23.6 and 21.6; 1000 x 4, 768 39.0 and 36.4; 1000 x 4, 2048
// 75 and 70.  What the exponentials cost is now in the product, where they are computed while the other workgroup of a CU multiplies.
extern "C" int32_t nvh_gemm_grouped_gated_nt(const void* x, int64_t x_row_stride, const int32_t* gather, const void* w, void* y, int64_t y_row_stride,
                                             const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* tile_rows, int64_t max_tiles, int64_t inter,
                                             int64_t K, int32_t act, const int32_t* pos_of_pair, const float* weights, int64_t top, float limit, float alpha,
                                             int32_t many, nvh_stream_t stream) {
    NVH_REQUIRE(x && w && y && tile_expert && tile_row0 && tile_rows, NVH_EINVAL, "nvh_gemm_grouped_gated_nt: null pointer");
    NVH_REQUIRE(max_tiles >= 0 && max_tiles < 65536 && inter > 0 && K > 0 && inter < (1 << 29) && K < (1 << 30) && x_row_stride >= K && y_row_stride >= inter && act >= 0 && act <= 3,
                NVH_EINVAL, "nvh_gemm_grouped_gated_nt: bad sizes");
    NVH_REQUIRE(act != 3 || limit > 0.f, NVH_EINVAL, "nvh_gemm_grouped_gated_nt: act 3 needs a limit above 0");
    NVH_REQUIRE(!weights || (act == 3 && gather && pos_of_pair && top > 0 && top < (1 << 20)), NVH_EINVAL, "nvh_gemm_grouped_gated_nt: weights go with act 3 and the rows of the choices");
    NVH_REQUIRE(K % 64 == 0 && inter % 2 == 0 && x_row_stride % 8 == 0 && y_row_stride % 2 == 0 && nvh_aligned16(x) && nvh_aligned16(w) && nvh_aligned16(y), NVH_ENOSYS,
                "nvh_gemm_grouped_gated_nt: whole k-tiles, pairs of columns and aligned rows only");
    if (max_tiles == 0) return NVH_OK;
    const GroupedArgs a{x, x_row_stride, gather, w, y, y_row_stride, tile_expert, tile_row0, tile_rows, (int)(2 * inter), (int)K, 1, 0,
                        act, pos_of_pair, weights, (int)top, limit, alpha};
    hipStream_t st = (hipStream_t)stream;
    if (!(many && launch_grouped_tall<false, true>(a, max_tiles, st)))
        gemm_grouped_short_bf16_kernel<false, true><<<dim3((unsigned)nvh_cdiv(a.N, SHORT_N), (unsigned)max_tiles), 256, SHORT_LDS, st>>>(a);
    NVH_CHECK_LAUNCH("nvh_gemm_grouped_gated_nt");
    return NVH_OK;
}

bool nvh_any::launch_short_product(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, bool out_f32, hipStream_t st) {
    if (K % 64 != 0 || N % 4 != 0 || ldx % 8 != 0 || ldy % 4 != 0 || !nvh_aligned16(x) || !nvh_aligned16(w) || !nvh_aligned16(y)) return false;
    const GroupedArgs a{x, ldx, nullptr, w, y, ldy, nullptr, nullptr, nullptr, (int)N, (int)K, 1, 0};
    const dim3 grid((unsigned)nvh_cdiv(N, SHORT_N), (unsigned)nvh_cdiv(M, nvh_any::GT));
    if (out_f32) gemm_short_bf16_kernel<true><<<grid, 256, SHORT_LDS, st>>>(a, (int)M);
    else gemm_short_bf16_kernel<false><<<grid, 256, SHORT_LDS, st>>>(a, (int)M);
    return true;
}

bool nvh_any::launch_short_heads(const void* x, int64_t ldx, int64_t x_head, const void* w, void* y, int64_t ldy, int64_t y_head, int64_t M, int64_t heads, int64_t N, int64_t K,
                                 const void* gate, int64_t ldg, hipStream_t st) {
    // (16-byte pieces of x and w, four columns of y and the gate at a time)
    if (K % 64 != 0 || N % 4 != 0 || ldx % 8 != 0 || x_head % 8 != 0 || ldy % 4 != 0 || y_head % 4 != 0 || !nvh_aligned16(x) || !nvh_aligned16(w) || !nvh_aligned16(y)) return false;
    if (gate && (ldg % 4 != 0 || !nvh_aligned16(gate))) return false;
    const GroupedArgs a{x, ldx, nullptr, w, y, ldy, nullptr, nullptr, nullptr, (int)N, (int)K, 1, 0};
    const dim3 grid((unsigned)nvh_cdiv(N, SHORT_N), (unsigned)nvh_cdiv(M, nvh_any::GT), (unsigned)heads);
    if (gate) gemm_heads_short_bf16_kernel<true><<<grid, 256, SHORT_LDS, st>>>(a, (int)M, x_head, y_head, (const bf16*)gate, ldg);
    else gemm_heads_short_bf16_kernel<false><<<grid, 256, SHORT_LDS, st>>>(a, (int)M, x_head, y_head, nullptr, 0);
    return true;
}

extern "C" int32_t nvh_gemm_grouped_any_nt(const void* x, int64_t x_row_stride, const int32_t* gather, const void* w, void* y, int64_t y_row_stride,
                                           const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* tile_rows, int64_t max_tiles,
                                           int64_t N, int64_t K, int32_t relu2, int32_t in_f32, int32_t out_f32, nvh_stream_t stream) {
    return grouped_product(x, x_row_stride, gather, w, y, y_row_stride, tile_expert, tile_row0, tile_rows, max_tiles, N, K, relu2, in_f32, out_f32, 0, stream);
}

extern "C" int32_t nvh_gemm_grouped_many_nt(const void* x, int64_t x_row_stride, const int32_t* gather, const void* w, void* y, int64_t y_row_stride,
                                            const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* tile_rows, int64_t max_tiles,
                                            int64_t N, int64_t K, int32_t relu2, int32_t in_f32, int32_t out_f32, nvh_stream_t stream) {
    return grouped_product(x, x_row_stride, gather, w, y, y_row_stride, tile_expert, tile_row0, tile_rows, max_tiles, N, K, relu2, in_f32, out_f32, 1, stream);
}

extern "C" int32_t nvh_glu_clamp_pairs(const void* gate_up, int64_t row_stride, const int32_t* pos_of_pair, const float* weights, void* y, int64_t y_stride,
                                       int64_t pairs, int64_t inter, float limit, float alpha, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(gate_up && pos_of_pair && y && pairs >= 0 && inter > 0 && row_stride >= 2 * inter && y_stride >= inter && limit > 0.f, NVH_EINVAL,
                "nvh_glu_clamp_pairs: bad argument");
    if (pairs == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    // One element a lane spreads few elements over the chip, eight a lane make wide accesses of many; between them, and where rows do not allow wide
    // accesses, a workgroup a pair.  us, one, eight a lane and a workgroup a pair: 300 x 768 bf16 2.4, 2.7, 2.6; 64 x 3072 2.3, 2.6, 3.7; 900 x 768 3.3,
    // 3.3, 3.1; 1400 x 768 fp32 4.3, 3.9, 3.6; 4000 x 768 8.2, 5.9, 6.4; 1000 x 3072 8.1, 5.9, 6.6; 3000 x 1001 8.7, none, 6.5.
    const int64_t total = pairs * inter;
    const bool wide = inter % 8 == 0 && row_stride % 8 == 0 && y_stride % 8 == 0 && nvh_aligned16(gate_up) && nvh_aligned16(y);
    const bool few = total < (1 << 19), vec = !few && wide && (inter > 1024 || total >= (act_f32 ? 1 << 21 : 1 << 20));
    const int64_t most = std::max<int64_t>((1ll << 31) / inter, 1);      // pairs a launch: a grid has fewer than 2^32 threads
    auto launch = [&](auto kernel, auto rows_kernel, auto type) {
        typedef decltype(type) A;
        if (!few && !vec) {
            rows_kernel<<<dim3((unsigned)pairs), 256, 0, st>>>((const A*)gate_up, row_stride, pos_of_pair, weights, (A*)y, y_stride, (int)inter, limit, alpha);
            return;
        }
        for (int64_t p0 = 0; p0 < pairs; p0 += most) {
            const int64_t n = std::min(most, pairs - p0);
            kernel<<<dim3((unsigned)nvh_cdiv(n * inter, vec ? 2048 : 256)), 256, 0, st>>>((const A*)gate_up, row_stride, pos_of_pair + p0, weights ? weights + p0 : nullptr, (A*)y, y_stride, n,
                                                                                           (int)inter, limit, alpha);
        }
    };
    if (act_f32) launch(vec ? &glu_clamp_pairs_kernel<float, 8> : &glu_clamp_pairs_kernel<float, 1>, &glu_clamp_rows_kernel<float>, 0.f);
    else launch(vec ? &glu_clamp_pairs_kernel<bf16, 8> : &glu_clamp_pairs_kernel<bf16, 1>, &glu_clamp_rows_kernel<bf16>, (bf16)0.f);
    NVH_CHECK_LAUNCH("nvh_glu_clamp_pairs");
    return NVH_OK;
}

extern "C" int32_t nvh_moe_combine(const void* y, int64_t y_row_stride, const int32_t* pos_of_pair, const float* weights, const void* shared,
                                   int64_t shared_stride, const float* shared_gate, int64_t shared_gate_stride, float* out, int64_t num_tokens, int64_t dim,
                                   int64_t top, int32_t act_f32, nvh_stream_t stream) {
    NVH_REQUIRE(y && pos_of_pair && out && num_tokens >= 0 && dim > 0 && top > 0 && y_row_stride >= dim, NVH_EINVAL, "nvh_moe_combine: bad argument");
    if (num_tokens == 0) return NVH_OK;
    hipStream_t st = (hipStream_t)stream;
    if (act_f32) moe_combine_kernel<float><<<dim3((unsigned)num_tokens), 256, 0, st>>>((const float*)y, y_row_stride, pos_of_pair, weights, (const float*)shared, shared_stride, shared_gate, shared_gate_stride, out, (int)dim, (int)top);
    else moe_combine_kernel<bf16><<<dim3((unsigned)num_tokens), 256, 0, st>>>((const bf16*)y, y_row_stride, pos_of_pair, weights, (const bf16*)shared, shared_stride, shared_gate, shared_gate_stride, out, (int)dim, (int)top);
    NVH_CHECK_LAUNCH("nvh_moe_combine");
    return NVH_OK;
}
