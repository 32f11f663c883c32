// The any-shape product as device functions, shared by the plain entry point (one weight matrix, rows as they lie) and
// the grouped one (a weight matrix per tile, rows gathered through an index): a tile of the grid is handed the rows it
// covers through `RowMap`, everything else is the same code, so a row's result never depends on which entry point, tile
// or batch it travelled in.
#pragma once
#include "common.h"

namespace nvh_any {

// Which rows a 64-row tile covers: row r of the tile (r < rows) is read from x row `src(r)` and written to y row `dst(r)`.
struct RowMap {
    const int32_t* gather;     // source row per destination row (null: the destination row itself)
    int row0;                  // first destination row of the tile
    int rows;                  // real rows of the tile (<= 64)
    __device__ __forceinline__ int64_t dst(int r) const { return row0 + r; }
    __device__ __forceinline__ int64_t src(int r) const { return gather ? gather[row0 + r] : row0 + r; }
};

__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

// ---------------------------------------------------------------------------------------------------------------
// y[M, N] = x[M, K] w[N, K]^T (+ bias[N]) (times sigmoid(gate[m, n]) when a gate is given; squared relu with `relu2`) for ANY M, N, K (ragged
// edges are zero-filled on the way into LDS and masked on the way out).  The order in which an output element sums over k depends on
// (N, K) only, never on M or on the row's place in the batch.  bf16: 64 x 64 tile per workgroup, four waves of 2 x 2 MFMA 16x16x32
// tiles, fp32 accumulation.  fp32: see gemm_any_f32_tile_body.
constexpr int GT = 64, GK = 64, GLD = GK + 8;

// What happens to a sum on its way out.
struct Epilogue {
    const bf16* bias;
    const bf16* gate;
    int64_t ldg;
    int relu2;
    __device__ __forceinline__ float operator()(float v, int64_t m, int n) const {
        if (bias) v += (float)bias[n];
        if (gate) v *= sigmoid((float)gate[m * ldg + n]);
        if (relu2) {
            v = fmaxf(v, 0.f);
            v *= v;
        }
        return v;
    }
};

template <bool OUT_F32, bool VEC>
__device__ __forceinline__ void gemm_any_bf16_tile_body(const bf16* __restrict__ x, int64_t ldx, const bf16* __restrict__ w, int64_t ldw, void* __restrict__ yv,
                                                        int64_t ldy, const RowMap rm, int n0, int N, int K, const Epilogue epi, bf16* lds) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int lr = tid >> 2, lc = (tid & 3) * 16;            // this thread's row and first column of the 64 x 64 tile
    // (VEC: rows beyond the tile's or the matrix's repeat a real one - their sums are not written; columns beyond K are zeroed on the way into LDS)
    const bf16* xrow = x + rm.src(min(lr, rm.rows - 1)) * ldx;
    const bf16* wrow = w + (int64_t)min(n0 + lr, N - 1) * ldw;
    // This thread's four 16-byte pieces of a k-step's tiles (x: 0, 1; w: 2, 3) are loaded two steps ahead: two register sets, two LDS
    // buffers, one barrier a step.  A load is issued on every path (past the end: the last columns once more), so the waits leave the
    // younger set in flight.
    bf16x8 pre_a[4], pre_b[4];
    auto gload = [&](int k0, bf16x8 (&pre)[4]) {
#pragma unroll
        for (int which = 0; which < 2; ++which)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const bf16* src = which ? wrow : xrow;
                const int kc = k0 + lc + half * 8;
                if constexpr (VEC) {
                    pre[which * 2 + half] = *reinterpret_cast<const bf16x8*>(src + min(kc, K - 8));
                } else {
                    bf16x8 v;
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = kc + e < K ? src[kc + e] : (bf16)0.f;
                    pre[which * 2 + half] = v;
                }
            }
    };
    auto step = [&](int k0, bf16* buf, bf16x8 (&pre)[4]) {
        bf16 *xs = buf, *ws = buf + GT * GLD;
#pragma unroll
        for (int which = 0; which < 2; ++which)
#pragma unroll
            for (int half = 0; half < 2; ++half)
                *reinterpret_cast<bf16x8*>((which ? ws : xs) + lr * GLD + lc + half * 8) = !VEC || k0 + lc + half * 8 < K ? pre[which * 2 + half] : bf16x8{};
        __syncthreads();
        gload(k0 + 2 * GK, pre);
#pragma unroll
        for (int ks = 0; ks < GK / 32; ++ks) {
            bf16x8 wf[2], xf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                wf[i] = *reinterpret_cast<const bf16x8*>(ws + (wn + i * 16 + fr) * GLD + ks * 32 + fq * 8);
                xf[i] = *reinterpret_cast<const bf16x8*>(xs + (wm + i * 16 + fr) * GLD + ks * 32 + fq * 8);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
        }
    };
    gload(0, pre_a);
    gload(GK, pre_b);
    int k0 = 0;
    for (; k0 + GK < K; k0 += 2 * GK) {
        step(k0, lds, pre_a);
        step(k0 + GK, lds + 2 * GT * GLD, pre_b);
    }
    if (k0 < K) step(k0, lds, pre_a);
    // lane holds, for weight tile i and row tile j: row m = wm + 16 j + fr, columns n = wn + 16 i + 4 fq + e
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = wm + j * 16 + fr;
            if (r >= rm.rows) continue;
            const int64_t m = rm.dst(r);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = n0 + wn + i * 16 + fq * 4 + e;
                if (n >= N) continue;
                const float v = epi(acc[i][j][e], m, n);
                if constexpr (OUT_F32) ((float*)yv)[m * ldy + n] = v;
                else ((bf16*)yv)[m * ldy + n] = (bf16)v;
            }
        }
}

template <bool OUT_F32>
__device__ __forceinline__ void gemm_any_bf16_tile(const bf16* __restrict__ x, int64_t ldx, const bf16* __restrict__ w, int64_t ldw,
                                                   const bf16* __restrict__ bias, void* __restrict__ yv, int64_t ldy, const RowMap rm, int n0, int N, int K,
                                                   int vec_ok, const bf16* __restrict__ gate = nullptr, int64_t ldg = 0, int relu2 = 0) {
    __shared__ __attribute__((aligned(16))) bf16 lds[4 * GT * GLD];
    const Epilogue epi{bias, gate, ldg, relu2};
    if (vec_ok) gemm_any_bf16_tile_body<OUT_F32, true>(x, ldx, w, ldw, yv, ldy, rm, n0, N, K, epi, lds);
    else gemm_any_bf16_tile_body<OUT_F32, false>(x, ldx, w, ldw, yv, ldy, rm, n0, N, K, epi, lds);
}

// The same tile when few of its rows are real (at most 16 NR; K a multiple of 32, 16-byte rows): a wave takes 16 columns and all rows, the
// operands go from memory to the matrix cores without LDS, U products of 32 ahead, so what a wave waits for is the weights' stream and
// not a barrier a step.  Sums in the same order as above: bit for bit the same results.
template <bool OUT_F32, int NR>
__device__ __forceinline__ void gemm_any_bf16_few_rows(const bf16* __restrict__ x, int64_t ldx, const bf16* __restrict__ w, int64_t ldw, void* __restrict__ yv,
                                                       int64_t ldy, const RowMap rm, int n0, int N, int K, const Epilogue epi) {
    constexpr int U = NR == 1 ? 8 : 4;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, fr = lane & 15, fq = lane >> 4;
    const int nw = n0 + wave * 16;
    if (nw >= N) return;
    const bf16* wp = w + (int64_t)min(nw + fr, N - 1) * ldw + fq * 8;
    const bf16* xp[NR];
    f32x4 acc[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        xp[j] = x + rm.src(min(16 * j + fr, rm.rows - 1)) * ldx + fq * 8;
        acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8 wa[U], xa[U][NR], wb[U], xb[U][NR];
    auto load = [&](int k0, bf16x8 (&wf)[U], bf16x8 (&xf)[U][NR]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + 32 * u, K - 32);
            wf[u] = *reinterpret_cast<const bf16x8*>(wp + k);
#pragma unroll
            for (int j = 0; j < NR; ++j) xf[u][j] = *reinterpret_cast<const bf16x8*>(xp[j] + k);
        }
    };
    auto multiply = [&](int k0, bf16x8 (&wf)[U], bf16x8 (&xf)[U][NR]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + 32 * u < K)
#pragma unroll
                for (int j = 0; j < NR; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf[u][j], acc[j], 0, 0, 0);
    };
    load(0, wa, xa);
    for (int k0 = 0; k0 < K; k0 += 64 * U) {
        load(k0 + 32 * U, wb, xb);
        multiply(k0, wa, xa);
        load(k0 + 64 * U, wa, xa);
        multiply(k0 + 32 * U, wb, xb);
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int r = 16 * j + fr;
        if (r >= rm.rows) continue;
        const int64_t m = rm.dst(r);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = nw + fq * 4 + e;
            if (n >= N) continue;
            const float v = epi(acc[j][e], m, n);
            if constexpr (OUT_F32) ((float*)yv)[m * ldy + n] = v;
            else ((bf16*)yv)[m * ldy + n] = (bf16)v;
        }
    }
}

// fp32: rows r0 .. r0 + 16 MR - 1 of the rows `rm` covers and columns n0 .. n0 + 16 NC - 1, on the matrix cores (16x16x4, products and sums in
// fp32).  The four waves of the workgroup split k: wave w takes the chunks of 32 numbered w, w + 4, ..., straight from memory (whole 128-byte
// lines a row, DEPTH chunks ahead, no barrier), and the four partial tiles meet in LDS as (p0 + p1) + (p2 + p3) - an order that depends on K alone.
// Bound by the matrix cores (124 TFLOP/s measured on independent products of this form) and the L1 in front of them once the grid covers the
// chip, below that by the chain of a wave's chunks.  Rows x columns x k, us a launch, before (64 x 64 tiles on the vector ALU, one LDS stage) and
// now: 1 x 1024 x 1024 97 -> 6.3, 64 x 4096 x 1024 115 -> 12.7, 301 x 1024 x 1024 108 -> 21, 301 x 6144 x 1024 162 -> 72 (53 TFLOP/s),
// 1000 x 32768 x 1024 1797 -> 1142 (59 TFLOP/s).
constexpr int F32_CHUNK = 32;
// Four consecutive sums of row r of the tile, from column n on, on their way out.
__device__ __forceinline__ void f32_finish(const f32x4& sum, const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, const RowMap& rm, int r, int n, int N,
                                           const float* __restrict__ gate, int64_t ldg, int relu2) {
    if (r >= rm.rows) return;
    const int64_t m = rm.dst(r);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (n + e >= N) continue;
        float v = sum[e] + (bias ? bias[n + e] : 0.f);
        if (gate) v *= sigmoid(gate[m * ldg + n + e]);
        if (relu2) {
            v = fmaxf(v, 0.f);
            v *= v;
        }
        y[m * ldy + n + e] = v;
    }
}
template <int MR, int NC, bool VEC>
__device__ __forceinline__ void gemm_any_f32_tile_body(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw,
                                                       const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, const RowMap rm, int r0, int n0, int N,
                                                       int K, const float* __restrict__ gate, int64_t ldg, int relu2, f32x4* lds) {
    constexpr int DEPTH = MR * NC == 1 ? 4 : 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, fr = lane & 15, fq = lane >> 4;
    const float *xp[MR], *wp[NC];
    f32x4 acc[NC][MR];
#pragma unroll
    for (int j = 0; j < MR; ++j) xp[j] = x + rm.src(min(r0 + 16 * j + fr, rm.rows - 1)) * ldx;      // (rows beyond the tile's repeat its last: not written)
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        wp[i] = w + (int64_t)min(n0 + 16 * i + fr, N - 1) * ldw;
#pragma unroll
        for (int j = 0; j < MR; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int chunks = (K + F32_CHUNK - 1) / F32_CHUNK;
    f32x4 xf[DEPTH][2][MR], wf[DEPTH][2][NC];
    auto load4 = [&](const float* row, int k) {
        if constexpr (VEC) {
            return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));                             // (K a multiple of 4)
        } else {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = row[min(k + e, K - 1)];
            return v;
        }
    };
    auto load = [&](int c, f32x4 (&xs)[2][MR], f32x4 (&ws)[2][NC]) {
        const int k = min(c, chunks - 1) * F32_CHUNK + 4 * fq;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int j = 0; j < MR; ++j) xs[half][j] = load4(xp[j], k + 16 * half);
#pragma unroll
            for (int i = 0; i < NC; ++i) ws[half][i] = load4(wp[i], k + 16 * half);
        }
    };
    auto multiply = [&](const f32x4 (&xs)[2][MR], const f32x4 (&ws)[2][NC]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NC; ++i)
#pragma unroll
                    for (int j = 0; j < MR; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ws[h][i][e], xs[h][j][e], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(wave + 4 * d, xf[d], wf[d]);
    // (no branch inside: the loads of a set go back to the registers it was read from, and only their age is waited for)
    int c0 = wave;
    for (; c0 + 4 * (DEPTH - 1) < K / F32_CHUNK; c0 += 4 * DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            multiply(xf[d], wf[d]);
            load(c0 + 4 * (d + DEPTH), xf[d], wf[d]);
            __builtin_amdgcn_sched_barrier(0);               // (left alone, all the loads sink to the end of the loop)
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        const int c = c0 + 4 * d;
        if (c >= chunks) break;
        if ((c + 1) * F32_CHUNK > K) {                       // the last chunk: what lies beyond K counts as zero on both sides
            const int k = c * F32_CHUNK + 4 * fq;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int h = e >> 2;
                const bool in = k + 16 * h + (e & 3) < K;
#pragma unroll
                for (int j = 0; j < MR; ++j) xf[d][h][j][e & 3] = in ? xf[d][h][j][e & 3] : 0.f;
#pragma unroll
                for (int i = 0; i < NC; ++i) wf[d][h][i][e & 3] = in ? wf[d][h][i][e & 3] : 0.f;
            }
        }
        multiply(xf[d], wf[d]);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < MR; ++j) lds[(wave * NC * MR + i * MR + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    // fragment (i, j) is finished by one wave: row r0 + 16 j + fr, columns n0 + 16 i + 4 fq + e
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < MR; ++j) {
            constexpr int F = NC * MR;
            const int f = i * MR + j;
            if (f % 4 != wave) continue;
            const f32x4 sum = (lds[f * 64 + lane] + lds[(F + f) * 64 + lane]) + (lds[(2 * F + f) * 64 + lane] + lds[(3 * F + f) * 64 + lane]);
            // (f32_finish, written out: through the function the compiler asks about the gate lane by lane, 16 x 192 x 128 a head 3.9 us instead of 3.7)
            const int r = r0 + 16 * j + fr;
            if (r >= rm.rows) continue;
            const int64_t m = rm.dst(r);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = n0 + 16 * i + 4 * fq + e;
                if (n >= N) continue;
                float v = sum[e] + (bias ? bias[n] : 0.f);
                if (gate) v *= sigmoid(gate[m * ldg + n]);
                if (relu2) {
                    v = fmaxf(v, 0.f);
                    v *= v;
                }
                y[m * ldy + n] = v;
            }
        }
}

// The same product through LDS (K a multiple of 32, 16-byte rows): every wave has a ring of STAGES chunks of its own there, filled by 16-byte LDS-DMA
// STAGES chunks ahead, so that neither registers nor barriers bound how much is on its way, and tiles can be larger: what bounds the form above is
// the operands' way to the CUs, which a 64 x 64 tile has half as much of as four 32 x 32 ones.  Chunks, products and sums as above: bit for bit the
// same results.
// us, the form above and this, rows x columns x k: 1 x 1024 x 1024 5.9 and 4.7, 64 x 1024 x 1024 11.6 and 5.2, 64 x 4096 x 1024 13.0 and 9.6,
// 301 x 1024 x 1024 21.2 and 13.9, 301 x 6144 x 1024 74 and 48 (79 TFLOP/s of the 124 that independent products reach), 512 x 6144 x 1024 112 and 67,
// 1 x 32000 x 1024 32.1 and 27.5, 1 x 12288 x 5120 49.5 and 46.0.
template <int MR, int NC, int STAGES>
constexpr int f32_ring_bytes() {
    return 4 * STAGES * 16 * (MR + NC) * 128;                // (at least the four waves' partial tiles, 1 KB a fragment: STAGES 2 (MR + NC) >= MR NC)
}
template <int MR, int NC, int STAGES>
__device__ __forceinline__ void gemm_any_f32_ring(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw,
                                                  const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, const RowMap rm, int r0, int n0, int N,
                                                  int K, const float* __restrict__ gate, int64_t ldg, int relu2, char* lds) {
    constexpr int STAGE = 16 * (MR + NC) * 128, PIECES = 2 * (MR + NC);
    static_assert(STAGES * 2 * (MR + NC) >= MR * NC && PIECES * (STAGES - 1) < 64, "the partial tile fits the ring; vmcnt is six bits");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, fr = lane & 15, fq = lane >> 4;
    char* ring = lds + wave * STAGES * STAGE;
    // A stage: 16 NC rows of w, then 16 MR of x, 32 k (128 bytes) each; 16-byte piece c of row r lies at place c ^ ((r >> 1) & 7), which spreads a
    // fragment read over all banks.  A DMA instruction brings 8 rows.
    const float* src[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const bool of_w = i < 2 * NC;
        const int r = 8 * (of_w ? i : i - 2 * NC) + (lane >> 3), piece = (lane & 7) ^ ((r >> 1) & 7);
        const float* row = of_w ? w + (int64_t)min(n0 + r, N - 1) * ldw : x + rm.src(min(r0 + r, rm.rows - 1)) * ldx;      // (repeated rows are not written)
        src[i] = row + 4 * piece + F32_CHUNK * wave;
    }
    const int chunks = K / F32_CHUNK, mine = (chunks - wave + 3) / 4;
    auto stage = [&](int j) {
        char* base = ring + j % STAGES * STAGE;
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            __builtin_amdgcn_global_load_lds((const GLOBAL_AS void*)(src[i] + 4 * F32_CHUNK * j), (LDS_AS void*)(base + 1024 * i), 16, 0, 0);
    };
    f32x4 acc[NC][MR];
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < MR; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < STAGES && j < mine; ++j) stage(j);
    for (int j = 0; j < mine; ++j) {
        const int ahead = min(STAGES - 1, mine - 1 - j);     // chunks behind this one that may still be on their way
        if (STAGES > 3 && ahead >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 3 ? 3 * PIECES : 0) : "memory");
        else if (STAGES > 2 && ahead >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 2 ? 2 * PIECES : 0) : "memory");
        else if (STAGES > 1 && ahead >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const char *ws = ring + j % STAGES * STAGE, *xs = ws + 16 * NC * 128;
        f32x4 xf[2][MR], wf[2][NC];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int r = 16 * i + fr;
                wf[h][i] = *reinterpret_cast<const f32x4*>(ws + r * 128 + (((4 * h + fq) ^ ((r >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int i = 0; i < MR; ++i) {
                const int r = 16 * i + fr;
                xf[h][i] = *reinterpret_cast<const f32x4*>(xs + r * 128 + (((4 * h + fq) ^ ((r >> 1) & 7)) << 4));
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the chunk is in registers: its stage is free
        __builtin_amdgcn_sched_barrier(0);
        if (j + STAGES < mine) stage(j + STAGES);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NC; ++i)
#pragma unroll
                    for (int m = 0; m < MR; ++m) acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[h][i][e], xf[h][m][e], acc[i][m], 0, 0, 0);
    }
    f32x4* part = reinterpret_cast<f32x4*>(ring);            // (this wave's ring: nobody else's DMA is under way in it)
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < MR; ++j) part[(i * MR + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    constexpr int RING = STAGES * STAGE / 16;                // (in f32x4)
    const f32x4* parts = reinterpret_cast<const f32x4*>(lds);
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < MR; ++j) {
            const int f = i * MR + j;
            if (f % 4 != wave) continue;
            const f32x4* p = parts + f * 64 + lane;
            f32_finish((p[0] + p[RING]) + (p[2 * RING] + p[3 * RING]), bias, y, ldy, rm, r0 + 16 * j + fr, n0 + 16 * i + 4 * fq, N, gate, ldg, relu2);
        }
}

template <int MR, int NC>
__device__ __forceinline__ void gemm_any_f32_tile(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw,
                                                  const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, const RowMap rm, int r0, int n0, int N, int K,
                                                  int vec_ok, const float* __restrict__ gate = nullptr, int64_t ldg = 0, int relu2 = 0) {
    __shared__ f32x4 lds[4 * MR * NC * 64];
    __syncthreads();                                         // (a tile before this one may still be read)
    if (vec_ok) gemm_any_f32_tile_body<MR, NC, true>(x, ldx, w, ldw, bias, y, ldy, rm, r0, n0, N, K, gate, ldg, relu2, lds);
    else gemm_any_f32_tile_body<MR, NC, false>(x, ldx, w, ldw, bias, y, ldy, rm, r0, n0, N, K, gate, ldg, relu2, lds);
}

// Whether rows of fp32 operands can be read 16 bytes at a time.
__host__ __forceinline__ int f32_vec_ok(const void* x, int64_t ldx, const void* w, int64_t K) {
    return K % 4 == 0 && ldx % 4 == 0 && nvh_aligned16(x) && nvh_aligned16(w);
}

// y = x w^T in bf16 through LDS rings (moe.hip), without a bias; false: a shape, stride or alignment that it does not take.
bool launch_short_product(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, bool out_f32, hipStream_t st);

// The same for a product per head (nvh_gemm_heads_nt), with its gate.
bool launch_short_heads(const void* x, int64_t ldx, int64_t x_head, const void* w, void* y, int64_t ldy, int64_t y_head, int64_t M, int64_t heads, int64_t N, int64_t K,
                        const void* gate, int64_t ldg, hipStream_t st);

}  // namespace nvh_any
