// Shared device helpers and host-side error plumbing for libnanovllm_hip.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <utility>
#include <stdint.h>
#include <stdio.h>
#include "../../include/nanovllm_hip.h"

typedef __bf16 bf16;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define GLOBAL_AS __attribute__((address_space(1)))
#define LDS_AS __attribute__((address_space(3)))

// ---- host side --------------------------------------------------------------------
void nvh_set_error(const char* fmt, ...);

#define NVH_REQUIRE(cond, code, ...)          \
    do {                                      \
        if (!(cond)) {                        \
            nvh_set_error(__VA_ARGS__);       \
            return (code);                    \
        }                                     \
    } while (0)

#define NVH_CHECK_LAUNCH(name)                                                   \
    do {                                                                         \
        hipError_t e__ = hipGetLastError();                                      \
        if (e__ != hipSuccess) {                                                 \
            nvh_set_error("%s: launch failed: %s", name, hipGetErrorString(e__)); \
            return NVH_ELAUNCH;                                                  \
        }                                                                        \
    } while (0)

// A kernel with more than 64 KB of dynamic LDS needs an attribute for it, on every device once: `granted` remembers them, a bit a device.  False: refused.
static inline bool nvh_grant_lds(std::atomic<uint64_t>& granted, const void* kernel, int bytes) {
    int dev = 0;
    const bool known = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64;
    if (known && (granted.load(std::memory_order_relaxed) >> dev & 1)) return true;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        (void)hipGetLastError();                             // (the caller reports it; not the next launch)
        return false;
    }
    if (known) granted.fetch_or(1ull << dev, std::memory_order_relaxed);
    return true;
}

// Merge per-range attention partials ([row][split][128] fp32 + [row][split][2] (max, sum)) into bf16 rows.
int32_t nvh_launch_attn_combine(const float* ws_acc, const float* ws_ml, void* out, int64_t rows, int num_splits,
                                const int32_t* ctx_lens, int hq, int min_range, const int32_t* seq_active, hipStream_t st);

// Device address, on the current GPU, of the built-in partial-result array of nvh_attn_decode_noalloc (resolved on
// first use; nvh_device_check resolves it ahead of time for callers that will run under graph capture).
int32_t nvh_noalloc_scratch(float** out);
// Device address, on the current GPU, of the arrival counters the decode attention uses to merge key ranges in its own
// launch (resolved on first use, or by nvh_device_check before a graph capture).
int32_t nvh_decode_arrivals(unsigned** out);
// nvh_attn_decode_fused_qkv whose sequences are dispatched in the given order (attention_decode.hip; null: as they lie), and nvh_embedding with
// one workgroup more that leaves that order, the longest context first (elementwise.hip).
#define NVH_ORDER_MAX 1024
int32_t nvh_attn_decode_fused_qkv_ordered(const void* qkv, int64_t token_stride, const void* q_norm_weight, const void* k_norm_weight, float eps,
                                          const int64_t* positions, const float* cos_sin, void* k_cache, void* v_cache, const int32_t* context_lens,
                                          const int32_t* block_tables, int64_t table_stride, int64_t batch, int64_t num_q_heads, int64_t num_kv_heads,
                                          int64_t head_dim, float softmax_scale, void* out, int32_t num_splits, int32_t min_range_keys, void* workspace,
                                          const int32_t* order, hipStream_t stream);
int32_t nvh_embedding_order(const int64_t* ids, const void* table, void* out, int64_t num_tokens, int64_t dim, int64_t vocab_start, int64_t vocab_rows,
                            const int32_t* context_lens, int32_t* order, int64_t batch, hipStream_t st);

// Decode attention over pieces that the step itself lays out (attention_decode.hip, "Pieces"): written by nvh_embedding_pieces (elementwise.hip), read by the
// attention of every layer.
struct NvhDecodePiece {
    int seq;                   // sequence | range << 16 | ranges << 24; 0xffff: none
    int start, end;            // its keys
    int context;               // of the sequence
    int page, position;        // of its first key; of the sequence's new token
    int next;                  // the piece that its workgroup goes on with; -1: none
    int follows;               // 1: a workgroup comes to it from another piece
};
struct NvhDecodePieces {
    NvhDecodePiece* pieces;    // [capacity], longest first
    unsigned* arrivals;        // [rows * kv heads], zero: ranges of a sequence that have left their partial result
    int capacity;              // nvh_piece_capacity()
};
#define NVH_PIECE_RANGES 8     // most pieces of a sequence
#define NVH_PIECE_TRIPS 8      // sequences of up to so many trips of 64 keys are not cut
#define NVH_CHAIN_TRIPS 6      // trips a workgroup from which on pieces are chained
static inline int nvh_pieces_per_head(int64_t num_kv_heads) { return num_kv_heads < 256 ? (int)(256 / num_kv_heads) : 1; }
// The captured step that a batch of so many rows runs in (ModelRunner.decode_buckets).  Whether there are pieces, and how many places for them beside one a
// sequence, decides where sequences are cut and so the last bits: both follow from this, not from the rows, so that a batch run eagerly is cut like the captured
// one (a padded row takes a place of its own and nothing else).
static inline int64_t nvh_captured_rows(int64_t rows) { return rows > 8 ? (rows + 15) / 16 * 16 : rows > 4 ? 8 : rows > 2 ? 4 : rows; }
static inline bool nvh_takes_pieces(int64_t rows, int64_t num_kv_heads) { return num_kv_heads > 0 && rows > 0 && nvh_captured_rows(rows) <= 2 * nvh_pieces_per_head(num_kv_heads); }
// Places in the list: one a sequence and some that cutting fills (pieces are made longer until they are enough).  Every place is a workgroup, and an empty one
// costs about 10 ns: up to one sequence a workgroup as many as cutting by one and a half shares can fill, above that a quarter (64 of 64..100 keys: 6 us a step more
// with two thirds).
static inline int nvh_piece_capacity(int64_t rows, int64_t num_kv_heads) {
    const int per_head = nvh_pieces_per_head(num_kv_heads);
    return (int)rows + (nvh_captured_rows(rows) <= per_head ? (2 * per_head + 2) / 3 : (per_head + 3) / 4);
}
// Room for the list of any up to `rows` sequences: fewer may take more places (with 8 kv heads 32 take 54 and 33 take 41), and a mixed step of `rows` lays one
// out for those of them that decode.
static inline int nvh_piece_room(int64_t rows, int64_t num_kv_heads) { return (int)rows + (2 * nvh_pieces_per_head(num_kv_heads) + 2) / 3; }
int32_t nvh_attn_decode_fused_qkv_pieces(const void* qkv, int64_t token_stride, const void* q_norm_weight, const void* k_norm_weight, float eps,
                                         const int64_t* positions, const float* cos_sin, void* k_cache, void* v_cache, const int32_t* context_lens,
                                         const int32_t* block_tables, int64_t table_stride, int64_t batch, int64_t num_q_heads, int64_t num_kv_heads,
                                         int64_t head_dim, float softmax_scale, void* out, void* workspace, const NvhDecodePieces& pieces, hipStream_t stream);
int32_t nvh_embedding_pieces(const int64_t* ids, const void* table, void* out, int64_t num_tokens, int64_t dim, int64_t vocab_start, int64_t vocab_rows,
                             const int32_t* context_lens, const int64_t* positions, const int32_t* block_tables, int64_t table_stride, int64_t batch, int64_t num_q_heads,
                             int64_t num_kv_heads, const NvhDecodePieces& pieces, hipStream_t st);

// nvh_attn_varlen, and whether another step's launches run beside it (attention_prefill.hip).
int32_t nvh_attn_varlen_beside(const void* q, int64_t q_token_stride, const void* k, const void* v, int64_t kv_token_stride, const int32_t* cu_seqlens_q,
                               const int32_t* cu_seqlens_k, const int32_t* block_tables, int64_t table_stride, int64_t batch, int64_t max_seqlen_q,
                               int64_t max_seqlen_k, int64_t total_q, int64_t num_q_heads, int64_t num_kv_heads, int64_t head_dim, float softmax_scale,
                               void* out, int32_t num_splits, void* workspace, bool beside, nvh_stream_t stream);

// Routing and measurement switches.  Every kernel choice in this library is a pure function of the call's shapes; the
// switches below exist for A/B measurements and for tests that compare two routes.  They are read from the environment
// (variable NVH_<name>) ONCE per process, and only when NVH_TUNING=1 is set, so that a stray variable in a user's
// environment cannot change routing; afterwards only nvh_set_switch() changes them.  A switch is either unset (-1) or holds
// a non-negative value (a variable that is set to something that is not a number counts as 1).
#define NVH_SWITCHES(X)                                                                                              \
    X(DECODE_TARGET_WGS) X(DECODE_FULL_WGS) X(DECODE_MERGE_IN_LAUNCH) X(ATTN_KS) X(VARLEN_LONG_SPLITS)             \
    X(ATTN_HEAD_MAJOR) X(ATTN_RB1) X(NORM_NO_WIDE) X(GEMM_NO_WIDE_STORE) X(GEMM_NO_XCD) X(GEMM_NO_NT)              \
    X(GEMM_NO_SKINNY) X(GEMM_M32_SKINNY) X(GEMM_FORCE_TILE) X(GEMM_NO_256) X(NO_KWAVES) X(KWAVES_KMIN)             \
    X(KWAVES_NO_8) X(GEMM_S128) X(GEMM_S64) X(GEMM_NO_ROUND_CUT) X(GEMM_NO_16x64) X(GEMM_NO_KGROUPS)               \
    X(QKV_NO_8WAVE) X(SWIGLU_NO_192) X(SWIGLU_NO_96) X(NO_FUSED_QKV) X(NO_NORM_GEMM) X(NORM_GEMM_KB)               \
    X(NORM_GEMM_ROWS) X(DECODE_SLABS) X(NO_FUSED_EXCHANGE) X(NO_FUSED_DECODE)        \
    X(LM_HEAD_NO_CUT) X(NO_ROWSCALE) X(NO_DECODE_PIECES) X(EXP_A) X(EXP_B) X(ATTN_ANY_NO_MFMA) X(ATTN_ANY_SPLIT_BELOW)
enum NvhSwitch : int {
#define NVH_SW_ENUM(n) SW_##n,
    NVH_SWITCHES(NVH_SW_ENUM)
#undef NVH_SW_ENUM
    SW_COUNT
};
int64_t nvh_switch(NvhSwitch s);                                   // -1: unset
static inline bool nvh_switch_on(NvhSwitch s) { return nvh_switch(s) >= 0; }
static inline int64_t nvh_switch_or(NvhSwitch s, int64_t dflt) { const int64_t v = nvh_switch(s); return v >= 0 ? v : dflt; }

static inline bool nvh_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
static inline int64_t nvh_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- device side ------------------------------------------------------------------
// f(0), f(1), .. f(N - 1) with constants: a loop whose body chooses by its index, written out whatever its length.
template <int... I, typename F>
__device__ __forceinline__ void nvh_static_for_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void nvh_static_for(F&& f) { nvh_static_for_of(std::make_integer_sequence<int, N>{}, f); }

// Sum / max over the 16 lanes of a DPP row (lanes 16r..16r+15); every lane of the row
// receives the result.  quad_perm[1,0,3,2], quad_perm[2,3,0,1], row_half_mirror, row_mirror.
#define NVH_DPP(x, ctrl) \
    __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (x)), (ctrl), 0xF, 0xF, true))

__device__ __forceinline__ float row16_sum(float x) {
    x += NVH_DPP(x, 0xB1);
    x += NVH_DPP(x, 0x4E);
    x += NVH_DPP(x, 0x141);
    x += NVH_DPP(x, 0x140);
    return x;
}
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, NVH_DPP(x, 0xB1));
    x = fmaxf(x, NVH_DPP(x, 0x4E));
    x = fmaxf(x, NVH_DPP(x, 0x141));
    x = fmaxf(x, NVH_DPP(x, 0x140));
    return x;
}
// With the lane 16 (32) places on, modulo 32 (64): rows (halves) of the wave exchanged on the vector ALU; a shuffle goes through the LDS unit and takes some
// 100 cycles of a chain.  Both lanes of a pair receive the same bits, those of x op shuffled x.
__device__ __forceinline__ float pair16_sum(float x) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float pair32_sum(float x) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float pair16_max(float x) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float pair32_max(float x) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
// Over the four lanes l, l + 16, l + 32, l + 48 (a row of results of the matrix cores).
__device__ __forceinline__ float rows_sum(float x) { return pair32_sum(pair16_sum(x)); }
__device__ __forceinline__ float rows_max(float x) { return pair32_max(pair16_max(x)); }
// Full 64-lane reductions (result in every lane).
__device__ __forceinline__ float wave_sum(float x) { return rows_sum(row16_sum(x)); }
__device__ __forceinline__ float wave_max(float x) { return rows_max(row16_max(x)); }

__device__ __forceinline__ float bf2f(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 f2bf(float v) { return (bf16)v; }

// Per-head RMSNorm -> bf16 -> x weight -> bf16 -> half-split RoPE -> bf16 for one head of 128 elements held
// by a 16-lane DPP row: lane c owns elements [8c, 8c+8).  The rotation partner (i +- 64) lives in lane c^8
// and arrives through a row rotation by 8.  cs_row: fp32 [cos(64) | sin(64)] of the token's position.
// Used by every kernel that applies the q/k epilogue, so they all produce identical bits.
__device__ __forceinline__ bf16x8 qknorm_rope_head_cs(bf16x8 x, bf16x8 w, f32x4 c0, f32x4 c1, f32x4 s0, f32x4 s1, int c, float eps) {
    float v[8];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        v[j] = bf2f(x[j]);
        ss += v[j] * v[j];
    }
    ss = row16_sum(ss);
    const float inv = 1.0f / sqrtf(ss / 128.0f + eps);
    bf16x8 out;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float n = bf2f(f2bf(bf2f(f2bf(v[j] * inv)) * bf2f(w[j])));
        const float p = NVH_DPP(n, 0x128);                       // row_ror:8 -> lane c^8's value
        const float cs = j < 4 ? c0[j] : c1[j - 4];
        const float sn = j < 4 ? s0[j] : s1[j - 4];
        // first half: x1*cos - x2*sin (own = x1); second half: x2*cos + x1*sin (own = x2)
        const float y = (c < 8) ? n * cs - p * sn : n * cs + p * sn;
        out[j] = f2bf(y);
    }
    return out;
}
__device__ __forceinline__ bf16x8 qknorm_rope_head(bf16x8 x, bf16x8 w, const float* __restrict__ cs_row, int c, float eps) {
    // lane c's cos / sin values: columns 8 (c & 7) .. + 7 of the position's row
    const f32x4 c0 = *reinterpret_cast<const f32x4*>(cs_row + 8 * (c & 7));
    const f32x4 c1 = *reinterpret_cast<const f32x4*>(cs_row + 8 * (c & 7) + 4);
    const f32x4 s0 = *reinterpret_cast<const f32x4*>(cs_row + 64 + 8 * (c & 7));
    const f32x4 s1 = *reinterpret_cast<const f32x4*>(cs_row + 64 + 8 * (c & 7) + 4);
    return qknorm_rope_head_cs(x, w, c0, c1, s0, s1, c, eps);
}

// Eight consecutive elements p[off .. off + 7] as floats; those at or beyond `valid` read as zero.  `vec`: 16-byte accesses are allowed.
template <typename A>
__device__ __forceinline__ void nvh_load8(const A* p, int64_t off, int valid, bool vec, float (&out)[8]) {
    if (vec && valid >= 8) {
        if constexpr (sizeof(A) == 2) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(p + off);
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = (float)v[i];
        } else {
            const f32x4 a = *reinterpret_cast<const f32x4*>(p + off), b = *reinterpret_cast<const f32x4*>(p + off + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                out[i] = a[i];
                out[4 + i] = b[i];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = i < valid ? (float)p[off + i] : 0.f;
    }
}

// From this many elements on an elementwise launch takes eight a lane (two workgroups a CU); fewer are faster one a lane (gelu, 64 x 3072: 3.1 and 2.2 us).
constexpr int64_t NVH_PIECES = 1 << 20;
// 0 silu, 1 gelu (tanh form), 2 squared relu.
__device__ __forceinline__ float nvh_activation(float g, int act) {
    if (act == 0) return g / (1.0f + expf(-g));
    if (act == 1) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    return g > 0.f ? g * g : 0.f;
}

// xIELU of bf16 rows (stream_f32.hip and, inside a product, gemm.hip): pos = softplus(p), neg = 1/2 + softplus(q).  The hardware's 2^x and log2: errors of about
// 1e-7 beside values of at least softplus' own size.
__device__ __forceinline__ float nvh_softplus_hw(float t) {
    return fmaxf(t, 0.f) + 0.6931471805599453f * __builtin_amdgcn_logf(1.0f + __builtin_amdgcn_exp2f(-fabsf(t) * 1.4426950408889634f));
}
__device__ __forceinline__ float nvh_xielu_hw(float z, float pos, float neg) {
    const float zn = fminf(z, 0.f);
    return (z > 0.f ? pos * z * z : neg * ((__builtin_amdgcn_exp2f(zn * 1.4426950408889634f) - 1.0f) - z)) + 0.5f * z;
}

// Elementwise launches over rows of `cols` columns: a lane (256 a workgroup) takes E consecutive columns, cols a multiple of E.  False: past the end.
template <int E>
__device__ __forceinline__ bool nvh_piece(int64_t rows, int cols, int64_t& row, int& c) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t per_row = (uint32_t)cols / E;
    if (i >= rows * per_row) return false;
    if (blockIdx.x < (1u << 24)) {                           // (uniform: a division in 64 bits costs more than the rest of such a kernel)
        const uint32_t r = (uint32_t)i / per_row;
        row = r;
        c = (int)(((uint32_t)i - r * per_row) * E);
    } else {
        row = i / per_row;
        c = (int)(i - row * per_row) * E;
    }
    return true;
}
// E consecutive elements (8: 16-byte accesses) on their way out.
template <typename A, int E>
__device__ __forceinline__ void nvh_store_piece(A* dst, const float (&v)[E]) {
    A out[E];
#pragma unroll
    for (int e = 0; e < E; ++e) out[e] = (A)v[e];
    if constexpr (E == 8) __builtin_memcpy(__builtin_assume_aligned(dst, 16), out, sizeof(out));
    else dst[0] = out[0];
}
template <typename A, int E>
__device__ __forceinline__ void nvh_load_piece(const A* src, float (&v)[E]) {
    if constexpr (E == 8) nvh_load8(src, 0, 8, true, v);
    else v[0] = (float)src[0];
}

// ---- packed steps --------------------------------------------------------------------------------
// The sequence that owns packed token t (cu: [batch + 1] ascending; null: token t is sequence t).
__device__ __forceinline__ int seq_of_token(const int32_t* cu, int batch, int64_t t) {
    if (!cu) return (int)t;
    int lo = 0, hi = batch - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cu[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// ---- rotary positions ---------------------------------------------------------------------------
// sin and cos of an fp32 angle through the hardware's sin(2 pi x) / cos(2 pi x): the turn count is reduced in float64 (an
// angle of thousands of radians keeps its fp32 value exactly), the functions themselves are good to about 1e-6 absolute.
// For the bf16 path; the library's sinf / cosf (used where everything is fp32) cost a few hundred instructions at such angles.
__device__ __forceinline__ void sincos_turns(float ang, float& sn, float& cs) {
    double rev = (double)ang * 0.15915494309189535;
    rev -= floor(rev);
    const float rf = (float)rev;
    sn = __builtin_amdgcn_sinf(rf);
    cs = __builtin_amdgcn_cosf(rf);
}

// The rotation's sine and cosine for activations of type A: the library functions where everything is fp32, the hardware
// path where the result is rounded to bf16 anyway.
template <typename A>
__device__ __forceinline__ void rot_sincos(float ang, float& sn, float& cs) {
    if constexpr (sizeof(A) == 4) {
        sn = sinf(ang);
        cs = cosf(ang);
    } else {
        sincos_turns(ang, sn, cs);
    }
}

// Index of the rotation partner of element i among `n` rotated dimensions, and the pair number.
__device__ __forceinline__ void pair_of(int i, int n, int interleaved, int& partner, int& pair, bool& first) {
    if (interleaved) {
        partner = i ^ 1;
        pair = i >> 1;
        first = (i & 1) == 0;
    } else {
        const int half = n >> 1;
        first = i < half;
        partner = first ? i + half : i - half;
        pair = first ? i : i - half;
    }
}

// ---- sampling pieces shared by the sampler kernels and the LM-head GEMM epilogue ------------------
struct ValIdx {
    float v;
    int64_t i;
};
__device__ __forceinline__ ValIdx better(ValIdx a, ValIdx b) {
    return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
// Philox4x32-10 counter generator.
__device__ __forceinline__ void philox(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
        c[1] = (uint32_t)p1;
        c[3] = (uint32_t)p0;
        c[0] = n0;
        c[2] = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// Scores of the exponential race for 4 consecutive columns col .. col+3 (col a multiple of 4) of `row`:
// z / T - ln(E), E ~ Exp(1) from Philox keyed by (seed; col / 4, row, offset).  score = z - ln(E), E = -ln(u), u uniform
// in (0,1): hardware log2 (1 ulp) is ample for noise.  23 random bits -> u = (k + 1/2) * 2^-23: every step is exact in
// fp32 and u stays inside [2^-24, 1 - 2^-24], so E is never 0; the clamp is the one the reference applies
// (layers/sampler.py:80, clamp_min_(1e-10)).
__device__ __forceinline__ void nvh_race_scores(const float (&z)[4], float inv_t, int64_t col, int64_t row, uint64_t seed, uint64_t offset,
                                                float (&sc)[4]) {
    if (inv_t == 0.f) {                                      // a greedy row (temperature 0): the plain logits race, no noise
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[e] = z[e];
        return;
    }
    uint32_t c[4] = {(uint32_t)(col >> 2), (uint32_t)row, (uint32_t)offset, (uint32_t)(offset >> 32)};
    philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    constexpr float LN2 = 0.6931471805599453f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float un = (float)(c[e] >> 9) * 0x1p-23f + 0x1p-24f;
        const float ex = fmaxf(-LN2 * __builtin_amdgcn_logf(un), 1e-10f);       // Exp(1) sample
        sc[e] = __builtin_fmaf(z[e], inv_t, -LN2 * __builtin_amdgcn_logf(ex));
    }
}

// Pick among `slices` candidates per row (sampler.hip): out[row] = index of the best.
int32_t nvh_launch_sample_final(const void* cand, int64_t* out, int64_t rows, int slices, hipStream_t st);
