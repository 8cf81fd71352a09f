// A prompt's tokens through the whole model, all tokens of a chunk at once.
//
// Semantics: fleet_prefill on tokens[0 .. n) at positions pos0 .. does what n
// calls of fleet_decode_step do without the lm_head (src/host/reference_decode.py:
// 210-302 per token and layer): the cache rows it writes and the last token's
// residual are what the steps leave. Norms, RoPE, routing and every projection are
// the same numbers by construction (each dot product exact and rounded once, to fp32,
// then bf16). Scores, softmax and the weighted sum of cache rows are fp64 as in the
// steps, but summed in another order (rounds of 128 positions here, chunks and
// batches there) before o_c is rounded to fp32. The two fp64 sums differ by some
// 1e-8 of an fp32 unit, so an o_c may round the other way, by one fp32 unit, and a
// head output whose bf16 rounding hangs on that unit would differ. No test has
// shown one (up to 1,100 tokens, every bit compared); nothing excludes it.
//
// Stepping reads every weight once per token (1.36 ms a step, 515 ms for 384
// tokens); here a weight is read once per chunk (384 tokens: 21.8 ms). The
// projections run as exact integer products of digits (digit_gemm.h); the
// attention's own products (q_c, scores, the weighted sum, W_UV), whose operands
// are fp32 or fp64, run on the fp64 matrix cores (v_mfma_f64_16x16x4).
//
// Operand layout of every fp64 MFMA below: lane l holds A[i = l % 16][k = l /
// 16] and B[k = l / 16][j = l % 16], and D[4 v + l / 16][l % 16] in register
// pair v. A sum over k may run in any order, so lane group q = l / 16 takes
// eight consecutive k of every 32 (one 16-byte load of bf16 feeds eight
// MFMAs), for both operands alike.
#include <cmath>

#include "attn_body.h"
#include "digit_gemm.h"
#include "expert_blocks.h"

namespace fleet_moe {
namespace pre {

using attn::kHeads;
using attn::kLora;
using attn::kNope;
using attn::kQDim;
using attn::kQkvRows;
using attn::kRope;
using attn::kRowElems;
using attn::kV;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kLanes;
constexpr int kChunkTokens = 528;       // tokens per chunk: h, partials and q of a chunk stay resident
constexpr int kQDimC = kLora + kRope;   // 576: q_c and q_pe of a head
constexpr int kSlots = kTopK + 1;

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mfma64(double a, double b, f64x4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Element e (0 .. 7) of a 16-byte bf16 chunk, widened.
__device__ __forceinline__ double widen(const u32x4& w, int e) {
    const uint32_t d = w[e >> 1];
    return (double)(e & 1 ? bf_hi(d) : bf_lo(d));
}

// Row i of a 16-row A tile under the permutation that gives lane group q the
// four consecutive rows 4 q .. 4 q + 3 of D (register pair v: row 4 q + v).
__device__ __forceinline__ int perm16(int i) { return 4 * (i & 3) + (i >> 2); }

struct Layout {
    size_t tab, ent, x, xn, xnf, qkv, q, oc, heads, ids, w, h, hs, part;
    size_t xd, headsd, hd, hsd;             // digit rows, 3 bytes a value
    size_t xm, headsm, hm, hsm;             // their exponents and error constants
    size_t total;
};

__host__ __device__ constexpr size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

__host__ constexpr Layout layout(int dense_inter) {
    const size_t T = kChunkTokens;
    const size_t hs = (size_t)(dense_inter > kSharedInter ? dense_inter : kSharedInter);
    Layout L{};
    L.tab = 0;
    L.ent = up256(sizeof(blocks::Table));
    L.x = L.ent + up256(T * kTopK * 4);
    L.xn = L.x + T * kHidden * 4;
    L.xnf = L.xn + T * kHidden * 2;
    L.qkv = L.xnf + T * kHidden * 4;
    L.q = L.qkv + up256(T * kQkvRows * 2);
    L.oc = L.q + T * kHeads * kQDimC * 4;
    L.heads = L.oc + T * kHeads * kLora * 4;
    L.ids = L.heads + T * kHeads * kV * 2;
    L.w = L.ids + up256(T * kTopK * 4);
    L.h = L.w + up256(T * kTopK * 4);
    L.hs = L.h + T * kTopK * kInter * 2;
    L.part = L.hs + up256(T * hs * 2);
    L.xd = L.part + T * kSlots * kHidden * 2;
    L.headsd = L.xd + T * kHidden * 3;
    L.hd = L.headsd + T * kHeads * kV * 3;
    L.hsd = L.hd + T * kTopK * kInter * 3;
    L.xm = L.hsd + up256(T * hs * 3);
    L.headsm = L.xm + up256(T * sizeof(digit::Meta));
    L.hm = L.headsm + up256(T * sizeof(digit::Meta));
    L.hsm = L.hm + up256(T * kTopK * sizeof(digit::Meta));
    L.total = L.hsm + up256(T * sizeof(digit::Meta));
    return L;
}
constexpr int kDenseInter = 10944;

// ---------------------------------------------------------------- norms

struct NormLds {
    double red[kWaves];
    uint32_t mx[kWaves];
    float sb[kWaves], rs[kWaves];
};

// A normed row's outputs: bf16, and its digits for the projections.
struct NormOut {
    uint16_t* xn;          // [T][H], or null (nothing follows)
    uint8_t* xd;           // [T][3 H]
    digit::Meta* xm;       // [T]
};

// RMSNorm of one 2048-vector held eight per thread (256 threads), the decode
// kernels' arithmetic; returns the eight bf16 results as a 16-byte chunk.
__device__ u32x4 norm_row(const float (&v)[8], const uint16_t* gamma, float eps, NormLds& S) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kLanes - 1);
    u32x4 g = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    if (gamma) {
        const uint2 a = ld_global_u2(gamma, 2 * tid), b = ld_global_u2(gamma, 2 * tid + 1);
        g = u32x4{a.x, a.y, b.x, b.y};
    }
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += (double)v[i] * v[i];
    ss = wave_sum64(ss);
    if (lane == 0) S.red[wave] = ss;
    __syncthreads();
    double ssq = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) ssq += S.red[w];
    const float var = (float)(ssq / (double)kHidden);
    const float inv = __fdiv_rn(1.0f, sqrt_rn(var + eps));
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = bf16r(bf16r(v[2 * i] * inv) * bf_lo(g[i]));
        const float b = bf16r(bf16r(v[2 * i + 1] * inv) * bf_hi(g[i]));
        o[i] = bf16_bits(a) | (bf16_bits(b) << 16);
    }
    return o;
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void widen8(const u32x4& c, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = bf_lo(c[i]);
        v[2 * i + 1] = bf_hi(c[i]);
    }
}

// Row t's normed chunk of this thread, and the row's digits.
__device__ void put_normed(const NormOut& O, int t, const u32x4& o, NormLds& S) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kLanes - 1);
    reinterpret_cast<u32x4*>(O.xn + (int64_t)t * kHidden)[tid] = o;
    const uint32_t w = digit::wave_umax(digit::absmax16(o));
    if (lane == 0) S.mx[wave] = w;
    __syncthreads();
    const uint32_t mx = max(max(S.mx[0], S.mx[1]), max(S.mx[2], S.mx[3]));
    int sx;
    const bool ok = digit::row_exponent(mx, sx);
    float sb0 = 0.f, res = 0.f;
    if (ok) digit::put_digits(O.xd + (int64_t)t * 3 * kHidden, tid, o, sx, sb0, res);
    sb0 = wave_sum(sb0);
    res = wave_sum(res);
    if (lane == 0) {
        S.sb[wave] = sb0;
        S.rs[wave] = res;
    }
    __syncthreads();
    if (tid == 0)
        O.xm[t] = digit::make_meta(mx, ok, sx, (S.sb[0] + S.sb[1]) + (S.sb[2] + S.sb[3]),
                                   (S.rs[0] + S.rs[1]) + (S.rs[2] + S.rs[3]));
}

// x = embed[token] (zeros and FLEET_MOE_ABORT_TOKEN outside the vocabulary,
// as fleet_embed), then layer 0's first norm. One workgroup per token.
__global__ __launch_bounds__(kThreads) void embed_norm_kernel(const uint16_t* embed,
                                                              const int32_t* tokens,
                                                              const uint16_t* gamma, float eps,
                                                              float* x, NormOut O,
                                                              uint32_t* status) {
    __shared__ NormLds S;
    const int t = blockIdx.x, tid = threadIdx.x;
    const int tok = tokens[t];
    u32x4 c = {0u, 0u, 0u, 0u};
    if (tok >= 0 && tok < attn::kVocab) {
        c = reinterpret_cast<const u32x4*>(embed + (int64_t)tok * kHidden)[tid];
    } else if (tid == 0) {
        __hip_atomic_fetch_or(status, FLEET_MOE_ABORT_TOKEN, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
    }
    float v[8];
    widen8(c, v);
    store8(x + (int64_t)t * kHidden + 8 * tid, v);
    put_normed(O, t, norm_row(v, gamma, eps, S), S);
}

// The normed row of x, also widened to fp32 for the router when xnf is not null.
__global__ __launch_bounds__(kThreads) void norm_kernel(const float* x, const uint16_t* gamma,
                                                        float eps, NormOut O, float* xnf) {
    __shared__ NormLds S;
    const int64_t at = (int64_t)blockIdx.x * kHidden;
    const int tid = threadIdx.x;
    float v[8];
    load8(x + at + 8 * tid, v);
    const u32x4 o = norm_row(v, gamma, eps, S);
    put_normed(O, blockIdx.x, o, S);
    if (xnf) {
        widen8(o, v);
        store8(xnf + at + 8 * tid, v);
    }
}

// The MoE layer's combine of one token, x = bf16(x + bf16(bf16(sum_k part_k) +
// shared)) with the routed terms in slot order, then the next layer's first
// norm (O.xn null after the last layer).
__global__ __launch_bounds__(kThreads) void combine_norm_kernel(const uint16_t* part, float* x,
                                                                const uint16_t* gamma, float eps,
                                                                NormOut O) {
    __shared__ NormLds S;
    const int t = blockIdx.x, tid = threadIdx.x;
    float v[8], y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    load8(x + (int64_t)t * kHidden + 8 * tid, v);
    u32x4 c[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        c[s] = reinterpret_cast<const u32x4*>(part + ((int64_t)t * kSlots + s) * kHidden)[tid];
    float p[8];
#pragma unroll
    for (int s = 0; s < kTopK; ++s) {
        widen8(c[s], p);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] += p[i];
    }
    widen8(c[kTopK], p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = bf16r(v[i] + bf16r(bf16r(y[i]) + p[i]));
    store8(x + (int64_t)t * kHidden + 8 * tid, v);
    if (O.xn) put_normed(O, t, norm_row(v, gamma, eps, S), S);
}

// ---------------------------------------------------------------- projections

// h = bf16(bf16(silu(g)) * u) of bf16 values
__device__ __forceinline__ float swiglu(float g, float u) { return bf16r(bf16r(silu_rn(g)) * u); }

__device__ __forceinline__ uint32_t pack2(float a, float b) {
    return bf16_bits(a) | (bf16_bits(b) << 16);
}

// A GEMM's token operand: bf16 rows of K values, their digits and exponents.
struct Rows {
    const uint16_t* x;
    const uint8_t* d;
    const digit::Meta* m;
};

// One workgroup: bf16 of its rows from `row0` of W x the tokens row(0 .. m - 1) of
// X. Returns the first of this wave's 16 rows, or -1 where another wave of the
// row tile holds the result. Waves past n_rows repeat the last rows.
template <int K, int NT, int KS, int NW, class Row>
__device__ __forceinline__ int product(const uint16_t* W, int row0, int n_rows, const Rows& X,
                                       int m, Row&& row,
                                       typename digit::Shape<NT, KS, NW>::Lds& L, float (&y)[NT][4]) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = threadIdx.x & 15, first = row0 + 16 * (wave / KS);
    const uint16_t* w = W + (int64_t)min(first, n_rows - 16) * K;
    digit::Acc<NT> acc;
    digit::gemm<K, NT, KS, NW>(w, [&](int i) { return X.d + (int64_t)row(min(i, m - 1)) * 3 * K; }, L,
                           acc);
    if (wave % KS != 0 || first >= n_rows) return -1;
    digit::Meta meta[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) meta[n] = X.m[row(min(16 * n + j, m - 1))];
    digit::finish<K, NT>(acc, meta, m, w, [&](int i) { return X.x + (int64_t)row(i) * K; }, y);
    return first;
}

enum Epi { kEpiBf16, kEpiResidual, kEpiSwiglu };

// Rows x tokens of a plain projection: out[t][row] = bf16 (kEpiBf16, pitch
// n_rows), x[t][row] = bf16(x + bf16(d)) (kEpiResidual, in place on fp32 x),
// or the SwiGLU of row pairs (kEpiSwiglu, pitch n_rows / 2). Grid (row tiles,
// token blocks of 16 NT); n_rows is a multiple of 16.
template <int K, int NT, int KS, int EPI>
__global__ __launch_bounds__(512) void proj_kernel(const uint16_t* W, int n_rows, Rows X, int T,
                                                   uint16_t* out, float* x) {
    using Sh = digit::Shape<NT, KS, 8>;
    __shared__ typename Sh::Lds L;
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    const int t0 = Sh::kTok * blockIdx.y, m = min(Sh::kTok, T - t0);
    float y[NT][4];
    const int row0 = product<K, NT, KS, 8>(W, Sh::kRows * blockIdx.x, n_rows, X, m,
                                        [&](int k) { return t0 + k; }, L, y);
    if (row0 < 0) return;
    const int row = row0 + 4 * q;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        if (16 * n + i >= m) continue;
        const int t = t0 + 16 * n + i;
        if constexpr (EPI == kEpiSwiglu) {
            *reinterpret_cast<uint32_t*>(out + (int64_t)t * (n_rows / 2) + row / 2) =
                pack2(swiglu(y[n][0], y[n][1]), swiglu(y[n][2], y[n][3]));
        } else if constexpr (EPI == kEpiResidual) {
            float4* p = reinterpret_cast<float4*>(x + (int64_t)t * n_rows + row);
            const float4 a = *p;
            *p = make_float4(bf16r(a.x + y[n][0]), bf16r(a.y + y[n][1]), bf16r(a.z + y[n][2]),
                             bf16r(a.w + y[n][3]));
        } else {
            *reinterpret_cast<uint2*>(out + (int64_t)t * n_rows + row) =
                make_uint2(pack2(y[n][0], y[n][1]), pack2(y[n][2], y[n][3]));
        }
    }
}

// ---------------------------------------------------------------- attention

// Per token: the cache row (kv_a_layernorm of c, RoPE of k_pe) and q_pe.
struct RopeLds {
    float v[kQkvRows];
    double red[kWaves];
};
__device__ void rope_cache(int t, const uint16_t* qkv, const uint16_t* gamma, float eps,
                           const float* cos, const float* sin, int pos0, uint16_t* cache, float* q,
                           RopeLds& S) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kLanes - 1);
    float* v = S.v;
    const int64_t pos = pos0 + t;
    const uint16_t* src = qkv + (int64_t)t * kQkvRows;
    for (int k = tid; k < kQkvRows / 2; k += kThreads) {
        const uint32_t w = reinterpret_cast<const uint32_t*>(src)[k];
        v[2 * k] = bf_lo(w);
        v[2 * k + 1] = bf_hi(w);
    }
    __syncthreads();
    uint16_t* row = cache + pos * kRowElems;
    const float c0 = v[kQDim + tid], c1 = v[kQDim + kThreads + tid];
    const double ss = wave_sum64((double)c0 * c0 + (double)c1 * c1);
    if (lane == 0) S.red[wave] = ss;
    __syncthreads();
    double ssq = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) ssq += S.red[w];
    const float inv = __fdiv_rn(1.0f, sqrt_rn((float)(ssq / (double)kLora) + eps));
    const float g0 = gamma ? bf_lo(gamma[tid]) : 1.f, g1 = gamma ? bf_lo(gamma[kThreads + tid]) : 1.f;
    row[tid] = (uint16_t)bf16_bits(bf16r(bf16r(c0 * inv) * g0));
    row[kThreads + tid] = (uint16_t)bf16_bits(bf16r(bf16r(c1 * inv) * g1));
    const float cs = cos[pos * kRope + lane], sn = sin[pos * kRope + lane];
    if (wave == 0) row[kLora + lane] = (uint16_t)bf16_bits(attn::rope_one(v + kQDim + kLora, cs, sn, lane));
#pragma unroll
    for (int k = 0; k < kHeads / kWaves; ++k) {
        const int h = wave + kWaves * k;
        q[((int64_t)t * kHeads + h) * kQDimC + kLora + lane] =
            attn::rope_one(v + h * (kNope + kRope) + kNope, cs, sn, lane);
    }
}

// q_c = W_UK^T q_nope, exact, rounded once to fp32. A wave: 64 columns of one
// head x 16 tokens; lane group q sums k = 32 q .. 32 q + 31, an 8-byte load of
// row k gives one A element of four column tiles (column 4 i + e of tile e).
// A workgroup: half of one head's columns for token block `block`. Bound by a
// wave's chain of MFMAs (64 cycles each), so a wave has 128 of them and all its
// weights in flight (8 / 384 tokens, with the launch of rope_cache: 16.0 / 27.1 us
// with 128 columns a wave, now 8.3 / 21.4).
__device__ void qc_block(int block, int h, int half, const uint16_t* qkv, const uint16_t* kv_b,
                         int T, float* q_out) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    const int t = 16 * block + i, col = kLora / 2 * half + 64 * wave;
    const uint16_t* wk = kv_b + ((int64_t)h * attn::kKvbRowsPerHead + 32 * q) * kLora + col;
    uint2 a[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) a[k] = ld_global_u2(wk + k * kLora, i);
    const uint16_t* xq = qkv + (int64_t)min(t, T - 1) * kQkvRows + h * (kNope + kRope) + 32 * q;
    u32x4 b[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) b[m] = reinterpret_cast<const u32x4*>(xq)[m];
    __builtin_amdgcn_sched_barrier(0);
    f64x4 acc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 32; ++k) {
        const double x = widen(b[k / 8], k % 8);
        acc[0] = mfma64((double)bf_lo(a[k].x), x, acc[0]);
        acc[1] = mfma64((double)bf_hi(a[k].x), x, acc[1]);
        acc[2] = mfma64((double)bf_lo(a[k].y), x, acc[2]);
        acc[3] = mfma64((double)bf_hi(a[k].y), x, acc[3]);
    }
    if (t >= T) return;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        *reinterpret_cast<float4*>(q_out + ((int64_t)t * kHeads + h) * kQDimC + col + 4 * (4 * v + q)) =
            make_float4((float)acc[0][v], (float)acc[1][v], (float)acc[2][v], (float)acc[3][v]);
}

// Both read the projection only, so they share a launch (rope_cache alone is
// the 5 us of an empty one): workgroups of q_c first, then one per token.
__global__ __launch_bounds__(kThreads, 2) void qc_rope_kernel(const uint16_t* qkv, const uint16_t* kv_b,
                                                           const uint16_t* gamma, float eps,
                                                           const float* cos, const float* sin, int T,
                                                           int pos0, uint16_t* cache, float* q) {
    __shared__ RopeLds S;
    const int n_qc = (T + 15) / 16 * 2 * kHeads, b = blockIdx.x;
    if (b < n_qc) qc_block(b / (2 * kHeads), b % kHeads, b / kHeads % 2, qkv, kv_b, T, q);
    else rope_cache(b - n_qc, qkv, gamma, eps, cos, sin, pos0, cache, q, S);
}

constexpr int kCus = 256;
constexpr int kMlaWaves = 8;
constexpr int kMlaPos = 16 * kMlaWaves;         // positions per round
constexpr int kMlaCols = kLora / kMlaWaves;     // columns of c per wave: 64
struct MlaLds {
    alignas(16) float q[kHeads][kQDimC + 4];
    double p[kHeads][kMlaPos + 2];
    double mx[kMlaWaves][kHeads];
    double ls[kMlaWaves][kHeads];
};

__device__ __forceinline__ double row_max64(double v) {
    v = fmax(v, dpp64<0xB1>(v));
    v = fmax(v, dpp64<0x4E>(v));
    v = fmax(v, dpp64<0x141>(v));
    return fmax(v, dpp64<0x140>(v));
}
__device__ __forceinline__ double row_sum64(double v) {
    v += dpp64<0xB1>(v);
    v += dpp64<0x4E>(v);
    v += dpp64<0x141>(v);
    return v + dpp64<0x140>(v);
}

// One token's 16 heads against cache rows 0 .. pos, all fp64 (the heads share
// the cached rows, so they are the 16 rows of A). Per 128 positions: wave w
// takes the scores of positions 16 w .. 16 w + 15 (144 MFMAs), the waves
// agree on the heads' running maxima, then wave w adds the positions'
// exp(s - m) c into columns 64 w .. 64 w + 63 (128 MFMAs; an 8-byte load of
// row k gives one B element of four column tiles, column 4 j + e of tile e).
// Tokens run from the last (the longest) to the first up to 256. A token is a serial
// chain of rounds, and up to a few hundred tokens leave matrix cores free: eight
// waves to a token instead of four halve its rounds (384 tokens: 99 -> 88 us).
// Past one token per CU, the workgroups that start second are the shortest and
// join CUs that hold middling ones; the longest have theirs alone (88 -> 76; 528
// tokens of a prompt 29.9 -> 29.0 ms).
__global__ __launch_bounds__(64 * kMlaWaves, 2) void mla_kernel(const float* q,
                                                                const uint16_t* cache, int pos0,
                                                                double scale, float* oc) {
    __shared__ MlaLds S;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & (kLanes - 1), i = lane & 15, g = lane >> 4;
    const int T = (int)gridDim.x, b = blockIdx.x;
    const int t = T > kCus && b < kCus ? T - kCus + b : T - 1 - b, n_pos = pos0 + t + 1;
    const float4* qs = reinterpret_cast<const float4*>(q + (int64_t)t * kHeads * kQDimC);
    for (int k = tid; k < kHeads * kQDimC / 4; k += 64 * kMlaWaves) {
        const int h = k / (kQDimC / 4), c = k - h * (kQDimC / 4);
        *reinterpret_cast<float4*>(&S.q[h][4 * c]) = qs[k];
    }
    double m[4], l[4];
    f64x4 o[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) { m[v] = -INFINITY; l[v] = 0.0; }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f64x4{0.0, 0.0, 0.0, 0.0};
    __syncthreads();
    for (int base = 0; base < n_pos; base += kMlaPos) {
        const int pos = base + 16 * wave + i;
        f64x4 s = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (base + 16 * wave < n_pos) {
            const u32x4* row = reinterpret_cast<const u32x4*>(
                cache + (int64_t)min(pos, n_pos - 1) * kRowElems) + g;
            f64x4 a4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) a4[e] = f64x4{0.0, 0.0, 0.0, 0.0};
            u32x4 b = ld_global(row);
#pragma unroll 3
            for (int k = 0; k < kQDimC / 32; ++k) {
                const u32x4 nb = ld_global(row + (k + 1 < kQDimC / 32 ? 4 * (k + 1) : 0));
                float qa[8];
                load8(&S.q[i][32 * k + 8 * g], qa);
#pragma unroll
                for (int e = 0; e < 8; ++e) a4[e & 3] = mfma64((double)qa[e], widen(b, e), a4[e & 3]);
                b = nb;
            }
#pragma unroll
            for (int v = 0; v < 4; ++v)
                s[v] = pos < n_pos ? ((a4[0][v] + a4[1][v]) + (a4[2][v] + a4[3][v])) * scale : -INFINITY;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double mv = row_max64(s[v]);
            if (i == 0) S.mx[wave][4 * v + g] = mv;
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double mn = m[v];
#pragma unroll
            for (int w = 0; w < kMlaWaves; ++w) mn = fmax(mn, S.mx[w][4 * v + g]);
            const double f = exp(m[v] - mn), p = exp(s[v] - mn);
            m[v] = mn;
            l[v] = fma(l[v], f, p);
            S.p[4 * v + g][16 * wave + i] = p;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e][v] *= f;
        }
        __syncthreads();
        const int ks = min(kMlaPos / 4, (n_pos - base + 3) >> 2);
        const uint16_t* col = cache + kMlaCols * wave;
        uint2 b = ld_global_u2(col + (int64_t)min(base + g, n_pos - 1) * kRowElems, i);
        for (int k = 0; k < ks; ++k) {
            const uint2 nb =
                ld_global_u2(col + (int64_t)min(base + 4 * (k + 1) + g, n_pos - 1) * kRowElems, i);
            const double a = S.p[i][4 * k + g];
            o[0] = mfma64(a, (double)bf_lo(b.x), o[0]);
            o[1] = mfma64(a, (double)bf_hi(b.x), o[1]);
            o[2] = mfma64(a, (double)bf_lo(b.y), o[2]);
            o[3] = mfma64(a, (double)bf_hi(b.y), o[3]);
            b = nb;
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const double s = row_sum64(l[v]);
        if (i == 0) S.ls[wave][4 * v + g] = s;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int h = 4 * v + g;
        double Ls = 0.0;
#pragma unroll
        for (int w = 0; w < kMlaWaves; ++w) Ls += S.ls[w][h];
        *reinterpret_cast<float4*>(oc + ((int64_t)t * kHeads + h) * kLora + kMlaCols * wave + 4 * i) =
            make_float4((float)(o[0][v] / Ls), (float)(o[1][v] / Ls), (float)(o[2][v] / Ls),
                        (float)(o[3][v] / Ls));
    }
}

// Head outputs bf16(W_UV o_c), exact. Grid (token blocks of 16, heads, quarters
// of the 128 rows), two waves per 16 rows, each with half of K: bound by the
// wave's chain of MFMAs (64 of 64 cycles each), all of whose operands are in
// flight at once (8 / 64 / 384 tokens: 12.4 / 12.9 / 20.1 us with two K halves
// in one wave and a few loads in flight, now 6.0 / 6.8 / 22.2).
__global__ __launch_bounds__(kThreads) void uv_kernel(const float* oc, const uint16_t* kv_b, int T,
                                                      uint16_t* heads) {
    __shared__ double part[2][4][kLanes];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    const int h = blockIdx.y, row0 = 32 * blockIdx.z + 16 * (wave & 1), half = wave >> 1;
    const int t = 16 * blockIdx.x + i;
    constexpr int kN = kLora / 64;          // 32-K loads per wave
    const u32x4* wp = reinterpret_cast<const u32x4*>(
        kv_b + ((int64_t)h * attn::kKvbRowsPerHead + kNope + row0 + perm16(i)) * kLora +
        kLora / 2 * half) + q;
    const float* xp = oc + ((int64_t)min(t, T - 1) * kHeads + h) * kLora + kLora / 2 * half + 8 * q;
    u32x4 a[kN];
    float x[kN][8];
#pragma unroll
    for (int s = 0; s < kN; ++s) {
        a[s] = ld_global(wp + 4 * s);
        load8(xp + 32 * s, x[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < kN; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = mfma64(widen(a[s], e), (double)x[s][e], acc);
    if (half == 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v) part[wave & 1][v][lane] = acc[v];
    }
    __syncthreads();
    if (half == 1 || t >= T) return;
    float d[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) d[v] = (float)(acc[v] + part[wave][v][lane]);
    *reinterpret_cast<uint2*>(heads + ((int64_t)t * kHeads + h) * kV + row0 + 4 * q) =
        make_uint2(pack2(d[0], d[1]), pack2(d[2], d[3]));
}

// ---------------------------------------------------------------- experts

// The sorted entries and blocks of a chunk's tokens, one workgroup. (Ids are
// clamped: logits that are not numbers can leave one outside the table. The order of
// an expert's entries does not matter: each entry's results are its own.)
__global__ __launch_bounds__(1024) void table_kernel(const int32_t* ids, int n, int tok,
                                                     blocks::Table* tab, int32_t* ent) {
    blocks::build<(kChunkTokens * kTopK + 1023) / 1024>(ids, n, tok, tab, ent);
}

struct ExpertParams {
    const uint16_t* experts;
    int64_t stride;
    const uint16_t* shared;
    const blocks::Table* tab;
    const int32_t* ent;
    const float* weights;
    Rows xn;                // [T][H]
    Rows hr;                // [T * 6][1408], in sorted order
    Rows hsr;               // [T][2816]
    uint16_t* h;            // hr's and hsr's bf16 rows, written by gate / up
    uint16_t* hs;
    uint16_t* part;         // [T][7][H]
    int T;
    int shared_wgs;         // workgroups of the shared expert's tiles, then those of routed ones
};

template <int NT, int KS, int NW>
__device__ __forceinline__ void gate_up_tile(const ExpertParams& P, const uint16_t* W, int tile,
                                             bool shared, int first, int m, void* lds) {
    using Sh = digit::Shape<NT, KS, NW>;
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    float y[NT][4];
    const int pitch = shared ? kSharedInter : kInter;
    const int row0 = product<kHidden, NT, KS, NW>(
        W, Sh::kRows * tile, 2 * pitch, P.xn, m,
        [&](int k) { return shared ? first + k : P.ent[first + k] / kTopK; },
        *static_cast<typename Sh::Lds*>(lds), y);
    if (row0 < 0) return;
    uint16_t* out = shared ? P.hs : P.h;
#pragma unroll
    for (int n = 0; n < NT; ++n)
        if (16 * n + i < m)
            *reinterpret_cast<uint32_t*>(out + (int64_t)(first + 16 * n + i) * pitch +
                                         (row0 + 4 * q) / 2) =
                pack2(swiglu(y[n][0], y[n][1]), swiglu(y[n][2], y[n][3]));
}

// gate / up and SwiGLU of every routed entry and of the shared expert, in
// blocks of at most 16 NTM tokens.
template <int NTM, int KS, int NW>
__global__ __launch_bounds__(64 * NW, NTM == 1 ? 3 : 2) void gate_up_kernel(ExpertParams P) {
    using Sh = digit::Shape<NTM, KS, NW>;
    __shared__ typename Sh::Lds L;
    int e = 0, tile = 0, first = 0, m = 0;
    const uint16_t* W;
    const bool shared = (int)blockIdx.x < P.shared_wgs;
    if (!shared) {
        if (!blocks::of(P.tab, (int)blockIdx.x - P.shared_wgs, Sh::kTok, 2 * kInter / Sh::kRows, e,
                        tile, first, m))
            return;
        W = P.experts + (int64_t)e * P.stride;
    } else {
        constexpr int kTiles = 2 * kSharedInter / Sh::kRows;
        const int b = blockIdx.x;
        tile = b % kTiles;
        first = Sh::kTok * (b / kTiles);
        m = min(Sh::kTok, P.T - first);
        W = P.shared;
    }
    if constexpr (NTM > 1) {
        if (m <= 16) return gate_up_tile<1, KS, NW>(P, W, tile, shared, first, m, &L);
        if (m <= 32) return gate_up_tile<2, KS, NW>(P, W, tile, shared, first, m, &L);
    }
    gate_up_tile<NTM, KS, NW>(P, W, tile, shared, first, m, &L);
}

template <int K, int NT, int KS, int NW>
__device__ __forceinline__ void down_tile(const ExpertParams& P, const uint16_t* W, int tile,
                                          int first, int m, void* lds) {
    using Sh = digit::Shape<NT, KS, NW>;
    constexpr bool shared = K == kSharedInter;
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    float y[NT][4];
    const int row0 = product<K, NT, KS, NW>(W, Sh::kRows * tile, kHidden, shared ? P.hsr : P.hr, m,
                                        [&](int k) { return first + k; },
                                        *static_cast<typename Sh::Lds*>(lds), y);
    if (row0 < 0) return;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        if (16 * n + i >= m) continue;
        const int j = first + 16 * n + i;
        int64_t slot;
        float w = 1.f;
        if (shared) {
            slot = (int64_t)j * kSlots + kTopK;
        } else {
            const int en = P.ent[j], t = en / kTopK;
            slot = (int64_t)t * kSlots + (en - t * kTopK);
            w = P.weights[en];
        }
        *reinterpret_cast<uint2*>(P.part + slot * kHidden + row0 + 4 * q) =
            make_uint2(pack2(w * y[n][0], w * y[n][1]), pack2(w * y[n][2], w * y[n][3]));
    }
}

template <int K, int NTM, int KS, int NW>
__device__ __forceinline__ void down_block(const ExpertParams& P, const uint16_t* W, int tile,
                                           int first, int m, void* lds) {
    if constexpr (NTM > 1) {
        if (m <= 16) return down_tile<K, 1, KS, NW>(P, W, tile, first, m, lds);
        if (m <= 32) return down_tile<K, 2, KS, NW>(P, W, tile, first, m, lds);
    }
    down_tile<K, NTM, KS, NW>(P, W, tile, first, m, lds);
}

// down and the routing weight of every routed entry, down of the shared expert.
template <int NTM, int KS, int NW>
__global__ __launch_bounds__(64 * NW, NTM == 1 ? 3 : 2) void down_kernel(ExpertParams P) {
    using Sh = digit::Shape<NTM, KS, NW>;
    __shared__ typename Sh::Lds L;
    constexpr int kTiles = kHidden / Sh::kRows;
    int e = 0, tile = 0, first = 0, m = 0;
    if ((int)blockIdx.x >= P.shared_wgs) {
        if (!blocks::of(P.tab, (int)blockIdx.x - P.shared_wgs, Sh::kTok, kTiles, e, tile, first, m))
            return;
        down_block<kInter, NTM, KS, NW>(P, P.experts + (int64_t)e * P.stride +
                                           (int64_t)2 * kInter * kHidden,
                                    tile, first, m, &L);
        return;
    }
    const int b = blockIdx.x;
    tile = b % kTiles;
    first = Sh::kTok * (b / kTiles);
    m = min(Sh::kTok, P.T - first);
    down_block<kSharedInter, NTM, KS, NW>(P, P.shared + (int64_t)2 * kSharedInter * kHidden, tile,
                                      first, m, &L);
}

// The two expert launches and the digits between them; `n` entries. The shared
// expert's workgroups come first: its blocks are full and its down rows twice as
// long, and started last they ran alone at the end of a launch (prompts of 4 / 8 /
// 64 / 384 tokens: 4.99 / 5.88 / 9.45 / 22.8 ms with the routed ones first, 4.64 /
// 5.39 / 8.95 / 22.5 so).
template <int NTM, int KG, int KD, int NW>
static void launch_experts(ExpertParams P, int n, uint8_t* hd, digit::Meta* hm, uint8_t* hsd,
                           digit::Meta* hsm, hipStream_t s) {
    constexpr int kTok = 16 * NTM;
    const int bx = blocks::most(n, kTok), sb = (P.T + kTok - 1) / kTok;
    constexpr int kGRows = digit::Shape<NTM, KG, NW>::kRows;
    constexpr int kDRows = digit::Shape<NTM, KD, NW>::kRows;
    P.shared_wgs = sb * (2 * kSharedInter / kGRows);
    hipLaunchKernelGGL((gate_up_kernel<NTM, KG, NW>),
                       dim3(P.shared_wgs + bx * (2 * kInter / kGRows)),
                       dim3(64 * NW), 0, s, P);
    hipLaunchKernelGGL((digit::digits2_kernel<kInter, kSharedInter>),
                       dim3((n + 3) / 4 + (P.T + 3) / 4), dim3(256), 0, s,
                       digit::Operand{P.h, n, hd, hm}, digit::Operand{P.hs, P.T, hsd, hsm});
    P.shared_wgs = sb * (kHidden / kDRows);
    hipLaunchKernelGGL((down_kernel<NTM, KD, NW>), dim3(P.shared_wgs + bx * (kHidden / kDRows)),
                       dim3(64 * NW), 0, s, P);
}

// The last token's residual, for the lm_head.
__global__ __launch_bounds__(kThreads) void copy_row_kernel(const float* x, float* out) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    out[k] = x[k];
}

template <int K, int NT, int KS, int EPI>
static void launch_proj_as(const uint16_t* W, int n_rows, const Rows& X, int T, uint16_t* out,
                           float* x, hipStream_t s) {
    using Sh = digit::Shape<NT, KS, 8>;
    hipLaunchKernelGGL((proj_kernel<K, NT, KS, EPI>),
                       dim3((n_rows + Sh::kRows - 1) / Sh::kRows, (T + Sh::kTok - 1) / Sh::kTok),
                       dim3(512), 0, s, W, n_rows, X, T, out, x);
}

// A projection over T tokens. Few tokens leave few workgroups, so four waves
// share a row tile's K (16 KB of weights each instead of 64: at 8 tokens qkv
// 33 -> 13 us, o_proj 29 -> 13); many give the CUs enough to do without. With
// 33 to 64 tokens, 2 waves suit the wide ones (qkv 25 -> 20 us at 64), 4 the
// 2048 rows of o_proj and down (14 against 18).
template <int K, int EPI>
static void launch_proj(const uint16_t* W, int n_rows, const Rows& X, int T, uint16_t* out,
                        float* x, hipStream_t s) {
    if (T <= 32 || (T <= 64 && n_rows <= kHidden))
        launch_proj_as<K, 1, 4, EPI>(W, n_rows, X, T, out, x, s);
    else if (T <= 64) launch_proj_as<K, 1, 2, EPI>(W, n_rows, X, T, out, x, s);
    else if (T <= 256 || K > kHidden) launch_proj_as<K, 2, 2, EPI>(W, n_rows, X, T, out, x, s);
    else launch_proj_as<K, 3, 1, EPI>(W, n_rows, X, T, out, x, s);
}

template <int K>
static void launch_digits(const uint16_t* x, int rows, uint8_t* d, digit::Meta* m, hipStream_t s) {
    hipLaunchKernelGGL((digit::digits_kernel<K>), dim3((rows + 3) / 4), dim3(256), 0, s, x, rows, d,
                       m);
}

}  // namespace pre
}  // namespace fleet_moe

using namespace fleet_moe;

int fleet_moe_check_dims(const fleet_moe_dims* d);
int fleet_moe_check_device(int min_cus);

static bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

extern "C" size_t fleet_prefill_workspace_bytes(const fleet_moe_dims* dims) {
    if (!dims || fleet_moe_check_dims(dims) != 0) return 0;
    return pre::layout(pre::kDenseInter).total;
}

extern "C" int fleet_prefill(const fleet_step_model* model, const fleet_step_layer* layers,
                             const int32_t* tokens, int32_t n_tokens, int32_t pos0, float* x_out,
                             uint32_t* status, void* workspace, size_t workspace_bytes,
                             const fleet_moe_dims* dims, hipStream_t stream) {
    using namespace pre;
    if (!model || !layers || !dims) return FLEET_MOE_ERR_ARG;
    if (int e = fleet_moe_check_dims(dims)) return e;
    if (model->n_layers < 1 || model->n_layers > FLEET_STEP_MAX_LAYERS || !model->embed ||
        !model->rope_cos || !model->rope_sin || model->max_pos < 1 ||
        model->max_pos > attn::kMaxPos || !tokens || !x_out || !status || !workspace ||
        n_tokens < 1 || pos0 < 0 || n_tokens > model->max_pos - pos0)
        return FLEET_MOE_ERR_ARG;
    if (!aligned(model->embed, 16) || !aligned(model->rope_cos, 4) ||
        !aligned(model->rope_sin, 4) || !aligned(tokens, 4) || !aligned(x_out, 4) ||
        !aligned(status, 4) || !aligned(workspace, 256))
        return FLEET_MOE_ERR_ARG;
    for (int i = 0; i < model->n_layers; ++i) {
        const fleet_step_layer& l = layers[i];
        if (!l.attn.qkv || !l.attn.kv_b || !l.attn.o_proj || !l.cache ||
            (!l.dense && (!l.moe.router || !l.moe.experts || !l.moe.shared)))
            return FLEET_MOE_ERR_ARG;
        if (!aligned(l.attn.norm_in, 8) || !aligned(l.attn.qkv, 16) ||
            !aligned(l.attn.kv_a_norm, 2) || !aligned(l.attn.kv_b, 16) ||
            !aligned(l.attn.o_proj, 16) || !aligned(l.cache, 16) || !aligned(l.moe.norm, 8) ||
            !aligned(l.dense, 16) || !aligned(l.moe.router, 16) || !aligned(l.moe.experts, 16) ||
            !aligned(l.moe.shared, 16))
            return FLEET_MOE_ERR_ARG;
        if (!l.dense && (l.moe.expert_stride < kExpertStride || l.moe.expert_stride % kChunk != 0))
            return FLEET_MOE_ERR_DIMS;
    }
    const Layout L = layout(kDenseInter);
    if (workspace_bytes < L.total) return FLEET_MOE_ERR_WORKSPACE;
    if (int e = fleet_moe_check_device(1)) return e;
    char* ws = static_cast<char*>(workspace);
    blocks::Table* tab = reinterpret_cast<blocks::Table*>(ws + L.tab);
    int32_t* ent = reinterpret_cast<int32_t*>(ws + L.ent);
    float* x = reinterpret_cast<float*>(ws + L.x);
    uint16_t* xn = reinterpret_cast<uint16_t*>(ws + L.xn);
    float* xnf = reinterpret_cast<float*>(ws + L.xnf);
    uint16_t* qkv = reinterpret_cast<uint16_t*>(ws + L.qkv);
    float* q = reinterpret_cast<float*>(ws + L.q);
    float* oc = reinterpret_cast<float*>(ws + L.oc);
    uint16_t* heads = reinterpret_cast<uint16_t*>(ws + L.heads);
    int32_t* ids = reinterpret_cast<int32_t*>(ws + L.ids);
    float* wts = reinterpret_cast<float*>(ws + L.w);
    uint16_t* h = reinterpret_cast<uint16_t*>(ws + L.h);
    uint16_t* hs = reinterpret_cast<uint16_t*>(ws + L.hs);
    uint16_t* part = reinterpret_cast<uint16_t*>(ws + L.part);
    auto bytes = [&](size_t o) { return reinterpret_cast<uint8_t*>(ws + o); };
    auto metas = [&](size_t o) { return reinterpret_cast<digit::Meta*>(ws + o); };
    const NormOut norm_out{xn, bytes(L.xd), metas(L.xm)}, no_out{nullptr, nullptr, nullptr};
    const Rows xr{xn, bytes(L.xd), metas(L.xm)}, headsr{heads, bytes(L.headsd), metas(L.headsm)},
        hr{h, bytes(L.hd), metas(L.hm)}, hsr{hs, bytes(L.hsd), metas(L.hsm)};
    const double mm = 0.1 * 0.707 * std::log(40.0) + 1.0;
    const double scale = std::pow(192.0, -0.5) * mm * mm;
    const float eps = dims->rms_eps;
    const int n_chunks = (n_tokens + kChunkTokens - 1) / kChunkTokens;
    const int chunk = (n_tokens + n_chunks - 1) / n_chunks;       // even chunks
    for (int c0 = 0; c0 < n_tokens; c0 += chunk) {
        const int T = n_tokens - c0 < chunk ? n_tokens - c0 : chunk;
        const int p0 = pos0 + c0;
        // Tokens per block of an expert. Narrow blocks take few registers and
        // little LDS, so three workgroups of four waves share a CU; wide ones split
        // a weight once for more tokens. Blocks of 16 / 48, ms: 96 tokens 10.7 /
        // 11.4, 129: 12.9 / 13.2, 136: 13.3 / 13.3, 144: 13.7 / 13.5, 176: 14.9 / 14.5,
        // 256: 18.8 / 17.0, 384: 25.8 / 21.8, 528: 34.7 / 28.6. (Blocks of 32, two workgroups a
        // CU: 14.0 against 14.1 at 160 and nowhere better by more; 384: 22.6.)
        const int block = T <= 136 ? 16 : 48;
        hipLaunchKernelGGL(embed_norm_kernel, dim3(T), dim3(kThreads), 0, stream, model->embed,
                           tokens + c0, layers[0].attn.norm_in, eps, x, norm_out, status);
        for (int i = 0; i < model->n_layers; ++i) {
            const fleet_step_layer& l = layers[i];
            launch_proj<kHidden, kEpiBf16>(l.attn.qkv, kQkvRows, xr, T, qkv, nullptr, stream);
            hipLaunchKernelGGL(qc_rope_kernel, dim3((T + 15) / 16 * 2 * kHeads + T), dim3(kThreads), 0,
                               stream, qkv, l.attn.kv_b, l.attn.kv_a_norm, eps, model->rope_cos,
                               model->rope_sin, T, p0, l.cache, q);
            hipLaunchKernelGGL(mla_kernel, dim3(T), dim3(64 * kMlaWaves), 0, stream, q, l.cache, p0,
                               scale, oc);
            hipLaunchKernelGGL(uv_kernel, dim3((T + 15) / 16, kHeads, 4), dim3(kThreads), 0,
                               stream, oc, l.attn.kv_b, T, heads);
            launch_digits<kHeads * kV>(heads, T, bytes(L.headsd), metas(L.headsm), stream);
            launch_proj<kHeads * kV, kEpiResidual>(l.attn.o_proj, kHidden, headsr, T, nullptr, x,
                                                   stream);
            hipLaunchKernelGGL(norm_kernel, dim3(T), dim3(kThreads), 0, stream, x, l.moe.norm, eps,
                               norm_out, l.dense ? nullptr : xnf);
            const bool last = i == model->n_layers - 1;
            const uint16_t* next = last ? nullptr : layers[i + 1].attn.norm_in;
            if (l.dense) {
                launch_proj<kHidden, kEpiSwiglu>(l.dense, 2 * kDenseInter, xr, T, hs, nullptr,
                                                 stream);
                launch_digits<kDenseInter>(hs, T, bytes(L.hsd), metas(L.hsm), stream);
                launch_proj<kDenseInter, kEpiResidual>(
                    l.dense + (int64_t)2 * kDenseInter * kHidden, kHidden, hsr, T, nullptr, x,
                    stream);
                if (!last)
                    hipLaunchKernelGGL(norm_kernel, dim3(T), dim3(kThreads), 0, stream, x, next,
                                       eps, norm_out, nullptr);
                continue;
            }
            if (int e = fleet_moe_router_topk(l.moe.router, xnf, T, nullptr, nullptr, ids, wts,
                                              dims, stream))
                return e;
            hipLaunchKernelGGL(table_kernel, dim3(1), dim3(1024), 0, stream, ids, T * kTopK,
                               block, tab, ent);
            ExpertParams P{};
            P.experts = l.moe.experts;
            P.stride = l.moe.expert_stride;
            P.shared = l.moe.shared;
            P.tab = tab;
            P.ent = ent;
            P.weights = wts;
            P.xn = xr;
            P.hr = hr;
            P.hsr = hsr;
            P.h = h;
            P.hs = hs;
            P.part = part;
            P.T = T;
            auto experts = [&](auto launch) {
                launch(P, T * kTopK, bytes(L.hd), metas(L.hm), bytes(L.hsd), metas(L.hsm), stream);
            };
            if (block == 16) experts(launch_experts<1, 1, 1, 4>);
            else experts(launch_experts<3, 1, 1, 8>);
            hipLaunchKernelGGL(combine_norm_kernel, dim3(T), dim3(kThreads), 0, stream, part, x,
                               next, eps, last ? no_out : norm_out);
        }
        if (c0 + T == n_tokens)
            hipLaunchKernelGGL(copy_row_kernel, dim3(kHidden / kThreads), dim3(kThreads), 0, stream,
                               x + (int64_t)(T - 1) * kHidden, x_out);
    }
    return (int)hipGetLastError();
}
