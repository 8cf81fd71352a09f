// Exactly rounded dot products of bf16 rows on the int8 matrix cores.
//
// Both operands are brought to fixed point and split into three balanced
// base-256 digits; the products of digits and their sums are exact integers
// (v_mfma_i32_16x16x64_i8, 16 cycles for 16 x 16 x 64 products), so what is
// left out is known and small, and a result is accepted when that cannot
// change its bf16 rounding. The rest (a few in 10^5) is evaluated as the
// decode kernels do it, in fp64.
//
// Per 16 x 16 x 64 products the fp64 matrix cores take 1024 cycles and more
// (v_mfma_f64_16x16x4); here the eight digit products that matter take 128, and
// a step of 16 x 64 weights about 160 vector instructions, most of them the split
// into digits, whatever the number of tokens: 640 issue cycles, against 770 in which a
// SIMD's share of HBM delivers those weights.
// Counters, experts' gate / up launch (share of the SIMDs' cycles): 8 tokens: vector
// ALU 55 %, matrix cores 11 %, 4.6 TB/s, 1.7 waves per SIMD; 64: 72 / 14 %, 5.1 TB/s,
// 2.3 waves; 384 (blocks of 48): 50 / 19 % (5 % at once), 3.5 TB/s, 1.55 waves, which
// wait for memory or LDS 30 % of their time and to issue 29 %. The vector ALU comes
// first, and no pipe is full: with two waves a SIMD they overlap by chance only.
// The 27-layer prompt of 384 tokens went from 50.7 ms on the fp64 cores to 21.8,
// 64 tokens from 24.0 to 9.0.
//
//   x (a token's row, K values): ix = round(x 2^sx), |ix| < 2^22, digits b2 b1
//     b0 (ix = b2 2^16 + b1 2^8 + b0, |b2| <= 64, |b1|, |b0| <= 128), one
//     exponent per row. bf16 values within 2^-14 of the largest are exact.
//   w (a weight row, 256 values at a time): floor(w 2^sw30), |.| < 2^30, its top
//     three bytes as digits a2 a1 a0 and its low byte summed (`low`), one
//     exponent per row and 256 values.
// The sum over k of (a2 2^16 + a1 2^8 + a0)(b2 2^16 + b1 2^8 + b0) without a0 b0,
// in units of 2^-(sw30 - 8) 2^-sx, differs from the exact dot product by at most
//   128 sum |b0|                    (a0 b0)
//   + 2^22 sum |x 2^sx - ix|        (x's rounding; |w 2^(sw30-8)| < 2^22)
//   + 2^22 (sum low + 256) / 256    (w's low byte and the half unit below it)
// and sums of 256 digit products stay below 2^23. b0 and low are zero unless a
// value is below 2^-6 / 2^-14 of its row's largest.
#pragma once
#include "moe_common.h"

namespace fleet_moe {
namespace digit {

constexpr int kStepK = 64;            // K of one MFMA
constexpr int kStepBytes = 3 * kStepK;   // a token's digits of a step: b0, b1, b2 planes
constexpr int kSliceSteps = 4;        // steps that share a weight exponent
constexpr int kSliceBytes = kSliceSteps * kStepBytes;         // a token's digits of a slice
constexpr int kSliceChunks = kSliceBytes / 16;

// A wave's turn buffer: 16 rows x one step (128 bytes, spread over the banks).
constexpr int kTurnPitch = 2 * kStepK + 16;

// A workgroup's shape: 16 NT tokens x 16 W / KS weight rows, W waves, KS of them
// sharing 16 rows' K slices (slice s is wave s % KS's). LDS holds two rounds of KS
// slices of the tokens' digits; the pitch spreads 16 tokens' chunks over all
// banks.
template <int NT, int KS, int W>
struct Shape {
    static constexpr int kWaves = W;
    static constexpr int kThreads = W * kLanes;
    static constexpr int kTok = 16 * NT;
    static constexpr int kRows = 16 * kWaves / KS;
    static constexpr int kPitch = KS * kSliceBytes + 16;
    struct Lds {
        alignas(16) uint8_t turn[W][16 * kTurnPitch];
        union {
            alignas(16) uint8_t x[2][kTok * kPitch];
            struct {
                double s[kWaves][NT][4][kLanes];
                float e[kWaves][2][4][kLanes];
            } part;
        };
    };
};

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A token row's exponent and error constant: c = 128 sum |b0| + 2^22 sum |x 2^sx
// - ix| (+inf: not representable, every result of the row is evaluated in
// fp64; -1: the row is zero, every result is).
struct Meta {
    float c;
    int32_t sx;
};

__device__ __forceinline__ double pow2(int e) {     // 2^e, -1022 <= e <= 1023
    return __longlong_as_double((long long)(1023 + e) << 52);
}

// ---------------------------------------------------------------- digits of token rows

// Exponent of a row from its largest |bf16| bits. Rows below 2^-87 or holding
// an infinity or NaN are left to the fp64 path.
__device__ __forceinline__ bool row_exponent(uint32_t maxbits, int& sx) {
    const int e = (int)(maxbits >> 7);
    sx = 148 - e;                     // |x| < 2^(e - 126): |x 2^sx| < 2^22
    return e >= 40 && e < 255;
}

__device__ __forceinline__ uint32_t absmax16(const u32x4& c) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        m = max(m, c[i] & 0x7fffu);
        m = max(m, (c[i] >> 16) & 0x7fffu);
    }
    return m;
}

// Digits of eight consecutive values (chunk `chunk` of the row) into the
// row's planes; adds to sum |b0| and sum |x 2^sx - ix|.
__device__ __forceinline__ void put_digits(uint8_t* row, int chunk, const u32x4& c, int sx,
                                           float& sb0, float& res) {
    const float scale = __uint_as_float((uint32_t)(127 + sx) << 23);
    uint32_t p[3][2] = {{0u, 0u}, {0u, 0u}, {0u, 0u}};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t d = c[i >> 1];
        const float f = (i & 1 ? bf_hi(d) : bf_lo(d)) * scale;
        const float r = __builtin_rintf(f);
        res += fabsf(f - r);
        const uint32_t u = (uint32_t)((int)r + 0x8080) ^ 0x8080u;
        sb0 += fabsf((float)(int8_t)(u & 0xffu));
#pragma unroll
        for (int k = 0; k < 3; ++k) p[k][i >> 2] |= ((u >> (8 * k)) & 0xffu) << (8 * (i & 3));
    }
    // lane group q of a step takes chunks q and q + 4 (64 contiguous bytes of
    // a weight row per load), so their digits lie side by side
    uint8_t* at = row + (chunk >> 3) * kStepBytes + (chunk & 3) * 16 + (chunk & 4) * 2;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        *reinterpret_cast<uint2*>(at + k * kStepK) = make_uint2(p[k][0], p[k][1]);
}

__device__ __forceinline__ Meta make_meta(uint32_t maxbits, bool ok, int sx, float sb0, float res) {
    Meta m;
    // (1 + 2^-7 covers the roundings of the two fp32 sums)
    m.c = maxbits == 0 ? -1.f : ok ? (128.f * sb0 + 4194304.f * res) * 1.0078125f : INFINITY;
    m.sx = ok ? sx : 0;
    return m;
}

__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
#pragma unroll
    for (int m = 1; m < kLanes; m <<= 1) v = max(v, (uint32_t)__shfl_xor((int)v, m));
    return v;
}

// The digits of one row of K values, by one wave.
template <int K>
__device__ __forceinline__ void digits_of_row(const uint16_t* x, int row, uint8_t* out, Meta* meta) {
    constexpr int C = K / kChunk, G = (C + kLanes - 1) / kLanes;
    const int lane = threadIdx.x & (kLanes - 1);
    const u32x4* src = reinterpret_cast<const u32x4*>(x + (int64_t)row * K);
    u32x4 c[G];
    uint32_t mx = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int k = lane + kLanes * g;
        c[g] = k < C ? src[k] : u32x4{0u, 0u, 0u, 0u};
        mx = max(mx, absmax16(c[g]));
    }
    mx = wave_umax(mx);
    int sx;
    const bool ok = row_exponent(mx, sx);
    float sb0 = 0.f, res = 0.f;
    if (ok) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int k = lane + kLanes * g;
            if (k < C) put_digits(out + (int64_t)row * 3 * K, k, c[g], sx, sb0, res);
        }
    }
    sb0 = wave_sum(sb0);
    res = wave_sum(res);
    if (lane == 0) meta[row] = make_meta(mx, ok, sx, sb0, res);
}

// Four rows of K values per workgroup.
template <int K>
__global__ __launch_bounds__(256) void digits_kernel(const uint16_t* x, int rows, uint8_t* out,
                                                     Meta* meta) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row < rows) digits_of_row<K>(x, row, out, meta);
}

// Two operands in one launch, workgroups of a's rows first: either alone is
// the 5 us that an empty launch takes here.
struct Operand {
    const uint16_t* x;
    int rows;
    uint8_t* d;
    Meta* m;
};
template <int KA, int KB>
__global__ __launch_bounds__(256) void digits2_kernel(Operand a, Operand b) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), rows_a = (a.rows + 3) & ~3;
    if (row < a.rows) digits_of_row<KA>(a.x, row, a.d, a.m);
    else if (row >= rows_a && row - rows_a < b.rows) digits_of_row<KB>(b.x, row - rows_a, b.d, b.m);
}

// ---------------------------------------------------------------- the GEMM

__device__ __forceinline__ i32x4 mfma8(const u32x4& a, const u32x4& b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a),
                                                 __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t xor_rows_max(uint32_t v) {   // over lanes l ^ 16, l ^ 32
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max((uint32_t)a[0], (uint32_t)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max((uint32_t)b[0], (uint32_t)b[1]);
}
__device__ __forceinline__ uint32_t xor_rows_sum(uint32_t v) {
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = (uint32_t)a[0] + (uint32_t)a[1];
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (uint32_t)b[0] + (uint32_t)b[1];
}

// Digits of 16 weights (two 16-byte chunks) scaled by 2^sw30: a[0..2], and the
// sum of the low bytes. The bias that balances the digits rides in the fma: the
// sum is exact down to its unit bit (f has 8 significant bits, the bias two).
__device__ __forceinline__ void split_weights(const u32x4& lo, const u32x4& hi, float sc,
                                              u32x4 (&a)[3], uint32_t& low) {
    constexpr float kBias = 8421376.f;          // 0x808000
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t w0 = j < 2 ? lo[2 * j] : hi[2 * j - 4];
        const uint32_t w1 = j < 2 ? lo[2 * j + 1] : hi[2 * j - 3];
        const uint32_t i0 = (uint32_t)(int)fmaf(bf_lo(w0), sc, kBias);
        const uint32_t i1 = (uint32_t)(int)fmaf(bf_hi(w0), sc, kBias);
        const uint32_t i2 = (uint32_t)(int)fmaf(bf_lo(w1), sc, kBias);
        const uint32_t i3 = (uint32_t)(int)fmaf(bf_hi(w1), sc, kBias);
        const uint32_t t0 = __builtin_amdgcn_perm(i1, i0, 0x05010400u);
        const uint32_t t1 = __builtin_amdgcn_perm(i1, i0, 0x07030602u);
        const uint32_t u0 = __builtin_amdgcn_perm(i3, i2, 0x05010400u);
        const uint32_t u1 = __builtin_amdgcn_perm(i3, i2, 0x07030602u);
        low = __builtin_amdgcn_sad_u8(__builtin_amdgcn_perm(u0, t0, 0x05040100u), 0u, low);
        a[0][j] = __builtin_amdgcn_perm(u0, t0, 0x07060302u) ^ 0x80808080u;
        a[1][j] = __builtin_amdgcn_perm(u1, t1, 0x05040100u) ^ 0x80808080u;
        a[2][j] = __builtin_amdgcn_perm(u1, t1, 0x07060302u);
    }
}

// Sums of one wave's 16 weight rows x 16 NT tokens: lane (j = l % 16, q = l / 16)
// holds rows 4 q + v of tokens 16 n + j in units of 2^(8 - sx), and per row the
// error terms es (largest 2^-sw of the slices: times a token's constant it bounds
// the sum over the slices) and er (w's own).
template <int NT>
struct Acc {
    f64x4 s[NT];
    f32x4 es, er;      // er: an fp32 sum of positive terms; finish() covers its rounding
};

// Orders a wave's own LDS accesses.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Max over the eight lanes of each aligned group of 8.
__device__ __forceinline__ uint32_t max8_lanes(uint32_t v) {
    v = max(v, (uint32_t)FLEET_DPP((int)v, 0xB1));
    v = max(v, (uint32_t)FLEET_DPP((int)v, 0x4E));
    return max(v, (uint32_t)FLEET_DPP((int)v, 0x141));
}

// One slice: split the weights in `raw`, multiply with the tokens' digits at `x`
// in LDS, fold the levels into A. raw[s][h]: step s of row 8 h + l / 8, chunk
// l % 8 (a load takes eight rows' 128-byte lines; in the MFMA's layout 16 lanes
// would touch 16 lines); a step's rows change to the MFMA's layout through the
// wave's turn buffer, one step ahead of their use. hook(s) runs once step s's
// registers are used (to refill them). Straight-line code: steps past the row's
// end hold zero weights, whose digits are zero.
template <int NT, int kPitch, class Hook>
__device__ __forceinline__ void slice(u32x4 (&raw)[kSliceSteps][2], const uint8_t* x,
                                      uint8_t* turn, Acc<NT>& A, Hook&& hook) {
    const int lane = threadIdx.x & (kLanes - 1), j = lane & 15, q = lane >> 4;
    uint8_t* const tw = turn + (lane >> 3) * kTurnPitch + 16 * (lane & 7);
    const uint8_t* const tr = turn + j * kTurnPitch + 16 * q;
    u32x4 w[2];
    auto turn_step = [&](int s) {
        *reinterpret_cast<u32x4*>(tw) = raw[s][0];
        *reinterpret_cast<u32x4*>(tw + 8 * kTurnPitch) = raw[s][1];
        wave_sync();
        w[0] = *reinterpret_cast<const u32x4*>(tr);
        w[1] = *reinterpret_cast<const u32x4*>(tr + 64);
        wave_sync();
    };
    // the slice's largest |w| per row: of rows 8 h + l / 8, then of row j
    uint32_t mx;
    {
        u16x2 m2[2] = {{0, 0}, {0, 0}};
#pragma unroll
        for (int s = 0; s < kSliceSteps; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    m2[h] = __builtin_elementwise_max(
                        m2[h], __builtin_bit_cast(u16x2, raw[s][h][d] & 0x7fff7fffu));
        const uint32_t m0 = max8_lanes(max((uint32_t)m2[0][0], (uint32_t)m2[0][1]));
        const uint32_t m1 = max8_lanes(max((uint32_t)m2[1][0], (uint32_t)m2[1][1]));
        const int src = (j & 7) << 5;                     // lane 8 (j % 8)
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)m0);
        const uint32_t b1 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)m1);
        mx = j < 8 ? b0 : b1;
    }
    const int e = (int)(mx >> 7);
    const bool ok = e >= 40 && e < 255;
    // |w| < 2^(e - 126): sw30 = 156 - e
    const float sc = ok ? __uint_as_float((uint32_t)(283 - e) << 23) : 0.f;
    i32x4 l4[NT], l3[NT], l2[NT], l1[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) l4[n] = l3[n] = l2[n] = l1[n] = i32x4{0, 0, 0, 0};
    uint32_t low = 0;
    turn_step(0);
    const uint8_t* xp = x + j * kPitch + 16 * q;
#pragma unroll
    for (int s = 0; s < kSliceSteps; ++s) {
        // (the barrier keeps the scheduler from splitting every step's weights
        // first, which spills)
        __builtin_amdgcn_sched_barrier(0);
        u32x4 a[3];
        split_weights(w[0], w[1], sc, a, low);
        hook(s);
        if (s + 1 < kSliceSteps) turn_step(s + 1);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            u32x4 b[3];
#pragma unroll
            for (int d = 0; d < 3; ++d)
                b[d] = *reinterpret_cast<const u32x4*>(xp + 16 * n * kPitch + s * kStepBytes +
                                                      d * kStepK);
            l4[n] = mfma8(a[2], b[2], l4[n]);
            l3[n] = mfma8(a[2], b[1], l3[n]);
            l2[n] = mfma8(a[2], b[0], l2[n]);
            l1[n] = mfma8(a[1], b[0], l1[n]);
            l3[n] = mfma8(a[1], b[2], l3[n]);
            l2[n] = mfma8(a[1], b[1], l2[n]);
            l1[n] = mfma8(a[0], b[1], l1[n]);
            l2[n] = mfma8(a[0], b[2], l2[n]);
        }
    }
    // fold: rows 4 q + v have their exponents in lanes 4 q + v
    low = xor_rows_sum(low);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int src = (4 * q + v) << 2;
        const int mr = __builtin_amdgcn_ds_bpermute(src, (int)mx);
        const int lr = __builtin_amdgcn_ds_bpermute(src, (int)low);
        const int er = mr >> 7;
        const bool okr = er >= 40 && er < 255;
        const double u = okr ? pow2(er - 148) : 0.0;        // 2^-(sw30 - 8)
        const float uf = okr ? __uint_as_float((uint32_t)(er - 21) << 23) : 0.f;
        A.es[v] = fmaxf(A.es[v], mr != 0 && !okr ? INFINITY : uf);
        A.er[v] += uf * (16384.f * (float)(lr + kSliceSteps * kStepK));
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const double hi = (double)((l4[n][v] << 8) + l3[n][v]);
            const double f = fma(hi, 65536.0, fma((double)l2[n][v], 256.0, (double)l1[n][v]));
            A.s[n][v] = fma(f, u, A.s[n][v]);
        }
    }
}

// The whole workgroup: w is the first of its wave's 16 weight rows, xd(i) the digit
// row of the workgroup's i-th token (i < 16 NT). While a round of KS slices is
// multiplied, the next one's weights (registers) and digits (registers, then the
// other LDS buffer) are on their way: a wave's loads complete in order, so digits
// loaded straight from memory would wait for the weights issued before them. The KS
// waves of a row tile add their sums in LDS; A is complete in those with wave % KS
// == 0.
template <int K, int NT, int KS, int W, class XD>
__device__ __forceinline__ void gemm(const uint16_t* w, XD&& xd,
                                     typename Shape<NT, KS, W>::Lds& L, Acc<NT>& A) {
    using Sh = Shape<NT, KS, W>;
    constexpr int kThreads = Sh::kThreads;
    static_assert(K % kStepK == 0, "whole steps");
    constexpr int S = K / kStepK;                        // steps
    constexpr int R = KS * kSliceSteps;                  // steps per round
    constexpr int kTokChunks = KS * kSliceChunks;
    constexpr int kChunks = Sh::kTok * kTokChunks, P = (kChunks + kThreads - 1) / kThreads;
    const int tid = threadIdx.x, lane = tid & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ks = wave % KS;
    // the 16 rows as a buffer: a load past it returns zeros and reads nothing
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(w), 0, 16 * K * 2, 0x00020000);
    const int wat = (lane >> 3) * (K * 2) + 16 * (lane & 7);
    // this thread's digit chunks of a round: chunk c of token t; threads without
    // one write to the padding
    const uint8_t* src[P];
    int at[P], col[P];       // LDS offset, offset within a round
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int p = tid + kThreads * i, t = p / kTokChunks, c = p - t * kTokChunks;
        const bool have = p < kChunks;
        src[i] = xd(have ? t : 0);
        at[i] = have ? t * Sh::kPitch + 16 * c : Sh::kPitch - 16;
        col[i] = 16 * c;
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) A.s[n] = f64x4{0.0, 0.0, 0.0, 0.0};
    A.es = A.er = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 raw[kSliceSteps][2], xs[P];
    auto load = [&](int s, int step) {          // step s of the slice, `step` of the row
        const int off = wat + (step < S ? step * 2 * kStepK : 1 << 30);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            raw[s][h] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * h * K, 0, 2);
    };
    // (a chunk past the row's end is never used: any of the row's stands in)
    auto load_x = [&](int s0) {
#pragma unroll
        for (int i = 0; i < P; ++i)
            xs[i] = ld_global(reinterpret_cast<const u32x4*>(
                src[i] + min(s0 * kStepBytes + col[i], S * kStepBytes - 16)));
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < P; ++i) *reinterpret_cast<u32x4*>(L.x[buf] + at[i]) = xs[i];
    };
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    // Workgroups start at different rounds: rows are 4 KB (2816 B) apart, and all
    // waves walking them from the left would meet in the same memory channels.
    constexpr int kRounds = (S + R - 1) / R;
    int s0 = (int)(blockIdx.x / 8 % kRounds) * R;
    load_x(s0);
#pragma unroll
    for (int s = 0; s < kSliceSteps; ++s) load(s, s0 + ks * kSliceSteps + s);
    put(0);
    barrier();
#pragma unroll 1
    for (int it = 0; it < kRounds; ++it) {
        const bool more = it + 1 < kRounds;
        const int buf = it & 1, nx = s0 + R < S ? s0 + R : 0;
        load_x(nx);
        // (the digits go to LDS half way, which frees their registers; after the
        // last round nothing reads them)
        slice<NT, Sh::kPitch>(raw, L.x[buf] + ks * kSliceBytes, L.turn[wave], A, [&](int s) {
            if (s == kSliceSteps / 2) put(buf ^ 1);
            load(s, more ? nx + ks * kSliceSteps + s : S);
        });
        s0 = nx;
        barrier();
    }
    if constexpr (KS > 1) {
        if (ks != 0) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
#pragma unroll
                for (int n = 0; n < NT; ++n) L.part.s[wave][n][v][lane] = A.s[n][v];
                L.part.e[wave][0][v][lane] = A.es[v];
                L.part.e[wave][1][v][lane] = A.er[v];
            }
        }
        barrier();
        if (ks == 0) {
#pragma unroll
            for (int k = 1; k < KS; ++k)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
#pragma unroll
                    for (int n = 0; n < NT; ++n) A.s[n][v] += L.part.s[wave + k][n][v][lane];
                    A.es[v] = fmaxf(A.es[v], L.part.e[wave + k][0][v][lane]);
                    A.er[v] += L.part.e[wave + k][1][v][lane];
                }
        }
    }
}

// Exact dot of a weight row and a token row (whole wave, every lane returns it).
template <int K>
__device__ __forceinline__ float exact_dot(const uint16_t* w, const uint16_t* x) {
    constexpr int C = K / kChunk, G = (C + kLanes - 1) / kLanes;
    const int lane = threadIdx.x & (kLanes - 1);
    double a = 0.0;
#pragma unroll 4
    for (int g = 0; g < G; ++g) {
        const int c = lane + kLanes * g;
        const bool in = c < C;
        const u32x4 z = {0u, 0u, 0u, 0u};
        const u32x4 wv = in ? ld_global(reinterpret_cast<const u32x4*>(w) + c) : z;
        const u32x4 xv = in ? ld_global(reinterpret_cast<const u32x4*>(x) + c) : z;
        a = dot8_x(wv, xv, a);
    }
    return (float)wave_sum64(a);
}

// bf16 of every dot product: y[n][v] is row 4 q + v of token 16 n + j. wbase:
// row 0 of the wave's 16 rows; xrow(i): the bf16 row of the wave's i-th token
// (wave-uniform i); meta[n]: this lane's tokens; m: tokens in use.
template <int K, int NT, class XRow>
__device__ __forceinline__ void finish(const Acc<NT>& A, const Meta (&meta)[NT], int m,
                                       const uint16_t* wbase, XRow&& xrow, float (&y)[NT][4]) {
    const int lane = threadIdx.x & (kLanes - 1), j = lane & 15;
    uint32_t bad = 0;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const bool have = 16 * n + j < m;
        const double sc = pow2(-meta[n].sx);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double s = A.s[n][v] * (256.0 * sc);
            const double err = fma((double)meta[n].c, (double)A.es[v], (double)A.er[v]) *
                               (1.0009765625 * sc);
            const float lo = (float)(s - err), hi = (float)(s + err);
            const bool zero = meta[n].c < 0.f && __builtin_isfinite(A.es[v]);
            y[n][v] = zero ? 0.f : bf16r(lo);
            const bool ok = zero || (bf16_bits(lo) == bf16_bits(hi) && __builtin_isfinite(lo) &&
                                     __builtin_isfinite(hi));
            bad |= have && !ok ? 1u << (4 * n + v) : 0u;
        }
    }
    for (uint64_t any = __ballot(bad != 0); any; any = __ballot(bad != 0)) {
        const int l = (int)__builtin_ctzll(any);
        const int k = __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)bad, l));
        const int n = k >> 2, v = k & 3;
        const float r = bf16r(exact_dot<K>(wbase + (int64_t)(4 * (l >> 4) + v) * K,
                                           xrow(16 * n + (l & 15))));
        if (lane == l) {
            bad &= ~(1u << k);
#pragma unroll
            for (int nn = 0; nn < NT; ++nn)
#pragma unroll
                for (int vv = 0; vv < 4; ++vv) y[nn][vv] = 4 * nn + vv == k ? r : y[nn][vv];
        }
    }
}

}  // namespace digit
}  // namespace fleet_moe
