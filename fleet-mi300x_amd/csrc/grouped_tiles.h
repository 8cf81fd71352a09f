// The grouped step's kernels for many tokens (launch_grouped draws the line):
// every unit -- the shared expert, each selected expert -- is cut into
// workgroups of 16 R W weight rows x up to 16 NT tokens, bf16 MFMA 16x16x32;
// experts with at most 8 tokens run the other plan's VALU items.
//
// HBM bound: 17.3 MB per selected expert and 34.6 MB for the shared one, at 31
// FLOP per byte and 256 tokens. A wave's weights go from HBM into registers (16
// R rows x 256 K, refilled for the next slice as they are used), so every weight
// byte is written to and read from LDS once, by its own wave, whatever the number
// of tokens; the token rows pass through LDS, two slices in turn, each read by
// the workgroup's four waves. Gate / up of 256 tokens streams 4.9 TB/s (65: 5.9):
// its waves wait for memory 80 % of their time, the matrix cores are busy 7 % and LDS
// 28 %, and 1.6 of the two waves a SIMD holds are there on average (the launch's end).
//
// Every sum is the other plan's, bit for bit (gemm): a token's result is the same
// in any block, at any place in the batch and from call to call. Walking K from
// eight different slices, which changes the sums with the workgroup, took
// 258 us where this takes 269 (256 tokens with the router; 128: 216 / 231; 65:
// 208 / 221). The other plan takes 474, 417 and 246.
//
// R = 2, NT = 4 holds 128 KB of weights in flight per CU. Other shapes, with K
// walked from any slice and the routed workgroups first (256 tokens 285 us): R =
// 1 and NT = 3: 335; NT = 2, R = 2: 292, but 332 against 272 under Zipf routing,
// whose popular experts fill blocks of 64. Persistent workgroups that carry the
// stream across tiles: 358. With one K step ahead (R = 1) in the down launch
// alone: 300. As it is now: chains taken slice by slice in turn 263 for 264 us; a
// VALU item's rows loaded during the one before 227 for 231 at 128 tokens and no
// gain at 256: not worth their lines.
//
// Launches: the tables (one workgroup), gate / up + SwiGLU, down + routing weight,
// combine; data crosses them as plain memory.
#pragma once

namespace fleet_moe {
namespace grouped {
namespace tiles {

constexpr int kSteps = 8;                     // MFMA steps (32 K) per slice
constexpr int kSliceK = 32 * kSteps;          // 256
constexpr int kPitch = kSliceK * 2 + 16;      // LDS bytes per token: 16 tokens' chunks hit 64 banks
using blocks::kXcds;

struct Table {
    blocks::Table b;
    int16_t ent[kMaxEntries];
};
static_assert(sizeof(Table) <= kTabBytes, "shares the place of the other plan's tables");

struct Params {
    const uint16_t* experts;
    const uint16_t* shared;
    int64_t stride;
    const float* weights;
    const uint16_t* x;
    const Table* tab;
    uint16_t* h;            // [T * 6][1408] in sorted order, then [T][2816]
    uint16_t* part;         // [T][7][H]: bf16(w bf16(d)) per slot, the shared expert's bf16(d)
    uint16_t* out;
    int T;
    int shared_wgs;         // workgroups of the shared expert's tiles, then those of routed ones
};

// One workgroup; ids outside [0, 64) are clamped and reported, as in the other
// plan. The entries of an expert come in no fixed order, which reaches no result:
// an entry's sums do not depend on its block or its place there.
__global__ __launch_bounds__(1024) void table_kernel(const int32_t* ids, int n, int tok, Header* hdr,
                                                     Table* tab) {
    const bool bad = blocks::build<2>(ids, n, tok, &tab->b, tab->ent);
    if (__ballot(bad) && (threadIdx.x & (kLanes - 1)) == 0) flag_abort(hdr, FLEET_MOE_ABORT_BAD_ID);
}
static_assert(kMaxEntries <= 2 * 1024, "two entries per thread");

// LDS of a workgroup: two slices of its tokens' rows, and per wave the turn buffer
// (two steps of 16 rows).
constexpr int kTurnPitch = 128 + 16;
template <int NT, int W>
struct Lds {
    alignas(16) uint8_t x[2][16 * NT * kPitch];
    alignas(16) uint8_t turn[W][16 * kTurnPitch];
};

// y[r][n][v] = row 16 r + 4 q + v of the wave's rows (from `w`) x token 16 n + l %
// 16; xrow(i): the row of `x` (bf16 [][K]) of the workgroup's i-th token.
// A weight load takes eight rows' 128-byte lines, eight lanes to a line. (In the
// MFMA's own layout, lane l = row l % 16, the four lanes of a row are 16 apart:
// every 16 lanes touch 16 lines, 64 bytes of each per load, and the stream stops
// at 4.9 TB/s.) Two such loads, 16 rows x two steps, change to the MFMA's layout
// through LDS.
// The sums are those of the other plan's MFMA items, bit for bit and whatever the
// block, the batch or the workgroup: one chain over the even slices, one over the
// odd, added; 2816 values as two halves of 1408, added. Which chain and which half
// come first is free (an addition's operands may change places), so workgroups
// start at different ones: rows are 4 KB (2816 B) apart, and all waves walking
// them from the left would meet in the same memory channels.
template <int K, int NT, int R, int W, class XRow>
__device__ __forceinline__ void gemm(const uint16_t* w, const uint16_t* x, XRow&& xrow,
                                     Lds<NT, W>& L, f32x4 (&y)[R][NT]) {
    constexpr int kChunks = K / kChunk;                  // 16-byte chunks per row
    constexpr int kTokChunks = kSliceK / kChunk;         // 32 per slice
    constexpr int P = 16 * NT * kTokChunks / (64 * W);
    constexpr int kHalves = K == kSharedInter ? 2 : 1, kHalfChunks = kChunks / kHalves;
    constexpr int kPer = (kHalfChunks / kTokChunks + 1) / 2;     // slices per chain
    constexpr int kChains = 2 * kHalves;
    static_assert(16 * NT * kTokChunks % (64 * W) == 0 && K % (64 * kHalves) == 0 &&
                      (2 * kPer - 1) * kTokChunks < kHalfChunks && kHalfChunks <= 2 * kPer * kTokChunks,
                  "whole chunks, whole lines, every slice holds some");
    const int tid = threadIdx.x, lane = tid & (kLanes - 1), j = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32x4* wp = reinterpret_cast<const u32x4*>(w) + (lane >> 3) * kChunks + (lane & 7);
    uint8_t* const turn = L.turn[wave];
    uint8_t* const tw = turn + (lane >> 3) * kTurnPitch + 16 * (lane & 7);
    const uint8_t* const tr = turn + j * kTurnPitch + 16 * q;
    uint32_t src[P];                                     // byte offsets from x: < 8 MB
    const int c = tid % kTokChunks;                      // 64 W is a multiple of 32
#pragma unroll
    for (int i = 0; i < P; ++i)
        src[i] = (uint32_t)(xrow((tid + 64 * W * i) / kTokChunks) * (2 * K) + 16 * c);
    const int dst = (tid / kTokChunks) * kPitch + 16 * c;
    constexpr int kDst = 64 * W / kTokChunks * kPitch;
    u32x4 raw[R][kSteps / 2][2], xs[P];
    // slice `i` of the chain taken ch-th: its first chunk and its chunks
    const int start = (int)(blockIdx.x / kXcds % kChains);
    struct Slice {
        int c0, n;
    };
    auto slice = [&](int ch, int i) {
        const int chain = ch ^ start, s = (2 * i + (chain & 1)) * kTokChunks;
        return Slice{(chain >> 1) * kHalfChunks + s, min(kTokChunks, kHalfChunks - s)};
    };
    auto load_w = [&](int p, Slice z) {                  // steps 2 p, 2 p + 1
        if (8 * p < z.n)                                 // uniform
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    raw[r][p][h] = ld_stream(wp + (16 * r + 8 * h) * kChunks + z.c0 + 8 * p);
    };
    auto load_x = [&](Slice z) {
        if (c < z.n)
#pragma unroll
            for (int i = 0; i < P; ++i) xs[i] = ld_global(reinterpret_cast<const u32x4*>(
                    reinterpret_cast<const uint8_t*>(x) + 16 * z.c0 + src[i]));
    };
    auto put = [&](int buf, Slice z) {
        if (c < z.n)
#pragma unroll
            for (int i = 0; i < P; ++i)
                *reinterpret_cast<u32x4*>(L.x[buf] + dst + i * kDst) = xs[i];
    };
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    Slice z = slice(0, 0);
    load_x(z);
#pragma unroll
    for (int p = 0; p < kSteps / 2; ++p) load_w(p, z);
    put(0, z);
    barrier();
    f32x4 lo[kHalves == 2 ? R : 1][kHalves == 2 ? NT : 1];      // the first half's sums
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < NT; ++n) y[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    int buf = 0;
#pragma unroll 1
    for (int ch = 0; ch < kChains; ++ch) {
        f32x4 t[R][NT];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < NT; ++n) t[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int i = 0; i < kPer; ++i, buf ^= 1) {
            const bool more = i + 1 < kPer || ch + 1 < kChains;
            const Slice nx = i + 1 < kPer ? slice(ch, i + 1) : slice(ch + 1, 0);
            if (more) load_x(nx);                        // uniform but for the tail's chunks
            const uint8_t* xp = L.x[buf] + j * kPitch + 16 * q;
#pragma unroll
            for (int p = 0; p < kSteps / 2; ++p) {
                if (8 * p < z.n) {                       // uniform
                    u32x4 a[R][2];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            *reinterpret_cast<u32x4*>(tw + 8 * h * kTurnPitch) = raw[r][p][h];
                        lds_wave_sync();
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            a[r][h] = *reinterpret_cast<const u32x4*>(tr + 64 * h);
                        lds_wave_sync();
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int n = 0; n < NT; ++n) {
                            const u32x4 b = *reinterpret_cast<const u32x4*>(xp + 16 * n * kPitch +
                                                                           64 * (2 * p + h));
#pragma unroll
                            for (int r = 0; r < R; ++r) t[r][n] = mfma16(a[r][h], b, t[r][n]);
                        }
                }
                if (p == kSteps / 4 && more) put(buf ^ 1, nx);
                if (more) load_w(p, nx);
            }
            z = nx;
            barrier();
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                if (ch % 2 == 0) {
                    if constexpr (kHalves == 2) lo[r][n] = y[r][n];
                    y[r][n] = t[r][n];
                } else {
                    y[r][n] += t[r][n];
                }
            }
    }
    if constexpr (kHalves == 2)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < NT; ++n) y[r][n] += lo[r][n];
}

// This workgroup's token block of a routed expert. few: the expert is a VALU unit.
// False past the last block.
__device__ __forceinline__ bool routed_block(const Params& P, int tok, int tiles, int& e, int& tile,
                                             int& first, int& m, bool& few) {
    if (!blocks::of(&P.tab->b, (int)blockIdx.x - P.shared_wgs, tok, tiles, e, tile, first, m))
        return false;
    few = is_v(P.tab->b.off[e + 1] - P.tab->b.off[e]);
    return true;
}

template <int NT, int R, int W>
__device__ __forceinline__ void g_tile(const Params& P, const uint16_t* wt, int tile, bool shared,
                                       int first, int m, void* lds) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    const int row0 = 16 * R * (W * tile + wave);
    f32x4 y[R][NT];
    gemm<kHidden, NT, R, W>(wt + (int64_t)row0 * kHidden, P.x, [&](int k) {
        const int j = first + min(k, m - 1);
        return shared ? j : P.tab->ent[j] / kTopK;
    }, *static_cast<Lds<NT, W>*>(lds), y);
    uint16_t* out = shared ? P.h + (int64_t)P.T * kTopK * kInter : P.h;
    const int pitch = shared ? kSharedInter : kInter;
#pragma unroll
    for (int n = 0; n < NT; ++n)
        if (16 * n + i < m)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const f32x4 d = y[r][n];
                *reinterpret_cast<uint32_t*>(out + (int64_t)(first + 16 * n + i) * pitch +
                                             (row0 + 16 * r + 4 * q) / 2) =
                    pack_bf16(bf16r(bf16r(silu_rn(bf16r(d[0]))) * bf16r(d[1])),
                              bf16r(bf16r(silu_rn(bf16r(d[2]))) * bf16r(d[3])));
            }
}

// Experts with at most 8 tokens: the other plan's VALU items (a wave each, one
// after the other), whose sums are another tree than the matrix cores'. Their
// tokens' rows sit in LDS, in front of the waves' reduction words.
constexpr int kFewRed = kVMax * kHidden * 2;
static_assert(kFewRed + 4 * kLanes * 4 <= (int)sizeof(Lds<4, 4>) && kInter <= kHidden, "rows fit");

template <int M, int ROWS, int W>
__device__ __forceinline__ void g_few(const Params& P, const uint16_t* wt, int tile, int first, int m,
                                      uint8_t* lds) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int k = tid; k < m * kRowChunks; k += 64 * W) {
        const int j = k / kRowChunks, c = k - j * kRowChunks;
        reinterpret_cast<u32x4*>(lds)[k] = ld_global(
            reinterpret_cast<const u32x4*>(P.x + (int64_t)(P.tab->ent[first + j] / kTopK) * kHidden) +
            c);
    }
    __syncthreads();
    float* const red = reinterpret_cast<float*>(lds + kFewRed) + kLanes * wave;
    const u32x4* rows = reinterpret_cast<const u32x4*>(wt) + (int64_t)ROWS * tile * kRowChunks;
    uint32_t* h = reinterpret_cast<uint32_t*>(P.h) + (int64_t)first * (kInter / 2) + ROWS / 4 * tile;
#pragma unroll 1
    for (int i = wave; i < ROWS / 4; i += W)
        g_pairs_v<M>(rows + 4 * i * kRowChunks, lds, m, red,
                     [&](int j, uint32_t word) { h[j * (kInter / 2) + i] = word; });
}

template <int M, int ROWS, int W>
__device__ __forceinline__ void d_few(const Params& P, const uint16_t* wt, int tile, int first, int m,
                                      uint8_t* lds) {
    constexpr int R = M <= 4 ? 8 : 4;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32x4* h = reinterpret_cast<const u32x4*>(P.h + (int64_t)first * kInter);
    for (int k = tid; k < m * kInterChunks; k += 64 * W)
        reinterpret_cast<u32x4*>(lds)[k] = ld_global(h + k);
    __syncthreads();
    float* const red = reinterpret_cast<float*>(lds + kFewRed) + kLanes * wave;
    const u32x4* rows = reinterpret_cast<const u32x4*>(wt) + (int64_t)ROWS * tile * kInterChunks;
#pragma unroll 1
    for (int i = wave; i < ROWS / R; i += W)
        d_rows_v<M, kInter, R>(rows + R * i * kInterChunks, lds, m, red,
                               [&](int j, int wp, float a, float b) {
            const int en = P.tab->ent[first + j], t = en / kTopK;
            const int64_t slot = (int64_t)t * kSlots + (en - t * kTopK);
            const float w = P.weights[en];
            *reinterpret_cast<uint32_t*>(P.part + slot * kHidden + ROWS * tile + R * i + 2 * wp) =
                pack_bf16(w * bf16r(a), w * bf16r(b));
        });
}

template <int NTM, int R, int W>
__global__ __launch_bounds__(64 * W, 2) void g_kernel(Params P) {
    __shared__ Lds<NTM, W> S;
    void* lds = &S;
    int e = 0, tile = 0, first = 0, m = 0;
    const uint16_t* wt;
    const bool shared = (int)blockIdx.x < P.shared_wgs;
    if (!shared) {
        bool few = false;
        if (!routed_block(P, 16 * NTM, 2 * kInter / (16 * R * W), e, tile, first, m, few)) return;
        wt = P.experts + (int64_t)e * P.stride;
        if (few) {
            uint8_t* const b = static_cast<uint8_t*>(lds);
            if (m == 1) return g_few<1, 16 * R * W, W>(P, wt, tile, first, m, b);
            if (m == 2) return g_few<2, 16 * R * W, W>(P, wt, tile, first, m, b);
            if (m <= 4) return g_few<4, 16 * R * W, W>(P, wt, tile, first, m, b);
            return g_few<8, 16 * R * W, W>(P, wt, tile, first, m, b);
        }
    } else {
        constexpr int kTiles = 2 * kSharedInter / (16 * R * W);
        const int b = blockIdx.x;
        tile = b % kTiles;
        first = 16 * NTM * (b / kTiles);
        m = min(16 * NTM, P.T - first);
        wt = P.shared;
    }
    if constexpr (NTM > 1)
        if (m <= 16) return g_tile<1, R, W>(P, wt, tile, shared, first, m, lds);
    if constexpr (NTM > 2)
        if (m <= 32) return g_tile<2, R, W>(P, wt, tile, shared, first, m, lds);
    if constexpr (NTM > 3)
        if (m <= 48) return g_tile<3, R, W>(P, wt, tile, shared, first, m, lds);
    g_tile<NTM, R, W>(P, wt, tile, shared, first, m, lds);
}

template <int K, int NT, int R, int W>
__device__ __forceinline__ void d_tile(const Params& P, const uint16_t* wt, int tile, int first,
                                       int m, void* lds) {
    constexpr bool shared = K == kSharedInter;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kLanes - 1), i = lane & 15, q = lane >> 4;
    const int row0 = 16 * R * (W * tile + wave);
    const uint16_t* h = shared ? P.h + (int64_t)P.T * kTopK * kInter : P.h;
    f32x4 y[R][NT];
    gemm<K, NT, R, W>(wt + (int64_t)row0 * K, h, [&](int k) { return first + min(k, m - 1); },
                      *static_cast<Lds<NT, W>*>(lds), y);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        if (16 * n + i >= m) continue;
        const int j = first + 16 * n + i;
        int64_t slot;
        float w = 1.f;
        if (shared) {
            slot = (int64_t)j * kSlots + kTopK;
        } else {
            const int en = P.tab->ent[j], t = en / kTopK;
            slot = (int64_t)t * kSlots + (en - t * kTopK);
            w = P.weights[en];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const f32x4 d = y[r][n];
            *reinterpret_cast<uint2*>(P.part + slot * kHidden + row0 + 16 * r + 4 * q) =
                make_uint2(pack_bf16(w * bf16r(d[0]), w * bf16r(d[1])),
                           pack_bf16(w * bf16r(d[2]), w * bf16r(d[3])));
        }
    }
}

template <int K, int NTM, int R, int W>
__device__ __forceinline__ void d_block(const Params& P, const uint16_t* wt, int tile, int first,
                                        int m, void* lds) {
    if constexpr (NTM > 1)
        if (m <= 16) return d_tile<K, 1, R, W>(P, wt, tile, first, m, lds);
    if constexpr (NTM > 2)
        if (m <= 32) return d_tile<K, 2, R, W>(P, wt, tile, first, m, lds);
    if constexpr (NTM > 3)
        if (m <= 48) return d_tile<K, 3, R, W>(P, wt, tile, first, m, lds);
    d_tile<K, NTM, R, W>(P, wt, tile, first, m, lds);
}

template <int NTM, int R, int W>
__global__ __launch_bounds__(64 * W, 2) void d_kernel(Params P) {
    __shared__ Lds<NTM, W> S;
    void* lds = &S;
    constexpr int kTiles = kHidden / (16 * R * W);
    int e = 0, tile = 0, first = 0, m = 0;
    if ((int)blockIdx.x >= P.shared_wgs) {
        bool few = false;
        if (!routed_block(P, 16 * NTM, kTiles, e, tile, first, m, few)) return;
        const uint16_t* wt = P.experts + (int64_t)e * P.stride + (int64_t)2 * kInter * kHidden;
        if (few) {
            uint8_t* const b = static_cast<uint8_t*>(lds);
            if (m == 1) return d_few<1, 16 * R * W, W>(P, wt, tile, first, m, b);
            if (m == 2) return d_few<2, 16 * R * W, W>(P, wt, tile, first, m, b);
            if (m <= 4) return d_few<4, 16 * R * W, W>(P, wt, tile, first, m, b);
            return d_few<8, 16 * R * W, W>(P, wt, tile, first, m, b);
        }
        d_block<kInter, NTM, R, W>(P, wt, tile, first, m, lds);
        return;
    }
    const int b = blockIdx.x;
    tile = b % kTiles;
    first = 16 * NTM * (b / kTiles);
    m = min(16 * NTM, P.T - first);
    d_block<kSharedInter, NTM, R, W>(P, P.shared + (int64_t)2 * kSharedInter * kHidden, tile, first, m,
                                  lds);
}

// out[t] = bf16(bf16(sum_k part[t][k]) + part[t][6]), k in slot order. A
// workgroup per token.
__global__ __launch_bounds__(256) void combine_kernel(const uint16_t* part, uint16_t* out) {
    const int t = blockIdx.x, tid = threadIdx.x;
    u32x4 c[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        c[s] = reinterpret_cast<const u32x4*>(part + ((int64_t)t * kSlots + s) * kHidden)[tid];
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int s = 0; s < kTopK; ++s) {
            a += bf_lo(c[s][i]);
            b += bf_hi(c[s][i]);
        }
        o[i] = pack_bf16(bf16r(bf16r(a) + bf_lo(c[kTopK][i])), bf16r(bf16r(b) + bf_hi(c[kTopK][i])));
    }
    uint32_t* p = reinterpret_cast<uint32_t*>(out + (int64_t)t * kHidden) + 4 * tid;
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = o[i];          // out is 4-byte aligned
}

template <int NTM, int R, int W>
static void launch(Params P, const int32_t* ids, Header* hdr, Table* tab, hipStream_t s) {
    constexpr int kTok = 16 * NTM;
    const int n = P.T * kTopK;
    hipLaunchKernelGGL(table_kernel, dim3(1), dim3(1024), 0, s, ids, n, kTok, hdr, tab);
    // The shared expert's workgroups come first: its blocks are full and its down
    // rows twice as long, and started last they ran alone at the end of a launch
    // (routing and experts of 84 / 128 / 256 tokens 240 / 244 / 286 us with the
    // routed ones first, now 217 / 216 / 258).
    const int bx = blocks::most(n, kTok), sb = (P.T + kTok - 1) / kTok;
    P.shared_wgs = sb * (2 * kSharedInter / (16 * R * W));
    hipLaunchKernelGGL((g_kernel<NTM, R, W>), dim3(P.shared_wgs + bx * (2 * kInter / (16 * R * W))),
                       dim3(64 * W), 0, s, P);
    P.shared_wgs = sb * (kHidden / (16 * R * W));
    hipLaunchKernelGGL((d_kernel<NTM, R, W>), dim3(P.shared_wgs + bx * (kHidden / (16 * R * W))),
                       dim3(64 * W), 0, s, P);
    hipLaunchKernelGGL(combine_kernel, dim3(P.T), dim3(256), 0, s, P.part, P.out);
}

}  // namespace tiles
}  // namespace grouped
}  // namespace fleet_moe
