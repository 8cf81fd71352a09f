// C-ABI plumbing shared by the entry points, and the standalone router.
//
// fleet_moe_router_topk runs the router GEMV and the greedy top-k for any
// number of tokens: one workgroup per token, fp64 accumulation of the exact
// bf16 x bf16 products (so the logits are the correctly rounded fp32 values and
// the routing is reproducible bit for bit), then softmax + top-k on wave 0 with
// ties to the lowest index.
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <vector>

#include "attn_body.h"

namespace fleet_moe {

int check_dims_impl(const fleet_moe_dims* d) {
    if (!d) return FLEET_MOE_ERR_ARG;
    if (d->hidden != kHidden || d->moe_inter != kInter || d->n_routed != kRouted ||
        d->n_shared != kShared || d->top_k != kTopK)
        return FLEET_MOE_ERR_DIMS;
    if (!(d->rms_eps > 0.f) || !(d->routed_scaling == d->routed_scaling))
        return FLEET_MOE_ERR_ARG;
    return 0;
}

namespace {
struct DeviceInfo {
    int checked = 0;
    int status = 0;
};
std::mutex g_mu;
std::vector<DeviceInfo> g_dev;
}  // namespace

// Per device, once: the code object is gfx950-only, and the kernels whose
// workgroups wait on each other launch one workgroup per CU over `min_cus` CUs.
int check_device_impl(int min_cus) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    std::lock_guard<std::mutex> lk(g_mu);
    if ((int)g_dev.size() <= dev) g_dev.resize(dev + 1);
    DeviceInfo& di = g_dev[dev];
    if (!di.checked) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, dev);
        if (e != hipSuccess) return (int)e;
        di.status = (strncmp(prop.gcnArchName, "gfx950", 6) == 0 &&
                     prop.multiProcessorCount >= min_cus)
                        ? 0
                        : FLEET_MOE_ERR_DEVICE;
        di.checked = 1;
    }
    return di.status;
}

namespace {
struct ResidentInfo {
    int dev;
    const void* fn;
    int status;
};
std::vector<ResidentInfo> g_resident;
}  // namespace

// Per device and kernel, once: the kernel's workgroups wait for each other's
// data, so all `grid` of them (one per CU, `threads` threads each) must be
// resident at the same time. That holds when the device has at least `grid`
// CUs and one workgroup fits on a CU with the kernel's registers and LDS;
// otherwise FLEET_MOE_ERR_DEVICE. (Work of other processes or streams holding
// CUs can still delay residency; the kernels' waits are bounded for that.)
int check_resident_impl(const void* fn, int threads, int grid) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (int st = check_device_impl(grid)) return st;
    std::lock_guard<std::mutex> lk(g_mu);
    for (const ResidentInfo& r : g_resident)
        if (r.dev == dev && r.fn == fn) return r.status;
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0);
    if (e != hipSuccess) return (int)e;
    const int st = per_cu >= 1 ? 0 : FLEET_MOE_ERR_DEVICE;
    g_resident.push_back(ResidentInfo{dev, fn, st});
    return st;
}

namespace router {

// 131,072 products of fp64 accumulation per token bound it (a product, a
// widening and an addition, ~17 cycles per 64 of them: 3.6 us on one CU), so
// the workgroup fills the CU: 16 waves, wave w rows 8 (w / 2) .. + 7, half w % 2
// of K, every load issued before the first product, and one reduction of eight
// sums per wave. (Four waves of 16 rows, a load and a reduction at a time: 9.2
// us for one token.) That workgroup is alone on its CU, also while one of its waves
// takes the softmax and the six picks. From four tokens to a CU on, four waves take
// a token instead and one token's picks run beside another's products (the whole
// call with 16 / 4 waves, us: 512 tokens 13.4 / 15.3, 900: 20.8 / 21.2, 1024: 21.2 /
// 21.3, 1536: 29.7 / 28.4, 8192: 144 / 122, 65,535: 1182 / 972).
constexpr int kThreads = 1024;
constexpr int kRowsPerWave = 8;
constexpr int kHalf = kHidden / 2;
constexpr int kManyThreads = 256;
constexpr int kManyRowsPerWave = 16;
constexpr int kManyTokens = 1024;

struct Params {
    const u32x4* router;
    const float* x;          // fp32[T][H]
    const float* bias;       // fp32[64] or null
    float* logits;           // fp32[T][64] or null
    int32_t* ids;            // int32[T][6]
    float* weights;          // fp32[T][6]
    uint16_t* xb;            // bf16 bits of x [T][H], or null
    float scaling;
};

// Eight fp32 values of a row, and their bf16 bits.
__device__ __forceinline__ void load_x8(const float* xt, int chunk, float (&v)[8]) {
    const float4* p = reinterpret_cast<const float4*>(xt) + 2 * chunk;
    const float4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ u32x4 bf16_x8(const float (&v)[8]) {
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = bf16_bits(v[2 * q]) | (bf16_bits(v[2 * q + 1]) << 16);
    return o;
}

__device__ __forceinline__ double dot8_xr(const u32x4& w, const float (&x)[8], double acc) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        acc += (double)(bf_lo(w[q]) * x[2 * q]);
        acc += (double)(bf_hi(w[q]) * x[2 * q + 1]);
    }
    return acc;
}

// Softmax and picks of token t from one logit per lane, by one wave.
__device__ __forceinline__ void pick(const Params& P, int t, float l, int* s_ids, float* s_w) {
    const int lane = threadIdx.x & (kLanes - 1);
    if (P.logits) P.logits[(int64_t)t * kRouted + lane] = l;
    wave_softmax_topk(l, kRouted, kTopK, P.scaling, s_ids, s_w, P.bias);
    // lanes < k read slots written by other lanes of this same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    if (lane < kTopK) {
        P.ids[(int64_t)t * kTopK + lane] = s_ids[lane];
        P.weights[(int64_t)t * kTopK + lane] = s_w[lane];
    }
}

__global__ __launch_bounds__(kThreads) void router_topk_kernel(Params P) {
    __shared__ double s_part[2][kRouted];
    __shared__ int s_ids[8];
    __shared__ float s_w[8];
    const int t = blockIdx.x;
    const int wave = threadIdx.x >> 6, half = wave & 1, row0 = kRowsPerWave * (wave >> 1);
    const int lane = threadIdx.x & (kLanes - 1);
    // lane: chunks lane and lane + 64 of its half
    const float* xt = P.x + (int64_t)t * kHidden + half * kHalf;
    float xr[2][8];
#pragma unroll
    for (int m = 0; m < 2; ++m) load_x8(xt, lane + kLanes * m, xr[m]);
    u32x4 w[kRowsPerWave][2];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
#pragma unroll
        for (int m = 0; m < 2; ++m)
            w[r][m] = P.router[(int64_t)(row0 + r) * kRowChunks + half * (kRowChunks / 2) + lane +
                               kLanes * m];
    if (P.xb && row0 == 0) {
        u32x4* o = reinterpret_cast<u32x4*>(P.xb + (int64_t)t * kHidden + half * kHalf);
#pragma unroll
        for (int m = 0; m < 2; ++m) o[lane + kLanes * m] = bf16_x8(xr[m]);
    }
    double acc[kRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        acc[r] = 0.0;
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[r] = dot8_xr(w[r][m], xr[m], acc[r]);
    }
    const double tot = attn::wave_msum64<kRowsPerWave>(acc);
    s_part[half][row0 + msum_index<kRowsPerWave>(lane)] = tot;   // lanes of an index agree
    __syncthreads();
    if (wave == 0) pick(P, t, (float)(s_part[0][lane] + s_part[1][lane]), s_ids, s_w);
}

__global__ __launch_bounds__(kManyThreads) void router_topk_many_kernel(Params P) {
    __shared__ float s_logit[kRouted];
    __shared__ int s_ids[8];
    __shared__ float s_w[8];
    const int t = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kLanes - 1);
    float xr[4][8];
#pragma unroll
    for (int m = 0; m < 4; ++m) load_x8(P.x + (int64_t)t * kHidden, lane + kLanes * m, xr[m]);
    if (P.xb) {
        u32x4* o = reinterpret_cast<u32x4*>(P.xb + (int64_t)t * kHidden) + lane;
#pragma unroll
        for (int m = 0; m < 4; ++m)
            if (m == wave) o[kLanes * m] = bf16_x8(xr[m]);
    }
    for (int r = wave * kManyRowsPerWave; r < (wave + 1) * kManyRowsPerWave; ++r) {
        const u32x4* row = P.router + (int64_t)r * kRowChunks;
        double acc = 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc = dot8_xr(row[lane + kLanes * m], xr[m], acc);
        acc = wave_sum64(acc);
        if (lane == 0) s_logit[r] = (float)acc;
    }
    __syncthreads();
    if (wave == 0) pick(P, t, s_logit[lane], s_ids, s_w);
}

}  // namespace router

namespace fold {

// x_out = bf16(x + bf16(p_0 + p_1 + ... + p_{n-1})), the partials added in
// fp32 in index order (one thread per hidden element; x may equal x_out).
constexpr int kThreads = 256;
__global__ __launch_bounds__(kThreads) void residual_fold_kernel(const float* x,
                                                                 const float* partials,
                                                                 int n_partials, float* x_out) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    float acc = partials[i];
    for (int p = 1; p < n_partials; ++p) acc += partials[(int64_t)p * kHidden + i];
    x_out[i] = bf16r(x[i] + bf16r(acc));
}

}  // namespace fold

namespace probe {

// Streaming read with the weight-load pattern of the MoE kernels: each wave
// reads 4 contiguous 1 KB wave-loads (16-byte non-temporal loads per lane)
// per step, grid-stride. The XOR of everything read is written only if it
// equals an improbable constant, so the loads cannot be dropped.
constexpr int kThreads = 256;
constexpr int kDepth = 4;
__global__ __launch_bounds__(kThreads) void stream_read_kernel(const u32x4* __restrict__ p,
                                                               size_t n16, uint32_t* sink) {
    const int lane = threadIdx.x & (kLanes - 1);
    const size_t wave = (blockIdx.x * (size_t)kThreads + threadIdx.x) / kLanes;
    const size_t nwaves = (gridDim.x * (size_t)kThreads) / kLanes;
    const size_t tile = (size_t)kDepth * kLanes;
    uint32_t acc = 0;
    for (size_t t = wave * tile; t < n16; t += nwaves * tile) {
        u32x4 v[kDepth];
#pragma unroll
        for (int d = 0; d < kDepth; ++d) v[d] = ld_stream(p + t + d * kLanes + lane);
#pragma unroll
        for (int d = 0; d < kDepth; ++d) acc ^= v[d].x ^ v[d].y ^ v[d].z ^ v[d].w;
    }
    if (acc == 0x9e3779b9u) sink[0] = acc;
}

}  // namespace probe
}  // namespace fleet_moe

using namespace fleet_moe;

int fleet_moe_check_dims(const fleet_moe_dims* d) { return check_dims_impl(d); }
int fleet_moe_check_device(int min_cus) { return check_device_impl(min_cus); }
int fleet_moe_check_resident(const void* fn, int threads, int grid) {
    return check_resident_impl(fn, threads, grid);
}

static bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

static int launch_router(const uint16_t* w_router, const float* x_norm, int32_t n_tokens,
                         const float* logit_bias, float* logits, int32_t* ids, float* weights,
                         uint16_t* x_bf16, const fleet_moe_dims* dims, hipStream_t stream) {
    if (int e = check_dims_impl(dims)) return e;
    if (!w_router || !x_norm || !ids || !weights || n_tokens < 1 || n_tokens > 65535)
        return FLEET_MOE_ERR_ARG;
    if (!aligned(w_router, 16) || !aligned(x_norm, 16) || !aligned(ids, 4) ||
        !aligned(weights, 4) || (logits && !aligned(logits, 4)) ||
        (logit_bias && !aligned(logit_bias, 4)) || (x_bf16 && !aligned(x_bf16, 16)))
        return FLEET_MOE_ERR_ARG;
    if (int e = check_device_impl(1)) return e;
    router::Params P;
    P.router = reinterpret_cast<const u32x4*>(w_router);
    P.x = x_norm;
    P.bias = logit_bias;
    P.logits = logits;
    P.ids = ids;
    P.weights = weights;
    P.xb = x_bf16;
    P.scaling = dims->routed_scaling;
    if (n_tokens < router::kManyTokens)
        hipLaunchKernelGGL(router::router_topk_kernel, dim3(n_tokens), dim3(router::kThreads), 0,
                           stream, P);
    else
        hipLaunchKernelGGL(router::router_topk_many_kernel, dim3(n_tokens),
                           dim3(router::kManyThreads), 0, stream, P);
    return (int)hipGetLastError();
}

extern "C" int fleet_moe_router_topk(const uint16_t* w_router, const float* x_norm,
                                     int32_t n_tokens, const float* logit_bias, float* logits,
                                     int32_t* ids, float* weights, const fleet_moe_dims* dims,
                                     hipStream_t stream) {
    return launch_router(w_router, x_norm, n_tokens, logit_bias, logits, ids, weights, nullptr, dims,
                         stream);
}

extern "C" int fleet_moe_router_topk_bf16(const uint16_t* w_router, const float* x_norm,
                                          int32_t n_tokens, const float* logit_bias,
                                          float* logits, int32_t* ids, float* weights,
                                          uint16_t* x_bf16, const fleet_moe_dims* dims,
                                          hipStream_t stream) {
    if (!x_bf16) return FLEET_MOE_ERR_ARG;
    return launch_router(w_router, x_norm, n_tokens, logit_bias, logits, ids, weights, x_bf16, dims,
                         stream);
}

extern "C" int fleet_moe_residual_fold(const float* x, const float* partials, int32_t n_partials,
                                       float* x_out, const fleet_moe_dims* dims,
                                       hipStream_t stream) {
    if (int e = check_dims_impl(dims)) return e;
    if (!x || !partials || !x_out || n_partials < 1 || n_partials > 64 || !aligned(x, 4) ||
        !aligned(partials, 4) || !aligned(x_out, 4))
        return FLEET_MOE_ERR_ARG;
    if (int e = check_device_impl(1)) return e;
    hipLaunchKernelGGL(fold::residual_fold_kernel, dim3(kHidden / fold::kThreads),
                       dim3(fold::kThreads), 0, stream, x, partials, n_partials, x_out);
    return (int)hipGetLastError();
}

extern "C" int fleet_moe_stream_read(const void* buf, size_t bytes, uint32_t* sink,
                                     hipStream_t stream) {
    if (!buf || !sink || !aligned(buf, 16) || !aligned(sink, 4) || bytes == 0 ||
        bytes % (16 * kLanes * probe::kDepth) != 0)
        return FLEET_MOE_ERR_ARG;
    if (int e = check_device_impl(1)) return e;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(probe::stream_read_kernel, dim3(2 * cus), dim3(probe::kThreads), 0, stream,
                       static_cast<const u32x4*>(buf), bytes / 16, sink);
    return (int)hipGetLastError();
}

extern "C" int fleet_moe_workspace_status(const void* workspace, uint32_t* status,
                                          hipStream_t stream) {
    if (!workspace || !status || !aligned(workspace, 256)) return FLEET_MOE_ERR_ARG;
    hipError_t e = hipMemcpyAsync(status, static_cast<const char*>(workspace) + 8,
                                  sizeof(uint32_t), hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess) return (int)e;
    return (int)hipStreamSynchronize(stream);
}

extern "C" const char* fleet_moe_error_string(int code) {
    switch (code) {
        case 0: return "success";
        case FLEET_MOE_ERR_DIMS: return "fleet_moe: unsupported model shape";
        case FLEET_MOE_ERR_ARG: return "fleet_moe: null, misaligned or out-of-range argument";
        case FLEET_MOE_ERR_WORKSPACE: return "fleet_moe: workspace too small";
        case FLEET_MOE_ERR_DEVICE:
            return "fleet_moe: device is not a gfx950 with enough CUs to hold one workgroup of "
                   "the kernel on each";
        case FLEET_MOE_ERR_CAPACITY:
            return "fleet_moe: more tokens than the static scratch of the no-allocation entry "
                   "point holds";
        case FLEET_MOE_ERR_CAPTURE:
            return "fleet_moe: the first no-allocation call on a device sets up its scratch and "
                   "must not be made under graph capture";
        default: return hipGetErrorString((hipError_t)code);
    }
}

extern "C" int fleet_moe_abi_version(void) { return 101; }
