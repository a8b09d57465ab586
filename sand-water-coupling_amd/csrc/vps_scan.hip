// vps_scan.hip -- the int32 array scan, its workspace, and the max reduction.
#include "vps_scan.h"

namespace vps {
namespace {

struct LoadI32 {
    static constexpr bool kWide = true;
    const int32_t* in;
    __device__ __forceinline__ int operator()(int64_t i) const { return in[i]; }
    __device__ __forceinline__ int4 four(int64_t i) const { return *(const int4*)(in + i); }
};
// clear != nullptr (the input itself, not aliased with out): the input is
// zeroed once read, ready for the next counting pass.
struct StoreI32 {
    static constexpr bool kWide = true;
    int32_t *out, *clear;
    __device__ __forceinline__ void four(int64_t i, int4 pre) const {
        *(int4*)(out + i) = pre;
        if (clear) *(int4*)(clear + i) = make_int4(0, 0, 0, 0);
    }
    __device__ __forceinline__ void operator()(int64_t i, int, int pre) const {
        out[i] = pre;
        if (clear) clear[i] = 0;
    }
};

__global__ void __launch_bounds__(256) k_max_f32(const float* in, int64_t n,
                                                 double* partials,
                                                 unsigned* counter,
                                                 double* out) {
    float m = -3.4e38f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * 256)
        m = fmaxf(m, in[i]);
    m = wave_max(m);
    __shared__ float sw[4];
    __shared__ bool last;
    if ((threadIdx.x & 63) == 0) sw[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = sw[0];
        for (int i = 1; i < 4; i++) t = fmaxf(t, sw[i]);
        partials[blockIdx.x] = t;
        __threadfence();
        last = atomicAdd(counter, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (last && threadIdx.x == 0) {
        __threadfence();
        double t = -3.4e38;
        for (unsigned i = 0; i < gridDim.x; i++) {
            const double v = __hip_atomic_load(&partials[i], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
            t = v > t ? v : t;
        }
        *out = t;
        *counter = 0;
    }
}

}  // namespace

int scan_workspace(vps_context* c, int64_t tiles, uint64_t** status, uint32_t** ticket,
                   uint32_t* epoch) {
    // the status words, then the ticket; zero words belong to no epoch
    if (c->scan_tmp.n < (size_t)tiles + 1 || c->scan_epoch >= (1u << 30) - 1) {
        VPS_TRY(dalloc(c, c->scan_tmp, (size_t)tiles + 1));
        VPS_HIP(c, hipMemsetAsync(c->scan_tmp.p, 0, c->scan_tmp.n * sizeof(uint64_t), c->stream));
        c->scan_epoch = 0;
    }
    *status = c->scan_tmp.p;
    *ticket = (uint32_t*)(c->scan_tmp.p + c->scan_tmp.n - 1);
    *epoch = ++c->scan_epoch;
    return VPS_OK;
}

int scan_exclusive_i32(vps_context* c, const int32_t* in, int32_t* out,
                       int64_t n, int32_t* total_dev, int32_t* clear_in) {
    if (n <= 0) {
        if (total_dev) VPS_HIP(c, hipMemsetAsync(total_dev, 0, 4, c->stream));
        return VPS_OK;
    }
    return scan_launch(c, LoadI32{in}, StoreI32{out, clear_in}, n, total_dev);
}

int reduce_max_f32(vps_context* c, const float* in, int64_t n, double* out) {
    int64_t nb = (n + 255) / 256;
    if (nb > 2048) nb = 2048;
    if (nb < 1) nb = 1;
    hipLaunchKernelGGL(k_max_f32, dim3((unsigned)nb), dim3(256), 0, c->stream,
                       in, n, c->partials.p, (unsigned*)&c->cg.p->counter[3],
                       out);
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

}  // namespace vps
