// Weighted residual of a field against data, and half its weighted square norm, in one pass.
//
// r = u - f (written over u) and loss = 1/2 sum_q w_q r_q^2.  HBM-bound: u, f and w read
// once, r written once, 32 B per point.  As a subtraction, a product and a dot product it read
// and wrote 64 B: with the transforms around it, on 32 768 hexes with 343 points (11.2e6
// points), a misfit and its gradient took 197 us so and take 149.  Each thread keeps its own
// FP64 sum, a workgroup leaves one partial sum, and a second kernel adds those in a fixed
// order, so the result does not vary from run to run.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ithaca_mf.h"

namespace imf {
namespace {

constexpr int kThreads = 256;

// Sum over the workgroup; complete in thread 0.
__device__ __forceinline__ double block_sum(double s)
{
    __shared__ double part[kThreads / 64];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < kThreads / 64; ++i) s += part[i];
    return s;
}

// V = double2 when all three arrays are aligned to it (n values in pairs, the odd last one
// by the last thread), else double.
template <typename V>
__global__ __launch_bounds__(kThreads) void residual_kernel(size_t n, double *__restrict__ u,
                                                            const double *__restrict__ f,
                                                            const double *__restrict__ w,
                                                            double *__restrict__ part)
{
    constexpr int W = sizeof(V) / sizeof(double);
    const size_t first = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const size_t step = (size_t)gridDim.x * kThreads;
    double s = 0.0;
    for (size_t i = first; i < n / W; i += step) {
        V x = ((const V *)u)[i];
        const V y = ((const V *)f)[i], wt = ((const V *)w)[i];
        if constexpr (W == 2) {
            x.x -= y.x;
            x.y -= y.y;
            s = fma(wt.x * x.x, x.x, s);
            s = fma(wt.y * x.y, x.y, s);
        } else {
            x -= y;
            s = fma(wt * x, x, s);
        }
        ((V *)u)[i] = x;
    }
    if (W == 2 && n % 2 && first == step - 1) {
        const double r = u[n - 1] - f[n - 1];
        u[n - 1] = r;
        s = fma(w[n - 1] * r, r, s);
    }
    s = block_sum(s);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(kThreads) void half_sum_kernel(int n, const double *__restrict__ part,
                                                            double *__restrict__ loss)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += kThreads) s += part[i];
    s = block_sum(s);
    if (threadIdx.x == 0) *loss = 0.5 * s;
}

}  // namespace
}  // namespace imf

extern "C" int imf_misfit_device(size_t n, double *d_u, const double *d_f, const double *d_w,
                                 double *d_part, double *d_loss, void *stream)
{
    if (!d_part || !d_loss || (n && (!d_u || !d_f || !d_w))) return IMF_ERR_ARG;
    using namespace imf;
    const hipStream_t s = (hipStream_t)stream;
    const bool pairs = (((uintptr_t)d_u | (uintptr_t)d_f | (uintptr_t)d_w) & 15) == 0;
    // enough workgroups to fill the chip several times over; a small field takes fewer
    const size_t want = (n / (pairs ? 2 : 1) + kThreads - 1) / kThreads;
    const int blocks = (int)std::min<size_t>(std::max<size_t>(want, 1), IMF_MISFIT_PARTS);
    if (pairs)
        residual_kernel<double2><<<blocks, kThreads, 0, s>>>(n, d_u, d_f, d_w, d_part);
    else
        residual_kernel<double><<<blocks, kThreads, 0, s>>>(n, d_u, d_f, d_w, d_part);
    if (hipGetLastError() != hipSuccess) return IMF_ERR_HIP;
    half_sum_kernel<<<1, kThreads, 0, s>>>(blocks, d_part, d_loss);
    return hipGetLastError() == hipSuccess ? IMF_OK : IMF_ERR_HIP;
}
