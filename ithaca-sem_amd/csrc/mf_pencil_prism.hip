// Pencil kernels of the prism operators (mf_pencil_kernels.hpp).
#include "mf_pencil_kernels.hpp"

namespace imf {

namespace {

__global__ void pencil_pack_kernel(long nElmt, int n0, int n1, int n2, const double *__restrict__ w0,
                                   const double *__restrict__ w1, const double *__restrict__ w2,
                                   const double *__restrict__ jac, const double *__restrict__ df,
                                   double *__restrict__ out)
{
    const int Q = n0 * n1 * n2;
    const long np = nElmt * Q, g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= np) return;
    const long e = g / Q;
    const int q = (int)(g - e * Q), i = q % n0, j = q / n0 % n1, k = q / (n0 * n1);
    const double jw = jac[g] * (w0[i] * w1[j] * w2[k]);
    double f[9];
#pragma unroll
    for (int d = 0; d < 9; ++d) f[d] = df[d * np + g];
    double *o = out + e * geo_stride(7l * Q, 8) + q;
    o[0] = jw;
    int n = 1;
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int y = x; y < 3; ++y)
            o[(long)Q * n++] = jw * fma(f[6 + x], f[6 + y], fma(f[3 + x], f[3 + y], f[x] * f[y]));
}

}  // namespace

hipError_t pencil_pack(long nElmt, const int *nq, const double *const *d_w, const double *jac,
                       const double *df, double *out, hipStream_t s)
{
    const long np = nElmt * nq[0] * nq[1] * nq[2];
    pencil_pack_kernel<<<(unsigned)((np + 255) / 256), 256, 0, s>>>(nElmt, nq[0], nq[1], nq[2], d_w[0],
                                                                    d_w[1], d_w[2], jac, df, out);
    return hipGetLastError();
}

PencilFn lookup_pencil_prism(int kind, int nm, int nq0) { return lookup_pencil<kPrism>(kind, nm, nq0); }

}  // namespace imf
