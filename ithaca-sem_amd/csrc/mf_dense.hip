// Operators of the collapsed shapes as dense products over the elements, on FP64 MFMA.
//
// The sum-factorised kernels of mf_{tri,tet,prism,pyr}.hip spend an LDS read of the table and
// one of the data on every multiply-add, and the collapsed directions' tables differ by mode,
// so neither can sit in a scalar register.  An element of these shapes has few modes
// (a tetrahedron of 5 modes per direction: 35 modes, 150 points), and at such sizes the
// element's whole matrix costs about as many multiply-adds as the factorised form:
//   BwdTrans, IProduct     M Q            (tetrahedron, 5 modes: 5 250; factorised 1 300)
//   Helmholtz, one set of  ng M^2         (8 575; factorised 9 650 with the pointwise part)
//   factors per element
// while every operand is used 16 times per load.  BwdTrans and IProduct then wait for HBM
// only; Helmholtz runs at the matrix cores' rate.
//
// One wave multiplies 16 elements by nt column tiles of 16: rows of A (the elements' inputs)
// come straight from global memory, two consecutive k per lane and 64 bytes per element and
// step; the matrix is staged in LDS chunk by chunk for the four waves of a workgroup, in the
// order the lanes read it (16 bytes per lane, no conflicts).  MFMA step c of a pair takes
// component c of both operands, so the order of k inside a step is the same for both.
#include "mf_dense.hpp"

#include <algorithm>

namespace imf {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double dv2 __attribute__((ext_vector_type(2)));
typedef dv2 dv2u __attribute__((aligned(8)));  // rows of A are 8-byte aligned

constexpr int KSTEP = 8;  // k per pair of MFMA steps

// steps per LDS chunk: four of one term (NT * 4 KB, at most 32 KB), one of several (NG * NT KB, at
// most 56 KB: Helmholtz tetrahedra of 8 modes, two workgroups per CU)
constexpr int chunk_steps(int ng) { return ng == 1 ? 4 : 1; }

// NT column tiles, NG geometry terms.
template <int NT, int NG>
__global__ __launch_bounds__(256) void dense_kernel(DenseArgs a)
{
    constexpr int CS = chunk_steps(NG), CH = CS * NG * NT * 64;  // 16-byte words per chunk
    constexpr int NL = (CH + 255) / 256;
    __shared__ dv2 tb[CH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kq = lane >> 4;
    const int K = a.sh.K, N = a.sh.N;
    const long e0 = ((long)blockIdx.x * 4 + wave) * 16;
    const long e = min(e0 + row, (long)a.nElmt - 1);  // rows past the end repeat the last
    const double *src = a.in + e * K + 2 * kq;
    const double *jp = a.jac + e * K + 2 * kq;        // kScalePoint only
    const double js = a.pre == kScaleElement ? a.jac[e] : 1.0;
    const dv2 *tab = reinterpret_cast<const dv2 *>(a.tab) +
                     (size_t)blockIdx.y * (a.sh.kp / KSTEP) * NG * NT * 64;

    double s[NG];
    if constexpr (NG > 1) {
        // lambda J, then J G^ab for (00, 01, 11) or (00, 01, 02, 11, 12, 22)
        constexpr int D = NG == 4 ? 2 : 3;
        double f[D][D];
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
            for (int d = 0; d < D; ++d) f[c][d] = a.df[(long)(c * D + d) * a.nElmt + e];
        const double J = a.jac[e];
        s[0] = a.lambda * J;
        int g = 1;
#pragma unroll
        for (int x = 0; x < D; ++x)
#pragma unroll
            for (int y = x; y < D; ++y) {
                double t = f[0][x] * f[0][y];
#pragma unroll
                for (int c = 1; c < D; ++c) t = fma(f[c][x], f[c][y], t);
                s[g++] = J * t;
            }
    }

    auto load_a = [&](int k, dv2 &v) {
        if (k + KSTEP <= K) {
            v = *reinterpret_cast<const dv2u *>(src + k);
            if (a.pre == kScalePoint) v *= *reinterpret_cast<const dv2u *>(jp + k);
        } else {
            const int k1 = k + 2 * kq;
            v.x = k1 < K ? src[k] : 0.0;
            v.y = k1 + 1 < K ? src[k + 1] : 0.0;
            if (a.pre == kScalePoint) {
                v.x *= k1 < K ? jp[k] : 0.0;
                v.y *= k1 + 1 < K ? jp[k + 1] : 0.0;
            }
        }
        if (NG == 1) v *= js;
    };

    d4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = d4{0, 0, 0, 0};
    dv2 nt_[NL], na[CS];
    auto fetch = [&](int k0) {
        const dv2 *p = tab + (size_t)(k0 / KSTEP) * NG * NT * 64;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            if (CH % 256 == 0 || i * 256 + (int)threadIdx.x < CH) nt_[i] = p[i * 256 + threadIdx.x];
#pragma unroll
        for (int c = 0; c < CS; ++c) load_a(k0 + c * KSTEP, na[c]);
    };
    fetch(0);
    for (int k0 = 0; k0 < a.sh.kp; k0 += CS * KSTEP) {
        dv2 av[CS];
#pragma unroll
        for (int i = 0; i < NL; ++i)
            if (CH % 256 == 0 || i * 256 + (int)threadIdx.x < CH) tb[i * 256 + threadIdx.x] = nt_[i];
#pragma unroll
        for (int c = 0; c < CS; ++c) av[c] = na[c];
        __syncthreads();
        if (k0 + CS * KSTEP < a.sh.kp) fetch(k0 + CS * KSTEP);
#pragma unroll
        for (int c = 0; c < CS; ++c)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const dv2 x = NG > 1 ? av[c] * s[g] : av[c];
                dv2 b[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) b[t] = tb[((c * NG + g) * NT + t) * 64 + lane];
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, b[t].x, acc[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, b[t].y, acc[t], 0, 0, 0);
            }
        __syncthreads();
    }
    // acc component r of a lane: element e0 + lane/16 + 4 r, column lane%16 of the tile
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const long er = e0 + (lane >> 4) + 4 * r;
        if (er >= a.nElmt) continue;
        const double jo = a.post == kScaleElement ? a.jac[er] : 1.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n = (blockIdx.y * NT + t) * 16 + row;
            if (n >= N) continue;
            double v = acc[t][r] * jo;
            if (a.post == kScalePoint) v *= a.jac[er * N + n];
            a.out[er * N + n] = v;
        }
    }
}

// Runs of a geometry term: the first, and for a pair of directions the one after it, of which
// half the difference counts.
__device__ __forceinline__ int first_run(int ng, int g, bool &pair)
{
    const int D = ng == 1 ? 0 : ng == 4 ? 2 : 3;
    int r = 1;
    pair = false;
    if (g == 0) return 0;
    for (int a = 0, h = 1; a < D; ++a)
        for (int b = a; b < D; ++b, ++h) {
            pair = b != a;
            if (h == g) return r;
            r += pair ? 2 : 1;
        }
    return r;
}

// One thread per entry of the fragment-ordered table, in its order:
// [column group][step][g][tile][lane][2], lane = 16 kq + column, k = 8 step + 2 kq + component.
__global__ void dense_pack_kernel(DenseShape sh, int transposed, const double *__restrict__ runs,
                                  double *__restrict__ tab)
{
    const int steps = sh.kp / KSTEP, per = sh.nt * 128;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)sh.ncg * steps * sh.ng * per) return;
    const int w = (int)(i % per), g = (int)(i / per) % sh.ng, step = (int)(i / per / sh.ng) % steps,
              cg = (int)(i / per / sh.ng / steps);
    const int comp = w & 1, lane = (w >> 1) & 63, t = w >> 7;
    const int k = step * KSTEP + 2 * (lane >> 4) + comp, n = (cg * sh.nt + t) * 16 + (lane & 15);
    double v = 0.0;
    if (k < sh.K && n < sh.N) {
        const long KN = (long)sh.K * sh.N;
        bool pair;
        const double *src = runs + first_run(sh.ng, g, pair) * KN +
                            (transposed ? (long)n * sh.K + k : (long)k * sh.N + n);
        v = pair ? 0.5 * (src[0] - src[KN]) : src[0];
    }
    tab[i] = v;
}

__global__ void dense_units_kernel(int M, int D, int nrun, double *__restrict__ in,
                                   double *__restrict__ jac, double *__restrict__ df)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = nrun * M;  // elements
    if (i >= (long)n * M) return;
    const int e = (int)(i / M), m = (int)(i - (long)e * M), run = e / M;
    in[i] = e - run * M == m ? 1.0 : 0.0;
    if (m) return;
    jac[e] = run ? 0x1p-200 : 1.0;
    double f[3] = {0.0, 0.0, 0.0};
    for (int a = 0, r = 1; a < D; ++a)
        for (int b = a; b < D; ++b) {
            if (r == run || (b != a && r + 1 == run)) {
                f[a] = 0x1p100;
                f[b] = r == run ? 0x1p100 : -0x1p100;
            }
            r += b != a ? 2 : 1;
        }
    for (int c = 0; c < D; ++c)
        for (int d = 0; d < D; ++d) df[(long)(c * D + d) * n + e] = c == 0 ? f[d] : 0.0;
}

template <int NG>
hipError_t launch_ng(const DenseArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.nElmt + 63) / 64), (unsigned)a.sh.ncg);
    switch (a.sh.nt) {
#define IMF_NT(n) \
    case n: dense_kernel<n, NG><<<grid, 256, 0, s>>>(a); break
        IMF_NT(1);
        IMF_NT(2);
        IMF_NT(3);
        IMF_NT(4);
        IMF_NT(5);
        IMF_NT(6);
        IMF_NT(7);
        IMF_NT(8);
#undef IMF_NT
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

DenseShape dense_shape(int K, int N, int ng)
{
    DenseShape sh;
    const int tiles = (N + 15) / 16;
    if (ng > 1 && tiles > 8) return sh;  // Helmholtz: one column group (at most 128 modes)
    sh.K = K;
    sh.N = N;
    sh.ng = ng;
    sh.ncg = (tiles + 7) / 8;
    sh.nt = (tiles + sh.ncg - 1) / sh.ncg;
    const int kc = chunk_steps(ng) * KSTEP;
    sh.kp = (K + kc - 1) / kc * kc;
    return sh;
}

int dense_runs(int D) { return D == 0 ? 1 : D == 2 ? 5 : 10; }

hipError_t dense_units(int M, int D, double *in, double *jac, double *df, hipStream_t s)
{
    const long n = (long)dense_runs(D) * M * M;
    dense_units_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(M, D, dense_runs(D), in, jac, df);
    return hipGetLastError();
}

hipError_t dense_pack(const DenseShape &sh, bool transposed, const double *runs, double *tab, hipStream_t s)
{
    const long n = (long)sh.tab_len();
    dense_pack_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(sh, transposed ? 1 : 0, runs, tab);
    return hipGetLastError();
}

hipError_t launch_dense(const DenseArgs &a, hipStream_t s)
{
    return a.sh.ng == 1 ? launch_ng<1>(a, s) : a.sh.ng == 4 ? launch_ng<4>(a, s) : launch_ng<7>(a, s);
}

}  // namespace imf
