// Collapsed-coordinate operators on pencils for compile-time orders (FP64).
//
// One element is owned by N0 N1 threads; a workgroup holds several elements, so that its
// lanes are nearly all used (prism of 6 points: 36 of 64 lanes with one element per wave,
// 252 of 256 with seven per workgroup).  Every one-dimensional contraction runs in registers
// on a line of the element held by one thread, re-oriented through LDS in between:
//   (p, q) lines  coefficients <-> eta2 points, the tables of each (p, q) read from LDS
//   (p, k) lines  q <-> j
//   (j, k) lines  p <-> i, and the eta0 derivative of the same line before it is written
//   (i, k) lines  the eta1 derivative
//   (i, j) lines  the eta2 derivative and the pointwise part, geometry read coalesced
// and the same back with D^T (dbdata = D bdata, checked when the operator is made), so the
// reference's four inner products become one D^T per direction and one (B0 B1 B2)^T.  The
// tables of eta0 (and eta1, tetrahedra excepted) are the same for all lanes and come through
// scalar registers.  The vertex and edge corrections of mf_{prism,tet,pyr}.hip enter the
// (p, q) and (p, k) steps as there.  The metric is kept in the reference coordinates and the
// collapse applied to the derivatives (as PhysDeriv does), so that a point needs 7 values
// instead of 10 and no metric is formed in the kernel.
//
// The runtime-size kernels read two LDS values per multiply-add, run one element per 256
// threads and form the metric from ten streamed values per point.  Helmholtz on curved
// elements, 12e6 points (at most 120 000 elements), one point more than modes, before / now
// in us for 3, 5 and 8 modes: tetrahedra 394/64, 989/194, 945/330; prisms 344/63, 655/153,
// 821/219; pyramids 359/60, 865/152, 1560/291 (the 7 values per point at the 4.8 TB/s of a
// copy: 48, 140, 148 us).  PhysDeriv of 8 modes: tetrahedra 531/227, prisms 366/261,
// pyramids 497/264, at the rate of a copy.
#pragma once

#include "mf_pencil.hpp"
#include "mf_prism.hpp"
#include "mf_pyr.hpp"
#include "mf_tet.hpp"

namespace imf {

template <int SH, int NM, int NQ>
struct PenCfg {
    static constexpr int N0 = NQ, N1 = SH == kTet ? NQ - 1 : NQ, N2 = NQ - 1;
    static constexpr int Q = N0 * N1 * N2, TPE = N0 * N1;
    static constexpr int TRI = NM * (NM + 1) / 2;
    static constexpr int M = SH == kPrism ? NM * TRI : SH == kTet ? NM * (NM + 1) * (NM + 2) / 6
                                                                  : NM * (NM + 1) * (2 * NM + 1) / 6;
    static constexpr int R1 = SH == kTet ? TRI : NM;         // rows of B1
    static constexpr int R2 = SH == kPrism ? TRI : M;        // rows of B2
    static constexpr int NP = SH == kTet ? TRI : NM * NM;    // (p, q) pairs
    static constexpr int NPX = SH == kTet ? NP + 2 : NP;     // and the two correction rows
    static constexpr int P0 = N0 | 1, P2 = N2 | 1;           // odd LDS row strides
    // offsets in the table image
    static constexpr int oB0 = 0, oD0 = 2 * NM * N0, oW0 = oD0 + N0 * N0, oB1 = oW0 + 2 * N0;
    static constexpr int oD1 = oB1 + 2 * R1 * N1, oW1 = oD1 + N1 * N1, oB2 = oW1 + 2 * N1;
    static constexpr int oD2 = oB2 + 2 * R2 * N2, oW2 = oD2 + N2 * N2, oX = oW2 + 2 * N2;
    static constexpr int oH0 = oX, oH1 = oH0 + N0, oG1 = oH1 + N1, oG2 = oG1 + N1;
    // one LDS buffer of an element
    static constexpr int cmax(int a, int b) { return a > b ? a : b; }
    static constexpr int S = cmax(cmax(N1 * N2 * P0, NPX * P2), cmax(M, NM * N1 * N2));
    // one wave where it holds four elements (no barriers between waves), else the block of 256
    // down to 64 threads with the most lanes used (a smaller one must use 3 % more: it shares
    // the staged tables among fewer elements)
    static constexpr int block()
    {
        if (64 / TPE >= 4) return 64;
        int best = 256, bu = 256 / TPE * TPE * 1000 / 256;
        for (int b = 192; b >= 64; b -= 64)
            if (b / TPE * TPE * 1000 / b > bu + 30) {
                bu = b / TPE * TPE * 1000 / b;
                best = b;
            }
        return best;
    }
    static constexpr int BLOCK = block(), EPB = BLOCK / TPE;
    static_assert(TPE <= 256 && NPX <= TPE && NM * N2 <= TPE, "lines per phase");
};

// (p, q) of a pair, its first mode, its number of modes and its B2 row (row of r = 0).
template <int SH, int NM>
__device__ __forceinline__ void pen_pair(int t, int &p, int &q, int &m0, int &len, int &row)
{
    if constexpr (SH == kPrism) {
        p = t / NM;
        q = t - p * NM;
        len = NM - p;
        row = p * NM - p * (p - 1) / 2;
        m0 = NM * row + q * len;
    } else if constexpr (SH == kPyr) {
        p = t / NM;
        q = t - p * NM;
        len = NM - max(p, q);
        // modes before (p, q): rows p' < p hold sum_q (NM - max(p', q))
        m0 = 0;
#pragma unroll
        for (int pp = 0; pp < NM; ++pp)
            if (pp < p) m0 += (pp + 1) * (NM - pp) + (NM - pp) * (NM - pp - 1) / 2;
        m0 += q <= p ? q * (NM - p) : (p + 1) * (NM - p) + (NM * (q - p - 1) - (q * (q - 1) - p * (p + 1)) / 2);
        row = m0;
    } else {
        p = 0;
        int s = 0;
#pragma unroll
        for (int pp = 1; pp < NM; ++pp) {
            const int st = pp * NM - pp * (pp - 1) / 2;
            if (st <= t) {
                p = pp;
                s = st;
            }
        }
        q = t - s;
        m0 = 0;
#pragma unroll
        for (int pp = 0; pp < NM; ++pp)
            if (pp < p) m0 += (NM - pp) * (NM - pp + 1) / 2;
        m0 += q * (NM - p) - q * (q - 1) / 2;
        len = NM - p - q;
        row = m0;
    }
}

template <int SH, int NM, int NQ, int KIND>
__global__ __launch_bounds__((PenCfg<SH, NM, NQ>::BLOCK)) void pencil_kernel(
    PencilArgs a, const double *__restrict__ tab, const double *__restrict__ in,
    const double *__restrict__ jac, const double *__restrict__ df,
    const double *__restrict__ geom, double *__restrict__ out)
{
    using C = PenCfg<SH, NM, NQ>;
    constexpr int N0 = C::N0, N1 = C::N1, N2 = C::N2, Q = C::Q, M = C::M, TPE = C::TPE;
    constexpr int P0 = C::P0, P2 = C::P2, EPB = C::EPB, S = C::S;
    constexpr bool FROM_MODES = KIND == kBwdTrans || KIND == kHelmholtz;
    constexpr bool TO_MODES = KIND == kIProduct || KIND == kHelmholtz || KIND == kIProdDeriv;
    constexpr bool DERIV = KIND == kHelmholtz || KIND == kPhysDeriv;
    constexpr bool MODES = FROM_MODES || TO_MODES;
    constexpr int LB1 = SH == kTet && MODES ? C::R1 * N1 : 0, LB2 = MODES ? C::R2 * N2 : 0;
    __shared__ double lds[EPB][3][S];
    __shared__ double lt[LB1 + LB2 + 1];
    const int es = threadIdx.x / TPE, t = threadIdx.x - es * TPE;
    const bool active = es < EPB;
    const long e0 = (long)blockIdx.x * EPB, e = e0 + es;
    const int nv = (int)min((long)EPB, (long)a.nElmt - e0);
    const bool valid = active && es < nv;
    double *BU = lds[active ? es : 0][0], *BD0 = lds[active ? es : 0][1], *BD1 = lds[active ? es : 0][2];
    const double *B0 = tab + C::oB0, *D0 = tab + C::oD0, *D1 = tab + C::oD1, *D2 = tab + C::oD2;
    const double *W2 = tab + C::oW2, *G2 = tab + C::oG2;
    const double *lB1 = lt, *lB2 = lt + LB1;
    const int ci = t % N0, cj = t / N0;  // this thread's (i, j) line
    const long nQ = (long)a.nElmt * Q;

    // Curved Helmholtz: the first NG arrays of this thread's geometry (w J, w J G^ab) travel
    // with the coefficients; as many as fit in 72 registers, the rest are read where used.
    constexpr int NG = KIND == kHelmholtz ? (72 / (2 * N2) > 7 ? 7 : 72 / (2 * N2)) : 0;
    constexpr long GS = geo_stride(7 * Q, 8);
    double gp[NG ? NG : 1][N2];
    if constexpr (KIND == kHelmholtz) {
        if (a.deformed && valid) {
#pragma unroll
            for (int c = 0; c < NG; ++c)
#pragma unroll
                for (int k = 0; k < N2; ++k)
                    gp[c][k] = __builtin_nontemporal_load(geom + e * GS + c * Q + k * TPE + t);
        }
    }
    if constexpr (MODES) {
        for (int i = threadIdx.x; i < LB1; i += C::BLOCK) lt[i] = tab[C::oB1 + i];
        for (int i = threadIdx.x; i < LB2; i += C::BLOCK) lt[LB1 + i] = tab[C::oB2 + i];
    }

    double u[N2];  // the (i, j) line
    if constexpr (FROM_MODES) {
        for (int i = threadIdx.x; i < nv * M; i += C::BLOCK) {
            const int sl = i / M;
            lds[sl][0][i - sl * M] = __builtin_nontemporal_load(in + e0 * M + i);
        }
        __syncthreads();
        // r -> k on (p, q) lines
        if (active && t < C::NPX) {
            double v[N2];
            if (SH == kTet && t >= C::NP) {
                // rows added to p = 1: X0 (with B1 of (0,0)) and X (with B1 of (0,1))
                const double c1 = BU[1];
                const double cn = t == C::NP ? 0.0 : BU[NM];
#pragma unroll
                for (int k = 0; k < N2; ++k) v[k] = fma(cn, lB2[k], c1 * lB2[N2 + k]);
#pragma unroll
                for (int r = 1; r < NM - 1; ++r) {
                    const double c = t == C::NP ? 0.0 : BU[NM + r];
#pragma unroll
                    for (int k = 0; k < N2; ++k) v[k] = fma(c, lB2[(r + 1) * N2 + k], v[k]);
                }
            } else {
                int p, q, m0, len, row;
                pen_pair<SH, NM>(t, p, q, m0, len, row);
#pragma unroll
                for (int k = 0; k < N2; ++k) v[k] = 0.0;
                for (int r = 0; r < len; ++r) {
                    const double c = BU[m0 + r];
#pragma unroll
                    for (int k = 0; k < N2; ++k) v[k] = fma(c, lB2[(row + r) * N2 + k], v[k]);
                }
                const bool cor = SH == kPrism ? p == 1 : SH == kPyr ? p + q > 0 && p <= 1 && q <= 1
                                                                    : t == 1;
                if (cor) {
                    const double c = BU[SH == kPrism ? q * NM + 1 : 1];
#pragma unroll
                    for (int k = 0; k < N2; ++k) v[k] = fma(c, lB2[N2 + k], v[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < N2; ++k) BD0[t * P2 + k] = v[k];
        }
        __syncthreads();
        // q -> j on (p, k) lines
        if (active && t < NM * N2) {
            const int p = t / N2, k = t - p * N2;
            double s[N1];
#pragma unroll
            for (int j = 0; j < N1; ++j) s[j] = 0.0;
            if constexpr (SH == kTet) {
                const int ps = p * NM - p * (p - 1) / 2;
                for (int q = 0; q < NM - p; ++q) {
                    const double x = BD0[(ps + q) * P2 + k];
#pragma unroll
                    for (int j = 0; j < N1; ++j) s[j] = fma(x, lB1[(ps + q) * N1 + j], s[j]);
                }
                if (p == 1) {
                    const double x0 = BD0[C::NP * P2 + k], x1 = BD0[(C::NP + 1) * P2 + k];
#pragma unroll
                    for (int j = 0; j < N1; ++j) s[j] = fma(x1, lB1[N1 + j], fma(x0, lB1[j], s[j]));
                }
            } else {
                const double *B1 = tab + C::oB1;
#pragma unroll
                for (int q = 0; q < NM; ++q) {
                    const double x = BD0[(p * NM + q) * P2 + k];
#pragma unroll
                    for (int j = 0; j < N1; ++j) s[j] = fma(x, B1[q * N1 + j], s[j]);
                }
            }
#pragma unroll
            for (int j = 0; j < N1; ++j) BD1[(p * N1 + j) * N2 + k] = s[j];
        }
        __syncthreads();
        // p -> i on (j, k) lines, t = j N2 + k, and the eta0 derivative of the line
        if (active && t < N1 * N2) {
            double x[NM], l[N0];
#pragma unroll
            for (int p = 0; p < NM; ++p) x[p] = BD1[p * N1 * N2 + t];
#pragma unroll
            for (int i = 0; i < N0; ++i) {
                double s = x[0] * B0[i];
#pragma unroll
                for (int p = 1; p < NM; ++p) s = fma(x[p], B0[p * N0 + i], s);
                l[i] = s;
                BU[t * P0 + i] = s;
            }
            if constexpr (DERIV) {
#pragma unroll
                for (int i = 0; i < N0; ++i) {
                    double s = l[0] * D0[i];
#pragma unroll
                    for (int b = 1; b < N0; ++b) s = fma(l[b], D0[b * N0 + i], s);
                    BD0[t * P0 + i] = s;
                }
            }
        }
        __syncthreads();
    }
    if constexpr (KIND == kPhysDeriv) {
#pragma unroll
        for (int k = 0; k < N2; ++k)
            u[k] = valid ? __builtin_nontemporal_load(in + e * Q + k * TPE + t) : 0.0;
        if (active)
#pragma unroll
            for (int k = 0; k < N2; ++k) BU[(cj * N2 + k) * P0 + ci] = u[k];
        __syncthreads();
        if (active && t < N1 * N2) {
            double l[N0];
#pragma unroll
            for (int i = 0; i < N0; ++i) l[i] = BU[t * P0 + i];
#pragma unroll
            for (int i = 0; i < N0; ++i) {
                double s = l[0] * D0[i];
#pragma unroll
                for (int b = 1; b < N0; ++b) s = fma(l[b], D0[b * N0 + i], s);
                BD0[t * P0 + i] = s;
            }
        }
    }
    if constexpr (DERIV) {
        // eta1 derivative on (i, k) lines
        if (active && t < N0 * N2) {
            const int i = t % N0, k = t / N0;
            double l[N1];
#pragma unroll
            for (int j = 0; j < N1; ++j) l[j] = BU[(j * N2 + k) * P0 + i];
#pragma unroll
            for (int j = 0; j < N1; ++j) {
                double s = l[0] * D1[j];
#pragma unroll
                for (int b = 1; b < N1; ++b) s = fma(l[b], D1[b * N1 + j], s);
                BD1[(j * N2 + k) * P0 + i] = s;
            }
        }
        __syncthreads();
    }

    // (i, j) lines: the pointwise part
    const int at = active ? cj * N2 * P0 + ci : 0;  // LDS position of (k = 0), stride P0
    if constexpr (KIND == kBwdTrans) {
        if (!valid) return;
        const double wij = a.scaled ? tab[C::oW0 + ci] * tab[C::oW1 + cj] : 1.0;
#pragma unroll
        for (int k = 0; k < N2; ++k) {
            double v = BU[at + k * P0];
            if (a.scaled) v *= wij * W2[k] * (a.deformed ? jac[e * Q + k * TPE + t] : jac[e]);
            __builtin_nontemporal_store(v, out + e * Q + k * TPE + t);
        }
        return;
    } else {
        // collapse of this line: h0 = (1 + eta0)/2, h1 = (1 + eta1)/2, g1 = 2/(1 - eta1)
        const double h0 = active ? tab[C::oH0 + ci] : 0.0, h1 = active ? tab[C::oH1 + cj] : 0.0;
        const double g1 = active && SH == kTet ? tab[C::oG1 + cj] : 1.0;
        const double wij = MODES && active ? tab[C::oW0 + ci] * tab[C::oW1 + cj] : 0.0;
        // xi derivatives from eta derivatives at point k (h2 = 2/(1 - eta2))
        auto chain = [&](double h2, double &x0, double &x1, double &x2) {
            if constexpr (SH == kPrism) {
                x0 *= h2;
                x2 = fma(h0, x0, x2);
            } else if constexpr (SH == kPyr) {
                x0 *= h2;
                x1 *= h2;
                x2 = fma(h1, x1, fma(h0, x0, x2));
            } else {
                x0 *= g1 * h2;
                const double hx = h0 * x0, xg = h2 * x1;
                x1 = hx + xg;
                x2 = fma(h1, xg, hx) + x2;
            }
        };
        // its transpose
        auto chain_t = [&](double h2, double &y0, double &y1, double &y2) {
            if constexpr (SH == kPrism) {
                y0 = h2 * fma(h0, y2, y0);
            } else if constexpr (SH == kPyr) {
                y0 = h2 * fma(h0, y2, y0);
                y1 = h2 * fma(h1, y2, y1);
            } else {
                y0 = g1 * h2 * fma(h0, y1 + y2, y0);
                y1 = h2 * fma(h1, y2, y1);
            }
        };
        double acc[N2], y2[N2];
        if constexpr (KIND == kHelmholtz || KIND == kPhysDeriv) {
            if constexpr (KIND == kHelmholtz) {
#pragma unroll
                for (int k = 0; k < N2; ++k) u[k] = BU[at + k * P0];
            }
            double J = 0.0, m[6] = {};
            if (KIND == kHelmholtz && valid && !a.deformed) {
                double f[9];
#pragma unroll
                for (int d = 0; d < 9; ++d) f[d] = df[(long)d * a.nElmt + e];
                J = jac[e] * wij;
                int n = 0;
#pragma unroll
                for (int x = 0; x < 3; ++x)
#pragma unroll
                    for (int y = x; y < 3; ++y)
                        m[n++] = J * fma(f[6 + x], f[6 + y], fma(f[3 + x], f[3 + y], f[x] * f[y]));
            }
            double o[KIND == kPhysDeriv ? 3 : 1][N2];
#pragma unroll
            for (int k = 0; k < N2; ++k) {
                double x2 = u[0] * D2[k];
#pragma unroll
                for (int b = 1; b < N2; ++b) x2 = fma(u[b], D2[b * N2 + k], x2);
                double x0 = BD0[at + k * P0], x1 = BD1[at + k * P0];
                const double h2 = G2[k];
                chain(h2, x0, x1, x2);
                if constexpr (KIND == kHelmholtz) {
                    double jw, g00, g01, g02, g11, g12, g22;
                    if (a.deformed) {
                        const double *g = geom + e * GS + k * TPE + t;
                        auto get = [&](int c) {
                            return c < NG ? gp[c < NG ? c : 0][k]
                                          : valid ? __builtin_nontemporal_load(g + c * Q) : 0.0;
                        };
                        jw = get(0);
                        g00 = get(1);
                        g01 = get(2);
                        g02 = get(3);
                        g11 = get(4);
                        g12 = get(5);
                        g22 = get(6);
                    } else {
                        const double w = W2[k];
                        jw = J * w;
                        g00 = m[0] * w;
                        g01 = m[1] * w;
                        g02 = m[2] * w;
                        g11 = m[3] * w;
                        g12 = m[4] * w;
                        g22 = m[5] * w;
                    }
                    double y0 = fma(g02, x2, fma(g01, x1, g00 * x0));
                    double y1 = fma(g12, x2, fma(g11, x1, g01 * x0));
                    y2[k] = fma(g22, x2, fma(g12, x1, g02 * x0));
                    chain_t(h2, y0, y1, y2[k]);
                    acc[k] = a.lambda * jw * u[k];
                    if (active) {
                        BD0[at + k * P0] = y0;
                        BD1[at + k * P0] = y1;
                    }
                } else if (valid) {
                    const long g = a.deformed ? e * Q + k * TPE + t : e, np = a.deformed ? nQ : a.nElmt;
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        o[c][k] = fma(x2, df[(3 * c + 2) * np + g],
                                      fma(x1, df[(3 * c + 1) * np + g], x0 * df[3 * c * np + g]));
                }
            }
            if constexpr (KIND == kPhysDeriv) {
                if (valid)
#pragma unroll
                    for (int c = 0; c < 3; ++c)
#pragma unroll
                        for (int k = 0; k < N2; ++k)
                            __builtin_nontemporal_store(o[c][k], out + c * nQ + e * Q + k * TPE + t);
                return;
            }
        } else if constexpr (KIND == kIProduct) {
#pragma unroll
            for (int k = 0; k < N2; ++k) {
                double v = valid ? __builtin_nontemporal_load(in + e * Q + k * TPE + t) : 0.0;
                if (a.scaled && valid)
                    v *= wij * W2[k] * (a.deformed ? __builtin_nontemporal_load(jac + e * Q + k * TPE + t) : jac[e]);
                if (active) BU[at + k * P0] = v;
            }
        } else {  // kIProdDeriv
#pragma unroll
            for (int k = 0; k < N2; ++k) {
                double y0 = 0.0, y1 = 0.0;
                y2[k] = 0.0;
                acc[k] = 0.0;
                if (valid) {
                    const long q = e * Q + k * TPE + t, g = a.deformed ? q : e, np = a.deformed ? nQ : a.nElmt;
                    const double x0 = __builtin_nontemporal_load(in + q), x1 = __builtin_nontemporal_load(in + nQ + q),
                                 x2 = __builtin_nontemporal_load(in + 2 * nQ + q);
                    const double wj = wij * W2[k] * (a.deformed ? jac[q] : jac[e]);
                    double v[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        v[c] = wj * fma(x2, df[(6 + c) * np + g], fma(x1, df[(3 + c) * np + g], x0 * df[c * np + g]));
                    y0 = v[0];
                    y1 = v[1];
                    y2[k] = v[2];
                    chain_t(G2[k], y0, y1, y2[k]);
                }
                if (active) {
                    BD0[at + k * P0] = y0;
                    BD1[at + k * P0] = y1;
                }
            }
        }
        if constexpr (KIND == kHelmholtz || KIND == kIProdDeriv) {
            // D2^T on the line, then D1^T on (i, k) lines added to it
#pragma unroll
            for (int k = 0; k < N2; ++k) {
                double s = acc[k];
#pragma unroll
                for (int b = 0; b < N2; ++b) s = fma(y2[b], D2[k * N2 + b], s);
                if (active) BU[at + k * P0] = s;
            }
            __syncthreads();
            if (active && t < N0 * N2) {
                const int i = t % N0, k = t / N0;
                double l[N1];
#pragma unroll
                for (int j = 0; j < N1; ++j) l[j] = BD1[(j * N2 + k) * P0 + i];
#pragma unroll
                for (int j = 0; j < N1; ++j) {
                    double s = BU[(j * N2 + k) * P0 + i];
#pragma unroll
                    for (int b = 0; b < N1; ++b) s = fma(l[b], D1[j * N1 + b], s);
                    BU[(j * N2 + k) * P0 + i] = s;
                }
            }
        }
        __syncthreads();
    }

    if constexpr (TO_MODES) {
        // D0^T and i -> p on (j, k) lines
        if (active && t < N1 * N2) {
            double s[N0];
#pragma unroll
            for (int i = 0; i < N0; ++i) s[i] = BU[t * P0 + i];
            if constexpr (KIND != kIProduct) {
                double l[N0];
#pragma unroll
                for (int i = 0; i < N0; ++i) l[i] = BD0[t * P0 + i];
#pragma unroll
                for (int i = 0; i < N0; ++i)
#pragma unroll
                    for (int b = 0; b < N0; ++b) s[i] = fma(l[b], D0[i * N0 + b], s[i]);
            }
#pragma unroll
            for (int p = 0; p < NM; ++p) {
                double v = s[0] * B0[p * N0];
#pragma unroll
                for (int i = 1; i < N0; ++i) v = fma(s[i], B0[p * N0 + i], v);
                BD1[p * N1 * N2 + t] = v;
            }
        }
        __syncthreads();
        // j -> q on (p, k) lines
        if (active && t < NM * N2) {
            const int p = t / N2, k = t - p * N2;
            double l[N1];
#pragma unroll
            for (int j = 0; j < N1; ++j) l[j] = BD1[(p * N1 + j) * N2 + k];
            if constexpr (SH == kTet) {
                const int ps = p * NM - p * (p - 1) / 2;
                for (int q = 0; q < NM - p; ++q) {
                    double s = 0.0;
#pragma unroll
                    for (int j = 0; j < N1; ++j) s = fma(l[j], lB1[(ps + q) * N1 + j], s);
                    BD0[(ps + q) * P2 + k] = s;
                }
                if (p == 1) {
                    double s0 = 0.0, s1 = 0.0;
#pragma unroll
                    for (int j = 0; j < N1; ++j) {
                        s0 = fma(l[j], lB1[j], s0);
                        s1 = fma(l[j], lB1[N1 + j], s1);
                    }
                    BD0[C::NP * P2 + k] = s0;
                    BD0[(C::NP + 1) * P2 + k] = s1;
                }
            } else {
                const double *B1 = tab + C::oB1;
#pragma unroll
                for (int q = 0; q < NM; ++q) {
                    double s = l[0] * B1[q * N1];
#pragma unroll
                    for (int j = 1; j < N1; ++j) s = fma(l[j], B1[q * N1 + j], s);
                    BD0[(p * NM + q) * P2 + k] = s;
                }
            }
        }
        __syncthreads();
        // k -> r on (p, q) lines
        if (active && t < C::NP) {
            int p, q, m0, len, row;
            pen_pair<SH, NM>(t, p, q, m0, len, row);
            double l[N2];
#pragma unroll
            for (int k = 0; k < N2; ++k) l[k] = BD0[t * P2 + k];
            for (int r = 0; r < len; ++r) {
                double s = 0.0;
#pragma unroll
                for (int k = 0; k < N2; ++k) s = fma(l[k], lB2[(row + r) * N2 + k], s);
                const int md = m0 + r;
                if constexpr (SH == kPrism) {
                    if (p == 0 && r == 1)  // the phi_1(eta0) part of the collapsed-edge mode
#pragma unroll
                        for (int k = 0; k < N2; ++k) s = fma(lB2[N2 + k], BD0[(NM + q) * P2 + k], s);
                } else if constexpr (SH == kPyr) {
                    if (md == 1)  // top vertex: (0,1), (1,0), (1,1)
#pragma unroll
                        for (int k = 0; k < N2; ++k)
                            s = fma(lB2[N2 + k], BD0[P2 + k] + BD0[NM * P2 + k] + BD0[(NM + 1) * P2 + k], s);
                } else {
                    const double *Y0 = BD0 + C::NP * P2, *Y = Y0 + P2;
                    if (md == 1) {  // top vertex
#pragma unroll
                        for (int k = 0; k < N2; ++k) s = fma(lB2[N2 + k], BD0[P2 + k] + Y0[k] + Y[k], s);
                    } else if (md == NM) {  // bottom vertex of the collapsed edge
#pragma unroll
                        for (int k = 0; k < N2; ++k) s = fma(lB2[k], Y[k], s);
                    } else if (md > NM && md < 2 * NM - 1) {  // singular edge
                        const double *rw = lB2 + (md - NM + 1) * N2;
#pragma unroll
                        for (int k = 0; k < N2; ++k) s = fma(rw[k], Y[k], s);
                    }
                }
                BU[md] = s;
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nv * M; i += C::BLOCK) {
            const int sl = i / M;
            __builtin_nontemporal_store(lds[sl][0][i - sl * M], out + e0 * M + i);
        }
    }
}

template <int SH, int NM, int NQ, int KIND>
hipError_t launch_pencil(const PencilArgs &a, hipStream_t s)
{
    using C = PenCfg<SH, NM, NQ>;
    const unsigned grid = (unsigned)((a.nElmt + C::EPB - 1) / C::EPB);
    pencil_kernel<SH, NM, NQ, KIND><<<grid, C::BLOCK, 0, s>>>(a, a.tab, a.in, a.jac, a.df, a.geom, a.out);
    return hipGetLastError();
}

template <int SH, int NM, int NQ>
PencilFn pencil_of(int kind)
{
    switch (kind) {
    case kBwdTrans: return &launch_pencil<SH, NM, NQ, kBwdTrans>;
    case kIProduct: return &launch_pencil<SH, NM, NQ, kIProduct>;
    case kHelmholtz: return &launch_pencil<SH, NM, NQ, kHelmholtz>;
    case kIProdDeriv: return &launch_pencil<SH, NM, NQ, kIProdDeriv>;
    case kPhysDeriv: return &launch_pencil<SH, NM, NQ, kPhysDeriv>;
    default: return nullptr;
    }
}

// nm = 2..8 with one or two points more than modes.
template <int SH>
PencilFn lookup_pencil(int kind, int nm, int nq0)
{
    switch (nm * 16 + nq0) {
#define IMF_P(m) \
    case m * 16 + m + 1: return pencil_of<SH, m, m + 1>(kind); \
    case m * 16 + m + 2: return pencil_of<SH, m, m + 2>(kind)
        IMF_P(2);
        IMF_P(3);
        IMF_P(4);
        IMF_P(5);
        IMF_P(6);
        IMF_P(7);
        IMF_P(8);
#undef IMF_P
    default: return nullptr;
    }
}

}  // namespace imf
