// Collapsed-shape operators as dense products over the elements (mf_dense.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace imf {

// out (nElmt x N) = sum_g diag(s_g) A (nElmt x K) T_g, T_g (K x N) the operator's matrix of
// one element.  A is the input, scaled by the Jacobian where `pre` says so; s_g are the
// element's geometry factors (ng = 1: s_0 = 1).
struct DenseShape {
    int K = 0, N = 0, ng = 0;   // ng = 1, 4 (2D Helmholtz) or 7 (3D Helmholtz)
    int nt = 0, ncg = 0;        // 16-wide column tiles per workgroup, column groups
    int kp = 0;                 // K rounded up to whole chunks of the kernel
    size_t tab_len() const { return (size_t)ncg * kp * ng * nt * 16; }
};

enum DenseScale : int { kScaleNone = 0, kScaleElement = 1, kScalePoint = 2 };

struct DenseArgs {
    DenseShape sh;
    int nElmt;
    int pre, post;       // DenseScale: Jacobian applied to the input / to the output
    double lambda;       // Helmholtz (ng > 1)
    const double *tab;   // fragment order (dense_pack)
    const double *in;
    double *out;
    const double *jac;   // GetJac layout
    const double *df;    // GetDerivFactors layout, one value per element (ng > 1)
};

// Sizes of the product for an element matrix of K x N and ng geometry terms; nt = 0 when the
// kernel does not take it.
DenseShape dense_shape(int K, int N, int ng);

// All terms into the fragment-ordered table, from the runs of dense_units (device): T_g row-major,
// K x N, or N x K where `transposed` is set.
hipError_t dense_pack(const DenseShape &sh, bool transposed, const double *runs, double *tab, hipStream_t s);

// Inputs that make an element kernel give its matrix: runs of M unit vectors with a Jacobian and
// (D > 0) D x D derivative factors per element.  Transforms: one run with unit Jacobians.
// Helmholtz with lambda = 1: the mass matrix (J = 1, no factors), then one run for each diagonal
// metric term and two for each pair.  A run's factors are one row, so that one metric term remains:
// e_a gives K_aa, e_a + e_b and e_a - e_b give K_aa + K_bb + (K_ab + K_ba) and the same with a
// minus sign.  They are 2^100 with J = 2^-200, which leaves the stiffness as it is and 2^-200 of
// the mass matrix beside it.
int dense_runs(int D);  // 1 for D = 0
hipError_t dense_units(int M, int D, double *in, double *jac, double *df, hipStream_t s);

hipError_t launch_dense(const DenseArgs &a, hipStream_t s);

}  // namespace imf
