// Pencil kernels of the collapsed shapes (prisms, tetrahedra, pyramids) for compile-time orders.
#pragma once

#include <hip/hip_runtime.h>

#include "imf_common.hpp"

namespace imf {

struct PencilArgs {
    int nElmt;
    int scaled;          // BwdTrans: times w J (the transpose of IProduct); IProduct: w J applied
    int deformed;        // geometry per point, else per element
    double lambda;
    const double *tab;   // the shape's table image (mf_{prism,tet,pyr}.hpp), then pencil_extra()
    const double *in;
    double *out;
    const double *jac;   // GetJac layout
    const double *df;    // GetDerivFactors layout
    const double *geom;  // deformed Helmholtz: packed by pencil_pack
};

using PencilFn = hipError_t (*)(const PencilArgs &, hipStream_t);

// Launcher of kind (kBwdTrans, kIProduct, kHelmholtz, kPhysDeriv, kIProdDeriv) for nm modes
// and nq0 points along eta0 with the reference's other counts (nq1 = nq0, or nq0 - 1 for
// tetrahedra; nq2 = nq0 - 1); null when there is none.
PencilFn lookup_pencil_prism(int kind, int nm, int nq0);
PencilFn lookup_pencil_tet(int kind, int nm, int nq0);
PencilFn lookup_pencil_pyr(int kind, int nm, int nq0);

// Doubles appended to the table image: (1 + z0)/2, (1 + z1)/2, 2/(1 - z1), 2/(1 - z2).
inline int pencil_extra(int nq0, int nq1, int nq2) { return nq0 + 2 * nq1 + nq2; }

// Deformed Helmholtz geometry: [e][GS], GS = geo_stride(7 Q, 8), of w J and w J G^ab in the
// reference coordinates (00, 01, 02, 11, 12, 22); w from the table image's three weight rows.
hipError_t pencil_pack(long nElmt, const int *nq, const double *const *d_w, const double *jac,
                       const double *df, double *out, hipStream_t s);

}  // namespace imf
