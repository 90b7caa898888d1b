// Which kernel or launch shape an operator takes by its sizes: rules that weigh two measured
// alternatives.  Plain C++, so that they can be checked without a device.
#pragma once

namespace imf {

// Hex Helmholtz: the number of elements from which a launch packs them into 256-thread workgroups (HexCfg); 0:
// never.  Many elements fill the lanes that an element of its own workgroup leaves idle, few are
// spread over more CUs and wait for no other element's barriers.  Narrow / wide in us, nq - 1 modes:
//   6 points FP64 deformed   16: 5.9/7.6   1 000: 8.0/8.8    4 000: 15.6/15.8   50 000: 131/118
//            FP64 regular    16: 5.6/6.7   1 000: 6.5/7.3    4 000: 11.3/10.9   50 000: 84/64
//   9 points FP64 deformed   16: 10.6/13.0 1 000: 17.9/18.9  1 500: 28.8/20.4   50 000: 585/536
//            FP32 deformed   16: 7.2/8.4   1 000: 12.0/12.9  1 500: 15.7/14.3   50 000: 265/237
//   7 points FP32 regular    16: 5.9/6.8   4 000: 10.8/11.2  8 000: 16.3/15.7   50 000: 74/69
// Never ahead at 12e6 points: 7 points FP64 deformed 133/150, 6 points FP32 deformed 74/79,
// 5 points FP64 70/70 and 121/127; BwdTrans, IProduct and PhysDeriv are bound by HBM (7 points:
// IProduct 51/70, PhysDeriv 76/101).
constexpr int helm_wide_from(int nq, bool f64, bool deformed)
{
    if (nq == 6) return f64 || !deformed ? 4000 : 0;
    if (nq == 7) return !f64 && !deformed ? 8000 : 0;
    return nq == 9 ? 1500 : 0;
}

// When a collapsed-shape operator takes dense products over its elements (mf_dense.hip).
struct DenseCase {
    int shape;            // kRouteTri ...
    bool helm;            // Helmholtz; else a transform
    bool from_modes;      // modes -> points (BwdTrans, transpose of IProduct); else points -> modes
    bool point_scale;     // points -> modes with a Jacobian per point
    bool pencil;          // a pencil kernel is the alternative, else the runtime-size kernel
    long M, Q, nElmt;     // modes and points of an element, elements
};
enum : int { kRouteTri = 0, kRouteTet = 1, kRoutePrism = 2, kRoutePyr = 3 };

// A dense product reads each table once per 64 elements and walks through K one chunk after
// another: about 3 us + K / 32 (0.6 + N / 48) us however few the elements are, flat until the
// chip is full.  The other kernels give an element to at most 256 threads: their time is short
// for few elements and grows with n.  So the dense product wins from some count on, which the
// rule states per class from times at 1 .. 120 000 elements (at most 12e6 points), 2 to 8 modes
// and 0, 1, 2, 4 or 8 points more, dense / other in us:
//   triangles, BwdTrans 8,10          n = 1000: 9.4 / 5.1    3 000: 9.7 / 5.8    30 000: 16 / 28
//   tetrahedra, Helmholtz 8,9         n = 256: 69 / 17       3 000: 70 / 39      20 833: 141 / 233
//               IProduct 8,9          n = 256: 61 / 9        10 000: 70 / 57     20 833: 99 / 109
//               IProduct 8,12         n = 256: 143 / 14      1 000: 143 / 50     8 264: 158 / 413
//               BwdTrans 8,12         n = 256: 18 / 12       1 000: 20 / 42      8 264: 98 / 317
// Triangles otherwise, and small elements, win at every count (tetrahedra 4,4: Helmholtz
// 7.5 / 15 at 64 elements, 34 / 423 at 120 000).  Over all 3 998 measured points the choice costs 1.005
// times the better of the two on average, 1.25 times or more in 22 of them.
inline bool dense_pays(const DenseCase &c)
{
    const bool tet = c.shape == kRouteTet, prism = c.shape == kRoutePrism;
    const long M = c.M, Q = c.Q, n = c.nElmt, nQ = n * Q;
    if (c.shape == kRouteTri) return c.helm || !c.from_modes || Q <= 16 || n >= 6000;
    if (c.helm) {
        // cost of the matrix M^2 (times the metric terms) against about Q per element
        if (c.pencil)
            return M * M < 27 * Q &&
                   (M <= (prism ? 10 : 20) || nQ >= (tet ? 300 : prism ? 800 : 550) * M * M);
        return M * M <= 1500 + 4 * Q + nQ / (prism ? 100 : 60);
    }
    if (c.from_modes) {
        // pencils run at the rate of the points written: 28 / 34 us for 120 000 tetrahedra 4,5
        if (c.pencil) return tet && M <= 20 && n >= 30000;
        // prisms of medium size fill the chip with the runtime-size kernel, which sums over no
        // shrinking mode ranges there (6,10: 101 / 98 us at 13 333 elements)
        return (Q <= 48 && M <= 30) ||
               ((!prism || M * Q <= 30000 || Q >= 1500) && nQ >= (prism ? 1200000 : 700000));
    }
    const double s = c.point_scale ? 1.7 : 1.0;  // the Jacobian per point is read beside the input
    if (c.pencil) return (tet || M <= 80) && n >= (tet ? 130 : prism ? 500 : 250) * s * M;
    const double few = prism ? Q * (14 + M / 3.0) : Q * (4 + M / 7.0), most = prism ? 6000 : 3500;
    return Q <= 40 || n >= (few < most ? few : most) * s;
}

}  // namespace imf
