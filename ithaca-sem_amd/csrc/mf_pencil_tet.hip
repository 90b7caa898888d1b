// Pencil kernels of the tet operators (mf_pencil_kernels.hpp).
#include "mf_pencil_kernels.hpp"

namespace imf {

PencilFn lookup_pencil_tet(int kind, int nm, int nq0) { return lookup_pencil<kTet>(kind, nm, nq0); }

}  // namespace imf
