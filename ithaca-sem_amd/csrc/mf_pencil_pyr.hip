// Pencil kernels of the pyramid operators (mf_pencil_kernels.hpp).
#include "mf_pencil_kernels.hpp"

namespace imf {

PencilFn lookup_pencil_pyr(int kind, int nm, int nq0) { return lookup_pencil<kPyr>(kind, nm, nq0); }

}  // namespace imf
