// Whole-iteration scan kernels over sites of one height, FIRE with the midpoint integrator.
#include "scan_iter.hpp"

namespace mafm {

template hipError_t launch_iter_sites<false, ITER_FLAT, true>(const IterLaunch&, int);
template hipError_t launch_iter_sites<true, ITER_FLAT, true>(const IterLaunch&, int);

}  // namespace mafm
