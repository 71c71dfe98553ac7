// Whole-iteration scan kernels over sites, FIRE with the midpoint integrator.
#include "scan_iter.hpp"

namespace mafm {

template hipError_t launch_iter_sites<false, ITER_SITES, true>(const IterLaunch&, int);
template hipError_t launch_iter_sites<true, ITER_SITES, true>(const IterLaunch&, int);

}  // namespace mafm
