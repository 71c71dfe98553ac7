// Whole-iteration scan kernels over sites, the other minimisers and integrators.
#include "scan_iter.hpp"

namespace mafm {

template hipError_t launch_iter_sites<false, ITER_SITES, false>(const IterLaunch&, int);
template hipError_t launch_iter_sites<true, ITER_SITES, false>(const IterLaunch&, int);

}  // namespace mafm
