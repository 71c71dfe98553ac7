// Whole-iteration scan kernels through force grids and over periodic images, and the
// launcher of all of them.
#include "scan_iter.hpp"

namespace mafm {

// the kernels of site tables are instantiated in scan_iter_{sites,flat}_{mid,gen}.hip
extern template hipError_t launch_iter_sites<false, ITER_SITES, true>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<false, ITER_SITES, false>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<true, ITER_SITES, true>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<true, ITER_SITES, false>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<false, ITER_FLAT, true>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<false, ITER_FLAT, false>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<true, ITER_FLAT, true>(const IterLaunch&, int);
extern template hipError_t launch_iter_sites<true, ITER_FLAT, false>(const IterLaunch&, int);

namespace {

template <int G, int RES, int MODE>
hipError_t launch_either(const IterLaunch& L, bool mid) {
    return mid ? launch_one<G, RES, false, MODE, true>(L) : launch_one<G, RES, false, MODE, false>(L);
}

template <int MODE>
hipError_t launch_sites(const IterLaunch& L, bool coul, bool mid, int G) {
    if (coul) return mid ? launch_iter_sites<true, MODE, true>(L, G) : launch_iter_sites<true, MODE, false>(L, G);
    return mid ? launch_iter_sites<false, MODE, true>(L, G) : launch_iter_sites<false, MODE, false>(L, G);
}

}  // namespace

// LDS bytes of one workgroup that scans molecules of n_min to n_max sites
size_t scan_iter_lds(int n_min, int n_max, int G, bool mid, bool images) {
    return iter_site_bytes(images ? ITER_IMAGES : ITER_SITES) * (size_t)G *
           padded_share(n_max, G, images ? 1 : resident_sites(n_min, G, mid));
}

// n_blocks workgroups of W waves (W = 1 .. 8), G lanes a pixel column (4 ..
// 64; a force grid 8, periodic images 8 .. 64); coul: some site carries a
// charge; mode: ITER_*
hipError_t launch_scan_iter(const ScanArgs& a, int G, bool coul, int mode, int n_blocks, int W, int n_min, int n_max,
                            hipStream_t st) {
    if (W < 1 || W > 8) return hipErrorInvalidValue;
    const bool mid = a.minimiser != MAFM_MIN_SD && a.integrator == MAFM_INT_MIDPOINT;
    const IterLaunch L = {a, n_blocks, W, n_min, n_max, st};
    if (mode == ITER_GRID) return G == 8 ? launch_either<8, 2, ITER_GRID>(L, mid) : hipErrorInvalidValue;
    if (mode == ITER_IMAGES) {
        switch (G) {
            case 8: return launch_either<8, 1, ITER_IMAGES>(L, mid);
            case 16: return launch_either<16, 1, ITER_IMAGES>(L, mid);
            case 32: return launch_either<32, 1, ITER_IMAGES>(L, mid);
            case 64: return launch_either<64, 1, ITER_IMAGES>(L, mid);
            default: return hipErrorInvalidValue;
        }
    }
    return mode == ITER_FLAT ? launch_sites<ITER_FLAT>(L, coul, mid, G) : launch_sites<ITER_SITES>(L, coul, mid, G);
}

}  // namespace mafm
