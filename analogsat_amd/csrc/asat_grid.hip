// The kernels of the few-workgroup persistent integrator (asat_grid.h), in a
// file of their own for its compile flags.
#include "asat_grid.h"

namespace asat {

template <typename T, int KT, bool SOLO>
static const void* grid_kernel_of(int cpt)
{
    if (cpt == 1) return (const void*)k_grid<T, KT, 1, SOLO>;
    if (cpt == 2) return (const void*)k_grid<T, KT, 2, SOLO>;
    if constexpr (!SOLO || sizeof(T) == 4) {
        if (cpt == 4) return (const void*)k_grid<T, KT, 4, SOLO>;
    }
    if constexpr (!SOLO && sizeof(T) == 4) {
        if (cpt == 8) return (const void*)k_grid<T, KT, 8, SOLO>;
    }
    return nullptr;
}

template <typename T, bool SOLO>
static const void* grid_kernel_k(int k, int cpt)
{
    return k == 3 ? grid_kernel_of<T, 3, SOLO>(cpt) : grid_kernel_of<T, 4, SOLO>(cpt);
}

const void* grid_kernel(int precision, int k, int cpt, bool solo)
{
    if (precision == ASAT_F64) return solo ? grid_kernel_k<double, true>(k, cpt) : grid_kernel_k<double, false>(k, cpt);
    return solo ? grid_kernel_k<float, true>(k, cpt) : grid_kernel_k<float, false>(k, cpt);
}

}  // namespace asat
