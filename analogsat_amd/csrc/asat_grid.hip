// The kernels of the few-workgroup persistent integrator (asat_grid.h), in a
// file of their own for its compile flags.
#include "asat_grid.h"

namespace asat {

template <typename T, int KT>
static const void* grid_kernel_of(int cpt)
{
    if (cpt == 1) return (const void*)k_grid<T, KT, 1>;
    if (cpt == 2) return (const void*)k_grid<T, KT, 2>;
    if (cpt == 4) return (const void*)k_grid<T, KT, 4>;
    if constexpr (sizeof(T) == 4) {
        if (cpt == 8) return (const void*)k_grid<T, KT, 8>;
    }
    return nullptr;
}

const void* grid_kernel(int precision, int k, int cpt)
{
    if (precision == ASAT_F64) return k == 3 ? grid_kernel_of<double, 3>(cpt) : grid_kernel_of<double, 4>(cpt);
    return k == 3 ? grid_kernel_of<float, 3>(cpt) : grid_kernel_of<float, 4>(cpt);
}

}  // namespace asat
