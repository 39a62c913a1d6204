// Pipelined GEMM kernels, complex double (the shapes of shape_info).
#include "gemm_plan.hpp"

namespace dmrg {
namespace pipe {

void launch_c128(const Launch &l, Shape s, dim3 grid, hipStream_t st) {
    switch(s) {
        case S64x64: launch_shape<double, true, 64, 64, 8, 2, 2, 4>(l, grid, st); break;
        case S64x32: launch_shape<double, true, 64, 32, 16, 2, 2, 3>(l, grid, st); break;
        case S32x32: launch_shape<double, true, 32, 32, 8, 2, 2, 4>(l, grid, st); break;
        default: throw Error(DMRG_ERR_ARG, "no such tile shape");
    }
}

void launch_grouped_c128(const Desc *d, const int *start, int n, int tiles, Shape s, hipStream_t st) {
    switch(s) {
        case S64x64: launch_grouped_shape<double, true, 64, 64, 8, 2, 2, 4>(d, start, n, tiles, st); break;
        case S32x32: launch_grouped_shape<double, true, 32, 32, 8, 2, 2, 4>(d, start, n, tiles, st); break;
        default: throw Error(DMRG_ERR_ARG, "no such grouped tile shape");
    }
}

} // namespace pipe
} // namespace dmrg
