// The prefill kernel's variants on 96 x 128 tiles (a file per tile shape, so that
// they compile side by side).
#include "qmm_kernel.hpp"

namespace eq {

bool qmm_run_t31(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups,
                 hipStream_t st) {
    return qmm_run_tile<3, 1>(bits, gs, scale_dtype, x_dtype, pw, a, workgroups, st);
}

}  // namespace eq
