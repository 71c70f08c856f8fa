// FP64 kernel (fused_f64.h): rho alone, standard bases.
#include "fused_f64.h"

namespace okmi_fused {

int launch_f64_p0(const F64Args& a, hipStream_t st)
{
    return launch_f64_units<0, true, false, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(a, st);
}

}  // namespace okmi_fused
