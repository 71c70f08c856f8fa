// FP64 kernel (fused_f64.h): the halves of second derivatives, standard bases.
#include "fused_f64.h"

namespace okmi_fused {

int launch_f64_p23(const F64Args& a, int pass, hipStream_t st)
{
    return pass == 2 ? launch_f64_units<2, true, false, 4, 8, 12, 16>(a, st)
                     : launch_f64_units<3, true, false, 4, 8, 12, 16>(a, st);
}

}  // namespace okmi_fused
