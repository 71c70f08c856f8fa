// FP64 fused density kernel (fused_f64.h): the passes with second derivatives.
#include "fused_f64.h"

namespace okmi_fused {

int launch_pass_f64_d2(const F64Args& a, int pass, int mpad, bool standard, hipStream_t st)
{
    switch (pass) {
    case 2: return standard ? launch_f64_u<2, true>(a, mpad / 4, st) : launch_f64_u<2, false>(a, mpad / 4, st);
    case 3: return standard ? launch_f64_u<3, true>(a, mpad / 4, st) : launch_f64_u<3, false>(a, mpad / 4, st);
    default: return standard ? launch_f64_u<4, true>(a, mpad / 4, st) : launch_f64_u<4, false>(a, mpad / 4, st);
    }
}

}  // namespace okmi_fused
