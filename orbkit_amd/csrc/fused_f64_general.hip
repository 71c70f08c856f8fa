// FP64 kernel (fused_f64.h): bases with l = 4 or general row maps.
#include "fused_f64.h"

namespace okmi_fused {

int launch_f64_general(const F64Args& a, int pass, hipStream_t st)
{
    switch (pass) {
    case 0: return launch_f64_units<0, false, false, 4, 8, 12, 16>(a, st);
    case 1: return launch_f64_units<1, false, false, 4, 8, 12, 16>(a, st);
    case 2: return launch_f64_units<2, false, false, 4, 8, 12, 16>(a, st);
    case 3: return launch_f64_units<3, false, false, 4, 8, 12, 16>(a, st);
    default: return launch_f64_units<4, false, false, 4, 8, 9, 10>(a, st);
    }
}

}  // namespace okmi_fused
