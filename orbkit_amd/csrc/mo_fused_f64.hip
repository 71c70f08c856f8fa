// FP64 kernel (fused_f64.h) with the MO values stored instead of reduced.
#include "fused_f64.h"

namespace okmi_fused {

int launch_mo_f64(const F64Args& a, int pass, bool standard, hipStream_t st)
{
    if (!standard) {
        switch (pass) {
        case 0: return launch_f64_units<0, false, true, 4, 8, 12, 16>(a, st);
        case 1: return launch_f64_units<1, false, true, 4, 8, 12, 16>(a, st);
        case 2: return launch_f64_units<2, false, true, 4, 8, 12, 16>(a, st);
        default: return launch_f64_units<3, false, true, 4, 8, 12, 16>(a, st);
        }
    }
    switch (pass) {
    case 0: return launch_f64_units<0, true, true, 1, 2, 4, 6, 8, 10, 12, 14, 16>(a, st);
    case 1: return launch_f64_units<1, true, true, 1, 2, 4, 6, 8, 10, 12, 14, 16>(a, st);
    case 2: return launch_f64_units<2, true, true, 4, 8, 12, 16>(a, st);
    default: return launch_f64_units<3, true, true, 4, 8, 12, 16>(a, st);
    }
}

}  // namespace okmi_fused
