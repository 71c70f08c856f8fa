// FP64 fused density kernel (fused_f64.h): rho, rho and first derivatives.
#include "fused_f64.h"

namespace okmi_fused {
namespace {

// mo_norm[m] += sum over tiles of part[tile][m], m < nmo: one workgroup per
// MO, each thread a fixed stride of tiles, then a tree in LDS (the order of
// the additions does not depend on timing)
__global__ void k_norm_reduce(const double* part, int64_t ntile, int mpad, int nmo, double* mo_norm)
{
    __shared__ double red[256];
    const int m = blockIdx.x;
    double s = 0.0;
    for (int64_t t = threadIdx.x; t < ntile; t += 256) s += part[t * mpad + m];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0 && m < nmo) mo_norm[m] += red[0];
}

}  // namespace

int launch_norm_reduce(const double* part, int64_t ntile, int mpad, int nmo, double* mo_norm, hipStream_t st)
{
    if (ntile <= 0 || nmo <= 0) return 0;
    hipLaunchKernelGGL(k_norm_reduce, dim3((unsigned)nmo), dim3(256), 0, st, part, ntile, mpad, nmo, mo_norm);
    return 0;
}

int launch_pass_f64(const F64Args& a, int pass, int mpad, bool standard, hipStream_t st)
{
    switch (pass) {
    case 0: return standard ? launch_f64_u<0, true>(a, mpad / 4, st) : launch_f64_u<0, false>(a, mpad / 4, st);
    case 1: return standard ? launch_f64_u<1, true>(a, mpad / 4, st) : launch_f64_u<1, false>(a, mpad / 4, st);
    default: return launch_pass_f64_d2(a, pass, mpad, standard, st);
    }
}

}  // namespace okmi_fused
