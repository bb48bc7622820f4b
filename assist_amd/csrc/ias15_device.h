// IAS15 tables and device helpers shared by the integration kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "ias15_tables.h"
#include "kernels.h"

namespace assist_gpu {

static __constant__ double cH[8] = IAS15_H_INIT;
static __constant__ double cRRI[28] = IAS15_RRINV_INIT;
static __constant__ double cC[21] = IAS15_C_INIT;
static __constant__ double cD[21] = IAS15_D_INIT;
static __constant__ double cPX[9 * 8] = IAS15_PX_INIT;
static __constant__ double cPV[9 * 7] = IAS15_PV_INIT;

// Kernel-argument pointer (constant address space, so loads through it are scalar loads; the
// host compilation pass only type-checks the kernel body, with a plain pointer).
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const IntegrateArgs* KArgs;
#else
typedef const IntegrateArgs* KArgs;
#endif
__device__ __forceinline__ KArgs launder(KArgs p) {
    asm volatile("" : "+s"(p));
    return p;
}

__device__ __forceinline__ void add_cs(double& p, double& cs, double in) {
    const double y = in - cs;
    const double t = p + y;
    cs = (t - p) - y;
    p = t;
}

// Re-expansion of the last accepted step's b (br) for a step of ratio q:
// e = Q(q) br (Taylor re-centring at h = 1, scaled by q^k); b = e + (br - er).
__device__ __forceinline__ void predict_e(const double br[7], double q, double e[7]) {
    const double q2 = q * q, q3 = q * q2, q4 = q2 * q2, q5 = q2 * q3, q6 = q3 * q3, q7 = q3 * q4;
    e[0] = q * (br[6] * 7.0 + br[5] * 6.0 + br[4] * 5.0 + br[3] * 4.0 + br[2] * 3.0 + br[1] * 2.0 + br[0]);
    e[1] = q2 * (br[6] * 21.0 + br[5] * 15.0 + br[4] * 10.0 + br[3] * 6.0 + br[2] * 3.0 + br[1]);
    e[2] = q3 * (br[6] * 35.0 + br[5] * 20.0 + br[4] * 10.0 + br[3] * 4.0 + br[2]);
    e[3] = q4 * (br[6] * 35.0 + br[5] * 15.0 + br[4] * 5.0 + br[3]);
    e[4] = q5 * (br[6] * 21.0 + br[5] * 6.0 + br[4]);
    e[5] = q6 * (br[6] * 7.0 + br[5]);
    e[6] = q7 * br[6];
}

}  // namespace assist_gpu
