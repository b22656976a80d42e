// mixed.hip -- instantiated run-time mixed-radix kernels (mixed_kernel.h) and their launcher.
#include <hip/hip_ext.h>

#include "registry.h"

namespace gfftx {

namespace {

typedef void (*MixKernel)(MixArgs);

template <typename T> MixKernel pick(const TileEntry& k)
{
    if (!k.loadT) {
        return k.real == REAL_POST ? mixed_kernel<T, MIX_EE, REAL_POST>
               : k.real == REAL_PRE ? mixed_kernel<T, MIX_EE, REAL_PRE>
                                    : mixed_kernel<T, MIX_EE, REAL_NONE>;
    }
    return k.storeT ? mixed_kernel<T, MIX_TT, REAL_NONE> : mixed_kernel<T, MIX_TE, REAL_NONE>;
}

MixKernel kernel_of(const TileEntry& k) { return k.prec == PREC_F64 ? pick<double>(k) : pick<float>(k); }

}  // namespace

hipError_t mixed_prepare(const TileEntry& k)
{
    if (k.lds_bytes <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel_of(k)), hipFuncAttributeMaxDynamicSharedMemorySize,
                               160 * 1024);
}

hipError_t launch_mixed(const TileEntry& k, const TileArgs& a, dim3 grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1)
{
    MixArgs x;
    x.a = a;
    x.m = *k.mix;
    const MixKernel f = kernel_of(k);
    if (t0) hipExtLaunchKernelGGL(f, grid, dim3(k.wg), k.lds_bytes, s, t0, t1, 0, x);
    else hipLaunchKernelGGL(f, grid, dim3(k.wg), k.lds_bytes, s, x);
    return hipGetLastError();
}

}  // namespace gfftx
