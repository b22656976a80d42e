// mixed.cpp -- launcher of the run-time mixed-radix kernels (mixed_kernel.h).
#include <hip/hip_ext.h>

#include "mixed_table.h"

namespace gfftx {

static MixKernel kernel_of(const TileEntry& k) { return k.prec == PREC_F64 ? mixed_f64(k) : mixed_f32(k); }

hipError_t mixed_prepare(const TileEntry& k)
{
    if (k.lds_bytes <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel_of(k)), hipFuncAttributeMaxDynamicSharedMemorySize,
                               160 * 1024);
}

hipError_t launch_mixed(const TileEntry& k, const TileArgs& a, dim3 grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1,
                        const ChirpArgs* c)
{
    MixArgs x;
    x.a = a;
    x.m = *k.mix;
    x.c = c ? *c : ChirpArgs{};
    const MixKernel f = kernel_of(k);
    if (t0) hipExtLaunchKernelGGL(f, grid, dim3(k.wg), k.lds_bytes, s, t0, t1, 0, x);
    else hipLaunchKernelGGL(f, grid, dim3(k.wg), k.lds_bytes, s, x);
    return hipGetLastError();
}

}  // namespace gfftx
