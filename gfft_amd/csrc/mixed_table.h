// mixed_table.h -- the run-time mixed-radix kernel of a tile: one translation unit per precision
// (mixed_f32.hip, mixed_f64.hip) instantiates them.
#pragma once
#include "registry.h"

namespace gfftx {

typedef void (*MixKernel)(MixArgs);

template <typename T> inline MixKernel mixed_pick(const TileEntry& k)
{
    if (!k.loadT) {
        return k.real == CHIRP_ALL ? mixed_kernel<T, MIX_EE, CHIRP_ALL>
               : k.real == REAL_POST ? mixed_kernel<T, MIX_EE, REAL_POST>
               : k.real == REAL_PRE ? mixed_kernel<T, MIX_EE, REAL_PRE>
                                    : mixed_kernel<T, MIX_EE, REAL_NONE>;
    }
    if (k.storeT) return k.real == CHIRP_OUT ? mixed_kernel<T, MIX_TT, CHIRP_OUT> : mixed_kernel<T, MIX_TT, REAL_NONE>;
    return k.real == CHIRP_IN     ? mixed_kernel<T, MIX_TE, CHIRP_IN>
           : k.real == CHIRP_TURN ? mixed_kernel<T, MIX_TE, CHIRP_TURN>
                                  : mixed_kernel<T, MIX_TE, REAL_NONE>;
}

MixKernel mixed_f32(const TileEntry& k);
MixKernel mixed_f64(const TileEntry& k);

}  // namespace gfftx
