// mixed_f32.hip -- run-time mixed-radix kernels (mixed_kernel.h) in FP32.
#include "mixed_table.h"

namespace gfftx {

MixKernel mixed_f32(const TileEntry& k) { return mixed_pick<float>(k); }

}  // namespace gfftx
