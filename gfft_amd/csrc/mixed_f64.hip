// mixed_f64.hip -- run-time mixed-radix kernels (mixed_kernel.h) in FP64.
#include "mixed_table.h"

namespace gfftx {

MixKernel mixed_f64(const TileEntry& k) { return mixed_pick<double>(k); }

}  // namespace gfftx
