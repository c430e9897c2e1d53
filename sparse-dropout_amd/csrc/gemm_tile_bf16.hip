// The tile kernels for bf16 operands.
#include "gemm_tile_launch.h"

namespace sd {
SD_TILE_INSTANCES(BF16)
}  // namespace sd
