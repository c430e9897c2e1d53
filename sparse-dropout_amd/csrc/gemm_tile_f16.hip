// The tile kernels for fp16 operands.
#include "gemm_tile_launch.h"

namespace sd {
SD_TILE_INSTANCES(F16)

int tile_threads(int shape) {
  return shape == kShapeOne ? FwdOne::THREADS : (shape == kShapeQuad ? FwdQuad::THREADS : FwdWide::THREADS);
}
}  // namespace sd
