// bf16 GEMM kernels for operands at any element address, 64x64 tile, 2x2 waves: all four loader pairs.
#include "agh_gemm_bf16_dl_launch.h"

namespace agh {
namespace gemm {
AGH_ANY_INSTANTIATE(64, 64, 2, 2)
}  // namespace gemm
}  // namespace agh
