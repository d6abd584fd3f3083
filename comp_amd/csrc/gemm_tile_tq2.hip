// The tiled matrix-core GEMM's TQ2_0 instantiations (gemm_tile.h).
#include "gemm_tile.h"

namespace komp {

hipError_t launch_gemm_tile_tq2(const GemmCall& c, const TilePlan& p, hipStream_t stream) {
  return gemm_tile::launch_fmt<FMT_TQ2_0>(c, p, stream);
}

}  // namespace komp
