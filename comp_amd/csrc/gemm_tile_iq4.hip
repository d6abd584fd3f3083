// The tiled matrix-core GEMM's IQ4_NL instantiations (gemm_tile.h).
#include "gemm_tile.h"

namespace komp {

hipError_t launch_gemm_tile_iq4(const GemmCall& c, const TilePlan& p, hipStream_t stream) {
  return gemm_tile::launch_fmt<FMT_IQ4_NL>(c, p, stream);
}

}  // namespace komp
