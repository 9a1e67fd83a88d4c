// The forward's products on the small fed tiles, half operands.
#include "gemm_fed_tiles.h"

namespace axn {
int launch_gemm_fed_nt_f16(const GemmArgs& args, int epilogue, bool out_f32, EdgeTile tile, hipStream_t stream) {
  return launch_fed_nt<true>(args, epilogue, out_f32, tile, stream);
}
}  // namespace axn
