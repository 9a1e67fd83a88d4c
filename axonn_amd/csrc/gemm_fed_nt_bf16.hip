// The forward's products on the small fed tiles, bfloat16 operands.
#include "gemm_fed_tiles.h"

namespace axn {
int launch_gemm_fed_nt_bf16(const GemmArgs& args, int epilogue, bool out_f32, EdgeTile tile, hipStream_t stream) {
  return launch_fed_nt<false>(args, epilogue, out_f32, tile, stream);
}
}  // namespace axn
