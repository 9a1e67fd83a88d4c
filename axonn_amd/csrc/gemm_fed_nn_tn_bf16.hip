// The gradients' products on the small fed tiles, bfloat16 operands.
#include "gemm_fed_tiles.h"

namespace axn {
int launch_gemm_fed_nn_tn_bf16(GemmLayout layout, const GemmArgs& args, bool out_f32, EdgeTile tile, hipStream_t stream) {
  return launch_fed_nn_tn<false>(layout, args, out_f32, tile, stream);
}
}  // namespace axn
