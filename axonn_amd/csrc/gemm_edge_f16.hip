// Edge-capable GEMMs on IEEE half operands (see gemm_edge.h).
#include "gemm_edge.h"

namespace axn {

int launch_gemm_edge_f16(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32, EdgeTile tile,
                         hipStream_t stream) {
  return launch_edge_layout<true>(layout, g, epilogue, out_f32, tile, stream);
}
int launch_gemm_edge_backward_f16(const GemmArgs& gw, const GemmArgs& gd, bool dw_f32, hipStream_t stream) {
  return launch_edge_backward<true>(gw, gd, dw_f32, stream);
}

}  // namespace axn
