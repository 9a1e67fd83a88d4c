// MFMA GEMMs of outputs that small tiles cover in one round of workgroups or two: fed_gemm on the tiles FED_*, any M, N,
// contraction and operand size.  Included once per element type and operand order (the instances of one take as long to
// compile as all of gemm_edge_bf16.hip).
#pragma once
#include <atomic>

#include "gemm_fed.h"

namespace axn {
namespace {

template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32, bool HALF, bool ODD>
__global__ void __launch_bounds__(512) gemm_fed_edge_kernel(const GemmArgs g) {
  fed_gemm<BM, BN, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, HALF, true, ODD>(g);
}

template <int BM, int BN, bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF, bool ODD = false>
int launch_fed(const GemmArgs& in, hipStream_t stream) {
  // odd output rows: as launch_edge_tile
  if constexpr (!ODD && AK && BKM && EPI == AXN_EPI_NONE && !OUT_F32)
    if (in.ldc % 2 != 0 && !in.beta && in.M > 80) return launch_fed<BM, BN, AK, BKM, EPI, OUT_F32, HALF, true>(in, stream);
  GemmArgs g = in;
  g.tiles_m = (int)ceil_div(g.M, BM);
  g.tiles_n = (int)ceil_div(g.N, BN);
  void (*kern)(const GemmArgs) = gemm_fed_edge_kernel<BM, BN, AK, BKM, EPI, OUT_F32, HALF, ODD>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, kFedLds<BM, BN>, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  const long long nwg = (long long)g.tiles_m * g.tiles_n * (g.splits > 1 ? g.splits : 1);
  hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(512), (kFedLds<BM, BN>), stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_fed_tile(const GemmArgs& g, EdgeTile tile, hipStream_t stream) {
  switch (tile) {
    case FED_64x64: return launch_fed<64, 64, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_96x64: return launch_fed<96, 64, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_64x128: return launch_fed<64, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_96x128: return launch_fed<96, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_128x128: return launch_fed<128, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_96x192: return launch_fed<96, 192, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_128x192: return launch_fed<128, 192, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_160x192: return launch_fed<160, 192, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_128x256: return launch_fed<128, 256, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    case FED_256x128: return launch_fed<256, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
    default: break;
  }
  set_error("gemm: no such tile");
  return AXN_EINVAL;
}

template <bool HALF>
int launch_fed_nt(const GemmArgs& g, int epilogue, bool out_f32, EdgeTile tile, hipStream_t stream) {
  if (out_f32) {
    if (epilogue == AXN_EPI_NONE && g.splits > 1)   // partial products
      return launch_fed_tile<true, true, AXN_EPI_NONE, true, HALF>(g, tile, stream);
    if (epilogue == AXN_EPI_BIAS) return launch_fed_tile<true, true, AXN_EPI_BIAS, true, HALF>(g, tile, stream);
    if (epilogue == AXN_EPI_BIAS_GELU) return launch_fed_tile<true, true, AXN_EPI_BIAS_GELU, true, HALF>(g, tile, stream);
  } else {
    switch (epilogue) {
      case AXN_EPI_NONE: return launch_fed_tile<true, true, AXN_EPI_NONE, false, HALF>(g, tile, stream);
      case AXN_EPI_BIAS: return launch_fed_tile<true, true, AXN_EPI_BIAS, false, HALF>(g, tile, stream);
      case AXN_EPI_BIAS_GELU: return launch_fed_tile<true, true, AXN_EPI_BIAS_GELU, false, HALF>(g, tile, stream);
      case AXN_EPI_GELU: return launch_fed_tile<true, true, AXN_EPI_GELU, false, HALF>(g, tile, stream);
    }
  }
  set_error("gemm: unsupported layout/epilogue/output combination");
  return AXN_EINVAL;
}

template <bool HALF>
int launch_fed_nn_tn(GemmLayout layout, const GemmArgs& g, bool out_f32, EdgeTile tile, hipStream_t stream) {
  if (layout == GEMM_NN)
    return out_f32 ? launch_fed_tile<true, false, AXN_EPI_NONE, true, HALF>(g, tile, stream)
                   : launch_fed_tile<true, false, AXN_EPI_NONE, false, HALF>(g, tile, stream);
  return out_f32 ? launch_fed_tile<false, false, AXN_EPI_NONE, true, HALF>(g, tile, stream)
                 : launch_fed_tile<false, false, AXN_EPI_NONE, false, HALF>(g, tile, stream);
}

}  // namespace
}  // namespace axn
