// MFMA GEMMs of shapes that are not made of whole tiles (ragged token counts, odd
// vocabularies, contractions that are not multiples of 64) and of operands of 2 GiB and more:
// solo_gemm with EDGE.  Included once per element type (gemm_edge_bf16.hip, gemm_edge_f16.hip:
// the instances of one type take as long to compile as all of gemm_bf16.hip).
//
// What bounds these: the same as the whole-tile kernels (MFMA issue and power), plus the work
// done for padding, at most one tile row and column.  They replaced a register-staged kernel
// (128 x 128 tiles, global -> VGPR -> LDS, one barrier per step, 32x32x16 MFMAs).  Measured on
// MI355X, bf16 unless stated, before -> after:
//   forward   777 x 14336 x 4096   165 -> 99 us (560 -> 920 TFLOP/s)
//   forward  3001 x 10240 x 2560   237 -> 166 us (fp16, fp32 result with bias)
//   backward of the same layer     468 -> 324 us (both products in one launch)
//   forward  2048 x 50264 x 2048   572 -> 355 us (740 -> 1190 TFLOP/s)
#pragma once
#include <atomic>

#include "gemm_solo.h"

namespace axn {
namespace {

template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32, bool HALF, bool ODD = false>
__global__ void __launch_bounds__(256) gemm_edge_kernel(const GemmArgs g) {
  solo_gemm<BM, BN, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, HALF, true, ODD>(g);
}

// Both gradients of a layer in one launch, as gemm_backward_kernel.  PARTS: the input gradient's contraction is
// in parts (fp32 partial products).
template <bool HALF, bool DW_F32, bool PARTS>
__global__ void __launch_bounds__(256) gemm_edge_backward_kernel(const GemmArgs gw, const GemmArgs gd) {
  const int b = (int)blockIdx.x;
  if (b >= gw.wg_first && b < gw.wg_first + gw.tiles_m * gw.tiles_n)
    solo_gemm<256, 256, false, false, AXN_EPI_NONE, DW_F32, HALF, true>(gw);
  else
    solo_gemm<256, 256, true, false, AXN_EPI_NONE, PARTS, HALF, true>(gd);
}

template <int BM, int BN, bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF, bool ODD = false>
int launch_edge_tile(const GemmArgs& in, hipStream_t stream) {
  // Only the forward's output rows can be odd (the others have the width of an input); those of heads over
  // vocabularies are, which have neither bias nor activation.  Up to 80 rows, few of a tile, the exchange costs what
  // the stores gain (us, plain / so: 78 x 1013, 448 6.6 / 7.3, 70 x 688, 1192 10.4 / 11.0; 65 to 80 rows 1.02 of the
  // time on average up to contractions of 1200 and 1.00 beyond, 81 to 96 rows 1.00, 113 to 128 0.94).
  if constexpr (!ODD && AK && BKM && EPI == AXN_EPI_NONE && !OUT_F32)
    if (in.ldc % 2 != 0 && !in.beta && in.M > 80) return launch_edge_tile<BM, BN, AK, BKM, EPI, OUT_F32, HALF, true>(in, stream);
  GemmArgs g = in;
  g.tiles_m = (int)ceil_div(g.M, BM);
  g.tiles_n = (int)ceil_div(g.N, BN);
  const long long nwg = (long long)g.tiles_m * g.tiles_n * (g.splits > 1 ? g.splits : 1);
  if (nwg > 0x7fffffffLL) {
    set_error("gemm: too many output tiles (%lld)", nwg);
    return AXN_ELIMIT;
  }
  constexpr size_t lds = 5 * BM * 64 * 2;   // five slots of the A tile's size
  void (*kern)(const GemmArgs) = gemm_edge_kernel<BM, BN, AK, BKM, EPI, OUT_F32, HALF, ODD>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(256), lds, stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_edge_kind(const GemmArgs& g, EdgeTile tile, hipStream_t stream) {
  if (tile == EDGE_128x128) return launch_edge_tile<128, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
  if (tile == EDGE_256x128) return launch_edge_tile<256, 128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
  return launch_edge_tile<256, 256, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
}

template <bool HALF>
int launch_edge_layout(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32, EdgeTile tile,
                       hipStream_t stream) {
  switch (layout) {
    case GEMM_NT:
      if (out_f32) {
        if (epilogue == AXN_EPI_NONE && g.splits > 1)   // partial products
          return launch_edge_kind<true, true, AXN_EPI_NONE, true, HALF>(g, tile, stream);
        if (epilogue == AXN_EPI_BIAS) return launch_edge_kind<true, true, AXN_EPI_BIAS, true, HALF>(g, tile, stream);
        if (epilogue == AXN_EPI_BIAS_GELU)
          return launch_edge_kind<true, true, AXN_EPI_BIAS_GELU, true, HALF>(g, tile, stream);
        break;
      }
      switch (epilogue) {
        case AXN_EPI_NONE:
          return launch_edge_kind<true, true, AXN_EPI_NONE, false, HALF>(g, tile, stream);
        case AXN_EPI_BIAS:
          return launch_edge_kind<true, true, AXN_EPI_BIAS, false, HALF>(g, tile, stream);
        case AXN_EPI_BIAS_GELU:
          return launch_edge_kind<true, true, AXN_EPI_BIAS_GELU, false, HALF>(g, tile, stream);
        case AXN_EPI_GELU:
          return launch_edge_kind<true, true, AXN_EPI_GELU, false, HALF>(g, tile, stream);
      }
      break;
    case GEMM_NN:
      if (epilogue != AXN_EPI_NONE || (out_f32 && g.splits <= 1)) break;
      if (out_f32) return launch_edge_kind<true, false, AXN_EPI_NONE, true, HALF>(g, tile, stream);
      return launch_edge_kind<true, false, AXN_EPI_NONE, false, HALF>(g, tile, stream);
    case GEMM_TN:
      if (epilogue != AXN_EPI_NONE) break;
      return out_f32 ? launch_edge_kind<false, false, AXN_EPI_NONE, true, HALF>(g, tile, stream)
                     : launch_edge_kind<false, false, AXN_EPI_NONE, false, HALF>(g, tile, stream);
  }
  set_error("gemm: unsupported layout/epilogue/output combination");
  return AXN_EINVAL;
}

template <bool HALF, bool DW_F32, bool PARTS>
int launch_edge_backward_kind(const GemmArgs& gw, const GemmArgs& gd, hipStream_t stream) {
  constexpr size_t lds = 5 * 256 * 64 * 2;
  void (*kern)(const GemmArgs, const GemmArgs) = gemm_edge_backward_kernel<HALF, DW_F32, PARTS>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  const unsigned nwg = (unsigned)(gw.tiles_m * gw.tiles_n + gd.tiles_m * gd.tiles_n * (PARTS ? gd.splits : 1));
  hipLaunchKernelGGL(kern, dim3(nwg), dim3(256), lds, stream, gw, gd);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <bool HALF>
int launch_edge_backward(const GemmArgs& gw, const GemmArgs& gd, bool dw_f32, hipStream_t stream) {
  if (gd.splits > 1)
    return dw_f32 ? launch_edge_backward_kind<HALF, true, true>(gw, gd, stream)
                  : launch_edge_backward_kind<HALF, false, true>(gw, gd, stream);
  return dw_f32 ? launch_edge_backward_kind<HALF, true, false>(gw, gd, stream)
                : launch_edge_backward_kind<HALF, false, false>(gw, gd, stream);
}

}  // namespace
}  // namespace axn
