// Weight gradients over few tokens: fed_gemm by workgroups that stay, one on a CU, and take a tile of every round.
//
// What bounds them on other kernels: a tile is 5 to 13 stages, about 0.7 us each, and its ramp (2 to 3 us until the first
// stage has come from HBM) and its stores are as long again.  Here the copying waves go on to the next tile's stages while
// the matrix waves store.  us (tokens x out x in), the other kernels / this: 447 x 12288 x 2048 44.7 / 34.3, 404 x 9600 x
// 2368 40.7 / 32.0, 320 x 16384 x 3584 64.2 / 59.8; where rounds_tile leaves it out 512 x 8192 x 3584 42.5 / 49.2, 1000 x
// 8192 x 3584 63.2 / 75.8.
// 128 x 128 and 160 x 192 tiles are behind these two (404 to 1014 tokens: 0 to 25 %).  The sums' order is the same.
#include <atomic>

#include "gemm_fed.h"

namespace axn {
namespace {

template <int BM, int BN, bool HALF>
__global__ void __launch_bounds__(512) gemm_fed_rounds_kernel(const GemmArgs g) {
  fed_gemm<BM, BN, false, false, AXN_EPI_NONE, false, HALF, true, false, true>(g);
}

template <int BM, int BN, bool HALF>
int launch_rounds(const GemmArgs& in, hipStream_t stream) {
  GemmArgs g = in;
  g.tiles_m = (int)ceil_div(g.M, BM);
  g.tiles_n = (int)ceil_div(g.N, BN);
  g.splits = 0;
  void (*kern)(const GemmArgs) = gemm_fed_rounds_kernel<BM, BN, HALF>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, kFedLds<BM, BN>, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  const int tiles = g.tiles_m * g.tiles_n;   // (rounds_tile: 65536 at most)
  hipLaunchKernelGGL(kern, dim3(tiles < 256 ? tiles : 256), dim3(512), (kFedLds<BM, BN>), stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

}  // namespace

int launch_gemm_fed_rounds(const GemmArgs& g, bool half, EdgeTile tile, hipStream_t stream) {
  if (g.N % 8 != 0 || g.ldc % 8 != 0) {   // the epilogue has no LDS for columns behind the last multiple of 8
    set_error("gemm_fed_rounds: rows of whole, aligned vectors expected (got N=%d, ldc=%lld)", g.N, (long long)g.ldc);
    return AXN_ESHAPE;
  }
  if (tile == FED_128x256) return half ? launch_rounds<128, 256, true>(g, stream) : launch_rounds<128, 256, false>(g, stream);
  return half ? launch_rounds<256, 128, true>(g, stream) : launch_rounds<256, 128, false>(g, stream);
}

}  // namespace axn
