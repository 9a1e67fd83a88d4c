// The gate and up projection of a gated MLP with their activation, silu(A B^T) * (A B2^T), in one launch for any number
// of rows: solo_gemm and fed_gemm with the gate/up epilogue and bounds.
//
// What bounds it: the same as any product of twice the columns.  What it saves against two products and the activation:
// a launch's ramp and last round (777 rows x 14336: 224 tiles of 256 x 256 each, 256 CUs), the activation's pass over
// both, and where nothing is saved for a backward pass the writing of both.  us, two products and the activation / this,
// operands from HBM: 777 x 14336 over 4096 188 / 161, 300 x 11008 over 4096 94 / 74, 150 x 8192 over 3072 50 / 38,
// 1000 x 4096 over 1024 34 / 22, 4000 x 10752 over 3072 477 / 393.  What it loses is the parts of a long contraction over few
// tiles (74 x 512 over 7752 30 / 71): callers leave those to two products (584 of 700 layers are taken, 0.73 of the time
// on average, 1.15 at worst).
#include <atomic>

#include "gemm_fed.h"

namespace axn {
namespace {

constexpr bool gate_up_is_fed(int bm, int bn) { return bm * bn <= 256 * 128; }

template <int BM, int BN, bool HALF>
__global__ void __launch_bounds__(gate_up_is_fed(BM, BN) ? 512 : 256) gemm_gate_up_edge_kernel(const GemmArgs g) {
  if constexpr (gate_up_is_fed(BM, BN)) fed_gemm<BM, BN, true, true, EPI_SWIGLU, false, HALF>(g);
  else solo_gemm<BM, BN, true, true, EPI_SWIGLU, false, HALF, true>(g);
}

template <int BM, int BN, bool HALF>
int launch_tile(const GemmArgs& in, hipStream_t stream) {
  constexpr bool fed = gate_up_is_fed(BM, BN);
  constexpr size_t lds = fed ? kFedLds<BM, BN> : 163840;
  GemmArgs g = in;
  g.tiles_m = (int)ceil_div(g.M, BM);
  g.tiles_n = (int)ceil_div(g.N, BN / 2);
  g.splits = 0;
  const long long nwg = (long long)g.tiles_m * g.tiles_n;
  if (nwg > 0x7fffffffLL) {
    set_error("gemm_swiglu: too many output tiles (%lld)", nwg);
    return AXN_ELIMIT;
  }
  void (*kern)(const GemmArgs) = gemm_gate_up_edge_kernel<BM, BN, HALF>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(fed ? 512 : 256), lds, stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// Tiles (rows, and columns of gate and up together) and their estimated time in us: a round of workgroups, a stage of
// it, a megabyte of operands (with a workgroup on every CU) and one of output.  Fitted to those 160 layers on every tile,
// 5 to 9 % rms; the pick has the time of the best tile (0.728 of the separate path's against 0.728).
struct GateUpTile {
  int bm, bn;
  float round, stage, operands, output;
  int (*launch[2])(const GemmArgs&, hipStream_t);
};
#define TILE(BM, BN, ROUND, STAGE, OPERANDS, OUTPUT) \
  {BM, BN, ROUND, STAGE, OPERANDS, OUTPUT, {launch_tile<BM, BN, false>, launch_tile<BM, BN, true>}}
constexpr GateUpTile kTiles[] = {
    TILE(256, 256, 3.93f, 1.199f, 0.007f, 0.37f), TILE(224, 256, 2.68f, 1.084f, 0.018f, 0.47f),
    TILE(192, 256, 2.99f, 1.009f, 0.024f, 0.32f), TILE(128, 256, 1.76f, 0.728f, 0.036f, 0.69f),
    TILE(128, 128, 1.73f, 0.461f, 0.057f, 0.82f), TILE(96, 128, 2.56f, 0.388f, 0.064f, 0.42f),
    TILE(64, 128, 1.97f, 0.315f, 0.100f, 0.58f),
};
#undef TILE

double tile_microseconds(const GateUpTile& t, const GemmArgs& g) {
  const long long w = ceil_div(g.M, t.bm) * ceil_div(g.N, t.bn / 2);
  const double rounds = (double)((w + 255) / 256), occupied = w >= 256 ? 1.0 : (double)w / 256;
  const double mb = ((double)g.M + 2.0 * (double)g.N) * (double)g.Kc * 2e-6;
  const double lines = g.Kc % 64 != 0 ? 1.3 : 1.0;   // rows that do not fill 128-byte lines
  return rounds * (t.round + t.stage * lines * (double)ceil_div(g.Kc, 64)) + t.operands * mb / occupied +
         t.output * (double)g.M * (double)g.N * 2e-6;
}

}  // namespace

int launch_gemm_swiglu_any(const GemmArgs& g, bool half, bool unless_largest, hipStream_t stream, bool& taken) {
  taken = true;
  if ((g.lda > g.ldb ? g.lda : g.ldb) >= kEdgeMaxLd / 2) {
    set_error("gemm_swiglu: row strides below %lld elements expected", (long long)(kEdgeMaxLd / 2));
    return AXN_ESHAPE;
  }
  const GateUpTile* best = kTiles;
  double us = tile_microseconds(*best, g) * (unless_largest ? 0.95 : 1.0);
  for (const GateUpTile& t : kTiles) {
    const double e = tile_microseconds(t, g);
    if (e < us) {
      us = e;
      best = &t;
    }
  }
  if (unless_largest && best == kTiles) {
    taken = false;
    return AXN_OK;
  }
  return best->launch[half ? 1 : 0](g, stream);
}

}  // namespace axn
