// bf16 MFMA GEMM for gfx950 (MI355X): the three shard GEMMs of the
// tensor-parallel Linear layer,
//   forward  Y  = X  W^T   (axonn/intra_layer/fully_connected.py:118)
//   dgrad    dX = dY W     (fully_connected.py:140)
//   wgrad    dW = dY^T X   (fully_connected.py:147-151)
// templated over the operand storage orders: an operand is "K-major" when the
// contraction index is contiguous in memory ([rows][Kc]) and "MN-major" when it
// is strided ([Kc][rows]).  No transposed copy of an operand is ever made.
//
//   * fp32 accumulation in registers; a workgroup owns a BM x BN output tile and
//     walks the contraction through LDS tiles.
//   * LDS layouts per storage order such that fragment reads are free of bank
//     conflicts on the 64-bank LDS; MN-major tiles are read with the transposing
//     ds_read_b64_tr_b16.
//   * The MFMA is issued with the operands swapped (D^T = B^T A^T), so that a lane
//     holds consecutive output columns of a row and writes 16 contiguous bytes.
//   * Workgroup ids are remapped so that each of the 8 XCDs (private L2 each)
//     works on a compact block of neighbouring tiles.
//
// One-wave-per-SIMD kernels (solo_gemm: gemm_*_solo_kernel at 256 x 256 and 128 x 128
// tiles, gemm_*_rest_kernel at 256 x 128, gemm_*_swiglu_kernel; shapes made of whole
// tiles, contraction % 64 == 0, operands below 2 GiB): 4 waves, one per SIMD, each a
// quarter of the tile on v_mfma_f32_16x16x32_{bf16,f16}; operand tiles go global -> LDS
// directly (buffer loads to LDS, 16 bytes per lane, no registers) into a ring of five
// 64-deep tiles; each wave pipelines its share of the copies and its LDS fragment reads
// between its own MFMAs; a permuted row order of the column operand's fragments leaves
// a lane with 8 consecutive output columns, stored straight from the accumulators.
// launch_shape / launch_whole choose the tile and cut a problem whose last round of
// large tiles would be at most half full into full rounds and a rest; a workspace
// variant splits the contraction of problems with few tiles over workgroups; the
// gate/up forward of a gated MLP gathers its column operand from two weight matrices
// and applies silu(gate) * up in the epilogue.
//
// Kernels with copying waves of their own (fed_gemm: the tiles of gemm_fed_tiles.h): rests, and outputs that small
// tiles cover in one round of workgroups or two, of any shape (fed_tile, gemm_plan).
//
// Everything else (ragged shapes, contractions that are not multiples of 64, operands of
// 2 GiB and more) runs on the same main loop with bounds: gemm_edge.h.
#include <atomic>
#include <cmath>
#include <functional>
#include <queue>
#include <vector>

#include "gemm_solo.h"

namespace axn {
namespace {

template <int TILE, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32>
__global__ void __launch_bounds__(256) gemm_bf16_solo_kernel(const GemmArgs g) {
  solo_gemm<TILE, TILE, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, false>(g);
}
template <int TILE, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32>
__global__ void __launch_bounds__(256) gemm_f16_solo_kernel(const GemmArgs g) {
  solo_gemm<TILE, TILE, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, true>(g);
}
// The 256 x 128 tile of the launches that finish a problem.  (As fed_gemm it takes longer, in one part or several: 260 input
// gradients, 260 weight gradients and 231 forwards that the estimates give this tile, with bounds and without, 1.04, 1.02 and
// 1.02 of the time on average, up to 1.16: 640 x 7936 over 3176 57.5 us, 63.9; 15872 x 256 over 4263 54.3, 61.8.  Whole
// problems of 65 to 128 large tiles 1.025; rests: launch_shape.)
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32>
__global__ void __launch_bounds__(256) gemm_bf16_rest_kernel(const GemmArgs g) {
  solo_gemm<256, 128, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, false>(g);
}
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32>
__global__ void __launch_bounds__(256) gemm_f16_rest_kernel(const GemmArgs g) {
  solo_gemm<256, 128, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, true>(g);
}

// Weight gradient and input gradient of one layer in one launch, 256 x 256 tiles: the
// workgroups [gw.wg_first, gw.wg_first + gw's) compute dW = dY^T X, the others dX = dY W.
// The host puts the problem with the longer tiles first; the dispatcher hands workgroups
// out in index order, so a CU takes a tile of the other product as soon as it is free.
// The second problem's last `quartered` tiles, those that would start when few are left, are four
// workgroups of 128 x 128 each, in the same order of sums: a tile that one CU would work on alone ends in
// less than half the time on four.  8192 x 5120 x 2560, 200 tiles of 128 stages and 320 of 80, the last 8
// of them alone on 56 idle CUs: 363 -> 343 us; 4096 x 2560 x 2560 104 -> 90, 4096 x 14336 x 2560 434 -> 416.
template <bool A_KMAJOR, bool B_KMAJOR, bool OUT_F32, bool HALF>
__device__ __forceinline__ void backward_tile(const GemmArgs& g, int pid) {
  const int whole = g.tiles_m * g.tiles_n - g.quartered;
  int tm, tn;
  if (pid < whole) {
    tile_of_workgroup(pid, g.tiles_m, g.tiles_n, tm, tn);
    solo_gemm<256, 256, A_KMAJOR, B_KMAJOR, AXN_EPI_NONE, OUT_F32, HALF>(g, tm, tn, 0);
  } else {
    const int q = pid - whole;
    tile_of_workgroup(whole + q / 4, g.tiles_m, g.tiles_n, tm, tn);
    solo_gemm<128, 128, A_KMAJOR, B_KMAJOR, AXN_EPI_NONE, OUT_F32, HALF>(g, 2 * tm + q % 4 / 2, 2 * tn + q % 2, 0);
  }
}
template <bool HALF, bool DW_F32>
__global__ void __launch_bounds__(256) gemm_backward_kernel(const GemmArgs gw, const GemmArgs gd) {
  const int b = (int)blockIdx.x;
  if (b >= gw.wg_first && b < gw.wg_first + gw.tiles_m * gw.tiles_n + 3 * gw.quartered)
    backward_tile<false, false, DW_F32, HALF>(gw, b - gw.wg_first);
  else
    backward_tile<true, false, false, HALF>(gd, b - gd.wg_first);
}

// The gate/up forward of a gated MLP: silu(A B^T) * (A B2^T), 256 rows x 128 columns of
// the output per workgroup (the MFMA work of a 256 x 256 tile).
__global__ void __launch_bounds__(256) gemm_bf16_swiglu_kernel(const GemmArgs g) {
  solo_gemm<256, 256, true, true, EPI_SWIGLU, false, false>(g);
}
__global__ void __launch_bounds__(256) gemm_f16_swiglu_kernel(const GemmArgs g) {
  solo_gemm<256, 256, true, true, EPI_SWIGLU, false, true>(g);
}

template <int TILE, bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_solo(const GemmArgs& in, hipStream_t stream) {
  GemmArgs g = in;
  g.tiles_m = g.M / TILE;
  g.tiles_n = g.N / TILE;
  // ring of 5 operand tiles: 160 KiB (all of a CU's LDS) or 80 KiB (two workgroups per CU)
  constexpr size_t lds = 5 * TILE * 64 * 2;
  void (*kern)(const GemmArgs) = gemm_bf16_solo_kernel<TILE, AK, BKM, EPI, OUT_F32>;
  if constexpr (HALF) kern = gemm_f16_solo_kernel<TILE, AK, BKM, EPI, OUT_F32>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  const int splits = g.splits > 1 ? g.splits : 1;
  hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_m * g.tiles_n * splits)), dim3(256), lds, stream,
                     g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_rest(const GemmArgs& in, hipStream_t stream) {
  GemmArgs g = in;
  g.tiles_m = g.M / 256;
  g.tiles_n = g.N / 128;
  constexpr size_t lds = 5 * 256 * 64 * 2;   // five slots of the A tile's size
  void (*kern)(const GemmArgs) = gemm_bf16_rest_kernel<AK, BKM, EPI, OUT_F32>;
  if constexpr (HALF) kern = gemm_f16_rest_kernel<AK, BKM, EPI, OUT_F32>;
  {
    static std::atomic<unsigned long long> lds_allowed{0};   // per template instance
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);
    if (rc != AXN_OK) return rc;
  }
  const int splits = g.splits > 1 ? g.splits : 1;
  hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_m * g.tiles_n * splits)), dim3(256), lds, stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// ---- shapes that are not made of whole tiles (gemm_edge.h) -----------------------------
// Estimated microseconds of one launch of `w` workgroups of a tile size that each walk `stages`
// 64-deep stages of operands of `mb` megabytes (short runs on MI355X, operands coming from HBM):
//   main loop   0.69 per stage of 128 x 128 tiles at one workgroup per CU, 1.2 + 0.936 per
//               stage at two; 2.5 + 0.737 of 256 x 128 tiles; 5.1 + 1.084 of 256 x 256 tiles;
//               times the rounds of workgroups;
//   operands    never faster than 1.7 + their bytes at 5.7 TB/s, which they reach only with a
//               workgroup on every CU (9 % of it with none, linear between).
// (256 x 128 tiles are the one-wave kernel's.)  The constants were fitted to 3479 launches: every tile size and split of 220 forward and
// input-gradient problems of 33 to 3000 tokens and 768 to 14336 features, ragged and whole.
// `epilogue`: what the output's epilogue adds to a round, on each of the four.
struct EpilogueTime {
  double us[4];
};
double launch_microseconds(EdgeTile tile, long long w, double stages, double mb, const EpilogueTime& epilogue = {}) {
  const double* e = epilogue.us;
  const double loop = tile == EDGE_256x256   ? (5.1 + 1.084 * stages + e[0]) * (double)((w + 255) / 256)
                      : tile == EDGE_256x128 ? (2.5 + 0.737 * stages + e[1]) * (double)((w + 255) / 256)
                      : w <= 256             ? 0.69 * stages + e[2]
                                             : (1.2 + 0.936 * stages + e[3]) * (double)((w + 511) / 512);
  const double occupied = w >= 256 ? 1.0 : (double)w / 256;
  const double stream = 1.74 + mb / (5.72 * (0.086 + 0.914 * occupied));
  return loop > stream ? loop : stream;
}

// One wave a SIMD has nothing to run beside its epilogue; two workgroups on a CU have each other's main loop.
// Bias, or (bias and) GELU, and each of an fp32 result and a saved pre-activation on top.  Fitted with the
// constants above held, to 2400 ragged forwards of 65 to 8192 rows, 64 to 16384 outputs and contractions of 192
// to 4096; over 5000 others the pick takes 0.3 % more than the best of the three tiles on average and 30 % at
// worst (without it 1.6 % and 69 %: 6144 x 2880 x 384 with bias 44 us on the large tile, 35 on the small).
EpilogueTime epilogue_time(const GemmArgs& g, int epilogue, bool out_f32) {
  if (epilogue == AXN_EPI_NONE) return {};
  const bool gelu = epilogue != AXN_EPI_BIAS;
  EpilogueTime t = gelu ? EpilogueTime{15.5, 7.8, 3.9, 1.4} : EpilogueTime{6.6, 3.3, 1.6, 0.0};
  const double more[4] = {1.9, 1.1, 0.7, 1.1};
  for (int i = 0; i < 4; ++i) t.us[i] += more[i] * ((out_f32 ? 1 : 0) + (gelu && g.Z != nullptr ? 1 : 0));
  return t;
}

// The same for an unsplit M x N output as launch_edge runs it: a last round of at most
// half of the CUs goes to smaller tiles (fed ones among them, which this leaves out).
double edge_microseconds(EdgeTile tile, long long M, long long N, long long Kc, const EpilogueTime& epilogue) {
  const int bm = tile == EDGE_128x128 ? 128 : 256, bn = tile == EDGE_256x256 ? 256 : 128;
  const long long w = ((M + bm - 1) / bm) * ((N + bn - 1) / bn), full = w / 256, rest = w % 256;
  const double stages = (double)((Kc + 63) / 64), mb = ((double)M + (double)N) * (double)Kc * 2e-6;
  if (tile == EDGE_256x256 && full > 0 && rest > 0 && rest <= 128)
    return launch_microseconds(tile, full * 256, stages, mb, epilogue) +
           launch_microseconds(rest <= 64 ? EDGE_128x128 : EDGE_256x128, 256, stages, 0.0, epilogue) + 3.0;
  return launch_microseconds(tile, w, stages, mb, epilogue);
}

EdgeTile edge_tile(long long M, long long N, long long Kc, const EpilogueTime& epilogue = {}, double* us = nullptr) {
  EdgeTile best = EDGE_256x256;
  double least = edge_microseconds(best, M, N, Kc, epilogue);
  for (EdgeTile t : {EDGE_256x128, EDGE_128x128}) {
    const double e = edge_microseconds(t, M, N, Kc, epilogue);
    if (e < least) {
      least = e;
      best = t;
    }
  }
  if (us != nullptr) *us = least;
  return best;
}

// Outputs made of whole 128 x 128 tiles but not of larger ones: whether the small tile without bounds is ahead
// of the larger ones with them.  Two workgroups share a CU and do not run in rounds, so its time grows
// evenly with their number.  Larger tiles have to be estimated 8 % faster, beyond one round of them, where the
// power cap stretches the estimate, 27 % (of 277 problems drawn those between 20 and 26 % took 1.01 of the small tile's
// time on average, up to 1.14; the ones beyond either line 0.92 and 0.90).  They do not add to the output: reading it in
// tiles that reach past its edge costs more than they gain (91 of them 1.01 on average, up to 1.22: 640 x
// 7040 x 6528 91 / 110).  us, small tile / larger ones, of M x N, contraction:
//   2048 x 50304, 2048  442 / 363      8192 x 5504, 2048  149 / 134   2048 x 5504, 8192 (weight gradient)  163 / 139
//   4096 x 50304, 768   398 / 298      4096 x 3200, 3200   83 / 67    3200 x 10240, 2560 (input gradient)  143 / 158
//   896 x 14336, 4096    99 / 82       8192 x 1920, 1920   52 / 46    2176 x 4096, 4096, GELU               83 / 87
bool small_tile_ahead(long long M, long long N, long long Kc, const EpilogueTime& epilogue) {
  const double w = (double)(M / 128) * (double)(N / 128), stages = (double)(Kc / 64);
  const double alone = 0.69 * stages + epilogue.us[2], shared = 1.2 + 0.936 * stages + epilogue.us[3];
  const double small = w <= 256 ? alone : w <= 512 ? alone + (shared - alone) * (w - 256) / 256 : shared * w / 512;
  double large = 0;
  if (edge_tile(M, N, Kc, epilogue, &large) == EDGE_128x128) return true;
  return small < large * (ceil_div(M, 256) * ceil_div(N, 256) <= 256 ? 1.08 : 1.27);
}

// ---- outputs of one round of small tiles, or two (gemm_fed_tiles.h) ------------------------
struct FedTile {
  EdgeTile tile;
  int bm, bn;
  // Estimated microseconds of a launch, for each operand order: a round of workgroups, a stage of it, a megabyte of
  // operands (with a workgroup on every CU) and one of output.
  float round[3], stage[3], operands[3], output[3];
};
// Fitted to 17288 launches on MI355X, cold operands: every tile, in 1 to 16 parts, of 1441 products of 1 to 8192 tokens
// and 256 to 14336 features as training and inference have them; 8 to 14 % rms, but alike for a problem's tiles.
constexpr FedTile kFedTiles[] = {
    {FED_64x64, 64, 64, {1.29f, 2.08f, 2.13f}, {0.175f, 0.208f, 0.077f}, {0.140f, 0.073f, 0.719f}, {0.79f, 0.70f, 0.00f}},
    {FED_96x64, 96, 64, {1.40f, 1.93f, 2.99f}, {0.276f, 0.295f, 0.270f}, {0.072f, 0.045f, 0.227f}, {0.65f, 0.63f, 0.05f}},
    {FED_64x128, 64, 128, {1.52f, 2.06f, 3.15f}, {0.330f, 0.343f, 0.277f}, {0.073f, 0.047f, 0.208f}, {0.58f, 0.61f, 0.11f}},
    {FED_96x128, 96, 128, {1.69f, 2.08f, 3.26f}, {0.400f, 0.417f, 0.371f}, {0.065f, 0.038f, 0.194f}, {0.51f, 0.56f, 0.14f}},
    {FED_128x128, 128, 128, {1.93f, 2.39f, 3.55f}, {0.470f, 0.504f, 0.425f}, {0.058f, 0.024f, 0.147f}, {0.47f, 0.51f, 0.15f}},
    {FED_96x192, 96, 192, {1.84f, 2.10f, 3.74f}, {0.512f, 0.533f, 0.491f}, {0.064f, 0.039f, 0.134f}, {0.46f, 0.51f, 0.13f}},
    {FED_128x192, 128, 192, {2.52f, 2.67f, 4.01f}, {0.564f, 0.595f, 0.528f}, {0.051f, 0.030f, 0.121f}, {0.45f, 0.48f, 0.15f}},
    {FED_160x192, 160, 192, {3.00f, 2.88f, 4.33f}, {0.609f, 0.662f, 0.620f}, {0.044f, 0.022f, 0.104f}, {0.41f, 0.44f, 0.15f}},
    {FED_128x256, 128, 256, {2.98f, 2.92f, 4.40f}, {0.683f, 0.686f, 0.627f}, {0.049f, 0.031f, 0.114f}, {0.39f, 0.42f, 0.15f}},
    {FED_256x128, 256, 128, {3.35f, 2.45f, 4.41f}, {0.748f, 0.784f, 0.678f}, {0.010f, 0.000f, 0.091f}, {0.39f, 0.46f, 0.16f}},
};

double fed_microseconds(const FedTile& t, GemmLayout layout, long long M, long long N, long long Kc, int parts,
                        double epilogue) {
  const long long w = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * parts;
  const double rounds = (double)((w + 255) / 256), occupied = w >= 256 ? 1.0 : (double)w / 256;
  const double mb = ((double)M + (double)N) * (double)Kc * 2e-6;
  const double out = (double)M * (double)N * (parts > 1 ? 4e-6 * parts : 2e-6);
  // rows of a contraction that does not fill 128-byte lines: the copies of a stage take two lines a row
  const double lines = layout != GEMM_TN && Kc % 64 != 0 ? 1.3 : 1.0;
  const double stages = (double)((Kc + 63) / 64 + parts - 1) / parts;
  return rounds * (t.round[layout] + t.stage[layout] * lines * stages + epilogue * (t.bm * t.bn) / 32768.0) +
         t.operands[layout] * mb / occupied + t.output[layout] * out;
}

// The best of them for a contraction in `parts`, or null.  More than two rounds of workgroups are left to larger
// tiles, and so are contractions of many stages to those of more than 64 columns: 64-column tiles read 128 bytes of a
// row of W or X at a time, which at some strides crowd onto few memory channels (446 x 2048 over 7168, rows of W of
// 4096 bytes, 41 us, 31 on larger tiles).  A weight gradient over few tokens is all stores, whatever its tile.
const FedTile* best_fed_tile(GemmLayout layout, long long M, long long N, long long Kc, int parts, double epilogue,
                             double* us) {
  const FedTile* best = nullptr;
  if (layout == GEMM_TN && Kc < 192) return best;
  for (const FedTile& t : kFedTiles) {
    const long long w = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * parts;
    if (w > (parts > 1 ? 256 : 512)) continue;
    if (t.bn == 64 && Kc > (layout == GEMM_NT ? 4096 : 2560) * parts) continue;
    const double e = fed_microseconds(t, layout, M, N, Kc, parts, epilogue);
    if (best == nullptr || e < *us) {
      best = &t;
      *us = e;
    }
  }
  return best;
}

// What an epilogue adds to a round of 256 x 128 tiles; a sum of parts has it in its own pass.
double fed_epilogue(const GemmArgs& g, int epilogue, bool out_f32) {
  if (epilogue == AXN_EPI_NONE) return 0.0;
  const bool gelu = epilogue != AXN_EPI_BIAS;
  return (gelu ? 7.8 : 3.3) + 1.1 * ((out_f32 ? 1 : 0) + (gelu && g.Z != nullptr ? 1 : 0));
}

// What the estimates above, of the other tiles, come to on cold operands: they leave out the output's way.  (Fitted to
// the same products, 10 % rms.)
double other_microseconds(GemmLayout layout, double us, long long M, long long N) {
  const double out = (double)M * (double)N * 2e-6;
  return layout == GEMM_TN ? 1.03 * us + 0.12 * out + 2.4 : layout == GEMM_NT ? 1.06 * us + 0.35 * out + 0.2 : 1.03 * us + 0.35 * out + 0.7;
}

// The fed tile of a contraction in one part, or null where the others are ahead or less than 5 % behind.  With the parts
// of gemm_plan: of 1500 products drawn anew (1 to 8192 tokens, 256 to 16384 features; a third each forwards, input and weight
// gradients) those that take a fed tile have 0.71 (forward), 0.73 and 0.77 of the time of the other tiles in one part, 0.82,
// 0.86 and 0.93 in several; 18 got 3 to 15 % slower (315 x 2304 x 9024, weight gradient, 26 -> 30 us; 640 x 2560 over 4480 with
// bias 32 -> 35).  us, before / so, outputs over contractions, operands from HBM: 512 x 8192, 3584 45.4 / 42.5; 777 x 6144, 4096
// 57 / 49; 250 x 1024, 1024 15.0 / 8.2; 2006 x 2432, 1088 20.9 / 18.6; weight gradient 2440 x 2240, 800 18.9 / 17.5.
const FedTile* fed_tile(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32) {
  if (g.splits > 1 || (g.lda > g.ldb ? g.lda : g.ldb) >= kEdgeMaxLd / 2) return nullptr;
  double us = 0, other = 0;
  const FedTile* t = best_fed_tile(layout, g.M, g.N, g.Kc, 1, fed_epilogue(g, epilogue, out_f32), &us);
  if (t == nullptr) return nullptr;
  edge_tile(g.M, g.N, g.Kc, epilogue_time(g, epilogue, out_f32), &other);
  return us < 0.95 * other_microseconds(layout, other, g.M, g.N) ? t : nullptr;
}

// The tile of a 16-bit weight gradient that is done in more than two rounds of workgroups that stay
// (gemm_fed_rounds.hip), or EDGE_256x256 where the others are ahead.  Such a launch saves what the tiles' ramps and
// stores cost a short contraction, and ends on a finer last round than 256 x 256 tiles; what it loses is their rate.
// Both sides are estimated in us: rounds, their stages, the output's and the operands' megabytes; the others' last round
// of up to 128 tiles is one of smaller ones.  Fitted to 700 gradients of 265 to 800 tokens over 1024 to 50264 and 512 to
// 8192 features with more than 512 tiles (7 and 5 % rms); 264 tokens and less are stores in any tile.  Of 700 drawn
// anew 309 are taken, with 0.92 of the time that they have elsewhere, 12 of them 3 to 7 % slower (counting half rounds of
// 256 x 256 tiles instead took 531, with 0.954 and 77 of them 3 to 18 % slower).  us, elsewhere / so, operands from HBM:
// 447 x 12288 x 2048 44.7 / 34.3, 404 x 9600 x 2368 40.7 / 32.0, 320 x 16384 x 3584 64.2 / 59.8, 748 x 6016 x 2880 45.0 / 42.2;
// left out 440 x 8288 x 3736 42.2 / 54.6, 708 x 8192 x 2304 36.0 / 44.5, 512 x 8192 x 3584 42.5 / 49.2, 768 x 8192 x 8192 112 /
// 138.  fp32 results and adding to one are bound by the output (382 x 4160 x 5632 fp32 35.6 / 39.7, 349 x 6784 x 4808 added
// to 46 / 57).
EdgeTile rounds_tile(const GemmArgs& g) {
  if (g.Kc <= 264 || g.Kc > 800 || g.beta || g.splits > 1 || (g.lda > g.ldb ? g.lda : g.ldb) >= kEdgeMaxLd / 2) return EDGE_256x256;
  if (g.N % 8 != 0 || g.ldc % 8 != 0) return EDGE_256x256;   // (columns that it does not store)
  const long long wide = ceil_div(g.M, 128) * ceil_div(g.N, 256), tall = ceil_div(g.M, 256) * ceil_div(g.N, 128);
  const long long tiles = wide <= tall ? wide : tall;
  if (tiles <= 512 || tiles > 65536) return EDGE_256x256;
  const double stages = (double)ceil_div(g.Kc, 64), out = (double)g.M * (double)g.N * 2e-6;
  const double in = ((double)g.M + (double)g.N) * (double)g.Kc * 2e-6;
  const double here = 7.3 + (double)ceil_div(tiles, 256) * (0.688 * stages - 1.22) + 0.27 * out + 0.16 * in;
  const long long tm = ceil_div(g.M, 256), tn = ceil_div(g.N, 256), full = tm * tn / 256, rest = tm * tn % 256;
  const bool cut = full > 0 && rest > 0 && rest <= 128 && (full * 256 % tm == 0 || full * 256 % tn == 0);
  const double last = rest == 0 ? 0.0 : !cut ? 0.78 + 1.217 * stages : rest > 64 ? 5.0 + 0.587 * stages : 3.8 + 0.28 * stages;
  const double others = 4.8 + (double)full * (0.78 + 1.217 * stages) + last + 0.234 * out + 0.101 * in;
  if (here > 0.95 * others) return EDGE_256x256;
  return wide <= tall ? FED_128x256 : FED_256x128;
}

int launch_fed(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32, bool half, EdgeTile tile,
               hipStream_t stream) {
  if (layout == GEMM_NT)
    return half ? launch_gemm_fed_nt_f16(g, epilogue, out_f32, tile, stream)
                : launch_gemm_fed_nt_bf16(g, epilogue, out_f32, tile, stream);
  return half ? launch_gemm_fed_nn_tn_f16(layout, g, out_f32, tile, stream)
              : launch_gemm_fed_nn_tn_bf16(layout, g, out_f32, tile, stream);
}

// `full` whole tile columns, or rows, of 256 x 256 tiles and the rest of a problem, or false if no cut gives them.
bool cut_problem(GemmLayout layout, const GemmArgs& g, bool out_f32, long long full, GemmArgs& g1, GemmArgs& g2) {
  const long long tm = ceil_div(g.M, 256), tn = ceil_div(g.N, 256);
  const int64_t esz = out_f32 ? 4 : 2;
  g1 = g2 = g;
  if (full % tm == 0) {  // whole tile columns
    const int64_t n1 = full / tm * 256;
    g1.N = (int)n1;
    g2.N = g.N - (int)n1;
    g2.B = layout == GEMM_NT ? g.B + n1 * g.ldb : g.B + n1;
    if (g.B2 != nullptr) g2.B2 = layout == GEMM_NT ? g.B2 + n1 * g.ldb : g.B2 + n1;
    g2.C = (char*)g.C + n1 * esz;
    g2.bias = bias_at(g, n1);
    if (g.Z != nullptr) g2.Z = g.Z + n1;
    return true;
  }
  if (full % tn != 0) return false;
  const int64_t m1 = full / tn * 256;   // whole tile rows
  g1.M = (int)m1;
  g2.M = g.M - (int)m1;
  g2.A = layout == GEMM_TN ? g.A + m1 : g.A + m1 * g.lda;
  if (g.A2 != nullptr) g2.A2 = layout == GEMM_TN ? g.A2 + m1 : g.A2 + m1 * g.lda;
  g2.C = (char*)g.C + m1 * g.ldc * esz;
  if (g.Z != nullptr) g2.Z = g.Z + m1 * g.ldc;
  return true;
}

// Full rounds and the rest, as launch_shape cuts whole-tile problems: a last round of at most half of the CUs goes to
// smaller tiles in a launch of its own (2048 x 50257 over 2048, 40 tiles of 1576 left: 128 x 128 tiles
// two to a CU 30 us, fed ones 21; weight gradient 24, 22).
int launch_edge(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32, bool half,
                hipStream_t stream) {
  const int64_t ld = g.lda > g.ldb ? g.lda : g.ldb;
  if (ld >= kEdgeMaxLd) return launch_gemm_far(layout, g, epilogue, out_f32, half, stream);
  const auto launch = [&](const GemmArgs& a, EdgeTile tile) {
    return half ? launch_gemm_edge_f16(layout, a, epilogue, out_f32, tile, stream)
                : launch_gemm_edge_bf16(layout, a, epilogue, out_f32, tile, stream);
  };
  if (ld >= kEdgeMaxLd / 2) return launch(g, EDGE_128x128);
  const EdgeTile tile = edge_tile(g.M, g.N, g.Kc, epilogue_time(g, epilogue, out_f32));
  const long long tiles = ceil_div(g.M, 256) * ceil_div(g.N, 256), full = tiles / 256 * 256, rest = tiles - full;
  GemmArgs g1, g2;
  if (tile == EDGE_256x256 && full > 0 && rest > 0 && rest <= 128 && cut_problem(layout, g, out_f32, full, g1, g2)) {
    const int rc = launch(g1, tile);
    if (rc != AXN_OK) return rc;
    if (const FedTile* t = fed_tile(layout, g2, epilogue, out_f32))
      return launch_fed(layout, g2, epilogue, out_f32, half, t->tile, stream);
    return launch(g2, rest > 64 ? EDGE_256x128 : EDGE_128x128);
  }
  return launch(g, tile);
}

// Kernel selection.  Problems made of whole 256 x 256 tiles, more than 128 of
// them (half of the CUs) and not just above one round of 256, take the
// one-wave-per-SIMD kernel at that tile size, 65..128 of them take it at 256 x 128;
// other problems made of whole 128 x 128 tiles take it at 128 x 128, or the larger tiles of
// gemm_edge.h where small_tile_ahead says so; ragged shapes, and operands too large for 32-bit
// byte offsets, take the kernels of gemm_edge.h.
template <bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_whole(const GemmArgs& g, hipStream_t stream) {
  const bool deep = g.Kc % 64 == 0;
  const bool whole256 = (g.M % 256 == 0) && (g.N % 256 == 0) && deep;
  const bool whole128 = (g.M % 128 == 0) && (g.N % 128 == 0) && deep;
  const long long tiles256 = ceil_div(g.M, 256) * ceil_div(g.N, 256);
  const long long tiles128 = ceil_div(g.M, 128) * ceil_div(g.N, 128);
  // The one-wave-per-SIMD kernel addresses its operands with 32-bit byte offsets.
  const int64_t a_span = (int64_t)(AK ? g.M : g.Kc) * g.lda * 2;
  const int64_t b_span = (int64_t)(BKM ? g.N : g.Kc) * g.ldb * 2;
  const bool small_spans = a_span < (1LL << 31) && b_span < (1LL << 31);
  // Up to 128 large tiles the small tile wins: four times as many workgroups, two per CU, still
  // fit in one round.  Beyond that its second round costs more than the idle CUs of the large one,
  // except just above one full round (257..320 large tiles), where the large tile's second round
  // would leave three quarters of the chip idle (measured: +10..14 % at 272..304 tiles, -3 % at 336).
  const bool large_tile = tiles256 > 128 && !(tiles256 > 256 && tiles256 <= 320);
  if (small_spans && whole256 && large_tile)
    return launch_solo<256, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
  // 65..128 large tiles: 256 x 128 tiles, one workgroup per CU on more than half of the CUs
  // (+4..11 % against the small tile, measured at 80, 96, 112 and 128 tiles).
  if (small_spans && whole256 && tiles256 > 64 && tiles256 <= 128)
    return launch_rest<AK, BKM, EPI, OUT_F32, HALF>(g, stream);
  if (small_spans && whole128 && tiles128 < (1LL << 31)) {
    bool small_tile = true;
    if constexpr (EPI != EPI_PAIR)
      small_tile = whole256 || g.beta || small_tile_ahead(g.M, g.N, g.Kc, epilogue_time(g, EPI, OUT_F32));
    if (small_tile) return launch_solo<128, AK, BKM, EPI, OUT_F32, HALF>(g, stream);
  }
  if constexpr (EPI == EPI_PAIR) {
    set_error("gemm_pair: needs whole 128 x 128 tiles, contractions that are multiples of 64 and "
              "operands below 2 GiB (got M=%d, N=%d, K=%d)", g.M, g.N, g.Kc);
    return AXN_ESHAPE;
  } else {
    constexpr GemmLayout layout = !AK ? GEMM_TN : BKM ? GEMM_NT : GEMM_NN;
    return launch_edge(layout, g, EPI, OUT_F32, HALF, stream);
  }
}

// Full rounds and the rest.  A problem of k * 256 + r large tiles with 0 < r <= 128 ends
// in a round that leaves at least half of the CUs idle.  It is cut along one output
// dimension into a part of exactly k rounds of large tiles and the remaining r tiles,
// which go to 256 x 128 tiles (2 r workgroups, one per CU) or, for r <= 64, to the small
// tile (4 r workgroups).
// Measured on 4096-row problems, K = 4096: +8..12 % at 272..384 tiles, +11..13 % at
// 544..576, +4 % at 640, +10 % at 800, +1 % at 896; with r > 128 the cut loses 2..3 %.
// The two parts run one after the other on the caller's stream.
template <bool AK, bool BKM, int EPI, bool OUT_F32, bool HALF>
int launch_shape(const GemmArgs& g, hipStream_t stream) {
  if constexpr (EPI != EPI_PAIR) {
    constexpr GemmLayout order = !AK ? GEMM_TN : BKM ? GEMM_NT : GEMM_NN;
    if constexpr (order == GEMM_TN && EPI == AXN_EPI_NONE && !OUT_F32)
      if (const EdgeTile t = rounds_tile(g); t != EDGE_256x256) return launch_gemm_fed_rounds(g, HALF, t, stream);
    if (const FedTile* t = fed_tile(order, g, EPI, OUT_F32))
      return launch_fed(order, g, EPI, OUT_F32, HALF, t->tile, stream);
    // output rows that are not 16-byte aligned (axn_gemm_any_n): the kernels with bounds store them
    if (g.ldc % 8 != 0) return launch_edge(order, g, EPI, OUT_F32, HALF, stream);
  }
  if (g.M % 256 == 0 && g.N % 256 == 0 && g.Kc % 64 == 0 && g.splits <= 1) {
    const long long tiles = (long long)(g.M / 256) * (g.N / 256);
    const long long full = tiles / 256 * 256, rest = tiles - full;
    if (full > 0 && rest > 0 && rest <= 128) {
      GemmArgs g1, g2;
      constexpr GemmLayout order = !AK ? GEMM_TN : BKM ? GEMM_NT : GEMM_NN;
      if (cut_problem(order, g, OUT_F32, full, g1, g2)) {
        const int rc = launch_whole<AK, BKM, EPI, OUT_F32, HALF>(g1, stream);
        if (rc != AXN_OK) return rc;
        // More than 64 tiles left: 256 x 128 tiles, one per CU on more than half of the CUs
        // (qkv forward +5 %, down dgrad +3 % against the small tile); fewer: the small tile,
        // whose 4 r workgroups still give every CU at most one (MLP shard dgrad, r = 64: -7 %
        // with the 256 x 128 tile).
        const int64_t a_span = (int64_t)(AK ? g2.M : g2.Kc) * g2.lda * 2;
        const int64_t b_span = (int64_t)(BKM ? g2.N : g2.Kc) * g2.ldb * 2;
        if (rest > 64 && a_span < (1LL << 31) && b_span < (1LL << 31)) {
          // From contractions of 2048 on (70 to 73 problems of whole tiles each) the tile with copying waves takes 0.992 of
          // the whole time in weight gradients, 1.005 in forwards, 1.008 in input gradients (0.96 to 1.04 in all three).
          if constexpr (order == GEMM_TN && EPI == AXN_EPI_NONE)
            if (g2.Kc >= 2048) return launch_fed(order, g2, EPI, OUT_F32, HALF, FED_256x128, stream);
          return launch_rest<AK, BKM, EPI, OUT_F32, HALF>(g2, stream);
        }
        if constexpr (EPI != EPI_PAIR) {
          if (const FedTile* t = fed_tile(order, g2, EPI, OUT_F32))
            return launch_fed(order, g2, EPI, OUT_F32, HALF, t->tile, stream);
        }
        return launch_whole<AK, BKM, EPI, OUT_F32, HALF>(g2, stream);
      }
    }
  }
  return launch_whole<AK, BKM, EPI, OUT_F32, HALF>(g, stream);
}

}  // namespace

namespace {

// Sum of the fp32 partial products of a split contraction, in split order, then the output's
// epilogue; 8 columns per lane.  Bound by its reads (512 x 8192, 2 parts: 7.3 us for 42 MB).
// ANY: N is not a multiple of 8, or the output's rows are not 16-byte aligned; the partial products'
// rows are padded to a multiple of 8.
template <int EPI, bool OUT_F32, bool HALF, bool ANY>
__global__ void __launch_bounds__(256)
    splitk_reduce_kernel(const float* __restrict__ ws, const GemmArgs g) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per_row = ceil_div(g.N, 8);
  if (idx >= (int64_t)g.M * per_row) return;
  const int64_t row = idx / per_row, col = (idx - row * per_row) * 8, part = (int64_t)g.M * per_row * 8;
  const float* p = ws + row * per_row * 8 + col;
  f32x4 a0 = __builtin_nontemporal_load((const f32x4*)p);
  f32x4 a1 = __builtin_nontemporal_load((const f32x4*)(p + 4));
  for (int s = 1; s < g.splits; ++s) {
    p += part;
    a0 += __builtin_nontemporal_load((const f32x4*)p);
    a1 += __builtin_nontemporal_load((const f32x4*)(p + 4));
  }
  float v[8] = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
  if constexpr (EPI == EPI_WIDEN) {
    using lp = std::conditional_t<HALF, _Float16, __bf16>;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)(lp)v[e];
  }
  if (ANY && col + 8 > g.N) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (col + e < g.N) store_one<EPI, OUT_F32, HALF>(v[e], g, (int)row, (int)col + e);
    return;
  }
  float bias[8];
  load_bias8<EPI, HALF>(bias, g, (int)col);
  store_row8<EPI, OUT_F32, HALF, ANY>(v, bias, g, (int)row, (int)col);
}

template <bool HALF, bool ANY>
int launch_reduce(const float* ws, const GemmArgs& g, int epilogue, bool out_f32, hipStream_t stream) {
  const int64_t lanes = (int64_t)g.M * ceil_div(g.N, 8);
  const dim3 grid((unsigned)((lanes + 255) / 256)), block(256);
#define REDUCE(EPI, F32) hipLaunchKernelGGL((splitk_reduce_kernel<EPI, F32, HALF, ANY>), grid, block, 0, stream, ws, g)
  if (out_f32) {
    if (epilogue == EPI_WIDEN) REDUCE(EPI_WIDEN, true);
    else if (epilogue == AXN_EPI_BIAS) REDUCE(AXN_EPI_BIAS, true);
    else if (epilogue == AXN_EPI_BIAS_GELU) REDUCE(AXN_EPI_BIAS_GELU, true);
    else REDUCE(AXN_EPI_NONE, true);
  } else {
    switch (epilogue) {
      case AXN_EPI_NONE: REDUCE(AXN_EPI_NONE, false); break;
      case AXN_EPI_BIAS: REDUCE(AXN_EPI_BIAS, false); break;
      case AXN_EPI_BIAS_GELU: REDUCE(AXN_EPI_BIAS_GELU, false); break;
      default: REDUCE(AXN_EPI_GELU, false);
    }
  }
#undef REDUCE
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <bool AK, bool BKM, bool HALF>
int launch_split(const GemmArgs& g, EdgeTile tile, hipStream_t stream) {
  if (tile == EDGE_256x256) return launch_solo<256, AK, BKM, AXN_EPI_NONE, true, HALF>(g, stream);
  if (tile == EDGE_256x128) return launch_rest<AK, BKM, AXN_EPI_NONE, true, HALF>(g, stream);
  return launch_solo<128, AK, BKM, AXN_EPI_NONE, true, HALF>(g, stream);
}

template <bool HALF>
int launch_layout(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32,
                  hipStream_t stream) {
  if (layout == GEMM_NT && g.M <= kStreamMaxRows && g.lda < kStreamMaxLd && g.ldb < kStreamMaxLd &&
      (!out_f32 || epilogue == AXN_EPI_BIAS || epilogue == AXN_EPI_BIAS_GELU))
    return launch_gemm_stream(g, epilogue, out_f32, HALF, stream);
  switch (layout) {
    case GEMM_NT:
      if (out_f32) {  // 16-bit product + fp32 bias promoted to fp32, as `x + bias` promotes it
        if (epilogue == AXN_EPI_BIAS) return launch_shape<true, true, AXN_EPI_BIAS, true, HALF>(g, stream);
        if (epilogue == AXN_EPI_BIAS_GELU)
          return launch_shape<true, true, AXN_EPI_BIAS_GELU, true, HALF>(g, stream);
        break;
      }
      switch (epilogue) {
        case AXN_EPI_NONE:
          return launch_shape<true, true, AXN_EPI_NONE, false, HALF>(g, stream);
        case AXN_EPI_BIAS:
          return launch_shape<true, true, AXN_EPI_BIAS, false, HALF>(g, stream);
        case AXN_EPI_BIAS_GELU:
          return launch_shape<true, true, AXN_EPI_BIAS_GELU, false, HALF>(g, stream);
        case AXN_EPI_GELU:
          return launch_shape<true, true, AXN_EPI_GELU, false, HALF>(g, stream);
      }
      break;
    case GEMM_NN:
      if (out_f32 || epilogue != AXN_EPI_NONE) break;
      return launch_shape<true, false, AXN_EPI_NONE, false, HALF>(g, stream);
    case GEMM_TN:
      if (epilogue != AXN_EPI_NONE) break;
      return out_f32 ? launch_shape<false, false, AXN_EPI_NONE, true, HALF>(g, stream)
                     : launch_shape<false, false, AXN_EPI_NONE, false, HALF>(g, stream);
  }
  set_error("gemm: unsupported layout/epilogue/output combination");
  return AXN_EINVAL;
}
}  // namespace

int launch_gemm_pair(const GemmArgs& g, bool half, hipStream_t stream) {
  if (g.k_first % 64 != 0 || g.k_first < 128 || (g.Kc - g.k_first) % 64 != 0 || g.Kc - g.k_first < 64 ||
      g.splits > 1) {
    set_error("gemm_pair: both contractions must be multiples of 64, the first at least 128 "
              "(got %d and %d)", g.k_first, g.Kc - g.k_first);
    return AXN_ESHAPE;
  }
  // the operand spans the kernels address with 32 bits, checked on the longer pair
  const int k_long = g.k_first > g.Kc - g.k_first ? g.k_first : g.Kc - g.k_first;
  if ((int64_t)k_long * g.ldb * 2 >= (1LL << 31)) {
    set_error("gemm_pair: operands must stay below 2 GiB");
    return AXN_ESHAPE;
  }
  return half ? launch_shape<true, false, EPI_PAIR, false, true>(g, stream)
              : launch_shape<true, false, EPI_PAIR, false, false>(g, stream);
}

int launch_gemm_swiglu(const GemmArgs& in, bool half, hipStream_t stream) {
  GemmArgs g = in;
  const int64_t a_span = (int64_t)g.M * g.lda * 2, b_span = (int64_t)g.N * g.ldb * 2;
  if (g.M % 256 != 0 || g.N % 128 != 0 || g.Kc % 64 != 0 || a_span >= (1LL << 31) ||
      b_span >= (1LL << 31)) {
    set_error("gemm_swiglu: needs M %% 256 == 0, N %% 128 == 0, K %% 64 == 0 and operands below "
              "2 GiB (got M=%d, N=%d, K=%d)", g.M, g.N, g.Kc);
    return AXN_ESHAPE;
  }
  if (g.lda < kEdgeMaxLd / 2 && g.ldb < kEdgeMaxLd / 2) {   // few large tiles, or a last round of few: others
    bool taken = false;
    const int rc = launch_gemm_swiglu_any(g, half, true, stream, taken);
    if (taken) return rc;
  }
  g.tiles_m = g.M / 256;
  g.tiles_n = g.N / 128;
  g.splits = 0;
  constexpr size_t lds = 5 * 256 * 64 * 2;
  void (*kern)(const GemmArgs) = half ? gemm_f16_swiglu_kernel : gemm_bf16_swiglu_kernel;
  {
    static std::atomic<unsigned long long> lds_allowed[2];   // bf16 and fp16 kernel
    const int rc = allow_lds((const void*)kern, lds, lds_allowed[half ? 1 : 0]);
    if (rc != AXN_OK) return rc;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)((long long)g.tiles_m * g.tiles_n)), dim3(256), lds,
                     stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// ---- input and weight gradient of one layer in one call ----------------------------
namespace {
// Rounds of 64-deep stages a launch of `tiles` 256 x 256 tiles over `stages` stages takes on
// 256 CUs the way launch_shape runs it (a rest of up to half a round costs about 0.7 of one).
double stages_alone(long long tiles, long long stages) {
  const long long full = tiles / 256, rest = tiles % 256;
  if (rest == 0) return (double)(full * stages);
  if (full > 0 && rest <= 128) return (full + 0.7) * stages;
  return (double)((full + 1) * stages);
}
// The same for one launch that holds both problems, longer tiles first: every CU takes the
// next tile when it is free (a heap of the CUs' busy times: a few thousand steps).  The last `quartered` tiles of the
// second problem are four of kQuarter of their stages each; last: how many of its tiles end with the launch.
constexpr double kQuarter = 0.5;   // 0.45 to 0.55 us a stage of a 128 x 128 tile alone on its CU, 1.04 to 1.3 of a large one
double stages_together(long long t1, long long s1, long long t2, long long s2, long long quartered = 0,
                       long long* last = nullptr) {
  if (s1 < s2) {
    std::swap(t1, t2);
    std::swap(s1, s2);
  }
  std::priority_queue<double, std::vector<double>, std::greater<double>> cus;
  for (int c = 0; c < 256; ++c) cus.push(0);
  double end = 0;
  long long at_end = 0;
  auto place = [&](long long tiles, double stages) {
    for (long long i = 0; i < tiles; ++i) {
      const double t = cus.top() + stages;
      cus.pop();
      cus.push(t);
      if (t > end) at_end = 0;
      end = t > end ? t : end;
      if (t == end) ++at_end;
    }
  };
  place(t1, (double)s1);
  place(t2 - quartered, (double)s2);
  place(4 * quartered, kQuarter * (double)s2);
  if (last != nullptr) *last = at_end;
  return end;
}

// Whether two tile sets run in one launch; the answers for the last few shapes of a thread
// are kept, a training loop asks for the same ones again and again.  The key holds all that
// `ends_earlier` looks at.
struct Together {
  bool together;
  int quartered = 0;
};
struct PlannedTogether {
  long long key[4];
  Together plan;
};
template <class F>
Together plan_together(PlannedTogether (&plans)[4], int& next, long long k0, long long k1, long long k2, long long k3,
                       F&& ends_earlier) {
  for (const PlannedTogether& p : plans)
    if (p.key[0] == k0 && p.key[1] == k1 && p.key[2] == k2 && p.key[3] == k3) return p.plan;
  PlannedTogether& p = plans[next];
  next = (next + 1) % 4;
  p = {{k0, k1, k2, k3}, ends_earlier()};
  return p.plan;
}
// The problem with the longer tiles takes the first workgroups.
void place_together(GemmArgs& gd, GemmArgs& gw, long long td, long long tw, long long sd, long long sw) {
  gw.tiles_m = (int)ceil_div(gw.M, 256), gw.tiles_n = (int)ceil_div(gw.N, 256), gw.wg_first = sw >= sd ? 0 : (int)td;
  gd.tiles_m = (int)ceil_div(gd.M, 256), gd.tiles_n = (int)ceil_div(gd.N, 256), gd.wg_first = sw >= sd ? (int)tw : 0;
  gw.splits = gd.splits = gw.quartered = gd.quartered = 0;
}

template <bool HALF>
int launch_backward(const GemmArgs& gd_in, const GemmArgs& gw_in, bool dw_f32, hipStream_t stream) {
  GemmArgs gd = gd_in, gw = gw_in;
  auto whole = [](const GemmArgs& g, bool ak, bool bk) {
    const int64_t a_span = (int64_t)(ak ? g.M : g.Kc) * g.lda * 2;
    const int64_t b_span = (int64_t)(bk ? g.N : g.Kc) * g.ldb * 2;
    return g.M % 256 == 0 && g.N % 256 == 0 && g.Kc % 64 == 0 && g.Kc >= 128 && a_span < (1LL << 31) &&
           b_span < (1LL << 31);
  };
  if (whole(gd, true, false) && whole(gw, false, false)) {
    const long long td = (long long)(gd.M / 256) * (gd.N / 256), tw = (long long)(gw.M / 256) * (gw.N / 256);
    const long long sd = gd.Kc / 64, sw = gw.Kc / 64;
    // one launch when that ends at least 5 % earlier than the two launches (measured on
    // MI355X at 8192 x 5120 x 2560: 320 tiles of 80 stages and 200 of 128)
    static thread_local PlannedTogether plans[4] = {};
    static thread_local int next_plan = 0;
    const Together plan = plan_together(plans, next_plan, td, tw, sd, sw, [&]() -> Together {
      if (td + tw > 4096) return {false};
      long long last = 0;
      const double end = stages_together(tw, sw, td, sd, 0, &last);
      if (end >= 0.95 * (stages_alone(td, sd) + stages_alone(tw, sw))) return {false};
      // few tiles that end the launch: a quarter each where that ends it 5 % earlier
      const bool few = last <= 64 && last < (sw >= sd ? td : tw);
      return {true, few && stages_together(tw, sw, td, sd, last) < 0.95 * end ? (int)last : 0};
    });
    if (plan.together) {
      place_together(gd, gw, td, tw, sd, sw);
      (sw >= sd ? gd : gw).quartered = plan.quartered;
      constexpr size_t lds = 5 * 256 * 64 * 2;
      void (*kern)(const GemmArgs, const GemmArgs) =
          dw_f32 ? gemm_backward_kernel<HALF, true> : gemm_backward_kernel<HALF, false>;
      {
        static std::atomic<unsigned long long> lds_allowed[2];   // per output type of dW
        const int rc = allow_lds((const void*)kern, lds, lds_allowed[dw_f32 ? 1 : 0]);
        if (rc != AXN_OK) return rc;
      }
      hipLaunchKernelGGL(kern, dim3((unsigned)(tw + td + 3 * plan.quartered)), dim3(256), lds, stream, gw, gd);
      AXN_HIP_TRY(hipGetLastError());
      return AXN_OK;
    }
  }
  // Ragged shapes: one launch of both tile sets where their 256 x 256 tiles, filled into the
  // CUs longest first, end at least 5 % before the two launches would by the estimate.
  const auto ragged = [](const GemmArgs& g) {
    return (g.M % 128 != 0 || g.N % 128 != 0 || g.Kc % 64 != 0) && g.lda < kEdgeMaxLd / 2 && g.ldb < kEdgeMaxLd / 2;
  };
  if (ragged(gd) && ragged(gw)) {
    const long long td = ceil_div(gd.M, 256) * ceil_div(gd.N, 256), tw = ceil_div(gw.M, 256) * ceil_div(gw.N, 256);
    const long long sd = ceil_div(gd.Kc, 64), sw = ceil_div(gw.Kc, 64);
    static thread_local PlannedTogether plans[4] = {};
    static thread_local int next_plan = 0;
    const Together plan = plan_together(plans, next_plan, gd.M, gd.N, gd.Kc, 0, [&]() -> Together {
      if (td + tw > 4096) return {false};
      double ud = 0, uw = 0;
      edge_tile(gd.M, gd.N, gd.Kc, {}, &ud);
      edge_tile(gw.M, gw.N, gw.Kc, {}, &uw);
      return {1.084 * stages_together(tw, sw, td, sd) + 15 < 0.95 * (ud + uw)};
    });
    if (plan.together) {
      place_together(gd, gw, td, tw, sd, sw);
      return HALF ? launch_gemm_edge_backward_f16(gw, gd, dw_f32, stream)
                  : launch_gemm_edge_backward_bf16(gw, gd, dw_f32, stream);
    }
  }
  const int rc = launch_shape<true, false, AXN_EPI_NONE, false, HALF>(gd, stream);
  if (rc != AXN_OK) return rc;
  return dw_f32 ? launch_shape<false, false, AXN_EPI_NONE, true, HALF>(gw, stream)
                : launch_shape<false, false, AXN_EPI_NONE, false, HALF>(gw, stream);
}
}  // namespace

int launch_gemm_backward(const GemmArgs& dgrad, const GemmArgs& wgrad, bool half, bool dw_f32,
                         hipStream_t stream) {
  return half ? launch_backward<true>(dgrad, wgrad, dw_f32, stream)
              : launch_backward<false>(dgrad, wgrad, dw_f32, stream);
}

int launch_gemm_bf16(GemmLayout layout, const GemmArgs& g, int epilogue,
                     bool out_f32, hipStream_t stream) {
  return launch_layout<false>(layout, g, epilogue, out_f32, stream);
}

int launch_gemm_f16(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32,
                    hipStream_t stream) {
  return launch_layout<true>(layout, g, epilogue, out_f32, stream);
}

namespace {
constexpr double kPartsMicroseconds = 2.96;
double part_microseconds(int64_t M, int64_t N) { return 2.02 * std::pow((double)M * (double)N * 1e-6, 0.763); }
}  // namespace

// Few output tiles leave most CUs without work: the contraction is cut into parts of at
// least 512, on the tile and into the number of parts with the smallest estimated time, each part
// a workgroup per tile.  On top of the launch (launch_microseconds) a split costs
// 2.96 + parts x 2.02 x (millions of output elements)^0.763 microseconds for writing the fp32
// partial products and for the pass that adds them.  Over the 220 problems the estimate was
// fitted to, its pick takes 1.3 % more than the fastest choice on average and 22 % at worst;
// the rule before (parts of whole shapes only, 2, 4 or 8 of them, on the two smaller tiles) left
// ragged ones unsplit: 60 x 3520 x 6848 78 -> 20 us, 479 x 832 x 13824 146 -> 31 us, 1111 x 2752 x
// 6336 70 -> 56 us.
// It looks at sizes only, not at strides: a caller asks for the workspace by size.
SplitPlan gemm_splits(GemmLayout layout, int64_t M, int64_t N, int64_t Kc, double* us) {
  SplitPlan plan = {1, EDGE_128x128};
  if (layout == GEMM_NT && stream_ahead(M, N, Kc)) return plan;
  const bool whole = M % 128 == 0 && N % 128 == 0 && Kc % 64 == 0;
  auto count = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const long long tiles[3] = {count(256, 256), count(256, 128), count(128, 128)};
  // beyond 128 large tiles an unsplit launch of them already has half of the CUs; a short
  // contraction over a ragged shape is left alone
  if (tiles[EDGE_256x256] > 128 || Kc < (whole ? 1024 : 1536)) return plan;
  const double mb = ((double)M + (double)N) * (double)Kc * 2e-6;
  const double part_cost = part_microseconds(M, N);
  const long long stages = (Kc + 63) / 64;
  double best = 1e30;
  for (EdgeTile tile : {EDGE_128x128, EDGE_256x128, EDGE_256x256})
    best = std::fmin(best, launch_microseconds(tile, tiles[tile], (double)stages, mb));
  for (int parts = 2; parts <= 16 && Kc / parts >= 512; ++parts)
    for (EdgeTile tile : {EDGE_128x128, EDGE_256x128, EDGE_256x256}) {
      if (tiles[tile] * parts > (tile == EDGE_128x128 ? 512 : 256)) continue;
      const double t = launch_microseconds(tile, tiles[tile] * parts, (double)((stages + parts - 1) / parts), mb) +
                       kPartsMicroseconds + parts * part_cost;
      if (t < best) {
        best = t;
        plan = {parts, tile};
      }
    }
  if (us != nullptr) *us = best;
  return plan;
}

// The parts that a sum of the fp32 products reads and writes, and the launch it is: fitted to 2 to 16 parts.
static double sum_microseconds(int64_t M, int64_t N, int parts) {
  return 2.5 + (double)M * (double)N * (4 * parts + 2) * 1e-6 / 7.0;
}

// (190 forwards with bias or GELU, of 9000 drawn, whose plan the epilogue changes: counted, 0.93 of the time that
// gemm_splits' parts take, 1.03 at worst; not counted 0.97, 68 of them 1.03 to 1.18.)
SplitPlan gemm_plan(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32) {
  const int64_t M = g.M, N = g.N, Kc = g.Kc;
  double other = 0;
  SplitPlan plan = gemm_splits(layout, M, N, Kc, &other);
  if (plan.parts <= 1) return plan;
  double least = 0.95 * other_microseconds(layout, other, M, N);
  // The input gradient of a layer whose gradients take one launch keeps the parts it has there.
  const bool kept = layout == GEMM_NN && (gemm_backward_parts(M, Kc, N, false) > 0 || gemm_backward_parts(M, Kc, N, true) > 0);
  const int most = plan.parts;   // what the workspace holds
  for (int parts = kept ? most : 1; parts <= most; ++parts) {
    double us = 0;
    const FedTile* t = best_fed_tile(layout, M, N, Kc, parts, parts > 1 ? 0 : fed_epilogue(g, epilogue, out_f32), &us);
    if (t == nullptr) continue;
    if (parts > 1) us += sum_microseconds(M, N, parts);
    if (us < least) {
      least = us;
      plan = {parts, t->tile};
    }
  }
  return plan;
}

static int launch_sum(const GemmArgs& in, int epilogue, bool half, bool out_f32, int parts, const float* ws,
                      hipStream_t stream) {
  GemmArgs out = in;
  out.splits = parts;
  if (out.N % 8 != 0 || out.ldc % 8 != 0)
    return half ? launch_reduce<true, true>(ws, out, epilogue, out_f32, stream)
                : launch_reduce<false, true>(ws, out, epilogue, out_f32, stream);
  return half ? launch_reduce<true, false>(ws, out, epilogue, out_f32, stream)
              : launch_reduce<false, false>(ws, out, epilogue, out_f32, stream);
}

int launch_gemm_splitk(GemmLayout layout, const GemmArgs& in, int epilogue, bool half, bool out_f32,
                       const SplitPlan& plan, float* ws, hipStream_t stream, bool widen) {
  if (widen) {
    epilogue = EPI_WIDEN;
    out_f32 = true;
  }
  GemmArgs g = in;
  g.C = ws;
  g.ldc = ceil_div(g.N, 8) * 8;   // whole vectors a row
  g.beta = 0;
  g.bias = nullptr;
  g.Z = nullptr;
  g.splits = plan.parts;
  g.k_split = g.Kc / plan.parts;
  if (plan.tile > EDGE_128x128) {
    const int rc = launch_fed(layout, g, AXN_EPI_NONE, true, half, plan.tile, stream);
    return rc ? rc : launch_sum(in, epilogue, half, out_f32, plan.parts, ws, stream);
  }
  const bool ak = layout != GEMM_TN, bkm = layout == GEMM_NT;
  const int bm = plan.tile == EDGE_128x128 ? 128 : 256, bn = plan.tile == EDGE_256x256 ? 256 : 128;
  const bool whole = g.M % bm == 0 && g.N % bn == 0 && g.Kc % (64 * plan.parts) == 0 &&
                     (int64_t)(ak ? g.M : g.Kc) * g.lda * 2 < (1LL << 31) &&
                     (int64_t)(bkm ? g.N : g.Kc) * g.ldb * 2 < (1LL << 31);
  int rc;
  if (!whole) {
    rc = half ? launch_gemm_edge_f16(layout, g, AXN_EPI_NONE, true, plan.tile, stream)
              : launch_gemm_edge_bf16(layout, g, AXN_EPI_NONE, true, plan.tile, stream);
  } else {
    switch (layout) {
      case GEMM_NT:
        rc = half ? launch_split<true, true, true>(g, plan.tile, stream)
                  : launch_split<true, true, false>(g, plan.tile, stream);
        break;
      case GEMM_NN:
        rc = half ? launch_split<true, false, true>(g, plan.tile, stream)
                  : launch_split<true, false, false>(g, plan.tile, stream);
        break;
      default:
        rc = half ? launch_split<false, false, true>(g, plan.tile, stream)
                  : launch_split<false, false, false>(g, plan.tile, stream);
    }
  }
  return rc ? rc : launch_sum(in, epilogue, half, out_f32, plan.parts, ws, stream);
}

// ---- both gradients in one launch, the input gradient's contraction in parts -----------
// An input gradient of few tiles and its weight gradient each end in a ramp and a last wave of their own; in one
// launch the shorter tiles fill what the longer leave.  us, two launches and the sum / one and the sum: 1722 x 5888
// x 1024 69 / 54, 1376 x 9088 x 2112 139 / 127, 599 x 32000 x 1088 128 / 121, 777 x 6144 x 4096 109 / 89.
namespace {
// Time until n1 tiles of s1 and then n2 of s2, each on the CU that is free first, are done.
double filled(long long n1, double s1, long long n2, double s2) {
  const long long rounds = n1 / 256, more = n1 % 256;   // `more` CUs have a tile of the first kind on top
  const auto room = [&](double t) {
    const double a = t - (double)(rounds + 1) * s1, b = t - (double)rounds * s1;
    return (double)more * (a > 0 ? std::floor(a / s2) : 0) + (double)(256 - more) * (b > 0 ? std::floor(b / s2) : 0);
  };
  double lo = (double)(rounds + (more > 0 ? 1 : 0)) * s1, hi = lo + (double)(n2 / 256 + 1) * s2;
  while (hi - lo > 0.25) {
    const double mid = 0.5 * (lo + hi);
    (room(mid) >= (double)n2 ? hi : lo) = mid;
  }
  return hi;
}

}  // namespace

// The parts are the input gradient's own, so that its bits are the same either way.  The estimate: 2.2 us and 1.45
// a stage of a time that lies between the work's average over the CUs and that of the fullest one (0.3 to 0.7), a
// tile counting 3 stages more than it has, 6 where it reads dW to add to it, and the parts' cost; fitted to 65
// problems of 64 to 3564 tokens with 2 to 16 parts each (7 % rms).  The two launches, whose estimate is 8 % low, and
// 15 % beyond 100 us, where the power cap stretches it, have to be slower (up to 20 %: of 1100 problems drawn 243
// more in one launch, 0.98 of the time of two, a twelfth of them 3 to 15 % slower).  Up to 192 rows a weight gradient
// is nearly all stores, and two launches are as fast (151 x 11392 x 4992: 75 us, 79 in one).
// Where that estimate is not enough, from 758 problems that it takes (481 of whole 128 x 128 x 64 tiles, whose two
// launches have kernels without bounds; us, two launches / one):
//   too few tiles in all to fill the CUs, which smaller tiles of a launch alone do        1536 x 3072 x 1024  37 / 44
//   at most 64 tiles of dX, unless they run beside one round of stores of dW + ...        256 x 11136 x 1664  45 / 50
//   more than 200 tiles of dX (nearly a round of their own) of a whole-tile problem, unless the estimate is well ahead
//                                                                                         512 x 11008 x 8192 186 / 196
//   adding to dW in tiles that reach past its edge where those of two launches do not      256 x 18560 x 5632 209 / 236
//   adding to more than 256 tiles of dW from at most 256 rows with bounds                  237 x 13312 x 5376 154 / 180
// The estimates of two launches know neither gemm_fed_tiles.h's tiles nor gemm_plan's parts, which make them faster than
// that; measured against what two launches do with both, free to take other parts, the rule holds: of 500 problems drawn
// anew that it takes, one launch has 0.877 of their time on average, 15 take 3 to 15 % longer (2549 x 4032 x 1088, added to an
// fp32 dW, 76 / 88; 284 x 15040 x 4800 123 / 139; 3223 x 11176 x 1920, fp32 dW, 283 / 296).
int gemm_backward_parts(int64_t M, int64_t N, int64_t K, bool add) {
  if (M <= 192) return 0;
  double apart_d = 0, apart_w = 0;
  const int parts = gemm_splits(GEMM_NN, M, K, N, &apart_d).parts;
  const long long tw = ceil_div(N, 256) * ceil_div(K, 256);
  if (parts <= 1 || tw > 65536 || gemm_splits(GEMM_TN, N, K, M).parts > 1) return 0;
  edge_tile(N, K, M, {}, &apart_w);
  if (add) apart_w += 0.5 * (double)N * (double)K * 2e-6 / 5.72;   // reading dW, half of it hidden
  const long long td = ceil_div(M, 256) * ceil_div(K, 256) * parts;
  const bool whole = M % 64 == 0 && N % 128 == 0 && K % 128 == 0, large = N % 256 == 0 && K % 256 == 0;
  if (td + tw <= 160 || (td <= 64 && !(add && tw <= 256))) return 0;
  if (add && (whole ? !large : M <= 256 && tw > 256)) return 0;
  const double d = (double)(ceil_div(ceil_div(N, 64), parts) + 3), w = (double)(ceil_div(M, 64) + (add ? 6 : 3));
  const double fullest = d >= w ? filled(td, d, tw, w) : filled(tw, w, td, d);
  const double average = ((double)td * d + (double)tw * w) / 256;
  const double us = 2.2 + 1.45 * (0.7 * fullest + 0.3 * average) + kPartsMicroseconds + parts * part_microseconds(M, K);
  const double apart = apart_d + apart_w;
  return us < apart * (apart < 100 ? 1.08 : whole && td > 200 ? 1.1 : 1.15) ? parts : 0;
}

int launch_gemm_backward_parts(const GemmArgs& dgrad, const GemmArgs& wgrad, bool half, bool dw_f32, int parts,
                               float* ws, hipStream_t stream) {
  GemmArgs gd = dgrad, gw = wgrad;
  const long long td = ceil_div(gd.M, 256) * ceil_div(gd.N, 256), tw = ceil_div(gw.M, 256) * ceil_div(gw.N, 256);
  place_together(gd, gw, td * parts, tw, ceil_div(ceil_div(gd.Kc, 64), parts), ceil_div(gw.Kc, 64));
  gd.C = ws;
  gd.ldc = ceil_div(gd.N, 8) * 8;
  gd.splits = parts;
  const int rc = half ? launch_gemm_edge_backward_f16(gw, gd, dw_f32, stream)
                      : launch_gemm_edge_backward_bf16(gw, gd, dw_f32, stream);
  if (rc) return rc;
  return launch_sum(dgrad, AXN_EPI_NONE, half, false, parts, ws, stream);
}

}  // namespace axn
