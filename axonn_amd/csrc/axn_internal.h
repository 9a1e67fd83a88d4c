// Internal declarations shared by the kernel translation units and the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

#include "axn.h"

namespace axn {

// Thread-local error text behind axn_last_error().
void set_error(const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);

#define AXN_HIP_TRY(expr)                                  \
  do {                                                     \
    hipError_t e__ = (expr);                               \
    if (e__ != hipSuccess) return ::axn::hip_fail(e__, #expr); \
  } while (0)

// ---- launches of many workgroups ---------------------------------------------------
// A launch has fewer than 2^32 threads in a dimension; beyond, the grid wraps without an error.  So the workgroups
// of a launch that may have that many go on in the next dimension, kMostBlocks (of up to 1024 threads) at a time, and
// some behind the last one with nothing to do.  (A constant: the size of the grid would be another load.)
constexpr int64_t kMostBlocks = 1 << 21;
inline dim3 grid_of(int64_t blocks) {
  return blocks <= kMostBlocks ? dim3((unsigned)blocks)
                               : dim3((unsigned)kMostBlocks, (unsigned)((blocks + kMostBlocks - 1) / kMostBlocks));
}
__device__ __forceinline__ int64_t block_number() { return (int64_t)blockIdx.y * kMostBlocks + blockIdx.x; }

// ---- exact-erf GELU -----------------------------------------------------------
// gelu(x) = x * Phi(x), Phi(x) = (1 + erf(x / sqrt 2)) / 2, the definition behind
// torch.nn.GELU() (approximate='none').  The library erff costs about 100 VALU
// operations per element with both of its branches taken in a wave, which made
// the fused epilogue as expensive as the GEMM's main loop.  Here
//   erfc(z) = t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-z^2),  t = 1 / (1 + p z),
// Abramowitz & Stegun 7.1.26, |error| <= 1.5e-7 absolute for z >= 0; the negative
// side uses Phi(-x) = 1 - Phi(x) without cancellation.  The same exponential
// serves the density in the derivative.
struct GeluTerms {
  float cdf;   // Phi(x)
  float expo;  // exp(-x^2 / 2)
};
__device__ __forceinline__ GeluTerms gelu_terms(float x) {
  const float z = fabsf(x) * 0.70710678118654752440f;
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, z, 1.0f));
  float p = 1.061405429f;
  p = fmaf(p, t, -1.453152027f);
  p = fmaf(p, t, 1.421413741f);
  p = fmaf(p, t, -0.284496736f);
  p = fmaf(p, t, 0.254829592f);
  const float e = __expf(-z * z);
  const float q = 0.5f * p * t * e;  // Phi(-|x|)
  GeluTerms r;
  r.cdf = x < 0.0f ? q : 1.0f - q;
  r.expo = e;
  return r;
}
// gelu(x) = max(x, 0) - |x| Phi(-|x|): no select between the two halves of Phi, and
// Phi(-|x|) = t (a1/2 + t (a2/2 + ...)) exp2(-x^2 log2(e) / 2), t = 1 / (1 + (p / sqrt 2) |x|),
// straight from x (the same approximation as gelu_terms with the constants folded:
// 11 full-rate operations, one reciprocal and one exp2 per element in the GEMM epilogue).
__device__ __forceinline__ float gelu_exact(float x) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f * 0.70710678118654752440f, ax, 1.0f));
  float p = 0.5f * 1.061405429f;
  p = fmaf(p, t, 0.5f * -1.453152027f);
  p = fmaf(p, t, 0.5f * 1.421413741f);
  p = fmaf(p, t, 0.5f * -0.284496736f);
  p = fmaf(p, t, 0.5f * 0.254829592f);
  const float e = __builtin_amdgcn_exp2f((x * x) * (-0.5f * 1.44269504088896340736f));
  const float q = (p * t) * e;  // Phi(-|x|)
  float pos;  // max(x, 0) as the one instruction (fmaxf adds a pass that quiets NaNs first;
              // a NaN x still gives NaN through the other operand)
  asm("v_max_f32 %0, 0, %1" : "=v"(pos) : "v"(x));
  return fmaf(-ax, q, pos);
}
// d/dx gelu(x) = Phi(x) + x phi(x), phi the standard normal density.
__device__ __forceinline__ float dgelu_exact(float x) {
  const GeluTerms g = gelu_terms(x);
  return fmaf(x * 0.39894228040143267794f, g.expo, g.cdf);
}

// sigmoid(x) = 1 / (1 + exp(-x)); exp overflows to +inf for x < -88 and the
// reciprocal then gives the correct limit 0.
__device__ __forceinline__ float sigmoid_f(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}

// ---- bf16 GEMM ------------------------------------------------------------
// C[M x N] (+)= A * B over a contraction of length Kc, bf16 operands, fp32
// accumulate.  Each operand is either "K-major" (stored [rows][Kc], the
// contraction index contiguous) or "MN-major" (stored [Kc][rows]).
struct GemmArgs {
  const uint16_t* A;
  const uint16_t* B;
  void* C;            // bf16 or fp32, row-major [M][N]
  const void* bias;   // [N] or null: fp32, or the operands' type if bias16
  int bias16;
  uint16_t* Z;        // optional pre-activation copy, bf16 [M][N], ld = ldc
  int M, N, Kc;
  int64_t lda, ldb, ldc;
  int tiles_m, tiles_n;
  int beta;  // 0: C = AB ; 1: C += AB
  // First workgroup of this problem in a launch that runs two problems (launch_gemm_backward), and how many of its
  // last tiles are four workgroups each.
  int wg_first, quartered;
  // Split of the contraction over workgroups (splits > 1): workgroup id / tiles is the
  // split, which covers k_split contraction elements and writes its fp32 partial
  // product to C + split * M * ldc.  0 or 1: no split.
  int splits, k_split;
  // Gate/up forward with the SwiGLU in the epilogue (launch_gemm_swiglu): B holds the gate
  // weights, B2 the up weights (same shape and ldb); C receives silu(gate) * up, G and U
  // (optional, ld = ldc) the two pre-activations; N counts the columns of C.
  const uint16_t* B2;
  uint16_t* G;
  uint16_t* U;
  // Two-term product C = A B + A2 B2 in one pass (launch_gemm_pair): the first k_first
  // elements of the contraction Kc come from (A, B), the others from (A2, B2), which have
  // the leading dimensions of A and B.
  const uint16_t* A2;
  int k_first;
  // Gate/up forward of a few rows (launch_gemm_stream_swiglu): output columns that start at the same line.
  int start_rows;
};

// Sizes go up to 2^31 - 1: what is rounded up to tiles or stages is computed in 64 bits.
__host__ __device__ constexpr int64_t ceil_div(int64_t n, int64_t by) { return (n + by - 1) / by; }
// The 64-deep stages of a contraction of kc that part `part` of `parts` covers.
struct StageRange {
  int first, count;
};
__host__ __device__ constexpr StageRange stages_of_part(int kc, int part, int parts) {
  const int all = (int)ceil_div(kc, 64);   // at most 2^25, times 16 parts 2^29
  if (parts <= 1) return {0, all};
  const int first = part * all / parts;
  return {first, (part + 1) * all / parts - first};
}
static_assert(stages_of_part(0x7fffffff, 0, 1).count == 1 << 25 && stages_of_part(0x7fffffff, 15, 16).first == 15 << 21 &&
                  stages_of_part(0x7fffffff, 15, 16).count == 1 << 21,
              "the longest contraction");

// Address of the bias of output column n.
inline const void* bias_at(const GemmArgs& g, int64_t n) {
  return g.bias == nullptr ? nullptr : (const char*)g.bias + n * (g.bias16 ? 2 : 4);
}

enum GemmLayout { GEMM_NT = 0, GEMM_NN = 1, GEMM_TN = 2 };
// GEMM_NT: A K-major, B K-major   (forward  Y  = X  W^T)
// GEMM_NN: A K-major, B MN-major  (dgrad    dX = dY W  )
// GEMM_TN: A MN-major, B MN-major (wgrad    dW = dY^T X)

int launch_gemm_bf16(GemmLayout layout, const GemmArgs& args, int epilogue,
                     bool out_f32, hipStream_t stream);
// The same kernels on IEEE half operands (v_mfma_f32_16x16x32_f16, half outputs).
int launch_gemm_f16(GemmLayout layout, const GemmArgs& args, int epilogue, bool out_f32,
                    hipStream_t stream);
// dX = dY W and dW (+)= dY^T X of one layer, args as for GEMM_NN and GEMM_TN.  Results are
// those of the two separate launches bit for bit; when the two problems' tile counts leave
// CUs idle one after the other but not together, they run as ONE launch (see gemm_bf16.hip).
int launch_gemm_backward(const GemmArgs& dgrad, const GemmArgs& wgrad, bool half, bool dw_f32,
                         hipStream_t stream);
// GEMMs of shapes that are not made of whole tiles (gemm_edge.h), on the tile the caller
// picks: any M, N, contraction and operand size, row strides below kEdgeMaxLd elements (half
// of that on the tiles of 256 rows).
// FED_*: tiles of gemm_fed_tiles.h, one workgroup on a CU.
enum EdgeTile {
  EDGE_256x256 = 0, EDGE_256x128 = 1, EDGE_128x128 = 2,
  FED_64x64, FED_96x64, FED_64x128, FED_96x128, FED_128x128, FED_96x192, FED_128x192, FED_160x192, FED_128x256, FED_256x128
};
constexpr int64_t kEdgeMaxLd = 1LL << 23;
// Split contraction for problems with few output tiles: into how many parts and on which
// tile (parts = 1: do not split), and the launch: partial products in fp32 to `ws`
// (parts * M * N floats, N rounded up to a multiple of 8), then one pass that adds them in part order, adds the old output if
// args.beta, applies the epilogue and stores args.C.
struct SplitPlan {
  int parts;
  EdgeTile tile;
};
SplitPlan gemm_splits(GemmLayout layout, int64_t M, int64_t N, int64_t Kc, double* us = nullptr);
// What a call with the workspace for gemm_splits' parts does: those parts or fewer, on the tile that is estimated to
// be fastest.
SplitPlan gemm_plan(GemmLayout layout, const GemmArgs& args, int epilogue, bool out_f32);
// widen (input gradient): the result is rounded to the operands' type and stored as fp32.
int launch_gemm_splitk(GemmLayout layout, const GemmArgs& args, int epilogue, bool half, bool out_f32,
                       const SplitPlan& plan, float* ws, hipStream_t stream, bool widen = false);
// The parts of the input gradient's contraction if both gradients of a layer (dY[M][N], W[N][K], X[M][K]) are
// estimated to be faster in one launch than in two, or 0; add: dW += ...; ws holds the parts, parts * M * K floats.
int gemm_backward_parts(int64_t M, int64_t N, int64_t K, bool add);
int launch_gemm_backward_parts(const GemmArgs& dgrad, const GemmArgs& wgrad, bool half, bool dw_f32, int parts,
                               float* ws, hipStream_t stream);
// Row strides from kEdgeMaxLd on, both operands addressed with 64 bits (gemm_far.hip).
int launch_gemm_far(GemmLayout layout, const GemmArgs& args, int epilogue, bool out_f32, bool half,
                    hipStream_t stream);
int launch_gemm_edge_bf16(GemmLayout layout, const GemmArgs& args, int epilogue, bool out_f32,
                          EdgeTile tile, hipStream_t stream);
int launch_gemm_edge_f16(GemmLayout layout, const GemmArgs& args, int epilogue, bool out_f32,
                         EdgeTile tile, hipStream_t stream);
// The same on a FED_* tile; row strides below kEdgeMaxLd / 2.
int launch_gemm_fed_nt_bf16(const GemmArgs& args, int epilogue, bool out_f32, EdgeTile tile, hipStream_t stream);
int launch_gemm_fed_nt_f16(const GemmArgs& args, int epilogue, bool out_f32, EdgeTile tile, hipStream_t stream);
int launch_gemm_fed_rounds(const GemmArgs& args, bool half, EdgeTile tile, hipStream_t stream);
int launch_gemm_fed_nn_tn_bf16(GemmLayout layout, const GemmArgs& args, bool out_f32, EdgeTile tile, hipStream_t stream);
int launch_gemm_fed_nn_tn_f16(GemmLayout layout, const GemmArgs& args, bool out_f32, EdgeTile tile, hipStream_t stream);
// Both gradients of a layer in one launch of 256 x 256 tiles; tiles_m, tiles_n and wg_first set.
int launch_gemm_edge_backward_bf16(const GemmArgs& wgrad, const GemmArgs& dgrad, bool dw_f32,
                                   hipStream_t stream);
int launch_gemm_edge_backward_f16(const GemmArgs& wgrad, const GemmArgs& dgrad, bool dw_f32,
                                  hipStream_t stream);

// Forward products of a few rows (gemm_stream.hip): a stream over the weights; row strides
// below kStreamMaxLd elements.
constexpr int64_t kStreamMaxRows = 64;
// Whether it is also ahead of tiles with the contraction in parts.  Those lose on many weights and win where a
// few workgroups would walk a long contraction; the line lies where they meet over 41397 shapes of 1 to 64 rows,
// 64 to 16384 outputs and contractions of 1024 to 65536 (cold weights, in rows of calls; the pick is 0.2 % off the
// faster one on average, 39 % at worst).  It moves with the share of the CUs that the stream's workgroups fill:
// 3072 outputs and more fill three quarters of them.  us, stream / tiles:
//   64 rows   512 x 4096 12.5 / 11.4    512 x 5120 15.9 / 12.7   4096 x 8192 23.5 / 24.0   4096 x 14336 47 / 37
//   32 rows   512 x 8192 13.5 / 14.5    512 x 28672 51 / 31      4096 x 28672 66 / 64      8192 x 65536 207 / 232
//   15 rows   3904 x 16256 24 / 40      64 x 14144 17.6 / 18.5   64 x 14656 (16 rows) 18.6 / 18.3
//   8 rows    512 x 14336 15.3 / 18.7   512 x 65536 56 / 55      4032 x 30336 40 / 58      4096 x 65536 84 / 143
inline bool stream_ahead(int64_t M, int64_t N, int64_t Kc) {
  if (M > kStreamMaxRows) return false;
  if (N >= 8192 || (N >= 4096 && M <= 32) || (N >= 3072 && M <= 16)) return true;
  if (N >= 3072) return M * Kc <= 524288;
  return Kc <= 65536 && (M <= 8 || M * Kc <= 225000);
}
constexpr int64_t kStreamMaxLd = 1LL << 24;
int launch_gemm_stream(const GemmArgs& args, int epilogue, bool out_f32, bool half, hipStream_t stream);
// The gate/up forward (launch_gemm_swiglu) of up to kStreamMaxRows rows, N a multiple of 8; the two products are
// those of launch_gemm_stream bit for bit.
int launch_gemm_stream_swiglu(const GemmArgs& args, bool half, hipStream_t stream);

// C = silu(A B^T) * (A B2^T) in one launch (both weight matrices [N][Kc], K-major), for
// M % 256 == 0, N % 128 == 0, Kc % 64 == 0 and operands below 2 GiB; AXN_ESHAPE otherwise.
int launch_gemm_swiglu(const GemmArgs& args, bool half, hipStream_t stream);
// The same for any M, N a multiple of 8 (gemm_gate_up.hip), on the tile that is estimated to be fastest; row strides
// below kEdgeMaxLd / 2.  unless_largest: nothing is launched (taken is false) where that is 256 x 256, or within 5 %.
int launch_gemm_swiglu_any(const GemmArgs& args, bool half, bool unless_largest, hipStream_t stream, bool& taken);

// C[M x N] = A B + A2 B2, A / A2 K-major [M][k1], [M][k2], B / B2 MN-major [k1][N], [k2][N]
// (two input-gradient products added in the accumulators): args.Kc = k1 + k2,
// args.k_first = k1.  Shapes of whole 128 x 128 tiles, k1 % 64 == 0 and >= 128,
// k2 % 64 == 0 and >= 64, operands below 2 GiB; AXN_ESHAPE otherwise.
int launch_gemm_pair(const GemmArgs& args, bool half, hipStream_t stream);

// ---- fp32 GEMM (full-precision layers) --------------------------------------
int launch_gemm_f32(GemmLayout layout, const float* A, const float* B, float* C,
                    const float* bias, float* Z, int M, int N, int Kc,
                    int epilogue, int beta, float* ws, size_t ws_bytes, hipStream_t stream);
// Workspace for a contraction in parts (0: it would not be split); ws == nullptr: no split.
size_t gemm_f32_workspace_bytes(GemmLayout layout, int64_t M, int64_t N, int64_t Kc);

// ---- elementwise backward of the bias/GELU epilogue ----------------------
size_t dgelu_dbias_workspace_bytes(int64_t M, int64_t N);
// wide: dY is fp32, rounded to dtype; dbias16: dbias has dtype.
int launch_dgelu_dbias(const void* dY, const void* Z, void* dZ, int dtype, bool wide, void* dbias, bool dbias16,
                       int64_t M, int64_t N, int64_t ld, int beta, void* ws, size_t ws_bytes, hipStream_t stream);
// dst = src, n (a multiple of 8) 16-bit elements as fp32.
int launch_widen(const void* src, float* dst, bool half, int64_t n, hipStream_t stream);

// dst[M][ld_dst] = src[M][N] (row stride ld) of 16-bit elements, zeros behind N; ld_dst a multiple of 8.
int launch_pad_rows16(const void* src, void* dst, int64_t M, int64_t N, int64_t ld, int64_t ld_dst,
                      hipStream_t stream);

// ---- SwiGLU activation of the Llama MLP and its backward -----------------------
int launch_swiglu_fwd(const void* gate, const void* up, void* out, int dtype, int64_t M,
                      int64_t N, int64_t ld, hipStream_t stream);
// ld: row stride of dout, gate and up; ld_out: of dgate and dup
int launch_swiglu_bwd(const void* dout, const void* gate, const void* up, void* dgate, void* dup,
                      int dtype, int64_t M, int64_t N, int64_t ld, int64_t ld_out,
                      hipStream_t stream);

// ---- embedding table: row gather, dense weight gradient, max_norm -------------------
size_t embedding_workspace_bytes(int64_t T, int64_t V);
int launch_embedding_fwd(const int64_t* ids, const void* W, void* out, int elem_bytes, int64_t T,
                         int64_t V, int64_t H, int64_t ldw, int64_t ldo, int* status,
                         hipStream_t stream);
int launch_embedding_bwd(const int64_t* ids, const void* dY, void* dW, int dy_dtype, int dw_dtype,
                         int64_t T, int64_t V, int64_t H, int64_t lddy, int64_t lddw,
                         int64_t padding_idx, int scale_by_freq, int beta, void* ws,
                         size_t ws_bytes, hipStream_t stream);
int launch_embedding_renorm(const int64_t* ids, void* W, int dtype, int64_t T, int64_t V,
                            int64_t H, int64_t ldw, float max_norm, float norm_type, void* ws,
                            size_t ws_bytes, hipStream_t stream);

// ---- multi-tensor optimizer ------------------------------------------------
size_t mt_scan_workspace_bytes(int64_t n, int64_t total);
int launch_mt_scan(const void* const* h_g, const int64_t* h_sizes, int64_t n,
                   int g_dtype, float inv_scale, float max_norm, float norm_type,
                   int accumulate, axn_scan_result* result, void* ws, size_t ws_bytes,
                   hipStream_t stream);
// The same with the partial results in the library's own device array (no workspace).
int launch_mt_scan_noalloc(const void* const* h_g, const int64_t* h_sizes, int64_t n,
                           int g_dtype, float inv_scale, float max_norm, float norm_type,
                           int accumulate, axn_scan_result* result, hipStream_t stream);
int launch_mt_adam(const void* const* h_g, void* const* h_p, void* const* h_m,
                   void* const* h_v, void* const* h_plow, const int64_t* h_sizes,
                   int64_t n, int g_dtype, int plow_dtype, float inv_scale,
                   const axn_scan_result* scan, const axn_adam_hparams& hp,
                   hipStream_t stream);
int launch_mt_scale(void* const* h_g, const int64_t* h_sizes, int64_t n,
                    int g_dtype, float inv_scale, const axn_scan_result* scan,
                    int use_clip, hipStream_t stream);


// The dynamic LDS size a kernel may ask for is an attribute of the kernel on a device: set
// on a kernel's first launch on each device, not on every launch.  `done` is the
// per-kernel-instance record (one bit per device).
inline int allow_lds(const void* kern, size_t lds, std::atomic<unsigned long long>& done) {
  int dev = 0;
  AXN_HIP_TRY(hipGetDevice(&dev));
  const unsigned long long bit = 1ull << (dev & 63);
  if (done.load(std::memory_order_acquire) & bit) return AXN_OK;
  AXN_HIP_TRY(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  done.fetch_or(bit, std::memory_order_release);
  return AXN_OK;
}

}  // namespace axn
