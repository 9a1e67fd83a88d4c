// 16-bit products whose operands have rows 2^23 elements or more apart, which the 32-bit offsets of
// the buffer copies in gemm_edge.h do not span: layers of that many features, and C callers' views
// (the tensor wrappers pack such views first).
//
// What bounds it: latency.  A wave owns 32 x 32 outputs and reads its fragments from global memory
// through 64-bit addresses, 16 bytes a lane where the contraction is contiguous and 2 where it is
// not, no LDS and no barrier.  It is there so that no stride is refused, not for speed: 16 tokens x
// 4096 x 4096 from rows 2^24 apart 46.6 us, the packed copy and the stream over the weights 21.0 us.
#include "gemm_solo.h"

namespace axn {
namespace {

// The 8 contraction elements k .. k + 7 of one row; zeros past the contraction.
template <bool KMAJOR>
__device__ __forceinline__ bf16x8 far_fragment(const uint16_t* base, int64_t ld, int row, int64_t k, int kc) {
  if (KMAJOR && k + 8 <= kc) return *(const bf16x8*)(base + row * ld + k);
  uint16_t v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = k + e < kc ? (KMAJOR ? base[row * ld + k + e] : base[(k + e) * ld + row]) : (uint16_t)0;
  return __builtin_bit_cast(bf16x8, v);
}

// Register v of acc[i][j] in lane (r, q): output row m0 + 16 i + 4 q + v, column n0 + 16 j + r.
template <int EPI, bool OUT_F32, bool HALF>
__device__ __forceinline__ void far_store(const f32x4 (&acc)[2][2], const GemmArgs& g, int64_t m0, int64_t n0) {
  const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t row = m0 + 16 * i + 4 * q + v, col = n0 + 16 * j + r;
        if (row < g.M && col < g.N) store_one<EPI, OUT_F32, HALF>(acc[i][j][v], g, (int)row, (int)col);
      }
}

template <bool AK, bool BKM, bool HALF>
__global__ void __launch_bounds__(64) gemm_far_kernel(const GemmArgs g, int epilogue, int out_f32) {
  const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
  const int64_t m0 = (int64_t)(blockIdx.x / g.tiles_n) * 32, n0 = (int64_t)(blockIdx.x % g.tiles_n) * 32;
  // Rows past the edge read the last one: their products are not stored.
  int row[2], col[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    row[i] = (int)(m0 + 16 * i + r < g.M ? m0 + 16 * i + r : g.M - 1);
    col[i] = (int)(n0 + 16 * i + r < g.N ? n0 + 16 * i + r : g.N - 1);
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int64_t k0 = 0; k0 < g.Kc; k0 += 32) {
    bf16x8 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[i] = far_fragment<AK>(g.A, g.lda, row[i], k0 + 8 * q, g.Kc);
      b[i] = far_fragment<BKM>(g.B, g.ldb, col[i], k0 + 8 * q, g.Kc);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if constexpr (HALF)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i]),
                                                             __builtin_bit_cast(f16x8, b[j]), acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }
  switch (epilogue) {
    case AXN_EPI_NONE:
      if (out_f32) far_store<AXN_EPI_NONE, true, HALF>(acc, g, m0, n0);
      else far_store<AXN_EPI_NONE, false, HALF>(acc, g, m0, n0);
      break;
    case AXN_EPI_BIAS:
      if (out_f32) far_store<AXN_EPI_BIAS, true, HALF>(acc, g, m0, n0);
      else far_store<AXN_EPI_BIAS, false, HALF>(acc, g, m0, n0);
      break;
    case AXN_EPI_BIAS_GELU:
      if (out_f32) far_store<AXN_EPI_BIAS_GELU, true, HALF>(acc, g, m0, n0);
      else far_store<AXN_EPI_BIAS_GELU, false, HALF>(acc, g, m0, n0);
      break;
    case AXN_EPI_GELU:
      far_store<AXN_EPI_GELU, false, HALF>(acc, g, m0, n0);
      break;
  }
}

template <bool HALF>
int launch_far(GemmLayout layout, const GemmArgs& in, int epilogue, bool out_f32, hipStream_t stream) {
  GemmArgs g = in;
  g.tiles_m = (int)ceil_div(g.M, 32);
  g.tiles_n = (int)ceil_div(g.N, 32);
  const long long nwg = (long long)g.tiles_m * g.tiles_n;
  if (nwg > 0x7fffffffLL) {
    set_error("gemm: too many output tiles (%lld)", nwg);
    return AXN_ELIMIT;
  }
  void (*kern)(const GemmArgs, int, int) = layout == GEMM_NT   ? gemm_far_kernel<true, true, HALF>
                                           : layout == GEMM_NN ? gemm_far_kernel<true, false, HALF>
                                                               : gemm_far_kernel<false, false, HALF>;
  hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(64), 0, stream, g, epilogue, out_f32 ? 1 : 0);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

}  // namespace

int launch_gemm_far(GemmLayout layout, const GemmArgs& g, int epilogue, bool out_f32, bool half,
                    hipStream_t stream) {
  return half ? launch_far<true>(layout, g, epilogue, out_f32, stream)
              : launch_far<false>(layout, g, epilogue, out_f32, stream);
}

}  // namespace axn
