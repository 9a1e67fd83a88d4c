// fp32 GEMMs for full-precision Linear layers on gfx950.  The reference's own
// layer tests run in fp32 (axonn/tests/test_intra_layer_fc.py:25); this is the
// same three products as the bf16 path (fully_connected.py:118, :140, :147-151)
// with fp32 operands, for any M, N, K >= 1.
//
// Three kernels.  gemm_f32_split_kernel forms each fp32 product from six bf16 products on LDS
// tiles and carries the large problems; gemm_f32_kernel and gemm_f32_copied_kernel use the fp32 matrix
// instruction, in the same order of sums: they give the same bits.
//
// gemm_f32_kernel: one wave per workgroup owns a (16 FM) x (16 FN) output tile and feeds
// v_mfma_f32_16x16x4_f32 (true fp32 products, fp32 accumulate) straight from
// global memory: no LDS, no barriers.  A 16 x 4 operand block wants, in lane l,
// the element of one row (r = l % 16) and contraction index q = l / 16; MFMA s of a
// 16-deep block takes contraction index 4 q + s from both operands.  Which row of
// the tile lane r of fragment i stands for is free as long as loads and stores
// agree; it is row FM r + i (column FN r + j), so that
//   * a contraction-contiguous operand is read with one 16-byte load per fragment
//     (indices 4 q .. 4 q + 3 of the lane's row),
//   * an operand stored the other way round is read with one FM- (FN-) float load
//     per contraction index (the lane's FM consecutive rows), and
//   * a lane stores FN consecutive output columns at once.
// Its tiles are chosen for many waves (latency hiding by occupancy and by U blocks of loads
// in flight per wave).  It takes any size and alignment, and is left with the short contractions of the rest.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "axn_internal.h"

namespace axn {
namespace {

typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

// Full-precision layers keep the library erff.
__device__ __forceinline__ float gelu_erff(float z) {
  return 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f));
}

template <int F>
struct VecOf {
  typedef float type __attribute__((ext_vector_type(F)));
};
template <>
struct VecOf<1> {
  typedef float type;
};
template <int F>
__device__ __forceinline__ float vec_get(const typename VecOf<F>::type& v, int i) {
  if constexpr (F == 1) return v;
  else return v[i];
}

// One 16-deep block of one operand for the F fragments of a lane: x[f][s] is the
// element of row F r + f (clamped to the last row) and contraction index k + s.
//   KMAJOR: element (row, k) at base[row * Kc + k]; else at base[k * rows + row]
//   VEC:    Kc % 4 == 0, a 16-byte aligned base and (unless KMAJOR) rows % F == 0:
//           vector loads
//   GUARD:  indices >= k_end read as zero (the end of a contraction, or of a part of one)
template <bool KMAJOR, int F, bool VEC, bool GUARD>
__device__ __forceinline__ void load_block(float (&x)[F][4], const float* __restrict__ base,
                                           int row0, int rows, int k, int Kc, int k_end) {
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int s = 0; s < 4; ++s) x[f][s] = 0.f;
  if (KMAJOR) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const float* p = base + (int64_t)min(row0 + f, rows - 1) * Kc;
      if (VEC) {  // the four indices are in or out together
        if (!GUARD || k < k_end) {
          const f32x4 v = *(const f32x4*)(p + k);
#pragma unroll
          for (int s = 0; s < 4; ++s) x[f][s] = v[s];
        }
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (!GUARD || k + s < k_end) x[f][s] = p[k + s];
      }
    }
  } else if (VEC) {  // the F rows are in or out together
    const float* p = base + min(row0, rows - F);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (!GUARD || k + s < k_end) {
        const typename VecOf<F>::type v = *(const typename VecOf<F>::type*)(p + (int64_t)(k + s) * rows);
#pragma unroll
        for (int f = 0; f < F; ++f) x[f][s] = vec_get<F>(v, f);
      }
  } else {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const float* p = base + min(row0 + f, rows - 1);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (!GUARD || k + s < k_end) x[f][s] = p[(int64_t)(k + s) * rows];
    }
  }
}

template <int FM, int FN>
__device__ __forceinline__ void clear(f32x4 (&acc)[FM][FN]) {
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// acc[i][j] += the products of contraction indices [k_begin, k_end) for rows arow + i and columns
// bcol + j of the lane, in fp32 MFMAs; this wave takes the 16 U-deep chunks first, first + STEP, ...
template <bool AK, bool BKM, int FM, int FN, int U, bool VEC, int STEP, bool LONG>
__device__ __forceinline__ void direct_tile(f32x4 (&acc)[FM][FN], const float* __restrict__ A,
                                            const float* __restrict__ B, int arow, int bcol, int M, int N,
                                            int Kc, int k_begin, int k_end, int first) {
  const int q = (threadIdx.x & 63) >> 4;
  auto blocks = [&](auto guard_, int k0, auto nblk_) {
    constexpr bool GUARD = decltype(guard_)::value;
    constexpr int NB = decltype(nblk_)::value;
    float a[NB][FM][4], b[NB][FN][4];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int k = k0 + 16 * u + 4 * q;
      load_block<AK, FM, VEC, GUARD>(a[u], A, arow, M, k, Kc, k_end);
      load_block<BKM, FN, VEC, GUARD>(b[u], B, bcol, N, k, Kc, k_end);
    }
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i][s], b[u][j][s], acc[i][j], 0, 0, 0);
  };
  const int whole = k_begin + (k_end - k_begin) / (16 * U) * (16 * U);  // the part made of whole chunks
  // LONG: the loops are left by a difference, for an index past the end of the longest contraction overflows an
  // int.  The test costs an instruction or two a chunk, but 12 % where the addresses are strided (256 x 4480 x 1992,
  // input gradient), and unsigned, 64-bit or counted indices leave fewer loads in flight: a variant of its own.
  for (int k0 = k_begin + first * 16 * U; k0 < whole; k0 += STEP * 16 * U) {
    blocks(std::false_type{}, k0, std::integral_constant<int, U>{});
    if (LONG && whole - k0 <= STEP * 16 * U) break;
  }
  for (int k0 = whole + first * 16; k0 < k_end; k0 += STEP * 16) {
    blocks(std::true_type{}, k0, std::integral_constant<int, 1>{});
    if (LONG && k_end - k0 <= STEP * 16) break;
  }
}

// Whether the lane's operands hold a non-zero number under `bound`.
template <bool AK, bool BKM, int FM, int FN, bool VEC>
__device__ __forceinline__ bool tiny_operands(const float* __restrict__ A, const float* __restrict__ B, int arow,
                                              int bcol, int M, int N, int Kc, int k_begin, int k_end, float bound) {
  const int q = (threadIdx.x & 63) >> 4;
  bool tiny = false;
  auto chunk = [&](auto guard_, int k0) {
    constexpr bool GUARD = decltype(guard_)::value;
    float a[FM][4], b[FN][4];
    load_block<AK, FM, VEC, GUARD>(a, A, arow, M, k0 + 4 * q, Kc, k_end);
    load_block<BKM, FN, VEC, GUARD>(b, B, bcol, N, k0 + 4 * q, Kc, k_end);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int i = 0; i < FM; ++i) tiny |= a[i][s] != 0.f && fabsf(a[i][s]) < bound;
#pragma unroll
      for (int j = 0; j < FN; ++j) tiny |= b[j][s] != 0.f && fabsf(b[j][s]) < bound;
    }
  };
  const int whole = k_begin + (k_end - k_begin) / 16 * 16;
  for (int k0 = k_begin; k0 < whole; k0 += 16) chunk(std::false_type{}, k0);
  if (whole < k_end) chunk(std::true_type{}, whole);
  return tiny;
}

// Stores FN results of a row, columns bcol ...
template <int EPI, int FN, bool VEC>
__device__ __forceinline__ void store_row(float (&x)[FN], float* __restrict__ C, const float* __restrict__ bias,
                                          float* __restrict__ Z, int row, int bcol, int M, int N, int beta) {
  using vec = typename VecOf<FN>::type;
  if (row >= M) return;
  const int64_t o = (int64_t)row * N + bcol;
  if (VEC) {  // N % FN == 0: the lane's FN columns are in or out together
    if (bcol >= N) return;
    if (EPI == AXN_EPI_BIAS || EPI == AXN_EPI_BIAS_GELU) {
      const vec bv = *(const vec*)(bias + bcol);
#pragma unroll
      for (int j = 0; j < FN; ++j) x[j] += vec_get<FN>(bv, j);
    }
    vec y;
    if (EPI == AXN_EPI_BIAS_GELU || EPI == AXN_EPI_GELU) {
      if (Z != nullptr) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (FN == 1) y = x[j];
          else y[j] = x[j];
        }
        *(vec*)(Z + o) = y;
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) x[j] = gelu_erff(x[j]);
    }
    if (beta) {
      const vec old = *(const vec*)(C + o);
#pragma unroll
      for (int j = 0; j < FN; ++j) x[j] += vec_get<FN>(old, j);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (FN == 1) y = x[j];
      else y[j] = x[j];
    }
    *(vec*)(C + o) = y;
  } else {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if (bcol + j >= N) continue;
      float t = x[j];
      if (EPI == AXN_EPI_BIAS || EPI == AXN_EPI_BIAS_GELU) t += bias[bcol + j];
      if (EPI == AXN_EPI_BIAS_GELU || EPI == AXN_EPI_GELU) {
        if (Z != nullptr) Z[o + j] = t;
        t = gelu_erff(t);
      }
      if (beta) t += C[o + j];
      C[o + j] = t;
    }
  }
}

// Stores a wave's 16 FM x 16 FN results at (m0, n0): register v of acc[i][j] in lane (r, q) is
// output row m0 + FM (4 q + v) + i, column n0 + FN r + j.
template <int EPI, int FM, int FN, bool VEC>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[FM][FN], float* __restrict__ C,
                                           const float* __restrict__ bias, float* __restrict__ Z, int m0,
                                           int n0, int M, int N, int beta) {
  const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float x[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) x[j] = acc[i][j][v];
      store_row<EPI, FN, VEC>(x, C, bias, Z, m0 + FM * (4 * q + v) + i, n0 + FN * r, M, N, beta);
    }
}

// WAVES > 1: the waves of a workgroup share one tile and take the 16 U-deep chunks of
// the contraction in turn; their partial sums meet in LDS and are added in wave order.
template <bool AK, bool BKM, int EPI, int FM, int FN, int U, bool VEC, int WAVES, bool LONG>
__global__ void __launch_bounds__(64 * WAVES)
    gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                    float* __restrict__ C, const float* __restrict__ bias,
                    float* __restrict__ Z, int M, int N, int Kc, int tiles_n, int beta) {
  const int lane = threadIdx.x & 63;
  const int wave = WAVES > 1 ? threadIdx.x >> 6 : 0;
  const int r = lane & 15;
  const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - tm * tiles_n;
  const int m0 = tm * 16 * FM, n0 = tn * 16 * FN;
  f32x4 acc[FM][FN];
  clear(acc);
  // Rows and columns past the edge read a valid one: their products land in output
  // elements that are never stored.
  direct_tile<AK, BKM, FM, FN, U, VEC, WAVES, LONG>(acc, A, B, m0 + FM * r, n0 + FN * r, M, N, Kc, 0, Kc, wave);

  if constexpr (WAVES > 1) {
    __shared__ f32x4 part[WAVES - 1][FM * FN][64];
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) part[wave - 1][i * FN + j][lane] = acc[i][j];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] += part[w][i * FN + j][lane];
  }

  store_tile<EPI, FM, FN, VEC>(acc, C, bias, Z, m0, n0, M, N, beta);
}

// ---- the native products with their operands copied to LDS ahead -----------------------
constexpr uint32_t kOutside = 0x80000000u;   // an offset behind every buffer: the copy writes zeros

// One operand of a unit, 32 contraction indices of 16 F rows (columns), in a wave's own LDS: 2 F copies of 1 KB.
//   KMAJOR: [row 16 i + r][32], row F r + i of the tile; the eight 16-byte pieces of a row are permuted by r / 2, so that
//           the 16 lanes of a fragment read hit 16 different bank groups
//   else    two blocks of 16 contraction indices, [4 s + q][16 F], index 4 q + s of the block
template <bool KMAJOR, int F>
struct Copied {
  static constexpr int COPIES = 2 * F, BYTES = 2048 * F;
  const char* base;
  int64_t left;           // bytes of the operand from there on
  uint32_t pitch, offset[KMAJOR ? 2 : 1];
  int index[2], Kc;       // KMAJOR: first contraction index of the lane's piece
  __device__ __forceinline__ void start(const float* from, int first, int rows, int K) {
    const int lane = threadIdx.x & 63;
    Kc = K;
    if constexpr (KMAJOR) {
      base = (const char*)(from + (int64_t)first * K);
      left = ((int64_t)rows - first) * K * 4;
      pitch = (uint32_t)K * 4;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        index[p] = 4 * ((lane & 7) ^ (4 * p + (lane >> 4)));
        offset[p] = (uint32_t)(F * (8 * p + (lane >> 3))) * pitch + (uint32_t)index[p] * 4;
      }
    } else {
      base = (const char*)(from + first);
      left = ((int64_t)rows * K - first) * 4;
      pitch = (uint32_t)rows * 4;
      if constexpr (F == 4) offset[0] = (uint32_t)(4 * (lane >> 4)) * pitch + 16 * (lane & 15);
      else if constexpr (F == 2) offset[0] = (uint32_t)(4 * ((lane >> 3) & 3) + (lane >> 5)) * pitch + 16 * (lane & 7);
      else offset[0] = (uint32_t)(4 * ((lane >> 2) & 3) + (lane >> 4)) * pitch + 16 * (lane & 3);
    }
  }
  // Starts the copies of contraction indices k .. k + 31; those behind the end come as zeros.
  __device__ __forceinline__ void copy(int k, char* lds) const {
    const int64_t skip = (int64_t)k * (KMAJOR ? 4 : pitch);
    const int64_t rest = left - skip;
    const int n = k >= Kc ? 0 : rest > 0x7fffffff ? 0x7fffffff : (int)rest;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (k >= Kc ? 0 : skip)), 0, n, 0x00020000);
#pragma unroll
    for (int j = 0; j < COPIES; ++j) {
      uint32_t at;
      if constexpr (KMAJOR) at = k + index[j & 1] < Kc ? offset[j & 1] + (uint32_t)(j >> 1) * pitch : kOutside;
      else at = offset[0] + (uint32_t)(16 * (j / F) + (F == 4 ? j % 4 : F == 2 ? 2 * (j % 2) : 0)) * pitch;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(lds + 1024 * j), 16, (int)at,
                                               0, 0, 0);
    }
  }
  // Where the lane's reads of block u start.
  __device__ __forceinline__ static uint32_t read_at(int u) {
    const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
    if constexpr (KMAJOR) return 128 * r + 16 * (((4 * u + q) ^ (r >> 1)) & 7);
    else return u * (BYTES / 2) + 64 * F * q + 4 * F * r;
  }
};

// An operand's fragments of a block of 16 contraction indices.  KMAJOR: k[i] holds indices 4 q .. 4 q + 3 of row i, else
// m[s] rows 0 .. F - 1 of index 4 q + s.
template <bool KMAJOR, int F>
struct Fragments {
  f32x4 k[F];
  __device__ __forceinline__ float at(int i, int s) const { return k[i][s]; }
};
template <int F>
struct Fragments<false, F> {
  typename VecOf<F>::type m[4];
  __device__ __forceinline__ float at(int i, int s) const { return vec_get<F>(m[s], i); }
};
// Both operands' fragments of the blocks that a step multiplies between two waits: four blocks (two units) at F = 1, two
// at F = 2, one of the two at F = 4.  pa, pb: where the lane's reads of blocks 0 and 1 of a unit start.
#define AXN_RD(size, to, from, at) "ds_read_" size " %" #to ", %" #from " offset:" #at "\n\t"
#define AXN_RD4(size, t0, t1, t2, t3, from, a0, a1, a2, a3) \
  AXN_RD(size, t0, from, a0) AXN_RD(size, t1, from, a1) AXN_RD(size, t2, from, a2) AXN_RD(size, t3, from, a3)
#define AXN_WAIT "s_waitcnt lgkmcnt(0)"
#define AXN_V4(x, y, z, w) "=&v"(x), "=&v"(y), "=&v"(z), "=&v"(w)
#define AXN_M(f) AXN_V4(f.m[0], f.m[1], f.m[2], f.m[3])
#define AXN_K(f) AXN_V4(f.k[0], f.k[1], f.k[2], f.k[3])
__device__ __forceinline__ void read_step(Fragments<true, 1> (&a)[4], Fragments<true, 1> (&b)[4], const uint32_t (&pa)[2],
                                          const uint32_t (&pb)[2]) {
  asm volatile(AXN_RD("b128", 0, 8, 0) AXN_RD("b128", 4, 10, 0) AXN_RD("b128", 1, 9, 0) AXN_RD("b128", 5, 11, 0)
               AXN_RD("b128", 2, 8, 4096) AXN_RD("b128", 6, 10, 4096) AXN_RD("b128", 3, 9, 4096) AXN_RD("b128", 7, 11, 4096) AXN_WAIT
               : AXN_V4(a[0].k[0], a[1].k[0], a[2].k[0], a[3].k[0]), AXN_V4(b[0].k[0], b[1].k[0], b[2].k[0], b[3].k[0])
               : "v"(pa[0]), "v"(pa[1]), "v"(pb[0]), "v"(pb[1]) : "memory");
}
__device__ __forceinline__ void read_step(Fragments<true, 1> (&a)[4], Fragments<false, 1> (&b)[4], const uint32_t (&pa)[2],
                                          const uint32_t (&pb)[2]) {
  asm volatile(AXN_RD("b128", 0, 20, 0) AXN_RD("b128", 1, 21, 0) AXN_RD("b128", 2, 20, 4096) AXN_RD("b128", 3, 21, 4096)
               AXN_RD4("b32", 4, 5, 6, 7, 22, 0, 256, 512, 768) AXN_RD4("b32", 8, 9, 10, 11, 22, 1024, 1280, 1536, 1792)
               AXN_RD4("b32", 12, 13, 14, 15, 22, 4096, 4352, 4608, 4864) AXN_RD4("b32", 16, 17, 18, 19, 22, 5120, 5376, 5632, 5888) AXN_WAIT
               : AXN_V4(a[0].k[0], a[1].k[0], a[2].k[0], a[3].k[0]), AXN_M(b[0]), AXN_M(b[1]), AXN_M(b[2]), AXN_M(b[3])
               : "v"(pa[0]), "v"(pa[1]), "v"(pb[0]) : "memory");
}
__device__ __forceinline__ void read_step(Fragments<true, 2> (&a)[2], Fragments<true, 2> (&b)[2], const uint32_t (&pa)[2],
                                          const uint32_t (&pb)[2]) {
  asm volatile(AXN_RD("b128", 0, 8, 0) AXN_RD("b128", 1, 8, 2048) AXN_RD("b128", 4, 10, 0) AXN_RD("b128", 5, 10, 2048)
               AXN_RD("b128", 2, 9, 0) AXN_RD("b128", 3, 9, 2048) AXN_RD("b128", 6, 11, 0) AXN_RD("b128", 7, 11, 2048) AXN_WAIT
               : AXN_V4(a[0].k[0], a[0].k[1], a[1].k[0], a[1].k[1]), AXN_V4(b[0].k[0], b[0].k[1], b[1].k[0], b[1].k[1])
               : "v"(pa[0]), "v"(pa[1]), "v"(pb[0]), "v"(pb[1]) : "memory");
}
__device__ __forceinline__ void read_step(Fragments<true, 2> (&a)[2], Fragments<false, 2> (&b)[2], const uint32_t (&pa)[2],
                                          const uint32_t (&pb)[2]) {
  asm volatile(AXN_RD("b128", 0, 12, 0) AXN_RD("b128", 1, 12, 2048) AXN_RD("b128", 2, 13, 0) AXN_RD("b128", 3, 13, 2048)
               AXN_RD4("b64", 4, 5, 6, 7, 14, 0, 512, 1024, 1536) AXN_RD4("b64", 8, 9, 10, 11, 14, 2048, 2560, 3072, 3584) AXN_WAIT
               : AXN_V4(a[0].k[0], a[0].k[1], a[1].k[0], a[1].k[1]), AXN_M(b[0]), AXN_M(b[1])
               : "v"(pa[0]), "v"(pa[1]), "v"(pb[0]) : "memory");
}
__device__ __forceinline__ void read_step(Fragments<false, 2> (&a)[2], Fragments<false, 2> (&b)[2], const uint32_t (&pa)[2],
                                          const uint32_t (&pb)[2]) {
  asm volatile(AXN_RD4("b64", 0, 1, 2, 3, 16, 0, 512, 1024, 1536) AXN_RD4("b64", 8, 9, 10, 11, 17, 0, 512, 1024, 1536)
               AXN_RD4("b64", 4, 5, 6, 7, 16, 2048, 2560, 3072, 3584) AXN_RD4("b64", 12, 13, 14, 15, 17, 2048, 2560, 3072, 3584) AXN_WAIT
               : AXN_M(a[0]), AXN_M(a[1]), AXN_M(b[0]), AXN_M(b[1]) : "v"(pa[0]), "v"(pb[0]) : "memory");
}
__device__ __forceinline__ void read_block(Fragments<true, 4>& a, Fragments<true, 4>& b, uint32_t pa, uint32_t pb) {
  asm volatile(AXN_RD4("b128", 0, 1, 2, 3, 8, 0, 2048, 4096, 6144) AXN_RD4("b128", 4, 5, 6, 7, 9, 0, 2048, 4096, 6144) AXN_WAIT
               : AXN_K(a), AXN_K(b) : "v"(pa), "v"(pb) : "memory");
}
__device__ __forceinline__ void read_block(Fragments<true, 4>& a, Fragments<false, 4>& b, uint32_t pa, uint32_t pb) {
  asm volatile(AXN_RD4("b128", 0, 1, 2, 3, 8, 0, 2048, 4096, 6144) AXN_RD4("b128", 4, 5, 6, 7, 9, 0, 1024, 2048, 3072) AXN_WAIT
               : AXN_K(a), AXN_M(b) : "v"(pa), "v"(pb) : "memory");
}
__device__ __forceinline__ void read_block(Fragments<false, 4>& a, Fragments<false, 4>& b, uint32_t pa, uint32_t pb) {
  asm volatile(AXN_RD4("b128", 0, 1, 2, 3, 8, 0, 1024, 2048, 3072) AXN_RD4("b128", 4, 5, 6, 7, 9, 0, 1024, 2048, 3072) AXN_WAIT
               : AXN_M(a), AXN_M(b) : "v"(pa), "v"(pb) : "memory");
}
#undef AXN_RD
#undef AXN_RD4
#undef AXN_WAIT
#undef AXN_V4
#undef AXN_M
#undef AXN_K

// Tile id of an output of tiles_m x tiles_n: the workgroups of a chiplet (every eighth) have neighbouring ones, in
// groups of eight rows.
__device__ __forceinline__ void chiplet_tile(unsigned id, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr unsigned kChiplets = 8, kRows = 8;
  const unsigned tiles = tiles_m * tiles_n, each = tiles / kChiplets, rest = tiles % kChiplets;
  const unsigned chiplet = id % kChiplets, t = chiplet * each + min(chiplet, rest) + id / kChiplets;
  const unsigned group = t / (kRows * tiles_n), first = group * kRows, high = min(kRows, tiles_m - first);
  const unsigned in = t - group * kRows * tiles_n;
  tm = first + in % high, tn = in / high;
}

// What bounds gemm_f32_kernel is that a wave waits for each chunk's loads before it multiplies, 1 to 2 us from HBM, and
// that an operand stored along the output is loaded 64 bytes a row and four bytes a lane.  Here a wave copies its own
// operands to its own part of LDS, whole lines and up to 24 KB ahead, and waits for nobody: no barrier in the loop.
// Its reads wait in the statement that issues them; a second workgroup on the CU (64 KB of LDS each up to F = 2) fills
// that.  us, operands from HBM, gemm_f32_kernel / this:
//   64 x 4096, contraction 1024, bias and GELU 18.0 / 10.9     1024 x 4096 weight gradient of 64 tokens  15.6 / 10.4
//   64 x 1024, contraction 4096               22.3 / 13.6      the same of 256 tokens                   45.6 / 21.9
//   256 x 4096, contraction 1024              41.0 / 26.6      1200 x 600, 1000 tokens                  41.2 / 23.4
//   64 x 1024, contraction 4096, input gradient 55.3 / 18.5    256 x 1024, contraction 4096, input gradient 63.9 / 29.8
// Twice the slots cost more (a workgroup a CU: 64 x 4096 above 13 -> 25 at F = 1); so do 32 x 32 tiles where 16 x 16 give a
// workgroup for every CU (64 x 1024 above 29).  256 x 4096 x 1024 are 14 us at the rate of the matrix cores.
//
// TOGETHER: the four waves of a workgroup have one tile and the 64-deep chunks of its contraction in turn (what is left,
// in blocks of 16); their sums are added in wave order.  Else a tile each, a square of two by two.
template <bool AK, bool BKM, int EPI, int F, int SLOTS, bool TOGETHER>
__global__ void __launch_bounds__(256)
    gemm_f32_copied_kernel(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                           const float* __restrict__ bias, float* __restrict__ Z, int M, int N, int Kc, int tiles_m,
                           int tiles_n, int beta) {
  using OA = Copied<AK, F>;
  using OB = Copied<BKM, F>;
  constexpr int UNIT = OA::BYTES + OB::BYTES, EACH = OA::COPIES + OB::COPIES;
  constexpr int STEP = F == 1 ? 2 : 1;   // units between two waits
  static_assert(SLOTS % STEP == 0 && (SLOTS - STEP) * EACH <= 63, "the count of a wait has six bits");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  chiplet_tile(blockIdx.x, tiles_m, tiles_n, tm, tn);
  if constexpr (!TOGETHER) tm = 2 * tm + (wave >> 1), tn = 2 * tn + (wave & 1);
  const int m0 = tm * 16 * F, n0 = tn * 16 * F;
  if (!TOGETHER && (m0 >= M || n0 >= N)) return;
  OA a;
  OB b;
  a.start(A, m0, M, Kc);
  b.start(B, n0, N, Kc);
  const int chunks = Kc / 64, own = (chunks - wave + 3) / 4, tail = chunks * 64 + 16 * wave;
  const int units = TOGETHER ? 2 * own + (tail < Kc) : (Kc + 31) / 32;
  auto index_of = [&](int u) {
    if constexpr (TOGETHER) return u < 2 * own ? 64 * (4 * (u >> 1) + wave) + 32 * (u & 1) : u == 2 * own ? tail : Kc;
    else return 32 * u;
  };
  char* const mine = lds + wave * SLOTS * UNIT;
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)mine;
  const uint32_t ra[2] = {at + OA::read_at(0), at + OA::read_at(1)};
  const uint32_t rb[2] = {at + OA::BYTES + OB::read_at(0), at + OA::BYTES + OB::read_at(1)};
  f32x4 acc[F][F];
  clear(acc);
#pragma unroll
  for (int u = 0; u < SLOTS; ++u) {
    a.copy(index_of(u), mine + u * UNIT);
    b.copy(index_of(u), mine + u * UNIT + OA::BYTES);
  }
  uint32_t slot = 0;
#pragma unroll 1
  for (int u = 0; u < units; u += STEP) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - STEP) * EACH) : "memory");
    Fragments<AK, F> fa[2 * STEP];
    Fragments<BKM, F> fb[2 * STEP];
    auto multiply = [&](int h) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[h].at(i, s), fb[h].at(j, s), acc[i][j], 0, 0, 0);
    };
    auto refill = [&]() {
#pragma unroll
      for (int v = 0; v < STEP; ++v) {
        a.copy(index_of(u + SLOTS + v), mine + slot + v * UNIT);
        b.copy(index_of(u + SLOTS + v), mine + slot + v * UNIT + OA::BYTES);
      }
    };
    const uint32_t pa[2] = {ra[0] + slot, ra[1] + slot}, pb[2] = {rb[0] + slot, rb[1] + slot};
    if constexpr (F == 4) {   // (two blocks' fragments would take half of the registers)
      read_block(fa[0], fb[0], pa[0], pb[0]);
      multiply(0);
      read_block(fa[1], fb[1], pa[1], pb[1]);
      refill();
    } else {
      read_step(fa, fb, pa, pb);
      refill();
      multiply(0);
    }
    if (!TOGETHER || u < 2 * own) {   // (else what is left: one block)
#pragma unroll
      for (int h = 1; h < 2 * STEP; ++h) multiply(h);
    }
    slot = slot + STEP * UNIT == SLOTS * UNIT ? 0 : slot + STEP * UNIT;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (TOGETHER) {
    // wave v adds and stores register v of every block
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) ((float*)mine)[((i * F + j) * 4 + v) * 64 + lane] = acc[i][j][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < F; ++i) {
      float x[F];
#pragma unroll
      for (int j = 0; j < F; ++j) {
        const int o = ((i * F + j) * 4 + wave) * 64 + lane;
        x[j] = ((const float*)lds)[o];
#pragma unroll
        for (int w = 1; w < 4; ++w) x[j] += ((const float*)(lds + w * SLOTS * UNIT))[o];
      }
      store_row<EPI, F, true>(x, C, bias, Z, m0 + F * (4 * q + wave) + i, n0 + F * r, M, N, beta);
    }
  } else {
    store_tile<EPI, F, F, true>(acc, C, bias, Z, m0, n0, M, N, beta);
  }
}

// ---- fp32 products on the 16-bit matrix units ---------------------------------
// v_mfma_f32_16x16x4_f32 runs at a sixteenth of the bf16 rate.  A float is the sum of three bf16
// numbers (8 significant bits each; the remainders are exact), so a product of floats is nine products
// of bf16, each exact in fp32.  The six that are not below 2^-24 of the whole are taken.  a1 b1 goes to
// one accumulator, the five smaller ones, least first, to another that is added at the end: its roundings
// are 2^-8 as large, so the sum sees one rounding per 32 contraction indices (the native instruction: one
// per 4).  Error against 64 bits, normal operands, native / this: contraction of 128 2.0e-7 / 6.6e-8,
// 1024 5.7e-7 / 1.9e-7, 4096 (native by four waves) 5.7e-7 / 4.0e-7; in one accumulator 4096 has 1.0e-6.
//
// Results that are one or two products (rows with as many non-zero elements) miss what the dropped products
// hold: against 64 bits, in 2^-24 of the sum of the magnitudes, native / this: one product 1.0 / 1.7 at most
// and 0.424 / 0.435 rms, two 2.0 / 2.7 and 0.521 / 0.537; from three on the native instruction's rounding of
// every product weighs more (rms of 3 0.602 / 0.585, of 8 0.902 / 0.642, of 64 2.40 / 0.86).  With two more of
// the three products one is 1.0 again and the kernel 16 to 22 % slower (2048 x 1024, contraction 4096: 97 us,
// 111), which dense sums, nearer to exact as they are, do not pay for.
//
// What three bf16 numbers cannot carry, and where the native products (direct_tile) take over, wave by wave:
//   * an infinity has no remainder, the largest floats round to one, and partial products far below the
//     result lose bits: a wave whose results hold a NaN, an infinity or a non-zero magnitude under 2^-64;
//   * the conversion rounds to multiples of 2^-133 (the matrix instruction itself keeps subnormals), so a
//     number under 2^-110 is off by up to 2^-134.  Times less than 2^16 that is nothing to a result of 2^-64
//     and more.  A workgroup that staged a larger number has its waves look through their operands for
//     numbers under 2^-110;
//   * a result of exactly zero may be one that was lost: those waves look for numbers under 2^-62 (a product
//     of two that are larger is a normal number).  Zero rows (padding) have none and keep their zeros.
// A look costs what reading the operands once more costs (2048 x 4096 x 1024 in a row of launches: 106 us, with
// half of the rows zero 142, with a zero row in every wave 198; four chunks of the look in flight made no
// difference); the largest magnitude, kept while staging, half an instruction an element (nothing
// measurable, 3 to 4 % of a weight gradient: 4096 x 2048 x 2048 170 -> 176 us).
//
// Four waves (2 x 2) own a 32 FM x 32 FN tile.  Each thread loads its share of a 32-deep stage into
// registers one stage ahead, splits it and writes three bf16 planes to LDS ([row][32], 64 bytes a row);
// splitting before LDS costs each element once a workgroup instead of once a wave.  Row rho of a plane is
// row F (rho % 32) + rho / 32 of the tile, for both storage orders: the thread that holds F consecutive
// rows of a contraction-strided operand writes to F places a bank apart from its neighbours', and a
// lane's fragments are F consecutive rows (columns), as direct_tile and store_tile have them.  A row's
// 16-byte pieces are permuted by part_of(rho) so that any 16 lanes of a fragment read hit 16 different
// 16-byte bank groups.
// LDS is single-buffered (48 KB for 128 x 128) so that two workgroups share a CU and fill each other's
// barriers.  2048 x 4096, contraction 1024: 86 us, 200 TFLOP/s of fp32 products (native 201 us), in a row of launches
// 110.  What bounds it is the work of a stage together, six products and both operands' splitting in every workgroup
// (matrix cores busy 47 % of the time, vector instructions 30 %, at 2.17 GHz): two LDS buffers with one barrier (one
// workgroup a CU) 122 us, splitting by truncation without the conversions 97, against 98 in the same run; the next
// stage's splitting between the matrix instructions 110 to 117 us against 107 to 112.
template <int F>
struct Planes {
  uint16_t at[3][32 * F][32];
};

__device__ __forceinline__ int part_of(int rho) {
  const int g = (rho >> 2) & 3;
  return ((g << 1) ^ ((g >> 1) * 3)) & 3;  // 0 2 3 1
}

// Four floats as three times four bf16.
__device__ __forceinline__ void split4(const float (&x)[4], uint2 (&out)[3]) {
  float rest[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    uint32_t u[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x2 v = {rest[2 * h], rest[2 * h + 1]};
      u[h] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
      if (p < 2) {
        rest[2 * h] -= __builtin_bit_cast(float, u[h] << 16);
        rest[2 * h + 1] -= __builtin_bit_cast(float, u[h] & 0xffff0000u);
      }
    }
    out[p] = uint2{u[0], u[1]};
  }
}

// Row group g (F rows) and quad (4 contraction indices) a thread stages, one of 32 x 8.
template <bool KMAJOR>
__device__ __forceinline__ void my_share(int& g, int& quad) {
  const int t = threadIdx.x;
  g = KMAJOR ? t >> 3 : t & 31;
  quad = KMAJOR ? t & 7 : t >> 5;
}

template <bool KMAJOR, int F>
__device__ __forceinline__ void put_stage(Planes<F>& lds, const float (&x)[F][4]) {
  int g, quad;
  my_share<KMAJOR>(g, quad);
  const int at = (((quad >> 1) ^ part_of(g)) << 3) + ((quad & 1) << 2);  // 32 i does not change part_of
#pragma unroll
  for (int i = 0; i < F; ++i) {
    uint2 p[3];
    split4(x[i], p);
#pragma unroll
    for (int s = 0; s < 3; ++s) *(uint2*)&lds.at[s][32 * i + g][at] = p[s];
  }
}

// The larger of m and the magnitudes (fmaxf would quiet NaNs first, an instruction each).
template <int F>
__device__ __forceinline__ float max_magnitude(float m, const float (&x)[F][4]) {
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int s = 0; s < 4; s += 2) asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(x[i][s]), "v"(x[i][s + 1]));
  return m;
}

// The parts of the five smaller products, least first.
constexpr int kPartA[5] = {2, 0, 1, 1, 0}, kPartB[5] = {0, 2, 1, 0, 1};

template <int FM, int FN>
__device__ __forceinline__ void split_stage(f32x4 (&acc)[FM][FN], f32x4 (&low)[FM][FN], const Planes<FM>& la,
                                            const Planes<FN>& lb) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, at = ((lane >> 4) ^ part_of(r)) << 3;
  const int ra = 16 * (wave >> 1) + r, rb = 16 * (wave & 1) + r;
  bf16x8 a[FM][3];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int p = 0; p < 3; ++p) a[i][p] = *(const bf16x8*)&la.at[p][32 * i + ra][at];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    bf16x8 b[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) b[p] = *(const bf16x8*)&lb.at[p][32 * j + rb][at];
#pragma unroll
    for (int t = 0; t < 5; ++t)
#pragma unroll
      for (int i = 0; i < FM; ++i)
        low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][kPartA[t]], b[kPartB[t]], low[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < FM; ++i)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][0], b[0], acc[i][j], 0, 0, 0);
  }
}

// parts > 1: workgroup id / tiles is the part, which covers k_part contraction indices and stores
// its products at C + part * M * N.
template <bool AK, bool BKM, int EPI, int FM, int FN, bool VEC>
__global__ void __launch_bounds__(256, 2)
    gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ B,
                          float* __restrict__ C, const float* __restrict__ bias, float* __restrict__ Z,
                          int M, int N, int Kc, int tiles_m, int tiles_n, int k_part, int beta) {
  __shared__ Planes<FM> la;
  __shared__ Planes<FN> lb;
  __shared__ int large;   // an operand of 2^16 and more was staged
  const int tiles = tiles_m * tiles_n;
  const int part = blockIdx.x / tiles, id = blockIdx.x - part * tiles;
  const int tm = id / tiles_n, tn = id - tm * tiles_n;
  const int m0 = tm * 32 * FM, n0 = tn * 32 * FN;
  // (unsigned: past the end of the longest contraction an int overflows; loops left by a difference are 2 %
  // slower here)
  const unsigned k_begin = part * k_part, k_end = min((unsigned)Kc, k_begin + k_part);
  C += (int64_t)part * M * N;

  f32x4 acc[FM][FN], low[FM][FN];
  clear(acc);
  clear(low);
  int ga, qa, gb, qb;
  my_share<AK>(ga, qa);
  my_share<BKM>(gb, qb);
  float xa[FM][4], xb[FN][4];
  // Rows past the edge read a valid one, indices past the end count as zero.
  auto fetch = [&](unsigned k0) {
    if (k0 + 32 <= k_end) {
      load_block<AK, FM, VEC, false>(xa, A, m0 + FM * ga, M, k0 + 4 * qa, Kc, k_end);
      load_block<BKM, FN, VEC, false>(xb, B, n0 + FN * gb, N, k0 + 4 * qb, Kc, k_end);
    } else {
      load_block<AK, FM, VEC, true>(xa, A, m0 + FM * ga, M, k0 + 4 * qa, Kc, k_end);
      load_block<BKM, FN, VEC, true>(xb, B, n0 + FN * gb, N, k0 + 4 * qb, Kc, k_end);
    }
  };
  float largest = 0.f;
  if (threadIdx.x == 0) large = 0;
  fetch(k_begin);
  for (unsigned k0 = k_begin; k0 < k_end; k0 += 32) {
    put_stage<AK, FM>(la, xa);
    put_stage<BKM, FN>(lb, xb);
    largest = max_magnitude(max_magnitude(largest, xa), xb);
    __syncthreads();
    if (k0 + 32 < k_end) fetch(k0 + 32);
    split_stage<FM, FN>(acc, low, la, lb);
    __syncthreads();
  }
  if (largest >= 0x1p16f) large = 1;
  __syncthreads();

  const int wave = threadIdx.x >> 6, r = threadIdx.x & 15;
  const int mw = m0 + 16 * FM * (wave >> 1), nw = n0 + 16 * FN * (wave & 1);
  bool odd = false, zero = false;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      acc[i][j] += low[i][j];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float c = fabsf(acc[i][j][v]);
        odd |= !(c == 0.f || (c >= 0x1p-64f && c <= 0x1.fffffep127f));
        zero |= c == 0.f;
      }
    }
  const bool zeros = __builtin_amdgcn_ballot_w64(zero) != 0;
  if (!__builtin_amdgcn_ballot_w64(odd) && (zeros || large))
    odd = tiny_operands<AK, BKM, FM, FN, VEC>(A, B, mw + FM * r, nw + FN * r, M, N, Kc, k_begin, k_end,
                                              zeros ? 0x1p-62f : 0x1p-110f);
  if (__builtin_amdgcn_ballot_w64(odd)) {
    clear(acc);
    direct_tile<AK, BKM, FM, FN, 1, VEC, 1, true>(acc, A, B, mw + FM * r, nw + FN * r, M, N, Kc, k_begin, k_end, 0);
  }
  store_tile<EPI, FM, FN, VEC>(acc, C, bias, Z, mw, nw, M, N, beta);
}

template <bool AK, bool BKM, int EPI, int FM, int FN, int U, int WAVES, bool LONG = false>
int launch_tile(const float* A, const float* B, float* C, const float* bias, float* Z, int M,
                int N, int Kc, int beta, hipStream_t stream) {
  const long long tiles_m = ceil_div(M, 16 * FM), tiles_n = ceil_div(N, 16 * FN);
  const long long nwg = tiles_m * tiles_n;
  if (nwg > 0x7fffffffLL) {
    set_error("gemm_f32: too many output tiles (%lld)", nwg);
    return AXN_ELIMIT;
  }
  // Vector accesses need whole groups (four along the contraction, FM rows, FN
  // columns) and 16-byte aligned bases.
  const uintptr_t ptrs = (uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)Z;
  const bool vec = Kc % 4 == 0 && (AK || M % FM == 0) && N % FN == 0 && (ptrs & 15u) == 0;
  if (vec)
    hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, EPI, FM, FN, U, true, WAVES, LONG>), dim3((unsigned)nwg),
                       dim3(64 * WAVES), 0, stream, A, B, C, bias, Z, M, N, Kc, (int)tiles_n, beta);
  else
    hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, EPI, FM, FN, U, false, WAVES, LONG>), dim3((unsigned)nwg),
                       dim3(64 * WAVES), 0, stream, A, B, C, bias, Z, M, N, Kc, (int)tiles_n, beta);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// Adds the parts of a split contraction in part order, then the epilogue.
template <int EPI, bool VEC>
__global__ void __launch_bounds__(256)
    f32_parts_kernel(const float* __restrict__ ws, float* __restrict__ C, const float* __restrict__ bias,
                     float* __restrict__ Z, int64_t MN, int N, int parts, int beta) {
  constexpr int W = VEC ? 4 : 1;
  using vec = typename VecOf<W>::type;
  const int64_t o = ((int64_t)blockIdx.x * 256 + threadIdx.x) * W;
  if (o >= MN) return;
  vec x = __builtin_nontemporal_load((const vec*)(ws + o));
  for (int p = 1; p < parts; ++p) x += __builtin_nontemporal_load((const vec*)(ws + p * MN + o));
  if (EPI == AXN_EPI_BIAS || EPI == AXN_EPI_BIAS_GELU) x += *(const vec*)(bias + o % N);
  if (EPI == AXN_EPI_BIAS_GELU || EPI == AXN_EPI_GELU) {
    if (Z != nullptr) *(vec*)(Z + o) = x;
    if constexpr (W == 1) x = gelu_erff(x);
    else
#pragma unroll
      for (int i = 0; i < W; ++i) x[i] = gelu_erff(x[i]);
  }
  if (beta) x += *(const vec*)(C + o);
  *(vec*)(C + o) = x;
}

// Problems of 2^32 multiply-adds and more may be split into bf16 products, with the contraction in as many
// parts as the estimate below finds fastest.  Smaller ones keep the native kernel and its bits, although by
// speed the line could lie lower (512 x 4096 x 1024 is 61 us natively and 41 split, 64 x 4096 x 1024 18 and
// 16): Adam divides a gradient by its own magnitude, so where one is next to zero the last bits of a product
// become 1e-2 of the learning rate, and small full-precision networks, whose steps the launches and the host
// bound, would take other steps than before for little.  (One step of a 1024 - 4096 - 1024 perceptron against
// 64 bits, largest difference of a weight over the weights' rms: batch 64 native 7e-4; batch 1024, which is
// above the line, native 3.2e-4, split 0.9e-4.)
constexpr double kSplitWork = 4294967296.0;

// Output tiles of the native kernel: the largest of 64 x 64, 32 x 32 and 16 x 16 (a loaded element is used
// 4, 2, 1 times) that still gives the chip's 1024 SIMDs a wave each; smaller tiles keep more loads in flight
// per wave.
struct NativeTiles {
  int size;
  long long count;
};
NativeTiles native_tiles(int64_t M, int64_t N) {
  const auto count = [&](int64_t t) { return (long long)((M + t - 1) / t) * ((N + t - 1) / t); };
  if (count(64) >= 1024) return {64, count(64)};
  if (count(32) >= 1024) return {32, count(32)};
  return {16, count(16)};
}

// Its estimated time in us: the products of whole tiles at a rate per tile size and storage order (NT, NN,
// TN), which the smallest tile reaches with 320, 1200 and 440 tiles.
double native_us(GemmLayout layout, int64_t M, int64_t N, int64_t Kc) {
  constexpr double kRate64[3] = {65, 70, 55}, kRate32[3] = {60, 55, 42}, kRate16[3] = {35, 30, 22};   // TFLOP/s
  constexpr double kFull16[3] = {320, 1200, 440};
  const NativeTiles t = native_tiles(M, N);
  double rate = t.size == 64 ? kRate64[layout] : t.size == 32 ? kRate32[layout] : kRate16[layout];
  if (t.size == 16 && t.count < kFull16[layout]) rate *= (double)t.count / kFull16[layout];
  return 2e-6 * (double)t.count * t.size * t.size * (double)Kc / rate;
}

// Parts of the contraction, by estimated time in us: a 32-deep stage takes 1.85 for a workgroup alone on
// its CU and 2.7 for two side by side, adding the parts takes a launch and their traffic.  Fitted to
// 30 problems from 8.6 to 69 GFLOP: 0.3 % off the best number of parts, and 2 % off the best of four tile
// sizes, on average.  2048 x 1024, contraction 4096: 1 part 217 us, 2 128, 4 99, 8 107.
// Thin outputs, whose 128 x 128 tiles are mostly padding, and few tiles over a long contraction without a
// workspace for parts are left to the native kernel where that is estimated to be faster (us, forward,
// native / split): 8 x 8192 over 65536 424 / 685, 15744 x 10 over 38831 679 / 1171, 128 x 128 over 2^18
// 1207 / 920 with a workspace and 14374 in one part.  Over 70 problems of 2^32 to 2^34.5 multiply-adds in the
// three storage orders the pick takes 0.5 % more than the faster of the two on average, 36 % at worst (41 %
// without a workspace); always split: 2.2 % and 73 % (140 % and 14 times).
struct F32Plan {
  int parts, k_part;   // parts 0: native
};
F32Plan plan_f32(GemmLayout layout, int64_t M, int64_t N, int64_t Kc, bool may_split) {
  constexpr int kCUs = 256, kMostParts = 16;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  F32Plan best = {0, 0};
  if ((double)M * (double)N * (double)Kc < kSplitWork || tiles * kMostParts > 0x7fffffffLL) return best;
  double least = native_us(layout, M, N, Kc);
  for (int p = 1; p <= (may_split ? kMostParts : 1); ++p) {
    const int64_t k_part = ((Kc + p - 1) / p + 31) / 32 * 32;
    if ((Kc + k_part - 1) / k_part != p) continue;
    const int64_t load = (tiles * p + kCUs - 1) / kCUs;   // workgroups on the fullest CU
    double us = (double)(k_part / 32) * ((double)(load / 2) * 2.7 + (double)(load % 2) * 1.85);
    if (p > 1) us += 3.0 + (p + 1) * (double)M * (double)N * 0.8e-6;
    if (us < least) least = us, best = {p, (int)(k_part < Kc ? k_part : Kc)};   // (one part of the longest: 2^31)
  }
  return best;
}

template <bool AK, bool BKM, int EPI>
int launch_split(const float* A, const float* B, float* C, const float* bias, float* Z, int M, int N,
                      int Kc, int beta, const F32Plan& plan, hipStream_t stream) {
  constexpr int F = 4;
  const int tiles_m = (int)ceil_div(M, 32 * F), tiles_n = (int)ceil_div(N, 32 * F);
  const dim3 grid((unsigned)((int64_t)tiles_m * tiles_n * plan.parts)), block(256);
  // as launch_tile's
  const uintptr_t ptrs = (uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)Z;
  const bool vec = Kc % 4 == 0 && (AK || M % F == 0) && N % F == 0 && (ptrs & 15u) == 0;
  if (vec)
    hipLaunchKernelGGL((gemm_f32_split_kernel<AK, BKM, EPI, F, F, true>), grid, block, 0, stream, A, B, C,
                       bias, Z, M, N, Kc, tiles_m, tiles_n, plan.k_part, beta);
  else
    hipLaunchKernelGGL((gemm_f32_split_kernel<AK, BKM, EPI, F, F, false>), grid, block, 0, stream, A, B, C,
                       bias, Z, M, N, Kc, tiles_m, tiles_n, plan.k_part, beta);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

template <int EPI>
int launch_parts(const float* ws, float* C, const float* bias, float* Z, int M, int N, int parts, int beta,
                 hipStream_t stream) {
  const int64_t MN = (int64_t)M * N;
  const uintptr_t ptrs = (uintptr_t)ws | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)Z;
  const bool vec = N % 4 == 0 && (ptrs & 15u) == 0;
  const int64_t lanes = vec ? MN / 4 : MN;
  const dim3 grid((unsigned)((lanes + 255) / 256)), block(256);
  if (vec)
    hipLaunchKernelGGL((f32_parts_kernel<EPI, true>), grid, block, 0, stream, ws, C, bias, Z, MN, N, parts, beta);
  else
    hipLaunchKernelGGL((f32_parts_kernel<EPI, false>), grid, block, 0, stream, ws, C, bias, Z, MN, N, parts, beta);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// With fewer than 4096 of the native kernel's tiles and a contraction of KMIN or more (256 for the smallest
// tile, 2048 for the middle one; measured: the split loses on the largest tile and on shorter contractions),
// four waves share a tile.
constexpr int kTogether16 = 256, kTogether32 = 2048;
template <bool AK, bool BKM, int EPI, int FM, int FN, int U, int KMIN>
int launch_waves(long long tiles, const float* A, const float* B, float* C, const float* bias,
                 float* Z, int M, int N, int Kc, int beta, hipStream_t stream) {
  if (tiles < 4096 && Kc >= KMIN)
    return launch_tile<AK, BKM, EPI, FM, FN, (U > 4 ? 4 : U), 4>(A, B, C, bias, Z, M, N, Kc, beta, stream);
  return launch_tile<AK, BKM, EPI, FM, FN, U, 1>(A, B, C, bias, Z, M, N, Kc, beta, stream);
}

// Whether gemm_f32_copied_kernel does a product faster than gemm_f32_kernel, and in which wave tiles: 16, 32 or 64
// square (1, 2, 4 blocks), 0 for neither.  In us, fitted to 260 sizes of 8 to 6200 tokens and 64 to 8192 features, cold
// operands, a layout and a tile each to 6 to 12 %; 5 % ahead counts.  What it picks takes 0.83 (forward), 0.53 (input
// gradient) and 0.83 (weight gradient) of the time of gemm_f32_kernel on average and 1 to 2 % more than the best.  That one
// stays ahead with short contractions (forward 924 x 336, contraction 164: 8.2 us, 8.9 here; weight gradients under 50 to
// 100 tokens: 5696 x 960, 72 tokens 16.5, 19.1): there its waves have all they multiply in flight at once.
// Weight gradients of up to 32 tokens are one unit a wave: with less than two 16 x 16 tiles for a SIMD its copy and its wait
// are all there is to them (128 x 128, 22 tokens 3.3 us, 3.7 here, added to 5.2, 7.2; 1088 x 128, 30 tokens, added to 5.6,
// 7.6; from 2300 tiles on 0.7 to 0.8 of the time).
int copied_blocks(GemmLayout layout, const NativeTiles& t, bool together, int64_t M, int64_t N, int64_t Kc) {
  if (layout == GEMM_TN && Kc <= 32 && t.size == 16 && t.count < 2048) return 0;
  struct Fit {
    double fixed, serial, load, round, out;   // a launch, a unit of a wave, of all on a CU, a round, 2^20 results or so
  };
  constexpr Fit kCopied[3][3] = {{{1.8, 0.098, 0.16, 1.6, 1.1}, {2.8, 0.31, 0.45, 1.1, 2.0}, {3.2, 2.1, 0.0, 4.2, 2.9}},
                                 {{1.7, 0.12, 0.18, 1.2, 0.0}, {1.2, 0.35, 0.45, 1.3, 0.21}, {1.9, 2.1, 0.0, 1.7, 0.7}},
                                 {{1e9, 0, 0, 0, 0}, {2.2, 0.22, 0.47, 0.51, 0.95}, {2.1, 2.0, 0.0, 1.7, 0.52}}};
  double least = 1e9;
  int best = 0;
  for (int i = 0; i < 3; ++i) {
    const int F = 1 << i, side = together ? 16 * F : 32 * F;
    const double each = together ? 2.0 * ((Kc + 255) / 256) : (double)((Kc + 31) / 32);
    const double load = (double)((((M + side - 1) / side) * ((N + side - 1) / side) + 255) / 256);
    const double rounds = F == 4 ? load : std::ceil(load / 2);
    const Fit& f = kCopied[layout][i];
    const double us = f.fixed + f.serial * rounds * each + f.load * load * each + f.round * rounds + f.out * M * N * 1e-6;
    if (us < least) least = us, best = F;
  }
  if (layout == GEMM_NN || (t.size == 32 && together)) return best;
  struct Direct {
    double fixed, chunk, chunks, load, bytes;   // a launch, a wave's 64 indices, a SIMD's, a wave on every SIMD, 1 MB loaded
  };
  // 16 x 16 tiles of a wave, of four waves, 32 x 32, 64 x 64
  constexpr Direct kDirect[2][4] = {{{2.6, 0.57, 0.0, 0.61, 0.068}, {3.3, 0.17, 0.65, 0.0, 0.023}, {4.7, 0.23, 0.0, 1.4, 0.12}, {16.0, 1.1, 0.0, 0.0, 0.2}},
                                    {{3.2, 0.0, 0.82, 0.15, 0.024}, {2.9, 0.86, 0.64, 0.16, 0.0}, {1.6, 4.0, 0.0, 1.1, 0.044}, {2.2, 4.9, 0.0, 3.1, 0.098}}};
  const Direct& d = kDirect[layout == GEMM_NT ? 0 : 1][t.size == 64 ? 3 : t.size == 32 ? 2 : together ? 1 : 0];
  const double chunks = Kc / (together ? 256.0 : 64.0), load = std::max(1.0, t.count * (together ? 4.0 : 1.0) / 1024);
  const double us = d.fixed + d.chunk * chunks + d.chunks * load * chunks + d.load * load + d.bytes * t.count * 2.0 * t.size * Kc * 4e-6;
  return least <= 0.95 * us ? best : 0;
}

template <bool AK, bool BKM, int EPI, int F, int SLOTS>
int launch_copied(bool together, const float* A, const float* B, float* C, const float* bias, float* Z, int M, int N, int Kc,
                  int beta, hipStream_t stream) {
  if constexpr (F == 1 && !AK) return AXN_EINVAL;   // (not picked)
  else {
    constexpr size_t kLds = 4 * SLOTS * F * 4096;
    const int side = together ? 16 * F : 32 * F, tiles_m = (int)ceil_div(M, side), tiles_n = (int)ceil_div(N, side);
    const auto kern = together ? gemm_f32_copied_kernel<AK, BKM, EPI, F, SLOTS, true> : gemm_f32_copied_kernel<AK, BKM, EPI, F, SLOTS, false>;
    static std::atomic<unsigned long long> allowed[2];   // per instance: devices it may have this LDS on
    if (const int rc = allow_lds((const void*)kern, kLds, allowed[together])) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)tiles_m * tiles_n)), dim3(256), kLds, stream, A, B, C, bias, Z, M, N, Kc,
                       tiles_m, tiles_n, beta);
    AXN_HIP_TRY(hipGetLastError());
    return AXN_OK;
  }
}

// Contractions whose loops would step past 2^31 - 1 (by four waves' chunks of 128 at most).
constexpr int kLongContraction = 0x7fffffff - 512;
static_assert((long long)kLongContraction + 4 * 16 * 8 <= 0x7fffffff, "the last step of the other variants");

template <bool AK, bool BKM, int EPI>
int launch_epi(const float* A, const float* B, float* C, const float* bias, float* Z, int M, int N,
               int Kc, int beta, float* ws, size_t ws_bytes, hipStream_t stream) {
  constexpr GemmLayout layout = !AK ? GEMM_TN : BKM ? GEMM_NT : GEMM_NN;
  const F32Plan plan = plan_f32(layout, M, N, Kc, ws != nullptr);
  if (plan.parts > 1) {
    const size_t need = (size_t)plan.parts * (size_t)M * (size_t)N * sizeof(float);
    if (ws_bytes < need) {
      set_error("gemm_f32: workspace too small (%zu bytes given, %zu needed)", ws_bytes, need);
      return AXN_EINVAL;
    }
    const int rc = launch_split<AK, BKM, AXN_EPI_NONE>(A, B, ws, nullptr, nullptr, M, N, Kc, 0, plan, stream);
    return rc ? rc : launch_parts<EPI>(ws, C, bias, Z, M, N, plan.parts, beta, stream);
  }
  if (plan.parts == 1)
    return launch_split<AK, BKM, EPI>(A, B, C, bias, Z, M, N, Kc, beta, plan, stream);
  const NativeTiles t = native_tiles(M, N);
  const uintptr_t ptrs = (uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)Z;
  if (N % 4 == 0 && (AK ? Kc % 4 == 0 : M % 4 == 0) && (ptrs & 15u) == 0 && std::max({M, N, Kc}) <= 1 << 22) {
    const bool together = t.size < 64 && t.count < 4096 && Kc >= (t.size == 32 ? kTogether32 : kTogether16);
    const int blocks = copied_blocks(layout, t, together, M, N, Kc);
    if (AK && blocks == 1)
      return launch_copied<AK, BKM, EPI, 1, 4>(together, A, B, C, bias, Z, M, N, Kc, beta, stream);
    if (blocks == 2) return launch_copied<AK, BKM, EPI, 2, 2>(together, A, B, C, bias, Z, M, N, Kc, beta, stream);
    if (blocks == 4) return launch_copied<AK, BKM, EPI, 4, 2>(together, A, B, C, bias, Z, M, N, Kc, beta, stream);
  }
  if (Kc > kLongContraction)
    return launch_tile<AK, BKM, EPI, 1, 1, 4, 4, true>(A, B, C, bias, Z, M, N, Kc, beta, stream);
  if (t.size == 64)
    return launch_tile<AK, BKM, EPI, 4, 4, 2, 1>(A, B, C, bias, Z, M, N, Kc, beta, stream);
  if (t.size == 32)
    return launch_waves<AK, BKM, EPI, 2, 2, 4, kTogether32>(t.count, A, B, C, bias, Z, M, N, Kc, beta, stream);
  return launch_waves<AK, BKM, EPI, 1, 1, 8, kTogether16>(t.count, A, B, C, bias, Z, M, N, Kc, beta, stream);
}

}  // namespace

size_t gemm_f32_workspace_bytes(GemmLayout layout, int64_t M, int64_t N, int64_t Kc) {
  const F32Plan plan = plan_f32(layout, M, N, Kc, true);
  return plan.parts > 1 ? (size_t)plan.parts * (size_t)M * (size_t)N * sizeof(float) : 0;
}

int launch_gemm_f32(GemmLayout layout, const float* A, const float* B, float* C,
                    const float* bias, float* Z, int M, int N, int Kc,
                    int epilogue, int beta, float* ws, size_t ws_bytes, hipStream_t stream) {
  switch (layout) {
    case GEMM_NT:
      switch (epilogue) {
        case AXN_EPI_NONE:
          return launch_epi<true, true, AXN_EPI_NONE>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
        case AXN_EPI_BIAS:
          return launch_epi<true, true, AXN_EPI_BIAS>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
        case AXN_EPI_BIAS_GELU:
          return launch_epi<true, true, AXN_EPI_BIAS_GELU>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
        default:
          return launch_epi<true, true, AXN_EPI_GELU>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
      }
    case GEMM_NN:
      return launch_epi<true, false, AXN_EPI_NONE>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
    default:
      return launch_epi<false, false, AXN_EPI_NONE>(A, B, C, bias, Z, M, N, Kc, beta, ws, ws_bytes, stream);
  }
}

}  // namespace axn
