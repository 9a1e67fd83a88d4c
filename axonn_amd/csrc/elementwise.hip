// Backward of the fused bias/GELU epilogue for gfx950: one HBM pass computing
//   dZ = dY * gelu'(Z)   and   dbias[n] = sum_m dZ[m, n]
// which is what autograd derives from the reference's `x + bias`
// (axonn/intra_layer/fully_connected.py:348) followed by the caller's exact-erf
// nn.GELU.  Lanes move 16 bytes (8 bf16 columns); column sums are kept in
// registers over a band's rows, combined through LDS, written as one fp32
// partial row per band and reduced over bands in a fixed order by a second
// kernel, so the result does not depend on scheduling.
//
// Also here: the SwiGLU activation of the Llama MLP, h = silu(gate) * up, and its
// backward, each one HBM pass.  The reference's Llama patch
// (axonn/models/transformers/modify_llama.py:76-95) swaps the three projections
// for its Linear and leaves `act_fn(gate_proj(x)) * up_proj(x)` to separate
// elementwise kernels with a bf16 rounding in between; here the product is formed
// in fp32 and rounded once.
#include "axn_internal.h"

namespace axn {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int EW_TX = 64;          // lanes along columns (8 columns each)
constexpr int EW_TY = 4;           // row phases per workgroup
constexpr int EW_COLS = EW_TX * 8; // 512 columns per workgroup
// Non-temporal loads of dY and Z: 12 % faster when the operands come from HBM (62 -> 55 us),
// 12 % slower when the memory-side cache holds them, which is the case in a training step
// (dY was written by the layer behind a moment ago): off.
constexpr bool DGELU_NT = false;
// SwiGLU has no sums to carry down the rows: one row piece per wave, the workgroups handed
// out in row-major order, so that the chip reads and writes one compact window of every
// operand (4096 x 14336 bf16 from HBM: forward 76 -> 59 us, backward 131 -> 98 us against
// 128-row bands, measured on MI355X).  Stores written through (nt + sc1), which gain 1 to
// 2 % in the optimizer's update kernel, change nothing in the forward and lose 6 % in the
// backward (two outputs): plain stores.
constexpr int SWIGLU_BAND = 4;

// 8 consecutive columns as floats, for bf16 / fp16 (16 bytes) and fp32 (32 bytes) rows.
// NT: non-temporal loads, for operands read once.  They are worth 15 % on the SwiGLU
// forward and 23 % on its backward and cost 12 % on dGELU (measured), so each kernel
// names its own.
template <bool NT, typename V>
__device__ __forceinline__ V load_vec(const void* p) {
  return NT ? __builtin_nontemporal_load((const V*)p) : *(const V*)p;
}
template <bool NT = false>
__device__ __forceinline__ void load8(const uint16_t* p, float (&x)[8]) {
  const bf16x8 v = load_vec<NT, bf16x8>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
template <bool NT = false>
__device__ __forceinline__ void load8(const _Float16* p, float (&x)[8]) {
  const f16x8 v = load_vec<NT, f16x8>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
template <bool NT = false>
__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
  const f32x4 a = load_vec<NT, f32x4>(p), b = load_vec<NT, f32x4>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = a[e];
    x[4 + e] = b[e];
  }
}
// Stores 8 columns rounded to the storage type and returns the stored values.
__device__ __forceinline__ void store8(uint16_t* p, float (&x)[8]) {
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = (__bf16)x[e];
    x[e] = (float)v[e];
  }
  *(bf16x8*)p = v;
}
__device__ __forceinline__ void store8(_Float16* p, float (&x)[8]) {
  f16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = (_Float16)x[e];
    x[e] = (float)v[e];
  }
  *(f16x8*)p = v;
}
__device__ __forceinline__ void store8(float* p, float (&x)[8]) {
  *(f32x4*)p = f32x4{x[0], x[1], x[2], x[3]};
  *(f32x4*)(p + 4) = f32x4{x[4], x[5], x[6], x[7]};
}

// Raw 8-column pieces of a row, so that a group of rows can be in flight as loads before
// any of it is converted.
template <typename T> struct Raw8;
template <> struct Raw8<uint16_t> { typedef bf16x8 type; };
template <> struct Raw8<_Float16> { typedef f16x8 type; };
template <> struct Raw8<float> { struct type { f32x4 lo, hi; }; };
template <typename T>
__device__ __forceinline__ typename Raw8<T>::type load_raw8(const T* p) {
  if constexpr (DGELU_NT && sizeof(T) == 2) {
    return __builtin_nontemporal_load((const typename Raw8<T>::type*)p);
  } else {
    return *(const typename Raw8<T>::type*)p;
  }
}
__device__ __forceinline__ void widen8(const bf16x8& v, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
__device__ __forceinline__ void widen8(const f16x8& v, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
__device__ __forceinline__ void widen8(const Raw8<float>::type& v, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = v.lo[e];
    x[4 + e] = v.hi[e];
  }
}

// A thread walks its rows in groups of EW_GROUP: the loads of the next group are issued
// before the stores of this one.  The memory counter of a wave is in order, so a load
// behind a store returns only after the store is acknowledged; with the loads in front,
// a wave waits for one store round trip per group and not per row (3 % at 8192 x 5120 bf16).
// Band b is the chunks b, b + bands, b + 2 bands, ...: all workgroups together walk down one compact
// window of the operands, where consecutive rows a band had each its own (us, from HBM, bf16: 8192 x 5120
// 56.5 -> 48.5, 8192 x 14336 153 -> 136, 5000 x 8192 69 -> 45, sums alone 24.6 -> 17.0).  What bounds it is the
// memory system, at 4.9 to 5.4 TB/s, beside about 24 operations an element.  Rows of different
// groups never overlap, so dZ may still alias dY.
constexpr int EW_GROUP = 4;
constexpr int EW_CHUNK = EW_TY * EW_GROUP;   // rows a workgroup has in flight
constexpr int EW_TURNS = 16;                 // most chunks a workgroup walks where that fills the chip

template <typename T, bool HAS_Z>
__global__ void __launch_bounds__(EW_TX* EW_TY)
    dgelu_dbias_kernel(const T* dY, const T* Z, T* dZ, float* partial, int64_t M,
                       int64_t N, int64_t ld) {
  typedef typename Raw8<T>::type raw;
  const int tx = threadIdx.x % EW_TX, ty = threadIdx.x / EW_TX;
  const int64_t col = (int64_t)blockIdx.x * EW_COLS + tx * 8;
  const int64_t step = (int64_t)gridDim.y * EW_CHUNK;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (col < N) {
    raw gy[EW_GROUP], gz[EW_GROUP];
    auto fetch = [&](int64_t first) {
#pragma unroll
      for (int u = 0; u < EW_GROUP; ++u) {
        const int64_t r = first + u * EW_TY;
        if (r < M) {
          gy[u] = load_raw8(dY + r * ld + col);
          if (HAS_Z) gz[u] = load_raw8(Z + r * ld + col);
        }
      }
    };
    int64_t first = (int64_t)blockIdx.y * EW_CHUNK + ty;
    fetch(first);
    while (first < M) {
      float g[EW_GROUP][8];
#pragma unroll
      for (int u = 0; u < EW_GROUP; ++u) {
        widen8(gy[u], g[u]);
        if (HAS_Z) {
          float z[8];
          widen8(gz[u], z);
#pragma unroll
          for (int e = 0; e < 8; ++e) g[u][e] *= dgelu_exact(z[e]);
        }
      }
      const int64_t next = first + step;
      if (next < M) fetch(next);
#pragma unroll
      for (int u = 0; u < EW_GROUP; ++u) {
        const int64_t r = first + u * EW_TY;
        if (r < M) {
          // g becomes what was stored: the sum of what wgrad reads
          if (HAS_Z) store8(dZ + r * ld + col, g[u]);
#pragma unroll
          for (int e = 0; e < 8; ++e) s[e] += g[u][e];
        }
      }
      first = next;
    }
  }
  if (partial == nullptr) return;
  __shared__ float red[EW_TY][EW_COLS];
#pragma unroll
  for (int e = 0; e < 8; ++e) red[ty][tx * 8 + e] = s[e];
  __syncthreads();
  for (int c = threadIdx.x; c < EW_COLS; c += EW_TX * EW_TY) {
    const int64_t gc = (int64_t)blockIdx.x * EW_COLS + c;
    if (gc < N)
      partial[(int64_t)blockIdx.y * N + gc] =
          (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  }
}

// Column sums over the band partials in a fixed order: 64 columns per workgroup, thread q of a
// column's 16 adds bands q, q + 16, ..., the 16 sums are then added in order.
__global__ void __launch_bounds__(1024)
    dbias_reduce_kernel(const float* partial, float* dbias, int64_t bands,
                        int64_t N, int beta) {
  __shared__ float red[16][64];
  const int tx = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int64_t c = (int64_t)blockIdx.x * 64 + tx;
  float s = 0.f;
  if (c < N)
#pragma unroll 4
    for (int64_t b = q; b < bands; b += 16) s += partial[b * N + c];
  red[q][tx] = s;
  __syncthreads();
  if (q == 0 && c < N) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[i][tx];
    dbias[c] = beta ? dbias[c] + t : t;
  }
}

template <typename T>
__global__ void __launch_bounds__(EW_TX* EW_TY)
    swiglu_fwd_kernel(const T* gate, const T* up, T* out, int64_t M, int64_t N, int64_t ld) {
  const int tx = threadIdx.x % EW_TX, ty = threadIdx.x / EW_TX;
  const int64_t col_blocks = (N + EW_COLS - 1) / EW_COLS;
  const int64_t band = blockIdx.x / col_blocks;
  const int64_t col = (int64_t)(blockIdx.x - band * col_blocks) * EW_COLS + tx * 8;
  if (col >= N) return;
  const int64_t r0 = band * SWIGLU_BAND;
  const int64_t r1 = (r0 + SWIGLU_BAND < M) ? r0 + SWIGLU_BAND : M;
  for (int64_t r = r0 + ty; r < r1; r += EW_TY) {
    const int64_t o = r * ld + col;
    float g[8], u[8];
    load8<true>(gate + o, g);
    load8<true>(up + o, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = g[e] * sigmoid_f(g[e]) * u[e];
    store8(out + o, g);
  }
}

// dgate = dout * up * silu'(gate),  dup = dout * silu(gate),
// silu'(x) = s (1 + x (1 - s)) with s = sigmoid(x).
template <typename T>
__global__ void __launch_bounds__(EW_TX* EW_TY)
    swiglu_bwd_kernel(const T* dout, const T* gate, const T* up, T* dgate, T* dup, int64_t M,
                      int64_t N, int64_t ld, int64_t ld_out) {
  const int tx = threadIdx.x % EW_TX, ty = threadIdx.x / EW_TX;
  const int64_t col_blocks = (N + EW_COLS - 1) / EW_COLS;
  const int64_t band = blockIdx.x / col_blocks;
  const int64_t col = (int64_t)(blockIdx.x - band * col_blocks) * EW_COLS + tx * 8;
  if (col >= N) return;
  const int64_t r0 = band * SWIGLU_BAND;
  const int64_t r1 = (r0 + SWIGLU_BAND < M) ? r0 + SWIGLU_BAND : M;
  for (int64_t r = r0 + ty; r < r1; r += EW_TY) {
    const int64_t o = r * ld + col;
    float d[8], g[8], u[8], dg[8], du[8];
    load8<true>(dout + o, d);
    load8<true>(gate + o, g);
    load8<true>(up + o, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sg = sigmoid_f(g[e]);
      du[e] = d[e] * g[e] * sg;
      dg[e] = d[e] * u[e] * sg * (1.0f + g[e] * (1.0f - sg));
    }
    store8(dgate + r * ld_out + col, dg);
    store8(dup + r * ld_out + col, du);
  }
}

}  // namespace

int launch_swiglu_fwd(const void* gate, const void* up, void* out, int dtype, int64_t M,
                      int64_t N, int64_t ld, hipStream_t stream) {
  const int64_t bands = (M + SWIGLU_BAND - 1) / SWIGLU_BAND;
  const int64_t blocks = bands * ((N + EW_COLS - 1) / EW_COLS);
  if (blocks > 0x7fffffffLL) {
    set_error("swiglu: too many elements (%lld x %lld)", (long long)M, (long long)N);
    return AXN_ELIMIT;
  }
  const dim3 grid((unsigned)blocks), block(EW_TX * EW_TY);
  if (dtype == AXN_F32)
    hipLaunchKernelGGL(swiglu_fwd_kernel<float>, grid, block, 0, stream, (const float*)gate,
                       (const float*)up, (float*)out, M, N, ld);
  else if (dtype == AXN_F16)
    hipLaunchKernelGGL(swiglu_fwd_kernel<_Float16>, grid, block, 0, stream, (const _Float16*)gate,
                       (const _Float16*)up, (_Float16*)out, M, N, ld);
  else
    hipLaunchKernelGGL(swiglu_fwd_kernel<uint16_t>, grid, block, 0, stream, (const uint16_t*)gate,
                       (const uint16_t*)up, (uint16_t*)out, M, N, ld);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

int launch_swiglu_bwd(const void* dout, const void* gate, const void* up, void* dgate, void* dup,
                      int dtype, int64_t M, int64_t N, int64_t ld, int64_t ld_out,
                      hipStream_t stream) {
  const int64_t bands = (M + SWIGLU_BAND - 1) / SWIGLU_BAND;
  const int64_t blocks = bands * ((N + EW_COLS - 1) / EW_COLS);
  if (blocks > 0x7fffffffLL) {
    set_error("swiglu: too many elements (%lld x %lld)", (long long)M, (long long)N);
    return AXN_ELIMIT;
  }
  const dim3 grid((unsigned)blocks), block(EW_TX * EW_TY);
  if (dtype == AXN_F32)
    hipLaunchKernelGGL(swiglu_bwd_kernel<float>, grid, block, 0, stream, (const float*)dout,
                       (const float*)gate, (const float*)up, (float*)dgate, (float*)dup, M, N, ld, ld_out);
  else if (dtype == AXN_F16)
    hipLaunchKernelGGL(swiglu_bwd_kernel<_Float16>, grid, block, 0, stream, (const _Float16*)dout,
                       (const _Float16*)gate, (const _Float16*)up, (_Float16*)dgate,
                       (_Float16*)dup, M, N, ld, ld_out);
  else
    hipLaunchKernelGGL(swiglu_bwd_kernel<uint16_t>, grid, block, 0, stream, (const uint16_t*)dout,
                       (const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)dgate,
                       (uint16_t*)dup, M, N, ld, ld_out);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

namespace {
// Bands of the dGELU + dbias pass: as many as leave a workgroup one to sixteen chunks of rows, at most 640
// workgroups where there is a choice (the sums' traffic grows with them; from eight chunks on there is none), and of
// those the number whose fullest CU has the fewest chunks to walk.  Bands of 128 consecutive rows left 64 to 500 rows
// to 8 to 32 CUs (us, before -> now): fp32 2048 x 4096 25.2 -> 20.2, 2900 x 6144 59.3 -> 40.0; bf16 256 x 4096 without
// sums 16 -> 9.  With no more than eight chunks 8192 x 5120 takes 640 workgroups, which are 3 for half of the CUs and 2
// for the others (bf16 51.7 us, with 470 48.5), 5000 x 8192 49.4 and 45.2.
int64_t dgelu_bands(int64_t M, int64_t N) {
  const int64_t cols = (N + EW_COLS - 1) / EW_COLS, chunks = (M + EW_CHUNK - 1) / EW_CHUNK;
  int64_t best = 0, least = 0;
  for (int64_t turns = 1; turns <= EW_TURNS; ++turns) {
    const int64_t bands = (chunks + turns - 1) / turns;
    if (bands * cols > 640 && turns < 8) continue;
    const int64_t walk = (bands * cols + 255) / 256 * turns;
    if (best == 0 || walk < least) best = bands, least = walk;
  }
  return best;
}
constexpr int EW_SUM_ROWS = 128;   // a workspace for a sum per so many rows is always enough
size_t band_sums_bytes(int64_t bands, int64_t N) { return (size_t)bands * (size_t)N * sizeof(float); }
}  // namespace

size_t dgelu_dbias_workspace_bytes(int64_t M, int64_t N) {
  if (M <= 0 || N <= 0) return 0;
  const int64_t bands = dgelu_bands(M, N), enough = (M + EW_SUM_ROWS - 1) / EW_SUM_ROWS;
  return band_sums_bytes(bands > enough ? bands : enough, N);
}

int launch_dgelu_dbias(const void* dY, const void* Z, void* dZ, int dtype,
                       float* dbias, int64_t M, int64_t N, int64_t ld, int beta,
                       void* ws, size_t ws_bytes, hipStream_t stream) {
  int64_t bands = dgelu_bands(M, N);
  if (dbias != nullptr && ws_bytes < band_sums_bytes(bands, N)) bands = (M + EW_SUM_ROWS - 1) / EW_SUM_ROWS;
  float* partial = nullptr;
  if (dbias != nullptr) {
    if (ws == nullptr || ws_bytes < band_sums_bytes(bands, N)) {
      set_error("dgelu_dbias: workspace too small (%zu bytes given, %zu needed)",
                ws_bytes, dgelu_dbias_workspace_bytes(M, N));
      return AXN_EINVAL;
    }
    partial = (float*)ws;
  }
  const dim3 grid((unsigned)((N + EW_COLS - 1) / EW_COLS), (unsigned)bands);
  if ((M + EW_SUM_ROWS - 1) / EW_SUM_ROWS > 65535) {   // (never fewer than bands where there are many)
    set_error("dgelu_dbias: too many rows (%lld)", (long long)M);
    return AXN_ELIMIT;
  }
  const dim3 block(EW_TX * EW_TY);
  if (dtype == AXN_F32) {
    const float *y = (const float*)dY, *z = (const float*)Z;
    if (Z != nullptr)
      hipLaunchKernelGGL((dgelu_dbias_kernel<float, true>), grid, block, 0, stream,
                         y, z, (float*)dZ, partial, M, N, ld);
    else
      hipLaunchKernelGGL((dgelu_dbias_kernel<float, false>), grid, block, 0, stream,
                         y, z, (float*)dZ, partial, M, N, ld);
  } else if (dtype == AXN_F16) {
    const _Float16 *y = (const _Float16*)dY, *z = (const _Float16*)Z;
    if (Z != nullptr)
      hipLaunchKernelGGL((dgelu_dbias_kernel<_Float16, true>), grid, block, 0, stream, y, z,
                         (_Float16*)dZ, partial, M, N, ld);
    else
      hipLaunchKernelGGL((dgelu_dbias_kernel<_Float16, false>), grid, block, 0, stream, y, z,
                         (_Float16*)dZ, partial, M, N, ld);
  } else {
    const uint16_t *y = (const uint16_t*)dY, *z = (const uint16_t*)Z;
    if (Z != nullptr)
      hipLaunchKernelGGL((dgelu_dbias_kernel<uint16_t, true>), grid, block, 0,
                         stream, y, z, (uint16_t*)dZ, partial, M, N, ld);
    else
      hipLaunchKernelGGL((dgelu_dbias_kernel<uint16_t, false>), grid, block, 0,
                         stream, y, z, (uint16_t*)dZ, partial, M, N, ld);
  }
  AXN_HIP_TRY(hipGetLastError());
  if (dbias != nullptr) {
    hipLaunchKernelGGL(dbias_reduce_kernel, dim3((unsigned)((N + 63) / 64)),
                       dim3(1024), 0, stream, partial, dbias, bands, N, beta);
    AXN_HIP_TRY(hipGetLastError());
  }
  return AXN_OK;
}

// ---- rows of any width, padded with zeros to a multiple of 8 elements -----------------
// Bound by its bytes: 8 elements a lane, the reads with the alignment of one element (2048 x 50257:
// 64 us, 6.4 TB/s).  The destination's rows are ld_dst elements apart, zeros up to there.
namespace {
struct __attribute__((packed, aligned(2))) Any8 {
  uint4 v;
};

__global__ void __launch_bounds__(256)
    pad_rows16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int64_t M, int64_t N,
                      int64_t ld, int64_t per_row) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * per_row) return;
  const int64_t row = idx / per_row, col = (idx - row * per_row) * 8;   // per_row groups of 8 in a padded row
  const uint16_t* from = src + row * ld + col;
  uint4 v = {0, 0, 0, 0};
  if (col + 8 <= N) {
    v = ((const Any8*)from)->v;
  } else {
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (col + e < N) w[e / 2] |= (uint32_t)from[e] << (16 * (e % 2));
    v = uint4{w[0], w[1], w[2], w[3]};
  }
  *(uint4*)(dst + idx * 8) = v;
}
}  // namespace

int launch_pad_rows16(const void* src, void* dst, int64_t M, int64_t N, int64_t ld, int64_t ld_dst,
                      hipStream_t stream) {
  const int64_t per_row = ld_dst / 8, groups = (M * per_row + 255) / 256;
  if (groups > 0x7fffffffLL) {
    set_error("pad_rows16: too many elements");
    return AXN_ELIMIT;
  }
  hipLaunchKernelGGL(pad_rows16_kernel, dim3((unsigned)groups), dim3(256), 0, stream, (const uint16_t*)src,
                     (uint16_t*)dst, M, N, ld, per_row);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

}  // namespace axn
