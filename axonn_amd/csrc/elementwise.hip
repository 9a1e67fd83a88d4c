// Backward of the fused bias/GELU epilogue for gfx950: one HBM pass computing
//   dZ = dY * gelu'(Z)   and   dbias[n] = sum_m dZ[m, n]
// which is what autograd derives from the reference's `x + bias`
// (axonn/intra_layer/fully_connected.py:348) followed by the caller's exact-erf
// nn.GELU.  Lanes move 16 bytes (8 bf16 columns); column sums are formed over
// bands of 128 rows, written as one fp32 partial row per band and reduced over
// bands in a fixed order by a second kernel, so the result does not depend on
// scheduling.
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
// SwiGLU has no sums to carry down the rows: one row piece per wave, the workgroups handed
// out in row-major order, so that the chip reads and writes one compact window of every
// operand (4096 x 14336 bf16 from HBM: forward 76 -> 59 us, backward 131 -> 98 us against
// 128-row bands, measured on MI355X).  Stores written through (nt + sc1), which gain 1 to
// 2 % in the optimizer's update kernel, change nothing in the forward and lose 6 % in the
// backward (two outputs): plain stores.
constexpr int SWIGLU_BAND = 4;

// 8 consecutive columns as floats, for bf16 / fp16 (16 bytes) and fp32 (32 bytes) rows.
// Non-temporal loads, for operands read once: worth 15 % on the SwiGLU forward and 23 % on its
// backward.  (dGELU is better off without: see dgelu_dbias_kernel.)
template <typename V>
__device__ __forceinline__ V load_vec(const void* p) {
  return __builtin_nontemporal_load((const V*)p);
}
__device__ __forceinline__ void load8(const uint16_t* p, float (&x)[8]) {
  const bf16x8 v = load_vec<bf16x8>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
__device__ __forceinline__ void load8(const _Float16* p, float (&x)[8]) {
  const f16x8 v = load_vec<f16x8>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}
__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
  const f32x4 a = load_vec<f32x4>(p), b = load_vec<f32x4>(p + 4);
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

// Raw 8-column pieces of a row (16-byte aligned), as they lie in memory.
typedef float f32x8 __attribute__((ext_vector_type(8), aligned(16)));
template <typename T> struct Raw8;
template <> struct Raw8<uint16_t> { typedef bf16x8 type; typedef __bf16 element; };
template <> struct Raw8<_Float16> { typedef f16x8 type; typedef _Float16 element; };
template <> struct Raw8<float> { typedef f32x8 type; typedef float element; };

// fp16(g * d) rounded once.
__device__ __forceinline__ _Float16 product_f16(float d, _Float16 g) {
  _Float16 r;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(r) : "v"(d), "v"(g));
  return r;
}

// A workgroup takes 128 columns of a band of 128 rows, 64 or 32 rows at a time: every thread one piece of 8 columns,
// which it stores and leaves in LDS, and then (512 threads) one column and phase whose sum it carries down the band:
// phase p adds rows p, p + 4, p + 8, ... one after the other, the four phases are added in pairs.  Two LDS buffers: the
// barrier behind the next rows is the one that frees these.
//
// Bound by memory: 252 MB of bf16 8192 x 5120 and their sums in 50 us from HBM (5.0 TB/s), 41 where the memory-side
// cache holds the operands.  The order of the sums is that of one workgroup of 256 threads walking 512 columns of a
// band row by row, which had 64 to 500 rows on 8 to 32 CUs; bands dealt out in chunks of 16 rows balance too,
// but add in another order, up to 1.6 times as far from 64 bits.  us with the sums, (HBM | cache), walk row by row,
// chunks, so:
//   bf16 8192 x 5120 62 | 51, 53 | 45, 50 | 41    2048 x 4096 22 | 21, 17 | 14, 15 | 14    256 x 4096 18, 7, 7
//   bf16 8192 x 14336 155, 135, 126               2900 x 6144 36 | 33, 26 | 23, 27 | 23    3001 x 10240 43 | 37, 40 | 34, 39 | 33
//   fp32 8192 x 5120 110, 101, 99                 2900 x 6144 64 | 46, 44 | 36, 48 | 37    5000 x 8192 108, 95, 87
//   sums alone, bf16 8192 x 5120 22, 18, 19       2900 x 6144 13.0, 12.4, 13.5             fp32 2900 x 6144 19.5, 15.8, 18.9
// 1024 threads are ahead of 512 by 2 % on 16-bit dGELU and behind by 3 to 8 % on fp32 and on sums alone (bf16 8192 x
// 5120 18.7 us, with 1024 19.6); 64 columns or 256 (fp32: 5 % slower), the loads of the next rows ahead of the stores and
// those of the whole band ahead of the first sums (2 to 5 % slower) were no faster.
// Non-temporal loads of dY and Z (bf16 8192 x 5120) are 10 % faster from HBM (47 us) and 12 % slower from the
// cache (47), which holds dY in a training step (the layer behind wrote it a moment ago): plain ones.
// Every thread has read its piece before it stores it, so dZ may alias dY.
constexpr int DG_BAND = 128, DG_COLS = 128, DG_PIECES = DG_COLS / 8;
template <typename T, bool HAS_Z>
constexpr int DG_THREADS = HAS_Z && sizeof(T) == 2 ? 1024 : 512;

// The workgroup's 128 columns.  Workgroups go to the 8 XCDs in turn, each with an L2 of its own: one XCD takes columns
// side by side, so that a 128-byte line that two of them share is read, and written, by one L2 (rows that do not
// start on lines share one line in three of 16-bit types).  fp32 (TURN): other columns in the next band, because
// 512 bytes of rows 4096 (32768) bytes apart lie in two of the 16 channels of an L2.  us in launch order, side by side,
// turned:   bf16 8192 x 5896 64, 54, 57   12000 x 8200 151, 117, 121   sums alone 8192 x 14344 49, 37, 42
//           fp32 16384 x 1024 44, 44, 34  4096 x 3048 34, 29, 27       sums alone 3000 x 8192 19, 23, 19
template <bool TURN>
__device__ __forceinline__ unsigned column_group() {
  const unsigned n = gridDim.x, xcd = blockIdx.x & 7, each = n >> 3;
  const unsigned at = xcd * each + min(xcd, n & 7u) + (blockIdx.x >> 3);
  return TURN ? (at + (blockIdx.y & 7) * max(each, 1u)) % n : at;
}

// WIDE: dY is fp32 (a 16-bit layer's fp32 bias makes its result, and so its gradient, fp32) and rounded to T on the way,
// as a cast before this pass would round it; without Z the rounded values are stored.  A cast of its own reads dY once
// more than that and its result is read twice: 3001 x 10240, fp16, sums alone: cast 34 us and 16.5 after it -> 37.
template <typename T, bool HAS_Z, bool WIDE>
__global__ void __launch_bounds__((DG_THREADS<T, HAS_Z>))
    dgelu_dbias_kernel(const void* dY, const T* Z, T* dZ, float* partial, int64_t M, int64_t N, int64_t ld) {
  typedef typename Raw8<T>::type raw;
  static_assert(!WIDE || sizeof(T) == 2, "rounds to a 16-bit type");
  typedef typename Raw8<T>::element element;
  constexpr int ROWS = DG_THREADS<T, HAS_Z> / DG_PIECES;   // at a time
  static_assert(ROWS % 4 == 0 && DG_BAND % ROWS == 0 && DG_THREADS<T, HAS_Z> >= 4 * DG_COLS, "a thread for each phase and column");
  // fp32: the sums take in the product unrounded, from its factors
  constexpr bool FACTORS = HAS_Z && std::is_same_v<T, float>;
  __shared__ __attribute__((aligned(16))) element rows[2][FACTORS ? 2 : 1][ROWS][DG_COLS];
  __shared__ float phases[4][DG_COLS];
  const int piece = threadIdx.x % DG_PIECES, row0 = threadIdx.x / DG_PIECES;
  const int c = threadIdx.x % DG_COLS, phase = threadIdx.x / DG_COLS;
  const unsigned at = column_group<sizeof(T) == 4>();
  const int64_t col0 = (blockIdx.z * kMostBlocks + at) * DG_COLS, band0 = (int64_t)blockIdx.y * DG_BAND;
  const int64_t col = col0 + piece * 8;
  float sum = 0.f;
#pragma unroll
  for (int step = 0; step < DG_BAND / ROWS; ++step) {
    const int64_t row = band0 + step * ROWS + row0;
    raw add = raw{}, factor = raw{};   // zeros outside
    if (row < M && col < N) {
      if constexpr (WIDE) {
        const f32x8 wide = *(const f32x8*)((const float*)dY + row * ld + col);
#pragma unroll
        for (int e = 0; e < 8; ++e) add[e] = (element)wide[e];
        if constexpr (!HAS_Z) *(raw*)(dZ + row * ld + col) = add;
      } else {
        add = *(const raw*)((const T*)dY + row * ld + col);
      }
      if constexpr (HAS_Z) {
        const raw z = *(const raw*)(Z + row * ld + col);
        raw out;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = dgelu_exact((float)z[e]);
          float g = (float)add[e] * d;
          if constexpr (FACTORS) {
            factor[e] = d;
            out[e] = g;
          } else if constexpr (std::is_same_v<T, _Float16>) {
            // stored: rounded to fp32 and then to fp16; added: the same, but in the first two columns of a piece
            // the product rounded once (what the sums of fp16 layers have been; one step apart on ties)
            asm("" : "+v"(g));
            out[e] = (_Float16)g;
            add[e] = e < 2 ? product_f16(d, add[e]) : out[e];
          } else {
            add[e] = out[e] = (__bf16)g;   // the sum of what wgrad reads
          }
        }
        *(raw*)(dZ + row * ld + col) = out;
      }
    }
    if (partial == nullptr) continue;
    *(raw*)&rows[step & 1][0][row0][piece * 8] = add;
    if constexpr (FACTORS) *(raw*)&rows[step & 1][1][row0][piece * 8] = factor;
    __syncthreads();
    if (phase >= 4) continue;
#pragma unroll
    for (int r = 0; r < ROWS; r += 4) {
      const float x = (float)rows[step & 1][0][phase + r][c];
      if constexpr (FACTORS)
        sum = __builtin_fmaf(x, rows[step & 1][1][phase + r][c], sum);
      else
        sum += x;
    }
  }
  if (partial == nullptr) return;
  if (phase < 4) phases[phase][c] = sum;
  __syncthreads();
  if (phase == 0 && col0 + c < N)
    partial[(int64_t)blockIdx.y * N + col0 + c] = (phases[0][c] + phases[1][c]) + (phases[2][c] + phases[3][c]);
}

// Column sums over the band partials in a fixed order: 64 columns per workgroup, the bands split in 4
// consecutive quarters summed by 4 threads each in band order (8 loads on their way), the quarters then
// combined as (q0 + q1) + (q2 + q3).  OUT: the sums' type (a 16-bit parameter's gradient straight away, where a cast
// would be one more launch).
template <typename OUT>
__global__ void __launch_bounds__(256)
    dbias_reduce_kernel(const float* partial, OUT* dbias, int64_t bands,
                        int64_t N, int beta) {
  __shared__ float red[4][64];
  const int tx = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int64_t c = block_number() * 64 + tx;
  const int64_t per = (bands + 3) / 4;
  const int64_t b1 = (q + 1) * per < bands ? (q + 1) * per : bands;
  float s = 0.f;
  if (c < N) {
    int64_t b = q * per;
    for (; b + 8 <= b1; b += 8) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = partial[(b + i) * N + c];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; b < b1; ++b) s += partial[b * N + c];
  }
  red[q][tx] = s;
  __syncthreads();
  if (q == 0 && c < N) {
    const float t = (red[0][tx] + red[1][tx]) + (red[2][tx] + red[3][tx]);
    dbias[c] = (OUT)(beta ? (float)dbias[c] + t : t);
  }
}

template <typename T>
__global__ void __launch_bounds__(EW_TX* EW_TY)
    swiglu_fwd_kernel(const T* gate, const T* up, T* out, int64_t M, int64_t N, int64_t ld) {
  const int tx = threadIdx.x % EW_TX, ty = threadIdx.x / EW_TX;
  const int64_t col_blocks = (N + EW_COLS - 1) / EW_COLS;
  const int64_t number = block_number(), band = number / col_blocks;
  const int64_t col = (number - band * col_blocks) * EW_COLS + tx * 8;
  if (col >= N) return;
  const int64_t r0 = band * SWIGLU_BAND;
  const int64_t r1 = (r0 + SWIGLU_BAND < M) ? r0 + SWIGLU_BAND : M;
  for (int64_t r = r0 + ty; r < r1; r += EW_TY) {
    const int64_t o = r * ld + col;
    float g[8], u[8];
    load8(gate + o, g);
    load8(up + o, u);
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
  const int64_t number = block_number(), band = number / col_blocks;
  const int64_t col = (number - band * col_blocks) * EW_COLS + tx * 8;
  if (col >= N) return;
  const int64_t r0 = band * SWIGLU_BAND;
  const int64_t r1 = (r0 + SWIGLU_BAND < M) ? r0 + SWIGLU_BAND : M;
  for (int64_t r = r0 + ty; r < r1; r += EW_TY) {
    const int64_t o = r * ld + col;
    float d[8], g[8], u[8], dg[8], du[8];
    load8(dout + o, d);
    load8(gate + o, g);
    load8(up + o, u);
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
  if (blocks > 0x7fffffffLL - kMostBlocks) {
    set_error("swiglu: too many elements (%lld x %lld)", (long long)M, (long long)N);
    return AXN_ELIMIT;
  }
  const dim3 grid = grid_of(blocks), block(EW_TX * EW_TY);
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
  if (blocks > 0x7fffffffLL - kMostBlocks) {
    set_error("swiglu: too many elements (%lld x %lld)", (long long)M, (long long)N);
    return AXN_ELIMIT;
  }
  const dim3 grid = grid_of(blocks), block(EW_TX * EW_TY);
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

size_t dgelu_dbias_workspace_bytes(int64_t M, int64_t N) {
  if (M <= 0 || N <= 0) return 0;
  return (size_t)((M + DG_BAND - 1) / DG_BAND) * (size_t)N * sizeof(float);
}

int launch_dgelu_dbias(const void* dY, const void* Z, void* dZ, int dtype, bool wide, void* dbias, bool dbias16,
                       int64_t M, int64_t N, int64_t ld, int beta, void* ws, size_t ws_bytes, hipStream_t stream) {
  const int64_t bands = (M + DG_BAND - 1) / DG_BAND;
  float* partial = nullptr;
  if (dbias != nullptr) {
    if (ws == nullptr || ws_bytes < dgelu_dbias_workspace_bytes(M, N)) {
      set_error("dgelu_dbias: workspace too small (%zu bytes given, %zu needed)",
                ws_bytes, dgelu_dbias_workspace_bytes(M, N));
      return AXN_EINVAL;
    }
    partial = (float*)ws;
  }
  const dim3 columns = grid_of((N + DG_COLS - 1) / DG_COLS), grid(columns.x, (unsigned)bands, columns.y);
  if (bands > 65535) {
    set_error("dgelu_dbias: too many rows (%lld)", (long long)M);
    return AXN_ELIMIT;
  }
#define AXN_DGELU(T, HAS_Z, WIDE)                                                                                       \
  hipLaunchKernelGGL((dgelu_dbias_kernel<T, HAS_Z, WIDE>), grid, dim3(DG_THREADS<T, HAS_Z>), 0, stream, dY, (const T*)Z, \
                     (T*)dZ, partial, M, N, ld)
#define AXN_DGELU_TYPE(T, WIDE)  \
  do {                           \
    if (Z != nullptr)            \
      AXN_DGELU(T, true, WIDE);  \
    else                         \
      AXN_DGELU(T, false, WIDE); \
  } while (0)
  if (dtype == AXN_F32)
    AXN_DGELU_TYPE(float, false);
  else if (dtype == AXN_F16 && wide)
    AXN_DGELU_TYPE(_Float16, true);
  else if (dtype == AXN_F16)
    AXN_DGELU_TYPE(_Float16, false);
  else if (wide)
    AXN_DGELU_TYPE(uint16_t, true);
  else
    AXN_DGELU_TYPE(uint16_t, false);
#undef AXN_DGELU_TYPE
#undef AXN_DGELU
  AXN_HIP_TRY(hipGetLastError());
  if (dbias != nullptr) {
#define AXN_REDUCE(OUT) \
  hipLaunchKernelGGL(dbias_reduce_kernel<OUT>, grid_of((N + 63) / 64), dim3(256), 0, stream, partial, (OUT*)dbias, bands, N, beta)
    if (!dbias16)
      AXN_REDUCE(float);
    else if (dtype == AXN_F16)
      AXN_REDUCE(_Float16);
    else
      AXN_REDUCE(__bf16);
#undef AXN_REDUCE
    AXN_HIP_TRY(hipGetLastError());
  }
  return AXN_OK;
}

// 16-bit elements as fp32: bound by its bytes.
namespace {
template <typename T>
__global__ void __launch_bounds__(256) widen_kernel(const T* __restrict__ src, float* __restrict__ dst, int64_t n8) {
  const int64_t i = block_number() * 256 + threadIdx.x;
  if (i >= n8) return;
  float x[8];
  load8(src + i * 8, x);
  store8(dst + i * 8, x);
}
}  // namespace
int launch_widen(const void* src, float* dst, bool half, int64_t n, hipStream_t stream) {
  const dim3 grid = grid_of((n / 8 + 255) / 256);
  if (half)
    hipLaunchKernelGGL(widen_kernel<_Float16>, grid, dim3(256), 0, stream, (const _Float16*)src, dst, n / 8);
  else
    hipLaunchKernelGGL(widen_kernel<uint16_t>, grid, dim3(256), 0, stream, (const uint16_t*)src, dst, n / 8);
  AXN_HIP_TRY(hipGetLastError());
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
  const int64_t idx = block_number() * 256 + threadIdx.x;
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
  if (groups > 0x7fffffffLL - kMostBlocks) {
    set_error("pad_rows16: too many elements");
    return AXN_ELIMIT;
  }
  hipLaunchKernelGGL(pad_rows16_kernel, grid_of(groups), dim3(256), 0, stream, (const uint16_t*)src,
                     (uint16_t*)dst, M, N, ld, per_row);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

}  // namespace axn
