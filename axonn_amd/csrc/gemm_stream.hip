// Forward products of a few tokens, Y[M, N] = X[M, K] W[N, K]^T with M up to a few dozen (token
// by token generation, small requests): the weights are read once and hardly computed
// with, so the kernel is a stream over W with the MFMAs on the side.
//
// One workgroup owns 16 R rows of W and all tokens; its waves take the contraction in turn,
// 64 elements (a 128-byte line of every row) at a time, each through a ring of its own in
// LDS: no barrier in the loop.  Straight loads into MFMA fragments were the first version:
// v_mfma_f32_16x16x32 wants 16 rows in 16 consecutive lanes, and a load whose neighbouring lanes
// lie in different lines runs at a quarter of the L1 rate (2.0 to 3.4 TB/s of weights).  Copies
// to LDS move whole lines (8 lanes each) and the fragments are read back swizzled
// (DeepOperand's layout: chunk c of row r at c ^ ((r >> 1) & 7)).  With W as the row operand a
// lane ends with 4 consecutive output columns of one token.  The waves' sums meet in LDS and
// are added in wave order, so results do not depend on timing.
//
// What bounds it: the weights' way from HBM, and the tokens' from L2, which every workgroup
// reads again (a CU takes about 60 KB/us in all).  So the workgroups are as tall as it takes
// to fit one round of the 256 CUs (launch_stream_rows).  Measured on MI355X, cold weights, us:
//   N x K            16 tokens         32 tokens   register-staged / bounded tile kernel, 16
//   4096 x 4096      8.0 (4.2 TB/s)    9.9         82 / 52
//   6144 x 4096      10.8 (4.7 TB/s)   13.0        75 / 54
//   14336 x 4096     19.6 (6.0 TB/s)   21.1        78 / 62
//   4096 x 14336     22.3 (5.3 TB/s)   29.8        247 / 161
//   (about 2.5 us of each are the launch; without the reads of X 16 tokens take 1 to 2 us less)
#include "gemm_solo.h"

namespace axn {
namespace {

// Gate/up forward: 4 consecutive columns of one row (of a multiple of 8), as store_swiglu8.
template <bool HALF>
__device__ __forceinline__ void store_swiglu4(const f32x4& vg, const f32x4& vu, const GemmArgs& g, int row, int col) {
  using lp = std::conditional_t<HALF, _Float16, __bf16>;
  typedef lp lpx4 __attribute__((ext_vector_type(4)));
  const int64_t o = (int64_t)row * g.ldc + col;
  lpx4 gate, up, out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    gate[e] = (lp)vg[e];
    up[e] = (lp)vu[e];
    const float x = (float)gate[e];
    out[e] = (lp)(x * sigmoid_f(x) * (float)up[e]);
  }
  if (g.G != nullptr) *(lpx4*)(g.G + o) = gate;
  if (g.U != nullptr) *(lpx4*)(g.U + o) = up;
  *(lpx4*)((uint16_t*)g.C + o) = out;
}

// D: lines of the contraction a wave has on their way (its ring's slots); DX: of those, slots for X.  With one, a
// line's part of X follows when the line before it is in registers: it comes from L2, and four waves have each other's
// latency, which rings too large for LDS leave room for.
template <int MT, int R, int NW, int D, int DX, int EPI, bool OUT_F32, bool HALF>
__device__ __forceinline__ void stream_gemm(const GemmArgs& g) {
  constexpr int GROUPS = R + MT;              // 16-row groups copied per line: W's, then X's
  constexpr uint32_t WLINE = R * 2048, XLINE = MT * 2048;   // bytes of a slot
  constexpr int COPIES = 2 * GROUPS;
  static_assert(DX == D || (DX == 1 && D == 2), "slots of X");
  // Gate/up forward: the first half of W's groups are rows of the gate weights, the second half the rows of
  // the up weights with the same indices.
  constexpr bool SWIGLU = EPI == EPI_SWIGLU;
  constexpr int RO = SWIGLU ? R / 2 : R;      // 16-column groups of the output
  static_assert(!SWIGLU || (R % 2 == 0 && !OUT_F32), "pairs of groups");
  static_assert(COPIES * (D - 1) < 64, "outstanding copies the wait can count");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * (16 * RO);
  char* const ring = lds + wave * (D * WLINE + DX * XLINE);
  char* const xring = ring + D * WLINE;

  // Copies: 8 rows of 128 bytes each.  Rows past the end are outside the buffer and come as
  // zeros; so do the chunks past the contraction's end in its last line.
  constexpr uint32_t kOutside = 0x80000000u;
  auto resource = [&](const uint16_t* base, int rows, int64_t ld, int row0) {
    const int64_t left = ((int64_t)(rows - 1 - row0) * ld + g.Kc) * 2;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + row0 * ld), 0, (int)(left < 0x7fffffff ? left : 0x7fffffff),
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rw = resource(g.B, g.N, g.ldb, n0), rx = resource(g.A, g.M, g.lda, 0);
  const __amdgpu_buffer_rsrc_t rw2 = SWIGLU ? resource(g.B2, g.N, g.ldb, n0) : rw;
  uint32_t vw[2], vx[2];   // copy h of a group: rows 8 h .. 8 h + 7
  int chunk[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 8 * h + (lane >> 3);
    chunk[h] = (lane & 7) ^ ((row >> 1) & 7);
    vw[h] = (uint32_t)(row * g.ldb * 2 + chunk[h] * 16);
    vx[h] = (uint32_t)(row * g.lda * 2 + chunk[h] * 16);
  }
  const uint32_t w_group = (uint32_t)(16 * g.ldb * 2), x_group = (uint32_t)(16 * g.lda * 2);
  const int lines = (g.Kc + 63) / 64;
  // Workgroups start at different lines: all at the same one, with power-of-two row strides,
  // they crowd onto few memory channels (N = 14336, R = 2: 27.7 -> 21.4 us).
  // (The gate/up forward starts where the two products of their own would: the same sums.)
  const unsigned start = SWIGLU ? (unsigned)n0 / (unsigned)g.start_rows : blockIdx.x;
  const int rot = (int)((start * 7u) % (unsigned)lines);
  const int mine = (lines - wave + NW - 1) / NW;   // lines wave, wave + NW, ... (may be 0 or less)
  // the wave's i-th line of W into slot i % D, of X into slot i % DX
  auto copy = [&](int i, bool of_w, bool of_x) {
    int line = wave + i * NW + rot;
    if (line >= lines) line -= lines;
    const int k0 = line * 64;
    char* const to = ring + (i % D) * WLINE;
    char* const xto = xring + (i % DX) * XLINE;
    const bool cut = k0 + 64 > g.Kc;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool out = cut && k0 + 8 * chunk[h] >= g.Kc;
      const uint32_t ow = out ? kOutside : vw[h], ox = out ? kOutside : vx[h];
#pragma unroll
      for (int j = 0; of_w && j < R; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(j < RO ? rw : rw2, LDS_PTR(void, to + j * 2048 + h * 1024), 16,
                                                 (int)ow, (int)(k0 * 2 + (j % RO) * w_group), 0, 2);   // non-temporal: read once (4 % on the kernel)
#pragma unroll
      for (int j = 0; of_x && j < MT; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, LDS_PTR(void, xto + j * 2048 + h * 1024), 16, (int)ox,
                                                 (int)(k0 * 2 + j * x_group), 0, 0);
    }
  };

  f32x4 acc[MT][R];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mfma = [&](const bf16x8& a, const bf16x8& b, f32x4& c) {
    if constexpr (HALF)
      c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                 0, 0, 0);
    else
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  };

  const uint32_t ring0 = (uint32_t)(uintptr_t)LDS_PTR(char, ring), xring0 = ring0 + D * WLINE;
  const uint32_t frag0 = (uint32_t)(r * 128 + ((q ^ ((r >> 1) & 7)) << 4));        // first 32 elements
  const uint32_t frag1 = (uint32_t)(r * 128 + (((4 + q) ^ ((r >> 1) & 7)) << 4));  // last 32
  // `then`: called when the line's fragments are in registers and its slots are free
  auto multiply_line = [&](int i, auto then) {
    const uint32_t at = ring0 + (uint32_t)(i % D) * WLINE, xat = xring0 + (uint32_t)(i % DX) * XLINE;
    bf16x8 f[GROUPS][2];
    static_for<GROUPS>([&](auto j_) {
      constexpr int J = decltype(j_)::value;
      const uint32_t from = J < R ? at : xat;
      f[J][0] = lds_read_b128<(J < R ? J : J - R) * 2048>(from + frag0);
      f[J][1] = lds_read_b128<(J < R ? J : J - R) * 2048>(from + frag1);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < GROUPS; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(f[j][h]));   // used behind the wait only
    then();
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i2 = 0; i2 < MT; ++i2)
#pragma unroll
        for (int j = 0; j < R; ++j) mfma(f[j][h], f[R + i2][h], acc[i2][j]);
  };

  auto nothing = [] {};
  if constexpr (DX == D) {
#pragma unroll
    for (int i = 0; i < D; ++i)
      if (i < mine) copy(i, true, true);
    int i = 0;
    for (; i + D < mine; ++i) {        // line i has landed when only the D - 1 behind it are on their way
      wait_vmcnt<COPIES * (D - 1)>();
      multiply_line(i, nothing);
      copy(i + D, true, true);         // into the slot whose fragments are in registers now
    }
    wait_vmcnt<0>();
    for (; i < mine; ++i) multiply_line(i, nothing);
  } else {
    // On their way, in this order: W's line i, X's line i, W's line i + 1.
    if (mine > 0) copy(0, true, true);
    if (mine > 1) copy(1, true, false);
    for (int i = 0; i < mine; ++i) {
      if (i + 1 < mine)
        wait_vmcnt<2 * R>();
      else
        wait_vmcnt<0>();
      multiply_line(i, [&] {
        if (i + 1 < mine) copy(i + 1, false, true);
        if (i + 2 < mine) copy(i + 2, true, false);
      });
    }
  }

  // The rings are free once every wave is here.
  __syncthreads();
  f32x4* part = (f32x4*)lds;         // [NW][MT * R][64]
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < R; ++j) part[(wave * (MT * R) + m * R + j) * 64 + lane] = acc[m][j];
  __syncthreads();
  auto total = [&](int b) {
    f32x4 s = part[b * 64 + lane];
#pragma unroll
    for (int v = 1; v < NW; ++v) s += part[(v * (MT * R) + b) * 64 + lane];
    return s;
  };
  if constexpr (SWIGLU) {
    for (int b = wave; b < MT * RO; b += NW) {
      const int m = b / RO, j = b % RO;
      const f32x4 gate = total(m * R + j), up = total(m * R + RO + j);
      const int row = 16 * m + r, col = n0 + 16 * j + 4 * q;
      if (row < g.M && col < g.N) store_swiglu4<HALF>(gate, up, g, row, col);
    }
    return;
  }
  for (int b = wave; b < MT * R; b += NW) {
    const f32x4 s = total(b);
    const int row = 16 * (b / R) + r, col = n0 + 16 * (b % R) + 4 * q;
    if (row >= g.M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < g.N) store_one<EPI, OUT_F32, HALF>(s[e], g, row, col + e);
  }
}

template <int MT, int R, int NW, int D, int EPI, bool OUT_F32, bool HALF>
__global__ void __launch_bounds__(NW * 64) gemm_stream_kernel(const GemmArgs g) {
  stream_gemm<MT, R, NW, D, D, EPI, OUT_F32, HALF>(g);
}
template <int MT, int R, int NW, int D, int DX, bool HALF>
__global__ void __launch_bounds__(NW * 64) gemm_gate_up_stream_kernel(const GemmArgs g) {
  stream_gemm<MT, R, NW, D, DX, EPI_SWIGLU, false, HALF>(g);
}

// The rings, or the waves' sums behind them.
constexpr size_t stream_lds(int MT, int R, int NW, int D, int DX) {
  const size_t ring = (size_t)NW * (D * R + DX * MT) * 2048, sums = (size_t)NW * MT * R * 1024;
  return ring > sums ? ring : sums;
}

template <int MT, int R, int NW, int D, bool HALF>
int launch_stream(const GemmArgs& g, int epilogue, bool out_f32, hipStream_t stream) {
  constexpr size_t lds = stream_lds(MT, R, NW, D, D);
  const dim3 grid((unsigned)ceil_div(g.N, 16 * R)), block(NW * 64);
#define STREAM(EPI, F32)                                                                   \
  {                                                                                        \
    void (*kern)(const GemmArgs) = gemm_stream_kernel<MT, R, NW, D, EPI, F32, HALF>;       \
    static std::atomic<unsigned long long> lds_allowed{0};                                 \
    const int rc = allow_lds((const void*)kern, lds, lds_allowed);                         \
    if (rc != AXN_OK) return rc;                                                           \
    hipLaunchKernelGGL(kern, grid, block, lds, stream, g);                                 \
  }
  if (out_f32) {
    if (epilogue == AXN_EPI_BIAS) STREAM(AXN_EPI_BIAS, true)
    else STREAM(AXN_EPI_BIAS_GELU, true)
  } else {
    switch (epilogue) {
      case AXN_EPI_NONE: STREAM(AXN_EPI_NONE, false) break;
      case AXN_EPI_BIAS: STREAM(AXN_EPI_BIAS, false) break;
      case AXN_EPI_BIAS_GELU: STREAM(AXN_EPI_BIAS_GELU, false) break;
      default: STREAM(AXN_EPI_GELU, false)
    }
  }
#undef STREAM
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

// The smallest R whose workgroups fit one round of the CUs: a second round costs more than
// taller workgroups (5120 x 4096, 16 tokens: 320 workgroups of 16 rows 12.3 us, 160 of 32
// rows 10.5; 4096 x 4096: 256 of 16 rows 8.0, 128 of 32 rows 10.1).
int stream_groups(int N) { return N <= 16 * 256 ? 1 : N <= 32 * 256 ? 2 : 4; }
template <int MT, int D1, int D2, bool HALF>
int launch_stream_rows(const GemmArgs& g, int epilogue, bool out_f32, hipStream_t stream) {
  const int groups = stream_groups(g.N);
  if (groups == 1) return launch_stream<MT, 1, 4, D1, HALF>(g, epilogue, out_f32, stream);
  if (groups == 2) return launch_stream<MT, 2, 4, D2, HALF>(g, epilogue, out_f32, stream);
  return launch_stream<MT, 4, 4, 2, HALF>(g, epilogue, out_f32, stream);
}

template <bool HALF>
int launch_stream_tokens(const GemmArgs& g, int epilogue, bool out_f32, hipStream_t stream) {
  if (g.M <= 16) return launch_stream_rows<1, 4, 3, HALF>(g, epilogue, out_f32, stream);
  if (g.M <= 32) return launch_stream_rows<2, 4, 2, HALF>(g, epilogue, out_f32, stream);
  return launch_stream_rows<4, 2, 2, HALF>(g, epilogue, out_f32, stream);
}

// The gate/up forward: R / 2 groups of 16 rows of either matrix a workgroup.  Two workgroups fit a CU with
// R up to 4, so that both matrices are one round of twice as many; taller ones read the tokens less often.
// us of 16 and 64 tokens (cold weights, N x K), two products and the activation before -> R = 2, 4, 8:
//              16 tokens                          64 tokens
//   2816 x 1024   11.8 -> 4.9, 5.9, 8.3           14.3 -> 6.5, 8.4, 13.7
//   5632 x 2048   16.0 -> 11.1, 10.0, 14.6        23.5 -> 18.2, 13.9, 22.7
//   8192 x 3072   23.1 -> 17.7, 17.7, 23.3        33.8 -> 28.6, 22.1, 32.9
//   11008 x 4096  38.6 -> 29.6, 34.6, 31.3        54.1 -> 47.9, 46.3, 38.5
//   14336 x 4096  45.2 -> 38.1, 37.8, 38.0        57.6 -> 63.0, 49.6, 43.2
// (R = 8 of more than 32 tokens with one slot for X a wave: with two its rings are larger than LDS.  With two slots
// and two waves, whose sums are twice as long, 40.8 and 43.7; 28672 x 8192 157, so 153.)  16384 x 4096 at 16 tokens:
// 40.2 us, 6.7 TB/s.
template <int MT, int R, int D, int DX, bool HALF>
int launch_gate_up_stream(const GemmArgs& in, hipStream_t stream) {
  constexpr int NW = 4;
  constexpr size_t lds = stream_lds(MT, R, NW, D, DX);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  GemmArgs g = in;
  g.start_rows = 16 * stream_groups(g.N);
  void (*kern)(const GemmArgs) = gemm_gate_up_stream_kernel<MT, R, NW, D, DX, HALF>;
  static std::atomic<unsigned long long> lds_allowed{0};
  const int rc = allow_lds((const void*)kern, lds, lds_allowed);
  if (rc != AXN_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(g.N, 8 * R)), dim3(NW * 64), lds, stream, g);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}
template <int MT, int D2, bool HALF>
int launch_stream_swiglu(const GemmArgs& g, hipStream_t stream) {
  if (g.N > 16 * 256 && g.N <= 32 * 256) return launch_gate_up_stream<MT, 4, 2, 2, HALF>(g, stream);
  if constexpr (MT > 1)
    if (g.N > 32 * 256) return launch_gate_up_stream<MT, 8, 2, MT == 4 ? 1 : 2, HALF>(g, stream);
  return launch_gate_up_stream<MT, 2, D2, D2, HALF>(g, stream);
}
template <bool HALF>
int launch_stream_swiglu_tokens(const GemmArgs& g, hipStream_t stream) {
  if (g.M <= 16) return launch_stream_swiglu<1, 3, HALF>(g, stream);
  if (g.M <= 32) return launch_stream_swiglu<2, 2, HALF>(g, stream);
  return launch_stream_swiglu<4, 2, HALF>(g, stream);
}

}  // namespace

int launch_gemm_stream_swiglu(const GemmArgs& g, bool half, hipStream_t stream) {
  return half ? launch_stream_swiglu_tokens<true>(g, stream) : launch_stream_swiglu_tokens<false>(g, stream);
}

int launch_gemm_stream(const GemmArgs& g, int epilogue, bool out_f32, bool half, hipStream_t stream) {
  return half ? launch_stream_tokens<true>(g, epilogue, out_f32, stream)
              : launch_stream_tokens<false>(g, epilogue, out_f32, stream);
}

}  // namespace axn
