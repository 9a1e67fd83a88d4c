// Device code of the one-wave-per-SIMD MFMA GEMM kernels (solo_gemm), shared by the
// translation units that instantiate it: gemm_bf16.hip (shapes made of whole tiles) and
// gemm_edge_bf16.hip, gemm_edge_f16.hip (every other shape).
#pragma once
#include <atomic>
#include <utility>

#include "axn_internal.h"

namespace axn {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int NUM_XCD = 8;      // MI355X: 8 accelerator dies, round-robin dispatch
// Internal epilogue of the gate/up forward: the tile's B rows are 64 gate rows and 64 up
// rows per wave, and the output is silu(gate) * up (not part of the public axn_epilogue).
constexpr int EPI_SWIGLU = 100;
// Internal: no epilogue, but the contraction runs through two operand pairs one after the
// other (C = A B + A2 B2).
constexpr int EPI_PAIR = 101;
// Internal, of the sum of parts: the result rounded to the 16-bit type and stored as fp32.
constexpr int EPI_WIDEN = 102;
#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// Calls f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>).
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// Workgroup id -> output tile, XCD aware.  Consecutive workgroup ids go to
// different XCDs, so ids are first regrouped per XCD into contiguous ranges and
// then walked in bands of GROUP_M tile rows.
__device__ __forceinline__ void tile_of_workgroup(int pid, int tiles_m,
                                                  int tiles_n, int& tm,
                                                  int& tn) {
  const int nwg = tiles_m * tiles_n;
  const int per = (nwg + NUM_XCD - 1) / NUM_XCD;
  int tall = nwg % NUM_XCD;
  if (tall == 0) tall = NUM_XCD;
  const int xcd = pid % NUM_XCD;
  const int local = pid / NUM_XCD;
  int t = (xcd < tall) ? xcd * per + local
                       : tall * per + (xcd - tall) * (per - 1) + local;
  constexpr int GROUP_M = 8;
  const int in_group = GROUP_M * tiles_n;
  const int group = t / in_group;
  const int first_m = group * GROUP_M;
  const int gsz = (tiles_m - first_m < GROUP_M) ? tiles_m - first_m : GROUP_M;
  const int r = t - group * in_group;
  tm = first_m + r % gsz;
  tn = r / gsz;
}

// A vector type whose loads and stores assume no more than the alignment of one element:
// rows of an output whose row stride is odd start anywhere.  The compiler still emits one
// 16-byte access (gfx950 runs with unaligned access enabled), so aligned rows cost the same.
template <typename V, int A>
struct Unaligned {
  typedef V type __attribute__((aligned(A)));
};

// The bias of 8 consecutive columns in fp32; a 16-bit one is widened here: a launch before the product that
// widens it costs more than the product of a small layer.
template <int EPI, bool HALF>
__device__ __forceinline__ void load_bias8(float (&bias)[8], const GemmArgs& g, int col) {
  using lpx8 = std::conditional_t<HALF, f16x8, bf16x8>;
  if (EPI != AXN_EPI_BIAS && EPI != AXN_EPI_BIAS_GELU) return;
  if (g.bias16) {
    const lpx8 b = *(const lpx8*)((const uint16_t*)g.bias + col);
#pragma unroll
    for (int e = 0; e < 8; ++e) bias[e] = (float)b[e];
  } else {
    const f32x4 b0 = *(const f32x4*)((const float*)g.bias + col);
    const f32x4 b1 = *(const f32x4*)((const float*)g.bias + col + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bias[e] = b0[e];
      bias[4 + e] = b1[e];
    }
  }
}

// Epilogue of 8 consecutive columns of one output row, held in fp32: bias,
// exact GELU with optional save of the pre-activation, accumulation into the
// existing output (beta), conversion and one 16- or 32-byte store.
// HALF: the 16-bit storage type is IEEE half instead of bfloat16.
// ANY: rows of C and Z have the alignment of one element (else 16 bytes).
// bias: the 8 columns', from load_bias8 (a load in here would be repeated for every row, behind the stores).
template <int EPI, bool OUT_F32, bool HALF, bool ANY = false>
__device__ __forceinline__ void store_row8(float (&v)[8], const float (&bias)[8], const GemmArgs& g, int row, int col) {
  using lp = std::conditional_t<HALF, _Float16, __bf16>;
  using lpx8 = std::conditional_t<HALF, f16x8, bf16x8>;
  using lpx8_mem = typename Unaligned<lpx8, ANY ? 2 : 16>::type;
  using f32x4_mem = typename Unaligned<f32x4, ANY ? 4 : 16>::type;
  const int64_t o = (int64_t)row * g.ldc + col;
  if (EPI == AXN_EPI_BIAS || EPI == AXN_EPI_BIAS_GELU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += bias[e];
  }
  if (EPI == AXN_EPI_BIAS_GELU || EPI == AXN_EPI_GELU) {
    if (g.Z != nullptr) {
      lpx8 z;
#pragma unroll
      for (int e = 0; e < 8; ++e) z[e] = (lp)v[e];
      *(lpx8_mem*)(g.Z + o) = z;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gelu_exact(v[e]);
  }
  if (OUT_F32) {
    float* C = (float*)g.C + o;
    f32x4 o0 = {v[0], v[1], v[2], v[3]}, o1 = {v[4], v[5], v[6], v[7]};
    if (g.beta) {
      o0 += *(const f32x4_mem*)C;
      o1 += *(const f32x4_mem*)(C + 4);
    }
    *(f32x4_mem*)C = o0;
    *(f32x4_mem*)(C + 4) = o1;
  } else {
    uint16_t* C = (uint16_t*)g.C + o;
    if (g.beta) {
      const lpx8 old = *(const lpx8_mem*)C;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += (float)old[e];
    }
    lpx8 y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (lp)v[e];
    *(lpx8_mem*)C = y;
  }
}

// An output row of 16-bit elements that starts 2 bytes off a 4-byte boundary (every second row of an odd row
// stride): a lane stores its predecessor's last element and its own first seven, on the boundary.  Stores off
// it cost 5 us a round of 256 x 256 tiles: 2048 x 50257, contraction 2048 418 us (50256 and 50258 columns,
// whose rows start on 4-byte boundaries, 385 and 388), this way 388 as well (in short
// runs 357 -> 337; 777 x 19999, 768 43.8 -> 36.3).
// y: the lane's 8 columns; before: the dword with the predecessor's last one (lead: there is none, the
// wave's first columns); end: nobody takes the lane's own last one.
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
// before <- the same of the lane whose byte index is `from`.  One statement that nothing moves across: of the
// builtin the compiler takes every row's exchange ahead of the first store, and spills.
__device__ __forceinline__ void lanes_16_down(uint32_t (&b)[4], int from) {
  asm volatile("ds_bpermute_b32 %0, %4, %0\n\tds_bpermute_b32 %1, %4, %1\n\tds_bpermute_b32 %2, %4, %2\n\t"
               "ds_bpermute_b32 %3, %4, %3\n\ts_waitcnt lgkmcnt(0)"
               : "+&v"(b[0]), "+&v"(b[1]), "+&v"(b[2]), "+&v"(b[3])
               : "v"(from));
}
__device__ __forceinline__ void lanes_16_down(uint32_t (&b)[3], int from) {
  asm volatile("ds_bpermute_b32 %0, %3, %0\n\tds_bpermute_b32 %1, %3, %1\n\tds_bpermute_b32 %2, %3, %2\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "+&v"(b[0]), "+&v"(b[1]), "+&v"(b[2])
               : "v"(from));
}
__device__ __forceinline__ void lanes_16_down(uint32_t (&b)[1], int from) {
  asm volatile("ds_bpermute_b32 %0, %1, %0\n\ts_waitcnt lgkmcnt(0)" : "+&v"(b[0]) : "v"(from));
}
__device__ __forceinline__ void lanes_16_down(uint32_t (&b)[2], int from) {
  asm volatile("ds_bpermute_b32 %0, %2, %0\n\tds_bpermute_b32 %1, %2, %1\n\ts_waitcnt lgkmcnt(0)"
               : "+&v"(b[0]), "+&v"(b[1])
               : "v"(from));
}
__device__ __forceinline__ void store_row8_odd(uint16_t* to, const u32x4& y, uint32_t before, bool lead, bool end) {
  typedef typename Unaligned<u32x4, 4>::type u32x4_mem;
  struct __attribute__((packed, aligned(4))) u32x3_mem {
    uint32_t d[3];
  };
  const bool off = ((uintptr_t)to & 2) != 0;
  u32x4 v = y;
  if (off) {
    v[0] = (y[0] << 16) | (before >> 16);
#pragma unroll
    for (int d = 1; d < 4; ++d) v[d] = (y[d] << 16) | (y[d - 1] >> 16);
  }
  if (off && lead) {
    *to = (uint16_t)y[0];
    *(u32x3_mem*)(to + 1) = u32x3_mem{{v[1], v[2], v[3]}};
  } else {
    *(u32x4_mem*)((char*)to - (off ? 2 : 0)) = v;
  }
  if (off && end) to[7] = (uint16_t)(y[3] >> 16);
}

// The same for one element.
template <int EPI, bool OUT_F32, bool HALF>
__device__ __forceinline__ void store_one(float x, const GemmArgs& g, int row, int col) {
  using lp = std::conditional_t<HALF, _Float16, __bf16>;
  const int64_t o = (int64_t)row * g.ldc + col;
  if (EPI == AXN_EPI_BIAS || EPI == AXN_EPI_BIAS_GELU)
    x += g.bias16 ? (float)((const lp*)g.bias)[col] : ((const float*)g.bias)[col];
  if (EPI == AXN_EPI_BIAS_GELU || EPI == AXN_EPI_GELU) {
    if (g.Z != nullptr) *((lp*)g.Z + o) = (lp)x;
    x = gelu_exact(x);
  }
  if (OUT_F32) {
    float* C = (float*)g.C + o;
    *C = g.beta ? x + *C : x;
  } else {
    lp* C = (lp*)g.C + o;
    if (g.beta) x += (float)*C;
    *C = (lp)x;
  }
}

// Epilogue of the gate/up forward for 8 consecutive columns of one row: both
// pre-activations are rounded to the 16-bit type (and stored, if asked for: the backward
// pass reads them), and the output is computed from the rounded values, so that it equals
// the separate activation kernel applied to the stored pre-activations bit for bit.
template <bool HALF>
__device__ __forceinline__ void store_swiglu8(const float (&vg)[8], const float (&vu)[8],
                                              const GemmArgs& g, int row, int col) {
  using lp = std::conditional_t<HALF, _Float16, __bf16>;
  using lpx8 = std::conditional_t<HALF, f16x8, bf16x8>;
  const int64_t o = (int64_t)row * g.ldc + col;
  lpx8 gate, up, out;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    gate[e] = (lp)vg[e];
    up[e] = (lp)vu[e];
    const float x = (float)gate[e];
    out[e] = (lp)(x * sigmoid_f(x) * (float)up[e]);
  }
  if (g.G != nullptr) *(lpx8*)(g.G + o) = gate;
  if (g.U != nullptr) *(lpx8*)(g.U + o) = up;
  *(lpx8*)((uint16_t*)g.C + o) = out;
}

// ---------------------------------------------------------------------------
// LDS fragment reads as inline assembly: the compiler neither waits for them nor
// orders them behind outstanding copies; the kernels place the waits themselves.
// ---------------------------------------------------------------------------
template <int IMM>
__device__ __forceinline__ bf16x8 lds_read_b128(uint32_t addr) {
  bf16x8 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(IMM));
  return v;
}
template <int IMM>
__device__ __forceinline__ s16x4 lds_read_tr16_b64(uint32_t addr) {
  s16x4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(IMM));
  return v;
}

// ---------------------------------------------------------------------------
// One-wave-per-SIMD kernel: 64-deep operand tiles, v_mfma_f32_16x16x32_bf16.
// ---------------------------------------------------------------------------
// Measured on MI355X, which runs these kernels power-limited: at equal FLOPs the
// 16x16x32 MFMA sustains about 10 % more clock than 32x32x16 (half the
// accumulator traffic per FLOP), and LDS fragment reads cost clock rather than
// issue slots.
//
// One operand tile: 256 rows x 64 deep (32 KiB), copied by 4 waves (8 copies
// each) and read as 16-row x 32-deep MFMA fragments (lane l: row l % 16,
// contraction elements 8 (l / 16) .. + 8).
//   K-major  tile [256][64] : 128-byte rows = whole cache lines of the operand;
//                             16-byte chunk c of row r lives at chunk c ^ ((r >> 1) & 7),
//                             which spreads the 16 lanes of a fragment quarter over
//                             all 64 banks
//   MN-major tile [64][256] : 512-byte rows; 64-byte chunk c of contraction row k
//                             lives at chunk c ^ (k & 3); read with the transposing
//                             ds_read_b64_tr_b16 (two per fragment)
// Tiles of other heights (multiples of 32 rows) differ in the MN-major swizzle alone: four contraction rows
// that are read together have to lie in four different 64-byte quarters of the 256 bytes that the banks span.
// Rows of an odd number of chunks do so by themselves, rows of 2, 6, 10 ... chunks with c ^ ((k >> 1) & 1).
//
// PERMUTED (the operand that supplies the output columns): fragment j holds the
// tile rows 32 (j / 2) + 8 (q / 4) + 4 (j % 2) + q % 4 in its lane-rows
// q = 0..15 instead of 16 j + q.  The MFMA result then leaves lane l with
// columns 8 (l / 16) .. + 3 of a 32-column group in block 2t and .. + 4 .. + 7
// in block 2t + 1: eight consecutive output columns per lane, stored from
// registers without a transpose through LDS.  Its K-major swizzle is
// chunk ^ (((r >> 1) & 1) | ((r >> 3) & 3) << 1), which again gives the 16 rows
// of a fragment quarter 16 distinct (row parity, chunk) pairs.
template <bool KMAJOR, bool PERMUTED, int ROWS_ /* a multiple of 32, up to 256 */>
struct DeepOperand {
  static constexpr int ROWS = ROWS_;
  static constexpr int PK = 64;
  static constexpr int BYTES = ROWS * PK * 2;      // 32 or 16 KiB
  static constexpr int NW = 4;
  static constexpr int DMA_N = BYTES / 1024 / NW;  // 8 or 4 copies per wave
  static constexpr int FR = ROWS / 32;             // 16-row fragments of a wave's half of the rows
  static constexpr int NADDR = KMAJOR ? 2 : (FR + 1) / 2;
  static constexpr int LPR = ROWS / 8;             // MN-major: lanes per contraction row of a copy

  __device__ __forceinline__ static int kmajor_swizzle(int row) {
    return PERMUTED ? (((row >> 1) & 1) | (((row >> 3) & 3) << 1)) : ((row >> 1) & 7);
  }
  __device__ __forceinline__ static int mnmajor_swizzle(int k) {
    return ROWS / 32 % 4 == 0 ? k & 3 : ROWS / 32 % 2 == 0 ? (k >> 1) & 1 : 0;
  }

  // Byte offset of this lane's 16 bytes for copy 0 of the tile at contraction
  // offset 0, and the uniform stride from copy i to i + 1.  Lane l of copy i
  // lands at tile + (4 i + wave) * 1024 + 16 l; the swizzle is applied here.
  __device__ __forceinline__ static uint32_t dma_offset(int64_t ld, int row0, int wave,
                                                        int lane, uint32_t& istride) {
    if constexpr (KMAJOR) {
      const int row = wave * 8 + (lane >> 3);              // + 32 i
      const int c = (lane & 7) ^ kmajor_swizzle(row);      // 32 i does not change the swizzle
      istride = (uint32_t)(32 * ld * 2);
      return (uint32_t)(((int64_t)(row0 + row) * ld + c * 8) * 2);
    } else {
      static_assert(64 % LPR == 0, "copies of whole contraction rows: 256 or 128 rows");
      constexpr int KPI = 64 / LPR;                    // contraction rows per copy: 2 or 4
      const int k = wave * KPI + lane / LPR;           // + 4 KPI i
      const int p16 = lane % LPR;
      const int c64 = (p16 >> 2) ^ (k & 3);            // 4 KPI i does not change k & 3
      istride = (uint32_t)(4 * KPI * ld * 2);
      return (uint32_t)(((int64_t)k * ld + row0 + (c64 * 4 + (p16 & 3)) * 8) * 2);
    }
  }

  // MN-major, tiles of any height: this lane's byte offset for copy i (contraction rows end inside a copy).
  __device__ __forceinline__ static uint32_t mnmajor_copy(int64_t ld, int wave, int lane, int i) {
    const int at = (NW * i + wave) * 1024 + 16 * lane, k = at / (ROWS * 2), b = at % (ROWS * 2);
    const int col = ((b >> 6) ^ mnmajor_swizzle(k)) * 32 + (b & 63) / 2;
    return (uint32_t)(((int64_t)k * ld + col) * 2);
  }

  // K-major: the 8 contraction elements 8 c .. 8 c + 7 of the tile that this lane copies
  // (the same for every copy of the tile).
  __device__ __forceinline__ static int dma_chunk(int wave, int lane) {
    return (lane & 7) ^ kmajor_swizzle(wave * 8 + (lane >> 3));
  }

  // Copy I of the tile (LDS kilobytes 4 I .. 4 I + 3); it reads the operand IO copy strides
  // behind copy 0 (IO = I unless the tile's rows are gathered from two places).
  template <int I, int IO = I>
  __device__ __forceinline__ static void dma_one(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff,
                                                 uint32_t tile_ofs, uint32_t istride,
                                                 char* lds_tile, int wave) {
    static_assert(I >= 0 && I < DMA_N && IO >= 0 && IO < DMA_N, "copy index");
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, lds_tile + (NW * I + wave) * 1024),
                                             16, (int)voff, (int)(tile_ofs + IO * istride), 0, 0);
  }

  // Per-lane LDS byte offsets (relative to the tile) the fragment reads start from.
  //   K-major : a[s] for the 32-deep step s; fragments add whole rows (frag_offset),
  //             which leave the swizzle unchanged.
  //   MN-major: a[i >> 1] for fragment i, step s adds 32 rows.  The 16 lanes of a
  //             block address contraction rows 8 (l / 16) + (l & 15) / 4 and 4
  //             columns each; the transposing read hands lane i of the block the
  //             column that lane 4 (i / 4) .. addressed, rows 8 (l / 16) + 0..3
  //             (second read: + 4..7).
  __device__ __forceinline__ static void read_bases(uint32_t (&a)[NADDR], int wrow0, int lane) {
    const int q = lane & 15;
    if (KMAJOR) {
      const int r = wrow0 + (PERMUTED ? 8 * (q >> 2) + (q & 3) : q);
      const int swz = kmajor_swizzle(r);
#pragma unroll
      for (int st = 0; st < 2; ++st)
        a[st] = (uint32_t)(r * 128 + (((st * 4 + (lane >> 4)) ^ swz) << 4));
    } else {
      const int kq = q >> 2;
      const int k = 8 * (lane >> 4) + kq;
#pragma unroll
      for (int h = 0; h < NADDR; ++h) {
        const int colbyte = (wrow0 + h * 32 + (PERMUTED ? 8 : 4) * (lane & 3)) * 2;
        a[h] = (uint32_t)(k * (ROWS * 2) + ((((colbyte >> 6) ^ mnmajor_swizzle(kq)) << 6) | (colbyte & 63)));
      }
    }
  }

  // Fragment I of the 32-deep step ST of the tile.
  template <int ST, int I>
  __device__ __forceinline__ static void read_frag(bf16x8& f, const uint32_t (&a)[NADDR]) {
    if constexpr (KMAJOR) {
      constexpr int row_ofs = PERMUTED ? 32 * (I >> 1) + 4 * (I & 1) : 16 * I;
      f = lds_read_b128<row_ofs * 128>(a[ST]);
    } else {
      constexpr int col_ofs = PERMUTED ? 4 * (I & 1) : 16 * (I & 1);  // elements
      const s16x4 lo = lds_read_tr16_b64<ST * 32 * ROWS * 2 + col_ofs * 2>(a[I >> 1]);
      const s16x4 hi = lds_read_tr16_b64<(ST * 32 + 4) * ROWS * 2 + col_ofs * 2>(a[I >> 1]);
      f = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

// With bounds: where the next A / B tile to copy starts and how many bytes of the operand lie
// behind that point.
struct OperandWalk {
  const char* at;
  int64_t left, step;
  __device__ __forceinline__ void start(const uint16_t* base, bool kmajor, int rows, int kc, int64_t ld, int row0,
                                        int k0) {
    const int64_t first = kmajor ? row0 * ld + k0 : k0 * ld + row0;
    // a row's last 8 elements are copied together: up to 7 of them are padding of the operand's rows
    const int64_t all = kmajor ? (int64_t)(rows - 1) * ld + ceil_div(kc, 8) * 8 : (int64_t)(kc - 1) * ld + ceil_div(rows, 8) * 8;
    at = (const char*)(base + first);
    left = (all - first) * 2;
    step = (kmajor ? (int64_t)64 : (int64_t)64 * ld) * 2;
  }
  // (left is positive: only stages that exist are copied; its halves are looked at one by
  // one because there is no scalar 64-bit order comparison)
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t resource() const {
    const uint32_t lo = (uint32_t)left;
    const uint32_t n = (uint32_t)(left >> 32) != 0u || lo > 0x7fffffffu ? 0x7fffffffu : lo;
    return __builtin_amdgcn_make_buffer_rsrc((void*)at, 0, (int)n, 0x00020000);
  }
  __device__ __forceinline__ void advance() {
    at += step;
    left -= step;
  }
};

// Passes fragments through a statement, so that no MFMA on them can move above it.
template <int N>
__device__ __forceinline__ void tie_fragments(bf16x8 (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}
// Waits for every outstanding LDS read of both operands' fragments.
template <int NA, int NB>
__device__ __forceinline__ void wait_all_fragments(bf16x8 (&fa)[NA], bf16x8 (&fb)[NB]) {
  asm volatile("s_waitcnt lgkmcnt(0)");
  tie_fragments(fa);
  tie_fragments(fb);
}
// The same for a row of accumulators (see the end of solo_gemm).
template <int N>
__device__ __forceinline__ void tie_accumulators(f32x4 (&a)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+a"(a[i]));
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Output of a wave's accumulators: rows m_first .., columns n_first .. of C.  With the permuted column fragments a
// lane owns, per block row i and block pair t, the 8 consecutive columns 32 t + 8 (l / 16) .. + 7 of row
// 16 i + l % 16: they go out straight from the registers, 64 contiguous bytes per row and instruction.
// EDGE: rows and columns inside the output only; tail: 8 floats a row in LDS that are the wave's own.
// APART: one block row after the other (left to itself the compiler works on several at once, and spills where a
// wave has 256 registers).
template <int EPI, bool OUT_F32, bool HALF, bool EDGE, bool ODD, bool APART = false, int FRM, int FRN>
__device__ __forceinline__ void store_blocks(f32x4 (&acc)[FRM][FRN], const GemmArgs& g, int split, int m_first,
                                             int n_first, int lane, [[maybe_unused]] float* tail) {
  constexpr int WTM = FRM * 16, WTN = FRN * 16;
  const int orow = m_first + (lane & 15), ocol = n_first + 8 * (lane >> 4);
  GemmArgs go = g;  // a split writes its own fp32 partial product
  if (OUT_F32 && g.splits > 1) go.C = (float*)g.C + (int64_t)split * g.M * g.ldc;
  constexpr int EP = EPI == EPI_PAIR ? (int)AXN_EPI_NONE : EPI;
  // EDGE: the columns behind the last multiple of 8 of the output go through LDS and are
  // stored one by one, which keeps that path out of the unrolled stores.
  float bias[FRN / 2][8];
#pragma unroll
  for (int t = 0; t < FRN / 2; ++t)
    if (!EDGE || ocol + 32 * t + 8 <= g.N) load_bias8<EP, HALF>(bias[t], g, ocol + 32 * t);
  static_assert(!ODD || (EDGE && EP == AXN_EPI_NONE && !OUT_F32), "store_row8_odd");
  if constexpr (ODD) {
    using lp = std::conditional_t<HALF, _Float16, __bf16>;
    using lpx8 = std::conditional_t<HALF, f16x8, bf16x8>;
#pragma unroll
    for (int i = 0; i < FRM; ++i) {
      const int row = orow + 16 * i;
      u32x4 y[FRN / 2];
      uint32_t before[FRN / 2];   // of each 8 columns: the dword with the one before them
#pragma unroll
      for (int t = 0; t < FRN / 2; ++t) {
        lpx8 y8;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y8[e] = (lp)acc[i][2 * t][e];
          y8[4 + e] = (lp)acc[i][2 * t + 1][e];
        }
        y[t] = __builtin_bit_cast(u32x4, y8);
        // it lies in the lane 16 further down; for lanes 0 .. 15 in lanes 48 .. 63 at t - 1
        before[t] = lane >= 48 ? (t > 0 ? y[t - 1][3] : 0u) : y[t][3];
      }
      lanes_16_down(before, ((lane + 48) & 63) * 4);
#pragma unroll
      for (int t = 0; t < FRN / 2; ++t) {
        const int col = ocol + 32 * t;
        if (row >= g.M || col >= g.N) continue;
        if (col + 8 > g.N) {
          f32x4* to = (f32x4*)(tail + ((lane & 15) + 16 * i) * 8);
          to[0] = acc[i][2 * t];
          to[1] = acc[i][2 * t + 1];
          continue;
        }
        store_row8_odd((uint16_t*)go.C + (int64_t)row * go.ldc + col, y[t], before[t], t == 0 && lane < 16,
                       (t == FRN / 2 - 1 && lane >= 48) || col + 16 > g.N);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < FRM; ++i) {
      if constexpr (APART) {
#pragma unroll
        for (int j = 0; j < FRN; ++j) asm volatile("" : "+a"(acc[i][j])::"memory");
      }
#pragma unroll
      for (int t = 0; t < FRN / 2; ++t) {
        const f32x4 lo = acc[i][2 * t], hi = acc[i][2 * t + 1];
        float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        const int row = orow + 16 * i, col = ocol + 32 * t;
        if constexpr (EDGE) {
          if (row >= g.M || col >= g.N) continue;
          if (col + 8 > g.N) {
            f32x4* to = (f32x4*)(tail + ((lane & 15) + 16 * i) * 8);
            to[0] = lo;
            to[1] = hi;
            continue;
          }
        }
        store_row8<EP, OUT_F32, HALF, EDGE>(v, bias[t], go, row, col);
      }
    }
  }
  if constexpr (EDGE) {
    const int end = g.N / 8 * 8, first = n_first;
    if (end < g.N && end >= first && end < first + WTN) {
#pragma unroll 1
      for (int k = lane; k < WTM * 8; k += 64) {
        const int row = m_first + k / 8, col = end + k % 8;
        if (row < g.M && col < g.N) store_one<EP, OUT_F32, HALF>(tail[k], go, row, col);
      }
    }
  }
}

// The gate/up forward: the tile's B rows are, per wave column, a half of gate rows and then the up rows with the same
// indices, so that a lane ends with a gate value in accumulator block j and the up value of the same output element in
// block j + FRN / 2.  Copy i brings 32 rows: those of the gate or the up weights from row 32 at on.
struct GateUpCopy {
  bool up;
  int at;
};
constexpr GateUpCopy gate_up_copy(int bn, int i) {
  const int a_half = bn / 64, of_one = a_half / 2;   // copies a wave column, of one of the two matrices
  return {i % a_half >= of_one, i / a_half * of_one + i % of_one};
}
template <bool HALF, bool EDGE, int FRM, int FRN>
__device__ __forceinline__ void store_gate_up(f32x4 (&acc)[FRM][FRN], const GemmArgs& g, int m_first, int n_first,
                                              int lane) {
  const int orow = m_first + (lane & 15), ocol = n_first + 8 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < FRM; ++i) {
    if constexpr (EDGE) {   // (one block row after the other, as store_blocks)
#pragma unroll
      for (int j = 0; j < FRN; ++j) asm volatile("" : "+a"(acc[i][j])::"memory");
    }
#pragma unroll
    for (int t = 0; t < FRN / 4; ++t) {
      const int row = orow + 16 * i, col = ocol + 32 * t;
      if (EDGE && (row >= g.M || col >= g.N)) continue;   // (N is a multiple of 8)
      const f32x4 gl = acc[i][2 * t], gh = acc[i][2 * t + 1];
      const f32x4 ul = acc[i][2 * t + FRN / 2], uh = acc[i][2 * t + 1 + FRN / 2];
      const float vg[8] = {gl[0], gl[1], gl[2], gl[3], gh[0], gh[1], gh[2], gh[3]};
      const float vu[8] = {ul[0], ul[1], ul[2], ul[3], uh[0], uh[1], uh[2], uh[3]};
      store_swiglu8<HALF>(vg, vu, g, row, col);
    }
  }
}

// TILE = 256: 4 waves, one per SIMD, each owning 128 x 128 of the 256 x 256 tile:
// 8 x 8 blocks of 16 x 16, 256 accumulator registers, 64 MFMAs per 32-deep step.
// A wave pipelines against itself: while the MFMAs of one step run on one
// register set (8 + 8 fragments), the fragments of the next step are read into
// the other, one fragment between two MFMAs.
//
// LDS holds a ring of 5 operand tiles (160 KiB); the tiles A0 B0 A1 B1 A2 ... of
// the contraction stages take the slots 0 1 2 3 4 0 1 ...  Stage p (64 deep):
//   step 0 : MFMAs | this wave's 8 copies of A(p+2) | reads of (p, 1)
//   step 1 : wait for own copies of A(p+1), B(p+1); barrier;
//            MFMAs | this wave's 8 copies of B(p+2) | reads of (p+1, 0)
// At the barrier every wave holds the last fragments of stage p in registers, so
// both of its slots are free: B(p+2) takes A(p)'s, A(p+3) (next step 0) B(p)'s.
// The copies come first in a step, the reads second: a tile has at least a whole
// stage (128 MFMAs per wave) to land.
//
// TILE = 128 is the same schedule on a 128 x 128 tile for problems that do not
// fill the chip with 256 x 256 tiles: 64 x 64 per wave (4 x 4 blocks, 16 MFMAs per
// step, 4 copies per tile and wave), an 80 KiB ring, two workgroups per CU.
//
// BM x BN = 256 x 128 is the tile of the launches that finish a problem after its full
// rounds of 256 x 256 tiles: a rest of r <= 128 large tiles makes 2 r <= 256 of these,
// one per CU, and needs 3/4 of the global -> LDS bytes per MFMA of the 128 x 128 tile.
// Its ring has five slots of the larger (A) tile's size.
//
// EDGE: any M, N and contraction, operands of any size.  The main loop is the same; what is
// added is
//   * copies of rows past the end of an operand: the buffer's byte count ends at the last
//     element, and lanes past it put zeros into LDS (measured: an out-of-range lane of a
//     load to LDS writes zeros, also where the scalar offset alone is past the end).  Zero
//     rows add nothing along a contraction-strided operand's contraction; elsewhere they
//     only reach output elements that are not stored, as do the columns of the next
//     row that a tile past the right edge of a contraction-strided operand reads;
//   * the last stage of a contraction that is not a multiple of 64: lanes of a
//     contraction-contiguous operand whose 8 elements lie past the end copy from an
//     out-of-range offset (kOutside), i.e. zeros;
//   * the buffer resource is rebased to the tile, and to the stage as the contraction
//     advances (five scalar instructions a tile), so that 32-bit offsets span the rows or the
//     contraction steps of one tile and not the whole operand: operands of any size, row
//     strides up to 2^22 elements (2^23 on the 128 x 128 tile).  A resource per copy instead
//     put 340 scalar and vector instructions into a stage and made it 60 % longer;
//   * stores of rows and columns inside the output only, with the alignment of one element.  ODD: the
//     output's row stride is odd (store_row8_odd; a kernel of its own: with both epilogues in one the
//     compiler converts what both store ahead of their branch, and spills).
template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32, bool HALF,
          bool EDGE = false, bool ODD = false>
__device__ __forceinline__ void solo_gemm(const GemmArgs& g, const int tm, const int tn, const int split) {
  constexpr uint32_t kOutside = 0x80000000u;
  constexpr int WTM = BM / 2, WTN = BN / 2, FRM = BM / 32, FRN = BN / 32;
  constexpr int PK = 64, NSLOT = 5;
  constexpr int NM = FRM * FRN;         // MFMAs per step
  using OA = DeepOperand<A_KMAJOR, false, BM>;
  using OB = DeepOperand<B_KMAJOR, true, BN>;
  constexpr uint32_t SLOT = OA::BYTES > OB::BYTES ? OA::BYTES : OB::BYTES;  // 32 or 16 KiB
  constexpr int NCA = OA::DMA_N, NCB = OB::DMA_N;  // copies per tile and wave
  constexpr int NFRAG = FRM + FRN;                 // fragment reads per step
  constexpr int READ_EVERY = (NM / 2) / NFRAG;     // a fragment read every .. MFMAs, first half of a step
  constexpr int COPY_EVERY_A = (NM / 2) / NCA;     // a copy every .. MFMAs, second half
  constexpr int COPY_EVERY_B = (NM / 2) / NCB;
  static_assert((BM <= 256 && BN == 256) || ((BM == 256 || BM == 128) && BN == 128), "tile sizes with a schedule below");
  static_assert(READ_EVERY >= 1 && COPY_EVERY_A >= 1 && COPY_EVERY_B >= 1, "schedule fits a step");
  // Gate/up forward (gate_up_copy): the tile covers 128 output columns.
  constexpr bool SWIGLU = EPI == EPI_SWIGLU;
  // Two-term product: stages 0 .. k_first / 64 - 1 copy from (A, B), the others from
  // (A2, B2); everything behind the copies is unchanged.
  constexpr bool PAIR = EPI == EPI_PAIR;
  static_assert(!EDGE || !PAIR, "whole tiles only");
  static_assert(!ODD || (A_KMAJOR && B_KMAJOR), "the forward");
  static_assert(!PAIR || (A_KMAJOR && !B_KMAJOR), "the two-term product is the dgrad layout");
  static_assert(!SWIGLU || (BN == 256 && A_KMAJOR && B_KMAJOR && !OUT_F32),
                "the gate/up forward runs on tiles of 256 columns with contraction-contiguous operands");

  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  f32x4 acc[FRM][FRN];

  // tm, tn: this workgroup's tile; for a split contraction its part, KP stages from stage s0 on.
  const int m0 = tm * BM, n0 = tn * (SWIGLU ? BN / 2 : BN);
  int KP, s0;
  if constexpr (EDGE) {
    static_assert(PK == 64, "stages_of_part");
    const StageRange part = stages_of_part(g.Kc, split, g.splits);
    s0 = part.first;
    KP = part.count;
  } else {
    KP = (g.splits > 1 ? g.k_split : g.Kc) / PK;
    s0 = split * KP;
  }

  const uint32_t a_bytes = (uint32_t)((int64_t)(A_KMAJOR ? g.M : g.Kc) * g.lda * 2);
  const uint32_t b_bytes = (uint32_t)((int64_t)(B_KMAJOR ? g.N : (PAIR ? g.k_first : g.Kc)) * g.ldb * 2);
  const __amdgpu_buffer_rsrc_t ra_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.A, 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.B, 0, (int)b_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb2_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(SWIGLU ? g.B2 : g.B), 0, (int)b_bytes, 0x00020000);
  // the pair the copies read from (PAIR only: switched once, two stages before the
  // first stage of the second pair)
  __amdgpu_buffer_rsrc_t ra_cur = ra_rsrc, rb_cur = rb_rsrc;
  [[maybe_unused]] __amdgpu_buffer_rsrc_t rb2_cur = rb2_rsrc;   // EDGE: the up weights'
  uint32_t a_is = 0, b_is = 0, va = 0, vb = 0;   // per-lane copy offsets of the current tile
  const uint32_t a_step = (uint32_t)((A_KMAJOR ? (int64_t)PK : (int64_t)PK * g.lda) * 2);
  const uint32_t b_step = (uint32_t)((B_KMAJOR ? (int64_t)PK : (int64_t)PK * g.ldb) * 2);
  uint32_t ka = 0, kb = 0;  // byte offsets of the next A / B tile to copy
  uint32_t wslot = 0;       // ring slot (byte offset) the next copied tile takes

  OperandWalk walk_a, walk_b, walk_b2;   // EDGE

  const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(char, lds);
  uint32_t ra0[OA::NADDR], rb0[OB::NADDR];
  OA::read_bases(ra0, wm * WTM, lane);
  OB::read_bases(rb0, wn * WTN, lane);
#pragma unroll
  for (int i = 0; i < OA::NADDR; ++i) ra0[i] += lds0;
#pragma unroll
  for (int i = 0; i < OB::NADDR; ++i) rb0[i] += lds0;

  auto next_slot = [&](uint32_t s_) { return s_ + SLOT == NSLOT * SLOT ? 0u : s_ + SLOT; };
  auto copy_a = [&](auto c_) {
    if constexpr (EDGE)
      OA::template dma_one<decltype(c_)::value>(ra_cur, va, 0, a_is, lds + wslot, wave);
    else if constexpr (PAIR)
      OA::template dma_one<decltype(c_)::value>(ra_cur, va, ka, a_is, lds + wslot, wave);
    else
      OA::template dma_one<decltype(c_)::value>(ra_rsrc, va, ka, a_is, lds + wslot, wave);
  };
  auto copy_b = [&](auto c_) {
    constexpr int I = decltype(c_)::value;
    if constexpr (SWIGLU) {
      constexpr GateUpCopy from = gate_up_copy(BN, I);
      if constexpr (EDGE)
        OB::template dma_one<I, from.at>(from.up ? rb2_cur : rb_cur, vb, 0, b_is, lds + wslot, wave);
      else
        OB::template dma_one<I, from.at>(from.up ? rb2_rsrc : rb_rsrc, vb, kb, b_is, lds + wslot, wave);
    } else if constexpr (EDGE) {
      OB::template dma_one<I>(rb_cur, vb, 0, b_is, lds + wslot, wave);
    } else if constexpr (PAIR) {
      OB::template dma_one<I>(rb_cur, vb, kb, b_is, lds + wslot, wave);
    } else {
      OB::template dma_one<I>(rb_rsrc, vb, kb, b_is, lds + wslot, wave);
    }
  };
  auto a_done = [&]() {
    if constexpr (EDGE) {
      walk_a.advance();
      ra_cur = walk_a.resource();
    } else {
      ka += a_step;
    }
    wslot = next_slot(wslot);
  };
  auto b_done = [&]() {
    if constexpr (EDGE) {
      walk_b.advance();
      rb_cur = walk_b.resource();
      if constexpr (SWIGLU) {
        walk_b2.advance();
        rb2_cur = walk_b2.resource();
      }
    } else {
      kb += b_step;
    }
    wslot = next_slot(wslot);
  };

  bf16x8 fa0[FRM], fb0[FRN], fa1[FRM], fb1[FRN];  // register sets of steps 0 / 1
  // fragment f of FRM + FRN (A fragments, then B fragments) of step ST of the stage
  // whose tiles sit at sa / sb, into register set ST
  auto read = [&](auto st_, auto f_, uint32_t sa, uint32_t sb) {
    constexpr int ST = decltype(st_)::value, f = decltype(f_)::value;
    bf16x8(&fa)[FRM] = ST ? fa1 : fa0;
    bf16x8(&fb)[FRN] = ST ? fb1 : fb0;
    if constexpr (f < FRM) {
      uint32_t ra[OA::NADDR];
#pragma unroll
      for (int i = 0; i < OA::NADDR; ++i) ra[i] = ra0[i] + sa;
      OA::template read_frag<ST, f>(fa[f], ra);
    } else {
      uint32_t rb[OB::NADDR];
#pragma unroll
      for (int i = 0; i < OB::NADDR; ++i) rb[i] = rb0[i] + sb;
      OB::template read_frag<ST, f - FRM>(fb[f - FRM], rb);
    }
  };
  uint32_t sa = 0, sb = SLOT;  // slots of the current stage's tiles

  // HAS2: stage p + 2 exists (its tiles are copied during this stage);
  // LAST: no stage follows.
  auto stage = [&](auto has2_, auto last_) {
    constexpr bool HAS2 = decltype(has2_)::value;
    constexpr bool LAST = decltype(last_)::value;
    const uint32_t na = next_slot(sb), nb = next_slot(na);  // slots of stage p + 1
    static_for<2>([&](auto st_) {
      constexpr int ST = decltype(st_)::value;
      bf16x8(&fa)[FRM] = ST ? fa1 : fa0;
      bf16x8(&fb)[FRN] = ST ? fb1 : fb0;
      wait_all_fragments(fa, fb);  // every read of this set was issued during the previous step
      if constexpr (ST == 1 && !LAST) {
        if (HAS2) wait_vmcnt<NCA>();  // A(p+2) may be in flight
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<NM>([&](auto m_) {
        constexpr int m = decltype(m_)::value;
        constexpr int i = m / FRN, j = m % FRN;
        // Inline assembly pins the register classes (accumulators in AGPRs, fragments
        // in VGPRs): with the builtin the allocator moves two-instruction
        // (transposed) fragments through AGPRs and spills.  No MFMA hazard can arise:
        // fragments come from LDS behind s_waitcnt, and an accumulator is touched
        // again only NM - 1 (at least 15) independent MFMAs later.
        // (fragments are opaque 16-byte registers: the mnemonic alone names the type)
        if constexpr (HALF)
          asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
                       : "+a"(acc[i][j])
                       : "v"(fb[j]), "v"(fa[i]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                       : "+a"(acc[i][j])
                       : "v"(fb[j]), "v"(fa[i]));
        constexpr int CE = ST == 0 ? COPY_EVERY_A : COPY_EVERY_B;  // step 0 copies A, step 1 B
        constexpr int NCX = ST == 0 ? NCA : NCB;
        // Copies in the first half of a step, fragment reads in the second: a copy is issued
        // as soon as the barrier (step 1) or the previous step (step 0) has freed its slot,
        // which gives the tile a quarter of a stage more to arrive than the other order
        // (measured: +2.6 % on the step, +7 % on the MLP shard); the reads still have half
        // a step to return.
        constexpr int mc = m;            // position in the copying half
        constexpr int mr = m - NM / 2;   // position in the reading half
        if constexpr (mr >= 0 && mr < NM / 2 && mr % READ_EVERY == 0 && mr / READ_EVERY < NFRAG) {
          if constexpr (ST == 0) read(std::integral_constant<int, 1>{},
                                      std::integral_constant<int, mr / READ_EVERY>{}, sa, sb);
          else if constexpr (!LAST) read(std::integral_constant<int, 0>{},
                                         std::integral_constant<int, mr / READ_EVERY>{}, na, nb);
        }
        // (an independent statement: a read and a copy may fall behind the same MFMA)
        static_assert((NM / 2) / CE >= NCX, "every copy of the tile has a place in the half step");
        if constexpr (HAS2 && mc >= 0 && mc < NM / 2 && mc % CE == CE - 1 && mc / CE < NCX) {
          if constexpr (ST == 0) copy_a(std::integral_constant<int, mc / CE>{});
          else copy_b(std::integral_constant<int, mc / CE>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (HAS2 && ST == 0) a_done();
      if constexpr (HAS2 && ST == 1) b_done();
    });
    sa = na;
    sb = nb;
  };
  using T = std::true_type;
  using F = std::false_type;

  uint32_t va_end = 0, vb_end = 0;   // EDGE: the copy offsets of the operand's last stage
  if constexpr (EDGE) {
    walk_a.start(g.A, A_KMAJOR, g.M, g.Kc, g.lda, m0, s0 * PK);
    walk_b.start(g.B, B_KMAJOR, g.N, g.Kc, g.ldb, n0, s0 * PK);
    ra_cur = walk_a.resource();
    rb_cur = walk_b.resource();
    if constexpr (SWIGLU) {
      walk_b2.start(g.B2, B_KMAJOR, g.N, g.Kc, g.ldb, n0, s0 * PK);
      rb2_cur = walk_b2.resource();
    }
    va = OA::dma_offset(g.lda, 0, wave, lane, a_is);
    vb = OB::dma_offset(g.ldb, 0, wave, lane, b_is);
    va_end = va;
    vb_end = vb;
    const int over = (int)((int64_t)(s0 + KP) * PK - g.Kc);   // contraction elements the last stage lacks
    if (over > 0) {
      if (A_KMAJOR && 8 * OA::dma_chunk(wave, lane) >= PK - over) va_end = kOutside;
      if (B_KMAJOR && 8 * OB::dma_chunk(wave, lane) >= PK - over) vb_end = kOutside;
    }
    if (KP == 1) {
      va = va_end;
      vb = vb_end;
    }
  } else {
    va = OA::dma_offset(g.lda, m0, wave, lane, a_is);
    vb = OB::dma_offset(g.ldb, n0, wave, lane, b_is);
    ka = (uint32_t)s0 * a_step;
    kb = (uint32_t)s0 * b_step;
  }

  // A0 B0 (A1 B1) up front.
  static_for<NCA>(copy_a); a_done();
  static_for<NCB>(copy_b); b_done();
  if (KP > 1) {
    if (EDGE && KP == 2) {
      va = va_end;
      vb = vb_end;
    }
    static_for<NCA>(copy_a); a_done();
    static_for<NCB>(copy_b); b_done();
  }
  // The accumulators are cleared here, while the first tiles are on their way: left
  // to itself the compiler clears them where they are first used, behind the wait.
#pragma unroll
  for (int i = 0; i < FRM; ++i)
#pragma unroll
    for (int j = 0; j < FRN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < FRM; ++i) tie_accumulators(acc[i]);
  if (KP > 1) {
    wait_vmcnt<NCA + NCB>();
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();

  static_for<NFRAG>([&](auto f_) { read(std::integral_constant<int, 0>{}, f_, sa, sb); });

  if constexpr (PAIR) {
    const int kp1 = g.k_first / PK;  // >= 2: the stages copied up front are of the first pair
    const uint32_t b2_bytes = (uint32_t)((int64_t)(g.Kc - g.k_first) * g.ldb * 2);
    for (int p = 0; p < KP - 2; ++p) {
      if (p == kp1 - 2) {  // this stage copies the tiles of stage kp1, the second pair's first
        ra_cur = __builtin_amdgcn_make_buffer_rsrc((void*)g.A2, 0, (int)a_bytes, 0x00020000);
        rb_cur = __builtin_amdgcn_make_buffer_rsrc((void*)g.B2, 0, (int)b2_bytes, 0x00020000);
        ka = 0;
        kb = 0;
      }
      stage(T{}, F{});
    }
  } else {
    for (int p = 0; p < KP - 2; ++p) {
      if (EDGE && p == KP - 3) {   // this stage copies the last stage's tiles
        va = va_end;
        vb = vb_end;
      }
      stage(T{}, F{});
    }
  }
  if (KP > 1) stage(F{}, F{});
  stage(F{}, T{});
  // The compiler does not know that the statements above are MFMAs: left alone it
  // copies an accumulator out of its AGPRs right behind the MFMA that writes it,
  // before the result has left the pipeline.  Every accumulator is therefore
  // passed through a statement that follows the last MFMA by more than its
  // latency; the epilogue can only read the values these statements return.
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < FRM; ++i) tie_accumulators(acc[i]);
  if constexpr (SWIGLU) {
    store_gate_up<HALF, EDGE>(acc, g, m0 + wm * WTM, n0 + wn * (WTN / 2), lane);
  } else {
    // (the ring slot behind the last stage's two is free: no wave reads or fills it any more)
    store_blocks<EPI, OUT_F32, HALF, EDGE, ODD>(acc, g, split, m0 + wm * WTM, n0 + wn * WTN, lane,
                                                (float*)(lds + sa) + wave * (WTM * 8));
  }
}

// The tile, and the part of the contraction, of a workgroup of a launch of its own or of a range of one.
template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32, bool HALF,
          bool EDGE = false, bool ODD = false>
__device__ __forceinline__ void solo_gemm(const GemmArgs& g) {
  int tm, tn, split = 0, pid = blockIdx.x - g.wg_first;
  if (g.splits > 1) {
    split = pid / (g.tiles_m * g.tiles_n);
    pid -= split * (g.tiles_m * g.tiles_n);
  }
  tile_of_workgroup(pid, g.tiles_m, g.tiles_n, tm, tn);
  solo_gemm<BM, BN, A_KMAJOR, B_KMAJOR, EPI, OUT_F32, HALF, EDGE, ODD>(g, tm, tn, split);
}

}  // namespace
}  // namespace axn
