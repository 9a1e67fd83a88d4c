// Embedding table lookup and its dense weight gradient for gfx950.
//
// Forward is a row gather, out[t, :] = W[ids[t], :]: one wave per 64 x 16 bytes of
// an output row, 16-byte loads and stores.
//
// Backward is dW[v, :] (+)= sum over the tokens t with ids[t] == v of dY[t, :].
// It is written as a gather as well, so that it needs no floating-point atomics
// and its result does not depend on the order in which workgroups run:
//   1. the token positions are sorted by id (stable LSD radix sort over the bits
//      of the vocabulary size, kernels below: no library call, no atomics on
//      floating-point data, nothing but kernel launches);
//   2. the first sorted slot of every id present is recorded in row_start[V] (by the
//      sort's last pass: the smallest slot a row's tokens land in);
//   3. one wave per 64 x 16 bytes of a dW row walks that row's run of sorted
//      slots, adds the dY rows in ascending token order in fp32 and stores the
//      row once; rows no token names are stored as zeros (beta = 0) or left alone
//      (beta = 1).  dW is never read unless beta = 1.  Where the table has at least twice as
//      many rows as there are tokens, the sort's launches write the zeros, to the whole table,
//      beside the sort, and step 3 takes one wave per sorted slot.
// The max_norm renormalisation of the looked-up rows reuses steps 1 and 2: one
// wave per row that occurs, so a row named by many tokens is scaled once.
#include "axn_internal.h"

#include <cstring>
#include <type_traits>

namespace axn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVES_PER_BLOCK = 4;
// LDS the weight-gradient kernel reserves per workgroup and never touches: 36 KB hold it at
// 16 waves per CU, where its stores stream best (all 32 resident: 263 us at 16384 tokens x 2048
// into 128256 rows; 16 to 20: 238 us; 12: 323 us; measured on MI355X).
constexpr int EMB_BWD_LDS = 36864;

// ---- forward ----------------------------------------------------------------
// Rows are moved as opaque 16-byte pieces: the element type only sets how many
// pieces a row has.  `pieces` = row bytes / 16, ld* in 16-byte pieces.
__global__ void __launch_bounds__(64 * WAVES_PER_BLOCK)
    embedding_fwd_kernel(const int64_t* __restrict__ ids, const u32x4* __restrict__ W,
                         u32x4* __restrict__ out, int64_t T, int64_t V, int64_t pieces,
                         int64_t ldw, int64_t ldo, int units_per_row, int* status) {
  const int lane = threadIdx.x & 63;
  const int64_t unit = block_number() * WAVES_PER_BLOCK + (threadIdx.x >> 6);
  const int64_t t = unit / units_per_row;
  if (t >= T) return;
  const int64_t piece = (unit % units_per_row) * 64 + lane;
  if (piece >= pieces) return;
  const int64_t id = ids[t];
  u32x4 v = {0u, 0u, 0u, 0u};
  if (id >= 0 && id < V)
    v = W[id * ldw + piece];
  else if (status != nullptr && piece == 0)
    *status = 1;
  __builtin_nontemporal_store(v, out + t * ldo + piece);
}

// One 16-byte store, non-temporal and written through (nt + sc1): the dense weight gradient
// is written once, row after row, and read much later.  (The s_nop: the wait states a store
// of more than 8 bytes needs before its data registers are written again are the
// compiler's to insert for its own stores, not for this one.)
template <typename V>
__device__ __forceinline__ void store_through(V v, void* p) {
  static_assert(sizeof(V) == 16, "one 16-byte store");
  asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// Zeros for a part of the gradient, written by the workgroups of a sort launch behind the
// `sort_blocks` that sort: a sort of a few thousand tokens keeps 32 workgroups busy for 25 us
// in three launches, and the rest of the chip writes the gradient meanwhile.
struct Fill {
  u32x4* first;          // 16-byte vectors
  int64_t count;
  int64_t sort_blocks;
};
constexpr int FILL_THREADS = 256;   // one vector a lane: see SORT_FILL_LDS
__device__ __forceinline__ bool fill_zeros(const Fill& fill) {
  const int64_t b = (int64_t)blockIdx.x - fill.sort_blocks;
  if (b < 0) return false;
  const int64_t i = b * FILL_THREADS + threadIdx.x;
  if (i < fill.count) store_through(u32x4{0u, 0u, 0u, 0u}, fill.first + i);
  return true;
}

// ---- sorting the token positions by id ---------------------------------------
// Stable least-significant-digit radix sort of (key, position) pairs, keys over [0, V]
// (V for an id outside [0, V): those sort behind every row), in 1 to 4 passes of at most
// 10 bits.  A workgroup of 4 waves owns 256 G consecutive slots, wave w the w-th quarter of
// them (G = 2 for batches up to 2^15 tokens, where short pieces give the sort more waves,
// G = 8 beyond, where they keep the count arrays small).  Per pass:
//   counts   hist[digit][workgroup] = slots of the workgroup whose key has that digit (pass
//            0: counted by the kernel that writes the keys; later passes: counted by the
//            previous pass's scatter with integer atomics, which add up to the same counts
//            in any order)
//   scan     exclusive prefix sum over the digit-major array: where the workgroup's slots
//            of a digit go (a launch of its own beyond 2^17 tokens; up to there the array is
//            small and every workgroup of the scatter sums what lies in front of it itself)
//   scatter  every wave counts the digits of its quarter, which places the quarters of a
//            digit one behind the other; then a wave walks its quarter 64 slots at a time
//            in slot order: lanes with equal digits find one another with one ballot per
//            digit bit, and a slot goes to (the running count of its digit) + (equal-digit
//            lanes before it).  Slots of equal digit keep their order, which is what makes
//            the sort stable and the order of every row's tokens ascending.
constexpr int SORT_SHORT_BATCH = 1 << 15;   // tokens up to which a wave's quarter is 128 slots
constexpr int SORT_FUSED_BATCH = 1 << 17;   // tokens (at most 64 workgroups) up to which no scan is launched
constexpr int SORT_WAVES = 4;        // waves per workgroup
constexpr int SORT_MAX_BITS = 10;    // digit width: 1024 counters per wave in LDS
constexpr int SORT_MAX_PASSES = 4;
// LDS of a workgroup in launches that also clear the gradient: 24 waves per CU, where a fill is fastest (7.3
// TB/s; 6.8 with 32).  What the kernels declare themselves comes off it.
constexpr int SORT_FILL_LDS = 27136;
constexpr int SORT_PREPARE_LDS = 4 << SORT_MAX_BITS, SORT_SCATTER_LDS = SORT_WAVES * (4 << SORT_MAX_BITS) + 64;

struct SortPlan {
  int passes;
  int bits[SORT_MAX_PASSES], shift[SORT_MAX_PASSES];
  int groups;                         // 64-slot groups per wave
  bool fused_scan;                    // the scatter derives the prefix sums itself
  int64_t nblk;                       // workgroups = units of the count arrays
  size_t hist_ofs[SORT_MAX_PASSES];   // in ints, from the start of the histogram area
  size_t hist_ints;
};

__device__ __forceinline__ int key_of_id(int64_t id, int64_t V) {
  return (id >= 0 && id < V) ? (int)id : (int)V;
}

// keys[i], vals[i] = i, pass 0's counts; row_start[v] = -1, status = 0, the later passes'
// counts cleared.  (row_start is not wanted where the gradient goes slot by slot.)
template <int G>
__global__ void __launch_bounds__(64 * SORT_WAVES)
    embedding_sort_prepare_kernel(const int64_t* __restrict__ ids, int* __restrict__ keys,
                                  int* __restrict__ vals, int* __restrict__ row_start, int* status,
                                  int* __restrict__ hist0, int* __restrict__ hist_rest,
                                  int64_t hist_rest_ints, int64_t T, int64_t V, int64_t nblk,
                                  int bits0, bool block_major, const Fill fill) {
  __shared__ int cnt[1 << SORT_MAX_BITS];
  if (fill_zeros(fill)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nthreads = fill.sort_blocks * blockDim.x;
  for (int64_t i = gtid; i < hist_rest_ints; i += nthreads) hist_rest[i] = 0;
  if (row_start != nullptr)
    for (int64_t i = gtid; i < V; i += nthreads) row_start[i] = -1;
  if (gtid == 0) *status = 0;
  const int nd = 1 << bits0;
  for (int d = threadIdx.x; d < nd; d += 64 * SORT_WAVES) cnt[d] = 0;
  __syncthreads();
  const int64_t blk = blockIdx.x;
  if (blk < nblk) {
    const int64_t first = (blk * SORT_WAVES + w) * (64 * G);
    int64_t id[G];   // all loads of the wave in flight at once
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t i = first + g * 64 + lane;
      id[g] = i < T ? ids[i] : 0;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t i = first + g * 64 + lane;
      if (i < T) {
        const int key = key_of_id(id[g], V);
        keys[i] = key;
        vals[i] = (int)i;
        atomicAdd(&cnt[key & (nd - 1)], 1);
      }
    }
  }
  __syncthreads();
  if (blk < nblk)
    for (int d = threadIdx.x; d < nd; d += 64 * SORT_WAVES)
      hist0[block_major ? blk * nd + d : (int64_t)d * nblk + blk] = cnt[d];
}

// Inclusive prefix sum across the 64 lanes in six data-parallel-primitive adds (no LDS
// round trip): shifts by 1, 2, 4, 8 inside the rows of 16 lanes (a lane the shift leaves
// without a source adds 0), then lane 15's total into rows 1 and 3, then lane 31's into
// rows 2 and 3.
__device__ __forceinline__ int wave_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);    // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);    // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);    // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
  return v;
}

// In-place exclusive prefix sum over n ints, one workgroup of 1024 threads: tiles of 65536
// entries, 4096 consecutive ones per wave held in registers as 16 rows of 64 lanes x 4 (every
// access of a wave covers 1 KiB of consecutive bytes, every load of a tile in flight at
// once, nothing read twice); rows are scanned across the lanes, the rows' totals along the
// wave, the waves' totals across the workgroup, and a running total goes from tile to tile.
__global__ void __launch_bounds__(1024) embedding_sort_scan_kernel(int* __restrict__ h, int64_t n) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  constexpr int ROWS = 16;                // 16-byte vectors per thread and tile
  __shared__ int wave_total[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int carry = 0;
  for (int64_t tile = 0; tile < n; tile += 1024 * ROWS * 4) {
    const int64_t lo = tile + (int64_t)w * (64 * ROWS * 4) + lane * 4;
    i32x4 v[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int64_t i = lo + 256 * j;
      if (i + 3 < n) {
        v[j] = *(const i32x4*)(h + i);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = i + e < n ? h[i + e] : 0;
      }
    }
    int excl[ROWS];   // sum of everything of this wave's part in front of v[j]
    int wave_sum = 0;
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int s = v[j][0] + v[j][1] + v[j][2] + v[j][3];
      const int incl = wave_inclusive_sum(s);
      excl[j] = wave_sum + incl - s;
      wave_sum += __builtin_amdgcn_readlane(incl, 63);
    }
    __syncthreads();   // the previous tile's totals have been read
    if (lane == 0) wave_total[w] = wave_sum;
    __syncthreads();
    int before = carry, all = 0;
    for (int k = 0; k < 16; ++k) {
      if (k < w) before += wave_total[k];
      all += wave_total[k];
    }
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int64_t i = lo + 256 * j;
      i32x4 o;
      o[0] = before + excl[j];
      o[1] = o[0] + v[j][0];
      o[2] = o[1] + v[j][1];
      o[3] = o[2] + v[j][2];
      if (i + 3 < n) {
        *(i32x4*)(h + i) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < n) h[i + e] = o[e];
      }
    }
    carry += all;
  }
}

// SCANNED: `base` holds the exclusive prefix sums of the counts (embedding_sort_scan_kernel
// has run); otherwise it holds the counts themselves and every workgroup derives its own
// part of the prefix sums from them - all digit-major rows in front of a digit's row and
// the row up to this workgroup - which for few workgroups costs less than a launch.
template <int G, bool SCANNED>
__global__ void __launch_bounds__(64 * SORT_WAVES)
    embedding_sort_scatter_kernel(const int* __restrict__ keys_in, const int* __restrict__ vals_in,
                                  int* __restrict__ keys_out, int* __restrict__ vals_out,
                                  const int* __restrict__ base, int* __restrict__ next_hist,
                                  int* __restrict__ row_start, int* status, int64_t T, int64_t V,
                                  int64_t nblk, int shift, int bits, int next_shift, int next_bits,
                                  const Fill fill) {
  __shared__ int cnt[SORT_WAVES][1 << SORT_MAX_BITS];
  if (fill_zeros(fill)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t blk = blockIdx.x;
  const int nd = 1 << bits;
  for (int d = threadIdx.x; d < SORT_WAVES * nd; d += 64 * SORT_WAVES) cnt[d / nd][d % nd] = 0;
  const int64_t first = (blk * SORT_WAVES + w) * (64 * G);
  int kreg[G], vreg[G];   // all loads of the wave in flight at once
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t i = first + g * 64 + lane;
    const bool active = i < T;
    kreg[g] = active ? keys_in[i] : 0;
    vreg[g] = active ? vals_in[i] : 0;
  }
  __syncthreads();
  // the digits of this wave's quarter
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (first + g * 64 + lane < T) atomicAdd(&cnt[w][(kreg[g] >> shift) & (nd - 1)], 1);
  __syncthreads();
  // counts -> first destination of each wave's slots of a digit; a thread sees to the
  // digits t, t + 256, t + 512, t + 768 (at most 1024 digits, 256 threads)
  int first_dest[4] = {0, 0, 0, 0};
  if constexpr (SCANNED) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = threadIdx.x + 256 * e;
      if (d < nd) first_dest[e] = base[(int64_t)d * nblk + blk];
    }
  } else {
    // The counts lie workgroup-major here ([workgroup][digit]: consecutive lanes read
    // consecutive words).  A digit's slots start behind every slot of a smaller digit (the
    // digits' totals, scanned over the workgroup in digit order) and behind the digit's
    // slots of the workgroups in front of this one.
    __shared__ int wave_total[4][SORT_WAVES];
    int tot[4] = {0, 0, 0, 0}, pre[4] = {0, 0, 0, 0};
#pragma unroll 8
    for (int64_t b = 0; b < nblk; ++b) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = threadIdx.x + 256 * e;
        const int c = d < nd ? base[b * nd + d] : 0;
        tot[e] += c;
        pre[e] += b < blk ? c : 0;
      }
    }
    int incl[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      incl[e] = wave_inclusive_sum(tot[e]);
      if (lane == 63) wave_total[e][w] = incl[e];
    }
    __syncthreads();
    int run = 0;   // slots of the digits in front of digit 256 e + 64 w
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int k = 0; k < SORT_WAVES; ++k) {
        if (k == w) first_dest[e] = run + incl[e] - tot[e] + pre[e];
        run += wave_total[e][k];
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = threadIdx.x + 256 * e;
    if (d < nd) {
      int run = first_dest[e];
#pragma unroll
      for (int k = 0; k < SORT_WAVES; ++k) {
        const int c = cnt[k][d];
        cnt[k][d] = run;
        run += c;
      }
    }
  }
  __syncthreads();
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int g = 0; g < G; ++g) {   // (every wave makes every trip: the barriers below)
    const bool active = first + g * 64 + lane < T;
    const int key = kreg[g];
    const int val = vreg[g];
    const int d = (key >> shift) & (nd - 1);
    uint64_t same = __ballot(active);   // the lanes whose slot has this lane's digit
    for (int b = 0; b < bits; ++b) {
      const bool bit = (d >> b) & 1;
      const uint64_t with = __ballot(active && bit);
      same &= bit ? with : ~with;
    }
    const int off = active ? cnt[w][d] : 0;
    __syncthreads();   // every lane has read its digit's count before any lane moves one on
    if (active && lane == 63 - __builtin_clzll(same)) cnt[w][d] = off + __builtin_popcountll(same);
    __syncthreads();
    // The ids of a text repeat (the most frequent one is a twentieth of all tokens), and an
    // atomic on one word is one at a time in L2: the lanes that would hit the same word are
    // joined first, and one of them goes (16384 such ids into 128256 rows: a scatter pass takes
    // 32 us without, 9 us with it; on ids drawn evenly both take 8).
    const int dest = off + __builtin_popcountll(same & below);
    if (next_hist != nullptr) {
      const int nx = (key >> next_shift) & ((1 << next_bits) - 1);
      const int nb = dest / (64 * G * SORT_WAVES);
      // equal next digit, and the same unit: the destinations of `same` are consecutive, so they
      // lie in at most two units, one of them odd
      uint64_t joined = same;
      for (int b = 0; b <= next_bits && __ballot(active) != 0; ++b) {
        const bool bit = ((b < next_bits ? nx >> b : nb) & 1) != 0;
        const uint64_t with = __ballot(active && bit);
        joined &= bit ? with : ~with;
      }
      if (active) {
        keys_out[dest] = key;
        vals_out[dest] = val;
        if ((joined & below) == 0)
          atomicAdd(&next_hist[SCANNED ? (int64_t)nx * nblk + nb : ((int64_t)nb << next_bits) + nx],
                    __builtin_popcountll(joined));
      }
    } else {
      // last pass: the slots are final, and a row's run starts at the smallest of them
      // (row_start holds -1 = the largest unsigned value until a slot arrives).  Lanes of one
      // digit take their slots in lane order, and equal keys are neighbours among them (the
      // passes before have sorted the other digits): only the first lane of a run goes.
      const uint64_t before = same & below;
      const int prev = before != 0 ? 63 - __builtin_clzll(before) : lane;
      const int prev_key = __shfl(key, prev, 64);
      if (active) {
        keys_out[dest] = key;
        vals_out[dest] = val;
        if (key < V) {
          if (row_start != nullptr && (prev == lane || prev_key != key))
            atomicMin((unsigned*)&row_start[key], (unsigned)dest);
        } else {
          *status = 1;   // an id outside the table
        }
      }
    }
  }
}

// ---- backward ------------------------------------------------------------------
// One 16-byte vector of a table row as fp32 values.
template <typename T>
struct Vec;
template <>
struct Vec<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load_cached(const float* p, float (&x)[4]) {
    const f32x4 v = *(const f32x4*)p;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = v[e];
  }
  static __device__ __forceinline__ void store(float* p, const float (&x)[4]) {
    store_through(f32x4{x[0], x[1], x[2], x[3]}, p);
  }
  static __device__ __forceinline__ void store_cached(float* p, const float (&x)[4]) {
    *(f32x4*)p = f32x4{x[0], x[1], x[2], x[3]};
  }
};
template <>
struct Vec<uint16_t> {
  static constexpr int N = 8;
  static __device__ __forceinline__ void load_cached(const uint16_t* p, float (&x)[8]) {
    const bf16x8 v = *(const bf16x8*)p;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
  }
  static __device__ __forceinline__ void store(uint16_t* p, const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__bf16)x[e];
    store_through(v, p);
  }
  static __device__ __forceinline__ void store_cached(uint16_t* p, const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__bf16)x[e];
    *(bf16x8*)p = v;
  }
};

template <>
struct Vec<_Float16> {
  static constexpr int N = 8;
  typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ void load_cached(const _Float16* p, float (&x)[8]) {
    const f16x8 v = *(const f16x8*)p;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
  }
  static __device__ __forceinline__ void store(_Float16* p, const float (&x)[8]) {
    f16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (_Float16)x[e];
    store_through(v, p);
  }
  static __device__ __forceinline__ void store_cached(_Float16* p, const float (&x)[8]) {
    f16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (_Float16)x[e];
    *(f16x8*)p = v;
  }
};

// VEC consecutive elements of a gradient row (VEC = 2, 4 or 8) as they lie in memory, so that
// several rows can be on their way before the first is added; 16 bytes per instruction where
// the type allows.  Gradient rows are read once: non-temporal.
template <typename T, int VEC>
struct RowPiece;
template <int VEC>
struct RowPiece<float, VEC> {
  static constexpr int W = VEC < 4 ? VEC : 4;
  typedef float fxv __attribute__((ext_vector_type(W)));
  fxv v[VEC / W];
  __device__ __forceinline__ void load(const float* p) {
#pragma unroll
    for (int h = 0; h < VEC / W; ++h) v[h] = __builtin_nontemporal_load((const fxv*)p + h);
  }
  __device__ __forceinline__ float get(int e) const { return v[e / W][e % W]; }
};
template <int VEC>
struct RowPiece<uint16_t, VEC> {
  typedef __bf16 bf16xv __attribute__((ext_vector_type(VEC)));
  bf16xv v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = __builtin_nontemporal_load((const bf16xv*)p); }
  __device__ __forceinline__ float get(int e) const { return (float)v[e]; }
};
template <int VEC>
__device__ __forceinline__ void add_old(const float* p, float (&x)[VEC]) {
  const f32x4 v = *(const f32x4*)p;
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] += v[e];
}
template <int VEC>
__device__ __forceinline__ void add_old(const uint16_t* p, float (&x)[VEC]) {
  const bf16x8 v = *(const bf16x8*)p;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] += (float)v[e];
}

// Adds the gradient rows whose positions lanes i .. i + B - 1 hold in `pos` to acc, in lane
// order.  All loads come first and under no condition (a lane past the row's end loads the
// row's last columns): with a condition per row the compiler pairs each load with its addition,
// and every row waits for the one before.  U pieces of 64 x VEC columns, `col0` this lane's
// first column.
template <typename TY, int VEC, int U, int B>
__device__ __forceinline__ void add_batch(float (&acc)[U][VEC], int i, int pos, const TY* dY, int64_t lddy,
                                          int64_t col0, int64_t H, bool scaled, float inv) {
  RowPiece<TY, VEC> g[B][U];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const TY* row = dY + (int64_t)__builtin_amdgcn_readlane(pos, i + b) * lddy;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t col = col0 + u * 64 * VEC;
      g[b][u].load(row + (col < H ? col : H - VEC));
    }
  }
  __builtin_amdgcn_sched_barrier(0);   // (the scheduler, too, would pair them, to save registers)
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < VEC; ++q)
        acc[u][q] = scaled ? __fmaf_rn(g[b][u].get(q), inv, acc[u][q]) : acc[u][q] + g[b][u].get(q);
}
// The same for lanes 0 .. n - 1, B rows on their way at a time.
template <typename TY, int VEC, int U, int B>
__device__ __forceinline__ void add_rows(float (&acc)[U][VEC], int n, int pos, const TY* dY, int64_t lddy,
                                         int64_t col0, int64_t H, bool scaled, float inv, int i = 0) {
  for (; i + B <= n; i += B) add_batch<TY, VEC, U, B>(acc, i, pos, dY, lddy, col0, H, scaled, inv);
  if constexpr (B > 1)
    if (i < n) add_rows<TY, VEC, U, B / 2>(acc, n, pos, dY, lddy, col0, H, scaled, inv, i);
}

template <typename TW, int VEC, int U>
__device__ __forceinline__ void store_rows(float (&acc)[U][VEC], TW* dst, int64_t col0, int64_t H, int beta) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (col0 + u * 64 * VEC >= H) break;
    if (beta != 0) add_old<VEC>(dst + u * 64 * VEC, acc[u]);
    Vec<TW>::store(dst + u * 64 * VEC, acc[u]);
  }
}

// Part of a 16-byte vector of the row.
template <typename TW, int VEC>
__device__ __forceinline__ void store_part(const float (&x)[VEC], TW* dst, int beta) {
  typedef std::conditional_t<sizeof(TW) == 4, float, __bf16> elem;
  typedef elem part __attribute__((ext_vector_type(VEC)));
  part o = beta != 0 ? *(const part*)dst : part{};
#pragma unroll
  for (int q = 0; q < VEC; ++q) o[q] = (elem)(x[q] + (float)o[q]);
  *(part*)dst = o;
}

// Table rows per token from which on the gradient is cleared by the sort's launches and then goes slot by
// slot.  Ids drawn evenly (the most rows written twice), 128256 rows x 2048, row by row -> slot by slot, us:
//   tokens          128256      64128       32064       16032       250
//   fp32            420 -> 458  319 -> 317  264 -> 240  234 -> 196  187 -> 147
//   bf16            237 -> 243  181 -> 164  153 -> 124  136 -> 101   99 -> 77
constexpr int64_t EMB_SLOT_ROWS = 2;
// Rows named by more than EMB_LONG_RUN tokens get waves of their own (below).
constexpr int EMB_LONG_RUN = 32;
// Workgroups that are resident together (256 CUs, 4 each: EMB_BWD_LDS).  Where all do not fit and those of the other
// rows take three quarters of the room at most, these start first: behind the long runs' they went where one
// ended first, several to a CU, and the launch waited for them.  Elsewhere the long runs, the longest chains, do.
// us, long runs first / so: 8192 tokens drawn evenly from 512 rows x 3640, fp32 into bf16 (256 and 928 workgroups) 75 / 44,
// 16384 from 1024 x 1832 84 / 50, 8192 from 3000 x 1832 (750, 480) 39 / 35; as in a text 16384 from 512 x 3640 186 / 172; but
// 2000 from 1024 x 3640 (1024, 456) 32 / 35.
constexpr int64_t EMB_RESIDENT = 4 * 256;

// The slots of `row` among the 64 from slot `first` on: their count, and this lane's position.
__device__ __forceinline__ int run_in_chunk(const int* __restrict__ keys, const int* __restrict__ vals,
                                            int64_t first, int64_t T, int row, int lane, int& pos) {
  const int64_t j = first + lane;
  const int key = j < T ? keys[j] : -1;
  pos = j < T ? vals[j] : 0;
  const uint64_t in = __ballot(key == row);
  return in == ~0ull ? 64 : __builtin_ctzll(~in);
}

// One wave per (row, U x 64 x VEC columns): VEC = one 16-byte store of the dW type
// per lane, U such pieces per lane, 64 x VEC columns apart, so that a wave has U
// independent loads in flight per gradient row and U KiB of stores behind one
// look-up of row_start (with one piece per wave the 8192 resident waves of the chip
// covered 8 MB per memory latency: 4.2 TB/s on a gradient that is mostly zeros).
//
// The order of a row's sum is fixed (token order), so a row named by many tokens is a
// chain of additions, and what it costs is how many gradient rows are on their way at once
// and how many waves share the row.  A row's slots are read 64 at a time, one per lane, and
// four (two) gradient rows are in flight.  Rows with more than EMB_LONG_RUN tokens are left to the
// launch's first `long_blocks` workgroups: one wave per (64 sorted slots, 16 x VEC columns)
// that looks for such runs among its slots and has 64 (32) gradient rows in flight, so that a
// long run is spread over all pieces of its row and starts first.  The whole call for 16384
// tokens x 2048 fp32 whose ids fall off like those of a text, into 128256 rows: 1394 us with one
// row in flight and every row on the same waves, 239 with pieces twice as wide and half as many rows in flight
// (the most frequent row, a twelfth of the tokens, was the launch's longest chain), 203 us so and slot by slot.
// (Twice as many waves that find no long run cost 1 to 6 % of tables with fewer than two rows a token whose ids
// are drawn evenly, 30000 x 512 x 3640 108 -> 113 us; as in a text these take 0.72 to 0.90 of the time.)
// What bounds it now is the store of the 1.05 GB gradient (147 us of 250 tokens, 153 us for a
// plain fill) and the way of 134 MB of gradient rows behind it.
//
// SLOTS: one wave per (sorted slot, U x 64 x VEC columns) instead, for a gradient whose other rows are
// zeros already (beta = 0: the sort's launches write them, see Fill) or stay as they are (beta = 1).  Only a
// run's first slot has work.  At most T rows are then written twice, but the zeros go at a fill's rate and under
// the sort.
template <typename TY, typename TW, int U, bool SLOTS>
__global__ void __launch_bounds__(64 * WAVES_PER_BLOCK, 4)
    embedding_bwd_kernel(const int* __restrict__ keys, const int* __restrict__ vals,
                         const int* __restrict__ row_start, const TY* __restrict__ dY, TW* dW,
                         int64_t T, int64_t V, int64_t H, int64_t lddy, int64_t lddw,
                         int64_t padding_idx, int units_per_row, int long_blocks, int long_at, int rows_at, int scale_by_freq,
                         int beta, int pieces_per_row) {
  constexpr int VEC = 16 / (int)sizeof(TW);
  constexpr int LV = VEC / 4;                                 // columns of a lane in a long run's wave
  constexpr int LONG_B = LV * (int)sizeof(TY) <= 4 ? 64 : 32; // its rows in flight: a chunk, or 64 registers
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // (units_per_row and the block numbers lie side by side and come with one load, not with a second one here)
  const int block = (int)block_number();   // (less than 2^31)
  if ((unsigned)(block - long_at) < (unsigned)long_blocks) {
    const int64_t unit = (int64_t)(block - long_at) * WAVES_PER_BLOCK + wave;
    const int64_t chunk = unit / pieces_per_row * 64;
    const int64_t col0 = (unit % pieces_per_row * 64 + lane) * LV;
    const int64_t j = chunk + lane;
    const int key = j < T ? keys[j] : -1;
    const bool starts = j < T && key < V && key != padding_idx && (j == 0 || keys[j - 1] != key) &&
                        j + EMB_LONG_RUN < T && keys[j + EMB_LONG_RUN] == key;
    for (uint64_t todo = __ballot(starts); todo != 0; todo &= todo - 1) {
      const int l = __builtin_ctzll(todo);
      const int row = __builtin_amdgcn_readlane(key, l);
      const int64_t first = chunk + l;
      int pos, n;
      float inv = 1.0f;
      if (scale_by_freq) {
        int64_t e = first;
        do {
          n = run_in_chunk(keys, vals, e, T, row, lane, pos);
          e += n;
        } while (n == 64);
        inv = 1.0f / (float)(e - first);
      }
      float acc[1][LV];
#pragma unroll
      for (int q = 0; q < LV; ++q) acc[0][q] = 0.f;
      n = run_in_chunk(keys, vals, first, T, row, lane, pos);
      for (int64_t at = first; n > 0; at += 64) {
        int next_pos = 0;   // looked up while this chunk's rows are added
        const int next_n = n == 64 ? run_in_chunk(keys, vals, at + 64, T, row, lane, next_pos) : 0;
        add_rows<TY, LV, 1, LONG_B>(acc, n, pos, dY, lddy, col0, H, scale_by_freq != 0, inv);
        n = next_n;
        pos = next_pos;
      }
      if (col0 < H) store_part<TW, LV>(acc[0], dW + row * lddw + col0, beta);
    }
    return;
  }
  // (the wave's number stays a vector here: row_start read through the scalar cache costs 7 %)
  // (a 64-bit division would be half of what a wave does for a row without tokens.  4 tokens, 146388 x 2240
  // bf16, beta: 55 us; 61 with the scalar unit's 64-bit quotient of the workgroup's first unit and a loop over its
  // other units)
  const int64_t unit0 = (int64_t)(block - rows_at) * WAVES_PER_BLOCK;
  int64_t row = unit0 + (int)(threadIdx.x >> 6);
  int rest = 0;
  if (units_per_row != 1) {   // (rows of up to 1024 fp32 or 2048 16-bit elements need no division)
    const int64_t unit = row;
    if (unit0 <= 0x7ffffff0)
      row = (uint32_t)unit / (uint32_t)units_per_row;
    else
      row = unit / units_per_row;
    rest = (int)(unit - row * units_per_row);
  }
  const int64_t col0 = ((int64_t)rest * (U * 64) + lane) * VEC;
  float acc[U][VEC];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[u][q] = 0.f;
  int s;
  if constexpr (SLOTS) {
    const int64_t slot = row;   // (fewer than 2^31)
    if (slot >= T) return;
    const int key = keys[slot], before = slot > 0 ? keys[slot - 1] : -1;
    if (key == before || key >= V || key == padding_idx) return;
    s = (int)slot;
    row = key;
  } else {
    if (row >= V) return;
    s = row_start[row];
  }
  if (SLOTS || (s >= 0 && row != padding_idx)) {
    int pos, n = 1;
    if (s + 1 >= T || keys[s + 1] != (int)row)   // most rows of a text have one token
      pos = vals[s];
    else
      n = run_in_chunk(keys, vals, s, T, (int)row, lane, pos);
    if (n > EMB_LONG_RUN) return;   // another wave's
    const float inv = scale_by_freq ? 1.0f / (float)n : 1.0f;
    constexpr int B = U * VEC * (int)sizeof(TY) > 64 ? 2 : 4;   // (at most 64 registers of a lane)
    add_rows<TY, VEC, U, B>(acc, n, pos, dY, lddy, col0, H, scale_by_freq != 0, inv);
  } else if (beta != 0) {
    return;  // nothing to add to this row
  }
  store_rows<TW, VEC, U>(acc, dW + row * lddw + col0, col0, H, beta);
}

// ---- max_norm ------------------------------------------------------------------
// One wave per row of the table; rows no token names are left alone.
// norm = (sum |w|^p)^(1/p) in fp32; rows with norm > max_norm are scaled by
// max_norm / (norm + 1e-7), as torch.embedding_renorm_ does.
template <typename TW>
__global__ void __launch_bounds__(64 * WAVES_PER_BLOCK)
    embedding_renorm_kernel(const int* __restrict__ row_start, TW* W, int64_t V, int64_t H,
                            int64_t ldw, float max_norm, float norm_type) {
  const int lane = threadIdx.x & 63;
  const int64_t row = block_number() * WAVES_PER_BLOCK + (threadIdx.x >> 6);
  if (row >= V) return;
  if (row_start[row] < 0) return;
  constexpr int N = Vec<TW>::N;
  TW* w = W + row * ldw;
  float sum = 0.f;
  for (int64_t c = (int64_t)lane * N; c < H; c += 64 * N) {
    float x[N];
    Vec<TW>::load_cached(w + c, x);
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const float a = fabsf(x[e]);
      if (norm_type == 1.0f)
        sum += a;
      else if (norm_type == 2.0f)
        sum = fmaf(a, a, sum);
      else
        sum += powf(a, norm_type);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  float norm;
  if (norm_type == 1.0f)
    norm = sum;
  else if (norm_type == 2.0f)
    norm = sqrtf(sum);
  else
    norm = powf(sum, 1.0f / norm_type);
  if (!(norm > max_norm)) return;
  const float scale = max_norm / (norm + 1e-7f);
  for (int64_t c = (int64_t)lane * N; c < H; c += 64 * N) {
    float x[N];
    Vec<TW>::load_cached(w + c, x);
#pragma unroll
    for (int e = 0; e < N; ++e) x[e] *= scale;
    Vec<TW>::store_cached(w + c, x);   // the lookup reads the row next
  }
}

// ---- workspace ---------------------------------------------------------------
constexpr size_t ALIGN = 256;
inline size_t round_up(size_t n) { return (n + ALIGN - 1) / ALIGN * ALIGN; }

struct Workspace {
  int *keys_a, *keys_b, *vals_a, *vals_b, *row_start, *status, *hist;
};

int bits_for(int64_t V) {  // keys run over [0, V]
  int b = 1;
  while ((1LL << b) <= V) ++b;
  return b;
}

// The passes of the sort: the key's bits in equal parts of at most SORT_MAX_BITS, and one
// digit-major count array [2^bits][segments] per pass.
SortPlan plan_sort(int64_t T, int64_t V) {
  SortPlan pl;
  const int total = bits_for(V);
  pl.passes = (total + SORT_MAX_BITS - 1) / SORT_MAX_BITS;
  pl.groups = T <= SORT_SHORT_BATCH ? 2 : 8;
  pl.fused_scan = T <= SORT_FUSED_BATCH;
  const int64_t per_block = 64 * pl.groups * SORT_WAVES;
  pl.nblk = (T + per_block - 1) / per_block;
  int shift = 0;
  size_t ofs = 0;
  for (int p = 0; p < SORT_MAX_PASSES; ++p) {
    pl.bits[p] = p < pl.passes ? total / pl.passes + (p < total % pl.passes ? 1 : 0) : 0;
    pl.shift[p] = shift;
    pl.hist_ofs[p] = ofs;
    shift += pl.bits[p];
    if (p < pl.passes) ofs += ((size_t)1 << pl.bits[p]) * (size_t)pl.nblk;
  }
  pl.hist_ints = ofs;
  return pl;
}

inline bool carve(void* ws, size_t ws_bytes, int64_t T, int64_t V, Workspace* out) {
  char* p = (char*)ws;
  const size_t tok = round_up((size_t)T * sizeof(int));
  out->keys_a = (int*)p; p += tok;
  out->keys_b = (int*)p; p += tok;
  out->vals_a = (int*)p; p += tok;
  out->vals_b = (int*)p; p += tok;
  out->row_start = (int*)p; p += round_up((size_t)V * sizeof(int));
  out->status = (int*)p; p += ALIGN;
  out->hist = (int*)p; p += round_up(plan_sort(T, V).hist_ints * sizeof(int));
  return (size_t)(p - (char*)ws) <= ws_bytes;
}

// Fills ws with the sorted (key, position) pairs and row_start; on return
// *keys and *vals point at the sorted arrays.
// With `zeros`, the launches also clear that many bytes there, about an equal share each, and row_start is left alone.
int sort_token_positions(const int64_t* ids, int64_t T, int64_t V, const Workspace& w,
                         const int** keys, const int** vals, hipStream_t stream, bool want_row_start = true,
                         void* zeros = nullptr, size_t zero_bytes = 0) {
  const SortPlan pl = plan_sort(T, V);
  if (pl.nblk >= (1LL << 31) ||
      pl.hist_ints >= ((size_t)1 << 40)) {
    set_error("embedding: too many tokens to sort (%lld)", (long long)T);
    return AXN_ELIMIT;
  }
  const dim3 block(64 * SORT_WAVES);
  const int64_t seg_blocks = pl.nblk;
  // (at least enough workgroups to fill row_start at a good rate when the batch is short)
  int64_t fill_blocks = (V + 4 * 256 - 1) / (4 * 256);
  if (fill_blocks > 1024) fill_blocks = 1024;
  const int64_t prep_blocks = seg_blocks > fill_blocks ? seg_blocks : (fill_blocks > 0 ? fill_blocks : 1);
  int* const row_start = want_row_start ? w.row_start : nullptr;
  // Shares end on whole waves' stores, 1 KB from a 128-byte line: stores across lines cost a third of the rate (482 MB
  // of 103213 x 1168 fp32 for 26 tokens 112 us, on lines 77).
  const int64_t vectors = (int64_t)(zero_bytes / 16), shares = 1 + (T > 0 ? pl.passes : 0);
  const int64_t ahead = (int64_t)(((uintptr_t)0 - (uintptr_t)zeros) % 128 / 16);   // to the first line
  auto end_of = [&](int64_t share) {
    const int64_t even = vectors / shares * (share + 1) - ahead;
    return share + 1 == shares ? vectors : even < 64 ? 0 : even / 64 * 64 + ahead;
  };
  auto fill_of = [&](int64_t share, int64_t sort_blocks) {
    const int64_t first = share == 0 ? 0 : end_of(share - 1), end = end_of(share);
    return Fill{(u32x4*)zeros + first, end - first, sort_blocks};
  };
  auto blocks_with = [](const Fill& fill) {
    return (unsigned)(fill.sort_blocks + (fill.count + FILL_THREADS - 1) / FILL_THREADS);
  };
  int* hist_rest = w.hist + pl.hist_ofs[1];
  const int64_t hist_rest_ints = pl.passes > 1 ? (int64_t)(pl.hist_ints - pl.hist_ofs[1]) : 0;
  {
    const Fill fill = fill_of(0, prep_blocks);
    void (*prepare)(const int64_t*, int*, int*, int*, int*, int*, int*, int64_t, int64_t, int64_t, int64_t, int,
                    bool, Fill) =
        pl.groups == 2 ? embedding_sort_prepare_kernel<2> : embedding_sort_prepare_kernel<8>;
    hipLaunchKernelGGL(prepare, dim3(blocks_with(fill)), block, vectors > 0 ? SORT_FILL_LDS - SORT_PREPARE_LDS : 0,
                       stream, ids, w.keys_a, w.vals_a, row_start, w.status, w.hist, hist_rest, hist_rest_ints, T, V,
                       pl.nblk, pl.bits[0], pl.fused_scan, fill);
  }
  AXN_HIP_TRY(hipGetLastError());
  const int *kin = w.keys_a, *vin = w.vals_a;
  int *kout = w.keys_b, *vout = w.vals_b;
  if (T > 0) {
    for (int p = 0; p < pl.passes; ++p) {
      int* hist = w.hist + pl.hist_ofs[p];
      const int64_t n = ((int64_t)1 << pl.bits[p]) * pl.nblk;
      if (!pl.fused_scan) {
        hipLaunchKernelGGL(embedding_sort_scan_kernel, dim3(1), dim3(1024), 0, stream, hist, n);
        AXN_HIP_TRY(hipGetLastError());
      }
      const bool more = p + 1 < pl.passes;
      void (*scatter)(const int*, const int*, int*, int*, const int*, int*, int*, int*, int64_t, int64_t,
                      int64_t, int, int, int, int, Fill) =
          pl.fused_scan ? (pl.groups == 2 ? embedding_sort_scatter_kernel<2, false>
                                          : embedding_sort_scatter_kernel<8, false>)
                        : embedding_sort_scatter_kernel<8, true>;
      const Fill fill = fill_of(p + 1, seg_blocks);
      hipLaunchKernelGGL(scatter, dim3(blocks_with(fill)), block,
                         vectors > 0 ? SORT_FILL_LDS - SORT_SCATTER_LDS : 0, stream, kin, vin, kout, vout,
                         (const int*)hist, more ? w.hist + pl.hist_ofs[p + 1] : nullptr, row_start,
                         w.status, T, V, pl.nblk, pl.shift[p], pl.bits[p], more ? pl.shift[p + 1] : 0,
                         more ? pl.bits[p + 1] : 0, fill);
      AXN_HIP_TRY(hipGetLastError());
      const int* tk = kin; kin = kout; kout = (int*)tk;
      const int* tv = vin; vin = vout; vout = (int*)tv;
    }
  }
  *keys = kin;
  *vals = vin;
  return AXN_OK;
}

}  // namespace

size_t embedding_workspace_bytes(int64_t T, int64_t V) {
  if (T < 0 || V <= 0) return 0;
  return 4 * round_up((size_t)T * sizeof(int)) + round_up((size_t)V * sizeof(int)) + ALIGN +
         round_up(plan_sort(T, V).hist_ints * sizeof(int));
}

int launch_embedding_fwd(const int64_t* ids, const void* W, void* out, int elem_bytes, int64_t T,
                         int64_t V, int64_t H, int64_t ldw, int64_t ldo, int* status,
                         hipStream_t stream) {
  const int per_piece = 16 / elem_bytes;
  const int64_t pieces = H / per_piece;
  const int upr = (int)((pieces + 63) / 64);
  const int64_t blocks = (T * upr + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
  if (blocks == 0) return AXN_OK;
  if (blocks >= (1LL << 31) - kMostBlocks) {
    set_error("embedding_fwd: too many tokens x columns (%lld blocks)", (long long)blocks);
    return AXN_ELIMIT;
  }
  hipLaunchKernelGGL(embedding_fwd_kernel, grid_of(blocks), dim3(64 * WAVES_PER_BLOCK), 0,
                     stream, ids, (const u32x4*)W, (u32x4*)out, T, V, pieces, ldw / per_piece,
                     ldo / per_piece, upr, status);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

int launch_embedding_bwd(const int64_t* ids, const void* dY, void* dW, int dy_dtype, int dw_dtype,
                         int64_t T, int64_t V, int64_t H, int64_t lddy, int64_t lddw,
                         int64_t padding_idx, int scale_by_freq, int beta, void* ws,
                         size_t ws_bytes, hipStream_t stream) {
  Workspace w;
  if (ws == nullptr || !carve(ws, ws_bytes, T, V, &w)) {
    set_error("embedding_bwd: workspace too small (%zu bytes given, %zu needed)", ws_bytes,
              embedding_workspace_bytes(T, V));
    return AXN_EINVAL;
  }
  // pieces of 64 lanes x one 16-byte dW vector per row; up to 4 of them per wave
  const int vec = dw_dtype == AXN_F32 ? 4 : 8;
  const int64_t pieces = (H / vec + 63) / 64;
  const int U = pieces >= 4 ? 4 : pieces >= 2 ? 2 : 1;
  const int upr = (int)((pieces + U - 1) / U);
  // waves for rows named by many tokens: one per 64 sorted slots and piece
  const int64_t long_pieces = (H / (vec / 4) + 63) / 64;
  const int64_t long_blocks =
      T > EMB_LONG_RUN ? ((T + 63) / 64 * long_pieces + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK : 0;
  // (a launch has fewer than 2^32 threads: one for each 16 bytes it clears, and those that sort)
  const int64_t clearing = 1 + (T > 0 ? plan_sort(T, V).passes : 0);
  const bool clears = lddw == H && V * (H / vec) / clearing < 0xd0000000LL;
  const bool slots = T <= V / EMB_SLOT_ROWS && (beta != 0 || clears);
  const int64_t row_blocks = ((slots ? T : V) * upr + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
  const int64_t blocks = row_blocks + long_blocks;
  const bool rows_first = row_blocks <= EMB_RESIDENT * 3 / 4 && blocks > EMB_RESIDENT;
  const size_t zero_bytes = slots && beta == 0 ? (size_t)V * (size_t)H * (dw_dtype == AXN_F32 ? 4 : 2) : 0;
  if (blocks >= (1LL << 31) - kMostBlocks) {
    set_error("embedding_bwd: too many rows x columns (%lld blocks)", (long long)blocks);
    return AXN_ELIMIT;
  }
  const int *keys = nullptr, *vals = nullptr;
  int rc = sort_token_positions(ids, T, V, w, &keys, &vals, stream, !slots, dW, zero_bytes);
  if (rc || blocks == 0) return rc;
  const dim3 grid = grid_of(blocks), block(64 * WAVES_PER_BLOCK);
#define AXN_EMB_BWD_US(TY, TW, UU, SLOTS)                                                       \
  hipLaunchKernelGGL((embedding_bwd_kernel<TY, TW, UU, SLOTS>), grid, block, EMB_BWD_LDS, stream, keys, vals,    \
                     w.row_start, (const TY*)dY, (TW*)dW, T, V, H, lddy, lddw, padding_idx, upr, \
                     (int)long_blocks, rows_first ? (int)row_blocks : 0, rows_first ? 0 : (int)long_blocks, \
                     scale_by_freq, beta, (int)long_pieces)
#define AXN_EMB_BWD_U(TY, TW, UU)           \
  do {                                      \
    if (slots)                              \
      AXN_EMB_BWD_US(TY, TW, UU, true);     \
    else                                    \
      AXN_EMB_BWD_US(TY, TW, UU, false);    \
  } while (0)
#define AXN_EMB_BWD(TY, TW)                 \
  do {                                      \
    if (U == 4)                             \
      AXN_EMB_BWD_U(TY, TW, 4);             \
    else if (U == 2)                        \
      AXN_EMB_BWD_U(TY, TW, 2);             \
    else                                    \
      AXN_EMB_BWD_U(TY, TW, 1);             \
  } while (0)
  if (dy_dtype == AXN_F32 && dw_dtype == AXN_F32)
    AXN_EMB_BWD(float, float);
  else if (dy_dtype == AXN_F32)
    AXN_EMB_BWD(float, uint16_t);
  else if (dw_dtype == AXN_F32)
    AXN_EMB_BWD(uint16_t, float);
  else
    AXN_EMB_BWD(uint16_t, uint16_t);
#undef AXN_EMB_BWD_US
#undef AXN_EMB_BWD_U
#undef AXN_EMB_BWD
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

int launch_embedding_renorm(const int64_t* ids, void* W, int dtype, int64_t T, int64_t V,
                            int64_t H, int64_t ldw, float max_norm, float norm_type, void* ws,
                            size_t ws_bytes, hipStream_t stream) {
  Workspace w;
  if (ws == nullptr || !carve(ws, ws_bytes, T, V, &w)) {
    set_error("embedding_renorm: workspace too small (%zu bytes given, %zu needed)", ws_bytes,
              embedding_workspace_bytes(T, V));
    return AXN_EINVAL;
  }
  const int *keys = nullptr, *vals = nullptr;
  int rc = sort_token_positions(ids, T, V, w, &keys, &vals, stream);
  if (rc) return rc;
  const dim3 grid = grid_of((V + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK), block(64 * WAVES_PER_BLOCK);
  if (dtype == AXN_F32)
    hipLaunchKernelGGL(embedding_renorm_kernel<float>, grid, block, 0, stream, w.row_start,
                       (float*)W, V, H, ldw, max_norm, norm_type);
  else if (dtype == AXN_F16)
    hipLaunchKernelGGL(embedding_renorm_kernel<_Float16>, grid, block, 0, stream, w.row_start,
                       (_Float16*)W, V, H, ldw, max_norm, norm_type);
  else
    hipLaunchKernelGGL(embedding_renorm_kernel<uint16_t>, grid, block, 0, stream, w.row_start,
                       (uint16_t*)W, V, H, ldw, max_norm, norm_type);
  AXN_HIP_TRY(hipGetLastError());
  return AXN_OK;
}

}  // namespace axn
