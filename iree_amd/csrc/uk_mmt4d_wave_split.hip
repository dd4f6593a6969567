// mmt4d of few tiles: K split over the eight waves of a workgroup.
//
// The macro-tile kernels give a workgroup 128 x 128 of the result and more, and
// K to all of its waves together. A problem of a few such tiles (a layer on some
// dozens of rows, a product of a few hundred rows and columns) then leaves most
// compute units idle, or K is split over workgroups, whose partial sums go
// through memory and cost a second launch (4 to 5 us).
//
// Here a workgroup owns 16 x 16 to 64 x 64 of the result and each of its waves
// every eighth pair of 64-byte steps of K, fetched straight into the registers
// that feed the matrix cores (packed tiles are in operand order) several steps
// ahead; no wave waits for another before the sums, which meet in LDS and are
// added in wave order: one launch, no scratch memory, the same bits whatever the
// tile.
//
// What bounds it: 3.5 us for a launch of one step; then what one compute unit
// takes in while the operands come from beyond its L2: packed ones 8 to 10 us per MB
// by the fit below (100 to 125 GB/s; f16 512x512 on 256 workgroups 100 from K = 1024 to
// 2048, 70 from there to 4096), row-major ones 13 to 17 (60 to 80 GB/s). That size
// decides the tile. Before and after, among other calls, operands in the last-level
// cache: bf16 128x608x1184 10.7 -> 4.0 us, 64x64x768 7.9 -> 3.5, f16 2208x160x1984
// 14.7 -> 8.0, 1024^3 10.8 -> 7.2; a linear layer of fp8 42x2602x5760 12.6 -> 7.1, f16
// 32x3117x1152 10.7 -> 5.0, 84 rows of bf16 1024x4288 13.0 -> 8.2; f32 416x971x1071
// with its packing 31.4 -> 22.8.
// Direct-to-LDS loads of both operands gave the same times (the load path is
// not what is full), more steps in flight as well.
#include "uk_mmt4d_wave_split.h"

#include <cmath>
#include <type_traits>

#include "uk_fp8.h"
#include "uk_mfma_cfg.h"

namespace uk {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr uint32_t kNowhere = 0x80000000u;   // past the end of every descriptor: the load gives zeros

// The product of one 16-byte piece per lane and operand (row lane % 16, bytes
// 16 (lane / 16) .. + 16 of 64 bytes of K) and the sum of the 16 x 16 results.
struct F8 {};
template <typename T> struct BlockProduct;
template <> struct BlockProduct<_Float16> {
  typedef floatx4 acc_t;
  __device__ static acc_t run(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
};
template <> struct BlockProduct<__bf16> {
  typedef floatx4 acc_t;
  __device__ static acc_t run(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct BlockProduct<int8_t> {
  typedef intx4 acc_t;
  __device__ static acc_t run(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(int4v, a), __builtin_bit_cast(int4v, b), c, 0, 0, 0);
  }
};
// (each instruction takes element e of the piece: both operands pair the same way)
template <> struct BlockProduct<float> {
  typedef floatx4 acc_t;
  __device__ static acc_t run(u32x4 a, u32x4 b, acc_t c) {
    const floatx4 x = __builtin_bit_cast(floatx4, a), y = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  }
};
template <> struct BlockProduct<F8> {
  typedef floatx4 acc_t;
  __device__ static acc_t run(u32x4 a, u32x4 b, acc_t c) {
    typedef long longx2 __attribute__((ext_vector_type(2)));
    const longx2 x = __builtin_bit_cast(longx2, a), y = __builtin_bit_cast(longx2, b);
    c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[0], y[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[1], y[1], c, 0, 0, 0);
  }
};

template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// MB x NB blocks of 16 x 16 results per workgroup; D steps of 64 bytes of K in
// flight per wave.
// kRowMajor: the left-hand side is a row-major matrix. (The 16 bytes of four
// adjacent lanes are then in four rows, which the load path takes as four
// requests: such a byte took 2.5 times as long as one of packed tiles. So its
// blocks come in with direct-to-LDS loads, in which the lanes of a quad fetch the
// 64 bytes of one row, and are read from there in operand order. A block lies
// in LDS row by row, the pieces of row r rotated by r / 4: the reads of 16 rows
// touch every bank alike.)
// kTiles: the result goes to a.tiles as well. (For itself: read from the arguments behind
// the last step, whether it does cost every call 0.1 us: bf16 linear layers of 202 rows
// 2624 -> 1401 7.88 us so and 7.78 compiled for itself, 96 rows 1664 -> 3978 6.76 and 6.65.)
template <typename T, typename out_t, int MB, int NB, int D, bool kRowMajor, bool kTiles>
__device__ __forceinline__ void mmt4d_wave_split_body(const WaveSplitArgs& a) {
  typedef typename BlockProduct<T>::acc_t acc_t;
  constexpr int F = MB * NB;
  static_assert(D % 2 == 0, "steps come in pairs");
  constexpr int kRingBytes = kRowMajor ? D * MB * 1024 : 0;     // of a wave
  constexpr int kSharedBytes = kWaves * (kRingBytes > F * 1024 ? kRingBytes : F * 1024);
  __shared__ __attribute__((aligned(1024))) char shared[kSharedBytes];
  acc_t (*const sums)[F][64] = (acc_t (*)[F][64])shared;
  const int lane = threadIdx.x & 63, l16 = lane & 15, kc = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn, plane;
  {
    // (workgroup ids go round-robin over the 8 XCDs: XCD x takes the x-th
    // contiguous slice of the tiles, plane by plane, the row tiles of one column
    // tile together)
    const int total = (int)gridDim.x, per = total / 8, rem = total % 8;
    const int xcd = (int)blockIdx.x % 8, idx = (int)blockIdx.x / 8;
    const int logical = xcd * per + (xcd < rem ? xcd : rem) + idx, tiles = a.tiles_m * a.tiles_n;
    plane = logical / tiles;
    tn = (logical - plane * tiles) / a.tiles_m;
    tm = logical - plane * tiles - tn * a.tiles_m;
  }
  // ---- where this lane's pieces of the operands lie --------------------------
  const int first_row = tm * MB * 16 / 32, first_col = a.silu ? tn * NB / 4 * 2 : tn * NB / 2;   // (outer ones)
  const __amdgpu_buffer_rsrc_t lhs_src = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.lhs + plane * a.lhs_batch + first_row * a.lhs_outer), 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t rhs_src = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.rhs + plane * a.rhs_batch + first_col * a.rhs_outer), 0, 0x7FFFFFFF, 0x00020000);
  // row of a block and piece of a step that this lane fetches of the left-hand side
  const int lhs_r = kRowMajor ? lane >> 2 : l16, lhs_c = kRowMajor ? ((lane & 3) - (lane >> 4)) & 3 : kc;
  uint32_t lhs_at[MB], rhs_at[NB];
#pragma unroll
  for (int x = 0; x < MB; ++x) {
    const int row = (tm * MB + x) * 16 + lhs_r;
    lhs_at[x] = row < a.rows ? (uint32_t)((row >> 5) - first_row) * (uint32_t)a.lhs_outer + (row & 31) * a.lhs_row + lhs_c * a.lhs_chunk
                             : kNowhere;
  }
#pragma unroll
  for (int y = 0; y < NB; ++y) {
    // (SiLU form: even blocks are gate columns, of even outer columns, and the
    // odd block behind one the same columns of the odd outer column)
    const int block = tn * NB + y;
    const int col = a.silu ? block / 4 * 2 + block % 2 : block / 2, half = a.silu ? block / 2 % 2 : block % 2;
    rhs_at[y] = col < a.outer_cols ? (uint32_t)(col - first_col) * (uint32_t)a.rhs_outer + half * 256 + l16 * 16 + kc * 512
                                   : kNowhere;
  }
  const uint32_t lhs_step = 4 * a.lhs_chunk;
  // ---- the products ----------------------------------------------------------
  // Steps are dealt to the waves in pairs (128 bytes of K: whole lines of a
  // row-major left-hand side). What lies past the end of K is zeros on both sides.
  const int groups = (a.k_chunks + 4 * kWaves * D - 1) / (4 * kWaves * D);
  acc_t acc[MB][NB];
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y) acc[x][y] = acc_t{0, 0, 0, 0};
  constexpr int kA = kRowMajor ? 2 : D;       // blocks of the left-hand side: one step ahead of LDS, or as loaded
  u32x4 fa[kA][MB], fb[D][NB];
  char* const ring = shared + wave * kRingBytes;
  auto load = [&](int group, int d) {
    const int step = ((group * (D / 2) + d / 2) * kWaves + wave) * 2 + d % 2;
    const bool lhs_exists = step * 4 + lhs_c < a.k_chunks, rhs_exists = step * 4 + kc < a.k_chunks;
#pragma unroll
    for (int x = 0; x < MB; ++x) {
      const uint32_t at = lhs_exists ? lhs_at[x] : kNowhere;
      if constexpr (kRowMajor)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            lhs_src, (__attribute__((address_space(3))) void*)(ring + (d * MB + x) * 1024), 16, at, step * lhs_step, 0, 0);
      else
        fa[d % kA][x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(lhs_src, at, step * lhs_step, 0));
    }
    if constexpr (kRowMajor) __builtin_amdgcn_sched_barrier(0);     // (the order that `read` counts on)
#pragma unroll
    for (int y = 0; y < NB; ++y)
      fb[d][y] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rhs_src, rhs_exists ? rhs_at[y] : kNowhere, step * 2048, 0));
    if constexpr (kRowMajor) __builtin_amdgcn_sched_barrier(0);
  };
  // (row-major) the blocks of step d from LDS; `behind`: loads issued after theirs
  auto read = [&](int d, auto behind) {
    if constexpr (kRowMajor) {
      wait_loads<decltype(behind)::value>();
#pragma unroll
      for (int x = 0; x < MB; ++x)
        fa[d % 2][x] = *(const u32x4*)(ring + (d * MB + x) * 1024 + l16 * 64 + ((kc + (l16 >> 2)) & 3) * 16);
    }
  };
  auto multiply = [&](int d) {
#pragma unroll
    for (int x = 0; x < MB; ++x)
#pragma unroll
      for (int y = 0; y < NB; ++y) acc[x][y] = BlockProduct<T>::run(fb[d][y], fa[d % kA][x], acc[x][y]);
  };
  typedef std::integral_constant<int, NB + (D - 1) * (MB + NB)> AllButOne;
  typedef std::integral_constant<int, NB + (D - 2) * (MB + NB)> AllButTwo;
#pragma unroll
  for (int d = 0; d < D; ++d) load(0, d);
  __builtin_amdgcn_sched_barrier(0);
  read(0, AllButOne());
#pragma unroll 1
  for (int g = 1; g < groups; ++g) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      // (the next step's blocks leave LDS while this one's are multiplied)
      __builtin_amdgcn_sched_barrier(0);
      read((d + 1) % D, AllButTwo());
      multiply(d);
      __builtin_amdgcn_sched_barrier(0);
      load(g, d);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (d + 1 < D) read(d + 1, std::integral_constant<int, 0>());
    multiply(d);
  }
  if constexpr (kRowMajor) __syncthreads();     // (the sums take the place of the rings)
  // ---- the waves' sums, in wave order ----------------------------------------
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y) sums[wave][x * NB + y][lane] = acc[x][y];
  __syncthreads();
  // Element e of lane l: row l % 16 of the block, column 4 (l / 16) + e.
  if (std::is_same<T, F8>::value && NB % 2 == 0 && a.silu) {
    if constexpr (NB % 2 == 0 && std::is_same<T, F8>::value) {
#pragma unroll
      for (int f0 = 0; f0 < F / 2; f0 += kWaves) {
        const int f = f0 + wave;
        if (f >= F / 2) break;
        const int x = f / (NB / 2), y = f % (NB / 2) * 2;
        const int block = tm * MB + x, pair = (tn * NB + y) / 2;
        if (block * 16 >= a.rows || pair / 2 * 2 >= a.outer_cols) continue;
        acc_t gate = {0, 0, 0, 0}, up = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          gate += sums[w][x * NB + y][lane];
          up += sums[w][x * NB + y + 1][lane];
        }
        float h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = silu_mul(gate[e] * a.gate_scale, up[e] * a.up_scale) * a.inv_out_scale;
        *(uint32_t*)(a.out + (block / 2) * a.out_outer + (int64_t)pair * 512 + (block % 2 * 16 + l16) * 16 + kc * 4) =
            pack4_e4m3(h[0], h[1], h[2], h[3]);
      }
    }
    return;
  }
  typedef out_t out4_t __attribute__((ext_vector_type(4), aligned(sizeof(out_t))));
#pragma unroll
  for (int f0 = 0; f0 < F; f0 += kWaves) {
    const int f = f0 + wave;
    if (f >= F) break;
    const int x = f / NB, y = f % NB;
    const int row = (tm * MB + x) * 16 + l16, col = (tn * NB + y) * 16 + kc * 4;
    const bool exists = row < a.out_rows && col < a.out_cols;
    if (!exists && !(kTiles && row < a.rows && col < a.outer_cols * 32)) continue;
    out_t* const dst = (out_t*)(a.out + plane * a.out_batch) + (row >> 5) * a.out_outer + (row & 31) * a.out_row +
                       (col >> 5) * a.out_tile + (col & 31) * a.out_col;
    const bool whole = a.out_col == 1 && col + 4 <= a.out_cols;
    acc_t sum = {0, 0, 0, 0};
    if (a.accumulate && (!kTiles || exists)) {
      if (whole) {
        const out4_t old = *(const out4_t*)dst;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = old[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < a.out_cols) sum[e] = dst[e * a.out_col];
      }
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w) sum += sums[w][f][lane];
    out4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (std::is_same<out_t, int32_t>::value) v[e] = sum[e];
      else v[e] = (out_t)(sum[e] * a.out_scale);
    }
    if constexpr (kTiles)
      *(out4_t*)((out_t*)a.tiles + (row >> 5) * a.tiles_outer + (int64_t)(col >> 5) * 1024 + (row & 31) * 32 + (col & 31)) = v;
    if (kTiles && !exists) continue;
    if (whole) {
      *(out4_t*)dst = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < a.out_cols) dst[e * a.out_col] = v[e];
    }
  }
}

// (the body is a function of its own: the host pass has no buffer descriptors)
template <typename T, typename out_t, int MB, int NB, int D, int kOcc, bool kRowMajor, bool kTiles>
__global__ __launch_bounds__(kWaves * 64, kOcc) void mmt4d_wave_split_kernel(WaveSplitArgs a) {
  mmt4d_wave_split_body<T, out_t, MB, NB, D, kRowMajor, kTiles>(a);
}

// Estimated time in microseconds on a tile of mb x nb blocks. Workgroups run in
// rounds of one per compute unit (several of a compute unit's are resident, which
// changes little): `first` for the first round of short ones, `round` for each
// further one, and beyond what the launch hides (`hidden`) the intake of a compute
// unit, in us per MB: rhs, lhs (packed) or rows (row-major), or all operands from
// memory, `memory`, whichever takes longer. f32 adds its matrix instructions.
// `store` is per MB of result. Fitted to 5000 problems (1 to 800 rows, 64 to 14336
// columns, K 64 to 14336, 7 forms and types): on 3000 others 7 to 8 % off on
// average, and the tile it picks is 0.7 % from the best of the five.
struct Tile {
  int mb, nb;
  float first, round, rhs, lhs, rows, hidden, memory, f32, store;
};
constexpr int kTiles = 5;
constexpr Tile kTile[kTiles] = {{1, 1, 3.53f, 0.83f, 8.1f, 8.5f, 12.7f, 0.84f, 0.215f, 0.130f, 0.27f},
                                {1, 2, 3.73f, 1.08f, 8.4f, 9.6f, 13.3f, 0.88f, 0.238f, 0.125f, 0.14f},
                                {2, 2, 3.72f, 1.01f, 9.2f, 9.2f, 15.2f, 0.81f, 0.260f, 0.135f, 0.25f},
                                {2, 4, 4.45f, 2.23f, 10.0f, 10.1f, 17.4f, 1.27f, 0.280f, 0.155f, 0.35f},
                                {4, 4, 4.36f, 2.59f, 10.3f, 10.2f, 16.6f, 0.78f, 0.290f, 0.175f, 0.36f}};

double estimate_us(const WaveSplitArgs& a, bool f32, int out_bytes, const Tile& t, int cus) {
  // (32 bits where they do: a call is as short as 3 us, and 64-bit divisions are slow)
  const uint32_t groups_m = (uint32_t)(a.rows + t.mb * 16 - 1) / (uint32_t)(t.mb * 16);
  const uint32_t groups_n = (uint32_t)(a.outer_cols * 2 + t.nb - 1) / (uint32_t)t.nb;
  const double groups = (double)groups_m * groups_n * a.batch;
  const double rounds = groups <= cus ? 1.0 : std::ceil(groups / cus);
  const double kb = a.k_chunks / 64.0;                    // KB of K, and MB of 1000 rows or columns
  double intake = rounds * kb * 0.016 * (t.nb * t.rhs + t.mb * (a.lhs_chunk == 16 ? t.rows : t.lhs));
  if (f32) intake += rounds * kb * t.mb * t.nb * t.f32;
  const double all = ((double)a.rows + a.outer_cols * 32.0) * a.batch * a.k_chunks * 16e-6 * t.memory;
  if (intake < all) intake = all;
  const double us = t.first + t.round * (rounds - 1) + (intake > t.hidden ? intake - t.hidden : 0.0) +
                    t.store * 1e-6 * a.rows * a.outer_cols * 32 * a.batch * out_bytes;
  // (operands that outgrow an L2 come from beyond it more than once; long ones are
  // under-estimated)
  return f32 || us < 8.0 ? us : us * (1.0 + 0.03 * (us - 8.0));
}

// Up to 64 rows of fp8 in packed tiles (a decode step of the MLP block) with 1.5 KB of K and
// weights of 16 MB and more: the intake of a compute unit and the time at memory's rate
// (both operands, `memory` us per MB) add up. Fitted to the geometric mean of the times with
// weights beyond the last-level cache and with three layers in turn, 7200 problems (1 to 64 rows, 512 to
// 28672 columns, K 768 to 14336), 6 to 9 % off on average. It decides the tile and, against
// macro tiles that keep K whole (few_rows_us), the kernel: the SiLU form 1.14 times as fast as with
// the estimate above on 75 other problems, with weights in the last-level cache and beyond it
// alike (32 rows x 2 x 8192 x 2048 9.3 -> 7.8 us with three layers in turn, 11.6 -> 8.7 beyond
// it); the plain form, 29 problems, as fast as before. 2 x 14336 x 4096 stays on macro tiles.
// Below these sizes and for the other types and forms it gave nothing, and costs a call of
// 4 us a tenth of them.
// (Weights past the caches by non-temporal loads, one workgroup having all rows: 5 to 8 %
// faster on 27 problems of 38 to 128 MB whose weights come from memory, 3 to 15 % slower where
// three layers stay in the last-level cache. The call cannot know, so not.)
struct RowsTile { float first, round, rhs, lhs, memory, store, silu; };
constexpr RowsTile kRowsTile[kTiles] = {
    {3.52f, 0.23f, 6.07f, 9.48f, 0.085f, 0.15f, 0.0f},  {3.34f, 0.19f, 7.77f, 9.98f, 0.090f, 0.31f, 0.17f},
    {3.36f, 0.30f, 6.16f, 11.7f, 0.086f, 0.16f, 0.06f}, {3.78f, 1.14f, 5.72f, 12.9f, 0.108f, 0.11f, -0.14f},
    {4.29f, 1.78f, 2.97f, 9.93f, 0.112f, 0.21f, 0.01f}};
double few_rows_estimate_us(const WaveSplitArgs& a, int out_bytes, int v, int cus) {
  const Tile& t = kTile[v];
  const RowsTile& f = kRowsTile[v];
  const uint32_t groups = (uint32_t)((a.rows + t.mb * 16 - 1) / (t.mb * 16)) * (uint32_t)((a.outer_cols * 2 + t.nb - 1) / t.nb);
  const double rounds = groups <= (uint32_t)cus ? 1.0 : (double)((groups + cus - 1) / cus);
  const double kb = a.k_chunks / 64.0, cols = a.outer_cols * 32.0;      // KB of K, and MB of 1000 rows or columns
  const double intake = rounds * kb * 0.016 * (t.nb * f.rhs + t.mb * f.lhs);
  const double memory = (a.rows + cols) * 1e-3 * kb * f.memory;
  return f.first + f.round * (rounds - 1) + intake + memory +
         f.store * 1e-6 * a.rows * (a.silu ? cols / 2 : cols) * out_bytes + (a.silu ? f.silu : 0.0f);
}

template <typename T, typename out_t, bool kRowMajor, bool kTiles>
int launch_tile(WaveSplitArgs a, int v, hipStream_t s) {
  void (*kernel)(WaveSplitArgs) = nullptr;
  switch (v) {
    case 0: kernel = mmt4d_wave_split_kernel<T, out_t, 1, 1, 8, 4, kRowMajor, kTiles>; break;
    case 1: kernel = mmt4d_wave_split_kernel<T, out_t, 1, 2, 6, 4, kRowMajor, kTiles>; break;
    case 2: kernel = mmt4d_wave_split_kernel<T, out_t, 2, 2, 4, 4, kRowMajor, kTiles>; break;
    case 3: kernel = mmt4d_wave_split_kernel<T, out_t, 2, 4, 4, 2, kRowMajor, kTiles>; break;
    default: kernel = mmt4d_wave_split_kernel<T, out_t, 4, 4, 2, 2, kRowMajor, kTiles>; break;
  }
  const Tile& t = kTile[v];
  a.tiles_m = (int)ceil_div((int64_t)a.rows, (int64_t)(t.mb * 16));
  a.tiles_n = (int)ceil_div((int64_t)a.outer_cols * 2, (int64_t)t.nb);
  const int64_t blocks = (int64_t)a.tiles_m * a.tiles_n * a.batch;
  if (blocks > 0x7FFFFFFF) return IREE_AMD_UK_STATUS_NOT_FOUND;
  note_macro_tile(t.mb * 16, t.nb * 16, 1);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kWaves * 64), 0, s, a);
  return check_hip(hipGetLastError(), "mmt4d_wave_split launch");
}

template <typename T, typename out_t>
int launch_type(const WaveSplitArgs& a, int v, hipStream_t s) {
  if (a.lhs_chunk == 16) return a.tiles ? IREE_AMD_UK_STATUS_NOT_FOUND : launch_tile<T, out_t, true, false>(a, v, s);
  return a.tiles ? launch_tile<T, out_t, false, true>(a, v, s) : launch_tile<T, out_t, false, false>(a, v, s);
}

}  // namespace

WaveSplitChoice choose_wave_split(const WaveSplitArgs& a, uint32_t type) {
  WaveSplitChoice best = {-1, 0.0, false, false, -1, 0.0};
  const bool f32 = type == IREE_AMD_UK_FLAG_MMT4D_TYPE_F32F32F32, f8 = type == IREE_AMD_UK_FLAG_MMT4D_TYPE_F8E4M3F8E4M3F32;
  // (unsigned 32-bit offsets within a workgroup's tile and along K: outer rows or columns
  // that run backwards are the other kernels')
  if ((a.silu && !f8) || a.lhs_outer < 0 || a.rhs_outer < 0 || a.lhs_outer > (1 << 28) || a.rhs_outer > (1 << 28) ||
      a.k_chunks < 1 || a.k_chunks > (1 << 18) ||
      a.rows < 1 || a.rows > (1 << 24) || a.outer_cols < 1 || a.outer_cols > (1 << 20))
    return best;
  const bool half_out = type == IREE_AMD_UK_FLAG_MMT4D_TYPE_F16F16F16 || type == IREE_AMD_UK_FLAG_MMT4D_TYPE_BF16BF16BF16;
  const int out_bytes = a.silu ? 1 : half_out ? 2 : 4;
  const int cus = device_cu_count();
  for (int v = 0; v < kTiles; ++v) {
    if (a.silu && kTile[v].nb == 1) continue;             // (gate and up columns side by side)
    const double us = estimate_us(a, f32, out_bytes, kTile[v], cus);
    if (best.tile < 0 || us < best.us) best = {v, us, false, false, v, us};
  }
  const int64_t weights = (int64_t)a.outer_cols * 512 * a.k_chunks;
  if (best.tile >= 0 && f8 && a.rows <= 64 && a.lhs_chunk != 16 && a.batch == 1 && a.k_chunks >= 96 && weights >= 16000000) {
    for (int v = 0; v < kTiles; ++v) {
      if (a.silu && kTile[v].nb == 1) continue;
      const double us = few_rows_estimate_us(a, out_bytes, v, cus);
      if (!best.few_rows || us < best.us) { best.tile = v; best.us = us; best.few_rows = true; }
    }
  }
  if (best.tile >= 0) {
    const Tile& t = kTile[best.tile];
    best.one_round = ceil_div((int64_t)a.rows, (int64_t)(t.mb * 16)) *
                         ceil_div((int64_t)a.outer_cols * 2, (int64_t)t.nb) * a.batch <= cus;
  }
  return best;
}

int launch_mmt4d_wave_split(const WaveSplitArgs& a, uint32_t type, int tile, hipStream_t s) {
  switch (type) {
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F16F16F32: return launch_type<_Float16, float>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_BF16BF16F32: return launch_type<__bf16, float>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F16F16F16: return launch_type<_Float16, _Float16>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_BF16BF16BF16: return launch_type<__bf16, __bf16>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_S8S8S32: return launch_type<int8_t, int32_t>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F8E4M3F8E4M3F32: return launch_type<F8, float>(a, tile, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F32F32F32: return launch_type<float, float>(a, tile, s);
    default: return IREE_AMD_UK_STATUS_NOT_FOUND;
  }
}

}  // namespace uk
