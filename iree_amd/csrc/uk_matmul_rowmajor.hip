// The whole data-tiled matmul (pack, pack, [pack C,] mmt4d, unpack) of a small
// problem as ONE launch, or two where K is split.
//
// Contract: include/iree_amd_uk.h, iree_amd_uk_matmul_data_tiled. The sequence
// it stands for is the reference's
// (compiler/src/iree/compiler/Codegen/Common/CPU/CPULowerToUKernels.cpp:339-480).
//
// What bounds such a call is not work but launches: a chain of 4 or 5 kernels
// that depend on each other costs about 5 us for each whatever it does. Here the
// first workgroups multiply straight from the row-major operands, the ones
// after them write the packed operands, which nothing in the launch waits for,
// and the matmul's epilogue stores both the tiles of the result and the matrix.
//
// Among other calls on one stream: f16 81x19x41 with C added 27.1 us as the chain,
// 7.4 here; i8 1024^3 21.0, 11.4.
//
// A step of K costs a workgroup 2.4 to 3.9 us: its 24 loads per thread, many of
// them of rows 64 bytes long, pass the compute unit's one load path. So a long
// K of few tiles is dealt to more workgroups, each with its own plane of partial
// sums, and a second launch adds the planes in order (2 us when it follows):
// bf16 64x29x3693 35.0 us whole, 8.7 in 8 slices.
//
// Multiplying workgroups: 4 waves on kRows x kRows of the result, 64 KiB of
// operands per K-step (128 KiB / kRows bytes of K), fetched for the next
// step while this one is multiplied: a wide step because a step costs a round
// trip to memory, and these problems have too few workgroups to hide it.
// An operand row of a step is kChunks chunks of 16 bytes of consecutive K in
// LDS, permuted within 16 by a hash of the row: fragment reads (16 consecutive
// rows, one chunk) and the stores of the right-hand side (rows 4 apart) hit 16
// different bank groups each. The right-hand side, whose rows run along N,
// is turned in registers: a thread loads 4 columns of the 16 / element-size
// rows of a chunk and stores 4 chunks.
//   kRows = 64: each wave a 32x32 quarter.
//   kRows = 32: each wave all of it for a quarter of K, summed in LDS in wave
//   order; four times as many workgroups and half as many steps.
#include <type_traits>

#include "uk_common.h"
#include "uk_mfma_cfg.h"

namespace uk {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// f32 on 16 rows: four v_mfma_f32_16x16x4_f32, element e of a lane's 16 bytes
// for the e-th; both operands pair the same way, so every k meets its partner.
struct F32Cfg16 {
  typedef floatx4 frag_t;
  typedef floatx4 acc_t;
  typedef float out_t;
  static constexpr int kElemBytes = 4;
  __device__ static acc_t mfma(frag_t a, frag_t b, acc_t c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
};

struct RowMajorArgs {
  const char* a;       // M x K
  const char* b;       // K x N
  char* c;             // M x N
  char* lhs;           // packed operands and result; null: not wanted
  char* rhs;
  char* out;
  int M, N, K, M0, N0, M1, N1, K1;
  int tiles_n, product_blocks, lhs_blocks;
  int accumulate;
  // K split: product block t + tiles * i multiplies the elements [i slice_k,
  // (i + 1) slice_k) of K for tile t into its own plane of partial sums (rows and
  // columns in whole tiles, accumulator type); partial is null without one.
  int tiles, slices, slice_k;
  void* partial;
};

// A 128-bit value moved down by `bytes` (0 to 15), zeros from above.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int bytes) {
  union { u32x4 v; unsigned __int128 x; } u;
  u.v = v;
  u.x >>= 8 * bytes;
  return u.v;
}

// Loads never leave the matrix and never branch: what lies past the end of a
// row is the 16 bytes (or 4 elements) that end there, moved down when they are
// stored; what lies past the last row is that row, replaced by zeros then. So
// all loads of a step are in flight together. (Rows of K are at least a chunk
// long, rows of N 4 elements.)
template <int kElemBytes>
__device__ __forceinline__ u32x4 load_chunk(const char* row, int k, int K) {
  constexpr int E = 16 / kElemBytes;
  u32x4 v;
  __builtin_memcpy(&v, row + (int64_t)(k + E <= K ? k : K - E) * kElemBytes, 16);   // (one load, aligned or not)
  return v;
}
template <int kElemBytes>
__device__ __forceinline__ u32x4 settle_chunk(u32x4 v, int k, int K, bool row_exists) {
  constexpr int E = 16 / kElemBytes;
  if (!row_exists || k >= K) return u32x4{0, 0, 0, 0};
  return k + E <= K ? v : shift_down(v, (k + E - K) * kElemBytes);
}

// Four consecutive elements of a row, in kElemBytes dwords.
template <int kElemBytes>
struct Four { uint32_t d[kElemBytes]; };
template <int kElemBytes>
__device__ __forceinline__ Four<kElemBytes> settle_four(Four<kElemBytes> r, int n, int N, bool row_exists) {
  if (!row_exists || n >= N) return Four<kElemBytes>{};
  if (n + 4 <= N) return r;
  u32x4 v = {0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < kElemBytes; ++i) v[i] = r.d[i];
  v = shift_down(v, (n + 4 - N) * kElemBytes);
#pragma unroll
  for (int i = 0; i < kElemBytes; ++i) r.d[i] = v[i];
  return r;
}

// Chunk of column e (0 to 3) from the 16 / kElemBytes rows of a four-column strip.
template <int kElemBytes>
__device__ __forceinline__ u32x4 column_chunk(const Four<kElemBytes>* rows, int e) {
  u32x4 v;
  if constexpr (kElemBytes == 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = rows[q].d[e];
  } else if constexpr (kElemBytes == 2) {
    const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = __builtin_amdgcn_perm(rows[2 * q + 1].d[e / 2], rows[2 * q].d[e / 2], sel);
  } else {
    const uint32_t sel = 0x0c0c0400u + 0x0101u * e;   // byte e of the second operand, then of the first
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t lo = __builtin_amdgcn_perm(rows[4 * q + 1].d[0], rows[4 * q].d[0], sel);
      const uint32_t hi = __builtin_amdgcn_perm(rows[4 * q + 3].d[0], rows[4 * q + 2].d[0], sel);
      v[q] = lo | hi << 16;
    }
  }
  return v;
}

// One workgroup's 256 chunks of a packed operand. Chunk r of the buffer is row
// i0 of the tile (i1, k1).
template <int kElemBytes>
__device__ void pack_block(const RowMajorArgs& p, int block) {
  constexpr int E = 16 / kElemBytes;
  const bool is_lhs = block < p.lhs_blocks;
  const uint32_t r = (uint32_t)(is_lhs ? block : block - p.lhs_blocks) * 256 + threadIdx.x;
  const uint32_t T0 = is_lhs ? p.M0 : p.N0, K1 = p.K1;
  if (r >= T0 * K1 * (uint32_t)(is_lhs ? p.M1 : p.N1)) return;
  const uint32_t tile = r / T0, i0 = r - tile * T0;
  const uint32_t i1 = tile / K1, k1 = tile - i1 * K1;
  const int i = (int)(i1 * T0 + i0), k = (int)k1 * E;
  u32x4 v = {0, 0, 0, 0};
  if (is_lhs) {
    if (i < p.M)
      v = settle_chunk<kElemBytes>(load_chunk<kElemBytes>(p.a + (int64_t)i * p.K * kElemBytes, k, p.K), k, p.K, true);
    *(u32x4*)(p.lhs + (int64_t)r * 16) = v;
  } else {
    typedef typename std::conditional<kElemBytes == 1, uint8_t,
                                      typename std::conditional<kElemBytes == 2, uint16_t, uint32_t>::type>::type elem_t;
    if (i < p.N) {
      const elem_t* q = (const elem_t*)p.b + i;
      elem_t x[E];
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = q[(int64_t)(k + e < p.K ? k + e : p.K - 1) * p.N];
#pragma unroll
      for (int e = 0; e < E; ++e)
        v[e * kElemBytes / 4] |= (k + e < p.K ? (uint32_t)x[e] : 0u) << (8 * (e * kElemBytes % 4));
    }
    *(u32x4*)(p.rhs + (int64_t)r * 16) = v;
  }
}

// What the sums of a result type are held in.
template <typename out_t>
struct Sum { typedef typename std::conditional<std::is_same<out_t, int32_t>::value, int32_t, float>::type type; };

// Adds the planes of a K split in order, then the old result, and stores the
// matrix and its tiles: one element per thread.
template <typename out_t>
__global__ __launch_bounds__(256) void matmul_rowmajor_sum_kernel(RowMajorArgs p, int rows, int cols) {
  typedef typename Sum<out_t>::type sum_t;
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x, plane = (int64_t)rows * cols;
  if (at >= plane) return;
  const int m = (int)(at / cols), n = (int)(at - (int64_t)m * cols);
  const int m1 = m / p.M0, m0 = m - m1 * p.M0, n1 = n / p.N0, n0 = n - n1 * p.N0;
  const bool in_matrix = m < p.M && n < p.N, in_tiles = p.out && m1 < p.M1 && n1 < p.N1;
  if (!in_matrix && !in_tiles) return;
  const sum_t* part = (const sum_t*)p.partial + at;
  out_t* const c = (out_t*)p.c + (int64_t)m * p.N + n;
  const sum_t old = p.accumulate && in_matrix ? (sum_t)*c : (sum_t)0;
  sum_t sum = 0;
#pragma unroll 8
  for (int i = 0; i < p.slices; ++i) sum += part[i * plane];
  const out_t v = (out_t)(sum + old);
  if (in_matrix) *c = v;
  if (in_tiles) ((out_t*)p.out)[(((int64_t)m1 * p.N1 + n1) * p.M0 + m0) * p.N0 + n0] = v;
}

template <typename Cfg, int kRows>
__global__ __launch_bounds__(256, 2) void matmul_rowmajor_kernel(RowMajorArgs p) {
  constexpr int kElemBytes = Cfg::kElemBytes;
  constexpr int E = 16 / kElemBytes;            // elements of a chunk
  constexpr int kChunks = 2048 / kRows;         // chunks of a row per step
  constexpr int kStep = kChunks * E;            // elements of K per step
  constexpr int kGroups = kRows / 4;            // four-column strips of the right-hand side
  typedef typename Cfg::frag_t frag_t;
  typedef typename Cfg::acc_t acc_t;
  typedef typename Cfg::out_t out_t;
  __shared__ u32x4 tile_a[2048], tile_b[2048];
  if ((int)blockIdx.x >= p.product_blocks) {
    pack_block<kElemBytes>(p, (int)blockIdx.x - p.product_blocks);
    return;
  }
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int slice = (int)blockIdx.x / p.tiles, tile = (int)blockIdx.x - slice * p.tiles;
  const int m_base = tile / p.tiles_n * kRows, n_base = tile % p.tiles_n * kRows;
  const int k_first = slice * p.slice_k, k_end = k_first + p.slice_k < p.K ? k_first + p.slice_k : p.K;
  auto place = [](int row, int chunk) { return row * kChunks + (chunk ^ ((row + (row >> 4)) & 15)); };

  // what this thread fetches of a step: chunk t % kChunks of 8 rows of A, and
  // two strips of 4 columns x E rows of B
  u32x4 next_a[8];
  Four<kElemBytes> next_b[2][E];
  const int my_row = m_base + t / kChunks, my_n = n_base + t % kGroups * 4;
  uint32_t row_at[8];                           // element offsets, 32 bits (operands of up to 64 MiB)
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int row = my_row + j * (kRows / 8);
    row_at[j] = (uint32_t)(row < p.M ? row : p.M - 1) * p.K;
  }
  const uint32_t col_at = my_n + 4 <= p.N ? my_n : p.N - 4, last_row = (uint32_t)(p.K - 1) * p.N;
  auto fetch = [&](int k_base) {
    const int ka = k_base + t % kChunks * E;
    const uint32_t at = ka + E <= p.K ? ka : p.K - E;
#pragma unroll
    for (int j = 0; j < 8; ++j) __builtin_memcpy(&next_a[j], p.a + (row_at[j] + at) * kElemBytes, 16);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t k_row = (uint32_t)(k_base + (t / kGroups + j * (256 / kGroups)) * E) * p.N;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint32_t r = k_row + (uint32_t)e * p.N;
        __builtin_memcpy(&next_b[j][e], p.b + ((r < last_row ? r : last_row) + col_at) * kElemBytes, 4 * kElemBytes);
      }
    }
  };
  fetch(k_first);

  // The wave's 2 x 2 blocks of 16x16: element r of a lane is row 4 (lane / 16) + r,
  // column lane % 16.
  const int wm = kRows == 64 ? wave / 2 * 32 : 0, wn = kRows == 64 ? wave % 2 * 32 : 0;
  const bool owner = kRows == 64 || wave == 0;   // stores the result
  // A step has sums of its own, one for every other instruction, which are added
  // to the whole at its end, and the old result last of all: the rounding error
  // of a sum grows with the number of terms it takes one by one.
  acc_t acc[2][2] = {}, old[2][2] = {};
  out_t* const c = (out_t*)p.c;
  if (p.accumulate && owner && !p.partial) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m_base + wm + i * 16 + lane / 16 * 4 + r, n = n_base + wn + j * 16 + lane % 16;
          if (m < p.M && n < p.N) old[i][j][r] = c[(int64_t)m * p.N + n];
        }
  }

  for (int k_base = k_first; k_base < k_end; k_base += kStep) {
    const int left = k_end - k_base;
    const int subs = left >= kStep ? kChunks / 4 : (left + 4 * E - 1) / (4 * E);   // of 4 chunks: one instruction's K
    if (k_base > k_first) __syncthreads();
    if (t % kChunks < subs * 4) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        tile_a[place(t / kChunks + j * (kRows / 8), t % kChunks)] = settle_chunk<kElemBytes>(
            next_a[j], k_base + t % kChunks * E, p.K, my_row + j * (kRows / 8) < p.M);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int chunk = t / kGroups + j * (256 / kGroups), k = k_base + chunk * E;
      if (chunk < subs * 4) {
        if (k + E > p.K || my_n + 4 > p.N) {
#pragma unroll
          for (int e = 0; e < E; ++e) next_b[j][e] = settle_four<kElemBytes>(next_b[j][e], my_n, p.N, k + e < p.K);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) tile_b[place(t % kGroups * 4 + e, chunk)] = column_chunk<kElemBytes>(next_b[j], e);
      }
    }
    __syncthreads();
    if (k_base + kStep < k_end) fetch(k_base + kStep);
    acc_t part[2][2][2] = {};
    auto multiply = [&](int s, acc_t (&sum)[2][2]) {
      union { u32x4 u; frag_t f; } fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[i].u = tile_a[place(wm + i * 16 + lane % 16, s * 4 + lane / 16)];
        fb[i].u = tile_b[place(wn + i * 16 + lane % 16, s * 4 + lane / 16)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) sum[i][j] = Cfg::mfma(fa[i].f, fb[j].f, sum[i][j]);
    };
    constexpr int kApart = kRows == 64 ? 1 : 4;   // (kRows = 32: a wave takes every fourth)
    for (int s = kRows == 64 ? 0 : wave; s < subs; s += 2 * kApart) {
      multiply(s, part[0]);
      if (s + kApart < subs) multiply(s + kApart, part[1]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += part[0][i][j] + part[1][i][j];
  }

  if constexpr (kRows == 32) {
    // the quarters of K, in wave order
    acc_t* const part = (acc_t*)tile_a;           // [wave - 1][block][lane]
    __syncthreads();
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) part[((wave - 1) * 4 + i) * 64 + lane] = acc[i / 2][i % 2];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i / 2][i % 2] += part[(w * 4 + i) * 64 + lane];
  }
  if (p.partial) {
    typedef typename Sum<out_t>::type sum_t;
    const int rows = p.tiles / p.tiles_n * kRows, cols = p.tiles_n * kRows;
    sum_t* const part = (sum_t*)p.partial + (int64_t)slice * rows * cols;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(int64_t)(m_base + wm + i * 16 + lane / 16 * 4 + r) * cols + n_base + wn + j * 16 + lane % 16] = acc[i][j][r];
    return;
  }
  out_t* const out = (out_t*)p.out;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n_base + wn + j * 16 + lane % 16;
    const int n1 = (int)((uint32_t)n / (uint32_t)p.N0), n0 = n - n1 * p.N0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m_base + wm + i * 16 + lane / 16 * 4 + r;
        const out_t v = (out_t)(acc[i][j][r] + old[i][j][r]);
        if (m < p.M && n < p.N) c[(int64_t)m * p.N + n] = v;
        if (out) {
          const int m1 = (int)((uint32_t)m / (uint32_t)p.M0), m0 = m - m1 * p.M0;
          if (m1 < p.M1 && n1 < p.N1) out[(((int64_t)m1 * p.N1 + n1) * p.M0 + m0) * p.N0 + n0] = v;
        }
      }
  }
}

// Estimated time in microseconds on kRows = side with K in `slices`. A step takes
// about as long whatever else runs, until a compute unit holds more than one
// workgroup; then the packed buffers and the result, and for a split the planes
// of sums, written and read, and the second launch. Fitted to 78 problems (f32,
// 16-bit and i8; 10 to 3900 rows and columns, K 200 to 4000) on both sides and
// 1 to 16 slices: 12 % off on average, and what it picks is 1.8 % from the best.
struct Estimate {
  int64_t tiles, steps;
  double step_us, bytes;
  template <typename Cfg>
  static Estimate of(const RowMajorArgs& p, int side) {
    constexpr bool kF32 = Cfg::kElemBytes == 4;   // (whose instructions take as long as a step's loads)
    const int64_t rows = (int64_t)p.M1 * p.M0, cols = (int64_t)p.N1 * p.N0;
    return {ceil_div(rows, (int64_t)side) * ceil_div(cols, (int64_t)side),
            ceil_div((int64_t)p.K * Cfg::kElemBytes, (int64_t)32768 / side),
            side == 64 ? (kF32 ? 3.9 : 3.0) : 2.8,
            (p.lhs ? 32.0 * rows * p.K1 : 0) + (p.rhs ? 32.0 * cols * p.K1 : 0) +
                (p.out ? 2.0 : 1.0) * rows * cols * sizeof(typename Cfg::out_t)};
  }
  double us(int cus, int side, int slices) const {
    const double load = (double)tiles * slices / cus;
    const double us = 4.3 + ceil_div(steps, (int64_t)slices) * step_us * (load > 1 ? load : 1) + bytes / 5.6e6;
    return slices > 1 ? us + 1.3 + 4.0 * slices * tiles * side * side / 2.8e6 : us;
  }
  // Below the time of every number of slices.
  double least_us(int cus) const { return 4.3 + (double)steps * step_us * tiles / cus + bytes / 5.6e6; }
};

// What the chain takes, from below: 5 us a launch when they follow each other,
// less 1, half a microsecond per MB of packed operands, and what the f32 matmul, which
// has no K split for so few tiles, takes beyond its launch (f32 172x54x2690 38.8
// us, estimated 37.4; bf16 1743x286x1222 25.3, 21.5; f16 54x163x733 17.0, 19.1).
// The rule: the estimate with 10 % added is below it. f16 54x163x733 8.6 us here;
// bf16 64x29x3693 21.2 as the chain, 35.0 here with K whole, 8.7 in 8 slices; f32
// 20x589x4022 43.6, 56.0, 13.5; i8 1024^3 18.7 and 11.5. Beyond it the chain wins:
// bf16 3421x599x980 24.4 as the chain, 36.7 here.
template <typename Cfg>
double chain_us(const RowMajorArgs& p) {
  const int launches = (p.lhs != nullptr) + (p.rhs != nullptr) + 1 + (p.out ? 1 + p.accumulate : 0);
  const double mb = 16e-6 * p.K1 * ((double)p.M1 * p.M0 + (double)p.N1 * p.N0);
  const double f32 = Cfg::kElemBytes == 4 ? 4 + 0.004 * p.K : 0;
  return 5.0 * launches - 1.0 + 0.5 * mb + (f32 < 13 ? f32 : 13);
}

// The fastest of both sides and 1 to max_slices slices of K; false when none takes
// limit_us or less. (A large problem, which is the chain's, is seen by least_us:
// the estimates of all slices took 0.5 us of every chain.)
template <typename Cfg>
bool choose(const RowMajorArgs& p, int max_slices, double limit_us, int* side, int* slices) {
  const int cus = device_cu_count();
  bool found = false;
  for (int try_side = 32; try_side <= 64; try_side += 32) {
    const Estimate e = Estimate::of<Cfg>(p, try_side);
    if (e.least_us(cus) > limit_us) continue;
    for (int n = 1; n <= max_slices && n <= e.steps; ++n) {
      const double us = e.us(cus, try_side, n);
      if (found ? us < limit_us : us <= limit_us) { found = true; limit_us = us; *side = try_side; *slices = n; }
    }
  }
  return found;
}

template <typename Cfg>
int launch(RowMajorArgs p, hipStream_t s) {
  const int64_t rows = (int64_t)p.M1 * p.M0, cols = (int64_t)p.N1 * p.N0;
  const double limit = chain_us<Cfg>(p) / 1.1;
  int side = 32, slices = 1;
  if (!choose<Cfg>(p, 16, limit, &side, &slices)) return IREE_AMD_UK_STATUS_NOT_FOUND;
  const int64_t elem_step = 32768 / Cfg::kElemBytes;              // elements of K per step, times the side
  auto lay_out = [&] {
    p.tiles_n = (int)ceil_div(cols, (int64_t)side);
    p.tiles = (int)(ceil_div(rows, (int64_t)side) * p.tiles_n);
    const int64_t step = elem_step / side;
    p.slice_k = (int)(ceil_div(ceil_div((int64_t)p.K, step), (int64_t)slices) * step);
    slices = (int)ceil_div((int64_t)p.K, (int64_t)p.slice_k);     // (no empty last slice)
  };
  lay_out();
  // (a graph keeps the addresses of its nodes: a call being captured takes no
  // memory that other calls on the stream use too)
  const bool may_split = slices > 1 && !scratch_under_capture(s);
  ScratchLease lease(s, may_split ? (size_t)slices * p.tiles * side * side * 4 : 0);
  if (slices > 1 && !lease.ptr()) {
    if (!choose<Cfg>(p, 1, limit, &side, &slices)) return IREE_AMD_UK_STATUS_NOT_FOUND;
    lay_out();
  }
  const int64_t plane = (int64_t)p.tiles * side * side;
  p.slices = slices;
  p.partial = slices > 1 ? lease.ptr() : nullptr;
  p.product_blocks = p.tiles * slices;
  p.lhs_blocks = p.lhs ? (int)ceil_div(rows * p.K1, (int64_t)256) : 0;
  const int rhs_blocks = p.rhs ? (int)ceil_div(cols * p.K1, (int64_t)256) : 0;
  const dim3 grid((unsigned)(p.product_blocks + p.lhs_blocks + rhs_blocks)), block(256);
  if (side == 32) hipLaunchKernelGGL((matmul_rowmajor_kernel<Cfg, 32>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((matmul_rowmajor_kernel<Cfg, 64>), grid, block, 0, s, p);
  const int st = check_hip(hipGetLastError(), "matmul_rowmajor launch");
  if (st || slices == 1) return st;
  const int padded_cols = p.tiles_n * side;
  hipLaunchKernelGGL(matmul_rowmajor_sum_kernel<typename Cfg::out_t>, dim3((unsigned)ceil_div(plane, (int64_t)256)),
                     block, 0, s, p, (int)(plane / padded_cols), padded_cols);
  return check_hip(hipGetLastError(), "matmul_rowmajor sum launch");
}

}  // namespace

int launch_matmul_rowmajor(const void* a, const void* b, void* c, void* lhs, void* rhs, void* out, int64_t M,
                           int64_t N, int64_t K, int M0, int N0, int K0, uint32_t flags, hipStream_t s) {
  Mmt4dTypeInfo ti;
  if (!mmt4d_type_info(flags, &ti) || ti.lhs_bits != ti.rhs_bits || ti.lhs_bits < 8) return IREE_AMD_UK_STATUS_NOT_FOUND;
  const int eb = ti.lhs_bits / 8;
  if (M <= 0 || N < 4 || K * eb < 16 || M > 65536 || N > 65536 || K > 65536) return IREE_AMD_UK_STATUS_NOT_FOUND;
  // (tiles that the chain's mmt4d would give to a matrix-core kernel as well:
  // others sum in the order of the element-wise kernel)
  const bool narrow = mmt4d_skinny_supported(flags, M0, N0, K0) && (M0 < 32 ? M <= M0 : N <= N0);
  if (K0 * eb != 16 || !(narrow || mmt4d_mfma_supported(flags, M0, N0, K0))) return IREE_AMD_UK_STATUS_NOT_FOUND;
  const int64_t M1 = ceil_div(M, (int64_t)M0), N1 = ceil_div(N, (int64_t)N0), K1 = ceil_div(K, (int64_t)K0);
  if (M1 * M0 * K1 * 16 > (64 << 20) || N1 * N0 * K1 * 16 > (64 << 20) || M1 * M0 * N1 * N0 > (16 << 20))
    return IREE_AMD_UK_STATUS_NOT_FOUND;
  // Buffers that share memory: the chain reads an operand completely before
  // the result is written, this kernel does not.
  struct Range { uintptr_t at; int64_t bytes; bool written; };
  const Range r[6] = {{(uintptr_t)a, M * K * eb, false},
                      {(uintptr_t)b, K * N * eb, false},
                      {(uintptr_t)c, M * N * ti.out_bytes, true},
                      {(uintptr_t)lhs, lhs ? M1 * M0 * K1 * 16 : 0, true},
                      {(uintptr_t)rhs, rhs ? N1 * N0 * K1 * 16 : 0, true},
                      {(uintptr_t)out, out ? M1 * M0 * N1 * N0 * ti.out_bytes : 0, true}};
  for (int i = 0; i < 6; ++i)
    for (int j = 0; j < i; ++j)
      if ((r[i].written || r[j].written) && r[i].at < r[j].at + r[j].bytes && r[j].at < r[i].at + r[i].bytes)
        return IREE_AMD_UK_STATUS_NOT_FOUND;
  if (!a || !b || !c || (uintptr_t)a % eb || (uintptr_t)b % eb || (uintptr_t)c % ti.out_bytes ||
      (uintptr_t)lhs % 16 || (uintptr_t)rhs % 16 || (uintptr_t)out % ti.out_bytes)
    return IREE_AMD_UK_STATUS_NOT_FOUND;
  RowMajorArgs p = {(const char*)a, (const char*)b, (char*)c, (char*)lhs, (char*)rhs, (char*)out,
                    (int)M, (int)N, (int)K, M0, N0, (int)M1, (int)N1, (int)K1, 0, 0, 0,
                    (flags & IREE_AMD_UK_FLAG_MMT4D_ACCUMULATE) != 0, 0, 1, 0, nullptr};
  switch (flags & IREE_AMD_UK_FLAG_MMT4D_TYPE_MASK) {
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F16F16F32: return launch<F16Cfg16>(p, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_BF16BF16F32: return launch<BF16Cfg16>(p, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F16F16F16: return launch<F16F16Cfg16>(p, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_BF16BF16BF16: return launch<BF16BF16Cfg16>(p, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_S8S8S32: return launch<S8Cfg16>(p, s);
    case IREE_AMD_UK_FLAG_MMT4D_TYPE_F32F32F32: return launch<F32Cfg16>(p, s);
    default: return IREE_AMD_UK_STATUS_NOT_FOUND;
  }
}

}  // namespace uk
