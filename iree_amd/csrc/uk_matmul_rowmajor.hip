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
// Called again and again on one stream, operands in the last-level cache, as the chain
// step by step, on tiles of 32 x 32 and 64 x 64 whose waves shared their operands
// through LDS, and here: f16 81x19x41 with C added 16.9, 7.5, 4.4 us; i8 1024^3 15.8,
// 10.6, 7.4; f16 1024^3 18.4, 22 to 24, 10.3; f16 2634x35x20 with C added 16.2, 8.2, 4.3.
//
// Multiplying workgroups: 16 or 32 rows x 64 columns of the result, K dealt to 8
// waves in steps of 64 bytes. A wave fetches its own steps straight into
// registers, two ahead, and waits for no other until the sums meet in LDS. A lane
// loads 4 columns of the 16 / element-size rows of the right-hand side that make a
// piece of a matrix-core operand, and turns them in registers into a piece of
// each column: column 4 i + y of the tile is column i of operand y, so that the
// sums of a lane are 4 consecutive columns again. Sharing the operands cost more
// than it saved: a step of 32 KB took 2.4 to 3.9 us, most of it waiting.
// What bounds it now: 3 to 3.5 us for a launch of one step, then the intake of the
// compute units that have work (loads of twice the columns gave the same times).
// A long K of few tiles is dealt to more workgroups, each with its own plane of
// partial sums, and a second launch adds the planes in order (2 us when it follows):
// bf16 64x29x3693 11.7 us whole, 6.7 in slices (14.3 as the chain).
#include <cmath>
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

constexpr int kThreads = 512;

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

// The bytes of a lane's piece move down by `bytes` (0 to 15), zeros from above.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int bytes) {
  const u32x4 a = bytes & 8 ? u32x4{v[2], v[3], 0, 0} : v;
  const u32x4 b = bytes & 4 ? u32x4{a[1], a[2], a[3], 0} : a;
  const uint32_t r = bytes & 3;
  return u32x4{__builtin_amdgcn_alignbyte(b[1], b[0], r), __builtin_amdgcn_alignbyte(b[2], b[1], r),
               __builtin_amdgcn_alignbyte(b[3], b[2], r), b[3] >> (8 * r)};
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

// Four consecutive elements of a row.
template <int kElemBytes>
struct Four { uint32_t d[kElemBytes]; };

// (of the matrix on tiles of 64 x 64: what lies past its ends, zeros)
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

// The piece of column e from the 16 / kElemBytes rows of a strip of 4 columns.
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

// One workgroup's kBlock chunks of a packed operand. Chunk r of the buffer is row
// i0 of the tile (i1, k1).
template <int kElemBytes, int kBlock = kThreads>
__device__ void pack_block(const RowMajorArgs& p, int block) {
  constexpr int E = 16 / kElemBytes;
  const bool is_lhs = block < p.lhs_blocks;
  const uint32_t r = (uint32_t)(is_lhs ? block : block - p.lhs_blocks) * kBlock + threadIdx.x;
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
  const out_t v = in_matrix ? (out_t)(sum + old) : (out_t)0;   // (padding of the tiles: zeros)
  if (in_matrix) *c = v;
  if (in_tiles) ((out_t*)p.out)[(((int64_t)m1 * p.N1 + n1) * p.M0 + m0) * p.N0 + n0] = v;
}

constexpr int kWaves = 8;
constexpr uint32_t kNowhere = 0x80000000u;   // past the end of every descriptor: the load gives zeros

// One workgroup: 16 MB rows x 64 columns of the result (of a slice of K).
template <typename Cfg, int MB>
__device__ __forceinline__ void multiply_tile(const RowMajorArgs& p) {
  constexpr int kElemBytes = Cfg::kElemBytes;
  constexpr int E = 16 / kElemBytes;            // elements of a piece, rows of the right-hand side per lane and step
  constexpr int kStep = 4 * E;                  // elements of K per step
  typedef typename Cfg::frag_t frag_t;
  typedef typename Cfg::acc_t acc_t;
  typedef typename Cfg::out_t out_t;
  typedef typename Sum<out_t>::type sum_t;
  typedef sum_t sum4_t __attribute__((ext_vector_type(4)));
  typedef sum_t sum4_unaligned_t __attribute__((ext_vector_type(4), aligned(4)));
  typedef out_t out4_t __attribute__((ext_vector_type(4), aligned(sizeof(out_t))));
  constexpr int F = MB * 4;                     // rows of a lane, 4 columns each
  constexpr int D = 2;                          // steps in flight
  typedef Four<kElemBytes> columns_t;
  __shared__ sum4_t sums[kWaves][F][64];
  __shared__ u32x4 turn[kWaves][MB][64];
  const int lane = threadIdx.x & 63, l16 = lane & 15, kc = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slice = (int)blockIdx.x / p.tiles, tile = (int)blockIdx.x - slice * p.tiles;
  const int m_base = tile / p.tiles_n * (MB * 16), n_base = tile % p.tiles_n * 64;
  const int k_first = slice * p.slice_k, k_end = k_first + p.slice_k < p.K ? k_first + p.slice_k : p.K;
  // This lane's columns: 4 of them, from n on; past the last ones the last ones again.
  const int n = n_base + l16 * 4, n_at = n + 4 <= p.N ? n : p.N - 4;
  const __amdgpu_buffer_rsrc_t a_src = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, 0x7FFFFFFF, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_src = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, 0x7FFFFFFF, 0x00020000);
  // (32-bit offsets: operands of up to 64 MiB)
  // The row and piece of a block of A that this lane fetches: the lanes of a quad the
  // 64 bytes of one row (of four rows they would be four requests). A block goes
  // through LDS into operand order, the pieces of row r rotated by r / 4 there.
  const int a_row = lane >> 2, a_piece = ((lane & 3) - (lane >> 4)) & 3;
  uint32_t a_at[MB];
#pragma unroll
  for (int x = 0; x < MB; ++x) {
    const int row = m_base + x * 16 + a_row;
    a_at[x] = (uint32_t)((row < p.M ? row : p.M - 1) * p.K + k_first + a_piece * E) * kElemBytes;
  }
  const uint32_t b_row = (uint32_t)p.N * kElemBytes;
  const uint32_t b_at = (uint32_t)(k_first + kc * E) * b_row + (uint32_t)n_at * kElemBytes;

  // what a step fetches: a piece of MB rows of A, 4 columns of E rows of B
  struct Step {
    u32x4 a[MB];
    columns_t b[E];
  };
  auto load_columns = [&](uint32_t at, uint32_t more) -> columns_t {
    columns_t r;
    if constexpr (kElemBytes == 1) {
      r.d[0] = __builtin_amdgcn_raw_buffer_load_b32(b_src, at, more, 0);
    } else if constexpr (kElemBytes == 2) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(b_src, at, more, 0);
      r.d[0] = v[0]; r.d[1] = v[1];
    } else {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(b_src, at, more, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) r.d[i] = v[i];
    }
    return r;
  };
  const int steps = (k_end - k_first) / kStep, tail = (k_end - k_first) % kStep;   // whole steps, elements left over
  // Steps are dealt to the waves one by one (the fewer a wave adds up one after the
  // other, the smaller the rounding error); what is past the last whole one is not
  // fetched.
  auto load = [&](Step& s, int i) {
    const int step = i * kWaves + wave;
    const bool exists = step < steps;
#pragma unroll
    for (int e = 0; e < E; ++e) s.b[e] = load_columns(exists ? b_at : kNowhere, exists ? (uint32_t)(step * kStep + e) * b_row : 0);
#pragma unroll
    for (int x = 0; x < MB; ++x)
      s.a[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_src, exists ? a_at[x] : kNowhere,
                                                                              exists ? step * 64 : 0, 0));
  };
  acc_t acc[MB][4];
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = acc_t{0, 0, 0, 0};
  auto multiply = [&](const Step& s) {
    // (a wave's LDS accesses are served in order)
    u32x4 fa[MB];
#pragma unroll
    for (int x = 0; x < MB; ++x) turn[wave][x][lane] = s.a[x];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int x = 0; x < MB; ++x) fa[x] = turn[wave][x][l16 * 4 + ((kc + (l16 >> 2)) & 3)];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const frag_t fb = __builtin_bit_cast(frag_t, column_chunk<kElemBytes>(s.b, y));
#pragma unroll
      for (int x = 0; x < MB; ++x) {
        // (f32, four instructions a step: each step has a sum of its own, for the
        // rounding error; 1.05 times as large on average without)
        if constexpr (kElemBytes == 4) acc[x][y] += Cfg::mfma(__builtin_bit_cast(frag_t, fa[x]), fb, acc_t{0, 0, 0, 0});
        else acc[x][y] = Cfg::mfma(__builtin_bit_cast(frag_t, fa[x]), fb, acc[x][y]);
      }
    }
  };
  // Row f of a lane after the sums.
  auto row_of = [&](int f) { return m_base + f / 4 * 16 + kc * 4 + f % 4; };
  constexpr int kOwn = (F + kWaves - 1) / kWaves;
  sum4_t old[kOwn];
  out_t* const c = (out_t*)p.c;
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    old[o] = sum4_t{0, 0, 0, 0};
    const int f = o * kWaves + wave;
    if (p.accumulate && !p.partial && f < F && row_of(f) < p.M) {
      const out4_t v = *(const out4_t*)(c + (int64_t)row_of(f) * p.N + n_at);
#pragma unroll
      for (int e = 0; e < 4; ++e) old[o][e] = (sum_t)v[e];
    }
  }
  // The step that ends inside itself: pieces that cross the end of K are those that
  // end there, moved down; rows past it the last one, replaced by zeros.
  const bool has_tail = tail > 0 && wave == steps % kWaves;
  const int k_tail = k_first + steps * kStep + kc * E, a_tail = k_first + steps * kStep + a_piece * E;   // (of B, of A)
  Step last;
  if (has_tail) {
#pragma unroll
    for (int x = 0; x < MB; ++x) {
      const int back = a_tail + E <= p.K ? 0 : a_tail + E - p.K;
      last.a[x] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                a_src, a_at[x] + (uint32_t)(steps * 64 - back * kElemBytes), 0, 0));
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = k_tail + e < k_end ? k_tail + e : k_end - 1;
      last.b[e] = load_columns((uint32_t)k * b_row + (uint32_t)n_at * kElemBytes, 0);
    }
  }
  const int rounds = steps > wave ? (steps - wave - 1) / kWaves + 1 : 0;      // steps of this wave
  if (rounds > 0) {
    Step ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load(ring[d], d);
#pragma unroll 1
    for (int i = 0; i + D < rounds; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        __builtin_amdgcn_sched_barrier(0);
        multiply(ring[d]);
        __builtin_amdgcn_sched_barrier(0);
        load(ring[d], i + D + d);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D; ++d) multiply(ring[d]);
  }
  if (has_tail) {
    const int left = k_end - k_tail;            // rows of this lane's that exist
#pragma unroll
    for (int x = 0; x < MB; ++x) {
      const int back = a_tail + E <= p.K ? 0 : a_tail + E - p.K;
      last.a[x] = a_tail < p.K ? shift_down(last.a[x], back * kElemBytes & 15) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e >= left) last.b[e] = columns_t{};
    multiply(last);
  }
  // ---- the waves' sums, by twos, then the old result --------------------
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sums[wave][x * 4 + r][lane] = sum4_t{acc[x][0][r], acc[x][1][r], acc[x][2][r], acc[x][3][r]};
  __syncthreads();
  out_t* const out = (out_t*)p.out;
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    const int f = o * kWaves + wave;
    if (f >= F) break;
    const int m = row_of(f);
    sum4_t part[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) part[w] = sums[w][f][lane];
#pragma unroll
    for (int apart = 1; apart < kWaves; apart *= 2)
#pragma unroll
      for (int w = 0; w < kWaves; w += 2 * apart) part[w] += part[w + apart];
    sum4_t sum = part[0];
    if (p.partial) {
      const int64_t cols = (int64_t)p.tiles_n * 64, rows = (int64_t)p.tiles / p.tiles_n * (MB * 16);
      if (n < p.N) *(sum4_unaligned_t*)((sum_t*)p.partial + ((int64_t)slice * rows + m) * cols + n_at) = sum;
      continue;
    }
    sum += old[o];
    out4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (out_t)sum[e];
    // (a repeated column is stored by the lane whose own it is: the others may be in
    // another workgroup, which then adds to it as well)
    const bool own = n_at == n;
    if (m < p.M && n < p.N) {
      out_t* const dst = c + (int64_t)m * p.N + n_at;
      if (own) {
        *(out4_t*)dst = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n_at + e >= n) dst[e] = v[e];
      }
    }
    if (out) {
      const int m1 = (int)((uint32_t)m / (uint32_t)p.M0), m0 = m - m1 * p.M0;
      if (m1 >= p.M1) continue;
      if (m >= p.M) v = out4_t{(out_t)0, (out_t)0, (out_t)0, (out_t)0};      // (padding of the tiles: zeros)
      auto place = [&](int col) -> out_t* {
        const int n1 = (int)((uint32_t)col / (uint32_t)p.N0), n0 = col - n1 * p.N0;
        return out + (((int64_t)m1 * p.N1 + n1) * p.M0 + m0) * p.N0 + n0;
      };
      if (p.N0 % 4 == 0 && own) {
        *(out4_t*)place(n) = v;
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n < p.N && n_at + e >= n) *place(n_at + e) = v[e];
        const int at = n + e;
        if (at >= p.N && at < p.N1 * p.N0) *place(at) = (out_t)0;
      }
    }
  }
}

template <typename Cfg, int MB>
__global__ __launch_bounds__(kThreads, 4) void matmul_rowmajor_kernel(RowMajorArgs p) {
  if ((int)blockIdx.x >= p.product_blocks) {
    pack_block<Cfg::kElemBytes>(p, (int)blockIdx.x - p.product_blocks);
    return;
  }
  multiply_tile<Cfg, MB>(p);
}

// The same on 64 x 64 of the result per workgroup: 4 waves, each a 32 x 32 quarter of it
// for all of K, which comes in steps of 512 bytes through LDS (64 KiB of both operands;
// chunk c of row r lies at c ^ hash(r) within 16, so that fragment reads, 16 rows of one
// chunk, and the turned stores hit 16 bank groups). The kernel above sums its 8 waves
// through LDS whatever K is; where K is a step or two and the result large, that is
// most of its time. Which of them: square_us.
template <typename Cfg>
__global__ __launch_bounds__(256, 2) void matmul_rowmajor_square_kernel(RowMajorArgs p) {
  constexpr int kRows = 64;
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
    pack_block<kElemBytes, 256>(p, (int)blockIdx.x - p.product_blocks);
    return;
  }
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int tile = (int)blockIdx.x;
  const int m_base = tile / p.tiles_n * kRows, n_base = tile % p.tiles_n * kRows;
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
  fetch(0);

  // The wave's 2 x 2 blocks of 16x16: element r of a lane is row 4 (lane / 16) + r,
  // column lane % 16.
  const int wm = wave / 2 * 32, wn = wave % 2 * 32;
  // A step has sums of its own, one for every other instruction, which are added
  // to the whole at its end, and the old result last of all: the rounding error
  // of a sum grows with the number of terms it takes one by one.
  acc_t acc[2][2] = {}, old[2][2] = {};
  out_t* const c = (out_t*)p.c;
  if (p.accumulate) {
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

  for (int k_base = 0; k_base < p.K; k_base += kStep) {
    const int left = p.K - k_base;
    const int subs = left >= kStep ? kChunks / 4 : (left + 4 * E - 1) / (4 * E);   // of 4 chunks: one instruction's K
    if (k_base > 0) __syncthreads();
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
    if (k_base + kStep < p.K) fetch(k_base + kStep);
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
    for (int s = 0; s < subs; s += 2) {
      multiply(s, part[0]);
      if (s + 1 < subs) multiply(s + 1, part[1]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += part[0][i][j] + part[1][i][j];
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
        const bool in_matrix = m < p.M && n < p.N;
        const out_t v = in_matrix ? (out_t)(acc[i][j][r] + old[i][j][r]) : (out_t)0;   // (padding of the tiles: zeros)
        if (in_matrix) c[(int64_t)m * p.N + n] = v;
        if (out) {
          const int m1 = (int)((uint32_t)m / (uint32_t)p.M0), m0 = m - m1 * p.M0;
          if (m1 < p.M1 && n1 < p.N1) out[(((int64_t)m1 * p.N1 + n1) * p.M0 + m0) * p.N0 + n0] = v;
        }
      }
  }
}

// Estimated time in microseconds on 16 mb rows x 64 columns with K in `slices`: the
// first round of workgroups, one per compute unit, each further one, an eighth of the
// steps of all of them (by element size), the result, C, and for a split the planes
// of sums and the launch that adds them. Fitted to half of 1300 problems (8 to 4096
// rows and columns, K 16 to 4096, six types) on 1 to 16 slices; on the other half
// 12 % off on average, and what it picks is 1 % from the best. A B beyond the 4 MB of an
// L2 comes from behind it, and in part for every row of workgroups anew, which those
// problems hardly had: with kBehind and kAgain 30 of 16328 others took over 20 % longer than
// as the chain, without them 102 (bf16 281x3489x3988 63.3 us in one launch, 38.4 as the
// chain; f16 45x4023x3840 38.1 and 27.3). f32, whose matrix instructions hide most of that, has
// less of it.
struct Shape {
  float first, round, step4, step1, step2, hidden, store, add, split, plane;
};
constexpr double kL2Mb = 4.0;
constexpr Shape kShapes[2] = {{3.47f, 0.30f, 0.82f, 0.99f, 0.78f, 0.26f, 0.42f, 0.18f, 2.10f, 1.12f},
                              {3.68f, 0.17f, 1.28f, 1.54f, 0.95f, 0.05f, 0.39f, 0.22f, 1.91f, 1.11f}};

struct Estimate {
  double groups, steps, step_us, other;
  const Shape& t;
  int cus;
  template <typename Cfg>
  static Estimate of(const RowMajorArgs& p, int mb, int cus) {
    const Shape& t = kShapes[mb - 1];
    const int rows = p.M1 * p.M0, cols = p.N1 * p.N0;
    const double groups = (double)((rows + 16 * mb - 1) / (16 * mb)) * ((cols + 63) / 64);
    const double result = (double)rows * cols * sizeof(typename Cfg::out_t) * 1e-6 * (p.out ? 2 : 1);
    const double b_mb = 1e-6 * cols * p.K * Cfg::kElemBytes, over = std::fmax(b_mb - kL2Mb, 0.0);
    const double kBehind = Cfg::kElemBytes == 4 ? 0.2 : 0.4, kAgain = Cfg::kElemBytes == 4 ? 0.02 : 0.08;    // us per MB
    const double again = kBehind * over + kAgain * std::fmin(over / kL2Mb, 1.0) * b_mb * ((rows + 16 * mb - 1) / (16 * mb));
    return {groups, std::ceil(p.K * (Cfg::kElemBytes / 64.0)),
            (Cfg::kElemBytes == 4 ? t.step4 : Cfg::kElemBytes == 1 ? t.step1 : t.step2) / 8.0,
            result * t.store + again + (p.accumulate ? t.add : 0.0), t, cus};
  }
  double us(int mb, int slices) const {
    const double rounds = std::ceil(groups * slices / cus), stream = rounds * std::ceil(steps / slices) * step_us;
    const double us = t.first + t.round * (rounds - 1) + (stream > t.hidden ? stream - t.hidden : 0.0) + other;
    return slices > 1 ? us + t.split + t.plane * groups * slices * mb * 4096e-6 : us;
  }
};

// What the chain takes: its launches, the packed operands and the result, the
// matrix instructions, and a share of K (fitted to the same problems, 11 % off on
// average). Without a packed result (the matmul writes the matrix, and reads the old one
// when it accumulates) a byte of the result costs a third. The rule: the estimate of one
// launch is below 0.9 of it (f32, not too large: 1.1). On 16328 other problems (32 to 4200 rows and
// columns, K 8 to 4200) that is 1.9 % from the best of all three on average, the noise of the
// timing among it, and 11 take over 20 % longer than as the chain (f16 2945x3940x145 without
// a packed result is one that the store counted twice sent to 64 x 64 tiles: 20.9 us as the
// chain, 32.7 there).
// A chain that does not pack A (its matmul reads the matrix, so there are two
// launches) was not among them; its estimate is from below.
template <typename Cfg>
double chain_us(const RowMajorArgs& p) {
  const int launches = (p.lhs != nullptr) + (p.rhs != nullptr) + 1 + (p.out ? 1 + p.accumulate : 0);
  const double rows = (double)p.M1 * p.M0, cols = (double)p.N1 * p.N0, bytes = (double)p.K * Cfg::kElemBytes;
  if (!p.lhs) {
    const double f32 = Cfg::kElemBytes == 4 ? 4 + 0.004 * p.K : 0;
    return 5.0 * launches - 1.0 + 0.5e-6 * (rows + cols) * bytes + (f32 < 13 ? f32 : 13);
  }
  const double giga = Cfg::kElemBytes == 4 ? 16.1 : Cfg::kElemBytes == 1 ? 3.0 : 2.8;
  const double store = p.out ? 0.62 : p.accumulate ? 0.35 : 0.2;
  return 3.17 + 2.40 * launches + 0.48e-6 * (rows + cols) * bytes + store * 1e-6 * rows * cols * sizeof(typename Cfg::out_t) +
         giga * 1e-9 * rows * cols * p.K + 0.16e-3 * bytes;
}

// The chain on full tiles whose matmul writes C beside the packed result
// (launch_matmul_chain): two launches. Fitted to 18000 problems (33 to 4096 rows and
// columns, K 16 to 4096), 11 to 12 % off on average; see times_shorter for what that leaves.
// f32 keeps the fit above, which counts an unpack (and a pack of C) that its chain no longer
// launches; it has not been fitted again.
template <typename Cfg>
bool full_tiles_chain(const RowMajorArgs& p) {
  return Cfg::kElemBytes != 4 && p.lhs && p.rhs && p.out && p.M0 == 32 && p.N0 == 32;
}
template <typename Cfg>
double full_tiles_chain_us(const RowMajorArgs& p) {
  constexpr bool kS8 = Cfg::kElemBytes == 1;
  const double rows = (double)p.M1 * p.M0, cols = (double)p.N1 * p.N0, bytes = (double)p.K * Cfg::kElemBytes;
  const double out_mb = rows * cols * 1e-6 * sizeof(typename Cfg::out_t);
  return (kS8 ? 11.1 : 9.6) + (kS8 ? 0.55e-6 : 0.48e-6) * (rows + cols) * bytes + 0.34 * out_mb +
         (kS8 ? 1.9e-9 : 2.9e-9) * rows * cols * p.K - (kS8 ? 0.79e-3 : 0.2e-3) * bytes +
         (p.accumulate ? 1.1 + (sizeof(typename Cfg::out_t) == 2 ? 0.8 : 0.43) * out_mb : 0.0);
}

// By how much the estimate of the chain has to be the shorter: by the bytes of a result and
// the rows of b (any, whole 128-byte lines, whole 8 KiB, where the chain packs each operand by
// a launch of its own as well). Time over estimate of one launch, over the same of the chain,
// where the estimates are within 1.6 of each other, has its middle at 0.86, 0.76 and 0.64 for f32
// results, 1.09, 1.01 and 0.90 for 16-bit ones, and is larger where C is added; the
// factors are those that gave the shortest times in all. Not for results of more than 24 MB (f32)
// or 6 MB, which lose by it (bf16 added to C 3874x4096x357 70 us in one launch, 52 as a chain).
// int8 that is not added to C: 0.93, with rows of whole 64 bytes 0.81 (8 KiB 0.89, where it
// gave nothing); of 300 other problems 7 instead of 16 over 5 % longer than before the chain's
// own estimate (715x3648x157 11.7 us in one launch, 14.9 as the chain).
template <typename Cfg>
double times_shorter(const RowMajorArgs& p) {
  constexpr bool kF32Out = sizeof(typename Cfg::out_t) == 4;
  const int64_t elems = (int64_t)p.M1 * p.M0 * p.N1 * p.N0;
  if (Cfg::kElemBytes == 1) return p.accumulate || p.N % 4096 == 0 ? 1.0 : p.N % 64 == 0 ? 1.2 : 1.05;
  if (elems > (kF32Out ? 6000000 : 3000000)) return 1.0;
  if (p.N % 4096 == 0) return kF32Out ? 1.4 : 1.2;
  if (p.N % 64 == 0) return kF32Out && !p.accumulate ? 1.25 : 1.1;
  return kF32Out ? 1.1 : 1.0;
}

// The fastest of both shapes and 1 to max_slices slices of K, whose time replaces *us;
// false when none takes *us or less.
template <typename Cfg>
bool choose(const RowMajorArgs& p, int max_slices, double* us, int* mb, int* slices) {
  const int cus = device_cu_count();
  // (f32 of a short K: its results, several hundred rows and columns, took 1.2 times as long)
  const double longer = Cfg::kElemBytes == 4 && p.K <= 300 ? 1.2 : 1.0;
  bool found = false;
  for (int rows = 1; rows <= 2; ++rows) {
    const Estimate e = Estimate::of<Cfg>(p, rows, cus);
    for (int n = 1; n <= max_slices && (n == 1 || n * 8 <= e.steps); n *= 2) {
      const double t = longer * e.us(rows, n);
      if (t <= *us) { found = true; *us = t; *mb = rows; *slices = n; }
      if (e.groups * n >= 4 * cus) break;
    }
  }
  return found;
}

// The kernel on 64 x 64: workgroups beyond one per compute unit run one after the
// other, each with a fixed part and its share of K; the result, C and the packed
// operands. Fitted to 2000 problems of up to 1200 bytes of K, 8 to 9 % off on average.
// (int8: a result beyond 8 MB costs more than that, by 0.2 us per MB stored; of 3400 other
// problems 22 took over 20 % longer than as the chain without it, 7 with it: 4016x3477x16 35.2
// us as the chain, 46.6 here, 3069x2476x45 26.4 and 30.2.)
// 16-bit types have no such kernel: it was the best for 13 of 525 of theirs, f32 203 of 482
// (1200x1500x100 16.1 us on 16 or 32 x 64, 12.5 here; 900x1300x300 17.2 and 20.9).
template <typename Cfg>
double square_us(const RowMajorArgs& p) {
  constexpr bool kF32 = Cfg::kElemBytes == 4;
  const double rows = (double)p.M1 * p.M0, cols = (double)p.N1 * p.N0, bytes = (double)p.K * Cfg::kElemBytes;
  const double load = std::fmax(1.0, std::ceil(rows / 64) * std::ceil(cols / 64) / device_cu_count());
  const double out_mb = rows * cols * 4e-6;
  return (kF32 ? 3.82 : 4.50) + load * ((kF32 ? 0.32 : 0.81) + (kF32 ? 3.47 : 2.49) / 512 * bytes) +
         (p.out ? 1.36 : 0.0) + (kF32 ? 0.205 : 0.221) * out_mb * (p.out ? 2 : 1) + (p.accumulate ? 0.42 * out_mb : 0.0) +
         (kF32 ? 0.62e-6 : 0.45e-6) * (rows + cols) * bytes + (kF32 ? 0.0 : 0.2 * std::fmax(0.0, out_mb * (p.out ? 2 : 1) - 8));
}

template <typename Cfg>
int launch_square(RowMajorArgs p, hipStream_t s) {
  const int64_t rows = (int64_t)p.M1 * p.M0, cols = (int64_t)p.N1 * p.N0;
  p.tiles_n = (int)ceil_div(cols, (int64_t)64);
  p.tiles = p.product_blocks = (int)(ceil_div(rows, (int64_t)64) * p.tiles_n);
  p.lhs_blocks = p.lhs ? (int)ceil_div(rows * p.K1, (int64_t)256) : 0;
  const int rhs_blocks = p.rhs ? (int)ceil_div(cols * p.K1, (int64_t)256) : 0;
  hipLaunchKernelGGL(matmul_rowmajor_square_kernel<Cfg>, dim3((unsigned)(p.product_blocks + p.lhs_blocks + rhs_blocks)),
                     dim3(256), 0, s, p);
  return check_hip(hipGetLastError(), "matmul_rowmajor launch");
}

template <typename Cfg>
int launch(RowMajorArgs p, hipStream_t s) {
  constexpr int kStep = 64 / Cfg::kElemBytes;                     // elements of K per step
  const int64_t rows = (int64_t)p.M1 * p.M0, cols = (int64_t)p.N1 * p.N0;
  // The chain on full tiles is taken where its estimate is the shorter by times_shorter: the
  // estimate of one launch is the longer by as much where the two are near each other, more
  // with f32 results and with rows of b of whole cache lines. On 1236 problems of 16-bit types
  // 1.1 % from the faster of the two on average and 3 over 10 % longer than before this chain
  // had an estimate of its own, without it 2.7 % and 41; on 400 others none (bf16 130x8192x523
  // 11.6 us in one launch, 21.1 as the chain; f16 480x4736x146 11.1 and 14.5; 838x2220x468
  // 13.6 and 16.3).
  // f32 (the chain as it was fitted packed the operands one after the other; in one launch
  // they take 2.0 to 3.5 us less) takes longer as the chain than estimated, for results of up
  // to 3 million elements; on 2343 problems 2.6 % from the best kernel on average and 5 over
  // 20 % longer than as the chain, with 0.9 of it 3.1 % and 4, and 531x2782x605 42.0 us as the
  // chain, 27.8 in one launch.
  const bool full = full_tiles_chain<Cfg>(p);
  const double chain = full ? full_tiles_chain_us<Cfg>(p) : chain_us<Cfg>(p);
  const bool together = p.lhs && p.rhs && p.out && p.M0 == 32 && p.N0 == 32;
  const bool slow_chain = Cfg::kElemBytes == 4 && rows * cols <= 3000000;
  const double limit = full                       ? times_shorter<Cfg>(p) * chain
                       : together && chain < 24.0 ? chain - 2.4
                                                  : (slow_chain ? 1.1 : 0.9) * chain;
  int mb = 1, slices = 1;
  double us = limit;
  const bool found = choose<Cfg>(p, 16, &us, &mb, &slices);
  if constexpr (Cfg::kElemBytes != 2) {
    if (p.K * Cfg::kElemBytes <= 1200 && square_us<Cfg>(p) < us) return launch_square<Cfg>(p, s);
  }
  if (!found) return IREE_AMD_UK_STATUS_NOT_FOUND;
  auto lay_out = [&] {
    p.tiles_n = (int)ceil_div(cols, (int64_t)64);
    p.tiles = (int)(ceil_div(rows, (int64_t)mb * 16) * p.tiles_n);
    p.slice_k = (int)ceil_div(ceil_div((int64_t)p.K, (int64_t)kStep), (int64_t)slices) * kStep;
    slices = (int)ceil_div((int64_t)p.K, (int64_t)p.slice_k);     // (no empty last slice)
  };
  lay_out();
  // (a graph keeps the addresses of its nodes: a call being captured takes no
  // memory that other calls on the stream use too)
  const bool may_split = slices > 1 && !scratch_under_capture(s);
  ScratchLease lease(s, may_split ? (size_t)slices * p.tiles * mb * 4096 : 0);
  if (slices > 1 && !lease.ptr()) {
    us = limit;
    if (!choose<Cfg>(p, 1, &us, &mb, &slices)) return IREE_AMD_UK_STATUS_NOT_FOUND;
    lay_out();
  }
  const int64_t plane = (int64_t)p.tiles * mb * 1024;
  p.slices = slices;
  p.partial = slices > 1 ? lease.ptr() : nullptr;
  p.product_blocks = p.tiles * slices;
  p.lhs_blocks = p.lhs ? (int)ceil_div(rows * p.K1, (int64_t)kThreads) : 0;
  const int rhs_blocks = p.rhs ? (int)ceil_div(cols * p.K1, (int64_t)kThreads) : 0;
  const dim3 grid((unsigned)(p.product_blocks + p.lhs_blocks + rhs_blocks));
  if (mb == 1) hipLaunchKernelGGL((matmul_rowmajor_kernel<Cfg, 1>), grid, dim3(kThreads), 0, s, p);
  else hipLaunchKernelGGL((matmul_rowmajor_kernel<Cfg, 2>), grid, dim3(kThreads), 0, s, p);
  const int st = check_hip(hipGetLastError(), "matmul_rowmajor launch");
  if (st || slices == 1) return st;
  const int padded_cols = p.tiles_n * 64;
  hipLaunchKernelGGL(matmul_rowmajor_sum_kernel<typename Cfg::out_t>, dim3((unsigned)ceil_div(plane, (int64_t)256)),
                     dim3(256), 0, s, p, (int)(plane / padded_cols), padded_cols);
  return check_hip(hipGetLastError(), "matmul_rowmajor sum launch");
}

// Buffers that share memory: a chain of launches reads an operand completely before
// the next buffer is written, the kernels that do several of its steps do not.
bool share_memory(const void* a, const void* b, const void* c, const void* lhs, const void* rhs, const void* out, int64_t M,
                  int64_t N, int64_t K, int eb, int ob, int64_t lhs_bytes, int64_t rhs_bytes, int64_t out_bytes) {
  struct Range { uintptr_t at; int64_t bytes; bool written; };
  const Range r[6] = {{(uintptr_t)a, M * K * eb, false},
                      {(uintptr_t)b, K * N * eb, false},
                      {(uintptr_t)c, M * N * ob, true},
                      {(uintptr_t)lhs, lhs ? lhs_bytes : 0, true},
                      {(uintptr_t)rhs, rhs ? rhs_bytes : 0, true},
                      {(uintptr_t)out, out ? out_bytes : 0, true}};
  for (int i = 0; i < 6; ++i)
    for (int j = 0; j < i; ++j)
      if ((r[i].written || r[j].written) && r[i].at < r[j].at + r[j].bytes && r[j].at < r[i].at + r[i].bytes) return true;
  return false;
}

}  // namespace

int launch_matmul_chain(const void* a, const void* b, void* c, void* lhs, void* rhs, void* out, int64_t M, int64_t N,
                        int64_t K, int M0, int N0, int K0, uint32_t flags, hipStream_t s) {
  Mmt4dTypeInfo ti;
  if (!a || !b || !c || !lhs || !rhs || !mmt4d_type_info(flags, &ti) || ti.lhs_bits != ti.rhs_bits || ti.lhs_bits < 8 ||
      M < 1 || N < 1 || K < 1 || M >= 1 << 30 || N >= 1 << 30 || K >= 1 << 30 || M0 < 1 || N0 < 1 || K0 < 1)
    return IREE_AMD_UK_STATUS_NOT_FOUND;
  const int eb = ti.lhs_bits / 8, ob = ti.out_bytes;
  const int64_t M1 = ceil_div(M, (int64_t)M0), N1 = ceil_div(N, (int64_t)N0), K1 = ceil_div(K, (int64_t)K0);
  if (K0 * eb != 16 || !mmt4d_mfma_supported(flags, M0, N0, K0) || (!out && (M0 != 32 || N0 != 32)) || (uintptr_t)c % ob ||
      (uintptr_t)out % ob ||
      share_memory(a, b, c, lhs, rhs, out, M, N, K, eb, ob, M1 * M0 * K1 * 16, N1 * N0 * K1 * 16, M1 * M0 * N1 * N0 * ob))
    return IREE_AMD_UK_STATUS_NOT_FOUND;
  int packed = launch_pack_operands(a, b, lhs, rhs, M, N, K, M0, N0, K0, eb, s);
  if (packed == IREE_AMD_UK_STATUS_NOT_FOUND && eb == 2 && N % 4096 == 0 && M0 == 32 && N0 == 32 &&
      !(((uintptr_t)a | (uintptr_t)b) % 2) && !(((uintptr_t)lhs | (uintptr_t)rhs) % 16)) {
    // (rows a power of two apart: each operand by the kernel that suits it)
    const uint32_t type = IREE_AMD_UK_FLAG_PACK_TYPE_F16F16;
    UK_RETURN_IF_ERROR(iree_amd_uk_pack(a, 0, K, 1, lhs, 0, K1 * M0 * K0, (int64_t)M0 * K0, M, K, M1, K1, M0, K0, 0, type,
                                        nullptr, s));
    packed = iree_amd_uk_pack(b, 0, N, 1, rhs, 0, K1 * N0 * K0, (int64_t)N0 * K0, K, N, N1, K1, N0, K0, 0,
                              type | IREE_AMD_UK_FLAG_PACK_TRANSPOSE_INNER | IREE_AMD_UK_FLAG_PACK_TRANSPOSE_OUTER, nullptr, s);
  }
  if (packed) return packed;
  if (!out)
    return iree_amd_uk_mmt4d_unpack(lhs, 0, K1 * M0 * K0, rhs, 0, K1 * N0 * K0, c, 0, N, M, N, M1, N1, K1, K0, flags, 1.0f,
                                    s);
  if (M0 == 32 && N0 == 32) {
    // The matmul writes the matrix beside the tiles (and adds to the matrix itself), and
    // the launch that would read the tiles back (and the one that packs C) is not needed:
    // bf16 1999 x 4099 x 3001 67.1 -> 63.3 us, f16 2048^3 with f16 results 34.6 -> 31.1,
    // 1000 x 4000 x 3000 added to C 51.0 -> 44.7, i8 4096^3 96.2 -> 85.7, 2000 x 3000 x 1000
    // 30.5 -> 26.0. What is left of the unpack is its store, at the rate of memory: all
    // workgroups of a round store at once.
    const iree_amd_uk_mmt4d_params_t p = {lhs, 0, K1 * M0 * K0, rhs, 0, K1 * N0 * K0, c, 0, N, M1, N1, K1, M0, N0, K0,
                                          flags, nullptr};
    const int st = launch_mmt4d_and_unpack_mfma(p, M, N, out, s);
    if (st != IREE_AMD_UK_STATUS_NOT_FOUND) {
      if (!st) note_kernel_path("mmt4d:mfma");
      return st;
    }
  }
  const uint32_t copy = ob == 2 ? IREE_AMD_UK_FLAG_PACK_TYPE_F16F16 : IREE_AMD_UK_FLAG_PACK_TYPE_I32I32;
  if (flags & IREE_AMD_UK_FLAG_MMT4D_ACCUMULATE)
    UK_RETURN_IF_ERROR(iree_amd_uk_pack(c, 0, N, 1, out, 0, N1 * M0 * N0, (int64_t)M0 * N0, M, N, M1, N1, M0, N0, 0, copy,
                                        nullptr, s));
  UK_RETURN_IF_ERROR(iree_amd_uk_mmt4d(lhs, 0, K1 * M0 * K0, rhs, 0, K1 * N0 * K0, out, 0, N1 * M0 * N0, M1, N1, K1, M0, N0,
                                       K0, flags, nullptr, s));
  return iree_amd_uk_unpack(out, 0, N1 * M0 * N0, (int64_t)M0 * N0, c, 0, N, 1, M1, N1, M0, N0, M, N,
                            ob == 2 ? IREE_AMD_UK_FLAG_UNPACK_TYPE_F16F16 : IREE_AMD_UK_FLAG_UNPACK_TYPE_I32I32, nullptr, s);
}

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
  if (share_memory(a, b, c, lhs, rhs, out, M, N, K, eb, ti.out_bytes, M1 * M0 * K1 * 16, N1 * N0 * K1 * 16,
                   M1 * M0 * N1 * N0 * ti.out_bytes))
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
