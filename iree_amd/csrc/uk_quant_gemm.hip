// Grouped int4-weight dequantising matmul on many rows (the prefill of a prompt;
// a few rows take the streaming kernels of uk_quant.hip and uk_quant_gemv.hip).
//
//   out[m][n] = sum_g s[n][g] * sum_{k in g} x[m][k] * (w[n][k] - zp[n][g])
//
// The same arithmetic as there: the matrix cores multiply the f16 activations
// by the small integers w - zp, exact in f16, into an f32 sum per GROUP, which
// is then multiplied by the group's f32 scale and added to the result in f32.
// (Scaling the weights to f16 first would let the matrix cores add everything,
// and would round every weight once more.)
//
// A workgroup owns 64 or 128 rows x 64 WN columns: four waves side by side, each
// 16 WN of the columns, one or two of them above each other, each 64 of the
// rows. A wave dequantises the weights of its columns in the registers that
// feed the matrix cores (12 vector instructions per 8 weights) and adds the
// scaled group sums (4 FMAs per 16x16 block and group): for 64 x 64 and a span
// of 128 k that is 64 MFMAs and 270 vector instructions, which share one issue
// port. Two waves per SIMD then take 2700 cycles where the MFMAs alone are
// 2048: vector issue bounds the kernel, and a wave tile twice as tall, which
// would halve the dequantisation, does not fit the registers that vector
// instructions can reach. (Two waves per SIMD: a workgroup of 128 rows, or two of
// 64, which fit a compute unit's LDS up to 128 columns, 64 with groups of 32.)
// Measured at 14336 columns, K = 4096, groups of 128: 128 / 256 / 512 / 2048 rows
// 29.5 / 42.2 / 70.7 / 286 us, 0.85 PFLOP/s at 512 (as passes of 32 rows over all
// the weights 46.2 / 91.3 / 183 / 727).
// K goes in spans of 128:
//   * weights: a 16-column x 128-k slab is one 16-byte load per lane (the tiled
//     layout's 1 KiB), straight to registers, one span ahead;
//   * activations: the rows' 256 bytes of the span go to LDS with direct loads
//     (16 adjacent lanes fetch one row: whole cache lines), into a ring of 4
//     spans (3 where LDS is short), each row's 16-byte chunks rotated by the row number so that the
//     fragment reads (16 rows, one chunk column) touch every bank once;
//   * scales and zero points of 4 groups at a time: 16 bytes of each column,
//     straight to LDS two spans ahead, and from there, one span ahead, as the
//     f32 scale and the pair of f16 offsets that the dequantisation adds.
// A lane holds one column of a block: its scale is one LDS read per 16 columns
// and group.
#include "uk_common.h"
#include "uk_i4.h"

namespace uk {
using namespace i4;
namespace {

struct I4GemmArgs {
  const uint16_t* x;      // [M][K] f16
  const uint8_t* w;       // tiled u4
  const uint16_t* scale;  // [N][G] f16
  const uint8_t* zp;      // [N][G] packed u4
  uint16_t* out;          // [M][N] f16
  float* partial;         // K split: f32 sums [slice][M][N] (else nullptr)
  int M, N, K, G;
  int spans, slice_spans; // K / 128 in all / per workgroup row blockIdx.y
  int tiles_m, tiles_n;
  int group_shift;        // log2(group size / what the kernel scales at a time), groups above 128
  uint32_t w_bytes;
};

constexpr int kParamGroups = 4;   // groups of scales and offsets per refill
// refills kept: a refill is written two spans before its first use
constexpr int param_bufs(int log2_ge) { return log2_ge == 5 ? 4 : 2; }

template <int WM, int MB, int WN, int kLog2Ge>
constexpr int i4_gemm_param_bytes() { return 64 * WN * (32 + param_bufs(kLog2Ge) * kParamGroups * 8); }
// spans of activations in LDS: 4, or what fits
template <int WM, int MB, int WN, int kLog2Ge>
constexpr int i4_gemm_ring() {
  return 4 * WM * MB * 4096 + i4_gemm_param_bytes<WM, MB, WN, kLog2Ge>() <= 160 * 1024 ? 4 : 3;
}
template <int WM, int MB, int WN, int kLog2Ge>
constexpr int i4_gemm_lds_bytes() {
  return i4_gemm_ring<WM, MB, WN, kLog2Ge>() * WM * MB * 4096 + i4_gemm_param_bytes<WM, MB, WN, kLog2Ge>();
}

template <int N>
__device__ __forceinline__ void gemm_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 8 nibbles of one dword -> 8 f16 integers (nibble - zero point) in k order: a
// byte permute puts both nibbles of a byte into the two halves, (t & mask) |
// 0x6400'6400 makes them 1024 + n and 1024 + 16 n', and one packed FMA with
// (1, 1/16) and the offsets (-1024 - zp, -64 - zp) the pair n - zp, n' - zp,
// every step exact.
__device__ __forceinline__ half8 dequant_in_order(uint32_t w, uint32_t mask, half2v offsets) {
  union { uint32_t u[4]; half2v p[4]; half8 h; } r;
  const half2v scale = {(_Float16)1.0f, (_Float16)0.0625f};
  r.u[0] = and_or_magic(__builtin_amdgcn_perm(w, w, 0x0c000c00u), mask);
  r.u[1] = and_or_magic(__builtin_amdgcn_perm(w, w, 0x0c010c01u), mask);
  r.u[2] = and_or_magic(__builtin_amdgcn_perm(w, w, 0x0c020c02u), mask);
  r.u[3] = and_or_magic(__builtin_amdgcn_perm(w, w, 0x0c030c03u), mask);
#pragma unroll
  for (int i = 0; i < 4; ++i) r.p[i] = __builtin_elementwise_fma(r.p[i], scale, offsets);
  return r.h;
}

// kLog2Ge: log2 of the k that one scale covers at a time (groups above 128: 128).
template <int WM, int MB, int WN, int kLog2Ge>
__device__ __forceinline__ void dequant_matmul_i4_gemm_body(const I4GemmArgs& a) {
  constexpr int BM = WM * MB * 16, BN = 64 * WN, kWaveCount = 4 * WM;
  constexpr int kStageBytes = BM * 256;                     // one span of the rows
  constexpr int kXLoads = BM / 4 / kWaveCount;              // 1 KiB loads (4 rows) per wave and span
  constexpr int kGroupsPerSpan = 128 >> kLog2Ge;            // 1, 2, 4
  constexpr int kQPerGroup = 4 / kGroupsPerSpan;            // MFMA K-steps per group
  constexpr int kChunkSpans = kParamGroups / kGroupsPerSpan;
  constexpr int kParamBufs = param_bufs(kLog2Ge);
  constexpr int kRing = i4_gemm_ring<WM, MB, WN, kLog2Ge>();
  static_assert(MB == 4, "two pairs of row blocks");
  constexpr int kWAhead = WN >= 2 ? 1 : 2;                  // spans that a slab of weights is requested ahead
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* const lds_raw = lds + kRing * kStageBytes;                                  // scales [BN] x 16 bytes, zero points alike
  float* const lds_scale = (float*)(lds_raw + 32 * BN);                             // [kParamBufs][4][BN]
  uint32_t* const lds_off = (uint32_t*)(lds_scale + kParamBufs * kParamGroups * BN);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kc = lane >> 4;
  const int wn = wave & 3, wm = wave >> 2;                  // this wave's columns and rows of the tile
  int tm, tn;
  {
    // (workgroup ids go round-robin over the 8 XCDs: XCD x takes the x-th
    // contiguous slice of the tiles, row tiles of one column tile together, so
    // that they share its weights in one L2)
    const int total = a.tiles_m * a.tiles_n, per = total / 8, rem = total % 8;
    const int xcd = (int)blockIdx.x % 8, idx = (int)blockIdx.x / 8;
    const int logical = xcd * per + (xcd < rem ? xcd : rem) + idx;
    tn = logical / a.tiles_m;
    tm = logical - tn * a.tiles_m;
  }
  const int m_base = tm * BM, n_base = tn * BN;
  const int s0 = (int)blockIdx.y * a.slice_spans;
  const int T = a.spans - s0 < a.slice_spans ? a.spans - s0 : a.slice_spans;

  // ---- activations: this wave's rows [wave * BM / 4, ...), 4 per load --------
  const __amdgpu_buffer_rsrc_t x_src =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (uint32_t)a.M * (uint32_t)a.K * 2u, 0x00020000);
  uint32_t x_off[kXLoads];
#pragma unroll
  for (int j = 0; j < kXLoads; ++j) {
    const int r = (wave * kXLoads + j) * 4 + (lane >> 4);    // row of the tile
    int row = m_base + r;
    row = row < a.M ? row : a.M - 1;                         // (rows past the end: loaded, not stored)
    x_off[j] = (uint32_t)row * (uint32_t)a.K * 2u + (uint32_t)((l16 - r) & 15) * 16u;
  }
  // (past the last span it is loaded again, into a slot nobody reads any more:
  // the number of loads in flight, which the waits count, stays the same)
  auto issue_x = [&](int span, int slot, int j) {
    const uint32_t at = (uint32_t)(s0 + (span < T ? span : T - 1)) * 256u;
    char* base = lds + slot * kStageBytes + wave * (kXLoads * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(x_src, (__attribute__((address_space(3))) void*)(base + j * 1024), 16,
                                             x_off[j], at, 0, 0);
  };
  // fragment (block x, K-step q): row 16 x + l16, chunk 4 q + kc
  uint32_t read_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) read_off[q] = (uint32_t)l16 * 256u + (uint32_t)((4 * q + kc + l16) & 15) * 16u;
  auto read_x = [&](int slot, int x, int q) -> half8 {
    return *(const half8*)(lds + slot * kStageBytes + wm * (MB * 4096) + read_off[q] + x * 4096);
  };

  // ---- weights: this wave's WN slabs of 16 columns ---------------------------
  const __amdgpu_buffer_rsrc_t w_src = __builtin_amdgcn_make_buffer_rsrc((void*)a.w, 0, a.w_bytes, 0x00020000);
  const uint32_t w_lane = (uint32_t)l16 * 64u + (uint32_t)kc * 16u;
  uint32_t w_base[WN];
#pragma unroll
  for (int y = 0; y < WN; ++y) {
    int cb = n_base / 16 + wn * WN + y;
    cb = cb * 16 < a.N ? cb : a.N / 16 - 1;
    w_base[y] = ((uint32_t)(cb >> 1) * (uint32_t)a.spans + (uint32_t)s0) * 2048u + (uint32_t)(cb & 1) * 1024u;
  }
  u32x4 raw[kWAhead][WN];     // slabs of span s in raw[s % kWAhead]
  auto load_w = [&](int span, int y, u32x4& dst) {
    const uint32_t at = (uint32_t)(span < T ? span : T - 1) * 2048u;
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(w_src, w_lane, w_base[y] + at, 0);
    dst = u32x4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
  };

  // ---- scales and offsets: one column per thread (the first BN) --------------
  // The 4 groups of a column are fetched as the 16 bytes that begin at the
  // 4-byte boundary before them (or end with the array): a column's groups
  // start anywhere. The arrays are whole 32 columns, i.e. whole 16 bytes.
  const bool p_thread = BN >= 64 * kWaveCount || wave < BN / 64;
  const int p_col = (int)threadIdx.x;
  const __amdgpu_buffer_rsrc_t s_src =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.scale, 0, (uint32_t)a.N * (uint32_t)a.G * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t z_src =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.zp, 0, (uint32_t)a.N * (uint32_t)a.G / 2u, 0x00020000);
  auto group_of = [&](int chunk, int i) -> uint32_t {    // index of a group in the arrays
    int n = n_base + p_col;
    n = n < a.N ? n : a.N - 1;
    int g = (chunk * kParamGroups + i) >> a.group_shift;
    g = g < a.G ? g : a.G - 1;
    return (uint32_t)n * (uint32_t)a.G + (uint32_t)g;
  };
  auto window = [&](uint32_t at, uint32_t bytes) -> uint32_t {
    at &= ~3u;
    return at < bytes - 16u ? at : bytes - 16u;
  };
  const uint32_t s_bytes = (uint32_t)a.N * (uint32_t)a.G * 2u, z_bytes = s_bytes / 4u;
  auto request_params = [&](int chunk) {
    if (!p_thread) return;
    const uint32_t at = group_of(chunk, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        s_src, (__attribute__((address_space(3))) void*)(lds_raw + wave * 1024), 16, window(at * 2, s_bytes), 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        z_src, (__attribute__((address_space(3))) void*)(lds_raw + BN * 16 + wave * 1024), 16, window(at / 2, z_bytes), 0,
        0, 0);
  };
  auto convert_params = [&](int chunk) {
    if (!p_thread) return;
    const uint32_t first = group_of(chunk, 0);
    const char* sw = lds_raw + p_col * 16 - window(first * 2, s_bytes);
    const char* zw = lds_raw + BN * 16 + p_col * 16 - window(first / 2, z_bytes);
#pragma unroll
    for (int i = 0; i < kParamGroups; ++i) {
      const uint32_t at = group_of(chunk, i);
      const uint32_t zp = (*(const uint8_t*)(zw + at / 2) >> (4 * (at & 1))) & 15u;
      const int to = ((chunk % kParamBufs) * kParamGroups + i) * BN + p_col;
      lds_scale[to] = __half2float(__ushort_as_half(*(const uint16_t*)(sw + at * 2)));
      lds_off[to] = 0xD400E400u | zp | (zp << 20);             // -(1024 + zp), -(64 + zp)
    }
  };
  // of group e (absolute) and column block y: the lane's scale, its offsets
  auto params_at = [&](int e, int y) -> int {
    return (((e / kParamGroups) % kParamBufs) * kParamGroups + e % kParamGroups) * BN + (wn * WN + y) * 16 + l16;
  };
  auto scale_of = [&](int e, int y) -> float { return lds_scale[params_at(e, y)]; };
  auto offsets_of = [&](int e, int y) -> half2v {
    union { uint32_t u; half2v h; } o;
    o.u = lds_off[params_at(e, y)];
    return o.h;
  };
  uint32_t mask;
  asm volatile("v_mov_b32 %0, 0x00f0000f" : "=v"(mask));

  floatx4 acc[MB][WN];
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int y = 0; y < WN; ++y) acc[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};

  half8 xf[MB][4];        // activation fragments of the span
  half8 wf[2][4];         // weight fragments of this column block and the next
  constexpr int kPairs = MB / 2, kRegions = WN * kPairs;

  // (scales and offsets of the first two spans, and what the step before the
  // first would have requested)
  {
    const int chunk = s0 / kChunkSpans, chunk1 = (s0 + 1) / kChunkSpans;
    request_params(chunk);
    gemm_wait_vmcnt<0>();
    convert_params(chunk);
    if (chunk1 != chunk) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (a lane's own 16 bytes: read before they are replaced)
      request_params(chunk1);
      gemm_wait_vmcnt<0>();
      convert_params(chunk1);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if ((s0 + 2) % kChunkSpans == 0) request_params((s0 + 2) / kChunkSpans);
  }
#pragma unroll
  for (int d = 0; d < kWAhead; ++d)
#pragma unroll
    for (int y = 0; y < WN; ++y) load_w(d, y, raw[d][y]);
#pragma unroll
  for (int d = 0; d < kRing - 1; ++d)
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) issue_x(d, d, j);
  __syncthreads();
  auto read_pair = [&](int from, int xp) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) xf[2 * xp + h][q] = read_x(from, 2 * xp + h, q);
  };
  read_pair(0, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    wf[0][q] = dequant_in_order(raw[0][0][q], mask, offsets_of(s0 * kGroupsPerSpan + q / kQPerGroup, 0));

  // One span. Its work is cut into regions of two row blocks times one column
  // block (8 MFMAs), and every region carries the same share of everything
  // else, issued behind its MFMAs: the FMAs that add the sums of the region
  // before, the dequantisation of the next column block, loads. The fences keep
  // the compiler from moving work between regions (it would otherwise hold the
  // sums of many of them).
  floatx4 part[kGroupsPerSpan][2];     // of the region before
  float part_scale[kGroupsPerSpan];
#pragma unroll
  for (int g = 0; g < kGroupsPerSpan; ++g) {
    part[g][0] = part[g][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    part_scale[g] = 0.f;
  }
  auto add_part = [&](int region) {
    const int y = region / kPairs, x = region % kPairs * 2;
#pragma unroll
    for (int g = 0; g < kGroupsPerSpan; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[x + h][y][v] = __builtin_fmaf(part[g][h][v], part_scale[g], acc[x + h][y][v]);
  };
  auto span_step = [&](auto parity, int i, int slot) {
    constexpr int P = decltype(parity)::value;
    const int free_slot = slot == 0 ? kRing - 1 : slot - 1;     // (the span before: read by every wave)
    const int next_slot = slot + 1 == kRing ? 0 : slot + 1;
    // The NEXT span of activations was requested kRing - 2 steps ago: it has
    // landed once only what was requested since is outstanding (all of the last
    // step, or the weights of its second half). The barrier publishes it and
    // frees the slot of the span before.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    gemm_wait_vmcnt<kRing == 4 ? kXLoads + WN : WN / 2>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int e0 = (s0 + i) * kGroupsPerSpan;
    // (requested by the step before, ahead of its weights and activations)
    if ((s0 + i + 2) % kChunkSpans == 0) {
      convert_params((s0 + i + 2) / kChunkSpans);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if ((s0 + i + 3) % kChunkSpans == 0) request_params((s0 + i + 3) / kChunkSpans);
    __builtin_amdgcn_sched_barrier(0);
    float sc[2][kGroupsPerSpan];
#pragma unroll
    for (int g = 0; g < kGroupsPerSpan; ++g) sc[0][g] = scale_of(e0 + g, 0);
#pragma unroll
    for (int y = 0; y < WN; ++y) {
      half8 (&f)[4] = wf[(P * WN + y) & 1];
      half8 (&fn)[4] = wf[(P * WN + y + 1) & 1];
      // where the next column block's words are, and their groups
      const u32x4 next_raw = y + 1 < WN ? raw[kWAhead == 1 ? 0 : P][y + 1] : raw[kWAhead == 1 ? 0 : P ^ 1][0];
      const int next_y = y + 1 < WN ? y + 1 : 0, next_e = y + 1 < WN ? e0 : e0 + kGroupsPerSpan;
      half2v off[kGroupsPerSpan];
#pragma unroll
      for (int g = 0; g < kGroupsPerSpan; ++g) off[g] = offsets_of(next_e + g, next_y);
      // (this column block's words have been used: its slab of the span ahead)
      load_w(i + kWAhead, y, raw[kWAhead == 1 ? 0 : P][y]);
      if (y + 1 < WN) {
#pragma unroll
        for (int g = 0; g < kGroupsPerSpan; ++g) sc[(y + 1) & 1][g] = scale_of(e0 + g, y + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int xp = 0; xp < kPairs; ++xp) {
        const int region = y * kPairs + xp;
        // (in the first half of the step)
        constexpr int kHalf = kRegions / 2;
        if (region < kHalf) {
#pragma unroll
          for (int j = region * kXLoads / kHalf; j < (region + 1) * kXLoads / kHalf; ++j) issue_x(i + kRing - 1, free_slot, j);
        }
        // Activation fragments: the second pair of row blocks of this span while
        // its first pair is multiplied for the first time, the first pair of the
        // next span once this one's has been multiplied for the last time.
        if (region == 0) read_pair(slot, 1);
        if (region == kRegions - 1) read_pair(next_slot, 0);
        floatx4 t[kGroupsPerSpan][2];
#pragma unroll
        for (int g = 0; g < kGroupsPerSpan; ++g) {
          t[g][0] = t[g][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = g * kQPerGroup; q < (g + 1) * kQPerGroup; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              t[g][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[2 * xp + h][q], f[q], t[g][h], 0, 0, 0);
        }
        add_part(region > 0 ? region - 1 : kRegions - 1);     // (zeros before the first)
#pragma unroll
        for (int q = xp * 4 / kPairs; q < (xp + 1) * 4 / kPairs; ++q)
          fn[q] = dequant_in_order(next_raw[q], mask, off[q / kQPerGroup]);
#pragma unroll
        for (int g = 0; g < kGroupsPerSpan; ++g) {
          part[g][0] = t[g][0];
          part[g][1] = t[g][1];
          part_scale[g] = sc[y & 1][g];
        }
        // (8 MFMAs, each with its share of the vector instructions behind it)
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (8 * kGroupsPerSpan + 48 / kPairs + 7) / 8, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  int slot = 0;
  int i = 0;
  if constexpr (WN % 2) {
    // (the two spans of weight fragments and words take turns)
    for (; i + 2 <= T; i += 2) {
      span_step(std::integral_constant<int, 0>(), i, slot);
      slot = slot + 1 == kRing ? 0 : slot + 1;
      span_step(std::integral_constant<int, 1>(), i + 1, slot);
      slot = slot + 1 == kRing ? 0 : slot + 1;
    }
  }
#pragma unroll 1
  for (; i < T; ++i) {
    span_step(std::integral_constant<int, 0>(), i, slot);
    slot = slot + 1 == kRing ? 0 : slot + 1;
  }
  add_part(kRegions - 1);
  gemm_wait_vmcnt<0>();      // (loads into LDS must not outlive the workgroup)

  // Register v of block (x, y): row 16 x + 4 kc + v, column l16.
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m_base + (wm * MB + x) * 16 + kc * 4 + v;
      if (m >= a.M) continue;
#pragma unroll
      for (int y = 0; y < WN; ++y) {
        const int n = n_base + (wn * WN + y) * 16 + l16;
        if (n >= a.N) continue;
        const int64_t at = (int64_t)m * a.N + n;
        if (a.partial) a.partial[(int64_t)blockIdx.y * a.M * a.N + at] = acc[x][y][v];
        else ((_Float16*)a.out)[at] = (_Float16)acc[x][y][v];
      }
    }
}

template <int WM, int MB, int WN, int kLog2Ge>
__global__ __launch_bounds__(256 * WM, 2) void dequant_matmul_i4_gemm_kernel(I4GemmArgs a) {
  dequant_matmul_i4_gemm_body<WM, MB, WN, kLog2Ge>(a);
}

template <int WM, int WN, int kLog2Ge>
int launch_gemm_instance(const I4GemmArgs& a, int slices, hipStream_t s) {
  constexpr int kLds = i4_gemm_lds_bytes<WM, 4, WN, kLog2Ge>();
  static_assert(kLds <= 160 * 1024, "LDS ring exceeds 160 KiB");
  void (*kernel)(I4GemmArgs) = dequant_matmul_i4_gemm_kernel<WM, 4, WN, kLog2Ge>;
  static PerDeviceOnce attr_set_on;
  int dev = 0;
  UK_RETURN_IF_HIP(hipGetDevice(&dev));
  if (!attr_set_on.done(dev)) {
    UK_RETURN_IF_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    attr_set_on.mark(dev);
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)slices), dim3(256 * WM), kLds, s, a);
  return check_hip(hipGetLastError(), "dequant_matmul_i4 gemm launch");
}

template <int WM, int WN>
int launch_gemm_shape(const I4GemmArgs& a, int log2_ge, int slices, hipStream_t s) {
  switch (log2_ge) {
    case 5: return launch_gemm_instance<WM, WN, 5>(a, slices, s);
    case 6: return launch_gemm_instance<WM, WN, 6>(a, slices, s);
    default: return launch_gemm_instance<WM, WN, 7>(a, slices, s);
  }
}

// Estimated time in microseconds on shape v with K in `slices`, by group size (32,
// 64, 128 and more). A span of 128 k of a workgroup takes `alone` in the last round
// when that gives a compute unit one workgroup at most, `shared` when it gives two
// to some, and `round` in the rounds before, which overlap with the next; `fixed`
// is what a workgroup needs before its first and after its last span. Then the
// result, and for a split the partial sums and the launch that adds them. Fitted to
// every shape and 1 to 8 slices on 3568 problems (33 to 700 rows, 256 to 14336
// columns, K 256 to 14336, groups of 32 to 256): 2.6 % off on average on 2941 other
// problems, where what it picks is 0.6 % slower than the best on average, 3.7 % in
// the 95th percentile and 29 % at most. (A count of vector instructions and bytes,
// which chose before: 3.9, 22 and 64 %. 203 x 3904 x 11776, groups of 128: 58 us as
// one slice of 64x128, 38 as four.)
constexpr int kShapes = 5;
struct GemmShape {
  int wm, wn;
  float alone[3], shared[3], round[3], fixed;
};
constexpr GemmShape kGemmShapes[kShapes] = {
    {2, 4, {2.80f, 2.14f, 1.80f}, {}, {2.11f, 1.42f, 1.20f}, 2.91f},
    {2, 2, {1.49f, 1.21f, 1.03f}, {}, {1.36f, 1.09f, 0.94f}, 1.70f},
    {1, 4, {2.06f, 1.42f, 1.13f}, {}, {1.77f, 1.20f, 0.95f}, 3.15f},
    {1, 2, {1.26f, 0.89f, 0.72f}, {0.0f, 1.30f, 1.05f}, {1.28f, 0.98f, 0.79f}, 1.38f},
    {1, 1, {0.92f, 0.66f, 0.56f}, {1.22f, 0.95f, 0.78f}, {1.10f, 0.85f, 0.72f}, 0.38f}};
// Workgroups of shape v on one compute unit: two of the narrower 64-row ones.
constexpr int workgroups_per_cu(int v, int log2_ge) {
  const GemmShape& t = kGemmShapes[v];
  return t.wm == 1 && (t.wn == 1 || (t.wn == 2 && log2_ge > 5)) ? 2 : 1;
}
static_assert(2 * i4_gemm_lds_bytes<1, 4, 1, 5>() <= 160 * 1024 && 2 * i4_gemm_lds_bytes<1, 4, 2, 6>() <= 160 * 1024 &&
              2 * i4_gemm_lds_bytes<1, 4, 2, 5>() > 160 * 1024 && 2 * i4_gemm_lds_bytes<1, 4, 4, 7>() > 160 * 1024,
              "workgroups_per_cu");
double gemm_estimate_us(const I4Args& p, int v, int log2_ge, int64_t tiles, int spans, int slices, int cus) {
  const GemmShape& t = kGemmShapes[v];
  const int64_t slice_spans = ceil_div((int64_t)spans, (int64_t)slices);
  slices = (int)ceil_div((int64_t)spans, slice_spans);                     // (as launched)
  const int64_t blocks = tiles * slices, slots = (int64_t)workgroups_per_cu(v, log2_ge) * cus;
  const int64_t before = ceil_div(blocks, slots) - 1, last = blocks - before * slots;
  const int g = log2_ge - 5;
  const double mb = (double)p.M * p.N * 1e-6;
  return 3.65 + slice_spans * (before * (double)t.round[g] + (last > cus ? t.shared[g] : t.alone[g])) +
         (before + 1) * (double)t.fixed + (slices > 1 ? 2.92 + 1.8 * mb * slices : 0.94 * mb);
}

}  // namespace

int launch_dequant_gemm_i4(const I4Args& p, hipStream_t s) {
  I4GemmArgs a;
  a.x = p.x; a.w = p.w; a.scale = p.scale; a.zp = (const uint8_t*)p.zp; a.out = p.out;
  a.partial = nullptr;
  a.M = p.M; a.N = p.N; a.K = p.K; a.G = p.G;
  a.spans = p.K / 128;
  a.w_bytes = p.w_bytes;
  const int log2_ge = p.log2_gs < 7 ? p.log2_gs : 7;
  a.group_shift = p.log2_gs - log2_ge;
  if ((int64_t)p.M * p.K * 2 >= (1ll << 31) || (int64_t)p.N * p.G * 2 >= (1ll << 31)) return IREE_AMD_UK_STATUS_NOT_FOUND;
  const int cus = device_cu_count();
  int best = -1, slices = 1;
  auto choose = [&](int max_slices) {
    best = -1;
    double best_us = 0;
    for (int v = 0; v < kShapes; ++v) {
      const int64_t tiles = ceil_div((int64_t)p.M, (int64_t)kGemmShapes[v].wm * 64) *
                            ceil_div((int64_t)p.N, (int64_t)kGemmShapes[v].wn * 64);
      if (tiles > 0x7FFFFFFF) continue;
      for (int n = 1; n <= max_slices; ++n) {
        if (n > 1 && a.spans / n < 4) break;
        const double us = gemm_estimate_us(p, v, log2_ge, tiles, a.spans, n, cus);
        if (best < 0 || us < best_us) { best = v; slices = n; best_us = us; }
      }
    }
    if (best < 0) return;
    a.slice_spans = (int)ceil_div(a.spans, slices);
    slices = (int)ceil_div(a.spans, a.slice_spans);
  };
  choose(8);
  if (best < 0) return IREE_AMD_UK_STATUS_NOT_FOUND;
  // A call being captured takes no scratch memory where the kernels for fewer
  // rows need none (K up to 4096, and what only this kernel serves): it need not
  // have been made before, and the graph may be replayed beside others.
  const bool may_split = slices > 1 && ((p.K > 4096 && p.K % 256 == 0) || !scratch_under_capture(s));
  ScratchLease lease(s, may_split ? (size_t)slices * p.M * p.N * 4 : 0);
  a.partial = (float*)lease.ptr();
  if (slices > 1 && !a.partial) choose(1);
  a.tiles_m = (int)ceil_div(p.M, kGemmShapes[best].wm * 64);
  a.tiles_n = (int)ceil_div(p.N, kGemmShapes[best].wn * 64);
  int st;
  switch (best) {
    case 0: st = launch_gemm_shape<2, 4>(a, log2_ge, slices, s); break;
    case 1: st = launch_gemm_shape<2, 2>(a, log2_ge, slices, s); break;
    case 2: st = launch_gemm_shape<1, 4>(a, log2_ge, slices, s); break;
    case 3: st = launch_gemm_shape<1, 2>(a, log2_ge, slices, s); break;
    default: st = launch_gemm_shape<1, 1>(a, log2_ge, slices, s); break;
  }
  if (st || slices == 1) return st;
  KSplitReduceArgs r;
  r.partials = a.partial;
  r.slices = slices;
  r.M = 1; r.N = 1;
  r.flat_elems = (int64_t)p.M * p.N;
  r.out = p.out;
  r.out_stride_bytes = 0;
  r.accumulate = 0;
  r.row_major_out = 0; r.out_rows = r.out_cols = 0;
  r.out_scale = 1.0f;
  r.acc_is_float = 1;
  r.out_kind = 1;   // f16
  return launch_ksplit_reduce(r, s);
}

}  // namespace uk
