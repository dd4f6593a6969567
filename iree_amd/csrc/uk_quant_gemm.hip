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
// A workgroup owns 128 or 64 rows x 256 columns, or 64 x 128: 8 or 4 waves side by
// side, each 32 of the columns and all of the rows, so that every weight is
// dequantised by one wave only, in the registers that feed the matrix cores (12
// vector instructions per 8 weights; adding a scaled group sum is one FMA per
// register). Vector and matrix instructions of a SIMD share its issue port, and how
// far they overlap depends on the instruction: with two waves, a
// v_mfma_f32_16x16x32_f16 and four vector instructions take 27.7 cycles (alone 16.8
// and 4.2 each), a v_mfma_f32_32x32x16_f16 and eight, twice that work, 41.5: hence
// the latter. For 128 x 256 and a span of 128 k a wave issues 32 of them and 176
// vector instructions, and reads its 32 fragments of the activations from LDS: about
// 2100 cycles of each of the three pipes of a compute unit, which take 3050 together.
// (Two rows of waves that each dequantise the weights, on the 16-row instruction, 277
// vector instructions: 4260.) Two waves per SIMD throughout: a single one issues an
// instruction only every 6 cycles or so (four waves of 128 x 64 each, with as few
// vector instructions per MFMA: 4050).
// Measured at 14336 columns, K = 4096, groups of 128, same box: 96 / 128 / 256 / 512 rows
// 32.4 / 33.0 / 44.4 / 72.5 -> 28.2 / 28.5 / 41.2 / 66.9 us, groups of 64 512 rows 79.5 -> 70.6;
// over 70 problems of 60 to 512 rows 5 % on average, 15 % at most. At 512 rows the clock is
// down at 1.9 GHz under the power limit.
// K goes in spans of 128:
//   * weights: a 32-column x 128-k tile is two 16-byte loads per lane (the tiled
//     layout's 2 KiB), straight to registers, two spans ahead;
//   * activations: the rows' 256 bytes of the span go to LDS with direct loads
//     (16 adjacent lanes fetch one row: whole cache lines), into a ring of 4
//     spans (3 where LDS is short), each row's 16-byte chunks in an order of its own
//     so that the fragment reads (16 rows, one chunk column) touch every bank once;
//   * scales and zero points of 4 groups at a time: 16 bytes of each column,
//     straight to LDS four spans ahead, and from there, three spans ahead, as the
//     f32 scale and the pair of f16 offsets that the dequantisation adds.
// A lane holds one column of a block: its scale is one LDS read per span and group.
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

typedef float floatx16 __attribute__((ext_vector_type(16)));
constexpr int kParamGroups = 4;   // groups of scales and offsets per refill
// refills kept: a refill is written three spans before its first use
constexpr int param_bufs(int log2_ge) { return log2_ge == 5 ? 4 : log2_ge == 6 ? 3 : 2; }

template <int WC, int kLog2Ge>
constexpr int i4_gemm_param_bytes() { return 32 * WC * (32 + param_bufs(kLog2Ge) * kParamGroups * 8); }
// spans of activations in LDS: 4, or what fits
template <int WC, int XB, int kLog2Ge>
constexpr int i4_gemm_ring() {
  return 4 * XB * 8192 + i4_gemm_param_bytes<WC, kLog2Ge>() <= 160 * 1024 ? 4 : 3;
}
template <int WC, int XB, int kLog2Ge>
constexpr int i4_gemm_lds_bytes() {
  return i4_gemm_ring<WC, XB, kLog2Ge>() * XB * 8192 + i4_gemm_param_bytes<WC, kLog2Ge>();
}

template <int N>
__device__ __forceinline__ void gemm_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Every load and LDS access of the wave (vmcnt and lgkmcnt 0, expcnt not waited for): as the
// builtin, which becomes one instruction with the wait of the barrier behind it.
__device__ __forceinline__ void gemm_wait_all() { __builtin_amdgcn_s_waitcnt(0x0070); }

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

// (workgroup ids go round-robin over the 8 XCDs: XCD x takes the x-th
// contiguous slice of the tiles, row tiles of one column tile together, so
// that they share its weights in one L2)
__device__ __forceinline__ void i4_gemm_tile(const I4GemmArgs& a, int* tm, int* tn) {
  const int total = a.tiles_m * a.tiles_n, per = total / 8, rem = total % 8;
  const int xcd = (int)blockIdx.x % 8, idx = (int)blockIdx.x / 8;
  const int logical = xcd * per + (xcd < rem ? xcd : rem) + idx;
  *tn = logical / a.tiles_m;
  *tm = logical - *tn * a.tiles_m;
}

// Scales and offsets of a workgroup's BN columns: one column per thread (the first BN).
// The 4 groups of a column are fetched as the 16 bytes that begin at the
// 4-byte boundary before them (or end with the array): a column's groups
// start anywhere. The arrays are whole 32 columns, i.e. whole 16 bytes.
template <int BN, int kWaveCount, int kLog2Ge>
struct I4GemmParams {
  static constexpr int kGroupsPerSpan = 128 >> kLog2Ge;
  static constexpr int kChunkSpans = kParamGroups / kGroupsPerSpan;
  static constexpr int kParamBufs = param_bufs(kLog2Ge);
  const I4GemmArgs& a;
  int n, wave, col;
  bool active;
  char* lds_raw;            // of a wave of 64 columns: their scales, 16 bytes each, zero points alike
  char* lds_spare;          // 64 BN bytes that are free before the first step
  float* lds_scale;         // [kParamBufs][4][BN]
  uint32_t* lds_off;
  uint32_t s_bytes, z_bytes;

  __device__ __forceinline__ I4GemmParams(const I4GemmArgs& args, int n_base, int w, char* raw, char* spare, float* scale,
                                          uint32_t* off)
      : a(args), wave(w), lds_raw(raw + w * 2048), lds_spare(spare + w * 2048), lds_scale(scale), lds_off(off) {
    col = (int)threadIdx.x;
    active = BN >= 64 * kWaveCount || wave < BN / 64;
    n = n_base + col;
    n = n < a.N ? n : a.N - 1;
    s_bytes = (uint32_t)a.N * (uint32_t)a.G * 2u;
    z_bytes = s_bytes / 4u;
  }
  __device__ __forceinline__ uint32_t group_of(int chunk, int i) const {    // index of a group in the arrays
    int g = (chunk * kParamGroups + i) >> a.group_shift;
    g = g < a.G ? g : a.G - 1;
    return (uint32_t)n * (uint32_t)a.G + (uint32_t)g;
  }
  __device__ __forceinline__ static uint32_t window(uint32_t at, uint32_t bytes) {
    at &= ~3u;
    return at < bytes - 16u ? at : bytes - 16u;
  }
  __device__ __forceinline__ void request(int chunk) const { request(chunk, lds_raw); }
  __device__ __forceinline__ void convert(int chunk) const { convert(chunk, lds_raw); }
  __device__ __forceinline__ void request(int chunk, char* raw) const {
    if (!active) return;
    const __amdgpu_buffer_rsrc_t s_src = __builtin_amdgcn_make_buffer_rsrc((void*)a.scale, 0, s_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t z_src = __builtin_amdgcn_make_buffer_rsrc((void*)a.zp, 0, z_bytes, 0x00020000);
    const uint32_t at = group_of(chunk, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        s_src, (__attribute__((address_space(3))) void*)raw, 16, window(at * 2, s_bytes), 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        z_src, (__attribute__((address_space(3))) void*)(raw + 1024), 16, window(at / 2, z_bytes), 0, 0, 0);
  }
  __device__ __forceinline__ void convert(int chunk, const char* raw) const {
    if (!active) return;
    const uint32_t first = group_of(chunk, 0);
    const char* sw = raw + (col & 63) * 16 - window(first * 2, s_bytes);
    const char* zw = raw + 1024 + (col & 63) * 16 - window(first / 2, z_bytes);
    // (all of them read before the first is written: one LDS latency instead of four)
    uint16_t sv[kParamGroups];
    uint32_t zv[kParamGroups];
#pragma unroll
    for (int i = 0; i < kParamGroups; ++i) {
      const uint32_t at = group_of(chunk, i);
      sv[i] = *(const uint16_t*)(sw + at * 2);
      zv[i] = (*(const uint8_t*)(zw + at / 2) >> (4 * (at & 1))) & 15u;
    }
#pragma unroll
    for (int i = 0; i < kParamGroups; ++i) {
      const int to = ((chunk % kParamBufs) * kParamGroups + i) * BN + col;
      lds_scale[to] = __half2float(__ushort_as_half(sv[i]));
      lds_off[to] = 0xD400E400u | zv[i] | (zv[i] << 20);       // -(1024 + zp), -(64 + zp)
    }
  }
  // The first three spans from s0: requested together ...
  __device__ __forceinline__ void request_first(int s0) const {
    const int first = s0 / kChunkSpans, last = (s0 + 2) / kChunkSpans;
    request(first);
    for (int chunk = first + 1; chunk <= last; ++chunk) request(chunk, lds_spare + (chunk - first - 1) * (BN * 32));
  }
  // ... and once they have landed, converted; then what the step before the first would
  // have requested.
  __device__ __forceinline__ void convert_first(int s0) const {
    const int first = s0 / kChunkSpans, last = (s0 + 2) / kChunkSpans;
    convert(first);
    for (int chunk = first + 1; chunk <= last; ++chunk) convert(chunk, lds_spare + (chunk - first - 1) * (BN * 32));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (a lane's own 16 bytes: read before they are replaced)
    if ((s0 + 3) % kChunkSpans == 0) request((s0 + 3) / kChunkSpans);
  }
  // of group e (absolute), column c of the workgroup
  __device__ __forceinline__ static int at(int e, int c) {
    return (((e / kParamGroups) % kParamBufs) * kParamGroups + e % kParamGroups) * BN + c;
  }
  __device__ __forceinline__ float scale(int e, int c) const { return lds_scale[at(e, c)]; }
  __device__ __forceinline__ half2v offsets(int e, int c) const {
    union { uint32_t u; half2v h; } o;
    o.u = lds_off[at(e, c)];
    return o.h;
  }
};

// WC waves side by side, each 32 of the columns and all 32 XB rows. kLog2Ge: log2 of the k that one scale covers at a time (groups above 128: 128).
template <int WC, int XB, int kLog2Ge>
__device__ __forceinline__ void dequant_matmul_i4_gemm_body(const I4GemmArgs& a) {
  constexpr int BM = XB * 32, BN = 32 * WC, kWaveCount = WC;
  constexpr int kStageBytes = BM * 256;                     // one span of the rows
  constexpr int kXLoads = BM / 4 / kWaveCount;              // 1 KiB loads (4 rows) per wave and span
  constexpr int kWLoads = 2;                                // weights: loads per wave and span
  constexpr int kGroupsPerSpan = 128 >> kLog2Ge;            // 1, 2, 4
  constexpr int kStepsPerGroup = 8 / kGroupsPerSpan;        // MFMA K-steps per group
  constexpr int kChunkSpans = kParamGroups / kGroupsPerSpan;
  constexpr int kParamBufs = param_bufs(kLog2Ge);
  constexpr int kRing = i4_gemm_ring<WC, XB, kLog2Ge>();
  static_assert(XB % 2 == 0, "row blocks take turns in two sets of registers");
  static_assert(BM / 4 % kWaveCount == 0, "every wave loads whole row quads");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* const lds_raw = lds + kRing * kStageBytes;                                  // scales and zero points as fetched, 32 BN bytes
  float* const lds_scale = (float*)(lds_raw + 32 * BN);                             // [kParamBufs][4][BN]
  uint32_t* const lds_off = (uint32_t*)(lds_scale + kParamBufs * kParamGroups * BN);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, l32 = lane & 31, kh = lane >> 5;
  int tm, tn;
  i4_gemm_tile(a, &tm, &tn);
  const int m_base = tm * BM, n_base = tn * BN;
  const int s0 = (int)blockIdx.y * a.slice_spans;
  const int T = a.spans - s0 < a.slice_spans ? a.spans - s0 : a.slice_spans;

  // ---- activations: this wave's rows [wave * BM / kWaveCount, ...), 4 per load ----
  // (a row's chunk c of 8 k lies at place c ^ (row % 16): the reads of 16 rows touch
  // every bank once)
  const __amdgpu_buffer_rsrc_t x_src =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (uint32_t)a.M * (uint32_t)a.K * 2u, 0x00020000);
  uint32_t x_off[kXLoads];
#pragma unroll
  for (int j = 0; j < kXLoads; ++j) {
    const int r = (wave * kXLoads + j) * 4 + (lane >> 4);    // row of the tile
    int row = m_base + r;
    row = row < a.M ? row : a.M - 1;                         // (rows past the end: loaded, not stored)
    x_off[j] = (uint32_t)row * (uint32_t)a.K * 2u + (uint32_t)((l16 ^ r) & 15) * 16u;
  }
  // (past the last span it is loaded again, into a slot nobody reads any more:
  // the number of loads in flight, which the waits count, stays the same)
  auto issue_x = [&](int span, int slot, int j) {
    const uint32_t at = (uint32_t)(s0 + (span < T ? span : T - 1)) * 256u;
    char* base = lds + slot * kStageBytes + wave * (kXLoads * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(x_src, (__attribute__((address_space(3))) void*)(base + j * 1024), 16,
                                             x_off[j], at, 0, 0);
  };
  // K-step 2 q + j of a span takes chunk 4 q + j (lanes 0..31) and 4 q + 2 + j (lanes
  // 32..63): the k of dword q of the weights' pieces 2 kh + j of 16 bytes.
  // Fragment (block x, K-step t): row 32 x + l32, that chunk.
  const uint32_t read_lane = (uint32_t)l32 * 256u + (uint32_t)((2 * kh) ^ l16) * 16u;
  half8 xf[2][8];         // of this row block and the next
  auto read_block = [&](int slot, int x) {
    const uint32_t at = (uint32_t)(slot * kStageBytes) + read_lane;
#pragma unroll
    for (int t = 0; t < 8; ++t)
      xf[x % 2][t] = *(const half8*)(lds + (at ^ (uint32_t)(t / 2 * 64 + t % 2 * 16)) + x * 8192);
  };

  // ---- weights: this wave's tile of 32 columns, two 16-byte pieces a lane --------
  const __amdgpu_buffer_rsrc_t w_src = __builtin_amdgcn_make_buffer_rsrc((void*)a.w, 0, a.w_bytes, 0x00020000);
  const uint32_t w_lane = (uint32_t)l32 * 64u + (uint32_t)kh * 32u;
  uint32_t w_base;
  {
    int cb = n_base / 32 + wave;
    cb = cb * 32 < a.N ? cb : a.N / 32 - 1;
    w_base = ((uint32_t)cb * (uint32_t)a.spans + (uint32_t)s0) * 2048u;
  }
  u32x4 raw[2][2];            // pieces of span s in raw[s % 2]
  auto load_w = [&](int span, u32x4 (&dst)[2]) {
    const uint32_t at = (uint32_t)(span < T ? span : T - 1) * 2048u;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(w_src, w_lane | (j * 16u), w_base + at, 0);
      dst[j] = u32x4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
    }
  };
  auto word_of = [](const u32x4 (&r)[2], int t) -> uint32_t { return r[t % 2][t / 2]; };

  // ---- scales and offsets ------------------------------------------------------
  const I4GemmParams<BN, kWaveCount, kLog2Ge> params(a, n_base, wave, lds_raw, lds + (kRing - 1) * kStageBytes, lds_scale,
                                                          lds_off);
  const int p_lane = wave * 32 + l32;
  uint32_t mask;
  asm volatile("v_mov_b32 %0, 0x00f0000f" : "=v"(mask));

  const floatx16 zeros = {};
  floatx16 acc[XB];
#pragma unroll
  for (int x = 0; x < XB; ++x) acc[x] = zeros;
  half8 wf[2][8];         // weight fragments of this span and the next

  static_assert(64 * BN <= kStageBytes, "the last slot of the ring holds two refills");
  params.request_first(s0);
  __builtin_amdgcn_sched_barrier(0);
  load_w(0, raw[0]);
  load_w(1, raw[1]);
#pragma unroll
  for (int d = 0; d < kRing - 1; ++d)
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) issue_x(d, d, j);
  __builtin_amdgcn_sched_barrier(0);
  gemm_wait_vmcnt<2 * kWLoads + (kRing - 1) * kXLoads>();
  params.convert_first(s0);
  // (the first span's rows come from every wave; and step 0 counts on all of this: its
  // wait for span 1 allows for a step's loads before it, its wait for a refill, which may
  // be the last thing requested here, for a step's activations behind it)
  gemm_wait_all();
  __syncthreads();
  read_block(0, 0);
#pragma unroll
  for (int t = 0; t < 8; ++t)
    wf[0][t] = dequant_in_order(word_of(raw[0], t), mask, params.offsets(s0 * kGroupsPerSpan + t / kStepsPerGroup, p_lane));

  // One span. Its work is cut into units of one row block times one group of k, each
  // with its share of the dequantisation of the next span behind its MFMAs; a
  // unit's sums are scaled and added when its last MFMA is done, under the other
  // wave's MFMAs. The fences keep the compiler from moving work between units (it would
  // otherwise hold the sums of many of them).
  auto span_step = [&](auto parity, int i, int slot) {
    constexpr int P = decltype(parity)::value;
    const int free_slot = slot == 0 ? kRing - 1 : slot - 1;     // (the span before: read by every wave)
    const int next_slot = slot + 1 == kRing ? 0 : slot + 1;
    const int e0 = (s0 + i) * kGroupsPerSpan;
    half8 (&f)[8] = wf[P];
    half8 (&fn)[8] = wf[P ^ 1];
    float sc[kGroupsPerSpan];
    half2v off[kGroupsPerSpan];
#pragma unroll
    for (int g = 0; g < kGroupsPerSpan; ++g) {
      sc[g] = params.scale(e0 + g, p_lane);
      off[g] = params.offsets(e0 + kGroupsPerSpan + g, p_lane);
    }
    // (this span's words have been used: the pieces of the span after the next)
    load_w(i + 2, raw[P]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < XB; ++x) {
      if (x == 1) {
        // The NEXT span of activations was requested kRing - 2 steps ago: it has
        // landed once only what was requested since is outstanding (the last step
        // and this one's weights, or those alone). The barrier publishes it and
        // frees the slot of the span before, whose fragments every wave has
        // multiplied. It comes behind the first row block so that the matrix pipes
        // have work while the waves meet.
        gemm_wait_vmcnt<kRing == 4 ? kXLoads + 2 * kWLoads : kWLoads>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        // (requested by the step before, ahead of its activations; published by the
        // next step's barrier, and the step behind that one is the first to read it)
        if ((s0 + i + 3) % kChunkSpans == 0) {
          gemm_wait_vmcnt<kXLoads + kWLoads>();
          params.convert((s0 + i + 3) / kChunkSpans);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        if ((s0 + i + 4) % kChunkSpans == 0) params.request((s0 + i + 4) / kChunkSpans);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (x >= 1) {
#pragma unroll
        for (int j = (x - 1) * kXLoads / (XB - 1); j < x * kXLoads / (XB - 1); ++j) issue_x(i + kRing - 1, free_slot, j);
      }
      // (the next row block's fragments, of the next span behind the last)
      if (x + 1 < XB) read_block(slot, x + 1);
      else read_block(next_slot, 0);
#pragma unroll
      for (int g = 0; g < kGroupsPerSpan; ++g) {
        constexpr int kUnits = XB * kGroupsPerSpan;
        const int unit = x * kGroupsPerSpan + g;
        floatx16 t = zeros;
#pragma unroll
        for (int k = g * kStepsPerGroup; k < (g + 1) * kStepsPerGroup; ++k)
          t = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[x % 2][k], f[k], t, 0, 0, 0);
#pragma unroll
        for (int k = unit * 8 / kUnits; k < (unit + 1) * 8 / kUnits; ++k) {
          fn[k] = dequant_in_order(word_of(raw[P ^ 1], k), mask, off[k / kStepsPerGroup]);
          asm volatile("" : "+v"(fn[k]));
        }
#pragma unroll
        for (int m = 0; m < kStepsPerGroup; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (96 / kUnits + kStepsPerGroup - 1) / kStepsPerGroup, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[x][v] = __builtin_fmaf(t[v], sc[g], acc[x][v]);
        asm volatile("" : "+v"(acc[x]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  int slot = 0;
  int i = 0;
  // (the two spans of weight fragments and words take turns)
  for (; i + 2 <= T; i += 2) {
    span_step(std::integral_constant<int, 0>(), i, slot);
    slot = slot + 1 == kRing ? 0 : slot + 1;
    span_step(std::integral_constant<int, 1>(), i + 1, slot);
    slot = slot + 1 == kRing ? 0 : slot + 1;
  }
  if (i < T) span_step(std::integral_constant<int, 0>(), i, slot);
  gemm_wait_vmcnt<0>();      // (loads into LDS must not outlive the workgroup)

  // Register v of block x: row 32 x + 8 (v / 4) + 4 kh + v % 4, column l32.
  const int n = n_base + wave * 32 + l32;
#pragma unroll
  for (int x = 0; x < XB; ++x)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = m_base + x * 32 + 8 * (v / 4) + 4 * kh + v % 4;
      if (m >= a.M || n >= a.N) continue;
      const int64_t at = (int64_t)m * a.N + n;
      if (a.partial) a.partial[(int64_t)blockIdx.y * a.M * a.N + at] = acc[x][v];
      else ((_Float16*)a.out)[at] = (_Float16)acc[x][v];
    }
}

// 64 x 64 on 16-row blocks: four waves side by side, each 16 of the columns and all of
// the rows. (On 32-row blocks a wave would own 32 columns, and two waves of a compute
// unit's matrix pipes would have none of such a tile.)
template <int kLog2Ge>
__device__ __forceinline__ void dequant_matmul_i4_gemm_small_body(const I4GemmArgs& a) {
  constexpr int BM = 64, BN = 64, MB = 4, kWaveCount = 4;
  constexpr int kStageBytes = BM * 256;                     // one span of the rows
  constexpr int kXLoads = BM / 4 / kWaveCount;              // 1 KiB loads (4 rows) per wave and span
  constexpr int kGroupsPerSpan = 128 >> kLog2Ge;            // 1, 2, 4
  constexpr int kQPerGroup = 4 / kGroupsPerSpan;            // MFMA K-steps per group
  constexpr int kChunkSpans = kParamGroups / kGroupsPerSpan;
  constexpr int kParamBufs = param_bufs(kLog2Ge);
  constexpr int kRing = i4_gemm_ring<2, 2, kLog2Ge>();
  static_assert(kRing == 4, "the waits count loads of a ring of 4");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* const lds_raw = lds + kRing * kStageBytes;                                  // scales and zero points as fetched, 32 BN bytes
  float* const lds_scale = (float*)(lds_raw + 32 * BN);                             // [kParamBufs][4][BN]
  uint32_t* const lds_off = (uint32_t*)(lds_scale + kParamBufs * kParamGroups * BN);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kc = lane >> 4;
  int tm, tn;
  i4_gemm_tile(a, &tm, &tn);
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
    return *(const half8*)(lds + slot * kStageBytes + read_off[q] + x * 4096);
  };

  // ---- weights: this wave's slab of 16 columns --------------------------------
  const __amdgpu_buffer_rsrc_t w_src = __builtin_amdgcn_make_buffer_rsrc((void*)a.w, 0, a.w_bytes, 0x00020000);
  const uint32_t w_lane = (uint32_t)l16 * 64u + (uint32_t)kc * 16u;
  uint32_t w_base;
  {
    int cb = n_base / 16 + wave;
    cb = cb * 16 < a.N ? cb : a.N / 16 - 1;
    w_base = ((uint32_t)(cb >> 1) * (uint32_t)a.spans + (uint32_t)s0) * 2048u + (uint32_t)(cb & 1) * 1024u;
  }
  u32x4 raw[2];               // slab of span s in raw[s % 2]
  auto load_w = [&](int span, u32x4& dst) {
    const uint32_t at = (uint32_t)(span < T ? span : T - 1) * 2048u;
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(w_src, w_lane, w_base + at, 0);
    dst = u32x4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
  };

  const I4GemmParams<BN, kWaveCount, kLog2Ge> params(a, n_base, wave, lds_raw, lds + (kRing - 1) * kStageBytes, lds_scale,
                                                          lds_off);
  const int p_lane = wave * 16 + l16;
  uint32_t mask;
  asm volatile("v_mov_b32 %0, 0x00f0000f" : "=v"(mask));

  floatx4 acc[MB];
#pragma unroll
  for (int x = 0; x < MB; ++x) acc[x] = floatx4{0.f, 0.f, 0.f, 0.f};

  half8 xf[MB][4];        // activation fragments of the span
  half8 wf[2][4];         // weight fragments of this span and the next
  static_assert(64 * BN <= kStageBytes, "the last slot of the ring holds two refills");
  params.request_first(s0);
  __builtin_amdgcn_sched_barrier(0);
  load_w(0, raw[0]);
  load_w(1, raw[1]);
#pragma unroll
  for (int d = 0; d < kRing - 1; ++d)
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) issue_x(d, d, j);
  __builtin_amdgcn_sched_barrier(0);
  gemm_wait_vmcnt<2 + (kRing - 1) * kXLoads>();
  params.convert_first(s0);
  // (as above: the first span's rows come from every wave, and the waits of step 0 allow
  // for loads that only later steps have behind them)
  gemm_wait_all();
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
    wf[0][q] = dequant_in_order(raw[0][q], mask, params.offsets(s0 * kGroupsPerSpan + q / kQPerGroup, p_lane));

  // One span, in two regions of two row blocks each (8 MFMAs), which carry the same
  // share of everything else, issued behind their MFMAs: the FMAs that add the sums
  // of the region before, the dequantisation of the next span, loads. The fences keep
  // the compiler from moving work between regions (it would otherwise hold the
  // sums of many of them).
  floatx4 part[kGroupsPerSpan][2];     // of the region before
  float part_scale[kGroupsPerSpan];
#pragma unroll
  for (int g = 0; g < kGroupsPerSpan; ++g) {
    part[g][0] = part[g][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    part_scale[g] = 0.f;
  }
  auto add_part = [&](int x) {
#pragma unroll
    for (int g = 0; g < kGroupsPerSpan; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[x + h][v] = __builtin_fmaf(part[g][h][v], part_scale[g], acc[x + h][v]);
  };
  auto span_step = [&](auto parity, int i, int slot) {
    constexpr int P = decltype(parity)::value;
    const int free_slot = slot == 0 ? kRing - 1 : slot - 1;     // (the span before: read by every wave)
    const int next_slot = slot + 1 == kRing ? 0 : slot + 1;
    // The NEXT span of activations was requested two steps ago: it has
    // landed once only the loads of the last step are outstanding. The barrier
    // publishes it and frees the slot of the span before.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    gemm_wait_vmcnt<kXLoads + 1>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int e0 = (s0 + i) * kGroupsPerSpan;
    // (requested by the step before, ahead of its weights and activations)
    if ((s0 + i + 3) % kChunkSpans == 0) {
      params.convert((s0 + i + 3) / kChunkSpans);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if ((s0 + i + 4) % kChunkSpans == 0) params.request((s0 + i + 4) / kChunkSpans);
    __builtin_amdgcn_sched_barrier(0);
    float sc[kGroupsPerSpan];
    half2v off[kGroupsPerSpan];
#pragma unroll
    for (int g = 0; g < kGroupsPerSpan; ++g) {
      sc[g] = params.scale(e0 + g, p_lane);
      off[g] = params.offsets(e0 + kGroupsPerSpan + g, p_lane);
    }
    // (this span's words have been used: the slab of the span after the next)
    load_w(i + 2, raw[P]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int xp = 0; xp < 2; ++xp) {
      if (xp == 0) {
#pragma unroll
        for (int j = 0; j < kXLoads; ++j) issue_x(i + kRing - 1, free_slot, j);
      }
      // Activation fragments: the second pair of row blocks of this span while
      // its first pair is multiplied, then the first pair of the next span.
      if (xp == 0) read_pair(slot, 1);
      else read_pair(next_slot, 0);
      floatx4 t[kGroupsPerSpan][2];
#pragma unroll
      for (int g = 0; g < kGroupsPerSpan; ++g) {
        t[g][0] = t[g][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = g * kQPerGroup; q < (g + 1) * kQPerGroup; ++q)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            t[g][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[2 * xp + h][q], wf[P][q], t[g][h], 0, 0, 0);
      }
      add_part(2 - 2 * xp);     // (zeros before the first)
#pragma unroll
      for (int q = 2 * xp; q < 2 * xp + 2; ++q) wf[P ^ 1][q] = dequant_in_order(raw[P ^ 1][q], mask, off[q / kQPerGroup]);
#pragma unroll
      for (int g = 0; g < kGroupsPerSpan; ++g) {
        part[g][0] = t[g][0];
        part[g][1] = t[g][1];
        part_scale[g] = sc[g];
      }
      // (8 MFMAs, each with its share of the vector instructions behind it)
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (8 * kGroupsPerSpan + 24 + 7) / 8, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  int slot = 0;
  int i = 0;
  // (the two spans of weight fragments and words take turns)
  for (; i + 2 <= T; i += 2) {
    span_step(std::integral_constant<int, 0>(), i, slot);
    slot = slot + 1 == kRing ? 0 : slot + 1;
    span_step(std::integral_constant<int, 1>(), i + 1, slot);
    slot = slot + 1 == kRing ? 0 : slot + 1;
  }
  if (i < T) span_step(std::integral_constant<int, 0>(), i, slot);
  add_part(2);
  gemm_wait_vmcnt<0>();      // (loads into LDS must not outlive the workgroup)

  // Register v of block x: row 16 x + 4 kc + v, column l16.
  const int n = n_base + wave * 16 + l16;
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m_base + x * 16 + kc * 4 + v;
      if (m >= a.M || n >= a.N) continue;
      const int64_t at = (int64_t)m * a.N + n;
      if (a.partial) a.partial[(int64_t)blockIdx.y * a.M * a.N + at] = acc[x][v];
      else ((_Float16*)a.out)[at] = (_Float16)acc[x][v];
    }
}

template <int WC, int XB, int kLog2Ge>
__global__ __launch_bounds__(64 * WC, 2) void dequant_matmul_i4_gemm_kernel(I4GemmArgs a) {
  dequant_matmul_i4_gemm_body<WC, XB, kLog2Ge>(a);
}
template <int kLog2Ge>
__global__ __launch_bounds__(256, 2) void dequant_matmul_i4_gemm_small_kernel(I4GemmArgs a) {
  dequant_matmul_i4_gemm_small_body<kLog2Ge>(a);
}

// WC = 2: the 64 x 64 kernel.
template <int WC, int XB, int kLog2Ge>
int launch_gemm_instance(const I4GemmArgs& a, int slices, hipStream_t s) {
  constexpr bool kSmall = WC == 2;
  constexpr int kLds = i4_gemm_lds_bytes<WC, XB, kLog2Ge>();
  static_assert(kLds <= 160 * 1024, "LDS ring exceeds 160 KiB");
  void (*kernel)(I4GemmArgs);
  if constexpr (kSmall) kernel = dequant_matmul_i4_gemm_small_kernel<kLog2Ge>;
  else kernel = dequant_matmul_i4_gemm_kernel<WC, XB, kLog2Ge>;
  static PerDeviceOnce attr_set_on;
  int dev = 0;
  UK_RETURN_IF_HIP(hipGetDevice(&dev));
  if (!attr_set_on.done(dev)) {
    UK_RETURN_IF_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    attr_set_on.mark(dev);
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)slices), dim3(kSmall ? 256 : 64 * WC), kLds, s, a);
  return check_hip(hipGetLastError(), "dequant_matmul_i4 gemm launch");
}

template <int WC, int XB>
int launch_gemm_shape(const I4GemmArgs& a, int log2_ge, int slices, hipStream_t s) {
  switch (log2_ge) {
    case 5:
      if constexpr (WC == 4) return IREE_AMD_UK_STATUS_NOT_FOUND;     // (serves_groups)
      else return launch_gemm_instance<WC, XB, 5>(a, slices, s);
    case 6: return launch_gemm_instance<WC, XB, 6>(a, slices, s);
    default: return launch_gemm_instance<WC, XB, 7>(a, slices, s);
  }
}

// Estimated time in microseconds on shape v with K in `slices`, by group size (32,
// 64, 128 and more). A span of 128 k of a workgroup takes `alone` in the last round
// when that gives a compute unit one workgroup at most, `shared` when it gives two
// to some, and `round` in the rounds before, which overlap with the next; `fixed`
// is what a workgroup needs before its first and after its last span. Then the
// result, and for a split the partial sums and the launch that adds them. Fitted to
// every shape and 1 to 8 slices on 600 problems (65 to 700 rows, 512 to 14336
// columns, K 512 to 14336, groups of 32 to 256) and 420 of a wider range; fitted to
// the former alone it is 2.9 % off on average on the latter, where what it picks is
// 0.7 % slower than the best on average, 4.1 % in the 95th percentile and 26 % at most.
struct GemmShape {
  int rows, cols;
  float alone[3], shared[3], round[3], fixed;
};
constexpr int kShapes = 4;
constexpr GemmShape kGemmShapes[kShapes] = {
    {64, 64, {0.84f, 0.63f, 0.54f}, {1.20f, 0.92f, 0.77f}, {1.14f, 0.86f, 0.75f}, 0.23f},
    {128, 256, {2.12f, 1.61f, 1.34f}, {}, {1.85f, 1.45f, 1.18f}, 3.57f},
    {64, 256, {1.50f, 1.11f, 0.93f}, {}, {1.46f, 1.09f, 0.94f}, 1.49f},
    {64, 128, {0.0f, 0.86f, 0.70f}, {0.0f, 1.25f, 1.05f}, {0.0f, 1.03f, 0.87f}, 1.10f}};
// (64 x 128 with groups of 32, of which a compute unit takes one workgroup, took 1.26 us a span
// alone and 1.33 in the rounds before the last: 64 x 64, of which it takes two, is never slower)
constexpr bool serves_groups(int v, int log2_ge) { return v != 3 || log2_ge > 5; }
// Workgroups of shape v on one compute unit: two of the smaller ones.
constexpr int workgroups_per_cu(int v) { return v == 0 || v == 3 ? 2 : 1; }
static_assert(2 * i4_gemm_lds_bytes<2, 2, 5>() <= 160 * 1024 && 2 * i4_gemm_lds_bytes<4, 2, 6>() <= 160 * 1024 &&
              2 * i4_gemm_lds_bytes<4, 2, 5>() > 160 * 1024 && 2 * i4_gemm_lds_bytes<8, 2, 7>() > 160 * 1024,
              "workgroups_per_cu");
double gemm_estimate_us(const I4Args& p, int v, int log2_ge, int64_t tiles, int spans, int slices, int cus) {
  const GemmShape& t = kGemmShapes[v];
  const int64_t slice_spans = ceil_div((int64_t)spans, (int64_t)slices);
  slices = (int)ceil_div((int64_t)spans, slice_spans);                     // (as launched)
  const int64_t blocks = tiles * slices, slots = (int64_t)workgroups_per_cu(v) * cus;
  const int64_t before = ceil_div(blocks, slots) - 1, last = blocks - before * slots;
  const int g = log2_ge - 5;
  const double mb = (double)p.M * p.N * 1e-6;
  return 3.72 + slice_spans * (before * (double)t.round[g] + (last > cus ? t.shared[g] : t.alone[g])) +
         (before + 1) * (double)t.fixed + (slices > 1 ? 3.11 + 1.67 * mb * slices : 0.80 * mb);
}

}  // namespace

int launch_dequant_gemm_i4(const I4Args& p, double limit_us, hipStream_t s) {
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
  double best_us = 0;
  auto choose = [&](int max_slices) {
    best = -1;
    for (int v = 0; v < kShapes; ++v) {
      if (!serves_groups(v, log2_ge)) continue;
      const int64_t tiles = ceil_div((int64_t)p.M, (int64_t)kGemmShapes[v].rows) *
                            ceil_div((int64_t)p.N, (int64_t)kGemmShapes[v].cols);
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
  if (best < 0 || (limit_us > 0 && best_us > limit_us)) return IREE_AMD_UK_STATUS_NOT_FOUND;
  // A call being captured takes no scratch memory where the kernels for fewer
  // rows need none (K up to 4096, and what only this kernel serves): it need not
  // have been made before, and the graph may be replayed beside others.
  const bool may_split = slices > 1 && ((p.K > 4096 && p.K % 256 == 0) || !scratch_under_capture(s));
  ScratchLease lease(s, may_split ? (size_t)slices * p.M * p.N * 4 : 0);
  a.partial = (float*)lease.ptr();
  if (slices > 1 && !a.partial) {
    choose(1);
    if (limit_us > 0 && best_us > limit_us) return IREE_AMD_UK_STATUS_NOT_FOUND;
  }
  a.tiles_m = (int)ceil_div(p.M, kGemmShapes[best].rows);
  a.tiles_n = (int)ceil_div(p.N, kGemmShapes[best].cols);
  int st;
  switch (best) {
    case 0: st = launch_gemm_shape<2, 2>(a, log2_ge, slices, s); break;
    case 1: st = launch_gemm_shape<8, 4>(a, log2_ge, slices, s); break;
    case 2: st = launch_gemm_shape<8, 2>(a, log2_ge, slices, s); break;
    default: st = launch_gemm_shape<4, 2>(a, log2_ge, slices, s); break;
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
