// mmt4d of few tiles (uk_mmt4d_wave_split.hip).
#ifndef IREE_AMD_UK_MMT4D_WAVE_SPLIT_H_
#define IREE_AMD_UK_MMT4D_WAVE_SPLIT_H_

#include "uk_common.h"

namespace uk {

// One problem, or `batch` of one shape as planes `*_batch` bytes apart. K comes
// in pieces of 16 bytes (tiles of K0 = 16 / element size).
struct WaveSplitArgs {
  const char* lhs;
  const char* rhs;
  char* out;
  int64_t lhs_batch, rhs_batch, out_batch;
  // piece c of row r at (r / 32) lhs_outer + (r % 32) lhs_row + c lhs_chunk bytes
  // (a row-major matrix, or tiles of up to 32 rows), piece c of column n at
  // (n / 32) rhs_outer + (n % 32) 16 + c 512
  int64_t lhs_outer, rhs_outer;
  int lhs_row, lhs_chunk;
  int rows, outer_cols;        // rows of the left-hand side that exist; columns / 32
  int k_chunks;
  // element (r, n) of the result, r < out_rows and n < out_cols, at
  // (r / 32) out_outer + (r % 32) out_row + (n / 32) out_tile + (n % 32) out_col
  // elements (SiLU form: 32 x 16 tiles of bytes, out_outer bytes per 32 rows)
  int64_t out_outer, out_row, out_tile;
  int out_col, out_rows, out_cols;
  // if not null, where the result goes as 32 x 32 tiles too, padding included, tiles_outer
  // elements per outer row
  char* tiles;
  int64_t tiles_outer;
  int accumulate, silu, batch;
  float gate_scale, up_scale, inv_out_scale, out_scale;
  int tiles_m, tiles_n;        // (set by the launch)
};

// The best tile for a problem, its estimated time and whether each of its workgroups
// has a compute unit; tile < 0: not served. The caller compares it with what else
// serves the call. few_rows: `us` is of the fit for up to 64 rows, and general_tile and
// general_us are what the fit for any number of rows gives (else the same as tile and us).
struct WaveSplitChoice { int tile; double us; bool one_round, few_rows; int general_tile; double general_us; };
WaveSplitChoice choose_wave_split(const WaveSplitArgs& a, uint32_t type);
int launch_mmt4d_wave_split(const WaveSplitArgs& a, uint32_t type, int tile, hipStream_t s);

}  // namespace uk

#endif  // IREE_AMD_UK_MMT4D_WAVE_SPLIT_H_
