// What the planner and the entry point of the W4A16 prefill kernel (ksq_w4a16_prefill.hip) share with the files that
// compile it (ksq_w4a16_prefill_f16.hip, ksq_w4a16_prefill_bf16.hip): arguments, and which forms there are.
#pragma once

#include "ksq_internal.h"

namespace ksq {

struct PrefillArgs {
  const void* weight;
  const void* sz;
  const void* act;
  void* out;
  const float* row_scale;  // bf16 route: 2^e per row of the re-encoded activations
  int M, N, K, KT, G, ntiles, mblocks, nblocks;
  int ksplit;          // grid.y: K split over workgroups
  float* partial;      // [ksplit][M][N] fp32, ksplit > 1 only
  Epilogue epi;
};

constexpr int kMaxRT = 8;  // 16-row MFMA tiles per wave at most: blocks of 128 rows

// The forms that are compiled, and with that the ones that the planner chooses from: `nw` waves side by side in `kg` k groups,
// `ct` column tiles a wave, `rt` row tiles.  Two k groups at every width and height; one k group (grids of more than one
// workgroup per CU) at three and four column tiles and 80 to 128 rows.  Each of these 36 is the planner's estimate of the
// fastest somewhere in M = 48 .. 4096, K = 256 .. 33000, N = 128 .. 57600; the least used ones, four waves and one k group at three
// column tiles, are up to 9 % ahead of the next there (M = 782, 3968 x 20736).
constexpr bool w4a16_prefill_form(int nw, int kg, int ct, int rt) {
  if (ct < 1 || ct > 4 || rt > kMaxRT) return false;
  return kg == 2 ? nw == 4 && rt >= 4 : kg == 1 && (nw == 4 || nw == 8) && ct >= 3 && rt >= 5;
}

// Launches one form; false if it is not one of them.  gpt = groups per k tile (1 or 2).
bool w4a16_prefill_launch_f16(const PrefillArgs& a, int gpt, const PrefillPlan& plan, dim3 grid, dim3 block, hipStream_t s);
bool w4a16_prefill_launch_bf16(const PrefillArgs& a, int gpt, const PrefillPlan& plan, dim3 grid, dim3 block, hipStream_t s);

}  // namespace ksq
