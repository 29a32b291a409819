// W4A16 prefill kernel (large M, MFMA-bound).
//
// Workgroup tile 64 to 128 rows x 64 to 512 columns, four or eight waves side by side: every wave owns RT x CT MFMA tiles
// of 16 x 16 (at most 128 x 64, fp32 accumulators in registers).  The height follows M: with 128 rows always, M = 140 at
// 4096 x 22016 took 46.7 us, in blocks of 80 36.4; M = 387 at 4096 x 12288 50 -> 45.  Activations go from global memory straight
// into LDS (no staging registers), 128 k at a time, two stages, one barrier per stage, in a layout that keeps both
// the global reads (four lanes per 64 contiguous bytes) and the LDS reads (no bank conflicts) at full rate.
// Weights never touch LDS: each wave
// reads its own column tiles straight from the fragment-order buffer (one 128-bit load per lane = the B operands of
// four 16x16x32 MFMAs), two k tiles ahead, and dequantises them in registers once per row block:
//   w = T((u - z) * s), rounded once -- the reference's dequantise-then-MMA semantics
//   (LK/cutlass_extensions/gemm/warp/mma_tensorop_dequantizer.h:206-245, 368-394), with no second rounding.
//   bit operations to 1024 + u / 64 + u, packed fp16 subtract of (bias + z) (exact), packed multiply by s.
// The matrix cores always run in fp16.  Rounding a dequantised weight to bf16 (8 significant bits) would cost up to
// 2^-8 per weight -- together with the bf16 rounding of the output more than the 1e-2 bound on the maximum relative
// error allows -- so bf16 activations are first re-encoded, exactly, as fp16 with one power-of-two exponent per row
// (a bf16 significand fits into fp16; the row exponent keeps every row inside the fp16 range whatever its
// magnitude); the row factor 2^e is applied to the fp32 accumulators in the epilogue.  The bf16 group scales are
// converted to fp16 after division by a power of two per column (the column's largest scale exponent, kept in
// every scale/zero word by the repack), which the epilogue puts back, so scales far outside the fp16 range work.
// Workgroups are numbered so that those sharing a row block of the activations run on the same XCD (own L2).
// The kernel and its launch by form, a template over the element type: compiled once per type (ksq_w4a16_prefill_f16.hip,
// ksq_w4a16_prefill_bf16.hip: the forms are half of the compile time of the library, and two files go side by side).
#pragma once

#include <type_traits>
#include <utility>

#include "ksq_internal.h"
#include "ksq_epilogue.h"
#include "ksq_w4a16_ops.h"
#include "ksq_w4a16_prefill.h"

namespace ksq {
namespace {

using namespace w4;
typedef __attribute__((address_space(3))) void* lds_ptr;

// RT = row tiles of 16 per workgroup: eight, or fewer where that divides the rows into as many blocks with less padding
// (every workgroup of M = 387 then has 112 rows instead of 128).
// CT = column tiles per wave: 4 (64 columns: tiles of 256 or 512 columns) or 3 (48 columns: 192 or 384), for
// widths whose number of tiles falls better on the compute units (a partly filled last round costs a full one);
// 2 or 1 (tiles of 128 or 64 columns) where a single row block has to be spread over the device (65 to 128 rows).
template <typename T, int GPT, int NW, int KG, int CT, int RT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void w4a16_prefill_kernel(PrefillArgs p) {
  static_assert(NW == 4 || NW == 8, "four or eight waves side by side");
  static_assert(CT >= 1 && CT <= 4, "one to four column tiles per wave");
  // KG = 2: two groups of four waves on the same 128 x 256 tile, the first on the even k tiles, the second on the
  // odd ones, each with its own pair of activation stages; the second group's accumulators reach the first through
  // LDS at the end.  For grids that put one workgroup on a CU: two waves per SIMD instead of one.
  static_assert(KG == 1 || (KG == 2 && NW == 4), "two k groups of four waves");
  static_assert(RT >= (KG == 2 ? 4 : 5) && RT <= kMaxRT, "row tiles per workgroup");  // five: the epilogue needs 17 KiB a stage
  constexpr int kH0 = (RT + 1) / 2, kH1 = RT / 2;  // row tiles of the two halves of a 32-k step
  constexpr int kFPW = (RT * 4 + NW - 1) / NW;  // activation blocks of a stage that one wave brings in (the last: fewer)
  constexpr int kPart = (kFPW + 3) / 4;         // of them in each quarter of a stage's loads
  using O = Ops<_Float16>;  // the matrix cores run in fp16 for both element types
  using DQ = Dequant<T>;
  constexpr bool kBF16 = sizeof(T) == 2 && !__is_same(T, _Float16);
  // 16-byte elements per activation stage (16 RT rows x 128 k): 32 KiB with eight.  Where the waves do not divide the blocks
  // (eight waves with five or seven row tiles) a stage has room for kFPW blocks from every wave, and the last ones' go unread:
  // a branch around those loads split every step for the compiler, which then spilled 31 registers with groups of 64 (us, with
  // the branch / without: M = 1774, 4096 x 16320 fp16 271 / 192, bf16 290 / 201; groups of 128, not spilled, 189 / 186; five
  // row tiles, M = 144, 4096 x 32976 50.7 / 51.9).
  constexpr int kStage = kFPW * NW * 64;
  constexpr int kEpiStride = 68;        // floats per row of the epilogue transpose (2-way conflicts at worst)
  // two activation stages as two separate objects: loads into one are then known not to alias reads of the other
  __shared__ u32x4 lds_a0[kStage];
  __shared__ u32x4 lds_a1[kStage];
  __shared__ u32x4 lds_a2[KG == 2 ? kStage : 1];
  __shared__ u32x4 lds_a3[KG == 2 ? kStage : 1];

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KG == 2 ? wave_all >> 2 : 0;           // k group of this wave
  const int wave = KG == 2 ? wave_all & 3 : wave_all;  // its place among the waves side by side
  const int c = lane & 15, j = lane >> 4;

  int mb, nb;
  if (!tile_of(tile_logical_id(blockIdx.x, gridDim.x), p.mblocks, p.nblocks, &mb, &nb)) return;  // rounding of the grid
  const int m0 = mb * (16 * RT);
  const int nt0 = (nb * NW + wave) * CT;

  __amdgpu_buffer_rsrc_t rs_w[CT], rs_sz[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int nt = nt0 + t;
    const bool ok = nt < p.ntiles;
    const size_t ntc = ok ? (size_t)nt : 0;
    rs_w[t] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(static_cast<const char*>(p.weight) + ntc * p.KT * 1024), 0, ok ? p.KT * 1024 : 0, 0x00020000);
    rs_sz[t] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p.sz) + ntc * p.G * 64), 0,
                                                 ok ? p.G * 64 : 0, 0x00020000);
  }
  const __amdgpu_buffer_rsrc_t rs_a =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.act), 0, (int)((size_t)p.M * p.K * 2), 0x00020000);
  // Activation stage in LDS: 4 RT blocks of 1 KiB, block (mt, q) = rows 4q .. 4q+3 of row tile mt, all 256 bytes of
  // the k tile.  A block is one global -> LDS load instruction (lane l lands at l * 16), with lane l on row l/4 % 4,
  // 32-k step l / 16 and 16-byte piece (l % 4) ^ q: every aligned group of four lanes reads 64 contiguous bytes of
  // one row (the memory pipeline then takes four lanes per clock instead of one), and the xor by q makes the 16
  // rows that one group of 16 lanes reads back for an MFMA operand (piece j of rows 0..15) fall on 16 different
  // bank groups.  Rows past M repeat row M - 1 (their results are never stored).  This wave brings in blocks
  // kFPW * wave .. kFPW * wave + kFPW - 1.
  unsigned a_off[8];  // kFPW of them in use: block i of this wave
#pragma unroll
  for (int i = 0; i < kFPW; ++i) {
    const int blk = kFPW * wave + i, mt = blk >> 2, q = blk & 3;
    int row = m0 + 16 * mt + 4 * q + ((lane >> 2) & 3);
    row = row < p.M ? row : p.M - 1;
    a_off[i] = (unsigned)row * p.K * 2u + 64u * (lane >> 4) + 16u * ((lane & 3) ^ q);
  }
  // where lane (c, j) finds piece j of row c of a (row tile, 32-k step) inside the stage, apart from
  // row tile * 256 + step * 16 (in 16-byte units)
  const int a_lane = (c >> 2) * 64 + (c & 3) * 4 + (j ^ (c >> 2));
  const unsigned w_voff = lane * 16u, sz_voff = c * 4u;

  f32x4 acc[RT][CT];
#pragma unroll
  for (int mt = 0; mt < RT; ++mt)
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[mt][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct BTile {
    u32x4 w[CT];
    uint32_t sz[CT][GPT];
  };
  BTile b0, b1;

  // k tiles of this workgroup: all of them, or (K split over grid.y, for grids that would leave most compute units
  // without a tile) the range of its split, whose raw fp32 tile goes to the workspace for the reduction kernel
  int kt0, kt1;
  split_range(p.KT, blockIdx.y, p.ksplit, &kt0, &kt1);

  // Loads are issued a few at a time between the matrix instructions (a burst of 16 memory instructions would hold the
  // wave in the issue queue of the memory pipeline, and the matrix cores with it): during a k tile first the activation
  // blocks of the next one (global -> LDS, no registers), a quarter of them at a time, and at its end, into the
  // registers that its own weights have left by then, the weights of the tile after the next.  They come from HBM and
  // would not arrive within one k tile of a small workgroup: a step waits for all loads but those (kWeightLoads).
  // 4096 x 22016 M = 70 28.0 -> 22.9 us, 4096 x 12288 M = 140 27.6 -> 24.0, 8192 x 8192 M = 200 39.6 -> 36.7; level at M = 4096.
  constexpr int kWeightLoads = CT * (1 + GPT);
  auto load_a = [&](u32x4* buf, int kt, int q) {
    if (kt >= kt1) kt = kt1 - 1;  // the scalar offset is not range-checked: past the end re-read the last tile (nobody uses it)
#pragma unroll
    for (int x = 0; x < kPart; ++x) {
      const int i = kPart * q + x;
      if (i < kFPW)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lds_ptr)(buf + (kFPW * wave + i) * 64), 16, a_off[i], kt * 256, 0, 0);
    }
  };
  auto load_w = [&](BTile& b, int kt, int t) {
    if (kt >= kt1) kt = p.KT;  // past the end of the resource: zero, without touching memory
    b.w[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_w[t], w_voff + kt * 1024u, 0, 0));
#pragma unroll
    for (int gi = 0; gi < GPT; ++gi)
      b.sz[t][gi] = __builtin_amdgcn_raw_buffer_load_b32(rs_sz[t], sz_voff + (kt * GPT + gi) * 64u, 0, 0);
  };

  uint32_t m_lo = Ops<_Float16>::kMaskLo, m_hi = Ops<_Float16>::kMaskHi, g_lo = Ops<_Float16>::kMagicLo,
           g_hi = Ops<_Float16>::kMagicHi;
  KSQ_PIN_SGPR(m_lo);
  KSQ_PIN_VGPR(g_lo);
  KSQ_PIN_VGPR(g_hi);
  KSQ_PIN_VGPR(m_hi);

  // Activation fragments are read from LDS three or four at a time (half of the row tiles of one 32-k step), one half ahead
  // of the matrix instructions that use them, so that the LDS latency hides behind 9 to 16 MFMAs (with three or four column tiles).
  auto read_half = [&](u32x4 (&a)[(RT + 1) / 2], const u32x4* buf, int ks, int h) {
#pragma unroll
    for (int i = 0; i < (h ? kH1 : kH0); ++i) a[i] = buf[(kH0 * h + i) * 256 + ks * 16 + a_lane];
  };
  auto mfma_row = [&](const u32x4& a, const u32x4 (&b)[CT], int mt) {
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[mt][t] = O::mfma(a, b[t], acc[mt][t]);
  };
  // One k tile.  After the barrier this tile's activations and weights have landed and are visible to
  // the whole workgroup, and every wave is done with the other buffer.
  auto step = [&](const u32x4* cur, u32x4* nxt, BTile& bt, int kt) __attribute__((always_inline)) {
    KSQ_WAIT_VMCNT(kWeightLoads);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    u32x4 a0[kH0], a1[kH0];
    read_half(a0, cur, 0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      u32x4 b[CT];
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const typename DQ::Consts k = DQ::prepare(bt.sz[t][GPT == 2 ? (ks >> 1) : 0]);
        b[t] = DQ::run(bt.w[t][ks], k, m_lo, m_hi, g_lo, g_hi);
      }
      read_half(a1, cur, ks, 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < kH0) mfma_row(a0[i], b, i);
        if (ks < 2 && i == 0) load_a(nxt, kt + KG, 2 * ks);
        if (ks == 3 && i < CT) load_w(bt, kt + 2 * KG, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (ks < 3) read_half(a0, cur, ks + 1, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < kH1) mfma_row(a1[i], b, kH0 + i);
        if (ks < 2 && i == 0) load_a(nxt, kt + KG, 2 * ks + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // The k loop of one k group over its pair of stages: k tiles kt0 + kg, kt0 + kg + KG, ...  Both groups pass the same
  // number of barriers (a step has one); with an odd number of k tiles the second group's last step has no tile.
  // (everything here has to be inlined: a call would put the accumulators, captured by reference, into memory; and
  // without a branch around a step, or the compiler's own waits no longer leave the weight loads in flight)
  auto k_loop = [&](u32x4* s0, u32x4* s1) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) load_a(s0, kt0 + kg, q);
#pragma unroll
    for (int t = 0; t < CT; ++t) load_w(b0, kt0 + kg, t);
    __builtin_amdgcn_sched_barrier(0);  // the wait of a step counts on this order
#pragma unroll
    for (int t = 0; t < CT; ++t) load_w(b1, kt0 + kg + KG, t);
    __builtin_amdgcn_sched_barrier(0);
    const int nsteps = (kt1 - kt0 + KG - 1) / KG, tiles = (kt1 - kt0 - kg + KG - 1) / KG;
    int st = 0;
    for (; st + 2 <= tiles; st += 2) {
      step(s0, s1, b0, kt0 + kg + st * KG);
      step(s1, s0, b1, kt0 + kg + (st + 1) * KG);
    }
    if (st < tiles) step(s0, s1, b0, kt0 + kg + st * KG);
    if (KG == 2 && tiles < nsteps) {
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __builtin_amdgcn_s_barrier();
    }
  };
  if (KG == 1 || kg == 0) k_loop(lds_a0, lds_a1);
  else k_loop(lds_a2, lds_a3);

  // ---- epilogue: transpose each 16-row slab through LDS so that every lane stores 16 contiguous bytes
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the last (unused) prefetch must not land on top of the transposes
  __syncthreads();
  float* epi = reinterpret_cast<float*>(wave < 4 ? lds_a0 : lds_a1) + (wave & 3) * (16 * kEpiStride);  // 4352 B
  if constexpr (KG == 2) {
    // wave w of the second group parks its accumulators in stage w; wave w of the first group, which owns the same
    // output tiles, adds them to its own and then uses that stage, and no other, for its transposes
    f32x4* park = reinterpret_cast<f32x4*>(wave == 0 ? lds_a0 : wave == 1 ? lds_a1 : wave == 2 ? lds_a2 : lds_a3);
    if (kg == 1) {
#pragma unroll
      for (int mt = 0; mt < RT; ++mt)
#pragma unroll
        for (int t = 0; t < CT; ++t) park[(mt * CT + t) * 64 + lane] = acc[mt][t];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int mt = 0; mt < RT; ++mt)
#pragma unroll
      for (int t = 0; t < CT; ++t) acc[mt][t] += park[(mt * CT + t) * 64 + lane];
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): all of them read before the transposes overwrite the stage
    epi = reinterpret_cast<float*>(park);
  }
  uint16_t* out = static_cast<uint16_t*>(p.out);
  const int ncol0 = nt0 * 16;
  float cf[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};  // bf16 scales: 2^E of this lane's eight columns
  if constexpr (kBF16) {
    const int col = ncol0 + (lane & 7) * 8;
    if (col + 8 <= p.N && (lane & 7) * 8 < 16 * CT) column_factors(p.sz, p.G, col, cf);
  }
#pragma unroll
  for (int mt = 0; mt < RT; ++mt) {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) epi[(4 * j + i) * kEpiStride + 16 * t + c] = acc[mt][t][i];
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own LDS writes have landed
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      const int rr = (lane >> 3) + 8 * pass, cc = (lane & 7) * 8;
      const float* src = epi + rr * kEpiStride + cc;
      const int row = m0 + 16 * mt + rr, col = ncol0 + cc;
      if (p.ksplit > 1) {  // the fp32 segment of this split; the reduction kernel finishes it
        if (row < p.M && col + 8 <= p.N && cc < 16 * CT) {
          f32x4* dst = reinterpret_cast<f32x4*>(p.partial + ((size_t)blockIdx.y * p.M + row) * p.N + col);
          dst[0] = f32x4{src[0], src[1], src[2], src[3]};
          dst[1] = f32x4{src[4], src[5], src[6], src[7]};
        }
        continue;
      }
      float rs = 1.f;
      if constexpr (kBF16) rs = p.row_scale[row < p.M ? row : p.M - 1];
      float vals[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) vals[q] = src[q] * rs * cf[q];
      epi_store_row8_wave<T>(p.epi, out, vals, row, col, p.N, row < p.M && col + 8 <= p.N && cc < 16 * CT, row < p.M, lane);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
  }
}

template <typename T, int GPT, int NW, int KG, int CT, int RT>
bool launch_form(const PrefillArgs& a, dim3 grid, dim3 block, hipStream_t s) {
  if constexpr (w4a16_prefill_form(NW, KG, CT, RT)) {
    hipLaunchKernelGGL((w4a16_prefill_kernel<T, GPT, NW, KG, CT, RT>), grid, block, 0, s, a);
    return true;
  } else {
    return false;
  }
}

// forms numbered by (waves and k groups: 4 x 1, 4 x 2, 8 x 1), column tiles 1 .. 4, row tiles 4 .. 8
constexpr int kFormIds = 3 * 4 * (kMaxRT - 3);
template <typename T, int GPT, int... ID>
bool launch_id(int id, const PrefillArgs& a, dim3 grid, dim3 block, hipStream_t s, std::integer_sequence<int, ID...>) {
  return ((id == ID && launch_form<T, GPT, ID % 3 == 2 ? 8 : 4, ID % 3 == 1 ? 2 : 1, ID / 3 % 4 + 1, ID / 12 + 4>(
                           a, grid, block, s)) ||
          ...);
}

template <typename T>
bool launch_typed(const PrefillArgs& a, int gpt, const PrefillPlan& p, dim3 grid, dim3 block, hipStream_t s) {
  if (!w4a16_prefill_form(p.nw, p.kg, p.ct, p.rt)) return false;
  const int id = (p.nw == 8 ? 2 : p.kg - 1) + 3 * (p.ct - 1) + 12 * (p.rt - 4);
  const auto ids = std::make_integer_sequence<int, kFormIds>();
  return gpt == 1 ? launch_id<T, 1>(id, a, grid, block, s, ids) : launch_id<T, 2>(id, a, grid, block, s, ids);
}

}  // namespace
}  // namespace ksq
