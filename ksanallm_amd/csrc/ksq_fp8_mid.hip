// FP8 e4m3 GEMM, medium M: out[m,n] = T((sum_k a[m,k] * w[n,k]) * w_scale[n] * a_scale[m]).
//
// Between the decode kernels (whose workgroups stream weights past activations held in registers) and the 256 x 256
// tiles (which need thousands of rows x columns to cover the device) a GEMM is bound by the bytes that the compute units
// have in flight: the weights come from HBM once, every CU has to hold a workgroup, and the rest is latency.  So:
//   * a workgroup is eight waves side by side on 16 MT rows x 128 WN columns; every wave has all the rows against WN
//     column tiles of its own, so a weight is read from memory and from LDS once.
//   * both operands go from memory straight into LDS, whole cache lines at a time, in a ring of R stages of 128 k
//     (R - 1 requested ahead), one barrier per stage.
//   * K is split over grid.y until the workgroups cover the device; a split stores its accumulators as they are (16
//     bytes per lane, whole KiB per wave and instruction) and fp8_mid_reduce_kernel adds them in split order.  (The
//     last workgroup to arrive doing that instead, through agent-scope stores and a counter, measured level or up to 25 %
//     slower: 4096 x 12288 at M = 64 18.5 -> 20.9 us.)
// K is any multiple of 16: the last stage masks the weights past K.
#include <cstdio>
#include <cstdlib>

#include "ksq_epilogue.h"
#include "ksq_internal.h"
#include "ksq_lds_dma.h"

namespace ksq {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
using ldsdma::lds_addr;
using ldsdma::load_lds_opaque;
using ldsdma::raw_rsrc;

struct Fp8MidArgs {
  const uint8_t* aq;  // [M][K]
  const uint8_t* wq;  // [N][K]
  const float* a_scale;
  const float* w_scale;
  void* out;
  f32x4* partial;  // [ksplit][row tiles of 16][ntiles][64], ksplit > 1 only
  int M, N, K, KS /* 128-byte k stages, rounded up */, mblocks, nblocks, mtiles, ntiles;
  int a_scale_per_row, w_scale_per_col;
  int ksplit;
  Epilogue epi;
};

__device__ inline i32x8 join(u32x4 lo, u32x4 hi) {
  i32x8 v;
  v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
  v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
  return v;
}

template <typename T, int MT, int WN, int R>
__global__ __launch_bounds__(512) void fp8_mid_kernel(Fp8MidArgs p) {
  static_assert(MT == 4 || MT == 8, "activation blocks are dealt out to eight waves");
  constexpr int kAct = MT * 128, kWave = WN * 128;  // 16-byte elements of a stage: activations, one wave's weights
  constexpr int kStage = kAct + 8 * kWave;
  constexpr int kAPW = MT / 4;                      // activation blocks (8 rows x 128 bytes) per wave and stage
  constexpr int kLoads = kAPW + 2 * WN;             // memory instructions per wave and stage
  constexpr int kEpiStride = 16 * WN + 4;
  __shared__ u32x4 ring[R * kStage];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, j = lane >> 4;

  int mb, nb;
  if (!tile_of(tile_logical_id(blockIdx.x, gridDim.x), p.mblocks, p.nblocks, &mb, &nb)) return;  // rounding of the grid
  const int m0 = mb * 16 * MT, nt0 = nb * 8 * WN + wave * WN;
  int s_begin, s_end;
  split_range(p.KS, blockIdx.y, p.ksplit, &s_begin, &s_end);

  const u32x4 rs_a = raw_rsrc(p.aq, (size_t)p.M * p.K), rs_w = raw_rsrc(p.wq, (size_t)p.N * p.K);
  // A block = one load instruction = 8 rows x the 128 bytes of a stage: eight lanes read one whole cache line (sixteen
  // rows of 64 bytes, which is what the operands of a matrix instruction look like, get a third of the rate out of a
  // compute unit: 35 against 84 bytes per ns measured).  Lane l lands at l * 16 and brings piece (l & 7) ^ x(row) of
  // row l >> 3, x = row ^ (row >> 3) over the 16 rows of a tile, so that the sixteen lanes which later read one piece
  // of sixteen rows fall on sixteen different bank groups.  Rows past M and N repeat the last one (never stored).
  unsigned a_off[kAPW], w_off[2 * WN];
  const unsigned kb0 = ((lane & 7) ^ (lane >> 3)) * 16u, kb1 = kb0 ^ 16u;  // of the rows 0 .. 7 and 8 .. 15 of a tile
#pragma unroll
  for (int i = 0; i < kAPW; ++i) {
    int row = m0 + 8 * (kAPW * wave + i) + (lane >> 3);
    row = row < p.M ? row : p.M - 1;
    a_off[i] = (unsigned)row * p.K;
  }
#pragma unroll
  for (int i = 0; i < 2 * WN; ++i) {
    int row = 16 * nt0 + 8 * i + (lane >> 3);
    row = row < p.N ? row : p.N - 1;
    w_off[i] = (unsigned)row * p.K;
  }
  const int f_lane0 = r * 8 + (j ^ (r & 7) ^ (r >> 3)), f_lane1 = f_lane0 ^ 4;  // pieces j and 4 + j of row r

  f32x4 acc[MT][WN];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < WN; ++t) acc[mt][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Memory instruction i of stage s into ring slot `slot`: kAPW activation blocks, then the wave's own weights.  In a
  // last stage that K ends inside of, pieces past K bring piece 0 of the row (masked below).
  auto load_item = [&](int slot, int s, int i) __attribute__((always_inline)) {
    const bool first = i < kAPW;
    const int block = first ? (kAPW == 2 ? i : wave) & 1 : (i - kAPW) & 1;  // which half of a 16-row tile
    unsigned kb = block ? kb1 : kb0;
    if (kb >= (unsigned)(p.K - s * 128)) kb = 0;
    u32x4* dst = ring + slot * kStage + (first ? (kAPW * wave + i) * 64 : kAct + wave * kWave + (i - kAPW) * 64);
    load_lds_opaque(first ? rs_a : rs_w, lds_addr(dst), (first ? a_off[first ? i : 0] : w_off[first ? 0 : i - kAPW]) + kb,
                    s * 128);
  };
  auto read_frag = [&](const u32x4* tile) __attribute__((always_inline)) { return join(tile[f_lane0], tile[f_lane1]); };

  // One stage.  On entry the loads of the AHEAD newest stages may be in flight; after the barrier stage s is visible to
  // every wave and every wave is done with the slot of stage s - 1, which stage s + R - 1 goes into.
  auto step = [&](int s, int slot, bool request) __attribute__((always_inline)) {
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const u32x4* act = ring + slot * kStage;
    const u32x4* wgt = act + kAct + wave * kWave;
    i32x8 bf[WN];
    i32x8 a_cur = read_frag(act);
#pragma unroll
    for (int t = 0; t < WN; ++t) bf[t] = read_frag(wgt + t * 128);
    i32x8 a_nxt = read_frag(act + 128);
    const int left = p.K - s * 128;
    if (left < 128) {  // the last stage of a K that is no multiple of 128: zero weights past K
#pragma unroll
      for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int q = 0; q < 8; ++q) bf[t][q] = 16 * j + (q < 4 ? 0 : 64) < left ? bf[t][q] : 0;
    }
    const int rslot = slot == 0 ? R - 1 : slot - 1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const i32x8 af = a_cur;
      a_cur = a_nxt;
      if (mt + 2 < MT) a_nxt = read_frag(act + (mt + 2) * 128);
      if (request) {
#pragma unroll
        for (int i = mt * kLoads / MT; i < (mt + 1) * kLoads / MT; ++i) load_item(rslot, s + R - 1, i);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < WN; ++t)
        acc[mt][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[t], acc[mt][t], 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int count = s_end - s_begin;
#pragma unroll
  for (int q = 0; q < R - 1; ++q)
    if (q < count) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) load_item(q, s_begin + q, i);
    }
  int s = s_begin, slot = 0;
  auto next = [&]() __attribute__((always_inline)) {
    ++s;
    slot = slot == R - 1 ? 0 : slot + 1;
  };
  while (s + R - 1 < s_end) {
    KSQ_WAIT_VMCNT((R - 2) * kLoads);
    step(s, slot, true);
    next();
  }
  // the last stages request nothing: one stage fewer in flight at each
  if constexpr (R >= 4) {
    if (s + 2 < s_end) {
      KSQ_WAIT_VMCNT(2 * kLoads);
      step(s, slot, false);
      next();
    }
  }
  if (s + 1 < s_end) {
    KSQ_WAIT_VMCNT(kLoads);
    step(s, slot, false);
    next();
  }
  if (s < s_end) {
    KSQ_WAIT_VMCNT(0);
    step(s, slot, false);
  }

  if (p.ksplit > 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < WN; ++t) {
        const int row_tile = mb * MT + mt;
        if (row_tile < p.mtiles && nt0 + t < p.ntiles)
          p.partial[(((size_t)blockIdx.y * p.mtiles + row_tile) * p.ntiles + nt0 + t) * 64 + lane] = acc[mt][t];
      }
    return;
  }
  // ---- epilogue: scales, then a transpose through LDS so that every lane stores eight contiguous columns
  __syncthreads();  // every wave is done with the ring
  float* epi = reinterpret_cast<float*>(ring) + wave * (16 * kEpiStride);
  epi_elem_t<T>* out = static_cast<epi_elem_t<T>*>(p.out);
  float ws[WN];
#pragma unroll
  for (int t = 0; t < WN; ++t) {
    const int col = 16 * (nt0 + t) + r;
    ws[t] = p.w_scale[p.w_scale_per_col ? (col < p.N ? col : p.N - 1) : 0];
  }
  constexpr int kSegs = 2 * WN;  // lanes per row, eight columns each; lanes past 16 rows idle (WN = 1)
  const int rr = lane / kSegs, cc = (lane % kSegs) * 8;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int t = 0; t < WN; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) epi[(4 * j + i) * kEpiStride + 16 * t + r] = acc[mt][t][i] * ws[t];
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own LDS writes have landed
    const int row = m0 + 16 * mt + rr, col = 16 * nt0 + cc;
    const bool row_ok = rr < 16 && row < p.M;
    const float* src = epi + (rr < 16 ? rr : 0) * kEpiStride + cc;
    const float as = p.a_scale[p.a_scale_per_row && row_ok ? row : 0];
    float vals[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) vals[q] = src[q] * as;
    epi_store_row8_wave<T, kSegs>(p.epi, out, vals, row, col, p.N, row_ok && col + 8 <= p.N, row_ok, lane);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // ... and its reads, before the next row tile overwrites the slab
  }
}

// Second half of a split: a workgroup per row tile x four column tiles, a wave per column tile: sums the
// splits in order, applies the column scales, and hands the sixteen rows through LDS to the lanes that store whole lines.
template <typename T>
__global__ __launch_bounds__(256) void fp8_mid_reduce_kernel(Fp8MidArgs p) {
  constexpr int kEpiStride = 68;
  __shared__ float slab[16 * kEpiStride];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, j = lane >> 4;
  const int groups = (p.ntiles + 3) / 4;
  const int row_tile = blockIdx.x / groups, nt0 = (blockIdx.x - row_tile * groups) * 4;
  const int nt = nt0 + wave < p.ntiles ? nt0 + wave : p.ntiles - 1;  // a tile past the last: summed, never stored
  const size_t stride = (size_t)p.mtiles * p.ntiles * 64;
  const f32x4* src0 = p.partial + ((size_t)row_tile * p.ntiles + nt) * 64 + lane;
  f32x4 sum[1];
  sum_splits(sum, p.ksplit, [&](int sp, int) { return src0[sp * stride]; });
  const int c = 16 * nt + r;
  const float ws = p.w_scale[p.w_scale_per_col ? (c < p.N ? c : p.N - 1) : 0];
#pragma unroll
  for (int i = 0; i < 4; ++i) slab[(4 * j + i) * kEpiStride + 16 * wave + r] = sum[0][i] * ws;
  __syncthreads();
  if (wave >= 2) return;  // two waves hold the sixteen rows' eight segments each
  const int rr = threadIdx.x >> 3, cc = (threadIdx.x & 7) * 8;
  const float* src = slab + rr * kEpiStride + cc;
  const int row = 16 * row_tile + rr, col = 16 * nt0 + cc;
  const float as = p.a_scale[p.a_scale_per_row && row < p.M ? row : 0];
  float vals[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) vals[q] = src[q] * as;
  epi_store_row8_wave<T>(p.epi, static_cast<epi_elem_t<T>*>(p.out), vals, row, col, p.N, row < p.M && col + 8 <= p.N,
                         row < p.M, lane);
}

}  // namespace

// ---- planning -----------------------------------------------------------------------------------------------------
// Which form, how many splits of K, and whether this kernel at all: the least estimated time in us.  The estimates are
// fitted to 12,000 measured points (23 shapes of N = 1024 .. 59136, K = 1024 .. 29568, M = 1 .. 2048, every form and
// split; 6 to 12 % rms per form).  Against the best of everything measured the choice loses 1.7 % on average; against
// the kernels that served these sizes before, M = 65 .. 2048 is 1.43 times as fast on average (M = 128: K = N = 4096
// 25.5 -> 14.5 us, 4096 x 12288 31.5 -> 20.0; M = 512, K = N = 4096 37 -> 19) and M = 17 .. 64 1.15 times.
//   form: fixed + rounds x (round + stages x (stage + load x busy)), busy = the share of the CUs that hold a workgroup:
//   memory and L2 are shared, so a stage takes longer on a full device
//   a split adds the reduction kernel and its bytes
namespace {
struct MidForm {
  int mt, wn, ring;
  double fixed, stage, load, round;
};
constexpr MidForm kForms[] = {
    {4, 1, 3, 4.36, 0.415, 0.088, 0.13},  // two workgroups per CU (72 KiB of LDS)
    {4, 1, 4, 2.66, 0.363, 0.155, 1.71},  // the others one: 96, 128, 128, 144 KiB
    {4, 2, 4, 2.62, 0.579, 0.293, 2.12},
    {8, 1, 4, 3.23, 0.533, 0.149, 1.52},
    {8, 2, 3, 2.83, 0.726, 0.363, 2.13},
};
constexpr double kReduce = 1.89, kReduceMB = 0.29;
constexpr size_t kMaxM = 2048;  // fitted up to here; the 256-row tiles win from about 1000 rows on anyway

constexpr size_t kMaxSplit = 12;

// The decode kernels at 17 .. 64 rows: a fixed part, the weights, the activations that every workgroup pulls (10 % rms)
double kstat_estimate(size_t m, size_t n, size_t k) {
  const double mb = n * 1e-6 * k, kk = k * 1e-3;
  return m <= 32 ? 3.41 + 0.215 * mb + 0.338 * kk : 3.06 + 0.235 * mb + 0.674 * kk;
}
}  // namespace

Fp8MidPlan fp8_mid_plan(size_t m, size_t n, size_t k, int cus_, size_t workspace_bytes) {
  Fp8MidPlan best{};
  if (m == 0 || m >= (1u << 24) || n % 8 != 0 || m * k >= 0x7FFFFF00ull || n * k >= 0x7FFFFF00ull || cus_ <= 0) return best;
  const size_t cus = (size_t)cus_, stages = (k + 127) / 128, mtiles = (m + 15) / 16, ntiles = (n + 15) / 16;
  int form = -1;
  size_t splits = 0;
  if (const char* e = tuning_env("KSQ_FP8_MID")) {  // tuning / test override: "0" = never, "form[,splits]" = always
    int f = -1, sp = 0;
    if (sscanf(e, "%d,%d", &f, &sp) >= 1 && f == 0) return best;
    if (f >= 1 && f <= (int)(sizeof(kForms) / sizeof(kForms[0]))) form = f - 1, splits = (size_t)sp;
  }
  if (const char* e = tuning_env("KSQ_FP8_PREFILL_TILE")) {  // a 128 x 256 tile is this kernel's, a 256 x 256 one is not
    if (atoi(e) == 256) return best;
    if (atoi(e) == 128) form = (int)(sizeof(kForms) / sizeof(kForms[0])) - 1;
  } else if (form < 0 && (tuning_env("KSQ_FP8_TAIL_KSPLIT") || tuning_env("KSQ_FP8_TAIL_QUARTERS") ||
                          tuning_env("KSQ_FP8_PREFILL_MIN_M"))) {
    return best;  // overrides of the 256-row kernel ask for that kernel
  }
  double limit = 1e30;
  if (form < 0) {
    if (m < 17 || m > kMaxM) return best;
    if (m <= 64) limit = kstat_estimate(m, n, k);
    else if (k % 128 == 0) limit = fp8_prefill_estimate(m, n, k, cus_);
    // else: the alternative is the streaming kernel, five to ten times as slow
  }
  // This runs in every call of these sizes (0.9 us with every estimate made in full): a form and split whose stages alone take
  // longer than the best so far goes no further.
  size_t split_stages[kMaxSplit + 1];
  for (size_t ks = 1; ks <= kMaxSplit; ++ks) split_stages[ks] = (stages + ks - 1) / ks;
  for (int f = 0; f < (int)(sizeof(kForms) / sizeof(kForms[0])); ++f) {
    if (form >= 0 && f != form) continue;
    const MidForm& fm = kForms[f];
    const size_t mb = (m + 16 * fm.mt - 1) / (16 * fm.mt), nb = (n + 128 * fm.wn - 1) / (128 * fm.wn);
    const size_t tiles = (mb * nb + 7) / 8 * 8;
    for (size_t ks = 1; ks <= kMaxSplit && (ks == 1 || ks * 4 <= stages || ks == splits); ++ks) {
      if (splits && ks != splits) continue;
      const size_t need = ks > 1 ? ks * mtiles * ntiles * 1024 : 0;
      if (need > workspace_bytes || ks > stages) break;
      const double reduce = ks > 1 ? kReduce + kReduceMB * 1e-6 * (double)(ks * mtiles * 16 * n * 4) : 0.0;
      if (fm.fixed + fm.round + (double)split_stages[ks] * fm.stage + reduce >= limit) continue;
      const size_t wgs = tiles * ks, rounds = (wgs + cus - 1) / cus;
      const double busy = (double)wgs / (double)(cus * rounds);
      const double t =
          fm.fixed + (double)rounds * (fm.round + (double)split_stages[ks] * (fm.stage + fm.load * busy)) + reduce;
      if (t < limit) {
        limit = t;
        best = Fp8MidPlan{true, fm.mt, fm.wn, fm.ring, (int)ks, need};
      }
    }
  }
  return best;
}

int fp8_launch_mid(int out_dtype, const Fp8MidPlan& plan, void* out, const void* act_q, const float* act_scale,
                   size_t act_scale_count, const void* w_q, const float* w_scale, size_t w_scale_count, size_t m,
                   size_t n, size_t k, void* workspace, hipStream_t s, const Epilogue& epi) {
  Fp8MidArgs a{};
  a.epi = epi;
  a.aq = static_cast<const uint8_t*>(act_q);
  a.wq = static_cast<const uint8_t*>(w_q);
  a.a_scale = act_scale;
  a.w_scale = w_scale;
  a.out = out;
  a.partial = static_cast<f32x4*>(workspace);
  a.M = (int)m;
  a.N = (int)n;
  a.K = (int)k;
  a.KS = (int)((k + 127) / 128);
  a.mtiles = (int)((m + 15) / 16);
  a.ntiles = (int)((n + 15) / 16);
  a.mblocks = (int)((m + 16 * plan.mt - 1) / (16 * plan.mt));
  a.nblocks = (int)((n + 128 * plan.wn - 1) / (128 * plan.wn));
  a.a_scale_per_row = act_scale_count > 1;
  a.w_scale_per_col = w_scale_count > 1;
  a.ksplit = plan.ksplit;
  const dim3 grid(tile_grid(a.mblocks, a.nblocks), (unsigned)plan.ksplit);
  note_launch("fp8_mid_kernel<mt=%d,wn=%d,ring=%d> grid=(%u,%u)", plan.mt, plan.wn, plan.ring, grid.x, grid.y);
#define KSQ_GO(T)                                                                                             \
  do {                                                                                                        \
    if (plan.mt == 4 && plan.wn == 1 && plan.ring == 3)                                                       \
      hipLaunchKernelGGL((fp8_mid_kernel<T, 4, 1, 3>), grid, dim3(512), 0, s, a);                             \
    else if (plan.mt == 4 && plan.wn == 1) hipLaunchKernelGGL((fp8_mid_kernel<T, 4, 1, 4>), grid, dim3(512), 0, s, a); \
    else if (plan.mt == 4) hipLaunchKernelGGL((fp8_mid_kernel<T, 4, 2, 4>), grid, dim3(512), 0, s, a);        \
    else if (plan.wn == 1) hipLaunchKernelGGL((fp8_mid_kernel<T, 8, 1, 4>), grid, dim3(512), 0, s, a);        \
    else hipLaunchKernelGGL((fp8_mid_kernel<T, 8, 2, 3>), grid, dim3(512), 0, s, a);                          \
    if (plan.ksplit > 1) {                                                                                    \
      const size_t units = (size_t)a.mtiles * ((a.ntiles + 3) / 4);                                           \
      hipLaunchKernelGGL(fp8_mid_reduce_kernel<T>, dim3((unsigned)units), dim3(256), 0, s, a);                 \
    }                                                                                                         \
  } while (0)
  if (out_dtype == KSQ_F16) KSQ_GO(_Float16);
  else if (out_dtype == KSQ_F32) KSQ_GO(float);
  else KSQ_GO(__bf16);
#undef KSQ_GO
  KSQ_HIP_TRY(hipGetLastError());
  return KSQ_OK;
}

}  // namespace ksq
