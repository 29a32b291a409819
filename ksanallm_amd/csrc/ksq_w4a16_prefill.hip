// W4A16 prefill: which form of the kernel (ksq_w4a16_prefill_kernel.h) takes a shape, the bf16 activations' conversion in
// front of it, and the sum of a K split behind it.
#include <cstdlib>

#include "ksq_internal.h"
#include "ksq_epilogue.h"
#include "ksq_w4a16_ops.h"
#include "ksq_w4a16_prefill.h"

namespace ksq {
namespace {

using namespace w4;

// Exponents of two bf16 elements as signed halves; infinities and NaN, which do not set a row's exponent, below all others
typedef short i16x2 __attribute__((ext_vector_type(2)));
__device__ inline i16x2 bf16_exponents(uint32_t v) {
  return __builtin_bit_cast(i16x2, v & 0x7F807F80u) + i16x2{0x80, 0x80};
}
// the power of two 2^e that a row is divided by, from the largest of its exponents (as above): the row maximum lands at 2^14.
// At least 2^-100, which keeps 2^-e and 2^e normal floats; rows that small lose bits that no output can show
__device__ inline int row_exponent(int largest) {
  const int e = (largest >> 7) - 1 - 127 - 14;
  return e < -100 ? -100 : e;
}
__device__ inline u32x4 bf16_to_f16(u32x4 v, float down) {
  u32x4 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float lo = __builtin_bit_cast(float, v[q] << 16) * down;
    const float hi = __builtin_bit_cast(float, v[q] & 0xFFFF0000u) * down;
    o[q] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)lo) |
           ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)hi) << 16);
  }
  return o;
}
template <int THREADS>
__device__ inline int row_max(i16x2 mx) {
  __shared__ int part[THREADS / 64];
  int m = mx[0] > mx[1] ? mx[0] : mx[1];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) m = part[w] > m ? part[w] : m;
  return m;
}

// bf16 [M][K] -> fp16 [M][K] * 2^-e[row] (exact: power-of-two shift of an 8-bit significand into 11 bits), with
// e[row] chosen so that the row maximum lands at 2^14; row_scale[row] = 2^e.  One workgroup per row; the row stays
// in registers between the maximum and the conversion (R chunks of eight elements per lane), so it is read once.
// Bound by its own launch and a row's round trip to memory.  Only the maximum's exponent counts, and packed 16-bit maxima
// find it at one and a half instructions an element instead of six (Llama-2-7B shapes at M = 387 and 1000, with the
// GEMM: K = 4096 46.6 -> 46.1 us, 49.8 -> 48.7; K = 11008 52.6 -> 51.3, 96.6 -> 94.6).
template <int THREADS, int R>
__global__ __launch_bounds__(THREADS) void bf16_rows_to_f16_kernel(const uint16_t* __restrict__ src,
                                                                   uint16_t* __restrict__ dst,
                                                                   float* __restrict__ row_scale, int K) {
  const size_t row = blockIdx.x;
  const u32x4* s = reinterpret_cast<const u32x4*>(src + row * K);
  u32x4* d = reinterpret_cast<u32x4*>(dst + row * K);
  const int nchunks = K / 8;  // K is a multiple of 128
  u32x4 v[R];
  i16x2 mx = {0, 0};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int ch = threadIdx.x + i * THREADS;
    v[i] = ch < nchunks ? s[ch] : u32x4{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) mx = __builtin_elementwise_max(mx, bf16_exponents(v[i][q]));
  const int e = row_exponent(row_max<THREADS>(mx));
  const float down = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);  // 2^-e, e in [-100, 113]
  if (threadIdx.x == 0) row_scale[row] = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int ch = threadIdx.x + i * THREADS;
    if (ch < nchunks) d[ch] = bf16_to_f16(v[i], down);
  }
}

// the same for rows longer than 32768 elements: two passes over global memory, eight elements per load
__global__ __launch_bounds__(1024) void bf16_rows_to_f16_long_kernel(const uint16_t* __restrict__ src,
                                                                     uint16_t* __restrict__ dst,
                                                                     float* __restrict__ row_scale, int K) {
  const size_t row = blockIdx.x;
  const u32x4* s = reinterpret_cast<const u32x4*>(src + row * K);
  u32x4* d = reinterpret_cast<u32x4*>(dst + row * K);
  const int nchunks = K / 8;
  i16x2 mx = {0, 0};
  for (int ch = threadIdx.x; ch < nchunks; ch += 1024) {
    const u32x4 v = s[ch];
#pragma unroll
    for (int q = 0; q < 4; ++q) mx = __builtin_elementwise_max(mx, bf16_exponents(v[q]));
  }
  const int e = row_exponent(row_max<1024>(mx));
  const float down = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
  if (threadIdx.x == 0) row_scale[row] = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
  for (int ch = threadIdx.x; ch < nchunks; ch += 1024) d[ch] = bf16_to_f16(s[ch], down);
}

// Second half of a K split: out[row, col .. col + 7] = epilogue(row factor x sum over the splits,
// in split order), one thread per segment of eight columns.
template <typename T>
__global__ __launch_bounds__(256) void w4a16_splitk_reduce_kernel(const float* __restrict__ partial, size_t split_stride,
                                                                  int ksplit, const float* __restrict__ row_scale,
                                                                  const void* sz, int G, uint16_t* out, int M, int N,
                                                                  Epilogue epi) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t segs = (size_t)N / 8;
  const size_t row = idx / segs;
  if (row >= (size_t)M) return;
  const int col = (int)(idx - row * segs) * 8;
  const f32x4* src = reinterpret_cast<const f32x4*>(partial + row * N + col);
  f32x4 sum[2];
  sum_splits(sum, ksplit, [&](int sp, int v) { return src[sp * (split_stride / 4) + v]; });
  const f32x4 lo = sum[0], hi = sum[1];
  const float rs = row_scale ? row_scale[row] : 1.f;
  float cf[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
  if (sz) column_factors(sz, G, col, cf);  // bf16 scales: the column's 2^E
  const float vals[8] = {lo[0] * rs * cf[0], lo[1] * rs * cf[1], lo[2] * rs * cf[2], lo[3] * rs * cf[3],
                         hi[0] * rs * cf[4], hi[1] * rs * cf[5], hi[2] * rs * cf[6], hi[3] * rs * cf[7]};
  const float mx = epi_store_row8<T>(epi, out, vals, (int)row, col, N);
  if (epi.row_absmax) atomicMax(reinterpret_cast<unsigned*>(epi.row_absmax) + row, __builtin_bit_cast(unsigned, mx));
}

}  // namespace

bool w4a16_prefill_supported(int dtype, size_t m, size_t n, size_t k, size_t g, int cus) {
  (void)g;
  // From 65 rows on.  49 to 64 rows as well where the columns alone fill the device several times over, or fill it with a
  // K long enough to split: there one 64-row block with the activations shared through LDS beats the decode
  // kernels, whose workgroups each pull all activations through their own loads (M = 64, decode / this: Llama-3-70B
  // gate_up 104 / 79 us, down 50 / 48, Llama-2-13B gate_up 37 / 33.5, Llama-2-7B gate_up even in fp16 and 31.5 / 31.1
  // in bf16; narrower shapes lose 10 to 60 %).  At 33 to 48 rows, three row tiles for the decode kernels and a quarter of
  // padding here, it is level or 5 to 10 % ahead on the wide shapes in fp16 (4096 x 22016 22.3 / 22.7, 4224 x 29440 28.9 /
  // 26.7, 70B gate_up 87 / 74); bf16, which pays the conversion launch, needs a long K for that (4096 x 32768 28.8 / 30.6),
  // and the long-K shapes do not win (70B down 39 / 42).
  const size_t ntiles = n / kTileN, kt = k / kTileK;
  const bool wide = ntiles >= 4 * (size_t)cus, long_k = ntiles >= 2 * (size_t)cus && kt >= 128;
  size_t min_m = wide && (dtype == KSQ_F16 || kt >= 48) ? 33 : wide || long_k ? 49 : 65;
  if (const char* e = tuning_env("KSQ_W4_PREFILL_MIN_M")) {  // tuning / test override
    const int v = atoi(e);
    if (v >= 1) min_m = (size_t)v;
  }
  return m >= min_m && n % 16 == 0 && m * k * 2 < 0x7FFFFF00ull && (k / kTileK) * 1024 < 0x7FFFFF00ull;
}

// bf16 route: fp16 copy of the activations + one float per row, in front of whatever else the plan needs
size_t w4a16_prefill_workspace_bytes(int dtype, size_t m, size_t k) {
  if (dtype != KSQ_BF16) return 0;
  return ((m * k * 2 + 255) / 256 * 256 + m * 4 + 255) / 256 * 256;
}

// ---- which form, which tile, which split: the smallest of these estimates (microseconds) -----------------------------
// Fitted by least squares to every form at 393 (M, K, N): the Llama-2-7B/13B and Llama-3-70B projections and random ones,
// M = 40 .. 4100, K = 512 .. 28288, N = 128 .. 57344 (rms 5 % for two k groups, 3 and 2 % for the others).  The choice is 1.0 %
// behind the fastest form of each case on average and 22 % at worst (2604 x 20096 x 384).  A k tile's time has a part for the
// workgroup, one for every row tile, and both grow with the share of the CUs in use, which share the L2s and the power.
// (A kernel of its own for 64 rows, four waves three k tiles ahead of themselves, was the fastest at none of them any more.)
namespace {

// two k groups, at most one workgroup per CU
double estimate_two_groups(int ct, int rt, size_t workgroups, int cus, size_t steps, size_t m, size_t n, size_t ksplit) {
  static const double kFixed[5] = {0, 5.08, 5.66, 6.12, 6.49}, kTile[5] = {0, 0.034, 0.163, 0.215, 0.299},
                      kRow[5] = {0, 0.064, 0.060, 0.085, 0.112}, kTileFill[5] = {0, 0.001, 0.085, 0.073, 0.027},
                      kRowFill[5] = {0, 0.018, 0.015, 0.024, 0.034};
  const double fill = (double)workgroups / (double)cus;
  // partial tiles out and in, and the second launch
  const double reduction =
      ksplit <= 1 ? 0.0 : 0.82 + 0.19 * (double)ksplit + 2.0 * (double)(ksplit * m * n) * 4.0 / 5.59e6;
  return kFixed[ct] + (double)steps * (kTile[ct] + kRow[ct] * rt + fill * (kTileFill[ct] + kRowFill[ct] * rt)) + reduction;
}

// eight waves side by side, rounds of one workgroup per CU
double estimate_eight_waves(int ct, int rt, size_t workgroups, int cus, size_t kt) {
  const size_t full = workgroups / (size_t)cus, rem = workgroups % (size_t)cus;
  const double fill = (double)rem / (double)cus;
  const double us =
      ct == 3 ? 7.54 + (double)kt * ((double)full * (0.551 + 0.264 * rt) + (rem ? 0.395 + 0.124 * rt + 0.121 * rt * fill : 0.0))
              : 7.77 + (double)kt * ((double)full * (0.669 + 0.350 * rt) + (rem ? 0.671 + 0.143 * rt + 0.153 * rt * fill : 0.0));
  // Grids of whole rounds: the fit, made mostly of grids with a rest, is some 4 % too high for them (no CU waits for the last
  // round's tail).  Where that decides against the next form -- 49 of 3960 shapes, four waves in 45 of them -- eight waves in
  // whole rounds were 2.5 % faster on average (48 measured): M = 4096, 4096 x 4096 107.9 against 113.0 us, M = 967, 1152 x 16336 36.6 against 38.9,
  // M = 2019, 4864 x 6080 98.9 against 107.4; slower in eight, by 7 % at most (M = 3516, 1280 x 44816 375 against 350).
  return rem == 0 ? 0.96 * us : us;
}

// four waves, rounds of two workgroups per CU
double estimate_four_waves(int ct, int rt, size_t workgroups, int cus, size_t kt) {
  const size_t two = 2 * (size_t)cus, full = workgroups / two, rem = workgroups % two;
  const double f1 = (double)rem / (double)cus, f2 = f1 - 1.0;  // share of the CUs with a first, a second workgroup
  double last = 0.0;
  if (ct == 3) {
    if (rem > 0) last = f1 <= 1.0 ? -0.124 + 0.122 * rt + 0.071 * rt * f1 : 0.313 + 0.204 * rt + 0.080 * rt * f2;
    return 7.98 + (double)kt * ((double)full * (0.296 + 0.293 * rt) + last);
  }
  if (rem > 0) last = f1 <= 1.0 ? 0.209 + 0.121 * rt + 0.072 * rt * f1 : 0.478 + 0.255 * rt + 0.100 * rt * f2;
  return 8.36 + (double)kt * ((double)full * (0.611 + 0.343 * rt) + last);
}

}  // namespace

// Tile shapes and K split; `workspace_bytes` is what remains behind the bf16 front part.  A function of ceil(M / 16), N, K
// and the workspace only, so the workspace can be sized by asking once per 16 rows.
PrefillPlan w4a16_prefill_plan(size_t m, size_t n, size_t k, int cus, size_t workspace_bytes) {
  PrefillPlan p{};
  m = (m + 15) / 16 * 16;
  const size_t ntiles = n / kTileN, kt = k / kTileK, mtiles = m / 16;
  auto need = [&](size_t x) { return x <= 1 ? (size_t)0 : x * m * n * 4; };
  auto env = [](const char* name, int lo, int hi) {  // tuning / test override, 0 = none
    const char* e = tuning_env(name);
    const int v = e ? atoi(e) : 0;
    return v >= lo && v <= hi ? v : 0;
  };
  const int want_rows = env("KSQ_W4_PREFILL_ROWS", 64, 128);

  // Row tiles per workgroup: every height that does not only pad the same number of blocks further.
  double best = 1e30;
  auto take = [&](double est, int rt, int nw, int kg, int ct, size_t c) {
    if (est >= best) return;
    best = est;
    p.rt = rt;
    p.nw = nw;
    p.kg = kg;
    p.ct = ct;
    p.ksplit = (int)c;
    p.partial_bytes = need(c);
  };
  for (int rt = 4; rt <= kMaxRT; ++rt) {
    const size_t mb = (mtiles + rt - 1) / rt;
    if (rt > 5 && mb == (mtiles + rt - 2) / (rt - 1)) continue;
    for (int ct = 1; ct <= 4; ++ct) {
      const size_t w = mb * ((ntiles + (size_t)(4 * ct) - 1) / (size_t)(4 * ct));
      // (workgroup ids go to the 8 XCDs in turn, y-slab after y-slab: what has to fit is every XCD's share)
      for (size_t c = 1; c <= 8 && (w + 7) / 8 * c <= (size_t)cus / 8 && (c == 1 || kt / c >= 8); ++c) {
        if (need(c) > workspace_bytes || (c > 1 && want_rows)) break;
        take(estimate_two_groups(ct, rt, w * c, cus, ((kt + c - 1) / c + 1) / 2 * 2, m, n, c), rt, 4, 2, ct, c);
      }
      if (!w4a16_prefill_form(4, 1, ct, rt)) continue;  // the same widths and heights with eight waves
      const size_t w8 = mb * ((ntiles + (size_t)(8 * ct) - 1) / (size_t)(8 * ct));
      take(estimate_four_waves(ct, rt, w, cus, kt), rt, 4, 1, ct, 1);
      take(estimate_eight_waves(ct, rt, w8, cus, kt), rt, 8, 1, ct, 1);
    }
  }
  if (want_rows) {  // tuning / test overrides; 64 rows: the two k groups with four row tiles
    if (want_rows == 64) {
      p.rt = p.nw = 4;
      p.ct = 4;
      if (const int v = env("KSQ_W4_PREFILL_NT", 1, 4)) p.ct = v;
    }
    if (const int v = env("KSQ_W4_PREFILL_WAVES", 4, 8)) p.nw = v == 8 ? 8 : 4;
    if (const int v = env("KSQ_W4_PREFILL_CT", 1, 4)) p.ct = v;
    if (const int v = env("KSQ_W4_PREFILL_RT", 4, kMaxRT)) p.rt = v;
    const size_t mb = (mtiles + p.rt - 1) / p.rt, nbw = (ntiles + (size_t)(4 * p.ct) - 1) / (size_t)(4 * p.ct);
    p.kg = want_rows == 64 || (p.nw == 4 && mb * nbw <= (size_t)cus) ? 2 : 1;
    const size_t want_split = (size_t)env("KSQ_W4_PREFILL_KSPLIT", 1, 8);
    size_t c = want_split && want_split <= kt ? want_split : 1;
    while (c > 1 && need(c) > workspace_bytes) --c;
    p.ksplit = (int)c;
    p.partial_bytes = need(c);
    if (const int v = env("KSQ_W4_PREFILL_KG", 1, 2)) p.kg = v;
    if (p.nw == 8) p.kg = 1;
    if (p.kg == 1) {  // what is compiled
      if (p.ct < 3) p.ct = 3;
      if (p.rt < 5) p.rt = 5;
    }
  }
  return p;
}

int w4a16_launch_prefill(int dtype, void* out, const void* act, const void* weight, const void* sz, size_t m,
                         size_t n, size_t k, size_t g, void* workspace, size_t workspace_bytes, hipStream_t s,
                         const Epilogue& epi) {
  KSQ_REQUIRE((reinterpret_cast<uintptr_t>(out) & 15) == 0 && n % 8 == 0, KSQ_ERR_INVALID_ARGUMENT,
              "prefill output must be 16-byte aligned");
  PrefillArgs a{};
  a.epi = epi;
  a.weight = weight;
  a.sz = sz;
  a.act = act;
  a.out = out;
  a.row_scale = nullptr;
  a.M = (int)m;
  a.N = (int)n;
  a.K = (int)k;
  a.KT = (int)(k / kTileK);
  a.G = (int)(k / g);
  a.ntiles = (int)(n / kTileN);
  const DeviceInfo* di = device_info();
  KSQ_REQUIRE(di != nullptr, KSQ_ERR_HIP, "no device");
  const size_t front = w4a16_prefill_workspace_bytes(dtype, m, k);
  KSQ_REQUIRE(front == 0 || (workspace != nullptr && workspace_bytes >= front), KSQ_ERR_WORKSPACE,
              "bf16 prefill needs its workspace");
  const PrefillPlan plan = w4a16_prefill_plan(m, n, k, di->cus, workspace ? workspace_bytes - front : 0);
  a.ksplit = plan.ksplit;
  a.partial = plan.ksplit > 1 ? reinterpret_cast<float*>(static_cast<char*>(workspace) + front) : nullptr;
  a.mblocks = (int)((m + 16 * plan.rt - 1) / (16 * plan.rt));
  const int bnt = plan.nw * plan.ct;
  a.nblocks = (a.ntiles + bnt - 1) / bnt;
  KSQ_REQUIRE((size_t)a.mblocks * a.nblocks < (1ull << 30), KSQ_ERR_UNSUPPORTED, "grid too large");
  const dim3 grid(tile_grid(a.mblocks, a.nblocks), (unsigned)plan.ksplit), block(64 * plan.nw * plan.kg);
  const int gpt = (int)(kTileK / g);
  if (dtype != KSQ_F16) note_launch("bf16_rows_to_f16_kernel grid=(%zu)", m);
  note_launch("w4a16_prefill_kernel<gpt=%d,rt=%d,nw=%d,kg=%d,ct=%d> grid=(%u,%u)", gpt, plan.rt, plan.nw, plan.kg, plan.ct, grid.x, grid.y);
  if (plan.ksplit > 1) note_launch("w4a16_splitk_reduce_kernel");
  bool launched;
  if (dtype == KSQ_F16) {
    launched = w4a16_prefill_launch_f16(a, gpt, plan, grid, block, s);
  } else {
    uint16_t* a16 = static_cast<uint16_t*>(workspace);
    float* row_scale = reinterpret_cast<float*>(static_cast<char*>(workspace) + (m * k * 2 + 255) / 256 * 256);
    const uint16_t* a_in = static_cast<const uint16_t*>(act);
    // (one chunk of eight elements per lane and more lanes, for few rows, measured the same)
    const dim3 rows((unsigned)m);
#define KSQ_ROWS(THREADS, R) hipLaunchKernelGGL((bf16_rows_to_f16_kernel<THREADS, R>), rows, dim3(THREADS), 0, s, a_in, a16, row_scale, (int)k)
    if (k <= 2048) KSQ_ROWS(256, 1);
    else if (k <= 4096) KSQ_ROWS(256, 2);
    else if (k <= 8192) KSQ_ROWS(256, 4);
    else if (k <= 16384) KSQ_ROWS(512, 4);
    else if (k <= 32768) KSQ_ROWS(1024, 4);
    else hipLaunchKernelGGL(bf16_rows_to_f16_long_kernel, rows, dim3(1024), 0, s, a_in, a16, row_scale, (int)k);
#undef KSQ_ROWS
    a.act = a16;
    a.row_scale = row_scale;
    launched = w4a16_prefill_launch_bf16(a, gpt, plan, grid, block, s);
  }
  KSQ_REQUIRE(launched, KSQ_ERR_UNSUPPORTED, "no prefill form with %d waves, %d k groups, %d x %d tiles", plan.nw, plan.kg, plan.rt,
              plan.ct);
  if (plan.ksplit > 1) {  // add the splits up and store
    const size_t stride = m * n;
    const dim3 rgrid((unsigned)((m * (n / 8) + 255) / 256));
    uint16_t* o = static_cast<uint16_t*>(out);
    if (dtype == KSQ_F16)
      hipLaunchKernelGGL(w4a16_splitk_reduce_kernel<_Float16>, rgrid, dim3(256), 0, s, a.partial, stride, plan.ksplit,
                         a.row_scale, (const void*)nullptr, a.G, o, (int)m, (int)n, epi);
    else
      hipLaunchKernelGGL(w4a16_splitk_reduce_kernel<__bf16>, rgrid, dim3(256), 0, s, a.partial, stride, plan.ksplit,
                         a.row_scale, sz, a.G, o, (int)m, (int)n, epi);
  }
  KSQ_HIP_TRY(hipGetLastError());
  return KSQ_OK;
}

}  // namespace ksq
