// ovh_linear for few rows, in one launch: quantise_a_u8 and the int8-nk GEMM
// (cpp/src/backend/cpu/gemm.cpp:379-504) with nothing in between.
//
// As two launches a small linear is bound by their fixed costs: ~2.7 us for the
// quantiser and ~7 us for the GEMM at 40 rows (M = 40, K = 2048, N = 1024: 0.6 us
// of memory time), the GEMM's mostly a chain of ring stages of which each waits
// for memory.  Here a workgroup owns 16 rows x 32 columns and all of K: it asks
// for everything it needs at once (its fp32 rows into registers, its 32 weight
// rows, one contiguous run of Kb KiB, into LDS by DMA), quantises the rows into
// LDS codes while the weights arrive, and after one barrier folds the Kb blocks
// without another wait.  Every column tile's workgroup quantises its rows again
// (16 rows x K from L2, ~1 us of its eight wavefronts), which is why the form
// stops at the sizes of linear_small_applies.
#include "gemm.h"
#include "ovh_common.h"
#include "quant.h"

namespace ovh {

namespace {

constexpr int kRows = 16, kWaves = 8, kThreads = 64 * kWaves;

// Row r's blocks 8 p + lane / 8, p < P, into codes and scales: quant_block_lane's
// bytes and scales, at half its instructions.  The two quotients of a block are
// worked out by one of its 8 lanes (lane p for pass p), without the general
// division's exponent scaling: 127 / amax by one Newton step and one residual
// correction, amax / 127 by one correction, both equal to the IEEE quotient for
// every significand while amax is in [2^-100, 2^120] (all 2^23 of them, for a
// reciprocal one unit off either way: tests/short_quotients.cpp).
// Rows with a NaN or an amax outside that range (zero is inside) go the general
// way.
template <int P>
__device__ __forceinline__ void quantise_row(const float (&v)[P][4], const int (&nvalid)[P],
                                             int8_t* codes, float (*scales)[kRows][4], int r,
                                             int lane) {
  const int g = lane >> 3, sub = lane & 7;
  auto at = [&](int p) __attribute__((always_inline)) {
    return reinterpret_cast<uint32_t*>(codes + (8 * p + g) * 512 + (sub >> 1) * 128 + r * 8 +
                                       (sub & 1) * 4);
  };
  float am[P], nan = 0.f, lo = 1.f, hi = 0.f;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    float m = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      m = fmaxf(m, fabsf(v[p][e]));
      nan = __fadd_rn(nan, v[p][e]);
    }
    am[p] = group8_max(m);
    lo = fminf(lo, am[p] == 0.f ? 1.f : am[p]);
    hi = fmaxf(hi, am[p]);
  }
  if (!__all(nan == nan && lo >= 0x1p-100f && hi <= 0x1p120f)) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      uint32_t q;
      const float s = quant_block_lane(v[p], nvalid[p], &q);
      *at(p) = q;
      if (sub == 0) scales[(8 * p + g) >> 2][r][(8 * p + g) & 3] = s;
    }
    return;
  }
#pragma unroll
  for (int p0 = 0; p0 < P; p0 += 8) {
    float a = am[p0];
#pragma unroll
    for (int i = 1; i < 8 && p0 + i < P; ++i) a = sub == i ? am[p0 + i] : a;
    const float y0 = __builtin_amdgcn_rcpf(a), y = fmaf(fmaf(-a, y0, 1.f), y0, y0);
    float inv = __fmul_rn(127.f, y);
    inv = fmaf(fmaf(-a, inv, 127.f), y, inv);
    inv = a > 0.f ? inv : 0.f;
    constexpr float c = 1.f / 127.f;
    const float s0 = __fmul_rn(a, c), s = fmaf(fmaf(-127.f, s0, a), c, s0);
    const int b = 8 * (p0 + sub) + g;
    if (p0 + sub < P) scales[b >> 2][r][b & 3] = s;
    const int ib = __float_as_int(inv);
    auto code = [&](int p, int lane_p_inv) __attribute__((always_inline)) {
      *at(p) = quant_pack4(v[p], __int_as_float(lane_p_inv), true);
    };
    // lane i of the 8 (ds_swizzle: and 0x18, or i)
    if (p0 + 0 < P) code(p0 + 0, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 0 << 5));
    if (p0 + 1 < P) code(p0 + 1, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 1 << 5));
    if (p0 + 2 < P) code(p0 + 2, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 2 << 5));
    if (p0 + 3 < P) code(p0 + 3, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 3 << 5));
    if (p0 + 4 < P) code(p0 + 4, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 4 << 5));
    if (p0 + 5 < P) code(p0 + 5, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 5 << 5));
    if (p0 + 6 < P) code(p0 + 6, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 6 << 5));
    if (p0 + 7 < P) code(p0 + 7, __builtin_amdgcn_ds_swizzle(ib, 0x18 | 7 << 5));
  }
}

// One 16 x 16 tile from the staged operands (wl: its half of the weight row
// tile, block b at 1024 b).
template <int KBM, bool ADD>
__device__ __forceinline__ void tile_16(int64_t M, int64_t N, int Kb, const int8_t* wl,
                                        const int8_t* cl, const float (*scales)[kRows][4],
                                        const float* __restrict__ ws, float* __restrict__ C,
                                        int64_t ldc, int64_t m16, int64_t n16, int lane) {
  const int q4 = lane >> 4, r = lane & 15;
  f32x4 f = {0.f, 0.f, 0.f, 0.f};
  const int8_t* const wf = wl + lane * 8;
  const int8_t* const cf = cl + lane * 8;
  // Groups of 8 blocks: a group's products are issued, the next group's fragments
  // read, then the group is folded.  The blocks past Kb in the last group have
  // zero codes and scales (the passes above wrote them), and their weights may be
  // anything: not folded.
  int64_t wa[8], ca[8];
  f32x4 sa[2];
  auto read = [&](int b0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      wa[i] = *reinterpret_cast<const int64_t*>(wf + (b0 + i) * 1024);
      ca[i] = *reinterpret_cast<const int64_t*>(cf + (b0 + i) * 512);
    }
    sa[0] = *reinterpret_cast<const f32x4*>(&scales[b0 >> 2][r][0]);
    sa[1] = *reinterpret_cast<const f32x4*>(&scales[(b0 >> 2) + 1][r][0]);
  };
  read(0);
  for (int b0 = 0; b0 < Kb; b0 += 8) {
    i32x4 acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      acc[i] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wa[i], ca[i], i32x4{0, 0, 0, 0}, 0, 0, 0);
    const f32x4 s0 = sa[0], s1 = sa[1];
    if (b0 + 8 < Kb) read(b0 + 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float s = i < 4 ? s0[i & 3] : s1[i & 3];
      if (b0 + i < Kb) {  // uniform
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = fmaf((float)acc[i][e], s, f[e]);
      }
    }
  }
  // lane: columns n16 + 4 q4 .. +3 of row m16 + r
  const int64_t m = m16 + r, nb = n16 + 4 * q4;
  if (m >= M || nb >= N) return;
  const f32x4 sw = *reinterpret_cast<const f32x4*>(ws + nb);  // padded past N
  float* const dst = C + m * ldc + nb;
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = __fmul_rn(f[e], sw[e]);
  if (nb + 4 <= N && ((uintptr_t)dst & 15u) == 0) {
    f32x4 x = f32x4{o[0], o[1], o[2], o[3]};
    if constexpr (ADD) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(dst);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = __fadd_rn(o[e], y[e]);
    }
    *reinterpret_cast<f32x4*>(dst) = x;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (nb + e < N) dst[e] = ADD ? __fadd_rn(o[e], dst[e]) : o[e];
  }
}

// COLS: columns per workgroup, 32 or 128 (a divisor of the weight's row padding).  KBM: Kb <= KBM, a multiple of 8.  VEC4: K % 4 == 0 and A 16-byte aligned.
template <int COLS, int KBM, bool ADD, bool VEC4>
__global__ __launch_bounds__(kThreads) void linear_small_kernel(
    int64_t M, int64_t N, int64_t K, int Kb, const float* __restrict__ A,
    const int8_t* __restrict__ W, const float* __restrict__ ws, float* __restrict__ C,
    int64_t ldc) {
  // the weights in an array of their own: the code stores below then need not
  // wait for their DMA
  __shared__ __attribute__((aligned(16))) int8_t wlds[COLS / 32 * KBM * 1024];
  // [block][k / 8 % 4][row][8], and [block / 4][row][block % 4]
  __shared__ __attribute__((aligned(16))) int8_t codes[KBM * 512];
  __shared__ __attribute__((aligned(16))) float scales[KBM / 4][kRows][4];
  constexpr int RPW = kRows / kWaves;  // rows per wavefront
  static_assert(kRowPad % COLS == 0 && COLS / 16 <= kWaves, "in-bounds weights; a tile a wavefront");
  constexpr int P = KBM / 8;  // passes of 8 blocks over a row
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n_tiles = (N + COLS - 1) / COLS;
  const int64_t mt = blockIdx.x / n_tiles, nt = blockIdx.x - mt * n_tiles;
  const int64_t m0 = mt * kRows, n0 = nt * COLS;

  // ---- this wavefront's rows (past M: the last row again, not stored)
  const int g = lane >> 3, sub = lane & 7;
  float v[RPW][P][4];
  int nvalid[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int64_t k0 = (int64_t)(8 * p + g) * 32 + sub * 4, rem = K - k0;
    nvalid[p] = rem >= 4 ? 4 : (rem > 0 ? (int)rem : 0);
  }
#pragma unroll
  for (int h = 0; h < RPW; ++h) {
    const int64_t r = m0 + RPW * wave + h;
    const float* row = A + (r < M ? r : M - 1) * K;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t k0 = (int64_t)(8 * p + g) * 32 + sub * 4;
      if constexpr (VEC4) {
        f32x4 x = {0.f, 0.f, 0.f, 0.f};
        if (nvalid[p]) x = *reinterpret_cast<const f32x4*>(row + k0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[h][p][e] = x[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[h][p][e] = e < nvalid[p] ? row[k0 + e] : 0.f;
      }
    }
  }
  // ---- the weight row tiles, block b by wavefront b % 8 (the scheduling barrier
  // keeps the loads above first: the quantiser waits for them alone).  Rows are
  // padded to a multiple of 128.
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < COLS / 32; ++t) {
    const int8_t* const wt = W + (nt * (COLS / 32) + t) * (int64_t)Kb * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int b = i * kWaves + wave;
      if (b < Kb)  // wavefront-uniform
        __builtin_amdgcn_global_load_lds(static_cast<const void*>(wt + (int64_t)b * 1024),
                                         (lds_void_t*)(wlds + (t * KBM + b) * 1024), 16, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- quantise: 8 lanes per block
#pragma unroll
  for (int h = 0; h < RPW; ++h)
    quantise_row<P>(v[h], nvalid, codes, scales, RPW * wave + h, lane);
  wait_vm_lgkm<0>();  // this wavefront's weights landed
  __syncthreads();    // and the others', and the codes written

  // ---- one 16 x 16 tile per wavefront, block by block
  if (wave < COLS / 16 && n0 + 16 * wave < N)
    tile_16<KBM, ADD>(M, N, Kb, wlds + (wave >> 1) * KBM * 1024 + (wave & 1) * 512, codes, scales, ws,
                      C, ldc, m0, n0 + 16 * wave, lane);
}

int64_t workgroups(int64_t M, int64_t N, int cols) {
  return (M + kRows - 1) / kRows * ((N + cols - 1) / cols);
}

bool vec4_rows(const float* A, const DeviceWeight& w) {
  return w.K % 4 == 0 && ((uintptr_t)A & 15u) == 0;
}

template <int COLS, int KBM>
hipError_t launch_small(int64_t M, const float* A, const DeviceWeight& w, float* C, int64_t ldc,
                        bool add, hipStream_t st) {
  const int64_t grid = workgroups(M, w.N, COLS);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kThreads), 0, st, M, w.N, w.K, (int)w.Kb,
                       A, w.q, w.scale, C, ldc);
    return hipGetLastError();
  };
  const bool vec4 = vec4_rows(A, w);
  if (add)
    return vec4 ? go(linear_small_kernel<COLS, KBM, true, true>)
                : go(linear_small_kernel<COLS, KBM, true, false>);
  return vec4 ? go(linear_small_kernel<COLS, KBM, false, true>)
              : go(linear_small_kernel<COLS, KBM, false, false>);
}

// Columns per workgroup, or 0 where two launches are faster.  A workgroup's time
// hardly depends on how many others are resident, so a form pays while one round
// of resident workgroups covers the call (us a call one launch / two): K <= 1024,
// 32 columns (three workgroups a CU) M = 64, N = 2048 7.9 / 10.6, at 768 workgroups
// 9.7 / 10.9, at 1024 11.3 / 10.6; 128 columns (one a CU) M = 333, N = 1501
// (252 workgroups) 7.9 / 10.6, at 384 12.1 / 10.7.  K = 2048, 32 columns (one a CU):
// M = 40, N = 1024 8.4 / 10.6, at 416 workgroups 15.8 / 10.9.  K = 3072: 12.0 / 10.7
// at 96 workgroups (the row quantisation alone is 1.5 us), not taken.  Rows loaded
// value by value (not VEC4) take four times the loads, and long ones not two
// workgroups a CU for the time of one: K = 1001, N = 1000, 32 columns, 224 workgroups
// 8.2 / 10.7, 320 11.8 / 10.3 (128 columns, 80 workgroups, 9.5), 128 columns at 240
// workgroups 9.7 / 10.7, at 256 10.9 / 10.6 (where K has a 128-k tail the two launches
// are slower: K = 850 13.4 of them); K = 250, 512 workgroups 7.6 / 10.6.
int small_cols(int64_t M, const DeviceWeight& w, bool vec4) {
  if (w.Kb > 64) return 0;
  if (w.Kb > 32) return workgroups(M, w.N, 32) <= 256 ? 32 : 0;
  const bool light = vec4 || w.Kb <= 24;
  if (workgroups(M, w.N, 32) <= (light ? 512 : 256)) return 32;
  return workgroups(M, w.N, 128) <= (light || w.Kb % 4 ? 256 : 240) ? 128 : 0;
}

}  // namespace

bool linear_small_applies(int64_t M, const float* A, const DeviceWeight& w, const float* C,
                          int64_t ldc) {
  if (w.Kb < 1 || M < 1 || M > 16384) return false;
  // C written while other workgroups still read A: not where they overlap
  const float *a1 = A + M * w.K, *c1 = C + (M - 1) * ldc + w.N;
  if (C < a1 && A < c1) return false;
  return small_cols(M, w, vec4_rows(A, w)) != 0;
}

hipError_t launch_linear_small(int64_t M, const float* A, const DeviceWeight& w, float* C,
                               int64_t ldc, bool add, hipStream_t st) {
  const int cols = small_cols(M, w, vec4_rows(A, w));
  if (cols == 32 && w.Kb <= 32) return launch_small<32, 32>(M, A, w, C, ldc, add, st);
  if (cols == 32 && w.Kb <= 64) return launch_small<32, 64>(M, A, w, C, ldc, add, st);
  if (cols == 128 && w.Kb <= 32) return launch_small<128, 32>(M, A, w, C, ldc, add, st);
  return hipErrorInvalidValue;
}

}  // namespace ovh
