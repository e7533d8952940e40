// Large-M form of the int8-nk GEMM: tiles of 128 weight rows n x BM activation
// rows m (64 or 128) on V_MFMA_I32_32X32X32_I8.
//
// What bounds it is instruction issue: the exact epilogue (gemm.hip) costs 8
// VALU instructions (4 conversions, 4 fmas) per 16 x 16 outputs and 32-k block,
// and a matrix instruction takes a slot of the same port (measured: a 16x16x32
// product with its 8 instructions 36.4 clocks per SIMD, 9 slots of 4; counters
// of the gate/up launch at M = 16384: VALU issue full).  So the tile and the
// loop are chosen for few instructions besides those 8:
//  * 32x32x32 products: a quarter of the matrix instructions;
//  * operands global -> LDS by DMA, weights and tile-major codes as they are
//    stored, row-major codes gathered 16 bytes a lane into the order the
//    fragment reads take; a block's fragments read while the block before it is
//    folded, across the stage barriers too (the ring's third stage), and every
//    product issued one fold ahead of its own: neither LDS nor matrix-core
//    latency shows in a wavefront's fold;
//  * a wavefront holds 64 x BM/2 outputs (BM 128: 161 registers, 3 wavefronts a
//    SIMD; BM 64: 110, 4), so fragment reads are 4 per 4 (or 3 per 2) products.
// Several workgroups share a CU, so one's epilogue runs beside another's loop.
// Against the 16x16x32 kernel's 128 x 64 tiles (MI355X, us, weights rotated):
// SiLU gate/up N = 6144, K = 1024: M = 768 30.2 -> 21.1, 1024 26.8 -> 22.8,
// 2048 41.4 -> 39.3, 8192 146 -> 131; q/k/v N = 4096: M = 1024 20.8 -> 18.2,
// 1536 27.4 -> 23.4, 8192 98.7 -> 95.5; head N = 8200: M = 3000 82.4 -> 71.1.
// Also measured and not taken: the operands widened to f16 on the way into LDS
// (no conversions in the fold; 256 x 256 tiles), which power limits to 1.7 GHz.
#include <type_traits>

#include "gemm.h"
#include "ovh_common.h"

namespace ovh {

namespace {

constexpr int kTile = 1024;      // bytes of a 32-row x 32-k block tile
constexpr int kBN = 128;         // weight rows n per workgroup
constexpr int kThreads = 256;
constexpr int kSB = 2;           // blocks per stage
constexpr int kNst = 3;          // stages in the ring

__device__ __forceinline__ i32x16 mfma_i8(i32x4 a, i32x4 b) {
  const i32x16 z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, z, 0, 0, 0);
}

// Workgroup id -> (n tile, m tile): XCD x (id % 8) takes the x-th contiguous
// range of the tiles numbered in groups of kGroupN n tiles, m-major inside a
// group, so the tiles an XCD runs at once share few weight and activation rows
// and every XCD gets the same number whatever n_tiles is.
constexpr int kGroupN = 8;
__device__ __forceinline__ bool wide_tile_of(int id, int n_tiles, int m_tiles, int& nt, int& mt) {
  const int total = n_tiles * m_tiles, per = (total + 7) >> 3;
  const int slot = id >> 3, p = (id & 7) * per + slot;
  if (slot >= per || p >= total) return false;
  const int g = p / (kGroupN * m_tiles), r = p - g * kGroupN * m_tiles;
  const int left = n_tiles - g * kGroupN, w = left < kGroupN ? left : kGroupN;
  mt = r / w;
  nt = g * kGroupN + (r - mt * w);
  return true;
}

template <int BM, int MODE, bool TILED>
__global__ __launch_bounds__(kThreads, BM == 128 ? 3 : 4) void gemm_wide_kernel(const GemmArgs a) {
  constexpr int FM = BM / 64;                               // 32-row tiles of m per wavefront
  constexpr int kStageBytes = (kBN + BM) / 32 * kSB * kTile;  // weight tiles, then code tiles
  constexpr int kScaleBytes = BM * 16;                      // 4 blocks' scales of the rows m
  constexpr int kScaleOff = kNst * kStageBytes;
  constexpr int kLdsBytes = kScaleOff + 2 * kScaleBytes;
  constexpr bool DUMP = MODE == kDumpBlocks;                // block products out, no scales
  constexpr int kOps = 2 + FM;                              // DMA ops of a stage per wavefront
  constexpr int kScaleWaves = DUMP ? 0 : BM / 64;           // wavefronts with a scale op
  __shared__ __attribute__((aligned(16))) int8_t lds[kLdsBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1, r32 = lane & 31, hf = lane >> 5;
  const int n_tiles = (a.N + kBN - 1) / kBN, m_tiles = (a.M + BM - 1) / BM;
  int nt, mt;
  if (!wide_tile_of(blockIdx.x, n_tiles, m_tiles, nt, mt)) return;  // padding workgroup
  const int n0 = nt * kBN, m0 = mt * BM;
  const int Kb = a.Kb, ns = Kb / kSB;

  // ---- DMA: wavefront w moves block w & 1 of the stage's row tiles w >> 1 and
  // (w >> 1) + 2 of both operands, and wavefronts 0 and 1 64 rows each of the
  // scales of 4 blocks with every second stage.  A tile lands in LDS as it is
  // stored (weights and tile-major codes), or, from row-major codes, as lane l:
  // row l % 32, k 16 (l / 32) .. +15 (rows past M repeat the last; row tiles
  // past the tile-major codes' last too; neither is stored).
  const int bb0 = wave & 1, rt0 = wave >> 1;
  const int8_t* const wbase = a.W + ((int64_t)(n0 / 32 + rt0) * Kb + bb0) * kTile;
  const int64_t w_row2 = 2 * (int64_t)Kb * kTile;
  const int a_last = (a.M + 31) / 32 - 1;
  const int8_t* abase[FM];
  int avoff[FM];
#pragma unroll
  for (int t = 0; t < FM; ++t) {
    const int rt = rt0 + 2 * t;
    if constexpr (TILED) {
      abase[t] = a.aq + ((int64_t)min(m0 / 32 + rt, a_last) * Kb + bb0) * kTile;
      avoff[t] = lane * 16;
    } else {
      abase[t] = a.aq + (int64_t)m0 * a.Kp + bb0 * 32;
      avoff[t] = (min(m0 + rt * 32 + r32, a.M - 1) - m0) * (int)a.Kp + hf * 16;
    }
  }
  constexpr int kAStep = TILED ? kSB * kTile : kSB * 32;
  const float* const sbase =
      DUMP ? nullptr : a.asc + (int64_t)min(m0 + (wave & (BM / 64 - 1)) * 64 + lane, a.M - 1) * Kb;
  auto issue = [&](int s, int slot) __attribute__((always_inline)) {
    int8_t* const base = lds + slot * kStageBytes;
    if ((s & 1) == 0 && wave < kScaleWaves)
      __builtin_amdgcn_global_load_lds(
          static_cast<const void*>(sbase + 2 * s),
          (lds_void_t*)(lds + kScaleOff + ((s >> 1) & 1) * kScaleBytes + wave * 1024), 16, 0, 0);
    const int8_t* const ws = wbase + (int64_t)s * (kSB * kTile);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(ws + t * w_row2 + lane * 16),
                                       (lds_void_t*)(base + ((rt0 + 2 * t) * kSB + bb0) * kTile),
                                       16, 0, 0);
#pragma unroll
    for (int t = 0; t < FM; ++t)
      __builtin_amdgcn_global_load_lds(
          static_cast<const void*>(abase[t] + (int64_t)s * kAStep + avoff[t]),
          (lds_void_t*)(base + ((kBN / 32 + rt0 + 2 * t) * kSB + bb0) * kTile), 16, 0, 0);
  };
  // stage s landed for every wavefront; younger: the stage after it (its scale
  // op counted for wavefronts 0 and 1 when that stage is an even one)
  auto wait_stage = [&](int s) __attribute__((always_inline)) {
    if (s + 1 >= ns)
      wait_vm_lgkm<0>();
    else if ((s & 1) && wave < kScaleWaves)
      wait_vm_lgkm<kOps + 1>();
    else
      wait_vm_lgkm<kOps>();
    __builtin_amdgcn_s_barrier();
  };

  f32x16 f[2][FM];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) f[i][j][e] = 0.f;

  // a weight row's 16 k as two 8-byte pieces, 128 bytes apart (interleaved
  // tile); a code row's the same, or one 16-byte read
  const int piece = (r32 >> 4) * 512 + (r32 & 15) * 8 + hf * 256;
  const int wrd = wn * 2 * kSB * kTile + piece;
  const int ard = (kBN / 32 + wm * FM) * kSB * kTile + (TILED ? piece : lane * 16);
  auto read16 = [](const int8_t* p) __attribute__((always_inline)) {
    const int64_t lo = *reinterpret_cast<const int64_t*>(p);
    const int64_t hi = *reinterpret_cast<const int64_t*>(p + 128);
    return i32x4{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
  };
  i32x4 af[2][2], bf[2][FM];  // [register set][row tile]
  auto read_frags = [&](int slot, int bb, int set) __attribute__((always_inline)) {
    const int8_t* const base = lds + slot * kStageBytes + bb * kTile;
#pragma unroll
    for (int i = 0; i < 2; ++i) af[set][i] = read16(base + wrd + i * kSB * kTile);
#pragma unroll
    for (int j = 0; j < FM; ++j)
      bf[set][j] = TILED ? read16(base + ard + j * kSB * kTile)
                         : *reinterpret_cast<const i32x4*>(base + ard + j * kSB * kTile);
  };
  f32x4 sc[FM], scn[FM];  // this chunk's and the next chunk's scales of the lane's rows
  auto read_scales = [&](int slot, f32x4 (&d)[FM]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < FM; ++j)
      d[j] = *reinterpret_cast<const f32x4*>(lds + kScaleOff + slot * kScaleBytes +
                                             (wm * FM * 32 + j * 32 + r32) * 16);
  };
  i32x16 p[2];
  // The four products of a block (registers of set S): product k + 1 is issued
  // (the last one: the next block's first), then product k is folded.
  auto block = [&](int s, int bb, auto set) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;
#pragma unroll
    for (int k = 0; k < 2 * FM; ++k) {
      const int i = k / FM, j = k % FM;
      if (k + 1 < 2 * FM)
        p[(k + 1) & 1] = mfma_i8(af[S][(k + 1) / FM], bf[S][(k + 1) % FM]);
      else
        p[0] = mfma_i8(af[S ^ 1][0], bf[S ^ 1][0]);
      if constexpr (DUMP) {
        const int m = m0 + (wm * FM + j) * 32 + r32;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int n = n0 + wn * 64 + i * 32 + 8 * (e >> 2) + 4 * hf + (e & 3);
          if (m < a.M && n < a.N)
            a.dump[((int64_t)m * a.N + n) * Kb + 2 * s + bb] = p[k & 1][e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          f[i][j][e] = fmaf((float)p[k & 1][e], sc[j][bb], f[i][j][e]);
        // folded here: without this the compiler sinks the folds past the stage
        // loop's branches and keeps every product in registers until then
        asm volatile("" : "+v"(f[i][j]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

#pragma unroll
  for (int s = 0; s < kNst; ++s)
    if (s < ns) issue(s, s);
  // stage 0: the two after it may be in flight
  if (ns > 2) {
    if (wave < kScaleWaves) wait_vm_lgkm<2 * kOps + 1>(); else wait_vm_lgkm<2 * kOps>();
  } else {
    wait_vm_lgkm<0>();
  }
  __builtin_amdgcn_s_barrier();
  read_frags(0, 0, 0);
  read_scales(0, sc);
  p[0] = mfma_i8(af[0][0], bf[0][0]);
  int slot = 0;  // of stage 2 c
  auto next = [](int s) __attribute__((always_inline)) { return s == kNst - 1 ? 0 : s + 1; };
  for (int s = 0; s < ns; s += 2) {  // one chunk of 4 blocks
    const int slot1 = next(slot), slot2 = next(slot1);
    read_frags(slot, 1, 1);
    block(s, 0, S0{});
    // every wavefront has stage s's last fragments in registers: its slot is
    // free once they have passed the barrier
    wait_stage(s + 1);
    if (s + 3 < ns) issue(s + 3, slot);
    read_frags(slot1, 0, 0);
    block(s, 1, S1{});
    read_frags(slot1, 1, 1);
    block(s, 2, S0{});
    if (s + 2 < ns) {
      wait_stage(s + 2);
      if (s + 4 < ns) issue(s + 4, slot1);
      read_frags(slot2, 0, 0);
      read_scales(((s >> 1) + 1) & 1, scn);
    }
    block(s, 3, S1{});
#pragma unroll
    for (int j = 0; j < FM; ++j) sc[j] = scn[j];
    slot = slot2;
  }

  if constexpr (DUMP) return;
  if constexpr (MODE == kSiluQuant) {
    // Row tile i of the wavefront holds 16 gate rows, then the 16 up rows
    // of the same h columns (weight_interleave16): elements e and e + 8 of a
    // lane are gate and up of h column 16 i + 8 (e / 4) + 4 hf + e % 4.  The
    // lane pair l, l ^ 32 holds a row's 32-column block.
    if (n0 + wn * 64 >= a.N) return;  // wavefront-uniform
    f32x4 ws[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        ws[i][g] = *reinterpret_cast<const f32x4*>(a.ws + n0 + wn * 64 + i * 32 + 8 * g + 4 * hf);
    const int64_t col = (int64_t)(n0 + wn * 64) / 2;  // h column of the block
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + wm * FM * 32 + j * 32 + r32;
      float g[16], u[16], h[16], am = 0.f, nan = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          g[8 * i + e] = __fmul_rn(f[i][j][e], ws[i][e >> 2][e & 3]);
          u[8 * i + e] = __fmul_rn(f[i][j][e + 8], ws[i][2 + (e >> 2)][e & 3]);
        }
      silu_up_lanes(g, u, h);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        am = fmaxf(am, fabsf(h[e]));
        nan = __fadd_rn(nan, h[e]);
      }
      am = fmaxf(am, __shfl_xor(am, 32));
      const bool ok = __all(nan == nan && (am == 0.f || (am >= 0x1p-100f && am <= 0x1p120f)));
      const float qinv = am > 0.f ? __fdiv_rn(127.0f, am) : 0.f;
      uint32_t c[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) c[t] = quant_pack4(h + 4 * t, qinv, ok);
      if (m >= a.M) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int g4 = 0; g4 < 2; ++g4)
          *reinterpret_cast<uint32_t*>(
              a.hq + act_index(m, col + 16 * i + 8 * g4 + 4 * hf, a.hKp, a.h_tiled)) =
              c[2 * i + g4];
      if (hf == 0) a.hsc[(int64_t)m * (a.hKp / 32) + col / 32] = __fdiv_rn(am, 127.0f);
    }
    return;
  }

  // column scale, optional residual add, slice-aware store (slice widths are
  // multiples of 64: a 32-column tile lies in one slice, chosen in scalars)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n32 = n0 + wn * 64 + i * 32;  // wavefront-uniform
    int s = 0;
#pragma unroll
    for (int t = 1; t < kMaxSlices; ++t)
      if (t < a.nslices && n32 >= a.start[t]) s = t;
    float* const out = a.out[s];
    const int64_t ld = a.ld[s];
    const int s0 = a.start[s], s1 = a.start[s + 1];
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + wm * FM * 32 + j * 32 + r32;
      if (m >= a.M) continue;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int nb = n32 + 8 * g + 4 * hf;
        if (nb >= a.N) continue;
        const f32x4 ws = *reinterpret_cast<const f32x4*>(a.ws + nb);
        float* dst = out + (int64_t)m * ld + (nb - s0);
        const int lim = s1 - nb;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = __fmul_rn(f[i][j][4 * g + e], ws[e]);
        if (lim >= 4 && ((uintptr_t)dst & 15u) == 0) {
          f32x4 v;
          if (MODE == kAccumulate) {
            const f32x4 c = *reinterpret_cast<const f32x4*>(dst);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fadd_rn(o[e], c[e]);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = o[e];
          }
          *reinterpret_cast<f32x4*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < lim) dst[e] = MODE == kAccumulate ? __fadd_rn(o[e], dst[e]) : o[e];
        }
      }
    }
  }
}

template <int BM, int MODE>
hipError_t launch_wide_mode(const GemmArgs& a, hipStream_t st) {
  const int64_t tiles = (((int64_t)a.N + kBN - 1) / kBN) * (((int64_t)a.M + BM - 1) / BM);
  const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
  if (a.a_tiled)
    hipLaunchKernelGGL((gemm_wide_kernel<BM, MODE, true>), grid, dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((gemm_wide_kernel<BM, MODE, false>), grid, dim3(kThreads), 0, st, a);
  return hipGetLastError();
}

}  // namespace

// Where the form is the faster one (swept with the weights rotated through 600 MB,
// both code layouts, against the 16x16x32 kernel's tiles for the same shape).  SiLU
// from 640 rows (M = 600 within 2 %, 512 row by row equal).  Stores where the 128 x
// 64 tiles fill the four workgroup slots of every CU, or between 1024 and 2048 rows
// about half of them (K = 1024, N = 3072, M = 1280, 480 tiles, the other kernel /
// this one: row-major codes 20.2 / 18.3 us, tile-major 18.2 / 17.2), and where K is
// long enough for the ring, whose three stages fill and drain for nothing below
// (N = 8200, M = 1024, row-major: K = 128 1.46 times the other's time, 256 1.17,
// 512 1.04; over all N from 1024 to 12000 0.98 to 1.28 times at K = 256, 0.89 to
// 1.14 at 512), except that 512 pays from 4096 rows and columns (0.84 to 1.0, once
// 1.05).  Below 2048 rows the other kernel's 128 x 64 tiles come out even at 1024
// rows of 6144 columns or more (K = 1024 22.3 / 23.3 us, N = 6144; 31.3 / 32.2, 8200)
// and over rows of more than 10240 columns (K = 768, N = 12000, M = 1536 47.3 /
// 53.5); from K = 1536 the two are level there.
bool wide_applies(const GemmArgs& a, GemmMode mode) {
  if (a.Kb % 4 || a.W16) return false;
  if (mode == kSiluQuant) return a.M >= 640;
  if (mode != kStore && mode != kAccumulate && mode != kDumpBlocks) return false;
  if (a.Kb < 24 && (a.Kb < 16 || a.M < 4096 || a.N < 4096)) return false;
  if (a.M < 2048 && a.Kb < 48 && (a.N > 10240 || (a.M < 1088 && a.N >= 6144))) return false;
  const int64_t tiles = (((int64_t)a.N + kBN - 1) / kBN) * (((int64_t)a.M + 63) / 64);
  return a.M >= 1024 && tiles >= (a.M < 2048 ? 480 : 1000);
}

// 64-row tiles, except for the SiLU form from 4096 rows, where its longer
// epilogue gains from the larger tile (M = 4096 72.7 against 69.1 us, 2048 39.3
// against 38.4, 3000 55.5 against 56.5, whose 1152 tiles end in a half-full round),
// as long as there are enough of those tiles (64- / 128-row tiles, K = 1024: N = 128,
// M = 4096, 32 tiles 11.8 / 17.9; N = 896, M = 5000, 280 tiles 19.3 / 23.9, M = 8192,
// 448 tiles 25.2 / 25.1).
hipError_t launch_gemm_wide(const GemmArgs& a, GemmMode mode, hipStream_t st) {
  switch (mode) {
    case kStore: return launch_wide_mode<64, kStore>(a, st);
    case kAccumulate: return launch_wide_mode<64, kAccumulate>(a, st);
    case kDumpBlocks: return launch_wide_mode<64, kDumpBlocks>(a, st);
    case kSiluQuant:
      if (a.N % 128 || !a.hq || !a.hsc || a.hKp < a.N / 2) return hipErrorInvalidValue;
      return a.M >= 4096 && a.N / 128 * (((int64_t)a.M + 127) / 128) >= 448
                 ? launch_wide_mode<128, kSiluQuant>(a, st)
                 : launch_wide_mode<64, kSiluQuant>(a, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ovh
