// Dense GEMMs of mid-size batches for gfx950: out [m, n] = A [m, k] . W [n, k]^T
// with bf16 operands, or e4m3 operands and UE8M0 scales (one per A row and
// 128 k, one per 128 W rows and 128 k), fp32 accumulation.
//
// What bounds such a call: not HBM alone.  A block reads its A rows as well as
// its W rows, and a CU takes in ~64 GB/s (55-65, fitted to the measured times
// of calls of one round, where the tiles' row bytes are known), against the
// ~23 GB/s that is its share of HBM.  So a tile of TM x TN costs a CU (TM + TN)
// x row bytes at that rate, and what matters is that all 256 CUs have a tile
// and that TM + TN is no larger than that takes.  The 128 x 256 tiles of
// gemm_fp8_moe.hip leave most CUs idle at these sizes, and the 16-row GEMV
// blocks read all of A for every 16 weight rows in the waves' own loads.  Here
// the tile is chosen per call (PickTile) from 16-row steps both ways.  Which
// calls run here, and both sides' times: dense_route.hpp, gemm_mfma.hip.
//
// A block is 4 multiplying and 4 loading waves: a wave issues in order, and a
// DMA that the full load queue does not take yet would hold back the MFMAs
// behind it (one kind of wave doing both: 5-15 % slower).  A K step is 256
// bytes of every tile row, moved into LDS by DMA (global_load_lds_dwordx4, 4
// rows x 256 bytes an instruction, the same number from every loading wave),
// kStages steps deep: one wait and one barrier a step.  16-byte chunk c of row
// r sits in slot c ^ (r & 15) of its 256 bytes, so that a fragment read (16
// rows, one chunk each) covers the 64 banks once.  The multiplying waves split
// the step's K, not the tile: each reads its share of every row, so an LDS
// byte is read once (bf16: four k quarters; e4m3: two 128-k halves, times two
// halves of the W rows), and the waves' sums meet in LDS at the end in a fixed
// order, from which whole output rows are stored.  The MFMA's first operand is
// W, so a lane's four results are four consecutive columns of one row.
//
// e4m3 NaN codes count as 0 and raise the code bit, as the reference decodes
// them (plugins/kernels/deepseek-v4-sm89/native/deepseek_fp8_gemm.cu:11-70):
// a code turns every sum over its row into a NaN, so an element that came out
// non-finite looks for codes in its two operand rows and, finding one, is
// summed again the reference's way.  A 0xFF scale's block adds nothing, also
// where the caller asked for no code check (the grouped GEMM): the sum from
// before the block's MFMA is kept, so its codes are never seen.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace pih_amd {
namespace {

enum : int { kTileBf16 = 0, kTileFp8 = 1 };
constexpr uint32_t SB = 256;  // bytes of a row per K step
constexpr uint32_t kGridStep = kWalkStep;  // ... in the kernel that walks tiles
constexpr uint32_t kThreads = 512;  // waves 0-3 multiply, waves 4-7 load
constexpr uint32_t kMaxKb = 64;  // e4m3: K / 128 the scale panels hold
constexpr uint32_t kOutPitch = 144;  // staged output rows: 128 bytes + 16
// bytes between the blocks of the waves' sums: the four 16-lane groups 16
// bytes off a bank period, so that a row's columns are read without conflicts
constexpr uint32_t kSumGroup = 272, kSumBlock = 4 * kSumGroup;

struct TileParams {
  const uint8_t* a;
  const uint8_t* w;
  const uint8_t* a_scale;
  const uint8_t* w_scale;
  void* out;
  uint32_t* err;
  uint32_t m, n, row_bytes, m_tiles, n_tiles, problems;
  uint32_t a_row_stride, a_prob_row;
  uint64_t out_row_stride;
  uint32_t out_prob_col;
  uint32_t out_f32, write_nonfinite, check_codes;
  uint32_t err_code, err_scale, err_nonfinite;
};

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Output element (A row ar, column col of problem prob) the reference's way,
// by a whole wave (every lane the same element): per 128-k block an fp32 sum
// of decoded e4m3 products in k order with NaN codes as 0, the blocks added
// in order, a block with a 0xFF scale skipped before it is read.  Lane b
// takes block b (a product of two codes is exact in fp32, so the FMA rounds
// as the reference's multiply and add).  False when neither operand row holds
// a code.  A call with one code in an A row or a W row (alone on the stream,
// us, A / W; clean 6-9): 4096 -> 1024 at M 16 16.8 / 16.1, 8192 -> 4096 at M 4
// 24 / 15, 2048 -> 4096 at M 64 23 / 22; with a lane per element, walking all
// of K alone, 2627 / 591, 5330 / 1051 and 1324 / 513.
__device__ __forceinline__ bool code_element(const TileParams& p, uint64_t ar, uint32_t prob, uint32_t col, float& sum,
                                             uint32_t& bits) {
  const uint32_t RB = p.row_bytes, KB = RB / 128, lane = threadIdx.x & 63, b = min(lane, KB - 1);
  const v4i* const ap = reinterpret_cast<const v4i*>(p.a + ar * RB) + b * 8;
  const v4i* const wp = reinterpret_cast<const v4i*>(p.w + ((uint64_t)prob * p.n + col) * RB) + b * 8;
  const uint32_t as = p.a_scale[ar * KB + b], ws = p.w_scale[((uint64_t)prob * (p.n / 128) + col / 128) * KB + b];
  const bool live = lane < KB, skip = as == 0xffu || ws == 0xffu;
  uint32_t nan = 0;
  float local = 0.0f;
#pragma unroll 1
  for (int c = 0; c < 8; ++c) {
    const v4i x = ap[c], y = wp[c];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t nx = e4m3_nan_bytes((uint32_t)x[q]), ny = e4m3_nan_bytes((uint32_t)y[q]);
      nan |= nx | ny;
      const int xa = (int)e4m3_nan_to_zero((uint32_t)x[q], nx), xw = (int)e4m3_nan_to_zero((uint32_t)y[q], ny);
      const v2f a0 = __builtin_amdgcn_cvt_pk_f32_fp8(xa, false), a1 = __builtin_amdgcn_cvt_pk_f32_fp8(xa, true);
      const v2f w0 = __builtin_amdgcn_cvt_pk_f32_fp8(xw, false), w1 = __builtin_amdgcn_cvt_pk_f32_fp8(xw, true);
      local = __builtin_fmaf(a0[0], w0[0], local);
      local = __builtin_fmaf(a0[1], w0[1], local);
      local = __builtin_fmaf(a1[0], w1[0], local);
      local = __builtin_fmaf(a1[1], w1[1], local);
    }
  }
  const int part = __builtin_bit_cast(int, local * ue8m0_value(as) * ue8m0_value(ws));
  const uint64_t add = __builtin_amdgcn_ballot_w64(live && !skip);
  sum = 0.0f;
#pragma unroll 1
  for (uint32_t i = 0; i < KB; ++i)
    if ((add >> i) & 1) sum = sum + __builtin_bit_cast(float, __builtin_amdgcn_readlane(part, i));
  bits = __builtin_amdgcn_ballot_w64(live && skip) ? kErrScale : 0u;
  if (__builtin_amdgcn_ballot_w64(live && !skip && nan)) bits |= kErrCode;
  return __builtin_amdgcn_ballot_w64(live && nan) != 0;
}

__device__ __forceinline__ bool finite4(v4f v) {
  return __builtin_isfinite(v[0]) && __builtin_isfinite(v[1]) && __builtin_isfinite(v[2]) && __builtin_isfinite(v[3]);
}

// four columns from `col` of output row `row`, or one of them
__device__ __forceinline__ void store4(const TileParams& p, uint32_t row, uint32_t prob, uint32_t col, v4f v) {
  const uint64_t o = (uint64_t)row * p.out_row_stride + (uint64_t)prob * p.out_prob_col + col;
  if (p.out_f32) *reinterpret_cast<v4f*>(static_cast<float*>(p.out) + o) = v;
  else
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + o) =
        uint2{f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3])};
}
__device__ __forceinline__ void store1(const TileParams& p, uint32_t row, uint32_t prob, uint32_t col, float v) {
  const uint64_t o = (uint64_t)row * p.out_row_stride + (uint64_t)prob * p.out_prob_col + col;
  if (p.out_f32) static_cast<float*>(p.out)[o] = v;
  else static_cast<uint16_t*>(p.out)[o] = (uint16_t)f32_to_bf16_bits(v);
}

// Element v at (row, col) after the look for codes; a non-finite one raises
// its bit and is stored unless the caller leaves such elements out.
__device__ __forceinline__ void store_looked_at(const TileParams& p, uint32_t row, uint32_t prob, uint32_t col, float v,
                                                uint32_t& bad) {
  const bool fin = __builtin_isfinite(v);
  if (!fin) bad |= kErrNonFinite;
  if (fin || !p.err_nonfinite || p.write_nonfinite) store1(p, row, prob, col, v);
}

// The non-finite element v at (row, col), by a whole wave, its lane `by`
// storing: e4m3 operands that hold a NaN code get the reference's sum and its
// bits.
__device__ __forceinline__ void store_nonfinite(const TileParams& p, uint32_t row, uint32_t prob, uint32_t col, float v,
                                                uint32_t by, uint32_t& bad) {
  float sum;
  uint32_t bits;
  const bool code = code_element(p, (uint64_t)row * p.a_row_stride + (uint64_t)prob * p.a_prob_row, prob, col, sum, bits);
  if ((threadIdx.x & 63) != by) return;
  if (code) bad |= bits;
  store_looked_at(p, row, prob, col, code ? sum : v, bad);
}

__device__ __forceinline__ void raise(const TileParams& p, uint32_t bad) {
  const uint32_t bits = ((bad & kErrCode) ? p.err_code : 0u) | ((bad & kErrScale) ? p.err_scale : 0u) |
                        ((bad & kErrNonFinite) ? p.err_nonfinite : 0u);
  // (the waves of a whole output may have the same to say: only one that
  // finds it unsaid adds to the queue at the flag)
  if (bits & ~__hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(p.err, bits);
}

// A block under a 0xFF scale adds nothing, whatever its codes: a lane's four
// results belong to one A row (scale byte as) and one 128-row W block (ws),
// and the sum before the MFMA is kept.  (Zeroed operands or a scale of 0
// would do for finite values only: a NaN code in the other operand, or in
// the skipped one, stays a NaN.)
__device__ __forceinline__ v4f without_ff_block(uint32_t ws, uint32_t as, v4f before, v4f after) {
  const bool skip = ws == 0xffu || as == 0xffu;
  return v4f{skip ? before[0] : after[0], skip ? before[1] : after[1], skip ? before[2] : after[2],
             skip ? before[3] : after[3]};
}

template <int OP, int MB, int NB>
struct TileShape {
  static constexpr uint32_t TM = 16 * MB, TN = 16 * NB, kStage = (TM + TN) * SB;
  // 256 bytes of W scales and TM x kMaxKb of A scales, each in whole DMAs
  static constexpr uint32_t kPanel = OP == kTileFp8 ? 256 + TM * kMaxKb : 0;
  static constexpr uint32_t kLds = 160 * 1024 - 512;
  static constexpr int kLoads = MB + NB;  // DMAs per wave and step
  static constexpr int kFit = (int)((kLds - kPanel) / kStage);
  // as deep as LDS allows, at most 8 steps and 63 loads in flight
  static constexpr int kStages = std::min(std::min(kFit, 8), 63 / kLoads + 1);
  static constexpr int kParts = OP == kTileFp8 ? 2 : 4;  // waves that share an output
  // accumulator sets a wave takes turns with, as far as registers go.  An
  // fp32 sum of K products rounds at every MFMA, by the size it has reached:
  // off 64 bits at K 4096 (bf16, fp32 output, normwise) 1.89e-7 with one set,
  // 1.34e-7 with two, 1.03e-7 with four; the GEMV's 8 waves 1.37e-7, its 16
  // waves of 2-4 rows 1.13e-7, a K split in eight 1.37e-7.  A call pays 1-2 %
  // (4096 -> 1024 at M 8 6.0 -> 6.15 us).  (e4m3: 5.5e-5 with any number, the
  // instruction's own rounding.)
  static constexpr int kSets = OP == kTileFp8 ? 1 : MB == 1 && NB <= 4 ? 4 : MB * NB <= 24 ? 2 : 1;
  static constexpr uint32_t kSums = kParts * MB * NB * kSumBlock;
  static constexpr uint32_t kRing = kStages * kStage > kSums ? kStages * kStage : kSums;
};

template <int OP, int MB, int NB>
__global__ __launch_bounds__(kThreads, 1) void tile_gemm_kernel(TileParams p) {
  using S = TileShape<OP, MB, NB>;
  constexpr uint32_t TM = S::TM, TN = S::TN;
  constexpr int ST = S::kStages, NL = S::kLoads;
  static_assert(ST >= 2, "two stages");
  constexpr bool kFp8 = OP == kTileFp8;
  // e4m3: the two wave pairs take half of the W blocks each, or of the A
  // blocks; with an odd number of both one pair does all (the loads bound it)
  constexpr bool kSplitN = kFp8 && NB % 2 == 0, kSplitM = kFp8 && !kSplitN && MB % 2 == 0;
  constexpr bool kOnePair = kFp8 && !kSplitN && !kSplitM;
  constexpr int MW = kSplitM ? MB / 2 : MB, NW = kSplitN ? NB / 2 : NB;  // a wave's blocks
  __shared__ __align__(16) uint8_t smem[S::kRing + S::kPanel];
  const uint32_t tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3;
  const bool loader = wave >= 4;
  const uint32_t lds0 = lds_addr(smem);

  // tile t of (problem, N tile, M tile), M fastest: the tiles that share W
  // rows run side by side on one XCD, which walks a contiguous range
  const uint32_t total = p.m_tiles * p.n_tiles * p.problems, per = (total + 7) / 8;
  const uint32_t t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || t >= total) return;
  const uint32_t mt = t % p.m_tiles, rest = t / p.m_tiles, nt = rest % p.n_tiles, prob = rest / p.n_tiles;
  const uint32_t row0 = mt * TM, col0 = nt * TN;
  const uint32_t RB = p.row_bytes, steps = RB / SB;
  uint32_t bad = 0;

  // tile rows past m read row m - 1; they are not stored
  auto a_row = [&](uint32_t r) -> uint64_t {
    return (uint64_t)min(row0 + r, p.m - 1) * p.a_row_stride + (uint64_t)prob * p.a_prob_row;
  };
  const uint8_t* const w_base = p.w + ((uint64_t)prob * p.n + col0) * RB;

  // ---- DMA sources: instruction i of wave w moves rows 16 i + 4 w + (l >> 4),
  // lane l's 16 bytes to slot l & 15 (chunk (l & 15) ^ (row & 15))
  const uint32_t drow = 4 * wv + lg, dchunk = (lr ^ drow) << 4;
  uint32_t a_off[MB], w_off[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) a_off[i] = (uint32_t)(a_row(16 * i + drow) * RB) + dchunk;
#pragma unroll
  for (int i = 0; i < NB; ++i) w_off[i] = (16 * i + drow) * RB + dchunk;
  auto issue = [&](uint32_t stage, uint32_t j, auto NT) __attribute__((always_inline)) {
    const uint32_t lds = lds0 + stage * S::kStage + wv * 1024;
    const uint8_t* ab = uniform_ptr(p.a + (uint64_t)j * SB);
    const uint8_t* wb = uniform_ptr(w_base + (uint64_t)j * SB);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if constexpr (decltype(NT)::value) dma16nt(wb, w_off[i], lds + TM * SB + i * 4096);
      else dma16(wb, w_off[i], lds + TM * SB + i * 4096);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) dma16(ab, a_off[i], lds + i * 4096);
  };

  // ---- e4m3: the tile's scales, whole panels by dword DMA ahead of the
  // first step: KB bytes of W scales, TM rows of KB bytes of A scales
  const uint32_t KB = RB / 128;  // e4m3 only
  const uint8_t* const pw = smem + S::kRing;
  const uint8_t* const pa = pw + 256;
  if (kFp8 && loader) {
    const uint32_t q4 = KB / 4;  // dwords per row (the launcher checks KB % 4)
    if (wv == 0) {
      const uint8_t* src = p.w_scale + ((uint64_t)prob * (p.n / 128) + col0 / 128) * KB;
      dma4v(src + 4 * min(lane, q4 - 1), lds0 + S::kRing);
    }
    for (uint32_t b = wv * 64; b < TM * q4; b += 256) {
      const uint32_t i = min(b + lane, TM * q4 - 1);
      dma4v(p.a_scale + a_row(i / q4) * KB + 4 * (i % q4), lds0 + S::kRing + 256 + 4 * b);
    }
  }

  // a wave's accumulators [set][W block][A block]; step j adds to set j % SETS
  constexpr int SETS = S::kSets;
  v4f acc[SETS][NW][MW];
#pragma unroll
  for (int t = 0; t < SETS; ++t)
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int r = 0; r < MW; ++r) acc[t][n][r] = v4f{0.f, 0.f, 0.f, 0.f};
  const uint32_t kh = wv & 1, half = wv >> 1;
  const uint32_t mb0 = kSplitM ? half * MW : 0, nb0 = kSplitN ? half * NW : 0;

  auto compute = [&](uint32_t stage, uint32_t j, auto FF, auto SET) __attribute__((always_inline)) {
    if (kOnePair && half) return;
    auto& sums = acc[decltype(SET)::value];
    const uint8_t* sa = smem + stage * S::kStage + (mb0 * 16 + lr) * SB;
    const uint8_t* sw = smem + stage * S::kStage + (TM + nb0 * 16 + lr) * SB;
    if constexpr (!kFp8) {
      const uint32_t at = ((4 * wv + lg) ^ lr) << 4;
      v4i wf[NW];
#pragma unroll
      for (int n = 0; n < NW; ++n) wf[n] = *reinterpret_cast<const v4i*>(sw + n * 4096 + at);
#pragma unroll
      for (int r = 0; r < MW; ++r) {
        const v4i af = *reinterpret_cast<const v4i*>(sa + r * 4096 + at);
#pragma unroll
        for (int n = 0; n < NW; ++n)
          sums[n][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wf[n]),
                                                              __builtin_bit_cast(v8bf, af), sums[n][r], 0, 0, 0);
      }
    } else {
      const uint32_t at0 = ((8 * kh + lg) ^ lr) << 4, at1 = ((8 * kh + 4 + lg) ^ lr) << 4;
      auto frag = [&](const uint8_t* s) __attribute__((always_inline)) -> v8i {
        const v4i x = *reinterpret_cast<const v4i*>(s + at0), y = *reinterpret_cast<const v4i*>(s + at1);
        return v8i{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
      };
      const uint32_t kb = 2 * j + kh;
      const uint32_t ws = pw[kb];
      v8i wf[NW];
#pragma unroll
      for (int n = 0; n < NW; ++n) wf[n] = frag(sw + n * 4096);
#pragma unroll
      for (int r = 0; r < MW; ++r) {
        const v8i af = frag(sa + r * 4096);
        const uint32_t as = pa[(mb0 * 16 + r * 16 + lr) * KB + kb];
#pragma unroll
        for (int n = 0; n < NW; ++n) {
          const v4f sum = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[n], af, sums[n][r], 0, 0, 0, (int)ws, 0,
                                                                           (int)as);
          sums[n][r] = decltype(FF)::value ? without_ff_block(ws, as, sums[n][r], sum) : sum;
        }
      }
    }
  };

  // ---- the K loop: ST stages.  A loading wave waits for its part of step
  // j's stage, meets the others at the barrier and sends for step j + ST - 1
  // (the last ST - 1 steps send for nothing and wait for less each); a
  // multiplying wave waits for its own LDS reads (the stage it has read may be
  // refilled once all are past the barrier), meets it and multiplies step j.
  const uint32_t lead = min((uint32_t)(ST - 1), steps);
  auto tail_wait = [&](int left) __attribute__((always_inline)) {
    // `left` further steps are in flight
#define PIH_TILE_WAIT(L) \
  case L:                \
    if constexpr ((L) < ST - 1) __builtin_amdgcn_s_waitcnt(vmcnt_at_most((L) * NL)); \
    break;
    switch (left) {
      PIH_TILE_WAIT(0) PIH_TILE_WAIT(1) PIH_TILE_WAIT(2) PIH_TILE_WAIT(3)
      PIH_TILE_WAIT(4) PIH_TILE_WAIT(5) PIH_TILE_WAIT(6)
    }
#undef PIH_TILE_WAIT
  };
  auto load_loop = [&](auto NT) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if ((uint32_t)s < lead) issue(s, s, NT);
    if constexpr (kFp8) {
      // the scale panels are older loads than the stages'
      if (lead == ST - 1) __builtin_amdgcn_s_waitcnt(vmcnt_at_most((ST - 1) * NL));
      else __builtin_amdgcn_s_waitcnt(vmcnt_at_most(0));
      __builtin_amdgcn_s_barrier();
    }
    uint32_t j = 0, ist = ST - 1;
    for (; j + (ST - 1) < steps; ++j) {
      __builtin_amdgcn_s_waitcnt(vmcnt_at_most((ST - 2) * NL));
      __builtin_amdgcn_s_barrier();
      issue(ist, j + (ST - 1), NT);
      ist = ist + 1 == ST ? 0 : ist + 1;
    }
#pragma unroll
    for (int left = ST - 2; left >= 0; --left) {
      if (j + left >= steps) continue;  // fewer steps than stages
      tail_wait(left);
      __builtin_amdgcn_s_barrier();
      ++j;
    }
  };
  auto multiply_loop = [&](auto FF) __attribute__((always_inline)) {
    uint32_t cst = 0;
    auto step = [&](uint32_t j, auto SET) __attribute__((always_inline)) {
      __builtin_amdgcn_s_waitcnt(kLdsRead);
      __builtin_amdgcn_s_barrier();
      compute(cst, j, FF, SET);
      cst = cst + 1 == ST ? 0 : cst + 1;
    };
    uint32_t j = 0;
    for (; j + SETS <= steps; j += SETS) {
      step(j, std::integral_constant<int, 0>{});
      if constexpr (SETS > 1) step(j + 1, std::integral_constant<int, 1>{});
      if constexpr (SETS > 2) {
        step(j + 2, std::integral_constant<int, 2>{});
        step(j + 3, std::integral_constant<int, 3>{});
      }
    }
    if constexpr (SETS > 1)
      if (j < steps) step(j, std::integral_constant<int, 0>{});
    if constexpr (SETS > 2) {
      if (j + 1 < steps) step(j + 1, std::integral_constant<int, 1>{});
      if (j + 2 < steps) step(j + 2, std::integral_constant<int, 2>{});
    }
    // the sets, pairwise
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int r = 0; r < MW; ++r) {
        if constexpr (SETS == 4) acc[0][n][r] = (acc[0][n][r] + acc[1][n][r]) + (acc[2][n][r] + acc[3][n][r]);
        else if constexpr (SETS == 2) acc[0][n][r] += acc[1][n][r];
      }
  };
  if (loader) {
    // one M tile reads each weight byte once: non-temporal, so that the A
    // rows every tile reads again stay in L2
    if (p.m_tiles == 1) load_loop(std::true_type{});
    else load_loop(std::false_type{});
  } else {
    bool ff = false;
    if constexpr (kFp8) {
      // a 0xFF scale anywhere in the panels; every wave looks through all of
      // them, which needs no exchange
      __builtin_amdgcn_s_barrier();
      uint32_t hit = 0;
      for (uint32_t i = lane; i < TM * KB / 16; i += 64) {
        const v4u v = reinterpret_cast<const v4u*>(pa)[i];
        hit |= ff_bytes(v.x) | ff_bytes(v.y) | ff_bytes(v.z) | ff_bytes(v.w);
      }
      if (lane < KB / 4) hit |= ff_bytes(reinterpret_cast<const uint32_t*>(pw)[lane]);
      ff = __builtin_amdgcn_ballot_w64(hit != 0) != 0;
      if (ff) bad |= kErrScale;
    }
    if (kFp8 && ff) multiply_loop(std::true_type{});
    else multiply_loop(std::false_type{});
  }

  // ---- the waves' sums, then whole rows.  Under the code check an element
  // that came out non-finite is only marked (bit row TN + column of a map
  // where the scale panels were), and the eight waves then share them out.
  const bool look = kFp8 && p.check_codes;
  uint32_t* const map = reinterpret_cast<uint32_t*>(smem + S::kRing);  // [0]: any
  constexpr uint32_t kMapWords = TM * TN / 32;
  static_assert(!kFp8 || (kMapWords + 1) * 4 <= S::kPanel, "the map fits the panels");
  __syncthreads();
  if (look)
    for (uint32_t i = tid; i <= kMapWords; i += kThreads) map[i] = 0;
  const uint32_t part = kFp8 ? kh : wv;
#pragma unroll
  for (int n = 0; n < NW && !loader && !(kOnePair && half); ++n)
#pragma unroll
    for (int r = 0; r < MW; ++r)
      *reinterpret_cast<v4f*>(smem + (part * MB * NB + (mb0 + r) * NB + nb0 + n) * kSumBlock + lg * kSumGroup + lr * 16) =
          acc[0][n][r];
  __syncthreads();
  constexpr uint32_t QR = TN / 4;  // 4-column groups per row
  // columns 4 cq .. + 3 of a row, summed over the waves
  auto sum4 = [&](uint32_t row, uint32_t cq) __attribute__((always_inline)) -> v4f {
    const uint8_t* s = smem + ((row >> 4) * NB + (cq >> 2)) * kSumBlock + (cq & 3) * kSumGroup + (row & 15) * 16;
    v4f v = *reinterpret_cast<const v4f*>(s);
#pragma unroll
    for (int q = 1; q < S::kParts; ++q) v += *reinterpret_cast<const v4f*>(s + q * MB * NB * kSumBlock);
    return v;
  };
  auto pick4 = [](v4f v, uint32_t i) __attribute__((always_inline)) -> float {
    return i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3];
  };
#pragma unroll 1
  for (uint32_t it = tid; it < TM * QR; it += kThreads) {
    const uint32_t row = it / QR, cq = it % QR;
    if (row0 + row >= p.m) continue;
    const v4f v = sum4(row, cq);
    if (finite4(v)) {
      store4(p, row0 + row, prob, col0 + cq * 4, v);
    } else {
#pragma unroll 1
      for (uint32_t i = 0; i < 4; ++i) {
        const float e = pick4(v, i);
        if (look && !__builtin_isfinite(e)) {
          const uint32_t at = row * TN + cq * 4 + i;
          atomicOr(&map[1 + at / 32], 1u << (at & 31));
          map[0] = 1;
        } else {
          store_looked_at(p, row0 + row, prob, col0 + cq * 4 + i, e, bad);
        }
      }
    }
  }
  if (look) {
    __syncthreads();
    if (map[0]) {
#pragma unroll 1
      for (uint32_t base = 0; base < kMapWords; base += 64) {
        // every eighth column of a row, the next one in the next row: an A
        // row's elements and a W row's are spread over the waves alike
        const uint32_t first = (base + lane) * 32 / TN, even = 0x01010101u << ((wave + first) & 7),
                       odd = 0x01010101u << ((wave + first + 1) & 7);
        const uint32_t share = TN >= 32 ? even : (even & 0xffffu) | (odd & 0xffff0000u);
        uint32_t mine = base + lane < kMapWords ? map[1 + base + lane] & share : 0u;
        uint64_t left;
        while ((left = __builtin_amdgcn_ballot_w64(mine != 0)) != 0) {
          const uint32_t l = (uint32_t)__builtin_ctzll(left);
          const uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)mine, l);
          const uint32_t at = (base + l) * 32 + (uint32_t)__builtin_ctz(word), row = at / TN, col = at % TN;
          if (lane == l) mine &= mine - 1;
          store_nonfinite(p, row0 + row, prob, col0 + col, pick4(sum4(row, col / 4), col & 3), 0, bad);
        }
      }
    }
  }
  if (bad) raise(p, bad);
}

// ------------------------------------------------ several tiles per CU
// The same operands and loading waves, for shapes of more tiles than CUs: a
// block per CU walks its tiles, and the four multiplying waves take a quarter
// of the tile each (2 x 2), so that nothing has to be summed across them: a
// wave stores its results from its registers and goes on, while the loading
// waves are already kStages - 1 steps into the next tile.  One barrier per K
// step for all waves, none per tile.
template <int OP, int MB, int NB, int SBW>
struct GridShape {
  static constexpr uint32_t TM = 16 * MB, TN = 16 * NB, kStage = (TM + TN) * SBW;
  static constexpr uint32_t kPanelOne = OP == kTileFp8 ? 256 + TM * kMaxKb : 0;  // two of them
  static constexpr uint32_t kLds = 160 * 1024 - 512;
  static constexpr int kLoads = (MB + NB) * (int)SBW / 256;
  static constexpr uint32_t kOut = 4 * 16 * kOutPitch;  // a 16-row x 128-byte piece of output per wave
  static constexpr int kFit = (int)((kLds - 2 * kPanelOne - kOut) / kStage);
  static constexpr int kStages = std::min(std::min(kFit, 8), 63 / kLoads + 1);
  // fragments read ahead of their MFMAs; an e4m3 fragment is 8 registers, and
  // three of them ahead spilled (128 x 128 tiles: 23.3 -> 25.5 us at M 2048,
  // 4096 -> 2048; bf16 256 x 128: 60.6 -> 57.2 us at 4096 -> 4096 with three)
  static constexpr int kAhead = OP == kTileBf16 ? 3 : 1;
  // accumulator sets (see TileShape): the two 32-k slices of a bf16 step each
  // have one where registers hold them; 12 and 16 row blocks (96 and 128
  // accumulator registers a set) have one chain, the rounding of an unsplit
  // sum on the 128 x 256 tiles
  static constexpr int kSets = OP == kTileBf16 && MB == 8 ? 2 : 1;
};

template <int OP, int MB, int NB, int SBW>
__global__ __launch_bounds__(kThreads, 1) void tile_grid_kernel(TileParams p) {
  using S = GridShape<OP, MB, NB, SBW>;
  constexpr uint32_t TM = S::TM, TN = S::TN;
  constexpr int ST = S::kStages, NL = S::kLoads;
  static_assert(ST >= 2 && MB % 2 == 0 && NB == 8 && ((MB + NB) * SBW) % 256 == 0, "shape");
  constexpr bool kFp8 = OP == kTileFp8;
  constexpr int MW = MB / 2, NW = NB / 2;
  constexpr int RPI = 1024 / SBW, IPB = 16 / RPI;  // rows per DMA instruction, instructions per 16 rows (all waves)
  __shared__ __align__(16) uint8_t smem[ST * S::kStage + 2 * S::kPanelOne + S::kOut];
  const uint32_t tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3;
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t RB = p.row_bytes, steps = RB / SBW, KB = RB / 128;
  const uint32_t total = p.m_tiles * p.n_tiles * p.problems, per = (total + 7) / 8;
  const uint32_t xcd = blockIdx.x & 7, jstep = gridDim.x >> 3;
  const uint32_t t_end = min((xcd + 1) * per, total);
  const uint32_t t_first = xcd * per + (blockIdx.x >> 3);
  if (t_first >= t_end) return;
  const uint32_t tiles = (t_end - t_first + jstep - 1) / jstep;
  auto tile_at = [&](uint32_t i, uint32_t& row0, uint32_t& col0, uint32_t& prob) __attribute__((always_inline)) {
    const uint32_t t = t_first + i * jstep, mt = t % p.m_tiles, rest = t / p.m_tiles;
    row0 = mt * TM;
    col0 = (rest % p.n_tiles) * TN;
    prob = rest / p.n_tiles;
  };

  if (wave >= 4) {
    // ---- loading waves.  Instruction q of wave w moves rows
    // RPI (4 q + w) + (l / (64 / RPI)) of the A rows followed by the W rows.
    constexpr uint32_t LPR = 64 / RPI;
    const uint32_t lrow = lane / LPR, lchunk = lane % LPR;
    uint32_t off[NL];
    const uint8_t* w_base = nullptr;
    uint32_t li = 0, lj = 0, ist = 0;  // next load: tile, step, stage
    static_assert((MB * IPB) % 4 == 0 && (NB * IPB) % 4 == 0, "every wave the same loads");
    constexpr int NLA = MB * IPB / 4;
    auto issue_next = [&]() __attribute__((always_inline)) {
      if (lj == 0) {
        uint32_t row0, col0, prob;
        tile_at(li, row0, col0, prob);
        w_base = p.w + ((uint64_t)prob * p.n + col0) * RB;
        auto a_row = [&](uint32_t r) -> uint64_t {
          return (uint64_t)min(row0 + r, p.m - 1) * p.a_row_stride + (uint64_t)prob * p.a_prob_row;
        };
#pragma unroll
        for (int q = 0; q < NL; ++q) {
          const uint32_t r = RPI * (4 * (q < NLA ? q : q - NLA) + wv) + lrow;
          const uint32_t c = SBW == 256 ? lchunk ^ (r & 15) : lchunk ^ ((r >> 1) & 7);
          off[q] = (q < NLA ? (uint32_t)(a_row(r) * RB) : r * RB) + (c << 4);
        }
        if constexpr (kFp8) {
          const uint32_t q4 = KB / 4, pan = lds0 + ST * S::kStage + (li & 1) * S::kPanelOne;
          if (wv == 0) {
            const uint8_t* src = p.w_scale + ((uint64_t)prob * (p.n / 128) + col0 / 128) * KB;
            dma4v(src + 4 * min(lane, q4 - 1), pan);
          }
          for (uint32_t b = wv * 64; b < TM * q4; b += 256) {
            const uint32_t i = min(b + lane, TM * q4 - 1);
            dma4v(p.a_scale + a_row(i / q4) * KB + 4 * (i % q4), pan + 256 + 4 * b);
          }
        }
      }
      const uint32_t lds = lds0 + ist * S::kStage + wv * 1024;
      const uint8_t* ab = uniform_ptr(p.a + (uint64_t)lj * SBW);
      const uint8_t* wb = uniform_ptr(w_base + (uint64_t)lj * SBW);
#pragma unroll
      for (int q = 0; q < NL; ++q) dma16(q < NLA ? ab : wb, off[q], lds + q * 4096);
      ist = ist + 1 == ST ? 0 : ist + 1;
      if (++lj == steps) {
        lj = 0;
        ++li;
      }
    };
    const uint32_t all = tiles * steps;
#pragma unroll 1
    for (uint32_t s = 0; s < min((uint32_t)(ST - 1), all); ++s) issue_next();
    uint32_t g = 0;
    for (; g + (ST - 1) < all; ++g) {
      __builtin_amdgcn_s_waitcnt(vmcnt_at_most((ST - 2) * NL));
      __builtin_amdgcn_s_barrier();
      issue_next();
    }
#pragma unroll
    for (int left = ST - 2; left >= 0; --left) {
      if (g + left >= all) continue;
      switch (left) {
#define PIH_TILE_WAIT(L) \
  case L:                \
    if constexpr ((L) < ST - 1) __builtin_amdgcn_s_waitcnt(vmcnt_at_most((L) * NL)); \
    break;
        PIH_TILE_WAIT(0) PIH_TILE_WAIT(1) PIH_TILE_WAIT(2) PIH_TILE_WAIT(3)
        PIH_TILE_WAIT(4) PIH_TILE_WAIT(5) PIH_TILE_WAIT(6)
#undef PIH_TILE_WAIT
      }
      __builtin_amdgcn_s_barrier();
      ++g;
    }
    __builtin_amdgcn_s_barrier();  // the multiplying waves' look past the last step
    return;
  }

  // ---- multiplying waves.  A step is GS groups of one A fragment times the
  // wave's NW W fragments of its K slice (32 bf16 or 128 e4m3 values); A
  // fragments are read kAhead groups ahead and W fragments a slice ahead, over
  // the step's end: the barrier that opens step j + 1 stands kAhead groups
  // before the end of step j, when every fragment of step j is in registers.
  const uint32_t wm = wv >> 1, wn = wv & 1;
  uint32_t bad = 0, cst = 0;
  constexpr int QS = kFp8 ? SBW / 128 : SBW / 64, GS = QS * MW;
  constexpr int D = S::kAhead, AR = D + 1;
  static_assert(D <= MW && GS % AR == 0, "fragment ring");
  using Frag = std::conditional_t<kFp8, v8i, v4i>;
  Frag af[AR], wf[2][NW];
  uint32_t as[AR], ws[2];
  const uint32_t a_lane = (wm * MW * 16 + lr) * SBW, w_lane = (TM + wn * NW * 16 + lr) * SBW;
  auto frag = [&](const uint8_t* s, int q) __attribute__((always_inline)) -> Frag {
    auto at = [&](uint32_t c) -> uint32_t { return (SBW == 256 ? c ^ lr : c ^ (lr >> 1)) << 4; };
    if constexpr (kFp8) {
      const v4i x = *reinterpret_cast<const v4i*>(s + at(8 * q + lg)), y = *reinterpret_cast<const v4i*>(s + at(8 * q + 4 + lg));
      return v8i{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    } else {
      return *reinterpret_cast<const v4i*>(s + at(4 * q + lg));
    }
  };
  auto read_a = [&](uint32_t stage, uint32_t j, const uint8_t* pan, int g, int slot) __attribute__((always_inline)) {
    const int r = g % MW, q = g / MW;
    af[slot] = frag(smem + stage * S::kStage + a_lane + r * 16 * SBW, q);
    if constexpr (kFp8) as[slot] = pan[256 + ((wm * MW + r) * 16 + lr) * KB + j * QS + q];
  };
  auto read_w = [&](uint32_t stage, uint32_t j, const uint8_t* pan, int q, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NW; ++n) wf[buf][n] = frag(smem + stage * S::kStage + w_lane + n * 16 * SBW, q);
    if constexpr (kFp8) ws[buf] = pan[j * QS + q];
  };
  const uint8_t* const panels = smem + ST * S::kStage;
  __builtin_amdgcn_s_barrier();
  read_w(0, 0, panels, 0, 0);
#pragma unroll
  for (int g = 0; g < D; ++g) read_a(0, 0, panels, g, g);
  for (uint32_t i = 0; i < tiles; ++i) {
    uint32_t row0, col0, prob;
    tile_at(i, row0, col0, prob);
    v4f sums[S::kSets][NW][MW];
#pragma unroll
    for (int t = 0; t < S::kSets; ++t)
#pragma unroll
      for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int r = 0; r < MW; ++r) sums[t][n][r] = v4f{0.f, 0.f, 0.f, 0.f};
    auto& acc = sums[0];
    const uint8_t* const pan = panels + (i & 1) * S::kPanelOne;
    // step j, whose first slice's W fragments are in wf[P]
    auto step = [&](uint32_t j, auto PAR, auto FF) __attribute__((always_inline)) {
      constexpr int P = decltype(PAR)::value;
      const uint32_t nst = cst + 1 == ST ? 0 : cst + 1;
      const bool wrap = j + 1 == steps;
      const uint32_t nj = wrap ? 0 : j + 1;
      const uint8_t* const npan = wrap ? panels + ((i + 1) & 1) * S::kPanelOne : pan;
#pragma unroll
      for (int g = 0; g < GS; ++g) {
        const int r = g % MW, q = g / MW, wb = (P + q) & 1;
        if (g != GS - D) {
          if (g < GS - D) read_a(cst, j, pan, g + D, (g + D) % AR);
          else read_a(nst, nj, npan, g + D - GS, (g + D) % AR);
          if (q + 1 < QS && r == MW - D) read_w(cst, j, pan, q + 1, wb ^ 1);
        }
        const Frag a = af[g % AR];
        const uint32_t sa = as[g % AR], sw = ws[wb];
#pragma unroll
        for (int n = 0; n < NW; ++n) {
          if constexpr (kFp8) {
            const v4f sum = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[wb][n], a, acc[n][r], 0, 0, 0, (int)sw,
                                                                             0, (int)sa);
            acc[n][r] = decltype(FF)::value ? without_ff_block(sw, sa, acc[n][r], sum) : sum;
          } else {
            sums[q % S::kSets][n][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(v8bf, wf[wb][n]), __builtin_bit_cast(v8bf, a), sums[q % S::kSets][n][r], 0, 0, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (g == GS - D) {
          __builtin_amdgcn_s_waitcnt(kLdsRead);
          __builtin_amdgcn_s_barrier();
          read_w(nst, nj, npan, 0, (P + QS) & 1);
          read_a(nst, nj, npan, 0, (g + D) % AR);
        }
      }
      cst = nst;
    };
    bool ff = false;
    if constexpr (kFp8) {
      uint32_t hit = 0;
      for (uint32_t e = lane; e < TM * KB / 16; e += 64) {
        const v4u v = reinterpret_cast<const v4u*>(pan + 256)[e];
        hit |= ff_bytes(v.x) | ff_bytes(v.y) | ff_bytes(v.z) | ff_bytes(v.w);
      }
      if (lane < KB / 4) hit |= ff_bytes(reinterpret_cast<const uint32_t*>(pan)[lane]);
      ff = __builtin_amdgcn_ballot_w64(hit != 0) != 0;
      if (ff) bad |= kErrScale;
    }
    auto run = [&](auto FF) __attribute__((always_inline)) {
      // one slice a step: two steps a trip, so that the W buffers are constant
#pragma unroll 1
      for (uint32_t j = 0; j < steps; j += QS % 2 ? 2 : 1) {
        step(j, std::integral_constant<int, 0>{}, FF);
        if constexpr (QS % 2) step(j + 1, std::integral_constant<int, 1>{}, FF);
      }
    };
    if (kFp8 && ff) run(std::true_type{});
    else run(std::false_type{});
    if constexpr (S::kSets == 2) {
#pragma unroll
      for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int r = 0; r < MW; ++r) acc[n][r] += sums[1][n][r];
    }
    const uint32_t orow = row0 + wm * MW * 16 + lr, ocol = col0 + wn * NW * 16 + 4 * lg;
    bool nonfin = false;
#pragma unroll
    for (int r = 0; r < MW; ++r)
#pragma unroll
      for (int n = 0; n < NW; ++n) nonfin |= orow + r * 16 < p.m && !finite4(acc[n][r]);
    if (!__builtin_amdgcn_ballot_w64(nonfin)) {
      // 16 rows x 128 bytes at a time through the wave's own LDS, so that
      // every store instruction writes whole 128-byte lines (8 rows)
      uint8_t* const st = smem + ST * S::kStage + 2 * S::kPanelOne + wv * (16 * kOutPitch);
      uint8_t* const put = st + lr * kOutPitch;
      const uint8_t* const get = st + (lane >> 3) * kOutPitch + (lane & 7) * 16;
      const uint32_t OSZ = p.out_f32 ? 4 : 2;
      const uint32_t grow = row0 + wm * MW * 16 + (lane >> 3);
      uint8_t* const gout = static_cast<uint8_t*>(p.out) +
                            ((uint64_t)grow * p.out_row_stride + (uint64_t)prob * p.out_prob_col + col0 + wn * NW * 16) * OSZ +
                            (lane & 7) * 16;
      const uint64_t pitch = p.out_row_stride * OSZ;
      auto flush = [&](int r, uint32_t at) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (grow + r * 16 + h * 8 < p.m)
            *reinterpret_cast<v4i*>(gout + (r * 16 + h * 8) * pitch + at) =
                *reinterpret_cast<const v4i*>(get + h * 8 * kOutPitch);
      };
#pragma unroll
      for (int r = 0; r < MW; ++r) {
        if (p.out_f32) {
#pragma unroll
          for (int n = 0; n < NW; ++n) {
            *reinterpret_cast<v4f*>(put + (n & 1) * 64 + lg * 16) = acc[n][r];
            if (n & 1) flush(r, (n >> 1) * 128);
          }
        } else {
#pragma unroll
          for (int n = 0; n < NW; ++n)
            *reinterpret_cast<uint2*>(put + n * 32 + lg * 8) =
                uint2{f32x2_to_bf16x2(acc[n][r][0], acc[n][r][1]), f32x2_to_bf16x2(acc[n][r][2], acc[n][r][3])};
          flush(r, 0);
        }
      }
    } else {
      // rare: one 16-column block at a time, its values picked by selects
#pragma unroll 1
      for (int b = 0; b < MW * NW * 4; ++b) {
        float v = 0.0f;
#pragma unroll
        for (int r = 0; r < MW; ++r)
#pragma unroll
          for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) v = b == (r * NW + n) * 4 + e ? acc[n][r][e] : v;
        const uint32_t row = orow + b / (4 * NW) * 16, col = ocol + b / 4 % NW * 16 + (b & 3);
        const bool in = row < p.m, look = kFp8 && p.check_codes && in && !__builtin_isfinite(v);
        if (in && !look) store_looked_at(p, row, prob, col, v, bad);
        if constexpr (kFp8) {
          // the wave takes its lanes' elements one after the other
          uint64_t left = __builtin_amdgcn_ballot_w64(look);
          while (left) {
            const uint32_t l = (uint32_t)__builtin_ctzll(left);
            left &= left - 1;
            store_nonfinite(p, (uint32_t)__builtin_amdgcn_readlane((int)row, l), prob,
                            (uint32_t)__builtin_amdgcn_readlane((int)col, l), v, l, bad);
          }
        }
      }
    }
  }
  if (bad) raise(p, bad);
}

template <int OP, int MB, int NB>
void launch_tile(TileParams p, hipStream_t s) {
  p.m_tiles = (p.m + 16 * MB - 1) / (16 * MB);
  p.n_tiles = p.n / (16 * NB);
  const uint32_t grid = (p.m_tiles * p.n_tiles * p.problems + 7) / 8 * 8;
  hipLaunchKernelGGL((tile_gemm_kernel<OP, MB, NB>), dim3(grid), dim3(kThreads), 0, s, p);
}

template <int OP, int MB, int NB, int SBW>
void launch_grid(TileParams p, uint32_t cus, hipStream_t s) {
  p.m_tiles = (p.m + 16 * MB - 1) / (16 * MB);
  p.n_tiles = p.n / (16 * NB);
  const uint32_t grid = std::min((p.m_tiles * p.n_tiles * p.problems + 7) / 8 * 8, cus / 8 * 8);
  hipLaunchKernelGGL((tile_grid_kernel<OP, MB, NB, SBW>), dim3(grid), dim3(kThreads), 0, s, p);
}

template <int OP, int MB>
void launch_nb(int nb, const TileParams& p, hipStream_t s) {
  switch (nb) {
    case 1: launch_tile<OP, MB, 1>(p, s); break;
    case 2: launch_tile<OP, MB, 2>(p, s); break;
    case 3:
      if constexpr (OP == kTileBf16) launch_tile<OP, MB, 3>(p, s);
      break;
    case 4: launch_tile<OP, MB, 4>(p, s); break;
    case 8:
      if constexpr (MB <= 4) launch_tile<OP, MB, 8>(p, s);
      break;
  }
}

template <int OP>
void launch_pick(const TilePick& t, const TileParams& p, hipStream_t s) {
  if (t.grid) {
    if (t.mb == 8) launch_grid<OP, 8, 8, kGridStep>(p, kCus, s);
    else if (t.mb == 12) launch_grid<OP, 12, 8, kGridStep>(p, kCus, s);
    else if constexpr (OP == kTileBf16) launch_grid<OP, 16, 8, kGridStep>(p, kCus, s);
    return;
  }
  switch (t.mb) {
    case 1: launch_nb<OP, 1>(t.nb, p, s); break;
    case 2: launch_nb<OP, 2>(t.nb, p, s); break;
    case 3: launch_nb<OP, 3>(t.nb, p, s); break;
    case 4: launch_nb<OP, 4>(t.nb, p, s); break;
    case 5: launch_nb<OP, 5>(t.nb, p, s); break;
    case 6: launch_nb<OP, 6>(t.nb, p, s); break;
    case 8: launch_nb<OP, 8>(t.nb, p, s); break;
  }
}

}  // namespace

bool TileGemmTakes(const TileGemmArgs& a) {
  const uint64_t rb = a.bf16 ? 2ull * a.k : a.k, osz = a.out_kind == kOutF32 ? 4 : 2;
  if (a.m == 0 || a.n == 0 || a.k == 0 || a.problems == 0 || rb % SB || a.n % (a.bf16 ? 16 : 128)) return false;
  if (a.out_kind != kOutBf16 && a.out_kind != kOutF32) return false;
  const uint64_t rows = (uint64_t)(a.m - 1) * a.a_row_stride + (uint64_t)(a.problems - 1) * a.a_prob_row + 1;
  const uint64_t stride = a.out_row_stride ? a.out_row_stride : a.n;
  // 32-bit byte offsets into A and within a W tile, 16-byte loads and stores
  if (rows > a.a_rows_total || rows * rb > 0xffffffffull || 128ull * rb > 0xffffffffull) return false;
  if ((uint64_t)a.n * a.problems / 16 * ((a.m + 15) / 16) > 0x3fffffffull) return false;
  if ((reinterpret_cast<uintptr_t>(a.a) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.out)) % 16 ||
      stride * osz % 16 || (uint64_t)a.out_prob_col * osz % 16)
    return false;
  if (a.bf16) return true;
  return a.k % 512 == 0 && a.k / 128 <= kMaxKb &&
         (reinterpret_cast<uintptr_t>(a.a_scale) | reinterpret_cast<uintptr_t>(a.w_scale)) % 4 == 0;
}

St LaunchTileGemm(const TileGemmArgs& a, const TilePick& t) {
  if (!a.a || !a.w || !a.out || !a.stream || (!a.bf16 && (!a.a_scale || !a.w_scale || !a.error_flag)))
    return Invalid("tile_gemm_null_argument");
  if (!TileGemmTakes(a)) return Invalid("tile_gemm_shape_invalid");
  TileParams p{};
  p.a = static_cast<const uint8_t*>(a.a);
  p.w = static_cast<const uint8_t*>(a.w);
  p.a_scale = a.a_scale;
  p.w_scale = a.w_scale;
  p.out = a.out;
  p.err = a.error_flag;
  p.m = a.m;
  p.n = a.n;
  p.row_bytes = a.bf16 ? 2 * a.k : a.k;
  p.problems = a.problems;
  p.a_row_stride = a.a_row_stride;
  p.a_prob_row = a.a_prob_row;
  p.out_row_stride = a.out_row_stride ? a.out_row_stride : a.n;
  p.out_prob_col = a.out_prob_col;
  p.out_f32 = a.out_kind == kOutF32;
  p.write_nonfinite = a.write_nonfinite;
  p.check_codes = a.check_codes;
  if (a.error_flag) {
    p.err_code = a.err_code_bit;
    p.err_scale = a.err_scale_bit;
    p.err_nonfinite = a.err_nonfinite_bit;
  }
  St s = RequireCleanLastError();
  if (!s.ok()) return s;
  if (a.bf16) launch_pick<kTileBf16>(t, p, a.stream);
  else launch_pick<kTileFp8>(t, p, a.stream);
  return AfterLaunch("tile_gemm_launch_failed");
}

}  // namespace pih_amd
