// W4A16 for decode batches on gfx950: y [m, n] = x [m, k] . W [n, k]^T with INT4
// weights (symmetric or asymmetric, a scale per 128 k), up to 8 problems of
// one m and k in a launch, tiles chosen per launch as in gemm_tile.hip.
//
// What bounds it: at m 16 a block's x rows are 4x the bytes of its 16 weight
// rows, so the weight-streaming blocks of gemv.hip spent their loads on x,
// and each of their waves loaded, unpacked and multiplied in turn.  Here four
// waves load (LDS DMA) and four unpack and multiply, and a block takes 16 NB
// weight rows against its x rows, with NB such that the tiles make about one
// round on the CUs.
//
// A K step is 512 values: 1024 bytes of an x row (one DMA instruction; 16-byte
// chunk c of row r in slot c ^ (r & 15) of its 256-byte quarter) and 256 bytes
// of a weight row (4 rows an instruction, slot c ^ (r & 15)).  Wave w of the
// multiplying four takes the step's 128-value group w: nibbles become bf16
// (128 + u) by two masks and four v_perm a word, x takes the same k order in
// registers, four MFMAs give sum x (128 + u), one more chain against ones
// gives sum x, and the group's scale and zero point are applied in fp32:
// acc += s (pq - (128 + z) sum x), the arithmetic of gemv_mid_kernel.  The
// scales and zero points of the tile's rows come into LDS once, ahead of the
// first step.  The waves' sums meet in LDS in wave order.
//
// Error codes as in gemv.hip: 12 reserved nibble (symmetric), 13 scale not
// finite and positive, 14 non-finite output, the first one stored.
#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"

namespace pih_amd {
namespace {

constexpr uint32_t kThreads = 512, kMaxGroup = 8;
constexpr uint32_t kMaxGroups = 96;  // K / 128 the panels hold
constexpr uint32_t kReservedNibble = 12, kBadScale = 13, kNonFinite = 14;

struct W4Problem {
  const uint8_t* x;
  const uint8_t* w;
  const uint8_t* scales;
  const uint8_t* zeros;
  uint16_t* out;
  uint32_t n, tile0;  // first tile of the problem in the launch
};
struct W4Params {
  W4Problem prob[kMaxGroup];
  uint32_t* err;
  uint32_t m, k, count, tiles;
};

// XI x rows a loading wave moves per step: 4 XI rows in all, whole 16-row MFMA
// operands
template <int XI, int NB>
struct W4Shape {
  static constexpr int MB = XI / 4;
  static constexpr uint32_t TM = 16 * MB, TN = 16 * NB, kX = 4 * XI * 1024, kStage = kX + TN * 256;
  static constexpr uint32_t kScales = TN * kMaxGroups * 2, kZeros = TN * ((kMaxGroups + 7) / 8) * 4;
  static constexpr uint32_t kPanel = (kScales + kZeros + 511) / 512 * 512;  // whole DMAs of each
  static constexpr int kLoads = XI + NB;
  static constexpr int kFit = (int)((160 * 1024 - 512 - kPanel) / kStage);
  static constexpr int kStages = std::min(std::min(kFit, 4), 63 / kLoads + 1);  // (8 deep: launches 0.5-0.8 us longer)
  static constexpr uint32_t kSums = 4 * MB * NB * 1024;
  static constexpr uint32_t kRing = kStages * kStage > kSums ? kStages * kStage : kSums;
  static_assert(kRing + kPanel <= 160 * 1024, "LDS");
};

template <bool SYM, int XI, int NB>
__global__ __launch_bounds__(kThreads, 1) void w4a16_tile_kernel(W4Params p) {
  using S = W4Shape<XI, NB>;
  constexpr int MB = S::MB;
  constexpr uint32_t TM = S::TM, TN = S::TN;
  constexpr int ST = S::kStages, NL = S::kLoads;
  static_assert(ST >= 2, "two stages");
  __shared__ __align__(16) uint8_t smem[S::kRing + S::kPanel];
  const uint32_t tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3;
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t t = blockIdx.x;
  uint32_t pi = 0;
#pragma unroll
  for (uint32_t i = 1; i < kMaxGroup; ++i)
    if (i < p.count && t >= p.prob[i].tile0) pi = i;
  W4Problem q = p.prob[0];
#pragma unroll
  for (uint32_t i = 1; i < kMaxGroup; ++i)
    if (pi == i) q = p.prob[i];
  const uint32_t n0 = (t - q.tile0) * TN, K = p.k, G = K / 128, ZW = (G + 7) / 8, steps = K / 512;
  const uint8_t* const w_base = q.w + (uint64_t)n0 * (K / 2);
  uint8_t* const panel = smem + S::kRing;
  uint8_t* const zpanel = panel + S::kScales;

  v4f acc[NB][MB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int a = 0; a < MB; ++a) acc[b][a] = v4f{0.f, 0.f, 0.f, 0.f};

  if (wave >= 4) {
    // ---- loading waves: the panels, then the steps (x row r of a step by
    // wave r & 3; weight rows 4 w + (l >> 4) of each 16-row block)
    auto panel_in = [&](const uint8_t* src, uint32_t dwords, uint32_t at) __attribute__((always_inline)) {
      for (uint32_t b = wv * 64; b < dwords; b += 256) dma4v(src + 4 * min(b + lane, dwords - 1), lds0 + at + 4 * b);
    };
    panel_in(q.scales + (uint64_t)n0 * G * 2, TN * G / 2, S::kRing);
    if constexpr (!SYM) panel_in(q.zeros + (uint64_t)n0 * ZW * 4, TN * ZW, S::kRing + S::kScales);
    uint32_t x_off[XI], w_off[NB];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const uint32_t r = 4 * i + wv;  // rows past m read row m - 1; they are not stored
      x_off[i] = min(r, p.m - 1) * (K * 2) + (((lane & 48u) | ((lane ^ r) & 15u)) << 4);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const uint32_t r = 16 * i + 4 * wv + lg;
      w_off[i] = r * (K / 2) + ((lr ^ (r & 15u)) << 4);
    }
    auto issue = [&](uint32_t stage, uint32_t j) __attribute__((always_inline)) {
      const uint32_t lds = lds0 + stage * S::kStage;
      const uint8_t* xb = uniform_ptr(q.x + (uint64_t)j * 1024);
      const uint8_t* wb = uniform_ptr(w_base + (uint64_t)j * 256);
#pragma unroll
      for (int i = 0; i < NB; ++i) dma16nt(wb, w_off[i], lds + S::kX + i * 4096 + wv * 1024);
#pragma unroll
      for (int i = 0; i < XI; ++i) dma16(xb, x_off[i], lds + (4 * i + wv) * 1024);
    };
    const uint32_t lead = min((uint32_t)(ST - 1), steps);
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if ((uint32_t)s < lead) issue(s, s);
    uint32_t j = 0, ist = ST - 1;
    for (; j + (ST - 1) < steps; ++j) {
      __builtin_amdgcn_s_waitcnt(vmcnt_at_most((ST - 2) * NL));
      __builtin_amdgcn_s_barrier();
      issue(ist, j + (ST - 1));
      ist = ist + 1 == ST ? 0 : ist + 1;
    }
#pragma unroll
    for (int left = ST - 2; left >= 0; --left) {
      if (j + left >= steps) continue;  // fewer steps than stages
#define PIH_W4_WAIT(L) \
  case L:              \
    if constexpr ((L) < ST - 1) __builtin_amdgcn_s_waitcnt(vmcnt_at_most((L) * NL)); \
    break;
      switch (left) {
        PIH_W4_WAIT(0) PIH_W4_WAIT(1) PIH_W4_WAIT(2) PIH_W4_WAIT(3) PIH_W4_WAIT(4) PIH_W4_WAIT(5) PIH_W4_WAIT(6)
      }
#undef PIH_W4_WAIT
      __builtin_amdgcn_s_barrier();
      ++j;
    }
  } else {
    // ---- multiplying waves: group 4 j + w of step j.  (Products in two chains
    // of two MFMAs: a chain waits for its last result each time.)
    uint32_t bad = 0, cst = 0;
    const v8bf ones = __builtin_bit_cast(v8bf, v4i{0x3f803f80, 0x3f803f80, 0x3f803f80, 0x3f803f80});
    const v4f zero4{0.f, 0.f, 0.f, 0.f};
    auto mma = [](v8bf x, v8bf y, v4f c) __attribute__((always_inline)) -> v4f {
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
    };
#pragma unroll 1
    for (uint32_t j = 0; j < steps; ++j) {
      __builtin_amdgcn_s_waitcnt(kLdsRead);
      __builtin_amdgcn_s_barrier();
      const uint8_t* sx = smem + cst * S::kStage + lr * 1024 + wv * 256;
      const uint8_t* sw = smem + cst * S::kStage + S::kX + lr * 256 + (((4 * wv + lg) ^ lr) << 4);
      const uint32_t g = 4 * j + wv;
      v4i wf[NB];
      uint32_t sb[NB], zb[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        wf[b] = *reinterpret_cast<const v4i*>(sw + b * 4096);
        sb[b] = *reinterpret_cast<const uint16_t*>(panel + ((b * 16 + lr) * G + g) * 2);
        if constexpr (!SYM) zb[b] = *reinterpret_cast<const uint32_t*>(zpanel + ((b * 16 + lr) * ZW + g / 8) * 4);
      }
      v8bf xf[MB][4];
      v4f xs[MB];
#pragma unroll
      for (int a = 0; a < MB; ++a) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          xf[a][i] = __builtin_bit_cast(
              v8bf, x_in_nibble_order(*reinterpret_cast<const v4i*>(sx + a * 16384 + (((4 * lg + i) ^ lr) << 4))));
        xs[a] = mma(xf[a][1], ones, mma(xf[a][0], ones, zero4)) + mma(xf[a][3], ones, mma(xf[a][2], ones, zero4));
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float sc;
        int zero;
        if constexpr (SYM) {
          sc = (float)__builtin_bit_cast(_Float16, (uint16_t)sb[b]);
          zero = 8;
        } else {
          sc = bf16_bits_to_f32(sb[b]);
          zero = (int)((zb[b] >> (4 * (g & 7u))) & 0xfu);
        }
        if (!(sc > 0.0f) || !__builtin_isfinite(sc)) bad = bad ? bad : kBadScale;
        v8bf qb[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t wd = (uint32_t)wf[b][i];
          if constexpr (SYM) {
            wd ^= 0x88888888u;  // two's complement nibble -> u = q + 8; reserved 8 -> 0
            if ((wd - 0x11111111u) & ~wd & 0x88888888u) bad = kReservedNibble;
          }
          qb[i] = __builtin_bit_cast(v8bf, nibbles_to_bf16(wd));
        }
        const float zc = 128.0f + (float)zero;
#pragma unroll
        for (int a = 0; a < MB; ++a) {
          const v4f pq = mma(xf[a][1], qb[1], mma(xf[a][0], qb[0], zero4)) + mma(xf[a][3], qb[3], mma(xf[a][2], qb[2], zero4));
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[b][a][i] = __builtin_fmaf(__builtin_fmaf(-zc, xs[a][i], pq[i]), sc, acc[b][a][i]);
        }
      }
      cst = cst + 1 == ST ? 0 : cst + 1;
    }
    if (bad) atomicCAS(p.err, 0u, bad);
  }

  // ---- the waves' sums in wave order; lane (lr, lg) of block (b, a) holds
  // rows 16 a + 4 lg + i of column 16 b + lr
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int a = 0; a < MB; ++a)
        *reinterpret_cast<v4f*>(smem + ((wv * NB + b) * MB + a) * 1024 + lane * 16) = acc[b][a];
  }
  __syncthreads();
  bool nonfinite = false;
#pragma unroll 1
  for (uint32_t it = tid; it < TM * TN / 2; it += kThreads) {
    const uint32_t row = it / (TN / 2), col = it % (TN / 2) * 2;  // two columns
    if (row >= p.m) continue;
    const uint8_t* s = smem + ((col >> 4) * MB + (row >> 4)) * 1024 + (((row & 15) >> 2) * 16 + (col & 15)) * 16 + (row & 3) * 4;
    float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      v0 += *reinterpret_cast<const float*>(s + w * (NB * MB * 1024));
      v1 += *reinterpret_cast<const float*>(s + w * (NB * MB * 1024) + 16);
    }
    nonfinite |= !__builtin_isfinite(v0) || !__builtin_isfinite(v1);
    *reinterpret_cast<uint32_t*>(q.out + (uint64_t)row * q.n + n0 + col) = f32x2_to_bf16x2(v0, v1);
  }
  if (nonfinite) atomicCAS(p.err, 0u, kNonFinite);
}

template <bool SYM, int XI>
void launch_nb(uint32_t nb, const W4Params& p, hipStream_t s) {
  const dim3 grid(p.tiles), block(kThreads);
  switch (nb) {
    case 1: hipLaunchKernelGGL((w4a16_tile_kernel<SYM, XI, 1>), grid, block, 0, s, p); break;
    case 2: hipLaunchKernelGGL((w4a16_tile_kernel<SYM, XI, 2>), grid, block, 0, s, p); break;
    case 3: hipLaunchKernelGGL((w4a16_tile_kernel<SYM, XI, 3>), grid, block, 0, s, p); break;
    case 4: hipLaunchKernelGGL((w4a16_tile_kernel<SYM, XI, 4>), grid, block, 0, s, p); break;
    case 6: hipLaunchKernelGGL((w4a16_tile_kernel<SYM, XI, 6>), grid, block, 0, s, p); break;
  }
}
template <bool SYM>
void launch_tile(uint32_t m, uint32_t nb, const W4Params& p, hipStream_t s) {
  if (m <= 16) launch_nb<SYM, 4>(nb, p, s);
  else launch_nb<SYM, 8>(nb, p, s);
}

}  // namespace

// Takes a launch when it is the faster one (W4a16TileBlocks), else leaves it
// (`taken` false) to the GEMV kernels.
St LaunchW4a16Tile(const W4a16Args* probs, uint32_t count, bool& taken) {
  taken = false;
  const W4a16Args& a0 = probs[0];
  const uint32_t m = a0.m, k = a0.k;
  if (count == 0 || count > kMaxGroup || k % 512 || k / 128 > kMaxGroups || 64ull * k > 0xffffffffull) return Ok();
  uint32_t n[kMaxGroup];
  uint64_t blocks16 = 0;
  uintptr_t at16 = 0, at4 = 0;
  for (uint32_t i = 0; i < count; ++i) {
    n[i] = probs[i].n;
    blocks16 += n[i] / 16;
    at16 |= reinterpret_cast<uintptr_t>(probs[i].x) | reinterpret_cast<uintptr_t>(probs[i].qweight);
    at4 |= reinterpret_cast<uintptr_t>(probs[i].scales) | reinterpret_cast<uintptr_t>(probs[i].out);
    if (!a0.symmetric) at4 |= reinterpret_cast<uintptr_t>(probs[i].zeros);
  }
  if (at16 % 16 || at4 % 4 || blocks16 > 0x7fffffffull) return Ok();
  const uint32_t nb = W4a16TileBlocks(m, k, n, count);
  if (!nb) return Ok();
  W4Params p{};
  for (uint32_t i = 0; i < count; ++i) {
    W4Problem& q = p.prob[i];
    q.x = reinterpret_cast<const uint8_t*>(probs[i].x);
    q.w = static_cast<const uint8_t*>(probs[i].qweight);
    q.scales = reinterpret_cast<const uint8_t*>(probs[i].scales);
    q.zeros = reinterpret_cast<const uint8_t*>(probs[i].zeros);
    q.out = probs[i].out;
    q.n = probs[i].n;
    q.tile0 = p.tiles;
    p.tiles += probs[i].n / (16 * nb);
  }
  p.err = a0.error_flag;
  p.m = m;
  p.k = k;
  p.count = count;
  taken = true;
  if (a0.symmetric) launch_tile<true>(m, nb, p, a0.stream);
  else launch_tile<false>(m, nb, p, a0.stream);
  return AfterLaunch("w4a16_tile_launch_failed");
}

}  // namespace pih_amd
