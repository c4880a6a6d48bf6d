// Prefill (grouped GEMM) path: activation quantisation, the two grouped GEMMs
// with fused epilogues, on CDNA4 matrix cores.
//
// Formats
//   FMT_FP8   W8A8: activations e4m3 with one float32 scale per row per 128 K
//             (s = amax/448, reference per_token_group_quant_fp8,
//             kernel/triton/fp8_block_linear.py:38-82), weights e4m3 with float32
//             128x128 block scales.  One v_mfma_f32_16x16x128_f8f6f4 covers exactly
//             one 128-deep scale block, so each MFMA result is folded into the
//             accumulator with the product of both scales (reference
//             _prefill_fp8_moe_kernel: acc += dot(a, w) * a_s * w_s).
//   FMT_MXFP4 activations e4m3 with a power-of-two scale per row per 128 K (the
//             DSV4 act_quant round trip of routed_experts_fp4_prefill), weights e2m1
//             with e8m0 per 32 K: v_mfma_scale_f32_16x16x128_f8f6f4 applies both
//             scales in hardware and accumulates directly.
//   FMT_BF16  bf16 activations and weights, v_mfma_f32_16x16x32_bf16.
//
// All three run prefill_qgemm_kernel, whose tiling, copies and schedule are
// described at its section below.  bf16 calls with an operand beyond 2 GiB,
// past the 31-bit offsets of that kernel's buffer descriptors, take the
// register-staged prefill_gemm_kernel, which addresses with 64 bits; the rest
// of this header describes it.
//
// Tiling: a workgroup computes a 128 (weight rows) x 128 (routes) tile with 4 waves
// (2 x 2), each 64 x 64 = 4 x 4 MFMA blocks.  Weights are the MFMA A operand, so a
// lane's four accumulators are four consecutive output features of one route and
// stores are 8-byte vectors.  K advances 128 per step; global->LDS copies of the
// next step overlap the MFMAs of the current one (double-buffered LDS).
//
// Gate/up: the weight tile holds gate rows [n0, n0+64) and up rows [I+n0, I+n0+64);
// wave column wn owns gate and up rows n0+32wn..+32, so SwiGLU pairs registers.
//
// Schedule: workgroups are ordered expert-major -- for each expert, each N tile,
// all M blocks of that expert -- so the blocks sharing a weight tile run together
// and read it from HBM about once; the expert's activation rows stay hot in the
// memory-side cache across its N tiles.  Shared-expert blocks come last.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "quant.h"

namespace ftmoe {

constexpr int kPBM = 128;   // routes per tile
constexpr int kPBN = 128;   // weight rows per tile
constexpr int kPThreads = 256;

// ----------------------------------------------------------------------------
// Activation quantisation: one wave per row, 2 values per lane per 128-group
// (group_scale / quant_value of quant.h).
// ----------------------------------------------------------------------------
// Maximum over each 16-lane row of the wave (DPP inside the row), in every lane.
__device__ __forceinline__ float row16_max_f32(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_f32<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_f32<0x141>(v));  // row_half_mirror
  return fmaxf(v, dpp_f32<0x140>(v));  // row_mirror
}

// One wave per row.  Lane l of load i holds 8 values (16 bytes) at
// 8 * (64 i + l): the 16 lanes of a row of the wave cover one 128-value group,
// whose amax is a DPP reduction inside the row.  kAhead loads of the row are
// in flight together; x is read once (nontemporal).
template <int MODE>
__global__ void __launch_bounds__(256) act_quant_kernel(const uint16_t* __restrict__ x, int rows, int K,
                                                        uint8_t* __restrict__ q, void* __restrict__ scales,
                                                        int sstride) {
  const int lane = lane_id();
  const int row = blockIdx.x * 4 + threadIdx.x / kWave;
  if (row >= rows) return;
  const u32x4* xr = reinterpret_cast<const u32x4*>(x + static_cast<size_t>(row) * K);
  uint2* qr = reinterpret_cast<uint2*>(q + static_cast<size_t>(row) * K);
  const int nv = K / 8;                  // 16-byte pieces of the row
  const int nload = (nv + kWave - 1) / kWave;
  constexpr int kAhead = 8;
  for (int i0 = 0; i0 < nload; i0 += kAhead) {
    u32x4 v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int p = (i0 + u) * kWave + lane;
      v[u] = (i0 + u < nload && p < nv) ? __builtin_nontemporal_load(xr + p) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (i0 + u >= nload) break;
      const int p = (i0 + u) * kWave + lane;
      const int gi = p / 16;  // the row's 16 lanes form group gi (uniform inside the row)
      float f[8];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        f[2 * w] = bf16_to_f32(static_cast<uint16_t>(v[u][w] & 0xffffu));
        f[2 * w + 1] = bf16_to_f32(static_cast<uint16_t>(v[u][w] >> 16));
      }
      float m = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) m = fmaxf(m, fabsf(f[w]));
      const float amax = row16_max_f32(m);
      if (p >= nv) continue;  // whole rows of lanes past the end (K not a multiple of 512)
      float mul;
      const float sc = group_scale<MODE>(amax, mul);
      uint32_t pk[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float q0 = quant_value<MODE>(f[4 * h], sc, mul), q1 = quant_value<MODE>(f[4 * h + 1], sc, mul);
        const float q2 = quant_value<MODE>(f[4 * h + 2], sc, mul), q3 = quant_value<MODE>(f[4 * h + 3], sc, mul);
        uint32_t w4 = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(q0, q1, 0, false));
        w4 = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(q2, q3, static_cast<int>(w4), true));
        pk[h] = w4;
      }
      qr[p] = uint2{pk[0], pk[1]};
      if ((lane & 15) == 0) {
        const size_t at = static_cast<size_t>(row) * sstride + gi;
        if (MODE == 0) static_cast<float*>(scales)[at] = sc;
        else static_cast<uint8_t*>(scales)[at] = static_cast<uint8_t>(sc);
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Grouped GEMM
// ----------------------------------------------------------------------------

constexpr int kPRow = 256;            // bytes of a weight or activation row per K step (128 values)
constexpr int kPStride = kPRow + 16;  // LDS row stride
constexpr int kPW = kPBN * kPStride;
constexpr int kPBuf = kPW + kPBM * kPStride;
constexpr int kPLds = 2 * kPBuf;

// Maps a workgroup to (expert or shared, M block, N tile); returns false when idle.
__device__ __forceinline__ bool map_tile(const PrefillGemmArgs& a, int wg, bool& shared, int& expert, int& mblock,
                                         int& ntile) {
  // blocks of the real experts only; ids == num_experts (the sentinel bucket of
  // the align contract) take no part in the GEMMs
  const int routed_wgs = (a.cum[a.num_experts] / kPBM) * a.ntiles;
  if (wg < routed_wgs) {
    // expert owning this workgroup: largest e with cum[e]/BM * ntiles <= wg
    int lo = 0, hi = a.num_experts;  // cum[num_experts] region (sentinel bucket) never has work here
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if ((a.cum[mid] / kPBM) * a.ntiles <= wg) lo = mid; else hi = mid;
    }
    const int b0 = a.cum[lo] / kPBM;
    const int nb = a.cum[lo + 1] / kPBM - b0;
    const int local = wg - b0 * a.ntiles;
    shared = false;
    expert = lo;
    ntile = local / nb;
    mblock = b0 + local % nb;
    return true;
  }
  const int sh0 = a.max_blocks * a.ntiles;
  if (a.shared_blocks > 0 && wg >= sh0 && wg < sh0 + a.shared_blocks * a.ntiles) {
    const int local = wg - sh0;
    shared = true;
    expert = 0;
    ntile = local / a.shared_blocks;
    mblock = local % a.shared_blocks;
    return true;
  }
  return false;
}

template <int GATE_UP>
__global__ void __launch_bounds__(kPThreads) prefill_gemm_kernel(PrefillGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ int s_row[kPBM];   // activation row of each tile column (-1: padding)
  __shared__ int s_route[kPBM]; // route (routed) or token (shared) of each column, -1: padding

  bool shared;
  int expert, mblock, ntile;
  if (!map_tile(a, blockIdx.x, shared, expert, mblock, ntile)) return;

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid / kWave;
  const int wn = wave >> 1, wm = wave & 1;
  const int r16 = lane & 15, g = lane >> 4;

  if (tid < kPBM) {
    int row = -1, route = -1;
    if (shared) {
      const int t = mblock * kPBM + tid;
      if (t < a.M) {
        route = t;
        row = a.x_token_rows ? t : a.numel + t;
      }
    } else {
      const int rr = a.sorted[mblock * kPBM + tid];
      if (rr < a.numel) {
        route = rr;
        row = a.x_token_rows ? rr / a.k : rr;
      }
    }
    s_row[tid] = row;
    s_route[tid] = route;
  }
  __syncthreads();

  const BankView bank = shared ? a.ws : a.w;
  const int n0 = GATE_UP ? ntile * (kPBN / 2) : ntile * kPBN;
  const size_t row_bytes = static_cast<size_t>(a.K) * 2;
  const uint8_t* wexp = bank.w + static_cast<size_t>(expert) * a.N * row_bytes;
  const int nkb = a.K / 128;

  auto wrow_of = [&](int r) -> int {  // weight row held in tile row r
    if (GATE_UP) return r < kPBN / 2 ? n0 + r : a.inter + n0 + (r - kPBN / 2);
    return n0 + r;
  };

  // ---- global -> register staging of one K step
  constexpr int kWChunks = kPBN * kPRow / 16;
  constexpr int kXChunks = kPBM * kPRow / 16;
  constexpr int kWPer = kWChunks / kPThreads;
  constexpr int kXPer = kXChunks / kPThreads;
  u32x4 wreg[kWPer], xreg[kXPer];

  auto load_step = [&](int kb) {
#pragma unroll
    for (int q = 0; q < kWPer; ++q) {
      const int c = tid + q * kPThreads;
      const int r = c / (kPRow / 16), col = c % (kPRow / 16);
      const uint8_t* p = wexp + static_cast<size_t>(wrow_of(r)) * row_bytes + static_cast<size_t>(kb) * kPRow + col * 16;
      wreg[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    }
#pragma unroll
    for (int q = 0; q < kXPer; ++q) {
      const int c = tid + q * kPThreads;
      const int r = c / (kPRow / 16), col = c % (kPRow / 16);
      const int row = s_row[r];
      const int src = row < 0 ? 0 : row;
      const uint8_t* p = a.xq + static_cast<size_t>(src) * row_bytes + static_cast<size_t>(kb) * kPRow + col * 16;
      xreg[q] = *reinterpret_cast<const u32x4*>(p);
    }
  };
  auto store_step = [&](int buf) {
    uint8_t* base = lds + buf * kPBuf;
#pragma unroll
    for (int q = 0; q < kWPer; ++q) {
      const int c = tid + q * kPThreads;
      const int r = c / (kPRow / 16), col = c % (kPRow / 16);
      *reinterpret_cast<u32x4*>(base + r * kPStride + col * 16) = wreg[q];
    }
#pragma unroll
    for (int q = 0; q < kXPer; ++q) {
      const int c = tid + q * kPThreads;
      const int r = c / (kPRow / 16), col = c % (kPRow / 16);
      *reinterpret_cast<u32x4*>(base + kPW + r * kPStride + col * 16) = xreg[q];
    }
  };

  // wave sub-tiles: weight rows (j) and route columns (i)
  int wrow_base[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (GATE_UP) wrow_base[j] = (j < 2) ? 32 * wn + 16 * j : kPBN / 2 + 32 * wn + 16 * (j - 2);
    else wrow_base[j] = 64 * wn + 16 * j;
  }
  const int xcol_base = 64 * wm;

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = zero;

  load_step(0);
  store_step(0);
  __syncthreads();

  for (int kb = 0; kb < nkb; ++kb) {
    const int cur = kb & 1;
    if (kb + 1 < nkb) load_step(kb + 1);
    const uint8_t* base = lds + cur * kPBuf;

    // four K=32 MFMAs per 128 step
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8 xf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint8_t* p = base + kPW + (xcol_base + 16 * i + r16) * kPStride + (g * 32 + s * 8) * 2;
        xf[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint8_t* p = base + (wrow_base[j] + r16) * kPStride + (g * 32 + s * 8) * 2;
        const bf16x8 wf = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[i], acc[j][i], 0, 0, 0);
      }
    }

    if (kb + 1 < nkb) store_step(cur ^ 1);
    __syncthreads();
  }

  // ---- epilogue: lane holds weight rows wrow_base[j] + g*4 + v of route column r16
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = xcol_base + 16 * i + r16;
    const int route = s_route[col];
    if (route < 0) continue;
    if (GATE_UP) {
      const int arow = shared ? a.numel + route : route;
      const float lim = shared ? a.sh_act_limit : a.act_limit;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float gg = bf16_round(acc[s][i][v]);
          float uu = bf16_round(acc[2 + s][i][v]);
          swiglu_clamp(lim, gg, uu);
          o[v] = act_apply(a.act_kind, gg) * uu;
        }
        const int n = n0 + 32 * wn + 16 * s + g * 4;
        uint2 pk;
        pk.x = pack_bf16x2(o[0], o[1]);
        pk.y = pack_bf16x2(o[2], o[3]);
        *reinterpret_cast<uint2*>(a.out + static_cast<size_t>(arow) * a.inter + n) = pk;
      }
    } else {
      const float wt = shared ? 1.0f : a.topk_w[route];
      uint16_t* dst = shared ? a.sh_out + static_cast<size_t>(route) * a.N : a.out + static_cast<size_t>(route) * a.N;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + wrow_base[j] + g * 4;
        uint2 pk;
        pk.x = pack_bf16x2(acc[j][i][0] * wt, acc[j][i][1] * wt);
        pk.y = pack_bf16x2(acc[j][i][2] * wt, acc[j][i][3] * wt);
        *reinterpret_cast<uint2*>(dst + n) = pk;
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Grouped GEMM on direct-to-LDS copies (FP8, MXFP4, bf16)
//
// A workgroup of 8 waves computes 256 weight rows x BM routes.  Wave w is row
// group rg = w/2 (64 weight rows: four 16-row MFMA tiles) and column half
// ch = w%2 (BM/2 routes: BM/32 16-column tiles); two waves share each SIMD, so
// one wave's MFMAs run while the other waits on LDS, folds scales or sits at
// the barrier.  Every operand of a K step -- weight rows, activation tile,
// weight scales, activation scales -- is copied global -> LDS by the LDS-DMA
// form of the global loads (no register staging) into a ring of kStages
// stages: the copies of the next kStages-1 steps are in flight while a step
// computes.  Waits are explicit (vmcnt of whole steps' copies) and the barrier
// is a bare s_barrier, so a barrier never drains copies in flight.  A K step
// is one 128-byte line of every row: 128 values of the quantised formats (64
// bytes of MXFP4 weights), 64 of bf16.
//
// Routes per tile (BM, prefill_block_size): 256 where the experts have that
// many routes; 128 and 64 for shorter batches, where a tile of 256 is mostly
// padding columns whose MFMAs, LDS reads and scale folds cost as much as real
// ones, while the bound is the stream of the weights.  The smaller tiles'
// stages leave room for a deeper ring.
//
// LDS lines (a weight row or an activation column of one K step: 128 bytes,
// 64 for MXFP4 weights) are stored as 16-byte chunks XOR-swizzled by the line
// index (swz_pair, swz_b, swz64: patterns measured free of LDS bank conflicts
// for the way each operand is read).
//
// Gate/up: row group rg owns gate rows n0+32rg+[0,32) and up rows
// I+n0+32rg+[0,32), so SwiGLU pairs registers; a workgroup covers 128
// intermediate features.  Down: rows at or past N (the last tile when
// N % 256 != 0) read zeros and are never stored.  The epilogues
// are VALU work with the matrix cores idle: the gate/up epilogue quantises
// without a division instruction (quant.h) and the down epilogue stores its
// outputs as whole 128-byte rows through LDS.
//
// Schedule (map_tile_q): the active workgroups are laid out XCD-major
// (workgroup b runs on XCD b % 8), so each XCD works through a contiguous range
// of the logical order, in which chunks of q_chunk() M blocks of one expert sweep
// its N tiles: the workgroups an XCD runs at once read several weight tiles and
// share the activations of a few M blocks.
// ----------------------------------------------------------------------------
constexpr int kQRows = 256;   // weight rows per workgroup
constexpr int kQThreads = 512;
constexpr int kXcds = 8;
constexpr int kQDynamicLds = 160 * 1024 - 4096;  // beside the tiles' route and weight lists
// M blocks per chunk of the schedule (see map_tile_q): [FP8, MXFP4][gate_up, down].
// Measured on C5 (interleaved A/B, ms): FP8 gate_up 4 -> 2.23-2.24, 8 -> 2.19-2.20,
// 16 -> 2.22, 2 -> 2.32; FP8 down 4 -> 1.25-1.26, 2 -> 1.20, 1 -> 1.22; MXFP4
// gate_up 4 -> 1.79 (2 and 8 slower by 4-7%); MXFP4 down 4 -> 1.04-1.06, 2 ->
// 1.02-1.04, 8 -> 1.09-1.10.  Tiles of 128 and 64 routes take twice and four
// times as many (the same routes).
constexpr int kQChunkSel[2][2] = {{8, 2}, {4, 2}};
template <int FMT, int GATE_UP, int BM>
constexpr int q_chunk() {
  return kQChunkSel[FMT == FMT_MXFP4 ? 1 : 0][GATE_UP ? 0 : 1] * (256 / BM);
}
// FP8: MFMAs between an MFMA and the fold of its result.  2 -> 3: H 3840, I 896, 32 experts, 2000 tokens
// 331 -> 329 us; H 2432, I 896, 63 experts, 3740 tokens 345 -> 342; H 7168, I 2048, 256 experts, 8192 tokens equal.
constexpr int kFoldLag = 3;

template <int FMT, int BM>
struct QLds {
  // as many stages as fit 160 KB beside the scales and the tile's lists
  static constexpr int kStages = FMT == FMT_MXFP4 ? (BM == 256 ? 3 : BM == 128 ? 4 : 5) : (BM == 256 ? 2 : 3);
  static constexpr bool kQuant = FMT != FMT_BF16;
  static constexpr int kStepK = kQuant ? 128 : 64;            // K values per step
  static constexpr int kALine = FMT == FMT_MXFP4 ? 64 : 128;  // weight bytes per row per K step
  static constexpr int kA = kQRows * kALine;
  static constexpr int kB = BM * 128;
  static constexpr int kStage = kA + kB;
  static constexpr int kRing = kStages * kStage;
  static constexpr int kACopies = kA / 1024 / 8;   // 1 KB copies per wave per step
  static constexpr int kBCopies = kB / 1024 / 8;
  // LDS-DMA instructions each wave issues per K step (uniform over waves; the
  // scale groups come on top)
  static constexpr int kDmaPerStep = kACopies + kBCopies;
  // Scales are copied for four K steps at once, 16 bytes of a row's float32
  // scales or e8m0 codes per lane (4 bytes of the activations' byte codes): a
  // copy per step fetched 4 bytes of every row's line, as many lines per step
  // as the weights and activations together (without any scale copies, timing
  // only, MXFP4 H 5120, I 1536, 12000 routes over 160 experts took 714 -> 648
  // us; in groups 658).  (The 16 columns of a tile then lie 16 bytes apart, which
  // is half of the banks: 12% of the FP8 gate_up's LDS cycles are conflicts.)
  // A group's buffer is written D steps before its first step: with three
  // buffers the one written is never in use; with two (what fits beside 256
  // routes) it is only where a tile's last group is shorter than D, and such a
  // tile does not run ahead into the next.
  static constexpr int kWS = FMT == FMT_FP8 ? 4 * 64 : FMT == FMT_MXFP4 ? kQRows * 16 : 0;
  static constexpr int kXS = FMT == FMT_FP8 ? BM * 16 : FMT == FMT_MXFP4 ? BM * 4 : 0;
  static constexpr int kGroup = kWS + kXS;
  static constexpr int kGroups = BM == 256 ? 2 : 3;
  // LDS before the expert list, whose entries are halved where 1024 of them
  // would not fit (prefill_block_size keeps such calls below 2^16 blocks)
  static constexpr int kFixed = kRing + kGroups * kGroup;
  using Blk = std::conditional_t<FMT == FMT_MXFP4 && BM == 256, uint16_t, int>;
  static_assert(kFixed + (kPrefillMaxRows + 1) * sizeof(Blk) <= kQDynamicLds, "the expert list fits beside the ring");
};

__device__ __forceinline__ int xcd_major(int b, int n) {
  const int per = n / kXcds, rem = n % kXcds;
  const int x = b % kXcds, i = b / kXcds;
  return x * per + min(x, rem) + i;
}

struct MNTile {
  int m, ntile;
};

// (M block, N tile) of position `local` in a group of nb M blocks x ntiles:
// chunks of kQChunk M blocks, each chunk sweeping all N tiles.
// (Returned by value, and from one call per mapping: results written through
// references from two calls lived in scratch memory, whose loads wait for the
// copies in flight.)
template <int kQChunk>
__device__ __forceinline__ MNTile chunked(int local, int nb, int ntiles) {
  const int full = nb / kQChunk, rem = nb - full * kQChunk;
  const int span = kQChunk * ntiles;
  const bool whole = local < full * span;
  const int c = whole ? local / span : full;
  const int w = local - c * span, in = whole ? kQChunk : rem;
  const int ntile = w / in;
  return {c * kQChunk + (w - ntile * in), ntile};
}

// Lane index as an asm result: the compiler can neither hoist nor merge it,
// so per-tile set-up code recomputes its lane-derived values instead of keeping
// them live (or spilled) across the K loop.
__device__ __forceinline__ int fresh_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

struct QTile {
  bool shared;  // the shared expert's blocks (tokens in order) instead of a routed expert's
  int expert, mblock, ntile;
};

// Workgroup b of the grid -> (expert or shared, M block, N tile).  Only the
// active workgroups -- routed blocks of the real experts, then the shared
// expert's blocks -- take part; they are laid out XCD-major over their own
// count, so every XCD gets the same share.  Returns false for idle ones.
// s_blk (LDS): the first M block of every expert, [num_experts] the routed
// total.  The owner of a position is found by the whole wave at once (one
// ballot per 64 experts): a binary search over the regions in global memory
// was a chain of dependent loads at every tile, each of whose waits drained
// the copies in flight.  A workgroup's first tile, with nothing in flight yet,
// takes that search in scalar registers instead of waiting for s_blk (small
// calls, whose workgroups have one tile: H 1280, I 640, 16 experts, 2048 tokens,
// gate_up 30.6 -> 29.9 us).
template <int kQChunk, int BM, bool kFirst, typename Blk>
__device__ __forceinline__ bool map_tile_q(const PrefillGemmArgs& a, const Blk* s_blk, int b, QTile& t) {
  const int E = a.num_experts;
  auto first_block = [&](int e) -> int {
    if constexpr (kFirst) return a.cum[e] / BM;
    else return __builtin_amdgcn_readfirstlane(static_cast<int>(s_blk[e]));
  };
  const int routed = first_block(E) * a.ntiles;
  const int total = routed + a.shared_blocks * a.ntiles;
  if (b >= total) return false;
  const int wg = xcd_major(b, total);
  int local = wg - routed, nb = a.shared_blocks, b0 = 0, owner = 0;
  const bool shared = wg >= routed;
  if (!shared) {  // owner: the largest e whose first tile is <= wg
    if constexpr (kFirst) {
      int hi = E;
      while (hi - owner > 1) {
        const int mid = (owner + hi) >> 1;
        if (first_block(mid) * a.ntiles <= wg) owner = mid;
        else hi = mid;
      }
    } else {
      owner = -1;
      for (int e0 = 0; e0 < E; e0 += 4 * kWave) {
        int first[4];  // four reads in flight (entries past the last expert: its neighbours)
        const int l = fresh_lane();
#pragma unroll
        for (int u = 0; u < 4; ++u) first[u] = s_blk[min(e0 + u * kWave + l, E)];
#pragma unroll
        for (int u = 0; u < 4; ++u) owner += __popcll(__ballot(e0 + u * kWave + l < E && first[u] * a.ntiles <= wg));
      }
      owner = __builtin_amdgcn_readfirstlane(owner);
    }
    b0 = first_block(owner);
    nb = first_block(owner + 1) - b0;
    local = wg - b0 * a.ntiles;
  }
  const MNTile mn = chunked<kQChunk>(local, nb, a.ntiles);
  t.shared = shared;
  t.expert = owner;
  t.mblock = b0 + mn.m;
  t.ntile = mn.ntile;
  return true;
}

// s_barrier without the memory fence of __syncthreads (which would wait for
// every copy in flight); the clobber keeps the compiler from moving LDS
// accesses across it.
__device__ __forceinline__ void bare_barrier() { asm volatile("s_barrier" ::: "memory"); }

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void wait_lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// LDS-DMA copies through a buffer descriptor: each lane's 16 (4) bytes at lane
// offset voff plus the wave-uniform soff land at dst + lane * 16 (4), dst
// wave-uniform; a lane offset at or past the descriptor's range reads zeros
// without memory traffic.
__device__ __forceinline__ void lds_buf16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void lds_buf4(__amdgpu_buffer_rsrc_t r, uint8_t* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, voff, soff, 0, 0);
}

// Chunk swizzles of the LDS lines, chosen by measurement (rocprofv3
// SQ_LDS_BANK_CONFLICT over ds_read_b128 patterns on gfx950): for 128-byte
// lines read as chunk pairs (2g, 2g+1) -- the FP8 and bf16 operands -- position
// c ^ swz_pair(line) is conflict-free while c ^ (line & 7) is not; for lines
// read as chunks (g, 4+g) -- the MXFP4 activations -- c ^ (line & 7) is
// conflict-free; for 64-byte lines read as chunk g -- the MXFP4 weights --
// c ^ ((line >> 1) & 3) is.
__device__ __forceinline__ int swz_pair(int line) { return ((line & 3) << 1) | ((line >> 2) & 1); }
template <int FMT>
__device__ __forceinline__ int swz_b(int line) { return FMT == FMT_MXFP4 ? (line & 7) : swz_pair(line); }
__device__ __forceinline__ int swz64(int line) { return (line >> 1) & 3; }

// Position of a running count in a ring of N.  (Unsigned: the signed remainders
// were a dozen more scalar operations at the head of every step, before its
// first LDS read; FP8 calls gained 0.3-0.8%.)
template <int N>
__device__ __forceinline__ int ring(int i) {
  return static_cast<int>(static_cast<unsigned>(i) % N);
}

// Empty asm that keeps the value's update at this point of the instruction
// stream (no code is emitted).
__device__ __forceinline__ void pin(f32x4& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) { return readlane_u64(v, 0); }

template <int FMT, int GATE_UP, int BM, bool NT>
__global__ void __launch_bounds__(kQThreads) prefill_qgemm_kernel(PrefillGemmArgs a) {
  using L = QLds<FMT, BM>;
  constexpr int S = L::kStages;
  constexpr int D = S - 1;       // prefetch distance in K steps
  constexpr int NCT = BM / 32;   // 16-column tiles per wave
  constexpr bool kQuant = L::kQuant;
  // ring of stages, scale groups, then the first M block of every expert ([num_experts + 1])
  extern __shared__ __attribute__((aligned(16))) uint8_t q_lds[];
  typename L::Blk* const s_blk = reinterpret_cast<typename L::Blk*>(q_lds + L::kFixed);
  // per tile parity: each route column's route (shared tiles: token); padding
  // columns hold a value at or past the tile's limit (col_limit)
  __shared__ int s_route[2][BM];
  __shared__ float s_wt[GATE_UP ? 1 : 2][BM];  // down: per tile parity, router weight of each column

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int rg = wave >> 1, ch = wave & 1;
  const int r16 = lane & 15, g = lane >> 4;
  const int K = a.K, nkb = K / L::kStepK, nsc = K / 128;
  const int ngrp = (nkb + 3) / 4;  // scale groups of a tile
  const uint32_t xsb = FMT == FMT_FP8 ? act_scale_stride(K) * 4u : 1u * act_scale_stride(K);  // bytes of a row's scales
  // bytes of a weight row and of an activation row
  const uint32_t rb = FMT == FMT_BF16 ? 2u * K : FMT == FMT_FP8 ? 1u * K : static_cast<uint32_t>(K) / 2;
  const uint32_t xb = FMT == FMT_BF16 ? 2u * K : 1u * K;

  // (published with the first tile's routes)
  for (int e = tid; e <= a.num_experts; e += kQThreads) s_blk[e] = static_cast<typename L::Blk>(a.cum[e] / BM);
  int v = blockIdx.x;
  QTile cur;
  constexpr int kChunk = q_chunk<FMT, GATE_UP, BM>();
  if (!map_tile_q<kChunk, BM, true>(a, s_blk, v, cur)) return;

  auto n0_of = [&](const QTile& t) -> int { return GATE_UP ? t.ntile * (kQRows / 2) : t.ntile * kQRows; };
  // first weight row of tile j of row group q, relative to the tile's first row n0
  auto trow_rel = [&](int q, int j) -> int {
    if (GATE_UP) return (j < 2 ? 0 : a.inter) + 32 * q + 16 * (j & 1);
    return 64 * q + 16 * j;
  };
  // columns of tile t with s_route at or past this are padding
  auto col_limit = [&](const QTile& t) -> int { return t.shared ? a.M : a.numel; };

  // ---- sources of the copies: buffer descriptors + 32-bit lane offsets of K
  // step 0 (step kb adds kb * step bytes as the scalar offset).  Weight rows,
  // weight scales and activation rows past their range (the last down tile's
  // rows past N, padding route columns) read zeros without memory traffic.
  const int xrows = a.x_token_rows ? a.M : a.numel + a.M;
  const __amdgpu_buffer_rsrc_t rsrc_x = make_rsrc(a.xq, static_cast<uint32_t>(xrows) * xb);
  // (the weights' and scales' ranges are kept as wave-uniform integers: as
  // descriptors carried from tile to tile they were held in vector registers,
  // and every copy ran as a loop over their distinct values)
  uint64_t wbase = 0;
  uint32_t wrange = 0;
  const __amdgpu_buffer_rsrc_t rsrc_wt = make_rsrc(a.topk_w, static_cast<uint32_t>(a.numel) * 4);
  // weights: copy c of wave w fills LDS rows of 1 KB block i = w*kACopies + c
  uint32_t avoff[L::kACopies];
#pragma unroll
  for (int c = 0; c < L::kACopies; ++c) {
    const int i = wave * L::kACopies + c;
    int R, q;
    if constexpr (FMT != FMT_MXFP4) {
      R = 8 * i + (lane >> 3);
      q = (lane & 7) ^ swz_pair(R);
    } else {
      R = 16 * i + (lane >> 2);
      q = (lane & 3) ^ swz64(R);
    }
    avoff[c] = static_cast<uint32_t>(trow_rel(R >> 6, (R >> 4) & 3) + (R & 15)) * rb + q * 16;
  }
  // scales: waves 0-3 copy their row group's weight scales (offsets fixed
  // relative to the tile), the next BM/64 waves 64 activation-scale columns each
  // (sbase, srange: the array this wave copies from; slanes lanes take part)
  const int slanes = wave < 4 ? (FMT == FMT_FP8 ? 4 : kWave) : wave < 4 + BM / 64 ? kWave : 0;
  const int sdst = __builtin_amdgcn_readfirstlane(wave < 4 ? wave * (L::kWS / 4)
                                                           : L::kWS + (wave - 4) * (L::kXS / (BM / 64)));
  uint64_t sbase = reinterpret_cast<uint64_t>(a.xs);
  uint32_t srange = kQuant ? static_cast<uint32_t>(xrows) * xsb : 0u;
  uint32_t svoff = 0;
  if (kQuant && wave < 4) {
    if constexpr (FMT == FMT_FP8) svoff = static_cast<uint32_t>(trow_rel(wave, lane & 3) / 128) * nsc * 4;
    else svoff = static_cast<uint32_t>(trow_rel(wave, lane >> 4) + (lane & 15)) * (K / 32);
  }
  // activations: copy c of wave w fills LDS columns of 1 KB block i = w*kBCopies + c
  uint32_t xvoff[L::kBCopies];
  auto setup = [&](const QTile& t, int b) {
    const BankView bank = t.shared ? a.ws : a.w;
    const int n0 = n0_of(t);
    wbase = uniform_u64(reinterpret_cast<uint64_t>(bank.w) + (static_cast<uint64_t>(t.expert) * a.N + n0) * rb);
    wrange = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a.N - n0) * rb);
    if (kQuant && wave < 4) {
      const uint32_t srow = FMT == FMT_FP8 ? static_cast<uint32_t>(nsc) * 4 : static_cast<uint32_t>(K) / 32;
      const int nrow = FMT == FMT_FP8 ? a.N / 128 : a.N, r0 = FMT == FMT_FP8 ? n0 / 128 : n0;
      const uint64_t at = reinterpret_cast<uint64_t>(bank.s) + (static_cast<uint64_t>(t.expert) * nrow + r0) * srow;
      sbase = uniform_u64(at);
      srange = __builtin_amdgcn_readfirstlane((nrow - r0) * srow);
    }
    // activation row of a column: gate_up the token, down the route (the
    // shared expert's tokens follow the routes)
    const int lim = col_limit(t);
    const uint32_t magic = !t.shared && a.x_token_rows ? a.k_magic : 0u;
    const int add = t.shared && !a.x_token_rows ? a.numel : 0;
    auto row_of = [&](int r) -> uint32_t {
      uint32_t q = static_cast<uint32_t>(r);
      if (magic) {
        q = __umulhi(q, magic);
        // the rounded-up reciprocal gives at most one too many, from r = 2^32 / k on
        q -= q * static_cast<uint32_t>(a.k) > static_cast<uint32_t>(r) ? 1u : 0u;
      }
      return q + add;
    };
    const int ln = fresh_lane();
    if (kQuant && wave >= 4 && wave < 4 + BM / 64) {
      const int r = s_route[b][64 * (wave - 4) + ln];
      svoff = r >= lim ? kOutOfRange : row_of(r) * xsb;
    }
#pragma unroll
    for (int c = 0; c < L::kBCopies; ++c) {
      const int col = 8 * (wave * L::kBCopies + c) + (ln >> 3);
      const int q = (ln & 7) ^ swz_b<FMT>(col);
      const int r = s_route[b][col];
      xvoff[c] = r >= lim ? kOutOfRange : row_of(r) * xb + q * 16;
    }
    if (!GATE_UP && !t.shared && wave < BM / 64) {
      const int r = s_route[b][64 * wave + ln];
      lds_buf4(rsrc_wt, reinterpret_cast<uint8_t*>(&s_wt[b][64 * wave]),
               r >= lim ? kOutOfRange : static_cast<uint32_t>(r) * 4, 0);
    }
  };

  // piece q of a K step's copies (weight copies, activation copies)
  constexpr int kPieces = L::kDmaPerStep;
  auto issue_piece = [&](int q, int kb, int stg) {
    uint8_t* st = q_lds + stg * L::kStage;
    if (q < L::kACopies) {
      lds_buf16(make_rsrc(reinterpret_cast<const void*>(wbase), wrange), st + (wave * L::kACopies + q) * 1024,
                avoff[q], static_cast<uint32_t>(kb) * L::kALine);
    } else {
      const int c = q - L::kACopies;
      lds_buf16(rsrc_x, st + L::kA + (wave * L::kBCopies + c) * 1024, xvoff[c], static_cast<uint32_t>(kb) * 128);
    }
  };
  // the scales of steps kb .. kb+3 (kb % 4 == 0; past the last step unused
  // values) into group buffer grp
  auto scale_group = [&](int grp) { return q_lds + __builtin_amdgcn_readfirstlane(L::kRing + grp * L::kGroup); };
  auto issue_scales = [&](int kb, int grp) {
    if constexpr (FMT == FMT_FP8) {
      // one instruction for both kinds, its descriptor chosen per wave by
      // scalar selects (with a branch per kind the compiler merged the two
      // into one copy whose descriptor sat in vector registers, which runs as
      // a loop over its distinct values)
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const void*>(sbase), srange);
      uint8_t* const gs = scale_group(grp) + sdst;
      if (lane < slanes) lds_buf16(rs, gs, svoff, static_cast<uint32_t>(kb) * 4);
    } else if constexpr (FMT == FMT_MXFP4) {
      uint8_t* const gs = scale_group(grp) + sdst;
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const void*>(sbase), srange);
      if (wave < 4) lds_buf16(rs, gs, svoff, static_cast<uint32_t>(kb) * 4);
      else if (wave < 4 + BM / 64) lds_buf4(rs, gs, svoff, static_cast<uint32_t>(kb));
    }
  };
  auto issue = [&](int kb, int stg, int gb) {
    if ((kb & 3) == 0) issue_scales(kb, ring<L::kGroups>(gb + (kb >> 2)));
#pragma unroll
    for (int q = 0; q < kPieces; ++q) issue_piece(q, kb, stg);
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[4][NCT];

  // K step kb from stage stg, scales from the groups that start at gb.  With
  // ikb >= 0 the copies of step ikb into stage istg (groups from igb) are issued
  // a few per column tile in the first tiles, between the LDS reads and MFMAs,
  // instead of as one burst before the step (a burst stalls the wave's in-order
  // issue until the memory pipeline takes it: measured 3% of the FP8 gate_up
  // GEMM; MXFP4 with 256-route tiles, which has no registers to spare, keeps the
  // burst).
  constexpr bool kSpread = FMT != FMT_MXFP4 || BM < 256;
  constexpr int kPer = NCT == 8 ? 2 : (kPieces + NCT - 1) / NCT;  // pieces per column tile
  auto compute = [&](int kb, int stg, int gb, int ikb, int istg, int igb) {
    const uint8_t* st = q_lds + stg * L::kStage;
    if (ikb >= 0 && (ikb & 3) == 0) issue_scales(ikb, ring<L::kGroups>(igb + (ikb >> 2)));
    const uint8_t* sg = scale_group(ring<L::kGroups>(gb + (kb >> 2)));
    const int sq = kb & 3;  // step of the group
    i32x8 wf[4];
    int wcode[4];
    float sw[4];
    // Row tile j reads weight row 64rg + 16j + r16.  The chunk swizzles depend on
    // the row's low 3 bits (those of r16) only, so every tile's reads are one
    // per-lane base of the step plus a compile-time offset.  (A base per tile took
    // seven more registers than the 256-route MXFP4 kernels have: they spilled,
    // and read one activation tile at a time.  With these and the scheduling
    // barrier below: H 4096, I 1536, 64 experts, 3000 tokens 588 -> 558 us; H 7168,
    // I 2048, 256 experts, 8192 tokens 3166 -> 3008.)
    const int w0 = 64 * rg + r16;
    const uint8_t* const w_lo = FMT == FMT_MXFP4 ? st + w0 * 64 + (g ^ swz64(r16)) * 16
                                                 : st + w0 * 128 + ((2 * g) ^ swz_pair(r16)) * 16;
    const uint8_t* const w_hi = st + w0 * 128 + ((2 * g + 1) ^ swz_pair(r16)) * 16;  // (not MXFP4)
    const uint8_t* const w_sc = FMT == FMT_FP8 ? sg + rg * 64 + sq * 4 : sg + w0 * 16 + sq * 4 + g;
    auto read_w = [&](int j) {
      if constexpr (FMT != FMT_MXFP4) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(w_lo + 2048 * j);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(w_hi + 2048 * j);
        wf[j] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        if constexpr (FMT == FMT_FP8) sw[j] = *reinterpret_cast<const float*>(w_sc + 16 * j);
      } else {
        const u32x4 v4 = *reinterpret_cast<const u32x4*>(w_lo + 1024 * j);
        wf[j] = i32x8{(int)v4[0], (int)v4[1], (int)v4[2], (int)v4[3], 0, 0, 0, 0};
        wcode[j] = w_sc[256 * j];
      }
    };
    // Column tile i reads route column (BM/2)ch + 16i + r16.  The chunk swizzle
    // depends on the column's low 3 bits (those of r16) only, so every tile's
    // reads are one per-lane base of the step plus a compile-time offset
    // (2048 B per tile for the codes, 256 or 64 B for the scales): no address
    // arithmetic per tile.  The f8f6f4 MFMA reads an fp8 lane group g as
    // K = 16g+[0,16) and 64+16g+[0,16), an fp4 lane group as the block
    // [32g, 32g+32); the bf16 MFMAs take chunk 2g of both operands, then
    // chunk 2g+1.
    const int c0 = (BM / 2) * ch + r16;
    const int q_lo = FMT == FMT_MXFP4 ? g ^ swz_b<FMT>(r16) : (2 * g) ^ swz_b<FMT>(r16);
    const int q_hi = FMT == FMT_MXFP4 ? (4 + g) ^ swz_b<FMT>(r16) : (2 * g + 1) ^ swz_b<FMT>(r16);
    const uint8_t* const x_lo = st + L::kA + c0 * 128 + q_lo * 16;
    const uint8_t* const x_hi = st + L::kA + c0 * 128 + q_hi * 16;
    const uint8_t* const x_sc = sg + L::kWS + (FMT == FMT_FP8 ? c0 * 16 + sq * 4 : c0 * 4 + sq);
    auto read_x = [&](int i, i32x8& xf, uint32_t& xs) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(x_lo + 2048 * i);
      const u32x4 hi = *reinterpret_cast<const u32x4*>(x_hi + 2048 * i);
      xf = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      if constexpr (FMT == FMT_FP8) xs = *reinterpret_cast<const uint32_t*>(x_sc + 256 * i);
      else if constexpr (FMT == FMT_MXFP4) xs = x_sc[64 * i];
    };
    // The next column tile's LDS reads are issued before this tile's MFMAs.
    // FP8: each scale fold is written kFoldLag MFMAs after its own MFMA (its
    // result register stays live that long), so the compiler can place the
    // fold's VALU work while the matrix core runs later MFMAs instead of
    // waiting out the MFMA result latency; pin() keeps the accumulator updates
    // in that order.
    i32x8 xf[2];
    uint32_t xs[2] = {0u, 0u};
    if constexpr (FMT != FMT_MXFP4) {
      // The step's first MFMA needs row tile 0 and column tile 0 only: those
      // reads are issued first (LDS returns in order), so after the barrier
      // each wave waits for four reads instead of the whole step's weight
      // tiles (FP8 GEMMs 1.7% faster; MXFP4, whose weight tiles are one read
      // each, 3% slower, so it keeps the weight tiles first)
      read_w(0);
      read_x(0, xf[0], xs[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 1; j < 4; ++j) read_w(j);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) read_w(j);
      read_x(0, xf[0], xs[0]);
    }
    // FP8: kFoldLag MFMA results in flight (tq, with their fold factors fq)
    constexpr int P = kFoldLag;
    f32x4 tq[P];
    float fq[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
      tq[q] = zero;
      fq[q] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < NCT; ++i) {
      if (ikb >= 0) {
#pragma unroll
        for (int q = kPer * i; q < kPer * i + kPer; ++q)
          if (q < kPieces) issue_piece(q, ikb, istg);
      }
      if (i + 1 < NCT) read_x(i + 1, xf[(i + 1) & 1], xs[(i + 1) & 1]);
      // (held here in the 256-route MXFP4 kernels: short of registers, the
      // compiler moved these reads behind the MFMAs, which then waited for each
      // pair of them.  Tile 0 is left to it: the barrier would add tile 1's reads
      // to the wait of the step's first MFMA)
      if (FMT == FMT_MXFP4 && BM == 256 && i > 0) __builtin_amdgcn_sched_barrier(0);
      if constexpr (FMT == FMT_BF16) {
        // two K = 32 MFMAs per tile pair, the dependent one four MFMAs later
        const auto half = [](const i32x8& r, int h) {
          return __builtin_bit_cast(bf16x8, i32x4{r[4 * h], r[4 * h + 1], r[4 * h + 2], r[4 * h + 3]});
        };
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(half(wf[j], h), half(xf[i & 1], h), acc[j][i], 0, 0, 0);
        // (keeps the later tiles' reads from being hoisted into spills)
        if constexpr (BM == 256) __builtin_amdgcn_sched_barrier(0);
        continue;
      }
      // FP8 fold factors of this column tile: a weight scale covers 128 rows,
      // so tiles j = 0, 1 (gate rows) share one and tiles 2, 3 (up rows)
      // another, and the down GEMM's 64 rows of a wave share one
      float fi[2] = {0.f, 0.f};
      if constexpr (FMT == FMT_FP8) fi[0] = __uint_as_float(xs[i & 1]) * sw[0];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (FMT == FMT_FP8) {
          const f32x4 t = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[j], xf[i & 1], zero, 0, 0, 0, 0, 0, 0);
          // the step's first MFMA goes out before anything that waits on the
          // later weight-tile reads (the up rows' scale factor among them)
          if (i == 0 && j == 0) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (GATE_UP) asm volatile("" : "+v"(sw[2]));
          }
          if (j == 1) fi[1] = GATE_UP ? __uint_as_float(xs[i & 1]) * sw[2] : fi[0];
          const int k = 4 * i + j;
          if (k >= P) {
            const int pi = (k - P) >> 2, pj = (k - P) & 3;
            acc[pj][pi] += tq[k % P] * fq[k % P];
            pin(acc[pj][pi]);
          }
          tq[k % P] = t;
          fq[k % P] = fi[j >> 1];
        } else if constexpr (FMT == FMT_MXFP4) {
          acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[j], xf[i & 1], acc[j][i], 4, 0, 0, wcode[j], 0,
                                                                       static_cast<int>(xs[i & 1]));
        }
      }
    }
    if constexpr (FMT == FMT_FP8) {
#pragma unroll
      for (int k = 4 * NCT - P; k < 4 * NCT; ++k) acc[k & 3][k >> 2] += tq[k % P] * fq[k % P];
    }
  };

  // ---- epilogue: lane holds rows trow + g*4 + v of route column (BM/2)ch + 16i + r16
  // (stg: an LDS stage that no copy targets before the next tile's K loop)
  auto epilogue = [&](const QTile& t, int b, uint8_t* stg) {
    const int n0 = n0_of(t);
    const int lim_col = col_limit(t);
    if constexpr (GATE_UP) {
      // SwiGLU, then the down GEMM's activation quantisation of this 128-feature
      // group (one K group of the down GEMM) per route: amax over the 32 features
      // of the wave (lanes g = 0..3 of a column) and over the 4 row groups (LDS).
      // bf16 pairs (v0,v1), (v2,v3) of each column tile and gate/up tile pair (bf16: stored at once)
      uint32_t pk[kQuant ? NCT : 1][2][2];
      float amax[NCT];
      // SiLU (every configuration here) runs as straight-line code with its
      // kind and the clamp of a clamped SwiGLU fixed at compile time; the other
      // kinds keep the runtime choice
      const float lim = t.shared ? a.sh_act_limit : a.act_limit;
      auto swiglu = [&](auto kind, auto clamp) {
#pragma unroll
        for (int i = 0; i < NCT; ++i) {
          float m = 0.f;
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            float o[4];
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
              // gate and up of one feature rounded to bf16 by one packed conversion
              const uint32_t gu = pack_bf16x2(acc[s2][i][v4], acc[2 + s2][i][v4]);
              float gg = __uint_as_float(gu << 16), uu = __uint_as_float(gu & 0xffff0000u);
              if constexpr (decltype(clamp)::value) {
                gg = fminf(gg, lim);
                uu = fminf(fmaxf(uu, -lim), lim);
              }
              float act;
              if constexpr (decltype(kind)::value != ACT_SILU) act = act_apply(a.act_kind, gg);
              else if constexpr (kQuant) act = act_fixed<ACT_SILU>(gg);
              else act = act_apply(ACT_SILU, gg);  // divides, as the decode does
              o[v4] = act * uu;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const uint32_t p2 = pack_bf16x2(o[2 * h], o[2 * h + 1]);
              pk[kQuant ? i : 0][s2][h] = p2;
              if constexpr (kQuant)
                m = fmaxf(m, fmaxf(fabsf(__uint_as_float(p2 << 16)), fabsf(__uint_as_float(p2 & 0xffff0000u))));
            }
          }
          if constexpr (!kQuant) {
            const int route = s_route[b][(BM / 2) * ch + 16 * i + r16];
            if (route < lim_col) {
              const size_t arow = t.shared ? a.numel + route : route;
              uint16_t* const dst = a.out + arow * a.inter + n0 + 32 * rg + g * 4;
              *reinterpret_cast<uint2*>(dst) = uint2{pk[0][0][0], pk[0][0][1]};
              *reinterpret_cast<uint2*>(dst + 16) = uint2{pk[0][1][0], pk[0][1][1]};
            }
          }
          if constexpr (kQuant) {
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            amax[i] = m;
          }
        }
      };
      if (a.act_kind == ACT_SILU) {
        if (lim > 0.f) swiglu(std::integral_constant<int, ACT_SILU>{}, std::true_type{});
        else swiglu(std::integral_constant<int, ACT_SILU>{}, std::false_type{});
      } else {
        swiglu(std::integral_constant<int, -1>{}, std::false_type{});
      }
      if constexpr (kQuant) {
        constexpr int QMODE = FMT == FMT_FP8 ? 0 : 1;
        float* const s_amax = reinterpret_cast<float*>(stg);  // [row group][column]
#pragma unroll
        for (int i = 0; i < NCT; ++i)
          if (g == 0) s_amax[rg * BM + (BM / 2) * ch + 16 * i + r16] = amax[i];
        // publish the amax (LDS only: the next tile's copies stay in flight)
        wait_lgkm0();
        bare_barrier();
        const int sst = act_scale_stride(a.inter);
#pragma unroll
        for (int i = 0; i < NCT; ++i) {
          const int col = (BM / 2) * ch + 16 * i + r16;
          const int route = s_route[b][col];
          if (route >= lim_col) continue;
          const float m = fmaxf(fmaxf(s_amax[col], s_amax[BM + col]), fmaxf(s_amax[2 * BM + col], s_amax[3 * BM + col]));
          float mul;
          const float sc = group_scale<QMODE>(m, mul);
          const int arow = t.shared ? a.numel + route : route;
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            float vals[4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              vals[2 * h] = quant_value<QMODE>(bf16_to_f32(static_cast<uint16_t>(pk[i][s2][h] & 0xffffu)), sc, mul);
              vals[2 * h + 1] = quant_value<QMODE>(bf16_to_f32(static_cast<uint16_t>(pk[i][s2][h] >> 16)), sc, mul);
            }
            uint32_t q4 = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(vals[0], vals[1], 0, false));
            q4 = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(vals[2], vals[3], static_cast<int>(q4), true));
            const int n = n0 + 32 * rg + 16 * s2 + g * 4;
            *reinterpret_cast<uint32_t*>(a.act_q + static_cast<size_t>(arow) * a.inter + n) = q4;
          }
          if (rg == 0 && g == 0) {
            const size_t at = static_cast<size_t>(arow) * sst + t.ntile;
            if (QMODE == 0) static_cast<float*>(a.act_s)[at] = sc;
            else static_cast<uint8_t*>(a.act_s)[at] = static_cast<uint8_t>(sc);
          }
        }
      }
    } else {
      // A lane holds 4 consecutive output rows of a route, so direct stores
      // write 32-byte pieces of 16 routes per instruction.  The outputs are
      // staged in LDS instead (CT column tiles per pass, each wave in its own
      // 128-byte-per-route area, 16-byte chunks swizzled by route so that
      // writes and reads are conflict-free) and stored as whole 128-byte rows
      // of this wave's 64 output rows, 8 routes per instruction: half the
      // store instructions and a quarter of the memory requests.  N is a
      // multiple of 128, so a wave's rows are all inside N or all past it.
      constexpr int CT = L::kStage >= 65536 ? 4 : L::kStage >= 32768 ? 2 : 1;
      static_assert(8 * 16 * CT * 128 <= L::kStage && NCT % CT == 0, "a pass's staging areas fit one stage");
      uint8_t* const mine = stg + wave * (16 * CT * 128);
      const int nrow0 = n0 + 64 * rg;
      const bool rows_in = nrow0 < a.N;
      uint16_t* const base = t.shared ? a.sh_out : a.out;
#pragma unroll
      for (int p = 0; p < NCT / CT; ++p) {
#pragma unroll
        for (int ii = 0; ii < CT; ++ii) {
          const int i = p * CT + ii;
          const int c = 16 * ii + r16;  // staging row of this lane's route
          const float wt = t.shared ? 1.0f : s_wt[b][(BM / 2) * ch + 16 * i + r16];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            uint2 pk2;
            pk2.x = pack_bf16x2(acc[j][i][0] * wt, acc[j][i][1] * wt);
            pk2.y = pack_bf16x2(acc[j][i][2] * wt, acc[j][i][3] * wt);
            // rows 16j + 4g .. +3 are bytes 32j + 8g of the route's 128
            const int chunk = (2 * j + (g >> 1)) ^ (c & 7);
            *reinterpret_cast<uint2*>(mine + c * 128 + chunk * 16 + (g & 1) * 8) = pk2;
          }
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int kk = 0; kk < 2 * CT; ++kk) {
          const int c = 8 * kk + (lane >> 3), chunk = lane & 7;
          const u32x4 v = *reinterpret_cast<const u32x4*>(mine + c * 128 + ((chunk ^ (c & 7)) * 16));
          const int route = s_route[b][(BM / 2) * ch + 16 * (p * CT + (c >> 4)) + (c & 15)];
          if (route < lim_col && rows_in) {
            u32x4* const dst = reinterpret_cast<u32x4*>(base + static_cast<size_t>(route) * a.N + nrow0 + 8 * chunk);
            if constexpr (NT) __builtin_nontemporal_store(v, dst);
            else *dst = v;
          }
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      }
    }
  };

  // ---- route lists.  The column routes of a tile (its align entries) and, for
  // the down GEMM, their router weights (setup) come by LDS-DMA too, so that no
  // wait of an ordinary load drains the copies in flight.
  auto fetch_routes = [&](const QTile& t, int b) {  // columns [64 wave, +64) by waves below BM/64
    if (wave >= BM / 64) return;
    const int ln = fresh_lane();
    if (t.shared) {
      s_route[b][64 * wave + ln] = t.mblock * BM + 64 * wave + ln;
    } else {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.sorted + static_cast<size_t>(t.mblock) * BM, BM * 4);
      lds_buf4(rs, reinterpret_cast<uint8_t*>(&s_route[b][64 * wave]), (64 * wave + ln) * 4, 0);
    }
  };

  // ---- persistent loop over this workgroup's tiles (v, v + grid, ...).  The
  // K pipeline runs over a ring of S LDS stages with copies D steps ahead; the
  // ring continues across tiles (global step g0 + kb), so the last D steps of a
  // tile issue the next tile's first D steps, which land while this tile's
  // epilogue runs.  The next tile's route list is copied at the start of a
  // tile and has landed (and been published by a step's barrier) before its
  // last D steps.
  fetch_routes(cur, 0);
  wait_vm<0>();
  __syncthreads();
  setup(cur, 0);
  int buf = 0, g0 = 0, gb = 0;  // gb: the tile's first scale group
  bool ahead = false;  // this tile's first D steps were issued during the previous tile
  for (;;) {
    if (!ahead) {
#pragma unroll
      for (int d = 0; d < D; ++d)
        if (d < nkb) issue(d, ring<S>(g0 + d), gb);
    }
    QTile nxt;
    const bool has_next = map_tile_q<kChunk, BM, false>(a, s_blk, v + static_cast<int>(gridDim.x), nxt);
    // the next tile's first steps ride in this tile's last D steps, unless its
    // first scale group's buffer would still be in use (kGroups 2 and a last
    // group shorter than D)
    const bool cross = has_next && nkb > D && (L::kGroups > 2 || (nkb & 3) == 0 || (nkb & 3) >= D);
    const int gbn = gb + ngrp;
    // (pinned: a known-zero accumulator would let the compiler schedule the
    // first step, which it peels, apart from the others, at a register cost)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NCT; ++i) {
        acc[j][i] = zero;
        pin(acc[j][i]);
      }
    // step 0 has landed once at most the copies of the D - 1 later steps (and
    // nothing older) are outstanding; what the previous epilogue stored is
    // newer than the copies and counts with them
    if (nkb >= D) wait_vm<(D - 1) * L::kDmaPerStep>();
    else wait_vm<0>();
    bare_barrier();
    if (has_next) fetch_routes(nxt, buf ^ 1);
    // steady steps: step kb + D of this tile is issued; step kb + 1 must have
    // landed at the end (later ones may still fly); every LDS read of the step
    // has returned before its MFMA used it
    int kb = 0;
    for (; kb < nkb - D; ++kb) {
      if constexpr (kSpread) {
        compute(kb, ring<S>(g0 + kb), gb, kb + D, ring<S>(g0 + kb + D), gb);
      } else {
        issue(kb + D, ring<S>(g0 + kb + D), gb);
        compute(kb, ring<S>(g0 + kb), gb, -1, 0, 0);
      }
      wait_vm<(D - 1) * L::kDmaPerStep>();
      wait_lgkm0();
      bare_barrier();
    }
    // The next tile's routes were copied before step D's copies, so from
    // nkb = 2D on the waits above covered them (at least D steady steps);
    // shorter tiles wait for them here.  (Its router weights are copied by
    // setup, before the copies of its first steps, and so have landed with the
    // first of those.)
    if (has_next && nkb < 2 * D) {
      wait_vm<0>();
      wait_lgkm0();
      bare_barrier();
    }
    if (cross) setup(nxt, buf ^ 1);
    for (; kb < nkb; ++kb) {
      if constexpr (kSpread) {
        compute(kb, ring<S>(g0 + kb), gb, cross ? kb + D - nkb : -1, ring<S>(g0 + kb + D), gbn);
      } else {
        if (cross) issue(kb + D - nkb, ring<S>(g0 + kb + D), gbn);
        compute(kb, ring<S>(g0 + kb), gb, -1, 0, 0);
      }
      if (kb + 1 < nkb) {
        if (cross) wait_vm<(D - 1) * L::kDmaPerStep>();
        else wait_vm<0>();
      }
      wait_lgkm0();
      bare_barrier();
    }
    // the stage of this tile's last step: the next tile's first D steps ride
    // in the other stages, and its step D is issued after the barrier that
    // starts its K loop
    epilogue(cur, buf, q_lds + (ring<S>(g0 + nkb + D)) * L::kStage);
    if (!has_next) break;
    ahead = cross;
    cur = nxt;
    buf ^= 1;
    g0 += nkb;
    gb = ring<L::kGroups>(gbn);
    v += static_cast<int>(gridDim.x);
    if (!ahead) setup(cur, buf);
  }
}

hipError_t launch_act_quant(int mode, const uint16_t* x, int rows, int K, int sstride, uint8_t* q, void* scales,
                            hipStream_t stream) {
  const dim3 grid((rows + 3) / 4), block(256);
  if (mode == 0)
    hipLaunchKernelGGL(act_quant_kernel<0>, grid, block, 0, stream, x, rows, K, q, scales, sstride);
  else
    hipLaunchKernelGGL(act_quant_kernel<1>, grid, block, 0, stream, x, rows, K, q, scales, sstride);
  return hipGetLastError();
}

template <int GU>
static hipError_t launch_gemm_t(const PrefillGemmArgs& a, hipStream_t stream) {
  static bool attr = false;
  const void* fn = reinterpret_cast<const void*>(prefill_gemm_kernel<GU>);
  if (!attr) {
    hipError_t err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kPLds);
    if (err != hipSuccess) return err;
    attr = true;
  }
  const int wgs = (a.max_blocks + a.shared_blocks) * a.ntiles;
  hipLaunchKernelGGL((prefill_gemm_kernel<GU>), dim3(wgs), dim3(kPThreads), kPLds, stream, a);
  return hipGetLastError();
}

// CUs of the current device, rounded down to a multiple of the XCD count
static int q_cu_count() {
  static int cached = 0;
  if (cached == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                  hipSuccess || n < kXcds)
      n = 256;
    cached = n / kXcds * kXcds;
  }
  return cached;
}

template <int FMT, int GU, int BM, bool NT = false>
static hipError_t launch_qgemm_t(PrefillGemmArgs a, hipStream_t stream) {
  // the ring, the scale groups, then one int per expert (and the total)
  const int lds = QLds<FMT, BM>::kFixed + (a.num_experts + 1) * static_cast<int>(sizeof(typename QLds<FMT, BM>::Blk));
  static bool attr = false;
  if (!attr) {
    const hipError_t err =
        hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_qgemm_kernel<FMT, GU, BM, NT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kQDynamicLds);
    if (err != hipSuccess) return err;
    attr = true;
  }
  a.ntiles = GU ? a.inter / (kQRows / 2) : (a.N + kQRows - 1) / kQRows;
  // persistent: one workgroup per CU (the LDS ring admits one), each walking
  // tiles b, b + grid, ...; the grid is a multiple of the XCD count, so a
  // workgroup's tiles all map to its own XCD's range
  const long long tiles = static_cast<long long>(a.max_blocks + a.shared_blocks) * a.ntiles;
  const int wgs = static_cast<int>(std::min<long long>(tiles, q_cu_count()));
  if (wgs <= 0) return hipSuccess;
  hipLaunchKernelGGL((prefill_qgemm_kernel<FMT, GU, BM, NT>), dim3(wgs), dim3(kQThreads), lds, stream, a);
  return hipGetLastError();
}

// Down outputs above this are stored nontemporally: they pass the 256 MB
// memory-side cache before the combine reads them.  Measured (us of the call,
// plain / nontemporal): FP8 145 MB 338 / 344, 303 MB 514.7 / 519.7, 397 MB 1098 /
// 1106, 470 MB 1825 / 1819, 1.06 GB 3862 / 3834; MXFP4 1.06 GB 3097 / 3059.  A
// test of the size inside the kernel cost the largest call 1%, so the choice is
// a variant's.
constexpr size_t kStreamedOutputs = size_t{448} << 20;

template <int FMT, int GU>
static hipError_t launch_qgemm_bm(const PrefillGemmArgs& a, hipStream_t stream) {
  if (a.block == 64) return launch_qgemm_t<FMT, GU, 64>(a, stream);
  if (a.block == 128) return launch_qgemm_t<FMT, GU, 128>(a, stream);
  if (a.block == 256) {
    const size_t out_bytes = (static_cast<size_t>(a.numel) + (a.shared_blocks ? a.M : 0)) * a.N * 2;
    if (!GU && out_bytes > kStreamedOutputs) return launch_qgemm_t<FMT, GU, 256, !GU>(a, stream);
    return launch_qgemm_t<FMT, GU, 256>(a, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_prefill_gemm(int fmt, int gate_up, const PrefillGemmArgs& a, hipStream_t stream) {
  if (fmt == FMT_FP8) return gate_up ? launch_qgemm_bm<FMT_FP8, 1>(a, stream) : launch_qgemm_bm<FMT_FP8, 0>(a, stream);
  if (fmt == FMT_MXFP4)
    return gate_up ? launch_qgemm_bm<FMT_MXFP4, 1>(a, stream) : launch_qgemm_bm<FMT_MXFP4, 0>(a, stream);
  if (fmt == FMT_BF16 && a.wide) return gate_up ? launch_gemm_t<1>(a, stream) : launch_gemm_t<0>(a, stream);
  if (fmt == FMT_BF16)
    return gate_up ? launch_qgemm_bm<FMT_BF16, 1>(a, stream) : launch_qgemm_bm<FMT_BF16, 0>(a, stream);
  return hipErrorInvalidValue;
}

}  // namespace ftmoe
