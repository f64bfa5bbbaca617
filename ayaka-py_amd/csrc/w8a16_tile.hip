// W8A16 GEMM for batches past the decode kernels on gfx950 (any M):
// out[M, N] = x[M, K] . dequant(w[N, K])^T.
//
// Bound: the 16-bit matrix cores. Design:
//  * Direct-to-LDS loads into two stage buffers of 64 K; the next stage lands while the
//    current one is multiplied. The weights stay e4m3 in LDS (half the bytes) and are
//    widened where they enter the MFMA, v_mfma_f32_32x32x16_{bf16,f16}.
//  * w * s is rounded to the activation type before the product (the reference's
//    numerics), two VALU instructions a weight: eight wavefronts, two a SIMD, so that one
//    wavefront's conversions run beside the other's MFMAs, and wavefront tiles with more
//    activation than weight rows, so that few wavefronts convert the same weight (256 x
//    256 as 64 x 128 wavefront tiles: 382 us on 4096 x 4096 x 14336, as 128 x 64: 429;
//    128 x 128 as 32 x 128 against 64 x 64: 462 and 491).
//  * 256 x 256, 256 x 128, 128 x 128 and 128 x 64 (n x m) tiles, two to four workgroups a
//    CU for the smaller ones, and a K split, chosen by w16_tile_plan.
// Measured against the register-staged 128 x 128 kernel this replaces (Llama-3-8B, bf16,
// 218 MB of weights, M = 1024): 274 -> 960 TFLOP/s over the four projections; 4096 x
// 14336 at M = 4096 reaches 1260 TFLOP/s, 88% of a bf16 library product on the same card.
#include "w8a16_tile.h"

#include "ayk_common.h"
#include "gemm_tiles.h"
#include "gemm_util.h"
#include "tile_store.h"

namespace ayk {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr int kStepK = 64;          // K elements per stage
constexpr int kWRowB = kStepK;      // weight bytes of one LDS row
constexpr int kXRowB = 2 * kStepK;  // activation bytes of one LDS row

template <bool BF16>
__device__ inline v16f mfma_16bit(const v4i& w, const v4i& x, const v16f& c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, w), __builtin_bit_cast(v8bf, x), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x), c, 0, 0, 0);
  }
}

// Eight e4m3 bytes -> w * s rounded to the activation type.
template <bool BF16>
__device__ inline v4i dequant8(uint32_t lo, uint32_t hi, float s) {
  float f[8];
  e4m3x4_to_f32(lo, f);
  e4m3x4_to_f32(hi, f + 4);
  v4i r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = f[2 * e] * s, b = f[2 * e + 1] * s;
    if constexpr (BF16) {
      r[e] = (int)pack_bf16x2(a, b);
    } else {
      const v2h t = {(_Float16)a, (_Float16)b};
      r[e] = __builtin_bit_cast(int, t);
    }
  }
  return r;
}

// ROW: one scale per weight row (bx >= K); else block scales with bx % 64 == 0.
// WN x WM wavefronts of (BN / WN) weight rows x (BM / WM) activation rows. kps > 0: the
// launch splits K, blockIdx.y takes [y kps, (y + 1) kps) and writes an fp32 partial.
template <bool BF16, bool ROW, int BN, int BM, int WN, int WM, int WGS>
__global__ __launch_bounds__(WN * WM * 64, WGS) void w8a16_tile_kernel(W16TileArgs g, int tiles_m, int64_t kps) {
  constexpr int kWaves = WN * WM;
  constexpr int TN = BN / WN, TM = BM / WM, FN = TN / 32, FM = TM / 32;
  constexpr int kWBytes = BN * kWRowB, kXBytes = BM * kXRowB, kStage = kWBytes + kXBytes;
  constexpr int kWDma = kWBytes / 1024 / kWaves, kXDma = kXBytes / 1024 / kWaves;  // direct loads per wavefront
  static_assert(kWDma >= 1 && kXDma >= 1 && kWBytes % (1024 * kWaves) == 0 && kXBytes % (1024 * kWaves) == 0, "whole loads");
  __shared__ __attribute__((aligned(1024))) uint8_t B0[kStage];
  __shared__ __attribute__((aligned(1024))) uint8_t B1[kStage];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave / WM, wm = wave % WM;
  const int h = lane >> 5, frow = lane & 31;
  int tm, tn;
  big_tile_coords(blockIdx.x, tiles_m, (int)cdiv(g.N, BN), tm, tn);
  const int64_t n_base = (int64_t)tn * BN, m_base = (int64_t)tm * BM;
  const int64_t k0 = kps > 0 ? (int64_t)blockIdx.y * kps : 0;
  const int klen = (int)(kps > 0 && g.K - k0 > kps ? kps : g.K - k0);
  const int ns = (klen + kStepK - 1) / kStepK;

  // Direct loads. Weights: one instruction covers 16 rows x 64 bytes; lane L writes row
  // L / 4, physical 16-byte chunk L % 4, which holds logical chunk (L % 4) ^ (row / 4 % 4).
  // Activations: 8 rows x 128 bytes; row L / 8, physical chunk L % 8 holds logical chunk
  // (L % 8) ^ (row / 2 % 8). Rows past N / M and chunks past K read zeros (they lie
  // beyond the descriptor's records).
  const int ldw = __builtin_amdgcn_readfirstlane((int)g.ldw), ldx = __builtin_amdgcn_readfirstlane((int)(2 * g.ldx));
  const OperandWindow ww = operand_window(n_base, g.N, g.ldw);
  const OperandWindow xw = operand_window(m_base, g.M, 2 * g.ldx);
  const __amdgpu_buffer_rsrc_t wr = uniform_rsrc(g.w + ww.base_offset + k0, ww.records);
  const __amdgpu_buffer_rsrc_t xr = uniform_rsrc(reinterpret_cast<const uint8_t*>(g.x) + xw.base_offset + 2 * k0, xw.records);
  const int wchunk = 16 * ((lane & 3) ^ ((lane >> 4) & 3));  // the lane's row / 4 % 4 is lane / 16
  const int wvoff = (lane >> 2) * ldw + wchunk;
  // row / 2 % 8 of row 8 i + lane / 8 is 4 (i % 2) + lane / 16
  const int xchunk_e = 16 * ((lane & 7) ^ (lane >> 4)), xchunk_o = 16 * ((lane & 7) ^ (4 + (lane >> 4)));
  const int xvoff_e = (lane >> 3) * ldx + xchunk_e, xvoff_o = (lane >> 3) * ldx + xchunk_o;
  constexpr int kPast = (int)0x80000000u;  // an offset past every window (records < 2^31)
  auto issue = [&](int s, uint8_t* dst) {
    const int k = s * kStepK;
    const int left = klen - k;  // K elements from this stage on
    const int wv = wchunk < left ? wvoff : kPast;
    const int xve = xchunk_e < 2 * left ? xvoff_e : kPast, xvo = xchunk_o < 2 * left ? xvoff_o : kPast;
#pragma unroll
    for (int j = 0; j < kWDma; ++j) {
      const int i = wave * kWDma + j;
      const int soff = __builtin_amdgcn_readfirstlane(16 * i * ldw + k);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(dst + 1024 * i), 16, wv, soff, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kXDma; ++j) {
      const int i = wave * kXDma + j;
      const int soff = __builtin_amdgcn_readfirstlane(8 * i * ldx + 2 * k);
      const bool odd = kXDma % 2 == 0 ? (j & 1) : (i & 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(dst + kWBytes + 1024 * i), 16,
                                               odd ? xvo : xve, soff, 0, 0);
    }
  };

  // The scales of this lane's weight rows: one each, or one each and stage.
  float sc[FN], sc_next[FN];
  int64_t srow[FN];
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    int64_t n = n_base + wn * TN + i * 32 + frow;
    n = n < g.N ? n : g.N - 1;
    srow[i] = (int64_t)((uint64_t)n / (uint64_t)g.by) * g.srs;
    sc[i] = ROW ? load_f32(g.scale, g.scale_dtype, srow[i]) : 1.0f;
  }
  auto block_scales = [&](int s, float (&v)[FN]) {  // bx % 64 == 0: a stage lies in one scale block
    const int64_t kb = (int64_t)((uint32_t)(k0 + (int64_t)s * kStepK) / (uint32_t)g.bx);
#pragma unroll
    for (int i = 0; i < FN; ++i) v[i] = load_f32(g.scale, g.scale_dtype, srow[i] + kb);
  };

  // Fragment reads: lane (frow, h) of a 32-K pair q takes K [32 q + 16 h, +16): one
  // 16-byte weight chunk and two activation chunks, the operands of two MFMAs.
  const int wsw = (frow >> 2) & 3, xsw = (frow >> 1) & 7;
  int woff[2], xoff[2][2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    woff[q] = frow * kWRowB + (((2 * q + h) ^ wsw) << 4);
#pragma unroll
    for (int c = 0; c < 2; ++c) xoff[q][c] = frow * kXRowB + (((4 * q + 2 * h + c) ^ xsw) << 4);
  }
  v16f acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  auto compute = [&](const uint8_t* buf) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      v4i wq[FN], xf[FM][2];
#pragma unroll
      for (int i = 0; i < FN; ++i) wq[i] = *reinterpret_cast<const v4i*>(buf + (wn * TN + 32 * i) * kWRowB + woff[q]);
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          xf[j][c] = *reinterpret_cast<const v4i*>(buf + kWBytes + (wm * TM + 32 * j) * kXRowB + xoff[q][c]);
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        v4i lo, hi;
        lo = dequant8<BF16>((uint32_t)wq[i][0], (uint32_t)wq[i][1], sc[i]);
        hi = dequant8<BF16>((uint32_t)wq[i][2], (uint32_t)wq[i][3], sc[i]);
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mfma_16bit<BF16>(lo, xf[j][0], acc[i][j]);
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mfma_16bit<BF16>(hi, xf[j][1], acc[i][j]);
      }
    }
  };

  if constexpr (!ROW) block_scales(0, sc);
  issue(0, B0);
  wait_vmcnt<0>();
  lds_barrier();
  // Stage s is visible in `cur` and nothing is in flight; stage s + 1 lands in `nxt`
  // (read by nobody since the last barrier) while stage s is multiplied.
  auto step = [&](int s, uint8_t* cur, uint8_t* nxt) {
    if (s + 1 < ns) {
      issue(s + 1, nxt);
      if constexpr (!ROW) block_scales(s + 1, sc_next);
    }
    compute(cur);
    wait_vmcnt<0>();
    lds_barrier();
    if constexpr (!ROW) {
#pragma unroll
      for (int i = 0; i < FN; ++i) sc[i] = sc_next[i];
    }
  };
  for (int s = 0; s < ns; s += 2) {
    step(s, B0, B1);
    if (s + 1 < ns) step(s + 1, B1, B0);  // workgroup-uniform
  }

  // Epilogue. D[n][m]: lane holds m = lane % 32 and n = 8 (r / 4) + 4 h + r % 4 of a tile.
  const int64_t n_w = n_base + wn * TN, m_w = m_base + wm * TM;
  if (kps > 0) {  // fp32 partials, read back by the reduce
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int64_t m = m_w + 32 * j + frow;
      if (m >= g.M) continue;
      float* prow = g.part + ((int64_t)blockIdx.y * g.M + m) * g.N;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
          const int64_t n = n_w + 32 * i + 8 * grp + 4 * h;
          const float v[4] = {acc[i][j][4 * grp], acc[i][j][4 * grp + 1], acc[i][j][4 * grp + 2], acc[i][j][4 * grp + 3]};
          store4_f32(prow + n, g.N - n, v);
        }
    }
    return;
  }
  // Every wavefront stages 32 (m) x TN (n) slabs in a private region of the stage buffers.
  constexpr int kRegion = 32 * TN * 2, kPerBuf = kStage / kRegion;
  static_assert(2 * kPerBuf >= kWaves, "the staging regions fit the stage buffers");
  uint8_t* region = wave < kPerBuf ? B0 + wave * kRegion : B1 + (wave - kPerBuf) * kRegion;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int grp = 0; grp < 4; ++grp) {
        const float v[4] = {acc[i][j][4 * grp], acc[i][j][4 * grp + 1], acc[i][j][4 * grp + 2], acc[i][j][4 * grp + 3]};
        stage_slab16<BF16, TN>(region, frow, 2 * (32 * i + 8 * grp + 4 * h), v);
      }
    store_slab16<TN>(region, static_cast<uint16_t*>(g.out), g.ldo, g.M, g.N, m_w + 32 * j, n_w, lane);
  }
}

// Fixed-order sum of the K-split partials, one rounding, for N or alignments the
// four-element reduce does not take.
__global__ __launch_bounds__(256) void w8a16_tile_reduce(const float* __restrict__ part, int64_t M, int64_t N, int split,
                                                         const void* __restrict__, int, void* __restrict__ out,
                                                         int out_dtype, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * N) return;
  float v = 0.0f;
  for (int s = 0; s < split; ++s) v += part[(int64_t)s * M * N + i];
  store_f32(out, out_dtype, i / N * ldo + i % N, v);
}

// Tile and K split of a shape: the pair with the smallest modelled time. The model, in
// microseconds, was fitted on 13 weight shapes from 2048 x 1024 to 37888 x 3584 and 13
// batches from 40 to 4096 (cold weights): a CU that runs u workgroups of a tile takes
// max(u tau, ceil(u / resident) lambda) per 64-K stage (throughput, or one round's
// latency) and an epilogue in proportion to its output; a split adds a reduce launch and
// the fp32 partials' traffic. Over those shapes its choice is 1.4% slower than the
// fastest tile and split on average, 15% at worst. It runs for every workspace query and
// launch: no division in its loops has a variable divisor (0.27 us a plan with them, 0.10 without).
struct TileConfig {
  int bn, bm, resident;
  float tau, lambda;
};
constexpr TileConfig kConfigs[4] = {
    {256, 256, 1, 1.31f, 1.43f}, {256, 128, 2, 0.83f, 1.0f}, {128, 128, 3, 0.49f, 0.72f}, {128, 64, 4, 0.32f, 0.53f}};
constexpr int kSplits[8] = {1, 2, 3, 4, 6, 8, 12, 16};
constexpr int kMinSplitK = 512;  // shorter K pieces never paid for the reduce
constexpr int kCus = 256;

int64_t stages(int64_t K) { return cdiv(K, kStepK); }
int64_t split_kps(int64_t K, int split) { return cdiv(stages(K), split) * kStepK; }

// Tiles of `side` rows (64, 128 or 256).
int64_t tile_count(int64_t rows, int side) { return side == 256 ? cdiv(rows, 256) : (side == 128 ? cdiv(rows, 128) : cdiv(rows, 64)); }
int64_t by_resident(int64_t n, int resident) {
  return resident == 1 ? n : (resident == 2 ? cdiv(n, 2) : (resident == 3 ? cdiv(n, 3) : cdiv(n, 4)));
}

size_t split_bytes(const W16TilePlan& p, int64_t M, int64_t N) {
  return p.split > 1 ? (size_t)p.split * (size_t)M * (size_t)N * sizeof(float) : 0;
}

}  // namespace

W16TilePlan w16_tile_plan(int64_t M, int64_t N, int64_t K, bool may_split) {
  W16TilePlan best{0, 1, 0.0f};
  bool first = true;
  int splits = 1;
  while (may_split && splits < 8 && K >= (int64_t)kMinSplitK * kSplits[splits]) ++splits;
  int64_t pieces[8];  // stages of one
  for (int i = 0; i < splits; ++i) pieces[i] = cdiv(stages(K), kSplits[i]);
  for (int c = 0; c < 4; ++c) {
    const TileConfig& t = kConfigs[c];
    const int64_t tiles = tile_count(M, t.bm) * tile_count(N, t.bn);
    for (int i = 0; i < splits; ++i) {
      const int s = kSplits[i];
      const int64_t wgs = cdiv(tiles * s, kCus);  // a CU
      const float u = (float)wgs, rounds = (float)by_resident(wgs, t.resident);
      const float stage = rounds * t.lambda > u * t.tau ? rounds * t.lambda : u * t.tau;
      float us = (float)pieces[i] * stage + 1.5f * u * (float)(t.bn * t.bm) / 65536.0f;
      if (s > 1) us += 5.0f + 1.6e-6f * (float)s * (float)M * (float)N;
      if (first || us < best.us) {
        first = false;
        best = {c, s, us};
      }
    }
  }
  best.split = (int)cdiv(K, split_kps(K, best.split));  // whole stages a piece may need fewer pieces
  return best;
}

namespace {

template <bool BF16, bool ROW>
void launch_config(const W16TileArgs& a, const W16TilePlan& p, hipStream_t st) {
  const TileConfig& t = kConfigs[p.config];
  const int tiles_m = (int)cdiv(a.M, t.bm);
  const dim3 grid((unsigned)(tiles_m * cdiv(a.N, t.bn)), (unsigned)p.split);
  const int64_t kps = p.split > 1 ? split_kps(a.K, p.split) : 0;
  switch (p.config) {
    case 0: hipLaunchKernelGGL((w8a16_tile_kernel<BF16, ROW, 256, 256, 4, 2, 1>), grid, dim3(512), 0, st, a, tiles_m, kps); break;
    case 1: hipLaunchKernelGGL((w8a16_tile_kernel<BF16, ROW, 256, 128, 8, 1, 1>), grid, dim3(512), 0, st, a, tiles_m, kps); break;
    case 2: hipLaunchKernelGGL((w8a16_tile_kernel<BF16, ROW, 128, 128, 4, 1, 3>), grid, dim3(256), 0, st, a, tiles_m, kps); break;
    default: hipLaunchKernelGGL((w8a16_tile_kernel<BF16, ROW, 128, 64, 4, 1, 4>), grid, dim3(256), 0, st, a, tiles_m, kps); break;
  }
}

}  // namespace

size_t w16_tile_workspace(int64_t M, int64_t N, int64_t K) { return split_bytes(w16_tile_plan(M, N, K), M, N); }

// The weights stream at no more than 4.4 TB/s beside a launch and its prologue.
float w16_tile_time(const W16TilePlan& p, int64_t N, int64_t K) {
  const float stream = 6.0f + (float)N * (float)K / 4.4e6f;
  return p.us > stream ? p.us : stream;
}

bool w16_tile_supported(const W16TileArgs& a) {
  // 32-bit offsets within a tile's rows; whole stages of one scale block.
  return (a.bx >= a.K || a.bx % kStepK == 0) && a.K < ((int64_t)1 << 30) && 256 * a.ldw < ((int64_t)1 << 31) &&
         512 * a.ldx < ((int64_t)1 << 31) && cdiv(a.M, 64) * cdiv(a.N, 128) < ((int64_t)1 << 31);
}

int w16_tile_launch(const W16TileArgs& a, W16TilePlan p, bool bf16, hipStream_t st, const char* op) {
  // A caller that brings no workspace gets the best plan without a split.
  if (p.split > 1 && (a.part == nullptr || a.part_bytes < split_bytes(p, a.M, a.N))) p = w16_tile_plan(a.M, a.N, a.K, false);
  const bool row = a.bx >= a.K;
  note_plan("w8a16 tile %dx%d split=%d", kConfigs[p.config].bn, kConfigs[p.config].bm, p.split);
  if (bf16) row ? launch_config<true, true>(a, p, st) : launch_config<true, false>(a, p, st);
  else row ? launch_config<false, true>(a, p, st) : launch_config<false, false>(a, p, st);
  if (int rc = check_launch(op)) return rc;
  if (p.split == 1) return AYK_OK;
  launch_split_reduce(w8a16_tile_reduce, a.part, a.M, a.N, p.split, nullptr, 0, a.out, bf16 ? AYK_BF16 : AYK_F16, a.ldo, st);
  return check_launch(op);
}

}  // namespace ayk
