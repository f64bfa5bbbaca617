// W8A8 GEMM on medium tiles, gfx950: out[M, N] = epilogue(a[M, K] . w[N, K]^T) for the
// batches between the decode kernels and the 256 x 256 pair kernels, for shapes whose
// 256 x 256 tiles leave CUs idle, and for every K, N, scale type and alignment that the
// pair kernels refuse. Recipes as in gemm.hip: per-row / per-tensor scales, 128 x 128
// block scales, MXFP8 codes, INT8.
//
// Bound: at these sizes the weight stream and its latency (M = 65 .. 255), then the matrix
// cores. Design:
//  * 256 x 256 (eight wavefronts), 128 x 128 and 128 x 64 (four, two or three workgroups a
//    CU) tiles on v_mfma_scale_f32_32x32x64_f8f6f4, weight = operand A: a lane's
//    accumulator column is one activation row.
//  * Direct-to-LDS loads (8 rows x 128 bytes an instruction) into two 128-K stage buffers;
//    the next stage lands while the current one is multiplied, and the other workgroups of
//    the CU run while one waits at its stage barrier.
//  * A K tail is zero-filled by the loads' bounds check, so any K % 16 == 0 takes the same
//    loop; rows past M and N likewise.
//  * Block scales: a 128-K stage is one scale block; its two MFMAs start from zero and one
//    fma an accumulator folds them with sa[m, kb] sb[n / 128, kb].
//  * MXFP8 codes: four stages' codes of a row are one 16-byte direct load into LDS (rows
//    that are only 4-byte aligned: one dword a stage; unaligned rows: the two dwords that
//    hold it).
//  * Tile and K split come from a fitted time model (mid_plan), which gemm.hip also holds
//    against the other kernels' (mid_time).
// Measured (kernel alone in a graph, against the kernels these shapes ran before; 4096 x
// 14336, 37888 x 3584): per-row M = 65 54.2 -> 26.2 us and 87 -> 37, M = 128 60.8 -> 31.7
// and 96 -> 39; MXFP8 M = 128 47.0 -> 33.6 and 83 -> 45; block-128 37888 x 3584 M = 128
// 76 -> 43; per-row 4096 x 4096 M = 1024 41.3 -> 25.9, 3072 x 1024 M = 65 21.2 -> 8.4.
#include "gemm_mid.h"

#include "ayk_common.h"
#include "gemm_tiles.h"
#include "gemm_util.h"
#include "tile_store.h"

namespace ayk {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kStageK = 128;     // K bytes per stage: two MFMA steps, one 128-K scale block
constexpr int kCodeOne = 127;    // UE8M0 code of 1.0
// Kernel modes for MX codes whose rows are only 4-byte aligned (K % 128 == 0), or not at all.
constexpr int kMidMx4 = 4, kMidMxAny = 5;
constexpr bool mx_mode(int mode) { return mode == kMidMx || mode == kMidMx4 || mode == kMidMxAny; }
// Stages whose codes are loaded together, and their LDS bytes a row (unaligned rows: the
// two aligned dwords that hold a stage's four codes).
constexpr int code_stages(int mode) { return mode == kMidMx ? 4 : 1; }
constexpr int code_bytes(int mode) { return mode == kMidMx ? 16 : (mode == kMidMx4 ? 4 : (mode == kMidMxAny ? 8 : 0)); }

// One 64-K step of a 32 x 32 tile. Lane half h holds K [16 h, +16) and [32 + 16 h, +16) of
// the step; the scaled MFMA applies the code of half b to K block [32 b, +32). INT8 sums
// travel in the accumulator registers bit for bit (exact int32).
template <int MODE, int SEL>
__device__ inline v16f mid_mma(const v8i& w, const v8i& a, const v16f& c, int cw, int ca) {
  if constexpr (MODE == kMidInt8) {
    v16i acc = __builtin_bit_cast(v16i, c);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_shufflevector(w, w, 0, 1, 2, 3), __builtin_shufflevector(a, a, 0, 1, 2, 3),
                                                acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_shufflevector(w, w, 4, 5, 6, 7), __builtin_shufflevector(a, a, 4, 5, 6, 7),
                                                acc, 0, 0, 0);
    return __builtin_bit_cast(v16f, acc);
  } else if constexpr (mx_mode(MODE)) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, 0, 0, SEL, cw, SEL, ca);
  } else {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, 0, 0, 0, kCodeOne, 0, kCodeOne);
  }
}

// WN x WM wavefronts of (BN / WN) weight rows x (BM / WM) activation rows. kps > 0: the
// launch splits K (whole 128-K stages), blockIdx.y takes [y kps, (y + 1) kps) and writes
// an fp32 partial without the bias.
template <int MODE, int BN, int BM, int WN, int WM, int WGS>
__global__ __launch_bounds__(WN * WM * 64, WGS) void fp8_mid_kernel(MidArgs g, int tiles_m, int64_t kps) {
  constexpr int kThreads = WN * WM * 64, kWaves = WN * WM;
  constexpr int TN = BN / WN, TM = BM / WM, FN = TN / 32, FM = TM / 32;
  constexpr int kRows = BN + BM, kStage = kRows * kStageK;
  constexpr int kWDma = BN / 8 / kWaves, kADma = BM / 8 / kWaves;  // direct loads per wavefront and stage
  static_assert(BN % (16 * kWaves) == 0 && BM % (16 * kWaves) == 0, "whole pairs of loads per wavefront");
  __shared__ __attribute__((aligned(1024))) uint8_t B0[kStage];
  __shared__ __attribute__((aligned(1024))) uint8_t B1[kStage];
  __shared__ float col_scale[BN], col_bias[BN];
  constexpr int CS = code_stages(MODE), kCodeB = code_bytes(MODE), kCodes = kCodeB ? kRows * kCodeB : 16;  // one chunk
  __shared__ __attribute__((aligned(1024))) uint8_t code_lds[2 * kCodes];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave / WM, wm = wave % WM;
  const int h = lane >> 5, frow = lane & 31;
  int tm, tn;
  big_tile_coords(blockIdx.x, tiles_m, (int)cdiv(g.N, BN), tm, tn);
  const int64_t n_base = (int64_t)tn * BN, m_base = (int64_t)tm * BM;
  const int64_t k0 = kps > 0 ? (int64_t)blockIdx.y * kps : 0;
  const int klen = (int)(kps > 0 && g.K - k0 > kps ? kps : g.K - k0);
  const int ns = (klen + kStageK - 1) / kStageK;

  // Direct loads: instruction i covers LDS rows 8 i .. 8 i + 7 (the BN weight rows, then the
  // BM activation rows) x 128 bytes. Lane L writes row 8 i + L / 8 at physical chunk L % 8,
  // which holds logical 16-byte chunk (L % 8) ^ (row / 2 % 8). Rows past N / M and chunks
  // past K read zeros (they lie beyond the descriptor's records).
  const int ldw = __builtin_amdgcn_readfirstlane((int)g.ldw), lda = __builtin_amdgcn_readfirstlane((int)g.lda);
  const OperandWindow ww = operand_window(n_base, g.N, g.ldw), aw = operand_window(m_base, g.M, g.lda);
  const __amdgpu_buffer_rsrc_t wr = uniform_rsrc(g.w + ww.base_offset + k0, ww.records);
  const __amdgpu_buffer_rsrc_t ar = uniform_rsrc(g.a + aw.base_offset + k0, aw.records);
  // row / 2 % 8 of row 8 i + L / 8 is 4 (i % 2) + L / 16
  const int chunk_e = 16 * ((lane & 7) ^ (lane >> 4)), chunk_o = 16 * ((lane & 7) ^ (4 + (lane >> 4)));
  constexpr int kPast = (int)0x80000000u;  // an offset past every window (records < 2^31)
  auto issue = [&](int s, uint8_t* dst) {
    const int left = klen - s * kStageK;  // K bytes from this stage on
    const int row = lane >> 3;
    const int ce = chunk_e < left ? chunk_e : kPast, co = chunk_o < left ? chunk_o : kPast;
    const int we = ce < 0 ? kPast : row * ldw + ce, wo = co < 0 ? kPast : row * ldw + co;
    const int ae = ce < 0 ? kPast : row * lda + ce, ao = co < 0 ? kPast : row * lda + co;
#pragma unroll
    for (int j = 0; j < kWDma; ++j) {
      const int i = wave * kWDma + j;
      const int soff = __builtin_amdgcn_readfirstlane(8 * i * ldw + s * kStageK);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(dst + 1024 * i), 16,
                                               (j & 1) ? wo : we, soff, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kADma; ++j) {
      const int i = wave * kADma + j;
      const int soff = __builtin_amdgcn_readfirstlane(8 * i * lda + s * kStageK);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (__attribute__((address_space(3))) void*)(dst + BN * kStageK + 1024 * i), 16,
                                               (j & 1) ? ao : ae, soff, 0, 0);
    }
  };

  // Activation rows of this lane's fragments, clamped to M.
  int64_t mrow[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int64_t m = m_base + wm * TM + 32 * j + frow;
    mrow[j] = m < g.M ? m : g.M - 1;
  }
  // Epilogue tables: the columns' weight scale and bias; a lane's rows' activation scale.
  float row_sa[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) row_sa[j] = 1.0f;
  if constexpr (MODE == kMidScaled || MODE == kMidInt8) {
#pragma unroll
    for (int j = 0; j < FM; ++j) row_sa[j] = load_f32(g.sa, g.sa_dtype, g.sa_vec ? mrow[j] : 0);
  }
  for (int t = tid; t < BN; t += kThreads) {
    const int64_t n = n_base + t < g.N ? n_base + t : g.N - 1;
    if constexpr (MODE == kMidScaled || MODE == kMidInt8) col_scale[t] = load_f32(g.sb, g.sb_dtype, g.sb_vec ? n : 0);
    col_bias[t] = g.bias && kps == 0 ? load_f32(g.bias, g.bias_dtype, n) : 0.0f;
  }

  // Per-stage scales. MX: the codes of this lane half's 32-K blocks, byte 2 t for step t.
  // Block: sa[m, kb] and sb[n / 128, kb] as raw words (a 32-row slab lies in one 128-row
  // block), decoded when used.
  struct Scales {
    int cw[FN], ca[FM];
    RawBits sa[FM], sb[FN];
  };
  const int64_t kblocks = cdiv(g.K, 128);
  const int64_t sa_ld = g.ld_sa > 0 ? g.ld_sa : kblocks, sb_ld = g.ld_sb > 0 ? g.ld_sb : kblocks;
  auto load_scales = [&](int s, Scales& v) {
    const int64_t kb = k0 / kStageK + s;
    if constexpr (MODE == kMidBlock) {
#pragma unroll
      for (int j = 0; j < FM; ++j) v.sa[j] = load_bits(g.sa, g.sa_dtype, g.sa_vec ? kb * g.M + mrow[j] : mrow[j] * sa_ld + kb);
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int64_t n = n_base + wn * TN + 32 * i;
        v.sb[i] = load_bits(g.sb, g.sb_dtype, (n < g.N ? n : g.N - 1) / 128 * sb_ld + kb);
      }
    }
  };
  // MX codes go through LDS for all wavefronts, one or two direct loads a row and chunk of
  // CS stages. A dword a row and stage straight into each wavefront's registers asked for
  // more cache lines than the operands themselves. The windows start at a 4-byte boundary
  // and end with the last row's last code (rounded up to a dword, which lies in its page).
  // `mis`: bytes from a window's start to the tile's first code.
  const uintptr_t cwp = reinterpret_cast<uintptr_t>(g.sb) + (uintptr_t)(n_base * g.ld_sb + k0 / 32);
  const uintptr_t cap = reinterpret_cast<uintptr_t>(g.sa) + (uintptr_t)(m_base * g.ld_sa + k0 / 32);
  const int cw_mis = __builtin_amdgcn_readfirstlane((int)(cwp & 3)), ca_mis = __builtin_amdgcn_readfirstlane((int)(cap & 3));
  const int cw_ld = __builtin_amdgcn_readfirstlane((int)g.ld_sb), ca_ld = __builtin_amdgcn_readfirstlane((int)g.ld_sa);
  auto code_records = [&](int64_t rows_left, int64_t ldc, int mis) {  // the tile's first row lies inside the operand
    const int64_t bytes = ((rows_left - 1) * ldc + (g.K - k0 + 31) / 32 + mis + 3) & ~(int64_t)3;
    return (int32_t)(bytes < 0x7FFFFFFC ? bytes : 0x7FFFFFFC);
  };
  const __amdgpu_buffer_rsrc_t cwr =
      uniform_rsrc(reinterpret_cast<const void*>(cwp - cw_mis), kCodeB ? code_records(g.N - n_base, g.ld_sb, cw_mis) : 0);
  const __amdgpu_buffer_rsrc_t car =
      uniform_rsrc(reinterpret_cast<const void*>(cap - ca_mis), kCodeB ? code_records(g.M - m_base, g.ld_sa, ca_mis) : 0);
  auto issue_codes = [&](int s) {  // the chunk that stage s begins
    if constexpr (kCodeB > 0) {
      if (s % CS) return;
      uint8_t* chunk = code_lds + (s / CS % 2) * kCodes;
      for (int t = wave; t < kRows / 64; t += kWaves) {
        const bool w_side = 64 * t < BN;
        const __amdgpu_buffer_rsrc_t rsrc = w_side ? cwr : car;
        const int voff = w_side ? (64 * t + lane) * cw_ld + cw_mis : (64 * t - BN + lane) * ca_ld + ca_mis;
        if constexpr (MODE == kMidMx) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(chunk + 1024 * t), 16, voff,
                                                   4 * s, 0, 0);
        } else {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(chunk + 256 * t), 4,
                                                   voff & ~3, 4 * s, 0, 0);
          if constexpr (MODE == kMidMxAny) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rsrc, (__attribute__((address_space(3))) void*)(chunk + 4 * kRows + 256 * t), 4, (voff & ~3) + 4, 4 * s, 0, 0);
          }
        }
      }
    }
  };
  auto read_codes = [&](int s, Scales& v) {
    if constexpr (kCodeB > 0) {
      const uint8_t* chunk = code_lds + (s / CS % 2) * kCodes;
      // Codes past K are 1.0: their operands are zeros, which a NaN code would turn into NaN.
      const int valid = (klen - s * kStageK + 31) / 32;
      const uint32_t past = MODE == kMidMxAny && valid < 4 ? 0xFFFFFFFFu << (8 * valid) : 0u;
      auto codes = [&](int row, int byte) -> int {  // byte: the row's first code, from its window's start
        uint32_t w;
        if constexpr (MODE == kMidMx) {
          w = *reinterpret_cast<const uint32_t*>(chunk + 16 * row + 4 * (s % CS));
        } else {
          w = *reinterpret_cast<const uint32_t*>(chunk + 4 * row);
          if constexpr (MODE == kMidMxAny) {
            const uint32_t hi = *reinterpret_cast<const uint32_t*>(chunk + 4 * kRows + 4 * row);
            w = __builtin_amdgcn_alignbyte(hi, w, (uint32_t)byte & 3);
            w = (w & ~past) | (0x7F7F7F7Fu & past);
          }
        }
        return (int)(w >> (8 * h));
      };
#pragma unroll
      for (int i = 0; i < FN; ++i) v.cw[i] = codes(wn * TN + 32 * i + frow, (wn * TN + 32 * i + frow) * cw_ld + cw_mis);
#pragma unroll
      for (int j = 0; j < FM; ++j) v.ca[j] = codes(BN + wm * TM + 32 * j + frow, (wm * TM + 32 * j + frow) * ca_ld + ca_mis);
    }
  };

  // Fragment of LDS rows row .. row + 31 at 64-K step t: logical chunks 4 t + h and 4 t + 2 + h.
  const int fsw = (frow >> 1) & 7;
  const int off_t[2][2] = {{frow * kStageK + ((h ^ fsw) << 4), frow * kStageK + (((2 + h) ^ fsw) << 4)},
                           {frow * kStageK + (((4 + h) ^ fsw) << 4), frow * kStageK + (((6 + h) ^ fsw) << 4)}};
  auto frag = [&](const uint8_t* buf, int row, int t) -> v8i {
    const v4i lo = *reinterpret_cast<const v4i*>(buf + row * kStageK + off_t[t][0]);
    const v4i hi = *reinterpret_cast<const v4i*>(buf + row * kStageK + off_t[t][1]);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  const v16f zero = {};
  v16f acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = zero;

  auto compute = [&](const uint8_t* buf, const Scales& v) {
    v8i wf[2][FN], af[2][FM];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < FN; ++i) wf[t][i] = frag(buf, wn * TN + 32 * i, t);
#pragma unroll
      for (int j = 0; j < FM; ++j) af[t][j] = frag(buf, BN + wm * TM + 32 * j, t);
    }
    if constexpr (MODE == kMidBlock) {
      float sa[FM], sb[FN];
#pragma unroll
      for (int j = 0; j < FM; ++j) sa[j] = bits_to_f32(v.sa[j], g.sa_dtype);
#pragma unroll
      for (int i = 0; i < FN; ++i) sb[i] = bits_to_f32(v.sb[i], g.sb_dtype);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          v16f part = mid_mma<MODE, 0>(wf[0][i], af[0][j], zero, 0, 0);
          part = mid_mma<MODE, 0>(wf[1][i], af[1][j], part, 0, 0);
          const float c = sa[j] * sb[i];
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(part[r], c, acc[i][j][r]);
        }
    } else {
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mid_mma<MODE, 0>(wf[0][i], af[0][j], acc[i][j], v.cw[i], v.ca[j]);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mid_mma<MODE, 2>(wf[1][i], af[1][j], acc[i][j], v.cw[i], v.ca[j]);
    }
  };

  Scales cur_s{}, next_s{};
  load_scales(0, cur_s);
  issue_codes(0);
  issue(0, B0);
  wait_vmcnt<0>();
  lds_barrier();
  // Stage s is visible in `cur` and nothing is in flight; stage s + 1 lands in `nxt`
  // (read by nobody since the last barrier) while stage s is multiplied. The code reads
  // come first: behind a direct load into the same LDS object they would wait for it.
  auto step = [&](int s, uint8_t* cur, uint8_t* nxt) {
    read_codes(s, cur_s);
    if (s + 1 < ns) {
      issue(s + 1, nxt);
      issue_codes(s + 1);
      load_scales(s + 1, next_s);
    }
    compute(cur, cur_s);
    wait_vmcnt<0>();
    lds_barrier();
    if constexpr (MODE == kMidBlock) cur_s = next_s;
  };
  for (int s = 0; s < ns; s += 2) {
    step(s, B0, B1);
    if (s + 1 < ns) step(s + 1, B1, B0);  // workgroup-uniform
  }

  // Epilogue: scales, bias, one rounding.
  const int64_t n_w = n_base + wn * TN, m_w = m_base + wm * TM;
  auto value = [&](int i, int j, int grp, float (&v)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = wn * TN + 32 * i + 8 * grp + 4 * h + q;
      float y = acc[i][j][4 * grp + q];
      if constexpr (MODE == kMidInt8) y = (float)__builtin_bit_cast(int, y);
      if constexpr (MODE == kMidScaled || MODE == kMidInt8) y = y * row_sa[j] * col_scale[c];
      asm volatile("" : "+v"(y));  // keep the fp32 product, sum and output conversion three roundings
      v[q] = y + col_bias[c];
      asm volatile("" : "+v"(v[q]));
    }
  };
  if (kps > 0 || g.out_dtype == AYK_F32) {
    float* base = kps > 0 ? g.ws + (int64_t)blockIdx.y * g.M * g.N : static_cast<float*>(g.out);
    const int64_t ldo = kps > 0 ? g.N : g.ldo;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int64_t m = m_w + 32 * j + frow;
      if (m >= g.M) continue;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
          const int64_t n = n_w + 32 * i + 8 * grp + 4 * h;
          float v[4];
          value(i, j, grp, v);
          store4_f32(base + m * ldo + n, g.N - n, v);
        }
    }
    return;
  }
  constexpr int kRegion = 32 * TN * 2, kPerBuf = kStage / kRegion;
  static_assert(2 * kPerBuf >= kWaves, "the staging regions fit the stage buffers");
  uint8_t* region = wave < kPerBuf ? B0 + wave * kRegion : B1 + (wave - kPerBuf) * kRegion;
  const bool bf16 = g.out_dtype == AYK_BF16;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int grp = 0; grp < 4; ++grp) {
        float v[4];
        value(i, j, grp, v);
        const int byte = 2 * (32 * i + 8 * grp + 4 * h);
        if (bf16) stage_slab16<true, TN>(region, frow, byte, v);
        else stage_slab16<false, TN>(region, frow, byte, v);
      }
    store_slab16<TN>(region, static_cast<uint16_t*>(g.out), g.ldo, g.M, g.N, m_w + 32 * j, n_w, lane);
  }
}

// Fixed-order sum of the K-split partials, bias, one rounding, for N or alignments the
// four-element reduce does not take.
__global__ __launch_bounds__(256) void mid_reduce(const float* __restrict__ part, int64_t M, int64_t N, int split,
                                                  const void* __restrict__ bias, int bias_dtype, void* __restrict__ out,
                                                  int out_dtype, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * N) return;
  const int64_t m = i / N, n = i - m * N;
  float v = 0.0f;
  for (int s = 0; s < split; ++s) v += part[(int64_t)s * M * N + i];
  if (bias) v += load_f32(bias, bias_dtype, n);
  store_f32(out, out_dtype, m * ldo + n, v);
}

// Tile and K split: the pair with the smallest modelled time. The model, in microseconds,
// was fitted per recipe on 13 weight shapes from 3072 x 1024 to 37888 x 3584 and 12 batches
// from 64 to 2048 (weights cold): a CU that runs u workgroups of a tile takes
// max(u tau, ceil(u / resident) lambda) per 128-K stage (throughput, or one round's
// latency) and `store` per 256 x 256 outputs; a split adds a reduce launch and the fp32
// partials' traffic. Its choice is 2-3% slower than the fastest tile and split on average.
struct MidPlan {
  int config, split;
  float us;
};
struct MidTile {
  int bn, bm, resident;
};
constexpr MidTile kTiles[3] = {{256, 256, 1}, {128, 128, 2}, {128, 64, 3}};
struct MidModel {
  float tau[3], lambda[3];
  float store, base, reduce, partial;
};
// Block scales have no 256 x 256 form (its partial sums do not fit the registers).
constexpr MidModel kModels[3] = {{{1.54f, 0.55f, 0.43f}, {1.54f, 0.97f, 0.77f}, 7.6f, 0.2f, 6.5f, 1.67e-6f},
                                 {{0.0f, 0.67f, 0.48f}, {0.0f, 1.19f, 0.91f}, 7.8f, 1.7f, 4.8f, 1.68e-6f},
                                 {{1.71f, 0.61f, 0.53f}, {1.71f, 1.03f, 0.91f}, 5.7f, 0.0f, 6.5f, 1.8e-6f}};
constexpr int kSplits[8] = {1, 2, 3, 4, 6, 8, 12, 16};
constexpr int kMinSplitK = 512;
constexpr int kCus = 256;

// K of one piece: whole stages; MXFP8: whole 512-K code chunks.
int64_t mid_kps(MidMode mode, int64_t K, int split) {
  const int64_t unit = mode == kMidMx ? 4 * kStageK : kStageK;
  return cdiv(cdiv(K, unit), split) * unit;
}

MidPlan mid_plan(MidMode mode, int64_t M, int64_t N, int64_t K, bool may_split) {
  const MidModel& m = kModels[mode == kMidInt8 ? kMidScaled : mode];
  MidPlan best{2, 1, 0.0f};
  bool first = true;
  for (int c = mode == kMidBlock ? 1 : 0; c < 3; ++c) {
    const MidTile& t = kTiles[c];
    const int64_t tiles = cdiv(M, t.bm) * cdiv(N, t.bn);
    for (const int s : kSplits) {
      // INT8 never splits: a partial would leave the exact int32 sum.
      if (s > 1 && (!may_split || mode == kMidInt8 || K < (int64_t)kMinSplitK * s)) break;
      const float u = (float)cdiv(tiles * s, kCus), rounds = (float)cdiv(cdiv(tiles * s, kCus), t.resident);
      const float stage = rounds * m.lambda[c] > u * m.tau[c] ? rounds * m.lambda[c] : u * m.tau[c];
      float us = m.base + (float)cdiv(cdiv(K, kStageK), s) * stage + m.store * u * (float)(t.bn * t.bm) / 65536.0f;
      if (s > 1) us += m.reduce + m.partial * (float)s * (float)M * (float)N;
      if (first || us < best.us) {
        first = false;
        best = {c, s, us};
      }
    }
  }
  best.split = (int)cdiv(K, mid_kps(mode, K, best.split));  // rounded-up pieces may need fewer of them
  return best;
}
size_t split_bytes(const MidPlan& p, int64_t M, int64_t N) {
  return p.split > 1 ? (size_t)p.split * (size_t)M * (size_t)N * sizeof(float) : 0;
}

template <int MODE>
void launch_tile(const MidArgs& g, const MidPlan& p, int64_t kps, hipStream_t st) {
  const MidTile& t = kTiles[p.config];
  const int tiles_m = (int)cdiv(g.M, t.bm);
  const dim3 grid((unsigned)(tiles_m * cdiv(g.N, t.bn)), (unsigned)p.split);
  if constexpr (MODE != kMidBlock) {
    if (p.config == 0) {
      hipLaunchKernelGGL((fp8_mid_kernel<MODE, 256, 256, 2, 4, 1>), grid, dim3(512), 0, st, g, tiles_m, kps);
      return;
    }
  }
  if (p.config == 1) hipLaunchKernelGGL((fp8_mid_kernel<MODE, 128, 128, 2, 2, 2>), grid, dim3(256), 0, st, g, tiles_m, kps);
  else hipLaunchKernelGGL((fp8_mid_kernel<MODE, 128, 64, 2, 2, 2>), grid, dim3(256), 0, st, g, tiles_m, kps);
}

}  // namespace

size_t mid_workspace(MidMode mode, int64_t M, int64_t N, int64_t K) {
  return split_bytes(mid_plan(mode, M, N, K, true), M, N);
}
// The weights stream at no more than 4.4 TB/s beside a launch and its prologue (only the
// smallest batches are near that; the plan itself does not depend on it).
float mid_time(MidMode mode, int64_t M, int64_t N, int64_t K) {
  const float us = mid_plan(mode, M, N, K, true).us, stream = 6.0f + (float)N * (float)K / 4.4e6f;
  return us > stream ? us : stream;
}

bool mid_supported(const MidArgs& g) {
  return g.K < ((int64_t)1 << 30) && 256 * g.lda < ((int64_t)1 << 31) && 256 * g.ldw < ((int64_t)1 << 31) &&
         256 * g.ld_sa < ((int64_t)1 << 31) && 256 * g.ld_sb < ((int64_t)1 << 31) &&
         cdiv(g.M, 64) * cdiv(g.N, 128) < ((int64_t)1 << 31);
}

int mid_launch(MidMode mode, const MidArgs& g, hipStream_t st, const char* op) {
  MidPlan p = mid_plan(mode, g.M, g.N, g.K, true);
  // A caller that brings no workspace gets the best plan without a split.
  if (p.split > 1 && (g.ws == nullptr || g.ws_bytes < split_bytes(p, g.M, g.N))) p = mid_plan(mode, g.M, g.N, g.K, false);
  const int64_t kps = p.split > 1 ? mid_kps(mode, g.K, p.split) : 0;
  note_plan("mid %dx%d split=%d", kTiles[p.config].bn, kTiles[p.config].bm, p.split);
  switch (mode) {
    case kMidScaled: launch_tile<kMidScaled>(g, p, kps, st); break;
    case kMidBlock: launch_tile<kMidBlock>(g, p, kps, st); break;
    case kMidInt8: launch_tile<kMidInt8>(g, p, kps, st); break;
    default:
      // 16-byte code loads need whole 512-K chunks and 16-byte aligned code rows, 4-byte ones
      // whole stages and 4-byte aligned rows.
      if (g.K % (4 * kStageK) == 0 && g.ld_sa % 16 == 0 && g.ld_sb % 16 == 0 && aligned16(g.sa) && aligned16(g.sb)) {
        launch_tile<kMidMx>(g, p, kps, st);
      } else if (g.K % kStageK == 0 && g.ld_sa % 4 == 0 && g.ld_sb % 4 == 0 &&
                 ((reinterpret_cast<uintptr_t>(g.sa) | reinterpret_cast<uintptr_t>(g.sb)) & 3) == 0) {
        launch_tile<kMidMx4>(g, p, kps, st);
      } else {
        launch_tile<kMidMxAny>(g, p, kps, st);
      }
  }
  if (int rc = check_launch(op)) return rc;
  if (p.split == 1) return AYK_OK;
  launch_split_reduce(mid_reduce, g.ws, g.M, g.N, p.split, g.bias, g.bias_dtype, g.out, g.out_dtype, g.ldo, st);
  return check_launch(op);
}

}  // namespace ayk
