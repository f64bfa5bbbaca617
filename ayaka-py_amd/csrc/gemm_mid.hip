// W8A8 GEMM on medium tiles, gfx950: out[M, N] = epilogue(a[M, K] . w[N, K]^T) for the
// batches between the decode kernels and the 256 x 256 pair kernels, for shapes whose
// 256 x 256 tiles leave CUs idle, and for every K, N, scale type and alignment that the
// pair kernels refuse. Recipes as in gemm.hip: per-row / per-tensor scales, 128 x 128
// block scales, MXFP8 codes, INT8.
//
// Bound: at these sizes the weight stream and its latency (M = 65 .. 255), then the matrix
// cores. Design:
//  * 256 x 256 (eight wavefronts), 128 x 128, 128 x 64 and 64 x 64 (four) tiles on
//    v_mfma_scale_f32_32x32x64_f8f6f4, weight = operand A: a lane's accumulator column is
//    one activation row.
//  * Direct-to-LDS loads (8 rows x 128 bytes an instruction) into a ring of two or four
//    128-K stage buffers. Two buffers leave room for several workgroups a CU, which run
//    while one waits at its stage barrier (throughput, the larger batches); four hide the
//    latency of a stage inside one workgroup (few tiles a CU, long K), which also saves
//    most K splits.
//  * A K tail is zero-filled by the loads' bounds check, so any K % 16 == 0 takes the same
//    loop; rows past M and N likewise.
//  * Block scales: a 128-K stage is one scale block; its two MFMAs start from zero and one
//    fma an accumulator folds them with sa[m, kb] sb[n / 128, kb].
//  * Scales and MXFP8 codes pass through LDS as well, a dword a row and stage (16-byte
//    aligned codes: 16 bytes for four stages; unaligned ones: the two dwords).
//  * Tile, ring and K split come from a fitted time model (mid_plan), which gemm.hip also
//    holds against the other kernels' (mid_time).
// Measured (kernel alone in a graph; the kernels these shapes ran at first -> two buffers
// only -> now): per-row 4096 x 14336 M = 128 60.8 -> 31.7 -> 25.5 us, 4096 x 4096 M = 128
// 33 -> 18.4 -> 10.9, M = 512 28 -> 25 -> 15.3, M = 1024 41.3 -> 25.9 -> 24.5; MXFP8 4096 x
// 14336 M = 128 47.0 -> 33.6 -> 27.4; block-128 4096 x 4096 M = 256 23.6 -> 17.1.
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
// Kernel modes of MXFP8 by its codes: kMidMx K % 512 == 0 and 16-byte aligned rows, kMidMx4
// K % 128 == 0 and 4-byte aligned rows, kMidMxAny the rest.
constexpr int kMidMx4 = 4, kMidMxAny = 5;
constexpr bool mx_mode(int mode) { return mode == kMidMx || mode == kMidMx4 || mode == kMidMxAny; }
// Dwords of LDS for a row's scales of one stage: the dword that holds its block scale or its
// four codes (unaligned code rows: the two dwords that do; kMidMx loads four stages at once).
constexpr int scale_words(int mode) { return mode == kMidBlock || mode == kMidMx4 ? 1 : (mode == kMidMxAny ? 2 : 0); }

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
// an fp32 partial without the bias. D stage buffers: D - 1 stages are in flight. F32:
// large fp32 outputs, whose rows pass through LDS (no K split).
template <int MODE, bool F32, int BN, int BM, int WN, int WM, int D, int WGS>
__global__ __launch_bounds__(WN * WM * 64, WGS) void fp8_mid_kernel(MidArgs g, int tiles_m, int64_t kps) {
  constexpr int kThreads = WN * WM * 64, kWaves = WN * WM;
  constexpr int TN = BN / WN, TM = BM / WM, FN = TN / 32, FM = TM / 32;
  constexpr int kRows = BN + BM, kStage = kRows * kStageK;
  constexpr int kWDma = BN / 8 / kWaves, kADma = BM / 8 / kWaves;  // direct loads per wavefront and stage
  static_assert(BN % (16 * kWaves) == 0 && BM % (16 * kWaves) == 0, "whole pairs of loads per wavefront");
  constexpr int kWords = scale_words(MODE), kWordRows = 64 * kWaves;  // each wavefront loads 64 rows' words
  constexpr int kOps = kWDma + kADma + kWords, kBuf = kStage + kWordRows * 4 * kWords;
  static_assert(kRows <= kWordRows, "a lane a row");
  static_assert((D == 2 || D == 4) && (D - 2) * kOps <= 63, "whole rings in a chunk of four stages; vmcnt range");
  // Distinct LDS objects with compile-time names, so that the compiler keeps the loads in
  // flight to one apart from the reads of another.
  __shared__ __attribute__((aligned(1024))) uint8_t B0[kBuf], B1[kBuf], B2[D == 4 ? kBuf : 16], B3[D == 4 ? kBuf : 16];
  constexpr bool kChunks = MODE == kMidMx;
  __shared__ __attribute__((aligned(1024))) uint8_t chunk[kChunks ? kWordRows * 16 : 16];
  __shared__ float col_scale[BN], col_bias[BN];
  auto buffer = [&](auto d) -> uint8_t* {
    constexpr int i = decltype(d)::value;
    if constexpr (i == 0) return B0;
    else if constexpr (i == 1) return B1;
    else if constexpr (i == 2) return B2;
    else return B3;
  };

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

  // Per-stage scales: block sa[m, kb] and sb[n / 128, kb], MX four codes a row. Every row's
  // dword goes through LDS, loaded by one lane behind the operands of its stage: straight
  // into each wavefront's registers they asked for more cache lines than the operands, and
  // any branch or register load among the direct loads costs the compiler its exact wait
  // counts. `word`: byte offset of this lane's row's first scale from the 4-byte aligned start
  // of its side's window, which ends with the last row's last scale (rounded up to a dword,
  // which lies in its page); `step`: bytes from one stage's scale to the next.
  const int64_t kblocks = cdiv(g.K, kStageK), kb0 = k0 / kStageK;
  const int sa_size = MODE == kMidBlock ? dtype_size(g.sa_dtype) : 1, sb_size = MODE == kMidBlock ? dtype_size(g.sb_dtype) : 1;
  const bool sa_cols = MODE == kMidBlock && g.sa_vec;
  const int64_t unit = MODE == kMidBlock ? kblocks : cdiv(g.K, 32);  // scales of a row
  const int64_t u0 = MODE == kMidBlock ? kb0 : k0 / 32;              // the first of this piece
  const int64_t sa_ld = sa_cols ? 1 : (g.ld_sa > 0 ? g.ld_sa : unit), sb_ld = g.ld_sb > 0 ? g.ld_sb : unit;
  const int64_t n_row0 = MODE == kMidBlock ? n_base / 128 : n_base;
  const uintptr_t sap = reinterpret_cast<uintptr_t>(g.sa) + (uintptr_t)((sa_cols ? u0 * g.M + m_base : m_base * sa_ld + u0) * sa_size);
  const uintptr_t sbp = reinterpret_cast<uintptr_t>(g.sb) + (uintptr_t)((n_row0 * sb_ld + u0) * sb_size);
  const uint32_t sa_mis = (uint32_t)__builtin_amdgcn_readfirstlane((int)(sap & 3)), sb_mis = (uint32_t)__builtin_amdgcn_readfirstlane((int)(sbp & 3));
  const uint32_t sa_step = (uint32_t)__builtin_amdgcn_readfirstlane((int)(MODE == kMidBlock ? (sa_cols ? g.M : 1) * sa_size : 4));
  const uint32_t sb_step = MODE == kMidBlock ? (uint32_t)sb_size : 4u;
  const uint32_t sa_row = (uint32_t)__builtin_amdgcn_readfirstlane((int)(sa_ld * sa_size));
  const uint32_t sb_row = (uint32_t)__builtin_amdgcn_readfirstlane((int)(sb_ld * sb_size));
  auto sa_byte = [&](int r) -> uint32_t { return sa_mis + (uint32_t)r * sa_row; };
  auto sb_byte = [&](int r) -> uint32_t {
    return sb_mis + (uint32_t)(MODE == kMidBlock ? ((int)(n_base & 127) + r) / 128 : r) * sb_row;
  };
  auto window = [&](int64_t rows_left, int64_t ld, int64_t size, uint32_t mis) {  // the tile's first row lies inside
    const int64_t bytes = (((rows_left - 1) * ld + unit - u0) * size + mis + 3) & ~(int64_t)3;
    return (int32_t)(bytes < 0x7FFFFFFC ? bytes : 0x7FFFFFFC);
  };
  const bool w_side = 64 * wave < BN;
  const int64_t sa_rows = sa_cols ? (unit - u0 - 1) * g.M + g.M - m_base : g.M - m_base;  // column-major: as one long row set
  const int32_t sa_records = sa_cols ? (int32_t)((((sa_rows * sa_size) + sa_mis + 3) & ~(int64_t)3)) : window(sa_rows, sa_ld, sa_size, sa_mis);
  const int32_t sb_records = window((MODE == kMidBlock ? cdiv(g.N, 128) : g.N) - n_row0, sb_ld, sb_size, sb_mis);
  const __amdgpu_buffer_rsrc_t word_rsrc = uniform_rsrc(reinterpret_cast<const void*>(w_side ? sbp - sb_mis : sap - sa_mis),
                                                        kWords || kChunks ? (w_side ? sb_records : sa_records) : 0);
  const int word_row = 64 * wave + lane;
  const uint32_t word = word_row >= kRows ? (uint32_t)kPast : (w_side ? sb_byte(word_row) : sa_byte(word_row - BN));
  const uint32_t word_step = w_side ? sb_step : sa_step;
  auto issue_words = [&](int s, uint8_t* dst) {
    if constexpr (kWords > 0) {
      const int voff = (int)((word + (uint32_t)s * word_step) & ~3u);
      uint8_t* words = dst + kStage + 256 * wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(word_rsrc, (__attribute__((address_space(3))) void*)words, 4, voff, 0, 0, 0);
      if constexpr (kWords == 2) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(word_rsrc, (__attribute__((address_space(3))) void*)(words + 4 * kWordRows), 4,
                                                 voff + 4, 0, 0, 0);
      }
    }
  };
  // The codes of stages 4 q .. 4 q + 3.
  auto issue_chunk = [&](int q) {
    if constexpr (kChunks) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(word_rsrc, (__attribute__((address_space(3))) void*)(chunk + 1024 * wave), 16,
                                               (int)word, 16 * q, 0, 0);
    }
  };
  v4i chunk_w[FN], chunk_a[FM];
  auto read_chunk = [&]() {
    if constexpr (kChunks) {
#pragma unroll
      for (int i = 0; i < FN; ++i) chunk_w[i] = *reinterpret_cast<const v4i*>(chunk + 16 * (wn * TN + 32 * i + frow));
#pragma unroll
      for (int j = 0; j < FM; ++j) chunk_a[j] = *reinterpret_cast<const v4i*>(chunk + 16 * (BN + wm * TM + 32 * j + frow));
    }
  };
  struct Scales {
    int cw[FN], ca[FM];    // MX: the codes of this lane half's 32-K blocks, byte 2 t for step t
    float sb[FN], sa[FM];  // block
  };
  auto read_scales = [&](int s, const uint8_t* buf, Scales& v) {
    if constexpr (kWords > 0) {  // (kMidMx: from the chunk)
      const uint32_t* words = reinterpret_cast<const uint32_t*>(buf + kStage);
      if constexpr (MODE == kMidBlock) {
        // (a 32-row slab lies in one 128-row block of the weight)
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const int r = wn * TN + 32 * i;
          v.sb[i] = bits_to_f32({words[r], ((sb_byte(r) + (uint32_t)s * sb_step) & 3) * 8}, g.sb_dtype);
        }
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          const int r = wm * TM + 32 * j + frow;
          v.sa[j] = bits_to_f32({words[BN + r], ((sa_byte(r) + (uint32_t)s * sa_step) & 3) * 8}, g.sa_dtype);
        }
      } else {
        // Codes past K are 1.0: their operands are zeros, which a NaN code would turn into NaN.
        const int valid = (klen - s * kStageK + 31) / 32;
        const uint32_t past = MODE == kMidMxAny && valid < 4 ? 0xFFFFFFFFu << (8 * valid) : 0u;
        auto codes = [&](int row, uint32_t byte) -> int {
          uint32_t w = words[row];
          if constexpr (MODE == kMidMxAny) {
            w = __builtin_amdgcn_alignbyte(words[kWordRows + row], w, byte & 3);
            w = (w & ~past) | (0x7F7F7F7Fu & past);
          }
          return (int)(w >> (8 * h));
        };
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const int r = wn * TN + 32 * i + frow;
          v.cw[i] = codes(r, sb_byte(r));
        }
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          const int r = wm * TM + 32 * j + frow;
          v.ca[j] = codes(BN + r, sa_byte(r));
        }
      }
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
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          v16f part = mid_mma<MODE, 0>(wf[0][i], af[0][j], zero, 0, 0);
          part = mid_mma<MODE, 0>(wf[1][i], af[1][j], part, 0, 0);
          const float c = v.sa[j] * v.sb[i];
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

  // The ring: stages 0 .. D - 2 in flight. Step s waits for stage s (the D - 2 younger ones
  // may still be in flight), passes a barrier (stage s is visible, and nobody reads stage
  // s - 1 any more), refills that buffer with stage s + D - 1 and multiplies stage s. Stages
  // past the last one load nothing that is used (operands: kPast), so the counts stay exact.
  // A round of U steps runs without a branch inside. kMidMx: the first step of a round reads
  // its four stages' codes, the second refills the chunk ahead of the data of a later stage.
  constexpr int U = kChunks ? 4 : D;
  auto prefetch = [&](int s, uint8_t* dst) {
    issue_words(s, dst);
    issue(s, dst);
  };
  issue_chunk(0);
  unrolled<D - 1>([&](auto d) { prefetch(decltype(d)::value, buffer(d)); });
  auto step = [&](int s, auto u) {
    constexpr int i = decltype(u)::value;
    const std::integral_constant<int, i % D> d;
    wait_vmcnt<(D - 2) * kOps>();
    lds_barrier();
    Scales v;
    read_scales(s, buffer(d), v);
    if constexpr (kChunks) {
      if constexpr (i == 0) read_chunk();
      if constexpr (i == 1) issue_chunk(s / 4 + 1);
#pragma unroll
      for (int t = 0; t < FN; ++t) v.cw[t] = (int)((uint32_t)chunk_w[t][i] >> (8 * h));
#pragma unroll
      for (int t = 0; t < FM; ++t) v.ca[t] = (int)((uint32_t)chunk_a[t][i] >> (8 * h));
    }
    prefetch(s + D - 1, buffer(std::integral_constant<int, (i + D - 1) % D>{}));
    // With one stage in flight its loads go first and the products stay in their step
    // (spread among each other they cost a 256 x 256 tile 13%); deeper rings gain from it.
    if constexpr (D == 2) __builtin_amdgcn_sched_barrier(0);
    compute(buffer(d), v);
    if constexpr (D == 2) __builtin_amdgcn_sched_barrier(0);
  };
  int s0 = 0;
  for (; s0 + U <= ns; s0 += U) {
    unrolled<U>([&](auto u) { step(s0 + decltype(u)::value, u); });
  }
  if constexpr (!kChunks) {  // (whole chunks only)
    unrolled<D - 1>([&](auto u) {
      if (s0 + decltype(u)::value < ns) step(s0 + decltype(u)::value, u);  // workgroup-uniform
    });
  }
  wait_vmcnt<0>();  // no direct load may still write LDS
  lds_barrier();    // no wavefront still reads a stage: the buffers become staging regions

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
  // Every wavefront stages 32 (m) x TN (n) slabs in a private region of the stage buffers.
  constexpr int kRegion = 32 * TN * (F32 ? 4 : 2), kPerBuf = kStage / kRegion;
  static_assert(2 * kPerBuf >= kWaves, "the staging regions fit the stage buffers");
  uint8_t* region = wave < kPerBuf ? B0 + wave * kRegion : B1 + (wave - kPerBuf) * kRegion;
  if constexpr (F32) {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
          float v[4];
          value(i, j, grp, v);
          stage_slab32<TN>(region, frow, 32 * i + 8 * grp + 4 * h, v);
        }
      store_slab32<TN>(region, static_cast<float*>(g.out), g.ldo, g.M, g.N, m_w + 32 * j, n_w, lane);
    }
    return;
  }
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

// Tile, stage buffers and K split: the triple with the smallest modelled time. The model, in
// microseconds, was fitted per recipe on 12 weight shapes from 3072 x 1024 to 37888 x 3584
// and 16 batches from 16 to 2048 (weights cold): a CU that runs u workgroups of a tile takes
// max(u tau, ceil(u / resident) lambda) per 128-K stage (throughput, or one round's
// latency) and `store` per 256 x 256 outputs; `cold` is the weights' share that no stage
// hides; a split adds a reduce launch and the fp32 partials' traffic. Its choice is 1-2%
// slower than the fastest triple on average (tau of the two-buffer tiles: from the launches of
// two rounds and more, above the fit, whose weight lies on the small ones). It runs for every
// workspace query and launch, so no division in its loops has a variable divisor (0.40 us a plan
// with them, 0.15 without).
struct MidTile {
  int bn, bm, resident;
};
constexpr int kConfigs = 6;
constexpr MidTile kTiles[kConfigs] = {{256, 256, 1}, {128, 128, 2}, {128, 64, 3}, {128, 128, 1}, {128, 64, 1}, {64, 64, 2}};
struct MidModel {
  float tau[kConfigs], lambda[kConfigs];  // 0: no such kernel
  float store, base, reduce, partial, cold;
};
constexpr MidModel kModels[3] = {
    {{1.25f, 0.44f, 0.32f, 0.50f, 0.27f, 0.19f}, {1.25f, 0.71f, 0.52f, 0.32f, 0.34f, 0.20f}, 9.0f, 2.9f, 3.4f, 1.68e-6f, 8.0e-8f},
    {{0.0f, 0.57f, 0.36f, 0.0f, 0.0f, 0.25f}, {0.0f, 0.99f, 0.74f, 0.0f, 0.0f, 0.33f}, 4.6f, 4.2f, 2.8f, 1.95e-6f, 7.0e-8f},
    {{1.71f, 0.55f, 0.37f, 0.33f, 0.37f, 0.22f}, {1.40f, 0.70f, 0.54f, 0.56f, 0.39f, 0.24f}, 3.8f, 2.8f, 3.5f, 1.92e-6f, 9.0e-8f}};
constexpr int kSplits[8] = {1, 2, 3, 4, 6, 8, 12, 16};
constexpr int kMinSplitK = 512;
constexpr int kCus = 256;

// K of one piece: whole stages; MXFP8: whole 512-K code chunks.
int64_t mid_kps(MidMode mode, int64_t K, int split) {
  const int64_t unit = mode == kMidMx ? 4 * kStageK : kStageK;
  return cdiv(cdiv(K, unit), split) * unit;
}

// Tiles of `side` rows (64, 128 or 256).
int64_t tile_count(int64_t rows, int side) { return side == 256 ? cdiv(rows, 256) : (side == 128 ? cdiv(rows, 128) : cdiv(rows, 64)); }
int64_t by_resident(int64_t n, int resident) { return resident == 1 ? n : (resident == 2 ? cdiv(n, 2) : cdiv(n, 3)); }

size_t split_bytes(const MidPlan& p, int64_t M, int64_t N) {
  return p.split > 1 ? (size_t)p.split * (size_t)M * (size_t)N * sizeof(float) : 0;
}

}  // namespace

MidPlan mid_plan(MidMode mode, int64_t M, int64_t N, int64_t K, bool may_split) {
  const MidModel& m = kModels[mode == kMidInt8 ? kMidScaled : mode];
  MidPlan best{5, 1, 0.0f};
  bool first = true;
  // INT8 never splits: a partial would leave the exact int32 sum.
  int splits = 1;
  while (may_split && mode != kMidInt8 && splits < 8 && K >= (int64_t)kMinSplitK * kSplits[splits]) ++splits;
  int64_t stages[8];
  for (int i = 0; i < splits; ++i) stages[i] = cdiv(cdiv(K, kStageK), kSplits[i]);
  for (int c = 0; c < kConfigs; ++c) {
    if (m.tau[c] == 0.0f) continue;
    const MidTile& t = kTiles[c];
    const int64_t tiles = tile_count(M, t.bm) * tile_count(N, t.bn);
    for (int i = 0; i < splits; ++i) {
      const int s = kSplits[i];
      const int64_t wgs = cdiv(tiles * s, kCus);  // a CU
      const float u = (float)wgs, rounds = (float)by_resident(wgs, t.resident);
      const float stage = rounds * m.lambda[c] > u * m.tau[c] ? rounds * m.lambda[c] : u * m.tau[c];
      float us = m.base + m.cold * (float)N * (float)K + (float)stages[i] * stage + m.store * u * (float)(t.bn * t.bm) / 65536.0f;
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

namespace {

template <int MODE, bool F32>
void launch_tile(const MidArgs& g, const MidPlan& p, int64_t kps, hipStream_t st) {
  const MidTile& t = kTiles[p.config];
  const int tiles_m = (int)cdiv(g.M, t.bm);
  const dim3 grid((unsigned)(tiles_m * cdiv(g.N, t.bn)), (unsigned)p.split);
#define AYK_MID(...) hipLaunchKernelGGL((fp8_mid_kernel<MODE, F32, __VA_ARGS__>), grid, dim3(threads), 0, st, g, tiles_m, kps)
  const unsigned threads = p.config == 0 ? 512 : 256;
  if constexpr (MODE == kMidBlock) {
    switch (p.config) {
      case 1: AYK_MID(128, 128, 2, 2, 2, 2); break;
      case 2: AYK_MID(128, 64, 2, 2, 2, 2); break;
      default: AYK_MID(64, 64, 2, 2, 4, 2); break;
    }
  } else {
    switch (p.config) {
      case 0: AYK_MID(256, 256, 2, 4, 2, 1); break;
      case 1: AYK_MID(128, 128, 2, 2, 2, 2); break;
      case 2: AYK_MID(128, 64, 2, 2, 2, 2); break;
      case 3: AYK_MID(128, 128, 2, 2, 4, 1); break;
      case 4: AYK_MID(128, 64, 2, 2, 4, 1); break;
      default: AYK_MID(64, 64, 2, 2, 4, 2); break;
    }
  }
#undef AYK_MID
}

// fp32 outputs of 4 MB and more pass through LDS up to K = 4096: below, the staging is a wait
// without a return (72 x 868 x 128: 4.8 -> 5.6 us), and past it the output is a small part of
// the launch.
template <int MODE>
void launch_mode(const MidArgs& g, const MidPlan& p, int64_t kps, hipStream_t st) {
  if (g.out_dtype == AYK_F32 && p.split == 1 && g.M * g.N >= (1 << 20) && g.K <= 4096) launch_tile<MODE, true>(g, p, kps, st);
  else launch_tile<MODE, false>(g, p, kps, st);
}

}  // namespace

size_t mid_workspace(MidMode mode, int64_t M, int64_t N, int64_t K) { return split_bytes(mid_plan(mode, M, N, K), M, N); }
// The weights stream at no more than 4.4 TB/s beside a launch and its prologue (only the
// smallest batches are near that; the plan itself does not depend on it).
float mid_time(const MidPlan& p, int64_t N, int64_t K) {
  const float stream = 6.0f + (float)N * (float)K / 4.4e6f;
  return p.us > stream ? p.us : stream;
}

bool mid_supported(MidMode mode, const MidArgs& g) {
  const int64_t lim = (int64_t)1 << 31;
  // 256 rows of the operands and of their scales (four bytes at most), and a column-major
  // scale table, within 32-bit offsets.
  return g.K < ((int64_t)1 << 30) && 256 * g.lda < lim && 256 * g.ldw < lim && 1024 * g.ld_sa < lim && 1024 * g.ld_sb < lim &&
         !(mode == kMidBlock && g.sa_vec && 4 * g.M * cdiv(g.K, 128) >= lim) && cdiv(g.M, 64) * cdiv(g.N, 64) < lim;
}

int mid_launch(MidMode mode, const MidArgs& g, MidPlan p, hipStream_t st, const char* op) {
  // A caller that brings no workspace gets the best plan without a split.
  if (p.split > 1 && (g.ws == nullptr || g.ws_bytes < split_bytes(p, g.M, g.N))) p = mid_plan(mode, g.M, g.N, g.K, false);
  const int64_t kps = p.split > 1 ? mid_kps(mode, g.K, p.split) : 0;
  note_plan("mid %dx%d%s split=%d", kTiles[p.config].bn, kTiles[p.config].bm, p.config >= 3 ? " ring" : "", p.split);
  const uintptr_t code_align = reinterpret_cast<uintptr_t>(g.sa) | reinterpret_cast<uintptr_t>(g.sb) | (uintptr_t)(g.ld_sa | g.ld_sb);
  switch (mode) {
    case kMidScaled: launch_mode<kMidScaled>(g, p, kps, st); break;
    case kMidBlock: launch_mode<kMidBlock>(g, p, kps, st); break;
    case kMidInt8: launch_mode<kMidInt8>(g, p, kps, st); break;
    default:
      if (g.K % (4 * kStageK) == 0 && (code_align & 15) == 0) {
        launch_mode<kMidMx>(g, p, kps, st);
      } else if (g.K % kStageK == 0 && (code_align & 3) == 0) {
        launch_mode<kMidMx4>(g, p, kps, st);
      } else {
        launch_mode<kMidMxAny>(g, p, kps, st);
      }
  }
  if (int rc = check_launch(op)) return rc;
  if (p.split == 1) return AYK_OK;
  launch_split_reduce(mid_reduce, g.ws, g.M, g.N, p.split, g.bias, g.bias_dtype, g.out, g.out_dtype, g.ldo, st);
  return check_launch(op);
}

}  // namespace ayk
