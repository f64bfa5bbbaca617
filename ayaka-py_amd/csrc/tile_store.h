// Output stores shared by the tiled GEMM kernels: a wavefront's 32 (m) x TN (n) slab of
// 32 x 32 MFMA tiles D[n][m], where lane (frow = lane % 32, h = lane / 32) holds column
// m = frow and rows n = 8 g + 4 h + q (register 4 g + q) of each tile.
#pragma once

#include "ayk_common.h"
#include "gemm_util.h"

namespace ayk {
namespace {

typedef int slab_chunk __attribute__((ext_vector_type(4)));

// Four consecutive 16-bit outputs of row m = frow at column byte `byte` (of TN * 2) into
// the wavefront's staging region; 16-byte chunks are XOR-swizzled by row, so the 32 rows
// of a write fall on distinct banks.
template <bool BF16, int TN>
__device__ inline void stage_slab16(uint8_t* region, int frow, int byte, const float (&v)[4]) {
  constexpr int kRowB = TN * 2, kChunks = kRowB / 16;
  uint8_t* dst = region + frow * kRowB + (((byte >> 4) ^ (frow & (kChunks - 1))) << 4) + (byte & 15);
  if constexpr (BF16) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  } else {
    *reinterpret_cast<uint2*>(dst) = make_uint2((uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16),
                                                (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16));
  }
}

// The staged slab to rows [m0, m0 + 32) x columns [n0, n0 + TN) of out (clipped to M, N),
// row by row in 16-byte pieces where the address allows, in 8-byte ones where only that does
// (N % 8 == 4: every other row, whose elements stored one by one cost MXFP8 2048 x 29692 x 288
// 104 us against 82, 2048 x 7492 x 128 23 against 16). The region belongs to the wavefront: no
// barrier, only its own LDS counter.
template <int TN>
__device__ inline void store_slab16(const uint8_t* region, uint16_t* out, int64_t ldo, int64_t M, int64_t N, int64_t m0,
                                    int64_t n0, int lane) {
  constexpr int kRowB = TN * 2, kChunks = kRowB / 16, kRowsPerStore = 64 / kChunks;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wavefront's own staging writes
#pragma unroll
  for (int r0 = 0; r0 < 32; r0 += kRowsPerStore) {
    const int rr = r0 + lane / kChunks, cc = lane % kChunks;
    const int64_t gm = m0 + rr, gn = n0 + 8 * cc;
    const slab_chunk val = *reinterpret_cast<const slab_chunk*>(region + rr * kRowB + ((cc ^ (rr & (kChunks - 1))) << 4));
    if (gm < M && gn < N) {
      uint16_t* p = out + gm * ldo + gn;
      if (gn + 8 <= N && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
        __builtin_nontemporal_store(val, reinterpret_cast<slab_chunk*>(p));
      } else {
#pragma unroll
        for (int q = 0; q < 8; q += 4) {
          if (gn + q + 4 <= N && (reinterpret_cast<uintptr_t>(p + q) & 7) == 0) {
            *reinterpret_cast<uint2*>(p + q) = make_uint2((uint32_t)val[q / 2], (uint32_t)val[q / 2 + 1]);
          } else {
#pragma unroll
            for (int c = q; c < q + 4; ++c)
              if (gn + c < N) p[c] = (uint16_t)((uint32_t)val[c / 2] >> (16 * (c % 2)));
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read back before the next slab overwrites it
}

// The same for fp32 slabs (a region of 32 * TN * 4 bytes): four consecutive outputs of row m =
// frow from column `col` on, then row by row in 16-byte pieces. A lane's own four outputs lie
// 32 rows apart from its neighbours': stored from the registers, an instruction writes 32 pieces
// of 32 bytes, which holds large outputs of a short K to half the memory's rate (MXFP8, from the
// registers and through LDS: 2742 x 32768 x 640 413 -> 156 us, 2039 x 16384 x 1280 145 -> 73). A
// 16-byte store to global memory needs 4-byte alignment only.
typedef float slab_f32 __attribute__((ext_vector_type(4)));
typedef slab_f32 slab_f32_any __attribute__((aligned(4)));

template <int TN>
__device__ inline void stage_slab32(uint8_t* region, int frow, int col, const float (&v)[4]) {
  constexpr int kChunks = TN / 4;
  *reinterpret_cast<float4*>(region + frow * TN * 4 + (((col >> 2) ^ (frow & (kChunks - 1))) << 4)) = make_float4(v[0], v[1], v[2], v[3]);
}

template <int TN>
__device__ inline void store_slab32(const uint8_t* region, float* out, int64_t ldo, int64_t M, int64_t N, int64_t m0,
                                    int64_t n0, int lane) {
  constexpr int kChunks = TN / 4, kRowsPerStore = 64 / kChunks;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wavefront's own staging writes
#pragma unroll
  for (int r0 = 0; r0 < 32; r0 += kRowsPerStore) {
    const int rr = r0 + lane / kChunks, cc = lane % kChunks;
    const int64_t gm = m0 + rr, gn = n0 + 4 * cc;
    const slab_f32 val = *reinterpret_cast<const slab_f32*>(region + rr * TN * 4 + ((cc ^ (rr & (kChunks - 1))) << 4));
    if (gm < M && gn < N) {
      float* p = out + gm * ldo + gn;
      if (gn + 4 <= N) {
        __builtin_nontemporal_store(val, reinterpret_cast<slab_f32_any*>(p));
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (gn + c < N) p[c] = val[c];
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read back before the next slab overwrites it
}

// Four consecutive fp32 values of one row (`left` columns remain in it).
__device__ inline void store4_f32(float* p, int64_t left, const float (&v)[4]) {
  if (left >= 4 && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < left) p[q] = v[q];
  }
}

}  // namespace
}  // namespace ayk
