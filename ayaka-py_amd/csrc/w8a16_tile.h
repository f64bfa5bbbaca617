// W8A16 GEMM of any M on gfx950: out[M, N] = x[M, K] . dequant(w[N, K])^T with e4m3
// weights, 16-bit activations and fp32 accumulation, LDS-tiled on
// v_mfma_f32_32x32x16_{bf16,f16}. The launcher that w8a16.hip's dispatch calls.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

namespace ayk {

struct W16TileArgs {
  const uint16_t* x;  // [M, K], row stride ldx (elements)
  int64_t ldx;
  const uint8_t* w;   // [N, K] e4m3, row stride ldw
  int64_t ldw;
  int64_t M, N, K;
  const void* scale;  // scale[(n / by) * srs + k / bx]
  int scale_dtype;
  int64_t srs, by, bx;
  void* out;          // [M, N] of the activation dtype, row stride ldo
  int64_t ldo;
  float* part;        // K-split partials [split, M, N] fp32
  size_t part_bytes;
};

// Tile and K split of a shape with their modelled time in microseconds, and the workspace
// bytes of the launch below (0: no K split); functions of the shape only.
struct W16TilePlan {
  int config, split;
  float us;
};
W16TilePlan w16_tile_plan(int64_t M, int64_t N, int64_t K, bool may_split = true);
float w16_tile_time(const W16TilePlan& p, int64_t N, int64_t K);
size_t w16_tile_workspace(int64_t M, int64_t N, int64_t K);
// Whether the tiled kernel takes this problem.
bool w16_tile_supported(const W16TileArgs& a);
// `p`: w16_tile_plan of the shape.
int w16_tile_launch(const W16TileArgs& a, W16TilePlan p, bool bf16, hipStream_t st, const char* op);

}  // namespace ayk
