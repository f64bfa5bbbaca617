// W8A8 GEMM on medium tiles: the launcher that gemm.hip's dispatch calls for batches and
// shapes that the 256 x 256 pair kernels do not take or do not fill the chip with.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

namespace ayk {

enum MidMode { kMidScaled = 0, kMidBlock = 1, kMidMx = 2, kMidInt8 = 3 };

struct MidArgs {
  const uint8_t* a;  // [M, K], row stride lda
  int64_t lda;
  const uint8_t* w;  // [N, K], row stride ldw
  int64_t ldw;
  int64_t M, N, K;
  const void* sa;    // scaled / int8: scalar or [M]; block: [M, ld_sa] or [K / 128, M]; MX: u8 [M, ld_sa]
  int sa_dtype, sa_vec;  // sa_vec: per row; block: column-major
  int64_t ld_sa;
  const void* sb;    // scaled / int8: scalar or [N]; block: [N / 128, ld_sb]; MX: u8 [N, ld_sb]
  int sb_dtype, sb_vec;
  int64_t ld_sb;
  const void* bias;
  int bias_dtype;
  void* out;
  int out_dtype;
  int64_t ldo;
  float* ws;         // K-split partials [split, M, N] fp32
  size_t ws_bytes;
};

// Tile and K split of a shape with their modelled time in microseconds, and the workspace
// bytes of the launch (0: no K split); functions of the mode and shape only.
struct MidPlan {
  int config, split;
  float us;
};
MidPlan mid_plan(MidMode mode, int64_t M, int64_t N, int64_t K, bool may_split = true);
float mid_time(const MidPlan& p, int64_t N, int64_t K);
size_t mid_workspace(MidMode mode, int64_t M, int64_t N, int64_t K);
// 32-bit offsets within a tile's rows.
bool mid_supported(MidMode mode, const MidArgs& g);
// `p`: mid_plan of the shape.
int mid_launch(MidMode mode, const MidArgs& g, MidPlan p, hipStream_t st, const char* op);

}  // namespace ayk
