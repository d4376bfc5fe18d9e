// Shared pieces of the convolution GEMMs (conv.hip, conv_lds.hip): the brick
// geometry, the epilogues' reductions and store policy, and the fp32
// LDS-staged GEMM's arguments.
#pragma once

#include "ctmr_common.hpp"

namespace ctmr {

// Cache-policy operands of the GEMMs' output stores (gfx950 encoding: bit 1 =
// NT, non-temporal; bit 4 = SC1, device scope).  Same values under every
// policy; measured on MI355X, default / NT / SC1, A/B twice in one run: the
// brick GEMMs (fp32 and bf16 LDS-staged) and the streaming GEMM take SC1
// (config-0 fp32 + bf16 GEMMs 0.462 / 0.505 / 0.451 ms, UNet step 17.72 /
// 17.80 / 17.69 ms, config-1 block 26.18 / 26.17 / 26.14 ms, config 2a and
// the decoder window within 0.5 % either way); the persistent 1x1 GEMM takes
// NT (config 2c 0.165 / 0.160 / 0.171 ms).
constexpr int kStoreSC1 = 16;
constexpr int kStoreNT = 2;

// No term after the bias (the epilogues' default `after_bias`).
struct NoTerm {
  template <typename Acc>
  __device__ void operator()(Acc&) const {}
};

// Final step of the group-norm partials of a stored tile: red[wave][c] holds
// the fp64 (sum, sum of squares) of column c of each wave's 64 x (NSUB*16)
// block over its rows (published by a barrier); each group's columns and
// waves are added in ascending order -- a fixed order for a given shape.
template <int NSUB, int WM, int WN>
__device__ __forceinline__ void combine_gn_partials(const double (*red)[64][2], int col0, int cout, int cpg,
                                                    int groups, double* __restrict__ stats_tile) {
  constexpr int kWaveCols = NSUB * 16;
  const int groups_here = (WN * kWaveCols) / cpg;
  for (int gl = threadIdx.x; gl < groups_here; gl += 256) {
    const int g = col0 / cpg + gl;
    if (g >= groups || g * cpg >= cout) continue;
    double a = 0.0, q = 0.0;
    for (int wm = 0; wm < WM; ++wm)
      for (int cc = 0; cc < cpg; ++cc) {
        const int col = gl * cpg + cc;
        const int wv = (col / kWaveCols) * WM + wm;
        a += red[wv][col % kWaveCols][0];
        q += red[wv][col % kWaveCols][1];
      }
    stats_tile[(int64_t)g * 2] = a;
    stats_tile[(int64_t)g * 2 + 1] = q;
  }
}

// One DPP lane move of an fp64 value (two 32-bit halves; every source lane
// lies inside the lane's row of 16).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// Sum over the 16 lanes of a row, in the tree of an xor butterfly (partners
// 1, 2, 4, 8): quad_perm [1,0,3,2] and [2,3,0,1] are xor 1 and xor 2; after
// them lane 7 - i of a half row holds the value lane i ^ 4 holds (fp32/fp64
// addition commutes), so the half-row mirror is the xor-4 step and the row
// mirror the xor-8 step.  VALU moves instead of LDS permutes.
__device__ __forceinline__ double row16_sum(double v) {
  v += dpp_f64<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f64<0x141>(v);  // row_half_mirror
  v += dpp_f64<0x140>(v);  // row_mirror
  return v;
}

// Bricks of output voxels and their 3x3x3 halos.
constexpr int kBD = 4, kBH = 8, kBW = 8;
constexpr int kHD = kBD + 2, kHH = kBH + 2, kHW = kBW + 2;
constexpr int kHaloVox = kHD * kHH * kHW;                 // 600
constexpr int kStageIters = (kHaloVox * 4 + 255) / 256;  // 16-byte pieces per thread

struct LdsArgs {
  const float* x;       // unpadded NDHWC input (channels [0, c1) of a two-source input)
  const float* x2;      // channels [c1, cin) of a two-source input, or null
  int c1;               // channels of x (cin for one source; a multiple of 16)
  const float* affine;  // (n, cin, 2) or null
  const char* wp;       // packed weight [tap][kblock][np][64 bytes]
  const float* bias;
  const float* res;
  float* y;             // output, or split partial planes
  int64_t x_bytes, w_bytes, plane;
  int n, d, h, w, cin, cout, np, kb;
  int tz, ty, tx;       // bricks per axis
  int n_tiles, split;
  int affine_on, silu_on, batch_bias, has_res, has_bias;
  double* stats;        // group-norm partials of the output (ctmr_conv3d_gn) or null
  int gn_groups, gn_cpg;
};

// conv_lds_kernel over one (a.x2 null) or two input tensors, with the staging
// transform xf (bit 0 affine, bit 1 SiLU) and `wsets` wave sets a workgroup.
void launch_conv_lds(int xf, int wsets, dim3 grid, hipStream_t st, const LdsArgs& a);

// The plane-marching conv of 8 input channels (conv_march.hip).
struct MarchArgs {
  const float* x;       // unpadded NDHWC input, 8 channels
  const float* affine;  // (n, 8, 2) or null
  const float* wp;      // packed im2col weight [kblock][np][16]
  const float* bias;    // null: none
  const float* res;     // null: none
  float* y;
  int n, d, h, w, od, oh, ow, cout, np;
  int tz, ty, tx, run;  // output tiles per axis; depths per tile
  int affine_on, silu_on, batch_bias;
  double* stats;        // group-norm partials per tile (stride 2) or null
  int gn_groups;
};

// Output rows and columns of its workgroup's tile.
constexpr int march_rows(int stride) { return stride == 1 ? 16 : 8; }
constexpr int march_cols(int stride) { return stride == 1 ? 32 : 16; }
void launch_conv_march(int stride, dim3 grid, hipStream_t st, const MarchArgs& a);

}  // namespace ctmr
