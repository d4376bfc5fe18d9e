// 3x3x3 convolutions of 8 input channels that walk the volume plane by plane:
// fp32 operands as three bf16 parts on bf16 MFMA.
#include "conv_gemm.hpp"

#include <type_traits>

namespace ctmr {

// ---------------------------------------------------------------------------
// 3b''. Plane-marching conv for 8 input channels (fp32; stride 1 with 8
// outputs, stride 2 with 17 .. 32: the label-condition encoder)
// ---------------------------------------------------------------------------
// A workgroup owns a tile of output rows and columns over a run of output
// depths and reads every input plane of the run once, double-buffered in LDS:
// affine, SiLU and the split into three bf16 parts (h, m, l; as the LDS-staged
// GEMM's) are done once per staged voxel.  A voxel is 48 bytes, [h | m | l] of
// its 8 channels, and the lines are a multiple of 256 bytes apart, so each of a
// lane's operands is one ds_read_b128 without bank conflicts.
//
// The contraction is v_mfma_f32_16x16x32_bf16 over 16 output columns of one
// line, K = 4 input lines x 8 channels: lane group g of the voxel operand holds
// halo line g of the row block.  Stride 1 needs lines 0 .. 2 for its first and
// 1 .. 3 for its second output row, so the 16 weight columns are 2 rows x 8
// outputs with zeros where a line is not in a row's window; stride 2 takes
// lines 0 .. 2 (the fourth's weights are zero; it re-reads line 2) and 16 of
// its 32 outputs per wave.  The split weights of all 27 taps stay in registers
// (108 of them) for the whole run.  A plane's operands, read once, serve every
// depth tap: kd = 0, 1, 2 add to the sums of the next, this and the previous
// output plane (stride 2: odd planes kd = 0 and 2, even planes kd = 1).
// Six part products, summed smallest first in fp32 per (plane, column tap); a
// result that they do not hold is summed again on FP32 MFMA (march_rerun).
//
// Bound by HBM and the matrix pipe about equally: 8 -> 8 channels at 256 x 256 x
// 128 moves 0.54 GB (115 us at a large copy's rate) against 112 us of MFMAs.
// Measured there with SiLU on the input, against the brick GEMM on FP32 MFMA and
// a SiLU pass: 695 -> 200 us; 8 -> 32 at stride 2, against im2col rows in memory,
// 907 -> 130 us.  What is left is latency: a workgroup alone takes about 3 us a
// plane, 1.5 of them MFMAs, the next plane's loads in flight for one plane only
// (registers allow no more).  Operands read one step ahead, or the next plane's
// split set between the products' MFMAs, measured no faster (192 and 203 us
// against 189 without SiLU).
// Caller's pointers are 4-byte aligned.
constexpr int kMarchVox = 48;
constexpr int kMarchPitch = 1792;  // 7 * 256 >= 34 (stride 1) or 33 (stride 2) voxels

template <int STRIDE>
struct March {
  static constexpr int TH = march_rows(STRIDE), TW = march_cols(STRIDE);  // output tile
  static constexpr int HH = STRIDE * (TH - 1) + 3, HW = STRIDE * (TW - 1) + 3;  // halo lines, columns
  static constexpr int kVox = HH * HW;
  static constexpr int kIters = (kVox + 255) / 256;
  static constexpr int kBuf = HH * kMarchPitch;
  static constexpr int kAcc = STRIDE == 1 ? 3 : 2;  // output planes in flight
};

// The sums of a wave's four row blocks (layout of `acc`) as fp32 products on
// FP32 MFMA (v_mfma_f32_16x16x4_f32), operands straight from memory: for a plane
// with a result that the part products do not hold (part_sum_keep; the bound on
// the cost as x3_rerun's, conv_lds.hip).  Lane group g holds line g of one output
// row's window (lane group 3 zeros on both sides: a zero weight must not meet an
// infinity), product j its channel j; stride 1 computes its two output rows one
// after the other.  oy: the output row of block 0; ox: this lane's output column;
// wbase: the first of the wave's output channels.
template <int STRIDE>
__device__ __forceinline__ void march_rerun(const MarchArgs& p, f4 (&sum)[4], int b, int oz, int oy, int ox, int wbase,
                                            int lrow, int lgrp) {
  const int wcol = min(STRIDE == 1 ? lrow & 7 : wbase + lrow, p.cout - 1);
#pragma clang loop unroll(disable)
  for (int r = 0; r < (STRIDE == 1 ? 2 : 1); ++r) {
    f4 part[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) part[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
    for (int k = 0; k < 9; ++k) {
      const int kd = k / 3, kw = k % 3, tap = (kd * 3 + min(lgrp, 2)) * 3 + kw;
      const f4a4* wp = reinterpret_cast<const f4a4*>(p.wp + ((int64_t)(tap >> 1) * p.np + wcol) * 16 + (tap & 1) * 8);
      f4 w[2] = {wp[0], wp[1]};
      const int gz = oz * STRIDE + kd - 1, gx = ox * STRIDE + kw - 1;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int gy = (oy + (STRIDE == 1 ? 2 * t + r : t)) * STRIDE + lgrp - 1;
        const bool in = lgrp < 3 && gz >= 0 && gz < p.d && gy >= 0 && gy < p.h && gx >= 0 && gx < p.w;
        const int64_t vox = in ? (((int64_t)b * p.d + gz) * p.h + gy) * p.w + gx : 0;
        const f4a4* xp = reinterpret_cast<const f4a4*>(p.x + vox * 8);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const f4 v = xp[e];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float s = v[j];
            if (p.affine_on) {
              const float* a = p.affine + (b * 8 + e * 4 + j) * 2;
              s = fmaf(s, a[0], a[1]);
            }
            if (p.silu_on) s = silu_f(s);
            part[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(lgrp < 3 ? w[e][j] : 0.f, in ? s : 0.f, part[t], 0, 0, 0);
          }
        }
      }
    }
    if (STRIDE == 2 || (lgrp >> 1) == r) {
#pragma unroll
      for (int t = 0; t < 4; ++t) sum[t] = part[t];
    }
  }
}

template <int STRIDE>
__global__ __launch_bounds__(256, 2) void conv_march_kernel(MarchArgs p) {
  using M = March<STRIDE>;
  __shared__ __attribute__((aligned(256))) char lds[2 * M::kBuf];
  __shared__ double red[4][16][2];  // group-norm sums: each wave's 16 output columns
  const int tid = threadIdx.x, lane = tid & 63, lrow = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order: tiles that share halo lines run on one XCD
  const int nb = gridDim.x, bid = blockIdx.x;
  const int xcd = bid & 7, slot = bid >> 3, per = nb >> 3, rem = nb & 7;
  const int tile = (xcd < rem) ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
  const int bx = tile % p.tx, by = (tile / p.tx) % p.ty;
  const int bz = (tile / (p.tx * p.ty)) % p.tz, b = tile / (p.tx * p.ty * p.tz);
  const int oz0 = bz * p.run, oz1 = min(oz0 + p.run, p.od);
  const int y0 = by * M::TH, x0 = bx * M::TW;

  // Weights: this lane's output column and halo line, all (kd, kw), split.
  // Stride 1: rows of 2 x 8 columns; stride 2: 16 of the outputs by wave parity.
  // `first` on: every load before the first split, one round of latency; a kd at
  // a time otherwise (the rerun's registers).
  u4 W[3][3][3];
  auto load_weights = [&](int ln, auto first) __attribute__((always_inline)) {
    const int wrow = STRIDE == 1 ? (ln & 15) >> 3 : 0;
    const int wcol = STRIDE == 1 ? ln & 7 : (wave & 1) * 16 + (ln & 15);
    const int kh = (ln >> 4) - wrow;
    const bool w_on = kh >= 0 && kh < 3 && wcol < p.cout;
    f4 raw[3][3][2];
    auto load_kd = [&](int kd) __attribute__((always_inline)) {
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) {
        const int tap = (kd * 3 + min(max(kh, 0), 2)) * 3 + kw;
        const f4a4* src = reinterpret_cast<const f4a4*>(p.wp + ((tap >> 1) * p.np + min(wcol, p.cout - 1)) * 16 +
                                                        (tap & 1) * 8);
        raw[kd][kw][0] = src[0];
        raw[kd][kw][1] = src[1];
      }
    };
    if constexpr (decltype(first)::value) {
#pragma unroll
      for (int kd = 0; kd < 3; ++kd) load_kd(kd);
    }
#pragma unroll
    for (int kd = 0; kd < 3; ++kd) {
      if constexpr (!decltype(first)::value) {
        __builtin_amdgcn_sched_barrier(0);
        load_kd(kd);
      }
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) {
        const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
        uint2 h[2], m[2], l[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) split_bf16x3(w_on ? raw[kd][kw][e] : zero, h[e], m[e], l[e]);
        W[kd][kw][0] = u4{h[0].x, h[0].y, h[1].x, h[1].y};
        W[kd][kw][1] = u4{m[0].x, m[0].y, m[1].x, m[1].y};
        W[kd][kw][2] = u4{l[0].x, l[0].y, l[1].x, l[1].y};
      }
    }
  };
  load_weights(lane, std::true_type{});

  // Staging: thread t holds halo voxels t + 256 i; offsets within a plane (the
  // host checks a plane spans under 2 GiB), -1 outside the volume.
  int goff[M::kIters], loff[M::kIters];
#pragma unroll
  for (int i = 0; i < M::kIters; ++i) {
    const int q = tid + 256 * i, hy = q / M::HW, hx = q % M::HW;
    const int gy = y0 * STRIDE - 1 + hy, gx = x0 * STRIDE - 1 + hx;
    const bool in = q < M::kVox && gy >= 0 && gy < p.h && gx >= 0 && gx < p.w;
    goff[i] = in ? (gy * p.w + gx) * 32 : -1;
    // stride 2: even columns first, then the odd ones, so a wave's 16 columns lie side by side
    const int px = STRIDE == 1 ? hx : (hx >> 1) + (hx & 1) * ((M::HW + 1) / 2);
    loff[i] = hy * kMarchPitch + px * kMarchVox;
  }
  const int plane_bytes = p.h * p.w * 32;
  u4 stage[M::kIters][2];
  auto load = [&](int z) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)p.x + ((int64_t)b * p.d + z) * plane_bytes), (short)0, plane_bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < M::kIters; ++i) {  // offset -1 is past the range: zeros
      stage[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, goff[i], 0, 0);
      stage[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, goff[i] < 0 ? -1 : goff[i] + 16, 0, 0);
    }
  };
  auto commit = [&](char* buf) {
#pragma unroll
    for (int i = 0; i < M::kIters; ++i) {
      uint2 h[2], m[2], l[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        f4 v = __builtin_bit_cast(f4, stage[i][e]);
        if (p.affine_on) {  // zero outside the volume, after the affine
          const float* a = p.affine + (b * 8 + e * 4) * 2;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float scaled = fmaf(v[j], a[2 * j], a[2 * j + 1]);
            v[j] = goff[i] < 0 ? 0.f : scaled;
          }
        }
        if (p.silu_on) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = silu_f(v[j]);
        }
        split_bf16x3(v, h[e], m[e], l[e]);
      }
      if (M::kVox % 256 == 0 || tid + 256 * i < M::kVox) {
        u4* dst = reinterpret_cast<u4*>(buf + loff[i]);
        dst[0] = u4{h[0].x, h[0].y, h[1].x, h[1].y};
        dst[1] = u4{m[0].x, m[0].y, m[1].x, m[1].y};
        dst[2] = u4{l[0].x, l[0].y, l[1].x, l[1].y};
      }
    }
  };

  // This wave's four row blocks: stride 1 rows 2 (4 (wave / 2) + t) .. + 1 of 16
  // columns (wave % 2); stride 2 row 4 (wave / 2) + t.
  const int line0 = 8 * (wave >> 1) + (STRIDE == 1 ? lgrp : min(lgrp, 2));
  const int abase = line0 * kMarchPitch + (lrow + (STRIDE == 1 ? (wave & 1) * 16 : 0)) * kMarchVox;
  constexpr int kLines = 2 * kMarchPitch;  // halo lines between row blocks (both strides)
  f4 acc[M::kAcc][4];
#pragma unroll
  for (int k = 0; k < M::kAcc; ++k)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[k][t] = f4{0.f, 0.f, 0.f, 0.f};

  // The plane's products: pairs(add) names the (sums, kd) pairs.  Two row blocks
  // at a time: at least two sums in turn on the matrix pipe.
  auto products = [&](const char* buf, auto pairs) {
    constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, iw[6] = {0, 2, 1, 0, 1, 0};  // lh hl mm mh hm hh
#pragma unroll
    for (int kw = 0; kw < 3; ++kw) {
      const int col = STRIDE == 1 ? kw * kMarchVox
                                  : (kw == 1 ? (M::HW + 1) / 2 * kMarchVox : (kw >> 1) * kMarchVox);
#pragma unroll
      for (int t0 = 0; t0 < 4; t0 += 2) {
        u4 A[2][3];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int q = 0; q < 3; ++q)
            A[t][q] = *reinterpret_cast<const u4*>(buf + abase + (t0 + t) * kLines + col + q * 16);
#pragma unroll
        for (int s = 0; s < 6; ++s)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            pairs([&](int k, int kd) {
              f4& c = acc[k][t0 + t];
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, W[kd][kw][iw[s]]),
                                                          __builtin_bit_cast(bf8, A[t][ia[s]]), c, 0, 0, 0);
            });
      }
    }
  };

  // Epilogue of a finished plane: lane l holds column l % 16 of its lines and
  // outputs ocol .. ocol + 3.
  const int orow = STRIDE == 1 ? 8 * (wave >> 1) + (lgrp >> 1) : 4 * (wave >> 1);
  const int ox = x0 + (STRIDE == 1 ? (wave & 1) * 16 : 0) + lrow;
  const int ocol = STRIDE == 1 ? (lgrp & 1) * 4 : (wave & 1) * 16 + lgrp * 4;
  f4 bias = f4{0.f, 0.f, 0.f, 0.f};
  if (p.bias && ocol < p.cout) {
    const float* bq = p.bias + (p.batch_bias ? b * p.cout : 0) + ocol;
    bias = f4{bq[0], bq[1], bq[2], bq[3]};
  }
  auto store = [&](f4 (&sum)[4], int oz) {
    PartSumProbe probe;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      probe.add(sum[t][0], sum[t][1]);
      probe.add(sum[t][2], sum[t][3]);
    }
    PartSumTest test;  // of the results to be stored
    if (__builtin_expect(__any(probe.maybe()), 0)) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int oy = y0 + orow + (STRIDE == 1 ? 2 * t : t);
#pragma unroll
        for (int j = 0; j < 4; ++j) test.add(oy < p.oh && ox < p.ow && ocol < p.cout ? sum[t][j] : 0.f);
      }
    }
    if (__builtin_expect(__any(test.any()), 0)) {
      // The weights are loaded again afterwards, and the lane's indices are
      // opaque copies: neither then holds registers in the loop or in here.
      int ln = threadIdx.x & 63;
      asm volatile("" : "+v"(ln));
      f4 again[4];
      march_rerun<STRIDE>(p, again, b, oz, y0 + (STRIDE == 1 ? 8 : 4) * (wave >> 1),
                          x0 + (STRIDE == 1 ? (wave & 1) * 16 : 0) + (ln & 15), (wave & 1) * 16, ln & 15, ln >> 4);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          sum[t][j] = part_sum_keep(sum[t][j], again[t][j]);
      load_weights(ln, std::false_type{});
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int oy = y0 + orow + (STRIDE == 1 ? 2 * t : t);
      if (oy >= p.oh || ox >= p.ow || ocol >= p.cout) continue;
      f4& v = sum[t];
      v += bias;
      const int64_t at = ((((int64_t)b * p.od + oz) * p.oh + oy) * p.ow + ox) * p.cout + ocol;
      if (p.res) v += *reinterpret_cast<const f4a4*>(p.res + at);
      *reinterpret_cast<f4a4*>(p.y + at) = v;
    }
    if (p.stats) {  // one column at a time: its lane sums over the row blocks, then the 16 columns of a line
#pragma clang loop unroll(disable)
      for (int j = 0; j < 4; ++j) {
        double a = 0.0, q = 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int oy = y0 + orow + (STRIDE == 1 ? 2 * t : t);
          const double v = j == 0 ? sum[t][0] : j == 1 ? sum[t][1] : j == 2 ? sum[t][2] : sum[t][3];
          if (oy < p.oh && ox < p.ow && ocol < p.cout) {
            a += v;
            q = fma(v, v, q);
          }
        }
        a = row16_sum(a);
        q = row16_sum(q);
        if (lrow == 0) {
          red[wave][lgrp * 4 + j][0] += a;
          red[wave][lgrp * 4 + j][1] += q;
        }
      }
    }
  };

  if (p.stats && lrow == 0) {  // read and added to by this lane only, until the last barrier
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave][lgrp * 4 + j][0] = red[wave][lgrp * 4 + j][1] = 0.0;
  }
  // Planes oz0 * STRIDE - 1 .. (oz1 - 1) * STRIDE + 1, those outside the volume
  // skipped: zeros add nothing.  One barrier per plane: a wave writes a buffer
  // after the barrier of the plane between, which every wave reaches only when
  // it has read the buffer's last plane.
  const int z_last = min((oz1 - 1) * STRIDE + 1, p.d - 1);
  int z = oz0 * STRIDE - 1;
  load(max(z, 0));
  int flip = 0;
  auto stage_plane = [&]() {  // publishes plane z, starts the next one's loads
    char* buf = lds + flip * M::kBuf;
    flip ^= 1;
    commit(buf);
    lds_barrier();
    if (z < z_last) load(z + 1);
    return (const char*)buf;
  };
  if constexpr (STRIDE == 1) {
    for (; z <= oz1; ++z) {
      if (z >= 0 && z <= z_last) {
        const char* buf = stage_plane();
        products(buf, [](auto add) { add(0, 2); add(1, 1); add(2, 0); });
      }
      if (z > oz0) store(acc[0], z - 1);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[0][t] = acc[1][t];
        acc[1][t] = acc[2][t];
        acc[2][t] = f4{0.f, 0.f, 0.f, 0.f};
      }
    }
  } else {
    if (z >= 0) {
      const char* buf = stage_plane();
      products(buf, [](auto add) { add(0, 0); });
    }
    ++z;
    for (int oz = oz0; oz < oz1; ++oz) {
      {
        const char* buf = stage_plane();  // plane 2 oz, always inside
        products(buf, [](auto add) { add(0, 1); });
      }
      ++z;
      if (z <= z_last) {
        const char* buf = stage_plane();
        products(buf, [](auto add) { add(0, 2); add(1, 0); });
      }
      ++z;
      store(acc[0], oz);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[0][t] = acc[1][t];
        acc[1][t] = f4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  if (p.stats) {  // a kernel argument: every thread reaches the barrier
    __syncthreads();
    const int cpg = p.cout / p.gn_groups;
    if (tid < p.gn_groups) {  // columns, then the waves that hold them (both rows of stride 1), ascending
      double a = 0.0, q = 0.0;
      for (int c = tid * cpg; c < (tid + 1) * cpg; ++c)
        for (int half = 0; half < (STRIDE == 1 ? 8 : 2); ++half) {
          const double* r = STRIDE == 1 ? red[half >> 1][(half & 1) * 8 + c] : red[half * 2 + (c >> 4)][c & 15];
          a += r[0];
          q += r[1];
        }
      double* out = p.stats + ((int64_t)tile * p.gn_groups + tid) * 2;
      out[0] = a;
      out[1] = q;
    }
  }
}

void launch_conv_march(int stride, dim3 grid, hipStream_t st, const MarchArgs& a) {
  if (stride == 1) hipLaunchKernelGGL((conv_march_kernel<1>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((conv_march_kernel<2>), grid, dim3(256), 0, st, a);
}

}  // namespace ctmr
