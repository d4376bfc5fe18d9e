// The fp32 LDS-staged implicit GEMM of 3x3x3 convolutions: fp32 operands as
// three bf16 parts on bf16 MFMA.
#include "conv_gemm.hpp"

#include <utility>

namespace ctmr {

// ---------------------------------------------------------------------------
// 3b. LDS-staged implicit GEMM (large stride-1 fp32 volumes)
// ---------------------------------------------------------------------------
// A workgroup owns a 4x8x8 brick of output voxels (wave m holds depth m) and
// 64 output channels.  For each 16-channel chunk it stages the brick's 6x10x10
// halo from the unpadded NDHWC input into LDS -- zero outside the volume,
// group-norm affine + SiLU applied on the way -- then runs all 27 taps.
//
// Products.  FP32 MFMA runs at a sixteenth of the bf16 rate, so each fp32
// operand v is staged as three bf16 parts h = bf16(v), m = bf16(v - h), l =
// bf16(v - h - m), round to nearest: both differences are exact and h + m + l
// holds all 24 significant bits at v's own exponent, for v from 2^-110 (l's
// last bit is then bf16's smallest, 2^-133) to bf16's largest.  Of the nine
// part products the six at or above 2^-17 of the full product run on
// v_mfma_f32_32x32x16_bf16 (hh, hm, mh, mm, hl, lh; each exact in fp32), the
// dropped ml, lm, ll are below 2^-24 together, and fewer fp32 roundings per sum
// (one per 16 channels and part product) leave the results closer to 64 bits
// than FP32 MFMA's.  Results outside what the parts hold (part_sum_keep: not
// finite, or below 2^-60) are summed again on FP32 MFMA (x3_rerun).
//
// Bound by the matrix pipe: 24 MFMAs of 32 cycles per wave, tap and chunk
// against 12 ds_read_b128, 1 KiB each.  A and B both come from LDS: a staged
// voxel (and a weight column) is 96 bytes, [h | m | l] of 16 channels, the two
// 16-byte halves of a part exchanged where bit 1 of the halo line (bit 4 of
// the column) is set, so the 16 lanes that ds_read_b128 serves at once (equal
// bit 5, equal parity of bits 2-4) hit 16 distinct bank groups.  The packed
// fp32 weights are split by the workgroup, four values per thread and tap, two
// taps ahead in a two-slot ring: one barrier per tap publishes the next slot.
// The next chunk's halo is in flight in registers meanwhile.
// Measured against the same tiling on FP32 MFMA: 128 -> 128 channels at 128^3
// with the norm and SiLU 13.0 -> 7.73 ms (240 TFLOP/s: 1440 in bf16 products,
// MFMA busy 81 % at the 1.65 GHz the power limit leaves), 64 -> 64 at 64^3 404
// -> 268 us (MFMA busy 70 %), no bank conflicts; one 32-column block, 32 -> 32 at
// 128 x 128 x 64, 302 us (192 TFLOP/s; a tap reads nine operands for six products,
// twelve for twelve with two blocks); distance from 64 bits over
// residual blocks 4.5e-7 .. 7.0e-7 -> 3.9e-7 .. 6.0e-7.
constexpr int kX3Row = 96;                                // a staged voxel or weight column
constexpr int kX3Halo = kHaloVox * kX3Row;                // 57600
constexpr int kX3Tap = 64 * kX3Row;                       // one tap's 64 columns
constexpr int kX3Set = kX3Halo + 2 * kX3Tap;              // 69888

typedef float f16v __attribute__((ext_vector_type(16)));
// Brick line of row r = lane % 32 of MFMA row block mb: mb + brick32_line(r)
// (column r % 8).
__device__ __forceinline__ int brick32_line(int r) { return ((r >> 3) & 1) * 4 + (r >> 4) * 2; }

// store_brick for 32x32 accumulator blocks: lane l of block (mb, nb) holds
// voxel (z0 + wave, y0 + mb + brick32_line(l % 32), x0 + l % 8) and output
// columns n0 + nb*32 + 8*q + 4*(l/32) + r in element 4*q + r.  Group-norm
// column sums: per lane over mb, then the 16-lane rows (row16_sum), whose
// eight partials per column (two per wave) combine in ascending order.
template <int NB, typename Args, typename AfterBias = NoTerm>
__device__ __forceinline__ void store_brick32(const Args& p, f16v (&acc)[2][NB], int b, int split_id, int z0, int y0,
                                              int x0, int n0, int wave, int lane, int tile_id,
                                              double (*red)[64][2], AfterBias after_bias = {}) {
  const int r32 = lane & 31, half = lane >> 5;
  const bool partial = p.split > 1;
  float* out = p.y + (partial ? (int64_t)split_id * p.plane : 0);
  const int z = z0 + wave, x = x0 + (r32 & 7);
  bool row_ok[2];
  int64_t base[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int y = y0 + mb + brick32_line(r32);
    row_ok[mb] = z < p.d && y < p.h && x < p.w;
    base[mb] = ((((int64_t)b * p.d + min(z, p.d - 1)) * p.h + min(y, p.h - 1)) * p.w + min(x, p.w - 1)) * p.cout +
               n0 + 4 * half;
  }
  if (!partial && p.has_bias) {
    const float* bias_b = p.bias + (p.batch_bias ? (int64_t)b * p.cout : 0) + n0 + 4 * half;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float bq = bias_b[nb * 32 + 8 * (i >> 2) + (i & 3)];
        acc[0][nb][i] += bq;
        acc[1][nb][i] += bq;
      }
  }
  after_bias(acc);
  if (!partial && p.has_res) {  // every residual load before the first store
    f4 rq[2][NB][4];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          rq[mb][nb][q] = *reinterpret_cast<const f4*>(p.res + base[mb] + nb * 32 + 8 * q);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][nb][i] += rq[mb][nb][i >> 2][i & 3];
  }
  {
    // buffer stores relative to the brick's first output plane, as store_brick's
    const int64_t origin = ((int64_t)b * p.d + min(z0, p.d - 1)) * p.h * (int64_t)p.w * p.cout;
    const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
        out + origin, (short)0, (int)min(max((int64_t)p.plane - origin, (int64_t)0) * 4, (int64_t)0x7fffffff),
        0x00020000);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (row_ok[mb]) {
            const f4 val = f4{acc[mb][nb][4 * q], acc[mb][nb][4 * q + 1], acc[mb][nb][4 * q + 2],
                              acc[mb][nb][4 * q + 3]};
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, val), ors,
                                                   (int)((base[mb] - origin + nb * 32 + 8 * q) * 4), 0, kStoreSC1);
          }
  }
  if (p.stats) {  // a kernel argument: every thread reaches the barriers
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const double d0 = row_ok[0] ? (double)acc[0][nb][i] : 0.0, d1 = row_ok[1] ? (double)acc[1][nb][i] : 0.0;
        const double q1 = row16_sum(d0 + d1), q2 = row16_sum(fma(d1, d1, d0 * d0));
        if ((lane & 15) == 0) {
          double* o = red[wave * 2 + ((lane >> 4) & 1)][nb * 32 + 8 * (i >> 2) + 4 * half + (i & 3)];
          o[0] = q1;
          o[1] = q2;
        }
      }
    __syncthreads();
    combine_gn_partials<2 * NB, 8, 1>(red, n0, p.cout, p.gn_cpg, p.gn_groups,
                                 p.stats + ((int64_t)b * p.tz * p.ty * p.tx + tile_id) * p.gn_groups * 2);
  }
}

// The wave's results that the part products do not hold (part_sum_keep), as
// fp32 products over chunks [c_begin, c_end).  Reached by volumes that hold an
// infinity, a NaN or values near either end of fp32's range, and one of those
// can reach every output of the layers after it (through a group norm), so the
// whole tile runs on FP32 MFMA
// (v_mfma_f32_32x32x2_f32), operands straight from memory: the cost stays a
// few times the finite one whatever the values.  Lane half h holds channels
// 8h .. 8h + 7 of a chunk, product j the pair of channels j and 8 + j.
// `buf`: the wave's 16 KiB of LDS (no wave reads the staged operands any more)
// keeps the part products' results meanwhile.
template <int XF, int NB>
__device__ __forceinline__ void x3_rerun(const LdsArgs& p, f16v (&acc)[2][NB], f16v* buf, int b, int z, int y0,
                                         int x0, int n0, int lane, int c_begin, int c_end) {
  const int r32 = lane & 31, half = lane >> 5, x = x0 + (r32 & 7), y = y0 + brick32_line(r32);
#pragma unroll
  for (int i = 0; i < 2 * NB; ++i) {
    buf[i * 64 + lane] = acc[i / NB][i % NB];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i / NB][i % NB][e] = 0.f;
  }
#pragma clang loop unroll(disable)
  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    const bool second = chunk * 16 >= p.c1;
    const int row = second ? p.cin - p.c1 : p.c1;
    const float* src = (second ? p.x2 + (chunk * 16 - p.c1) : p.x + chunk * 16) + 8 * half;
    float sc[8], of[8];
    if constexpr ((XF & 1) != 0) {
      const float* a = p.affine + ((int64_t)b * p.cin + chunk * 16 + 8 * half) * 2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sc[j] = a[2 * j];
        of[j] = a[2 * j + 1];
      }
    }
#pragma clang loop unroll(disable)
    for (int tap = 0; tap < 27; ++tap) {
      const int gz = z + tap / 9 - 1, gx = x + tap % 3 - 1;
      f4a4 A[2][2], B[NB][2];
      bool in[2];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int gy = y + mb + (tap / 3) % 3 - 1;
        in[mb] = gz >= 0 && gz < p.d && gy >= 0 && gy < p.h && gx >= 0 && gx < p.w;
        const int64_t vox = in[mb] ? (((int64_t)b * p.d + gz) * p.h + gy) * p.w + gx : 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) A[mb][q] = *reinterpret_cast<const f4a4*>(src + vox * row + 4 * q);
      }
      const float* wb = reinterpret_cast<const float*>(p.wp) +
                        (((int64_t)tap * p.kb + chunk) * p.np + n0 + r32) * 16 + 8 * half;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 2; ++q) B[nb][q] = *reinterpret_cast<const f4a4*>(wb + nb * 32 * 16 + 4 * q);
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          float v = A[mb][j >> 2][j & 3];
          if constexpr ((XF & 1) != 0) v = fmaf(v, sc[j], of[j]);
          if constexpr ((XF & 2) != 0) v = silu_f(v);
          v = in[mb] ? v : 0.f;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(B[nb][j >> 2][j & 3], v, acc[mb][nb], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 2 * NB; ++i) {
    const f16v was = buf[i * 64 + lane];
#pragma unroll
    for (int e = 0; e < 16; ++e)
      acc[i / NB][i % NB][e] = part_sum_keep(was[e], acc[i / NB][i % NB][e]);
  }
}

// TWO: the input is two tensors (ctmr_conv3d_cat); the one-tensor kernel keeps
// precomputed byte offsets and a single descriptor.  XF: the staging
// transform, bit 0 the GN affine and bit 1 SiLU (p.affine_on, p.silu_on), as
// template flags so the transform is branch-free code.  WS = 2: a K split of
// two ranges inside the workgroup -- wave set s (waves 4s .. 4s + 3, each set
// with its own halo and weight slots) runs the chunks of range s of one brick,
// and set 0 adds set 1's sums after the bias, the order of the split reduction
// (bias, range 0, range 1, residual), with no partial planes in memory; both
// sets run the same chunk count, so every barrier is the workgroup's.  NB: 32-
// column blocks a workgroup computes, two, or one for 32 outputs.
template <bool TWO, int XF, int WS, int NB = 2>
__global__ __launch_bounds__(256 * WS, WS == 1 ? 2 : 1) void conv_lds_kernel(LdsArgs p) {
  static_assert(WS == 1 || WS == 2, "one or two wave sets");
  __shared__ __attribute__((aligned(256))) char lds_sets[WS * kX3Set];
  const int set = WS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  char* const lds = lds_sets + set * kX3Set;
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order (as conv_kernel): neighbouring bricks share halo planes.
  const int nb = gridDim.x, bid = blockIdx.x;
  const int xcd = bid & 7, slot = bid >> 3, per = nb >> 3, rem = nb & 7;
  const int tile = (xcd < rem) ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
  const int n_tile = tile % p.n_tiles;
  int rest = tile / p.n_tiles;
  const int bx = rest % p.tx;
  rest /= p.tx;
  const int by = rest % p.ty;
  rest /= p.ty;
  const int bz = rest % p.tz;
  rest /= p.tz;
  const int b = rest % p.n;
  const int split_id = rest / p.n;
  const int z0 = bz * kBD, y0 = by * kBH, x0 = bx * kBW;
  const int r32 = lane & 31, half = lane >> 5;

  // Staging: piece i of thread t is channels 4*(t&3)..+3 of the chunk at halo
  // voxel (t>>2) + 64i.  Offsets are relative to the first staged plane, so
  // they stay within 32 bits (the host checks 6 planes fit).  goff[i] is the
  // piece's byte offset; with TWO it is the piece's voxel index instead: a
  // chunk comes from x (chunks below c1 / 16) or from x2, whose rows hold the
  // remaining channels, and the byte offset follows from the chunk's source.
  const int part = tid & 3;
  const int zb = max(z0 - 1, 0);
  const int c2 = p.cin - p.c1;
  const int kb1 = p.c1 >> 4;
  const int64_t vbase = ((int64_t)b * p.d + zb) * p.h * p.w;     // first staged voxel
  const int64_t vtotal = (int64_t)p.n * p.d * p.h * p.w;
  const __amdgpu_buffer_rsrc_t xrsrc1 = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.x + vbase * p.c1), (short)0, (int)min((vtotal - vbase) * p.c1 * 4, (int64_t)0x7fffffff),
      0x00020000);
  const __amdgpu_buffer_rsrc_t xrsrc2 = TWO ? __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.x2 + vbase * c2), (short)0, (int)min((vtotal - vbase) * c2 * 4, (int64_t)0x7fffffff),
      0x00020000) : xrsrc1;
  int goff[kStageIters];
  unsigned valid = 0, swap = 0;  // swap: pieces on halo lines with bit 1 set
#pragma unroll
  for (int i = 0; i < kStageIters; ++i) {
    const int hv = (tid >> 2) + 64 * i;
    goff[i] = 0;
    if (hv < kHaloVox) {
      const int hz = hv / (kHH * kHW), hr = hv - hz * (kHH * kHW);
      const int hy = hr / kHW, hx = hr - hy * kHW;
      const int gz = z0 - 1 + hz, gy = y0 - 1 + hy, gx = x0 - 1 + hx;
      if ((hy >> 1) & 1) swap |= 1u << i;
      if (gz >= 0 && gz < p.d && gy >= 0 && gy < p.h && gx >= 0 && gx < p.w) {
        valid |= 1u << i;
        const int vox = ((gz - zb) * p.h + gy) * p.w + gx;
        goff[i] = TWO ? vox : vox * p.cin * 4 + part * 16;
      }
    }
  }
  // Source of a chunk: descriptor, row bytes (TWO) and the chunk's byte offset in a row.
  struct ChunkSrc {
    __amdgpu_buffer_rsrc_t rs;
    int row, so;
  };
  auto chunk_src = [&](int chunk) {
    ChunkSrc c;
    const bool second = TWO && chunk >= kb1;
    c.rs = second ? xrsrc2 : xrsrc1;
    c.row = (second ? c2 : p.c1) * 4;
    c.so = __builtin_amdgcn_readfirstlane((second ? chunk - kb1 : chunk) * 64);
    return c;
  };
  auto piece_off = [&](int i, const ChunkSrc& c) { return TWO ? goff[i] * c.row + part * 16 : goff[i]; };

  // A: LDS bytes of this lane's voxel of row block 0 at tap (0, 0, 0), half
  // `half` of part h; av[v] where bit 1 of (block + kh) is v.
  const int avox = (wave * kHH + brick32_line(r32)) * kHW + (r32 & 7);
  const char* const av[2] = {lds + avox * kX3Row + 16 * (half ^ (r32 >> 4)),
                             lds + avox * kX3Row + 16 * (half ^ (r32 >> 4) ^ 1)};
  // B: this lane's column of column block 0 in slot 0.
  const int n0 = n_tile * 32 * NB;
  const char* const bv = lds + kX3Halo + r32 * kX3Row + 16 * (half ^ (r32 >> 4));
  // Weight split: thread t takes channels 4*(t&3)..+3 of column t>>2.
  char* const bw = lds + kX3Halo + (tid >> 2) * kX3Row + 16 * ((part >> 1) ^ ((tid >> 6) & 1)) + 8 * (part & 1);
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.wp, (short)0, (int)min(p.w_bytes, (int64_t)0x7fffffff), 0x00020000);
  const int boff = n0 * 64 + tid * 16;
  const int bchunk = p.np * 64;

  f16v acc[2][NB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int kpart = split_id * WS + set, kparts = p.split * WS;
  const int c_begin = __builtin_amdgcn_readfirstlane((int)((int64_t)kpart * p.kb / kparts));
  const int c_end = __builtin_amdgcn_readfirstlane((int)((int64_t)(kpart + 1) * p.kb / kparts));

  u4 stage[kStageIters];
  // GN affine of this thread's four channels of a chunk: (scale, offset) pairs.
  auto load_affine = [&](int chunk, f4& sc, f4& of) {
    sc = f4{1.f, 1.f, 1.f, 1.f};
    of = f4{0.f, 0.f, 0.f, 0.f};
    if constexpr ((XF & 1) != 0) {
      const f4* q = reinterpret_cast<const f4*>(p.affine + ((int64_t)b * p.cin + chunk * 16 + part * 4) * 2);
      const f4 a0 = q[0], a1 = q[1];
      sc = f4{a0[0], a0[2], a1[0], a1[2]};
      of = f4{a0[1], a0[3], a1[1], a1[3]};
    }
  };
  // Piece i as staged: GN affine, SiLU, zero outside the volume.
  auto transform = [&](int i, const f4& sc, const f4& of) {
    f4 v = __builtin_bit_cast(f4, stage[i]);
    const bool in = (valid >> i) & 1u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float t = v[j];
      if constexpr ((XF & 1) != 0) t = fmaf(t, sc[j], of[j]);
      if constexpr ((XF & 2) != 0) t = silu_f(t);
      v[j] = in ? t : 0.f;
    }
    stage[i] = __builtin_bit_cast(u4, v);
  };
  auto commit = [&](int i) {
    const int hv = (tid >> 2) + 64 * i;
    if (hv >= kHaloVox) return;
    uint2 h, m, l;
    split_bf16x3(__builtin_bit_cast(f4, stage[i]), h, m, l);
    char* o = lds + hv * kX3Row + 16 * ((part >> 1) ^ ((swap >> i) & 1)) + 8 * (part & 1);
    *reinterpret_cast<uint2*>(o) = h;
    *reinterpret_cast<uint2*>(o + 32) = m;
    *reinterpret_cast<uint2*>(o + 64) = l;
  };
  auto load_w = [&](int tap, int chunk) {
    const int so = __builtin_amdgcn_readfirstlane((tap * p.kb + chunk) * bchunk);
    return __builtin_amdgcn_raw_buffer_load_b128(brsrc, boff, so, 0);
  };
  auto put_w = [&](u4 w, char* dst) {
    if (NB == 1 && tid >= 128) return;  // the columns of a whole block only
    uint2 h, m, l;
    split_bf16x3(__builtin_bit_cast(f4, w), h, m, l);
    *reinterpret_cast<uint2*>(dst) = h;
    *reinterpret_cast<uint2*>(dst + 32) = m;
    *reinterpret_cast<uint2*>(dst + 64) = l;
  };
  auto read_a = [&](bf8 (&A)[2], int tap, int pt) {
    const int kd = tap / 9, kh = (tap / 3) % 3, kw = tap % 3;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
      A[mb] = *reinterpret_cast<const bf8*>(av[((mb + kh) >> 1) & 1] + ((kd * kHH + kh + mb) * kHW + kw) * kX3Row +
                                            pt * 32);
  };
  auto read_b = [&](bf8 (&B)[NB], const char* slot, int pt) {
#pragma unroll
    for (int n = 0; n < NB; ++n) B[n] = *reinterpret_cast<const bf8*>(slot + n * 32 * kX3Row + pt * 32);
  };
  auto mma = [&](const bf8 (&A)[2], const bf8 (&B)[NB]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(B[j], A[i], acc[i][j], 0, 0, 0);
  };

  // Prologue: the first chunk's halo and its first two taps' weights.
  {
    const ChunkSrc c = chunk_src(c_begin);
#pragma unroll
    for (int i = 0; i < kStageIters; ++i)
      stage[i] = __builtin_amdgcn_raw_buffer_load_b128(c.rs, piece_off(i, c), c.so, 0);
  }
  // raw[t % 3]: the weights of tap t + 2 before step t, of tap t + 5 after it
  u4 raw[3] = {load_w(0, c_begin), load_w(1, c_begin), u4{0u, 0u, 0u, 0u}};
  int cur = 0, nxt = kX3Tap;  // slot offsets of the tap in the registers and of the next
  {
    f4 sc, of;
    load_affine(c_begin, sc, of);
#pragma unroll
    for (int i = 0; i < kStageIters; ++i) {
      transform(i, sc, of);
      commit(i);
    }
  }
  put_w(raw[0], bw);
  put_w(raw[1], bw + kX3Tap);
#pragma unroll
  for (int i = 0; i < 3; ++i) raw[i] = load_w(i + 2, c_begin);
  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    lds_barrier();  // the chunk's halo and the weights of its first two taps are in LDS
    bf8 Ah[2], Am[2], Al[2], Bh[NB], Bm[NB], Bl[NB];
    read_a(Al, 0, 2);
    read_b(Bh, bv + cur, 0);
    read_a(Am, 0, 1);
    read_a(Ah, 0, 0);
    read_b(Bm, bv + cur, 1);
    read_b(Bl, bv + cur, 2);
    // Unconditional (see conv_kernel): the last chunk re-reads itself.
    const int next = min(chunk + 1, c_end - 1);
    const ChunkSrc nx = chunk_src(next);
    f4 nsc, nof;
    load_affine(next, nsc, nof);
    const auto tap_step = [&](auto tap) __attribute__((always_inline)) {
      constexpr int t = decltype(tap)::value;
      // Every wave holds tap t in registers and tap t + 1's slot is written:
      // tap t's slot takes tap t + 2 (of the next chunk from tap 25 on).
      lds_barrier();
      put_w(raw[t % 3], bw + cur);
      raw[t % 3] = t + 5 < 27 ? load_w(t + 5, chunk) : load_w(t + 5 - 27, next);
      // The next chunk's halo, one 16-byte piece every other tap.
      if constexpr ((t & 1) && (t >> 1) < kStageIters)
        stage[t >> 1] = __builtin_amdgcn_raw_buffer_load_b128(nx.rs, piece_off(t >> 1, nx), nx.so, 0);
      if constexpr (t >= 6 && !(t & 1) && ((t - 6) >> 1) < kStageIters) transform((t - 6) >> 1, nsc, nof);
      constexpr bool more = t + 1 < 27;
      const char* const bn = bv + nxt;
      __builtin_amdgcn_s_setprio(1);
      mma(Al, Bh);
      if constexpr (more) read_a(Al, t + 1, 2);
      mma(Am, Bh);
      mma(Ah, Bh);
      if constexpr (more) read_b(Bh, bn, 0);
      mma(Am, Bm);
      if constexpr (more) read_a(Am, t + 1, 1);
      mma(Ah, Bm);
      if constexpr (more) read_b(Bm, bn, 1);
      mma(Ah, Bl);
      if constexpr (more) read_a(Ah, t + 1, 0);
      if constexpr (more) read_b(Bl, bn, 2);
      __builtin_amdgcn_s_setprio(0);
      // Tap 26 is in registers and every wave has passed its reads: the next
      // chunk's halo (the last chunk writes its own again, unread).
      if constexpr (t == 26) {
#pragma unroll
        for (int i = 0; i < kStageIters; ++i) commit(i);
      }
      const int sw = cur;
      cur = nxt;
      nxt = sw;
    };
    [&]<int... T>(std::integer_sequence<int, T...>) __attribute__((always_inline)) {
      (tap_step(std::integral_constant<int, T>{}), ...);
    }(std::make_integer_sequence<int, 27>{});
  }

  PartSumProbe probe;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; e += 2) probe.add(acc[i][j][e], acc[i][j][e + 1]);
  lds_barrier();
  static_assert(4 * 64 * 256 <= kX3Set, "a set's results fit its staging buffers");
  PartSumTest test;
  if (__any(probe.maybe())) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) test.add(acc[i][j][e]);
  }
  if (__any(test.any()))
    x3_rerun<XF>(p, acc, reinterpret_cast<f16v*>(lds) + wave * 128 * NB, b, z0 + wave, y0, x0, n0, lane, c_begin,
                 c_end);

  // The statistics' reduction buffer and the hand-over below reuse the halos.
  double (*const red)[64][2] = reinterpret_cast<double (*)[64][2]>(lds_sets);
  const int tile_id = (bz * p.ty + by) * p.tx + bx;
  if constexpr (WS == 2) {
    // Set 1 hands its sums to set 0 through LDS past the statistics' 8 KiB
    // once every wave has finished its last chunk, then ends; the barriers
    // after that wait only for set 0's waves.
    f16v* const xs = reinterpret_cast<f16v*>(lds_sets + 8192);
    static_assert(8192 + 4 * 4 * 64 * 64 <= WS * kX3Set, "hand-over buffer");
    __syncthreads();
    if (set == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) xs[(wave * 4 + i) * 64 + lane] = acc[i >> 1][i & 1];
    }
    __syncthreads();
    if (set == 1) return;
    store_brick32(p, acc, b, split_id, z0, y0, x0, n0, wave, lane, tile_id, red, [&](f16v (&a)[2][2]) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i >> 1][i & 1] += xs[(wave * 4 + i) * 64 + lane];
    });
  } else {
    store_brick32(p, acc, b, split_id, z0, y0, x0, n0, wave, lane, tile_id, red);
  }
}

// conv_lds_kernel for a staging transform xf (bit 0 affine, bit 1 SiLU).
template <bool TWO, int WS, int NB = 2>
static void launch_lds(int xf, dim3 grid, hipStream_t st, const LdsArgs& a) {
  const dim3 block(256 * WS);
  switch (xf) {
    case 0: hipLaunchKernelGGL((conv_lds_kernel<TWO, 0, WS, NB>), grid, block, 0, st, a); break;
    case 1: hipLaunchKernelGGL((conv_lds_kernel<TWO, 1, WS, NB>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((conv_lds_kernel<TWO, 2, WS, NB>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((conv_lds_kernel<TWO, 3, WS, NB>), grid, block, 0, st, a); break;
  }
}


void launch_conv_lds(int xf, int wsets, dim3 grid, hipStream_t st, const LdsArgs& a) {
  if (a.x2) {
    if (wsets == 2) launch_lds<true, 2>(xf, grid, st, a);
    else launch_lds<true, 1>(xf, grid, st, a);
  } else {
    if (wsets == 2) launch_lds<false, 2>(xf, grid, st, a);
    else if (a.cout == 32) launch_lds<false, 1, 1>(xf, grid, st, a);
    else launch_lds<false, 1>(xf, grid, st, a);
  }
}

}  // namespace ctmr
