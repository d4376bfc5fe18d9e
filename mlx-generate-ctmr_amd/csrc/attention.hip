// Flash attention for 32-wide heads on gfx950 matrix cores: fp32 operands as
// three bf16 parts, and the reference's split-fp16 form.
//
// Computes softmax(Q K^T * scale) V per (batch item, head) without writing the
// scores, as _flash_attention.flash_attention does (_flash_attention.py:1-27,
// 320-360): an online softmax over key blocks with a running row maximum and
// sum, exp2 of log2(e)-scaled scores (the scale is folded into Q once).
//
// MI355X layout.  One wave owns 16 queries and walks its keys in blocks of 32.
// Both products run on 16x16x32 MFMA (bf16 or fp16 parts of the fp32 operands,
// fp32 accumulation) in the transposed form:
//   S^T = K Q^T   (rows = keys, columns = queries; k runs over the 32 head dims)
//   O^T += V^T P^T (rows = head dims, columns = queries; k runs over the block's keys)
// With the MFMA result layout (lane l, register r -> row 4*(l/16)+r, column
// l%16) a lane's S^T registers are 4 keys of ONE query, so
//   * the per-query max/sum need only 2 cross-lane steps (lanes l^16, l^32),
//   * the S^T registers, split, are already P^T's B operand for the next product
//     (k slot 8g + 4u + r is key 16u + 4g + r), and
//   * the running-output rescale is one scalar per lane.
// Everything accumulates in FP32; keys are visited in ascending blocks within one,
// two or four parts chosen from the shape, so a shape's results are always the
// same bits, whatever else runs on the device.
#include "ctmr_common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace ctmr {
namespace {

constexpr int kHeadDim = 32;
constexpr int kWaves = 8;     // waves per workgroup
constexpr int kKeyTiles = 2;  // 16-key tiles per key block
constexpr int kBlock = 16 * kKeyTiles;
constexpr float kLazyMax = 8.0f;  // log2 headroom before the softmax reference max moves

struct AttnArgs {
  const float* q;
  const float* k;
  const float* v;
  float* out;
  int64_t ldq, ldk, ldv, ldo;
  int lq, lk, heads;
  float qscale;  // scale * log2(e)
};

// Maximum over lanes l, l^16, l^32, l^48 (the four lane groups holding one
// query's scores): v_permlane16_swap / v_permlane32_swap of a value with
// itself yield the pair {x[l], x[l^16]} / {x[l], x[l^32]} (VALU, no LDS round
// trip as with ds_bpermute).
__device__ __forceinline__ float lane_group_max(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

// Keys of every part but the last of a split in KS: an equal share, rounded up
// to whole key blocks, so only the last block is ragged (halves to 64 keys).
template <int KS>
__device__ __forceinline__ int attention_part_keys(int lk) {
  constexpr int kUnit = KS == 2 ? 64 : kBlock;
  return ((lk + KS - 1) / KS + kUnit - 1) / kUnit * kUnit;
}

// Whether a wave's staging piece j of KS (flash_attention_kernel) is of K.
template <int KS>
__device__ __forceinline__ bool wave_piece_is_k(int wave, int j) {
  return KS == 1 ? wave < kWaves / 2 : j < KS / 2;
}

// Online softmax of one 32-key block, shared by both kernels: scores -> P^T in
// place, running reference max m and sum l, and the factor alpha the outputs
// must be scaled by before this block's P V products.  A lane holds keys
// 16u + 4g + r (u < 2, r < 4) of its query.  The reference m[t] of a query
// moves only when the block's max exceeds it by more than kLazyMax (in log2
// units; always on the first block, where m = -inf): P = 2^(s - m) then stays
// below 2^8, and in most blocks alpha is exactly 1, so the output rescale is
// skipped (output / sum is the same quotient for any reference).  The decision
// is per query, so every tiling computes the same bits.  RAGGED masks keys at
// or past k_end (the last block only).
template <bool RAGGED>
__device__ __forceinline__ void block_softmax(f4 (&s)[kKeyTiles], float& m, float& l, float& alpha, int k0, int k_end,
                                              int g) {
  if constexpr (RAGGED) {
#pragma unroll
    for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (k0 + u * 16 + 4 * g + r >= k_end) s[u][r] = -INFINITY;
  }
  float bm = s[0][0];
#pragma unroll
  for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) bm = fmaxf(bm, s[u][r]);
  bm = lane_group_max(bm);
  // Every block holds at least one real key, so bm is finite and the first
  // block moves the reference (alpha = 2^-inf = 0).  Arguments are <= 8:
  // the hardware exp2 (v_exp_f32) differs from exp2f only below 2^-126,
  // far under the resolution of the running sum (>= 1).
  const bool move = bm > m + kLazyMax;
  const float mn = move ? bm : m;
  alpha = move ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;
  m = mn;
  float ps = 0.f;
#pragma unroll
  for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = __builtin_amdgcn_exp2f(s[u][r] - mn);
      s[u][r] = p;
      ps += p;
    }
  l = l * alpha + ps;
}

// Operand schemes of flash_attention_kernel.
//  * kFp32: q, k, v and P as three bf16 parts h, m, l that together hold an
//    fp32 value's 24 bits (split_bf16x3), the six part products at or above
//    2^-17 of the full one on bf16 MFMA (FP32 MFMA runs at a sixteenth of its
//    rate).  Rows with an output outside what the parts hold (part_sum_keep) are
//    computed again on FP32 MFMA (attention_rerun).
//  * kF16x2: the reference's split-fp16 arithmetic (_flash_attention.py:
//    140-290, 314-317): hi = fp16(x), lo = fp16((x - hi) * 2^11) of q (after
//    scale * log2(e)), k, v and P, with
//      S = Kh Qh + (Kh Ql + Kl Qh) * 2^-11          (per 32-key block)
//      O = Vh Ph + (Vh Pl + Vl Ph) * 2^-11
//    the cross terms of O kept in their own accumulator over all key blocks
//    and added at the end, as the reference does.
constexpr int kFp32 = 3, kF16x2 = 2;  // the value is the number of parts

constexpr int kThreads = 64 * kWaves;
constexpr int kRow = 96;                   // LDS bytes of a 32-value row (64 used): conflict-free b128 reads of 16 rows
constexpr int kPlane = kBlock * kRow;      // one part of one operand of a key block

// The parts of four values, 8 bytes each.
template <int SCH>
__device__ __forceinline__ void split_parts(f4 v, uint2 (&p)[SCH]) {
  if constexpr (SCH == kFp32) {
    split_bf16x3(v, p[0], p[1], p[2]);
  } else {
    h4 hi, lo;
    split_f16x4(v, hi, lo);
    p[0] = __builtin_bit_cast(uint2, hi);
    p[1] = __builtin_bit_cast(uint2, lo);
  }
}

template <int SCH>
__device__ __forceinline__ f4 mfma32(const u4& a, const u4& b, f4 c) {
  if constexpr (SCH == kFp32)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// The six part products of one MFMA tile, smallest first.
__device__ __forceinline__ f4 mfma_x3(const u4 (&a)[3], const u4 (&b)[3], f4 c) {
  c = mfma32<kFp32>(a[2], b[0], c);
  c = mfma32<kFp32>(a[0], b[2], c);
  c = mfma32<kFp32>(a[1], b[1], c);
  c = mfma32<kFp32>(a[1], b[0], c);
  c = mfma32<kFp32>(a[0], b[1], c);
  return mfma32<kFp32>(a[0], b[0], c);
}

// A wave's 16 queries over all keys as fp32 products on FP32 MFMA
// (v_mfma_f32_16x16x4_f32), keys and values straight from memory: for waves with
// an output that the part products do not hold (part_sum_keep).  One NaN or infinity among the keys reaches
// every query of its head, so the cost must stay a few times the finite one.
// Two passes, the scores' maximum and then the probabilities, so that a score of
// -inf is a key without weight wherever it stands.  S^T product j takes dims j
// and 4 + j ... of each lane group g's dims 8g .. 8g + 7, P V product (u, r) the
// keys 16u + 4g + r.  q: this lane's query row; out: dims 4g + r and 16 + 4g + r.
template <typename Rows>
__device__ __forceinline__ void attention_rerun(const AttnArgs& a, const float* q, const float* K, const float* V,
                                                Rows rows_rsrc, int col, int g, f4 (&out)[2]) {
  f4 qv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) qv[i] = *reinterpret_cast<const f4*>(q + 8 * g + 4 * i) * a.qscale;
  auto scores = [&](int k0, f4 (&s)[kKeyTiles]) {
    const __amdgpu_buffer_rsrc_t rk = rows_rsrc(K, a.ldk, k0);
#pragma unroll
    for (int u = 0; u < kKeyTiles; ++u) {
      const int row = min(u * 16 + col, a.lk - k0);  // rows past the end: zeros
      const int off = (int)(((int64_t)row * a.ldk + 8 * g) * 4);
      f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const f4 kv = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rk, off + 16 * i, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[e], qv[i][e], acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) s[u][r] = k0 + u * 16 + 4 * g + r < a.lk ? acc[r] : -INFINITY;
    }
  };
  float m = -INFINITY;
#pragma clang loop unroll(disable)
  for (int k0 = 0; k0 < a.lk; k0 += kBlock) {
    f4 s[kKeyTiles];
    scores(k0, s);
#pragma unroll
    for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) m = fmaxf(m, s[u][r]);
  }
  m = lane_group_max(m);
  float l = 0.f;
  out[0] = out[1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
  for (int k0 = 0; k0 < a.lk; k0 += kBlock) {
    f4 s[kKeyTiles];
    scores(k0, s);
    const __amdgpu_buffer_rsrc_t rv = rows_rsrc(V, a.ldv, k0);
#pragma unroll
    for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = u * 16 + 4 * g + r;
        const float pr = k0 + key < a.lk ? __builtin_amdgcn_exp2f(s[u][r] - m) : 0.f;
        l += pr;
        const int off = (int)(((int64_t)min(key, a.lk - k0) * a.ldv + col) * 4);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          out[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, off + 64 * j, 0, 0)), pr, out[j], 0, 0, 0);
      }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
#pragma unroll
  for (int j = 0; j < 2; ++j) out[j] *= 1.0f / l;
}

// A workgroup of eight waves: KS key parts x (8 / KS) query groups of 16
// queries (KS = 2 or 4 for small grids: part p takes the keys from
// p * attention_part_keys on).  Each step the threads of a part load a 32-key
// block of K and V as fp32, split it once for all the part's waves and publish
// it in LDS in MFMA operand order (K rows of 32 dims; V transposed, 32 dims x
// 32 keys in P^T's k order), one block ahead, one barrier a step.  The fp32
// loads of the next block, or of the next two with key parts, are in flight
// during a step.
// Sharing the blocks is what the time followed: with every wave loading its
// own operands the kernel took as long on fp16 MFMA as on FP32 MFMA, and 16
// queries a wave 1.6 times 32 queries a wave at any occupancy.  Measured, that
// form (its separate split pass included) / this one us: 2048 tokens x 8 heads
// x 2 fp32 87 / 70, split fp16 86 / 53; 4158 x 8 244 / 173, 237 / 143; 4800 x
// 16 553 / 334, 500 / 263.  Now bound by a step's chain (barrier, LDS reads,
// S^T, softmax, split, P V), which four waves a SIMD cover in part: VALU issues
// in 54 % of the cycles (168 operations a wave and block), the MFMAs take 30 %
// (fp32) or 19 %, LDS bank conflicts 16 %.  32 queries a wave halve the LDS
// reads but leave half the waves: 67, 70; 193, 177 us.
// A small grid is bound by the latency of its steps: 1024 tokens x 8 heads 16.2
// / 15.2, 33.4 / 13.8; 256 x 16 x 2 7.2 / 7.8, 13.4 / 6.8 (with two parts and
// one block in flight 21.6, 18.8; 8.8, 7.6).
template <int SCH, int KS>
__global__ __launch_bounds__(kThreads, SCH == kFp32 && KS == 1 ? 6 : 4) void flash_attention_kernel(AttnArgs a) {
  static_assert(KS == 1 || KS == 2 || KS == 4, "one, two or four key parts");
  constexpr int kGroups = kWaves / KS, kPartThreads = kThreads / KS;
  constexpr int kAhead = KS == 1 ? 1 : 2;  // blocks in registers beyond the one in LDS
  constexpr int kBuf = 2 * SCH * kPlane;  // K planes, then V planes
  constexpr int NO = SCH == kF16x2 ? 4 : 2;  // output accumulators per query tile
  __shared__ __attribute__((aligned(16))) char lds[2][KS][kBuf];
  static_assert(kGroups * (KS - 1) * (2 + 4 * NO) * 64 * 4 <= 2 * KS * kBuf, "the hand-over fits");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int b = blockIdx.y / a.heads, h = blockIdx.y % a.heads;
  const int part = wave / kGroups, group = wave % kGroups;
  const int q0 = (blockIdx.x * kGroups + group) * 16;
  // Wave-uniform.  Every wave reaches every barrier: a query group past the
  // end runs on clamped rows and stores nothing.
  const int part_keys = KS == 1 ? a.lk : attention_part_keys<KS>(a.lk);
  const int k_begin = min(a.lk, part * part_keys), k_end = min(a.lk, k_begin + part_keys);
  const int steps = (min(part_keys, a.lk) + kBlock - 1) / kBlock;  // part 0's, the most of any part

  const float* Q = a.q + (int64_t)b * a.lq * a.ldq + h * kHeadDim;
  const float* K = a.k + (int64_t)b * a.lk * a.ldk + h * kHeadDim;
  const float* V = a.v + (int64_t)b * a.lk * a.ldv + h * kHeadDim;
  // K and V rows of a key block through a buffer descriptor built per block
  // from wave-uniform values: base = row k0, range = the rows left before lk,
  // so rows at or past lk read as zero (masked below).  The host keeps lk * ld
  // * 4 within 31 bits.
  auto rows_rsrc = [&](const float* base, int64_t ld, int k0) {
    const int64_t left = (int64_t)max(a.lk - k0, 0) * ld * 4;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)min(k0, a.lk) * ld), (short)0, (int)left,
                                             0x00020000);
  };
  // Staging: a part's 512 pieces of four values, KS per thread.  Piece i < 256
  // is dims 4 (i % 8) .. +3 of key i / 8; piece 256 + i is dim i % 32 of the
  // keys 4 (i / 32) .. +3, which are slots 8 g' + 4 u .. +3 of V^T's k order
  // (u = i / 128, g' = (i / 32) % 4: P^T's k slot 8 g + 4 u + r is key 16 u +
  // 4 g + r).
  const int st = threadIdx.x % kPartThreads;
  // Rows past lk take row lk's offset, out of range: where lk < 32 a row of the
  // block can lie past 2^32 bytes, and its offset must not wrap into the range.
  unsigned goff[KS];
  int loff[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j) {
    const int id = st + j * kPartThreads;
    if (id < 256) {
      goff[j] = (unsigned)(((int64_t)min(id >> 3, a.lk) * a.ldk + 4 * (id & 7)) * 4);
      loff[j] = (id >> 3) * kRow + 8 * (id & 7);
    } else {
      const int i = id - 256, kq = i >> 5;
      goff[j] = (unsigned)(((int64_t)min(4 * kq, a.lk) * a.ldv + (i & 31)) * 4);
      loff[j] = SCH * kPlane + (i & 31) * kRow + 16 * (kq & 3) + 8 * (kq >> 2);
    }
  }
  const unsigned vrow = (unsigned)(a.ldv * 4);
  auto fetch = [&](int k0, f4 (&raw)[KS]) {
    const __amdgpu_buffer_rsrc_t rk = rows_rsrc(K, a.ldk, k0), rv = rows_rsrc(V, a.ldv, k0);
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      if (wave_piece_is_k<KS>(wave, j)) {  // wave-uniform
        raw[j] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rk, (int)goff[j], 0, 0));
      } else {
        unsigned off = goff[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          raw[j][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, (int)off, 0, 0));
          off = __builtin_elementwise_add_sat(off, vrow);
        }
      }
    }
  };
  auto publish = [&](char* buf, const f4 (&raw)[KS]) {
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      uint2 p[SCH];
      split_parts<SCH>(raw[j], p);
#pragma unroll
      for (int i = 0; i < SCH; ++i) *reinterpret_cast<uint2*>(buf + loff[j] + i * kPlane) = p[i];
    }
  };

  // The first blocks and Q in one round of latency.
  f4 raw0[KS], raw[kAhead][KS];
  fetch(k_begin, raw0);
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(k_begin + (1 + i) * kBlock, raw[i]);

  // Q^T as the B operand of S^T = K Q^T: query q0 + col, dims 8g .. 8g+7.
  u4 qf[SCH];
  {
    const f4* p = reinterpret_cast<const f4*>(Q + (int64_t)min(q0 + col, a.lq - 1) * a.ldq + 8 * g);
    f4 v0 = p[0] * a.qscale, v1 = p[1] * a.qscale;
    // opaque: the scaled values are rounded to fp32 before they are split
    asm volatile("" : "+v"(v0), "+v"(v1));
    uint2 p0[SCH], p1[SCH];
    split_parts<SCH>(v0, p0);
    split_parts<SCH>(v1, p1);
#pragma unroll
    for (int i = 0; i < SCH; ++i) qf[i] = u4{p0[i].x, p0[i].y, p1[i].x, p1[i].y};
  }

  // acc[0..1]: dims 16j + 4g + r; split fp16: acc[2..3] the 2^11-scaled cross
  // terms.
  f4 acc[NO];
#pragma unroll
  for (int j = 0; j < NO; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f, alpha;

  const int rd = col * kRow + 16 * g;  // this lane's 16 bytes of row `col`
  // One key block from `buf`: S^T, the softmax, the split of P, P V.
  auto block = [&](const char* buf, int k0, auto ragged) {
    f4 s[kKeyTiles];
#pragma unroll
    for (int u = 0; u < kKeyTiles; ++u) {
      u4 kf[SCH];
#pragma unroll
      for (int i = 0; i < SCH; ++i) kf[i] = *reinterpret_cast<const u4*>(buf + i * kPlane + u * 16 * kRow + rd);
      const f4 z = {0.f, 0.f, 0.f, 0.f};
      if constexpr (SCH == kFp32) {
        s[u] = mfma_x3(kf, qf, z);
      } else {
        const f4 hh = mfma32<SCH>(kf[0], qf[0], z);
        f4 cr = mfma32<SCH>(kf[0], qf[1], z);
        cr = mfma32<SCH>(kf[1], qf[0], cr);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[u][r] = fmaf(cr[r], 1.0f / 2048.0f, hh[r]);
      }
    }
    block_softmax<decltype(ragged)::value>(s, m, l, alpha, k0, k_end, g);
    // acc *= alpha, skipped (same bits: every factor is exactly 1) unless a
    // lane of the wave moved its reference.
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int j = 0; j < NO; ++j) acc[j] *= alpha;
    }
    u4 pf[SCH];
    if constexpr (SCH == kFp32) {
      uint2 p0[SCH], p1[SCH];
      split_parts<SCH>(s[0], p0);
      split_parts<SCH>(s[1], p1);
#pragma unroll
      for (int i = 0; i < SCH; ++i) pf[i] = u4{p0[i].x, p0[i].y, p1[i].x, p1[i].y};
    } else {
      h8 ph, pl;
#pragma unroll
      for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) ph[4 * u + r] = (_Float16)s[u][r];
      // The low halves below read hi from these packed registers (an opaque
      // copy: otherwise the compiler converts each p to fp16 a second time).
      asm volatile("" : "+v"(ph));
      // lo = fp16((p - hi) * 2^11) = fp16(2^11 p - 2^11 hi): both products and
      // their difference are exact in fp32, so one rounding of the fused form
      // (v_fma_mix) gives the same half.
#pragma unroll
      for (int u = 0; u < kKeyTiles; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          pl[4 * u + r] = (_Float16)__builtin_fmaf((float)ph[4 * u + r], -2048.0f, s[u][r] * 2048.0f);
      pf[0] = __builtin_bit_cast(u4, ph);
      pf[1] = __builtin_bit_cast(u4, pl);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u4 vf[SCH];
#pragma unroll
      for (int i = 0; i < SCH; ++i)
        vf[i] = *reinterpret_cast<const u4*>(buf + (SCH + i) * kPlane + j * 16 * kRow + rd);
      if constexpr (SCH == kFp32) {
        acc[j] = mfma_x3(vf, pf, acc[j]);
      } else {
        acc[j] = mfma32<SCH>(vf[0], pf[0], acc[j]);
        acc[2 + j] = mfma32<SCH>(vf[0], pf[1], acc[2 + j]);
        acc[2 + j] = mfma32<SCH>(vf[1], pf[0], acc[2 + j]);
      }
    }
  };

  publish(lds[0][part], raw0);
  auto step = [&](int i, f4 (&ahead)[KS]) {
    // Block i is published, and every wave is done with block i - 1, whose
    // buffer takes block i + 1 (past the part's keys: other keys or zeros,
    // never used).
    lds_barrier();
    publish(lds[(i + 1) & 1][part], ahead);
    const int k0 = k_begin + i * kBlock;
    fetch(k0 + (1 + kAhead) * kBlock, ahead);
    if (k0 + kBlock <= k_end) block(lds[i & 1][part], k0, std::false_type{});
    else if (k0 < k_end) block(lds[i & 1][part], k0, std::true_type{});
  };
  for (int i = 0; i < steps; i += kAhead) {
    step(i, raw[0]);
    if constexpr (kAhead == 2) {
      if (i + 1 < steps) step(i + 1, raw[1]);
    }
  }

  if constexpr (KS > 1) {
    // The later parts' waves hand their running max, sum and accumulators to
    // the first's, which rescales and adds them part by part, ascending.
    constexpr int kSlot = (2 + 4 * NO) * 64;  // one wave's
    float* const xch = reinterpret_cast<float*>(&lds[0][0][0]) + group * (KS - 1) * kSlot + lane;
    lds_barrier();
    if (part > 0) {
      float* o = xch + (part - 1) * kSlot;
      o[0] = m;
      o[64] = l;
#pragma unroll
      for (int j = 0; j < NO; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[(2 + 4 * j + e) * 64] = acc[j][e];
    }
    lds_barrier();
    if (part > 0) return;
#pragma unroll
    for (int k = 0; k < KS - 1; ++k) {
      const float* o = xch + k * kSlot;
      const float m1 = o[0];
      const float mm = fmaxf(m, m1);  // the first part always holds keys: finite
      const float a0 = exp2f(m - mm), a1 = exp2f(m1 - mm);  // a1 = 0 for an empty part
      m = mm;
      l = l * a0 + o[64] * a1;
#pragma unroll
      for (int j = 0; j < NO; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = acc[j][e] * a0 + o[(2 + 4 * j + e) * 64] * a1;
    }
  }

  // The four lane groups hold partial sums of the same query; xor pairs add
  // commutatively, so every lane ends with the same bits.
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  const float inv = 1.0f / l;
  const int query = q0 + col;
  f4 o[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    o[j] = acc[j];
    if constexpr (SCH == kF16x2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[j][r] = acc[j][r] + acc[2 + j][r] * (1.0f / 2048.0f);
    }
    o[j] *= inv;
  }
  if constexpr (SCH == kFp32) {
    PartSumTest test;
#pragma unroll
    for (int e = 0; e < 8; ++e) test.add(o[e >> 2][e & 3]);
    const bool bad = test.any();
    if (__any(bad && query < a.lq)) {
      f4 again[2];
      attention_rerun(a, Q + (int64_t)min(query, a.lq - 1) * a.ldq, K, V, rows_rsrc, col, g, again);
      if (bad) {
        o[0] = again[0];
        o[1] = again[1];
      }
    }
  }
  if (query >= a.lq) return;
  float* const dst = a.out + ((int64_t)b * a.lq + query) * a.ldo + h * kHeadDim;
  *reinterpret_cast<f4*>(dst + 4 * g) = o[0];       // dims 4g .. 4g+3
  *reinterpret_cast<f4*>(dst + 16 + 4 * g) = o[1];  // dims 16 + 4g .. 16 + 4g+3
}

template <int SCH, int KS>
int launch_attention(const AttnArgs& a, int n, hipStream_t stream) {
  const int64_t per_block = (int64_t)(kWaves / KS) * 16;
  dim3 grid((unsigned)ceil_div(a.lq, per_block), (unsigned)(n * a.heads));
  hipLaunchKernelGGL((flash_attention_kernel<SCH, KS>), grid, dim3(kThreads), 0, stream, a);
  return check_launch("flash_attention_kernel");
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

// Key parts, from the shape only: two when there are at least 128 keys and the
// grid of two parts stays under two rounds of 512 workgroups; four when their
// grid, 32 queries a workgroup, leaves every workgroup a CU of its own.
// Measured, one / two parts us: 4158 tokens x 8 heads 210 / 178 (fp32), 160 /
// 144 (split fp16); 3000 x 16 154 / 137, 118 / 110.  Two / four: 512 x 8 12.8 /
// 9.6, 11.2 / 8.8; 648 x 8 16.6 / 12.3, 14.7 / 11.2.
int attention_key_parts(int n, int lq, int lk, int heads) {
  if (lk < 128) return 1;
  if (ceil_div(lq, 32) * n * heads <= 256) return 4;
  return ceil_div(lq, 64) * n * heads < 1024 ? 2 : 1;
}

}  // namespace ctmr

namespace ctmr {
namespace {

// Argument checks shared by both entry points (messages name the caller).
int check_attn(const ctmr_attn_desc* d, const float* q, const float* k, const float* v, const float* out,
               const char* fn) {
  if (!d || !q || !k || !v || !out) {
    set_error("%s: null argument", fn);
    return CTMR_E_INVALID;
  }
  if (d->head_dim != kHeadDim) {
    set_error("%s: head_dim %d unsupported (32 only)", fn, d->head_dim);
    return CTMR_E_UNSUPPORTED;
  }
  const char* bad = nullptr;
  int code = CTMR_E_INVALID;
  const int64_t width = (int64_t)d->heads * kHeadDim;
  if (d->query_tiles < 0 || d->query_tiles > 2)
    bad = "query_tiles must be 0, 1 or 2";
  else if (d->n < 1 || d->lq < 1 || d->lk < 1 || d->heads < 1)
    bad = "n, lq, lk and heads must be >= 1";
  else if ((int64_t)d->n * d->heads > 65535)
    bad = "n * heads exceeds 65535";
  else if (d->ldq < width || d->ldk < width || d->ldv < width || d->ldo < width)
    bad = "row stride below heads * head_dim";
  else if ((d->ldq | d->ldk | d->ldv | d->ldo) & 3)
    bad = "row strides must be multiples of 4 floats";
  else if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out))
    bad = "q, k, v and out must be 16-byte aligned";
  else if ((int64_t)d->lk * std::max(d->ldk, d->ldv) * 4 > 0x7fffffffll)
    bad = "lk * row stride exceeds 2^31 bytes", code = CTMR_E_UNSUPPORTED;
  else if (!std::isfinite(d->scale))
    bad = "scale must be finite";
  if (bad) {
    set_error("%s: %s", fn, bad);
    return code;
  }
  return CTMR_OK;
}

template <int SCH>
int run_attention(const ctmr_attn_desc* d, const float* q, const float* k, const float* v, float* out, void* stream) {
  const AttnArgs a{q, k, v, out, d->ldq, d->ldk, d->ldv, d->ldo, d->lq, d->lk, d->heads,
                   (float)((double)d->scale * 1.4426950408889634)};
  hipStream_t st = (hipStream_t)stream;
  switch (attention_key_parts(d->n, d->lq, d->lk, d->heads)) {
    case 1: return launch_attention<SCH, 1>(a, d->n, st);
    case 2: return launch_attention<SCH, 2>(a, d->n, st);
    default: return launch_attention<SCH, 4>(a, d->n, st);
  }
}

// What ctmr_flash_attention_f16x2_workspace_bytes answers, and the least a
// caller's workspace must hold: six fp16 planes (Q, K and V, hi and lo), each in
// whole 256 bytes.  Nothing is written to it.
int64_t split_workspace_bytes(const ctmr_attn_desc* d) {
  const int64_t items = (int64_t)d->n * d->heads * kHeadDim * 2;
  return 2 * round_up(items * d->lq, 256) + 4 * round_up(items * round_up(d->lk, kBlock), 256);
}

}  // namespace
}  // namespace ctmr

extern "C" int ctmr_flash_attention(const ctmr_attn_desc* d, const float* q, const float* k, const float* v,
                                    float* out, void* stream) {
  using namespace ctmr;
  if (const int rc = check_attn(d, q, k, v, out, "ctmr_flash_attention")) return rc;
  return run_attention<kFp32>(d, q, k, v, out, stream);
}

extern "C" int64_t ctmr_flash_attention_f16x2_workspace_bytes(const ctmr_attn_desc* d) {
  using namespace ctmr;
  if (!d || d->n < 1 || d->lq < 1 || d->lk < 1 || d->heads < 1) return -1;
  return split_workspace_bytes(d);
}

extern "C" int ctmr_flash_attention_f16x2(const ctmr_attn_desc* d, const float* q, const float* k, const float* v,
                                          float* out, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace ctmr;
  if (const int rc = check_attn(d, q, k, v, out, "ctmr_flash_attention_f16x2")) return rc;
  const int64_t need = split_workspace_bytes(d);
  const bool none = !workspace && workspace_bytes == 0;
  if (!none && (!workspace || workspace_bytes < need)) {
    set_error("ctmr_flash_attention_f16x2: workspace of %lld bytes needed, %lld given", (long long)need,
              (long long)(workspace ? workspace_bytes : 0));
    return CTMR_E_INVALID;
  }
  if (((uintptr_t)workspace & 255u) != 0)
    return fail(CTMR_E_INVALID, "ctmr_flash_attention_f16x2: workspace must be 256-byte aligned");
  return run_attention<kF16x2>(d, q, k, v, out, stream);
}
