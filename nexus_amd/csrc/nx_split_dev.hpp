// nx_split_dev.hpp — operands of the split-activation MFMA kernels
// (nx_mfv.hip, nx_mfd.hip): f32 activations as two fp16 halves against
// quantized codes that enter the matrix cores as exact fp16 values.
#pragma once

#include "nx_device.hpp"
#include "nx_internal.hpp"

namespace nx {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 4 x 4 transpose of dwords across the four 16-lane groups: on return
// c[k] of lane group g holds what c[g] of lane group k held (register
// swaps between lane halves, then between neighbouring lane groups)
__device__ __forceinline__ void transpose_groups(uint32_t (&c)[4]) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const auto v = __builtin_amdgcn_permlane32_swap(c[k], c[k + 2], false, false);
    c[k] = v[0];
    c[k + 2] = v[1];
  }
#pragma unroll
  for (int k = 0; k < 4; k += 2) {
    const auto v = __builtin_amdgcn_permlane16_swap(c[k], c[k + 1], false, false);
    c[k] = v[0];
    c[k + 1] = v[1];
  }
}

// a DPP move within a row of 16 lanes
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// (q - 8) sc for the 8 codes of a dword holding q ^ 8, times 2^-14 (2^10 in
// the scales) or any 2^k that keeps |.| fp16: s1 = {sc 2^(24+k)}, s16 = s1 / 16,
// off = {-8 sc 2^k}
__device__ __forceinline__ f16x8 operand4(uint32_t cw, f16x2 s1, f16x2 s16, f16x2 off) {
  cw ^= 0x88888888u;
  const uint32_t c8 = cw >> 8;
  const f16x2 a = __builtin_bit_cast(f16x2, cw & 0x000F000Fu) * s1 + off;
  const f16x2 b = __builtin_bit_cast(f16x2, cw & 0x00F000F0u) * s16 + off;
  const f16x2 c = __builtin_bit_cast(f16x2, c8 & 0x000F000Fu) * s1 + off;
  const f16x2 d = __builtin_bit_cast(f16x2, c8 & 0x00F000F0u) * s16 + off;
  // a: elements 0, 2; c: 1, 3; b: 4, 6; d: 5, 7 (nibble 2 i of the dword is
  // element i, nibble 2 i + 1 element 4 + i)
  return f16x8{a[0], a[1], c[0], c[1], b[0], b[1], d[0], d[1]};
}

// n sc for the 8 unsigned codes of a dword, scaled as above
__device__ __forceinline__ f16x8 operand4u(uint32_t cw, f16x2 s1, f16x2 s16) {
  const uint32_t c8 = cw >> 8;
  const f16x2 a = __builtin_bit_cast(f16x2, cw & 0x000F000Fu) * s1;
  const f16x2 b = __builtin_bit_cast(f16x2, cw & 0x00F000F0u) * s16;
  const f16x2 c = __builtin_bit_cast(f16x2, c8 & 0x000F000Fu) * s1;
  const f16x2 d = __builtin_bit_cast(f16x2, c8 & 0x00F000F0u) * s16;
  return f16x8{a[0], a[1], c[0], c[1], b[0], b[1], d[0], d[1]};
}

// q 2^-9 for the 8 signed bytes of two code dwords, in element order
__device__ __forceinline__ f16x8 operand8(uint32_t lo, uint32_t hi) {
  lo ^= 0x80808080u;
  hi ^= 0x80808080u;
  const f16x2 s = {32768.0f16, 32768.0f16}, off = {-0.25f16, -0.25f16};
  const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(lo, lo, 0x0C010C00u)) * s + off;
  const f16x2 b = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(lo, lo, 0x0C030C02u)) * s + off;
  const f16x2 c = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(hi, hi, 0x0C010C00u)) * s + off;
  const f16x2 d = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(hi, hi, 0x0C030C02u)) * s + off;
  return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// One row's chunk of 256 activations, in the 16 lanes of a row (lane j16 holds
// elements 64 q + 4 j16 .. + 3 in v[q]), as fp16 halves hi + lo scaled into
// [2^13, 2^14) by a power of two; returns the factor that takes the scale off.
// put(u, g, half, hi, lo): this lane's four values, half `half` of the operand
// of MFMA u, lane group g, in the order of operand4 (Q8_0: operand8).  The
// elements of (u, g): Q4_K 32 g + 8 u (u < 4) or 128 + 32 g + 8 (u - 4), the
// dwords of sub-blocks g and g + 4; Q2_K 64 g + 8 u, segment g; Q4_0 and Q8_0
// 32 u + 8 g, a quarter of block u.
// put_sum(g, i, hl): for the min term, the sub-block sum that is value i of
// lane group g, X 2^-6 as (hi, lo): Q4_K sub-blocks g and g + 4, Q2_K the four
// of segment g.  (Several lanes put the same sum.)
template <int FMT, typename Put, typename PutSum>
__device__ __forceinline__ float split16(const f32x4 (&v)[4], int j16, Put put, PutSum put_sum) {
  constexpr bool Q4K = FMT == NX_FMT_Q4_K, Q2K = FMT == NX_FMT_Q2_K, Q80 = FMT == NX_FMT_Q8_0;
  float mx = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    // (fmaxf would first quiet each operand: two more instructions per pair)
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(v[q].x), "v"(v[q].y));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(v[q].z), "v"(v[q].w));
  }
  mx = fmaxf(mx, dpp_f<0x128>(mx));  // row_ror 8, 4, 2, 1
  mx = fmaxf(mx, dpp_f<0x124>(mx));
  mx = fmaxf(mx, dpp_f<0x122>(mx));
  mx = fmaxf(mx, dpp_f<0x121>(mx));
  // max|x| < 2^E; an infinity or NaN ends as NaN through x' - hi or hi
  int E = mx < INFINITY ? __builtin_amdgcn_frexp_expf(mx) : 0;
  E = max(E, -112);  // 2^126 and 2^-126 at most: smaller maxima keep their bits down to 2^-126
  const float up = __builtin_amdgcn_ldexpf(1.0f, 14 - E);
  const int kd = (j16 >> 1) & 3, s0 = j16 >> 3;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f16x2 h[2], l[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      // operand order of a 4-bit dword's half: elements 0, 2, 1, 3
      const int e0 = Q80 ? 2 * i : i, e1 = Q80 ? 2 * i + 1 : i + 2;
      h[i] = f16x2{(_Float16)(v[q][e0] * up), (_Float16)(v[q][e1] * up)};
      asm("" : "+v"(h[i]));  // converted once: l reads the packed halves
      l[i] = f16x2{(_Float16)fmaf(v[q][e0], up, -(float)h[i][0]),
                   (_Float16)fmaf(v[q][e1], up, -(float)h[i][1])};
    }
    // elements 64 q + 4 j16 .. + 3 are half j16 % 2 of dword kd of 32-element
    // sub-block s
    const int s = 2 * q + s0;
    const int u = Q4K ? 4 * (s >> 2) + kd : Q2K ? 4 * s0 + kd : s;
    const int g = Q4K ? s & 3 : Q2K ? q : kd;
    put(u, g, j16 & 1, f16x4{h[0][0], h[0][1], h[1][0], h[1][1]},
        f16x4{l[0][0], l[0][1], l[1][0], l[1][1]});
    if constexpr (Q4K || Q2K) {
      // the sub-block's lanes: quad pairs, quads (16 elements), the half row
      float X = fmaf(v[q].y, up, v[q].x * up);
      X = fmaf(v[q].w, up, fmaf(v[q].z, up, X));
      X += dpp_f<0xB1>(X);
      X += dpp_f<0x4E>(X);
      if constexpr (Q4K) X += dpp_f<0x141>(X);
      const float xq = X * 0.015625f;  // |X| <= 32 x 2^14
      const _Float16 xh = (_Float16)xq;
      put_sum(g, Q4K ? s >> 2 : j16 >> 2, f16x2{xh, (_Float16)(xq - (float)xh)});
    }
  }
  return __builtin_amdgcn_ldexpf(1.0f, E - 14);
}

// One row's chunk of activations as operands: value p of MFMA u, lane group g
// at 16 ((2 u + (hi 0, lo 1)) 4 + g) + 2 p, so the four lane groups of a row
// read 64 contiguous bytes; then the min term's operands (8 bytes per lane
// group in Q4_K, 16 in Q2_K) and the unscale factor.
constexpr int REC_XM = 1024, REC_SX = 1088;
static_assert(REC_SX + 64 == REC_BYTES, "a record is whole 128-byte lines");

// the record of one (row, chunk), written by its 16 lanes
template <int FMT>
__device__ __forceinline__ void write_record(uint8_t *rec, const f32x4 (&v)[4], int j16) {
  const float un = split16<FMT>(
      v, j16,
      [&](int u, int g, int half, f16x4 h, f16x4 l) {
        uint8_t *o = rec + 128 * u + 16 * g + 8 * half;
        *reinterpret_cast<f16x4 *>(o) = h;
        *reinterpret_cast<f16x4 *>(o + 64) = l;
      },
      [&](int g, int i, f16x2 hl) {
        *reinterpret_cast<f16x2 *>(rec + REC_XM + (FMT == NX_FMT_Q2_K ? 16 : 8) * g + 4 * i) = hl;
      });
  *reinterpret_cast<float *>(rec + REC_SX) = un;
}

// row i of a split job (x [n][256] -> n records), in 16 lanes
template <int FMT>
__device__ __forceinline__ void split_row(const SplitJob &job, size_t i) {
  const int j = threadIdx.x & 15;
  const float *src = job.x + min(i, job.n - 1) * 256 + 4 * j;
  f32x4 v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const f32x4 *>(src + 64 * q);
  if (i < job.n) write_record<FMT>(job.rec + i * REC_BYTES, v, j);  // all 16 lanes or none
}
__device__ __forceinline__ void split_rows(const SplitJob &job, size_t i) {
  if (job.fmt == NX_FMT_Q4_K)
    split_row<NX_FMT_Q4_K>(job, i);
  else if (job.fmt == NX_FMT_Q8_0)
    split_row<NX_FMT_Q8_0>(job, i);
  else if (job.fmt == NX_FMT_Q2_K)
    split_row<NX_FMT_Q2_K>(job, i);
  else
    split_row<NX_FMT_Q4_0>(job, i);
}

}  // namespace nx
