// nx_mfd.hip — dense matvec of several tokens on MFMA for Q4_K, Q4_0 and
// Q8_0 matrices (InferenceEngine::matvec, src/engine/mod.rs:775-801, on the
// q/k/v/o projections and the output head of a batch or a prompt).
//
// The decode GEMV costs about one instruction per weight and token, so
// beyond a few tokens its time grows with the tokens and it re-reads the
// matrix per token group: 4096 x 4096 Q4_K took 869 us for 509 tokens.  Here
// the products run on the matrix cores at the GEMV's precision:
//
//   - Codes are exact fp16 values: a nibble pair of a code dword masked in
//     place is the subnormal n 2^-24 (or 16 n 2^-24) per 16-bit half, and one
//     packed fma makes (n - 8) sc 2^-14 of it (Q4_0: 2^-9), at most 9 bits.
//     Q8_0's bytes likewise, (q + 128) 2^-24 to q 2^-9.  The operands must be
//     normal numbers: the MFMA aligns products by the exponents of its
//     inputs, and a subnormal's leading zeros are bits lost there (Q4_0 with
//     codes left at 2^-24: 8e-5 relative error against 64 bits).
//   - Activations are scaled per token and 256-column chunk by a power of two
//     (chunk maximum in [2^13, 2^14)) and split into hi + lo fp16 halves, 22
//     bits and a sign; both halves go through v_mfma_f32_16x16x32_f16, which
//     accumulates in f32.
//   - Q4_K (src/quant/mod.rs:820-849): w = d sc (q - 8) + (8 d sc - dmin m),
//     so a chunk's 8 sub-blocks accumulate together, the sub-block sums X_s
//     enter one K = 16 MFMA against 8 sc_s and one against m_s, and d and
//     dmin apply once per chunk.  Q4_0 and Q8_0 (src/quant/mod.rs:689-745): one
//     MFMA pair per 32-weight block, whose f16 scale applies to its result.
//
// Work: a workgroup of 8 waves, KW chunk groups of RW = 8 / KW waves, owns 16 R
// RW rows and 16 NT tokens (NT = RW).  Group k takes chunks k, k + KW, ... of
// K; each of its waves converts one token tile of the chunk into the group's
// LDS stage (operand layout), then multiplies all of the stage's token tiles
// with its own R row tiles of 16.  So a workgroup converts no activation
// twice, its x loads are whole 256-byte runs, and the next chunk's x and
// codes are in flight while a chunk is computed.  The groups' partial sums
// meet in LDS at the end, added in group order.  No workspace: the call stays
// valid under stream capture.
//
// Bound by instruction issue: a wave's share of the conversion (about 450
// instructions per token tile and chunk) and of the operands, with two waves
// per SIMD (registers, LDS) to cover each other's waits.  Counters, 4096 x 4096
// Q4_K, 509 tokens: 60% of the issue slots taken, the matrix cores busy 25% of
// the time, waves waiting 27% of theirs for memory or a barrier and 36% for
// issue; 32000 x 4096 Q8_0, 13 tokens: 38%, 7%, 32% and 43%.  Measured against
// the GEMV (us): 4096 x 4096 Q4_K, 5 tokens 12.8 -> 9.2, 64 tokens 112 -> 17.0,
// 509 tokens 874 -> 54-64; 32000 x 4096 Q8_0, 13 tokens 159 -> 44.5 (3.2 TB/s of
// weights).  Error against
// 64 bits 2.1e-7 (Q4_K) and 1.1e-7 (Q4_0, Q8_0), the GEMV's 3.0e-7 and 2.7e-7.
#include "nx_internal.hpp"
#include "nx_split_dev.hpp"

namespace nx {

namespace {

struct MfdArgs {
  const uint8_t *qs, *meta;
  uint32_t qs_bytes, meta_bytes;
  int rows, cols, nseg, nchunk, T;
  const float *x;
  float *out;
  int nrb, ntb;  // row blocks, token blocks
};

// one (row tile, chunk) of a lane.  Q4_K: the code halves of sub-blocks g and
// g + 4 and the block's 16 header bytes; Q4_0: halves of blocks 2 g and
// 2 g + 1; Q8_0: both halves of blocks 2 g and 2 g + 1; the two with the
// chunk's 8 f16 scales
template <int FMT>
struct MfdStep {
  u32x4_t q[FMT == NX_FMT_Q8_0 ? 4 : 2];
  u32x4_t m;
};

// One token tile and chunk in LDS: the A operands of the 8 MFMAs, value p of
// lane L = token + 16 g of MFMA u.  Q4_K: lane group g holds elements
// 32 g + 8 u (u < 4) or 128 + 32 g + 8 (u - 4), the dwords of its sub-blocks g
// and g + 4; Q4_0 and Q8_0: elements 32 u + 8 g, a quarter of block u.  Strides
// in bytes: the padding spreads a staging write's lanes over the banks.
template <int FMT>
struct MfdStage {
  static constexpr int SG = FMT == NX_FMT_Q4_K ? 256 : 288;  // lane group
  static constexpr int SH = 4 * SG;                          // hi, lo
  static constexpr int SU = 2 * SH + 64;                     // MFMA
  alignas(16) uint8_t a[8 * SU];
  // Q4_K: lane L's sub-block sums g and g + 4, X 2^-6 as (hi, lo) each
  uint2 xm[FMT == NX_FMT_Q4_K ? 64 : 1];
  alignas(16) float sx[16];  // unscale factors
};

template <int FMT, int R, int KW>
__global__ __launch_bounds__(64 * MD_WAVES, 2) void k_mfd(const MfdArgs a) {
  constexpr bool Q4K = FMT == NX_FMT_Q4_K, Q80 = FMT == NX_FMT_Q8_0;
  constexpr int RW = MD_WAVES / KW, NT = RW;
  constexpr int NRED = RW * R * NT;  // 16 x 16 tiles of the workgroup
  using Stage = MfdStage<FMT>;
  __shared__ union {
    Stage st[KW][NT];
    float red[KW][NRED][4][64];
  } sh;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / RW, rw = wave % RW;
  const int l16 = lane & 15, g = lane >> 4;
  // workgroup L runs on XCD L % 8: the token blocks of one row block follow
  // each other on one XCD, so its L2 serves the re-reads of the rows
  const int L = (int)blockIdx.x, j = L >> 3;
  const int tb = j % a.ntb, rb = (j / a.ntb) * 8 + (L & 7);
  if (rb >= a.nrb) return;  // workgroup-uniform
  const int row0 = (rb * RW + rw) * 16 * R;

  const __amdgpu_buffer_rsrc_t rq = make_rsrc(a.qs, a.qs_bytes), rm = make_rsrc(a.meta, a.meta_bytes);
  const uint32_t prq = panel_row_bytes(a.nseg, 32), prm = panel_row_bytes(a.nseg, Q80 ? 2 : 4);
  constexpr int SPC = Q80 ? 8 : 4;  // segments per chunk
  // rows past the matrix and tokens past the batch read the last one's data
  // and are not stored; a chunk past the row reads the last chunk's
  MfdStep<FMT> w[R];
  auto issue = [&](int c) {
    c = min(c, a.nchunk - 1);
    const int j0 = SPC * c, grp = j0 >> 6, gsz = min(64, a.nseg - (grp << 6));
    const uint32_t pbase = (uint32_t)grp * (uint32_t)a.rows;
    const int sbase = (int)(pbase * prq + (uint32_t)((j0 & 63) * 16));
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = min(row0 + 16 * r + l16, a.rows - 1);
      const int vq = (int)((uint32_t)row * prq + (Q80 ? 32u : 16u) * (uint32_t)g);
#pragma unroll
      for (int i = 0; i < (Q80 ? 4 : 2); ++i) {
        // Q8_0: [2 t + h] = half h of block 2 g + t; else half i of segment g
        const int h = Q80 ? (i & 1) : i, t = Q80 ? (i >> 1) : 0;
        w[r].q[i] = __builtin_amdgcn_raw_buffer_load_b128(rq, vq, sbase + h * 16 * gsz + 16 * t, 0);
      }
      w[r].m = __builtin_amdgcn_raw_buffer_load_b128(
          rm, (int)((pbase + (uint32_t)row) * prm + (uint32_t)((j0 & 63) * (Q80 ? 2 : 4))), 0, 0);
    }
  };
  // this wave's token tile: lane's token 4 p + g, columns 64 q + 4 l16 .. + 3
  f32x4 xr[4][4];
  const float *xrow[4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    xrow[p] = a.x + (size_t)min((tb * NT + rw) * 16 + 4 * p + g, a.T - 1) * a.cols + 4 * l16;
  auto load_x = [&](int c) {
    c = min(c, a.nchunk - 1);
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        xr[p][q] = *reinterpret_cast<const f32x4 *>(xrow[p] + (size_t)c * MD_K + 64 * q);
  };
  auto stage_x = [&]() {
    Stage &st = sh.st[kg][rw];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int tok = 4 * p + g;
      st.sx[tok] = split16<FMT>(
          xr[p], l16,
          [&](int u, int gq, int half, f16x4 hi, f16x4 lo) {
            uint8_t *o = st.a + u * Stage::SU + gq * Stage::SG + 16 * tok + 8 * half;
            *reinterpret_cast<f16x4 *>(o) = hi;
            *reinterpret_cast<f16x4 *>(o + Stage::SH) = lo;
          },
          [&](int gq, int i, f16x2 hl) { (&st.xm[tok + 16 * gq].x)[i] = __builtin_bit_cast(uint32_t, hl); });
    }
  };
  // between staging and use: the waves of a group share its stage
  auto sync = [&]() {
    if constexpr (RW > 1)
      __syncthreads();
    else
      wave_handoff();
  };

  f32x4 acc[R][NT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&]() {
    const Stage *st = sh.st[kg];
    f32x4 y[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int n = 0; n < NT; ++n) y[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // MFMA u + 1's operands are read while u's are multiplied (R NT = 8 of
    // four token tiles: no registers for that)
    constexpr bool AHEAD = R * NT < 8 || NT < 4;
    const uint32_t la = g * Stage::SG + 16 * l16;
    f16x8 ahi[1 + AHEAD][NT], alo[1 + AHEAD][NT];
    auto operands = [&](int u) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        ahi[u & AHEAD][n] = *reinterpret_cast<const f16x8 *>(st[n].a + u * Stage::SU + la);
        alo[u & AHEAD][n] = *reinterpret_cast<const f16x8 *>(st[n].a + u * Stage::SU + Stage::SH + la);
      }
      if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (AHEAD) operands(0);
    if constexpr (Q4K) {
      // get_scale_min_k4 (src/quant/mod.rs:1163-1170) of sub-blocks g, g + 4:
      // sc 2^10, sc 2^6 and -8 sc 2^-14
      f16x2 s1[R][2], s16[R][2], off[R][2];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t p03 = w[r].m.y, p8b = w[r].m.w;
        const uint32_t sc[2] = {(p03 >> (8 * g)) & 63,
                                ((p8b >> (8 * g)) & 15) | (((p03 >> (8 * g + 6)) & 3) << 4)};
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const _Float16 f = (_Float16)(float)(sc[v] << 10);
          s1[r][v] = f16x2{f, f};
          s16[r][v] = s1[r][v] * f16x2{0.0625f16, 0.0625f16};
          off[r][v] = s16[r][v] * f16x2{-0x1p-17f16, -0x1p-17f16};
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int v = u >> 2;
        if (!AHEAD || u < 7) operands(u + AHEAD);
        const f16x8(&hi)[NT] = ahi[u & AHEAD], (&lo)[NT] = alo[u & AHEAD];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const f16x8 b = operand4(w[r].q[v][u & 3], s1[r][v], s16[r][v], off[r][v]);
#pragma unroll
          for (int n = 0; n < NT; ++n) y[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[n], b, y[r][n], 0, 0, 0);
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            y[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[n], b, y[r][n], 0, 0, 0);
            // one step's operands live at a time: left free, the compiler
            // forms every step's operands first and spills
            asm volatile("" : "+v"(y[r][n]));
          }
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        // 8 sc X at the codes' 2^-14 (X enters 2^-6): sc 2^-5; and m
        const uint32_t p47 = w[r].m.z, p8b = w[r].m.w;
        const uint32_t mn0 = (p47 >> (8 * g)) & 63;
        const uint32_t mn1 = ((p8b >> (8 * g + 4)) & 15) | (((p47 >> (8 * g + 6)) & 3) << 4);
        const _Float16 k15 = (_Float16)0x1p-15f;
        const _Float16 b0 = s1[r][0][0] * k15, b1 = s1[r][1][0] * k15;
        const _Float16 m0 = (_Float16)(float)mn0, m1 = (_Float16)(float)mn1;
        const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[r].m.x & 0xFFFF));
        const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[r].m.x >> 16));
        const float dd = d * 16384.0f, dm = dmin * 64.0f;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const f16x4 xm = *reinterpret_cast<const f16x4 *>(&st[n].xm[lane]);
          const f32x4 sx = *reinterpret_cast<const f32x4 *>(&st[n].sx[4 * g]);
          // (never onto y: nx_mfv.hip)
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          const f32x4 yx = __builtin_amdgcn_mfma_f32_16x16x16f16(xm, f16x4{b0, b0, b1, b1}, zero, 0, 0, 0);
          const f32x4 ym = __builtin_amdgcn_mfma_f32_16x16x16f16(xm, f16x4{m0, m0, m1, m1}, zero, 0, 0, 0);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            acc[r][n][k] = fmaf(sx[k], fmaf(dd, y[r][n][k], fmaf(dd, yx[k], -dm * ym[k])), acc[r][n][k]);
        }
      }
    } else {
      // the blocks' codes from the lane groups that loaded them: lane group
      // g gets its 8 elements of every block (nx_split_dev.hpp)
      constexpr int NW = Q80 ? 2 : 1;
      uint32_t cq[R][2][NW][4];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (Q80) {
            const u32x4_t q0 = w[r].q[2 * h], q1 = w[r].q[2 * h + 1];
            const uint32_t lo[4] = {q0.x, q0.z, q1.x, q1.z}, hi[4] = {q0.y, q0.w, q1.y, q1.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) cq[r][h][0][k] = lo[k], cq[r][h][NW - 1][k] = hi[k];
          } else {
            const u32x4_t q0 = w[r].q[h];
            cq[r][h][0][0] = q0.x, cq[r][h][0][1] = q0.y, cq[r][h][0][2] = q0.z, cq[r][h][0][3] = q0.w;
          }
#pragma unroll
          for (int v = 0; v < NW; ++v) transpose_groups(cq[r][h][v]);
        }
      // codes at 2^-9
      const f16x2 s1 = {32768.0f16, 32768.0f16}, s16 = {2048.0f16, 2048.0f16};
      const f16x2 off = {-0x1p-6f16, -0x1p-6f16};
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (!AHEAD || b < 7) operands(b + AHEAD);
        const f16x8(&hi)[NT] = ahi[b & AHEAD], (&lo)[NT] = alo[b & AHEAD];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const f16x8 bq = Q80 ? operand8(cq[r][b & 1][0][b >> 1], cq[r][b & 1][NW - 1][b >> 1])
                               : operand4(cq[r][b & 1][0][b >> 1], s1, s16, off);
          const uint32_t dw = w[r].m[b >> 1];
          const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(b & 1 ? dw >> 16 : dw & 0xFFFFu));
          f32x4 z[NT];
#pragma unroll
          for (int n = 0; n < NT; ++n)
            z[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[n], bq, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int n = 0; n < NT; ++n) z[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[n], bq, z[n], 0, 0, 0);
#pragma unroll
          for (int n = 0; n < NT; ++n) {
#pragma unroll
            for (int k = 0; k < 4; ++k) y[r][n][k] = fmaf(d, z[n][k], y[r][n][k]);
            asm volatile("" : "+v"(y[r][n]));  // as for Q4_K
          }
        }
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const f32x4 sx = *reinterpret_cast<const f32x4 *>(&st[n].sx[4 * g]);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int k = 0; k < 4; ++k) acc[r][n][k] = fmaf(sx[k] * 512.0f, y[r][n][k], acc[r][n][k]);
      }
    }
  };

  const int nstep = (a.nchunk + KW - 1) / KW;
  load_x(kg);
  __builtin_amdgcn_sched_barrier(0);  // x ahead of the codes here too, as the loop's waits count
  issue(kg);
  __builtin_amdgcn_sched_barrier(0);
#pragma clang loop unroll(disable)
  for (int i = 0; i < nstep; ++i) {
    const int c = i * KW + kg;
    // the loop carries each load as one register tuple: split into its
    // elements, the compiler copies them at the back edge, which waits there
    // for the loads in flight (4096 x 4096 Q4_K, 509 tokens: 58 us)
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(xr[p][q]));
    stage_x();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int q = 0; q < (Q80 ? 4 : 2); ++q) asm volatile("" : "+v"(w[r].q[q]));
      asm volatile("" : "+v"(w[r].m));
    }
    sync();
    load_x(c + KW);
    __builtin_amdgcn_sched_barrier(0);
    if (c < a.nchunk) compute();  // wave-uniform
    __builtin_amdgcn_sched_barrier(0);
    issue(c + KW);
    sync();
  }

  // the groups' partial sums, added in group order
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int k = 0; k < 4; ++k) sh.red[kg][(rw * R + r) * NT + n][k][lane] = acc[r][n][k];
  __syncthreads();
  for (int i = tid; i < NRED * 256; i += 64 * MD_WAVES) {
    const int tile = i >> 8, k = (i >> 6) & 3, ln = i & 63;
    const int row = (rb * RW * R + tile / NT) * 16 + (ln & 15);
    const int tok = (tb * NT + tile % NT) * 16 + 4 * (ln >> 4) + k;
    float sum = 0.f;
#pragma unroll
    for (int kk = 0; kk < KW; ++kk) sum += sh.red[kk][tile][k][ln];
    if (row < a.rows && tok < a.T) a.out[(size_t)tok * a.rows + row] = sum;
  }
}

template <int FMT>
void (*mfd_pick(MfdShape s))(MfdArgs) {
  if (s.kw == 2) return s.r == 2 ? k_mfd<FMT, 2, 2> : k_mfd<FMT, 1, 2>;
  if (s.kw == 4) return s.r == 2 ? k_mfd<FMT, 2, 4> : k_mfd<FMT, 1, 4>;
  return s.r == 4 ? k_mfd<FMT, 4, 8> : s.r == 2 ? k_mfd<FMT, 2, 8> : k_mfd<FMT, 1, 8>;
}

}  // namespace

bool mfd_takes(int fmt, const RolePlane &pl, const float *x, int T) {
  return mfd_sizes(fmt, pl.rows, pl.cols, T) && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
         (uint64_t)pl.rows * pl.row_qs < 0x7FFFFFF0ull;
}

int launch_mfd(nx_ctx *c, int fmt, const RolePlane &pl, const float *x, int T, float *out) {
  MfdArgs a{};
  a.qs = pl.qs;
  a.meta = pl.meta;
  a.qs_bytes = (uint32_t)pl.rows * pl.row_qs;
  a.meta_bytes = (uint32_t)pl.rows * pl.row_meta;
  a.rows = pl.rows;
  a.cols = pl.cols;
  a.nseg = pl.nseg;
  a.nchunk = pl.cols / MD_K;
  a.T = T;
  a.x = x;
  a.out = out;
  const MfdShape s = mfd_shape(pl.rows, a.nchunk, T, c->num_cu);
  a.ntb = (T + s.tokens() - 1) / s.tokens();
  a.nrb = (pl.rows + s.rows() - 1) / s.rows();
  const auto kern = fmt == NX_FMT_Q4_K   ? mfd_pick<NX_FMT_Q4_K>(s)
                    : fmt == NX_FMT_Q4_0 ? mfd_pick<NX_FMT_Q4_0>(s)
                                         : mfd_pick<NX_FMT_Q8_0>(s);
  const long blocks = (long)((a.nrb + 7) / 8) * 8 * a.ntb;
  return launch(c, "mfd_matrix", [&] { go(c, kern, dim3((unsigned)blocks), dim3(64 * MD_WAVES), 0, a); });
}

}  // namespace nx
