// nx_mfv.hip — few-token grouped matvec on MFMA for Q4_K, Q4_0, Q8_0 and Q2_K experts: decode
// batches whose experts see a handful of tokens each (2 to ~128 tokens),
// with or without a shared expert (as wide as the routed ones) that sees
// every token.
//
// The decode GEMV's exact integer dot costs about one instruction per
// weight per token, so its time grows with the tokens an expert sees; the
// prefill GEMM dequantizes every weight into its operands, which costs the
// same at 8 tokens as at 128.  Here the weights are never dequantized:
//
//   sum_i w_i x_i over a 32-weight sub-block s of a Q4_K block
//     = (d sc_s) sum_i (q_i - 8) x_i  +  (8 d sc_s - dmin m_s) sum_i x_i
//
// (src/quant/mod.rs:820-849: w_i = d sc_s q_i - dmin m_s).  The operand of
// weight i is (q_i - 8) sc_s, exact in fp16 (nx_split_dev.hpp), so one
// v_mfma_f32_16x16x32_f16 may span several sub-blocks and the 8 MFMAs of a
// block accumulate together; d and dmin apply once per block.  sum_s 8 sc_s X_s
// and sum_s m_s X_s are one more MFMA each, on the staged sub-block sums X_s.
// Q4_0 (w_i = d (q_i - 8), src/quant/mod.rs:723-745) and Q8_0 (w_i = d q_i,
// src/quant/mod.rs:689-703): one MFMA pair per 32-weight block, whose f16 scale
// applies to its result; a 4 x 4 dword transpose across the lane groups hands
// every lane group its 8 weights of each block.  Q2_K (w_i = d sc q_i - dmin m
// per 16-weight sub-block, src/quant/mod.rs:913-937): as Q4_K without the 8.
//
// Activations keep close to fp32 precision: per row and 256-element chunk
// they are scaled by a power of two so the chunk maximum lies in
// [2^13, 2^14), split into x' = hi + lo with hi = fp16(x') and lo =
// fp16(x' - hi), and both halves go through the MFMA (two MFMAs per
// operand, chained).  hi + lo carries 22 bits of x' and a sign.
//
// Work: the activations are split once per row, not per workgroup, into
// operand records in memory: x's by workgroups that ride along with the routing
// kernels, the gated rows' by k_mfv_swiglu.  A wave of k_mfv owns one chunk of
// one expert's tile of 16 pairs (the permutation's tile list with tile_m = 16):
// it holds the chunk's operands in registers and streams row tiles of 16
// weight rows past them, the codes of the next MV_D steps in flight.  The waves
// of a workgroup take the chunks of one K slice (at most 8) side by side, so
// the 128-byte lines that two chunks' codes and eight chunks' scales share are
// read at about the same time, and add their results through LDS every pass
// of four steps.  Slices write partial sums, which the SwiGLU kernel (gate/up) and the
// weighted combine (down) add in slice order.
//
// Bound by the weight stream, then by instruction issue: Mixtral Q4_K, 32
// tokens, gate/up (529 MB) 127 us, of which the loads alone take 123 and the
// arithmetic alone 99.  Against workgroups of 256 rows that staged their
// activations in LDS and walked a slice of 4 chunks (us, layer): Mixtral 32
// tokens 250 -> 214, DeepSeek 27 tokens 1071 -> 831, Qwen3 61 tokens 119.8 ->
// 109.2; error against 64 bits 9.3e-7 -> 3.8e-7 (Q4_K), 7.8e-5 -> 2.1e-7 (Q4_0,
// whose codes were fp16 subnormals).  A wave per 64 rows that walked the chunks
// itself read each line's halves a chunk apart, too late for the L2: 370 us.
#include "nx_internal.hpp"
#include "nx_split_dev.hpp"

namespace nx {

namespace {

constexpr int MV_M = 16;   // pairs per tile

struct MfvArgs {
  const uint8_t *qs0, *qs1, *meta0, *meta1;  // role planes (gate, up) or (down, -)
  size_t qs_stride, meta_stride;             // per expert
  uint32_t row_qs, row_meta;
  int rows, nseg, nchunk;                    // nchunk = cols / 256
  const uint8_t *rec;         // operand records [row][chunk]
  const int32_t *perm_token;  // gate/up: pair -> token row of x; down: null (pair row)
  const int32_t *offsets;     // [E + 1]
  const int32_t *tiles;       // [0] = tile count, [1] unused, then (expert, first pair within it)
  // the shared expert (tiles of expert E; pairs T k + t, t the token), with
  // the routed experts' row layout
  const uint8_t *sqs0, *sqs1, *smeta0, *smeta1;
  int E, T, k;
  float *out;                 // partial sums: [slice][pair][out_stride]
  int out_stride;             // gate/up: 2 F (gate rows, then up rows); down: H
  size_t out_split;           // floats between slices
  int ks;                     // chunks per K slice, the waves of a workgroup
  int nks;                    // K slices
};

// one (row tile, chunk) step of a lane.  Q4_K: the code halves of sub-blocks g
// and g + 4 and the block's 16 header bytes (d, dmin, scales12); Q4_0: halves
// of blocks 2 g and 2 g + 1; Q8_0: both halves of blocks 2 g and 2 g + 1; the
// two with the chunk's 8 f16 scales; Q2_K: segment g's 16 code bytes and its
// scale-plane entry {f16 d, f16 dmin, the segment's four scale/min bytes}
template <int FMT>
struct MfvStep {
  static constexpr int NQ = FMT == NX_FMT_Q8_0 ? 4 : FMT == NX_FMT_Q2_K ? 1 : 2;
  u32x4_t q[NQ];
  u32x4_t m;
};

constexpr int MV_STEPS = 4;  // (row tile, matrix) steps per pass of the loop
constexpr int MV_D = 4;      // steps in flight, at most MV_STEPS (2, 3 or 6: within 3%)

template <bool GATEUP, int FMT>
__global__ __launch_bounds__(64 * MV_KW, 2) void k_mfv(const MfvArgs a) {
  constexpr bool Q4K = FMT == NX_FMT_Q4_K, Q2K = FMT == NX_FMT_Q2_K, Q80 = FMT == NX_FMT_Q8_0;
  constexpr bool BLK = !Q4K && !Q2K;  // one MFMA per 32-weight block
  constexpr int D = MV_D, NQ = MfvStep<FMT>::NQ;
  constexpr int RT = GATEUP ? MV_STEPS / 2 : MV_STEPS;  // row tiles per pass
  extern __shared__ f32x4 red[];  // [pass parity][wave][step][lane]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The work is a line of (tile, slice, pass of RT row tiles), cut into the runs
  // of the workgroups (mfv_run).  (Workgroups of a fixed run of rows, sized on the
  // host from the expected tile count, left CUs idle wherever the routing
  // drew another: Mixtral 32 tokens 223 us, Qwen3 61 tokens 135 us.)  Passes are
  // as short as the steps in flight allow: a run of one or two passes more than
  // the others' is the round's tail.  Equal runs of 8-step passes took (layer, 8
  // experts, top 2) 1024 x 2048 Q8_0 256 tokens 97 us, now 75; 2048 x 1280 Q4_K
  // 128 tokens 68, now 56.
  const int ntile = a.tiles[0], npass = (a.rows >> 4) / RT;
  int buf = 0;  // the sums' buffer of this pass: red + 0 or + ks MV_STEPS 64
  // rounds of the segments (a tile's K slice) from `first` on
  for (int first = 0, left = ntile * a.nks; left > 0; first += gridDim.x, left -= gridDim.x) {
    const MfvRun run = mfv_run((int)blockIdx.x, (int)gridDim.x, left, npass);
    for (int un = run.u0; un < run.u1;) {
      const int s = un / npass, pass0 = un - s * npass;
      const int pass1 = min(npass, pass0 + (run.u1 - un));
      un += pass1 - pass0;
      const int seg = first + run.seg0 + s, tile = seg / a.nks, slice = seg - tile * a.nks;
      // tile t: expert tiles[2 + 2t] (E: the shared expert), first pair
      // tiles[3 + 2t] within the expert
      const int e = __builtin_amdgcn_readfirstlane(a.tiles[2 + 2 * tile]);
      const int m0 = __builtin_amdgcn_readfirstlane(a.tiles[3 + 2 * tile]);
      const bool routed = e < a.E;
      const int pair0 = __builtin_amdgcn_readfirstlane(routed ? a.offsets[e] + m0 : a.T * a.k + m0);
      const int cnt = __builtin_amdgcn_readfirstlane(
          min(MV_M, routed ? a.offsets[e + 1] - pair0 : a.T - m0));
      // this wave's chunk; past the row's end (the last slice) it adds zeros
      const int c = slice * a.ks + wave;
      const bool in_row = c < a.nchunk;
      const int rt0 = pass0 * RT, rt1 = pass1 * RT;

      const int l16 = lane & 15, g = lane >> 4;
      __amdgpu_buffer_rsrc_t rq[GATEUP ? 2 : 1], rm[GATEUP ? 2 : 1];
      {
        const uint32_t nq = (uint32_t)a.rows * a.row_qs, nm = (uint32_t)a.rows * a.row_meta;
        rq[0] = make_rsrc(routed ? a.qs0 + (size_t)e * a.qs_stride : a.sqs0, nq);
        rm[0] = make_rsrc(routed ? a.meta0 + (size_t)e * a.meta_stride : a.smeta0, nm);
        if constexpr (GATEUP) {
          rq[1] = make_rsrc(routed ? a.qs1 + (size_t)e * a.qs_stride : a.sqs1, nq);
          rm[1] = make_rsrc(routed ? a.meta1 + (size_t)e * a.meta_stride : a.smeta1, nm);
        }
      }
      // The planes are in panels of 64 segments (nx_device.hpp): the chunk's
      // panel grp starts at grp * rows * prq (codes) and grp * rows * prm
      // (scales), prq and prm a row's bytes in a panel, and holds gsz segments
      // of each row.  Per-lane parts of the offsets stay in registers; the rest
      // goes in the scalar offset.  Steps past the run's rows (the
      // pipeline's tail) and chunks past the row read at OOB.
      constexpr int SPC = Q80 ? 8 : 4;                               // segments per chunk
      constexpr int QU = Q2K ? 16 : 32, MU = Q80 ? 2 : Q2K ? 8 : 4;  // plane bytes per segment
      const uint32_t prq = panel_row_bytes(a.nseg, QU), prm = panel_row_bytes(a.nseg, MU);
      const int j0 = SPC * (in_row ? c : 0), grp = j0 >> 6, gsz = min(64, a.nseg - (grp << 6));
      const uint32_t vq = (uint32_t)l16 * prq + (Q80 ? 32u : 16u) * (uint32_t)g;
      const uint32_t vm = (uint32_t)l16 * prm + (Q2K ? 8u * (uint32_t)g : 0u);
      const uint32_t sq0 = (uint32_t)grp * (uint32_t)a.rows * prq + (uint32_t)((j0 & 63) * 16);
      const uint32_t sm0 = (uint32_t)grp * (uint32_t)a.rows * prm + (uint32_t)((j0 & 63) * MU);
      // step i of the pass from row tile rt: gate/up row tile rt + i / 2 of gate
      // (i even) or up
      auto issue = [&](MfvStep<FMT> &w, int rt, int i) {
        rt += GATEUP ? i >> 1 : i;
        const int mt = GATEUP ? i & 1 : 0;
        const bool in = in_row && rt < rt1;  // wave-uniform
        const uint32_t past = in ? 0u : OOB;
        const uint32_t sq = in ? sq0 + 16u * rt * prq : 0u, smo = in ? sm0 + 16u * rt * prm : 0u;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          // Q8_0: [2 t + h] = half h of block 2 g + t; Q4: half q of segment g
          const int h = Q80 ? (q & 1) : q, t = Q80 ? (q >> 1) : 0;
          w.q[q] = __builtin_amdgcn_raw_buffer_load_b128(rq[mt], (int)(vq | past),
                                                         (int)(sq + (in ? h * 16 * gsz + 16 * t : 0)), 0);
        }
        if constexpr (Q2K) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(rm[mt], (int)(vm | past), (int)smo, 0);
          w.m = u32x4_t{v[0], v[1], 0, 0};
        } else {
          w.m = __builtin_amdgcn_raw_buffer_load_b128(rm[mt], (int)(vm | past), (int)smo, 0);
        }
      };
      // the first steps go out ahead of the chain of loads that finds the pairs'
      // records
      MfvStep<FMT> ring[MV_STEPS];  // slot i: step i of a pass; D of them live
#pragma unroll
      for (int i = 0; i < D; ++i) issue(ring[i], rt0, i);
      __builtin_amdgcn_sched_barrier(0);

      // ---- activations: lane's row of the tile (absent pairs take the last
      // one's, and are not stored)
      const int m = min(l16, cnt - 1);
      const int xr = a.perm_token ? (routed ? a.perm_token[pair0 + m] : m0 + m) : pair0 + m;
      const uint8_t *rec = a.rec + ((size_t)xr * a.nchunk + (in_row ? c : 0)) * REC_BYTES;
      f16x8 hi[8], lo[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        hi[u] = *reinterpret_cast<const f16x8 *>(rec + 128 * u + 16 * g);
        lo[u] = *reinterpret_cast<const f16x8 *>(rec + 128 * u + 64 + 16 * g);
      }
      u32x4_t xm = {0, 0, 0, 0};
      if constexpr (Q4K) {
        const uint2 v = *reinterpret_cast<const uint2 *>(rec + REC_XM + 8 * g);
        xm.x = v.x;
        xm.y = v.y;
      } else if constexpr (Q2K) {
        xm = *reinterpret_cast<const u32x4_t *>(rec + REC_XM + 16 * g);
      }
      const float sxl = *reinterpret_cast<const float *>(rec + REC_SX);
      float sx[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) sx[k] = in_row ? __shfl(sxl, 4 * g + k, 64) : 0.f;

      float *out = a.out + (size_t)slice * a.out_split + (size_t)(pair0 + 4 * g) * a.out_stride + l16;
#pragma clang loop unroll(disable)
      for (int rt = rt0; rt < rt1; rt += RT) {
#pragma unroll
        for (int i = 0; i < MV_STEPS; ++i) {
          MfvStep<FMT> &w = ring[i];
#pragma unroll
          for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(w.q[q]));
          asm volatile("" : "+v"(w.m));
          f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f}, res;
          // MFMA u of operand b, both halves
          auto mfma = [&](int u, f16x8 b, f32x4 y4) {
            y4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[u], b, y4, 0, 0, 0);
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[u], b, y4, 0, 0, 0);
          };
          if constexpr (BLK) {
            // the loads give lane group g blocks 2 g and 2 g + 1; transposed
            // across the lane groups, it holds its 8 weights of every block
            constexpr int NW = Q80 ? 2 : 1;
            uint32_t cq[2][NW][4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              if constexpr (Q80) {
                const u32x4_t q0 = w.q[2 * h], q1 = w.q[2 * h + 1];
                cq[h][0][0] = q0.x, cq[h][0][1] = q0.z, cq[h][0][2] = q1.x, cq[h][0][3] = q1.z;
                cq[h][NW - 1][0] = q0.y, cq[h][NW - 1][1] = q0.w, cq[h][NW - 1][2] = q1.y, cq[h][NW - 1][3] = q1.w;
              } else {
                const u32x4_t q0 = w.q[h];
                cq[h][0][0] = q0.x, cq[h][0][1] = q0.y, cq[h][0][2] = q0.z, cq[h][0][3] = q0.w;
              }
#pragma unroll
              for (int v = 0; v < NW; ++v) transpose_groups(cq[h][v]);
            }
            // codes at 2^-9
            const f16x2 s1 = {32768.0f16, 32768.0f16}, s16 = {2048.0f16, 2048.0f16};
            const f16x2 off = {-0x1p-6f16, -0x1p-6f16};
#pragma unroll
            for (int b = 0; b < 8; ++b) {
              const f16x8 bq = Q80 ? operand8(cq[b & 1][0][b >> 1], cq[b & 1][NW - 1][b >> 1])
                                   : operand4(cq[b & 1][0][b >> 1], s1, s16, off);
              const uint32_t dw = w.m[b >> 1];
              const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(b & 1 ? dw >> 16 : dw & 0xFFFFu));
              const f32x4 z = mfma(b, bq, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
              for (int k = 0; k < 4; ++k) y[k] = fmaf(d, z[k], y[k]);
              // one step's operands live at a time: left free, the compiler
              // forms every step's operands first and spills
              asm volatile("" : "+v"(y));
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) res[k] = sx[k] * 512.0f * y[k];
          } else {
            // scales into the operands, sc 2^10 and sc 2^6 (2^-14 with the codes'
            // 2^-24); mins for their own MFMA
            constexpr int NV = Q2K ? 4 : 2;
            uint32_t scv[NV], mnv[NV];
            if constexpr (Q2K) {
#pragma unroll
              for (int v = 0; v < NV; ++v) {
                scv[v] = (w.m.y >> (8 * v)) & 15;
                mnv[v] = (w.m.y >> (8 * v + 4)) & 15;
              }
            } else {
              // get_scale_min_k4 (src/quant/mod.rs:1163-1170) of sub-blocks g, g + 4
              const uint32_t p03 = w.m.y, p47 = w.m.z, p8b = w.m.w;
              scv[0] = (p03 >> (8 * g)) & 63;
              mnv[0] = (p47 >> (8 * g)) & 63;
              scv[NV - 1] = ((p8b >> (8 * g)) & 15) | (((p03 >> (8 * g + 6)) & 3) << 4);
              mnv[NV - 1] = ((p8b >> (8 * g + 4)) & 15) | (((p47 >> (8 * g + 6)) & 3) << 4);
            }
            f16x2 s1[NV], s16[NV], off[NV];
            _Float16 mn[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
              const _Float16 f = (_Float16)(float)(scv[v] << 10);
              s1[v] = f16x2{f, f};
              s16[v] = s1[v] * f16x2{0.0625f16, 0.0625f16};
              off[v] = s16[v] * f16x2{-0x1p-17f16, -0x1p-17f16};  // -8 sc 2^-14
              mn[v] = (_Float16)(float)mnv[v];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              f16x8 b;
              if constexpr (Q2K)  // the 2-bit codes of half u / 4 widened to nibbles (no offset)
                b = operand4u((w.q[0][u & 3] >> (2 * (u >> 2))) & 0x33333333u, s1[u >> 1], s16[u >> 1]);
              else
                b = operand4(w.q[(u >> 2) % NQ][u & 3], s1[(u >> 2) % NV], s16[(u >> 2) % NV], off[(u >> 2) % NV]);
              y = mfma(u, b, y);
              asm volatile("" : "+v"(y));  // as above
            }
            const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(w.m.x & 0xFFFF));
            const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(w.m.x >> 16));
            const float dd = d * 16384.0f, dm = dmin * 64.0f;  // X enters 2^-6
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            f32x4 rest;  // what the offsets and mins add
            if constexpr (Q2K) {
              const f32x4 ym = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  __builtin_bit_cast(f16x8, xm), f16x8{mn[0], mn[0], mn[1], mn[1], mn[NV - 2], mn[NV - 2], mn[NV - 1], mn[NV - 1]},
                  zero, 0, 0, 0);
#pragma unroll
              for (int k = 0; k < 4; ++k) rest[k] = -dm * ym[k];
            } else {
              // 8 sc X at the codes' 2^-14 (X enters 2^-6): sc 2^-5; and m.  On
              // accumulators of their own: the result of an MFMA of one shape, taken
              // as another shape's accumulator, is read before it is complete unless
              // enough instructions lie between, and the compiler (ROCm 7.2) puts no
              // wait there.  16x16x32 and 16x16x16 back to back on one accumulator
              // lose the first in two of the four registers.
              const f16x4 xa = __builtin_bit_cast(f16x4, uint2{xm.x, xm.y});
              const _Float16 k15 = (_Float16)0x1p-15f;
              const _Float16 b0 = s1[0][0] * k15, b1 = s1[NV - 1][0] * k15;
              const f32x4 yx = __builtin_amdgcn_mfma_f32_16x16x16f16(xa, f16x4{b0, b0, b1, b1}, zero, 0, 0, 0);
              const f32x4 ym = __builtin_amdgcn_mfma_f32_16x16x16f16(
                  xa, f16x4{mn[0], mn[0], mn[NV - 1], mn[NV - 1]}, zero, 0, 0, 0);
#pragma unroll
              for (int k = 0; k < 4; ++k) rest[k] = fmaf(dd, yx[k], -dm * ym[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) res[k] = sx[k] * fmaf(dd, y[k], rest[k]);
          }
          __builtin_amdgcn_sched_barrier(0);
          issue(ring[(i + D) % MV_STEPS], i + D < MV_STEPS ? rt : rt + RT, (i + D) % MV_STEPS);
          __builtin_amdgcn_sched_barrier(0);
          red[buf + (wave * MV_STEPS + i) * 64 + lane] = res;
        }
        // The slice's sums: every pass the waves leave their chunks' results in one
        // of two buffers, and wave w adds those of steps w, w + ks, ... in chunk
        // order.  One barrier per pass: a buffer is written again only after the
        // next pass's barrier.
        __syncthreads();
        for (int t = wave; t < MV_STEPS; t += a.ks) {
          const f32x4 *r = red + buf + t * 64 + lane;
          f32x4 sum = *r;
          for (int v = 1; v < a.ks; ++v) {
            r += MV_STEPS * 64;
#pragma unroll
            for (int k = 0; k < 4; ++k) sum[k] += (*r)[k];
          }
          // lane holds row (lane % 16), pairs 4g .. 4g+3
          float *o = out + (GATEUP ? 16 * (rt + (t >> 1)) + (t & 1) * a.rows : 16 * (rt + t));
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (4 * g + k < cnt) o[(size_t)k * a.out_stride] = sum[k];
        }
        buf ^= a.ks * MV_STEPS * 64;
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_mfv_split(const SplitJob job) {
  split_rows(job, (size_t)blockIdx.x * 16 + (threadIdx.x >> 4));
}

// Records of silu(sum_s gate_s[p][f]) * sum_s up_s[p][f] over the K slices of
// the gate/up pass, summed in slice order: 16 lanes per (pair, chunk of 256
// columns).  The slices are loaded SB at a time (past the last clamped to it)
// before any is added, so up to SB slices take one round of loads.
template <int FMT, int SB>
__global__ __launch_bounds__(256) void k_mfv_swiglu(const float *__restrict__ part, int nslice,
                                                    size_t slice_stride, size_t n, int F,
                                                    uint8_t *__restrict__ rec) {
  const size_t i = (size_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15, nchunk = F / MV_K;
  const size_t ic = min(i, n - 1), p = ic / nchunk;
  const float *src = part + p * 2 * F + (ic - p * nchunk) * MV_K + 4 * j;
  f32x4 v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 g = {0.f, 0.f, 0.f, 0.f}, u = g;
    for (int s0 = 0; s0 < nslice; s0 += SB) {
      f32x4 gv[SB], uv[SB];
#pragma unroll
      for (int k = 0; k < SB; ++k) {
        const float *o = src + (size_t)min(s0 + k, nslice - 1) * slice_stride + 64 * q;
        gv[k] = *reinterpret_cast<const f32x4 *>(o);
        uv[k] = *reinterpret_cast<const f32x4 *>(o + F);
      }
#pragma unroll
      for (int k = 0; k < SB; ++k) {
        const bool first = s0 + k == 0, in = s0 + k < nslice;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          g[c] = first ? gv[k][c] : (in ? g[c] + gv[k][c] : g[c]);
          u[c] = first ? uv[k][c] : (in ? u[c] + uv[k][c] : u[c]);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) v[q][c] = silu_mul(g[c], u[c]);
  }
  if (i < n) write_record<FMT>(rec + i * REC_BYTES, v, j);
}

template <int FMT>
int run_mfv(nx_ctx *c, const MfvPlan &p) {
  const nx_experts *ex = p.ex;
  const bool shared = ex->Fs > 0;
  const int H = ex->H, F = ex->F, cd = F / MV_K;
  const MfvSizes z = mfv_sizes(shape_of(ex), p.T, p.k);
  const size_t pairs = z.pairs;
  const int nks_g = z.nks_g, nks_d = z.nks_d;
  void *vp;
  NX_TRY(ws_get(c, WS_MFV_PART, z.bytes, &vp));
  float *ppart = static_cast<float *>(vp);
  uint8_t *rec = static_cast<uint8_t *>(vp) + z.act_at;
  for (int pass = 0; pass < 2; ++pass) {
    const bool gateup = pass == 0;
    const RolePlane &R0 = ex->role[gateup ? NX_ROLE_GATE : NX_ROLE_DOWN];
    const RolePlane &R1 = ex->role[gateup ? NX_ROLE_UP : NX_ROLE_DOWN];
    MfvArgs a{};
    a.qs0 = R0.qs;
    a.qs1 = R1.qs;
    a.meta0 = R0.meta;
    a.meta1 = R1.meta;
    a.qs_stride = R0.qs_stride;
    a.meta_stride = R0.meta_stride;
    a.row_qs = R0.row_qs;
    a.row_meta = R0.row_meta;
    a.rows = R0.rows;
    a.nseg = R0.nseg;
    a.nchunk = R0.cols / MV_K;
    a.rec = gateup ? p.rec : rec;
    a.offsets = p.offsets;
    a.tiles = p.tiles;
    a.E = ex->E;
    a.T = p.T;
    a.k = p.k;
    if (shared) {
      const RolePlane &S0 = ex->shared[gateup ? NX_ROLE_GATE : NX_ROLE_DOWN];
      const RolePlane &S1 = ex->shared[gateup ? NX_ROLE_UP : NX_ROLE_DOWN];
      a.sqs0 = S0.qs;
      a.sqs1 = S1.qs;
      a.smeta0 = S0.meta;
      a.smeta1 = S1.meta;
    }
    a.perm_token = gateup ? p.perm_token : nullptr;
    a.out = ppart;
    a.out_stride = gateup ? 2 * F : H;
    a.out_split = pairs * a.out_stride;
    a.ks = gateup ? z.ks_g : z.ks_d;
    a.nks = gateup ? nks_g : nks_d;
    // At most 8 waves per CU.  Registers allow 12 (Q8_0: 8), but with as many
    // workgroups as fit the layers whose slices leave room got slower: 32 experts
    // of 2560 x 1536, top 4, Q2_K 12 tokens 63 -> 77 us; 16 of 4096 x 2304, top
    // 4, Q4_K 6 tokens 76 -> 84 us.
    const dim3 grid((unsigned)(c->num_cu * (MV_KW / a.ks))), block(64 * a.ks);
    const uint32_t lds = 2 * a.ks * MV_STEPS * 64 * sizeof(f32x4);
    if (gateup) {
      NX_TRY(launch(c, "mfv_gateup", [&] { go(c, k_mfv<true, FMT>, grid, block, lds, a); }));
      const size_t n = pairs * cd;
      auto swiglu = [&](auto kern) {
        return launch(c, "mfv_swiglu", [&] {
          go(c, kern, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, ppart, nks_g, pairs * 2 * F, n, F, rec);
        });
      };
      NX_TRY(nks_g <= 1 ? swiglu(k_mfv_swiglu<FMT, 1>)
                        : nks_g <= 2 ? swiglu(k_mfv_swiglu<FMT, 2>) : swiglu(k_mfv_swiglu<FMT, 4>));
    } else {
      NX_TRY(launch(c, "mfv_down", [&] { go(c, k_mfv<false, FMT>, grid, block, lds, a); }));
    }
  }
  return launch_combine(c, ppart, p.rw, p.rcnt, p.inv, p.T, p.k, H, shared, p.out, nks_d,
                        pairs * (size_t)H, p.residual);
}

}  // namespace

int mfv_max_tiles(int T, int k, int E, bool shared) {
  const long pairs = (long)T * k;
  return (int)((pairs + MV_M - 1) / MV_M + std::min<long>(E, pairs) +
               (shared ? (T + MV_M - 1) / MV_M : 0));
}

int mfv_records(nx_ctx *c, const nx_experts *ex, int T, int k, uint8_t **rec) {
  const MfvSizes z = mfv_sizes(shape_of(ex), T, k);
  void *p;
  NX_TRY(ws_get(c, WS_MFV_PART, z.bytes, &p));
  *rec = static_cast<uint8_t *>(p) + z.x_at;
  return NX_OK;
}

int launch_mfv_split(nx_ctx *c, const SplitJob &job) {
  return launch(c, "mfv_split", [&] {
    go(c, k_mfv_split, dim3((unsigned)((job.n + 15) / 16)), dim3(256), 0, job);
  });
}

int launch_mfv(nx_ctx *c, const MfvPlan &p) {
  const nx_experts *ex = p.ex;
  if (!mfv_supports(shape_of(ex)))
    return fail(NX_ERR_UNSUPPORTED,
                "the split-activation MFMA path takes Q4_K and Q2_K experts, or Q4_0 and Q8_0 "
                "experts whose hidden and FFN widths are multiples of 256");
  const bool shared = ex->Fs > 0;
  if (shared && ex->Fs != ex->F)
    return fail(NX_ERR_UNSUPPORTED,
                "the split-activation MFMA path takes a shared expert as wide as the routed ones");
  switch (ex->fmt) {
  case NX_FMT_Q4_0: return run_mfv<NX_FMT_Q4_0>(c, p);
  case NX_FMT_Q8_0: return run_mfv<NX_FMT_Q8_0>(c, p);
  case NX_FMT_Q2_K: return run_mfv<NX_FMT_Q2_K>(c, p);
  default: return run_mfv<NX_FMT_Q4_K>(c, p);
  }
}

}  // namespace nx
