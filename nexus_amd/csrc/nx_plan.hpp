// nx_plan.hpp — what a call's sizes alone decide: the path that AUTO takes, the
// split-activation path's workspace and runs, and the dense matvec's kernel.
//
// Plain C++ (no HIP): the CPU tests compile this header on its own.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

#include "../../include/nexus_hip.h"

namespace nx {

// an expert layer's format and widths (Fs: the shared expert's, or 0)
struct MoeShape {
  int fmt, E, H, F, Fs;
};

// ---- split-activation path (nx_mfv.hip)
constexpr int MV_K = 256;        // K positions per chunk
constexpr int MV_KW = 8;         // chunks per K slice, at most: one per wave
constexpr int REC_BYTES = 1152;  // operand record of a row's chunk (nx_split_dev.hpp)

// whether the path takes these experts: whole 256-weight chunks in both
// products (Q4_K and Q2_K always)
inline bool mfv_supports(const MoeShape &s) {
  if (s.fmt == NX_FMT_Q4_K || s.fmt == NX_FMT_Q2_K) return true;
  return (s.fmt == NX_FMT_Q4_0 || s.fmt == NX_FMT_Q8_0) && s.H % MV_K == 0 && s.F % MV_K == 0;
}

// Chunks per K slice: as many slices of at most MV_KW chunks as the row needs,
// of equal size (but for the last one's remainder)
inline int mv_slice_chunks(int nchunk) {
  if (nchunk <= 0) return 1;  // (no such layer is supported)
  const int n = (nchunk + MV_KW - 1) / MV_KW;
  return (nchunk + n - 1) / n;
}

// The path's workspace is one buffer.  At its start lie the gate/up sums, then
// the down sums; x's records follow the gate/up sums, and the gated rows'
// records end the buffer.  The SwiGLU kernel writes those when x's records are
// dead, the down pass its sums when the gate/up sums are, so each pair that is
// in use at one time lies apart.
struct MfvSizes {
  size_t pairs;
  int ks_g, ks_d, nks_g, nks_d;  // chunks per K slice, slices
  size_t x_at, act_at, bytes;    // offsets of x's and the gated rows' records; the buffer
};

inline MfvSizes mfv_sizes(const MoeShape &s, int T, int k) {
  // routed pairs, then one pair per token for the shared expert
  const size_t pairs = (size_t)T * k + (s.Fs > 0 ? (size_t)T : 0);
  const int cg = s.H / MV_K, cd = s.F / MV_K;
  MfvSizes z{};
  z.pairs = pairs;
  z.ks_g = mv_slice_chunks(cg);
  z.ks_d = mv_slice_chunks(cd);
  z.nks_g = (cg + z.ks_g - 1) / z.ks_g;
  z.nks_d = (cd + z.ks_d - 1) / z.ks_d;
  const size_t gate = (size_t)z.nks_g * pairs * 2 * s.F * sizeof(float);
  const size_t down = (size_t)z.nks_d * pairs * s.H * sizeof(float);
  const size_t xrec = (size_t)T * cg * REC_BYTES, arec = pairs * cd * REC_BYTES;
  z.x_at = gate;
  z.bytes = std::max({gate + xrec, gate + arec, down + arec});
  z.act_at = z.bytes - arec;
  return z;
}

// its workspace, but the routes'
inline size_t mfv_bytes(const MoeShape &s, int T, int k) { return mfv_sizes(s, T, k).bytes; }

// A workgroup's run of k_mfv's work, nseg segments (a tile's K slice) of npass
// passes each: units [u0, u1) of the line of passes from segment seg0 on.  With as
// many segments as workgroups or more, each takes one whole segment, the
// workgroups consecutive ones, and the rest is for the next round: the tiles of
// an expert stream its rows at about the same time, from the caches (DeepSeek
// 2048 tokens, a line of segments per workgroup against rounds: Q4_K 8.13 -> 6.36
// ms, Q8_0 12.95 -> 8.7).  In the last round, with fewer segments than workgroups,
// each workgroup stays in one of them: a run that crosses into another waits a
// second time for the chain of loads that finds the pairs, about two passes'
// time.  Where whole segments would leave some workgroups more than that much
// extra, the line is cut into equal runs.
struct MfvRun {
  int seg0, u0, u1;
};
constexpr MfvRun mfv_run(int block, int nblocks, int nseg, int npass) {
  if (nseg >= nblocks) return {block, 0, npass};
  if (nseg <= 0) return {0, 0, 0};
  const int work = nseg * npass, share = work / nblocks, over = work - share * nblocks;
  const int least = nblocks / nseg;  // workgroups of a segment, at least
  if ((npass + least - 1) / least <= share + 2) {
    // the first `more` segments have one workgroup more
    const int more = nblocks - least * nseg, past = more * (least + 1);
    const int n = block < past ? least + 1 : least;
    const int seg = block < past ? block / n : more + (block - past) / n;
    const int at = block < past ? block - seg * n : block - past - (seg - more) * n;
    return {seg, npass * at / n, npass * (at + 1) / n};
  }
  return {0, share * block + over * block / nblocks, share * (block + 1) + over * (block + 1) / nblocks};
}

// ---- AUTO
// The path of a call on T tokens, top k.  aligned: x on 16 bytes, which the
// split path needs and the others do not.  scratch: the bytes its workspace may
// take (SIZE_MAX where it is allocated).
//
// AUTO takes bf16 operands on the grouped GEMM: fp16's range ends at 65504,
// which SwiGLU activations of real models can pass; bf16 keeps float32's range,
// runs as fast here, and stays within the MFMA bar.
inline int auto_path(const MoeShape &s, int T, int k, bool aligned, size_t scratch) {
  if (s.fmt == NX_FMT_F16 || s.fmt == NX_FMT_BF16) return NX_PATH_GEMV;
  const bool shared = s.Fs > 0;
  // Tokens per active expert, with the active count expected under
  // uniform routing, E (1 - (1 - k/E)^T).
  const double kk = std::min(1.0, (double)k / s.E);
  const double act = std::max(1.0, s.E * (1.0 - std::pow(1.0 - kk, (double)T)));
  const double tpe = (double)T * k / act;
  // The split path streams the active experts' weights at 4.3 TB/s behind
  // about 30 us of launches, so it wins over wider ranges where an expert is
  // large: `large` from 7 M weights a matrix (measured at 4096 x 1792 and up).
  // In the fixed scratch array of nx_moe_forward_noalloc a batch that its
  // workspace would not fit keeps the narrower ranges, whose other paths
  // need less.
  const bool split_fmt = aligned && mfv_supports(s);
  const bool fits = split_fmt && (scratch == SIZE_MAX || mfv_bytes(s, T, k) + (size_t)T * k * 64 +
                                                                 (size_t)s.E * 64 + (1u << 20) <=
                                                             scratch);
  const double weights = (double)s.H * s.F;
  const bool large = fits && weights >= 7e6;
  const bool q8 = s.fmt == NX_FMT_Q8_0;
  if (s.fmt == NX_FMT_Q2_K) {
    // The GEMV or the split-activation path (Q2_K has no grouped GEMM).
    // Measured (us, GEMV / split): Mixtral 2 tokens 93 / 84, 4: 174 / 112, 8:
    // 276 / 153, 32: 797 / 170, 128: 2840 / 364; Qwen3 4 tokens 46 / 40, 8: 77 /
    // 52, 128: 588 / 97; DeepSeek with its shared expert 2 tokens 121 / 104, 4:
    // 305 / 175.  (The limits are those of a slower split kernel.)
    if (!split_fmt) return NX_PATH_GEMV;
    if (shared) return (s.Fs == s.F && T >= 4) ? NX_PATH_MFMA_SPLIT : NX_PATH_GEMV;
    return (tpe >= 1.8 || ((long)T * k >= 64 && tpe >= 1.2)) ? NX_PATH_MFMA_SPLIT : NX_PATH_GEMV;
  }
  if (split_fmt && shared && s.Fs == s.F && (large || s.fmt == NX_FMT_Q4_K)) {
    // A shared expert sees every token: the GEMV walks it a token pair at
    // a time, the split-activation path 16 tokens at a time.  Measured
    // (DeepSeek shapes, us, GEMV / split / grouped GEMM): Q4_K 2 tokens 107 /
    // 117 / 238, 4: 263 / 183 / 283, 8: 874 / 331 / 580, 27: - / 814 / 1223,
    // 128: - / 1543 / 2046, 256 (8 per routed expert): - / 1702 / 2141, 384
    // (12): - / 1853 / 2195; Q4_0 2: 98 / 123 / 235, 4: 237 / 200 / 293, 27: - /
    // 839 / 1187, 384: - / 1870 / 2147; Q8_0 4: 315 / 313 / 370, 8: 847 / 529 /
    // 650, 128: - / 2398 / 2559, 256: - / 2696 / 2700, 384: - / 2934 / 2772.
    if (tpe >= (large && !q8 ? 12.0 : 8.0)) return NX_PATH_MFMA_BF16;
    return T >= (q8 ? 6 : 4) ? NX_PATH_MFMA_SPLIT : NX_PATH_GEMV;
  }
  if (split_fmt && !shared) {
    // The GEMV re-reads an expert's weights per pair of its tokens, the
    // split-activation path reads them once per 16 tokens, and the grouped
    // GEMM once, at bf16 operands.  Measured (us, GEMV / split / grouped
    // GEMM, means over four to thirty routings: the GEMV's time hangs on how the
    // tokens pair up) by tokens per expert.  Mixtral Q4_K 1.1: 90 / 94 / 176,
    // 1.3: 150 / 115 / 223, 2.2: 382 / 172 / 296, 8: - / 213 / 305, 12: - / 225 /
    // 307, 16: - / 271 / 314; Q4_0 1.3: 99 / 114 / 216, 1.46: 130 / 132 / 243,
    // 1.64: 160 / 144 / -, 12: - / 232 / 300; Q8_0 1.5: 193 / 213 / 286, 2.0: 300
    // / 265 / 338, 8: - / 344 / 364, 12: - / 370 / 368, 16: - / 463 / 369; Qwen3
    // Q4_K 1.1: 51 / 44 / 68, 1.3: 124 / 61 / 93, 8: - / 123 / 152, 12.5: - / 136 /
    // 154, 16: - / 154 / 156.  16 experts of 4096 x 2304, top 4, 1.3: Q4_K 61 /
    // 57, Q4_0 51 / 61; 1.46: Q4_0 68 / 65; 2.0: Q8_0 129 / 111.
    // Layers of 7 M weights, 4 experts of 2048 x 3584: Q4_K 6 pairs 34 / 36, 8
    // pairs 40 / 37, Q8_0 10 pairs 42 / 43; 8 of 4096 x 1792: Q4_K 6 pairs 37 /
    // 39, 8 pairs 45 / 43, Q8_0 14 pairs 52 / 56, 16 pairs 61 / 56.  Smaller ones:
    // 8 of 1024 x 2048 Q4_K 1.5: 34 / 32, 1.6: 41 / 32, Q8_0 2.2: 33 / 37, 3.1: 40
    // / 38; 8 of 512 x 1024 Q4_K 1.6: 30 / 30, 2.2: 36 / 31, Q8_0 3.1: 35 / 36; 64
    // of 1024 x 768, top 8, Q4_K 1.1: 31 / 31, 1.3: 47 / 37, Q8_0 1.28: 38 / 42,
    // 1.36: 49 / 45.
    const long pairs = (long)T * k;
    if (tpe >= (large && !q8 ? 13.0 : 12.0)) return NX_PATH_MFMA_BF16;
    // the least tokens per expert of a large layer; the smallest of them with a
    // few pairs are bound by the launches, of which the GEMV has fewer
    const double least = q8 ? 2.0 : s.fmt == NX_FMT_Q4_0 ? 1.5 : 1.28;
    const bool few = weights < 9e6 && pairs < (q8 ? 16 : 8);
    if (tpe >= 3.0 || (pairs >= 64 && tpe >= 1.2) || (fits && pairs >= 40 && tpe >= (q8 ? 1.3 : 1.25)) ||
        (large && !few && tpe >= least) || (fits && !q8 && !few && weights >= 2e6 && tpe >= 1.6))
      return NX_PATH_MFMA_SPLIT;
    return NX_PATH_GEMV;
  }
  if (s.fmt == NX_FMT_F32) {
    // f32 weights keep their precision on the GEMV; the bf16 grouped GEMM
    // only once experts see 32 tokens on average
    const long active_max = std::min<long>(s.E, (long)T * k);
    return ((long)T * k >= 32 * active_max) ? NX_PATH_MFMA_BF16 : NX_PATH_GEMV;
  }
  // The grouped GEMM from ~3 tokens per routed expert (Mixtral Q8_0 and
  // Q4_0 at 8 and 16 tokens, Qwen3 Q8_0 at 32), or from 6 tokens when a
  // shared expert sees them all: the GEMV passes over the shared expert
  // per pair of tokens and over the routed experts per token group
  // (DeepSeek shapes with a shared expert: GEMV 0.29 / 0.81 / 10.5 ms
  // at 4 / 8 / 32 tokens, grouped GEMM 0.36 / 0.61 / 1.44 ms).
  return (tpe >= 3.0 || (shared && T >= 6)) ? NX_PATH_MFMA_BF16 : NX_PATH_GEMV;
}

// ---- dense matvec on MFMA (nx_mfd.hip)
constexpr int MD_K = 256;    // columns per chunk
constexpr int MD_WAVES = 8;  // waves per workgroup

// Whether a matrix and token count run there.  From five tokens: the GEMV's time
// grows with every two tokens, and at five it is behind at nearly every size
// (us, GEMV / MFMA: 512 x 512 Q4_K 14.2 / 5.7, 1024 x 2048 Q4_0 16.7 / 5.5, 4096
// x 14336 Q4_K 45 / 26, 32000 x 4096 Q8_0 70 / 40); up to four tokens a call
// gives each token the bits of a call of its own.  Not so where the GEMV's rows
// are one round of its workgroups and few rows leave each MFMA workgroup alone
// with a long row: up to 256 rows and six tokens, Q4_K of more than 40 chunks (256
// x 11008 18.1 / 20.0, x 14336 19.4 / 23.4; 384 rows 30 / 23; 7 tokens 25 / 23;
// 40 chunks 17.5 / 17.6) and Q8_0 of 17 to 32 (256 x 5120 9.7 / 10.4, x 7168 10.6
// / 12.7, x 8192 11.1 / 13.0; 16 chunks 10.7 / 8.2, 40: 17.7 / 15.3; 384 rows 14.4 /
// 12.8).  Q4_0 is level at 56 chunks (19.5 / 19.7).
inline bool mfd_sizes(int fmt, int rows, int cols, int T) {
  if (fmt != NX_FMT_Q4_K && fmt != NX_FMT_Q4_0 && fmt != NX_FMT_Q8_0) return false;
  if (T <= 4 || cols % MD_K != 0) return false;
  const int n = cols / MD_K;
  if (T <= 6 && rows <= 256 && ((fmt == NX_FMT_Q4_K && n > 40) || (fmt == NX_FMT_Q8_0 && n > 16 && n <= 32)))
    return false;
  return true;
}

// A workgroup's shape: r row tiles of 16 per wave, kw chunk groups of 8 / kw
// waves and as many token tiles.
struct MfdShape {
  int r, kw;
  int rows() const { return 16 * r * (MD_WAVES / kw); }
  int tokens() const { return 16 * (MD_WAVES / kw); }
};

// One workgroup fits a CU (its stage fills the LDS), so a shape costs its
// rounds of the CUs times its steps of kw chunks.  Step times (us, one
// MI355X, all rows and tokens of a shape in use, the formats within 10%):
// a step costs its 8 waves about 4 us of conversion, staging and waits, and
// little more for more rows or token tiles, so the larger shapes win where
// they fill the CUs.  4096 x 4096 Q4_K, 1 x 8 / 2 x 8 / 4 x 8 / 2 x 4 / 1 x 2 /
// 2 x 2: 16 tokens 11.1 / 12.0 / 16.7 / 23.8 / 41.8 / 53.1 us; 64 tokens 40.3
// / 24.5 / 18.2 / 24.4 / 41.8 / 53.4; 509 tokens 330 / 187 / 135 / 98 / 91 /
// 62.
inline MfdShape mfd_shape(int rows, int nchunk, int T, int num_cu) {
  static const struct {
    MfdShape s;
    double step_us;
  } shapes[] = {{{1, 8}, 4.0}, {{2, 8}, 4.5}, {{4, 8}, 6.8}, {{1, 4}, 4.4},
                {{2, 4}, 5.2}, {{1, 2}, 4.8}, {{2, 2}, 6.2}};
  MfdShape s{1, 8};
  double best = 0.0;
  for (const auto &t : shapes) {
    const long wgs = (long)((rows + t.s.rows() - 1) / t.s.rows()) * ((T + t.s.tokens() - 1) / t.s.tokens());
    const double us = t.step_us * (double)((wgs + num_cu - 1) / num_cu) *
                      (double)((nchunk + t.s.kw - 1) / t.s.kw);
    if (best == 0.0 || us < best) best = us, s = t.s;
  }
  return s;
}

}  // namespace nx
