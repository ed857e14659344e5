"""What a call's sizes decide (nexus_amd/csrc/nx_plan.hpp): the path AUTO takes,
the split-activation path's workspace and runs, and the dense matvec's kernel.
CPU only: the header is plain
C++ and is compiled on its own with the host compiler.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "nexus_amd", "csrc")
GXX = shutil.which("g++")

pytestmark = pytest.mark.skipif(GXX is None, reason="no host C++ compiler")


def run(tmp_path, body):
    """Compiles `body` as main()'s statements over the header and runs it."""
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text('#include <cstdio>\n#include <vector>\n#include "nx_plan.hpp"\nusing namespace nx;\n'
                   "int main() {\n  int bad = 0;\n" + body + "\n  return bad ? 1 : 0;\n}\n")
    r = subprocess.run([GXX, "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-2000:]}"
    return r.stdout


def test_any_width_has_a_path_in_the_scratch_array(tmp_path):
    """Every format and width that an expert set may have gets a path, with and
    without a limit on the workspace; a layer that is not in whole 256-weight
    chunks (narrower than one among them) never the split path."""
    run(tmp_path, r"""
  const int fmts[] = {NX_FMT_F32, NX_FMT_F16, NX_FMT_BF16, NX_FMT_Q4_0, NX_FMT_Q8_0, NX_FMT_Q4_K, NX_FMT_Q2_K};
  for (int fmt : fmts)
    for (int H : {1, 32, 96, 128, 224, 256, 288, 512, 4096})
      for (int F : {1, 32, 96, 128, 224, 256, 288, 512, 14336})
        for (int Fs : {0, 32, F})
          for (int T : {1, 2, 3, 5, 8, 33, 1000})
            for (int k : {1, 2, 8})
              for (size_t scratch : {(size_t)64 << 20, SIZE_MAX}) {
                const bool super = fmt == NX_FMT_Q4_K || fmt == NX_FMT_Q2_K;
                if (super && (H % 256 || F % 256)) continue;  // refused when created
                const int p = auto_path({fmt, 8, H, F, Fs}, T, k, true, scratch);
                const bool chunks = H % 256 == 0 && F % 256 == 0 && fmt != NX_FMT_F32 &&
                                    fmt != NX_FMT_F16 && fmt != NX_FMT_BF16;
                if (p == NX_PATH_AUTO || (p == NX_PATH_MFMA_SPLIT && !chunks)) {
                  std::printf("fmt %d H %d F %d Fs %d T %d k %d: path %d\n", fmt, H, F, Fs, T, k, p);
                  ++bad;
                }
              }
""")


def test_unaligned_inputs_stay_off_the_split_path(tmp_path):
    """The split path reads x in 16-byte runs.  Calls on other addresses take
    the rule of the formats without it: the grouped GEMM (Q2_K: none) from 3
    tokens per expert or 6 with a shared expert, the GEMV below."""
    run(tmp_path, r"""
  for (int fmt : {NX_FMT_Q4_0, NX_FMT_Q8_0, NX_FMT_Q4_K, NX_FMT_Q2_K})
    for (int H : {256, 1024, 4096})
      for (int F : {256, 2048, 14336})
        for (int Fs : {0, 32 * 8, F})
          for (int T = 1; T < 400; ++T)
            for (size_t scratch : {(size_t)64 << 20, SIZE_MAX}) {
              const double tpe = T * 2 / (8 * (1.0 - std::pow(0.75, (double)T)));
              const int want = fmt != NX_FMT_Q2_K && (tpe >= 3.0 || (Fs && T >= 6)) ? NX_PATH_MFMA_BF16
                                                                                    : NX_PATH_GEMV;
              const int p = auto_path({fmt, 8, H, F, Fs}, T, 2, false, scratch);
              if (p != want) {
                std::printf("fmt %d H %d F %d Fs %d T %d: path %d\n", fmt, H, F, Fs, T, p);
                ++bad;
              }
            }
""")


def test_split_workspace(tmp_path):
    """The split path's buffer: x's records apart from the gate/up sums, the
    gated rows' records apart from both passes' sums, all inside it and on
    128-byte lines.  It is never larger than f32 gated rows and the sums of both
    passes side by side, in K slices of 4 and 3 chunks: a call of the
    no-allocation entry point that fitted with those still does."""
    run(tmp_path, r"""
  for (int cg = 1; cg <= 64; ++cg)
    for (int cd = 1; cd <= 112; ++cd)
      for (int k : {1, 2, 4, 8})
        for (int shared = 0; shared < 2; ++shared)
          for (int T : {1, 3, 17, 4099}) {
            const MoeShape s{NX_FMT_Q4_K, 64, 256 * cg, 256 * cd, shared ? 256 * cd : 0};
            const MfvSizes z = mfv_sizes(s, T, k);
            const size_t p = z.pairs, f = sizeof(float);
            const size_t gate = z.nks_g * p * 2 * s.F * f, down = z.nks_d * p * s.H * f;
            const size_t xrec = (size_t)T * cg * REC_BYTES, arec = p * cd * REC_BYTES;
            const size_t most = ((cg + 3) / 4 * 2 * s.F + s.F + (size_t)((cd + 2) / 3) * s.H) * p * f;
            bool ok = p == (size_t)T * (k + shared) && z.ks_g >= 1 && z.ks_g <= MV_KW && z.ks_d >= 1 &&
                      z.ks_d <= MV_KW && z.nks_g * z.ks_g >= cg && (z.nks_g - 1) * z.ks_g < cg &&
                      z.nks_d * z.ks_d >= cd && (z.nks_d - 1) * z.ks_d < cd;
            ok = ok && z.x_at >= gate && z.x_at + xrec <= z.bytes && z.act_at >= gate && z.act_at >= down &&
                 z.act_at + arec <= z.bytes && z.x_at % 128 == 0 && z.act_at % 128 == 0 && z.bytes <= most;
            if (!ok) {
              std::printf("cg %d cd %d k %d shared %d T %d: %zu bytes, at most %zu\n", cg, cd, k, shared, T,
                          z.bytes, most);
              ++bad;
            }
          }
""")


def test_split_runs_cover_the_line_once(tmp_path):
    """The workgroups' runs of the split kernel cover the whole line, each unit
    once; whole segments but in the last round, where none is longer than an
    equal share and two passes."""
    run(tmp_path, r"""
  for (int nb : {256, 512, 304, 1})
    for (int nseg = 0; nseg <= 1100; nseg += nseg < 40 ? 1 : 13)
      for (int npass : {2, 4, 5, 8, 20, 32, 64, 112, 448}) {
        std::vector<int> seen((size_t)nseg * npass);
        for (int first = 0, left = nseg; left > 0; first += nb, left -= nb)
          for (int b = 0; b < nb; ++b) {
            const MfvRun r = mfv_run(b, nb, left, npass);
            const long share = ((long)left * npass + nb - 1) / nb;
            if (r.u1 < r.u0 || r.u1 - r.u0 > (left >= nb ? npass : share + 2)) ++bad;
            for (int u = r.u0; u < r.u1; ++u) ++seen.at((size_t)(first + r.seg0) * npass + u);
          }
        for (int v : seen)
          if (v != 1) {
            std::printf("%d workgroups, %d segments of %d\n", nb, nseg, npass);
            ++bad;
            break;
          }
      }
""")


# fmt, E, H, F, shared F, top k, token counts at which AUTO's path changes:
# the GEMV below the first, the split path from it, the grouped GEMM from the second
AUTO_LIMITS = [
    ("Q4_K", 8, 4096, 14336, 0, 2, 3, 52),   # 1.30 and 13 tokens per expert
    ("Q4_0", 8, 4096, 14336, 0, 2, 5, 52),   # 1.64
    ("Q8_0", 8, 4096, 14336, 0, 2, 7, 48),   # 2.02 and 12
    ("Q4_0", 16, 4096, 2304, 0, 4, 5, 52),
    ("Q8_0", 16, 4096, 2304, 0, 4, 7, 48),
    ("Q4_K", 8, 4096, 1792, 0, 2, 4, 52),    # 7.3 M weights: from 8 pairs
    ("Q4_K", 4, 2048, 3584, 0, 2, 4, 26),
    ("Q4_0", 4, 2048, 3584, 0, 2, 4, 26),
    ("Q8_0", 8, 4096, 1792, 0, 2, 8, 48),    # ... from 16 pairs
    ("Q8_0", 4, 2048, 3584, 0, 2, 6, 24),    # ... or 3 tokens per expert
    ("Q4_K", 8, 1024, 2048, 0, 2, 5, 48),    # 2.1 M weights: 1.64
    ("Q8_0", 8, 1024, 2048, 0, 2, 12, 48),   # 3.1
    ("Q4_K", 8, 512, 1024, 0, 2, 12, 48),
    ("Q4_K", 64, 1024, 768, 0, 8, 5, 96),    # 40 pairs at 1.28
    ("Q8_0", 64, 1024, 768, 0, 8, 6, 96),    # 1.36
    ("Q4_K", 128, 2048, 768, 0, 8, 8, 192),  # 64 pairs
    ("Q4_K", 256, 7168, 2048, 2048, 8, 4, 384),  # a shared expert: 4 tokens, 12 per expert
    ("Q4_0", 256, 7168, 2048, 2048, 8, 4, 384),
    ("Q8_0", 256, 7168, 2048, 2048, 8, 6, 256),  # 6 tokens, 8 per expert
    ("Q4_K", 16, 512, 512, 512, 4, 4, 32),       # a small one: 8 per expert
    ("Q4_0", 16, 512, 512, 512, 4, 6, 6),        # ... without the split path
    ("Q4_K", 16, 512, 512, 1024, 4, 6, 6),       # a shared expert of another width
]


def test_auto_limits(tmp_path):
    """Where AUTO changes its path, over 1 to 512 tokens."""
    rows = ",".join("{{NX_FMT_%s, %d, %d, %d, %d}, %d, %d, %d}" % r for r in AUTO_LIMITS)
    run(tmp_path, r"""
  const struct { MoeShape s; int k, split, gemm; } rows[] = {""" + rows + r"""};
  for (const auto &r : rows)
    for (int T = 1; T <= 512; ++T) {
      const int want = T < r.split ? NX_PATH_GEMV : T < r.gemm ? NX_PATH_MFMA_SPLIT : NX_PATH_MFMA_BF16;
      const int p = auto_path(r.s, T, r.k, true, SIZE_MAX);
      if (p != want) {
        std::printf("fmt %d, %d experts of %d x %d, T %d: path %d\n", r.s.fmt, r.s.E, r.s.H, r.s.F, T, p);
        ++bad;
      }
    }
""")


def test_auto_in_the_scratch_array(tmp_path):
    """Within a limit on the workspace AUTO takes the split path over its wider
    ranges only where that fits, and otherwise as without the wider ranges."""
    run(tmp_path, r"""
  const size_t limit = (size_t)64 << 20;
  const MoeShape s{NX_FMT_Q4_K, 64, 2304, 4096, 0};
  for (int T = 1; T <= 300; ++T) {
    const int p = auto_path(s, T, 8, true, limit), free = auto_path(s, T, 8, true, SIZE_MAX);
    if (mfv_bytes(s, T, 8) > limit && free == NX_PATH_MFMA_SPLIT && T * 8 >= 12 * 64 && p != NX_PATH_MFMA_BF16) ++bad;
    if (mfv_bytes(s, T, 8) + (2u << 20) < limit && p != free) ++bad;
  }
  if (auto_path(s, 101, 8, true, limit) != NX_PATH_MFMA_BF16) ++bad;
  if (auto_path(s, 101, 8, true, SIZE_MAX) != NX_PATH_MFMA_SPLIT) ++bad;
""")


def test_dense_kernel(tmp_path):
    """The dense matvec runs on the matrix cores from five tokens of whole
    256-column chunks, but for up to six tokens of at most 256 long rows."""
    run(tmp_path, r"""
  for (int fmt : {NX_FMT_F32, NX_FMT_F16, NX_FMT_BF16, NX_FMT_Q2_K, NX_FMT_Q4_0, NX_FMT_Q8_0, NX_FMT_Q4_K})
    for (int rows : {1, 16, 255, 256, 257, 4096})
      for (int cols = 32; cols <= 14336; cols += 32)
        for (int T : {1, 4, 5, 6, 7, 16, 512}) {
          const bool fits = fmt == NX_FMT_Q4_0 || fmt == NX_FMT_Q8_0 || fmt == NX_FMT_Q4_K;
          const bool small = rows <= 256 && T <= 6;
          const bool gemv = small && ((fmt == NX_FMT_Q4_K && cols > 10240) ||
                                      (fmt == NX_FMT_Q8_0 && cols > 4096 && cols <= 8192));
          if (mfd_sizes(fmt, rows, cols, T) != (fits && T >= 5 && cols % 256 == 0 && !gemv)) {
            std::printf("fmt %d, %d x %d, T %d\n", fmt, rows, cols, T);
            ++bad;
          }
        }
""")


def test_dense_instances(tmp_path):
    """The sizes of the dense matvec's instance test choose each of the seven
    instances on 256 CUs, over several steps with a ragged last one."""
    from test_gpu_matvec_mfma import INSTANCES

    assert len({c[:2] for c in INSTANCES}) == 7
    rows = ",".join("{%d, %d, %d, %d, %d}" % c for c in INSTANCES)
    run(tmp_path, r"""
  const struct { int r, kw, rows, cols, T; } cases[] = {""" + rows + r"""};
  for (const auto &c : cases) {
    const int n = c.cols / MD_K;
    const MfdShape s = mfd_shape(c.rows, n, c.T, 256);
    for (int fmt : {NX_FMT_Q4_K, NX_FMT_Q4_0, NX_FMT_Q8_0})
      if (!mfd_sizes(fmt, c.rows, c.cols, c.T)) ++bad;
    if (s.r != c.r || s.kw != c.kw || n <= s.kw || n % s.kw == 0 || c.rows % s.rows() == 0 || c.T % s.tokens() == 0) {
      std::printf("%d x %d, %d tokens: %d x %d\n", c.rows, c.cols, c.T, s.r, s.kw);
      ++bad;
    }
  }
""")
