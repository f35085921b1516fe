// Which kernel runs a product of more than 64 rows: a rule of the host alone (standard C++,
// no HIP), so that it can be checked without a device.
#pragma once

#include <math.h>
#ifdef T2I_TUNING
#include <stdio.h>
#include <stdlib.h>
#endif

#include <algorithm>

namespace t2i_host {

// Rows from which a product is a prompt batch: the LDS-tiled kernels serve it whatever its
// shape (N a multiple of 128); from 65 rows they do where they are faster.
constexpr int PROMPT_ROWS = 512;

// What runs an M x K x N product without a fused norm: the decode linear's tiles (NONE),
// the 64 x 128 kernel (TILES64) or a form of the ring kernel (RING: row fragments a wave,
// columns a lane, waves along N, k slices).
struct PromptPlan {
  enum Kind { NONE, TILES64, RING } kind;
  int cfg[4];
};

// A kernel's time (us) as a fit, g = K / 128 groups: with up to `res` workgroups on each of the
// 256 CUs, level o (o workgroups on the fullest CU) is one[o] = {at its start, a group, across
// the level, a group of that}; with more it is many = {fixed, a group, a round of 256 res, a
// group of that, the last round's idle share, a group of that}.
struct PromptFit {
  int rows, cols, res;
  double one[3][4], many[6];
  double us(int M, int K, int N) const {
    const double t = (double)((M + rows - 1) / rows) * (N / cols), g = K / 128, slots = 256.0 * res;
    if (t <= slots) {
      const int o = std::max(1, (int)ceil(t / 256)) - 1;
      const double share = t / 256 - o;
      return one[o][0] + one[o][1] * g + share * (one[o][2] + one[o][3] * g);
    }
    const double r = t / slots, idle = ceil(r) - r;
    return many[0] + many[1] * g + r * (many[2] + many[3] * g) + idle * (many[4] + many[5] * g);
  }
};

// The ring kernel's forms: 64 x 128 tiles (two workgroups a CU), 64 x 128 with K in two slices,
// 128 x 256 (its estimate is the least sure, 5 to 95 % of the fit -7 to +8 %: it is taken from
// 3 % on).  One fit serves own and given row sums, which differ by 1 %; with given ones the
// first form is nowhere the fastest, and is not built for them.
struct PromptForm {
  int cfg[4];
  PromptFit fit;
  double over;
  bool given;
};
constexpr PromptForm PROMPT_FORMS[] = {
    {{4, 2, 4, 1}, {64, 128, 2, {{5.25, 0.8, 0.17, 0.06}, {4.86, 1.28, 1.3, 0.07}}, {1.77, 0.22, 4.61, 1.22, 2.79, 0.47}}, 1.0, false},
    {{4, 2, 4, 2}, {64, 128, 1, {{5.56, 0.56, -0.45, 0.17}}, {0.44, 0.15, 4.73, 0.62, 4.49, 0.51}}, 1.0, true},
    {{8, 2, 8, 1}, {128, 256, 1, {{8.28, 1.51, 2.43, 0.27}}, {1.98, 0.31, 9.43, 1.7, 5.67, 1.16}}, 1.03, true},
};
// The 64 x 128 kernel, with its own row sums and with given ones (which save it a third of its
// MFMAs).
constexpr PromptFit TILES64_FIT[2] = {
    {64, 128, 3, {{-1.64, 1.1, 2.95, 0.02}, {4.55, 1.29, 0.23, 0.2}, {6.01, 1.83, -0.96, 0.37}},
     {4.46, 0.02, 2.37, 2.05, -1.16, 0.4}},
    {64, 128, 3, {{-2.09, 1.08, 3.39, -0.02}, {4.35, 1.21, 1.11, 0.07}, {6.5, 1.66, -0.76, 0.24}},
     {5.92, -0.1, 2.15, 1.84, -1.71, 0.49}},
};

// Whether the plan's kernel exists and can run a product of N columns, on given row sums or its
// own.  The launchers refuse a product that fails this (columns past the last whole tile would
// stay unwritten).
inline bool prompt_form_serves(const PromptPlan& pl, int N, bool sums) {
  if (pl.kind == PromptPlan::TILES64) return N % 128 == 0;
  if (pl.kind == PromptPlan::RING)
    for (const PromptForm& f : PROMPT_FORMS)
      if (std::equal(f.cfg, f.cfg + 4, pl.cfg)) return N % f.fit.cols == 0 && (f.given || !sums);
  return false;
}

// The kernel for an M x K x N product of more than 64 rows: the one of the least estimated time.
// Fits and choice are from a sweep of M = 65 .. 8192 over the decoders' eight projection shapes,
// every kernel graph-launched on both kinds of row sums and behind the fused q|k|v epilogue (572
// measured choices): the fits are within 4 to 8 % of nine times in ten, the choice is within 8 %
// of the fastest (11 % at 1024 x 2048 -> 12288), and 3 choices are 3 to 4 % slower than the
// kernel that served the product before the ring kernel came.  The decode tiles (fewer than 512
// rows) are 1.5 + 1 + 0.143 g a round of 256 workgroups of 16 rows x 64 columns.  A form of 32 x
// 64 tiles with K in four slices was measured nowhere faster by more than 0.2 %.
// sums: the rows' sums are given.  The choice depends on M, K, N and that alone, so a
// projection's fused and plain forms give the same bits.  Products of two to four groups lie
// outside the sweep: no ring launch was measured under 8.5 us (K = 256: 173 rows -> 5120 7.7 on
// the decode tiles, 8.9 on the ring; 410 -> 6144 17.0, 9.9).
inline PromptPlan plan_prompt(int M, int K, int N, bool sums) {
  PromptPlan best{PromptPlan::NONE, {0, 0, 0, 0}};
  const bool prompt = M >= PROMPT_ROWS;
  if (M <= 64 || N % 128) return best;
  // the ring kernel addresses its tensors with 32-bit byte offsets
  const bool ring = (double)K * N / 2 < 4e9 && (double)M * K / 16 < 4e9;
  if (prompt) best.kind = PromptPlan::TILES64;
#ifdef T2I_TUNING
  // a form for every product that it can serve, the 64 x 128 kernel or the decode tiles for the rest
  if (const char* env = getenv("T2I_PROMPT")) {
    PromptPlan o{PromptPlan::RING, {0, 0, 0, 0}};
    if (ring && sscanf(env, "%d,%d,%d,%d", &o.cfg[0], &o.cfg[1], &o.cfg[2], &o.cfg[3]) == 4 &&
        prompt_form_serves(o, N, sums))
      return o;
    return best;
  }
#endif
  if (!ring) return best;
  const double g = K / 128;
  double least = prompt ? TILES64_FIT[sums].us(M, K, N) : 1.5 + ceil((M + 15) / 16 * (N / 64.0) / 256) * (1 + 0.143 * g);
  for (const PromptForm& f : PROMPT_FORMS) {
    if (!prompt_form_serves({PromptPlan::RING, {f.cfg[0], f.cfg[1], f.cfg[2], f.cfg[3]}}, N, sums)) continue;
    const double us = f.over * std::max(8.5, f.fit.us(M, K, N));
    if (us < least) {
      least = us;
      best = PromptPlan{PromptPlan::RING, {f.cfg[0], f.cfg[1], f.cfg[2], f.cfg[3]}};
    }
  }
  return best;
}

}  // namespace t2i_host
