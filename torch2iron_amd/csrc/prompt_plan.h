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

// Whether the plan's kernel can run a product of N columns; batch: with what only a prompt
// batch's calls have (given row sums, output sums, the fused q|k|v epilogue), which needs
// tiles of whole 128-column pieces.  The launchers refuse a product that fails this.
inline bool prompt_form_serves(const PromptPlan& pl, int N, bool batch) {
  if (pl.kind == PromptPlan::NONE) return false;
  if (pl.kind == PromptPlan::RING && (pl.cfg[1] < 1 || pl.cfg[1] > 8 || pl.cfg[2] < 1 || pl.cfg[2] > 16)) return false;
  const int cols = pl.kind == PromptPlan::TILES64 ? 128 : 16 * pl.cfg[1] * pl.cfg[2];
  return N % cols == 0 && !(batch && cols % 128);
}

// The kernel for an M x K x N product of more than 64 rows, from a fit of every form's time
// (us; g = K / 128 groups, R rounds of the chip's 256 CUs) to a sweep of M = 65 .. 8192 over
// the decoders' eight projection shapes, graph-launched.  Each line's constants are the fit;
// the fits are within 15 % of the sweep and the choice within 8 % of the fastest form.
//   decode tiles of 16 rows (fewer than 512 rows):  3.5 + 0.00085 x (16-row x 64-column tiles) x g
//   2,2,2,4: 32 x 64, K in 4 slices (fewer than 512 rows):  2.5 + R (3.3 + 0.28 g)
//   4,2,4,2: 64 x 128, K in 2 slices:  2.5 + R (4 + 0.66 g)
//   4,2,4,1: 64 x 128, two workgroups a CU:  2 + 5.5 + 1.22 g a pair, 4 + 0.88 g a single
//   8,2,8,1: 128 x 256:  3 + 6.5 + g (1.36 .. 1.8 with the round's fill) a round, and a tenth for
//     its one workgroup a CU with the fused q|k|v epilogue (5000 rows, K = 1024: 82 against 81 us)
//   the 64 x 128 kernel of three workgroups a CU (512 rows and more):  3 + 1.05 g, 2 + 1.65 g,
//   2.5 + 2.3 g with one, two, three on a CU
// The choice depends on M, K and N alone, so a projection's fused and plain forms give the
// same bits.
inline PromptPlan plan_prompt(int M, int K, int N) {
  PromptPlan best{PromptPlan::NONE, {0, 0, 0, 0}};
  const double g = K / 128;
  double cost = 1e30;
  auto offer = [&](double c, PromptPlan::Kind kind, int a, int b, int d, int e) {
    if (c < cost) {
      cost = c;
      best = PromptPlan{kind, {a, b, d, e}};
    }
  };
  const bool prompt = M >= PROMPT_ROWS;
  if (M <= 64) return best;
  if (prompt && N % 128) return best;
  // the ring kernel addresses its tensors with 32-bit byte offsets
  const bool ring = (double)K * N / 2 < 4e9 && (double)M * K / 16 < 4e9;
#ifdef T2I_TUNING
  // a form for every product that it can serve, the 64 x 128 kernel or the decode tiles for the rest
  if (const char* env = getenv("T2I_PROMPT")) {
    PromptPlan o{PromptPlan::RING, {0, 0, 0, 0}};
    if (ring && sscanf(env, "%d,%d,%d,%d", &o.cfg[0], &o.cfg[1], &o.cfg[2], &o.cfg[3]) == 4 &&
        prompt_form_serves(o, N, false))
      return o;
    return PromptPlan{prompt ? PromptPlan::TILES64 : PromptPlan::NONE, {0, 0, 0, 0}};
  }
#endif
  if (!prompt) offer(3.5 + 0.00085 * ((M + 15) / 16) * (N / 64.0) * g, PromptPlan::NONE, 0, 0, 0, 0);
  const double t64 = (double)((M + 63) / 64) * (N / 128);
  if (prompt)
    offer(t64 <= 256 ? 3 + 1.05 * g : t64 <= 512 ? 2 + 1.65 * g : std::max(1.0, t64 / 768) * (2.5 + 2.3 * g),
          PromptPlan::TILES64, 0, 0, 0, 0);
  if (!ring) return best;
  if (!prompt && N % 64 == 0)
    offer(2.5 + ceil((M + 31) / 32 * (N / 64) / 256.0) * (3.3 + 0.28 * g), PromptPlan::RING, 2, 2, 2, 4);
  if (N % 128 == 0) {
    const double pairs = floor(t64 / 512), rest = t64 - 512 * pairs;
    offer(2.5 + ceil(t64 / 256) * (4 + 0.66 * g), PromptPlan::RING, 4, 2, 4, 2);
    offer(2 + pairs * (5.5 + 1.22 * g) + (rest == 0 ? 0 : rest <= 256 ? 4 + 0.88 * g : 5.5 + 1.22 * g), PromptPlan::RING,
          4, 2, 4, 1);
  }
  if (N % 256 == 0) {
    const double t = (double)((M + 127) / 128) * (N / 256), r = ceil(t / 256);
    offer(1.1 * (3 + (r - 1) * (6.5 + 1.8 * g) + 6.5 + g * (1.36 + 0.44 * (t - (r - 1) * 256) / 256)), PromptPlan::RING, 8,
          2, 8, 1);
  }
  return best;
}

}  // namespace t2i_host
