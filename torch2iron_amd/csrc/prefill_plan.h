// Which prompt-attention kernel a call runs: a rule of the host alone (standard C++, no HIP),
// so that it can be checked without a device.
#pragma once

#include <math.h>

#include <algorithm>

namespace t2i_host {

// Whether the kernel of 128-row blocks (two row sets a wave, two workgroups a CU) is taken
// over the one of 64-row blocks (three a CU): B sequences of T rows from position p0, Hkv kv
// heads of Q q heads.  From both kernels' times at 2515 calls (1 to 4096 rows from 0 to 6000
// on, 1 to 500 sequences, 1, 2, 4 and 8 q heads a kv head, graph-launched):
//   n1, n2    blocks of 64 and of 128 rows.  A block of 128 costs 1.47 of 64 in the long run,
//             so padding decides short chunks (64 x 20 rows from 500, 8 kv heads of 2: as many
//             blocks either way, 25.6 us with 64 rows and 31.3 with 128);
//   even, k   n2 in blocks of the longest one's length (a block's work grows from p0 to p0 + T
//             keys: with few of them the longest block is the call), and a block's mean 64-key
//             blocks (under 1.5 what a workgroup starts with outweighs its products);
//   idle      the share of a last round of workgroups that is empty;
//   gain      log of the times' ratio, a fit of these with a standard error of 0.11: taken
//             from 8 % on.  Whole blocks of six key blocks and more need no estimate from 512
//             of the longest one's length on (0.999 to 1.69 times there).
// Of those calls it sends 870 to the 128-row blocks: 7 are 2 to 8 % slower than with 64-row
// ones, the rest 0.98 to 1.72 times as fast, the median 1.22.  (us, 64-row / 128-row: 1999 rows
// from 6001, 32 / 8 heads 386 / 278; 16 x 250 rows from 500, 16 / 8: 45.4 / 35.5; 16 x 512 rows
// from 0, 16 / 8: 42.0 / 39.7; and kept with 64-row blocks: 312 x 1 row from 0, 8 / 8 12.0 /
// 19.7, 56 x 129 rows from 0, 8 / 8 18.6 / 22.5, 2000 rows from 0, 16 / 8 49.3 / 58.5.)
inline bool prefill_wide(int B, int T, int p0, int Hkv, int Q) {
  const double heads = (double)B * Hkv, last = (double)p0 + T, mean = p0 + 0.5 * T;
  const double n1 = heads * ((T + 64 / Q - 1) / (64 / Q)), n2 = heads * ((T + 128 / Q - 1) / (128 / Q));
  const double even = n2 * mean / last, k = mean / 64;
  if (k < 1.5 || even < 380) return false;
  if (k >= 6 && even >= 512 && n1 >= 1.7 * n2) return true;
  auto idle = [](double n, double slots) { return std::min(1.0, ceil(n / slots) * slots / n - 1.0); };
  const double gain = log(n1 / n2) - 0.52 - 0.244 / (1 + k) - 44 / even - 0.276 * idle(n2, 512) +
                      0.127 * idle(n1, 768) + 0.3 * (p0 + 64) / (last + 64);
  return gain >= log(1.08);
}

}  // namespace t2i_host
