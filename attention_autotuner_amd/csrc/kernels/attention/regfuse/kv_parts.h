// Host side of the kv split of the attention forward: into how many parts a launch cuts the kv range.
//
// A row block walks its kv range alone, so a problem with fewer row blocks than the chip has CUs leaves CUs idle for the
// length of that walk: 72 row blocks of 128 rows against 4160 kv rows (batch 3, 12 heads, 192 queries, d 128) take 84 us
// in one part, 35 us in three or six.  Every part costs a second kernel and a round trip of its fp32 output, so a problem
// that fills the chip, or whose walk is short, stays in one part.
//
// The estimate below is the launch's time in microseconds, fitted on 3 700 launches of 38 tile shapes (d 64 ... 256, 26
// problems, both walks, 1 ... 32 parts; mean error 12 % there).  It knows matrix work only: on 136 problems outside the fit it is
// 7 to 25 % low, more where the stream from memory bounds a launch.  Over the launches of the fit the parts it picks are 2 % slower on the
// mean than the best ones; the simplest rule, one block per CU, is 5 % and up to twice the time on long kv ranges, where
// a second block per CU pays.  autotuner/gfx950_space.py holds the same estimate to choose between tile shapes.
#pragma once
#include <stdint.h>
#include <cmath>

namespace aat {

constexpr int kMi355xCus = 256;
constexpr int kMaxKvParts = 64;

struct ForwardShape {                      // what of a configuration the estimate depends on
  int Br, Bc, Kd, D, waves, blocks_per_cu, single_buffers;
};

// Blocks of `waves` waves that share a CU.
constexpr int forward_blocks_per_cu(int waves, int waves_per_eu, int lds_bytes) {
  const int by_regs = waves_per_eu * 4 / waves, by_lds = 160 * 1024 / lds_bytes;
  const int n = by_regs < by_lds ? by_regs : by_lds;
  return n < 1 ? 1 : n;
}

inline double forward_estimate_us(const ForwardShape& c, int B, int H, int Seq_q, int Seq_k, int causal, int parts) {
  // a kv tile's matrix work at the rate a CU sustains next to a softmax, and what short rows (small d) cost on top
  const double tile = (double)c.Br * c.Bc * 2.0 * (c.Kd + c.D) / 4.5e6 * (1.0 + 17.0 / c.D);
  const double alone = 4.55 / c.waves * tile;                        // a block that has its CU to itself
  const double shared = (c.Br >= 512 ? 0.72 : c.Br >= 256 ? 0.77 : c.Br >= 128 ? 0.87 : 1.25) * (1.0 + 0.034 * c.single_buffers) * tile;
  const double start = 0.7 + 2.6e-5 * c.Br * (c.Kd + c.D);           // first loads, output
  const int row_blocks = (Seq_q + c.Br - 1) / c.Br;
  const int tiles = ((Seq_k + c.Bc - 1) / c.Bc + parts - 1) / parts;
  const double per_cu = (double)B * H * row_blocks * parts / kMi355xCus;
  double us = start + tiles * alone;
  if (per_cu > 1.0) {
    // row blocks of all lengths, dealt out longest first: the CUs end together, and no sooner than the longest block
    const bool triangle = causal && Seq_q == Seq_k;
    const double walked = triangle ? (row_blocks + 1) / (2.0 * row_blocks) : 1.0;
    const double queue = per_cu < 3.0 ? std::ceil(per_cu) : per_cu + (triangle ? 0.3 : 0.6);
    const double rounds = per_cu < 3.0 * c.blocks_per_cu ? std::ceil(queue / c.blocks_per_cu) : queue / c.blocks_per_cu;
    us = std::fmax(triangle ? us : rounds * us, start + queue * walked * tiles * shared);
  }
  if (parts > 1) us += 4.0 + 1.6e-6 * parts * B * H * Seq_q * c.D;   // the merge kernel and the partial outputs' round trip
  return us;
}

inline int choose_kv_parts(const ForwardShape& c, int B, int H, int Seq_q, int Seq_k, int causal) {
  // fewer than 1024 kv rows are walked in less than the merge costs; two or more blocks per CU fill the chip
  const int64_t blocks = (int64_t)B * H * ((Seq_q + c.Br - 1) / c.Br);
  if (Seq_k < 1024 || blocks >= 2 * kMi355xCus) return 1;
  int best = 1;
  double best_us = forward_estimate_us(c, B, H, Seq_q, Seq_k, causal, 1);
  for (int parts = 2; parts <= kMaxKvParts && parts * 256 <= Seq_k; ++parts) {
    const double us = forward_estimate_us(c, B, H, Seq_q, Seq_k, causal, parts);
    if (us < best_us) {
      best = parts;
      best_us = us;
    }
  }
  return best;
}

}  // namespace aat
