// neon_exact_routes.hpp -- which of the exact kernels a call takes, by its
// sizes.  Every route gives the same bits.  Plain integer functions without HIP
// headers: a host program checks the lines against what was measured
// (tests/cpp/exact_routes.cpp).
#pragma once

#include <cstdint>

namespace neon {

// ---- experts of a batch: (row, slot) pairs B k over E experts ------------------
// Three forms: pair by pair (k_moe_gate_up, k_moe_down), grouped on the vector
// units (k_moe_gate_up_bt, k_moe_down_bt: at most 64 pairs, an expert's rows read
// once) and four pairs of an expert at a time on the fp32 matrix instructions
// (k_xm_gate_up, k_xm_down: H, I <= 4096, at most kXmMaxPairs).
constexpr int kXmMaxPairs = 1280;
constexpr int kXmGuColumns = 72;  // intermediate columns of a k_xm_gate_up block

// Sharing an expert's rows makes one block of what were many, so it needs
// column blocks: pairs x blocks >= 1280 (five per CU) and, for a batch that spreads
// over all experts, E x blocks >= 150.  us per call, pair by pair / grouped /
// matrix, H, I, E, k: 512, 512, 8, 4 B = 16 20 / 36 / 25, B = 64 58 / - / 67; 1024,
// 1024, 8, 2 B = 64 62 / - / 61, B = 128 114 / - / 116; 1024, 2048, 16, 2 B = 16 33 /
// 39 / 34; 4096, 4096, 4, 1 B = 8 40 / 48 / 54; 2880, 2880, 8, 4 B = 4 (640) 44 / 52 /
// 48, B = 8 (1280) 82 / 78 / 69.
inline int xm_blocks(int I) { return (I + kXmGuColumns - 1) / kXmGuColumns; }
inline bool moe_wide(int B, int k, int E, int I) {
  const int64_t blocks = xm_blocks(I);
  return B >= 2 && B * (int64_t)k * blocks >= 1280 && E * blocks >= 150;
}

// The matrix form from 1.5 pairs per expert on (an instruction takes four pairs
// of an expert whether there are four or one), from 2 where an expert has fewer
// than 36 column blocks.  us per call, pair by pair / matrix, 2880, 2880, k = 4:
// E = 32 B = 9 93 / 102, 10 106 / 108, 12 124 / 120, 16 166 / 136, 64 616 / 309; E =
// 128 B = 32 318 / 338, 48 472 / 435, 64 625 / 477; 2048, 2048, 32, 4 B = 12 57 / 64,
// 16 78 / 73, 64 305 / 193; 2048, 1408, 64, 6 B = 16 92 / 102, 21 127 / 120.  The
// line is for rows that spread.  Rows that all choose the same k experts leave it
// k x blocks blocks: 2880, k = 4 (160) B = 16 139 / 131, 64 558 / 486, but 2048, k = 4
// (116) B = 64 242 / 353 and 1024, 2048, 16, 2 (58) B = 64 94 / 158 (spread 111 / 88).
inline bool xm_moe_wanted(int B, int k, int E, int H, int I) {
  const int64_t pairs = B * (int64_t)k;
  const bool many = xm_blocks(I) >= 36;
  return pairs <= kXmMaxPairs && E <= 256 && H <= 4096 && I <= 4096 && moe_wide(B, k, E, I) &&
         2 * pairs >= (many ? 3 : 4) * E;
}

// The grouped form from more than one pair per expert on, where the matrix form
// is not taken and an expert has at least 36 column blocks: up to one, few pairs
// share an expert and a second read of one comes from the Infinity Cache.  It costs
// rows that spread up to 3% and saves rows alike 5%.  20b steps of 12 layers, ms,
// pair by pair / grouped / matrix, rows that spread (and all rows alike): B = 8
// 1.77 / 1.92 / 1.94 (1.74 / 1.72 / 1.62), 9 2.24 / 2.30 / 2.26 (2.20 / 2.09 / 2.27),
// 11 2.47 / 2.49 / 2.41 (2.41 / 2.26 / 2.33), 12 2.59 / 2.58 / 2.47 (2.53 / 2.34 /
// 2.33).  us per call, 2048, 2048, 32, 4 B = 12 57 / 63 / 64 (52 / 54 / 80).
inline bool moe_grouped_wanted(int B, int k, int E, int I) {
  const int64_t pairs = B * (int64_t)k;
  return pairs <= 64 && pairs > E && xm_blocks(I) >= 36 && moe_wide(B, k, E, I);
}

}  // namespace neon
