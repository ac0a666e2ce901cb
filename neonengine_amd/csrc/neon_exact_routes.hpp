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
// (116) B = 64 242 / 353, 1024, 2048, 16, 2 (58) B = 64 94 / 158 (spread 111 / 88)
// and 160, 512, 32, 3 (24) B = 311 158 / 358 (spread 153 / 121).
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

// ---- decode attention: B rows, Hq / Hkv heads, S key splits of a span of keys ----
// The matrix form (k_xa_attn) costs the same for 1 and for 8 query heads per kv
// head; the vector form (k_attn_split) has work per head and blocks that all wait
// for a slot.  The span is the cache's rows or the window, whichever is less; how
// many keys a row holds is not known here.  us, vector / matrix, span full (an
// eighth full):
//   one split (a vector block per query head):
//     8 heads per kv head, 128 keys: B Hq = 1024 10.7 / 8.3 (10.7 / 7.7), 4096 35 / 12
//     4: 512 6.5 / 8.2, 1024 10.7 / 8.6; 2: 1024 10.7 / 11.8, 2048 19.9 / 17.9
//     1: 512 6.5 / 11.7, 2048 23.2 / 29.7
//   several (a block per kv head and split):
//     8, 2048 keys: B Hkv S = 256 8.9 / 9.0, 512 15.7 / 11.1, 2048 44.7 / 21.6;
//     8192 keys: 256 13.3 / 15.8, 512 24.9 / 21.3, 2048 83.4 / 51.2
//     4, 2048 keys: 512 8.7 / 10.7, 1024 14.6 / 14.2, 2048 23.8 / 21.1
//     1, 2048 keys: 512 8.1 / 10.3, 1024 13.5 / 13.9, 2048 21.7 / 21.0, 4096 37 / 33
//     longer splits, 2048 blocks: 4, 4096 keys 32.6 / 32.5 (17.6 / 13.2), 8192 keys
//     44 / 51; 1, 4096 keys 30 / 32 (16.6 / 12.5), 8192 keys 41 / 51; 4096 blocks:
//     1, 4096 keys 50 / 53 (27 / 18), 8192 keys 69 / 100 (30 / 24)
inline bool attn_on_matrix(int B, int Hq, int Hkv, int S, int span) {
  const int G = Hq / Hkv;
  const int64_t heads = B * (int64_t)Hq, blocks = B * (int64_t)Hkv * S;
  if (S == 1) return G >= 4 ? heads > 512 : G == 2 && heads >= 2048;
  return G == 8 ? blocks >= 512 : span <= (G == 4 ? 128 : 64) * S && blocks >= 2048;
}

// ---- prompt rows: the fewest of a wide pass --------------------------------------
// A wide pass (neon_exact_prompt.hip) takes an expert's pairs 16 at a time and
// pays for a whole tile of every expert that any row chose, so it costs about as
// much for few rows as for many: 49 rows' worth of the passes of 16 for what does
// not depend on the experts, and one row's more for every 2.25 million of E H I / k.
// ms, four layers, passes of 16 / wide, H = I = 2880, top-4: E = 8 40 rows 1.91 / 2.10,
// 64 2.87 / 2.17; E = 32 24 rows 1.54 / 3.70, 64 3.17 / 3.77, 80 3.94 / 3.91, 128
// 6.23 / 4.44; E = 128 24 rows 2.00 / 6.86, 128 8.90 / 11.06, 160 11.07 / 11.34, 192
// 13.2 / 11.7; E = 32 top-1 128 rows 3.49 / 3.92, 192 5.18 / 4.25; 512, 32, top-4 48
// rows 0.67 / 0.72, 64 0.85 / 0.74; 4096, 8, top-2 64 rows 3.01 / 3.17, 80 3.75 / 3.25.
inline int64_t xg_min_rows(int E, int k, int H, int I) {
  return 49 + E * (int64_t)H * I / (k * (int64_t)2250000);
}

}  // namespace neon
