// The lines of neon_exact_routes.hpp against what was measured on both sides
// of them: a call must not take a form that was timed slower there.
#include "neon_exact_routes.hpp"

#include <cstdio>

enum Form { PAIRS, GROUPED, MATRIX };

static Form form(int B, int k, int E, int H, int I) {
  if (neon::xm_moe_wanted(B, k, E, H, I)) return MATRIX;
  return neon::moe_grouped_wanted(B, k, E, I) ? GROUPED : PAIRS;
}

int main() {
  int bad = 0, n = 0;
  auto expect = [&](const char* what, int got, int want) {
    ++n;
    if (got != want) {
      std::printf("%s: form %d, expected %d\n", what, got, want);
      ++bad;
    }
  };
#define MOE(B, k, E, H, I, want) expect(#want " B=" #B " k=" #k " E=" #E " H=" #H " I=" #I, form(B, k, E, H, I), want)
  // small experts: pair by pair at any batch that was timed
  MOE(3, 4, 8, 512, 512, PAIRS);
  MOE(16, 4, 8, 512, 512, PAIRS);
  MOE(64, 4, 8, 512, 512, PAIRS);
  MOE(8, 2, 2, 1024, 1024, PAIRS);
  MOE(64, 2, 8, 1024, 1024, PAIRS);
  MOE(12, 2, 16, 1024, 2048, PAIRS);
  MOE(16, 2, 16, 1024, 2048, PAIRS);
  MOE(8, 1, 4, 4096, 4096, PAIRS);
  MOE(12, 4, 32, 2048, 2048, PAIRS);
  MOE(6, 4, 16, 2880, 2880, PAIRS);
  MOE(3, 4, 8, 2880, 2880, PAIRS);
  MOE(16, 6, 64, 2048, 1408, PAIRS);
  // few pairs per expert
  MOE(1, 4, 32, 2880, 2880, PAIRS);
  MOE(8, 4, 32, 2880, 2880, PAIRS);
  MOE(16, 4, 128, 2880, 2880, PAIRS);
  MOE(47, 4, 128, 2880, 2880, PAIRS);
  MOE(9, 4, 32, 2880, 2880, GROUPED);
  MOE(11, 4, 32, 2880, 2880, GROUPED);
  // past the matrix form's row length
  MOE(16, 4, 8, 4128, 2880, GROUPED);
  MOE(16, 4, 8, 2880, 4128, GROUPED);
  MOE(17, 4, 8, 4128, 2880, PAIRS);
  // the matrix form
  MOE(12, 4, 32, 2880, 2880, MATRIX);
  MOE(64, 4, 32, 2880, 2880, MATRIX);
  MOE(48, 4, 128, 2880, 2880, MATRIX);
  MOE(16, 4, 4, 2880, 2880, MATRIX);
  MOE(8, 4, 8, 2880, 2880, MATRIX);
  MOE(8, 4, 16, 2880, 2880, MATRIX);
  MOE(16, 4, 32, 2048, 2048, MATRIX);
  MOE(22, 6, 64, 2048, 1408, MATRIX);
  MOE(32, 2, 16, 1024, 2048, MATRIX);
  MOE(64, 1, 4, 4096, 4096, MATRIX);
  MOE(32, 8, 128, 1024, 512, MATRIX);
  MOE(320, 4, 32, 2880, 2880, MATRIX);
  MOE(321, 4, 32, 2880, 2880, PAIRS);
  MOE(65535, 16, 256, 8192, 8192, PAIRS);
#define ATTN(B, Hq, Hkv, S, span, want) expect("attn B=" #B " heads " #Hq "/" #Hkv " S=" #S " span " #span, neon::attn_on_matrix(B, Hq, Hkv, S, span), want)
  // one split
  ATTN(8, 64, 8, 1, 128, 0);
  ATTN(16, 64, 8, 1, 128, 1);
  ATTN(64, 64, 8, 1, 256, 1);
  ATTN(64, 16, 2, 1, 256, 1);
  ATTN(16, 32, 8, 1, 128, 0);
  ATTN(32, 32, 8, 1, 128, 1);
  ATTN(64, 16, 8, 1, 128, 0);
  ATTN(72, 16, 8, 1, 128, 0);
  ATTN(128, 16, 8, 1, 128, 1);
  ATTN(65, 8, 8, 1, 128, 0);
  ATTN(256, 8, 8, 1, 128, 0);
  // several
  ATTN(1, 64, 8, 32, 4096, 0);
  ATTN(2, 64, 8, 32, 4096, 1);
  ATTN(8, 64, 8, 8, 512, 1);
  ATTN(16, 64, 8, 32, 32768, 1);
  ATTN(2, 8, 8, 32, 4096, 0);
  ATTN(8, 8, 8, 8, 512, 0);
  ATTN(8, 32, 8, 8, 512, 0);
  ATTN(8, 32, 8, 32, 8192, 0);
  ATTN(8, 32, 8, 32, 4096, 1);
  ATTN(32, 8, 8, 32, 4096, 0);
  ATTN(8, 8, 8, 32, 2048, 1);
  ATTN(32, 32, 8, 8, 512, 1);
#define WIDE(rows, E, k, H, I, want) expect(#rows " rows E=" #E " k=" #k " H=" #H " I=" #I, rows >= neon::xg_min_rows(E, k, H, I), want)
  WIDE(24, 32, 4, 2880, 2880, 0);
  WIDE(64, 32, 4, 2880, 2880, 0);
  WIDE(96, 32, 4, 2880, 2880, 1);
  WIDE(24, 128, 4, 2880, 2880, 0);
  WIDE(128, 128, 4, 2880, 2880, 0);
  WIDE(160, 128, 4, 2880, 2880, 0);
  WIDE(174, 128, 4, 2880, 2880, 1);
  WIDE(192, 128, 4, 2880, 2880, 1);
  WIDE(80, 64, 4, 2880, 2880, 0);
  WIDE(112, 64, 4, 2880, 2880, 1);
  WIDE(48, 16, 4, 2880, 2880, 0);
  WIDE(64, 16, 4, 2880, 2880, 1);
  WIDE(40, 8, 4, 2880, 2880, 0);
  WIDE(64, 8, 4, 2880, 2880, 1);
  WIDE(128, 32, 1, 2880, 2880, 0);
  WIDE(192, 32, 1, 2880, 2880, 1);
  WIDE(48, 32, 4, 512, 512, 0);
  WIDE(64, 32, 4, 512, 512, 1);
  WIDE(48, 64, 6, 2048, 1408, 0);
  WIDE(80, 64, 6, 2048, 1408, 1);
  WIDE(64, 8, 2, 4096, 4096, 0);
  WIDE(96, 8, 2, 4096, 4096, 1);
  std::printf("%d calls, %d on the wrong form\n", n, bad);
  return bad != 0;
}
