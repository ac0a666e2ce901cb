// Walks the expert input addresses of the 4x4x1 kernels over every row length
// they serve: each read stays inside its row, and lane block b of group g holds
// the four pieces of unit 16 g + b where the row has that unit.
#define __host__
#define __device__
#include "neon_exact_index.hpp"

#include <cstdio>

int main() {
  int bad = 0, rows = 0;
  for (int U = 1; U <= 128; ++U) {
    const int ng = neon::xm_groups(32 * U);
    if (ng == 0) {
      std::printf("U=%d: not served\n", U);
      return 1;
    }
    ++rows;
    for (int g = 0; g < ng; ++g)
      for (int b = 0; b < 16; ++b) {
        const neon::XmPieces at = neon::xm_pieces(g, b, U);
        for (int q = 0; q < 4; ++q) {
          const int piece = at.first + q * at.step;
          if (piece < 0 || piece >= 4 * U) {
            std::printf("U=%d group %d unit %d piece %d: reads piece %d of %d\n", U, g, b, q, piece,
                        4 * U);
            ++bad;
          } else if (16 * g + b < U) {
            // where the writer put the piece's first element
            const int elem = 32 * (16 * g + b) + 8 * q;
            if (neon::xm_act_at(elem, U) != 8 * piece) {
              std::printf("U=%d element %d: stored at %d, read at %d\n", U, elem,
                          neon::xm_act_at(elem, U), 8 * piece);
              ++bad;
            }
          }
        }
      }
  }
  if (neon::xm_groups(32 * 129) != 0) ++bad;
  std::printf("%d row lengths, %d wrong addresses\n", rows, bad);
  return bad != 0;
}
