// neon_exact_index.hpp -- which 16-byte piece of an expert input row a lane of
// the 4x4x1 kernels (neon_exact.hip) reads.  Plain integer functions without
// HIP headers: a host program walks them over every row length
// (tests/cpp/exact_index.cpp).
#pragma once

namespace neon {

// Groups of 16 units that the kernels are built for (0: K not covered).  3, 5
// and 7 groups run as 4, 6 and 8: the last of those may lie past the row.
__host__ __device__ inline int xm_groups(int K) {
  const int ng = (K / 32 + 15) / 16;
  return ng <= 1 ? 1 : ng <= 2 ? 2 : ng <= 4 ? 4 : ng <= 6 ? 6 : ng <= 8 ? 8 : 0;
}

// Place of element j of an act row of U units: the 16-byte pieces of a group's
// units are stored piece by piece ([piece][unit]), so that the 16 lanes of an
// input row read 256 contiguous bytes per load.
__host__ __device__ inline int xm_act_at(int j, int U) {
  const int g = j >> 9, b = (j >> 5) & 15, q = (j >> 3) & 3, left = U - 16 * g;
  return (g << 9) + (q * (left < 16 ? left : 16) + b) * 8 + (j & 7);
}

// Pieces of unit 16 g + b of such a row: piece q sits at first + q step.  A
// group or a unit past the row reads the last group or unit instead, and its
// value is dropped.
struct XmPieces {
  int first, step;
};
__host__ __device__ inline XmPieces xm_pieces(int g, int b, int U) {
  const int last = (U - 1) >> 4;
  g = g < last ? g : last;
  const int nb = U - 16 * g < 16 ? U - 16 * g : 16;
  return XmPieces{64 * g + (b < nb ? b : nb - 1), nb};
}

}  // namespace neon
