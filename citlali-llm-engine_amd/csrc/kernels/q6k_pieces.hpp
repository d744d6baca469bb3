// q6k_pieces.hpp -- which 16-byte pieces the tile kernels read of a matrix of
// Q6_K blocks.  Plain arithmetic, so that host code can check it.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define CITLALI_PIECES __host__ __device__ constexpr
#else
#define CITLALI_PIECES constexpr
#endif

namespace citlali::hip {

constexpr int kQ6KBlockBytes = 210;
constexpr int kQ6KPieces = 14;   // aligned pieces that cover a block at any even offset in its first one

// A tile's step reads one block of each of its rows.  skew: how far the block
// of the tile's first row lies behind its piece's first byte; row_offset: the
// distance from that block to the block of another row.  Offset of that
// row's piece p from the first row's first piece; a piece may begin before its
// block and end behind it.
CITLALI_PIECES int q6k_piece(int skew, int row_offset, int p) { return ((row_offset + skew) & ~15) + 16 * p; }

// Blocks of a row of nb whose pieces may reach outside the matrix: its first
// block where it does not begin with a piece, its last where it does not end
// with one.  (lo, hi): such blocks of a tile, -1 for none.
struct Q6KEnds {
    int lo, hi;
};
CITLALI_PIECES Q6KEnds q6k_ends(uintptr_t w, int rows, int nb, bool first_tile, bool last_tile) {
    const uint32_t end = (uint32_t)w + (uint32_t)rows * (uint32_t)(nb * kQ6KBlockBytes);
    return Q6KEnds{first_tile && (w & 15) != 0 ? 0 : -1, last_tile && (end & 15) != 0 ? nb - 1 : -1};
}

}  // namespace citlali::hip
