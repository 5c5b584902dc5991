// Row addressing of a tile's clamped loads in the streaming compress.
#pragma once

#include <stdint.h>

#ifdef __HIP__
#define BS_HD __host__ __device__ __forceinline__
#else
#define BS_HD inline
#endif

namespace bs {

// The wave-uniform part of the row that round k of a tile loads (row 8k of the
// tile, to which a lane adds lane/8 if that row is inside the matrix): 0, the
// tile's first row, for a round that lies past the `rows_in_tile` (>= 1) rows
// of the tile inside the matrix.  Clamping the lane's part alone is not
// enough: in a last tile row of 56 rows or fewer, row 8k itself can lie past
// the matrix.
BS_HD int64_t row_step(int k, int64_t rows_in_tile)
{
    return 8 * k < rows_in_tile ? 8 * k : 0;
}

}  // namespace bs
