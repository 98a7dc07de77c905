// The library's i8 tile kernels (matmul_tile.h), in a file of their own so that the types
// compile in parallel; matmul_i8.hip launches them.
#include "matmul_tile.h"

ASC_TILE_KERNELS_I8(ASC_TILE_DEFINE, , asc_tile_)
