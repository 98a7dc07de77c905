// The library's bf16 tile kernels (matmul_tile.h), in a file of their own so that the types
// compile in parallel; matmul.hip launches them.
#include "matmul_tile.h"

ASC_TILE_KERNELS_BF16(ASC_TILE_DEFINE, , asc_tile_)
