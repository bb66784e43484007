// The tile GEMM's kernels for bfloat16 storage.
#include "gemm_tiles_kernels.h"

namespace omni {
template hipError_t tile_group_of<kBF16>(int, int, TileGroup&, const TileChoice&, float*, bool, hipStream_t);
template bool tile_pair_of<kBF16>(int, TilePair&, hipStream_t, hipError_t*);
template hipError_t tile_down_of<kBF16>(const TileProduct&, const SelectArgs&, const TileChoice&, float*, hipStream_t, bool*, int*);
}  // namespace omni
