// oit_tiles_k.hip - the tile path's composites for one layer count
// (OIT_TILE_K, one object per value: they compile side by side).
#include "oit_tiles.hpp"

namespace oit {

template <>
hipError_t tile_resolve_k<OIT_TILE_K>(const TileBuf& tb, const TileSrc& src, const TileDst& dst, int mode, bool tail,
                                      hipStream_t s) {
  return TileResolve<OIT_TILE_K>::run(tb, src, dst, mode, tail, s);
}

template <>
hipError_t tile_batch_k<OIT_TILE_K>(const BatchArgs& a, const TileBuf& tb, bool tail, hipStream_t s) {
  return tail ? TileBatch<OIT_TILE_K>::go<true>(a, tb, s) : TileBatch<OIT_TILE_K>::go<false>(a, tb, s);
}

}  // namespace oit
