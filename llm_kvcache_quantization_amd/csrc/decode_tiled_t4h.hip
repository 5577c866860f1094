// Instantiations of decode_tiled_kernel (decode_tiled.h) for INT4_SYM K and V with per-token fp16
// scales.
#include "decode_tiled.h"

namespace kvq {

TiledFn tiled_kernel_t4h(int fam, bool pack8) {
  switch (fam) {
    case kTiledT4h: return tiled_pick<KTokT<true, 1, true>, VTokT<true, false, true>>(pack8);
    case kTiledT4hg16: return tiled_pick<KTokT<true, 2, true>, VTokT<true, false, true>>(pack8);
    case kTiledT4hs: return tiled_pick<KTokT<true, 1, true>, VTokT<true, true, true>>(pack8);
    case kTiledT4hg16s: return tiled_pick<KTokT<true, 2, true>, VTokT<true, true, true>>(pack8);
    default: return TiledFn{nullptr, nullptr, -1, -1};
  }
}

}  // namespace kvq
