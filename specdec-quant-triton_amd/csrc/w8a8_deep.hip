// Instantiations of the many-row W8A8 / W4A8 kernel (packed weight layouts 1 and 2).  LDS rings:
// deep ones where one workgroup runs per CU (64 and 128 rows), two slots where two or three do.
#include "w8a8_deep.hpp"

namespace specq {

const void* w8a8_deep_fn(int tile, int layout) {
  if (layout == 1) {
    switch (tile) {
      case kDeep64: return reinterpret_cast<const void*>(&w8a8_deep_kernel<2, 4, 3, 1>);
      case kDeep128: return reinterpret_cast<const void*>(&w8a8_deep_kernel<4, 4, 4, 1>);
      case kDeep128Pair: return reinterpret_cast<const void*>(&w8a8_deep_kernel<4, 4, 2, 1>);
      case kDeepMix: return reinterpret_cast<const void*>(&w8a8_deep_mix_kernel<1>);
    }
  }
  if (layout == 2 && tile == kDeep128Pair) return reinterpret_cast<const void*>(&w8a8_deep_kernel<4, 4, 2, 2>);
  return nullptr;
}

}  // namespace specq
