// Instantiations of the many-row W8A8 / W4A8 kernel (packed weight layouts 1 and 2).  LDS rings:
// deep ones where one workgroup runs per CU (64 and 128 rows), two slots where two or three do.
#include "w8a8_deep.hpp"

namespace specq {

namespace {

template <int FM, int FN, int NSL, int WL>
const void* pick(bool wide) {
  return wide ? reinterpret_cast<const void*>(&w8a8_deep_wide_kernel<FM, FN, NSL, WL>)
              : reinterpret_cast<const void*>(&w8a8_deep_kernel<FM, FN, NSL, WL>);
}

}  // namespace

const void* w8a8_deep_fn(int tile, int layout, bool wide) {
  if (layout == 1) {
    switch (tile) {
      case kDeep64: return pick<2, 4, 3, 1>(wide);
      case kDeep128: return pick<4, 4, 4, 1>(wide);
      case kDeep128Pair: return pick<4, 4, 2, 1>(wide);
      case kDeepMix:
        return wide ? reinterpret_cast<const void*>(&w8a8_deep_mix_wide_kernel<1>)
                    : reinterpret_cast<const void*>(&w8a8_deep_mix_kernel<1>);
    }
  }
  if (layout == 2 && tile == kDeep128Pair) return pick<4, 4, 2, 2>(wide);
  return nullptr;
}

}  // namespace specq
