// Instantiations of the many-row W4A16 kernel, one per weight layout.
#include "w4a16_deep.hpp"

namespace specq {

const void* w4a16_deep_fn(int layout, bool wide) {
  switch (layout + (wide ? 3 : 0)) {
    case 0: return reinterpret_cast<const void*>(&w4a16_deep_kernel<0>);
    case 1: return reinterpret_cast<const void*>(&w4a16_deep_kernel<1>);
    case 2: return reinterpret_cast<const void*>(&w4a16_deep_kernel<2>);
    case 3: return reinterpret_cast<const void*>(&w4a16_deep_wide_kernel<0>);
    case 4: return reinterpret_cast<const void*>(&w4a16_deep_wide_kernel<1>);
    case 5: return reinterpret_cast<const void*>(&w4a16_deep_wide_kernel<2>);
  }
  return nullptr;
}

}  // namespace specq
