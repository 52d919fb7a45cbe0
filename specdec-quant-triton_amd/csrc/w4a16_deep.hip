// Instantiations of the many-row W4A16 kernel, one per weight layout.
#include "w4a16_deep.hpp"

namespace specq {

const void* w4a16_deep_fn(int layout) {
  switch (layout) {
    case 0: return reinterpret_cast<const void*>(&w4a16_deep_kernel<0>);
    case 1: return reinterpret_cast<const void*>(&w4a16_deep_kernel<1>);
    case 2: return reinterpret_cast<const void*>(&w4a16_deep_kernel<2>);
  }
  return nullptr;
}

}  // namespace specq
