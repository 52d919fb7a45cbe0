// Instantiations of the LDS-staged-activation W8A8 kernel: BLOCK_N = 128, weight layout 1
// (packed K-step-major fragments), token tiles of 2 .. 19 x 16 rows.
#include "w8a8_tiles.hpp"

namespace specq {

const void* w8a8_ws_fn_n128_l1(int mt, bool keep) {
  switch (mt) {
    case 2: return w8a8_ws_pick<2, 3, 1>(keep);
    case 3: return w8a8_ws_pick<3, 3, 1>(keep);
    case 4: return w8a8_ws_pick<4, 3, 1>(keep);
    case 5: return w8a8_ws_pick<5, 3, 1>(keep);
    case 6: return w8a8_ws_pick<6, 3, 1>(keep);
    case 7: return w8a8_ws_pick<7, 3, 1>(keep);
    case 8: return w8a8_ws_pick<8, 3, 1>(keep);
    case 9: return w8a8_ws_pick<9, 3, 1>(keep);
    case 10: return w8a8_ws_pick<10, 3, 1>(keep);
    case 11: return w8a8_ws_pick<11, 3, 1>(keep);
    case 12: return w8a8_ws_pick<12, 3, 1>(keep);
    case 13: return w8a8_ws_pick<13, 3, 1>(keep);
    case 14: return w8a8_ws_pick<14, 3, 1>(keep);
    case 15: return w8a8_ws_pick<15, 3, 1>(keep);
    case 16: return w8a8_ws_pick<16, 3, 1>(keep);
    case 17: return w8a8_ws_pick<17, 3, 1>(keep);
    case 18: return w8a8_ws_pick<18, 3, 1>(keep);
    case 19: return w8a8_ws_pick<19, 3, 1>(keep);
    default: return nullptr;
  }
}

}  // namespace specq
