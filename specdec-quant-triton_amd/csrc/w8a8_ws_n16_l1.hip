// Instantiations of the LDS-staged-activation W8A8 kernel: BLOCK_N = 16, weight layout 1
// (packed K-step-major fragments), token tiles of 2 .. 19 x 16 rows.
#include "w8a8_tiles.hpp"

namespace specq {

const void* w8a8_ws_fn_n16_l1(int mt, bool keep) {
  switch (mt) {
    case 2: return w8a8_ws_pick<2, 0, 1>(keep);
    case 3: return w8a8_ws_pick<3, 0, 1>(keep);
    case 4: return w8a8_ws_pick<4, 0, 1>(keep);
    case 5: return w8a8_ws_pick<5, 0, 1>(keep);
    case 6: return w8a8_ws_pick<6, 0, 1>(keep);
    case 7: return w8a8_ws_pick<7, 0, 1>(keep);
    case 8: return w8a8_ws_pick<8, 0, 1>(keep);
    case 9: return w8a8_ws_pick<9, 0, 1>(keep);
    case 10: return w8a8_ws_pick<10, 0, 1>(keep);
    case 11: return w8a8_ws_pick<11, 0, 1>(keep);
    case 12: return w8a8_ws_pick<12, 0, 1>(keep);
    case 13: return w8a8_ws_pick<13, 0, 1>(keep);
    case 14: return w8a8_ws_pick<14, 0, 1>(keep);
    case 15: return w8a8_ws_pick<15, 0, 1>(keep);
    case 16: return w8a8_ws_pick<16, 0, 1>(keep);
    case 17: return w8a8_ws_pick<17, 0, 1>(keep);
    case 18: return w8a8_ws_pick<18, 0, 1>(keep);
    case 19: return w8a8_ws_pick<19, 0, 1>(keep);
    default: return nullptr;
  }
}

}  // namespace specq
