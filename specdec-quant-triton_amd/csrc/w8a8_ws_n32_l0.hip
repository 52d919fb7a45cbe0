// Instantiations of the LDS-staged-activation W8A8 kernel: BLOCK_N = 32, weight layout 0
// (row-major), token tiles of 2 .. 19 x 16 rows.
#include "w8a8_tiles.hpp"

namespace specq {

const void* w8a8_ws_fn_n32_l0(int mt, bool keep) {
  switch (mt) {
    case 2: return w8a8_ws_pick<2, 1, 0>(keep);
    case 3: return w8a8_ws_pick<3, 1, 0>(keep);
    case 4: return w8a8_ws_pick<4, 1, 0>(keep);
    case 5: return w8a8_ws_pick<5, 1, 0>(keep);
    case 6: return w8a8_ws_pick<6, 1, 0>(keep);
    case 7: return w8a8_ws_pick<7, 1, 0>(keep);
    case 8: return w8a8_ws_pick<8, 1, 0>(keep);
    case 9: return w8a8_ws_pick<9, 1, 0>(keep);
    case 10: return w8a8_ws_pick<10, 1, 0>(keep);
    case 11: return w8a8_ws_pick<11, 1, 0>(keep);
    case 12: return w8a8_ws_pick<12, 1, 0>(keep);
    case 13: return w8a8_ws_pick<13, 1, 0>(keep);
    case 14: return w8a8_ws_pick<14, 1, 0>(keep);
    case 15: return w8a8_ws_pick<15, 1, 0>(keep);
    case 16: return w8a8_ws_pick<16, 1, 0>(keep);
    case 17: return w8a8_ws_pick<17, 1, 0>(keep);
    case 18: return w8a8_ws_pick<18, 1, 0>(keep);
    case 19: return w8a8_ws_pick<19, 1, 0>(keep);
    default: return nullptr;
  }
}

}  // namespace specq
