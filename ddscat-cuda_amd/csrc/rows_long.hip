// x-pass shapes for padded x axes of 270 to 768 points (rows.hpp).  The
// components of pass 5 are loaded and transformed one after another (VN of 18
// to 35 values), real and imaginary parts crossing LDS in turn, in finish
// groups of two outputs: 3 to 5 % faster than whole exchanges and groups of
// four at 270 to 480 points.
#include "rows.hpp"

namespace ddhip {
#define X_BOTH(R1, R2) X_FWD(R1, R2, 16), X_INV(R1, R2, 16, 2, true, false)
static const RowShape kShapes[] = {
    X_BOTH(18, 15), X_FWD(18, 16, 16), X_BOTH(20, 15), X_FWD(20, 16, 16), X_BOTH(18, 18), X_BOTH(20, 18),
    X_BOTH(16, 24), X_BOTH(20, 20), X_BOTH(24, 18), X_BOTH(25, 18), X_BOTH(32, 15), X_BOTH(27, 18), X_FWD(25, 20, 16),
    X_FWD(32, 16, 16), X_BOTH(27, 20), X_BOTH(24, 24), X_BOTH(25, 24), X_BOTH(32, 20), X_BOTH(27, 24), X_BOTH(30, 24),
    X_BOTH(30, 25), X_BOTH(32, 24),
    // a factor 7
    X_BOTH(20, 14), X_BOTH(21, 14), X_BOTH(24, 14), X_BOTH(25, 14), X_BOTH(27, 14), X_BOTH(28, 14), X_BOTH(28, 15),
    X_BOTH(32, 14), X_BOTH(35, 14), X_BOTH(28, 18),
    // 512 points: 32 rows, 256 bytes of a1 per kx (256^3: 506 us against 551 with 16 rows)
    X_INV(32, 16, 32, 2, true, false), X_INV(32, 16, 16, 2, true, false), X_INV(32, 24, 16, 4, true, false),
    X_INV(25, 20, 16, 2, false, false),
    // 16 lanes along x: the finish reads and writes whole 128-byte lines, and
    // 16 x 18 took 144^3 from 531 to 500 us against 18 x 16, 16 x 20 160^3 from 720
    // to 691 against 20 x 16 (pass 1, which only reads x, is the same either way)
    X_INV(16, 18, 16, 2, true, false), X_INV(16, 20, 16, 2, true, false),
};
const RowShape* row_shapes_long(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
