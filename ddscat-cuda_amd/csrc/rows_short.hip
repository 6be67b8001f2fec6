// x-pass shapes for padded x axes of 24 to 256 points (rows.hpp): two-level
// register transforms, R1 lanes per row, at most 18 to 25 values per lane.
// 32 rows per workgroup where R1 is small (workgroups of 128 threads and
// more), 16 rows (one 128-byte line of a1 per kx) otherwise.  16 lanes where
// 16 divides the length, so that the finish of pass 5 touches whole 128-byte
// lines of the vectors: 8 right-hand sides of 48 x 96 x 96 553 -> 533 us with 16 x 6
// in place of 12 x 8, 40 x 80 x 80 340 -> 333 (16 x 5, 10 x 8), 72^3 506 -> 500.
#include "rows.hpp"

namespace ddhip {
#define X_BOTH(R1, R2, C) X_FWD(R1, R2, C), X_INV(R1, R2, C, 4, false, true)
static const RowShape kShapes[] = {
    X_BOTH(6, 4, 32),   X_BOTH(6, 5, 32),   X_BOTH(4, 8, 32),   X_BOTH(6, 6, 32),   X_BOTH(8, 5, 32),
    X_BOTH(8, 6, 32),   X_BOTH(10, 5, 32),  X_BOTH(9, 6, 32),   X_BOTH(10, 6, 32),  X_BOTH(8, 8, 32),
    X_BOTH(12, 6, 16),  X_BOTH(16, 5, 16),  X_BOTH(10, 9, 16),  X_BOTH(16, 6, 16),  X_BOTH(10, 10, 16),
    X_BOTH(12, 9, 16),  X_BOTH(12, 10, 16), X_BOTH(16, 8, 16),  X_BOTH(16, 9, 16),  X_BOTH(15, 10, 16),
    X_BOTH(16, 10, 16), X_BOTH(18, 9, 16),  X_BOTH(15, 12, 16), X_BOTH(16, 12, 16), X_FWD(20, 10, 16),
    X_FWD(18, 12, 16),  X_BOTH(16, 15, 16), X_FWD(25, 10, 16),  X_BOTH(16, 16, 16),
    // a factor 7
    X_BOTH(7, 4, 32), X_BOTH(7, 6, 32), X_BOTH(8, 7, 32), X_BOTH(10, 7, 32), X_BOTH(12, 7, 16), X_BOTH(14, 7, 16),
    X_BOTH(16, 7, 16), X_BOTH(14, 9, 16), X_BOTH(14, 10, 16), X_BOTH(14, 12, 16), X_BOTH(14, 14, 16),
    X_BOTH(15, 14, 16), X_BOTH(16, 14, 16), X_BOTH(18, 14, 16),
    // one component at a time (200 points: 72 -> 65 us, 216: 77 -> 73 us on 128 x 128 rows)
    X_INV(20, 10, 16, 5, false, false), X_INV(18, 12, 16, 3, false, false), X_INV(25, 10, 16, 5, false, false),
};
const RowShape* row_shapes_short(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
