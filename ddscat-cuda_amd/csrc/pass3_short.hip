// Green-pass plans for padded z axes of 24 to 160 points (pass3_wave.hpp),
// the fastest of two to four measured per length on 96 x 96 x N grids.  Two
// stages, one exchange each way; T lanes per column fill 54 to 64 lanes of a
// wave and hold at most 16 values per component; the larger radix first (its
// zero half folds away), and T the larger of the two where that saves
// registers (90 points: 10 lanes of 10 values 31 us, 9 lanes of 20 50 us).
// 150 points take three stages: 15 lanes leave a third of the 15-point
// butterflies' lanes idle (54 against 46 us).
#include "pass3_wave.hpp"

namespace ddhip {
static const P3Shape kShapes[] = {
    P3_PLAN(6, 6, 4), P3_PLAN(6, 6, 5), P3_PLAN(8, 4, 8), P3_PLAN(6, 6, 6), P3_PLAN(8, 8, 5), P3_PLAN(8, 8, 6),
    P3_PLAN(5, 10, 5), P3_PLAN(9, 6, 9), P3_PLAN(10, 10, 6), P3_PLAN(8, 8, 8), P3_PLAN(9, 8, 9), P3_PLAN(10, 8, 10),
    P3_PLAN(10, 10, 9), P3_PLAN(12, 12, 8), P3_PLAN(10, 10, 10), P3_PLAN(12, 12, 9), P3_PLAN(12, 12, 10),
    P3_PLAN(8, 16, 8), P3_PLAN(12, 12, 12), P3_PLAN(30, 6, 5, 5), P3_PLAN(16, 16, 10),
    // a factor 7
    P3_PLAN(7, 4, 7), P3_PLAN(7, 6, 7), P3_PLAN(8, 8, 7), P3_PLAN(10, 10, 7), P3_PLAN(12, 12, 7), P3_PLAN(14, 14, 7),
    P3_PLAN(14, 14, 8), P3_PLAN(14, 14, 9), P3_PLAN(14, 14, 10),
};
const P3Shape* p3_shapes_short(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
