// Green-pass plans for padded z axes of 360 to 768 points (pass3_wave.hpp),
// the fastest of three to eight measured per length on whole MATVECs of cubes
// (N, N, N): three stages, mostly of 8 to 12 values (up to 18 where the length
// splits no better), one column per wave or two; two stages of 18 to 21 values
// at 400 points (20 x 20: 1,538 us at 200^3, three stages 1,570 and more), 378 and
// 420; 768 points 16 16 3 (9,785 at 384^3, 16 8 6 9,796, 8 8 12 9,865, 12 8 8 10,760).
// 360 points 20 18
// -> 12 5 6: 180^3 1,187 -> 1,053 us; 384 8 6 8 -> 8 8 6: 192^3 1,332 -> 1,249;
// 432 8 6 9 -> 12 4 9: 216^3 1,996 -> 1,960.
#include "pass3_wave.hpp"

namespace ddhip {
static const P3Shape kShapes[] = {
    P3_PLAN(30, 12, 5, 6), P3_PLAN(64, 8, 8, 6), P3_PLAN(20, 20, 20), P3_PLAN(54, 12, 4, 9), P3_PLAN(50, 10, 5, 9),
    P3_PLAN(64, 10, 6, 8), P3_PLAN(54, 6, 9, 9), P3_PLAN(50, 10, 10, 5), P3_PLAN(64, 8, 8, 8), P3_PLAN(60, 12, 5, 9),
    P3_PLAN(64, 8, 8, 9), P3_PLAN(60, 10, 6, 10), P3_PLAN(64, 16, 8, 5), P3_PLAN(54, 18, 6, 6),
    P3_PLAN(60, 10, 6, 12), P3_PLAN(50, 10, 15, 5), P3_PLAN(64, 16, 16, 3),
    // a factor 7 (504 points 8 9 7 -> 14 4 9: 252^3 3,135 -> 2,965 us)
    P3_PLAN(56, 8, 6, 7), P3_PLAN(50, 10, 5, 7), P3_PLAN(21, 18, 21), P3_PLAN(56, 8, 7, 7), P3_PLAN(21, 20, 21),
    P3_PLAN(64, 8, 8, 7), P3_PLAN(49, 10, 7, 7), P3_PLAN(63, 14, 4, 9),
};
const P3Shape* p3_shapes_long(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
