// Green-pass plans for padded z axes of 360 to 768 points (pass3_wave.hpp),
// the fastest of two to three measured per length on 96 x 96 x N grids: two
// stages up to 400 points, then three, one column per wave (768 points as 16
// 16 3: 16 values per lane; with four stages of 12 values 10 % slower).
#include "pass3_wave.hpp"

namespace ddhip {
static const P3Shape kShapes[] = {
    P3_PLAN(20, 20, 18), P3_PLAN(64, 8, 6, 8), P3_PLAN(20, 20, 20), P3_PLAN(54, 8, 6, 9), P3_PLAN(50, 10, 5, 9),
    P3_PLAN(64, 10, 6, 8), P3_PLAN(54, 6, 9, 9), P3_PLAN(50, 10, 10, 5), P3_PLAN(64, 8, 8, 8), P3_PLAN(60, 12, 5, 9),
    P3_PLAN(64, 8, 8, 9), P3_PLAN(60, 10, 6, 10), P3_PLAN(64, 16, 8, 5), P3_PLAN(54, 18, 6, 6),
    P3_PLAN(60, 10, 6, 12), P3_PLAN(50, 10, 15, 5), P3_PLAN(64, 16, 16, 3),
    // a factor 7, the faster of a two- and a three-stage plan each (336^3 grid
    // points: 345 against 393 us, 448^3: 765, 988, 420^3: 744, 813)
    P3_PLAN(56, 8, 6, 7), P3_PLAN(50, 10, 5, 7), P3_PLAN(21, 18, 21), P3_PLAN(56, 8, 7, 7), P3_PLAN(21, 20, 21),
    P3_PLAN(64, 8, 8, 7), P3_PLAN(49, 10, 7, 7), P3_PLAN(63, 8, 9, 7),
};
const P3Shape* p3_shapes_long(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
