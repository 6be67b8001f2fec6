// Green-pass plans for padded z axes of 162 to 324 points (pass3_wave.hpp),
// the fastest of two to three measured per length on 96 x 96 x N grids.  Two
// stages of up to 20 values per lane and component beat three stages of 10 to
// 12 wherever the length splits into factors that small (288 points: 95
// against 108 us), although they run at 2 to 3 instead of 4 waves per SIMD:
// each stage more costs another LDS exchange each way.  (162 points: 9 lanes of
// 18 values 59 to 73 us, 18 lanes in three stages 55 us.)
#include "pass3_wave.hpp"

namespace ddhip {
static const P3Shape kShapes[] = {
    P3_PLAN(18, 6, 3, 9), P3_PLAN(15, 12, 15), P3_PLAN(16, 16, 12), P3_PLAN(10, 20, 10), P3_PLAN(18, 18, 12),
    P3_PLAN(16, 16, 15), P3_PLAN(25, 10, 5, 5), P3_PLAN(16, 16, 16), P3_PLAN(30, 10, 3, 9), P3_PLAN(18, 18, 16),
    P3_PLAN(20, 20, 15), P3_PLAN(20, 20, 16), P3_PLAN(18, 18, 18),
    // a factor 7: here three stages of 7 to 14 values beat two of 18 to 21
    // (252^3 grid points: 152 against 181 us, 280^3: 226, 257, 294^3: 258, 301)
    P3_PLAN(14, 14, 12), P3_PLAN(14, 14, 14), P3_PLAN(15, 14, 15), P3_PLAN(16, 14, 16), P3_PLAN(21, 6, 6, 7),
    P3_PLAN(56, 8, 5, 7), P3_PLAN(49, 6, 7, 7),
};
const P3Shape* p3_shapes_medium(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
