// Green-pass plans for padded z axes of 162 to 324 points (pass3_wave.hpp),
// the fastest of five to eight measured per length on whole MATVECs of cubes
// (N, N, N), among those that round no worse.  Two stages of up to 20 values
// per lane and component, where the length splits into factors that small,
// against three stages of 9 to 12, which leave room for more waves but cost
// another LDS exchange each way: two win to 192 points (90^3 points: 512 against
// 540 us and more) and at 240 and 288 (144^3: 538, 547), three at 200 (100^3 x 4:
// 729 -> 704 us), 216 (108^3 x 4: 891 -> 844) and 324 (162^3: 855 -> 827).  Lanes a
// column beyond its butterflies repeat the last one: 16 lanes at 196 points
// (98^3 x 4: 701 -> 658) and 21 at 320 (160^3: 751 -> 713), where 14 and 20 cost
// registers for the column index.
#include "pass3_wave.hpp"

namespace ddhip {
static const P3Shape kShapes[] = {
    P3_PLAN(18, 6, 3, 9), P3_PLAN(15, 12, 15), P3_PLAN(16, 16, 12), P3_PLAN(20, 10, 2, 10), P3_PLAN(27, 8, 9, 3),
    P3_PLAN(16, 16, 15), P3_PLAN(25, 10, 5, 5), P3_PLAN(16, 16, 16), P3_PLAN(30, 10, 3, 9), P3_PLAN(18, 18, 16),
    P3_PLAN(20, 20, 15), P3_PLAN(21, 20, 16), P3_PLAN(54, 6, 9, 6),
    // a factor 7: here three stages of 7 to 14 values beat two of 18 to 21
    // (252^3 grid points: 152 against 181 us, 280^3: 226, 257, 294^3: 258, 301)
    P3_PLAN(14, 14, 12), P3_PLAN(16, 14, 14), P3_PLAN(15, 14, 15), P3_PLAN(16, 14, 16), P3_PLAN(21, 6, 6, 7),
    P3_PLAN(56, 8, 5, 7), P3_PLAN(49, 6, 7, 7),
};
const P3Shape* p3_shapes_medium(int& n) {
  n = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
  return kShapes;
}
}  // namespace ddhip
