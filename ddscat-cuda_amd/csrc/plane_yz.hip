// Plane kernels for padded z axes of 24 to 108 points (plane_yz.hpp): the
// Green-pass plans of pass3_short.hip, and the two-level splits of the y axis.
#include "plane_yz.hpp"
#include "solver_common.hpp"

namespace ddhip {

static const YzShape kShapes[] = {
    YZ_PLAN(6, 6, 4),    YZ_PLAN(7, 4, 7),    YZ_PLAN(6, 6, 5),   YZ_PLAN(8, 4, 8),    YZ_PLAN(6, 6, 6),
    YZ_PLAN(8, 8, 5),    YZ_PLAN(7, 6, 7),    YZ_PLAN(8, 8, 6),   YZ_PLAN(5, 10, 5),   YZ_PLAN(9, 6, 9),
    YZ_PLAN(8, 8, 7),    YZ_PLAN(10, 10, 6),  YZ_PLAN(8, 8, 8),   YZ_PLAN(10, 10, 7),  YZ_PLAN(9, 8, 9),
    YZ_PLAN(10, 8, 10),  YZ_PLAN(12, 12, 7),  YZ_PLAN(10, 10, 9), YZ_PLAN(12, 12, 8),  YZ_PLAN(14, 14, 7),
    YZ_PLAN(10, 10, 10), YZ_PLAN(12, 12, 9),
};
// 2NY = R2 R1, R2 even
struct YzSplit {
  int R2, R1;
};
static const YzSplit kSplits[] = {{6, 4},  {4, 7},  {6, 5},  {8, 4},  {6, 6},  {8, 5},  {6, 7},   {8, 6},
                                  {10, 5}, {6, 9},  {8, 7},  {10, 6}, {8, 8},  {10, 7}, {8, 9},   {8, 10},
                                  {12, 7}, {10, 9}, {12, 8}, {14, 7}, {10, 10}, {12, 9}};

constexpr size_t YZ_LDS = 160 * 1024;  // per CU

static const YzShape* z_shape(int L) {
  for (const YzShape& s : kShapes)
    if (s.L == L) return &s;
  return nullptr;
}
static const YzSplit* y_split(int L) {
  for (const YzSplit& s : kSplits)
    if (s.R2 * s.R1 == L) return &s;
  return nullptr;
}

static size_t lds_bytes(const MatvecPlan& m, const YzShape* z) {
  return ((size_t)m.gy * z->pitch() + m.gy + m.gz) * sizeof(float2);
}

// The plane kernel where a plane fits LDS and there are planes enough to share
// the CUs: any number up to 80 KB (36 x 36), 32 planes up to 104 KB (one
// right-hand side of 12 x 45 x 45: 26.1 us by the passes, 27.3 here; 16: 27.3
// either way; 24: 31.9 and 29.0), 96 above (24 x 50 x 50 35.3 and 34.4, 12 x 50 x
// 50 28.0 and 31.6, 48 x 54 x 54 44.1 and 43.0).  The number of right-hand sides
// does not enter, so that a batch rounds like its members.
// (56 x 56 planes were slower at one right-hand side: 46 and 52 us at 56^3.)
// No upper limit on the number of planes: 256 x 16 x 16 36 us, 47 by the passes, 256
// x 32 x 32 51 and 57, with 8 right-hand sides 239 and 326, 500 x 54 x 54 342 and 423.
int plane_yz_setup(Context& c) {
  c.mv.plane = 0;
  const YzShape* z = z_shape(c.mv.gz);
  if (!z || !y_split(c.mv.gy)) return 0;
  const size_t lds = lds_bytes(c.mv, z);
  const int planes = c.mv.gx;
  if (lds > YZ_LDS || planes < (lds <= 80 * 1024 ? 0 : lds <= 104 * 1024 ? 32 : 96)) return 0;
  c.mv.plane = 1;
  DDH_TRY(hipFuncSetAttribute(z->kernel(!c.ipbc), hipFuncAttributeMaxDynamicSharedMemorySize, (int)YZ_LDS),
          "plane kernel LDS", 206);
  return 0;
}

void plane_yz_stages(const Context& c, FftPlan& y, FftPlan& z) {
  const YzSplit* s = y_split(c.mv.gy);
  y = FftPlan{c.mv.gy, 2, {s->R2, s->R1}};
  z = z_shape(c.mv.gz)->stages();
}

int plane_yz_launch(Context& c, hipStream_t st, const MvBatch& bt) {
  const MatvecPlan& m = c.mv;
  const YzShape* z = z_shape(m.gz);
  const YzSplit* y = y_split(m.gy);
  YzGeo q{};
  q.R1 = y->R1; q.R2 = y->R2;
  q.cp = z->pitch();
  q.mz = (1u << 18) / (unsigned)c.nz + 1;
  q.m1 = (1u << 18) / (unsigned)q.R1 + 1;
  q.ny = c.ny; q.nz = c.nz; q.nzp = m.nzp; q.p1 = m.p1; q.gx = m.gx;
  q.nrhs = bt.nrhs;
  // Threads: the fewest rounds of z columns (64 / T per wave, two thirds of the
  // kernel) and of level items, under a cap that leaves room for the
  // workgroups whose LDS fits a CU.
  const size_t lds = lds_bytes(m, z);
  const int wgs = 2 * c.nx * bt.nrhs, fit = wgs <= 256 ? 1 : std::min(4, (int)(YZ_LDS / lds));
  const int items = 3 * c.nz * std::max(q.R1, q.R2);
  const auto rounds = [](int n, int per) { return (n + per - 1) / per; };
  int threads = 0, best = 0;
  for (int w = 1; w <= YZ_MAX_THREADS / 64 / fit; ++w) {
    const int cost = 3 * rounds(m.gy, w * z->seq) + rounds(items, 64 * w);
    if (!threads || cost < best) { threads = 64 * w; best = cost; }
  }
  const unsigned blocks = (unsigned)((c.nx + 7) / 8 * 8 * 2 * bt.nrhs);
  const float2 *green = c.green, *twy = m.twy, *twz = m.twz;
  float2* a1 = bt.a1;
  BatchArgs ba = bt.k;
  GreenGeo gg = green_geo(c);
  void* args[] = {&a1, (void*)&green, (void*)&twy, (void*)&twz, &ba, &gg, &q};
  DDH_TRY(hipLaunchKernel(z->kernel(!c.ipbc), dim3(blocks), dim3((unsigned)threads), args, lds, st),
          "MATVEC plane kernel", 23);
  return 0;
}

}  // namespace ddhip
