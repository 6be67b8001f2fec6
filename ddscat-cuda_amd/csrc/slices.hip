// SLICES (low-memory) MATVEC backend for gfx950.
//
// Same operator as FFT3D (ddscat_cuda_unified/cuda/ddscat_matvec_cuda.cu:136-214,
// 361-404) with the kernels of FFT3D.  Pass 1 leaves the x spectra of all
// rows in a1 [3][2NX][NY][nzp] (6 NAT complex); every kx plane is then on its
// own until pass 5, so passes 2 to 4 run over slabs of kx planes (H planes and
// their H mirrors, which read the same Green entries) held in a small a2:
//   y-FFT (+i) into the slab's [3][2H][2NY][nzp], z-FFT, Green multiply and
//   inverse z-FFT in place, inverse y-FFT back into the planes of a1.
// Slabs alternate between two HIP streams, each with its own a2, so that one
// slab's memory-bound y passes run beside the other's Green pass.
#include "solver_common.hpp"
#include <algorithm>

namespace ddhip {

struct SliceState {
  float2* a2[2] = {nullptr, nullptr};
  hipStream_t side[2] = {nullptr, nullptr};
  hipEvent_t ev_in = nullptr, ev_done[2] = {nullptr, nullptr};
  int H = 0;  // half-planes per slab
  int nslab = 0;
};
static SliceState g_sl[MAX_TARGETS + 1];  // one per target slot

int slices_setup(Context& c) {
  if (int rc = matvec_plan(c, "SLICES plan")) return rc;
  MatvecPlan& m = c.mv;
  if (m.gy > 2048) {
    set_error("SLICES plan", "padded grid axis exceeds the LDS FFT limit (2N <= 2048)");
    return 206;
  }
  SliceState& s = g_sl[c.slot];
  s = SliceState{};
  // Slabs: one (the whole a2, no side streams) up to 64 MiB, where a launch
  // costs as much as its work (64^3: 53 us against 117 in four slabs and 169
  // in eight; 90 x 75 x 81: 107 against 151), then as many of 64 MiB, between
  // four, whose two buffers are half of a2, and eight, above which the
  // smaller slabs only add launches (256^3: 2,709 us in eight, 2,717 in 32;
  // 384^3: 9,595 and 9,834).
  const size_t one = (size_t)64 << 20, all = matvec_a2_count(c) * sizeof(float2);
  const int n = all <= one ? 1 : (int)std::min<size_t>(8, std::max<size_t>(4, (all + one - 1) / one));
  s.H = (c.nx + n - 1) / n;
  s.nslab = (c.nx + s.H - 1) / s.H;
  DDH_TRY(hipMalloc((void**)&c.a1, matvec_a1_count(c) * sizeof(float2)), "malloc SLICES x spectra", 204);
  for (int i = 0; i < std::min(2, s.nslab); ++i)
    DDH_TRY(hipMalloc((void**)&s.a2[i], (size_t)6 * s.H * m.p2 * sizeof(float2)), "malloc SLICES slab", 204);
  if (s.nslab == 1) return 0;
  for (int i = 0; i < 2; ++i) {
    DDH_TRY(hipStreamCreateWithFlags(&s.side[i], hipStreamNonBlocking), "create SLICES stream", 206);
    DDH_TRY(hipEventCreateWithFlags(&s.ev_done[i], hipEventDisableTiming), "create SLICES event", 206);
  }
  DDH_TRY(hipEventCreateWithFlags(&s.ev_in, hipEventDisableTiming), "create SLICES event", 206);
  return 0;
}

void slices_release(Context& c) {
  SliceState& s = g_sl[c.slot];
  for (int i = 0; i < 2; ++i) {
    if (s.side[i]) {
      hipStreamSynchronize(s.side[i]);
      hipStreamDestroy(s.side[i]);
    }
    if (s.a2[i]) hipFree(s.a2[i]);
    if (s.ev_done[i]) hipEventDestroy(s.ev_done[i]);
  }
  if (s.ev_in) hipEventDestroy(s.ev_in);
  s = SliceState{};
}

void slices_slab(const Context& c, int h0, MvBatch& bt) {
  const SliceState& s = g_sl[c.slot];
  bt.slab = KxSlab{h0, std::min(s.H, c.nx - h0), c.mv.gx};
  bt.a2 = s.a2[h0 / s.H & 1];
}

int slices_matvec(Context& c, int cwhat, const float2* x, float2* y, const float2* adia, const float2* aoff,
                  int layout, hipStream_t st, const int* act) {
  SliceState& s = g_sl[c.slot];
  if (!s.H) { set_error("SLICES MATVEC", "backend not prepared"); return 20; }
  MvBatch bt;
  bt.a1 = c.a1;
  bt.k.active = act;
  matvec_support(c, layout, bt.k);
  if (int rc = matvec_end_pass(c, 1, cwhat, x, y, adia, aoff, layout, st, bt)) return rc;
  if (plane_yz_runs(c)) {
    if (int rc = plane_yz_launch(c, st, bt)) return rc;
  } else if (s.nslab == 1) {
    slices_slab(c, 0, bt);
    if (int rc = matvec_slab(c, st, bt)) return rc;
  } else {
    DDH_TRY(hipEventRecord(s.ev_in, st), "SLICES record", 25);
    for (int i = 0; i < 2; ++i) DDH_TRY(hipStreamWaitEvent(s.side[i], s.ev_in, 0), "SLICES wait", 25);
    for (int k = 0; k < s.nslab; ++k) {
      slices_slab(c, k * s.H, bt);
      if (int rc = matvec_slab(c, s.side[k & 1], bt)) return rc;
    }
    for (int i = 0; i < 2; ++i) {
      DDH_TRY(hipEventRecord(s.ev_done[i], s.side[i]), "SLICES record", 25);
      DDH_TRY(hipStreamWaitEvent(st, s.ev_done[i], 0), "SLICES wait", 25);
    }
  }
  if (int rc = matvec_end_pass(c, 5, cwhat, x, y, adia, aoff, layout, st, bt)) return rc;
  DDH_LAUNCH_OK("SLICES register passes", 29);
  c.matvec_count++;
  return 0;
}

}  // namespace ddhip
