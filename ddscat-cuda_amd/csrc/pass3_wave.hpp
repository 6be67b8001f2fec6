// Green pass of FFT3D (pass 3): z-FFT, symmetric 3x3 Green multiply, inverse
// z-FFT, in place on the contiguous z columns of a2[3][2NX][p2: 2NY][nzp].
//
// A column's three components sit in the registers of T lanes of one
// wavefront (fft_wave.hpp), 64 / T columns per wave, and nothing in the
// kernel synchronises a workgroup after the twiddle table is loaded: the
// columns of a wave are loaded, transformed and stored independently of every
// other wave, so memory, LDS and VALU phases of different waves overlap.
//
// What bounds it: VALU issue, 60 % of the cycles at 256 points (128^3), 76 % at
// 512 and 98 % at 768, where the power limit also holds the clock at 1.7 GHz;
// 95 % of the instructions are FP32 arithmetic.  Measured against the kernels
// this one replaced, which walked z with the plane stride and synchronised
// 256- to 768-thread workgroups at every exchange (bytes: a2 in and out and the
// octant once):
//   128^3, 256 points: 148 -> 128 us (4.0 TB/s; 136 to 139 in runs of a few MATVECs)
//   256^3, 512 points: 1,830 -> 1,110 us (3.6 TB/s; 1,090 to 1,330, with the clock)
//   384^3, 768 points: 7,700 -> 4,110 us (3.3 TB/s; to 4,480)
#pragma once
#include "fft_wave.hpp"
#include "mv_device.hpp"
#include <type_traits>

namespace ddhip {

constexpr int P3_WAVES = 4;  // waves per workgroup (1 to 8 measured within 4 %)

// Column order.  Workgroups go round-robin over the 8 XCDs by linear id; the
// columns that read the same Green octant entries (kx and 2NX - kx, ky and
// 2NY - ky) are given to workgroups 8 ids apart, and so are the B right-hand
// sides of a batch, so the entries come from HBM once and from that XCD's L2
// for the others.
//  aligned: blocks of `per` consecutive ky of one kx, in groups of four
//           mirrors (+-kx, block b and nkb - 1 - b);
//  flat:    blocks of `per` consecutive columns slot 2NY + ky of the half
//           slot < H, in groups of two (+-kx); taken where 2NY leaves more
//           than an eighth of an aligned block's lanes idle.
struct P3Cols {
  KxSlab sl;  // the planes of a2
  int per;    // columns per workgroup
  int flat;
  int nkb;    // aligned: ky blocks per kx; flat: blocks per half
  int groups; // groups of mirrors
  int nrhs;
};
inline P3Cols p3_cols(const KxSlab& sl, int gy, int per, int nrhs) {
  P3Cols q;
  q.sl = sl;
  q.per = per;
  q.nrhs = nrhs;
  const int nkb = (gy + per - 1) / per;
  q.flat = (long long)8 * nkb * per > (long long)9 * gy;
  if (q.flat) {
    q.nkb = (int)(((long long)sl.H * gy + per - 1) / per);
    q.groups = q.nkb;
  } else {
    q.nkb = nkb;
    q.groups = sl.H * ((nkb + 1) / 2);
  }
  return q;
}
inline unsigned p3_blocks(const P3Cols& q) { return (unsigned)((q.groups + 7) / 8 * 8 * (q.flat ? 2 : 4) * q.nrhs); }
// right-hand side of this workgroup and (plane slot, ky) of its column `col`; ky < 0 past the end
__device__ __forceinline__ void p3_column(const P3Cols& q, int col, int gy, int& rb, int& ps, int& ky) {
  const int x8 = (int)blockIdx.x & 7, sq = (int)blockIdx.x >> 3, nm = q.flat ? 2 : 4;
  const int sp = sq / q.nrhs;
  rb = sq - sp * q.nrhs;
  const int g = sp / nm, slot = sp - g * nm, grp = g * 8 + x8;
  ky = -1;
  ps = 0;
  if (grp >= q.groups) return;
  int half;
  if (q.flat) {
    const int hc = grp * q.per + col;
    half = hc / gy;
    if (half >= q.sl.H) return;
    ky = hc - half * gy;
  } else {
    const int hb = (q.nkb + 1) / 2;
    half = grp / hb;
    const int b0 = grp - half * hb, b = (slot & 1) ? q.nkb - 1 - b0 : b0;
    if ((slot & 1) && b == b0) return;
    ky = b * q.per + col;
    if (ky >= gy) { ky = -1; return; }
  }
  const int mx = q.flat ? slot : slot >> 1;
  ps = half + mx * q.sl.H;
}

// Green points are loaded in groups of two (12 registers each; groups of one
// and four points 133 and 129 us against 122 at 128^3).  MIRROR: octant stored (IPBC=0), else the whole
// grid (one kernel with both forms of the multiply keeps a second copy of the
// column live across the branch: 256 instead of 161 registers at 16 x 16)
// z-FFT, Green multiply and inverse z-FFT of a column held as stage-0 inputs
// in v; xb: the column's exchange slots; g0: byte offset of its Green entries
template <class PL, bool MIRROR>
__device__ __forceinline__ void p3_transform(float2 (&v)[3][PL::V], float2* xb, const float2* tw, int j,
                                             const char* gb, unsigned g0) {
  constexpr int L = PL::L, SL = PL::S - 1, RL = PL::rad(SL);
#pragma unroll
  for (int c = 0; c < 3; ++c) w_forward<PL, +1>(v[c], xb, tw, j);
#pragma unroll
  for (int b = 0; b < PL::nb(SL); ++b)
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int e = b * RL + r, k = w_bfly<PL, SL>(j, b) + r * (L / RL);
      // a point lies in the mirrored half k > L / 2 when 2 r >= RL, but for
      // k = L / 2 itself and, with an odd RL, the middle group's first half
      const bool up = MIRROR && 2 * r + 1 >= RL;
      const bool mixed = MIRROR && (2 * r == RL || 2 * r + 1 == RL);
      const bool hi = up && (!mixed || k > L / 2);
      const Green6 G = green_at_b(gb, g0 + (unsigned)(hi ? L - k : k) * 48u);
      float2 g13 = G.xz, g23 = G.yz;
      if (mixed) {
        const float sz = hi ? -1.f : 1.f;
        g13 = cscale(g13, sz);
        g23 = cscale(g23, sz);
      } else if (up) {
        g13 = make_float2(-g13.x, -g13.y);
        g23 = make_float2(-g23.x, -g23.y);
      }
      const float2 p0 = v[0][e], p1 = v[1][e], p2 = v[2][e];
      v[0][e] = cdot3(G.xx, p0, G.xy, p1, g13, p2);
      v[1][e] = cdot3(G.xy, p0, G.yy, p1, g23, p2);
      v[2][e] = cdot3(g13, p0, g23, p1, G.zz, p2);
      if (e & 1) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int c = 0; c < 3; ++c) w_inverse<PL, -1>(v[c], xb, tw, j);
}
// The waves per SIMD that 6 V registers of column data leave room for are
// asked of the compiler: left alone it ends a few registers above a step now
// and then (18 x 16 points at 170 instead of 168, 2 waves instead of 3: 385 us
// against 326 on a 200 x 162 x 144 grid).
template <class PL>
constexpr int p3_waves_per_simd() {
  return PL::V <= 12 ? 4 : PL::V <= 18 ? 3 : 2;
}
template <class PL, bool MIRROR>
__global__ __launch_bounds__(64 * P3_WAVES) __attribute__((amdgpu_waves_per_eu(p3_waves_per_simd<PL>()))) void kw_pass3(
    float2* __restrict__ a2, const float2* __restrict__ green, const float2* __restrict__ twg, int nz, int nzp, int p2, int gy,
    BatchArgs ba, GreenGeo gg, P3Cols q) {
  constexpr int L = PL::L, T = PL::T, V = PL::V, SEQ = PL::SEQ, R0 = PL::rad(0);
  static_assert(R0 % 2 == 0, "the zero half of a padded column is a compile-time set");
  __shared__ float2 tw[L];
  __shared__ float2 xbuf[P3_WAVES * SEQ * PL::SLOTS];
  for (int i = threadIdx.x; i < L; i += 64 * P3_WAVES) tw[i] = twg[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, seq = lane / T, j = lane - seq * T;
  if (T * SEQ < 64 && seq >= SEQ) return;
  int rb, ps, ky;
  p3_column(q, w * SEQ + seq, gy, rb, ps, ky);
  if (ky < 0 || (ba.active && !ba.active[rb])) return;
  const int kx = q.sl.kx(ps);
  float2* const xb = xbuf + (w * SEQ + seq) * PL::SLOTS;
  // workgroup-uniform base per component, 32-bit byte offsets per lane (the
  // launcher checks that a component and the Green array span < 4 GiB)
  char* const cb = reinterpret_cast<char*>(a2 + rb * ba.a2s);
  const size_t csb = (size_t)(2 * q.sl.H) * p2 * sizeof(float2);
  const unsigned o0 = ((unsigned)ps * (unsigned)p2 + (unsigned)ky * (unsigned)nzp) * 8u;
  // stage-0 inputs: v[c][b R0 + r] = x_c[j + T b + r L / R0], zero for r >= R0 / 2
  float2 v[3][V];
#pragma unroll
  for (int b = 0; b < PL::nb(0); ++b) {
    const unsigned o = o0 + 8u * (unsigned)w_bfly<PL, 0>(j, b);
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        v[c][b * R0 + r] = 2 * r < R0 ? *reinterpret_cast<const float2*>(cb + c * csb + (o + 8u * (r * (L / R0))))
                                      : make_float2(0.f, 0.f);
  }
  // Octant mirror signs (cu:109-115): G at a mirrored point is D G D with
  // D = diag(sx, sy, sz), so sx and sy go onto components 0 and 1 of the
  // column before and after, and sz onto the off-diagonals of its upper half.
  const int ir = min(kx, gg.mx - kx), jr = min(ky, gg.my - ky);
  const float sx = kx <= gg.tx ? 1.f : -1.f, sy = ky <= gg.ty ? 1.f : -1.f;
#pragma unroll
  for (int e = 0; e < PL::nb(0) * R0; ++e)
    if (2 * (e % R0) < R0) {
      v[0][e] = cscale(v[0][e], sx);
      v[1][e] = cscale(v[1][e], sy);
    }
  const unsigned g0 = ((unsigned)ir * (unsigned)gg.oy + (unsigned)jr) * (unsigned)gg.oz * 48u;
  p3_transform<PL, MIRROR>(v, xb, tw, j, reinterpret_cast<const char*>(green), g0);
#pragma unroll
  for (int b = 0; b < PL::nb(0); ++b) {
    const unsigned ob = o0 + 8u * (unsigned)w_bfly<PL, 0>(j, b);
#pragma unroll
    for (int r = 0; 2 * r < R0; ++r) {
      const unsigned o = ob + 8u * (r * (L / R0));
      *reinterpret_cast<float2*>(cb + o) = cscale(v[0][b * R0 + r], sx);
      *reinterpret_cast<float2*>(cb + csb + o) = cscale(v[1][b * R0 + r], sy);
      *reinterpret_cast<float2*>(cb + 2 * csb + o) = v[2][b * R0 + r];
    }
  }
  // the padding up to nzp, so that the column's last 128-byte line is written whole
  for (int n = nz + j; n < nzp; n += T)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      *reinterpret_cast<float2*>(cb + c * csb + o0 + 8u * (unsigned)n) = make_float2(0.f, 0.f);
}

template <class PL>
static void launch_kw_pass3(Context& c, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const P3Cols q = p3_cols(bt.slab, m.gy, P3_WAVES * PL::SEQ, bt.nrhs);
  const auto kernel = c.ipbc ? &kw_pass3<PL, false> : &kw_pass3<PL, true>;
  hipLaunchKernelGGL(kernel, dim3(p3_blocks(q)), dim3(64 * P3_WAVES), 0, st, bt.a2, c.green, m.twz, c.nz, m.nzp, m.p2, m.gy,
                     bt.k, green_geo(c), q);
}
struct P3Shape {
  int L;
  void (*fn)(Context&, const MvBatch&, hipStream_t);
  FftPlan (*stages)();
};
// P3_PLAN(lanes per column, radices...)
#define P3_PLAN(...) P3Shape{WPlan<__VA_ARGS__>::L, &launch_kw_pass3<WPlan<__VA_ARGS__>>, &w_stages<WPlan<__VA_ARGS__>>}
const P3Shape* p3_shapes_short(int& n);   // up to 160 points
const P3Shape* p3_shapes_medium(int& n);  // 162 to 324
const P3Shape* p3_shapes_long(int& n);    // 360 to 768

}  // namespace ddhip
