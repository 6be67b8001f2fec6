// Device pieces shared by the register MATVEC kernels: site maps, the 3x3
// Green product, and the finish of the last pass.
//
// Compact vectors: when every lattice row's occupied sites form one interval
// [rowlo, rowlo + count) (true for convex targets), the compact index of
// (row g, ix) is rowptr[g] + ix - rowlo[g] and no per-site index is read;
// otherwise a full-site -> compact map (qmap, -1 for void sites) is used.
#pragma once
#include "state.hpp"

namespace ddhip {

struct SiteMap {
  const int* rowptr;
  const int* rowlo;
  const int* qmap;
  int contiguous;
};

// whether any of rows q0 .. q0 + C - 1 (q = iy nzp + iz) is in the support; uniform
template <int C>
__device__ __forceinline__ bool rows_in_support(const BatchArgs& ba, int q0, int ny, int nzp) {
  if (!ba.ysup) return true;
  const int zt = 1 << ba.zsh;
  int iy = q0 / nzp, iz = q0 - iy * nzp;
  bool any = false;
  for (int n = 0; n < C && iy < ny; n += zt) {
    const int2 r = ba.ysup[iz >> ba.zsh];
    any |= iy >= r.x && iy < r.y;
    iz += zt;
    if (iz >= nzp) { iz -= nzp; ++iy; }
  }
  return any;
}

// compact index of site (row g, ix), or -1 when void
__device__ __forceinline__ int compact_index(const SiteMap& m, int g, int ix, int nx) {
  if (m.contiguous) {
    const int lo = m.rowlo[g], q0 = m.rowptr[g], cnt = m.rowptr[g + 1] - q0;
    const int d = ix - lo;
    return (d >= 0 && d < cnt) ? q0 + d : -1;
  }
  return m.qmap[(size_t)g * nx + ix];
}

// g0 p0 + g1 p1 + g2 p2 as two FMA chains (6 instructions per part)
__device__ __forceinline__ float2 cdot3(float2 g0, float2 p0, float2 g1, float2 p1, float2 g2, float2 p2) {
  float re = g0.x * p0.x, im = g0.x * p0.y;
  re = fmaf(-g0.y, p0.y, re);
  im = fmaf(g0.y, p0.x, im);
  re = fmaf(g1.x, p1.x, re);
  im = fmaf(g1.x, p1.y, im);
  re = fmaf(-g1.y, p1.y, re);
  im = fmaf(g1.y, p1.x, im);
  re = fmaf(g2.x, p2.x, re);
  im = fmaf(g2.x, p2.y, im);
  re = fmaf(-g2.y, p2.y, re);
  im = fmaf(g2.y, p2.x, im);
  return make_float2(re, im);
}
// Green entry at byte offset off
__device__ __forceinline__ Green6 green_at_b(const char* __restrict__ g, unsigned off) {
  const float4 a = *reinterpret_cast<const float4*>(g + off);
  const float4 b = *reinterpret_cast<const float4*>(g + off + 16u);
  const float4 c = *reinterpret_cast<const float4*>(g + off + 32u);
  return Green6{make_float2(a.x, a.y), make_float2(a.z, a.w), make_float2(b.x, b.y),
                make_float2(b.z, b.w), make_float2(c.x, c.y), make_float2(c.z, c.w)};
}
// d x - (inv.x + inv.y) w: the convolution's scale as a float and the rest
// (matvec_scale), which enters where a product is rounded anyway
__device__ __forceinline__ float2 scaled_site(float2 d, float2 x, float2 w, float2 inv) {
  const float re = fmaf(d.x, x.x, -fmaf(d.y, x.y, w.x * inv.y));
  const float im = fmaf(d.x, x.y, fmaf(d.y, x.x, -(w.y * inv.y)));
  return make_float2(fmaf(-w.x, inv.x, re), fmaf(-w.y, inv.x, im));
}
// one site of the finish (cu:116-118): r = d x - w / G + offdiag(a) x, conjugated in and out with cj
__device__ __forceinline__ void finish_site(const float2* x, const float2* d, const float2* a, float2 w1, float2 w2,
                                            float2 w3, float2 inv, bool cj, float2& r1, float2& r2, float2& r3) {
  float2 x1 = x[0], x2 = x[1], x3 = x[2];
  const float2 a23 = a[0], a31 = a[1], a12 = a[2];
  if (cj) { x1.y = -x1.y; x2.y = -x2.y; x3.y = -x3.y; }
  r1 = cadd(scaled_site(d[0], x1, w1, inv), cadd(cmul(a31, x3), cmul(a12, x2)));
  r2 = cadd(scaled_site(d[1], x2, w2, inv), cadd(cmul(a12, x1), cmul(a23, x3)));
  r3 = cadd(scaled_site(d[2], x3, w3, inv), cadd(cmul(a23, x2), cmul(a31, x1)));
  if (cj) { r1.y = -r1.y; r2.y = -r2.y; r3.y = -r3.y; }
}
// finish of row g (cu:116-118): y = adia x - w/G + offdiag(aoff) x on the
// unpadded outputs; w0..w2[n2] hold the inverse-transformed components at
// row index ix(n2) for n2 < H, kept(n2, ix) says whether ix < nx (compact
// or full layout, conj for 'C').  Site indices are resolved first with the
// layout test outside the element loop; the loads then run unconditionally
// in groups of FG outputs (an unoccupied site reads entry 0 and stores
// nothing), so each group's 9 FG loads are in flight together instead of
// waiting on per-output branches.
template <int H, int FG, typename IX, typename KEPT>
__device__ __forceinline__ void p5_finish_at(const float2* w0, const float2* w1, const float2* w2, IX ixof, KEPT kept,
                                             int g, const float2* __restrict__ x, float2* __restrict__ y,
                                             const float2* __restrict__ adia, const float2* __restrict__ aoff,
                                             const int16_t* __restrict__ iocc, const SiteMap& sm, int nx, int nat,
                                             int nat0, int compact, int cj, float2 inv) {
  size_t o[H];
  bool st[H], zr[H];
  if (!compact) {
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int ix = ixof(n2);
      st[n2] = kept(n2, ix);
      o[n2] = st[n2] ? (size_t)g * nx + ix : 0;
      zr[n2] = iocc && iocc[o[n2]] == 0;
    }
  } else if (sm.contiguous) {
    const int lo = sm.rowlo[g], q0 = sm.rowptr[g], cnt = sm.rowptr[g + 1] - q0;
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int ix = ixof(n2), d = ix - lo;
      st[n2] = kept(n2, ix) && d >= 0 && d < cnt;
      o[n2] = st[n2] ? (size_t)(q0 + d) : 0;
      zr[n2] = false;
    }
  } else {
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int ix = ixof(n2);
      const int q = kept(n2, ix) ? sm.qmap[(size_t)g * nx + ix] : -1;
      st[n2] = q >= 0;
      o[n2] = st[n2] ? (size_t)q : 0;
      zr[n2] = false;
    }
  }
  const size_t sd = compact ? (size_t)nat0 : (size_t)nat;
#pragma unroll
  for (int g0 = 0; g0 < H; g0 += FG) {
    float2 xv[FG][3], dv[FG][3], av[FG][3];
#pragma unroll
    for (int j = 0; j < FG && g0 + j < H; ++j)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const size_t e = o[g0 + j] + k * sd;
        xv[j][k] = x[e];
        dv[j][k] = adia[e];
        av[j][k] = aoff[e];
      }
#pragma unroll
    for (int j = 0; j < FG && g0 + j < H; ++j) {
      const int n2 = g0 + j;
      float2 r1, r2, r3;
      finish_site(xv[j], dv[j], av[j], w0[n2], w1[n2], w2[n2], inv, cj != 0, r1, r2, r3);
      if (zr[n2]) r1 = r2 = r3 = make_float2(0.f, 0.f);
      if (st[n2]) {
        const size_t e = o[n2];
        y[e] = r1; y[e + sd] = r2; y[e + 2 * sd] = r3;
      }
    }
  }
}

}  // namespace ddhip
