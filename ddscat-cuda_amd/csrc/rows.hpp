// x passes of FFT3D: pass 1 (x rows -> a1) and pass 5 (a1 -> finished y).
//
// a1[3][2NX][NY][nzp] keeps z contiguous, so these two passes transpose: a
// workgroup takes C lattice rows that follow each other in z (row q = iy nzp +
// iz; those with iz >= NZ are padding, so that runs start on 128-byte lines), reads or writes them along x with lanes running over x, and touches a1
// with lanes running over the C rows, 8 C contiguous bytes per kx.  The
// change of lane order costs nothing: it happens in the LDS exchange between
// the two levels of the register transform (fft_reg.hpp), which one side
// writes and the other reads with its own thread mapping.  Exchange layout
// (k2 R1 + n1) (C + 1) + s: lanes over s are consecutive and lanes over n1 or
// k2 an odd number of words apart, so neither side conflicts.
#pragma once
#include "fft_reg.hpp"
#include "mv_device.hpp"

namespace ddhip {

// (iy, iz) of row q0 + s, q0 the workgroup's first row (divided once, as a
// scalar); false past the end, which gets row 0.  iz >= NZ: padding row.
__device__ __forceinline__ bool row_of(int q0, int s, int ny, int nzp, int& iy, int& iz) {
  iy = q0 / nzp;
  iz = q0 - iy * nzp + s;
  while (iz >= nzp) {
    iz -= nzp;
    ++iy;
  }
  const bool in = iy < ny;
  iy = in ? iy : 0;
  iz = in ? iz : 0;
  return in;
}

template <int R1, int R2, int C>
__global__ __launch_bounds__(R1 * C) void kx_fwd(const float2* __restrict__ x, float2* __restrict__ a1, SiteMap sm,
                                                 const float2* __restrict__ twg, int nx, int ny, int nz, int nzp, int ks,
                                                 int nat, int nat0, int compact, int cj, BatchArgs ba) {
  constexpr int L = R1 * R2, RT = R1 * C, P = C + 1, G = Reg2<R1, R2>::G, VN = Reg2<R1, R2>::VN;
  __shared__ float2 twL[L];
  __shared__ float buf[L * P];  // real and imaginary parts cross in turn
  const int rb = blockIdx.z;
  if (ba.active && !ba.active[rb]) return;
  x += rb * ba.xs;
  a1 += rb * ba.a1s;
  const int c = blockIdx.y, q0 = blockIdx.x * C;
  if (!rows_in_support<C>(ba, q0, ny, nzp)) return;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  // load side: lanes over x
  const int t = threadIdx.x % R1, s = threadIdx.x / R1;
  int iy, iz;
  const bool live = row_of(q0, s, ny, nzp, iy, iz) && iz < nz;
  const int g = live ? iy + ny * iz : 0;
  // site of each unpadded input n = t + R1 n2 (n2 < H), resolved with the
  // layout test outside the element loop; the loads then run unconditionally
  // (an empty site or a row past the end reads entry 0 and is zeroed), so
  // they are in flight together instead of waiting on per-element branches
  constexpr int H = (R2 + 1) / 2;
  size_t o[H];
  bool ok[H];
  if (!compact) {
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int n = t + R1 * n2;
      ok[n2] = live && lower_half<R2>(n2, n, nx);
      o[n2] = ok[n2] ? (size_t)g * nx + n : 0;
    }
  } else if (sm.contiguous) {
    const int lo = sm.rowlo[g], p0 = sm.rowptr[g], cnt = sm.rowptr[g + 1] - p0;
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int n = t + R1 * n2, d = n - lo;
      ok[n2] = live && lower_half<R2>(n2, n, nx) && d >= 0 && d < cnt;
      o[n2] = ok[n2] ? (size_t)(p0 + d) : 0;
    }
  } else {
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      const int n = t + R1 * n2;
      const int q = live && lower_half<R2>(n2, n, nx) ? sm.qmap[(size_t)g * nx + n] : -1;
      ok[n2] = q >= 0;
      o[n2] = ok[n2] ? (size_t)q : 0;
    }
  }
  float2 v[VN];
  const float2* xc = x + (size_t)c * (compact ? nat0 : nat);
#pragma unroll
  for (int n2 = 0; n2 < H; ++n2) {
    const float2 val = xc[o[n2]];
    v[n2] = ok[n2] ? val : make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int n2 = H; n2 < R2; ++n2) v[n2] = make_float2(0.f, 0.f);
  if (cj) {
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) v[n2].y = -v[n2].y;
  }
  __syncthreads();
  dft_reg<R2, +1>(v);
#pragma unroll
  for (int k2 = 1; k2 < R2; ++k2) v[k2] = cmul(v[k2], twL[t * k2]);
  // store side: lanes over the rows
  const int s2 = threadIdx.x % C, t2 = threadIdx.x / C;
  float re[G * R1];
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) buf[(k2 * R1 + t) * P + s] = v[k2].x;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t2, i)) continue;
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) re[i * R1 + n1] = buf[((t2 + R1 * i) * R1 + n1) * P + s2];
  }
  __syncthreads();
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) buf[(k2 * R1 + t) * P + s] = v[k2].y;
  __syncthreads();
  // padding rows are stored too (zeros): a 128-byte line written in part costs
  // a read of the rest
  if (!row_of(q0, s2, ny, nzp, iy, iz)) return;
  float2* out = a1 + (size_t)c * L * ks + (size_t)iy * nzp + iz;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t2, i)) continue;
    float2 u[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1)
      u[n1] = make_float2(re[i * R1 + n1], buf[((t2 + R1 * i) * R1 + n1) * P + s2]);
    dft_reg<R1, +1>(u);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) out[(size_t)((t2 + R1 * i) + R2 * k1) * ks] = u[k1];
  }
}

// FG: outputs per finish load group.  SPL: real and imaginary parts cross in
// turn (half the LDS).  EARLY: all three components are loaded before the
// first is transformed (6 VN registers, for VN up to 16).
template <int R1, int R2, int C, int FG, bool SPL, bool EARLY>
__global__ __launch_bounds__(R1 * C) void kx_inv(const float2* __restrict__ a1, const float2* __restrict__ twg,
                                                 const float2* __restrict__ x, float2* __restrict__ y,
                                                 const float2* __restrict__ adia, const float2* __restrict__ aoff,
                                                 const int16_t* __restrict__ iocc, SiteMap sm, int nx, int ny, int nz,
                                                 int nzp, int ks, int nat, int nat0, int compact, int cj, float2 inv,
                                                 BatchArgs ba) {
  constexpr int L = R1 * R2, RT = R1 * C, P = C + 1, G = Reg2<R1, R2>::G, VN = G * R1, H = (R2 + 1) / 2;
  __shared__ float2 twL[L];
  __shared__ float buf[(SPL ? 1 : 2) * L * P];
  float2* const buf2 = reinterpret_cast<float2*>(buf);
  const int rb = blockIdx.y;
  if (ba.active && !ba.active[rb]) return;
  a1 += rb * ba.a1s;
  x += rb * ba.xs;
  y += rb * ba.xs;
  adia += rb * ba.os;
  aoff += rb * ba.os;
  const int q0 = blockIdx.x * C;
  if (!rows_in_support<C>(ba, q0, ny, nzp)) return;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  const int s2 = threadIdx.x % C, t2 = threadIdx.x / C;  // load side: lanes over the rows
  const int t = threadIdx.x % R1, s = threadIdx.x / R1;  // finish side: lanes over x
  int iy, iz;
  row_of(q0, s2, ny, nzp, iy, iz);
  const float2* src = a1 + (size_t)iy * nzp + iz;
  float2 v[EARLY ? 3 : 1][VN], w[3][H];
  auto load = [&](int c, float2* d) {
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1)
        d[i * R1 + k1] = reg2_owns<R1, R2>(t2, i) ? src[((size_t)c * L + (t2 + R1 * i) + R2 * k1) * ks]
                                                  : make_float2(0.f, 0.f);
  };
  if (EARLY) {
#pragma unroll
    for (int c = 0; c < 3; ++c) load(c, v[EARLY ? c : 0]);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float2* d = v[EARLY ? c : 0];
    if (!EARLY) load(c, d);
    float2 u[R2];
    if (c == 0) __syncthreads();  // twiddles
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if (!reg2_owns<R1, R2>(t2, i)) continue;
      const int k2 = t2 + R1 * i;
      dft_reg<R1, -1>(d + i * R1);
#pragma unroll
      for (int n1 = 1; n1 < R1; ++n1) {
        const float2 tw = twL[n1 * k2];
        d[i * R1 + n1] = cmul(d[i * R1 + n1], make_float2(tw.x, -tw.y));
      }
    }
    if (c) __syncthreads();  // the previous component's reads
    if constexpr (SPL) {
#pragma unroll
      for (int i = 0; i < G; ++i)
        if (reg2_owns<R1, R2>(t2, i)) {
#pragma unroll
          for (int n1 = 0; n1 < R1; ++n1) buf[((t2 + R1 * i) * R1 + n1) * P + s2] = d[i * R1 + n1].x;
        }
      __syncthreads();
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) u[k2].x = buf[(k2 * R1 + t) * P + s];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < G; ++i)
        if (reg2_owns<R1, R2>(t2, i)) {
#pragma unroll
          for (int n1 = 0; n1 < R1; ++n1) buf[((t2 + R1 * i) * R1 + n1) * P + s2] = d[i * R1 + n1].y;
        }
      __syncthreads();
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) u[k2].y = buf[(k2 * R1 + t) * P + s];
    } else {
#pragma unroll
      for (int i = 0; i < G; ++i)
        if (reg2_owns<R1, R2>(t2, i)) {
#pragma unroll
          for (int n1 = 0; n1 < R1; ++n1) buf2[((t2 + R1 * i) * R1 + n1) * P + s2] = d[i * R1 + n1];
        }
      __syncthreads();
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) u[k2] = buf2[(k2 * R1 + t) * P + s];
    }
    dft_reg<R2, -1>(u);
    // the kept outputs are materialised here: otherwise the last butterflies
    // sink into the finish and hold its loads and their inputs live at once
#pragma unroll
    for (int n2 = 0; n2 < H; ++n2) {
      w[c][n2] = u[n2];
      asm volatile("" : "+v"(w[c][n2].x), "+v"(w[c][n2].y));
    }
  }
  if (!row_of(q0, s, ny, nzp, iy, iz) || iz >= nz) return;
  p5_finish_at<H, FG>(
      w[0], w[1], w[2], [=](int n2) { return t + R1 * n2; },
      [=](int n2, int ix) { return lower_half<R2>(n2, ix, nx); }, iy + ny * iz, x, y, adia, aoff, iocc, sm, nx, nat,
      nat0, compact, cj, inv);
}

struct RowArgs {
  int cj, compact;
  const float2* x;
  float2* y;
  const float2 *adia, *aoff;
};
template <int R1, int R2, int C>
static void launch_kx_fwd(Context& c, const RowArgs& a, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const SiteMap sm{c.rowptr, c.rowlo, c.qmap, c.rows_contiguous};
  const int nrows = c.ny * m.nzp;
  hipLaunchKernelGGL((kx_fwd<R1, R2, C>), dim3((nrows + C - 1) / C, 3, (unsigned)bt.nrhs), dim3(R1 * C), 0, st, a.x,
                     bt.a1, sm, m.twx, c.nx, c.ny, c.nz, m.nzp, m.p1, c.nat, c.nat0, a.compact, a.cj, bt.k);
}
template <int R1, int R2, int C, int FG, bool SPL, bool EARLY>
static void launch_kx_inv(Context& c, const RowArgs& a, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const SiteMap sm{c.rowptr, c.rowlo, c.qmap, c.rows_contiguous};
  const int nrows = c.ny * m.nzp;
  hipLaunchKernelGGL((kx_inv<R1, R2, C, FG, SPL, EARLY>), dim3((nrows + C - 1) / C, (unsigned)bt.nrhs), dim3(R1 * C),
                     0, st, bt.a1, m.twx, a.x, a.y, a.adia, a.aoff, a.compact ? nullptr : c.iocc, sm, c.nx, c.ny, c.nz,
                     m.nzp, m.p1, c.nat, c.nat0, a.compact, a.cj, m.scale, bt.k);
}
struct RowShape {
  int L, pass;  // padded length, pass 1 or 5
  void (*fn)(Context&, const RowArgs&, const MvBatch&, hipStream_t);
  int R1, R2;
};
// the shapes of one length and pass: the first is the default, further ones
// are autotuner candidates
#define X_FWD(R1, R2, C) RowShape{(R1) * (R2), 1, &launch_kx_fwd<R1, R2, C>, R1, R2}
#define X_INV(R1, R2, C, FG, SPL, EARLY) RowShape{(R1) * (R2), 5, &launch_kx_inv<R1, R2, C, FG, SPL, EARLY>, R1, R2}
const RowShape* row_shapes_short(int& n);  // up to 256 points
const RowShape* row_shapes_long(int& n);   // 270 to 768

}  // namespace ddhip
