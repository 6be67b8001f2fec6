// Register column kernels: the y passes (2 and 4) of FFT3D and the three
// transforms of the SLICES backend, on the two-level and Stockham register
// FFTs of fft_reg.hpp.  The x passes of FFT3D are in rows.hpp, its Green pass
// in pass3_wave.hpp; the tables of all register kernels meet at the end.
#include "fft_reg.hpp"
#include "mv_device.hpp"
#include "pass3_wave.hpp"
#include "rows.hpp"
#include "solver_common.hpp"
#include <type_traits>

namespace ddhip {

// ------------------------------------------------------------ passes 2, 4
// element j of component c of a MATVEC input as BatchArgs' gather fields
// name it, or 0 when !take (the SLICES z-forward pass reads x itself, compact
// or conjugated).  MAP: compact input through the site map.  Branch-free: a
// lane that takes nothing loads site 0 and discards it, so a thread's
// site-map loads, then its x loads, issue back to back.
template <bool MAP>
__device__ __forceinline__ float2 gathered(const BatchArgs& ba, int c, size_t j, bool take) {
  j = take ? j : 0;
  float2 v;
  if constexpr (MAP) {
    const int q = ba.gmap[j];
    take = take && q >= 0;
    v = ba.gsrc[(size_t)c * ba.gcs + (q >= 0 ? q : 0)];
  } else {
    v = ba.gsrc[(size_t)c * ba.gcs + j];
  }
  if (!take) v = make_float2(0.f, 0.f);
  if (ba.gconj) v.y = -v.y;
  return v;
}

// Columns of a strided transform: column q = o ni + i (i < ni) of component c
// starts at c cin + o ins + i of the input and c cout + o outs + i of the
// output, and its elements follow at `pitch`.  Columns of different o share
// workgroups, so a short inner extent ni costs no idle lanes.
struct Cols {
  int ni, total, pitch;
  size_t ins, outs, cin, cout;
};
// o and i of column q0 + s, q0 the workgroup's first column (divided once, as a scalar)
__device__ __forceinline__ void column_of(const Cols& q, int q0, int s, int& o, int& i) {
  o = q0 / q.ni;
  i = q0 - o * q.ni + s;
  while (i >= q.ni) {
    i -= q.ni;
    ++o;
  }
}
// nin inputs -> nout outputs per column.
// GA (DIR = +1, one o: the SLICES z pass): input element n of column i is
// gathered(ba, c, n pitch + i).
template <int R1, int R2, int C, int DIR, bool GA = false>
__global__ __launch_bounds__(R1 * C) void kr_passy(const float2* __restrict__ in, float2* __restrict__ out,
                                               const float2* __restrict__ twg, Cols q, int nin, int nout,
                                               BatchArgs ba) {
  constexpr int L = R1 * R2, RT = R1 * C, P = C + 1, G = Reg2<R1, R2>::G, VN = Reg2<R1, R2>::VN;
  __shared__ float2 twL[L];
  __shared__ float2 buf[L * P];
  const int rb = blockIdx.z / 3;
  if (ba.active && !ba.active[rb]) return;
  in += rb * (DIR > 0 ? ba.a1s : ba.a2s);
  out += rb * (DIR > 0 ? ba.a2s : ba.a1s);
  const int s = threadIdx.x % C, t = threadIdx.x / C;
  const int q0 = xcd_tile<C>((int)blockIdx.x, (int)gridDim.x, false) * C, c = blockIdx.z % 3;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  const bool live = q0 + s < q.total;
  int o, col;
  column_of(q, q0, live ? s : 0, o, col);
  const int gx = q.pitch;
  const float2* src = in + c * q.cin + o * q.ins + col;
  float2* dst = out + c * q.cout + o * q.outs + col;
  float2 v[VN];
  if (DIR > 0) {
    auto load = [&](auto mapc) {
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int n = t + R1 * n2;
        const bool take = live && lower_half<R2>(n2, n, nin);
        if constexpr (GA)
          v[n2] = gathered<decltype(mapc)::value>(ba, c, (size_t)n * gx + col, take);
        else
          v[n2] = take ? src[(size_t)n * gx] : make_float2(0.f, 0.f);
      }
    };
    if (GA && ba.gmap)
      load(std::true_type{});
    else
      load(std::false_type{});
    __syncthreads();
    fft2_fwd<R1, R2, +1>(v, buf, twL, t, s, P);
    if (live) {
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int k1 = 0; k1 < R1; ++k1)
          if (reg2_owns<R1, R2>(t, i)) dst[(size_t)((t + R1 * i) + R2 * k1) * gx] = v[i * R1 + k1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1)
        v[i * R1 + k1] = (live && reg2_owns<R1, R2>(t, i)) ? src[(size_t)((t + R1 * i) + R2 * k1) * gx]
                                                           : make_float2(0.f, 0.f);
    __syncthreads();
    fft2_inv<R1, R2, -1>(v, buf, twL, t, s, P);
    if (live) {
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int n = t + R1 * n2;
        if (lower_half<R2>(n2, n, nout)) dst[(size_t)n * gx] = v[n2];
      }
    }
  }
}

// ------------------------------------------------ passes 2, 4, L = M * 256
// Column pass of kr_passy for L = M * 256 (M = 2, 3) by decimation in time
// over 256-point register FFTs (16 x 16): thread group m of M transforms
// x[M n1 + m], the twiddle w_L^{m k1} and an M-point DFT through LDS leave
// group m holding X[k1 + 256 m].  16 values per thread, real and imaginary
// parts exchanged in turn (256-point FFTs and the M-point combine), so a
// 768-point column tile of C = 8 needs about 36 KB of LDS instead of the
// 61 KB of the two-level 32 x 24 shape.  DIR = +1: nin (<= L/2, pruned)
// inputs -> L spectral outputs; DIR = -1: L spectral inputs -> nout (<= L/2).
// GA as in kr_passy.
template <int M, int C, int DIR, bool GA = false>
__global__ __launch_bounds__(M * 16 * C) void kr_passym(const float2* __restrict__ in, float2* __restrict__ out,
                                                    const float2* __restrict__ twg, Cols q, int nin, int nout,
                                                    BatchArgs ba) {
  constexpr int R = 16, S = R * R, L = M * S, GT = R * C, RT = M * GT;
  constexpr int PS = M * C + 1;  // 256-point exchange: M C sequences per workgroup (floats)
  constexpr int PC = C + 1;      // M-point exchange layout (u S + k1) PC + s, u < M (floats)
  constexpr int XB = S * PS > M * S * PC ? S * PS : M * S * PC;
  __shared__ float2 twL[L];
  __shared__ float2 twS[S];
  __shared__ float xf[XB];
  const int rb = blockIdx.z / 3;
  if (ba.active && !ba.active[rb]) return;
  in += rb * (DIR > 0 ? ba.a1s : ba.a2s);
  out += rb * (DIR > 0 ? ba.a2s : ba.a1s);
  const int m = threadIdx.x / GT, lt = threadIdx.x % GT;
  const int s = lt % C, t = lt / C, sv = m * C + s;
  const int q0 = xcd_tile<C>((int)blockIdx.x, (int)gridDim.x, false) * C, c = blockIdx.z % 3;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  for (int i = threadIdx.x; i < S; i += RT) twS[i] = twg[M * i];
  const bool live = q0 + s < q.total;
  int o, col;
  column_of(q, q0, live ? s : 0, o, col);
  const int gx = q.pitch;
  const float2* src = in + c * q.cin + o * q.ins + col;
  float2* dst = out + c * q.cout + o * q.outs + col;
  float2 v[R];
  // M-point DFT across the groups, through LDS in two halves: the real
  // parts cross first and are held (M R floats), then each output reads the
  // imaginary parts at its k1 and combines (DIR: sign of the M-point DFT;
  // the inverse then applies the conjugate twiddle w_L^{-m k1})
  auto combine = [&](auto dirc) {
    constexpr int D = decltype(dirc)::value;
    float zr[M][R];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i) xf[(m * S + t + R * i) * PC + s] = v[i].x;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int u = 0; u < M; ++u) zr[u][i] = xf[(u * S + t + R * i) * PC + s];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i) xf[(m * S + t + R * i) * PC + s] = v[i].y;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i) {
      float2 z[M];
#pragma unroll
      for (int u = 0; u < M; ++u) z[u] = make_float2(zr[u][i], xf[(u * S + t + R * i) * PC + s]);
      v[i] = dft_m_out<M, D>(z, m);
      if (D < 0) {
        float2 w = twL[m * (t + R * i)];
        w.y = -w.y;
        v[i] = cmul(v[i], w);
      }
    }
  };
  if (DIR > 0) {
    auto load = [&](auto mapc) {
#pragma unroll
      for (int n2 = 0; n2 < R; ++n2) {
        const int n = M * (t + R * n2) + m;
        const bool take = live && n2 < R / 2 && n < nin;
        if constexpr (GA)
          v[n2] = gathered<decltype(mapc)::value>(ba, c, (size_t)n * gx + col, take);
        else
          v[n2] = take ? src[(size_t)n * gx] : make_float2(0.f, 0.f);
      }
    };
    if (GA && ba.gmap)
      load(std::true_type{});
    else
      load(std::false_type{});
    __syncthreads();
    fft2_fwd_s<R, R, +1>(v, xf, twS, t, sv, PS);  // v[i] = Y_m[t + 16 i]
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = cmul(v[i], twL[m * (t + R * i)]);
    combine(std::integral_constant<int, +1>{});  // v[i] = X[t + 16 i + 256 m]
    if (live) {
#pragma unroll
      for (int i = 0; i < R; ++i) dst[(size_t)(t + R * i + S * m) * gx] = v[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = live ? src[(size_t)(t + R * i + S * m) * gx] : make_float2(0.f, 0.f);
    combine(std::integral_constant<int, -1>{});  // v[i] = W_m[t + 16 i]
    __syncthreads();
    fft2_inv_s<R, R, -1>(v, xf, twS, t, sv, PS);  // v[n2] = x[M (t + 16 n2) + m]
    if (live) {
#pragma unroll
      for (int n2 = 0; n2 < R / 2; ++n2) {
        const int n = M * (t + R * n2) + m;
        if (n < nout) dst[(size_t)n * gx] = v[n2];
      }
    }
  }
}

// -------------------------------------------------- SLICES Green pass
// Column (kx, kz = k0 + plane) of a slice batch [planes][3][NY][2NX],
// transform along y.  Element n of component c is at col[n es + c cs]; the
// transform has nf nonzero inputs and kept outputs.  The Green entry of point
// k is at pb + step min(k, mf - k); the off-diagonal signs are c12, c13, c23
// times the parity of k (k <= tf) for the components that involve y (octant
// mirror rules for IPBC=0, cu:166-186; IPBC=1 has no mirrors and all signs +1).
struct P3Col {
  float2* col;
  size_t es, cs;
  int nf;
  size_t pb, step;
  int mf, tf;
  float c12, c13, c23;
};
// a2 points at plane 0 of the batch, k0 is the batch's first kz
__device__ __forceinline__ P3Col p3_col(float2* a2, int kx, int kz, int ny, int gx, int k0, const GreenGeo& gg) {
  P3Col q;
  const int ir = kx < gx ? min(kx, gg.mx - kx) : 0;
  const float sx = kx <= gg.tx ? 1.f : -1.f;
  const int kr = min(kz, gg.mz - kz);
  const float sz = kz <= gg.tz ? 1.f : -1.f;
  q.col = a2 + (size_t)(kz - k0) * 3 * ny * gx + kx;
  q.es = gx;
  q.cs = (size_t)ny * gx;
  q.nf = ny;
  q.pb = (size_t)ir + (size_t)gg.ox * gg.oy * kr;
  q.step = gg.ox;
  q.mf = gg.my; q.tf = gg.ty;
  q.c12 = sx; q.c13 = sx * sz; q.c23 = sz;
  return q;
}
// Green multiply of point k along the transform: p0..p2 in, G p out
__device__ __forceinline__ void p3_green(const P3Col& q, const float2* __restrict__ green, int k, float2& p0,
                                         float2& p1, float2& p2) {
  const int kr = min(k, q.mf - k);
  const float sf = k <= q.tf ? 1.f : -1.f;
  const Green6 G = green_at(green, q.pb + q.step * kr);
  const float2 g12 = cscale(G.xy, q.c12 * sf);
  const float2 g13 = cscale(G.xz, q.c13);
  const float2 g23 = cscale(G.yz, q.c23 * sf);
  const float2 a = p0, b = p1, c = p2;
  p0 = cadd(cadd(cmul(G.xx, a), cmul(g12, b)), cmul(g13, c));
  p1 = cadd(cadd(cmul(g12, a), cmul(G.yy, b)), cmul(g23, c));
  p2 = cadd(cadd(cmul(g13, a), cmul(g23, b)), cmul(G.zz, c));
}

// y-FFT, Green multiply at kz and inverse y-FFT over a batch of kz planes
// starting at k0 (grid rows = planes of the batch).
template <int R1, int R2, int C>
__global__ __launch_bounds__(R1 * C) void kr_sly(float2* __restrict__ a2, const float2* __restrict__ green,
                                               const float2* __restrict__ twg, int ny, int gx, int k0,
                                               const int* __restrict__ act, GreenGeo gg) {
  constexpr int L = R1 * R2, RT = R1 * C, P = C + 1, G = Reg2<R1, R2>::G, VN = Reg2<R1, R2>::VN;
  __shared__ float2 twL[L];
  __shared__ float2 buf[L * P];
  if (act && !*act) return;  // inactive right-hand side of a batch
  const int s = threadIdx.x % C, t = threadIdx.x / C;
  // Grid order puts Green-sharing blocks on one XCD (workgroups go round-robin
  // over the 8 XCDs by linear id): column tile b and its mirror NT-1-b are
  // h = ceil(NT/2) grid columns apart (NT = column tiles).
  const int NT = gridDim.x, h = (NT + 1) / 2;
  const int tile = (int)blockIdx.x < h ? (int)blockIdx.x : NT - 1 - ((int)blockIdx.x - h);
  const int kx = tile * C + s;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  const bool live = kx < gx;
  const P3Col q = p3_col(a2, kx, k0 + (int)blockIdx.y, ny, gx, k0, gg);
  float2 v0[VN], v1[VN], v2[VN];
#pragma unroll
  for (int n2 = 0; n2 < R2; ++n2) {
    const int n = t + R1 * n2;
    const bool ok = live && lower_half<R2>(n2, n, q.nf);
    const size_t o = (size_t)n * q.es;
    v0[n2] = ok ? q.col[o] : make_float2(0.f, 0.f);
    v1[n2] = ok ? q.col[o + q.cs] : make_float2(0.f, 0.f);
    v2[n2] = ok ? q.col[o + 2 * q.cs] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft2_fwd<R1, R2, +1>(v0, buf, twL, t, s, P);
  __syncthreads();
  fft2_fwd<R1, R2, +1>(v1, buf, twL, t, s, P);
  __syncthreads();
  fft2_fwd<R1, R2, +1>(v2, buf, twL, t, s, P);
  // 3x3 symmetric Green multiply.  Each octant entry serves up to eight
  // mirror points; the mirrors along the transform are in this block and the
  // others run on the same XCD at about the same time (grid order above), so
  // repeats hit in L2.
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
      const int e = i * R1 + k1;
      p3_green(q, green, (t + R1 * i) + R2 * k1, v0[e], v1[e], v2[e]);
    }
  }
  __syncthreads();
  fft2_inv<R1, R2, -1>(v0, buf, twL, t, s, P);
  __syncthreads();
  fft2_inv<R1, R2, -1>(v1, buf, twL, t, s, P);
  __syncthreads();
  fft2_inv<R1, R2, -1>(v2, buf, twL, t, s, P);
  if (live) {
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int n = t + R1 * n2;
      if (lower_half<R2>(n2, n, q.nf)) {
        const size_t o = (size_t)n * q.es;
        q.col[o] = v0[n2];
        q.col[o + q.cs] = v1[n2];
        q.col[o + 2 * q.cs] = v2[n2];
      }
    }
  }
}

// The same for 512- and 768-point y axes with register Stockham transforms
// (fft_reg.hpp, SkPlan): a column of L = 2 NY points is held by T = L / V
// threads with V values per component.  C columns per workgroup, thread (col,
// j) at threadIdx.x = j C + col so that a wave's loads run along kx.
// Addresses are a workgroup-uniform base per component plus a 32-bit byte
// offset per lane (one register per address instead of two); the launcher
// checks that the Green array spans less than 4 GiB.
template <class PL, int C, int NBUF, int K, int WPE, int GS, bool RC>
__global__ __launch_bounds__(PL::T * C) __attribute__((amdgpu_waves_per_eu(WPE))) void kr_sly_s(
    float2* __restrict__ a2, const float2* __restrict__ green, const float2* __restrict__ twg, int ny, int gx, int k0,
    const int* __restrict__ act, GreenGeo gg) {
  constexpr int L = PL::L, T = PL::T, V = PL::V, NTH = T * C, R0 = PL::rad(0), RL = PL::rad(PL::S - 1);
  __shared__ float2 twL[L];
  __shared__ float2 xb[NBUF * K * L * C];
  if (act && !*act) return;
  const int col = threadIdx.x % C, j = threadIdx.x / C;
  const int tile = xcd_tile<C>((int)blockIdx.x, (int)gridDim.x, true);
  const int kx = tile * C + col;
  for (int i = threadIdx.x; i < L; i += NTH) twL[i] = twg[i];
  const bool live = kx < gx;
  const int kz = k0 + (int)blockIdx.y;
  const P3Col q = p3_col(a2, kx, kz, ny, gx, k0, gg);
  // uniform base of the tile's first column; lane offset (col + n es) * 8 bytes
  char* const cb = reinterpret_cast<char*>(a2 + (size_t)(kz - k0) * 3 * ny * gx + (size_t)tile * C);
  const size_t csb = q.cs * sizeof(float2);
  const unsigned esb = (unsigned)(q.es * sizeof(float2));
  const unsigned lane0 = (unsigned)(col * sizeof(float2));
  // stage-0 gathers: v[c][b R0 + r] = x_c[j + T b + r L / R0]; the upper
  // half (r >= R0 / 2) is the zero padding
  float2 v[3][V];
#pragma unroll
  for (int b = 0; b < V / R0; ++b)
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      const unsigned o = lane0 + (unsigned)sk_gather<PL, 0>(j + T * b, r) * esb;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        v[c][b * R0 + r] = (live && 2 * r < R0) ? *reinterpret_cast<const float2*>(cb + c * csb + o)
                                                : make_float2(0.f, 0.f);
    }
  __syncthreads();
  // K = 3: the three components advance stage by stage together; K = 1: one after another
  SkLds<PL, C, NBUF, K, RC> lx{xb};
  // 3x3 symmetric Green multiply at k = i + r L / R_last (octant point
  // pb + step min(k, mf - k), 48 bytes each)
  const char* const gb = reinterpret_cast<const char*>(green);
  const unsigned pb48 = (unsigned)q.pb * 48u, st48 = (unsigned)q.step * 48u;
#pragma unroll
  for (int c = 0; c < 3; c += K) sk_forward<PL, C, NBUF, K, +1>(v[c], lx, twL, j, col);
#pragma unroll
  for (int b = 0; b < V / RL; ++b)
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int e = b * RL + r, k = j + T * b + r * (L / RL);
      const float sf = k <= q.tf ? 1.f : -1.f;
      const Green6 G = green_at_b(gb, pb48 + (unsigned)min(k, q.mf - k) * st48);
      const float2 g12 = cscale(G.xy, q.c12 * sf);
      const float2 g13 = cscale(G.xz, q.c13);
      const float2 g23 = cscale(G.yz, q.c23 * sf);
      const float2 p0 = v[0][e], p1 = v[1][e], p2 = v[2][e];
      v[0][e] = cdot3(G.xx, p0, g12, p1, g13, p2);
      v[1][e] = cdot3(g12, p0, G.yy, p1, g23, p2);
      v[2][e] = cdot3(g13, p0, g23, p1, G.zz, p2);
      // at most GS points' Green loads (12 registers each) in flight
      if ((e + 1) % GS == 0) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int c = 0; c < 3; c += K) sk_inverse<PL, C, NBUF, K, -1>(v[c], lx, twL, j, col);
  if (live) {
#pragma unroll
    for (int b = 0; b < V / R0; ++b)
#pragma unroll
      for (int r = 0; 2 * r < R0; ++r) {
        const unsigned o = lane0 + (unsigned)sk_gather<PL, 0>(j + T * b, r) * esb;
#pragma unroll
        for (int c = 0; c < 3; ++c) *reinterpret_cast<float2*>(cb + c * csb + o) = v[c][b * R0 + r];
      }
  }
}

// ------------------------------------------------------------------ host --
// ------------------------------------------------ SLICES x passes (register)
// Rows of a batch of kz planes, row r = (b 3 + c) NY + iy for plane
// kz = k0 + b and component c.  DIR = +1: x-FFT of zwork row
// [c][kz][iy] (NX values, zero-padded to 2NX) into slice row r (2NX
// spectral values).  DIR = -1: inverse x-FFT of slice row r back into the
// zwork row (its NX unpadded outputs).  A row past the end is clamped to
// the last row for loading and never stored.
template <int R1, int R2, int C, int DIR>
__global__ __launch_bounds__(R1 * C) void kr_slx(float2* __restrict__ zw, float2* __restrict__ sl,
                                             const float2* __restrict__ twg, int nx, int ny, int gz, int k0,
                                             int nrows, const int* __restrict__ act) {
  if (act && !*act) return;  // inactive right-hand side of a batch
  constexpr int L = R1 * R2, RT = R1 * C, P = row_stride<R1, R2>(), G = Reg2<R1, R2>::G, VN = Reg2<R1, R2>::VN;
  __shared__ float2 twL[L];
  __shared__ float buf[C * P];  // split exchange, row layout
  const int t = threadIdx.x % R1, s = threadIdx.x / R1;
  const int r = blockIdx.x * C + s;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  const bool live = r < nrows;
  const int rr = live ? r : nrows - 1;
  const int iy = rr % ny, bc = rr / ny, c = bc % 3, b = bc / 3;
  float2* zrow = zw + (((size_t)c * gz + k0 + b) * ny + iy) * nx;
  float2* srow = sl + (size_t)rr * L;
  float2 v[VN];
  if (DIR > 0) {
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int n = t + R1 * n2;
      v[n2] = lower_half<R2>(n2, n, nx) ? zrow[n] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft2_fwd_s<R1, R2, +1, 1>(v, buf, twL, t, s, P);
    if (live) {
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int k1 = 0; k1 < R1; ++k1)
          if (reg2_owns<R1, R2>(t, i)) srow[(t + R1 * i) + R2 * k1] = v[i * R1 + k1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1)
        v[i * R1 + k1] = reg2_owns<R1, R2>(t, i) ? srow[(t + R1 * i) + R2 * k1] : make_float2(0.f, 0.f);
    __syncthreads();
    fft2_inv_s<R1, R2, -1, 1>(v, buf, twL, t, s, P);
    if (live) {
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int n = t + R1 * n2;
        if (lower_half<R2>(n2, n, nx)) zrow[n] = v[n2];
      }
    }
  }
}

template <int R1, int R2, int C>
static void launch_slx(Context& c, int dir, float2* zw, float2* sl, int k0, int nb, hipStream_t st,
                       const int* act) {
  const MatvecPlan& m = c.mv;
  const int nrows = nb * 3 * c.ny;
  const dim3 grid((nrows + C - 1) / C);
  if (dir > 0)
    hipLaunchKernelGGL((kr_slx<R1, R2, C, +1>), grid, dim3(R1 * C), 0, st, zw, sl, m.twx, c.nx, c.ny, m.gz, k0, nrows,
                       act);
  else
    hipLaunchKernelGGL((kr_slx<R1, R2, C, -1>), grid, dim3(R1 * C), 0, st, zw, sl, m.twx, c.nx, c.ny, m.gz, k0, nrows,
                       act);
}
using SlxLaunch = void (*)(Context&, int, float2*, float2*, int, int, hipStream_t, const int*);
struct SlxShape {
  int L;
  SlxLaunch fn;
};
// the default row shape of each register length (passes 1 and 5 of FFT3D)
static const SlxShape kSlxShapes[] = {
    {32, &launch_slx<4, 8, 64>},     {48, &launch_slx<8, 6, 32>},     {60, &launch_slx<10, 6, 32>},
    {64, &launch_slx<8, 8, 32>},     {72, &launch_slx<12, 6, 16>},    {80, &launch_slx<10, 8, 32>},
    {96, &launch_slx<12, 8, 16>},    {100, &launch_slx<10, 10, 32>},  {108, &launch_slx<12, 9, 16>},
    {120, &launch_slx<12, 10, 16>},  {128, &launch_slx<8, 16, 32>},   {144, &launch_slx<12, 12, 16>},
    {150, &launch_slx<15, 10, 16>},  {160, &launch_slx<16, 10, 16>},  {180, &launch_slx<15, 12, 16>},
    {192, &launch_slx<16, 12, 16>},  {240, &launch_slx<16, 15, 16>},  {256, &launch_slx<16, 16, 16>},
    {512, &launch_slx<32, 16, 8>},   {768, &launch_slx<32, 24, 8>},
};

int slices_x_reg(Context& c, int dir, float2* zw, float2* sl, int k0, int nb, hipStream_t st, const int* act) {
  if (c.fft_generic) return 0;
  for (const SlxShape& r : kSlxShapes)
    if (r.L == c.mv.gx) {
      r.fn(c, dir, zw, sl, k0, nb, st, act);
      return 1;
    }
  return 0;
}

// ------------------------------------------------ SLICES z passes (register)
// Column FFTs along z over the NX NY columns of a plane (kr_passy with one
// "row", columns at element stride NX NY).  dir = +1: in [3][NZ][NY][NX]
// (the full-layout vector) -> out = zwork [3][2NZ][NY][NX]; dir = -1: zwork ->
// out [3][NZ][NY][NX] (the NZ unpadded outputs).
// one right-hand side (grid z = the 3 components, so RHS index 0) whose
// active flag, when given, is *act
static BatchArgs one_rhs(const int* act) {
  BatchArgs ba;
  ba.active = act;
  return ba;
}
// ba: one_rhs(act), with the gather fields set when the forward pass reads
// the MATVEC's x itself (compact or conjugated)
static Cols slz_cols(const Context& c, int dir) {
  const int plane = c.nx * c.ny;
  const size_t full = (size_t)c.mv.gz * plane, half = (size_t)c.nz * plane;
  return Cols{plane, plane, plane, 0, 0, dir > 0 ? half : full, dir > 0 ? full : half};
}
template <int R1, int R2, int C>
static void launch_slz(Context& c, int dir, const float2* in, float2* out, hipStream_t st, const BatchArgs& ba) {
  const MatvecPlan& m = c.mv;
  const Cols q = slz_cols(c, dir);
  const dim3 grid((q.total + C - 1) / C, 1, 3), block(R1 * C);
  if (dir > 0 && ba.gsrc)
    hipLaunchKernelGGL((kr_passy<R1, R2, C, +1, true>), grid, block, 0, st, in, out, m.twz, q, c.nz, m.gz, ba);
  else if (dir > 0)
    hipLaunchKernelGGL((kr_passy<R1, R2, C, +1>), grid, block, 0, st, in, out, m.twz, q, c.nz, m.gz, ba);
  else
    hipLaunchKernelGGL((kr_passy<R1, R2, C, -1>), grid, block, 0, st, in, out, m.twz, q, m.gz, c.nz, ba);
}
template <int M, int C>
static void launch_slz_m(Context& c, int dir, const float2* in, float2* out, hipStream_t st, const BatchArgs& ba) {
  const MatvecPlan& m = c.mv;
  const Cols q = slz_cols(c, dir);
  const dim3 grid((q.total + C - 1) / C, 1, 3), block(M * 16 * C);
  if (dir > 0 && ba.gsrc)
    hipLaunchKernelGGL((kr_passym<M, C, +1, true>), grid, block, 0, st, in, out, m.twz, q, c.nz, m.gz, ba);
  else if (dir > 0)
    hipLaunchKernelGGL((kr_passym<M, C, +1>), grid, block, 0, st, in, out, m.twz, q, c.nz, m.gz, ba);
  else
    hipLaunchKernelGGL((kr_passym<M, C, -1>), grid, block, 0, st, in, out, m.twz, q, m.gz, c.nz, ba);
}
using SlzLaunch = void (*)(Context&, int, const float2*, float2*, hipStream_t, const BatchArgs&);
struct SlzShape {
  int L;
  SlzLaunch fn;
};
// the default column shape of each register length (passes 2 and 4 of FFT3D);
// 512 and 768 points by decimation over 256-point FFTs (kr_passym, the faster
// y pass of FFT3D at those lengths)
static const SlzShape kSlzShapes[] = {
    {32, &launch_slz<4, 8, 64>},     {48, &launch_slz<8, 6, 32>},     {60, &launch_slz<10, 6, 32>},
    {64, &launch_slz<8, 8, 32>},     {72, &launch_slz<12, 6, 16>},    {80, &launch_slz<10, 8, 32>},
    {96, &launch_slz<12, 8, 16>},    {100, &launch_slz<10, 10, 32>},  {108, &launch_slz<12, 9, 16>},
    {120, &launch_slz<12, 10, 16>},  {128, &launch_slz<8, 16, 32>},   {144, &launch_slz<12, 12, 16>},
    {150, &launch_slz<15, 10, 16>},  {160, &launch_slz<16, 10, 16>},  {180, &launch_slz<15, 12, 16>},
    {192, &launch_slz<16, 12, 16>},  {240, &launch_slz<16, 15, 16>},  {256, &launch_slz<16, 16, 16>},
    {512, &launch_slz_m<2, 16>},     {768, &launch_slz_m<3, 16>},
};

int slices_z_reg_length(int L) {
  for (const SlzShape& r : kSlzShapes)
    if (r.L == L) return 1;
  return 0;
}

int slices_z_reg(Context& c, int dir, const float2* in, float2* out, hipStream_t st, const int* act, bool gather,
                 int compact, int cj) {
  if (c.fft_generic) return 0;
  BatchArgs ba = one_rhs(act);
  if (gather && dir > 0) {
    ba.gsrc = in;
    ba.gmap = compact ? c.qmap : nullptr;
    ba.gcs = compact ? (size_t)c.nat0 : (size_t)c.nat;
    ba.gconj = cj;
  }
  for (const SlzShape& r : kSlzShapes)
    if (r.L == c.mv.gz) {
      r.fn(c, dir, in, out, st, ba);
      return 1;
    }
  return 0;
}

// ------------------------------------------------- SLICES y pass (register)
// y-FFT, Green multiply at kz and inverse y-FFT of nb slice planes starting
// at kz = k0, with the register kernels of pass 3 (column setup p3_col<true>)
template <int R1, int R2, int C>
static void launch_sly(Context& c, float2* sl, int k0, int nb, hipStream_t st, const int* act) {
  const MatvecPlan& m = c.mv;
  hipLaunchKernelGGL((kr_sly<R1, R2, C>), dim3((m.gx + C - 1) / C, nb), dim3(R1 * C), 0, st, sl, c.green, m.twy, c.ny,
                     m.gx, k0, act, green_geo(c));
}
template <class PL, int C, int NBUF, int K, int WPE, int GS, bool RC>
static void launch_sly_s(Context& c, float2* sl, int k0, int nb, hipStream_t st, const int* act) {
  const MatvecPlan& m = c.mv;
  hipLaunchKernelGGL((kr_sly_s<PL, C, NBUF, K, WPE, GS, RC>), dim3((m.gx + C - 1) / C, nb), dim3(PL::T * C), 0, st, sl,
                     c.green, m.twy, c.ny, m.gx, k0, act, green_geo(c));
}
using SlyLaunch = void (*)(Context&, float2*, int, int, hipStream_t, const int*);
struct SlyShape {
  int L;
  SlyLaunch fn;
  bool off32 = false;  // addresses the Green array with 32-bit byte offsets
};
// the default pass-3 shape of each register length
static const SlyShape kSlyShapes[] = {
    {32, &launch_sly<4, 8, 64>},     {48, &launch_sly<8, 6, 32>},     {60, &launch_sly<10, 6, 32>},
    {64, &launch_sly<8, 8, 32>},     {72, &launch_sly<12, 6, 16>},    {80, &launch_sly<10, 8, 32>},
    {96, &launch_sly<12, 8, 16>},    {100, &launch_sly<10, 10, 32>},  {108, &launch_sly<12, 9, 16>},
    {120, &launch_sly<12, 10, 16>},  {128, &launch_sly<8, 16, 32>},   {144, &launch_sly<12, 12, 16>},
    {150, &launch_sly<15, 10, 16>},  {160, &launch_sly<16, 10, 16>},  {180, &launch_sly<15, 12, 16>},
    {192, &launch_sly<16, 12, 16>},  {240, &launch_sly<16, 15, 16>},  {256, &launch_sly<16, 16, 16>},
    {512, &launch_sly_s<SkPlan<8, 8, 8, 8>, 8, 2, 1, 4, 4, true>, true},
    {768, &launch_sly_s<SkPlan<12, 12, 4, 4, 4>, 8, 2, 1, 2, 4, false>, true},
};

int slices_y_green_reg(Context& c, float2* sl, int k0, int nb, hipStream_t st, const int* act) {
  if (c.fft_generic) return 0;
  for (const SlyShape& r : kSlyShapes)
    if (r.L == c.mv.gy) {
      // the slice buffers are small; a Green array of 4 GiB or more takes
      // the LDS-staged kernel
      if (r.off32 && green_points(c.nx, c.ny, c.nz, c.ipbc) * 6 * sizeof(float2) >= ((size_t)1 << 32)) return 0;
      r.fn(c, sl, k0, nb, st, act);
      return 1;
    }
  return 0;
}

// ------------------------------------------------ passes 2 and 4 of FFT3D
// a1[3][2NX][NY][nzp] <-> a2[3][2NX][2NY][nzp]: y columns of one kx plane,
// lanes over z, elements nzp apart.  The padding columns of a plane go through
// too, so that every tile starts on a 128-byte line and writes whole ones
// (8 right-hand sides of an 80 x 96 x 75 grid: 158 us per pass without, 118 us with).
static Cols y_cols(const Context& c, int dir) {
  const MatvecPlan& m = c.mv;
  const size_t i = dir > 0 ? m.p1 : m.p2, o = dir > 0 ? m.p2 : m.p1;
  return Cols{m.nzp, m.nzp * m.gx, m.nzp, i, o, i * m.gx, o * m.gx};
}
template <int R1, int R2, int C>
static void launch_y(Context& c, int dir, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const Cols q = y_cols(c, dir);
  const dim3 grid((q.total + C - 1) / C, 1, 3 * (unsigned)bt.nrhs), block(R1 * C);
  if (dir > 0)
    hipLaunchKernelGGL((kr_passy<R1, R2, C, +1>), grid, block, 0, st, bt.a1, bt.a2, m.twy, q, c.ny, m.gy, bt.k);
  else
    hipLaunchKernelGGL((kr_passy<R1, R2, C, -1>), grid, block, 0, st, bt.a2, bt.a1, m.twy, q, m.gy, c.ny, bt.k);
}
template <int M, int C>
static void launch_y_m(Context& c, int dir, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const Cols q = y_cols(c, dir);
  const dim3 grid((q.total + C - 1) / C, 1, 3 * (unsigned)bt.nrhs), block(M * 16 * C);
  if (dir > 0)
    hipLaunchKernelGGL((kr_passym<M, C, +1>), grid, block, 0, st, bt.a1, bt.a2, m.twy, q, c.ny, m.gy, bt.k);
  else
    hipLaunchKernelGGL((kr_passym<M, C, -1>), grid, block, 0, st, bt.a2, bt.a1, m.twy, q, m.gy, c.ny, bt.k);
}
struct YShape {
  int L;
  void (*fn)(Context&, int, const MvBatch&, hipStream_t);
};
#define Y_SHAPE(R1, R2, C) YShape{(R1) * (R2), &launch_y<R1, R2, C>}
// One shape per padded length 2N, N = 2^a 3^b 5^c from 12 to 256 and a few
// above (two-level, R1 threads per column, at most 25 values each, C columns
// per workgroup; 512 and 768 points by decimation, 20 and 30 % faster there).
// Lengths with a factor 7 and those above 768 use the LDS-staged kernels.
static const YShape kYShapes[] = {
    Y_SHAPE(6, 4, 32), Y_SHAPE(6, 5, 32), Y_SHAPE(4, 8, 64), Y_SHAPE(6, 6, 32), Y_SHAPE(8, 5, 32), Y_SHAPE(8, 6, 32),
    Y_SHAPE(10, 5, 32), Y_SHAPE(9, 6, 32), Y_SHAPE(10, 6, 32), Y_SHAPE(8, 8, 32), Y_SHAPE(12, 6, 16),
    Y_SHAPE(10, 8, 32), Y_SHAPE(10, 9, 32), Y_SHAPE(12, 8, 16), Y_SHAPE(10, 10, 32), Y_SHAPE(12, 9, 16),
    Y_SHAPE(12, 10, 16), Y_SHAPE(8, 16, 32), Y_SHAPE(12, 12, 16), Y_SHAPE(15, 10, 16), Y_SHAPE(16, 10, 16),
    Y_SHAPE(18, 9, 16), Y_SHAPE(15, 12, 16), Y_SHAPE(16, 12, 16), Y_SHAPE(20, 10, 16), Y_SHAPE(18, 12, 16),
    Y_SHAPE(16, 15, 16), Y_SHAPE(25, 10, 16), Y_SHAPE(16, 16, 32), Y_SHAPE(18, 15, 16), Y_SHAPE(18, 16, 16),
    Y_SHAPE(20, 15, 16), Y_SHAPE(20, 16, 16), Y_SHAPE(18, 18, 16), Y_SHAPE(20, 18, 16), Y_SHAPE(24, 16, 16),
    Y_SHAPE(20, 20, 16), Y_SHAPE(24, 18, 16), Y_SHAPE(25, 18, 16), Y_SHAPE(24, 20, 16), Y_SHAPE(27, 18, 16),
    Y_SHAPE(25, 20, 16), YShape{512, &launch_y_m<2, 16>}, Y_SHAPE(27, 20, 8), Y_SHAPE(24, 24, 8), Y_SHAPE(25, 24, 8),
    Y_SHAPE(32, 20, 8), Y_SHAPE(27, 24, 8), Y_SHAPE(30, 24, 8), Y_SHAPE(30, 25, 8), YShape{768, &launch_y_m<3, 16>},
};

// candidate `cand` of the table entries that `match`
template <class Shape, class Match>
static const Shape* nth(const Shape* t, int n, int cand, Match match) {
  for (int i = 0; i < n; ++i)
    if (match(t[i]) && cand-- == 0) return &t[i];
  return nullptr;
}
static const RowShape* row_shape(int L, int pass, int cand) {
  int n;
  const RowShape* t = L <= 256 ? row_shapes_short(n) : row_shapes_long(n);
  return nth(t, n, cand, [=](const RowShape& r) { return r.L == L && r.pass == pass; });
}
static const P3Shape* p3_shape(int L, int cand) {
  int n;
  const P3Shape* t = L <= 160 ? p3_shapes_short(n) : L <= 324 ? p3_shapes_medium(n) : p3_shapes_long(n);
  return nth(t, n, cand, [=](const P3Shape& r) { return r.L == L; });
}
static const YShape* y_shape(int L, int cand) {
  return nth(kYShapes, (int)(sizeof(kYShapes) / sizeof(kYShapes[0])), cand, [=](const YShape& r) { return r.L == L; });
}

int reg_candidates(int L, int which) {
  int n = 0;
  while (which == 3 ? p3_shape(L, n) != nullptr
                    : (which == 1 || which == 5) ? row_shape(L, which, n) != nullptr : y_shape(L, n) != nullptr)
    ++n;
  return n;
}

// launches register pass `which` (1..5) with shape `cand` of its axis length;
// returns 1 when launched, 0 when the caller should use the generic kernel
int reg_pass(Context& c, int which, int cand, int cj, int compact, const float2* x, float2* y, const float2* adia,
             const float2* aoff, hipStream_t st, const MvBatch& bt) {
  const MatvecPlan& m = c.mv;
  if (cand < 0) return 0;
  if (which == 1 || which == 5) {
    const RowShape* r = row_shape(m.gx, which, cand);
    if (r) r->fn(c, RowArgs{cj, compact, x, y, adia, aoff}, bt, st);
    return r != nullptr;
  }
  if (which == 3) {
    // the wave kernel addresses a component of a2 and the Green array with
    // 32-bit byte offsets; larger grids take the LDS-staged kernel
    const size_t lim = (size_t)1 << 32, comp = (size_t)m.gx * m.p2 * sizeof(float2);
    if (comp >= lim || green_points(c.nx, c.ny, c.nz, c.ipbc) * 6 * sizeof(float2) >= lim) return 0;
    const P3Shape* r = p3_shape(m.gz, cand);
    if (r) r->fn(c, bt, st);
    return r != nullptr;
  }
  const YShape* r = y_shape(m.gy, cand);
  if (r) r->fn(c, which == 2 ? +1 : -1, bt, st);
  return r != nullptr;
}

}  // namespace ddhip
