// Register column kernels: the y passes (2 and 4) on the two-level register
// FFTs of fft_reg.hpp.  The x passes are in rows.hpp, the Green pass in
// pass3_wave.hpp; the tables of all register kernels meet at the end.
#include "fft_reg.hpp"
#include "mv_device.hpp"
#include "pass3_wave.hpp"
#include "rows.hpp"
#include "solver_common.hpp"
#include <type_traits>

namespace ddhip {

// ------------------------------------------------------------ passes 2, 4
// The columns of a y pass: column q = slot ni + i (i < ni) of component c, its
// elements `pitch` apart.  The a1 side counts planes by kx, the a2 side by
// slot.  Columns of different planes share workgroups, so a short inner
// extent ni costs no idle lanes.
struct Cols {
  int ni, total, pitch;
  size_t p1, p2, c1, c2;  // plane and component strides in a1 and a2
  KxSlab sl;
};
// Tile of this workgroup.  Where tiles share 128-byte lines (z runs of no whole
// lines, tiles of less than one) neighbours run on one XCD: MATVECs with the
// tiles dealt out over the XCDs, and so, 80 x 80 x 20 with 8 right-hand sides 174 ->
// 137 us, 80 x 80 x 28 243 -> 209, 100^3 181 -> 175, 120^3 302 -> 292; on whole lines
// 128^3 and 192^3 were up to 1 % slower so.
template <int C>
__device__ __forceinline__ int y_tile(const Cols& q) {
  return C < 16 || q.pitch % 16 ? xcd_run((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
}
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
template <int R1, int R2, int C, bool SPL, int DIR>
__global__ __launch_bounds__(R1 * C) void kr_passy(const float2* __restrict__ in, float2* __restrict__ out,
                                               const float2* __restrict__ twg, Cols q, int nin, int nout,
                                               BatchArgs ba) {
  constexpr int L = R1 * R2, RT = R1 * C, P = C + 1, G = Reg2<R1, R2>::G, VN = Reg2<R1, R2>::VN;
  __shared__ float2 twL[L];
  __shared__ float2 buf[SPL ? (L * P + 1) / 2 : L * P];
  float* const bufs = reinterpret_cast<float*>(buf);
  const int rb = blockIdx.z / 3;
  if (ba.active && !ba.active[rb]) return;
  in += rb * (DIR > 0 ? ba.a1s : ba.a2s);
  out += rb * (DIR > 0 ? ba.a2s : ba.a1s);
  const int s = threadIdx.x % C, t = threadIdx.x / C;
  const int q0 = y_tile<C>(q) * C, c = blockIdx.z % 3;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  const bool live = q0 + s < q.total;
  int o, col;
  column_of(q, q0, live ? s : 0, o, col);
  const int gx = q.pitch;
  const size_t o1 = c * q.c1 + q.sl.kx(o) * q.p1 + col, o2 = c * q.c2 + o * q.p2 + col;
  const float2* src = in + (DIR > 0 ? o1 : o2);
  float2* dst = out + (DIR > 0 ? o2 : o1);
  float2 v[VN];
  if (DIR > 0) {
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int n = t + R1 * n2;
      v[n2] = live && lower_half<R2>(n2, n, nin) ? src[(size_t)n * gx] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    if constexpr (SPL)
      fft2_fwd_s<R1, R2, +1>(v, bufs, twL, t, s, P);
    else
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
    if constexpr (SPL)
      fft2_inv_s<R1, R2, -1>(v, bufs, twL, t, s, P);
    else
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
// SUP: only the inputs or outputs in the row support.
template <int M, int C, int DIR, bool SUP>
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
  const int q0 = y_tile<C>(q) * C, c = blockIdx.z % 3;
  for (int i = threadIdx.x; i < L; i += RT) twL[i] = twg[i];
  for (int i = threadIdx.x; i < S; i += RT) twS[i] = twg[M * i];
  const bool live = q0 + s < q.total;
  int o, col;
  column_of(q, q0, live ? s : 0, o, col);
  const int2 sup = SUP ? ba.ysup[col >> ba.zsh] : make_int2(0, DIR > 0 ? nin : nout);
  const int gx = q.pitch;
  const size_t o1 = c * q.c1 + q.sl.kx(o) * q.p1 + col, o2 = c * q.c2 + o * q.p2 + col;
  const float2* src = in + (DIR > 0 ? o1 : o2);
  float2* dst = out + (DIR > 0 ? o2 : o1);
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
#pragma unroll
    for (int n2 = 0; n2 < R; ++n2) {
      const int n = M * (t + R * n2) + m;
      v[n2] = live && n2 < R / 2 && (!SUP || n >= sup.x) && n < sup.y ? src[(size_t)n * gx] : make_float2(0.f, 0.f);
    }
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
        if ((!SUP || n >= sup.x) && n < sup.y) dst[(size_t)n * gx] = v[n2];
      }
    }
  }
}

// ------------------------------------------------------------------ host --
// ------------------------------------------------ passes 2 and 4
// a1[3][2NX][NY][nzp] <-> a2[3][2H][2NY][nzp]: y columns of one kx plane,
// lanes over z, elements nzp apart.  The padding columns of a plane go through
// too, so that every tile starts on a 128-byte line and writes whole ones
// (8 right-hand sides of an 80 x 96 x 75 grid: 158 us per pass without, 118 us with).
static Cols y_cols(const Context& c, const KxSlab& sl) {
  const MatvecPlan& m = c.mv;
  const size_t p1 = m.p1, p2 = m.p2;
  return Cols{m.nzp, m.nzp * 2 * sl.H, m.nzp, p1, p2, p1 * m.gx, p2 * 2 * sl.H, sl};
}
template <int R1, int R2, int C, bool SPL = false>
static void launch_y(Context& c, int dir, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const Cols q = y_cols(c, bt.slab);
  const dim3 grid((q.total + C - 1) / C, 1, 3 * (unsigned)bt.nrhs), block(R1 * C);
  if (dir > 0)
    hipLaunchKernelGGL((kr_passy<R1, R2, C, SPL, +1>), grid, block, 0, st, bt.a1, bt.a2, m.twy, q, c.ny, m.gy, bt.k);
  else
    hipLaunchKernelGGL((kr_passy<R1, R2, C, SPL, -1>), grid, block, 0, st, bt.a2, bt.a1, m.twy, q, m.gy, c.ny, bt.k);
}
template <int M, int C>
static void launch_y_m(Context& c, int dir, const MvBatch& bt, hipStream_t st) {
  const MatvecPlan& m = c.mv;
  const Cols q = y_cols(c, bt.slab);
  const dim3 grid((q.total + C - 1) / C, 1, 3 * (unsigned)bt.nrhs), block(M * 16 * C);
  if (dir > 0) {
    const auto kernel = bt.k.ysup ? &kr_passym<M, C, +1, true> : &kr_passym<M, C, +1, false>;
    hipLaunchKernelGGL(kernel, grid, block, 0, st, bt.a1, bt.a2, m.twy, q, c.ny, m.gy, bt.k);
  } else {
    const auto kernel = bt.k.ysup ? &kr_passym<M, C, -1, true> : &kr_passym<M, C, -1, false>;
    hipLaunchKernelGGL(kernel, grid, block, 0, st, bt.a2, bt.a1, m.twy, q, m.gy, c.ny, bt.k);
  }
}
struct YShape {
  int L;
  void (*fn)(Context&, int, const MvBatch&, hipStream_t);
  int rad[3];        // its stages in order
  bool sup = false;  // the kernel honours BatchArgs::ysup
};
#define Y_SHAPE(R1, R2, C) YShape{(R1) * (R2), &launch_y<R1, R2, C>, {R2, R1, 1}}
#define Y_SPLIT(R1, R2, C) YShape{(R1) * (R2), &launch_y<R1, R2, C, true>, {R2, R1, 1}}
// One shape per padded length 2N, N = 2^a 3^b 5^c 7^d from 12 to 256 and a few
// above (two-level, R1 threads per column, up to 25 values each to 500 points and
// 24 to 35 above, C columns per workgroup; 512 and 768 points by decimation, 20
// and 30 % faster there).
// The real and imaginary parts cross in turn (Y_SPLIT), with half the LDS and
// twice the workgroups on a CU for two further barriers, at the lengths where
// that gained a percent or more of a MATVEC: 192^3 1,249 -> 1,165 us, 200^3
// 1,536 -> 1,413, 216^3 1,974 -> 1,809, 240^3 2,582 -> 2,520, 144^3 539 -> 529,
// 162^3 827 -> 811 (96^3 to 140^3: 0 to 2 % slower, 250^3 2,825 and 2,984).
// 32 columns where z runs are often no whole lines long and 16 columns then
// straddle two (144, 150 and 180 points: 8 right-hand sides of 64 x 72 x 72 445 ->
// 436 us, 64 x 75 x 64 377 -> 369, 64 x 90 x 72 535 -> 529; 120, 160 and 192 points
// within a percent either way).
// Lengths of other sizes use the LDS-staged kernels (the y passes of a 70^3
// grid: 34 us each against 14 to 16 here, 196^3: 470 against 213 to 235).
static const YShape kYShapes[] = {
    Y_SHAPE(6, 4, 32), Y_SHAPE(6, 5, 32), Y_SHAPE(4, 8, 64), Y_SHAPE(6, 6, 32), Y_SHAPE(8, 5, 32), Y_SHAPE(8, 6, 32),
    Y_SHAPE(10, 5, 32), Y_SHAPE(9, 6, 32), Y_SHAPE(10, 6, 32), Y_SHAPE(8, 8, 32), Y_SHAPE(12, 6, 16),
    Y_SHAPE(10, 8, 32), Y_SHAPE(10, 9, 32), Y_SHAPE(12, 8, 16), Y_SHAPE(10, 10, 32), Y_SHAPE(12, 9, 16),
    Y_SHAPE(12, 10, 16), Y_SHAPE(8, 16, 32), Y_SHAPE(12, 12, 32), Y_SHAPE(15, 10, 32), Y_SHAPE(16, 10, 16),
    Y_SHAPE(18, 9, 16), Y_SHAPE(15, 12, 32), Y_SHAPE(16, 12, 16), Y_SHAPE(20, 10, 16), Y_SHAPE(18, 12, 16),
    Y_SHAPE(16, 15, 16), Y_SHAPE(25, 10, 16), Y_SHAPE(16, 16, 32), Y_SHAPE(18, 15, 16), Y_SPLIT(18, 16, 16),
    Y_SHAPE(20, 15, 16), Y_SHAPE(20, 16, 16), Y_SPLIT(18, 18, 16), Y_SHAPE(20, 18, 16), Y_SPLIT(24, 16, 16),
    Y_SPLIT(20, 20, 16), Y_SPLIT(24, 18, 16), Y_SPLIT(25, 18, 16), Y_SPLIT(24, 20, 16), Y_SHAPE(27, 18, 16),
    Y_SHAPE(25, 20, 16), YShape{512, &launch_y_m<2, 16>, {16, 16, 2}, true}, Y_SHAPE(27, 20, 8), Y_SHAPE(24, 24, 8), Y_SHAPE(25, 24, 8),
    Y_SHAPE(32, 20, 8), Y_SHAPE(27, 24, 8), Y_SHAPE(30, 24, 8), Y_SHAPE(30, 25, 8), YShape{768, &launch_y_m<3, 16>, {16, 16, 3}, true},
    // a factor 7
    Y_SHAPE(7, 4, 32), Y_SHAPE(7, 6, 32), Y_SHAPE(8, 7, 32), Y_SHAPE(10, 7, 32), Y_SHAPE(12, 7, 16),
    Y_SHAPE(14, 7, 16), Y_SHAPE(14, 8, 16), Y_SHAPE(14, 9, 16), Y_SHAPE(14, 10, 16), Y_SHAPE(14, 12, 16),
    Y_SHAPE(14, 14, 32), Y_SHAPE(15, 14, 16), Y_SHAPE(16, 14, 16), Y_SHAPE(18, 14, 16), Y_SHAPE(20, 14, 16),
    Y_SHAPE(21, 14, 16), Y_SHAPE(21, 16, 16), Y_SHAPE(25, 14, 16), Y_SHAPE(27, 14, 16), Y_SHAPE(28, 14, 16),
    Y_SPLIT(30, 14, 16), Y_SHAPE(28, 16, 16), Y_SHAPE(35, 14, 8), Y_SHAPE(28, 18, 8),
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

bool reg_row_support(int L, int cand) {
  const YShape* y = cand < 0 ? nullptr : y_shape(L, cand);
  return y && y->sup;
}

FftPlan reg_stages(int L, int which, int cand) {
  if (which == 3) {
    const P3Shape* r = p3_shape(L, cand);
    return r ? r->stages() : FftPlan{};
  }
  if (which == 1 || which == 5) {
    const RowShape* r = row_shape(L, which, cand);
    return r ? FftPlan{L, 2, {r->R2, r->R1}} : FftPlan{};
  }
  const YShape* y = y_shape(L, cand);
  return y ? FftPlan{L, 3, {y->rad[0], y->rad[1], y->rad[2]}} : FftPlan{};
}

int reg_candidates(int L, int which) {
  int n = 0;
  while (which == 3 ? p3_shape(L, n) != nullptr
                    : (which == 1 || which == 5) ? row_shape(L, which, n) != nullptr : y_shape(L, n) != nullptr)
    ++n;
  return n;
}

bool reg_green_reach(const Context& c, const KxSlab& sl) {
  const size_t lim = (size_t)1 << 32, comp = (size_t)(2 * sl.H) * c.mv.p2 * sizeof(float2);
  return comp < lim && green_points(c.nx, c.ny, c.nz, c.ipbc) * 6 * sizeof(float2) < lim;
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
    if (!reg_green_reach(c, bt.slab)) return 0;
    const P3Shape* r = p3_shape(m.gz, cand);
    if (r) r->fn(c, bt, st);
    return r != nullptr;
  }
  const YShape* r = y_shape(m.gy, cand);
  if (r) r->fn(c, which == 2 ? +1 : -1, bt, st);
  return r != nullptr;
}

}  // namespace ddhip
