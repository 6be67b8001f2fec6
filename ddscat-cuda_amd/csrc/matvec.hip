// FFT3D Green-tensor MATVEC for gfx950.
//
// y = adia o x + offdiag(aoff) x - (1/G) F-[ Ghat . F+[pad(x)] ]
// (ddscat_cuda_unified/cuda/ddscat_matvec_cuda.cu:104-118, 406-415; CPU
// semantics ddscat_cuda_unified/fortran/cprod_cuda.f90:446-607), computed as
// five pruned, LDS-staged 1-D FFT passes over the zero-padded 2NX x 2NY x 2NZ
// grid.  Only the non-zero input half of each axis is read and only the
// needed output half is written:
//
//   pass 1  x-FFT (+i)   x[3][NAT] or compact x      -> a1[3][2NX][p1: NY][nzp]
//   pass 2  y-FFT (+i)   a1                            -> a2[3][2NX][p2: 2NY][nzp]
//   pass 3  z-FFT (+i), 3x3 Green multiply, z-FFT (-i), keep iz < NZ (in place in a2)
//   pass 4  y-FFT (-i)   a2, keep iy < NY              -> a1
//   pass 5  x-FFT (-i), keep ix < NX, finish with x, adia, aoff -> y
//
// The work arrays keep z contiguous (pitch nzp), so that the heaviest pass,
// the z transforms around the Green multiply, streams whole columns; passes 1
// and 5 transpose between x rows and z runs on the way through LDS.  This
// file holds the LDS-staged kernels for every axis length; lengths with a
// register shape use the kernels of rows.hpp, matvec_reg.hip and
// pass3_wave.hpp, which read and write the same arrays.
#include "state.hpp"
#include "fft_gain.hpp"
#include "fft_reg.hpp"
#include "mv_device.hpp"
#include <vector>
#include <cmath>
#include <algorithm>
#include <array>
#include <map>
#include <type_traits>

namespace ddhip {

static constexpr int MV_THREADS = 256;
static constexpr int PER_WIDE = 16;   // passes 2, 4
static constexpr int PER_NARROW = 8;  // passes 1, 5, and 3 (three components in LDS)
// Wide tiles: long axes (a 256-thread tile would hold fewer than 8 columns,
// i.e. rows of < 64 contiguous bytes) run passes 2-4 with 1024-thread
// workgroups and up to the device's per-workgroup LDS, so each tile reads
// rows of 8-16 columns; passes 1 and 5 with 512 threads and half the LDS, two
// workgroups to a CU (with 1024 and all of it, 450 x 48 x 48 took 234 us, not 218).
static constexpr int WIDE_THREADS = 1024;
static constexpr int ROW_THREADS = 512;

// x / d as a multiplication, exact for x d < 2^32
struct FastDiv {
  unsigned m;  // ceil(2^32 / d); 0 for d = 1
};
static FastDiv fast_div_by(int d) { return FastDiv{(unsigned)((((uint64_t)1 << 32) + d - 1) / (uint64_t)d)}; }
__device__ __forceinline__ int fast_div(int x, FastDiv d) { return d.m ? (int)__umulhi((unsigned)x, d.m) : x; }

// The x passes: rows q = iy NZ + iz, rx of them per workgroup, interleaved in
// LDS at an odd pitch, so that the vectors are walked with lanes over x and the
// work arrays with lanes over the rows (runs of consecutive z), without
// conflicts.  MATVECs, rows one after another in LDS and often 1 to 5 of them
// before: 280 x 48 x 48 193 -> 138 us, 512 x 96 x 96 1,204 -> 984, 400 x 128 x 128
// 1,607 -> 1,327, 1,024 x 64 x 64 1,407 -> 945, 5 x 128 x 128 with four right-hand
// sides 214 -> 86.
struct RowTile {
  int rx, nr, iy0, z0, nz;  // rows per workgroup, rows of this one, and where it starts
  FastDiv dz, dr;           // by nz and rx
  __device__ __forceinline__ void row(int r, int& iy, int& iz) const {
    const int d = fast_div(z0 + r, dz);
    iy = iy0 + d;
    iz = z0 + r - d * nz;
  }
};
__device__ __forceinline__ RowTile row_tile(int rx, int ny, int nz, FastDiv dz, FastDiv dr) {
  const int q0 = xcd_run((int)blockIdx.x, (int)gridDim.x) * rx, iy0 = q0 / nz;
  return RowTile{rx, min(rx, ny * nz - q0), iy0, q0 - iy0 * nz, nz, dz, dr};
}

// ---------------------------------------------------------------- pass 1 --
template <int PER, int NT = MV_THREADS>
__global__ __launch_bounds__(NT) void k_pass1_xfwd(
    const float2* __restrict__ x, float2* __restrict__ a1, SiteMap map, const float2* __restrict__ twg, FftPlan p,
    int nx, int ny, int nz, int nzp, int ks, int rx, FastDiv dx, FastDiv dz, FastDiv dr, int nat, int nat0, int compact,
    int conj_in, BatchArgs ba) {
  extern __shared__ float2 sm[];
  const int rb = blockIdx.z;
  if (ba.active && !ba.active[rb]) return;
  x += rb * ba.xs;
  a1 += rb * ba.a1s;
  const int L = p.L, rp = rx | 1;  // L = 2 nx
  float2* tw = sm;
  float2* buf = sm + L;
  const int c = blockIdx.y;
  const RowTile t = row_tile(rx, ny, nz, dz, dr);
  const int T = blockDim.x;
  for (int i = threadIdx.x; i < L; i += T) tw[i] = twg[i];
  const float2* xs = x + (size_t)c * (compact ? nat0 : nat);
  for (int idx = threadIdx.x; idx < nx * rx; idx += T) {
    const int r = fast_div(idx, dx), e = idx - r * nx;
    float2 v = make_float2(0.f, 0.f);
    if (r < t.nr) {
      int iy, iz;
      t.row(r, iy, iz);
      const int g = iy + ny * iz;
      const int o = compact ? compact_index(map, g, e, nx) : g * nx + e;
      if (o >= 0) v = xs[o];
      if (conj_in) v.y = -v.y;
    }
    buf[e * rp + r] = v;
    buf[(e + nx) * rp + r] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft_run<+1, true, PER>(buf, tw, p, rx, rp, 1);
  float2* out = a1 + (size_t)c * L * ks;
  for (int idx = threadIdx.x; idx < rx * L; idx += T) {
    const int k = fast_div(idx, t.dr), r = idx - k * rx;
    if (r >= t.nr) continue;
    int iy, iz;
    t.row(r, iy, iz);
    out[(size_t)k * ks + (size_t)iy * nzp + iz] = buf[k * rp + r];
  }
}

// ------------------------------------------------------------- pass 2, 4 --
// a1 [3][gx][p1: ny][nzp] <-> a2 [3][2H][p2: gy][nzp], FFT along the middle axis of
// a plane, cy columns per workgroup: column q = slot ni + iz of ni per plane,
// NZ rounded up to whole tiles or, where that leaves lanes idle, NZ itself with
// tiles that cross planes (MATVECs, whole tiles before: 280 x 280 x 1 241 -> 102 us,
// 512 x 512 x 1 583 -> 203, 512 x 512 x 20 2,080 -> 1,715, 64 x 400 x 4 101 -> 72).
template <int DIR, int PER, int NT = MV_THREADS>
__global__ __launch_bounds__(NT) void k_pass_y(
    const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ twg,
    FftPlan p, KxSlab sl, int nin, int nout, int nz, int nzp, int ins,
    int outs, int cy_log2, int ni, FastDiv dn, BatchArgs ba) {
  extern __shared__ float2 sm[];
  const int rb = blockIdx.z / 3;
  if (ba.active && !ba.active[rb]) return;
  in += rb * (DIR > 0 ? ba.a1s : ba.a2s);
  out += rb * (DIR > 0 ? ba.a2s : ba.a1s);
  const int L = p.L;
  const int cy = 1 << cy_log2;
  float2* tw = sm;
  float2* buf = sm + L;
  const int c = blockIdx.z % 3, q0 = blockIdx.x * cy, slot0 = q0 / ni;
  const int T = blockDim.x;
  for (int i = threadIdx.x; i < L; i += T) tw[i] = twg[i];
  // this thread's column: T is a multiple of cy
  const int i = q0 - slot0 * ni + (threadIdx.x & (cy - 1)), d = fast_div(i, dn);
  const int slot = slot0 + d, iz = i - d * ni;
  const bool live = iz < nz && slot < 2 * sl.H;
  const size_t pl1 = (size_t)c * sl.gx + sl.kx(live ? slot : 0), pl2 = (size_t)c * (2 * sl.H) + slot;
  const float2* src = in + (DIR > 0 ? pl1 : pl2) * ins + iz;
  for (int idx = threadIdx.x; idx < L * cy; idx += T) {
    const int e = idx >> cy_log2;
    float2 v = make_float2(0.f, 0.f);
    if (e < nin && live) v = src[(size_t)e * nzp];
    buf[idx] = v;
  }
  __syncthreads();
  fft_run<DIR, true, PER>(buf, tw, p, cy, cy, 1);
  if (!live) return;
  float2* dst = out + (DIR > 0 ? pl2 : pl1) * outs + iz;
  for (int idx = threadIdx.x; idx < nout * cy; idx += T) {
    const int e = idx >> cy_log2;
    dst[(size_t)e * nzp] = buf[idx];
  }
}

// ---------------------------------------------------------------- pass 3 --
// cz contiguous z columns (slot 2NY + ky) per workgroup, interleaved in LDS at
// an odd pitch cp: global memory and the Green row are walked with lanes over z,
// the butterflies with lanes over the columns, and neither conflicts.  cz fills
// the workgroup also where L is short.  Whole MATVECs against columns one after
// another in LDS, at most 16 of them: 128 x 128 x 1 92 -> 44 us, 128 x 128 x 10
// 117 -> 65, 48 x 48 x 280 305 -> 237, 48 x 48 x 1,024 1,053 -> 789.
template <int PER, int NT = MV_THREADS>
__global__ __launch_bounds__(NT) void k_pass3_z_green(
    float2* __restrict__ a2, const float2* __restrict__ green, const float2* __restrict__ twg,
    FftPlan p, int nz, int nzp, int p2, KxSlab sl, int gy, int cz, FastDiv dz, FastDiv dl, FastDiv dy, BatchArgs ba,
    GreenGeo gg) {
  extern __shared__ float2 sm[];
  const int rb = blockIdx.z;
  if (ba.active && !ba.active[rb]) return;
  a2 += rb * ba.a2s;
  const int L = p.L, cp = cz | 1;  // L = 2 nz
  float2* tw = sm;
  float2* b0 = sm + L;
  float2* b1 = b0 + cp * L;
  float2* b2 = b1 + cp * L;
  const int ncol = 2 * sl.H * gy, q0 = blockIdx.x * cz, nc = min(cz, ncol - q0);
  const int slot0 = q0 / gy, ky0 = q0 - slot0 * gy;
  const int T = blockDim.x;
  const size_t cstride = (size_t)(2 * sl.H) * p2;
  const auto column = [&](int r, int& slot, int& ky) {
    const int d = fast_div(ky0 + r, dy);
    slot = slot0 + d;
    ky = ky0 + r - d * gy;
  };
  const auto address = [&](int r) {
    int slot, ky;
    column(r, slot, ky);
    return (size_t)slot * p2 + (size_t)ky * nzp;
  };
  for (int i = threadIdx.x; i < L; i += T) tw[i] = twg[i];
  for (int idx = threadIdx.x; idx < nz * cz; idx += T) {
    const int r = fast_div(idx, dz), e = idx - r * nz;
    const float2 z = make_float2(0.f, 0.f);
    float2 v0 = z, v1 = z, v2 = z;
    if (r < nc) {
      const size_t o = address(r) + e;
      v0 = a2[o];
      v1 = a2[o + cstride];
      v2 = a2[o + 2 * cstride];
    }
    const int li = e * cp + r, lu = li + nz * cp;
    b0[li] = v0; b1[li] = v1; b2[li] = v2;
    b0[lu] = z; b1[lu] = z; b2[lu] = z;
  }
  __syncthreads();
  fft_run<+1, true, PER>(b0, tw, p, cz, cp, 1);
  fft_run<+1, true, PER>(b1, tw, p, cz, cp, 1);
  fft_run<+1, true, PER>(b2, tw, p, cz, cp, 1);
  // symmetric 3x3 multiply; trimmed-octant reconstruction for IPBC=0
  // (cu:109-115), whole grid for IPBC=1
  for (int idx = threadIdx.x; idx < L * nc; idx += T) {
    const int r = fast_div(idx, dl), kz = idx - r * L;
    int slot, ky;
    column(r, slot, ky);
    const int kx = sl.kx(slot);
    const int ir = min(kx, gg.mx - kx), jr = min(ky, gg.my - ky), kr = min(kz, gg.mz - kz);
    const float sx = kx <= gg.tx ? 1.f : -1.f, sy = ky <= gg.ty ? 1.f : -1.f;
    const float sz = kz <= gg.tz ? 1.f : -1.f;
    const Green6 G = green_at(green, (size_t)kr + (size_t)gg.oz * ((size_t)jr + (size_t)gg.oy * ir));
    const float2 g12 = cscale(G.xy, sx * sy);
    const float2 g13 = cscale(G.xz, sx * sz);
    const float2 g23 = cscale(G.yz, sy * sz);
    const int li = kz * cp + r;
    const float2 p0 = b0[li], p1 = b1[li], p2 = b2[li];
    b0[li] = cadd(cadd(cmul(G.xx, p0), cmul(g12, p1)), cmul(g13, p2));
    b1[li] = cadd(cadd(cmul(g12, p0), cmul(G.yy, p1)), cmul(g23, p2));
    b2[li] = cadd(cadd(cmul(g13, p0), cmul(g23, p1)), cmul(G.zz, p2));
  }
  __syncthreads();
  fft_run<-1, true, PER>(b0, tw, p, cz, cp, 1);
  fft_run<-1, true, PER>(b1, tw, p, cz, cp, 1);
  fft_run<-1, true, PER>(b2, tw, p, cz, cp, 1);
  for (int idx = threadIdx.x; idx < nz * nc; idx += T) {
    const int r = fast_div(idx, dz), e = idx - r * nz;
    const size_t o = address(r) + e;
    const int li = e * cp + r;
    a2[o] = b0[li];
    a2[o + cstride] = b1[li];
    a2[o + 2 * cstride] = b2[li];
  }
}

// ---------------------------------------------------------------- pass 5 --
// One component after another in LDS, the kept half of each waiting in registers;
// `three`: all of them at once, in launches of up to 256 workgroups that have
// the room, which then wait for one round of loads and not for three (5 x 24 x 24
// 25.9 -> 24.5 us, 400 x 10 x 10 67 -> 65).
template <int PER, int NT = MV_THREADS>
__global__ __launch_bounds__(NT, 4) void k_pass5_xinv_finish(
    const float2* __restrict__ a1, const float2* __restrict__ twg, FftPlan p,
    const float2* __restrict__ x, float2* __restrict__ y, const float2* __restrict__ adia,
    const float2* __restrict__ aoff, const int16_t* __restrict__ iocc, SiteMap map, int nx, int ny, int nz, int nzp,
    int ks, int rx, FastDiv dx, FastDiv dz, FastDiv dr, int three, int nat, int nat0, int compact, int cj, float2 inv,
    BatchArgs ba) {
  constexpr int KEEP = PER / 2;  // kept outputs per thread and component
  extern __shared__ float2 sm[];
  const int rb = blockIdx.y;
  if (ba.active && !ba.active[rb]) return;
  a1 += rb * ba.a1s;
  x += rb * ba.xs;
  y += rb * ba.xs;
  adia += rb * ba.os;
  aoff += rb * ba.os;
  const int L = p.L, rp = rx | 1;
  float2* tw = sm;
  float2* buf = sm + L;
  const RowTile t = row_tile(rx, ny, nz, dz, dr);
  const int T = blockDim.x;
  for (int i = threadIdx.x; i < L; i += T) tw[i] = twg[i];
  const size_t cs = (size_t)L * ks;
  // components c0 .. c0 + NC - 1 of the tile, bs apart in LDS
  const int bs = three ? rp * L : 0;
  const auto load = [&](int c0, auto nc) {
    constexpr int NC = decltype(nc)::value;
    for (int idx = threadIdx.x; idx < rx * L; idx += T) {
      const int k = fast_div(idx, t.dr), r = idx - k * rx;
      float2 v[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) v[c] = make_float2(0.f, 0.f);
      if (r < t.nr) {
        int iy, iz;
        t.row(r, iy, iz);
        const float2* src = a1 + c0 * cs + (size_t)k * ks + (size_t)iy * nzp + iz;
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = src[c * cs];
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) buf[(c0 + c) * bs + k * rp + r] = v[c];
    }
    __syncthreads();
  };
  if (three) load(0, std::integral_constant<int, 3>{});
  float2 w[3][KEEP];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (!three) {
      if (c) __syncthreads();
      load(c, std::integral_constant<int, 1>{});
    }
    fft_run<-1, true, PER>(buf + c * bs, tw, p, rx, rp, 1);
#pragma unroll
    for (int j = 0; j < KEEP; ++j) {
      const int idx = threadIdx.x + j * T, r = fast_div(idx, dx), ix = idx - r * nx;
      w[c][j] = r < rx ? buf[c * bs + ix * rp + r] : make_float2(0.f, 0.f);
    }
  }
  const size_t sd = compact ? (size_t)nat0 : (size_t)nat;
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    const int idx = threadIdx.x + j * T, r = fast_div(idx, dx), ix = idx - r * nx;
    if (r >= t.nr) continue;
    int iy, iz;
    t.row(r, iy, iz);
    const int g = iy + ny * iz;
    const int o = compact ? compact_index(map, g, ix, nx) : g * nx + ix;
    if (o < 0) continue;
    float2 r1, r2, r3;
    if (iocc && iocc[o] == 0) {
      r1 = r2 = r3 = make_float2(0.f, 0.f);
    } else {
      float2 xv[3], dv[3], av[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const size_t q = (size_t)o + c * sd;
        xv[c] = x[q];
        dv[c] = adia[q];
        av[c] = aoff[q];
      }
      finish_site(xv, dv, av, w[0][j], w[1][j], w[2][j], inv, cj != 0, r1, r2, r3);
    }
    y[o] = r1; y[o + sd] = r2; y[o + 2 * sd] = r3;
  }
}

// ------------------------------------------------------------------ host --
static int pow2floor(int v) {
  int p = 1;
  while (p * 2 <= v) p *= 2;
  return p;
}
static int ilog2(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

bool fft_make_plan(int L, FftPlan& p) {
  p = FftPlan{};
  p.L = L;
  int m = L;
  std::vector<int> r;
  while (m % 8 == 0) { r.push_back(8); m /= 8; }
  while (m % 4 == 0) { r.push_back(4); m /= 4; }
  while (m % 2 == 0) { r.push_back(2); m /= 2; }
  while (m % 3 == 0) { r.push_back(3); m /= 3; }
  while (m % 5 == 0) { r.push_back(5); m /= 5; }
  while (m % 7 == 0) { r.push_back(7); m /= 7; }
  if (m != 1 || (int)r.size() > FFT_MAX_STAGES || L < 2) return false;
  p.nst = (int)r.size();
  for (int i = 0; i < p.nst; ++i) p.rad[i] = r[i];
  return true;
}

void fft_twiddles_host(int L, float2* out) {
  const double twopi = 6.283185307179586476925286766559;
  for (int m = 0; m < L; ++m) {
    const double a = twopi * (double)m / (double)L;
    out[m] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
}

static int upload_twiddles(int L, float2** dst) {
  std::vector<float2> h(L);
  fft_twiddles_host(L, h.data());
  DDH_TRY(hipMalloc((void**)dst, (size_t)L * sizeof(float2)), "twiddle alloc", 1);
  DDH_TRY(hipMemcpy(*dst, h.data(), (size_t)L * sizeof(float2), hipMemcpyHostToDevice), "twiddle H2D", 1);
  return 0;
}

// per-workgroup LDS bytes of the current device (160 KB on gfx950)
static size_t lds_limit() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
    return 64 * 1024;
  return (size_t)v;
}

// lets the wide-tile kernels take more than 64 KB of dynamic LDS
static int allow_big_lds(size_t bytes) {
  const void* const wide[] = {(const void*)k_pass1_xfwd<PER_NARROW, ROW_THREADS>,
                              (const void*)k_pass5_xinv_finish<PER_NARROW, ROW_THREADS>,
                              (const void*)k_pass_y<+1, PER_WIDE, WIDE_THREADS>,
                              (const void*)k_pass_y<-1, PER_WIDE, WIDE_THREADS>,
                              (const void*)k_pass3_z_green<PER_NARROW, WIDE_THREADS>};
  for (const void* k : wide)
    if (const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        e != hipSuccess) {
      set_hip_error("MATVEC plan (wide LDS tiles)", e);
      return 1;
    }
  return 0;
}

int matvec_plan(Context& c, const char* name) {
  MatvecPlan& m = c.mv;
  m = MatvecPlan{};
  m.nx = c.nx; m.ny = c.ny; m.nz = c.nz; m.nat = c.nat; m.nat0 = c.nat0;
  m.gx = 2 * c.nx; m.gy = 2 * c.ny; m.gz = 2 * c.nz;
  m.ngrid = (size_t)m.gx * m.gy * m.gz;
  if (!fft_make_plan(m.gx, m.px) || !fft_make_plan(m.gy, m.py) || !fft_make_plan(m.gz, m.pz)) {
    set_error(name, "2*NX, 2*NY, 2*NZ must factor into 2, 3, 5 and 7");
    return 206;
  }
  const int wide = PER_WIDE * MV_THREADS, narrow = PER_NARROW * MV_THREADS;
  if (m.gx > wide || m.gy > wide || m.gz > narrow / 1 || m.gx > narrow) {
    set_error(name, "padded grid axis exceeds the LDS FFT limit (2N <= 2048)");
    return 206;
  }
  const int nrows = c.ny * c.nz;
  const size_t lds_max = lds_limit();
  // rows per workgroup of the LDS-staged x passes: what 256 threads hold at short
  // axes, at long ones 16 (a 128-byte line of a1 per kx) or what 512 threads
  // hold in half the LDS; fewer, but for an element a thread, where that leaves
  // less than 512 workgroups (2,048 of them: 280 x 48 x 48 135 -> 168 us).
  // Where at most 256 remain they take 512 threads too (targets of 4 x 4 to 16 x
  // 16 rows: 5 to 10 % of a MATVEC; with more workgroups it loses as much).
  const auto tiles = [&](int rx) { return (nrows + rx - 1) / rx; };
  int& rx = m.rx;
  rx = PER_NARROW * MV_THREADS / m.gx;
  if (rx < 16) rx = std::min(16, PER_NARROW * ROW_THREADS / m.gx);
  while (rx > 1 && (size_t)m.gx * (1 + (rx | 1)) * sizeof(float2) > lds_max / 2) --rx;
  while (rx > 1 && tiles(rx) < 512 && rx / 2 * m.gx >= MV_THREADS) rx /= 2;
  const bool full = rx * m.gx > PER_NARROW * MV_THREADS, few = tiles(rx) <= 256 && rx * m.gx >= ROW_THREADS;
  m.tx = full || few ? ROW_THREADS : MV_THREADS;
  m.cy = std::min(16, pow2floor(std::max(1, wide / m.gy)));
  // columns of the LDS-staged Green pass: as many as the workgroup has room for
  // (8 values a thread) in 1,024 workgroups or more, but at least 4 columns, an
  // element for every thread, and no thread idle in the last round of them (400 x
  // 10 x 10: 15 columns 75 us, 25 67)
  const auto green_columns = [&](int elements) {
    const int ncol = m.gx * m.gy, least = std::max(4, (MV_THREADS + m.gz - 1) / m.gz);
    const int cz = std::max(1, std::min(elements / m.gz, std::max(least, ncol / 1024)));
    const int rounds = (cz * m.gz + MV_THREADS - 1) / MV_THREADS;
    return std::max(cz, std::min(elements, rounds * MV_THREADS) / m.gz);
  };
  m.cz = green_columns(narrow);
  m.ty = m.tz = MV_THREADS;
  if (m.cy < 8) {
    int cw = std::min(16, pow2floor(std::max(1, PER_WIDE * WIDE_THREADS / m.gy)));
    while (cw > 1 && (size_t)(m.gy + cw * m.gy) * sizeof(float2) > lds_max) cw /= 2;
    if (cw > m.cy) { m.cy = cw; m.ty = WIDE_THREADS; }
  }
  if (m.cz < 8) {
    int cw = green_columns(PER_NARROW * WIDE_THREADS);
    while (cw > 1 && (size_t)(m.gz + 3 * (cw | 1) * m.gz) * sizeof(float2) > lds_max) --cw;
    if (cw > m.cz) { m.cz = cw; m.tz = WIDE_THREADS; }
  }
  if (std::max({m.tx, m.ty, m.tz}) > MV_THREADS && allow_big_lds(lds_max)) return 206;
  if (upload_twiddles(m.gx, &m.twx) || upload_twiddles(m.gy, &m.twy) || upload_twiddles(m.gz, &m.twz)) return 206;
  // z runs start on 128-byte lines; on half lines where whole ones would pad by
  // more than a twentieth (16 right-hand sides of 48 x 50 x 50: 357 us at a pitch of
  // 64, 332 at 56; of 72 x 80 x 120: 1,827 at 128, 1,724 at 120; NZ = 108, which 112
  // pads by 4 %: 350 us, 361 unpadded); on quarter lines where half ones would
  // pad by more than a tenth (8 right-hand sides of 80 x 80 x 36: 314 us at 40, 290
  // at 36, of 80 x 80 x 50: 482 at 56, 460 at 52; but of 80 x 80 x 75, padded by 7 %: 607
  // at 80, 639 at 76) and for targets of few planes
  const auto up = [&](int n) { return (c.nz + n - 1) / n * n; };
  const auto pads = [&](int n, int part) { return part * (up(n) - c.nz) > c.nz; };
  m.nzp = c.nz <= 32 ? up(4) : !pads(16, 20) ? up(16) : !pads(8, 10) ? up(8) : up(4);
  // an odd number of 128-byte lines per kx plane: passes 1 and 5 step through
  // the planes, and an even step hits fewer memory channels (pass 4 at 256^3
  // 505 us with the power of two it has unpadded, 456 so; an odd number of
  // 256-byte blocks 0 to 4 % slower on MATVECs of 16 right-hand sides)
  const auto odd_lines = [](int n) { return ((n + 15) / 16 | 1) * 16; };
  m.p1 = odd_lines(c.ny * m.nzp);
  m.p2 = odd_lines(m.gy * m.nzp);
  return 0;
}

int matvec_setup(Context& c) {
  if (int rc = matvec_plan(c, "MATVEC plan")) return rc;
  DDH_TRY(hipMalloc((void**)&c.a1, matvec_a1_count(c) * sizeof(float2)), "malloc FFT work a1", 204);
  DDH_TRY(hipMalloc((void**)&c.a2, matvec_a2_count(c) * sizeof(float2)), "malloc FFT work a2", 204);
  return 0;
}

size_t matvec_a1_count(const Context& c) { return (size_t)3 * c.mv.gx * c.mv.p1; }
size_t matvec_a2_count(const Context& c) { return (size_t)3 * c.mv.gx * c.mv.p2; }

void matvec_release(Context& c) {
  for (float2** p : {&c.mv.twx, &c.mv.twy, &c.mv.twz, &c.a1, &c.a2}) {
    if (*p) hipFree(*p);
    *p = nullptr;
  }
}

// Pass 5's factor for the kernels in use: 1 / G without the gain of the transforms
// (fft_gain.hpp), in double and then as a float and the rest.
static void matvec_scale(Context& c, int kind5, const KxSlab& sl) {
  MatvecPlan& m = c.mv;
  const FftPlan* staged[6] = {nullptr, &m.px, &m.py, &m.pz, &m.py, &m.px};
  const int lens[6] = {0, m.gx, m.gy, m.gz, m.gy, m.gx}, plane = plane_yz_runs(c);
  int key[6] = {plane};
  for (int p = 1; p <= 5; ++p) key[p] = c.fft_generic ? -1 : p == 5 ? kind5 : m.kind[p];
  if (key[3] >= 0 && !reg_green_reach(c, sl)) key[3] = -1;
  if (std::equal(key, key + 6, m.scale_key)) return;
  const auto gain = [&](int p) { return fft_gain(key[p] >= 0 ? reg_stages(lens[p], p, key[p]) : *staged[p]); };
  double g = 1.0 + 0.5 * (gain(1) + gain(5));
  if (plane) {
    FftPlan y, z;
    plane_yz_stages(c, y, z);
    g *= (1.0 + fft_gain(y)) * (1.0 + fft_gain(z));
  } else {
    g *= (1.0 + 0.5 * (gain(2) + gain(4))) * (1.0 + gain(3));
  }
  const double f = 1.0 / ((double)m.ngrid * g);
  m.scale.x = (float)f;
  m.scale.y = (float)(f - (double)m.scale.x);
  std::copy(key, key + 6, m.scale_key);
}

// One MATVEC pass with kernel choice `kind` (-1: LDS-staged, >= 0: register shape).
static int launch_pass(Context& c, int which, int kind, int cj, int compact, const float2* x, float2* y,
                       const float2* adia, const float2* aoff, hipStream_t st, const MvBatch& bt) {
  const MatvecPlan& m = c.mv;
  const int nrows = c.ny * c.nz;
  const unsigned nb = (unsigned)bt.nrhs;
  float2 *a1 = bt.a1, *a2 = bt.a2;
  const SiteMap sm{c.rowptr, c.rowlo, c.qmap, c.rows_contiguous};
  if (which == 5) matvec_scale(c, kind, bt.slab);
  if (!c.fft_generic && kind >= 0 && reg_pass(c, which, kind, cj, compact, x, y, adia, aoff, st, bt)) return 0;
  switch (which) {
    case 1: {
      const dim3 grid((nrows + m.rx - 1) / m.rx, 3, nb);
      const size_t lds = (size_t)m.gx * (1 + (m.rx | 1)) * sizeof(float2);
      const auto kernel = m.tx == ROW_THREADS ? &k_pass1_xfwd<PER_NARROW, ROW_THREADS> : &k_pass1_xfwd<PER_NARROW>;
      hipLaunchKernelGGL(kernel, grid, dim3(m.tx), lds, st, x, a1, sm, m.twx, m.px, c.nx, c.ny, c.nz, m.nzp, m.p1,
                         m.rx, fast_div_by(c.nx), fast_div_by(c.nz), fast_div_by(m.rx), c.nat, c.nat0, compact,
                         cj, bt.k);
      DDH_LAUNCH_OK("MATVEC pass 1 (x FFT)", 21);
      break;
    }
    case 2:
    case 4: {
      const bool fwd = which == 2, wide = m.ty == WIDE_THREADS;
      // whole tiles per plane, unless that leaves more than a ninth of them idle
      const int whole = (c.nz + m.cy - 1) / m.cy * m.cy, ni = 8 * whole > 9 * c.nz ? c.nz : whole;
      const dim3 grid((unsigned)((2 * bt.slab.H * ni + m.cy - 1) / m.cy), 1, 3 * nb);
      const size_t lds = (size_t)(m.gy + m.cy * m.gy) * sizeof(float2);
      const int lg = ilog2(m.cy);
      const FastDiv dn = fast_div_by(ni);
      if (fwd) {
        const auto kernel = wide ? &k_pass_y<+1, PER_WIDE, WIDE_THREADS> : &k_pass_y<+1, PER_WIDE>;
        hipLaunchKernelGGL(kernel, grid, dim3(m.ty), lds, st, a1, a2, m.twy, m.py, bt.slab, c.ny, m.gy, c.nz, m.nzp, m.p1,
                           m.p2, lg, ni, dn, bt.k);
      } else {
        const auto kernel = wide ? &k_pass_y<-1, PER_WIDE, WIDE_THREADS> : &k_pass_y<-1, PER_WIDE>;
        hipLaunchKernelGGL(kernel, grid, dim3(m.ty), lds, st, a2, a1, m.twy, m.py, bt.slab, m.gy, c.ny, c.nz, m.nzp, m.p2,
                           m.p1, lg, ni, dn, bt.k);
      }
      DDH_LAUNCH_OK("MATVEC y FFT", fwd ? 22 : 24);
      break;
    }
    case 3: {
      dim3 grid((2 * bt.slab.H * m.gy + m.cz - 1) / m.cz, 1, nb);
      const size_t lds = (size_t)(m.gz + 3 * (m.cz | 1) * m.gz) * sizeof(float2);
      const FastDiv dz = fast_div_by(c.nz), dl = fast_div_by(m.gz), dy = fast_div_by(m.gy);
      if (m.tz == WIDE_THREADS)
        hipLaunchKernelGGL((k_pass3_z_green<PER_NARROW, WIDE_THREADS>), grid, dim3(WIDE_THREADS), lds, st, a2,
                           c.green, m.twz, m.pz, c.nz, m.nzp, m.p2, bt.slab, m.gy, m.cz, dz, dl, dy, bt.k, green_geo(c));
      else
        hipLaunchKernelGGL(k_pass3_z_green<PER_NARROW>, grid, dim3(MV_THREADS), lds, st, a2, c.green, m.twz, m.pz,
                           c.nz, m.nzp, m.p2, bt.slab, m.gy, m.cz, dz, dl, dy, bt.k, green_geo(c));
      DDH_LAUNCH_OK("MATVEC pass 3 (z FFT + Green)", 23);
      break;
    }
    default: {
      const dim3 grid((nrows + m.rx - 1) / m.rx, nb);
      size_t lds = (size_t)m.gx * (1 + 3 * (m.rx | 1)) * sizeof(float2);
      const int three = lds <= 64 * 1024 && grid.x * nb <= 256;
      if (!three) lds = (size_t)m.gx * (1 + (m.rx | 1)) * sizeof(float2);
      const auto kernel =
          m.tx == ROW_THREADS ? &k_pass5_xinv_finish<PER_NARROW, ROW_THREADS> : &k_pass5_xinv_finish<PER_NARROW>;
      hipLaunchKernelGGL(kernel, grid, dim3(m.tx), lds, st, a1, m.twx, m.px, x, y, adia, aoff,
                         compact ? nullptr : c.iocc, sm, c.nx, c.ny, c.nz, m.nzp, m.p1, m.rx, fast_div_by(c.nx),
                         fast_div_by(c.nz), fast_div_by(m.rx), three, c.nat, c.nat0, compact, cj, m.scale, bt.k);
      DDH_LAUNCH_OK("MATVEC pass 5 (x inverse FFT + finish)", 25);
      break;
    }
  }
  return 0;
}

void matvec_support(const Context& c, int layout, BatchArgs& k) {
  const MatvecPlan& m = c.mv;
  const bool honoured = !c.fft_generic && !plane_yz_runs(c) && m.kind[1] >= 0 && m.kind[5] >= 0 &&
                        reg_row_support(m.gy, m.kind[2]) && reg_row_support(m.gy, m.kind[4]);
  k.ysup = layout && honoured ? c.ysup : nullptr;
  k.zsh = m.zsh;
}

int matvec_launch(Context& c, int cwhat, const float2* x, float2* y, const float2* adia,
                  const float2* aoff, int layout, hipStream_t st, hipEvent_t* ev, const MvBatch* btp) {
  const int cj = (cwhat == 'C') ? 1 : 0;
  const int compact = layout ? 1 : 0;
  MvBatch bt = btp ? *btp : MvBatch{};
  if (!bt.a1) bt.a1 = c.a1;
  if (!bt.a2) bt.a2 = c.a2;
  matvec_support(c, layout, bt.k);
  bt.slab = KxSlab{0, c.nx, c.mv.gx};
  for (int p = 1; p <= 5; ++p) {
    if (ev) hipEventRecord(ev[p - 1], st);
    if (plane_yz_runs(c) && p >= 2 && p <= 4) {
      if (p != 3) continue;
      if (int rc = plane_yz_launch(c, st, bt)) return rc;
      continue;
    }
    if (int rc = launch_pass(c, p, c.mv.kind[p], cj, compact, x, y, adia, aoff, st, bt)) return rc;
  }
  DDH_LAUNCH_OK("MATVEC register passes", 20);
  if (ev) hipEventRecord(ev[5], st);
  c.matvec_count += (unsigned)bt.nrhs;
  return 0;
}

int matvec_slab(Context& c, hipStream_t st, const MvBatch& bt) {
  for (int p = 2; p <= 4; ++p)
    if (int rc = launch_pass(c, p, c.mv.kind[p], 0, 0, nullptr, nullptr, nullptr, nullptr, st, bt)) return rc;
  return 0;
}

int matvec_end_pass(Context& c, int which, int cwhat, const float2* x, float2* y, const float2* adia,
                    const float2* aoff, int layout, hipStream_t st, const MvBatch& bt) {
  return launch_pass(c, which, c.mv.kind[which], cwhat == 'C' ? 1 : 0, layout ? 1 : 0, x, y, adia, aoff, st, bt);
}

// Autotuner: a pass whose axis length has several register shapes runs each a
// few times on the prepared grid (compact vectors, stream events); the fastest
// is kept in c.mv.kind.  A pass with one shape takes it, a pass without one the
// LDS-staged kernel (slower wherever there is a shape).  Choices are cached per
// grid for the life of the process, so re-preparing the same grid (for instance
// every target orientation of a DDSCAT run) does not re-time.
namespace {
struct TuneKey {
  int nx, ny, nz, ipbc;  // IPBC=1 reads the whole-grid Green in pass 3, not the octant
  bool operator<(const TuneKey& o) const {
    return nx != o.nx ? nx < o.nx : ny != o.ny ? ny < o.ny : nz != o.nz ? nz < o.nz : ipbc < o.ipbc;
  }
};
std::map<TuneKey, std::array<int, 6>>& tune_cache() {
  static std::map<TuneKey, std::array<int, 6>> m;
  return m;
}
}  // namespace

int matvec_autotune(Context& c) {
  MatvecPlan& m = c.mv;
  const int lens[6] = {0, m.gx, m.gy, m.gz, m.gy, m.gx};
  for (int p = 1; p <= 5; ++p) m.kind[p] = reg_candidates(lens[p], p) > 0 ? 0 : -1;
  m.tuned = 0;
  if (int rc = plane_yz_setup(c)) return rc;
  if (!c.autotune || c.fft_generic || !c.sx || !c.sy || !c.adia_c || !c.aoff_c) return 0;
  const TuneKey key{c.nx, c.ny, c.nz, c.ipbc};
  auto it = tune_cache().find(key);
  if (it != tune_cache().end()) {
    for (int p = 1; p <= 5; ++p) m.kind[p] = it->second[p];
    m.tuned = 1;
    return 0;
  }
  hipStream_t st = c.stream;
  const size_t cb = (size_t)3 * c.nat0 * sizeof(float2);
  DDH_TRY(hipMemsetAsync(c.sx, 0, cb, st), "autotune", 20);
  DDH_TRY(hipMemsetAsync(c.adia_c, 0, cb, st), "autotune", 20);
  DDH_TRY(hipMemsetAsync(c.aoff_c, 0, cb, st), "autotune", 20);
  hipEvent_t e0, e1;
  DDH_TRY(hipEventCreate(&e0), "autotune", 20);
  if (hipEventCreate(&e1) != hipSuccess) { hipEventDestroy(e0); set_error("autotune", "event"); return 20; }
  MvBatch bt;
  bt.a1 = c.a1;
  bt.a2 = c.a2;
  bt.slab = KxSlab{0, c.nx, m.gx};
  if (c.backend == BACKEND_SLICES) slices_slab(c, 0, bt);
  int rc = 0;
  for (int p = 1; p <= 5 && !rc; ++p) {
    const int ncand = reg_candidates(lens[p], p);
    if (ncand < 2) continue;
    float best = 1e30f;
    int best_kind = m.kind[p];
    for (int k = 0; k < ncand && !rc; ++k) {
      for (int w = 0; w < 2 && !rc; ++w) rc = launch_pass(c, p, k, 0, 1, c.sx, c.sy, c.adia_c, c.aoff_c, st, bt);
      hipEventRecord(e0, st);
      for (int r = 0; r < 5 && !rc; ++r) rc = launch_pass(c, p, k, 0, 1, c.sx, c.sy, c.adia_c, c.aoff_c, st, bt);
      hipEventRecord(e1, st);
      if (rc || hipEventSynchronize(e1) != hipSuccess) { rc = rc ? rc : 20; break; }
      float ms = 0.f;
      hipEventElapsedTime(&ms, e0, e1);
      if (ms < best) { best = ms; best_kind = k; }
    }
    m.kind[p] = best_kind;
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (rc) return rc;
  std::array<int, 6> k6;
  for (int p = 0; p < 6; ++p) k6[p] = m.kind[p];
  tune_cache()[key] = k6;
  m.tuned = 1;
  return 0;
}

}  // namespace ddhip
