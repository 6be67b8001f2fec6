// Passes 2 to 4 in one kernel for kx planes that fit LDS: y-FFT, z-FFT, Green
// multiply, inverse z-FFT and inverse y-FFT of a plane of a1, in place.
//
// A workgroup holds the plane's 2NY padded z columns as pl[row][3][NZ] (pitch
// cp).  The y transforms are two-level, 2NY = R2 R1: level 1 does R2-point
// DFTs of the NY inputs of one y column (pruned: R2 is even) and leaves
// twiddled results in rows k2 R1 + n1, level 2 does the R1-point DFTs of rows
// k2 R1 ... in place, so row k2 R1 + k1 ends with ky = k2 + R2 k1 and neither
// level needs registers across a barrier; lanes run over z.  The z columns
// then go through p3_transform by single wavefronts, a column's own 3 NZ slots
// serving as its exchange buffer once its values are in registers.  Four
// barriers per plane, and nothing of a2 crosses memory.
//
// What bounds it: a plane sits on one CU, where VALU issue of the z columns is
// two thirds of the time (32^3, one right-hand side: 1.3 + 0.9 us the y levels,
// 4.5 the columns, 1.5 the inverse levels); a small cube has fewer planes than
// CUs, so the time is one plane's.  Against passes 2, 3
// and 4 as kernels of their own, whole MATVECs:
//   16^3 20.7 -> 16.3 us, 32^3 23.0 -> 20.5, 45^3 41 -> 35;
//   32 right-hand sides: 32^3 129 -> 110 us, 36^3 259 -> 174, 54^3 878 -> 632.
#pragma once
#include "pass3_wave.hpp"

namespace ddhip {

struct YzGeo {
  int R1, R2;        // 2NY = R2 (level 1) R1 (level 2)
  int cp;            // LDS pitch of a row
  unsigned mz, m1;   // x / NZ = x mz >> 18, x / R1 = x m1 >> 18 (x < 2^12)
  int ny, nz, nzp, p1, gx;
  int nrhs;
};
__device__ __forceinline__ int yz_div(int x, unsigned magic) { return (int)(((unsigned)x * magic) >> 18); }

// item -> (component, outer index, z) of 3 n nz items, z fastest
__device__ __forceinline__ void yz_item(const YzGeo& q, int it, int n, int& c, int& o, int& z) {
  const int per = n * q.nz;
  c = (it >= per) + (it >= 2 * per);
  const int r = it - c * per;
  o = yz_div(r, q.mz);
  z = r - o * q.nz;
}
template <int R>
__device__ __forceinline__ void yz_fwd1(const YzGeo& q, const float2* src, size_t cs, float2* pl, const float2* tw) {
  for (int it = threadIdx.x; it < 3 * q.R1 * q.nz; it += blockDim.x) {
    int c, t, z;
    yz_item(q, it, q.R1, c, t, z);
    const float2* p = src + c * cs + z;
    float2 v[R];
#pragma unroll
    for (int n2 = 0; n2 < R; ++n2) v[n2] = 2 * n2 < R ? p[(t + q.R1 * n2) * q.nzp] : make_float2(0.f, 0.f);
    dft_reg<R, +1>(v);
    float2* o = pl + t * q.cp + c * q.nz + z;
    o[0] = v[0];
#pragma unroll
    for (int k2 = 1; k2 < R; ++k2) o[k2 * q.R1 * q.cp] = cmul(v[k2], tw[t * k2]);
  }
}
template <int R>
__device__ __forceinline__ void yz_fwd2(const YzGeo& q, float2* pl) {
  for (int it = threadIdx.x; it < 3 * q.R2 * q.nz; it += blockDim.x) {
    int c, k2, z;
    yz_item(q, it, q.R2, c, k2, z);
    float2* o = pl + k2 * R * q.cp + c * q.nz + z;
    float2 v[R];
#pragma unroll
    for (int n1 = 0; n1 < R; ++n1) v[n1] = o[n1 * q.cp];
    dft_reg<R, +1>(v);
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) o[k1 * q.cp] = v[k1];
  }
}
template <int R>
__device__ __forceinline__ void yz_inv2(const YzGeo& q, float2* pl, const float2* tw) {
  for (int it = threadIdx.x; it < 3 * q.R2 * q.nz; it += blockDim.x) {
    int c, k2, z;
    yz_item(q, it, q.R2, c, k2, z);
    float2* o = pl + k2 * R * q.cp + c * q.nz + z;
    float2 v[R];
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) v[k1] = o[k1 * q.cp];
    dft_reg<R, -1>(v);
    o[0] = v[0];
#pragma unroll
    for (int n1 = 1; n1 < R; ++n1) {
      const float2 w = tw[n1 * k2];
      o[n1 * q.cp] = cmul(v[n1], make_float2(w.x, -w.y));
    }
  }
}
template <int R>
__device__ __forceinline__ void yz_inv1(const YzGeo& q, const float2* pl, float2* dst, size_t cs) {
  for (int it = threadIdx.x; it < 3 * q.R1 * q.nz; it += blockDim.x) {
    int c, t, z;
    yz_item(q, it, q.R1, c, t, z);
    const float2* o = pl + t * q.cp + c * q.nz + z;
    float2 v[R];
#pragma unroll
    for (int k2 = 0; k2 < R; ++k2) v[k2] = o[k2 * q.R1 * q.cp];
    dft_reg<R, -1>(v);
    float2* p = dst + c * cs + z;
#pragma unroll
    for (int n2 = 0; 2 * n2 < R; ++n2) p[(t + q.R1 * n2) * q.nzp] = v[n2];
  }
}
// the radices of yz_split: level 1 even (its inputs' zero half is a compile-time set)
#define YZ_LEVEL1(fn, ...)                        \
  switch (q.R2) {                                 \
    case 4: fn<4>(__VA_ARGS__); break;            \
    case 6: fn<6>(__VA_ARGS__); break;            \
    case 8: fn<8>(__VA_ARGS__); break;            \
    case 10: fn<10>(__VA_ARGS__); break;          \
    case 12: fn<12>(__VA_ARGS__); break;          \
    default: fn<14>(__VA_ARGS__); break;          \
  }
#define YZ_LEVEL2(fn, ...)                        \
  switch (q.R1) {                                 \
    case 4: fn<4>(__VA_ARGS__); break;            \
    case 5: fn<5>(__VA_ARGS__); break;            \
    case 6: fn<6>(__VA_ARGS__); break;            \
    case 7: fn<7>(__VA_ARGS__); break;            \
    case 8: fn<8>(__VA_ARGS__); break;            \
    case 9: fn<9>(__VA_ARGS__); break;            \
    default: fn<10>(__VA_ARGS__); break;          \
  }

constexpr int YZ_MAX_THREADS = 1024;
template <class PL, bool MIRROR>
__global__ __launch_bounds__(YZ_MAX_THREADS) void kw_plane_yz(float2* __restrict__ a1, const float2* __restrict__ green,
                                                              const float2* __restrict__ twyg,
                                                              const float2* __restrict__ twzg, BatchArgs ba, GreenGeo gg,
                                                              YzGeo q) {
  constexpr int L = PL::L, T = PL::T, V = PL::V, SEQ = PL::SEQ, R0 = PL::rad(0);
  extern __shared__ float2 sm[];
  const int gy = 2 * q.ny;
  float2 *pl = sm, *twy = sm + gy * q.cp, *twz = twy + gy;
  // workgroups go round-robin over the 8 XCDs: the right-hand sides and the
  // mirror of a plane, which read the same Green entries, 8 ids apart
  const int sq = (int)blockIdx.x >> 3, per = 2 * q.nrhs, grp = sq / per, rem = sq - grp * per;
  const int half = grp * 8 + ((int)blockIdx.x & 7), mir = rem / q.nrhs, rb = rem - mir * q.nrhs;
  if (half >= q.gx / 2 || (ba.active && !ba.active[rb])) return;
  const int kx = mir ? (half == 0 ? q.gx / 2 : q.gx - half) : half;
  float2* const plane = a1 + rb * ba.a1s + (size_t)kx * q.p1;
  const size_t cs = (size_t)q.gx * q.p1;
  for (int i = threadIdx.x; i < gy; i += blockDim.x) twy[i] = twyg[i];
  for (int i = threadIdx.x; i < L; i += blockDim.x) twz[i] = twzg[i];
  __syncthreads();
  YZ_LEVEL1(yz_fwd1, q, plane, cs, pl, twy)
  __syncthreads();
  YZ_LEVEL2(yz_fwd2, q, pl)
  __syncthreads();
  {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6, seq = lane / T, j = lane - seq * T;
    const int ir = min(kx, gg.mx - kx);
    const float sx = kx <= gg.tx ? 1.f : -1.f;
    if (seq < SEQ)
      for (int row = w * SEQ + seq; row < gy; row += nw * SEQ) {
        float2* const col = pl + row * q.cp;
        const int k2 = yz_div(row, q.m1), ky = k2 + q.R2 * (row - k2 * q.R1);
        const int jr = min(ky, gg.my - ky);
        const float sy = ky <= gg.ty ? 1.f : -1.f;
        float2 v[3][V];
#pragma unroll
        for (int b = 0; b < PL::nb(0); ++b) {
          const int i = w_bfly<PL, 0>(j, b);
#pragma unroll
          for (int r = 0; r < R0; ++r) {
            const int e = b * R0 + r;
            if (2 * r < R0) {
              v[0][e] = cscale(col[i + r * (L / R0)], sx);
              v[1][e] = cscale(col[L / 2 + i + r * (L / R0)], sy);
              v[2][e] = col[L + i + r * (L / R0)];
            } else {
              v[0][e] = v[1][e] = v[2][e] = make_float2(0.f, 0.f);
            }
          }
        }
        wave_sync();
        p3_transform<PL, MIRROR>(v, col, twz, j, reinterpret_cast<const char*>(green),
                                 ((unsigned)ir * (unsigned)gg.oy + (unsigned)jr) * (unsigned)gg.oz * 48u);
        wave_sync();
#pragma unroll
        for (int b = 0; b < PL::nb(0); ++b) {
          const int i = w_bfly<PL, 0>(j, b);
#pragma unroll
          for (int r = 0; 2 * r < R0; ++r) {
            const int e = b * R0 + r;
            col[i + r * (L / R0)] = cscale(v[0][e], sx);
            col[L / 2 + i + r * (L / R0)] = cscale(v[1][e], sy);
            col[L + i + r * (L / R0)] = v[2][e];
          }
        }
      }
  }
  __syncthreads();
  YZ_LEVEL2(yz_inv2, q, pl, twy)
  __syncthreads();
  YZ_LEVEL1(yz_inv1, q, pl, plane, cs)
}

// LDS pitch of a row for a z plan: its three components, at least one
// exchange buffer, and such that the columns of a wave start T slots apart in the banks
template <class PL>
int yz_pitch() {
  int cp = 3 * (PL::L / 2);
  if (cp < PL::SLOTS) cp = PL::SLOTS;
  while (cp % 32 != PL::T % 32) ++cp;
  return cp;
}
struct YzShape {
  int L, seq;     // padded z axis, columns per wave
  int (*pitch)();
  FftPlan (*stages)();
  const void* (*kernel)(bool mirror);
};
template <class PL>
const void* yz_kernel(bool mirror) {
  return mirror ? reinterpret_cast<const void*>(&kw_plane_yz<PL, true>)
                : reinterpret_cast<const void*>(&kw_plane_yz<PL, false>);
}
#define YZ_PLAN(...) YzShape{WPlan<__VA_ARGS__>::L, WPlan<__VA_ARGS__>::SEQ, &yz_pitch<WPlan<__VA_ARGS__>>, &w_stages<WPlan<__VA_ARGS__>>, \
  &yz_kernel<WPlan<__VA_ARGS__>>}
const YzShape* yz_shapes(int& n);

}  // namespace ddhip
