// Wave-private register Stockham FFTs for gfx950.
//
// One wavefront transforms one or more sequences of length L = R0 R1 (R2 (R3))
// by itself: T lanes per sequence, 64 / T sequences per wave, no workgroup
// barrier anywhere, so the waves of a CU drift apart and one wave's loads and
// stores run under another's butterflies.  Stage s of radix R and span
// P = R0 ... R_{s-1}: butterfly i (i < L / R) of lane j (i = j + T b) gathers
// u_r = d[i + r L / R], multiplies by w_{PR}^{r (i mod P)}, does the R-point
// DFT and scatters y_r to (i - i mod P) R + i mod P + r P; after the last
// stage d is in natural order.  Stages exchange through LDS slots private to
// the wave: LDS instructions of one wave execute in order, so only the
// compiler has to be kept from moving them (wave_sync).  The inverse runs the
// transposed stages backwards, from the forward's output distribution to its
// input distribution.
// A stage's butterflies need be no multiple of T, so L is not tied to powers of
// two.
#pragma once
#include "fft_reg.hpp"

namespace ddhip {

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int T_, int R0, int R1, int R2 = 1, int R3 = 1>
struct WPlan {
  static constexpr int L = R0 * R1 * R2 * R3, T = T_, S = R3 > 1 ? 4 : R2 > 1 ? 3 : 2;
  static constexpr int rad(int s) { return s == 0 ? R0 : s == 1 ? R1 : s == 2 ? R2 : R3; }
  static constexpr int span(int s) { return s == 0 ? 1 : span(s - 1) * rad(s - 1); }
  static constexpr int nbf(int s) { return L / rad(s); }           // butterflies of stage s
  static constexpr int nb(int s) { return (nbf(s) + T - 1) / T; }  // and per lane
  static constexpr int vals(int s) { return s == S ? 0 : nb(s) * rad(s) > vals(s + 1) ? nb(s) * rad(s) : vals(s + 1); }
  static constexpr int V = vals(0);            // register values per lane
  static constexpr int SEQ = 64 / T;           // sequences per wave
  static constexpr int PAD = R0 % 2 == 0 ? R0 : 0;  // one padding slot per R0 points when R0 is even
  static constexpr int SLOTS = PAD ? L + L / R0 : L;  // LDS slots of one sequence
  static_assert(T <= 64 && nb(0) >= 1, "a sequence sits in one wave");
};
template <class PL>
FftPlan w_stages() {
  FftPlan p{PL::L, PL::S, {}};
  for (int s = 0; s < PL::S; ++s) p.rad[s] = PL::rad(s);
  return p;
}
// LDS slot of point idx: one slot of padding per R0 points, so the stride-R0
// scatter of stage 0 (odd stride after padding) and the unit-stride gathers
// both spread over the banks
template <class PL>
__device__ __forceinline__ constexpr int w_slot(int idx) {
  return PL::PAD ? idx + idx / (PL::PAD ? PL::PAD : 1) : idx;
}
// Butterfly b of lane j in stage s.  Where the stage's butterflies are no
// multiple of T, the lanes past the last one repeat it: they gather, compute
// and write what its own lane does, which costs nothing and keeps the code
// free of branches (guarded writes split it into blocks across which the
// compiler hoisted loads: 222 instead of 150 registers at 54 points).
template <class PL, int s>
__device__ __forceinline__ int w_bfly(int j, int b) {
  const int i = j + PL::T * b;
  return PL::nbf(s) % PL::T == 0 || PL::T * (b + 1) <= PL::nbf(s) ? i : min(i, PL::nbf(s) - 1);
}
// LDS pointer of the scatter position r = 0 of butterfly i of stage s; the
// others follow at compile-time distances (the padding is constant over
// multiples of R0, and within one run of R0 points in stage 0)
template <class PL, int s>
__device__ __forceinline__ float2* w_scatter_at(float2* xb, int i) {
  constexpr int R = PL::rad(s), P = PL::span(s);
  const int k = i % P;
  return xb + w_slot<PL>((i - k) * R + k);
}
template <class PL, int s>
__device__ __forceinline__ constexpr int w_scatter_step(int r) {
  return s == 0 ? r : w_slot<PL>(r * PL::span(s));
}
// and of the gather positions of stage s >= 1 (L / R is a multiple of R0)
template <class PL, int s>
__device__ __forceinline__ constexpr int w_gather_step(int r) {
  return w_slot<PL>(r * (PL::L / PL::rad(s)));
}
template <class PL, int s>
__device__ __forceinline__ void w_scatter(const float2* v, float2* __restrict__ xb, int j) {
#pragma unroll
  for (int b = 0; b < PL::nb(s); ++b) {
    float2* p = w_scatter_at<PL, s>(xb, w_bfly<PL, s>(j, b));
#pragma unroll
    for (int r = 0; r < PL::rad(s); ++r) p[w_scatter_step<PL, s>(r)] = v[b * PL::rad(s) + r];
  }
}
template <class PL, int s>
__device__ __forceinline__ void w_scatter_read(float2* v, float2* __restrict__ xb, int j) {
#pragma unroll
  for (int b = 0; b < PL::nb(s); ++b) {
    const float2* p = w_scatter_at<PL, s>(xb, w_bfly<PL, s>(j, b));
#pragma unroll
    for (int r = 0; r < PL::rad(s); ++r) v[b * PL::rad(s) + r] = p[w_scatter_step<PL, s>(r)];
  }
}
template <class PL, int s>
__device__ __forceinline__ void w_gather(float2* v, const float2* __restrict__ xb, int j) {
#pragma unroll
  for (int b = 0; b < PL::nb(s); ++b) {
    const float2* p = xb + w_slot<PL>(w_bfly<PL, s>(j, b));
#pragma unroll
    for (int r = 0; r < PL::rad(s); ++r) v[b * PL::rad(s) + r] = p[w_gather_step<PL, s>(r)];
  }
}
template <class PL, int s>
__device__ __forceinline__ void w_gather_write(const float2* v, float2* __restrict__ xb, int j) {
#pragma unroll
  for (int b = 0; b < PL::nb(s); ++b) {
    float2* p = xb + w_slot<PL>(w_bfly<PL, s>(j, b));
#pragma unroll
    for (int r = 0; r < PL::rad(s); ++r) p[w_gather_step<PL, s>(r)] = v[b * PL::rad(s) + r];
  }
}
// twiddle w_{PR}^{r (i mod P)} of stage s from the length-L table
template <class PL, int s, int DIR>
__device__ __forceinline__ void w_twiddle(float2* v, const float2* __restrict__ tw, int j) {
  constexpr int R = PL::rad(s), P = PL::span(s), NB = PL::nb(s), TS = PL::L / (P * R);
  if constexpr (P > 1) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int k = w_bfly<PL, s>(j, b) % P;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        float2 w = tw[r * k * TS];
        if (DIR < 0) w.y = -w.y;
        v[b * R + r] = cmul(v[b * R + r], w);
      }
    }
  }
}
template <class PL, int s, int DIR>
__device__ __forceinline__ void w_dft(float2* v) {
#pragma unroll
  for (int b = 0; b < PL::nb(s); ++b) dft_reg<PL::rad(s), DIR>(v + b * PL::rad(s));
}
// forward: v[b R0 + r] = x[j + T b + r L / R0] in, v[b R + r] = X[j + T b + r L / R] out (R the last radix)
template <class PL, int DIR, int s = 0>
__device__ __forceinline__ void w_forward(float2* v, float2* __restrict__ xb, const float2* __restrict__ tw, int j) {
  w_twiddle<PL, s, DIR>(v, tw, j);
  w_dft<PL, s, DIR>(v);
  if constexpr (s + 1 < PL::S) {
    wave_sync();
    w_scatter<PL, s>(v, xb, j);
    wave_sync();
    w_gather<PL, s + 1>(v, xb, j);
    w_forward<PL, DIR, s + 1>(v, xb, tw, j);
  }
}
// inverse (sign DIR): the forward's output distribution in, its input distribution out
template <class PL, int DIR, int s = PL::S - 1>
__device__ __forceinline__ void w_inverse(float2* v, float2* __restrict__ xb, const float2* __restrict__ tw, int j) {
  w_dft<PL, s, DIR>(v);
  w_twiddle<PL, s, DIR>(v, tw, j);
  if constexpr (s > 0) {
    wave_sync();
    w_gather_write<PL, s>(v, xb, j);
    wave_sync();
    w_scatter_read<PL, s - 1>(v, xb, j);
    w_inverse<PL, DIR, s - 1>(v, xb, tw, j);
  }
}

}  // namespace ddhip
