// Register-resident two-level FFTs for gfx950.
//
// A length L = R1 * R2 transform of one sequence is shared by R1 threads.
// With n = n1 + R1 n2 and k = k2 + R2 k1,
//   X[k2 + R2 k1] = sum_n1 W_R1^{n1 k1} W_L^{n1 k2} sum_n2 x[n1 + R1 n2] W_R2^{n2 k2}.
// Forward: thread n1 holds x[n1 + R1 n2] (n2 < R2) in registers, does the
// R2-point DFT, multiplies by W_L^{n1 k2}, writes to LDS; after one barrier
// thread t holds, for each owned k2 = t + R1 i (i < R2/R1), the R1 values
// n1 and does the R1-point DFT, ending with X[k2 + R2 k1] in registers.
// Inverse runs the same two steps backwards from that distribution and ends
// with y[n1 + R1 n2] on thread n1.  One LDS exchange per transform; the
// R-point DFTs are fully unrolled with compile-time twiddles.
#pragma once
#include "common.hpp"
#include "fft_device.hpp"

namespace ddhip {

// cos(2 pi m / 32), m any integer
__host__ __device__ constexpr float cos32(int m) {
  constexpr float C[9] = {1.0f,
                          0.98078528040323044913f,
                          0.92387953251128675613f,
                          0.83146961230254523708f,
                          0.70710678118654752440f,
                          0.55557023301960222474f,
                          0.38268343236508977173f,
                          0.19509032201612826785f,
                          0.0f};
  m &= 31;
  return m <= 8 ? C[m] : m <= 16 ? -C[16 - m] : m <= 24 ? -C[m - 16] : C[32 - m];
}
__host__ __device__ constexpr float sin32(int m) { return cos32(m - 8); }

// cos / sin of 2 pi m / N for any N, evaluated at compile time: the angle is
// reduced to [-pi/4, pi/4] by octant and expanded in Taylor series to double
// precision, so a table entry is exact to float rounding.
constexpr double kTwoPi = 6.283185307179586476925286766559;
constexpr double taylor_sin(double x) {
  double t = x, s = x;
  for (int k = 1; k < 12; ++k) {
    t *= -x * x / ((2.0 * k) * (2.0 * k + 1.0));
    s += t;
  }
  return s;
}
constexpr double taylor_cos(double x) {
  double t = 1.0, s = 1.0;
  for (int k = 1; k < 12; ++k) {
    t *= -x * x / ((2.0 * k - 1.0) * (2.0 * k));
    s += t;
  }
  return s;
}
// (cos, sin) of 2 pi m / N via the octant o = round(8 m / N) and r = 2 pi m / N - o pi / 4
constexpr double cos_frac(long m, long N, bool want_sin) {
  m %= N;
  if (m < 0) m += N;
  const long o = (8 * m + N / 2) / N;  // nearest eighth of a turn
  const double r = kTwoPi * ((double)m / (double)N) - (double)o * (kTwoPi / 8.0);
  const double c = taylor_cos(r), s = taylor_sin(r);
  const double h = 0.70710678118654752440;
  // rotate (c, s) by o * 45 degrees
  double cr = c, sr = s;
  switch (o & 7) {
    case 0: cr = c; sr = s; break;
    case 1: cr = h * (c - s); sr = h * (c + s); break;
    case 2: cr = -s; sr = c; break;
    case 3: cr = -h * (c + s); sr = h * (c - s); break;
    case 4: cr = -c; sr = -s; break;
    case 5: cr = h * (s - c); sr = -h * (c + s); break;
    case 6: cr = s; sr = -c; break;
    default: cr = h * (c + s); sr = h * (s - c); break;
  }
  return want_sin ? sr : cr;
}
template <int N>
struct TwTable {
  float c[N], s[N];
  constexpr TwTable() : c(), s() {
    for (int m = 0; m < N; ++m) {
      c[m] = (float)cos_frac(m, N, false);
      s[m] = (float)cos_frac(m, N, true);
    }
  }
};
template <int N>
struct Tw {
  static constexpr TwTable<N> t{};
};

// multiply by e^{DIR 2 pi i m / N}, m compile-time after unrolling
template <int N, int DIR>
__device__ __forceinline__ float2 twc(float2 a, int m) {
  float c, s;
  if constexpr (32 % N == 0) {
    const int q = m * (32 / N);
    c = cos32(q);
    s = DIR * sin32(q);
  } else {
    const int q = m % N;
    c = Tw<N>::t.c[q];
    s = DIR * Tw<N>::t.s[q];
  }
  return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
}

template <int R, int DIR>
__device__ __forceinline__ void dft_reg(float2* a);

// N = P * Q composition: n = n1 + P n2, k = k2 + Q k1
template <int P, int Q, int DIR>
__device__ __forceinline__ void dft_comp(float2* a) {
  constexpr int N = P * Q;
  float2 b[N];
#pragma unroll
  for (int n1 = 0; n1 < P; ++n1) {
    float2 t[Q];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) t[n2] = a[n1 + P * n2];
    dft_reg<Q, DIR>(t);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) b[n1 * Q + k2] = (n1 * k2 == 0) ? t[k2] : twc<N, DIR>(t[k2], n1 * k2);
  }
#pragma unroll
  for (int k2 = 0; k2 < Q; ++k2) {
    float2 t[P];
#pragma unroll
    for (int n1 = 0; n1 < P; ++n1) t[n1] = b[n1 * Q + k2];
    dft_reg<P, DIR>(t);
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) a[k2 + Q * k1] = t[k1];
  }
}

template <int R, int DIR>
__device__ __forceinline__ void dft_reg(float2* a) {
  if constexpr (R == 1) {
  } else if constexpr (R == 2) {
    dft2<DIR>(a);
  } else if constexpr (R == 4) {
    dft4<DIR>(a);
  } else if constexpr (R == 8) {
    dft8<DIR>(a);
  } else if constexpr (R == 3) {
    dft3<DIR>(a);
  } else if constexpr (R == 5) {
    dft5<DIR>(a);
  } else if constexpr (R == 7) {
    dft7<DIR>(a);
  } else if constexpr (R == 16) {
    dft_comp<4, 4, DIR>(a);
  } else if constexpr (R == 32) {
    dft_comp<4, 8, DIR>(a);
  } else if constexpr (R % 8 == 0 && R > 8) {
    dft_comp<R / 8, 8, DIR>(a);
  } else if constexpr (R % 4 == 0 && R > 4) {
    dft_comp<R / 4, 4, DIR>(a);
  } else if constexpr (R % 5 == 0 && R > 5) {
    dft_comp<R / 5, 5, DIR>(a);
  } else if constexpr (R % 3 == 0 && R > 3) {
    dft_comp<R / 3, 3, DIR>(a);
  } else if constexpr (R % 2 == 0 && R > 2) {
    dft_comp<R / 2, 2, DIR>(a);
  } else {
    static_assert(R == 1, "unsupported register DFT size");
  }
}

// Work split of a length L = R1 * R2 transform over R1 threads.  The first
// step is one R2-point DFT per thread; the second step's R2 DFTs of length R1
// go round-robin to the threads: thread t owns k2 = t + R1 i for i < G while
// k2 < R2 (all of them when R1 divides R2).  A thread's register array holds
// VN values.  LDS exchange layout for C sequences: element (row, s) at
// row * P + s, row = k2 * R1 + n1, P = C + 1 (pad against bank conflicts).
template <int R1, int R2>
struct Reg2 {
  static constexpr int L = R1 * R2;
  static constexpr int G = (R2 + R1 - 1) / R1;
  static constexpr int VN = R2 > G * R1 ? R2 : G * R1;
};
// Tile of block bx of n.  Blocks go round-robin over the 8 XCDs by linear id, and
// each XCD has its own L2: the blocks of one XCD (ids 8 apart) take a run of
// neighbours, so that tiles which share a 128-byte line share it there.
__device__ __forceinline__ int xcd_run(int bx, int n) {
  const int x = bx & 7, q = n >> 3, rem = n & 7;
  return x * q + min(x, rem) + (bx >> 3);
}

// The padded axes have length L = R1 R2 = 2N with data (forward input) and
// kept results (inverse output) in n < N.  Element n = t + R1 n2 of thread t
// (t < R1) lies below N for every t when 2 n2 + 1 < R2 and above it when
// 2 n2 + 1 > R2; only the middle element of an odd R2 depends on t.  With
// the test in this form the zero half of a forward input is a compile-time
// constant (its butterflies fold away) and the discarded half of an inverse
// output is never computed.
template <int R2>
__device__ __forceinline__ bool lower_half(int n2, int n, int N) {
  return (2 * n2 + 1 < R2) || (2 * n2 + 1 == R2 && n < N);
}
template <int R1, int R2>
__device__ __forceinline__ bool reg2_owns(int t, int i) {
  return Reg2<R1, R2>::G * R1 == R2 || t + R1 * i < R2;
}

// LDS exchange index of element (k2, n1) of sequence s: lanes run over s, P = C + 1
template <int R1>
__device__ __forceinline__ int lidx(int k2, int n1, int s, int P) {
  return (k2 * R1 + n1) * P + s;
}

// forward: v[n2] = x[t + R1 n2] (n2 < R2) in; v[i R1 + k1] = X[(t + R1 i) + R2 k1]
// out for the groups i the thread owns
template <int R1, int R2, int DIR>
__device__ __forceinline__ void fft2_fwd(float2* v, float2* __restrict__ lds, const float2* __restrict__ twL, int t,
                                         int s, int P) {
  dft_reg<R2, DIR>(v);
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) {
    float2 w = twL[t * k2];
    if (DIR < 0) w.y = -w.y;
    lds[lidx<R1>(k2, t, s, P)] = k2 == 0 ? v[0] : cmul(v[k2], w);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < Reg2<R1, R2>::G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
    const int k2 = t + R1 * i;
    float2 u[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) u[n1] = lds[lidx<R1>(k2, n1, s, P)];
    dft_reg<R1, DIR>(u);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) v[i * R1 + k1] = u[k1];
  }
}

// inverse of the forward distribution: v[i R1 + k1] = Y[(t + R1 i) + R2 k1] in
// (owned groups), v[n2] = y[t + R1 n2] out (direction DIR, normally -1)
template <int R1, int R2, int DIR>
__device__ __forceinline__ void fft2_inv(float2* v, float2* __restrict__ lds, const float2* __restrict__ twL, int t,
                                         int s, int P) {
#pragma unroll
  for (int i = 0; i < Reg2<R1, R2>::G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
    const int k2 = t + R1 * i;
    float2 u[R1];
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) u[k1] = v[i * R1 + k1];
    dft_reg<R1, DIR>(u);
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      float2 w = twL[n1 * k2];
      if (DIR < 0) w.y = -w.y;
      lds[lidx<R1>(k2, n1, s, P)] = n1 == 0 ? u[0] : cmul(u[n1], w);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) v[k2] = lds[lidx<R1>(k2, t, s, P)];
  dft_reg<R2, DIR>(v);
}

// Split-exchange form of fft2_fwd: the real and the imaginary parts cross
// LDS in turn, so the exchange buffer holds L*P floats instead of L*P
// float2.  Half the LDS per workgroup doubles the workgroups a CU can hold
// for kernels whose occupancy LDS limits (pass 1); two more barriers.
template <int R1, int R2, int DIR>
__device__ __forceinline__ void fft2_fwd_s(float2* v, float* __restrict__ lds, const float2* __restrict__ twL, int t,
                                           int s, int P) {
  constexpr int G = Reg2<R1, R2>::G;
  dft_reg<R2, DIR>(v);
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) {
    float2 w = twL[t * k2];
    if (DIR < 0) w.y = -w.y;
    v[k2] = cmul(v[k2], w);
  }
  float re[G * R1];
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) lds[lidx<R1>(k2, t, s, P)] = v[k2].x;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) re[i * R1 + n1] = lds[lidx<R1>(t + R1 * i, n1, s, P)];
  }
  __syncthreads();
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) lds[lidx<R1>(k2, t, s, P)] = v[k2].y;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
    float2 u[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) u[n1] = make_float2(re[i * R1 + n1], lds[lidx<R1>(t + R1 * i, n1, s, P)]);
    dft_reg<R1, DIR>(u);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) v[i * R1 + k1] = u[k1];
  }
}

// Split-exchange form of fft2_inv (real and imaginary parts cross LDS in turn).
template <int R1, int R2, int DIR>
__device__ __forceinline__ void fft2_inv_s(float2* v, float* __restrict__ lds, const float2* __restrict__ twL, int t,
                                           int s, int P) {
  constexpr int G = Reg2<R1, R2>::G;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
    const int k2 = t + R1 * i;
    float2 u[R1];
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) u[k1] = v[i * R1 + k1];
    dft_reg<R1, DIR>(u);
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      float2 w = twL[n1 * k2];
      if (DIR < 0) w.y = -w.y;
      v[i * R1 + n1] = cmul(u[n1], w);
    }
  }
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) lds[lidx<R1>(t + R1 * i, n1, s, P)] = v[i * R1 + n1].x;
  }
  __syncthreads();
  float re[R2];
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) re[k2] = lds[lidx<R1>(k2, t, s, P)];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (!reg2_owns<R1, R2>(t, i)) continue;
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) lds[lidx<R1>(t + R1 * i, n1, s, P)] = v[i * R1 + n1].y;
  }
  __syncthreads();
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) v[k2] = make_float2(re[k2], lds[lidx<R1>(k2, t, s, P)]);
  dft_reg<R2, DIR>(v);
}

// e^{DIR 2 pi i q / M} for M = 2, 3
template <int M, int DIR>
__device__ __forceinline__ float2 root_m(int q) {
  if (M == 2) return make_float2(q ? -1.f : 1.f, 0.f);
  constexpr float h = 0.8660254037844386f;  // sqrt(3) / 2
  return q == 0 ? make_float2(1.f, 0.f) : make_float2(-0.5f, ((q == 1) == (DIR > 0)) ? h : -h);
}
// output m of an M-point DFT (sign DIR) of z[0..M)
template <int M, int DIR>
__device__ __forceinline__ float2 dft_m_out(const float2* z, int m) {
  float2 r = z[0];
#pragma unroll
  for (int q = 1; q < M; ++q) r = cadd(r, cmul(root_m<M, DIR>((q * m) % M), z[q]));
  return r;
}

}  // namespace ddhip
