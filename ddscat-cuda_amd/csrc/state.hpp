// Device-resident state of one prepared target (Green tensor, FFT work
// buffers, occupancy maps, solver workspace).  The reference C ABI is
// stateful and single-instance (ddscat_cuda_unified/cuda/ddscat_matvec_cuda.cu:20-56);
// the library keeps one default Context for it.
#pragma once
#include "common.hpp"
#include <vector>

namespace ddhip {

enum Backend { BACKEND_FFT3D = 0, BACKEND_SLICES = 1 };
enum Precision { PREC_MIXED = 0, PREC_FP32 = 1 };

struct MatvecPlan {
  int nx = 0, ny = 0, nz = 0, nat = 0, nat0 = 0;
  int gx = 0, gy = 0, gz = 0;
  size_t ngrid = 0;
  FftPlan px{}, py{}, pz{};
  float2 *twx = nullptr, *twy = nullptr, *twz = nullptr;  // device twiddle tables
  // tile parameters
  int rx = 1, cy = 1, cz = 1;
  int tx = 256, ty = 256, tz = 256;  // workgroup sizes of the LDS-staged x, y and z passes
  // z pitch and kx plane strides (elements) of the FFT3D work arrays
  // a1 [3][gx][p1: ny][nzp] and a2 [3][gx][p2: gy][nzp]
  int nzp = 0, p1 = 0, p2 = 0;
  // FFT kernel per pass 1..5: index into the register shapes of that pass's
  // axis length, or -1 for the LDS-staged kernel (chosen by the autotuner)
  int kind[6] = {-1, -1, -1, -1, -1, -1};
  int zsh = 0;    // log2 of the z run length of the row support (c.ysup)
  int plane = 0;  // passes 2 to 4 by the plane kernel (plane_yz.hpp)
  // pass 5's factor of the convolution, a float and the rest, for the kernels of scale_key (matvec_scale)
  float2 scale{0.f, 0.f};
  int scale_key[6] = {-2, -2, -2, -2, -2, -2};
  int tuned = 0;
};

// Convergence record of the last solve (batched: one entry per RHS;
// single-RHS solvers: RHS 0), read by ddscat_hip_solve_log.
// What a failed reliable-residual check (gap >= 1e-3 or false convergence,
// cu:543-556) does to QMRCCG: REPLACE takes the true residual as the
// recursive one and keeps the Lanczos recurrence (default); RESTART restarts
// the recurrence from the true residual, as the reference does.
enum ReliableMode { RELIABLE_REPLACE = 0, RELIABLE_RESTART = 1 };

struct SolveLog {
  enum { RESTART = 1, REPLACE = 2 };  // action column of a check row
  std::vector<std::vector<double>> resid;   // recursive residual after each iteration
  std::vector<std::vector<double>> checks;  // (iteration, true residual, gap, action) per reliable check
  std::vector<int> restarts;
  void reset(int n) {
    resid.assign(n, {});
    checks.assign(n, {});
    restarts.assign(n, 0);
  }
  void iter(int r, double v) {
    if (r >= 0 && r < (int)resid.size()) resid[r].push_back(v);
  }
  void check(int r, double true_res, double gap, int action) {
    if (r < 0 || r >= (int)resid.size()) return;
    checks[r].insert(checks[r].end(), {(double)resid[r].size(), true_res, gap, (double)action});
    if (action == RESTART) ++restarts[r];
  }
};

// Prepared targets the library holds at once: slot 0 is the reference ABI's
// single target; slots 1..MAX_TARGETS serve multi-target batched solves
// (ddscat_hip_select_target, ddscat_hip_solve_targets).
constexpr int MAX_TARGETS = 64;

struct Context {
  int slot = 0;  // index of this context among the held targets
  bool ready = false;
  int nx = 0, ny = 0, nz = 0, ipbc = 0, nat = 0, nat0 = 0;
  int backend = BACKEND_FFT3D;
  int precision = PREC_MIXED;
  MatvecPlan mv;
  hipStream_t stream = nullptr;
  // Spectral Green tensor, point-interleaved complex64: the trimmed octant
  // of (nx+1)(ny+1)(nz+1) points for IPBC=0, the whole grid of 2nx 2ny 2nz for IPBC=1
  float2* green = nullptr;
  size_t green_count = 0;
  // FFT3D work: a1 [3][gx][p1: ny][nzp], a2 [3][gx][p2: gy][nzp]
  float2 *a1 = nullptr, *a2 = nullptr;
  // occupancy
  int16_t* iocc = nullptr;     // [nat]
  int* occ = nullptr;          // [nat0] occupied site j, increasing
  int* rowptr = nullptr;       // [ny*nz+1] compact range of each (iy,iz) row
  int* rowlo = nullptr;        // [ny*nz] first occupied ix of each row
  int* qmap = nullptr;         // [nat] full site -> compact index (-1 void); built when rows are not intervals
  int2* ysup = nullptr;        // occupied iy range of each z run (BatchArgs::ysup); nullptr where it is nearly all
  int rows_contiguous = 0;     // every row's occupied sites form one interval
  int fft_generic = 0;         // 1: force the LDS-staged generic FFT kernels
  int autotune = 1;            // 1: time the FFT kernel candidates per pass at prepare
  // full-layout operator and vector staging
  float2 *adia = nullptr, *aoff = nullptr;      // [3*nat]
  float2 *adia_c = nullptr, *aoff_c = nullptr;  // [3*nat0]
  float2 *xfull = nullptr, *yfull = nullptr;    // [3*nat]
  // solver storage (compact, 3*nat0 each)
  float2 *sx = nullptr, *sy = nullptr, *sb = nullptr, *wrk = nullptr;
  int wrk_vectors = 0;
  double* red = nullptr;        // reduction partials
  double* scal = nullptr;       // device scalar block (doubles)
  double* hscal = nullptr;      // pinned host mirror
  bool solution_valid = false;
  unsigned long long matvec_count = 0;
  int restarts = 0;               // reliable-residual restarts of the last single-RHS solve
  SolveLog log;                   // convergence record of the last solve
  int reliable_mode = RELIABLE_REPLACE;  // QMRCCG's response to a failed reliable check
  double forced_gap = 0.0;        // added once to the next reliable check's gap (test hook)
  double green_build_ms = 0.0;
};

Context& ctx();                 // the selected target's context
Context& ctx_at(int slot);      // target slot 0..MAX_TARGETS
int selected_target();
void select_target(int slot);
void release_context(Context& c);
int  ensure_solver_workspace(Context& c, int nvec);
void release_solver_workspace(Context& c);

// Several right-hand sides through one MATVEC launch sequence: RHS r uses
// x + r*xs, y + r*xs, adia + r*os, aoff + r*os (os = 0: shared operators) and
// its own FFT work a1 + r*a1s, a2 + r*a2s; RHS with active[r] == 0 are
// skipped (every workgroup of theirs exits at once).  Kernel-side view:
struct BatchArgs {
  size_t xs = 0, os = 0, a1s = 0, a2s = 0;
  const int* active = nullptr;
  // Support of a compact vector: occupied iy range [x, y) of each 1 << zsh
  // consecutive iz; nullptr: all rows.  Pass 1 leaves the rows of a1 outside
  // it unwritten and pass 2 takes them as zero; pass 4 leaves them unwritten
  // and pass 5, which has no site there, does not read them.
  const int2* ysup = nullptr;
  int zsh = 0;
};
// The kx planes of a2: 2 H slots, slot s < H holding kx = h0 + s and slot H + s
// its mirror 2NX - kx (the plane of the same Green entries; for kx = 0, which
// is its own mirror, kx = NX).  H = NX is every plane (FFT3D); SLICES runs
// passes 2 to 4 over slabs of a few H.
struct KxSlab {
  int h0 = 0, H = 0, gx = 0;
  __host__ __device__ int kx(int slot) const {
    if (slot < H) return h0 + slot;
    const int h = h0 + slot - H;
    return h == 0 ? gx / 2 : gx - h;
  }
};
struct MvBatch {
  int nrhs = 1;
  KxSlab slab;           // the planes passes 2 to 4 run on
  BatchArgs k;
  float2* a1 = nullptr;  // nullptr: the context's single-RHS buffers
  float2* a2 = nullptr;
};

// MATVEC: y = A x.  layout 0: full [3][nat] vectors (iocc mask applied);
// layout 1: compact [3][nat0] vectors (adia_c/aoff_c).  conj_mode: 'N' or 'C'.
// ev (optional): 6 events recorded before passes 1..5 and after pass 5.
int matvec_launch(Context& c, int cwhat, const float2* x, float2* y, const float2* adia,
                  const float2* aoff, int layout, hipStream_t st, hipEvent_t* ev = nullptr,
                  const MvBatch* bt = nullptr);
int matvec_setup(Context& c);
// sets the row support in k for a call of this layout, where the kernels of the plan honour it
void matvec_support(const Context& c, int layout, BatchArgs& k);
void matvec_release(Context& c);
// FFT work elements per RHS: a1 [3][gx][p1: ny][nzp], a2 [3][gx][p2: gy][nzp]
size_t matvec_a1_count(const Context& c);
size_t matvec_a2_count(const Context& c);
// register-FFT shapes available for pass `which` (1..5) on a padded axis length (0: none)
int reg_candidates(int L, int which);
// stages of shape `cand` of pass `which`
FftPlan reg_stages(int L, int which, int cand);
// whether the wave kernel of the Green pass, which addresses a component of a2
// and the Green array with 32-bit byte offsets, reaches the planes sl
bool reg_green_reach(const Context& c, const KxSlab& sl);
// whether y-pass shape `cand` of a padded length leaves the rows outside the row support alone
bool reg_row_support(int L, int cand);
// register-FFT pass `which` (1..5) with shape `cand` of its axis length; 1 = launched
int reg_pass(Context& c, int which, int cand, int cj, int compact, const float2* x, float2* y, const float2* adia,
             const float2* aoff, hipStream_t st, const MvBatch& bt);
// passes 2 to 4 on the planes bt.slab of a1, through the slab's planes in bt.a2
int matvec_slab(Context& c, hipStream_t st, const MvBatch& bt);
// SLICES: bt's slab and a2: the slab of planes from half-plane h0 and its buffer
void slices_slab(const Context& c, int h0, MvBatch& bt);
// the plane kernel in place of passes 2 to 4, in place on every plane of bt.a1:
// whether the prepared grid takes it (c.mv.plane), and its launch
int plane_yz_setup(Context& c);
// whether it runs now: the LDS-staged family can be chosen on a prepared target
inline bool plane_yz_runs(const Context& c) { return c.mv.plane && !c.fft_generic; }
int plane_yz_launch(Context& c, hipStream_t st, const MvBatch& bt);
// its stages along y and z
void plane_yz_stages(const Context& c, FftPlan& y, FftPlan& z);
// pass 1 (x -> a1) or 5 (a1 -> y) alone
int matvec_end_pass(Context& c, int which, int cwhat, const float2* x, float2* y, const float2* adia,
                    const float2* aoff, int layout, hipStream_t st, const MvBatch& bt);
// axis lengths, pitches and twiddles of c.mv
int matvec_plan(Context& c, const char* name);
// times every FFT kernel candidate of each pass and stores the fastest in c.mv.kind
int matvec_autotune(Context& c);

// Green tensor build on device, result in c.green (octant for IPBC=0, whole
// grid for IPBC=1).  gamma, pyd, pzd and the wave-vector components matter
// only for IPBC=1 (replica sums, cu:634-643).
struct GreenBuild {
  int ipbc = 0, idipint = 0;
  double gamma = 0.0, pyd = 0.0, pzd = 0.0;
  double ak[3] = {0.0, 0.0, 0.0};
  double dx[3] = {1.0, 1.0, 1.0};
};
int green_build(Context& c, const GreenBuild& b);
// number of direct interactions the IPBC=1 replica sums would evaluate (upper
// bound over the lag grid); 0 for IPBC=0
double green_pbc_work(const Context& c, const GreenBuild& b);

// The resident spectral Green tensor c.green is stored point-interleaved:
// the six components (xx, xy, xz, yy, yz, zz) of octant point
// (ir, jr, kr) sit at green[6p .. 6p+5], so a MATVEC reads them as three
// 16-byte loads from one 48-byte run.  The axis that the Green pass transforms
// runs fastest: p = kr + (NZ+1)(jr + (NY+1) ir).  The reference layout
// ([6][NZ+1][NY+1][NX+1], CXZC) is converted at the ABI edges.
struct Green6 {
  float2 xx, xy, xz, yy, yz, zz;
};
__device__ __forceinline__ Green6 green_at(const float2* __restrict__ g, size_t p) {
  const float4* q = reinterpret_cast<const float4*>(g) + 3 * p;
  const float4 a = q[0], b = q[1], c = q[2];
  return Green6{make_float2(a.x, a.y), make_float2(a.z, a.w), make_float2(b.x, b.y),
                make_float2(b.z, b.w), make_float2(c.x, c.y), make_float2(c.z, c.w)};
}
// Where the Green entry of spectral point (kx, ky, kz) lives, and its signs.
// IPBC=0 stores the octant and rebuilds the rest by mirror symmetry
// (cu:109-115): index min(k, 2N - k) per axis, the off-diagonal components
// flip sign with the mirrored axes' parities.  IPBC=1 stores the whole grid.
// Both use the same instructions:
//   r = min(k, m - k),  sign = (k <= t) ? +1 : -1,
//   point = rz + oz (ry + oy rx)
// octant: m = 2N, t = N, o = N+1; full grid: m = t = 2^30 (no mirror, all
// signs +1), o = 2N.
struct GreenGeo {
  int ox, oy, oz;
  int mx, my, mz;
  int tx, ty, tz;
};
inline GreenGeo green_geo(const Context& c) {
  constexpr int NOMIRROR = 1 << 30;
  if (c.ipbc) return GreenGeo{2 * c.nx, 2 * c.ny, 2 * c.nz, NOMIRROR, NOMIRROR, NOMIRROR, NOMIRROR, NOMIRROR, NOMIRROR};
  return GreenGeo{c.nx + 1, c.ny + 1, c.nz + 1, 2 * c.nx, 2 * c.ny, 2 * c.nz, c.nx, c.ny, c.nz};
}
// number of spectral Green points stored: octant or whole padded grid
inline size_t green_points(int nx, int ny, int nz, int ipbc) {
  return ipbc ? (size_t)(2 * nx) * (2 * ny) * (2 * nz) : (size_t)(nx + 1) * (ny + 1) * (nz + 1);
}

// component-major [6][rz][ry][rx] (x fastest) <-> the resident layout, device to device
int green_interleave(Context& c, const float2* comp_major, float2* resident, hipStream_t st);
int green_deinterleave(Context& c, const float2* resident, float2* comp_major, hipStream_t st);

}  // namespace ddhip
