// DG upwind advection on a Cartesian periodic mesh (GLL nodal basis,
// Gauss quadrature), EvaluationDGAdvection::do_inner_loop / do_rk_stage of
// legacy/include/evaluation_dg_advect.h:285-715, plus what the reference
// does not have: per-point velocity, the adjoint (transposed) operator and
// the gradient with respect to the velocity.
//
// kind 0  r = M^{-1} L(u),  L(u)_K = (grad v, a u)_K - <v, (a.n) u_upwind>;
//         optional fused LSRK stage np = upd + c_np r, tm = np + c_tm r.
// kind 1  L^T y:  (v, a.grad y)_K - <v, max(a.n,0) (y^- - y^+)>  (downwind
//         coupling), so that A^T w = L^T (M^{-1} w).
// kind 2  M^{-1} x = Sinv^T W^{-1} Sinv x (cell-local collocation inverse).
// kind 3  velocity gradient of mu^T L(a) u with mu = M^{-1} lambda:
//         cell: (d mu/dx_d) u JxW at every q-point; face (upper face of each
//         cell, normal velocity b = a.n):  -(mu^- - mu^+) u_upwind JxW_f.
// kind 4  kinds 1 and 3 of the same mu in one pass (they share the sweeps and
//         derivatives of mu), the velocity read from the caller's arrays and
//         stored into the operator's on the way (set_cell, set_face).
// kind 5  kind 0 that reads and stores the velocity so.
// One thread per line of N points of a cell (N^2 threads), cells_per_block
// cells in a workgroup, the cell's values in LDS between the sweeps.
//
// What bounds it: the stored velocity and the vectors at large sizes, and for
// N <= 4 as much the vector unit's issue slots (N = 4, FP32, 47x51x45 cells:
// 693 vector instructions a thread were 30 of 41 us).  So no quadrature weight
// is multiplied in the kernels: in the collocation space of the Gauss points
// the tangential weights of every term cancel against those of W^{-1}, and what
// is left (w_j / w_i, the cell size, the lifting l_i(0) / w_i of the face
// fluxes) is folded into the 1D matrices on the host, one per direction; the
// inverse mass matrix is one 1D matrix per direction instead of two.  The sweeps
// end so that the first and the last run on the z lines that are loaded and
// stored (consecutive dofs across lanes), and the y derivative starts from the
// registers of the y value sweep: 7 phases instead of 10.  Measured, before ->
// after: apply FP64 p = 3 48^3 62.7 -> 55.7 us (5.8 TB/s, as a large elementwise
// kernel), p = 7 24x25x26 74 -> 62, FP32 p = 3 47x51x45 29.3 -> 27.5; transpose
// FP64 p = 3 90 -> 83; LSRK stage FP64 p = 3 95 -> 79, p = 8 22x21x20 104 -> 81; velocity gradient
// FP64 p = 3 108 -> 74, FP32 51 -> 39.
#include "sfk_device.h"
#include "sfk_kernels.h"

namespace sfk {

constexpr int kAdvMaxThreads = 256;

// LDS values per cell: two blocks (A, B) and six face layers; kind 2 one block,
// kind 4 three blocks and nine layers
template <int N, typename T, int KIND>
constexpr int adv_lds_values()
{
  if (KIND == 2) return CellLds<N, T>::CS;
  return KIND == 4 ? 3 * CellLds<N, T>::CS + 9 * N * N : 2 * CellLds<N, T>::CS + 6 * N * N;
}
template <int N, typename T, int KIND>
constexpr int adv_waves()
{
  constexpr int cb = full_cells(N);
  return lds_waves_per_simd(cb * adv_lds_values<N, T, KIND>() * (int)sizeof(T), cb * N * N);
}

// face lifting of one direction, l_i(0) f0 + l_i(1) f1 at point i by parity:
// e[i] (f0 + f1) + o[i] (f0 - f1), the mirrored point with - o[i]
template <int N, typename T>
struct AdvLift {
  T e[(N + 1) / 2], o[(N + 1) / 2];
};

// 1D matrices of an advection operator, weights and cell size folded in
template <int N, typename T>
struct AdvTab {
  Eo<N, T> Sf;       // GLL values -> Gauss points
  Eo<N, T> If;       // Gauss points -> GLL values (inverse of Sf)
  Eo<N, T> Sw;       // S^T W: Gauss points -> test functions
  Eo<N, T> Mi, Mij;  // S^{-1} W^{-1} S^{-T}, and that divided by JxW's cell part
  Eo<N, T> Dw[3];    // ij W^{-1} D^T W (forward)
  Eo<N, T> Da[3];    // ij jxw D (adjoint)
  Eo<N, T> Dg[3];    // ij jxw W D (velocity gradient)
  AdvLift<N, T> tr;  // traces: v0, v1 = sum of l_i(0), l_i(1) times the values
  AdvLift<N, T> Lw[3], La[3]; // -1/2 ij W^{-1} l, and that times jxw
  T w[N];            // Gauss weights
};

template <int N, typename T>
static AdvTab<N, T> make_advtab(const Tables1D &t, const double ij[3])
{
  AdvTab<N, T> a{};
  // products in extended precision: one rounding per entry
  using R = long double;
  const R jxw = 1 / (R(ij[0]) * ij[1] * ij[2]);
  const std::vector<R> w(t.weights.begin(), t.weights.end());
  std::vector<double> m(N * N);
  auto eo = [&](bool forward, auto entry) {
    for (int i = 0; i < N; ++i)
      for (int q = 0; q < N; ++q) m[i * N + q] = (double)entry(i, q);
    return make_eo<N, T>(m, forward);
  };
  auto lift = [&](auto l0) { // l0(i): the factor of f0; that of f1 mirrors it
    AdvLift<N, T> L{};
    for (int i = 0; i < (N + 1) / 2; ++i) {
      L.e[i] = T((l0(i) + l0(N - 1 - i)) / 2);
      L.o[i] = T((l0(i) - l0(N - 1 - i)) / 2);
    }
    return L;
  };
  auto minv = [&](int i, int q) {
    R v = 0;
    for (int k = 0; k < N; ++k) v += (R)t.Sinv[k * N + i] * t.Sinv[k * N + q] / w[k];
    return v;
  };
  a.Sf = make_eo<N, T>(t.S, true);
  a.If = make_eo<N, T>(t.Sinv, true);
  a.Sw = eo(false, [&](int i, int q) { return t.S[i * N + q] * w[q]; });
  a.Mi = eo(true, minv);
  a.Mij = eo(true, [&](int i, int q) { return minv(i, q) / jxw; });
  a.tr = lift([&](int i) { return t.fv0[i]; });
  for (int d = 0; d < 3; ++d) {
    a.Dw[d] = eo(false, [&](int i, int q) { return ij[d] * (t.D[i * N + q] * w[q] / w[i]); });
    a.Da[d] = eo(true, [&](int i, int q) { return ij[d] * jxw * t.D[i * N + q]; });
    a.Dg[d] = eo(true, [&](int i, int q) { return ij[d] * jxw * (t.D[i * N + q] * w[q]); });
    a.Lw[d] = lift([&](int i) { return -(R)ij[d] * (t.fv0[i] / w[i]) / 2; });
    a.La[d] = lift([&](int i) { return -ij[d] * jxw * (t.fv0[i] / w[i]) / 2; });
  }
  for (int i = 0; i < N; ++i) a.w[i] = T(w[i]);
  return a;
}

template <int N, typename T>
__device__ __forceinline__ const SFK_CONST_AS AdvTab<N, T> &atab(const AdvTab<N, T> *p)
{
  return *(const SFK_CONST_AS AdvTab<N, T> *)opaque_ptr(p);
}

template <int N, typename T>
struct AdvArgs {
  const AdvTab<N, T> *dt; // tables in device memory (read through atab)
  const T *src, *upd, *aux;
  T *dst, *tm, *dst2;
  T c_np, c_tm;
  const T *cell_vel, *face_vel;
  T *set_cell, *set_face; // kinds 4 and 5: the velocity read is stored here
  T vel[3];
  T jxwf[3];
  long long ncells;
  int nx, ny, nz;
  int cb;    // cells per workgroup
  int order; // block order (logical_block)
};

// velocity component DIR at the points of line l, and the normal velocities
// a.n (outward from the cell) on its two ends: the lower face's value is stored
// with the lower neighbour
template <int N, typename T>
struct AdvVel {
  T v[N], n0, n1;
};
template <int N, int DIR, typename T, bool VAR>
__device__ __forceinline__ void load_velocity(const AdvArgs<N, T> &a, long long cell, int lower, int l, AdvVel<N, T> &v)
{
  if constexpr (VAR) {
    constexpr int N2 = N * N, N3 = N2 * N;
    const T *p = a.cell_vel + (cell * 3 + DIR) * N3 + line_base<N, N, DIR>(l);
#pragma unroll
    for (int i = 0; i < N; ++i) v.v[i] = p[i * line_stride<N, N, DIR>()];
    const T *f = a.face_vel + (long long)DIR * a.ncells * N2 + l;
    v.n0 = -f[(long long)lower * N2];
    v.n1 = f[cell * N2];
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) v.v[i] = a.vel[DIR];
    v.n0 = -a.vel[DIR];
    v.n1 = a.vel[DIR];
  }
}

// Stores of results that no workgroup of the launch reads: non-temporal where
// that pays, which for the stage is where one store instruction covers whole
// cache lines, and for the velocity gradients also in FP64 from N = 4 on.
// Measured, plain -> non-temporal: time step (5 stages) FP64 p = 3 47x51x45 396 ->
// 374 us, but p = 2 72x70x68 659 -> 788, FP32 p = 4 40x37x42 214 -> 261; velocity
// gradient repeated into the same arrays FP64 p = 3 48^3 105 -> 74 us, p = 4 130 ->
// 98, p = 6 112 -> 86, FP32 p = 3 42 -> 39, but p = 1 126 -> 159, p = 6 47 -> 54;
// within forward, loss and backward pass FP32 p = 3 254 -> 251, but p = 2 399 ->
// 431, FP64 p = 2 688 -> 721.
template <int N, typename T>
constexpr bool adv_nt_grad()
{
  return (sizeof(T) == 8 && N >= 4) || N * N * sizeof(T) % 64 == 0;
}
template <int N, typename T>
constexpr bool adv_nt_stage()
{
  return N * N * sizeof(T) % 128 == 0;
}
template <bool NT, typename T>
__device__ __forceinline__ void store_result(T v, T *p)
{
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// How kinds 4 and 5 store the velocity: for N < 4 as a copy of its own
// (copy_velocity: a second, contiguous load, non-temporal stores), else from the
// registers that the lines are computed from.  Forward pass, loss and backward
// pass, copy / registers: p = 1 90x85x80 FP32 232 / 259 us, FP64 395 / 420; p = 2
// 72x70x68 FP32 399 / 442, FP64 721 / 746; but p = 3 47x51x45 FP32 264 / 253,
// FP64 453 / 431; p = 6 28x27x29 FP32 290 / 274, FP64 520 / 474 (p = 4 FP32 303 /
// 312).  With separate set, apply, transpose and gradient calls p = 3 took 345
// (FP32) and 617 us.
template <int N, typename T>
constexpr bool adv_flat_copy()
{
  return N < 4;
}

template <int N, int DIR, typename T>
__device__ __forceinline__ void store_velocity(const AdvArgs<N, T> &a, long long cell, int l, const AdvVel<N, T> &v)
{
  constexpr int N2 = N * N, N3 = N2 * N;
  T *p = a.set_cell + (cell * 3 + DIR) * N3 + line_base<N, N, DIR>(l);
#pragma unroll
  for (int i = 0; i < N; ++i) p[i * line_stride<N, N, DIR>()] = v.v[i];
  a.set_face[((long long)DIR * a.ncells + cell) * N2 + l] = v.n1;
}

// Part of three of the copy of the caller's velocity into the operator's: the
// workgroup at traversal position cell0 copies the values of CB cells in index
// order (which for block order 2 need not be the cells it computes), so that
// loads and stores are contiguous over the workgroup.
template <int N, typename T>
struct AdvCopy {
  T v[N], f;
};
template <int N, typename T, bool STORE>
__device__ __forceinline__ void copy_velocity(const AdvArgs<N, T> &a, long long cell0, int CB, int t, int part,
                                              AdvCopy<N, T> &c)
{
  constexpr int N2 = N * N, N3 = N2 * N;
  if constexpr (!adv_flat_copy<N, T>()) return;
  const int nt = CB * N2;
  if (t >= nt) return;
  const long long base = cell0 * (3 * N3) + (long long)part * N * nt + t, end = a.ncells * (3 * N3);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (base + i * nt < end) {
      if constexpr (STORE) store_result<true>(c.v[i], a.set_cell + base + i * nt);
      else c.v[i] = a.cell_vel[base + i * nt];
    }
  }
  const long long fb = cell0 * N2 + t;
  if (fb < a.ncells * N2) {
    if constexpr (STORE) store_result<true>(c.f, a.set_face + part * a.ncells * N2 + fb);
    else c.f = a.face_vel[part * a.ncells * N2 + fb];
  }
}

// traces at both ends of a line of Gauss values
template <int N, typename L, typename T>
__device__ __forceinline__ void line_traces(const L &tr, const T (&q)[N], T &v0, T &v1)
{
  T e = 0, o = 0;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    e += tr.e[i] * (q[i] + q[N - 1 - i]);
    o += tr.o[i] * (q[i] - q[N - 1 - i]);
  }
  if constexpr (N % 2 == 1) e += tr.e[N / 2] * q[N / 2];
  v0 = e + o;
  v1 = e - o;
}

// r = D g plus the lifting of the end values f0, f1 (D odd: eo_apply<N, -1>
// with the lifting added to its two parity sums)
template <int N, typename E, typename L, typename T>
__device__ __forceinline__ void derivative_lift(const E &t, const L &lw, const T (&g)[N], T f0, T f1, T (&r)[N])
{
  constexpr int mid = N / 2;
  const T fs = f0 + f1, fd = f0 - f1;
  T e[mid], o[mid];
#pragma unroll
  for (int k = 0; k < mid; ++k) {
    e[k] = g[k] + g[N - 1 - k];
    o[k] = g[k] - g[N - 1 - k];
  }
#pragma unroll
  for (int q = 0; q < mid; ++q) {
    T p = lw.o[q] * fd, s = lw.e[q] * fs;
#pragma unroll
    for (int k = 0; k < mid; ++k) {
      p += t.A[k][q] * e[k];
      s += t.B[k][q] * o[k];
    }
    if constexpr (N % 2 == 1) p += t.C[q] * g[mid];
    r[q] = s + p;
    r[N - 1 - q] = s - p;
  }
  if constexpr (N % 2 == 1) {
    T m = lw.e[mid] * fs;
#pragma unroll
    for (int k = 0; k < mid; ++k) m += t.E[k] * o[k];
    r[mid] = m;
  }
}

// r = v r plus the lifting of the end values f0, f1
template <int N, typename L, typename T>
__device__ __forceinline__ void scale_lift(const L &lw, const T (&v)[N], T f0, T f1, T (&r)[N])
{
  const T fs = f0 + f1, fd = f0 - f1;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const T s = lw.e[i] * fs;
    r[i] = v[i] * r[i] + (s + lw.o[i] * fd);
    r[N - 1 - i] = v[N - 1 - i] * r[N - 1 - i] + (s - lw.o[i] * fd);
  }
  if constexpr (N % 2 == 1) r[N / 2] = v[N / 2] * r[N / 2] + lw.e[N / 2] * fs;
}

// One face layer line per item (6 N of them): the layer of neighbour f that
// touches this cell (GLL nodal: the layer is the trace), swept in the second
// tangential direction on its way into F[f][fa].  Adjacent items are adjacent
// in the first, so that their loads share cache lines.
template <int N, typename T, typename E>
__device__ __forceinline__ void face_lines(const E &S, const T *src, T *F, int item, int f, int d, int layer, int nbr)
{
  constexpr int N2 = N * N, N3 = N2 * N;
  const int r = item % N;
  const T *p = src + (long long)nbr * N3 + (d == 0 ? r * N + layer : (d == 1 ? layer * N + r : layer * N2 + r));
  const int st = d == 2 ? N : N2;
  T u[N], v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) u[i] = p[i * st];
  eo_apply<N, 1>(S, u, v);
#pragma unroll
  for (int i = 0; i < N; ++i) F[f * N2 + i * N + r] = v[i];
}

// sweep of NF layers in the first tangential direction
template <int N, int NF, typename T, typename E>
__device__ __forceinline__ void face_sweep(const E &S, T *F, int l)
{
  for (int it = l; it < NF * N; it += N * N) {
    T u[N], v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) u[i] = F[it * N + i];
    eo_apply<N, 1>(S, u, v);
#pragma unroll
    for (int i = 0; i < N; ++i) F[it * N + i] = v[i];
  }
}

template <int N, int DIR, typename E, typename T>
__device__ __forceinline__ void sweep_line(const E &M, T *A, int l)
{
  T u[N], v[N];
  cl_read<N, DIR>(A, l, u);
  eo_apply<N, 1>(M, u, v);
  cl_write<N, DIR>(A, l, v);
}

// forward (kind 0) and transposed weak form (kind 1) in direction DIR from the
// line's Gauss values q
template <int N, int DIR, bool ADJ, typename Tb, typename T>
__device__ __forceinline__ void adv_dir(const Tb &tb, const T (&q)[N], const AdvVel<N, T> &v, const T *F, int l,
                                        T (&r)[N])
{
  constexpr int N2 = N * N;
  T v0, v1;
  line_traces<N>(tb.tr, q, v0, v1);
  const T d0 = v0 - F[2 * DIR * N2 + l], d1 = v1 - F[(2 * DIR + 1) * N2 + l];
  if constexpr (!ADJ) {
    T g[N];
#pragma unroll
    for (int i = 0; i < N; ++i) g[i] = v.v[i] * q[i];
    // (u^- + u^+) a.n + |a.n| (u^- - u^+), evaluation_dg_advect.h:403-404 (the
    // factor -1/2 is in the lifting)
    const T s0 = v0 + F[2 * DIR * N2 + l], s1 = v1 + F[(2 * DIR + 1) * N2 + l];
    derivative_lift<N>(tb.Dw[DIR], tb.Lw[DIR], g, s0 * v.n0 + fabs(v.n0) * d0, s1 * v.n1 + fabs(v.n1) * d1, r);
  } else {
    eo_apply<N, -1>(tb.Da[DIR], q, r);
    // 2 max(a.n, 0) (y^- - y^+)
    scale_lift<N>(tb.La[DIR], v.v, (v.n0 > T(0) ? T(2) * v.n0 : T(0)) * d0, (v.n1 > T(0) ? T(2) * v.n1 : T(0)) * d1,
                  r);
  }
}

template <int N, typename T, int KIND, bool VAR, bool STAGE>
__global__ void __launch_bounds__(kAdvMaxThreads) __attribute__((amdgpu_waves_per_eu(1, adv_waves<N, T, KIND>())))
advect_kernel(const AdvArgs<N, T> a)
{
  constexpr int N2 = N * N, N3 = N * N * N;
  constexpr bool ADJ = KIND == 1;
  const int CB = a.cb;
  // dynamic LDS: A [CB][CS], B [CB][CS] (padded cell blocks), F [CB][6][N2]
  // (M^{-1}: A only)
  constexpr int CS = CellLds<N, T>::CS;
  T *sA = dyn_lds<T>();
  const int t = threadIdx.x, c = t / N2, l = t % N2;
  const long long cell0 = (long long)logical_block(blockIdx.x, gridDim.x, a.order) * CB;
  const bool act = c < CB && cell0 + c < a.ncells;
  // the cell at this traversal position and its periodic neighbour cells
  int nbr[6] = {0, 0, 0, 0, 0, 0};
  const long long cell = act ? locate_cell((unsigned)cell0, (unsigned)c, a.nx, a.ny, a.nz, a.order, nbr) : 0;
  T *A = sA + (act ? c : 0) * CS;
  T *B = sA + (CB + (act ? c : 0)) * CS;
  T *F = sA + (KIND == 4 ? 3 : 2) * CB * CS + (act ? c : 0) * (KIND == 4 ? 9 : 6) * N2;

  if constexpr (KIND == 2) {
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], v[N];
#pragma unroll
      for (int k = 0; k < N; ++k) u[k] = a.src[cell * N3 + k * N2 + l];
      eo_apply<N, 1>(tb.Mij, u, v);
      cl_write<N, 2>(A, l, v);
    }
    __syncthreads();
    if (act) sweep_line<N, 0>(atab(a.dt).Mi, A, l);
    __syncthreads();
    if (act) sweep_line<N, 1>(atab(a.dt).Mi, A, l);
    __syncthreads();
    if (act) {
      T u[N];
      cl_read<N, 2>(A, l, u);
#pragma unroll
      for (int k = 0; k < N; ++k) a.dst[cell * N3 + k * N2 + l] = u[k];
    }
    return;
  } else if constexpr (KIND == 3) {
    // velocity gradient: A <- u at q-points, B <- mu at q-points,
    // F[0..2] <- u^+ on the upper faces, F[3..5] <- mu^+ on the upper faces
    T bn[3] = {0, 0, 0}, wl = 0;
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], m[N], v[N];
#pragma unroll
      for (int k = 0; k < N; ++k) u[k] = a.src[cell * N3 + k * N2 + l];
#pragma unroll
      for (int k = 0; k < N; ++k) m[k] = a.aux[cell * N3 + k * N2 + l];
      for (int it = l; it < 6 * N; it += N2) {
        const int fi = it / N, d = fi % 3;
        face_lines<N>(tb.Sf, fi < 3 ? a.src : a.aux, F, it, fi, d, 0, d == 0 ? nbr[1] : (d == 1 ? nbr[3] : nbr[5]));
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) bn[d] = a.face_vel[((long long)d * a.ncells + cell) * N2 + l];
      wl = a.dt->w[l % N] * a.dt->w[l / N];
      eo_apply<N, 1>(tb.Sf, u, v);
      cl_write<N, 2>(A, l, v);
      eo_apply<N, 1>(tb.Sf, m, v);
      cl_write<N, 2>(B, l, v);
    }
    __syncthreads();
    if (act) {
      const auto &tb = atab(a.dt);
      sweep_line<N, 0>(tb.Sf, A, l);
      sweep_line<N, 0>(tb.Sf, B, l);
      face_sweep<N, 6>(tb.Sf, F, l);
    }
    __syncthreads();
    // cell gradients of line l in direction DIR: the x and y lines go
    // through LDS below, so that every store writes consecutive dofs across
    // lanes (FP64 p3 48^3: 168 -> 151 us)
    T gx[N], gy[N];
    auto do_dir = [&](auto dirc, const T(&uq)[N], const T(&mq)[N], T(&g)[N]) {
      constexpr int DIR = decltype(dirc)::value;
      const auto &tb = atab(a.dt);
      eo_apply<N, -1>(tb.Dg[DIR], mq, g);
#pragma unroll
      for (int i = 0; i < N; ++i) g[i] *= wl * uq[i];
      T u0, um, m0, mm;
      line_traces<N>(tb.tr, uq, u0, um);
      line_traces<N>(tb.tr, mq, m0, mm);
      const T up = F[DIR * N2 + l], mp = F[(3 + DIR) * N2 + l];
      const T sg = bn[DIR] > T(0) ? T(1) : (bn[DIR] < T(0) ? T(-1) : T(0));
      const T uh = T(0.5) * (um + up) + T(0.5) * sg * (um - up);
      store_result<adv_nt_grad<N, T>()>(-(mm - mp) * uh * (wl * a.jxwf[DIR]),
                                           a.dst2 + ((long long)DIR * a.ncells + cell) * N2 + l);
    };
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], uq[N], mq[N];
      cl_read<N, 1>(A, l, u);
      eo_apply<N, 1>(tb.Sf, u, uq);
      cl_write<N, 1>(A, l, uq);
      cl_read<N, 1>(B, l, u);
      eo_apply<N, 1>(tb.Sf, u, mq);
      cl_write<N, 1>(B, l, mq);
      do_dir(std::integral_constant<int, 1>(), uq, mq, gy);
    }
    __syncthreads();
    if (act) {
      T uq[N], mq[N], gz[N];
      cl_read<N, 0>(A, l, uq);
      cl_read<N, 0>(B, l, mq);
      do_dir(std::integral_constant<int, 0>(), uq, mq, gx);
      cl_read<N, 2>(A, l, uq);
      cl_read<N, 2>(B, l, mq);
      do_dir(std::integral_constant<int, 2>(), uq, mq, gz);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(gz[m], a.dst + (cell * 3 + 2) * N3 + l + m * N2);
    }
    // x and y gradients: written into the cell blocks (their q-point values
    // are no longer needed) and stored as z lines, lane l at dof l + m N^2
    __syncthreads();
    if (act) {
      cl_write<N, 0>(A, l, gx);
      cl_write<N, 1>(B, l, gy);
    }
    __syncthreads();
    if (act) {
      T v[N];
      cl_read<N, 2>(A, l, v);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(v[m], a.dst + (cell * 3 + 0) * N3 + l + m * N2);
      cl_read<N, 2>(B, l, v);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(v[m], a.dst + (cell * 3 + 1) * N3 + l + m * N2);
    }
    return;
  } else if constexpr (KIND == 4) {
    // A <- u, B <- mu at q-points, C <- the sum of L^T mu, F[0..5] <- mu of the
    // six neighbours, F[6..8] <- u of the upper ones
    T *C = sA + (2 * CB + (act ? c : 0)) * CS;
    AdvVel<N, T> vx, vy, vz;
    T wl = 0;
    AdvCopy<N, T> cp;
    copy_velocity<N, T, false>(a, cell0, CB, t, 0, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], m[N], v[N];
#pragma unroll
      for (int k = 0; k < N; ++k) m[k] = a.aux[cell * N3 + k * N2 + l];
#pragma unroll
      for (int k = 0; k < N; ++k) u[k] = a.src[cell * N3 + k * N2 + l];
      for (int it = l; it < 9 * N; it += N2) {
        const int f = it / N, d = f < 6 ? f / 2 : f - 6;
        const int below = d == 0 ? nbr[0] : (d == 1 ? nbr[2] : nbr[4]);
        const int above = d == 0 ? nbr[1] : (d == 1 ? nbr[3] : nbr[5]);
        const bool up = f >= 6 || f % 2;
        face_lines<N>(tb.Sf, f < 6 ? a.aux : a.src, F, it, f, d, up ? 0 : N - 1, up ? above : below);
      }
      load_velocity<N, 1, T, true>(a, cell, nbr[2], l, vy);
      wl = a.dt->w[l % N] * a.dt->w[l / N];
      eo_apply<N, 1>(tb.Sf, m, v);
      cl_write<N, 2>(B, l, v);
      eo_apply<N, 1>(tb.Sf, u, v);
      cl_write<N, 2>(A, l, v);
    }
    copy_velocity<N, T, true>(a, cell0, CB, t, 0, cp);
    __syncthreads();
    copy_velocity<N, T, false>(a, cell0, CB, t, 1, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      load_velocity<N, 2, T, true>(a, cell, nbr[4], l, vz);
      sweep_line<N, 0>(tb.Sf, A, l);
      sweep_line<N, 0>(tb.Sf, B, l);
      face_sweep<N, 9>(tb.Sf, F, l);
    }
    copy_velocity<N, T, true>(a, cell0, CB, t, 1, cp);
    __syncthreads();
    T gx[N], gy[N];
    auto do_dir = [&](auto dirc, const T(&uq)[N], const T(&mq)[N], const AdvVel<N, T> &v, T(&g)[N], T(&r)[N]) {
      constexpr int DIR = decltype(dirc)::value;
      const auto &tb = atab(a.dt);
      T u0, u1, m0, m1;
      line_traces<N>(tb.tr, uq, u0, u1);
      line_traces<N>(tb.tr, mq, m0, m1);
      const T d0 = m0 - F[2 * DIR * N2 + l], d1 = m1 - F[(2 * DIR + 1) * N2 + l], up = F[(6 + DIR) * N2 + l];
      if constexpr (!adv_flat_copy<N, T>()) store_velocity<N, DIR>(a, cell, l, v);
      eo_apply<N, -1>(tb.Da[DIR], mq, r);
#pragma unroll
      for (int i = 0; i < N; ++i) g[i] = r[i] * (uq[i] * (wl * tb.w[i]));
      const T sg = v.n1 > T(0) ? T(1) : (v.n1 < T(0) ? T(-1) : T(0));
      const T uh = T(0.5) * (u1 + up) + T(0.5) * sg * (u1 - up);
      store_result<adv_nt_grad<N, T>()>(-d1 * uh * (wl * a.jxwf[DIR]),
                                        a.dst2 + ((long long)DIR * a.ncells + cell) * N2 + l);
      scale_lift<N>(tb.La[DIR], v.v, (v.n0 > T(0) ? T(2) * v.n0 : T(0)) * d0, (v.n1 > T(0) ? T(2) * v.n1 : T(0)) * d1,
                    r);
    };
    copy_velocity<N, T, false>(a, cell0, CB, t, 2, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], uq[N], mq[N], r[N];
      load_velocity<N, 0, T, true>(a, cell, nbr[0], l, vx);
      cl_read<N, 1>(A, l, u);
      eo_apply<N, 1>(tb.Sf, u, uq);
      cl_write<N, 1>(A, l, uq);
      cl_read<N, 1>(B, l, u);
      eo_apply<N, 1>(tb.Sf, u, mq);
      cl_write<N, 1>(B, l, mq);
      do_dir(std::integral_constant<int, 1>(), uq, mq, vy, gy, r);
      cl_write<N, 1>(C, l, r);
    }
    copy_velocity<N, T, true>(a, cell0, CB, t, 2, cp);
    __syncthreads();
    if (act) {
      T uq[N], mq[N], gz[N], r[N], b[N];
      cl_read<N, 2>(A, l, uq);
      cl_read<N, 2>(B, l, mq);
      do_dir(std::integral_constant<int, 2>(), uq, mq, vz, gz, r);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(gz[m], a.dst + (cell * 3 + 2) * N3 + l + m * N2);
      cl_read<N, 2>(C, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      cl_write<N, 2>(C, l, r);
    }
    __syncthreads();
    if (act) {
      const auto &tb = atab(a.dt);
      T uq[N], mq[N], r[N], b[N];
      cl_read<N, 0>(A, l, uq);
      cl_read<N, 0>(B, l, mq);
      do_dir(std::integral_constant<int, 0>(), uq, mq, vx, gx, r);
      cl_read<N, 0>(C, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      eo_apply<N, 1>(tb.Sw, r, b);
      cl_write<N, 0>(C, l, b);
    }
    __syncthreads();
    // the x and y gradients leave through A and B as z lines (see kind 3)
    if (act) {
      cl_write<N, 0>(A, l, gx);
      cl_write<N, 1>(B, l, gy);
      sweep_line<N, 1>(atab(a.dt).Sw, C, l);
    }
    __syncthreads();
    if (act) {
      T v[N], o[N];
      cl_read<N, 2>(A, l, v);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(v[m], a.dst + (cell * 3 + 0) * N3 + l + m * N2);
      cl_read<N, 2>(B, l, v);
#pragma unroll
      for (int m = 0; m < N; ++m) store_result<adv_nt_grad<N, T>()>(v[m], a.dst + (cell * 3 + 1) * N3 + l + m * N2);
      cl_read<N, 2>(C, l, v);
      eo_apply<N, 1>(atab(a.dt).Sw, v, o);
#pragma unroll
      for (int m = 0; m < N; ++m) __builtin_nontemporal_store(o[m], a.tm + cell * N3 + l + m * N2);
    }
    return;
  } else {
    // ------------------------------------------------ L: z values + faces
    // The velocities of a direction are loaded two phases before their use.
    AdvVel<N, T> vx, vy, vz;
    AdvCopy<N, T> cp;
    if constexpr (KIND == 5) copy_velocity<N, T, false>(a, cell0, CB, t, 0, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], v[N];
#pragma unroll
      for (int k = 0; k < N; ++k) u[k] = a.src[cell * N3 + k * N2 + l];
      for (int it = l; it < 6 * N; it += N2) {
        const int f = it / N;
        const int below = f == 0 ? nbr[0] : (f == 2 ? nbr[2] : nbr[4]);
        const int above = f == 1 ? nbr[1] : (f == 3 ? nbr[3] : nbr[5]);
        face_lines<N>(tb.Sf, a.src, F, it, f, f / 2, f % 2 ? 0 : N - 1, f % 2 ? above : below);
      }
      load_velocity<N, 1, T, VAR>(a, cell, nbr[2], l, vy);
      eo_apply<N, 1>(tb.Sf, u, v);
      cl_write<N, 2>(A, l, v);
    }
    if constexpr (KIND == 5) copy_velocity<N, T, true>(a, cell0, CB, t, 0, cp);
    __syncthreads();
    if constexpr (KIND == 5) copy_velocity<N, T, false>(a, cell0, CB, t, 1, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      load_velocity<N, 2, T, VAR>(a, cell, nbr[4], l, vz);
      sweep_line<N, 0>(tb.Sf, A, l);
      face_sweep<N, 6>(tb.Sf, F, l);
    }
    if constexpr (KIND == 5) copy_velocity<N, T, true>(a, cell0, CB, t, 1, cp);
    __syncthreads();
    if constexpr (KIND == 5) copy_velocity<N, T, false>(a, cell0, CB, t, 2, cp);
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], q[N], r[N];
      load_velocity<N, 0, T, VAR>(a, cell, nbr[0], l, vx);
      cl_read<N, 1>(A, l, u);
      eo_apply<N, 1>(tb.Sf, u, q);
      cl_write<N, 1>(A, l, q);
      if constexpr (KIND == 5 && !adv_flat_copy<N, T>()) store_velocity<N, 1>(a, cell, l, vy);
      adv_dir<N, 1, ADJ>(tb, q, vy, F, l, r);
      cl_write<N, 1>(B, l, r);
    }
    if constexpr (KIND == 5) copy_velocity<N, T, true>(a, cell0, CB, t, 2, cp);
    __syncthreads();
    if (act) {
      const auto &tb = atab(a.dt);
      T q[N], r[N], b[N];
      cl_read<N, 2>(A, l, q);
      if constexpr (KIND == 5 && !adv_flat_copy<N, T>()) store_velocity<N, 2>(a, cell, l, vz);
      adv_dir<N, 2, ADJ>(tb, q, vz, F, l, r);
      cl_read<N, 2>(B, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      cl_write<N, 2>(B, l, r);
    }
    __syncthreads();
    // back to the dofs: forward by collocation (evaluation_dg_advect.h:619-624)
    if (act) {
      const auto &tb = atab(a.dt);
      T q[N], r[N], b[N];
      cl_read<N, 0>(A, l, q);
      if constexpr (KIND == 5 && !adv_flat_copy<N, T>()) store_velocity<N, 0>(a, cell, l, vx);
      adv_dir<N, 0, ADJ>(tb, q, vx, F, l, r);
      cl_read<N, 0>(B, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      if constexpr (!ADJ) eo_apply<N, 1>(tb.If, r, b);
      else eo_apply<N, 1>(tb.Sw, r, b);
      cl_write<N, 0>(B, l, b);
    }
    __syncthreads();
    if (act) {
      const auto &tb = atab(a.dt);
      if constexpr (!ADJ) sweep_line<N, 1>(tb.If, B, l);
      else sweep_line<N, 1>(tb.Sw, B, l);
    }
    __syncthreads();
    if (act) {
      const auto &tb = atab(a.dt);
      T u[N], o[N];
      const long long g0 = cell * N3 + l;
      if constexpr (STAGE) {
        T up[N];
#pragma unroll
        for (int m = 0; m < N; ++m) up[m] = a.upd[g0 + m * N2];
        cl_read<N, 2>(B, l, u);
        eo_apply<N, 1>(tb.If, u, o);
        // evaluation_dg_advect.h:651-667
#pragma unroll
        for (int m = 0; m < N; ++m) {
          const long long g = g0 + m * N2;
          const T vnp = up[m] + a.c_np * o[m];
          store_result<adv_nt_stage<N, T>()>(vnp, a.dst + g);
          if (a.c_tm != T(0)) store_result<adv_nt_stage<N, T>()>(vnp + a.c_tm * o[m], a.tm + g);
        }
      } else {
        cl_read<N, 2>(B, l, u);
        if constexpr (!ADJ) eo_apply<N, 1>(tb.If, u, o);
        else eo_apply<N, 1>(tb.Sw, u, o);
        // written once, read by nobody in this launch: non-temporal stores
        // keep L2 for the velocity and neighbour layers other workgroups
        // re-read (forward p = 3, 48^3: 73 -> 60 us on MI355X)
#pragma unroll
        for (int m = 0; m < N; ++m) __builtin_nontemporal_store(o[m], a.dst + g0 + m * N2);
      }
    }
  }
}

template <int N, typename T>
static size_t advect_lds_per_cell_n(int kind)
{
  return size_t(kind == 2 ? adv_lds_values<N, T, 2>() : kind == 4 ? adv_lds_values<N, T, 4>() : adv_lds_values<N, T, 0>()) *
         sizeof(T);
}

template <int N, typename T>
static hipError_t launch_advect_n(const AdvectLaunch &L, hipStream_t s)
{
  AdvArgs<N, T> a{};
  a.dt = (const AdvTab<N, T> *)L.dtab;
  a.src = (const T *)L.src;
  a.upd = (const T *)L.upd;
  a.aux = (const T *)L.aux;
  a.dst = (T *)L.dst;
  a.tm = (T *)L.tm;
  a.dst2 = (T *)L.dst2;
  a.c_np = T(L.c_np);
  a.c_tm = T(L.c_tm);
  a.cell_vel = (const T *)L.cell_vel;
  a.face_vel = (const T *)L.face_vel;
  a.set_cell = (T *)L.set_cell;
  a.set_face = (T *)L.set_face;
  const double jxw = 1. / (L.inv_jac[0] * L.inv_jac[1] * L.inv_jac[2]);
  for (int d = 0; d < 3; ++d) {
    a.vel[d] = T(L.vel[d]);
    a.jxwf[d] = T(jxw * L.inv_jac[d]);
  }
  a.ncells = L.ncells;
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  const int CB = L.cb > 0 ? L.cb : full_cells(N);
  if (CB * N * N > kAdvMaxThreads) return hipErrorInvalidConfiguration;
  a.cb = CB;
  a.order = L.order;
  const size_t lds = size_t(CB) * advect_lds_per_cell_n<N, T>(L.kind);
  const dim3 grid((unsigned)((L.ncells + CB - 1) / CB)), block(((CB * N * N + 63) / 64) * 64);
  const bool var = L.cell_vel != nullptr;
  decltype(&advect_kernel<N, T, 0, false, false>) kern = nullptr;
  switch (L.kind) {
  case 0:
    if (var) kern = L.stage ? advect_kernel<N, T, 0, true, true> : advect_kernel<N, T, 0, true, false>;
    else kern = L.stage ? advect_kernel<N, T, 0, false, true> : advect_kernel<N, T, 0, false, false>;
    break;
  case 1: kern = var ? advect_kernel<N, T, 1, true, false> : advect_kernel<N, T, 1, false, false>; break;
  case 2: kern = advect_kernel<N, T, 2, false, false>; break;
  case 3: kern = advect_kernel<N, T, 3, true, false>; break;
  case 4: kern = advect_kernel<N, T, 4, true, false>; break;
  case 5: kern = advect_kernel<N, T, 5, true, false>; break;
  default: return hipErrorInvalidValue;
  }
  const hipError_t e = allow_dynamic_lds((const void *)kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, block, lds, s, a);
  return hipGetLastError();
}

template <typename T>
static hipError_t dispatch_advect(const AdvectLaunch &L, hipStream_t s)
{
  switch (L.tables->n) {
#define SFK_CASE(NN) \
  case NN: return launch_advect_n<NN, T>(L, s);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

template <int N, typename T>
static hipError_t upload_advtab(const Tables1D &t, const double ij[3], void **dev)
{
  const AdvTab<N, T> h = make_advtab<N, T>(t, ij);
  const hipError_t e = hipMalloc(dev, sizeof(h));
  if (e != hipSuccess) {
    *dev = nullptr;
    return e;
  }
  return hipMemcpy(*dev, &h, sizeof(h), hipMemcpyHostToDevice);
}

hipError_t upload_advect_tables(const Tables1D &t, const double ij[3], bool fp32, void **dev)
{
  switch (t.n) {
#define SFK_CASE(NN) \
  case NN: return fp32 ? upload_advtab<NN, float>(t, ij, dev) : upload_advtab<NN, double>(t, ij, dev);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

size_t advect_lds_per_cell(int n, bool fp32)
{
  switch (n) {
#define SFK_CASE(NN) \
  case NN: return fp32 ? advect_lds_per_cell_n<NN, float>(0) : advect_lds_per_cell_n<NN, double>(0);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return size_t(2 * n * n * n + 6 * n * n) * (fp32 ? 4 : 8);
  }
}

hipError_t launch_advect(const AdvectLaunch &L, hipStream_t s)
{
  return L.fp32 ? dispatch_advect<float>(L, s) : dispatch_advect<double>(L, s);
}

} // namespace sfk
