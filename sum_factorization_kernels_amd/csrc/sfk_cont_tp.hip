// Continuous Q_p Laplacian on an affine Cartesian mesh with a constant
// coefficient, evaluated as a sum of Kronecker products of the assembled
// 1D element matrices (tensor-product form).
//
// With Gauss quadrature of p+1 points per direction the element mass and
// stiffness matrices of the GLL-Lagrange basis are integrated exactly, so
// the cell operator of legacy/include/evaluation_cell_laplacian.h:264-503
// (value sweeps, collocation gradient, q-point operator G = diag(JxW J_d^2),
// transposed sweeps) equals
//   A_cell = c_x K (x) M (x) M + c_y M (x) K (x) M + c_z M (x) M (x) K,
//   M_ij = sum_q w_q phi_i(x_q) phi_j(x_q),  K_ij = sum_q w_q phi_i'(x_q) phi_j'(x_q),
//   c_d = JxW J_d^2 (the same constants as the cell kernel's cdiag),
// and on a structured grid of cells the assembled operator is the same sum
// with the assembled (banded) 1D matrices M^G, K^G in place of M, K.  The
// kernel applies it direction by direction on the global node grid,
//   a = M_y u,  b = c_y K_y u;   c = M_x a,  d = M_x b + c_x K_x a;
//   A u = M_z d + c_z K_z c,
// so nodes shared by cells are summed inside each 1D sweep: no scatter,
// colouring or atomics.  Every 1D sweep is the even-odd contraction of an
// element line (eo_apply) plus, for the element's first node (shared with
// the element before it), the last row of the element matrix applied to the
// element before: outputs of a line are its nodes 0..p-1.  Results equal the
// quadrature form up to rounding (the test suite pins both against the
// oracle at 1e-12).  Dirichlet nodes are 0 on input and output.
//
// A workgroup owns a tile of TX x TY nodes (BX x BY cells) in x/y and marches
// through a range of cells in z, one layer (p node planes) at a time:
//   phase Y  y lines of the input from HBM (lanes on consecutive x:
//            coalesced), for the tile's rows and a halo of p+1 columns (the x
//            sweep needs the cell before the tile and the tile's last node)
//            -> a, b in LDS;
//   phase X  x lines of a, b from LDS -> registers -> c, d over a, b;
//   phase Z  one thread per node column: z line of c, d (the layer's first
//            plane kept in registers from the layer before), z sweep, stores
//            of the p finished planes (coalesced); the sum for the shared
//            plane is carried in a register to the next layer.
// A z range that starts above z = 0 first rebuilds the carried state from the
// cell below (one plane, then one layer without stores).  Optionally the
// Chebyshev update of do_cheby_iter<true> (evaluation_dg_laplacian.h:485-502)
// is fused into phase Z: the assembled value of a node is final there, and all
// its streams are coalesced.
//
// What bounds it, and why it is built this way (Q6 64^3 FP64 unless stated;
// 913 MB of vectors, 160-190 us at the rate of a plain copy):
// * c, d overwrite a, b (four barriers per layer instead of two): half the
//   LDS, so two or more workgroups share a CU and one computes while another
//   waits.  With four arrays one workgroup of 13 waves ran per CU.
// * Every load and store of the layer loop is an unconditional buffer access;
//   lanes without work carry an offset beyond the buffer, which reads 0 and
//   stores nothing.  Loads and stores share one completion counter, and from
//   divergent branches the compiler could only wait for all of them: every
//   layer then waited for its own stores to reach memory.  Now the wait for
//   the y lines counts past the stores issued after them.  It also makes
//   Dirichlet rows, tile edges and the y boundary one code path.
// * Idle threads repeat the last work item instead of being masked, and row
//   and plane strides are re-derived at each use: 536 instead of about 900
//   instructions per layer and thread, 20 instead of 60 of them scalar spills.
// * The row pitch is 1 modulo the banks and items run over the rows of one
//   cell, then its x neighbours, so the lanes of an LDS pass of phase X fall
//   on consecutive banks (conflicts 0.21 -> 0.05 of the LDS cycles).
// * The fused forms keep the input values of phase Y in a third LDS array for
//   phase Z instead of reading them again: with 10 MB of streams per layer in
//   flight on an XCD the second read missed its 4 MB L2 (29 % more HBM reads).
// Measured before -> after: matvec FP64 282 -> 264 us (3.5 TB/s; 3.9 TB/s with
// the halo), FP32 172 -> 127 us; three-term Chebyshev step FP64 675 -> 443 us
// (4.1 TB/s), FP32 358 -> 244 us; Q3 101x107x100 FP32 96 -> 58 us.
#include <cmath>
#include <type_traits>

#include "sfk_device.h"
#include "sfk_kernels.h"


namespace sfk {

// tables of the tensor-product operator (device memory, read through the
// constant address space like DevTab)
template <int N, typename T>
struct TpTab {
  Eo<N, T> M;    // element mass
  Eo<N, T> K[3]; // c_d K, d = x, y, z
  T mrow[N];     // last row of M
  T krow[3][N];  // last row of c_d K
  // diagonals of the assembled 1D matrices at local node index i (i = 0: a
  // vertex shared by two cells): the operator's diagonal at node (i, j, k)
  // is dk[0][i] dm[j] dm[k] + dm[i] dk[1][j] dm[k] + dm[i] dm[j] dk[2][k]
  T dm[N];
  T dk[3][N];
};

template <int N, typename T>
__device__ __forceinline__ const SFK_CONST_AS TpTab<N, T> &tptab(const void *p)
{
  return *(const SFK_CONST_AS TpTab<N, T> *)opaque_ptr(p);
}

constexpr int round64(int v) { return (v + 63) / 64 * 64; }

template <int N, typename T, int BX, int BY>
struct TpCfg {
  static constexpr int p = N - 1;
  static constexpr int TX = BX * p, TY = BY * p;
  static constexpr int HX = TX + p + 1;   // columns of phase Y (halo of p before, 1 after)
  static constexpr int NYI = p * BY * HX; // work items of phase Y (p planes): the most of all phases
  static constexpr int NXI = p * TY * BX; // phase X
  static constexpr int NZI = TX * TY;     // phase Z (node columns)
  static constexpr int THREADS = round64(NYI);
  static_assert(THREADS <= 1024, "one phase-Y item per thread");
  // LDS banks in units of T (32 banks of 4 bytes): a row pitch of 1 modulo
  // the banks puts the p rows of a cell, and with them the rows of its x
  // neighbours (p further), on consecutive banks; the plane pitch continues
  // that sequence from one plane to the next when BY = 1
  static constexpr int LW = 128 / (int)sizeof(T);
  static constexpr int RPA = (HX - 2) / LW * LW + LW + 1;
  static constexpr int PSA = TY * RPA + ((p * BX - TY * RPA) % LW + LW) % LW;
  static constexpr int LA = p * PSA;      // one of a, b (c, d)
  // input values at the nodes (fused forms), one spare column per row
  static constexpr int RPU = (TX + 1) | 1;
  static constexpr int PSU = TY * RPU;
  static constexpr int LU = p * PSU;
  static constexpr int lds_values(bool fused) { return 2 * LA + (fused ? LU : 0); }
};

// The next layer's y lines are loaded before phase X of the current one where
// the registers allow it; without that prefetch the matvec needs 28 registers
// less (FP64), which from degree 7 on decides whether two workgroups fit a CU.
// The fused forms hold their streams instead (Q6 64^3 FP64 Chebyshev step: 457
// us without, 502 us with it).
template <int N, typename T, int CHEBY>
constexpr bool tp_prefetch()
{
  return CHEBY == 0 && (sizeof(T) == 4 || N <= 7);
}
// The fused forms' streams (rhs, previous iterate, ...) are loaded before
// phase X (hidden behind it) or, where that would spill, at the start of
// phase Z (FP64 from degree 7; the six-stream form in FP64).
template <int N, typename T, int CHEBY>
constexpr bool tp_streams_early()
{
  return sizeof(T) == 4 || (N <= 7 && CHEBY != 1);
}
// Waves per SIMD asked of the compiler.  FP64 up to degree 6: 4 (128
// registers), i.e. two workgroups of 8 waves or four of 4 waves per CU; asking
// for 5 or 6 spilled (Q6 matvec 264 -> 312 us).  Degrees 7 and 8 hold 4 only
// in the matvec's 8-wave tiles (Chebyshev step of Q7 46x44x45: 301 us at 3,
// 310 us at 4 with spills).  FP32 needs at most 95 registers by itself.
template <int N, typename T, int CHEBY, int THREADS>
constexpr int tp_waves()
{
  if (sizeof(T) == 4) return 1;
  if (N <= 7) return 4;
  return (CHEBY == 0 || CHEBY == 5) && THREADS > 256 ? 4 : 3;
}

template <typename T>
struct TpArgs {
  const void *tab;
  const T *src;
  T *dst;
  const T *rhs, *diag; // fused Chebyshev
  T *tm;
  const T *prev;       // three-term Chebyshev: the previous iterate (or null: zero)
  T c_np, c_tm;
  // three-term Chebyshev, CHEBY 3 / 4: the input / the previous iterate is
  // the first iterate s_rhs D^{-1} rhs, formed in the kernel from rhs
  // instead of read (CHEBY 3: src points to rhs)
  T s_rhs;
  double *dot_part;  // CHEBY 5: src . dst summed over the grid (grid_sums) into dot_out
  unsigned *dot_ticket;
  double *dot_out;
  int nx, ny, nz;    // cells
  int gx, gy, gz;    // nodes
  int ntx, nty;      // tiles per direction
  int zc;            // cells in z per workgroup
  int order;         // block order (logical_block)
  long long vstride; // elements between right-hand sides
};

// element line with the shared first node: in[0..2p] = values at nodes
// e p - p .. e p + p; out[i] = (A u_e)[i] + (i == 0 ? (A u_{e-1})[p] : 0),
// i < p, for A = M (W = 0) or c_d K (W = 1 + d).  The table pointer is
// re-derived here and a scheduling barrier closes the contraction, so each
// matrix lives in scalar registers only while it is used (held for a whole
// phase, the tables of two matrices and their rows exceed the SGPR file).
template <int N, typename T, int W>
__device__ __forceinline__ void line_one(const void *tab, const T (&in)[2 * N - 1], T (&o)[N - 1])
{
  constexpr int p = N - 1;
  const auto &tb = tptab<N, T>(tab);
  const auto &E = W == 0 ? tb.M : tb.K[W > 0 ? W - 1 : 0];
  const auto &R = W == 0 ? tb.mrow : tb.krow[W > 0 ? W - 1 : 0];
  T ue[N], r[N];
#pragma unroll
  for (int i = 0; i < N; ++i) ue[i] = in[p + i];
  eo_apply<N, 1>(E, ue, r);
  T v = R[0] * in[0];
#pragma unroll
  for (int j = 1; j < N; ++j) v = R[j] * in[j] + v;
  o[0] = r[0] + v;
#pragma unroll
  for (int i = 1; i < p; ++i) o[i] = r[i];
  __builtin_amdgcn_sched_barrier(0);
}


// the same value, unknown to the compiler: keeps multiples of a stride from
// being hoisted out of the layer loop into scalar registers it then spills
__device__ __forceinline__ unsigned opaque_s(unsigned v)
{
  __asm__ volatile("" : "+s"(v));
  return v;
}

// CHEBY: 0 matvec; 1 the Chebyshev step of do_cheby_iter<true>
// (evaluation_dg_laplacian.h:485-502): tm = c_tm tm + c_np diag (A u - rhs),
// dst = u - tm; 2 the same recurrence in three-term form with the
// operator's own inverse diagonal (solver smoother): with tm = prev - u,
// dst = u - c_tm (prev - u) - c_np D^{-1} (A u - rhs), four streams instead
// of six, and dst may be prev (each node is read, then written, by one
// thread); 3 and 4 the three-term step whose input (3) or previous iterate
// (4) is the first iterate s_rhs D^{-1} rhs, formed from rhs in the kernel;
// 5 the matvec with the workgroup's partial sum of src . dst
template <int N, typename T, int BX, int BY, int CHEBY>
__global__ void __launch_bounds__((TpCfg<N, T, BX, BY>::THREADS))
__attribute__((amdgpu_waves_per_eu(tp_waves<N, T, CHEBY, TpCfg<N, T, BX, BY>::THREADS>(), 8)))
cont_tp_kernel(const TpArgs<T> a)
{
  using C = TpCfg<N, T, BX, BY>;
  constexpr int p = N - 1, TX = C::TX, TY = C::TY, HX = C::HX, RPA = C::RPA, PSA = C::PSA, ES = (int)sizeof(T);
  // three-term form (2, 3, 4); 3: the input, 4: the previous iterate is
  // s_rhs D^{-1} rhs (the first iterate, never stored)
  constexpr bool TT = CHEBY >= 2 && CHEBY <= 4, RSRC = CHEBY == 3, RPREV = CHEBY == 4, DOT = CHEBY == 5;
  constexpr bool FUSED = CHEBY != 0; // phase Z needs the input at its nodes
  // the Dirichlet nodes beyond a tile's end: the update's loads of a layer's
  // planes in flight together, from where there are planes enough (Q1 FP32 with it
  // 8 % slower; the matvec has nothing to load, and the code cost it up to 8 %)
  constexpr bool TOGETHER = CHEBY == 1 ? N > 2 : TT && N > 3;
  constexpr bool PF = tp_prefetch<N, T, CHEBY>(), EARLY = tp_streams_early<N, T, CHEBY>();
  T *sA = dyn_lds<T>(); // a, then c; b, then d follow at C::LA
  T *sU = sA + 2 * C::LA;

  const unsigned L = logical_block(blockIdx.x, gridDim.x, a.order);
  const int tx = (int)(L % (unsigned)a.ntx);
  const unsigned r0 = L / (unsigned)a.ntx;
  const int ty = (int)(r0 % (unsigned)a.nty);
  const int chunk = (int)(r0 / (unsigned)a.nty);
  const int ex0 = tx * BX, ey0 = ty * BY;
  const int x0 = ex0 * p, y0 = ey0 * p;
  const int ez_begin = chunk * a.zc;
  const int ez_end = ez_begin + a.zc < a.nz ? ez_begin + a.zc : a.nz;
  const int gx = a.gx, gy = a.gy, gz = a.gz;
  // (the host checks that the p+1 planes of a layer hold less than 2^31 bytes)
  const int plane = gx * gy;
  const unsigned plane_bytes = (unsigned)plane * ES, row_bytes = (unsigned)gx * ES;
  const long long layer_size = (long long)p * plane;
  const T *src = a.src + (long long)blockIdx.y * a.vstride;
  T *dst = a.dst + (long long)blockIdx.y * a.vstride;
  const int it = threadIdx.x;

  // ---- phase Y: this thread's y line (tp_line); the grid's last plane (ys =
  // p-1 of the last layer) is Dirichlet
  TpLine o;
  unsigned top_plane;
  int ys;
  T *ya, *yu = nullptr;
  T dxz = T(0), exz = T(0), dxz0 = T(0), exz0 = T(0);
  {
    const int i = it < C::NYI ? it : C::NYI - 1; // idle threads repeat the last item
    const int xh = i % HX, rest = i / HX, eyl = rest % BY;
    ys = rest / BY;
    const int ey = ey0 + eyl, X = x0 - p + xh;
    o = tp_line(p, ES, gx, a.ny, plane, ys, ey, X);
    top_plane = ys == p - 1 ? kOob : 0u;
    ya = sA + ys * PSA + eyl * p * RPA + xh;
    if constexpr (FUSED) {
      // halo columns share the spare slot after the tile's last column
      const int xu = xh >= p && xh < p + TX ? xh - p : TX;
      yu = sU + ys * C::PSU + eyl * p * C::RPU + xu;
    }
    if constexpr (RSRC) {
      // x/z factors of the line's diagonal: D = dxz dm[j % p] + exz dk_y[j % p]
      // at its row j (row j of a line is node j % p of its cell; index 0 is
      // the shared vertex)
      const auto &tb = tptab<N, T>(a.tab);
      const int jx = xh % p, jz = (ys + 1) % p;
      dxz = tb.dk[0][jx] * tb.dm[jz] + tb.dm[jx] * tb.dk[2][jz];
      exz = tb.dm[jx] * tb.dm[jz];
      dxz0 = tb.dk[0][jx] * tb.dm[0] + tb.dm[jx] * tb.dk[2][0]; // in a layer's plane 0
      exz0 = tb.dm[jx] * tb.dm[0];
    }
  }
  T u[2 * N - 1];
  auto load_lines = [&](const T *base, unsigned bytes, unsigned v0, unsigned v1, unsigned vm, unsigned vl) {
    const Rsrc r = make_rsrc(base, bytes);
    const unsigned rb = opaque_s(row_bytes);
#pragma unroll
    for (int j = 0; j < 2 * N - 1; ++j)
      u[j] = buf_load<T>(r, j == 0 ? v0 : (j <= p ? v1 : (j < 2 * p ? vm : vl)), (unsigned)j * rb);
  };
  // (live false: nothing is read, the loads only keep the loop uniform)
  auto load_y = [&](int ez, bool live) {
    const unsigned m = ez == a.nz - 1 ? top_plane : 0u;
    load_lines(src + ((long long)ez * layer_size + tp_line_base(p, gx, plane)), live ? kAll : 0u, o.first | m, o.low | m,
               o.mid | m, o.last | m);
  };
  auto phase_y = [&](bool plane0) {
    T un[FUSED ? p : 1]; // the input (RSRC: the right-hand side) at the line's own nodes
    if constexpr (FUSED)
#pragma unroll
      for (int i = 0; i < p; ++i) un[i] = u[p + i];
    if constexpr (RSRC) {
      const auto &tb = tptab<N, T>(a.tab);
#pragma unroll
      for (int j = 0; j < 2 * N - 1; ++j)
        u[j] *= a.s_rhs / ((plane0 ? dxz0 : dxz) * tb.dm[j % p] + (plane0 ? exz0 : exz) * tb.dk[1][j % p]);
    }
    T va[N - 1], vb[N - 1];
    line_one<N, T, 0>(a.tab, u, va); // a = M_y u
    line_one<N, T, 2>(a.tab, u, vb); // b = c_y K_y u
    __syncthreads();                 // phase Z of the layer before has read c, d
#pragma unroll
    for (int i = 0; i < p; ++i) {
      ya[i * RPA] = va[i];
      ya[C::LA + i * RPA] = vb[i];
    }
    if constexpr (FUSED)
#pragma unroll
      for (int i = 0; i < p; ++i) yu[i * C::RPU] = un[i];
    __syncthreads();
  };

  // ---- phase X: rows of one cell run fastest over the threads, then its x
  // neighbours, the rows of the next cells in y, the planes
  T *xa;
  {
    const int i = it < C::NXI ? it : C::NXI - 1;
    const int yi = i % p, r1 = i / p, exl = r1 % BX, r2 = r1 / BX, eyl = r2 % BY, xs = r2 / BY;
    xa = sA + xs * PSA + (eyl * p + yi) * RPA + exl * p;
  }
  auto phase_x = [&]() {
    // c = M a;  d = M b + c_x K a, one input line at a time (registers)
    T cm[N - 1], dm[N - 1], ck[N - 1];
    T ua[2 * N - 1];
#pragma unroll
    for (int j = 0; j < 2 * N - 1; ++j) ua[j] = xa[j];
    line_one<N, T, 0>(a.tab, ua, cm);
    line_one<N, T, 1>(a.tab, ua, ck);
    T ub[2 * N - 1];
#pragma unroll
    for (int j = 0; j < 2 * N - 1; ++j) ub[j] = xa[C::LA + j];
    line_one<N, T, 0>(a.tab, ub, dm);
#pragma unroll
    for (int i = 0; i < p; ++i) dm[i] += ck[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < p; ++i) {
      xa[i] = cm[i];
      xa[C::LA + i] = dm[i];
    }
    __syncthreads();
  };

  // ---- phase Z: this thread's node column
  const int zt = it < C::NZI ? it : C::NZI - 1;
  const int Xt = zt % TX, Yt = zt / TX;
  const int X = x0 + Xt, Y = y0 + Yt;
  const bool has = it < C::NZI && X < gx && Y < gy; // the thread stores this column
  const bool inner = has && X > 0 && X < gx - 1 && Y > 0 && Y < gy - 1;
  // the tile ends exactly at the last (Dirichlet) node: its zeros are
  // written by the threads of the nodes before it
  const bool xtra_x = has && Xt == TX - 1 && X + 1 == gx - 1;
  const bool xtra_y = has && Yt == TY - 1 && Y + 1 == gy - 1;
  const bool xtra = xtra_x || xtra_y;
  const unsigned coff = has ? (unsigned)((Y * gx + X) * ES) : kOob;
  const T *za = sA + Yt * RPA + Xt, *zu = sU + Yt * C::RPU + Xt;
  T cp = T(0), dp = T(0), yp = T(0), up = T(0); // carried: c, d, the shared plane's sum, the input
  double dot_acc = 0.;
  // streams of the fused forms at this column, plane k of the layer
  constexpr int NCH = CHEBY == 1 || TT ? p : 1;
  T q_r[NCH], q_d[CHEBY == 1 ? NCH : 1], q_t[NCH];
  auto load_streams = [&](int ez) {
    const long long zb = (long long)ez * layer_size;
    const unsigned pb = opaque_s(plane_bytes);
    if constexpr (CHEBY == 1 || (TT && !RSRC)) {
      const Rsrc r = make_rsrc(a.rhs + zb);
#pragma unroll
      for (int k = 0; k < p; ++k) q_r[k] = buf_load<T>(r, coff, k * pb);
    }
    if constexpr (CHEBY == 1) {
      // c_tm == 0: tm is not read
      const Rsrc rd = make_rsrc(a.diag + zb), rt = make_rsrc(a.tm + zb, a.c_tm != T(0) ? kAll : 0u);
#pragma unroll
      for (int k = 0; k < p; ++k) q_d[k] = buf_load<T>(rd, coff, k * pb);
#pragma unroll
      for (int k = 0; k < p; ++k) q_t[k] = buf_load<T>(rt, coff, k * pb);
    }
    if constexpr (TT && !RSRC && !RPREV) {
      // no previous iterate: the zero vector
      const Rsrc r = make_rsrc(a.prev ? a.prev + zb : src, a.prev ? kAll : 0u);
#pragma unroll
      for (int k = 0; k < p; ++k) q_t[k] = buf_load<T>(r, coff, k * pb);
    }
  };
  // three-term form: the inverse diagonal of this node column in plane k of a
  // cell, D = d1 dm[k] + d2 dk[2][k] with the x/y factors d1, d2 of the
  // column (0 off the interior columns); the same in every layer, so formed
  // once
  T dinvk[TT ? p : 1];
  if constexpr (TT) {
    const auto &tb = tptab<N, T>(a.tab);
    const int ix = inner ? X % p : 0, iy = inner ? Y % p : 0;
    const T d1 = tb.dk[0][ix] * tb.dm[iy] + tb.dm[ix] * tb.dk[1][iy];
    const T d2 = tb.dm[ix] * tb.dm[iy];
#pragma unroll
    for (int k = 0; k < p; ++k) dinvk[k] = inner ? T(1) / (d1 * tb.dm[k] + d2 * tb.dk[2][k]) : T(0);
  }
  // Dirichlet node at element g outside the layer loop's columns and planes
  // (A u = 0 there; three-term form: the inverse diagonal is 0 too, and a
  // first iterate formed from rhs is 0)
  auto put_zero = [&](int Z, unsigned off) {
    const long long g = (long long)Z * plane + off / ES;
    if constexpr (TT) {
      const T us = RSRC ? T(0) : src[g];
      const T pv = !RSRC && !RPREV && a.prev ? a.prev[g] : T(0);
      dst[g] = us - a.c_tm * (pv - us);
    } else if constexpr (CHEBY == 1) {
      const T t = (a.c_tm != T(0) ? a.c_tm * a.tm[g] : T(0)) + a.c_np * a.diag[g] * (T(0) - a.rhs[g]);
      a.tm[g] = t;
      dst[g] = src[g] - t;
    } else {
      dst[g] = T(0);
    }
  };
  // the same in the p planes of a layer (kOob: none)
  auto put_zeros = [&](int ez, unsigned off) {
    const long long zb = (long long)ez * layer_size;
    const unsigned pb = opaque_s(plane_bytes);
    const Rsrc rd = make_rsrc(dst + zb), rt = make_rsrc(CHEBY == 1 ? a.tm + zb : dst);
    T s[FUSED && !DOT && !RSRC ? p : 1], r[CHEBY == 1 ? p : 1], d[CHEBY == 1 ? p : 1], t[CHEBY == 1 || TT ? p : 1];
    if constexpr (CHEBY == 1 || (TT && !RSRC)) {
      const Rsrc rs = make_rsrc(src + zb);
#pragma unroll
      for (int k = 0; k < p; ++k) s[k] = buf_load<T>(rs, off, k * pb);
    }
    if constexpr (CHEBY == 1) {
      const Rsrc rr = make_rsrc(a.rhs + zb), rg = make_rsrc(a.diag + zb), rm = make_rsrc(a.tm + zb, a.c_tm != T(0) ? kAll : 0u);
#pragma unroll
      for (int k = 0; k < p; ++k) {
        r[k] = buf_load<T>(rr, off, k * pb);
        d[k] = buf_load<T>(rg, off, k * pb);
        t[k] = buf_load<T>(rm, off, k * pb);
      }
    }
    if constexpr (TT && !RSRC && !RPREV) {
      const Rsrc rp = make_rsrc(a.prev ? a.prev + zb : src, a.prev ? kAll : 0u);
#pragma unroll
      for (int k = 0; k < p; ++k) t[k] = buf_load<T>(rp, off, k * pb);
    }
#pragma unroll
    for (int k = 0; k < p; ++k) {
      if constexpr (TT) {
        const T us = RSRC ? T(0) : s[RSRC ? 0 : k];
        const T pv = RSRC || RPREV ? T(0) : t[k];
        buf_store<0>(rd, off, k * pb, us - a.c_tm * (pv - us));
      } else if constexpr (CHEBY == 1) {
        const T tn = (a.c_tm != T(0) ? a.c_tm * t[k] : T(0)) + a.c_np * d[k] * (T(0) - r[k]);
        buf_store<0>(rt, off, k * pb, tn);
        buf_store<0>(rd, off, k * pb, s[k] - tn);
      } else {
        buf_store<0>(rd, off, k * pb, T(0));
      }
    }
  };
  auto put_xtra = [&](int Z) {
    if (xtra_x) put_zero(Z, coff + ES);
    if (xtra_y) put_zero(Z, coff + row_bytes);
    if (xtra_x && xtra_y) put_zero(Z, coff + row_bytes + ES);
  };
  auto phase_z = [&](int ez, bool store) {
    if (!EARLY && store) load_streams(ez);
    T c[N], d[N], o[N], us[FUSED ? N : 1];
    c[0] = cp;
    d[0] = dp;
#pragma unroll
    for (int k = 1; k < N; ++k) {
      c[k] = za[(k - 1) * PSA];
      d[k] = za[C::LA + (k - 1) * PSA];
    }
    if constexpr (FUSED) {
      us[0] = up;
#pragma unroll
      for (int k = 1; k < N; ++k) us[k] = zu[(k - 1) * C::PSU];
      up = us[p];
    }
    T om[N], ok[N];
    eo_apply<N, 1>(tptab<N, T>(a.tab).M, d, om);
    __builtin_amdgcn_sched_barrier(0);
    eo_apply<N, 1>(tptab<N, T>(a.tab).K[2], c, ok);
#pragma unroll
    for (int k = 0; k < N; ++k) o[k] = om[k] + ok[k];
    o[0] += yp;
    cp = c[p];
    dp = d[p];
    yp = o[p];
    if (!store) return;
    const long long zb = (long long)ez * layer_size;
    if constexpr (FUSED && !DOT) {
      // Dirichlet columns: phase Y took 0 for their values, the update takes
      // what the vector holds
      if (has && !inner) {
#pragma unroll
        for (int k = 0; k < p; ++k) us[k] = src[zb + (long long)k * plane + coff / ES];
      }
    }
    const unsigned pb = opaque_s(plane_bytes);
    const Rsrc rd = make_rsrc(dst + zb), rt = make_rsrc(CHEBY == 1 ? a.tm + zb : dst);
#pragma unroll
    for (int k = 0; k < p; ++k) {
      const bool above = k > 0 || ez > 0; // not the grid's first plane
      const T v = inner && above ? o[k] : T(0);
      if constexpr (TT) {
        const T dinv = above ? dinvk[k] : T(0);
        const T rhs = RSRC ? us[k] : q_r[k];
        const T z1 = a.s_rhs * dinv * rhs; // the first iterate, when formed here
        const T ui = RSRC ? z1 : us[k];
        const T pv = RPREV ? z1 : (RSRC ? T(0) : q_t[k]);
        const T t = a.c_tm * (pv - ui) + a.c_np * dinv * (v - rhs);
        buf_store<0>(rd, coff, k * pb, ui - t);
      } else if constexpr (CHEBY == 1) {
        const T res = v - q_r[k];
        const T t = (a.c_tm != T(0) ? a.c_tm * q_t[k] : T(0)) + a.c_np * q_d[k] * res;
        buf_store<0>(rt, coff, k * pb, t);
        buf_store<0>(rd, coff, k * pb, us[k] - t);
      } else {
        buf_store<1>(rd, coff, k * pb, v);
        if constexpr (DOT) dot_acc += double(us[k]) * double(v);
      }
    }
    // the grid's last column, row and corner.  With an update, the layer's planes
    // together, so that its loads are in flight together.  One plane after another,
    // each waited for its own, every layer of a tile at the grid's end took p
    // more round trips to memory: six-stream Chebyshev step Q6 15x13x12 FP32 15.6
    // -> 10.9 us, Q3 84x72x73 FP32 156 -> 96, Q7 36x31x31 FP64 333 -> 247
    if (xtra) {
      if constexpr (TOGETHER) {
#pragma unroll 1
        for (int e = 0; e < 3; ++e) {
          const unsigned off = e == 0   ? (xtra_x ? coff + ES : kOob)
                               : e == 1 ? (xtra_y ? coff + row_bytes : kOob)
                                        : (xtra_x && xtra_y ? coff + row_bytes + ES : kOob);
          put_zeros(ez, off);
        }
      } else {
#pragma unroll 1
        for (int k = 0; k < p; ++k) put_xtra(ez * p + k);
      }
    }
  };

  // one layer; next: the layer to prefetch (ez itself: none)
  auto layer = [&](int ez, bool store, int next) {
    if (!PF) load_y(ez, true);
    phase_y(false);
    if (PF) load_y(next, next > ez);
    if (EARLY && store) load_streams(ez);
    phase_x();
    phase_z(ez, store);
  };
  if (ez_begin > 0) {
    // carried state at plane ez_begin p: c, d of the plane below the cell
    // below (slot 0; zero at the grid's first plane), then that cell's layer
    // without stores
    const int e0 = ez_begin - 1;
    const bool on = ys == 0 && e0 > 0;
    auto below = [&](unsigned v) { return on ? v : kOob; };
    load_lines(src + ((long long)e0 * layer_size + tp_line_base(p, gx, 0)), kAll, below(o.first), below(o.low),
               below(o.mid), below(o.last));
    phase_y(true);
    if (PF) load_y(e0, true);
    phase_x();
    cp = za[0];
    dp = za[C::LA];
    if constexpr (FUSED) up = zu[0];
    layer(e0, false, ez_begin);
  } else {
    if (PF) load_y(ez_begin, true);
    if constexpr (FUSED && !DOT) up = has ? src[coff / ES] : T(0); // the first plane (Dirichlet)
  }
  // (vmcnt(0): entering the loop with no access pending, so that the wait
  // for a layer's y lines inside it counts only what the loop issued)
  __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll 1
  for (int ez = ez_begin; ez < ez_end; ++ez) layer(ez, true, ez + 1 < ez_end ? ez + 1 : ez);
  // the grid's last z plane (Dirichlet)
  if (ez_end == a.nz && has) {
    put_zero(gz - 1, coff);
    put_xtra(gz - 1);
  }
  if constexpr (DOT) {
    // workgroup sum of this thread's src . dst terms: within each wave by
    // lane exchanges, then over the waves through LDS (free after the march)
    double v = dot_acc;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    double *red = reinterpret_cast<double *>(sA);
    const int wave = threadIdx.x / 64, nw = C::THREADS / 64;
    if (threadIdx.x % 64 == 0) red[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      v = 0.;
      for (int w = 0; w < nw; ++w) v += red[w];
    }
    double sum[1] = {v};
    if (grid_sums<1, C::THREADS>(sum, a.dot_part, a.dot_ticket, blockIdx.y * gridDim.x + blockIdx.x,
                                 gridDim.x * gridDim.y, red))
      *a.dot_out = sum[0];
  }
}

// ------------------------------------------------------------------ host

template <int N, typename T>
static TpTab<N, T> make_tptab(const Tables1D &t, const double inv_jac[3])
{
  // element matrices on [0,1] from the basis values S[i][q] and the basis
  // derivatives G = S D at the Gauss points
  std::vector<double> M(N * N, 0.), K(N * N, 0.), G(N * N, 0.);
  for (int i = 0; i < N; ++i)
    for (int q = 0; q < N; ++q) {
      double g = 0.;
      for (int m = 0; m < N; ++m) g += t.S[i * N + m] * t.D[m * N + q];
      G[i * N + q] = g;
    }
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j) {
      double m = 0., k = 0.;
      for (int q = 0; q < N; ++q) {
        m += t.weights[q] * t.S[i * N + q] * t.S[j * N + q];
        k += t.weights[q] * G[i * N + q] * G[j * N + q];
      }
      M[i * N + j] = m;
      K[i * N + j] = k;
    }
  // symmetrize (exact in exact arithmetic) and impose the centro-symmetry
  // the even-odd form relies on
  auto sym = [&](std::vector<double> &A) {
    std::vector<double> B(N * N);
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j)
        B[i * N + j] = 0.25 * (A[i * N + j] + A[j * N + i] + A[(N - 1 - i) * N + (N - 1 - j)] +
                               A[(N - 1 - j) * N + (N - 1 - i)]);
    A = B;
  };
  sym(M);
  sym(K);
  const double jxw = 1. / (inv_jac[0] * inv_jac[1] * inv_jac[2]);
  TpTab<N, T> tb{};
  tb.M = make_eo<N, T>(M, true);
  for (int d = 0; d < 3; ++d) {
    const double c = inv_jac[d] * inv_jac[d] * jxw;
    std::vector<double> Kd(N * N);
    for (int i = 0; i < N * N; ++i) Kd[i] = c * K[i];
    tb.K[d] = make_eo<N, T>(Kd, true);
    for (int j = 0; j < N; ++j) tb.krow[d][j] = T(Kd[(N - 1) * N + j]);
  }
  for (int j = 0; j < N; ++j) tb.mrow[j] = T(M[(N - 1) * N + j]);
  for (int i = 0; i < N; ++i) {
    // node i of a cell; i = 0 is also node p of the cell before it
    const double m = i == 0 ? M[0] + M[N * N - 1] : M[i * N + i];
    const double k = i == 0 ? K[0] + K[N * N - 1] : K[i * N + i];
    tb.dm[i] = T(m);
    for (int d = 0; d < 3; ++d) tb.dk[d][i] = T(inv_jac[d] * inv_jac[d] * jxw * k);
  }
  return tb;
}

template <int N, typename T>
static hipError_t upload_tp(const Tables1D &t, const double inv_jac[3], void **dev)
{
  const TpTab<N, T> h = make_tptab<N, T>(t, inv_jac);
  hipError_t e = hipMalloc(dev, sizeof(h));
  if (e != hipSuccess) {
    *dev = nullptr;
    return e;
  }
  e = hipMemcpy(*dev, &h, sizeof(h), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(*dev);
    *dev = nullptr;
  }
  return e;
}

hipError_t upload_tp_tables(const Tables1D &t, const double inv_jac[3], bool fp32, void **dev)
{
  switch (t.n) {
#define SFK_CASE(NN) \
  case NN: return fp32 ? upload_tp<NN, float>(t, inv_jac, dev) : upload_tp<NN, double>(t, inv_jac, dev);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

template <int N, typename T, int BX, int BY>
static hipError_t launch_tp_shape(const TpLaunch &L, hipStream_t s)
{
  using C = TpCfg<N, T, BX, BY>;
  constexpr int p = N - 1;
  TpArgs<T> a{};
  a.tab = L.tptab;
  a.src = (const T *)L.src;
  a.dst = (T *)L.dst;
  a.rhs = (const T *)L.rhs;
  a.diag = (const T *)L.diag;
  a.tm = (T *)L.tm;
  a.prev = (const T *)L.prev;
  const bool rsrc = L.cheby == 2 && L.src_from_rhs, rprev = L.cheby == 2 && L.prev_from_rhs;
  if (rsrc && rprev) return hipErrorInvalidValue;
  if (rsrc) a.src = (const T *)L.rhs;
  a.dot_part = L.dot_part;
  a.dot_ticket = L.dot_ticket;
  a.dot_out = L.dot_out;
  a.s_rhs = T(L.s_rhs);
  a.c_np = T(L.c_np);
  a.c_tm = T(L.c_tm);
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  a.gx = a.nx * p + 1;
  a.gy = a.ny * p + 1;
  a.gz = a.nz * p + 1;
  a.ntx = (a.nx + BX - 1) / BX;
  a.nty = (a.ny + BY - 1) / BY;
  a.zc = L.zc > 0 ? (L.zc < a.nz ? L.zc : a.nz) : a.nz;
  a.order = L.order;
  a.vstride = L.vstride;
  if (!tp_offsets_fit(N, a.gx, a.gy, (int)sizeof(T))) return hipErrorInvalidValue;
  const long long nchunks = (a.nz + a.zc - 1) / a.zc;
  const long long blocks = (long long)a.ntx * a.nty * nchunks;
  if (blocks <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  const size_t lds = size_t(C::lds_values(L.cheby != 0 || L.dot_part)) * sizeof(T);
  // the matvec with src . dst (CHEBY 5) exists for FP64 only (the solver's
  // outer matvec)
  decltype(&cont_tp_kernel<N, T, BX, BY, 0>) kdot = nullptr;
  if constexpr (std::is_same<T, double>::value) kdot = cont_tp_kernel<N, T, BX, BY, 5>;
  if (L.dot_part && (L.cheby != 0 || L.nrhs != 1 || !kdot || !L.dot_ticket || !L.dot_out)) return hipErrorInvalidValue;
  auto kern = rsrc ? cont_tp_kernel<N, T, BX, BY, 3>
              : rprev ? cont_tp_kernel<N, T, BX, BY, 4>
              : L.dot_part ? kdot
              : L.cheby == 2 ? cont_tp_kernel<N, T, BX, BY, 2>
                            : (L.cheby == 1 ? cont_tp_kernel<N, T, BX, BY, 1> : cont_tp_kernel<N, T, BX, BY, 0>);
  hipError_t e = allow_dynamic_lds((const void *)kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, L.nrhs), dim3(C::THREADS), lds, s, a);
  return hipGetLastError();
}

// Tile shapes (BX, BY) per points per direction N, from 1 (shape 0: tp_plan
// chooses).  Wide in x (the x halo of p+1 columns costs (p+1)/(BX p)), with
// BY p BX as large as fits, and first the tiles whose phase Y fills 4 or 8 waves,
// which spread evenly over the SIMDs (Q6 52x50x52 FP64: 13 x 1 cells in 8 waves 129
// us, 7 x 1 in 5 waves 177 us, 16 x 1 in 10 waves 195 us).  From N = 6 on few
// widths do: the tiles of 5, 6 and 7 waves are there for meshes whose cells in x
// they divide better (Q6 42x36x37 FP32 six-stream step: 11 x 1 in 7 waves 86 us, 5 x
// 1 in 4 waves 88 us, 13 x 1 in 8 waves more), and Q6's 24 x 1 in 15 waves, which leaves room for two
// workgroups a CU in FP32 only, for rows that it covers with one tile less.
#define SFK_TP_SHAPES(X)                                                        \
  X(2, 1, 30, 8) X(2, 2, 126, 4) X(2, 3, 62, 4) X(2, 4, 30, 16)                  \
  X(3, 1, 30, 2) X(3, 2, 62, 2) X(3, 3, 30, 4) X(3, 4, 14, 4)                    \
  X(4, 1, 27, 1) X(4, 2, 8, 3) X(4, 3, 27, 2) X(4, 4, 12, 2)                     \
  X(5, 1, 14, 1) X(5, 2, 30, 1) X(5, 3, 9, 3) X(5, 4, 14, 2) X(5, 5, 6, 2)       \
  X(6, 1, 9, 1) X(6, 2, 19, 1) X(6, 3, 16, 1) X(6, 4, 11, 1)                     \
  X(7, 1, 13, 1) X(7, 2, 11, 1) X(7, 3, 5, 1) X(7, 4, 9, 1) X(7, 5, 24, 1) X(7, 6, 7, 1) \
  X(8, 1, 4, 1) X(8, 2, 9, 1) X(8, 3, 7, 1) X(8, 4, 4, 2)                        \
  X(9, 1, 6, 1) X(9, 2, 2, 1) X(9, 3, 4, 1) X(9, 4, 3, 1)

int tp_shape_count(int n)
{
  int c = 1;
#define SFK_X(NN, SH, BXX, BYY) c += n == NN ? 1 : 0;
  SFK_TP_SHAPES(SFK_X)
#undef SFK_X
  return c;
}

void tp_shape(int n, int shape, int *bx, int *by)
{
  *bx = *by = 0;
#define SFK_X(NN, SH, BXX, BYY) \
  if (n == NN && shape == SH) { \
    *bx = BXX;                  \
    *by = BYY;                  \
  }
  SFK_TP_SHAPES(SFK_X)
#undef SFK_X
}

// LDS of a workgroup of the matvec
static size_t tp_lds_bytes(int n, int shape, bool fp32)
{
  size_t v = 0;
#define SFK_X(NN, SH, BXX, BYY) \
  if (n == NN && shape == SH)   \
    v = fp32 ? TpCfg<NN, float, BXX, BYY>::lds_values(false) * 4 : TpCfg<NN, double, BXX, BYY>::lds_values(false) * 8;
  SFK_TP_SHAPES(SFK_X)
#undef SFK_X
  return v;
}

// a CU (lds_max bytes) holds two workgroups of the matvec: below that the
// kernel's phases have nothing to overlap with (Q6 52x50x52 FP64 on 24 x 1
// cells, one workgroup of 94 KB per CU: 196 us instead of 129 us)
bool tp_shape_fits(int n, int shape, bool fp32, size_t lds_max)
{
  return 2 * tp_lds_bytes(n, shape, fp32) <= lds_max;
}

// Modelled cost of a schedule, in work items x layers per CU.  A workgroup
// costs its items, half of them rounded up to whole sets of four waves (the
// wave that a SIMD has more than the others is waited for at every barrier),
// and more where fewer than 16 waves of a CU are there to overlap;
// its range of cells in z costs 1.2 layers more when it starts above the
// bottom and 0.6 for its start; and a CU with few workgroups still needs the
// latency of a layer, about what 500 items cost, per set of resident ones.
double tp_cost(int n, const int nc[3], int shape, int zc, const Chip &chip)
{
  int bx = 0, by = 0;
  tp_shape(n, shape, &bx, &by);
  if (bx <= 0 || zc <= 0) return 1e300;
  const int p = n - 1, items = p * by * (bx * p + p + 1), waves = (items + 63) / 64;
  const long long tiles = (long long)((nc[0] + bx - 1) / bx) * ((nc[1] + by - 1) / by);
  const long long chunks = (nc[2] + zc - 1) / zc, per_cu = (tiles * chunks + chip.cus - 1) / chip.cus;
  const long long slots = 16 / waves > 0 ? 16 / waves : 1;
  const long long resident = (per_cu < slots ? per_cu : slots) * waves;
  double work = double(per_cu) * (0.5 * items + 0.5 * 256 * ((waves + 3) / 4));
  if (resident < 16) work *= std::sqrt(16. / double(resident));
  const double latency = double((per_cu + slots - 1) / slots) * 500.;
  return (zc + (chunks > 1 ? 1.8 : 0.6)) * (work > latency ? work : latency);
}

// cells in z per workgroup worth trying: the mesh in 1, 2, 3, ... parts
std::vector<int> tp_zc_candidates(int nz)
{
  std::vector<int> v;
  for (int k : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64, 96, 128})
    if (k <= nz && (v.empty() || (nz + k - 1) / k != v.back())) v.push_back((nz + k - 1) / k);
  if (v.back() != 1) v.push_back(1);
  return v;
}

// the schedule of shape 0 and / or zc 0 (automatic): the cheapest by tp_cost.
// Untuned Q6 64^3 FP64 380 -> 266 us (the tuner finds 264).  Its weak side are
// meshes with fewer workgroups than CUs: Q4 16^3 it takes 14 x 1 tiles and 2 cells
// in z (8.1 us), the tuner 6 x 2 and 1 (7.7 us).
void tp_plan(int n, bool fp32, const int nc[3], const Chip &chip, int *shape, int *zc)
{
  if (*shape > 0 && *zc > 0) return;
  const std::vector<int> zcs = *zc > 0 ? std::vector<int>{*zc < nc[2] ? *zc : nc[2]} : tp_zc_candidates(nc[2]);
  const int s0 = *shape > 0 ? *shape : 1, s1 = *shape > 0 ? *shape : tp_shape_count(n) - 1;
  double best = -1.;
  int bs = s0, bz = zcs[0];
  // (where no tile leaves room for two workgroups: the smallest one)
  for (int sh = s0 + 1; sh <= s1; ++sh)
    if (tp_lds_bytes(n, sh, fp32) < tp_lds_bytes(n, bs, fp32)) bs = sh;
  for (int sh = s0; sh <= s1; ++sh) {
    if (*shape == 0 && !tp_shape_fits(n, sh, fp32, chip.lds)) continue;
    for (int z : zcs) {
      const double c = tp_cost(n, nc, sh, z, chip);
      if (best < 0. || c < best) {
        best = c;
        bs = sh;
        bz = z;
      }
    }
  }
  *shape = bs;
  *zc = bz;
}

template <typename T>
static hipError_t launch_tp_t(const TpLaunch &L, hipStream_t s)
{
  const int shape = L.shape;
#define SFK_X(NN, SH, BXX, BYY) \
  if (L.n == NN && shape == SH) return launch_tp_shape<NN, T, BXX, BYY>(L, s);
  SFK_TP_SHAPES(SFK_X)
#undef SFK_X
  return hipErrorInvalidValue;
}

long long tp_launch_blocks(const TpLaunch &L)
{
  int bx = 0, by = 0;
  tp_shape(L.n, L.shape, &bx, &by);
  if (bx <= 0 || by <= 0) return 0;
  const int nz = L.nc[2], zc = L.zc > 0 ? (L.zc < nz ? L.zc : nz) : nz;
  return (long long)((L.nc[0] + bx - 1) / bx) * ((L.nc[1] + by - 1) / by) * ((nz + zc - 1) / zc);
}

hipError_t launch_cont_tp(const TpLaunch &L, hipStream_t s)
{
  return L.fp32 ? launch_tp_t<float>(L, s) : launch_tp_t<double>(L, s);
}

} // namespace sfk
