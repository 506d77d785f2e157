// Cell-batched sum-factorization kernels for the Laplacian family:
//   Mode::Local  element-local Laplacian (EvaluationCellLaplacian,
//                legacy/include/evaluation_cell_laplacian.h:264-503),
//   Mode::Cont   continuous Q_p Laplacian on a structured node grid with
//                homogeneous Dirichlet rows (colored stores or atomic scatter-add),
//   Mode::DG     DG-SIPG on a Cartesian periodic mesh with the fused
//                Chebyshev update (EvaluationDGLaplacian::do_inner_loop,
//                legacy/include/evaluation_dg_laplacian.h:129-510): degrees
//                above 8 and the reference-compatible x sweep.
//
// One workgroup processes CB cells; each cell gets N*N threads.  Thread l of
// a cell owns line l of every direction (x-line (j,k), y-line (i,k), z-line
// (i,j), all with index l = hi*N + lo), so each 1D sweep is a register-
// resident even-odd contraction fed by one LDS read and one LDS write per
// point.  Phase order (barriers between phases):
//   L  global -> z-line registers, z value sweep -> LDS A;  DG: neighbour
//      face layers (value + Hermite normal derivative) -> LDS F
//   V1 x value sweep on A;  DG: face arrays, first in-plane sweep
//   V2 y value sweep on A;  DG: face arrays, second in-plane sweep
//   Gx x gradient, cell term, x-face terms, transposed gradient -> B
//   Gy same for y, B += ...
//   Gz same for z, + B, transposed z value sweep -> A
//   By transposed y value sweep
//   Bx transposed x value sweep -> global (DG: fused Chebyshev update;
//      Cont: colored stores or atomic scatter-add)
#include "sfk_device.h"
#include "sfk_kernels.h"

namespace sfk {

enum class Mode { Local = 0, Cont = 1, DG = 2 };

template <int N>
constexpr int threads_per_block()
{
  return ((full_cells(N) * N * N + 63) / 64) * 64;
}
constexpr int kCellMaxThreads = 256;
template <int N, typename T, bool FACES>
constexpr int cell_waves()
{
  constexpr int cb = full_cells(N);
  return lds_waves_per_simd(cb * (2 * N * N * N + (FACES ? 12 * N * N : 0)) * (int)sizeof(T), cb * N * N);
}

template <int N, typename T>
struct CellArgs {
  const DevTab<N, T> *dt; // tables in device memory (read through ctab)
  const T *src;
  T *dst;
  const T *rhs, *diag; // Chebyshev
  T *tm;
  T c_np, c_tm;
  const T *coef;   // coefficient times quadrature weight per cell q-point (optional)
  long long ncells;
  int nx, ny, nz;  // cells per direction
  int gx, gy, gz;  // node grid (continuous)
  T cdiag[3];      // ij_d^2 * JxW
  T ij[3];         // 1/h_d
  T jxwf[3];       // JxW of a face normal to d (without weights)
  T tau[3];        // penalty (p+1)^2 / h_d
  int nrhs;
  long long vstride; // elements between right-hand sides
  // continuous: colour of this launch and the row/segment decomposition
  // (a workgroup = CB consecutive cells of one x row; colour = parity of
  // (row y, row z, segment) so that a launch writes every node at most once)
  int color, nseg, nss, nry, nrz;
  int cb;    // cells per workgroup (continuous colored: cells per segment)
  int order; // block order (logical_block)
};

// face terms of SIPG along one line (Cartesian): the thread owns line l of
// direction DIR, q[] are the values at the Gauss points of the line; adds
// value and normal-derivative test contributions to r[] (the transposed
// gradient sweep output).  Signs as in evaluation_dg_laplacian.h:237-252.
template <int N, int DIR, typename T>
__device__ __forceinline__ void sipg_faces(const CellArgs<N, T> &a, const T (&q)[N], const T *F, int l,
                                           T (&r)[N])
{
  constexpr int N2 = N * N;
  const auto &tb = ctab(a.dt);
  T v0 = 0, v1 = 0, d0 = 0, d1 = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v0 += tb.fv0[i] * q[i];
    v1 += tb.fv1[i] * q[i];
    d0 += tb.fd0[i] * q[i];
    d1 += tb.fd1[i] * q[i];
  }
  const T up0 = F[(2 * DIR) * N2 + l], dp0 = F[(6 + 2 * DIR) * N2 + l];
  const T up1 = F[(2 * DIR + 1) * N2 + l], dp1 = F[(6 + 2 * DIR + 1) * N2 + l];
  const T wf = tb.w[l % N] * tb.w[l / N];
  const T ij = a.ij[DIR], jf = a.jxwf[DIR] * wf, tau = a.tau[DIR];
  const T jump0 = v0 - up0, jump1 = v1 - up1;
  const T tv0 = (T(0.5) * ij * (d0 + dp0) + jump0 * tau) * jf;
  const T td0 = T(0.5) * ij * jf * jump0;
  const T tv1 = (T(-0.5) * ij * (d1 + dp1) + jump1 * tau) * jf;
  const T td1 = T(-0.5) * ij * jf * jump1;
#pragma unroll
  for (int i = 0; i < N; ++i)
    r[i] += tb.fv0[i] * tv0 + tb.fd0[i] * td0 + tb.fv1[i] * tv1 + tb.fd1[i] * td1;
}

// gradient phase of one direction: read Q line, collocation derivative,
// cell term, faces, transposed derivative
template <int N, int DIR, typename T, Mode MODE, bool COEF>
__device__ __forceinline__ void grad_phase(const CellArgs<N, T> &a, const T *Acell, const T *F, int l,
                                           long long cell, T (&r)[N])
{
  const auto &tb = ctab(a.dt);
  T q[N], g[N];
  lds_read_line<N, N, DIR>(Acell, l, q);
  eo_apply<N, -1>(tb.Df, q, g);
  const T c = a.cdiag[DIR];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    T f;
    if constexpr (COEF) f = c * a.coef[cell * (N * N * N) + line_base<N, N, DIR>(l) + i * line_stride<N, N, DIR>()];
    else f = c * line_weight<N, DIR>(tb.w, l, i);
    g[i] *= f;
  }
  eo_apply<N, -1>(tb.Db, g, r);
  if constexpr (MODE == Mode::DG) sipg_faces<N, DIR, T>(a, q, F, l, r);
}

// Colored store of a continuous segment.  A workgroup owns CB consecutive
// cells of one x row (a "segment"); the units (row y, row z, segment) are
// coloured by the parity of each index, so two units of one colour share no
// node and a launch writes every node at most once.  The colours are
// launched in ascending order; for every node the unit with the smallest
// colour among those that touch it stores (Dirichlet nodes: 0) and later
// ones add, which makes a zero fill and atomics unnecessary.
//
// The segment's output is (p+1)^2 node rows of ncs*p+1 consecutive nodes
// (ncs cells).  The threads' x lines are merged into those rows in LDS (the
// first x-plane of cell c+1, left in sB by its threads, is added to the last
// x-plane of cell c), and the rows are then written with consecutive lanes
// on consecutive nodes: a store instruction covers a few cache lines
// instead of one row per lane.  Values added to are all loaded before the
// first store.  Called by every thread of the workgroup (barrier inside);
// sA (the A sweep array, dead at this point) holds the rows.
// NR right-hand sides (nr of them present) share the index arithmetic: arrays
// of right-hand side r at sA + r rs, its vector at dst + r a.vstride.
template <int N, typename T, int NR = 1>
__device__ __forceinline__ void cont_store_colored(const CellArgs<N, T> &a, T (&o)[NR][N], T *sA, const T *sB, int rs,
                                                   int nr, bool act, int c, int l, int cy, int cz, int seg, int cx0,
                                                   int cx_end, T *dst)
{
  constexpr int p = N - 1, N2 = N * N, N3 = N2 * N;
  const int ncs = cx_end - cx0, Lx = ncs * p + 1;
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (c + 1 < ncs) o[r][p] += sB[r * rs + (c + 1) * N3 + l];
      T *row = sA + r * rs + l * Lx + c * p;
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (i > 0 || c == 0) row[i] = o[r][i];
    }
  }
  // per-row terms of the segment's N2 node rows, made once per row instead
  // of once per node: the index of the row's first node, a Dirichlet-row
  // bit (4), and the y/z part of the smallest colour of the units covering
  // the row (rows [ylo,yhi] x [zlo,zhi], each range one or two entries; the
  // segment part is added per node)
  __shared__ long long s_rbase[N2];
  __shared__ int s_rflag[N2];
  if ((int)threadIdx.x < N2) {
    const int rw = (int)threadIdx.x, j = rw % N, k = rw / N;
    const int ylo = (j == 0 && cy > 0) ? cy - 1 : cy, yhi = (j == p && cy + 1 < a.ny) ? cy + 1 : cy;
    const int zlo = (k == 0 && cz > 0) ? cz - 1 : cz, zhi = (k == p && cz + 1 < a.nz) ? cz + 1 : cz;
    const int py = ylo == yhi ? (ylo & 1) : 0, pz = zlo == zhi ? (zlo & 1) : 0;
    const int Y = cy * p + j, Z = cz * p + k;
    const bool bd = Y == 0 || Z == 0 || Y == a.gy - 1 || Z == a.gz - 1;
    s_rbase[rw] = ((long long)Z * a.gy + Y) * a.gx + (long long)cx0 * p;
    s_rflag[rw] = py + 2 * pz + (bd ? 4 : 0);
  }
  __syncthreads();
  // blockDim.x >= CB (p+1)^2 and N2 (ncs p + 1) <= CB N3: N rounds cover the rows
  const int total = N2 * Lx;
  // idx / Lx as (idx * mlx) >> 20 with mlx = ceil(2^20 / Lx): exact while
  // idx * (mlx - 2^20 / Lx) < 2^20 / Lx, i.e. for idx < 2^20 / Lx, which
  // holds here (idx < N blockDim.x <= 2304, Lx <= 8 * 64 + 1)
  const unsigned mlx = ((1u << 20) + unsigned(Lx) - 1u) / unsigned(Lx);
  int mode[N]; // 0 nothing, 1 store, 2 add
  long long gi[N];
  T val[NR][N], old[NR][N];
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const int idx = (int)threadIdx.x + r * (int)blockDim.x;
    mode[r] = 0;
    gi[r] = 0;
#pragma unroll
    for (int q = 0; q < NR; ++q) val[q][r] = old[q][r] = T(0);
    if (idx < total) {
      const int rw = (int)((unsigned(idx) * mlx) >> 20), xi = idx - rw * Lx;
      const int fl = s_rflag[rw];
      int ps = seg & 1;
      if ((xi == 0 && seg > 0) || (xi == Lx - 1 && seg + 1 < a.nseg)) ps = 0;
      const int m = (fl & 3) + 4 * ps;
      const int X = cx0 * p + xi;
      const bool bd = (fl & 4) || X == 0 || X == a.gx - 1;
      gi[r] = s_rbase[rw] + xi;
#pragma unroll
      for (int q = 0; q < NR; ++q) val[q][r] = bd ? T(0) : sA[q * rs + idx];
      mode[r] = m == a.color ? 1 : (bd ? 0 : 2);
    }
  }
  // the loads in a loop of their own, so that they are all in flight
  // together (interleaved with the index arithmetic above, the compiler
  // waited for each before the next)
#pragma unroll
  for (int q = 0; q < NR; ++q)
    if (q < nr)
#pragma unroll
      for (int r = 0; r < N; ++r)
        if (mode[r] == 2) old[q][r] = dst[q * a.vstride + gi[r]];
#pragma unroll
  for (int q = 0; q < NR; ++q)
    if (q < nr)
#pragma unroll
      for (int r = 0; r < N; ++r) {
        if (mode[r] == 1) dst[q * a.vstride + gi[r]] = val[q][r];
        else if (mode[r] == 2) dst[q * a.vstride + gi[r]] = old[q][r] + val[q][r];
      }
}

// A workgroup's cells of the continuous operator: the row-segment
// decomposition of a colour >= 0, or cells in index order (atomic scatter)
struct ContPos {
  int seg, cx, cy, cz, cx0, cx_end;
  long long cell0;
  bool act;
};
template <int N, typename T>
__device__ __forceinline__ ContPos cont_position(const CellArgs<N, T> &a, unsigned blk, int c)
{
  const int CB = a.cb;
  ContPos q{};
  if (a.color >= 0) {
    const int si = (int)(blk % a.nss);
    const int rest = (int)(blk / a.nss);
    q.seg = (a.color >> 2 & 1) + 2 * si;
    q.cy = (a.color & 1) + 2 * (rest % a.nry);
    q.cz = (a.color >> 1 & 1) + 2 * (rest / a.nry);
    q.cx0 = q.seg * CB;
    q.cx_end = q.cx0 + CB < a.nx ? q.cx0 + CB : a.nx;
    q.cx = q.cx0 + c;
    q.cell0 = ((long long)q.cz * a.ny + q.cy) * a.nx + q.cx0;
    q.act = c < CB && q.cx < q.cx_end;
  } else {
    // cell0's coordinates are uniform; cell0 + c is c steps further in x
    // unless that crosses the end of the row
    q.cell0 = (long long)blk * CB;
    q.act = c < CB && q.cell0 + c < a.ncells;
    CellXYZ x = traverse_xyz((unsigned)q.cell0, a.nx, a.ny, a.nz, 0);
    if (x.x + c < (unsigned)a.nx) x.x += c;
    else x = traverse_xyz((unsigned)(q.cell0 + c), a.nx, a.ny, a.nz, 0);
    q.cx = (int)x.x;
    q.cy = (int)x.y;
    q.cz = (int)x.z;
  }
  return q;
}

template <int N, typename T, Mode MODE, bool CHEBY, bool REFX, bool COEF>
__global__ void __launch_bounds__(kCellMaxThreads) __attribute__((amdgpu_waves_per_eu(1, cell_waves<N, T, MODE == Mode::DG>())))
cell_kernel(const CellArgs<N, T> a)
{
  constexpr int N2 = N * N, N3 = N * N * N, p = N - 1;
  constexpr bool FACES = MODE == Mode::DG;
  const int CB = a.cb;
  // dynamic LDS: A [CB][N3], B [CB][N3], F [CB][12][N2] (DG only)
  T *sA = dyn_lds<T>();
  T *sB = sA + CB * N3;
  T *sF = sB + CB * N3;

  const int t = threadIdx.x;
  const int c = t / N2, l = t % N2;
  const unsigned blk = logical_block(blockIdx.x, gridDim.x, a.order);
  long long cell0 = (long long)blk * CB;
  ContPos q{};
  bool act = c < CB && cell0 + c < a.ncells;
  if constexpr (MODE == Mode::Cont) {
    q = cont_position(a, blk, c);
    cell0 = q.cell0;
    act = q.act;
  }
  // DG: the cell at this traversal position and its periodic face neighbours
  int nbr[6] = {0, 0, 0, 0, 0, 0};
  long long cell = cell0 + c;
  if constexpr (MODE == Mode::DG) {
    if (act) cell = locate_cell((unsigned)cell0, (unsigned)c, a.nx, a.ny, a.nz, a.order, nbr);
  }
  T *A = sA + (act ? c : 0) * N3;
  T *B = sB + (act ? c : 0) * N3;
  T *F = sF + (FACES && act ? c * 12 * N2 : 0);

  // right-hand side rr = blockIdx.y (a loop over the right-hand sides here
  // would keep every 1D table live across it and spill scalar registers)
  {
    const long long rr = blockIdx.y;
    const T *src = a.src + rr * a.vstride;
    T *dst = a.dst + rr * a.vstride;
    // ---------------------------------------------------------------- L
    if (act) {
      const auto &tb = ctab(a.dt);
      T u[N], v[N];
      if constexpr (MODE == Mode::Cont) {
        // (staging the segment's node rows through LDS for coalesced loads
        // measured slower: the extra barrier costs more than it saves)
        const int X = q.cx * p + l % N, Y = q.cy * p + l / N;
        const bool bxy = X == 0 || Y == 0 || X == a.gx - 1 || Y == a.gy - 1;
        const long long g0 = (long long)q.cz * p * a.gy * a.gx + (long long)Y * a.gx + X;
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const int Z = q.cz * p + k;
          const bool bd = bxy || Z == 0 || Z == a.gz - 1;
          u[k] = bd ? T(0) : src[g0 + (long long)k * a.gy * a.gx];
        }
      } else {
#pragma unroll
        for (int k = 0; k < N; ++k) u[k] = src[cell * N3 + k * N2 + l];
      }
      eo_apply<N, 1>(tb.Sf, u, v);
      lds_write_line<N, N, 2>(A, l, v);
    }
    if constexpr (FACES) {
      // neighbour layers: value layer and Hermite normal derivative
      // w0*(inner - face) (evaluation_dg_laplacian.h:196-203, 272-283);
      // thread l of a cell loads face point l of all six faces (twelve
      // independent loads, issued together)
      if (act) {
        T uf[6], ui[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
          const int d = f / 2, s = f % 2;
          const T *nb = src + (long long)nbr[f] * N3;
          const int lf = s ? 0 : p, li = s ? 1 : p - 1;
          const int of = d == 0 ? face_dof<N, 0>(lf, l) : (d == 1 ? face_dof<N, 1>(lf, l) : face_dof<N, 2>(lf, l));
          const int oi = d == 0 ? face_dof<N, 0>(li, l) : (d == 1 ? face_dof<N, 1>(li, l) : face_dof<N, 2>(li, l));
          uf[f] = nb[of];
          ui[f] = nb[oi];
        }
        const T hd = ctab(a.dt).hd;
#pragma unroll
        for (int f = 0; f < 6; ++f) {
          F[f * N2 + l] = uf[f];
          F[(6 + f) * N2 + l] = (f % 2 ? -hd : hd) * (ui[f] - uf[f]);
        }
      }
    }
    __syncthreads();
    // --------------------------------------------------------------- V1
    if (act) {
      const auto &tb = ctab(a.dt);
      T u[N], v[N];
      lds_read_line<N, N, 0>(A, l, u);
      eo_apply<N, 1>(tb.Sf, u, v);
      lds_write_line<N, N, 0>(A, l, v);
      if constexpr (FACES) {
        for (int it = l; it < 12 * N; it += N2) {
          T *fl = F + (it / N) * N2 + (it % N) * N; // lo-direction line
#pragma unroll
          for (int i = 0; i < N; ++i) u[i] = fl[i];
          eo_apply<N, 1>(tb.Sf, u, v);
#pragma unroll
          for (int i = 0; i < N; ++i) fl[i] = v[i];
        }
      }
    }
    __syncthreads();
    // --------------------------------------------------------------- V2
    if (act) {
      const auto &tb = ctab(a.dt);
      T u[N], v[N];
      lds_read_line<N, N, 1>(A, l, u);
      eo_apply<N, 1>(tb.Sf, u, v);
      lds_write_line<N, N, 1>(A, l, v);
      if constexpr (FACES) {
        for (int it = l; it < 12 * N; it += N2) {
          T *fl = F + (it / N) * N2 + (it % N); // hi-direction line
#pragma unroll
          for (int i = 0; i < N; ++i) u[i] = fl[i * N];
          eo_apply<N, 1>(tb.Sf, u, v);
#pragma unroll
          for (int i = 0; i < N; ++i) fl[i * N] = v[i];
        }
      }
    }
    __syncthreads();
    // --------------------------------------------------------------- Gx
    if (act) {
      const auto &tb = ctab(a.dt);
      T r[N];
      grad_phase<N, 0, T, MODE, COEF>(a, A, F, l, cell, r);
      lds_write_line<N, N, 0>(B, l, r);
    }
    __syncthreads();
    // --------------------------------------------------------------- Gy
    if (act) {
      const auto &tb = ctab(a.dt);
      T r[N], b[N];
      grad_phase<N, 1, T, MODE, COEF>(a, A, F, l, cell, r);
      lds_read_line<N, N, 1>(B, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      lds_write_line<N, N, 1>(B, l, r);
    }
    __syncthreads();
    // --------------------------------------------------------------- Gz
    if (act) {
      const auto &tb = ctab(a.dt);
      T r[N], b[N], o[N];
      grad_phase<N, 2, T, MODE, COEF>(a, A, F, l, cell, r);
      lds_read_line<N, N, 2>(B, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] += b[i];
      eo_apply<N, 1>(tb.Sb, r, o);
      lds_write_line<N, N, 2>(A, l, o);
    }
    __syncthreads();
    // --------------------------------------------------------------- By
    // DG Chebyshev: this thread's x line of rhs, diag, tmp and the input,
    // loaded one phase ahead of the update that uses them
    T crhs[CHEBY ? N : 1], cdiag[CHEBY ? N : 1], ctm[CHEBY ? N : 1], csrc[CHEBY ? N : 1];
    if (act) {
      if constexpr (MODE == Mode::DG && CHEBY) {
        const long long g0 = cell * N3 + l * N;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          crhs[i] = a.rhs[g0 + i];
          cdiag[i] = a.diag[g0 + i];
          ctm[i] = a.c_tm != T(0) ? a.tm[g0 + i] : T(0); // c_tm == 0: tm not read
          csrc[i] = src[g0 + i];
        }
      }
      const auto &tb = ctab(a.dt);
      T u[N], v[N];
      lds_read_line<N, N, 1>(A, l, u);
      eo_apply<N, 1>(tb.Sb, u, v);
      lds_write_line<N, N, 1>(A, l, v);
    }
    __syncthreads();
    // --------------------------------------------------------------- Bx
    T oo[1][N];
    T(&o)[N] = oo[0];
    if (act) {
      const auto &tb = ctab(a.dt);
      T u[N];
      lds_read_line<N, N, 0>(A, l, u);
      if constexpr (REFX)
        eo_apply<N, 1>(tb.Sf, u, o); // evaluation_dg_laplacian.h:481-483
      else
        eo_apply<N, 1>(tb.Sb, u, o);
      if constexpr (MODE == Mode::Cont) {
        // x-merge: the first x-plane of cell c+1 is the last one of cell c
        if (a.color >= 0) B[l] = o[0];
      }
    }
    if constexpr (MODE == Mode::Cont) {
      if (a.color >= 0) {
        __syncthreads();
        cont_store_colored<N, T>(a, oo, sA, sB, 0, 1, act, c, l, q.cy, q.cz, q.seg, q.cx0, q.cx_end, dst);
      } else if (act) {
        const int Y = q.cy * p + l % N, Z = q.cz * p + l / N;
        const bool byz = Y == 0 || Z == 0 || Y == a.gy - 1 || Z == a.gz - 1;
        const long long g0 = ((long long)Z * a.gy + Y) * a.gx + (long long)q.cx * p;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int X = q.cx * p + i;
          if (!(byz || X == 0 || X == a.gx - 1)) atomicAdd(dst + g0 + i, o[i]);
        }
      }
    }
    if (act) {
      const auto &tb = ctab(a.dt);
      if constexpr (MODE == Mode::Cont) {
      } else if constexpr (CHEBY) {
        // r = A u - rhs; tm = c_tm*tm + c_np*diag*r; dst = u - tm
        // (evaluation_dg_laplacian.h:485-502)
        const long long g0 = cell * N3 + l * N;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const long long g = g0 + i;
          const T res = o[i] - crhs[i];
          const T base = a.c_np * cdiag[i] * res;
          const T tmv = a.c_tm != T(0) ? a.c_tm * ctm[i] + base : base;
          a.tm[g] = tmv;
          dst[g] = csrc[i] - tmv;
        }
      } else {
        const long long g0 = cell * N3 + l * N;
        // written once, read by nobody in this launch: non-temporal stores
#pragma unroll
        for (int i = 0; i < N; ++i) __builtin_nontemporal_store(o[i], dst + g0 + i);
      }
    }
  }
}

// Continuous Laplacian with a coefficient per q-point, NR right-hand sides per
// workgroup.  Phases (barrier between):
//   L   z line of the input -> z value sweep -> A
//   V1  x value sweep on A
//   Gy  y value sweep -> A; y gradient, coefficient, transposed gradient -> B
//   Gx  the same for x on A, B += ...
//   Gz  the same for z, + B, transposed z value sweep -> A
//   By  transposed y value sweep on A
//   Bx  transposed x value sweep, colored stores or atomic adds
// What bounds it: VALU issue and the latency between the phases.  Two
// right-hand sides share the coefficient, the table loads, the index
// arithmetic of the colored store and the barriers; the coefficient holds the
// quadrature weight (one product per point and direction instead of four) and
// the y gradient follows its value sweep in registers (15 LDS accesses per
// point instead of 16, 7 phases instead of 8).  Measured, before -> after (all
// right-hand sides of one apply): p = 2 80x70x75, 8, FP32 401 -> 300 us; p = 4
// 40x37x42, 3, FP64 181 -> 163 us; p = 5 24x26x28, 5, FP32 132 -> 114 us; p = 8
// 24^3, 1, FP64 143 -> 134 us, but 8, FP32 467 -> 465 us: there the workgroups a
// CU holds, and the tails of the 8 launches (15 %), set the time.
// PART: the last workgroup's right-hand sides may be fewer than NR; the others' work
// is left out (tested at run time, which cost full pairs up to 4 %)
template <int N, typename T, int NR, bool PART>
__global__ void __launch_bounds__(kCellMaxThreads)
__attribute__((amdgpu_waves_per_eu(1, lds_waves_per_simd(NR * full_cells(N) * 2 * N * N * N * (int)sizeof(T), full_cells(N) * N * N))))
cont_coef_kernel(const CellArgs<N, T> a)
{
  constexpr int N2 = N * N, N3 = N2 * N, p = N - 1;
  const int CB = a.cb, rs = 2 * CB * N3; // arrays of one right-hand side
  T *sA = dyn_lds<T>(), *sB = sA + CB * N3;
  const int t = threadIdx.x, c = t / N2, l = t % N2;
  const ContPos q = cont_position(a, logical_block(blockIdx.x, gridDim.x, a.order), c);
  const bool act = q.act;
  T *A = sA + (act ? c : 0) * N3, *B = sB + (act ? c : 0) * N3;
  const int r0 = (int)blockIdx.y * NR, nr = a.nrhs - r0 < NR ? a.nrhs - r0 : NR;
  const T *src = a.src + r0 * a.vstride;
  T *dst = a.dst + r0 * a.vstride;
  const T *coef = a.coef + (q.cell0 + (act ? c : 0)) * N3;

  if (act) {
    const int X = q.cx * p + l % N, Y = q.cy * p + l / N;
    const bool bxy = X == 0 || Y == 0 || X == a.gx - 1 || Y == a.gy - 1;
    const long long plane = (long long)a.gy * a.gx, g0 = (long long)q.cz * p * plane + (long long)Y * a.gx + X;
    T u[NR][N], v[N];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int Z = q.cz * p + k;
        u[r][k] = bxy || Z == 0 || Z == a.gz - 1 || r >= nr ? T(0) : src[r * a.vstride + g0 + k * plane];
      }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      eo_apply<N, 1>(ctab(a.dt).Sf, u[r], v);
      lds_write_line<N, N, 2>(A + r * rs, l, v);
    }
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T u[N], v[N];
      lds_read_line<N, N, 0>(A + r * rs, l, u);
      eo_apply<N, 1>(ctab(a.dt).Sf, u, v);
      lds_write_line<N, N, 0>(A + r * rs, l, v);
    }
  }
  // the coefficient of this thread's line of direction DIR
  auto load_coef = [&](auto dirc, T(&k)[N]) {
    constexpr int DIR = decltype(dirc)::value;
    const T *kl = coef + line_base<N, N, DIR>(l);
#pragma unroll
    for (int i = 0; i < N; ++i) k[i] = kl[i * line_stride<N, N, DIR>()];
  };
  // r = D^T (cdiag k) D v
  auto grad = [&](int dir, const T(&k)[N], const T(&v)[N], T(&r)[N]) {
    T g[N];
    eo_apply<N, -1>(ctab(a.dt).Df, v, g);
#pragma unroll
    for (int i = 0; i < N; ++i) g[i] *= a.cdiag[dir] * k[i];
    eo_apply<N, -1>(ctab(a.dt).Db, g, r);
  };
  using dir0 = std::integral_constant<int, 0>;
  using dir1 = std::integral_constant<int, 1>;
  using dir2 = std::integral_constant<int, 2>;
  T k[N];
  if (act) load_coef(dir1(), k);
  __syncthreads();
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T u[N], v[N], w[N];
      lds_read_line<N, N, 1>(A + r * rs, l, u);
      eo_apply<N, 1>(ctab(a.dt).Sf, u, v);
      lds_write_line<N, N, 1>(A + r * rs, l, v);
      grad(1, k, v, w);
      lds_write_line<N, N, 1>(B + r * rs, l, w);
    }
    load_coef(dir0(), k);
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T v[N], w[N], b[N];
      lds_read_line<N, N, 0>(A + r * rs, l, v);
      grad(0, k, v, w);
      lds_read_line<N, N, 0>(B + r * rs, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) w[i] += b[i];
      lds_write_line<N, N, 0>(B + r * rs, l, w);
    }
    load_coef(dir2(), k);
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T v[N], w[N], b[N];
      lds_read_line<N, N, 2>(A + r * rs, l, v);
      grad(2, k, v, w);
      lds_read_line<N, N, 2>(B + r * rs, l, b);
#pragma unroll
      for (int i = 0; i < N; ++i) w[i] += b[i];
      eo_apply<N, 1>(ctab(a.dt).Sb, w, v);
      lds_write_line<N, N, 2>(A + r * rs, l, v);
    }
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T u[N], v[N];
      lds_read_line<N, N, 1>(A + r * rs, l, u);
      eo_apply<N, 1>(ctab(a.dt).Sb, u, v);
      lds_write_line<N, N, 1>(A + r * rs, l, v);
    }
  }
  __syncthreads();
  T o[NR][N];
  if constexpr (PART)
#pragma unroll
    for (int i = 0; i < N; ++i) o[NR - 1][i] = T(0);
  if (act) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (PART && r >= nr) break;
      T u[N];
      lds_read_line<N, N, 0>(A + r * rs, l, u);
      eo_apply<N, 1>(ctab(a.dt).Sb, u, o[r]);
      // x-merge: the first x-plane of cell c+1 is the last one of cell c
      if (a.color >= 0) B[r * rs + l] = o[r][0];
    }
  }
  if (a.color >= 0) {
    __syncthreads();
    cont_store_colored<N, T, NR>(a, o, sA, sB, rs, nr, act, c, l, q.cy, q.cz, q.seg, q.cx0, q.cx_end, dst);
  } else if (act) {
    const int Y = q.cy * p + l % N, Z = q.cz * p + l / N;
    const bool byz = Y == 0 || Z == 0 || Y == a.gy - 1 || Z == a.gz - 1;
    const long long g0 = ((long long)Z * a.gy + Y) * a.gx + (long long)q.cx * p;
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (r < nr)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int X = q.cx * p + i;
          if (!(byz || X == 0 || X == a.gx - 1)) atomicAdd(dst + r * a.vstride + g0 + i, o[r][i]);
        }
  }
}

// Diagonal of the Cartesian Laplacian (local or continuous, optionally with
// a per-q coefficient): diag_i = sum_d sum_q c_d k_q w_q (dphi_i/dxi_d)^2
// prod_{e!=d} phi_i^2 -- a sum-factorized contraction of the weights with
// the squared 1D matrices (G1 = S D: basis derivative at Gauss points).
template <int N, typename T>
struct DiagArgs {
  Eo<N, T> S2b, G2b; // backward contractions with S^2 and G1^2
  Eo<N, T> S1b;      // load vector: backward contraction with S
  T fval, jxw;
  T w[N];
  const T *coef;
  T *diag;
  long long ncells;
  int nx, ny, nz, gx, gy, gz;
  T cdiag[3];
  int cont;
};

// LOAD: b_i = sum_q f JxW_q phi_i(x_q) instead of the diagonal; COEF: with a
// coefficient.  Kernels of their own: as run-time choices, their loads and
// registers cost the plain diagonal 25 % (Q6 FP64 1.2e7 nodes: 328 us)
template <int N, typename T, bool LOAD, bool COEF>
__global__ void __launch_bounds__(threads_per_block<N>()) diag_kernel(const DiagArgs<N, T> a)
{
  constexpr int CB = full_cells(N);
  constexpr int N2 = N * N, N3 = N * N * N, p = N - 1;
  __shared__ T sA[CB * N3];
  __shared__ T sR[CB * N3];
  const int t = threadIdx.x, c = t / N2, l = t % N2;
  const long long cell = (long long)blockIdx.x * CB + c;
  const bool act = c < CB && cell < a.ncells;
  T *A = sA + (act ? c : 0) * N3;
  T *R = sR + (act ? c : 0) * N3;
  for (int d = 0; d < (LOAD ? 1 : 3); ++d) {
    if (act) {
      // weights c_d w_q k_q on x-line l (the coefficient holds the quadrature weight)
      T u[N], v[N];
      const T f = LOAD ? a.fval * a.jxw : a.cdiag[d];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if constexpr (COEF) u[i] = f * a.coef[cell * N3 + l * N + i];
        else u[i] = f * line_weight<N, 0>(a.w, l, i);
      }
      if constexpr (LOAD) eo_apply<N, 1>(a.S1b, u, v);
      else if (d == 0) eo_apply<N, 1>(a.G2b, u, v);
      else eo_apply<N, 1>(a.S2b, u, v);
      lds_write_line<N, N, 0>(A, l, v);
    }
    __syncthreads();
    if (act) {
      T u[N], v[N];
      lds_read_line<N, N, 1>(A, l, u);
      if constexpr (LOAD) eo_apply<N, 1>(a.S1b, u, v);
      else if (d == 1) eo_apply<N, 1>(a.G2b, u, v);
      else eo_apply<N, 1>(a.S2b, u, v);
      lds_write_line<N, N, 1>(A, l, v);
    }
    __syncthreads();
    if (act) {
      T u[N], v[N], r[N];
      lds_read_line<N, N, 2>(A, l, u);
      if constexpr (LOAD) eo_apply<N, 1>(a.S1b, u, v);
      else if (d == 2) eo_apply<N, 1>(a.G2b, u, v);
      else eo_apply<N, 1>(a.S2b, u, v);
      if (d > 0) lds_read_line<N, N, 2>(R, l, r);
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] = d > 0 ? r[i] + v[i] : v[i];
      lds_write_line<N, N, 2>(R, l, r);
    }
    __syncthreads();
  }
  if (act) {
    T r[N];
    lds_read_line<N, N, 2>(R, l, r); // z-line l = j*N + i
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if (a.cont) {
        const int cx = (int)(cell % a.nx);
        const long long rr = cell / a.nx;
        const int cy = (int)(rr % a.ny), cz = (int)(rr / a.ny);
        const int X = cx * p + l % N, Y = cy * p + l / N, Z = cz * p + k;
        const bool bd = X == 0 || Y == 0 || Z == 0 || X == a.gx - 1 || Y == a.gy - 1 || Z == a.gz - 1;
        if (!bd) atomicAdd(a.diag + ((long long)Z * a.gy + Y) * a.gx + X, r[k]);
      } else {
        a.diag[cell * N3 + k * N2 + l] = r[k];
      }
    }
  }
}

// Gradient of lambda^T A(k) u with respect to the per-q coefficient of the
// continuous Laplacian: g_q = sum_rhs JxW_q sum_d ij_d^2 (du/dxi_d)(dlambda/dxi_d)
// at every cell quadrature point.
template <int N, typename T>
struct CoefGradArgs {
  const DevTab<N, T> *dt;
  const T *u, *lam;
  T *grad;
  long long ncells;
  int nx, ny, nz, gx, gy, gz;
  T cdiag[3];
  int nrhs;
  long long vstride;
};

// Phases per right-hand side (barrier between): z lines of u and lambda (the
// next pair's loads are in flight meanwhile), value sweeps in z -> U, Lm; x
// value sweeps; y value sweeps, y derivatives; x and z derivatives.  Each
// thread sums the products of its own lines in registers over all right-hand
// sides, one accumulator line per direction; they meet in LDS once at the end,
// where the quadrature weight is applied.  What bounds it: VALU issue and LDS.
// 14 LDS accesses per point and pair and 4 barriers, where accumulating in LDS
// direction by direction took 21 and 7, and one product per point and
// direction instead of four.  Measured, before -> after: p = 8 24^3, 8 pairs,
// FP32 360 -> 231 us, FP64 585 -> 451 us; p = 2 80x70x75, 8 pairs, FP64 449 -> 265
// us; p = 4 40x37x42, 3 pairs, FP32 123 -> 77 us.
template <int N, typename T>
__global__ void __launch_bounds__(threads_per_block<N>()) coef_grad_kernel(const CoefGradArgs<N, T> a)
{
  constexpr int CB = full_cells(N);
  constexpr int N2 = N * N, N3 = N * N * N, p = N - 1;
  __shared__ T sU[CB * N3];
  __shared__ T sL[CB * N3];
  const int t = threadIdx.x, c = t / N2, l = t % N2;
  const unsigned cell0 = blockIdx.x * (unsigned)CB;
  const bool act = c < CB && cell0 + c < a.ncells;
  T *U = sU + (act ? c : 0) * N3;
  T *Lm = sL + (act ? c : 0) * N3;
  CellXYZ q = traverse_xyz(cell0, a.nx, a.ny, a.nz, 0);
  if (q.x + c < (unsigned)a.nx) q.x += c;
  else q = traverse_xyz(act ? cell0 + c : cell0, a.nx, a.ny, a.nz, 0);
  const int X = (int)q.x * p + l % N, Y = (int)q.y * p + l / N, Z0 = (int)q.z * p;
  const bool bxy = !act || X == 0 || Y == 0 || X == a.gx - 1 || Y == a.gy - 1;
  const long long plane = (long long)a.gy * a.gx, g0 = (long long)Z0 * plane + (long long)Y * a.gx + X;
  T u[N], w[N];
  auto load = [&](int r) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const bool bd = bxy || Z0 + k == 0 || Z0 + k == a.gz - 1;
      const long long g = r * a.vstride + g0 + k * plane;
      u[k] = bd ? T(0) : a.u[g];
      w[k] = bd ? T(0) : a.lam[g];
    }
  };
  T ax[N], ay[N], az[N];
#pragma unroll
  for (int i = 0; i < N; ++i) ax[i] = ay[i] = az[i] = T(0);
  auto add = [&](const T(&x)[N], const T(&y)[N], T(&acc)[N]) {
    T gx[N], gy[N];
    eo_apply<N, -1>(ctab(a.dt).Df, x, gx);
    eo_apply<N, -1>(ctab(a.dt).Df, y, gy);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = gx[i] * gy[i] + acc[i];
  };
  // FP64 at N = 12 to 14: the next pair's registers would cost a third of the
  // resident waves (N = 12, 3e6 nodes, one pair 83 us instead of 54; N = 13 78 and
  // 52; N = 15 and 16 are 3 % faster with it)
  constexpr bool AHEAD = sizeof(T) == 4 || N < 12 || N > 14;
  if (AHEAD) load(0);
  for (int r = 0; r < a.nrhs; ++r) {
    if (!AHEAD) load(r);
    if (act) {
      T v[N], z[N];
      eo_apply<N, 1>(ctab(a.dt).Sf, u, v);
      eo_apply<N, 1>(ctab(a.dt).Sf, w, z);
      lds_write_line<N, N, 2>(U, l, v);
      lds_write_line<N, N, 2>(Lm, l, z);
    }
    __syncthreads();
    if (AHEAD && r + 1 < a.nrhs) load(r + 1);
    if (act) {
      T x[N], v[N];
      lds_read_line<N, N, 0>(U, l, x);
      eo_apply<N, 1>(ctab(a.dt).Sf, x, v);
      lds_write_line<N, N, 0>(U, l, v);
      lds_read_line<N, N, 0>(Lm, l, x);
      eo_apply<N, 1>(ctab(a.dt).Sf, x, v);
      lds_write_line<N, N, 0>(Lm, l, v);
    }
    __syncthreads();
    if (act) {
      T x[N], v[N], z[N];
      lds_read_line<N, N, 1>(U, l, x);
      eo_apply<N, 1>(ctab(a.dt).Sf, x, v);
      lds_write_line<N, N, 1>(U, l, v);
      lds_read_line<N, N, 1>(Lm, l, x);
      eo_apply<N, 1>(ctab(a.dt).Sf, x, z);
      lds_write_line<N, N, 1>(Lm, l, z);
      add(v, z, ay);
    }
    __syncthreads();
    if (act) {
      T x[N], y[N];
      lds_read_line<N, N, 0>(U, l, x);
      lds_read_line<N, N, 0>(Lm, l, y);
      add(x, y, ax);
      lds_read_line<N, N, 2>(U, l, x);
      lds_read_line<N, N, 2>(Lm, l, y);
      add(x, y, az);
    }
    __syncthreads();
  }
  if (act) {
#pragma unroll
    for (int i = 0; i < N; ++i) ax[i] *= a.cdiag[0];
    lds_write_line<N, N, 0>(U, l, ax);
  }
  __syncthreads();
  if (act) {
    T v[N];
    lds_read_line<N, N, 1>(U, l, v);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = a.cdiag[1] * ay[i] + v[i];
    lds_write_line<N, N, 1>(U, l, v);
  }
  __syncthreads();
  if (act) {
    T v[N];
    lds_read_line<N, N, 2>(U, l, v);
    T *out = a.grad + (long long)(cell0 + c) * N3 + l;
#pragma unroll
    for (int k = 0; k < N; ++k) out[k * N2] = (a.cdiag[2] * az[k] + v[k]) * line_weight<N, 2>(ctab(a.dt).w, l, k);
  }
}


template <int N, typename T>
static hipError_t launch_coef_grad_n(const CoefGradLaunch &L, hipStream_t s)
{
  CoefGradArgs<N, T> a{};
  a.dt = (const DevTab<N, T> *)L.dtab;
  a.u = (const T *)L.u;
  a.lam = (const T *)L.lambda;
  a.grad = (T *)L.grad;
  a.ncells = L.ncells;
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  a.gx = L.nc[0] * (N - 1) + 1;
  a.gy = L.nc[1] * (N - 1) + 1;
  a.gz = L.nc[2] * (N - 1) + 1;
  const double jxw = 1. / (L.inv_jac[0] * L.inv_jac[1] * L.inv_jac[2]);
  for (int d = 0; d < 3; ++d) a.cdiag[d] = T(L.inv_jac[d] * L.inv_jac[d] * jxw);
  a.nrhs = L.nrhs;
  a.vstride = L.vstride;
  constexpr int CB = full_cells(N);
  hipLaunchKernelGGL((coef_grad_kernel<N, T>), dim3((unsigned)((L.ncells + CB - 1) / CB)),
                     dim3(threads_per_block<N>()), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------- launch

// continuous scatter schedule: colored (no atomics, no zero fill) unless the
// caller asks for the atomic variant or, by default, each of the 8 colour
// launches would hold fewer workgroups than the chip has CUs
static bool cont_colored(const CellLaunch &L, int cb)
{
  if (L.cont_scatter >= 0) return L.cont_scatter == 1;
  return L.ncells / cb >= 8 * 256;
}

template <int N, typename T>
static hipError_t launch_cell_n(const CellLaunch &L, hipStream_t stream)
{
  CellArgs<N, T> a{};
  a.dt = (const DevTab<N, T> *)L.dtab;
  a.src = (const T *)L.src;
  a.dst = (T *)L.dst;
  a.rhs = (const T *)L.rhs;
  a.diag = (const T *)L.diag;
  a.tm = (T *)L.tm;
  a.c_np = T(L.c_np);
  a.c_tm = T(L.c_tm);
  a.coef = (const T *)L.coef;
  a.ncells = L.ncells;
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  a.gx = L.nc[0] * (N - 1) + 1;
  a.gy = L.nc[1] * (N - 1) + 1;
  a.gz = L.nc[2] * (N - 1) + 1;
  const double jxw = 1. / (L.inv_jac[0] * L.inv_jac[1] * L.inv_jac[2]);
  for (int d = 0; d < 3; ++d) {
    a.cdiag[d] = T(L.inv_jac[d] * L.inv_jac[d] * jxw);
    a.ij[d] = T(L.inv_jac[d]);
    a.jxwf[d] = T(jxw * L.inv_jac[d]);
    a.tau[d] = T(double(N * N) * L.inv_jac[d]);
  }
  a.nrhs = L.nrhs;
  a.vstride = L.vstride;
  const int CB = L.cb > 0 ? L.cb : full_cells(N);
  if (CB * N * N > kCellMaxThreads) return hipErrorInvalidConfiguration;
  a.cb = CB;
  a.order = L.order;
  constexpr int N3 = N * N * N;
  const size_t lds = size_t(CB) * (2 * N3 + (L.mode == 2 ? 12 * N * N : 0)) * sizeof(T);
  const unsigned blocks = (unsigned)((L.ncells + CB - 1) / CB);
  const dim3 grid(blocks, L.nrhs), block(((CB * N * N + 63) / 64) * 64);
  auto launch = [&](auto kern, dim3 g, size_t bytes) {
    const hipError_t e = allow_dynamic_lds((const void *)kern, bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, g, block, bytes, stream, a);
    return hipGetLastError();
  };
  if (L.mode == 0) {
    return launch(L.coef ? cell_kernel<N, T, Mode::Local, false, false, true>
                         : cell_kernel<N, T, Mode::Local, false, false, false>, grid, lds);
  } else if (L.mode == 1) {
    // two right-hand sides per workgroup at low degrees, where their shared
    // index arithmetic and coefficient outweigh the halved number of resident
    // workgroups (8 right-hand sides, p = 2 80x70x75 FP32: 370 -> 297 us, p = 4
    // 40x37x42 156 -> 150 us, p = 8 24^3 462 -> 493 us; FP64 p = 1 227 -> 184 us,
    // p = 3 50x52x55 263 -> 290 us), and only where each colour's launch still
    // fills the chip (2 right-hand sides FP32 p = 4 35x30x30, 450 pairs a colour:
    // 72 us one by one, 82 us in pairs; 55x47x48, 1728: 174 and 153 us; p = 3
    // 46x40x40 with 4, 1200: 99.5 and 103 us; p = 1 73x64x64 with 2, 1024: 53 and 49
    // us).  The atomic scatter gains nothing from pairs (p = 3 24x21x22 with 8: 117
    // and 120 us).
    constexpr int NR2 = N <= (std::is_same<T, float>::value ? 5 : 2) ? 2 : 1;
    a.nseg = (a.nx + CB - 1) / CB;
    const bool colored = cont_colored(L, CB);
    const long long pairs = (long long)((a.nseg + 1) / 2) * ((a.ny + 1) / 2) * ((a.nz + 1) / 2) * ((L.nrhs + 1) / 2);
    const bool two = L.coef && L.nrhs > 1 && NR2 == 2 && colored && pairs >= (N == 2 ? 1000 : 1300);
    auto kern = cell_kernel<N, T, Mode::Cont, false, false, false>;
    if (two) kern = L.nrhs % 2 ? cont_coef_kernel<N, T, NR2, NR2 == 2> : cont_coef_kernel<N, T, NR2, false>;
    else if (L.coef) kern = cont_coef_kernel<N, T, 1, false>;
    const size_t klds = two ? 2 * lds : lds;
    const unsigned ny = two ? (L.nrhs + 1) / 2 : L.nrhs;
    if (!colored) {
      a.color = -1;
      const hipError_t e = vec_fill(std::is_same<T, float>::value, L.dst, L.vstride * L.nrhs, 0., stream);
      if (e != hipSuccess) return e;
      return launch(kern, dim3(blocks, ny), klds);
    }
    // colours in ascending order: the first unit to touch a node stores it
    for (int color = 0; color < 8; ++color) {
      const int ps = color >> 2 & 1, py = color & 1, pz = color >> 1 & 1;
      a.color = color;
      a.nss = (a.nseg - ps + 1) / 2;
      a.nry = (a.ny - py + 1) / 2;
      a.nrz = (a.nz - pz + 1) / 2;
      const long long nb = (long long)a.nss * a.nry * a.nrz;
      if (nb == 0) continue;
      const hipError_t e = launch(kern, dim3((unsigned)nb, ny), klds);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  if (L.refx)
    return launch(L.cheby ? cell_kernel<N, T, Mode::DG, true, true, false> : cell_kernel<N, T, Mode::DG, false, true, false>,
                  grid, lds);
  // (up to degree 8 the operator runs as a sum of Kronecker products)
  if constexpr (N - 1 > kMaxDegreeTp)
    return launch(L.cheby ? cell_kernel<N, T, Mode::DG, true, false, false> : cell_kernel<N, T, Mode::DG, false, false, false>,
                  grid, lds);
  else return hipErrorInvalidValue;
}

template <int N, typename T>
static hipError_t launch_diag_n(const CellLaunch &L, hipStream_t stream)
{
  DiagArgs<N, T> a{};
  const Tables1D &t = *L.tables;
  std::vector<double> S2(N * N), G2(N * N);
  for (int i = 0; i < N; ++i)
    for (int q = 0; q < N; ++q) {
      double g = 0.;
      for (int m = 0; m < N; ++m) g += t.S[i * N + m] * t.D[m * N + q];
      S2[i * N + q] = t.S[i * N + q] * t.S[i * N + q];
      G2[i * N + q] = g * g;
    }
  a.S2b = make_eo<N, T>(S2, false);
  a.G2b = make_eo<N, T>(G2, false);
  a.S1b = make_eo<N, T>(t.S, false);
  a.fval = T(L.load_value);
  for (int i = 0; i < N; ++i) a.w[i] = T(t.weights[i]);
  a.coef = (const T *)L.coef;
  a.diag = (T *)L.dst;
  a.ncells = L.ncells;
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  a.gx = L.nc[0] * (N - 1) + 1;
  a.gy = L.nc[1] * (N - 1) + 1;
  a.gz = L.nc[2] * (N - 1) + 1;
  const double jxw = 1. / (L.inv_jac[0] * L.inv_jac[1] * L.inv_jac[2]);
  for (int d = 0; d < 3; ++d) a.cdiag[d] = T(L.inv_jac[d] * L.inv_jac[d] * jxw);
  a.jxw = T(jxw);
  a.cont = L.mode == 1;
  constexpr int CB = full_cells(N);
  const unsigned blocks = (unsigned)((L.ncells + CB - 1) / CB);
  auto kern = L.load ? diag_kernel<N, T, true, false>
                     : (L.coef ? diag_kernel<N, T, false, true> : diag_kernel<N, T, false, false>);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads_per_block<N>()), 0, stream, a);
  return hipGetLastError();
}

template <typename T>
static hipError_t dispatch_cell(const CellLaunch &L, hipStream_t s, bool diag)
{
  switch (L.tables->n) {
#define SFK_CASE(NN) \
  case NN: return diag ? launch_diag_n<NN, T>(L, s) : launch_cell_n<NN, T>(L, s);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_cell(const CellLaunch &L, hipStream_t stream)
{
  return L.fp32 ? dispatch_cell<float>(L, stream, false) : dispatch_cell<double>(L, stream, false);
}

hipError_t launch_cell_diagonal(const CellLaunch &L, hipStream_t stream)
{
  return L.fp32 ? dispatch_cell<float>(L, stream, true) : dispatch_cell<double>(L, stream, true);
}

template <typename T>
static hipError_t dispatch_coef_grad(const CoefGradLaunch &L, hipStream_t s)
{
  switch (L.tables->n) {
#define SFK_CASE(NN) \
  case NN: return launch_coef_grad_n<NN, T>(L, s);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_coef_gradient(const CoefGradLaunch &L, hipStream_t stream)
{
  return L.fp32 ? dispatch_coef_grad<float>(L, stream) : dispatch_coef_grad<double>(L, stream);
}

} // namespace sfk
