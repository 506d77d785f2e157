// DG Laplacian with precomputed 1D matrices on Cartesian cells
// (legacy/include/precomputed_dg_laplacian.h:96-377, do_inner_loop):
//
//   A u = f_x (M (x) M (x) L~) u + f_y (M (x) L~ (x) M) u + f_z (L~ (x) M (x) M) u
//
// (x fastest on the right), L = 1D Laplace matrix with the cell's own
// interior-penalty face terms, M = 1D mass matrix, both symmetric and
// centro-symmetric in the Hermite-like basis; L~ adds the coupling of rows
// 0, 1 (n-1, n-2) to the lower (upper) neighbour's two face layers through
// the constants v1, v2 (:139-148, :175-188, :215-224).  f_d =
// inv_jac_d^2 / (inv_jac_x inv_jac_y inv_jac_z) (1 on the reference's unit
// cells).  Periodic in every direction.
//
// The Cartesian DG-SIPG operator is the same sum with the penalty (p+1)^2/h
// instead of p(p+1)/h and runs here too (degree <= 8): (p+1)-point Gauss
// quadrature integrates its 1D mass and stiffness exactly.
//
// One workgroup = cb cells in a row of the traversal (block order 2: slabs of
// z-layers), n^2 threads per cell; thread l owns
// line l of every direction.  Phases (barrier between):
//   0  z line of u from global memory; U <- u, P <- L~_z u (z lines)
//   1  r = L~_x u (x line, registers), Q <- L~_y u (y line)
//   2  P <- M_x P, Q <- M_x Q, U <- r (x lines)
//   3  P <- M_y P, Q <- Q + M_y U (y lines)
//   4  z line of M_z Q + P -> dst, or the fused Chebyshev update of
//      evaluation_dg_laplacian.h:485-502 on the way out.
// (f_z M_y M_x L~_z + M_z (M_x f_y L~_y + M_y f_x L~_x); the factors f_d are
// in the tables of L.)
//
// What bounds it: LDS accesses and HBM about equally.  Starting and ending on
// z lines, whose lanes touch consecutive dofs, both the block load and the
// store go straight between registers and memory: 17 LDS accesses per point
// and 4 barriers, where a coalesced copy through LDS on both ends took 20 and
// 5.  Measured, before -> after, on vectors in turn,
// matvec: p = 3 56x50x55 FP64 41.0 -> 36.3 us (4.3 TB/s), FP32 24 -> 19.6 us; p = 5
// 31x37x29 FP64 33.3 -> 29.3 us, FP32 18.4 -> 16 us; p = 7 22x25x24 FP32 21.4
// -> 15.8 us; Chebyshev step p = 5 FP64 80 -> 70 us, p = 8 20x21x22 78 -> 62 us.
// Tried and not kept: workgroups that loop over several blocks and load the
// next one early (no faster at 4 to 64 workgroups per CU).
#include <type_traits>

#include "sfk_device.h"
#include "sfk_kernels.h"

namespace sfk {

namespace {

constexpr int kPcMaxThreads = 256;

template <int N, typename T>
struct PcTab {
  Eo<N, T> L[3], M; // f_d L, M; symmetric: the same table serves both contraction directions
  T v1[3], v2[3];   // neighbour coupling, times f_d
  T f[3];           // direction factors
  T ld[N], md[N];   // diagonals of L and M (operator diagonal)
};

// LDS block of a cell (x fastest): for n = 4, 8 rows are padded by one
// value, so that the x lines of consecutive rows, and with the plane pitch
// the y lines too, fall on different banks (passes per access relative to the
// conflict-free count, over the kernel's mix: n = 4 FP64 1.76 -> 1.24, n = 8
// 3.88 -> 1.24).  Odd n gains nothing from it, and for n = 6 the workgroup
// per CU that the larger block costs outweighs 1.84 -> 1.61 (p = 5 FP64 29.3
// us unpadded, 32.4 us padded).
template <int N>
struct PcLds {
  static constexpr int NP = N == 4 || N == 8 ? N + 1 : N, PP = N * NP, CS = N * PP;
};
template <int N, int DIR>
__device__ __forceinline__ int pc_base(int l)
{
  using C = PcLds<N>;
  return DIR == 0 ? (l / N) * C::PP + (l % N) * C::NP : (DIR == 1 ? (l / N) * C::PP + l % N : (l / N) * C::NP + l % N);
}
template <int N, int DIR, typename T>
__device__ __forceinline__ void pc_read(const T *cell, int l, T (&v)[N])
{
  constexpr int st = DIR == 0 ? 1 : (DIR == 1 ? PcLds<N>::NP : PcLds<N>::PP);
  const T *q = cell + pc_base<N, DIR>(l);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = q[i * st];
}
template <int N, int DIR, typename T>
__device__ __forceinline__ void pc_write(T *cell, int l, const T (&v)[N])
{
  constexpr int st = DIR == 0 ? 1 : (DIR == 1 ? PcLds<N>::NP : PcLds<N>::PP);
  T *q = cell + pc_base<N, DIR>(l);
#pragma unroll
  for (int i = 0; i < N; ++i) q[i * st] = v[i];
}

template <int N, typename T>
__device__ __forceinline__ const SFK_CONST_AS PcTab<N, T> &pctab(const PcTab<N, T> *p)
{
  return *(const SFK_CONST_AS PcTab<N, T> *)opaque_ptr(p);
}

template <int N, typename T>
constexpr int pc_waves()
{
  constexpr int cb = precomp_cells(N, sizeof(T) == 4);
  return lds_waves_per_simd(3 * cb * PcLds<N>::CS * (int)sizeof(T), cb * N * N);
}

template <int N, typename T>
struct PcArgs {
  const PcTab<N, T> *pt;
  const T *src;
  T *dst;
  const T *rhs, *diag;
  T *tm;
  T c_np, c_tm;
  long long ncells, nvec;
  int nx, ny, nz;
  int cb, order;
};

// index inside a cell of point k of line l in direction DIR (x fastest)
template <int N, int DIR>
__device__ __forceinline__ int pc_idx(int l, int k)
{
  return line_base<N, N, DIR>(l) + k * line_stride<N, N, DIR>();
}

// rows 0, 1 couple to the lower neighbour's layers n-1, n-2; rows n-1, n-2
// to the upper neighbour's layers 0, 1 (same adds as the reference)
template <int N, typename T>
__device__ __forceinline__ void pc_couple(T (&o)[N], const T (&nb)[4], T v1, T v2)
{
  o[0] += v1 * nb[0] + v2 * nb[1];
  o[1] += v2 * nb[0];
  o[N - 1] += v1 * nb[2] + v2 * nb[3];
  o[N - 2] += v2 * nb[2];
}

// the two face layers of the lower and of the upper neighbour at face point l
template <int N, int DIR, typename T>
__device__ __forceinline__ void pc_load_layers(const T *src, const int (&nbr)[6], int l, T (&nb)[4])
{
  constexpr long long N3 = N * N * N;
  const T *lo = src + nbr[2 * DIR] * N3 + pc_idx<N, DIR>(l, N - 2);
  const T *hi = src + nbr[2 * DIR + 1] * N3 + pc_idx<N, DIR>(l, 0);
  if constexpr (DIR == 0 && N % 2 == 0) {
    // adjacent in memory, at even positions: one load each
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const T2 a = *(const T2 *)lo, b = *(const T2 *)hi;
    nb[0] = a.y;
    nb[1] = a.x;
    nb[2] = b.x;
    nb[3] = b.y;
  } else {
    constexpr int st = line_stride<N, N, DIR>();
    nb[0] = lo[st];
    nb[1] = lo[0];
    nb[2] = hi[0];
    nb[3] = hi[st];
  }
}

// How the vectors are read and written: kLines as z lines; kFlatStore: the matvec's
// results leave through LDS as the block's consecutive values; kFlat: that at both
// ends.  Where a z line's lanes cover parts of cache lines (n^2 values: 32 to 200
// B), the pieces cost HBM more than LDS saves once the vectors exceed the Infinity
// Cache, the non-temporal stores of the matvec most.  Matvec, lines / flat stores /
// flat: n = 2 FP64 3e6 unknowns 15.1 / 14.5 / 15.5 us, 3e7 175 / 162 / 164; n = 3
// FP64 6e6 32 / 26 / 27.5, 2e7 132 / 107 / 105, FP32 1e7 28.5 / 27.1 / 27.9, 3e7
// 103 / 94 / 90; n = 5 FP64 2e7 107 / 101 / 98, FP32 2e7 45.7 / 47.5 / 50, 3e7 97 /
// 86 / 84; n = 6 FP32 2e7 43.8 / 45.9 / 47.9, 3e7 83.5 / 78.3 / 78.4; n = 7 and
// above, and n = 6 FP64: lines 3 to 13 % faster.  Chebyshev step (six streams),
// lines / flat: n = 5 FP32 6e6 24.8 / 28.2, 1.5e7 94 / 83, 3e7 182 / 167; n = 3 FP32
// 36 / 30; n = 5 FP64 and n >= 6: lines 1 to 30 % faster.  (Plain instead of
// non-temporal stores: 5 to 30 % slower at most sizes.)  "Large" is the size of one
// vector, pc_large_bytes: two of the matvec's, six of the step's fill most of the
// 256 MB Infinity Cache.
enum PcForm { kLines = 0, kFlatStore = 1, kFlat = 2 };
template <int N, typename T>
constexpr PcForm pc_form(bool cheby, bool large)
{
  const bool fp32 = sizeof(T) == 4;
  if (cheby) return N <= 3 || (N == 5 && fp32 && large) ? kFlat : kLines;
  if (N == 2) return fp32 ? kLines : kFlatStore;
  if (N == 3) return large ? kFlat : kFlatStore;
  if (N == 5 && !fp32) return kFlatStore;
  return (N == 5 || N == 6) && fp32 && large ? kFlat : kLines;
}
constexpr long long pc_large_bytes(bool cheby) { return cheby ? 36LL << 20 : 104LL << 20; }

template <int N, typename T, bool COUPLE, bool CHEBY, PcForm FORM>
__global__ void __launch_bounds__(kPcMaxThreads) __attribute__((amdgpu_waves_per_eu(1, pc_waves<N, T>())))
precomp_kernel(PcArgs<N, T> a)
{
  constexpr int N2 = N * N, N3 = N2 * N;
  const int cb = a.cb;
  constexpr int CS = PcLds<N>::CS;
  constexpr bool FLAT = FORM == kFlat, FLAT_ST = FORM != kLines;
  const long long c0 = (long long)logical_block(blockIdx.x, gridDim.x, a.order) * cb;
  const long long voff = (long long)blockIdx.y * a.nvec;
  const T *src = a.src + voff;
  const int t = threadIdx.x, c = t / N2, l = t - c * N2;
  const bool act = c < cb && c0 + c < a.ncells;
  // (the divisions of the cell's coordinates on the scalar unit)
  int nbr[6] = {0, 0, 0, 0, 0, 0};
  const long long cell = act ? locate_cell((unsigned)c0, (unsigned)c, a.nx, a.ny, a.nz, FLAT_ST ? 0 : a.order, nbr) : 0;
  T *U = dyn_lds<T>() + (act ? c : 0) * CS;
  T *P = U + cb * CS, *Q = P + cb * CS;
  const long long g0 = cell * N3 + l; // this thread's z line: g0 + k N2
  // FLAT: the block's nval consecutive values lie in LDS as in memory
  static_assert(!FLAT_ST || CS == N3, "unpadded");
  const long long rem = a.ncells - c0;
  const int nval = (rem < cb ? (int)rem : cb) * N3;

  T u[N], nb[3][4], keep[FLAT ? N : 1];
  auto load_layers = [&]() {
    if constexpr (COUPLE) {
      pc_load_layers<N, 2>(src, nbr, l, nb[2]);
      pc_load_layers<N, 1>(src, nbr, l, nb[1]);
      pc_load_layers<N, 0>(src, nbr, l, nb[0]);
    }
  };
  if constexpr (FLAT) {
    if (act) load_layers(); // in flight together with the block's own values
    // blockDim.x >= cb n^2: n rounds cover the block
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int i = t + k * (int)blockDim.x;
      keep[k] = src[c0 * N3 + (i < nval ? i : nval - 1)];
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int i = t + k * (int)blockDim.x;
      if (i < nval) dyn_lds<T>()[i] = keep[k];
    }
    __syncthreads();
  }
  if (act) {
    if constexpr (FLAT) pc_read<N, 2>(U, l, u);
    else
#pragma unroll
      for (int k = 0; k < N; ++k) u[k] = src[g0 + k * N2];
    if constexpr (!FLAT) {
      load_layers();
      pc_write<N, 2>(U, l, u);
    }
    const auto &pt = pctab(a.pt);
    T o[N];
    eo_apply<N, 1>(pt.L[2], u, o);
    if constexpr (COUPLE) pc_couple(o, nb[2], pt.v1[2], pt.v2[2]);
    pc_write<N, 2>(P, l, o);
  }
  __syncthreads();
  T r[N];
  if (act) {
    const auto &pt = pctab(a.pt);
    T v[N], o[N];
    pc_read<N, 0>(U, l, v);
    eo_apply<N, 1>(pt.L[0], v, r);
    if constexpr (COUPLE) pc_couple(r, nb[0], pt.v1[0], pt.v2[0]);
    pc_read<N, 1>(U, l, v);
    eo_apply<N, 1>(pt.L[1], v, o);
    if constexpr (COUPLE) pc_couple(o, nb[1], pt.v1[1], pt.v2[1]);
    pc_write<N, 1>(Q, l, o);
  }
  __syncthreads();
  if (act) {
    const auto &pt = pctab(a.pt);
    T v[N], o[N];
    pc_read<N, 0>(P, l, v);
    eo_apply<N, 1>(pt.M, v, o);
    pc_write<N, 0>(P, l, o);
    pc_read<N, 0>(Q, l, v);
    eo_apply<N, 1>(pt.M, v, o);
    pc_write<N, 0>(Q, l, o);
    pc_write<N, 0>(U, l, r);
  }
  __syncthreads();
  // fused update: its streams are loaded one phase ahead
  T s_rhs[CHEBY ? N : 1], s_diag[CHEBY ? N : 1], s_tm[CHEBY ? N : 1];
  if constexpr (CHEBY) {
    if (FLAT || act)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int i = t + k * (int)blockDim.x;
        const long long g = FLAT ? c0 * N3 + (i < nval ? i : nval - 1) : g0 + k * N2;
        s_rhs[k] = a.rhs[g];
        s_diag[k] = a.diag[g];
        s_tm[k] = a.c_tm != T(0) ? a.tm[g] : T(0); // c_tm == 0: tm not read
      }
  }
  if (act) {
    const auto &pt = pctab(a.pt);
    T v[N], o[N];
    pc_read<N, 1>(P, l, v);
    eo_apply<N, 1>(pt.M, v, o);
    pc_write<N, 1>(P, l, o);
    pc_read<N, 1>(U, l, v);
    eo_apply<N, 1>(pt.M, v, o);
    pc_read<N, 1>(Q, l, v);
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = v[i] + o[i];
    pc_write<N, 1>(Q, l, o);
  }
  __syncthreads();
  if (act) {
    const auto &pt = pctab(a.pt);
    T v[N], o[N];
    pc_read<N, 2>(Q, l, v);
    eo_apply<N, 1>(pt.M, v, o);
    pc_read<N, 2>(P, l, v);
    if constexpr (FLAT_ST) {
#pragma unroll
      for (int k = 0; k < N; ++k) o[k] += v[k];
      pc_write<N, 2>(U, l, o);
    }
#pragma unroll
    for (int k = 0; k < (FLAT_ST ? 0 : N); ++k) {
      const long long g = g0 + k * N2;
      const T au = o[k] + v[k];
      if constexpr (CHEBY) {
        // r = A u - rhs; tm = c_tm tm + c_np diag r; dst = u - tm
        const T res = au - s_rhs[k];
        T tmv = a.c_np * s_diag[k] * res;
        if (a.c_tm != T(0)) tmv = a.c_tm * s_tm[k] + tmv;
        a.tm[g] = tmv;
        a.dst[g] = u[k] - tmv;
      } else {
        __builtin_nontemporal_store(au, a.dst + voff + g); // written once
      }
    }
  }
  if constexpr (FLAT_ST) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int i = t + k * (int)blockDim.x;
      if (i >= nval) break;
      const long long g = c0 * N3 + i;
      if constexpr (!CHEBY) {
        __builtin_nontemporal_store(dyn_lds<T>()[i], a.dst + voff + g);
      } else {
        const T res = dyn_lds<T>()[i] - s_rhs[k];
        T tmv = a.c_np * s_diag[k] * res;
        if (a.c_tm != T(0)) tmv = a.c_tm * s_tm[k] + tmv;
        a.tm[g] = tmv;
        a.dst[g] = keep[k] - tmv;
      }
    }
  }
}

// diag(A) = f_x L_ii M_jj M_kk + f_y M_ii L_jj M_kk + f_z M_ii M_jj L_kk
// (the coupling is off-diagonal), the same pattern in every cell
template <int N, typename T>
__global__ void __launch_bounds__(256) precomp_diag_kernel(const PcTab<N, T> *ptp, long long n, T *diag)
{
  constexpr int N3 = N * N * N;
  const auto &pt = pctab(ptp);
  for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (long long)gridDim.x * blockDim.x) {
    const int d = (int)(g % N3);
    const int i = d % N, j = (d / N) % N, k = d / (N * N);
    diag[g] = pt.f[0] * pt.ld[i] * pt.md[j] * pt.md[k] + pt.f[1] * pt.md[i] * pt.ld[j] * pt.md[k] +
              pt.f[2] * pt.md[i] * pt.md[j] * pt.ld[k];
  }
}

template <int N, typename T>
hipError_t launch_precomp_n(const PrecompLaunch &L, hipStream_t s)
{
  PcArgs<N, T> a{};
  a.pt = (const PcTab<N, T> *)L.ptab;
  a.src = (const T *)L.src;
  a.dst = (T *)L.dst;
  a.rhs = (const T *)L.rhs;
  a.diag = (const T *)L.diag;
  a.tm = (T *)L.tm;
  a.c_np = T(L.c_np);
  a.c_tm = T(L.c_tm);
  a.ncells = L.ncells;
  a.nvec = L.ncells * N * N * N;
  a.nx = L.nc[0];
  a.ny = L.nc[1];
  a.nz = L.nc[2];
  const int CB = L.cb > 0 ? L.cb : precomp_cells(N, sizeof(T) == 4);
  if (CB * N * N > kPcMaxThreads) return hipErrorInvalidConfiguration;
  if (L.cheby && L.nrhs != 1) return hipErrorInvalidValue;
  a.cb = CB;
  a.order = L.order;
  const size_t lds = size_t(3) * CB * PcLds<N>::CS * sizeof(T);
  const dim3 grid((unsigned)((L.ncells + CB - 1) / CB), (unsigned)L.nrhs), block(((CB * N * N + 63) / 64) * 64);
  decltype(&precomp_kernel<N, T, true, false, kLines>) kern;
  const bool large = a.nvec * (long long)sizeof(T) >= pc_large_bytes(L.cheby);
  auto pick = [&](auto cheby, auto big) {
    constexpr bool C = decltype(cheby)::value;
    constexpr PcForm F = pc_form<N, T>(C, decltype(big)::value);
    kern = L.couple ? precomp_kernel<N, T, true, C, F> : precomp_kernel<N, T, false, C, F>;
  };
  using no = std::false_type;
  using yes = std::true_type;
  if (L.cheby) large ? pick(yes(), yes()) : pick(yes(), no());
  else large ? pick(no(), yes()) : pick(no(), no());
  const hipError_t e = allow_dynamic_lds((const void *)kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, block, lds, s, a);
  return hipGetLastError();
}

template <int N, typename T>
size_t precomp_lds_per_cell_n()
{
  return size_t(3) * PcLds<N>::CS * sizeof(T);
}

template <int N, typename T>
hipError_t launch_precomp_diag_n(const PrecompLaunch &L, hipStream_t s)
{
  const long long n = L.ncells * N * N * N;
  const long long blocks = (n + 255) / 256;
  const unsigned g = (unsigned)(blocks < 65536 ? blocks : 65536);
  hipLaunchKernelGGL((precomp_diag_kernel<N, T>), dim3(g), dim3(256), 0, s, (const PcTab<N, T> *)L.ptab, n,
                     (T *)L.dst);
  return hipGetLastError();
}

template <int N, typename T>
hipError_t upload_pctab(const Precomp1D &pc, const double f[3], void **dev)
{
  PcTab<N, T> h{};
  h.M = make_eo<N, T>(pc.mass, true);
  for (int d = 0; d < 3; ++d) {
    std::vector<double> L(pc.lap);
    for (double &v : L) v *= f[d];
    h.L[d] = make_eo<N, T>(L, true);
    h.v1[d] = T(f[d] * pc.v1);
    h.v2[d] = T(f[d] * pc.v2);
    h.f[d] = T(f[d]);
  }
  for (int i = 0; i < N; ++i) {
    h.ld[i] = T(pc.lap[i * N + i]);
    h.md[i] = T(pc.mass[i * N + i]);
  }
  hipError_t e = hipMalloc(dev, sizeof(h));
  if (e != hipSuccess) return e;
  return hipMemcpy(*dev, &h, sizeof(h), hipMemcpyHostToDevice);
}

} // namespace

#define SFK_PC_DISPATCH(fn, n, ...)                                                                \
  switch (n) {                                                                                     \
  case 2: return fn<2, T>(__VA_ARGS__);                                                            \
  case 3: return fn<3, T>(__VA_ARGS__);                                                            \
  case 4: return fn<4, T>(__VA_ARGS__);                                                            \
  case 5: return fn<5, T>(__VA_ARGS__);                                                            \
  case 6: return fn<6, T>(__VA_ARGS__);                                                            \
  case 7: return fn<7, T>(__VA_ARGS__);                                                            \
  case 8: return fn<8, T>(__VA_ARGS__);                                                            \
  case 9: return fn<9, T>(__VA_ARGS__);                                                            \
  default: return hipErrorInvalidValue;                                                            \
  }

template <typename T>
static hipError_t dispatch_precomp(const PrecompLaunch &L, hipStream_t s)
{
  SFK_PC_DISPATCH(launch_precomp_n, L.n, L, s)
}
template <typename T>
static hipError_t dispatch_precomp_diag(const PrecompLaunch &L, hipStream_t s)
{
  SFK_PC_DISPATCH(launch_precomp_diag_n, L.n, L, s)
}
template <typename T>
static hipError_t dispatch_pctab(int n, const Precomp1D &pc, const double f[3], void **dev)
{
  SFK_PC_DISPATCH(upload_pctab, n, pc, f, dev)
}
#undef SFK_PC_DISPATCH

hipError_t launch_precomp(const PrecompLaunch &L, hipStream_t s)
{
  return L.fp32 ? dispatch_precomp<float>(L, s) : dispatch_precomp<double>(L, s);
}

hipError_t launch_precomp_diagonal(const PrecompLaunch &L, hipStream_t s)
{
  return L.fp32 ? dispatch_precomp_diag<float>(L, s) : dispatch_precomp_diag<double>(L, s);
}

hipError_t upload_precomp_tables(int n, const Precomp1D &pc, const double f[3], bool fp32, void **dev)
{
  return fp32 ? dispatch_pctab<float>(n, pc, f, dev) : dispatch_pctab<double>(n, pc, f, dev);
}

size_t precomp_lds_per_cell(int n, bool fp32)
{
  switch (n) {
#define SFK_CASE(NN) \
  case NN: return fp32 ? precomp_lds_per_cell_n<NN, float>() : precomp_lds_per_cell_n<NN, double>();
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9)
#undef SFK_CASE
  default: return size_t(3) * n * n * n * (fp32 ? 4 : 8);
  }
}

} // namespace sfk
