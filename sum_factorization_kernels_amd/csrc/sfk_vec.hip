// Vector kernels: fill, convert, FP64-accumulated dot products, axpby,
// the Chebyshev vector update for operators whose matvec cannot fuse it
// (continuous Q_p: the assembled value of a node is complete only after all
// cells have scattered), Dirichlet masking, layout converters between the
// canonical and the reference's lane-interleaved layout, and the batched 1D
// even-odd kernel.  All grid-stride loops; every block exits.
#include "sfk_device.h"
#include "sfk_kernels.h"

namespace sfk {

namespace {
constexpr int kThreads = 256;

inline unsigned grid_for(long long n, int per_thread = 1)
{
  long long b = (n + (long long)kThreads * per_thread - 1) / ((long long)kThreads * per_thread);
  if (b < 1) b = 1;
  if (b > 65535LL * 8) b = 65535LL * 8;
  return (unsigned)b;
}

template <typename T>
__global__ void fill_kernel(T *x, long long n, T v)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] = v;
}

template <typename S, typename D>
__global__ void convert_kernel(const S *x, D *y, long long n)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = D(x[i]);
}

template <typename T>
__global__ void __launch_bounds__(kThreads) dot_partial_kernel(const T *x, const T *y, long long n, double *partials)
{
  __shared__ double red[kThreads];
  double s = 0.;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    s += double(x[i]) * double(y[i]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(kThreads) dot_final_kernel(const double *partials, int n, double *result)
{
  __shared__ double red[kThreads];
  double s = 0.;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += partials[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *result = red[0];
}

// The passes of a CG iteration over r, q, z are bound by memory; each sums its
// inner products over the grid itself (grid_sums), so that an iteration has no
// launch for a final sum and no copy of the scalars to the host (Q4 32^3 FP64:
// five of those took 23 of 212 us).  The tickets of all workgroups meet at one
// address, 12 ns each (1049 workgroups of 256: r -= alpha q took 22.8 us), so the
// grid is one workgroup a CU, and every thread has kSumUnroll pairs of each vector
// in flight.  With 2.1e6 values: the update 13.3 us (before, with the final sum and
// the copy, 19.5), z.r and z.q 12.7 us (18.8); 256 x 1024 threads with 4 pairs 13.9
// and 13.8, 512 x 512 with 4 pairs 15.2 and 14.3.
constexpr int kSumThreads = 512, kSumUnroll = 8, kSumBlocks = 256;

static unsigned sum_grid(long long n)
{
  const long long b = (n + 2 * kSumThreads - 1) / (2 * kSumThreads);
  return (unsigned)(b < 1 ? 1 : (b < kSumBlocks ? b : kSumBlocks));
}

// sum over the workgroup's threads, in thread 0
__device__ __forceinline__ double block_sum(double t, double *red)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
  __syncthreads();
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = t;
  __syncthreads();
  t = 0.;
  if (threadIdx.x == 0)
    for (int w = 0; w < kSumThreads / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

template <typename T>
struct Pair {
  T x, y;
};

// r -= alpha q, alpha = *zr / *pq (device scalars: no host round trip),
// optionally rs = (float) r, *rr = r.r; the three scalars also to the host
__global__ void __launch_bounds__(kSumThreads) cg_update_kernel(long long n, const double *zr, const double *pq,
                                                                const double *q, double *r, float *rs, double *rr,
                                                                double *host, double *partials, unsigned *ticket)
{
  __shared__ double red[kSumThreads / 64 + 1];
  const double alpha = *zr / *pq;
  const long long t = blockIdx.x * (long long)kSumThreads + threadIdx.x, stride = gridDim.x * (long long)kSumThreads;
  const long long pairs = n / 2;
  Pair<double> *r2 = reinterpret_cast<Pair<double> *>(r);
  const Pair<double> *q2 = reinterpret_cast<const Pair<double> *>(q);
  Pair<float> *rs2 = reinterpret_cast<Pair<float> *>(rs);
  double acc = 0.;
  for (long long i0 = t; i0 < pairs; i0 += kSumUnroll * stride) {
    Pair<double> rv[kSumUnroll], qv[kSumUnroll];
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u)
      if (i0 + u * stride < pairs) rv[u] = r2[i0 + u * stride], qv[u] = q2[i0 + u * stride];
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u) {
      const long long i = i0 + u * stride;
      if (i >= pairs) break;
      rv[u].x -= alpha * qv[u].x;
      rv[u].y -= alpha * qv[u].y;
      r2[i] = rv[u];
      if (rs) rs2[i] = {float(rv[u].x), float(rv[u].y)};
      acc += rv[u].x * rv[u].x + rv[u].y * rv[u].y;
    }
  }
  if (n % 2 == 1 && t == 0) {
    const double v = r[n - 1] - alpha * q[n - 1];
    r[n - 1] = v;
    if (rs) rs[n - 1] = float(v);
    acc += v * v;
  }
  double sum[1] = {block_sum(acc, red)};
  if (grid_sums<1, kSumThreads>(sum, partials, ticket, blockIdx.x, gridDim.x, red)) {
    *rr = sum[0];
    const double h[3] = {*pq, sum[0], *zr};
    for (int i = 0; i < 3; ++i) __hip_atomic_store(host + i, h[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// z.r and z.q (z FP32 or FP64)
template <typename Z>
__global__ void __launch_bounds__(kSumThreads) dot2_kernel(long long n, const Z *z, const double *r, const double *q,
                                                           double *result, double *partials, unsigned *ticket)
{
  __shared__ double red[kSumThreads / 64 + 1];
  const long long t = blockIdx.x * (long long)kSumThreads + threadIdx.x, stride = gridDim.x * (long long)kSumThreads;
  const long long pairs = n / 2;
  const Pair<Z> *z2 = reinterpret_cast<const Pair<Z> *>(z);
  const Pair<double> *r2 = reinterpret_cast<const Pair<double> *>(r), *q2 = reinterpret_cast<const Pair<double> *>(q);
  double a = 0., b = 0.;
  for (long long i0 = t; i0 < pairs; i0 += kSumUnroll * stride) {
    Pair<Z> zv[kSumUnroll];
    Pair<double> rv[kSumUnroll], qv[kSumUnroll];
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u) {
      const long long i = i0 + u * stride;
      if (i < pairs) zv[u] = z2[i], rv[u] = r2[i], qv[u] = q2[i];
    }
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u) {
      if (i0 + u * stride >= pairs) break;
      a += double(zv[u].x) * rv[u].x + double(zv[u].y) * rv[u].y;
      b += double(zv[u].x) * qv[u].x + double(zv[u].y) * qv[u].y;
    }
  }
  if (n % 2 == 1 && t == 0) {
    a += double(z[n - 1]) * r[n - 1];
    b += double(z[n - 1]) * q[n - 1];
  }
  a = block_sum(a, red);
  double sum[2] = {a, block_sum(b, red)};
  if (grid_sums<2, kSumThreads>(sum, partials, ticket, blockIdx.x, gridDim.x, red)) {
    result[0] = sum[0];
    result[1] = sum[1];
  }
}

// the Lanczos vector passes of vec_lanczos_*
__global__ void lanczos_next_kernel(long long n, const double *w, const double *ww, const double *isq, double *v,
                                    double *t)
{
  const double f = 1. / sqrt(*ww);
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double vi = f * w[i];
    v[i] = vi;
    t[i] = vi * isq[i];
  }
}

__global__ void __launch_bounds__(kSumThreads) lanczos_dot_kernel(long long n, double *w, const double *isq,
                                                                  const double *v, double *alpha, double *partials,
                                                                  unsigned *ticket)
{
  __shared__ double red[kSumThreads / 64 + 1];
  double acc = 0.;
#pragma unroll 4
  for (long long i = blockIdx.x * (long long)kSumThreads + threadIdx.x; i < n;
       i += gridDim.x * (long long)kSumThreads) {
    const double wi = w[i] * isq[i];
    w[i] = wi;
    acc += wi * v[i];
  }
  double sum[1] = {block_sum(acc, red)};
  if (grid_sums<1, kSumThreads>(sum, partials, ticket, blockIdx.x, gridDim.x, red)) *alpha = sum[0];
}

__global__ void __launch_bounds__(kSumThreads) lanczos_update_kernel(long long n, double *w, const double *v,
                                                                     const double *v0, const double *alpha,
                                                                     const double *bb, double *ww, double *partials,
                                                                     unsigned *ticket)
{
  __shared__ double red[kSumThreads / 64 + 1];
  const double a = *alpha, b = bb ? sqrt(*bb) : 0.;
  double acc = 0.;
#pragma unroll 4
  for (long long i = blockIdx.x * (long long)kSumThreads + threadIdx.x; i < n;
       i += gridDim.x * (long long)kSumThreads) {
    double wi = w[i] - a * v[i];
    if (bb) wi -= b * v0[i];
    w[i] = wi;
    acc += wi * wi;
  }
  double sum[1] = {block_sum(acc, red)};
  if (grid_sums<1, kSumThreads>(sum, partials, ticket, blockIdx.x, gridDim.x, red)) *ww = sum[0];
}

template <typename T>
__global__ void axpby_kernel(long long n, T a, const T *x, T b, T *y)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = b != T(0) ? a * x[i] + b * y[i] : a * x[i]; // b == 0: y is write-only
}

// p = (double) zs + b p
__global__ void axpby_widen_kernel(long long n, const float *zs, double b, double *p)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = double(zs[i]) + b * p[i];
}

// x += a p, then p = z + b p (z FP32 or FP64; x, p FP64): the iterate's
// update of one CG iteration folded into the next search direction's pass.
// a = *an / *ad, b = -*bn / *ad (device scalars)
template <typename Z>
__global__ void xp_update_kernel(long long n, const double *an, const double *ad, const double *bn, const Z *z,
                                 double *p, double *x)
{
  const double a = *an / *ad, b = -*bn / *ad;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double pi = p[i];
    x[i] += a * pi;
    p[i] = double(z[i]) + b * pi;
  }
}

template <typename T>
__global__ void cheby_kernel(long long n, const T *au, const T *rhs, const T *sol_old, const T *diag,
                             T *sol_new, T *tm, T c_np, T c_tm)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    // a null au or sol_old stands for the zero vector (the first step of a
    // recurrence started from zero): not read
    const T res = (au ? au[i] : T(0)) - rhs[i];
    // c_tm == 0 starts a recurrence: the previous tm is not read
    const T t = (c_tm != T(0) ? c_tm * tm[i] : T(0)) + c_np * diag[i] * res;
    tm[i] = t;
    sol_new[i] = (sol_old ? sol_old[i] : T(0)) - t;
  }
}

// z = c a b (elementwise)
template <typename T>
__global__ void mul_scaled_kernel(long long n, T c, const T *a, const T *b, T *z)
{
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    z[i] = c * a[i] * b[i];
}

template <typename T>
__global__ void dirichlet_kernel(T *x, int gx, int gy, int gz)
{
  const long long n = (long long)gx * gy * gz;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int X = (int)(i % gx);
    const long long r = i / gx;
    const int Y = (int)(r % gy), Z = (int)(r / gy);
    if (X == 0 || Y == 0 || Z == 0 || X == gx - 1 || Y == gy - 1 || Z == gz - 1) x[i] = T(0);
  }
}

__global__ void layout_kernel(int n3, int nx, int ny, int nz, int lanes, const double *in, double *out,
                              int to_canonical)
{
  const long long total = (long long)nx * ny * nz * n3;
  const int nxb = nx / lanes;
  for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < total; g += (long long)gridDim.x * blockDim.x) {
    const int dof = (int)(g % n3);
    const long long cell = g / n3;
    const int ix = (int)(cell % nx);
    const long long r = cell / nx;
    const int iy = (int)(r % ny), iz = (int)(r / ny);
    const long long il =
        (((long long)iz * ny + iy) * nxb + ix / lanes) * (long long)lanes * n3 + (long long)dof * lanes + ix % lanes;
    if (to_canonical) out[g] = in[il];
    else out[il] = in[g];
  }
}

template <int N>
__global__ void apply1d_kernel(Eo<N, double> t, int sym, long long n_lines, long long line_stride, int stride,
                               const double *in, double *out)
{
  for (long long li = blockIdx.x * (long long)blockDim.x + threadIdx.x; li < n_lines; li += (long long)gridDim.x * blockDim.x) {
    double u[N], v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) u[i] = in[li * line_stride + (long long)i * stride];
    if (sym > 0) eo_apply<N, 1>(t, u, v);
    else eo_apply<N, -1>(t, u, v);
#pragma unroll
    for (int i = 0; i < N; ++i) out[li * line_stride + (long long)i * stride] = v[i];
  }
}
} // namespace

hipError_t vec_fill(bool fp32, void *x, long long n, double v, hipStream_t s)
{
  if (fp32) hipLaunchKernelGGL(fill_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (float *)x, n, (float)v);
  else hipLaunchKernelGGL(fill_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (double *)x, n, v);
  return hipGetLastError();
}

hipError_t vec_copy_convert(bool to_fp32, const void *x, void *y, long long n, hipStream_t s)
{
  if (to_fp32)
    hipLaunchKernelGGL((convert_kernel<double, float>), dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (const double *)x, (float *)y, n);
  else
    hipLaunchKernelGGL((convert_kernel<float, double>), dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (const float *)x, (double *)y, n);
  return hipGetLastError();
}

hipError_t vec_dot(bool fp32, const void *x, const void *y, long long n, double *result_dev, double *partials,
                   int n_partials, hipStream_t s)
{
  unsigned g = grid_for(n, 8);
  if ((int)g > n_partials) g = n_partials;
  if (fp32)
    hipLaunchKernelGGL(dot_partial_kernel<float>, dim3(g), dim3(kThreads), 0, s, (const float *)x, (const float *)y, n, partials);
  else
    hipLaunchKernelGGL(dot_partial_kernel<double>, dim3(g), dim3(kThreads), 0, s, (const double *)x, (const double *)y, n, partials);
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kThreads), 0, s, (const double *)partials, (int)g, result_dev);
  return hipGetLastError();
}

hipError_t vec_cg_update(long long n, const double *zr, const double *pq, const void *q, void *r, void *rs,
                         double *rr, double *host, double *partials, unsigned *ticket, hipStream_t s)
{
  hipLaunchKernelGGL(cg_update_kernel, dim3(sum_grid(n)), dim3(kSumThreads), 0, s, n, zr, pq, (const double *)q,
                     (double *)r, (float *)rs, rr, host, partials, ticket);
  return hipGetLastError();
}

hipError_t vec_dot2(bool z_fp32, long long n, const void *z, const void *r, const void *q, double *result_dev,
                    double *partials, unsigned *ticket, hipStream_t s)
{
  if (z_fp32)
    hipLaunchKernelGGL(dot2_kernel<float>, dim3(sum_grid(n)), dim3(kSumThreads), 0, s, n, (const float *)z,
                       (const double *)r, (const double *)q, result_dev, partials, ticket);
  else
    hipLaunchKernelGGL(dot2_kernel<double>, dim3(sum_grid(n)), dim3(kSumThreads), 0, s, n, (const double *)z,
                       (const double *)r, (const double *)q, result_dev, partials, ticket);
  return hipGetLastError();
}

hipError_t vec_lanczos_next(long long n, const void *w, const double *ww, const void *isq, void *v, void *t,
                            hipStream_t s)
{
  hipLaunchKernelGGL(lanczos_next_kernel, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (const double *)w, ww,
                     (const double *)isq, (double *)v, (double *)t);
  return hipGetLastError();
}

hipError_t vec_lanczos_dot(long long n, void *w, const void *isq, const void *v, double *alpha, double *partials,
                           unsigned *ticket, hipStream_t s)
{
  hipLaunchKernelGGL(lanczos_dot_kernel, dim3(sum_grid(n)), dim3(kSumThreads), 0, s, n, (double *)w,
                     (const double *)isq, (const double *)v, alpha, partials, ticket);
  return hipGetLastError();
}

hipError_t vec_lanczos_update(long long n, void *w, const void *v, const void *v0, const double *alpha,
                              const double *bb, double *ww, double *partials, unsigned *ticket, hipStream_t s)
{
  hipLaunchKernelGGL(lanczos_update_kernel, dim3(sum_grid(n)), dim3(kSumThreads), 0, s, n, (double *)w,
                     (const double *)v, (const double *)v0, alpha, bb, ww, partials, ticket);
  return hipGetLastError();
}

hipError_t vec_xp_update(bool z_fp32, long long n, const double *an, const double *ad, const double *bn,
                         const void *z, void *p, void *x, hipStream_t s)
{
  if (z_fp32)
    hipLaunchKernelGGL(xp_update_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, an, ad, bn,
                       (const float *)z, (double *)p, (double *)x);
  else
    hipLaunchKernelGGL(xp_update_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, an, ad, bn,
                       (const double *)z, (double *)p, (double *)x);
  return hipGetLastError();
}

hipError_t vec_axpby_widen(long long n, const void *zs, double b, void *p, hipStream_t s)
{
  hipLaunchKernelGGL(axpby_widen_kernel, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (const float *)zs, b, (double *)p);
  return hipGetLastError();
}

hipError_t vec_axpby(bool fp32, long long n, double a, const void *x, double b, void *y, hipStream_t s)
{
  if (fp32)
    hipLaunchKernelGGL(axpby_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (float)a, (const float *)x, (float)b, (float *)y);
  else
    hipLaunchKernelGGL(axpby_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, a, (const double *)x, b, (double *)y);
  return hipGetLastError();
}

hipError_t vec_mul_scaled(bool fp32, long long n, double c, const void *a, const void *b, void *z, hipStream_t s)
{
  if (fp32)
    hipLaunchKernelGGL(mul_scaled_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (float)c,
                       (const float *)a, (const float *)b, (float *)z);
  else
    hipLaunchKernelGGL(mul_scaled_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, c,
                       (const double *)a, (const double *)b, (double *)z);
  return hipGetLastError();
}

hipError_t vec_cheby_update(bool fp32, long long n, const void *au, const void *rhs, const void *sol_old,
                            const void *diag, void *sol_new, void *tm, double c_np, double c_tm, hipStream_t s)
{
  if (fp32)
    hipLaunchKernelGGL(cheby_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (const float *)au,
                       (const float *)rhs, (const float *)sol_old, (const float *)diag, (float *)sol_new, (float *)tm,
                       (float)c_np, (float)c_tm);
  else
    hipLaunchKernelGGL(cheby_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, n, (const double *)au,
                       (const double *)rhs, (const double *)sol_old, (const double *)diag, (double *)sol_new,
                       (double *)tm, c_np, c_tm);
  return hipGetLastError();
}

hipError_t vec_zero_dirichlet(bool fp32, void *x, const int g[3], hipStream_t s)
{
  const long long n = (long long)g[0] * g[1] * g[2];
  if (fp32) hipLaunchKernelGGL(dirichlet_kernel<float>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (float *)x, g[0], g[1], g[2]);
  else hipLaunchKernelGGL(dirichlet_kernel<double>, dim3(grid_for(n, 4)), dim3(kThreads), 0, s, (double *)x, g[0], g[1], g[2]);
  return hipGetLastError();
}

hipError_t layout_convert(int degree, const int nc[3], int lanes, const double *in, double *out, bool to_canonical,
                          hipStream_t s)
{
  const int n = degree + 1;
  const long long total = (long long)nc[0] * nc[1] * nc[2] * n * n * n;
  hipLaunchKernelGGL(layout_kernel, dim3(grid_for(total, 4)), dim3(kThreads), 0, s, n * n * n, nc[0], nc[1], nc[2],
                     lanes, in, out, to_canonical ? 1 : 0);
  return hipGetLastError();
}

// y = x w_q: bound by memory; kWeightRounds coalesced values per thread, the
// position in the cell of a workgroup's first value is uniform and the threads'
// follow by 32-bit arithmetic.  Takes the place of a device copy when a
// coefficient is set and saves every later apply one multiplication per q-point
// (Q8, 8e6 nodes: FP32 15.1 us, the copy 13.4; FP64 28.5 us, the copy 31.9; with
// the weights loaded before the values 16.8 and 30.5.  Set and one apply together
// take no longer than a copy and the apply that multiplied).
constexpr int kWeightRounds = 8;
template <int N, typename T>
__global__ void __launch_bounds__(kThreads) weight_kernel(const DevTab<N, T> *dt, const T *x, T *y, long long n)
{
  constexpr unsigned N3 = N * N * N;
  const long long i0 = blockIdx.x * (long long)(kThreads * kWeightRounds);
  const unsigned q0 = (unsigned)(i0 % N3);
  T v[kWeightRounds];
#pragma unroll
  for (int r = 0; r < kWeightRounds; ++r) {
    const long long i = i0 + r * kThreads + threadIdx.x;
    v[r] = x[i < n ? i : n - 1];
  }
  // the weights while the values are on their way
  const auto &w = ctab(dt).w;
  __shared__ T sw[N];
  if (threadIdx.x < N) sw[threadIdx.x] = w[threadIdx.x];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kWeightRounds; ++r) {
    const long long i = i0 + r * kThreads + threadIdx.x;
    const unsigned q = (q0 + r * kThreads + threadIdx.x) % N3;
    if (i < n) y[i] = v[r] * (sw[q % N] * (sw[q / N % N] * sw[q / (N * N)]));
  }
}

hipError_t weight_qdata(int n, bool fp32, const void *dtab, const void *x, void *y, long long count, hipStream_t s)
{
  const long long blocks = (count + kThreads * kWeightRounds - 1) / (kThreads * kWeightRounds);
  if (blocks <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const unsigned g = (unsigned)blocks;
  switch (n) {
#define SFK_CASE(NN)                                                                                             \
  case NN:                                                                                                       \
    if (fp32)                                                                                                    \
      hipLaunchKernelGGL((weight_kernel<NN, float>), dim3(g), dim3(kThreads), 0, s,                              \
                         (const DevTab<NN, float> *)dtab, (const float *)x, (float *)y, count);                  \
    else                                                                                                         \
      hipLaunchKernelGGL((weight_kernel<NN, double>), dim3(g), dim3(kThreads), 0, s,                             \
                         (const DevTab<NN, double> *)dtab, (const double *)x, (double *)y, count);               \
    break;
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int N, typename T>
static hipError_t upload_devtab(const Tables1D &t, void **dev)
{
  const DevTab<N, T> h = make_devtab<N, T>(t);
  hipError_t e = hipMalloc(dev, sizeof(h));
  if (e != hipSuccess) {
    *dev = nullptr;
    return e;
  }
  return hipMemcpy(*dev, &h, sizeof(h), hipMemcpyHostToDevice);
}

hipError_t upload_device_tables(const Tables1D &t, bool fp32, void **dev)
{
  switch (t.n) {
#define SFK_CASE(NN) \
  case NN: return fp32 ? upload_devtab<NN, float>(t, dev) : upload_devtab<NN, double>(t, dev);
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
}

hipError_t apply_1d(int nn, const std::vector<double> &M, int sym, bool forward, long long n_lines,
                    long long line_stride, int stride, const double *in, double *out, hipStream_t s)
{
  const unsigned g = grid_for(n_lines);
  switch (nn) {
#define SFK_CASE(NN)                                                                                          \
  case NN:                                                                                                    \
    hipLaunchKernelGGL(apply1d_kernel<NN>, dim3(g), dim3(kThreads), 0, s, make_eo<NN, double>(M, forward), sym, \
                       n_lines, line_stride, stride, in, out);                                                \
    break;
    SFK_CASE(2) SFK_CASE(3) SFK_CASE(4) SFK_CASE(5) SFK_CASE(6) SFK_CASE(7) SFK_CASE(8) SFK_CASE(9) \
    SFK_CASE(10) SFK_CASE(11) SFK_CASE(12) SFK_CASE(13) SFK_CASE(14) SFK_CASE(15) SFK_CASE(16)
#undef SFK_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

} // namespace sfk
