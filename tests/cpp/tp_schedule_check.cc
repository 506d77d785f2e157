// The tensor-product launches of an operator with an automatic schedule: what
// they run on is the cost model's choice, and filling a launch does not ask the
// model again (it allocates; nothing may be allocated here); and the tile that
// sfk_op_tile_shape names for tile_shape 0 is the one they run on.  Without a
// device.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "sfk_op.h"

static long g_allocations = 0;
void *operator new(std::size_t n)
{
  ++g_allocations;
  void *p = std::malloc(n ? n : 1);
  if (!p) std::abort();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

using namespace sfk;

static int check(sfk_op *op, bool cheby, int shape, int zc)
{
  TpLaunch L;
  const long before = g_allocations;
  for (int i = 0; i < 100; ++i) fill_tp_launch(op, L, cheby);
  const long allocated = g_allocations - before;
  const int n = op->d.degree + 1;
  tp_plan(n, op->d.precision == SFK_FP32, op->d.n_cells, current_chip(), &shape, &zc);
  if (allocated == 0 && L.shape == shape && L.zc == zc) return 0;
  std::printf("degree %d, %d cells in z, %s: tile %d, %d cells (planned %d, %d), %ld allocations in 100 launches\n",
              n - 1, op->d.n_cells[2], cheby ? "Chebyshev" : "matvec", L.shape, L.zc, shape, zc, allocated);
  return 1;
}

static int check_tile(sfk_op *op)
{
  TpLaunch L;
  fill_tp_launch(op, L);
  int bx = 0, by = 0, lx = 0, ly = 0;
  tp_shape(op->d.degree + 1, L.shape, &lx, &ly);
  if (sfk_op_tile_shape(op, 0, nullptr, &bx, &by) == SFK_OK && bx == lx && by == ly) return 0;
  std::printf("degree %d, %d cells in z, z_cells %d: tile 0 is %d x %d, the launch's %d x %d\n", op->d.degree,
              op->d.n_cells[2], op->tp_zc, bx, by, lx, ly);
  return 1;
}

int main()
{
  int bad = 0;
  const int meshes[][3] = {{1, 1, 1}, {3, 2, 5}, {16, 16, 16}, {101, 67, 90}, {128, 128, 128}};
  for (int degree = 1; degree <= 8; ++degree)
    for (const auto &nc : meshes)
      for (int prec : {SFK_FP64, SFK_FP32}) {
        sfk_op_desc d{};
        d.kind = SFK_CONT_LAPLACE;
        d.degree = degree;
        d.basis = SFK_BASIS_GLL;
        d.geometry = SFK_GEOM_CARTESIAN;
        d.precision = prec;
        d.n_rhs = 1;
        for (int k = 0; k < 3; ++k) d.n_cells[k] = nc[k], d.inv_jac[k] = 1.;
        sfk_op *op = nullptr;
        if (sfk_op_create(&d, &op) != SFK_OK) return std::printf("create: %s\n", sfk_last_error()), EXIT_FAILURE;
        for (bool cheby : {false, true}) bad += check(op, cheby, 0, 0);
        bad += check_tile(op);
        for (int asked : {0, 1, 2})
          for (int zc : {0, 2}) {
            const sfk_schedule s{0, 1, 2, asked, zc};
            if (sfk_op_set_schedule(op, &s) != SFK_OK) return std::printf("set: %s\n", sfk_last_error()), EXIT_FAILURE;
            for (bool cheby : {false, true}) bad += check(op, cheby, asked, zc);
            if (asked == 0) bad += check_tile(op);
          }
        sfk_op_destroy(op);
      }
  std::printf("%d violations\n", bad);
  return bad ? EXIT_FAILURE : EXIT_SUCCESS;
}
