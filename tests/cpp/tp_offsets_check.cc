// The tensor-product kernel's y-line offsets (sfk_tp_offsets.h) on meshes at
// the limit of what it takes: with the range rule of raw buffer accesses (lane
// offset below num_records minus the uniform offset), every interior node of a
// line must be read at its own address and every other entry must be out of
// range.  Prints the first violation.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "sfk_tp_offsets.h"

using namespace sfk;

static bool check(int p, int es, int nx, int ny)
{
  const int n = p + 1, gx = nx * p + 1, gy = ny * p + 1, plane = gx * gy;
  const long long row_bytes = (long long)gx * es;
  for (int below = 0; below < 2; ++below) // the layer's planes 1..p, and plane 0 (its offsets: ys = 0)
    for (int ys : {0, p - 1})
      for (int ey : {0, 1, 2, 3, ny / 2, ny - 2, ny - 1, ny, ny + 1})
        for (int X : {-1, 0, 1, p, gx / 2, gx - 2, gx - 1, gx}) {
          if (ey < 0 || (below && ys != 0)) continue;
          const TpLine o = tp_line(p, es, gx, ny, plane, ys, ey, X);
          const long long base = tp_line_base(p, gx, below ? 0 : plane);
          for (int j = 0; j < 2 * n - 1; ++j) {
            const unsigned v = j == 0 ? o.first : (j <= p ? o.low : (j < 2 * p ? o.mid : o.last));
            const long long u = j * row_bytes, row = (long long)(ey - 1) * p + j;
            const bool node = ey < ny && X > 0 && X < gx - 1 && row > 0 && row < gy - 1;
            const bool in_range = (long long)v + u + es <= (long long)kAll;
            const bool out_of_range = (long long)v >= (long long)kAll - u;
            const long long z = below ? 0 : 1 + ys;
            const long long want = (z * plane + row * gx + X) * es;
            const bool ok = node ? in_range && base * es + v + u == want : out_of_range;
            if (!ok) {
              std::printf("p %d, %d bytes, %d x %d cells: plane %lld row %lld column %d (ey %d): offset %u + %lld\n", p,
                          es, nx, ny, z, row, X, ey, v, u);
              return false;
            }
          }
        }
  return true;
}

int main()
{
  int bad = 0, count = 0;
  for (int p = 1; p <= 8; ++p)
    for (int es : {4, 8})
      for (int nx : {1, 2, 3, 63, 64, 682, 1831, 4001, 20011}) {
        // the largest ny that the kernel takes with this nx
        const int gx = nx * p + 1, n = p + 1;
        const long long most = ((1LL << 31) - 1) / ((long long)n * gx * es);
        int ny = (int)((most - 1) / p);
        while (ny > 0 && !tp_offsets_fit(n, gx, ny * p + 1, es)) --ny;
        if (ny < 1) continue;
        if (tp_offsets_fit(n, gx, (ny + 1) * p + 1, es)) {
          std::printf("p %d nx %d: the limit moved\n", p, nx);
          ++bad;
        }
        for (int m : {ny, ny - 1, ny - 7, ny / 2, 3, 2, 1})
          if (m >= 1) ++count, bad += !check(p, es, nx, m);
      }
  std::printf("%d meshes, %d violations\n", count, bad);
  return bad ? EXIT_FAILURE : EXIT_SUCCESS;
}
