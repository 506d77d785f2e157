// The automatic tile of the tensor-product kernel is one that sfk_op_set_schedule
// and sfk_tune accept under the same LDS limit (tp_shape_fits), for every limit
// under which there is one; and fewer CUs are counted with.  Without a device.
#include <cstdio>
#include <cstdlib>

#include "sfk_kernels.h"

using namespace sfk;

int main()
{
  int bad = 0, none = 0;
  const int meshes[][3] = {{1, 1, 1}, {16, 16, 16}, {64, 64, 64}, {101, 67, 90}};
  for (int n = 2; n <= 9; ++n)
    for (bool fp32 : {false, true})
      for (const auto &nc : meshes)
        for (size_t lds : {size_t(32768), size_t(65536), size_t(98304), size_t(131072), size_t(163840)}) {
          bool any = false;
          for (int sh = 1; sh < tp_shape_count(n); ++sh) any = any || tp_shape_fits(n, sh, fp32, lds);
          int shape = 0, zc = 0;
          tp_plan(n, fp32, nc, Chip{lds, 256}, &shape, &zc);
          none += !any;
          if (shape >= 1 && shape < tp_shape_count(n) && zc >= 1 && (!any || tp_shape_fits(n, shape, fp32, lds)))
            continue;
          std::printf("n %d, %s, %zu bytes: tile %d, %d cells\n", n, fp32 ? "FP32" : "FP64", lds, shape, zc);
          ++bad;
        }
  const int nc[3] = {64, 64, 64};
  if (!(tp_cost(7, nc, 1, 64, Chip{163840, 32}) > tp_cost(7, nc, 1, 64, Chip{163840, 256}))) ++bad;
  std::printf("%d violations, %d cases without a tile\n", bad, none);
  return bad ? EXIT_FAILURE : EXIT_SUCCESS;
}
