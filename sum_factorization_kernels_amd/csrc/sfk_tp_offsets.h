// Byte offsets of the tensor-product kernel's buffer accesses (plain C++, no
// HIP).  A raw buffer access is in range where the lane's offset is below
// num_records minus the uniform offset; lanes without work carry kOob, which
// is beyond every buffer described here.
#pragma once

namespace sfk {

constexpr unsigned kOob = 0x80000000u, kAll = 0x7fffffffu;

// Meshes the kernel takes: the p+1 planes of a layer (gx x gy nodes of es
// bytes) hold less than 2^31 bytes.
constexpr bool tp_offsets_fit(int n, int gx, int gy, int es) { return (long long)n * gx * gy * es < (1LL << 31); }

// A thread's y line is column X of the layer's plane 1 + ys, rows (ey-1) p ..
// (ey+1) p.  Its entry j is at the lane offset below plus j rows, counted from
// element tp_line_base of the layer: row -p of plane 1, so that offsets are
// never negative and all that a layer reads ends below p planes and p rows of
// it, which the mesh limit above covers (counted from plane 0, the last rows of
// the last plane lay beyond 2^31 bytes on the largest meshes and read 0).
// Entry 0 is a node with a value if ey >= 2, entries 1..p if ey >= 1, the last
// one if the cell is not the last in y; the others are Dirichlet nodes or
// outside the grid.
struct TpLine {
  unsigned first, low, mid, last;
};
constexpr long long tp_line_base(int p, int gx, int plane) { return plane - (long long)p * gx; }
constexpr TpLine tp_line(int p, int es, int gx, int ny, int plane, int ys, int ey, int X)
{
  const bool ok = ey < ny && X > 0 && X < gx - 1;
  const unsigned o = ((unsigned)ys * (unsigned)plane + (unsigned)ey * (unsigned)p * (unsigned)gx + (unsigned)X) * (unsigned)es;
  return {ok && ey >= 2 ? o : kOob, ok && ey >= 1 ? o : kOob, ok ? o : kOob, ok && ey + 1 < ny ? o : kOob};
}

} // namespace sfk
