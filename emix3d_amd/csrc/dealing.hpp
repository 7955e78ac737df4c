// Which line group a workgroup of the line solvers takes.  Workgroups go to
// the eight XCDs round robin by their linear id, each XCD with its own L2;
// the functions here choose the groups so that those sharing cache lines
// meet in one L2.  Include after emx_internal.hpp.
#pragma once

namespace emx {

// Line group of workgroup x (of gx along the lines) for LG lines per
// wavefront, for workgroups in their round-robin order.  A group of 8
// doubles (64 bytes) shares each 128-byte cache line with its neighbour: the
// two halves of a line go to workgroups whose ids differ by 8, the same XCD,
// dispatched together.
template <int LG>
__host__ __device__ __forceinline__ int line_group(int x, int gx) {
  if constexpr (LG >= 16) {
    return x;
  } else {
    const int base = x & ~15;
    if (base + 16 > gx) return x;  // the last, incomplete set of 16
    const int r = x & 15;
    return base + 2 * (r & 7) + (r >> 3);
  }
}

// Workgroup local (of ngroup in its grid) -> line group g, row-major over
// (group along the lines, outer index).  A grid's rows start anywhere in a
// 128-byte cache line (its nx is any size), so neighbouring groups along a
// row share a cache line at every point.  Within each set of 8K workgroups
// (K = 16, fewer in the grid's last set), XCD x takes the K consecutive
// groups xK .. xK+K-1, in order, so that all but one of their shared lines
// are fetched once into that XCD's L2 and read there by the neighbour
// dispatched next.  A bijection on [0, ngroup): the last local % 8 ids of
// the grid keep their own group.
__host__ __device__ __forceinline__ int xcd_run_group(int local, int ngroup) {
  constexpr int K = 16;
  const int base = local & ~(8 * K - 1);
  const int left = (ngroup - base) >> 3;  // groups per XCD in this set
  const int k = left < K ? left : K;
  const int r = local - base;
  if (r >= 8 * k) return local;
  return base + (r & 7) * k + (r >> 3);
}

// The part z, line group x and outer index y of workgroup (x, y, z) of a
// (gx, gy, gz) launch, in place.
//
// run: groups are dealt by xcd_run_group, for launches of more workgroups
// than the chip holds at once.  Rows that start inside a cache line share it
// with their neighbours (stage at 187 x 151 x 129: 1183 us round robin,
// 1139 us in runs), and where they do not, a run's neighbouring segments
// still arrive in order (256^3: 4165 and 4073 us).  A small launch would
// only pay for the divisions (64^3 gradient and divergence: 43.2 us round
// robin, 43.7 us in runs).  INTERLEAVED: the parts of a group read fields in
// common and run next to each other.
template <int LG, bool INTERLEAVED>
__host__ __device__ __forceinline__ void deal_lines(int run, int gx, int gy, int gz, int& x,
                                                    int& y, int& z) {
  if (!run) {
    x = line_group<LG>(x, gx);
    return;
  }
  int g;
  if constexpr (INTERLEAVED) {
    g = xcd_run_group(x + gx * (y + gy * z), gx * gy * gz);
    z = g % gz;
    g /= gz;
  } else {
    g = xcd_run_group(x + gx * y, gx * gy);
  }
  x = g % gx;
  y = g / gx;
}

}  // namespace emx
