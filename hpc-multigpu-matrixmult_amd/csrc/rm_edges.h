// Rules of the row-major GEMM tiles at the ends of matrices and launches (gemm_rm.h), as plain
// arithmetic that host code can ask too.
#pragma once

#ifdef __HIPCC__
#define RM_BOTH __host__ __device__ __forceinline__
#else
#define RM_BOTH inline
#endif

// The last k rows of B whose 16-byte loads (CH elements) may end past the last row's end, so that
// they are taken element by element. Row r of K reaches past it by over - (K - 1 - r) * ldb
// elements, over = CH - n % CH: with ldb below over, a row before the last reaches past it too
// (n = ldb = 1 in FP32: the last three). `aligned`: all rows of B start on 16-byte boundaries, and
// a load past n ends on the boundary behind the row's last element, in memory that holds the row.
template <int CH>
RM_BOTH int rm_checked_rows(int n, long ldb, bool aligned) {
  const int over = n % CH ? CH - n % CH : 0;
  if (over == 0 || aligned) return 0;
  return over <= ldb ? 1 : over <= 2 * ldb ? 2 : 3;
}

// Workgroups of a launch over `total` tiles: `wanted` of them, or, at 0, one per tile. HIP launches
// fewer than 2^32 threads in one dimension, which a column of more than 2^30 rows would exceed
// (256 rows a tile, 1024 threads): then as many as there can be, a whole number of them on each of
// the 8 XCDs, walk the tiles.
inline int rm_grid(int wanted, int total, int threads) {
  const int most = (int)(0xffffffffu / (unsigned)threads / 8 * 8);
  const int g = wanted > 0 && wanted < total ? wanted : total;
  return g < most ? g : most;
}
