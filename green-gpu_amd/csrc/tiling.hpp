// Workgroup -> output-tile mapping shared by the GEMM kernels.
#pragma once

#include "zgemm.hpp"

namespace ggpu {

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2); the linear id is remapped so that every XCD receives a contiguous range
// of logical tiles, ordered m-tile fastest, then n-tile, then batch: the
// workgroups that share a B panel (same n-tile) and an A panel (same batch)
// run on the same XCD at the same time.
constexpr int NXCD = 8;
__device__ inline int64_t xcd_logical(int64_t id, int64_t total) {
  const int64_t xcd = id % NXCD, slot = id / NXCD;
  const int64_t per = total / NXCD, rem = total % NXCD;
  return (xcd < rem) ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
}

// Logical tile -> (m-tile, n-tile, batch b0, batch b1).  Default order:
// m-tile fastest, then n-tile, then batch b1, then b0.  With d.batch_major b0
// runs fastest and b1 slowest: chosen when every b0 shares A, so the
// workgroups reusing one A panel run back to back and find it in L2 instead of
// re-reading A from memory once per batch.
struct TileCoord { int mt, nt; int64_t b0, b1; };
__device__ inline TileCoord tile_coord(const GemmDesc& d, int tiles_m, int tiles_n) {
  int64_t lg = xcd_logical(blockIdx.x, gridDim.x);
  TileCoord c;
  if (d.batch_major) {
    c.b0 = lg % d.nb0;
    lg /= d.nb0;
    c.mt = (int)(lg % tiles_m);
    lg /= tiles_m;
    c.nt = (int)(lg % tiles_n);
    c.b1 = lg / tiles_n;
  } else {
    c.mt = (int)(lg % tiles_m);
    lg /= tiles_m;
    c.nt = (int)(lg % tiles_n);
    lg /= tiles_n;
    c.b1 = lg % d.nb1;
    c.b0 = lg / d.nb1;
  }
  return c;
}

}  // namespace ggpu
