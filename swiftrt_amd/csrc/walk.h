// The order in which a launch's workgroups take the tiles of a result (gemm_waves.h, gemm_short.h): host arithmetic, plain C++.
#pragma once
#include <stdint.h>

namespace srt {
namespace waves {

// Workgroup id runs on XCD id % 8 (each has its own L2), which takes the id / 8-th of its consecutive eighth of the tiles, the shorter
// side of the grid of tiles fastest, so that an XCD's tiles share rows and columns (along_rows: always the columns of tiles fastest).
struct Walk {
  uint32_t tiles, chunk;    // in total, per XCD
  uint32_t fast, slow;      // extents of the grid of tiles, in walk order
  uint32_t fast_rcp, slow_rcp;   // ceil(2^32 / extent): quotients of indexes below 2^16 by one multiplication (0: divide)
  int fast_is_m;
};

// A launch counts its threads in 32 bits along each dimension of the grid.
constexpr uint64_t kMostThreads = (1ull << 32) - 1;
constexpr uint32_t kWalkThreads = 256;   // of a workgroup of a walk too long for one tile a unit (those of 512 threads have no more tiles than units)

inline Walk make_walk(int M, int N, int batch, int edge, bool along_rows = false) {
  Walk w;
  const uint32_t tm = ((uint32_t)M + (uint32_t)edge - 1) / (uint32_t)edge, tn = ((uint32_t)N + (uint32_t)edge - 1) / (uint32_t)edge;
  w.fast_is_m = tm <= tn && !along_rows;
  w.fast = w.fast_is_m ? tm : tn;
  w.slow = w.fast_is_m ? tn : tm;
  const uint64_t matrix = (uint64_t)tm * tn, most = kMostThreads / kWalkThreads / 8 * 8;   // (whole eighths: 8 chunk workgroups run)
  w.tiles = matrix <= most / (uint64_t)batch ? (uint32_t)(matrix * (uint64_t)batch) : 0u;   // (0: too many for the walk's one grid dimension)
  w.chunk = (w.tiles + 7) / 8;
  // (exact while index x extent < 2^32: the reciprocal is too large by less than extent / 2^32)
  auto rcp = [&](uint32_t d) { return w.tiles <= 0xffffu && d > 1 ? (uint32_t)((0x100000000ull + d - 1) / d) : 0u; };
  w.fast_rcp = rcp(w.fast);
  w.slow_rcp = rcp(w.slow);
  return w;
}

}  // namespace waves
}  // namespace srt
