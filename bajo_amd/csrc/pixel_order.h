// The order in which a camera launch of the top level takes its pixels.
// (Host code can include it by itself.)
#pragma once

#include <stdint.h>

#ifndef BJ_HD
#define BJ_HD inline
#endif

namespace bj {

// The pixel that index r of a camera launch of R < 2^31 rays traces: views in
// order, a view in tiles of 8 x 8 pixels (narrower and lower ones at its right
// and bottom edges), so that a wave's rays stay close together and walk the
// same nodes (256 instances of a 67,280-triangle mesh, three 640 x 360 views:
// 426 us against 482 row by row).  A view that the launch cuts short is traced
// row by row.  A view of several bands of rows is less than 2^28 pixels wide,
// so 32 bits hold a band's pixels; one band may be as wide as the launch.
BJ_HD uint64_t camera_pixel(uint64_t r, uint64_t R, uint32_t w, uint32_t h) {
  const uint64_t ppv = (uint64_t)w * h;
  const uint64_t start = r / ppv * ppv;
  if (start + ppv > R) return r;
  uint32_t k = (uint32_t)(r - start);
  const uint32_t band = h > 8u ? k / (8u * w) : 0u;
  k -= band * 8u * w;
  const uint32_t rows = h - 8u * band < 8u ? h - 8u * band : 8u;
  const uint32_t tile = k / (8u * rows);
  k -= tile * 8u * rows;
  const uint32_t cols = w - 8u * tile < 8u ? w - 8u * tile : 8u;
  const uint32_t y = k / cols, x = k - y * cols;
  return start + (uint64_t)(8u * band + y) * w + 8u * tile + x;
}

}  // namespace bj
