// fs_conv_rows.h -- byte offsets into the few input rows that a tile of a
// 3x3 convolution reads, for buffer loads whose offsets have 32 bits.  An
// image may be larger than they reach (8 columns of 128 channels: from 2^20
// rows on), its rows around a tile are not: offsets count from the first of them.
#ifndef FS_CONV_ROWS_H
#define FS_CONV_ROWS_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fs {

// Rows y0 - 1 .. y0 + rows of an image of H rows, those of them inside it, in a
// source at half the resolution when up.
struct ConvRows {
  int64_t start;     // of the first row, in bytes from the image's
  uint32_t bytes;    // from there to the end of the last
  uint32_t skip;     // start, modulo 2^32
};
__host__ __device__ inline ConvRows conv_rows(int y0, int rows, int H, int up, int rowbytes) {
  const int first = (y0 > 0 ? y0 - 1 : 0) >> up, last = (y0 + rows < H ? y0 + rows : H - 1) >> up;
  ConvRows r;
  r.start = static_cast<int64_t>(first) * rowbytes;
  r.bytes = static_cast<uint32_t>(last - first + 1) * static_cast<uint32_t>(rowbytes);
  r.skip = static_cast<uint32_t>(first) * static_cast<uint32_t>(rowbytes);
  return r;
}

// Offset of row y (full resolution) from the window's start.
__host__ __device__ inline uint32_t conv_row_offset(int y, int up, uint32_t rowbytes,
                                                    uint32_t skip) {
  return static_cast<uint32_t>(y >> up) * rowbytes - skip;
}

}  // namespace fs

#endif
