// CPU check of csrc/fs_conv_rows.h against 64-bit offsets from the image's start:
// every row a tile reads, on images up to four times larger than 32-bit offsets
// reach.  Built by tests/test_conv_rows.py with hipcc's host pass.  Prints
// "rows mismatches rows-beyond-4-GiB".
#include <cstdint>
#include <cstdio>

#include "fs_conv_rows.h"

int main() {
  long rows = 0, bad = 0, far = 0;
  for (int H : {2, 4, 6, 8, 30, 1 << 10, (1 << 20) + 2, 3 << 20, (1 << 23) - 2, 1 << 24})
    for (int up = 0; up < 2; up++)
      for (int rowbytes : {64, 256, 1024, 2048, 5120}) {
        const int64_t image = static_cast<int64_t>(H >> up) * rowbytes;
        for (int k = 0; k < 200; k++) {
          // tiles of two rows: from the top, from the bottom, spread between
          const int n = H / 2, q = k < 50 ? k : k < 100 ? n - 1 - (k - 50) : static_cast<int>(
              static_cast<int64_t>(n) * (k - 100) / 100);
          if (q < 0 || q >= n) continue;
          const int y0 = 2 * q;
          const fs::ConvRows w = fs::conv_rows(y0, 2, H, up, rowbytes);
          if (w.start < 0 || w.start + w.bytes > image) bad++;
          for (int yy = y0 - 1; yy <= y0 + 2; yy++) {
            if (yy < 0 || yy >= H) continue;
            const uint32_t at = fs::conv_row_offset(yy, up, static_cast<uint32_t>(rowbytes), w.skip);
            const int64_t want = static_cast<int64_t>(yy >> up) * rowbytes;
            rows++;
            far += want >= 1ll << 32;
            if (w.start + at != want || static_cast<int64_t>(at) + rowbytes > w.bytes ||
                at >= 0x7FFF0000u)
              bad++;
          }
        }
      }
  std::printf("%ld %ld %ld\n", rows, bad, far);
  return 0;
}
