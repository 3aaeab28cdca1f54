// Walks the weight gradient's pixel positions as a loader wave does and checks
// that each stays the position of its linear index and that every shifted pixel lies
// in the batch.
#include <cstdio>
#include <initializer_list>

#include "gvm_nn_pixels.h"

int main() {
  using gvm::PixelPos;
  constexpr int kRange = 8192, kChunk = gvm::kWgradChunk;
  long checked = 0;
  for (int H = 1; H <= 20; H++)
    for (int W = 1; W <= 20; W++)
      for (int B : {1, 2, 3, 8, 16, 33, 64, 130, 1024}) {
        const int HW = H * W, npix = B * HW;
        const int step_b = kChunk / HW, step_p = kChunk % HW;
        for (int kbeg = 0; kbeg < npix; kbeg += kRange) {
          const int kend = npix < kbeg + kRange ? npix : kbeg + kRange;
          const int chunks = (kend - kbeg + kChunk - 1) / kChunk;
          for (int first : {-1, 0, 62, 63, 64, 126, 127, 128}) {
            PixelPos pos{};
            pos.start(kbeg + first, HW);
            for (int c = 0; c <= chunks + 1; c++) {  // two chunks are loaded ahead
              if (pos.q != kbeg + first + c * kChunk || pos.p < 0 || pos.p >= HW ||
                  (long)pos.b * HW + pos.p != pos.q) {
                std::printf("%d x %d x %d: q %d b %d p %d\n", B, H, W, pos.q, pos.b, pos.p);
                return 1;
              }
              for (int shift : {-W, 0, W}) {
                const int s = pos.shifted(shift, HW, npix);
                if (s < 0) continue;
                checked++;
                if (s >= HW || pos.b < 0 || pos.b >= B) {
                  std::printf("%d x %d x %d: reads pixel %d of image %d\n", B, H, W, s, pos.b);
                  return 1;
                }
              }
              pos.next(HW, step_b, step_p);
            }
          }
        }
      }
  std::printf("ok %ld\n", checked);
  return 0;
}
