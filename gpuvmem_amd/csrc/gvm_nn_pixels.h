// Pixel positions of the weight gradient's chunks (gvm_nn.hip).  Plain integer code that
// the host compiles too, so that a test can walk it.
#pragma once

namespace gvm {

constexpr int kWgradChunk = 128;  // pixels staged at a time

// Linear pixel index of a batch as (image, pixel of its plane), advanced by chunks.  q may
// start before the first pixel; 0 <= p < HW at all times.
struct PixelPos {
  int q, b, p;
  constexpr void start(int q0, int HW) {
    q = q0;
    b = q0 / HW;
    p = q0 - b * HW;
    if (p < 0) {
      p += HW;
      b--;
    }
  }
  // step_b, step_p: kWgradChunk pixels as whole images and pixels of the next.  (A chunk
  // may hold many images: a loop over them took 156 us for 1,000 x 1,000 channels of one
  // pixel.)
  constexpr void next(int HW, int step_b, int step_p) {
    q += kWgradChunk;
    b += step_b;
    p += step_p;
    if (p >= HW) {
      p -= HW;
      b++;
    }
  }
  // the pixel `shift` away in the same plane, or -1: none, or no pixel of the batch
  constexpr int shifted(int shift, int HW, int npix) const {
    const int s = p + shift;
    return q >= 0 && q < npix && s >= 0 && s < HW ? s : -1;
  }
};

}  // namespace gvm
