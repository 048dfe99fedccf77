// Private to the library: the LDS-staged 3x3 convolution (nx_conv.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nx {
// y = [relu](conv3x3(x, w) + bias), arguments as nx_conv3x3_fwd; false if no
// kernel takes these channels or pointers or the pixels are too few to pay,
// else true with the launch's status in *err.  Bitwise k_conv3x3's results.
bool conv3x3_lds(const uint16_t* x, const uint16_t* w, const float* bias, uint16_t* y, int n,
                 int h, int wd, int cin, int cout, int relu, hipStream_t s, hipError_t* err);
}  // namespace nx
