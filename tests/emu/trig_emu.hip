// Host build of device_trig.h's double-precision functions (test infrastructure).
#include <cstdint>

#include "../../axomae_amd/csrc/device_trig.h"

using namespace nova_hip;

// The float results for n arguments: sin and cos of x, acos of y and atan2(y, x), four floats each.
extern "C" void emu_trig(const float *x, const float *y, int64_t n, float *out) {
  for (int64_t i = 0; i < n; i++) {
    sincos_turns(x[i], out[4 * i], out[4 * i + 1]);
    out[4 * i + 2] = (float)acos_moderate(y[i]);
    out[4 * i + 3] = (float)atan2_moderate(y[i], x[i]);
  }
}
