// Two-factor FFT passes, one mesh, FP32.
#define P3M_FFT_TWO_SINGLE
#include "fft_two_launch.hpp"

namespace p3m {
namespace fft {
P3M_INST(float)
}  // namespace fft
}  // namespace p3m
