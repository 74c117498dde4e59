// Two-factor FFT passes, one mesh, FP64.
#define P3M_FFT_TWO_SINGLE
#include "fft_two_launch.hpp"

namespace p3m {
namespace fft {
P3M_INST(double)
}  // namespace fft
}  // namespace p3m
