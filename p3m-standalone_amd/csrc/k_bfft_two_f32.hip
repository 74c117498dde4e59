// Two-factor FFT passes, batches, FP32.
#define P3M_FFT_TWO_BATCH
#include "fft_two_launch.hpp"

namespace p3m {
namespace fft {
P3M_INST(float)
}  // namespace fft
}  // namespace p3m
