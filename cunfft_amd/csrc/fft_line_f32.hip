// fft_line_f32.hip -- FP32 instances of the register-resident FFT passes.
#include <type_traits>

#include "fft_line.hpp"

namespace cunfft {

template void launch_fft_line<float>(const FftPass<float> &, int64_t, size_t, hipStream_t);
template void launch_fft_line_batch<float>(const FftPass<float> *, const BlockMap *, uint32_t, bool, int, size_t,
                                          hipStream_t);

}  // namespace cunfft
