// fft_line_f64.hip -- FP64 instances of the register-resident FFT passes.
#include <type_traits>

#include "fft_line.hpp"

namespace cunfft {

template void launch_fft_line<double>(const FftPass<double> &, int64_t, size_t, hipStream_t);
template void launch_fft_line_batch<double>(const FftPass<double> *, const BlockMap *, uint32_t, bool, int, size_t,
                                          hipStream_t);

}  // namespace cunfft
