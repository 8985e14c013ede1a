// FP64 instantiations of the FFT passes (fft.hpp).
#include "fft.hpp"

namespace nfft_hip {

template void launch_fft_pass<double>(cplx<double> *, const cplx<double> *, cplx<double> *,
                                     const FftPass<double> &, int, hipStream_t, int, cplx<double> *);

}  // namespace nfft_hip
