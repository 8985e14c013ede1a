// FP32 instantiations of the FFT passes (fft.hpp).
#include "fft.hpp"

namespace nfft_hip {

template void launch_fft_pass<float>(cplx<float> *, const cplx<float> *, cplx<float> *,
                                     const FftPass<float> &, int, hipStream_t, int, cplx<float> *);

}  // namespace nfft_hip
