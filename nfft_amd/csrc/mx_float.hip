// Matrix-core B / B^T kernels instantiated for float (kernel templates in mx.hpp).
#include "mx.hpp"

namespace nfft_hip {
template void launch_mx_interp<float>(const cplx<float> *, cplx<float> *, const Engine<float> &, hipStream_t, int,
                                   const BinGeom *);
template void launch_mx_spread<float>(const cplx<float> *, const Engine<float> &, hipStream_t, int, const BinGeom *,
                                   cplx<float> *);
template void launch_mx_gather<float>(const Engine<float> &, cplx<float> *, hipStream_t, int, const BinGeom *,
                                   cplx<float> *);
}  // namespace nfft_hip
