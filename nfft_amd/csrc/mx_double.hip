// Matrix-core B / B^T kernels instantiated for double (kernel templates in mx.hpp).
#include "mx.hpp"

namespace nfft_hip {
template void launch_mx_interp<double>(const cplx<double> *, cplx<double> *, const Engine<double> &, hipStream_t, int,
                                   const BinGeom *);
template void launch_mx_spread<double>(const cplx<double> *, const Engine<double> &, hipStream_t, int, const BinGeom *,
                                   cplx<double> *);
template void launch_mx_gather<double>(const Engine<double> &, cplx<double> *, hipStream_t, int, const BinGeom *,
                                   cplx<double> *);
}  // namespace nfft_hip
