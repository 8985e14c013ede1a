// Index arithmetic of the matrix-core kernels' bins and planes, without HIP
// headers, so that a host compiler takes it too.
#pragma once

#if defined(__HIPCC__)
#define NFFT_HD __host__ __device__
#else
#define NFFT_HD
#endif

namespace nfft_hip {

// Ragged bins: first cell of bin b of nb over n cells, and the bin of cell c
// (n <= kMxMaxN, so that the products fit an int)
constexpr int kMxMaxN = 32767;
NFFT_HD inline int mx_lo(int b, int n, int nb) { return b * n / nb; }
NFFT_HD inline int mx_bin(int c, int n, int nb) { return ((c + 1) * nb - 1) / n; }
// widest window of the 3-D matrix-core kernels: m = kMxMaxM
constexpr int kMxMaxM = 6;

// B walks down a column with planes ra .. ra + mx_ring(W) - 1 in registers
// (plane p: the grid's p - m) and the next one ahead of its use; its nodes lie
// in up to kMxSpan dimension-0 cells at a time.
constexpr int kMxSpan = 4;
NFFT_HD constexpr int mx_ring(int W) { return W + kMxSpan - 1; }

// Grid plane of plane p, 0 <= p <= n0 - 1 + mx_ring(2 m + 2): the plane ahead
// of the last cell's lies up to m + 4 cells past the axis, which is a whole
// period and more for the shortest axes (n0 = 2 m + 3 = 5)
NFFT_HD inline int mx_plane(int p, int m, int n0) {
  int c = p - m;
  c += c < 0 ? n0 : 0;
  c -= c >= n0 ? n0 : 0;
  c -= c >= n0 ? n0 : 0;
  return c;
}

}  // namespace nfft_hip
