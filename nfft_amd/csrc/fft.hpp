// F: the d-dimensional unnormalised DFT of the oversampled grid (the role
// FFTW plays for the reference: kernel/nfft/nfft.c:6030-6031 plans,
// FFTW_FORWARD = sign -1 for trafo, FFTW_BACKWARD = sign +1 for adjoint),
// done as one pass per dimension with D and D^T fused into the passes at the
// ends and the zero band of the padded grid pruned:
//
//   trafo   passes t = d-1 .. 0.  The first reads f_hat, applies the
//           deconvolution factors and places the values in the band
//           (k - N_t/2) mod n_t of each line (D, reference
//           kernel/nfft/nfft.c:2786-2831); every pass handles only lines whose
//           not-yet-transformed coordinates lie in their band, and reads only
//           the band along its own axis (the rest is known to be zero).
//   adjoint passes t = 0 .. d-1.  Each keeps only the band of its axis (all
//           D^T reads, nfft.c:2874-2903) and handles only lines whose already
//           transformed coordinates lie in the band; the last writes f_hat
//           with the deconvolution factors applied (D^T).
//
// Each workgroup transforms `lines_per_block` whole lines by a self-sorting
// Stockham schedule.  Stage with radix R after sub-transforms of size Ns:
//   v_r = X[j + r n/R] * w^(r (j mod Ns))  with w = exp(sign 2 pi i / (Ns R))
//   v   = DFT_R(v)
//   Y[(j div Ns) Ns R + (j mod Ns) + r Ns] = v_r
// The first stage takes its butterflies straight from memory and the last one
// writes them straight back (its outputs are j + r n/R, whole runs along the
// line), so a line of two stages crosses LDS once and one of three twice; the
// radices go up to 16 to keep it at that (256 = 16 x 16, 150 = 15 x 10).
// Stages between run in place: every butterfly is read into registers, then
// all are written.  Twiddles come from a table exp(-2 pi i k / n) built in
// FP64 on the host.
//
// Bound: the latency of one load - LDS - store chain per workgroup, four
// workgroups deep (grids up to 128 MB stay in the last-level cache), and the
// strided axes' short segments.  Per pass before (every stage in place in LDS,
// run-time divisions by each length, lines staged in and out) and now:
//   256^3 FP32, trafo passes        52 + 59 + 108 us -> 20 + 25 + 44
//   256^3 FP64, adjoint passes      162 + 74 + 54 us -> 101 + 48 + 30
//   180 x 150 x 120 FP32, trafo     70 + 80 + 105 us -> 11 + 14 + 23
//   1024^2 FP32, adjoint            27 us -> 13
//   2^22 FP32 (2048 x 2048 halves)  118 us -> 26 each; its halves move 16
//     bytes per cache line with two lines per workgroup, 64 with eight
#pragma once

#include "engine.hpp"

namespace nfft_hip {

// elements per thread of a pass, and of one workgroup's lines
constexpr int kFftPer = 16;
template <typename R> constexpr int fft_cap() { return sizeof(R) == 4 ? 4096 : 2048; }

template <typename R>
__device__ __forceinline__ cplx<R> cmul(cplx<R> a, cplx<R> b) {
  return cplx<R>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename R>
__device__ __forceinline__ cplx<R> cadd(cplx<R> a, cplx<R> b) {
  return cplx<R>{a.x + b.x, a.y + b.y};
}
template <typename R>
__device__ __forceinline__ cplx<R> csub(cplx<R> a, cplx<R> b) {
  return cplx<R>{a.x - b.x, a.y - b.y};
}
// multiply by sign * i
template <typename R, int SIGN>
__device__ __forceinline__ cplx<R> mul_si(cplx<R> a) {
  return SIGN > 0 ? cplx<R>{-a.y, a.x} : cplx<R>{a.y, -a.x};
}

template <typename R, int SIGN>
__device__ __forceinline__ void dft2(cplx<R> *v) {
  cplx<R> a = v[0], b = v[1];
  v[0] = cadd<R>(a, b);
  v[1] = csub<R>(a, b);
}

template <typename R, int SIGN>
__device__ __forceinline__ void dft4(cplx<R> &v0, cplx<R> &v1, cplx<R> &v2, cplx<R> &v3) {
  cplx<R> s02 = cadd<R>(v0, v2), d02 = csub<R>(v0, v2);
  cplx<R> s13 = cadd<R>(v1, v3), d13 = mul_si<R, SIGN>(csub<R>(v1, v3));
  v0 = cadd<R>(s02, s13);
  v2 = csub<R>(s02, s13);
  v1 = cadd<R>(d02, d13);
  v3 = csub<R>(d02, d13);
}

template <typename R, int SIGN>
__device__ __forceinline__ void dft8(cplx<R> *v) {
  // even / odd radix-4 halves, then combine with w8^k, w8 = exp(sign 2 pi i/8)
  cplx<R> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  cplx<R> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<R, SIGN>(e0, e1, e2, e3);
  dft4<R, SIGN>(o0, o1, o2, o3);
  const R h = R(0.70710678118654752440084436210484903928);
  // o1 *= (1 + sign i)/sqrt2 ; o2 *= sign i ; o3 *= (-1 + sign i)/sqrt2
  cplx<R> t1 = cadd<R>(o1, mul_si<R, SIGN>(o1));
  t1 = cplx<R>{t1.x * h, t1.y * h};
  cplx<R> t2 = mul_si<R, SIGN>(o2);
  cplx<R> t3 = csub<R>(mul_si<R, SIGN>(o3), o3);
  t3 = cplx<R>{t3.x * h, t3.y * h};
  v[0] = cadd<R>(e0, o0);
  v[4] = csub<R>(e0, o0);
  v[1] = cadd<R>(e1, t1);
  v[5] = csub<R>(e1, t1);
  v[2] = cadd<R>(e2, t2);
  v[6] = csub<R>(e2, t2);
  v[3] = cadd<R>(e3, t3);
  v[7] = csub<R>(e3, t3);
}

// exp(2 pi i k / N), k < N, evaluated by the compiler: series of sin and cos
// on the first octant
template <int N> struct Roots {
  double c[N] = {}, s[N] = {};
  constexpr Roots() {
    for (int k = 0; k < N; k++) {
      // 8 k = o N + f: octant o, angle (pi / 4) (f / N) into it
      const int o = 8 * k / N, f = 8 * k - o * N;
      const double x = 0.78539816339744830961566084581987572 * ((o & 1) ? N - f : f) / N;
      double sn = 0, cs = 0, t = 1;
      for (int i = 0; i < 24; i++) {
        (i & 1 ? sn : cs) += (i & 2) ? -t : t;
        t *= x / (i + 1);
      }
      const bool sw = (o + 1) & 2;  // octants 1, 2, 5, 6: sine and cosine change places
      const double a = sw ? sn : cs, b = sw ? cs : sn;
      c[k] = o >= 2 && o < 6 ? -a : a;
      s[k] = o >= 4 ? -b : b;
    }
  }
};

// odd prime: outputs k and RAD - k share the sums over the pairs r, RAD - r
template <typename R, int RAD, int SIGN>
__device__ __forceinline__ void dft_odd(cplx<R> *v) {
  constexpr Roots<RAD> w;
  constexpr int H = RAD / 2;
  cplx<R> t[H], u[H];
#pragma unroll
  for (int r = 1; r <= H; r++) {
    t[r - 1] = cadd<R>(v[r], v[RAD - r]);
    u[r - 1] = csub<R>(v[r], v[RAD - r]);
  }
  cplx<R> s = v[0];
#pragma unroll
  for (int r = 0; r < H; r++) s = cadd<R>(s, t[r]);
#pragma unroll
  for (int k = 1; k <= H; k++) {
    cplx<R> a = v[0], b = cplx<R>{0, 0};
#pragma unroll
    for (int r = 1; r <= H; r++) {
      const R c = R(w.c[(r * k) % RAD]), sn = R(SIGN * w.s[(r * k) % RAD]);
      a = cplx<R>{fma(c, t[r - 1].x, a.x), fma(c, t[r - 1].y, a.y)};
      b = cplx<R>{fma(sn, u[r - 1].x, b.x), fma(sn, u[r - 1].y, b.y)};
    }
    v[k] = cplx<R>{a.x - b.y, a.y + b.x};
    v[RAD - k] = cplx<R>{a.x + b.y, a.y - b.x};
  }
  v[0] = s;
}

template <typename R, int RAD, int SIGN>
__device__ __forceinline__ void dft(cplx<R> *v);

// RAD = N1 N2: N2 transforms of length N1, roots of unity, N1 of length N2
template <typename R, int N1, int N2, int SIGN>
__device__ __forceinline__ void dft_split(cplx<R> *v) {
  constexpr int N = N1 * N2;
  constexpr Roots<N> w;
  cplx<R> y[N1][N2];
#pragma unroll
  for (int b = 0; b < N2; b++) {
    cplx<R> x[N1];
#pragma unroll
    for (int a = 0; a < N1; a++) x[a] = v[N2 * a + b];
    dft<R, N1, SIGN>(x);
#pragma unroll
    for (int a = 0; a < N1; a++) {
      const int e = a * b;
      if (e == 0) y[a][b] = x[a];
      else if (4 * e == N) y[a][b] = mul_si<R, SIGN>(x[a]);
      else if (8 * e == N || 8 * e == 3 * N) {
        // (+-1 +- i) / sqrt 2
        const R h = R(0.70710678118654752440084436210484903928);
        const cplx<R> i = mul_si<R, SIGN>(x[a]);
        const cplx<R> u = 8 * e == N ? cadd<R>(i, x[a]) : csub<R>(i, x[a]);
        y[a][b] = cplx<R>{u.x * h, u.y * h};
      }
      else y[a][b] = cmul<R>(x[a], cplx<R>{R(w.c[e % N]), R(SIGN * w.s[e % N])});
    }
  }
#pragma unroll
  for (int a = 0; a < N1; a++) {
    dft<R, N2, SIGN>(y[a]);
#pragma unroll
    for (int b = 0; b < N2; b++) v[a + N1 * b] = y[a][b];
  }
}

template <typename R, int RAD, int SIGN>
__device__ __forceinline__ void dft(cplx<R> *v) {
  if constexpr (RAD == 1) return;
  else if constexpr (RAD == 2) dft2<R, SIGN>(v);
  else if constexpr (RAD == 4) dft4<R, SIGN>(v[0], v[1], v[2], v[3]);
  else if constexpr (RAD == 8) dft8<R, SIGN>(v);
  else if constexpr (RAD == 6) dft_split<R, 3, 2, SIGN>(v);
  else if constexpr (RAD == 9) dft_split<R, 3, 3, SIGN>(v);
  else if constexpr (RAD == 10) dft_split<R, 5, 2, SIGN>(v);
  else if constexpr (RAD == 12) dft_split<R, 3, 4, SIGN>(v);
  else if constexpr (RAD == 15) dft_split<R, 5, 3, SIGN>(v);
  else if constexpr (RAD == 16) dft_split<R, 4, 4, SIGN>(v);
  else dft_odd<R, RAD, SIGN>(v);
}

// a div d and a mod d for 0 <= a < 2^14: the rounded quotient of a + 1/2 stays
// on the right side of the integers, 1 / (2 d) away, by a factor of 50
struct DivMod {
  float inv;
  int d;
  __device__ explicit DivMod(int d_) : inv(1.0f / (float)d_), d(d_) {}
  __device__ __forceinline__ void operator()(int a, int &q, int &r) const {
    q = (int)(((float)a + 0.5f) * inv);
    r = a - q * d;
  }
};

// LDS layout of the staged lines: element k of line ll sits at
// ll * ls + k + (k >> 4) with an odd line stride ls = n + n/16 + 1, so that
// neither the strided accesses of the first Stockham stages (stride RAD
// within a line) nor the staging of adjacent lines (one element per line)
// fall into the same LDS bank.
__device__ __forceinline__ int lds_idx(int ll, int k, int ls) { return ll * ls + k + (k >> 4); }

// multiplies the inputs of a butterfly by w^(r step), r = 1 .. RAD - 1
template <typename R, int RAD, int SIGN>
__device__ __forceinline__ void stage_twiddle(cplx<R> *v, const cplx<R> *tw, int step) {
#pragma unroll
  for (int r = 1; r < RAD; r++) {
    cplx<R> w = tw[r * step];
    if (SIGN > 0) w.y = -w.y;
    v[r] = cmul<R>(v[r], w);
  }
}

// First stage (Ns = 1) over nlines lines of length n: butterflies from
// load(line, j, v) into LDS.  Threads run along the line or, ACROSS, over the
// lines first.
template <typename R, int RAD, int SIGN, typename Load>
__device__ __forceinline__ void stage_first(cplx<R> *__restrict__ buf, int n, int ls, int nlines,
                                            bool across, Load load) {
  const int q = n / RAD;
  const DivMod dm(across ? nlines : q);
#pragma unroll 1
  for (int b = threadIdx.x; b < nlines * q; b += blockDim.x) {
    int ll, j;
    dm(b, across ? j : ll, across ? ll : j);
    cplx<R> v[RAD];
    load(ll, j, q, v);
    __builtin_amdgcn_sched_barrier(0);
    dft<R, RAD, SIGN>(v);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < RAD; r++) buf[lds_idx(ll, j * RAD + r, ls)] = v[r];
  }
  __syncthreads();
}

// Last stage (Ns = n / RAD): butterflies from LDS to store(line, j, q, v).
template <typename R, int RAD, int SIGN, typename Store>
__device__ __forceinline__ void stage_last(const cplx<R> *__restrict__ buf, int n, int ls,
                                           int nlines, bool across, const cplx<R> *tw,
                                           Store store) {
  const int q = n / RAD;
  const DivMod dm(across ? nlines : q);
#pragma unroll 1
  for (int b = threadIdx.x; b < nlines * q; b += blockDim.x) {
    int ll, j;
    dm(b, across ? j : ll, across ? ll : j);
    cplx<R> v[RAD];
#pragma unroll
    for (int r = 0; r < RAD; r++) v[r] = buf[lds_idx(ll, j + r * q, ls)];
    stage_twiddle<R, RAD, SIGN>(v, tw, j);
    __builtin_amdgcn_sched_barrier(0);
    dft<R, RAD, SIGN>(v);
    __builtin_amdgcn_sched_barrier(0);
    store(ll, j, q, v);
  }
}

// A stage between, in place in LDS.  A thread holds at most
// ceil(kFftPer / RAD) butterflies.
template <typename R, int RAD, int SIGN>
__device__ __forceinline__ void stage_inplace(cplx<R> *__restrict__ buf, int n, int ls, int nlines,
                                              int Ns, const cplx<R> *tw) {
  constexpr int SL = (kFftPer + RAD - 1) / RAD;
  const int q = n / RAD;
  const int nbf = nlines * q;
  const int span = Ns * RAD;
  const int twstep = n / span;
  const DivMod dq(q), dns(Ns);
  cplx<R> v[SL][RAD];
  int at[SL];
#pragma unroll
  for (int i = 0; i < SL; i++) {
    const int b = threadIdx.x + i * blockDim.x;
    at[i] = -1;
    if (b < nbf) {
      int ll, j, jd, jm;
      dq(b, ll, j);
      dns(j, jd, jm);
#pragma unroll
      for (int r = 0; r < RAD; r++) v[i][r] = buf[lds_idx(ll, j + r * q, ls)];
      stage_twiddle<R, RAD, SIGN>(v[i], tw, jm * twstep);
      __builtin_amdgcn_sched_barrier(0);
      dft<R, RAD, SIGN>(v[i]);
      at[i] = (ll << 16) + jd * span + jm;
    }
    // one butterfly's twiddles at a time
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SL; i++) {
    if (at[i] >= 0) {
#pragma unroll
      for (int r = 0; r < RAD; r++)
        buf[lds_idx(at[i] >> 16, (at[i] & 0xffff) + r * Ns, ls)] = v[i][r];
    }
  }
  __syncthreads();
}

// A Stockham stage of any radix (a prime factor above 13, known only at run
// time), same math as stage_inplace: each output of a butterfly is its own
// sum over the RAD inputs, read from LDS, with the radix-RAD DFT factor
// exp(sign 2 pi i r k / RAD) taken from the line's twiddle table at
// (r k mod RAD) n / RAD.  All outputs are held in registers until every
// thread has read its inputs, then written.  O(n RAD) work per line.
template <typename R, int SIGN>
__device__ __forceinline__ void stage_generic(cplx<R> *__restrict__ buf, int n, int ls, int nlines,
                                              int Ns, int RAD, const cplx<R> *tw) {
  constexpr int PER = kFftPer;
  const int q = n / RAD;
  const int span = Ns * RAD;
  const int twstep = n / span;
  const int tot = nlines * n;
  cplx<R> out[PER];
  int dll[PER], dpos[PER];
#pragma unroll
  for (int u = 0; u < PER; u++) {
    __builtin_amdgcn_sched_barrier(0);
    const int o = threadIdx.x + u * blockDim.x;
    dll[u] = -1;
    if (o < tot) {
      const int ll = o / n;
      const int pos = o - ll * n;
      // output pos = jd span + jm + k Ns of butterfly j = jd Ns + jm
      const int jd = pos / span;
      const int rr = pos - jd * span;
      const int k = rr / Ns;
      const int jm = rr - k * Ns;
      const int j = jd * Ns + jm;
      R sr = 0, si = 0;
      for (int r = 0; r < RAD; r++) {
        cplx<R> x = buf[lds_idx(ll, j + r * q, ls)];
        // stage twiddle w^(r jm) and the DFT factor, one table entry each
        cplx<R> w = tw[jm * r * twstep];
        cplx<R> f = tw[((r * k) % RAD) * q];
        if (SIGN > 0) {
          w.y = -w.y;
          f.y = -f.y;
        }
        x = cmul<R>(cmul<R>(x, w), f);
        sr += x.x;
        si += x.y;
      }
      out[u] = cplx<R>{sr, si};
      dll[u] = ll;
      dpos[u] = pos;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; u++)
    if (dll[u] >= 0) buf[lds_idx(dll[u], dpos[u], ls)] = out[u];
  __syncthreads();
}

// Band position of grid index k along a dimension (n, N): the f_hat
// coordinate ks in [0, N) with k = (ks - N/2) mod n, or -1 outside the band.
__device__ __forceinline__ int band_coord(int k, int n, int N) {
  const int h = N / 2;
  if (k < N - h) return k + h;
  if (k >= n - h) return k - (n - h);
  return -1;
}

// coordinates of line L0 + ll, the last one fastest: its offsets in the grid
// and in f_hat and the deconvolution factor of the other dimensions
// (the factors are FP64 in both families, a value is multiplied by their
// rounded product: as FP32 factors, rounded one by one, they made a sixth of
// the squared error of a 3-D FP32 transform)
struct LineInfo {
  long in, out;  // offsets in the pass's input and output
  double fac;
  int sub;
};

template <typename R, typename I>
__device__ __forceinline__ LineInfo line_info(const FftPass<R> &P, I L) {
  LineInfo li;
  li.sub = 0;
  if (P.four) {  // four-step halves: the sub-line index (j1 or k2) runs fastest
    li.sub = (int)(L % (I)P.nsub);
    L /= (I)P.nsub;
  }
  long go = 0, fo = 0;
  double fac = 1.0;
  for (int s = P.nod - 1; s >= 0; s--) {
    const int c = s > 0 ? (int)(L % (I)P.cnt[s]) : (int)L;
    if (s > 0) L /= (I)P.cnt[s];
    int k = c;
    if (P.band[s]) {
      k = c - P.N_od[s] / 2;
      k += k < 0 ? P.n_od[s] : 0;
    }
    go += (long)k * P.gstr[s];
    if (P.in_mode == kFromCoeffs || P.out_mode == kToCoeffs) {
      fo += (long)c * P.fstr[s];
      fac *= P.phi_od[s][c];
    }
  }
  li.in = P.in_mode == kFromCoeffs ? fo : go;
  li.out = P.out_mode == kToCoeffs ? fo : go;
  li.fac = fac;
  return li;
}

#define NFFT_FFT_RADIX(RAD_, CALL)  \
  switch (RAD_) {                   \
    case 1: { constexpr int RAD = 1; CALL; break; }    \
    case 2: { constexpr int RAD = 2; CALL; break; }    \
    case 4: { constexpr int RAD = 4; CALL; break; }    \
    case 8: { constexpr int RAD = 8; CALL; break; }    \
    case 16: { constexpr int RAD = 16; CALL; break; }  \
    default:                                           \
      if constexpr (KIND != kPow2) {                   \
        switch (RAD_) {                                \
          case 3: { constexpr int RAD = 3; CALL; break; }    \
          case 5: { constexpr int RAD = 5; CALL; break; }    \
          case 6: { constexpr int RAD = 6; CALL; break; }    \
          case 7: { constexpr int RAD = 7; CALL; break; }    \
          case 9: { constexpr int RAD = 9; CALL; break; }    \
          case 10: { constexpr int RAD = 10; CALL; break; }  \
          case 11: { constexpr int RAD = 11; CALL; break; }  \
          case 12: { constexpr int RAD = 12; CALL; break; }  \
          case 13: { constexpr int RAD = 13; CALL; break; }  \
          case 15: { constexpr int RAD = 15; CALL; break; }  \
          default: break;                              \
        }                                              \
      }                                                \
  }

// radices of a kernel: powers of two; all up to 16; those and generic stages
enum FftKind { kPow2, kSmooth, kGeneric };

// gsrc / gdst: the grid buffer the pass reads and the one it writes (the
// same buffer except in the second half of a four-step axis).  NT: the
// largest workgroup, which handles up to kFftPer NT elements.
template <typename R, int SIGN, int NT, FftKind KIND>
__global__ __launch_bounds__(NT, NT > 512 ? 4 : (sizeof(R) == 4 ? 4 : 2)) void k_fft_pass(
    const cplx<R> *gsrc, cplx<R> *gdst, const cplx<R> *__restrict__ fin, cplx<R> *__restrict__ fout,
    FftPass<R> P) {
  // right-hand side blockIdx.y of a batched launch
  gsrc += (long)blockIdx.y * P.bs_g;
  gdst += (long)blockIdx.y * P.bs_g;
  if (fin) fin += (long)blockIdx.y * P.bs_c;
  if (fout) fout += (long)blockIdx.y * P.bs_c;
  // consecutive groups of lines run on one XCD: where a group's accesses are
  // shorter than a cache line, its neighbours' meet them in that L2
  const unsigned per = (gridDim.x + 7) / 8, rem = gridDim.x - 8 * (per - 1);
  const unsigned xcd = blockIdx.x & 7, ix = blockIdx.x >> 3;
  const unsigned blk = ix + (xcd < rem ? xcd * per : rem * per + (xcd - rem) * (per - 1));
  const int ls = lds_line_stride(P.len);
  const int n = P.len;
  const long L0 = (long)blk * P.lines_per_block;
  const int TL = (int)min((long)P.lines_per_block, P.nlines - L0);
  // LDS: lines, their offsets, the line length's twiddle table where it fits
  extern __shared__ __align__(16) unsigned char fft_smem[];
  cplx<R> *buf = reinterpret_cast<cplx<R> *>(fft_smem);
  cplx<R> *twl = buf + (long)P.lines_per_block * ls;
  LineInfo *info = reinterpret_cast<LineInfo *>(twl + (P.twiddle_in_lds ? n : 0));
  const cplx<R> *tw = P.twiddle;
  if (P.twiddle_in_lds) {
    for (int k = threadIdx.x; k < n; k += blockDim.x) twl[k] = P.twiddle[k];
    tw = twl;
  }
  for (int ll = threadIdx.x; ll < TL; ll += blockDim.x)
    info[ll] = P.nlines < (1l << 31) ? line_info<R, unsigned>(P, (unsigned)(L0 + ll))
                                     : line_info<R, unsigned long>(P, (unsigned long)(L0 + ll));
  __syncthreads();

  // element k of a line: its position along the axis is ia k + ib sub at the
  // input and oa k + ob sub at the output (the two differ from k only in
  // four-step halves).  A wave walks along a line where its elements are
  // adjacent in memory, across lines otherwise.
  const int ia = P.four == 1 ? P.fn1 : 1, ib = P.four == 1 ? 1 : (P.four == 2 ? P.fn1 : 0);
  const int oa = P.four == 1 ? P.fn1 : (P.four == 2 ? P.fn2 : 1), ob = P.four ? 1 : 0;
  const int nax = P.four ? P.nfull : n;
  const bool across = !(P.stride == 1 && P.four != 1);
  const bool across_out = !(P.stride == 1 && P.four == 0);

  auto load = [&](int ll, int j, int q, auto &v) {
    constexpr int RAD = sizeof(v) / sizeof(v[0]);
    const LineInfo &li = info[ll];
    const int k0 = ia * j + ib * li.sub;
    if (P.in_mode == kFromCoeffs) {
      double ph[RAD];
#pragma unroll
      for (int r = 0; r < RAD; r++) {
        const int ks = band_coord(k0 + ia * r * q, nax, P.Nband);
        v[r] = cplx<R>{R(0), R(0)};
        ph[r] = 0.0;
        if (ks >= 0) {
          v[r] = fin[li.in + (long)ks * P.fstr_ax];
          ph[r] = P.phi_ax[ks];
        }
      }
#pragma unroll
      for (int r = 0; r < RAD; r++) {
        const R f = (R)(li.fac * ph[r]);
        v[r] = cplx<R>{v[r].x * f, v[r].y * f};
      }
    } else {
      const cplx<R> *src = gsrc + li.in + (long)k0 * P.stride;
      const long step = (long)(ia * q) * P.stride;
#pragma unroll
      for (int r = 0; r < RAD; r++) {
        v[r] = cplx<R>{R(0), R(0)};
        if (P.in_mode == kFromGrid || band_coord(k0 + ia * r * q, nax, P.Nband) >= 0)
          v[r] = src[r * step];
      }
    }
  };
  auto store = [&](int ll, int j, int q, auto &v) {
    constexpr int RAD = sizeof(v) / sizeof(v[0]);
    const LineInfo &li = info[ll];
    const int k0 = oa * j + ob * li.sub;
    if (P.four == 1) {
      // w_n^(j1 k2), stored where its product goes
#pragma unroll
      for (int r0 = 0; r0 < RAD; r0 += 4) {
        cplx<R> w[4];
#pragma unroll
        for (int r = 0; r < 4 && r0 + r < RAD; r++) w[r] = P.twiddle_full[k0 + oa * (r0 + r) * q];
#pragma unroll
        for (int r = 0; r < 4 && r0 + r < RAD; r++) {
          if (SIGN > 0) w[r].y = -w[r].y;
          v[r0 + r] = cmul<R>(v[r0 + r], w[r]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (P.out_mode == kToCoeffs) {
#pragma unroll
      for (int r = 0; r < RAD; r++) {
        const int ks = band_coord(k0 + oa * r * q, nax, P.Nband);
        if (ks >= 0) {
          const R f = (R)(li.fac * P.phi_ax[ks]);
          fout[li.out + (long)ks * P.fstr_ax] = cplx<R>{v[r].x * f, v[r].y * f};
        }
      }
    } else {
      cplx<R> *dst = gdst + li.out + (long)k0 * P.stride;
      const long step = (long)(oa * q) * P.stride;
#pragma unroll
      for (int r = 0; r < RAD; r++)
        if (P.out_mode == kToGrid || band_coord(k0 + oa * r * q, nax, P.Nband) >= 0)
          dst[r * step] = v[r];
    }
  };

  NFFT_FFT_RADIX(P.radix[0], (stage_first<R, RAD, SIGN>(buf, n, ls, TL, across, load)))
  int Ns = P.radix[0];
  for (int st = 1; st + 1 < P.nstages; st++) {
    const int rad = P.radix[st];
    // (opaque: the quotients by every radix would otherwise be computed ahead
    // of the loop and kept in registers)
    int n = P.len;
    asm volatile("" : "+s"(n));
    if (KIND == kGeneric && rad > 16) {
      if constexpr (KIND == kGeneric) stage_generic<R, SIGN>(buf, n, ls, TL, Ns, rad, tw);
    } else {
      NFFT_FFT_RADIX(rad, if constexpr (RAD > 1) (stage_inplace<R, RAD, SIGN>(buf, n, ls, TL, Ns, tw)))
    }
    Ns *= rad;
  }
  NFFT_FFT_RADIX(P.radix[P.nstages - 1],
                 (stage_last<R, RAD, SIGN>(buf, n, ls, TL, across_out, tw, store)))
}
#undef NFFT_FFT_RADIX

// Lines per workgroup: as many as its kFftPer elements per thread allow, but
// fewer when the launch would leave the GPU short of workgroups (small grids:
// aim for 1024 of them over all right-hand sides), keeping at least 2 lines (4
// along a strided axis, so that each load covers 32 contiguous bytes or more).
template <typename R>
void launch_fft_pass(cplx<R> *g, const cplx<R> *fhat_in, cplx<R> *fhat_out, const FftPass<R> &p0,
                     int sign, hipStream_t s, int nb, cplx<R> *g2) {
  if (p0.nlines <= 0) return;
  FftPass<R> p = p0;
  const bool strided = p.stride != 1 || p.four;
  bool pow2 = true, generic = false;
  for (int i = 0; i < p.nstages; i++) {
    const int r = p.radix[i];
    pow2 = pow2 && (r & (r - 1)) == 0;
    generic = generic || r > 16;
  }
  // A strided axis whose lines are so long that fewer than 64 bytes of
  // adjacent ones fit: a workgroup four times the size, if that many still
  // fill the CUs (a 2^22-point half: 118 us before, 36 with workgroups twice the
  // size and two per CU, 26 with four times).
  const long seg = 64 / (long)sizeof(cplx<R>);
  const long fit_big = std::min<long>(256, 4 * fft_cap<R>() / p.len);
  const bool big = strided && !generic && fft_cap<R>() / p.len < seg && p.nlines * (long)nb / fit_big >= 256;
  if (big) {
    p.lines_per_block = (int)std::max(std::min(4L, fit_big), fit_big >> std::max(0, -p0.lpb_shift));
  } else {
    const long fit = std::max<long>(1, std::min<long>(256, fft_cap<R>() / p.len));
    long want = std::max<long>(1, p0.nlines * (long)nb / 1024);
    want = p0.lpb_shift >= 0 ? want << p0.lpb_shift : std::max<long>(1, want >> -p0.lpb_shift);
    const long floor_lines = std::min<long>(fit, strided ? 4 : 2);
    p.lines_per_block = (int)std::max(floor_lines, std::min(fit, want));
  }
  const size_t lines = sizeof(cplx<R>) * (size_t)p.lines_per_block * lds_line_stride(p.len);
  const size_t table = sizeof(cplx<R>) * (size_t)p.len;
  const size_t info = sizeof(LineInfo) * (size_t)p.lines_per_block;
  p.twiddle_in_lds = lines + table + info <= (size_t)(big ? 160 : 64) * 1024 ? 1 : 0;
  const size_t lds = lines + info + (p.twiddle_in_lds ? table : 0);
  const long blocks = ceil_div(p.nlines, p.lines_per_block);
  // threads: the butterflies of the stage that has most
  int most = 1;
  const int tile = p.lines_per_block * p.len;
  for (int i = 0; i < p.nstages; i++)
    most = std::max(most, p.radix[i] > 16 ? tile : tile / p.radix[i]);
  constexpr int NT = fft_cap<R>() / kFftPer;
  const int nt = std::min((big ? 4 : 1) * NT, (most + 63) / 64 * 64);
  auto pick = [&](auto sg, auto nt_c) {
    constexpr int S = decltype(sg)::value, T = decltype(nt_c)::value;
    if constexpr (T == NT)
      if (generic) return k_fft_pass<R, S, T, kGeneric>;
    return pow2 ? k_fft_pass<R, S, T, kPow2> : k_fft_pass<R, S, T, kSmooth>;
  };
  using neg = std::integral_constant<int, -1>;
  using pos = std::integral_constant<int, 1>;
  using small_t = std::integral_constant<int, NT>;
  using big_t = std::integral_constant<int, 4 * NT>;
  auto fn = sign < 0 ? (big ? pick(neg{}, big_t{}) : pick(neg{}, small_t{}))
                     : (big ? pick(pos{}, big_t{}) : pick(pos{}, small_t{}));
  cplx<R> *src = p.src ? g2 : g;
  cplx<R> *dst = p.dst ? g2 : g;
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks, (unsigned)nb), dim3((unsigned)nt), lds, s,
                     (const cplx<R> *)src, dst, fhat_in, fhat_out, p);
}

}  // namespace nfft_hip
