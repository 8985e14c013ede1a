// B^T for d = 2 on the matrix cores.
//
// The taps of a bin's nodes fall on the E0 x E1 cells of its tile, at most
// 16 T along each dimension (T = 2, 3).  A node's window over those positions
// is its W values at its offset in the bin and zeros elsewhere, and
//
//   tile[e0][e1] += sum_k psi0_k[e0] (psi1_k[e1] f_k)
//
// is a product over the nodes k: four nodes per 16 x 16 x 4 product, T x T
// blocks of 16 x 16 cells for the real and the imaginary part, all of which a
// wavefront holds in registers.  Blocks that none of the four nodes reaches
// are skipped (nodes arrive sorted by cell, so the four are neighbours; about
// three of four blocks remain).  No LDS tile, no
// read-modify-write, no atomics: each wavefront of an item walks its share of
// the nodes, and the wavefronts' sums meet in LDS in a fixed order when the
// tile is written out.
//
// NR right-hand sides of a batch share the windows and the skip masks; per
// right-hand side the operations and their order are those of NR = 1, so the
// results are bit-identical.
//
// Bound: matrix cores and vector ALUs together, as in mx.hpp.
// Measured per launch, against the run-merging kernel (FP32) and LDS atomics
// (FP64): 2^20 clustered nodes on 1024^2, m = 4 FP32 138 -> 62 us, m = 6 FP64
// 577 -> 154; 128512 radial nodes on 512^2, m = 4 FP32 30 -> 14; 32 right-hand
// sides of 206336 such nodes 441 -> 306.
//
// FP32 errors against FP64, adjoint on 256^2 cells with 2^18 radial nodes (1e-7;
// kernels before / one sum over 64 nodes / two): m = 2 1.32 / 1.36 / 1.29, m = 3
// 1.38 / 1.41 / 1.34, m = 4 1.54 / 1.56, m = 5 1.94 / 1.83, m = 6 2.07 / 2.21 /
// 2.07.  Two sums cost single right-hand sides nothing and batches their second
// right-hand side per workgroup (registers): 32 of 206336 nodes, m = 3, 359 ->
// 429 us (467 with both).
#pragma once

#include "mx_util.hpp"

namespace nfft_hip {

template <typename R, int W, int T, int NR, bool SHARED, bool TWO>
__global__ __launch_bounds__(64 * kMx2dWaves<R>, sizeof(R) == 8 && T == 3 && !SHARED ? 1 : 2) void k_spread_mx2d(
    const cplx<R> *__restrict__ fin, cplx<R> *__restrict__ g, const int *__restrict__ perm,
    const int *__restrict__ cell, const R *__restrict__ frac, const int4 *__restrict__ subs,
    BinGeom gg, WinParams<R> wp, cplx<R> *__restrict__ tiles) {
  using C = cplx<R>;
  constexpr int NC = 32, NWV = kMx2dWaves<R>, P = 16 * T + 4;
  constexpr int kWin = 2 * NC * P;  // window rows of a wavefront's chunk: (dimension, node)
  constexpr size_t kWinBytes = sizeof(R) * NWV * kWin, kTileBytes = sizeof(C) * 256 * T * T;
  // a tile per wavefront where they fit in place of the window rows, else one
  constexpr bool OWN = kTileBytes * NWV <= kWinBytes;
  static_assert(OWN || kTileBytes <= kWinBytes, "the tile takes the place of the window rows");
  __shared__ __align__(16) unsigned char smem[kWinBytes];
  __shared__ __align__(16) C sf[NWV][NR][NC];
  __shared__ __align__(16) R spoly[SHARED ? 1 : 2 * (W / 2) * kMxCoef<R>];
  // right-hand sides c0 .. c0 + nrhs - 1 of a batched launch
  const int c0 = blockIdx.y * NR;
  const int nrhs = NR == 1 ? 1 : min(NR, gg.nrhs - c0);
  fin += (long)c0 * gg.bs_f;
  g += (long)c0 * gg.bs_g;
  if (tiles) tiles += (long)c0 * gg.bs_t;
  const int4 sp = subs[blockIdx.x];
  int lo[2];
  bin_corner<2>(sp.x, gg, lo);
  const int E0 = gg.E[0], E1 = gg.E[1], tot = E0 * E1;
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  R *win = reinterpret_cast<R *>(smem) + wv * kWin;
  // this lane evaluates dimension t of the chunk's node me
  const int me = lane & (NC - 1), t = lane >> 5;
  if constexpr (!SHARED) {
    mx_load_poly<R, 2, W>(spoly, wp.poly, threadIdx.x, 64 * NWV);
    __syncthreads();
  }
  // the wavefront's share of the nodes, whole groups of four
  const int part = ((sp.z + NWV - 1) / NWV + 3) & ~3;
  const int first = min(sp.z, wv * part), cntw = min(sp.z, first + part) - first;
  // FP32 sums over at most kMx2dOneSum nodes (one sum over all nodes of a dense
  // cell would lose up to a bit).  TWO, long shares: the sums of these run over
  // the share.  Shares of up to twice as many: groups of four add to two sums
  // in turn, except where one is no further off than the kernels before (see
  // the head) or registers lack (three blocks).
  constexpr int H = sizeof(R) == 4 && !TWO && T == 2 && mx2d_two_sums(W / 2 - 1) ? 2 : 1;
  mx4<R> acc[H][NR][T][T][2], sum[TWO ? NR : 1][TWO ? T : 1][TWO ? T : 1][2];
#pragma unroll
  for (int c = 0; c < NR; c++)
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++)
#pragma unroll
        for (int x = 0; x < 2; x++) {
#pragma unroll
          for (int h = 0; h < H; h++) acc[h][c][a][b][x] = mx4<R>{0, 0, 0, 0};
          if constexpr (TWO) sum[c][a][b][x] = mx4<R>{0, 0, 0, 0};
        }
  auto fold = [&]() {
    if constexpr (TWO) {
#pragma unroll
      for (int c = 0; c < NR; c++)
#pragma unroll
        for (int a = 0; a < T; a++)
#pragma unroll
          for (int b = 0; b < T; b++)
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
              for (int i = 0; i < 4; i++) {
                sum[c][a][b][x][i] += acc[0][c][a][b][x][i];
                mx_clear(acc[0][c][a][b][x], i);
              }
    }
  };
  if (cntw > 0) {
    const int *cellp = cell + t * gg.M + sp.y + first;
    const R *fracp = frac + t * gg.M + sp.y + first;
    const int *permp = perm + sp.y + first;
    const int last = cntw - 1, lot = t == 0 ? lo[0] : lo[1];
    // node data one chunk ahead, node indices two (lanes of dimension 0)
    int c = cellp[min(me, last)];
    R fr = fracp[min(me, last)];
    C fv[NR];
    int pnext = 0;
    auto load_f = [&](int p) {
#pragma unroll
      for (int r = 0; r < NR; r++) fv[r] = r < nrhs ? fin[(long)r * gg.bs_f + p] : C{0, 0};
    };
    if (t == 0) {
      load_f(permp[min(me, last)]);
      pnext = permp[min(NC + me, last)];
    }
    for (int base = 0; base < cntw; base += NC) {
      const int shift = c - lot;
      {
        const R *poly = wp.poly;
        // (read again for every chunk: held over the loop the coefficients
        // would take all registers)
        asm volatile("" : "+s"(poly));
        mx_window_row<R, W, P>(win + lane * P, shift, fr - R(0.5), [&](int w) {
          if constexpr (SHARED) return poly + w * (poly_deg_v<R> + 1);
          else return spoly + (t * (W / 2) + w) * kMxCoef<R>;
        });
      }
      const int cnt = min(NC, cntw - base);
      if (t == 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) sf[wv][r][me] = me < cnt ? fv[r] : C{0, 0};
      }
      // nodes that reach block u of dimension 0 (low half) and 1 (high half)
      unsigned long long reach[T];
#pragma unroll
      for (int u = 0; u < T; u++) reach[u] = __ballot(shift < 16 * u + 16 && shift + W > 16 * u);
      const int nn = min(base + NC + me, last);
      c = cellp[nn];
      fr = fracp[nn];
      if (t == 0) {
        load_f(pnext);
        pnext = permp[min(base + 2 * NC + me, last)];
      }
      __builtin_amdgcn_wave_barrier();
      auto four = [&](int k, auto set) {
        constexpr int h = decltype(set)::value;
        const R *row = win + (k + q) * P + j;
        R p0[T], p1[T];
#pragma unroll
        for (int u = 0; u < T; u++) {
          p0[u] = row[16 * u];
          p1[u] = row[NC * P + 16 * u];
        }
        C v[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) v[r] = sf[wv][r][k + q];
#pragma unroll
        for (int b = 0; b < T; b++) {
          if (((reach[b] >> (32 + k)) & 15) == 0) continue;
          R br[NR], bi[NR];
#pragma unroll
          for (int r = 0; r < NR; r++) {
            br[r] = p1[b] * v[r].x;
            bi[r] = p1[b] * v[r].y;
          }
#pragma unroll
          for (int a = 0; a < T; a++) {
            if (((reach[a] >> k) & 15) == 0) continue;
#pragma unroll
            for (int r = 0; r < NR; r++) {
              acc[h][r][a][b][0] = mx_mul(p0[a], br[r], acc[h][r][a][b][0]);
              acc[h][r][a][b][1] = mx_mul(p0[a], bi[r], acc[h][r][a][b][1]);
            }
          }
        }
      };
      for (int k = 0; k < cnt; k += 4 * H) {
        four(k, std::integral_constant<int, 0>{});
        if constexpr (H == 2)
          if (k + 4 < cnt) four(k + 4, std::integral_constant<int, 1>{});
      }
      __builtin_amdgcn_wave_barrier();
      if ((base + NC) % kMx2dOneSum == 0 && base + NC < cntw) fold();
    }
  }
  // the wavefronts' sums, in their order
  C *tile0 = reinterpret_cast<C *>(smem);
#pragma unroll
  for (int r = 0; r < NR; r++) {
    for (int w = 0; w < (OWN ? 1 : NWV); w++) {
      __syncthreads();
      if (!OWN && w != wv) continue;
      C *tile = tile0 + (OWN ? wv * tot : 0);
#pragma unroll
      for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int e0 = 16 * a + mx_row<R>(q, i), e1 = 16 * b + j;
            if (e0 < E0 && e1 < E1) {
              C s = C{acc[0][r][a][b][0][i], acc[0][r][a][b][1][i]};
              if constexpr (H == 2) s = C{s.x + acc[1][r][a][b][0][i], s.y + acc[1][r][a][b][1][i]};
              if constexpr (TWO) s = C{s.x + sum[r][a][b][0][i], s.y + sum[r][a][b][1][i]};
              if (w > 0) {
                const C o = tile[e0 * E1 + e1];
                s = C{o.x + s.x, o.y + s.y};
              }
              tile[e0 * E1 + e1] = s;
            }
          }
    }
    __syncthreads();
    if (r < nrhs)
      flush_tile<R, 2>(
          [&](int x) {
            C v = tile0[x];
            if constexpr (OWN) {
#pragma unroll
              for (int w = 1; w < NWV; w++) {
                const C o = tile0[w * tot + x];
                v = C{v.x + o.x, v.y + o.y};
              }
            }
            return v;
          },
          tiles ? tiles + (long)r * gg.bs_t : tiles, g + (long)r * gg.bs_g, lo, gg, tot, sp.w,
          threadIdx.x, 64 * NWV);
  }
}

}  // namespace nfft_hip
