// B and B^T for d = 3 on the matrix cores.
//
// The bins are narrow enough that the taps of all their nodes fall on 16 grid
// positions along each of the two last dimensions (bin edge at most 17 - W,
// W = 2m + 2 taps; 7 cells at m = 4).  A node's window over those positions
// is its W values at its offset in the bin and zeros elsewhere, and both
// transforms become products with 16 x 16 operands:
//
//   B^T  T_i[e1][e2] += sum_k (psi0_k[i] psi1_k[e1]) (psi2_k[e2] f_k)
//        for the W planes i of four nodes k of one dimension-0 cell: one
//        16 x 16 x 4 product per plane and real / imaginary part, the tile
//        planes staying in registers.  Nodes arrive sorted by their
//        dimension-0 cell along a whole column of bins, so a wavefront keeps
//        a ring of W planes and writes a plane out when the nodes have passed
//        it: no LDS tile, no read-modify-write, no atomics.
//   B    C[e1][k] += psi0_k[i] (sum_e2 g_i[e1][e2] psi2_k[e2])
//        for 16 nodes k: four 16 x 16 x 4 products per plane and part, then
//        f_k = sum_e1 psi1_k[e1] C[e1][k].  A wavefront walks down the column
//        with the planes its nodes reach in registers.
//
// Bound: the matrix cores and the vector ALUs together.  A node costs W planes
// x 2 parts x 16 x 16 multiply-adds, of which (W/16)^2 meet a nonzero window:
// at m = 4 160 cycles of a SIMD in FP32 (v_mfma_f32_16x16x4_f32, 32 cycles
// each), 320 in FP64; vector instructions do not overlap with these (measured:
// 5.5 cycles each between FP32 products), so the kernels are built to issue
// few of them per node.  Measured against the LDS-tile kernels (spread_impl.hpp,
// spread_runs.hpp), m = 4, 256^3 grid:
//   B^T, FP32, 2^24 kooshball nodes   4.01 + 0.25 ms -> 1.77 + 0.27 (reduction)
//   B^T, FP64, 2^21 uniform nodes     3.49 + 1.87 ms -> 0.75 + 0.50
//   B,   FP64, 2^21 uniform nodes     7.03 ms -> 0.96
//   B,   FP32, 2^24 kooshball nodes   1.62 ms -> 1.96; such sets and short
//     windows keep the LDS tiles, over slabs of these bins (bin_nodes): 1.53
// FP32 sums are cut so that no product sums more than 128 nodes (B^T) or the 16
// positions of one plane (B): single sums over an item or a window lost up to a
// bit (kooshball adjoint 3.0e-7 against FP64, 1.9e-7 as it is).
// FP64 on sparse nodes (6 per column and plane) is bound by its grid traffic:
// 256 / 49 grid cells read or written per cell, 41 planes per 32.
#pragma once

#include "mx_util.hpp"

namespace nfft_hip {

// B^T of one work item: a run of nodes of one column (dimension-1 and -2
// bins), sorted by dimension-0 cell.  Two wavefronts per item, each
// evaluating the windows of 16 nodes of a chunk of 32 (lane = node + 16
// dimension) into LDS and owning half of the ring's planes; both read the
// windows back as the products' operands, four nodes of one dimension-0 cell
// at a time (fewer where the cell's nodes or the chunk end; the missing ones
// enter with value zero).  Output: the item's planes of 16 x 16 cells in
// scratch, summed into the grid by k_mx_gather3.
template <typename R, int W, bool SHARED>
__global__ __launch_bounds__(128, sizeof(R) == 4 ? (W <= 10 ? 4 : 3) : 2) void k_mx_spread3(
    const cplx<R> *__restrict__ fin, cplx<R> *__restrict__ tiles, const int *__restrict__ perm,
    const int *__restrict__ cell, const R *__restrict__ frac, const int4 *__restrict__ subs,
    const int4 *__restrict__ info, BinGeom gg, WinParams<R> wp) {
  constexpr int NC = 32, H = W / 2;
  __shared__ __align__(16) R win[3 * NC * kMxPitch];
  __shared__ __align__(16) cplx<R> sf[NC];
  __shared__ int sc0[NC];
  __shared__ __align__(16) R spoly[SHARED ? 1 : 3 * (W / 2) * kMxCoef<R>];
  // right-hand side blockIdx.y of a batched launch
  fin += (long)blockIdx.y * gg.bs_f;
  tiles += (long)blockIdx.y * gg.bs_t;
  const int4 sp = subs[blockIdx.x];
  const int4 nf = info[sp.w];  // first plane in scratch, first node's cell, planes
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int me = wv * 16 + j;  // node of the chunk whose windows this lane evaluates
  const int t = q < 3 ? q : 0;
  const int col = sp.x / gg.nb[0];
  const int b1 = col / gg.nb[2], b2 = col - b1 * gg.nb[2];
  const int lo = t == 1 ? mx_lo(b1, gg.n[1], gg.nb[1]) : mx_lo(b2, gg.n[2], gg.nb[2]);
  if constexpr (!SHARED) {
    mx_load_poly<R, 3, W>(spoly, wp.poly, threadIdx.x, 128);
    __syncthreads();
  }
  // FP32: a product's sum runs over 4 chunks (2 where more nodes reach a cell),
  // the sums of these over the item (one sum over the thousands of nodes of a
  // dense item would lose a bit)
  constexpr bool TWO = sizeof(R) == 4;
  constexpr int FOLD = W >= 14 ? 2 : 4;
  mx4<R> acc[H][2], sum[TWO ? H : 1][2];
#pragma unroll
  for (int i = 0; i < H; i++) {
    acc[i][0] = acc[i][1] = mx4<R>{0, 0, 0, 0};
    if constexpr (TWO) sum[i][0] = sum[i][1] = mx4<R>{0, 0, 0, 0};
  }
  const int *cellp = cell + t * gg.M + sp.y;
  const R *fracp = frac + t * gg.M + sp.y;
  const int *permp = perm + sp.y;
  const int last = sp.z - 1;
  // node data one chunk ahead, node indices two
  int c = cellp[min(me, last)];
  R fr = fracp[min(me, last)];
  cplx<R> fv = cplx<R>{0, 0};
  int pnext = 0;
  if (q == 3) {
    fv = fin[permp[min(me, last)]];
    pnext = permp[min(NC + me, last)];
  }
  // the plane of a node's tap i is slot (its cell + i) mod W of the ring,
  // slots H wv .. H wv + H - 1 in this wavefront: lane i of a 16-lane row
  // reads the weight of own slot i, so that the products need no case per
  // rotation
  int a0 = nf.y;              // dimension-0 cell of the nodes at hand
  int rot = a0 % W - H * wv;  // own slot of its first plane, which no later cell reaches
  auto tap_of_slot = [&]() {
    const int i = (j < H ? j : 0) - rot;
    return i < 0 ? i + W : i;
  };
  int t0 = tap_of_slot();
  cplx<R> *out = tiles + (long)nf.x * 256 + j;
  auto flush = [&]() {
#pragma unroll
    for (int s = 0; s < H; s++)
      if (rot == s) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          // (opaque copies: the compiler otherwise keeps the accumulators as
          // (re, im) pairs across the node loop and moves all of them around
          // every product, 40 moves per 20 of them)
          R vr = acc[s][0][r], vi = acc[s][1][r];
          if constexpr (TWO) {
            vr += sum[s][0][r];
            vi += sum[s][1][r];
            mx_clear(sum[s][0], r);
            mx_clear(sum[s][1], r);
          }
          asm("" : "+v"(vr));
          asm("" : "+v"(vi));
          out[mx_row<R>(q, r) * 16] = cplx<R>{vr, vi};
          mx_clear(acc[s][0], r);
          mx_clear(acc[s][1], r);
        }
      }
    out += 256;
    rot = rot + 1 < W - H * wv ? rot + 1 : -H * wv;
  };
  for (int base = 0; base < sp.z; base += NC) {
    if (q < 3) {
      const R *poly = wp.poly;
      // (the coefficients are read again for every chunk: held over the
      // loop they would take all registers)
      asm volatile("" : "+s"(poly));
      mx_window_row<R, W>(win + (t * NC + me) * kMxPitch, t == 0 ? 0 : c - lo, fr - R(0.5),
                          [&](int w) {
                            if constexpr (SHARED) return poly + w * (poly_deg_v<R> + 1);
                            else return spoly + (t * (W / 2) + w) * kMxCoef<R>;
                          });
      if (q == 0) sc0[me] = c;
    } else {
      sf[me] = fv;
    }
    const int nn = min(base + NC + me, last);
    c = cellp[nn];
    fr = fracp[nn];
    if (q == 3) {
      fv = fin[pnext];
      pnext = permp[min(base + 2 * NC + me, last)];
    }
    __syncthreads();
    const int cnt = min(NC, sp.z - base);
    const int c0 = sc0[lane & (NC - 1)];
    for (int k = 0; k < cnt;) {
      // the nodes k .. end - 1 of one cell
      const int ak = __builtin_amdgcn_readlane(c0, k);
      const unsigned long long same = __ballot(lane < cnt && c0 == ak) >> k;
      const int end = k + (int)__builtin_ctzll(~same);
      if (a0 < ak) {
        for (; a0 < ak; a0++) flush();
        t0 = tap_of_slot();
      }
      auto four = [&](int idx, bool live) {
        const R *row = win + idx * kMxPitch;
        const R p0 = row[t0], p1 = row[NC * kMxPitch + j], p2 = row[2 * NC * kMxPitch + j];
        const cplx<R> v = sf[idx];
        const R br = live ? p2 * v.x : R(0), bi = live ? p2 * v.y : R(0);
        R a[H];
        mx_weights<R, H>(a, p0, p1);
#pragma unroll
        for (int i = 0; i < H; i++) {
          acc[i][0] = mx_mul(a[i], br, acc[i][0]);
          acc[i][1] = mx_mul(a[i], bi, acc[i][1]);
        }
      };
      for (; k + 4 <= end; k += 4) four(k + q, true);
      if (k < end) four(min(k + q, NC - 1), k + q < end);
      k = end;
    }
    if constexpr (TWO) {
      if ((base / NC) % FOLD == FOLD - 1) {
#pragma unroll
        for (int s = 0; s < H; s++)
#pragma unroll
          for (int x = 0; x < 2; x++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
              sum[s][x][r] += acc[s][x][r];
              mx_clear(acc[s][x], r);
            }
      }
    }
    __syncthreads();
  }
  for (int i = 0; i < W; i++) flush();
}

// B of one work item (the items of k_mx_spread3), 16 nodes at a time.  The
// products' second operand is the grid: a wavefront keeps the planes that the
// nodes at hand reach in registers, a ring of W + kMxSpan - 1 planes of which
// a chunk's nodes of up to kMxSpan dimension-0 cells use W .. W + kMxSpan - 1,
// and loads each plane once as the nodes move on (the next one ahead of its
// use).  FP32: both parts in one wavefront; FP64: the real parts in one, the
// imaginary parts in the other.
template <typename R> constexpr int kMxParts = sizeof(R) == 4 ? 1 : 2;

template <typename R, int W, bool SHARED>
__global__ __launch_bounds__(64 * kMxParts<R>, sizeof(R) == 4 && W <= 10 ? 3 : 2) void k_mx_interp3(
    const cplx<R> *__restrict__ g, cplx<R> *__restrict__ fout, const int *__restrict__ perm,
    const int *__restrict__ cell, const R *__restrict__ frac, const int4 *__restrict__ subs,
    BinGeom gg, WinParams<R> wp) {
  constexpr int NW = kMxParts<R>, NP = 2 / NW, NC = 16 * NW;
  constexpr int Z = kMxSpan - 1, RW = mx_ring(W);
  static_assert(W + 2 * Z <= kMxPitch, "zeros before and after the dimension-0 taps");
  // window rows: dimension 1, 0 (taps from position Z on), 2.  (A lane whose
  // node is not of the cells at hand reads outside its dimension-0 row, at
  // most a bin's cells away and so inside win, and drops its result.)
  __shared__ __align__(16) R win[3 * NC * kMxPitch];
  __shared__ int sc0[NC];
  __shared__ __align__(16) R spoly[SHARED ? 1 : 3 * (W / 2) * kMxCoef<R>];
  g += (long)blockIdx.y * gg.bs_g;
  fout += (long)blockIdx.y * gg.bs_f;
  const int4 sp = subs[blockIdx.x];
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const int wv = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int me = wv * 16 + j;
  // dimension whose windows this lane evaluates, and its place in win
  const int t = q < 3 ? q : 0, tp = t == 2 ? 2 : 1 - t;
  const int col = sp.x / gg.nb[0];
  const int b1 = col / gg.nb[2], b2 = col - b1 * gg.nb[2];
  const int lo1 = mx_lo(b1, gg.n[1], gg.nb[1]), lo2 = mx_lo(b2, gg.n[2], gg.nb[2]);
  const int shift0 = t == 0 ? 0 : (t == 1 ? lo1 : lo2);
  if constexpr (!SHARED) {
    mx_load_poly<R, 3, W>(spoly, wp.poly, threadIdx.x, 64 * NW);
    __syncthreads();
  }
  // this lane's grid cells: row e1 = j, columns e2 = 4 q + s
  long goff[4];
  {
    int c1 = lo1 - gg.m + j;
    c1 += c1 < 0 ? gg.n[1] : (c1 >= gg.n[1] ? -gg.n[1] : 0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      int c2 = lo2 - gg.m + 4 * q + s;
      c2 += c2 < 0 ? gg.n[2] : (c2 >= gg.n[2] ? -gg.n[2] : 0);
      goff[s] = (long)c1 * gg.n[2] + c2;
    }
  }
  const long plane = (long)gg.n[1] * gg.n[2];
  auto load_plane = [&](int p, R (&d)[NP][4]) {
    const int c0 = mx_plane(p, gg.m, gg.n[0]);
    const cplx<R> *gp = g + (long)c0 * plane;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      if constexpr (NP == 2) {
        const cplx<R> v = gp[goff[s]];
        d[0][s] = v.x;
        d[1][s] = v.y;
      } else {
        d[0][s] = reinterpret_cast<const R *>(gp + goff[s])[wv];
      }
    }
  };
  int ra = cell[sp.y];  // the ring holds planes ra .. ra + RW - 1, plane p in slot p mod RW
  int rot = ra % RW;
  R ring[RW][NP][4], next[NP][4];
#pragma unroll
  for (int s = 0; s < RW; s++) load_plane(ra + (s < rot ? s - rot + RW : s - rot), ring[s]);
  load_plane(ra + RW, next);
  const int *cellp = cell + t * gg.M + sp.y;
  const R *fracp = frac + t * gg.M + sp.y;
  const int last = sp.z - 1;
  int c = cellp[min(me, last)];
  R fr = fracp[min(me, last)];
  for (int base = 0; base < sp.z; base += NC) {
    if (q < 3) {
      const R *poly = wp.poly;
      asm volatile("" : "+s"(poly));  // as in k_mx_spread3
      mx_window_row<R, W>(win + (tp * NC + me) * kMxPitch, t == 0 ? Z : c - shift0, fr - R(0.5),
                          [&](int w) {
                            if constexpr (SHARED) return poly + w * (poly_deg_v<R> + 1);
                            else return spoly + (t * (W / 2) + w) * kMxCoef<R>;
                          });
      if (q == 0) sc0[me] = c;
    }
    const int nn = min(base + NC + me, last);
    c = cellp[nn];
    fr = fracp[nn];
    int pj[NW];
#pragma unroll
    for (int h = 0; h < NW; h++)
      pj[h] = perm[sp.y + min(base + 16 * h + j, last)];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NW; h++) {
      const int cnt = min(16, sp.z - base - 16 * h);
      const int c0 = sc0[16 * h + j];
      const R *rows = win + 16 * h * kMxPitch;
      R a2[4];
#pragma unroll
      for (int s = 0; s < 4; s++) a2[s] = rows[(2 * NC + j) * kMxPitch + 4 * q + s];
      for (int k = 0; k < cnt;) {
        // nodes k .. end - 1: cells ak .. az
        const int ak = __builtin_amdgcn_readlane(c0, k);
        const int end = __popcll(__ballot(lane < cnt && c0 <= ak + Z));
        const int az = __builtin_amdgcn_readlane(c0, end - 1);
        for (; ra < az - Z; ra++) {
#pragma unroll
          for (int s = 0; s < RW; s++)
            if (rot == s) {
#pragma unroll
              for (int u = 0; u < 4; u++)
#pragma unroll
                for (int x = 0; x < NP; x++) ring[s][x][u] = next[x][u];
            }
          rot = rot + 1 < RW ? rot + 1 : 0;
          load_plane(ra + 1 + RW, next);
        }
        mx4<R> acc[NP];
#pragma unroll
        for (int x = 0; x < NP; x++) acc[x] = mx4<R>{0, 0, 0, 0};
        const R *w0 = rows + (NC + j) * kMxPitch + Z - c0;
#pragma unroll
        for (int s = 0; s < RW; s++) {
          const int p = ra + (s < rot ? s - rot + RW : s - rot);
          if (p >= ak && p < az + W) {
            const R w = w0[p];
            mx4<R> z[NP] = {};
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
              for (int x = 0; x < NP; x++) z[x] = mx_mul(ring[s][x][u], a2[u], z[x]);
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
              for (int x = 0; x < NP; x++) acc[x][u] = fma(w, z[x][u], acc[x][u]);
          }
        }
        // rows e1, columns nodes: four rows in the lane, 16 over its column
        R out[NP] = {};
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const R p1 = rows[j * kMxPitch + mx_row<R>(q, u)];
#pragma unroll
          for (int x = 0; x < NP; x++) out[x] = fma(acc[x][u], p1, out[x]);
        }
#pragma unroll
        for (int x = 0; x < NP; x++) out[x] = mx_col_sum(out[x]);
        if (lane >= k && lane < end) {
          if constexpr (NP == 2) fout[pj[h]] = cplx<R>{out[0], out[1]};
          else reinterpret_cast<R *>(fout + pj[h])[wv] = out[0];
        }
        k = end;
      }
    }
    __syncthreads();
  }
}

// Sums the planes of the items of a spreading bin that has several (dense
// bins, up to hundreds of items) into one tile of the bin's planes, so that
// the reduction below reads one tile per bin.  A workgroup owns one plane of
// one such bin; a thread one cell.
template <typename R>
__global__ __launch_bounds__(256) void k_mx_sum3(cplx<R> *__restrict__ tiles,
                                                 const int4 *__restrict__ info,
                                                 const int4 *__restrict__ bin_info,
                                                 const int *__restrict__ multi,
                                                 const int *__restrict__ sp_first,
                                                 const int *__restrict__ sp_count, BinGeom gg) {
  tiles += (long)blockIdx.z * gg.bs_t;
  const int bin = multi[blockIdx.x];
  const int4 bi = bin_info[bin];  // first plane in scratch, dimension-0 cell, planes
  const int pl = blockIdx.y;
  if (pl >= bi.z) return;
  const int first = sp_first[bin], cnt = sp_count[bin];
  __shared__ int list[256];  // first to last: planes of the items that cover this one
  __shared__ int wsum[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  R ar = 0, ai = 0;
  for (int s0 = 0; s0 < cnt; s0 += 256) {
    const int s = s0 + threadIdx.x;
    int at = -1;
    if (s < cnt) {
      const int4 nf = info[first + s];
      const int p = pl - (nf.y - bi.y);
      if (p >= 0 && p < nf.z) at = nf.x + p;
    }
    const unsigned long long in = __ballot(at >= 0);
    if (lane == 0) wsum[wv] = __popcll(in);
    __syncthreads();
    int k = __popcll(in & ((1ull << lane) - 1));
    for (int w = 0; w < wv; w++) k += wsum[w];
    if (at >= 0) list[k] = at;
    const int n = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    for (int i = 0; i < n; i += 8) {
      cplx<R> v[8];
#pragma unroll
      for (int u = 0; u < 8; u++)
        v[u] = i + u < n ? tiles[(long)list[i + u] * 256 + threadIdx.x] : cplx<R>{0, 0};
      // (in pairs first: shorter FP32 sums)
#pragma unroll
      for (int w = 1; w < 8; w *= 2)
#pragma unroll
        for (int u = 0; u < 8; u += 2 * w) v[u] = cplx<R>{v[u].x + v[u + w].x, v[u].y + v[u + w].y};
      ar += v[0].x;
      ai += v[0].y;
    }
    __syncthreads();
  }
  tiles[((long)bi.x + pl) * 256 + threadIdx.x] = cplx<R>{ar, ai};
}

// Tile reduction: every grid cell as the sum of the bins' planes that cover
// it.  A workgroup owns one plane c0 and one dimension-1 bin's rows and up to
// 256 cells of dimension 2; a thread owns one dimension-2 cell of all those
// rows.  Tile rows of 16 cells are read whole by one workgroup, so each tile
// plane is read by the three workgroups of its dimension-1 neighbourhood
// only; these are adjacent in the launch order of one XCD and meet in its L2.
// Bound: the latency of bin information -> tile values, so the next bins'
// information and the values of CH neighbours along dimension 2 are in flight
// together.  One neighbour at a time -> as it is: 256^3 FP64, 2^21 uniform
// nodes 595 -> 495 us (1.9 GB read, 0.27 GB written); 256^3 FP32 kooshball 319 ->
// 219; 180 x 150 x 120 FP32 100 -> 46 (also by workgroups of 128 threads, which
// rows of 120 cells fill).
template <typename R, int W>
__global__ __launch_bounds__(256) void k_mx_gather3(const cplx<R> *__restrict__ tiles,
                                                    const int4 *__restrict__ bin_info,
                                                    cplx<R> *__restrict__ g, BinGeom gg,
                                                    int chunks, int total) {
  constexpr int ROWS = 17 - W;
  // dimension-2 neighbours whose values are in flight together
  constexpr int CH = ROWS * sizeof(R) <= 72 ? 3 : 1;
  tiles += (long)blockIdx.y * gg.bs_t;
  g += (long)blockIdx.y * gg.bs_g;
  // consecutive work of one XCD is consecutive in (plane, bin)
  const int per = (total + 7) / 8;
  int w = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || w >= total) return;
  const int ch = w % chunks;
  w /= chunks;
  const int b1 = w % gg.nb[1], c0 = w / gg.nb[1];
  const int n0 = gg.n[0], n1 = gg.n[1], n2 = gg.n[2];
  const int nb1 = gg.nb[1], nb2 = gg.nb[2], nb0 = gg.nb[0];
  const int c2 = ch * (int)blockDim.x + threadIdx.x;
  if (c2 >= n2) return;
  const int lo1 = mx_lo(b1, n1, nb1), rows = mx_lo(b1 + 1, n1, nb1) - lo1;
  const int b2 = mx_bin(c2, n2, nb2);
  const int bB = c0 / gg.bs[0];
  const int s1 = gg.mx_span[1], s2 = gg.mx_span[2], s0 = gg.mx_span[0];
  // neighbour jj of span: all bins, or the bins around the own one
  auto nbr = [](int b, int jj, int span, int nb) {
    if (span == nb) return jj;
    int v = b + jj - span / 2;
    v += v < 0 ? nb : 0;
    return v >= nb ? v - nb : v;
  };
  R ar[ROWS], ai[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; i++) ar[i] = ai[i] = R(0);
  // tile column of this cell in the dimension-2 neighbours j2 .. j2 + CH - 1,
  // 16 or more where the cell lies outside
  int bb2[CH], e2[CH];
  for (int j2 = 0; j2 < s2; j2 += CH) {
#pragma unroll
    for (int u = 0; u < CH; u++) {
      e2[u] = 16;
      bb2[u] = 0;
      if (j2 + u < s2) {
        bb2[u] = nbr(b2, j2 + u, s2, nb2);
        e2[u] = c2 - mx_lo(bb2[u], n2, nb2) + gg.m;
        e2[u] += e2[u] < 0 ? n2 : (e2[u] >= n2 ? -n2 : 0);
      }
    }
    // the dimension-1 and -0 neighbours (j1, j0), a step ahead
    int e1 = 0, e1_next = 0;
    int4 bi[CH], bi_next[CH];
    auto fetch = [&](int it) {
      const int j1 = it / s0, j0 = it - j1 * s0;
      const int bb1 = nbr(b1, j1, s1, nb1), bb0 = nbr(bB, j0, s0, nb0);
      e1_next = lo1 - mx_lo(bb1, n1, nb1) + gg.m;  // tile row of the first owned row
      e1_next += e1_next < 0 ? n1 : (e1_next >= n1 ? -n1 : 0);
      // planes of that bin: none beyond its cells' windows
      const int f0 = bb0 * gg.bs[0], h0 = min(n0, f0 + gg.bs[0]) - f0;
      int d0 = c0 - f0 + gg.m;
      d0 += d0 < 0 ? n0 : (d0 >= n0 ? -n0 : 0);
#pragma unroll
      for (int u = 0; u < CH; u++) {
        bi_next[u] = make_int4(0, 0, 0, 0);
        if (d0 < h0 + W - 1 && e2[u] < 16)
          bi_next[u] = bin_info[(bb1 * nb2 + bb2[u]) * nb0 + bb0];
      }
    };
    fetch(0);
    for (int it = 0; it < s1 * s0; it++) {
      e1 = e1_next;
#pragma unroll
      for (int u = 0; u < CH; u++) bi[u] = bi_next[u];
      if (it + 1 < s1 * s0) fetch(it + 1);
      cplx<R> v[CH][ROWS];
#pragma unroll
      for (int u = 0; u < CH; u++) {
        int pl = c0 - bi[u].y + gg.m;
        pl += pl < 0 ? n0 : (pl >= n0 ? -n0 : 0);
        const bool in = pl < bi[u].z;
        const cplx<R> *tp = tiles + ((long)bi[u].x + pl) * 256 + e2[u];
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
          int e = e1 + i;
          e -= e >= n1 ? n1 : 0;
          v[u][i] = cplx<R>{0, 0};
          if (in && e < 16 && i < rows) v[u][i] = tp[e * 16];
        }
      }
#pragma unroll
      for (int u = 0; u < CH; u++)
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
          ar[i] += v[u][i].x;
          ai[i] += v[u][i].y;
        }
    }
  }
  cplx<R> *gp = g + ((long)c0 * n1 + lo1) * n2 + c2;
#pragma unroll
  for (int i = 0; i < ROWS; i++)
    if (i < rows) gp[(long)i * n2] = cplx<R>{ar[i], ai[i]};
}

// ==================================================================== dispatch
template <typename R, int M_>
void mx_spread3(const cplx<R> *f, cplx<R> *tiles, const Engine<R> &e, const BinGeom &gg,
                hipStream_t s, int nb) {
  auto fn = e.win.poly_shared ? k_mx_spread3<R, 2 * M_ + 2, true> : k_mx_spread3<R, 2 * M_ + 2, false>;
  hipLaunchKernelGGL(fn, dim3((unsigned)e.sp_nsub, (unsigned)nb), dim3(128), 0, s, f,
                     tiles, e.perm, e.cell, e.frac, e.sp_subs, e.mx_info, gg, e.win);
}

template <typename R, int M_>
void mx_interp3(const cplx<R> *g, cplx<R> *f, const Engine<R> &e, const BinGeom &gg,
                hipStream_t s, int nb) {
  constexpr int W = 2 * M_ + 2;
  auto fn = e.win.poly_shared ? k_mx_interp3<R, W, true> : k_mx_interp3<R, W, false>;
  hipLaunchKernelGGL(fn, dim3((unsigned)e.nsub, (unsigned)nb), dim3(64 * kMxParts<R>), 0, s, g, f,
                     e.perm, e.cell, e.frac, e.subs, gg, e.win);
}

template <typename R, int M_>
void mx_gather3(const cplx<R> *tiles, cplx<R> *g, const Engine<R> &e, const BinGeom &gg,
                hipStream_t s, int nb) {
  if (e.mx_multi_n > 0)
    hipLaunchKernelGGL((k_mx_sum3<R>),
                       dim3((unsigned)e.mx_multi_n, (unsigned)(gg.bs[0] + 2 * M_ + 1), (unsigned)nb),
                       dim3(256), 0, s, const_cast<cplx<R> *>(tiles), e.mx_info, e.mx_bin_info,
                       e.mx_multi, e.sp_first, e.sp_count, gg);
  const int chunks = (gg.n[2] + 255) / 256;
  const int threads = (gg.n[2] + 64 * chunks - 1) / (64 * chunks) * 64;  // of 256 at most
  const int total = gg.n[0] * gg.nb[1] * chunks;
  const unsigned blocks = 8u * (unsigned)((total + 7) / 8);
  hipLaunchKernelGGL((k_mx_gather3<R, 2 * M_ + 2>), dim3(blocks, (unsigned)nb),
                     dim3((unsigned)threads), 0, s, tiles, e.mx_bin_info, g, gg, chunks, total);
}

// the launches of window cut-off m (1 .. kMxMaxM)
#define NFFT_MX_DISPATCH(FN, ...)              \
  switch (gg.m) {                              \
    case 1: FN<R, 1>(__VA_ARGS__); break;      \
    case 2: FN<R, 2>(__VA_ARGS__); break;      \
    case 3: FN<R, 3>(__VA_ARGS__); break;      \
    case 4: FN<R, 4>(__VA_ARGS__); break;      \
    case 5: FN<R, 5>(__VA_ARGS__); break;      \
    case 6: FN<R, 6>(__VA_ARGS__); break;      \
    default: break;                            \
  }

template <typename R>
void launch_mx_spread(const cplx<R> *f, const Engine<R> &e, hipStream_t s, int nb,
                      const BinGeom *gb, cplx<R> *tiles) {
  if (e.sp_nsub == 0) return;
  const BinGeom &gg = gb ? *gb : e.geom;
  if (!tiles) tiles = e.tiles;
  NFFT_MX_DISPATCH(mx_spread3, f, tiles, e, gg, s, nb)
}

template <typename R>
void launch_mx_interp(const cplx<R> *g, cplx<R> *f, const Engine<R> &e, hipStream_t s, int nb,
                      const BinGeom *gb) {
  if (e.nsub == 0) return;
  const BinGeom &gg = gb ? *gb : e.geom;
  NFFT_MX_DISPATCH(mx_interp3, g, f, e, gg, s, nb)
}

template <typename R>
void launch_mx_gather(const Engine<R> &e, cplx<R> *g, hipStream_t s, int nb, const BinGeom *gb,
                      cplx<R> *tiles) {
  const BinGeom &gg = gb ? *gb : e.geom;
  if (!tiles) tiles = e.tiles;
  NFFT_MX_DISPATCH(mx_gather3, tiles, g, e, gg, s, nb)
}
#undef NFFT_MX_DISPATCH

}  // namespace nfft_hip
