// Register-blocked complex contractions for many or large tiles: the forms
// of the grouped mode product and hole contraction whose launch fills the
// card, where operand traffic and not latency decides.
//
// gc_block (hole contraction): a workgroup owns a macro tile of NT x NT
// output tiles of 16 x 16; every wavefront holds all of it in registers and
// walks its own share of the reduction, so each element of the bra and the
// ket is loaded once per macro tile, and the shares are summed in LDS in
// wavefront order.  One wavefront per 16 x 16 tile (gc_grouped) reads each
// operand once per tile of the other index, from workgroups that the
// dispatcher spreads over XCDs with L2s of their own.  A reduction may be
// shared by several workgroups; their partial tiles are summed in order by
// gc_block_sum.  4096 order-3 complex128 tensors with legs 8-64 (4.3 GB of
// operands): 1552 -> 1086 us, 3.9 TB/s, where a large copy reaches 4.9; 1000
// complex64 tensors of legs 3-61: 418 -> 318 us.
//
// gm_block (mode product): a wavefront owns 2 x 2 output tiles, so X is read
// once per 32 columns and M once per 32 rows.  The 4096 tensors' products:
// 1284 -> 1222 us (3.5 TB/s read and written).
//
// Descriptors pass gm_lean_ok / gc_lean_ok (32-bit offsets, see gemm_ops.hip).
#include <algorithm>
#include <type_traits>

#include "gemm_dev.hpp"
#include "gemm_ops.hpp"

namespace qtg {

namespace {

// --------------------------------------------------------- hole contraction
// This wavefront's share [kbeg, kend) of NR x NC tiles at columns j0 of the
// bra and l0 of the ket, KS k-steps of four per stage, the next stage's
// operands in flight behind the current MFMAs (4 per tile and k-step, 64
// cycles each in FP64): the loads of a stage stand in straight-line code and
// nothing touches their values before the stage that uses them.  Columns past
// the tensor are clamped into it (never stored); only the last, partial stage
// masks k past the share.
template <typename T, int NT, int NR, int NC, int KS>
__device__ inline void gc_block_product(const GcDesc& d, int j0, int l0, int kbeg, int kend,
                                        const cplx<T>* __restrict__ X, const cplx<T>* __restrict__ Y,
                                        typename MF<T>::v4 (&cr)[NT][NT], typename MF<T>::v4 (&ci)[NT][NT]) {
  const int lane = threadIdx.x & 63, li = lane & 15, kk = lane >> 4;
  const uint32_t bef = (uint32_t)d.bef, aft = (uint32_t)d.aft;
  const uint32_t xs = bef * (uint32_t)d.nx, ys = bef * (uint32_t)d.ny;  // stride of a
  const uint32_t xmax = (bef - 1u) + (aft - 1u) * xs, ymax = (bef - 1u) + (aft - 1u) * ys;
  uint32_t xrow[NR], yrow[NC];
#pragma unroll
  for (int t = 0; t < NR; ++t) xrow[t] = (uint32_t)min(j0 + t * 16 + li, d.nx - 1) * bef;
#pragma unroll
  for (int t = 0; t < NC; ++t) yrow[t] = (uint32_t)min(l0 + t * 16 + li, d.ny - 1) * bef;
  const cplx<T>* xp = X + d.x;
  const cplx<T>* yp = Y + d.y;
  const int k0 = kbeg + kk;
  uint32_t b = (uint32_t)k0 % bef;
  const uint32_t a0 = (uint32_t)k0 / bef;
  uint32_t px = b + a0 * xs, py = b + a0 * ys;
  const uint32_t q4 = 4u / bef, r4 = 4u % bef;
  const uint32_t dx = r4 + q4 * xs, dy = r4 + q4 * ys;
  auto load = [&](cplx<T>(&xv)[KS][NR], cplx<T>(&yv)[KS][NC]) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint32_t ox = min(px, xmax), oy = min(py, ymax);
#pragma unroll
      for (int t = 0; t < NR; ++t) xv[u][t] = ld32(xp, xrow[t] + ox);
#pragma unroll
      for (int t = 0; t < NC; ++t) yv[u][t] = ld32(yp, yrow[t] + oy);
      b += r4;
      const bool carry = b >= bef;
      b -= carry ? bef : 0u;
      px += dx + (carry ? xs - bef : 0u);
      py += dy + (carry ? ys - bef : 0u);
    }
  };
  auto kstep = [&](const cplx<T>(&xv)[NR], const cplx<T>(&yv)[NC]) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const T nxi = -xv[i].im;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        cr[i][j] = MF<T>::mma(xv[i].re, yv[j].re, cr[i][j]);
        ci[i][j] = MF<T>::mma(xv[i].re, yv[j].im, ci[i][j]);
        cr[i][j] = MF<T>::mma(xv[i].im, yv[j].im, cr[i][j]);
        ci[i][j] = MF<T>::mma(nxi, yv[j].re, ci[i][j]);
      }
    }
  };
  // one stage that starts at k; the share's last stage masks its tail
  auto stage = [&](int k, cplx<T>(&xv)[KS][NR], cplx<T>(&yv)[KS][NC]) {
    if (k + 4 * KS <= kend) {
#pragma unroll
      for (int u = 0; u < KS; ++u) kstep(xv[u], yv[u]);
      return;
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (k + 4 * u >= kend) break;
      const bool kv = k + 4 * u + kk < kend;
#pragma unroll
      for (int t = 0; t < NR; ++t) xv[u][t] = mk<T>(kv ? xv[u][t].re : (T)0, kv ? xv[u][t].im : (T)0);
#pragma unroll
      for (int t = 0; t < NC; ++t) yv[u][t] = mk<T>(kv ? yv[u][t].re : (T)0, kv ? yv[u][t].im : (T)0);
      kstep(xv[u], yv[u]);
    }
  };
  if (kbeg >= kend) return;
  cplx<T> xa[KS][NR], ya[KS][NC], xb[KS][NR], yb[KS][NC];
  load(xa, ya);
  if (kend - kbeg <= 4 * KS) {
    stage(kbeg, xa, ya);
    return;
  }
  for (int k = kbeg; k < kend; k += 8 * KS) {
    load(xb, yb);
    stage(k, xa, ya);
    load(xa, ya);
    if (k + 4 * KS < kend) stage(k + 4 * KS, xb, yb);
  }
}

// W wavefronts per workgroup.  Grouped: wgs[blockIdx.x] names the
// workgroup's descriptor and its index t within it.  One
// contraction alone (wgs null): the descriptor `one`, t = blockIdx.x.  The
// index runs over macro tiles, and per macro tile over the S = ksplit
// workgroups that share its reduction; with S > 1 each leaves its macro tile
// in `part` (NT x NT tiles of 256 per workgroup).
template <typename T, int NT, int W>
__global__ void __launch_bounds__(64 * W)
    gc_block(const GcDesc* __restrict__ descs, const GcBlockWg* __restrict__ wgs, GcDesc one, int S1,
             const cplx<T>* __restrict__ X0, const cplx<T>* __restrict__ X1, cplx<T>* O, cplx<T>* part) {
  constexpr int NB = NT > 1 ? 2 : 1;  // LDS buffers: one barrier per tile
  __shared__ cplx<T> red[NB * W * 256];
  typedef typename MF<T>::v4 v4;
  unsigned t = blockIdx.x;
  int di = 0;
  int64_t p0 = blockIdx.x;
  if (wgs) {
    const GcBlockWg w = wgs[blockIdx.x];
    di = w.desc;
    t = (unsigned)w.t;
    p0 = w.part;
  }
  const GcDesc d = wgs ? descs[di] : one;
  const int S = wgs ? d.ksplit : S1;
  const unsigned s = S > 1 ? t % (unsigned)S : 0u;
  if (S > 1) t /= (unsigned)S;
  const unsigned MJ = (unsigned)(d.nx + 16 * NT - 1) / (16u * NT);
  const unsigned lm = MJ == 1 ? t : t / MJ, jm = t - lm * MJ;
  const int j0 = (int)jm * 16 * NT, l0 = (int)lm * 16 * NT;
  const int nrb = min(NT, (d.nx - j0 + 15) >> 4), ncb = min(NT, (d.ny - l0 + 15) >> 4);
  const int wave = wave_id(), lane = threadIdx.x & 63;
  // this wavefront's share of K (a multiple of 4 long, except the last)
  const int K = d.bef * d.aft, nch = W * S;
  const int chunk = ((K + nch - 1) / nch + 3) & ~3;
  const int64_t kb64 = (int64_t)((int)s * W + wave) * chunk;
  const int kbeg = (int)min((int64_t)K, kb64), kend = min(K, kbeg + chunk);
  const cplx<T>* xbase = (d.sel & 1) ? X1 : X0;
  const cplx<T>* ybase = (d.sel & 2) ? X1 : X0;
  v4 cr[NT][NT], ci[NT][NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) cr[i][j] = ci[i][j] = v4{0, 0, 0, 0};
  if constexpr (NT == 1) {
    gc_block_product<T, 1, 1, 1, 4>(d, j0, l0, kbeg, kend, xbase, ybase, cr, ci);
  } else {
    if (nrb == 1 && ncb == 1) gc_block_product<T, NT, 1, 1, 4>(d, j0, l0, kbeg, kend, xbase, ybase, cr, ci);
    else if (nrb == 1) gc_block_product<T, NT, 1, 2, 2>(d, j0, l0, kbeg, kend, xbase, ybase, cr, ci);
    else if (ncb == 1) gc_block_product<T, NT, 2, 1, 2>(d, j0, l0, kbeg, kend, xbase, ybase, cr, ci);
    else gc_block_product<T, NT, 2, 2, 2>(d, j0, l0, kbeg, kend, xbase, ybase, cr, ci);
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    if (i >= nrb) break;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (j >= ncb) break;
      cplx<T>* buf = red + (NB > 1 ? ((i * NT + j) & 1) * W * 256 : 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) buf[wave * 256 + q * 64 + lane] = mk<T>(cr[i][j][q], ci[i][j][q]);
      __syncthreads();
      if (threadIdx.x < 256) {
        const int e = threadIdx.x, el = e & 63, q = e >> 6;
        cplx<T> v = buf[e];
#pragma unroll
        for (int w = 1; w < W; ++w) v = cadd(v, buf[w * 256 + e]);
        const int row = j0 + i * 16 + MF<T>::drow(el, q), col = l0 + j * 16 + (el & 15);
        if (S > 1) {
          part[((p0 * NT + j) * NT + i) * 256 + e] = v;
        } else if (row < d.nx && col < d.ny) {
          const int64_t o = d.out + row + (int64_t)col * d.nx;
          if (d.acc) v = cadd(v, O[o]);
          O[o] = v;
        }
      }
    }
    // buffers alternate over (i NT + j) & 1: with an odd number of tiles in
    // this row and an even NT the next row starts on the buffer just read
    if (NB > 1 && (ncb & 1) && i + 1 < nrb) __syncthreads();
  }
}

// Sums the S partial macro tiles (2 x 2 tiles) of a macro tile: 16
// workgroups each, 64 elements a workgroup; a wavefront adds a sixteenth of
// the partials in order, then the first adds the wavefronts' sums.
// sums[blockIdx.x / 16]: descriptor, macro tile and its first partial.
template <typename T>
__global__ void __launch_bounds__(1024)
    gc_block_sum(const GcDesc* __restrict__ descs, const GcBlockWg* __restrict__ sums, GcDesc one, int S1,
                 const cplx<T>* __restrict__ part, cplx<T>* O) {
  __shared__ cplx<T> red[15 * 64];
  const unsigned b = blockIdx.x >> 4, sub = blockIdx.x & 15u;
  int di = 0;
  unsigned macro = b;
  int64_t p0 = (int64_t)b * S1;
  if (sums) {
    const GcBlockWg w = sums[b];
    di = w.desc;
    macro = (unsigned)w.t;
    p0 = w.part;
  }
  const GcDesc d = sums ? descs[di] : one;
  const int S = sums ? d.ksplit : S1;
  const unsigned MJ = (unsigned)(d.nx + 31) / 32u;
  const unsigned lm = macro / MJ, jm = macro - lm * MJ;
  const int tile = (int)(sub >> 2), i = tile & 1, j = tile >> 1;
  const int lane = threadIdx.x & 63, e = (int)(sub & 3u) * 64 + lane, g = wave_id();
  const int r0 = (int)jm * 32 + i * 16, c0 = (int)lm * 32 + j * 16;
  if (r0 >= d.nx || c0 >= d.ny) return;  // the whole workgroup
  const int per = (S + 15) >> 4, s0 = min(S, g * per), s1 = min(S, s0 + per);
  const cplx<T>* p = part + (p0 * 4 + tile) * 256 + e;
  cplx<T> v = czero<T>();
#pragma unroll 8
  for (int s = s0; s < s1; ++s) v = cadd(v, p[(int64_t)s * 1024]);
  if (g > 0) red[(g - 1) * 64 + lane] = v;
  __syncthreads();
  if (g > 0) return;
#pragma unroll
  for (int k = 0; k < 15; ++k) v = cadd(v, red[k * 64 + lane]);
  const int row = r0 + MF<T>::drow(lane, e >> 6), col = c0 + (lane & 15);
  if (row < d.nx && col < d.ny) {
    const int64_t o = d.out + row + (int64_t)col * d.nx;
    if (d.acc) v = cadd(v, O[o]);
    O[o] = v;
  }
}

// ----------------------------------------------------- summed contractions
// One workgroup per macro tile and share: its wavefronts split the
// concatenated reduction of all segments evenly, so a sum over many small
// contractions (the summed matrices of a sweep) is as wide as one long one
// and needs neither a matrix per segment nor a pass to add them.  FP32
// products keep what a matrix per segment gave: a segment's share is added,
// with its coefficient, in FP64.
template <typename T, int NT, int W>
__global__ void __launch_bounds__(64 * W)
    gc_sum_kernel(const GcSum* __restrict__ tasks, const GcSeg* __restrict__ segs, const cplx<T>* __restrict__ X0,
                  const cplx<T>* __restrict__ X1, cplx<double>* O, cplx<double>* part) {
  typedef typename MF<T>::v4 v4;
  constexpr int NB = NT > 1 ? 2 : 1;
  __shared__ cplx<double> red[NB * W * 256];
  const GcSum d = tasks[blockIdx.x];
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int TJ = (d.n + 16 * NT - 1) / (16 * NT), lt = d.tile / TJ, jt = d.tile - lt * TJ;
  const int j0 = jt * 16 * NT, l0 = lt * 16 * NT;
  const int nrb = min(NT, (d.n - j0 + 15) >> 4), ncb = min(NT, (d.n - l0 + 15) >> 4);
  const int K = d.bef * d.aft, nseg = d.seg1 - d.seg0;
  const int64_t Kt = (int64_t)K * nseg;
  const int64_t nch = (int64_t)W * d.S;
  const int64_t chunk = ((Kt + nch - 1) / nch + 3) & ~(int64_t)3;
  const int64_t kb = min(Kt, ((int64_t)d.share * W + wave) * chunk), ke = min(Kt, kb + chunk);
  GcDesc g{};
  g.bef = d.bef;
  g.nx = g.ny = d.n;
  g.aft = d.aft;
  v4 cr[NT][NT], ci[NT][NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) cr[i][j] = ci[i][j] = v4{0, 0, 0, 0};
  constexpr bool kFlush = std::is_same<T, float>::value;
  typedef MF<double>::v4 dv4;
  dv4 dr[NT][NT], di[NT][NT];  // kFlush: the sum over segments
  if constexpr (kFlush) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) dr[i][j] = di[i][j] = dv4{0, 0, 0, 0};
  }
  int sg = kb < ke ? (int)(kb / K) : nseg;
  for (; sg < nseg && (int64_t)sg * K < ke; ++sg) {
    const int64_t s0 = (int64_t)sg * K;
    const GcSeg e = segs[d.seg0 + sg];
    g.x = e.x;
    g.y = e.y;
    const int lo = (int)(max(kb, s0) - s0), hi = (int)(min(ke, s0 + K) - s0);
    const cplx<T>* X = (e.sel & 1) ? X1 : X0;
    const cplx<T>* Y = (e.sel & 2) ? X1 : X0;
    if constexpr (NT == 1) {
      gc_block_product<T, 1, 1, 1, 4>(g, j0, l0, lo, hi, X, Y, cr, ci);
    } else {
      if (nrb == 1 && ncb == 1) gc_block_product<T, NT, 1, 1, 4>(g, j0, l0, lo, hi, X, Y, cr, ci);
      else if (nrb == 1) gc_block_product<T, NT, 1, 2, 2>(g, j0, l0, lo, hi, X, Y, cr, ci);
      else if (ncb == 1) gc_block_product<T, NT, 2, 1, 2>(g, j0, l0, lo, hi, X, Y, cr, ci);
      else gc_block_product<T, NT, 2, 2, 2>(g, j0, l0, lo, hi, X, Y, cr, ci);
    }
    if constexpr (kFlush) {
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double vr = cr[i][j][q], vi = ci[i][j][q];
            dr[i][j][q] += e.are * vr - e.aim * vi;
            di[i][j][q] += e.are * vi + e.aim * vr;
          }
          cr[i][j] = ci[i][j] = v4{0, 0, 0, 0};
        }
    }
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    if (i >= nrb) break;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (j >= ncb) break;
      cplx<double>* buf = red + (NB > 1 ? ((i * NT + j) & 1) * W * 256 : 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (kFlush) buf[wave * 256 + q * 64 + lane] = mk<double>(dr[i][j][q], di[i][j][q]);
        else buf[wave * 256 + q * 64 + lane] = mk<double>(cr[i][j][q], ci[i][j][q]);
      }
      __syncthreads();
      if (threadIdx.x < 256) {
        const int e = threadIdx.x, el = e & 63;
        cplx<double> v = buf[e];
#pragma unroll
        for (int w = 1; w < W; ++w) v = cadd(v, buf[w * 256 + e]);
        const int row = j0 + i * 16 + MF<T>::drow(el, e >> 6), col = l0 + j * 16 + (el & 15);
        if (d.S > 1) {
          part[((((int64_t)d.part + d.share) * NT + j) * NT + i) * 256 + e] = v;
        } else if (row < d.n && col < d.n) {
          const int64_t o = row + (int64_t)col * d.n;
          if (d.add >= 0) v = cadd(v, O[d.add + o]);
          O[d.out + o] = v;
        }
      }
    }
    if (NB > 1 && (ncb & 1) && i + 1 < nrb) __syncthreads();  // as in gc_block
  }
}

// The shares of a macro tile, added in order: one workgroup per 16 x 16 tile.
template <typename T, int NT>
__global__ void __launch_bounds__(256)
    gc_sum_add(const GcSum* __restrict__ sums, const cplx<double>* __restrict__ part, cplx<double>* O) {
  const GcSum d = sums[blockIdx.x / (NT * NT)];
  const int sub = blockIdx.x % (NT * NT), i = sub % NT, j = sub / NT;
  const int TJ = (d.n + 16 * NT - 1) / (16 * NT), lt = d.tile / TJ, jt = d.tile - lt * TJ;
  const int e = threadIdx.x, el = e & 63;
  const int row = (jt * NT + i) * 16 + MF<T>::drow(el, e >> 6), col = (lt * NT + j) * 16 + (el & 15);
  if (row >= d.n || col >= d.n) return;
  const cplx<double>* p = part + (((int64_t)d.part * NT + j) * NT + i) * 256 + e;
  cplx<double> v = czero<double>();
#pragma unroll 8
  for (int s = 0; s < d.S; ++s) v = cadd(v, p[(int64_t)s * (NT * NT * 256)]);
  const int64_t o = row + (int64_t)col * d.n;
  if (d.add >= 0) v = cadd(v, O[d.add + o]);
  O[d.out + o] = v;
}

// ------------------------------------------------------------- mode product
// out(b,i,a) = sum_l op(M)(i,l) X(b,l,a) (+ out) on RB x CB tiles of
// 16 rows (flattened (b, a)) x 16 columns i, KS k-steps of four per stage,
// staged as in gc_block_product.  TR (bef >= 4): accumulated transposed, so a
// lane holds one row and the 16 lanes of a store write 16 consecutive
// elements.  Rows and columns past the range are clamped into it (never
// stored); the last, partial stage masks X past K.
template <typename T, int RB, int CB, int KS, bool TR>
__device__ inline void gm_block_tiles(const GmDesc& d, uint32_t r0, int c0, const cplx<T>* __restrict__ X,
                                      const cplx<T>* __restrict__ M, cplx<T>* O) {
  typedef typename MF<T>::v4 v4;
  const int lane = threadIdx.x & 63, li = lane & 15, kk = lane >> 4;
  const uint32_t bef = (uint32_t)d.bef, R = bef * (uint32_t)d.aft;
  const int nin = d.nin, nout = d.nout;
  uint32_t xrow[RB], mrow[CB];
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    const uint32_t r = min(r0 + (uint32_t)(t * 16 + li), R - 1u);
    const uint32_t a = r / bef;
    xrow[t] = (r - a * bef) + a * bef * (uint32_t)nin;
  }
  const uint32_t mks = d.op == GM_N ? (uint32_t)nout : 1u;
  const T msign = d.op == GM_H ? (T)-1 : (T)1;
#pragma unroll
  for (int t = 0; t < CB; ++t) {
    const int j = min(c0 + t * 16 + li, nout - 1);
    mrow[t] = d.op == GM_N ? (uint32_t)j : (uint32_t)j * (uint32_t)nin;
  }
  const cplx<T>* xp = X + d.x;
  const cplx<T>* mp = M + d.m;
  v4 cr[RB][CB], ci[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) cr[i][j] = ci[i][j] = v4{0, 0, 0, 0};
  auto load = [&](int k, cplx<T>(&xv)[KS][RB], cplx<T>(&mv)[KS][CB]) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint32_t kc = (uint32_t)min(k + 4 * u + kk, nin - 1);
      const uint32_t ox = kc * bef, om = kc * mks;
#pragma unroll
      for (int t = 0; t < RB; ++t) xv[u][t] = ld32(xp, xrow[t] + ox);
#pragma unroll
      for (int t = 0; t < CB; ++t) mv[u][t] = ld32(mp, mrow[t] + om);
    }
  };
  auto kstep = [&](const cplx<T>(&xv)[RB], const cplx<T>(&mv)[CB]) {
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const T mr = mv[j].re, mi = msign * mv[j].im;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const T nxi = -xv[i].im;
        if constexpr (TR) {
          cr[i][j] = MF<T>::mma(mr, xv[i].re, cr[i][j]);
          ci[i][j] = MF<T>::mma(mr, xv[i].im, ci[i][j]);
          cr[i][j] = MF<T>::mma(mi, nxi, cr[i][j]);
          ci[i][j] = MF<T>::mma(mi, xv[i].re, ci[i][j]);
        } else {
          cr[i][j] = MF<T>::mma(xv[i].re, mr, cr[i][j]);
          ci[i][j] = MF<T>::mma(xv[i].im, mr, ci[i][j]);
          cr[i][j] = MF<T>::mma(nxi, mi, cr[i][j]);
          ci[i][j] = MF<T>::mma(xv[i].re, mi, ci[i][j]);
        }
      }
    }
  };
  auto stage = [&](int k, cplx<T>(&xv)[KS][RB], const cplx<T>(&mv)[KS][CB]) {
    if (k + 4 * KS <= nin) {
#pragma unroll
      for (int u = 0; u < KS; ++u) kstep(xv[u], mv[u]);
      return;
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (k + 4 * u >= nin) break;
      const bool kv = k + 4 * u + kk < nin;
#pragma unroll
      for (int t = 0; t < RB; ++t) xv[u][t] = mk<T>(kv ? xv[u][t].re : (T)0, kv ? xv[u][t].im : (T)0);
      kstep(xv[u], mv[u]);
    }
  };
  cplx<T> xa[KS][RB], xb[KS][RB];
  cplx<T> ma[KS][CB], mb[KS][CB];
  load(0, xa, ma);
  for (int k = 0; k < nin; k += 8 * KS) {
    load(k + 4 * KS, xb, mb);
    stage(k, xa, ma);
    load(k + 8 * KS, xa, ma);
    if (k + 4 * KS < nin) stage(k + 4 * KS, xb, mb);
  }
  cplx<T>* ob = O + d.out;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
#pragma unroll
    for (int j = 0; j < CB; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t r = r0 + (uint32_t)(i * 16 + (TR ? li : MF<T>::drow(lane, q)));
        const int col = c0 + j * 16 + (TR ? MF<T>::drow(lane, q) : li);
        if (r < R && col < nout) {
          const uint32_t a = r / bef;
          cplx<T>* o = at32(ob, (r - a * bef) + (uint32_t)col * bef + a * bef * (uint32_t)nout);
          cplx<T> v = mk<T>(cr[i][j][q], ci[i][j][q]);
          if (d.acc) v = cadd(v, *o);
          *o = v;
        }
      }
    }
  }
}

// Four tasks (wavefronts) per workgroup.  A task is 2 x 2 tiles; its last
// column block may hold one column.
template <typename T>
__global__ void __launch_bounds__(256)
    gm_block(const GmDesc* __restrict__ descs, const int32_t* __restrict__ wgdesc, int64_t ntasks,
             const cplx<T>* __restrict__ X, const cplx<T>* __restrict__ M, cplx<T>* O) {
  const int64_t task = (int64_t)blockIdx.x * 4 + wave_id();
  if (task >= ntasks) return;
  const GmDesc d = descs[wgdesc[task]];
  const uint32_t t = (uint32_t)(task - d.tile0);
  const uint32_t CT = (uint32_t)(d.nout + 31) / 32u;
  const uint32_t rt = CT == 1 ? t : t / CT;
  const int c0 = (int)(t - rt * CT) * 32;
  const uint32_t r0 = rt * 32u;
  const bool two = d.nout - c0 > 16;
  if (d.bef >= 4) {
    if (two) gm_block_tiles<T, 2, 2, 1, true>(d, r0, c0, X, M, O);
    else gm_block_tiles<T, 2, 1, 1, true>(d, r0, c0, X, M, O);
  } else {
    if (two) gm_block_tiles<T, 2, 2, 1, false>(d, r0, c0, X, M, O);
    else gm_block_tiles<T, 2, 1, 1, false>(d, r0, c0, X, M, O);
  }
}

}  // namespace

template <typename T>
int launch_gc_sum(int nt, const GcSum* tasks, int64_t ntasks, const GcSum* sums, int64_t nsums, const GcSeg* segs,
                  const void* x0, const void* x1, void* obase, void* part, hipStream_t s, const KernelTiming* kt) {
  if (ntasks <= 0) return QTG_OK;
#define QTG_GCS(NT, W)                                                                                              \
  launch_timed(gc_sum_kernel<T, NT, W>, dim3((unsigned)ntasks), dim3(64 * W), 0, s, kt, tasks, segs,                \
               (const cplx<T>*)x0, (const cplx<T>*)x1, (cplx<double>*)obase, (cplx<double>*)part);                  \
  if (nsums > 0)                                                                                                    \
    hipLaunchKernelGGL((gc_sum_add<T, NT>), dim3((unsigned)(nsums * NT * NT)), dim3(256), 0, s, sums,               \
                       (const cplx<double>*)part, (cplx<double>*)obase)
  if (nt == 1) {
    QTG_GCS(1, 8);
  } else {
    QTG_GCS(2, 4);
  }
#undef QTG_GCS
  QTG_LAUNCH_CHECK();
  return QTG_OK;
}
template int launch_gc_sum<double>(int, const GcSum*, int64_t, const GcSum*, int64_t, const GcSeg*, const void*,
                                   const void*, void*, void*, hipStream_t, const KernelTiming*);
template int launch_gc_sum<float>(int, const GcSum*, int64_t, const GcSum*, int64_t, const GcSeg*, const void*,
                                  const void*, void*, void*, hipStream_t, const KernelTiming*);

template <typename T>
int launch_gm_block(const GmDesc* descs, const int32_t* wgdesc, int64_t ntasks, const void* x, const void* m, void* o,
                    hipStream_t s) {
  if (ntasks <= 0) return QTG_OK;
  hipLaunchKernelGGL(gm_block<T>, dim3((unsigned)((ntasks + 3) / 4)), dim3(256), 0, s, descs, wgdesc, ntasks,
                     (const cplx<T>*)x, (const cplx<T>*)m, (cplx<T>*)o);
  QTG_LAUNCH_CHECK();
  return QTG_OK;
}
template int launch_gm_block<double>(const GmDesc*, const int32_t*, int64_t, const void*, const void*, void*,
                                     hipStream_t);
template int launch_gm_block<float>(const GmDesc*, const int32_t*, int64_t, const void*, const void*, void*,
                                    hipStream_t);

template <typename T>
int launch_gc_block(const GcDesc* descs, const GcBlockWg* wgs, int64_t nwg, const GcBlockWg* sums, int64_t nsums,
                    const void* x0, const void* x1, void* obase, void* part, hipStream_t s) {
  if (nwg <= 0) return QTG_OK;
  const GcDesc none{};
  hipLaunchKernelGGL((gc_block<T, 2, 4>), dim3((unsigned)nwg), dim3(256), 0, s, descs, wgs, none, 1,
                     (const cplx<T>*)x0, (const cplx<T>*)x1, (cplx<T>*)obase, (cplx<T>*)part);
  if (nsums > 0)
    hipLaunchKernelGGL(gc_block_sum<T>, dim3((unsigned)(16 * nsums)), dim3(1024), 0, s, descs, sums, none, 1,
                       (const cplx<T>*)part, (cplx<T>*)obase);
  QTG_LAUNCH_CHECK();
  return QTG_OK;
}
template int launch_gc_block<double>(const GcDesc*, const GcBlockWg*, int64_t, const GcBlockWg*, int64_t, const void*,
                                     const void*, void*, void*, hipStream_t);
template int launch_gc_block<float>(const GcDesc*, const GcBlockWg*, int64_t, const GcBlockWg*, int64_t, const void*,
                                    const void*, void*, void*, hipStream_t);

// A reduction of up to kOneWgK elements stays in one workgroup per tile, 16
// wavefronts.  A split takes two launches and the slot's event besides, 4 us
// more of the host: two products and a contraction of 552 elements (7 x 7
// complex128 output) 17.7 against 21.4 us.  In a row of contractions alone the
// split is level there (K = 520 to 750, 13-14 us either way for most shapes) and
// ahead where `bef` is a multiple of eight (24 x 24, K = 576: 21 against 14.6);
// at K = 1024 (32 x 32) it takes 14, at 2048 (64 x 64) 14.5.  Beyond the line, K
// is split over workgroups toward 512 of them (two per CU), with shares of at
// least 32 elements per wavefront (K = 4096, 64 x 64: 15 us) and the partial
// tiles within max_part_elems (0: no split over workgroups).  One wavefront per
// tile (gc_single) took 4891 us at K = 65536, 64 x 64 complex128; this takes 46,
// of which the operands' 134 MB at the card's copy rate are 28.
GcOnePlan plan_gc_one(const GcDesc& d, int64_t max_part_elems) {
  constexpr int64_t kOneWgK = 768;
  const int64_t K = (int64_t)d.bef * d.aft;
  const int64_t m2 = gc_block_macros(d);
  GcOnePlan p{};
  p.S = 1;
  if (K > kOneWgK) {
    int64_t S = std::min<int64_t>((512 + m2 - 1) / m2, K / 128);
    S = std::min<int64_t>(S, max_part_elems / (m2 * 1024));
    // workgroup macro * S + s: with 8 | S the macro tiles of a share, which
    // read the same operands, land on one XCD (blockIdx mod 8)
    if (S > 8) S &= ~(int64_t)7;
    if (S > 1) {
      p.S = (int)S;
      p.macro = m2;
      return p;
    }
  }
  p.macro = (int64_t)((d.nx + 15) / 16) * ((d.ny + 15) / 16);
  return p;
}

template <typename T>
int launch_gc_one(const GcDesc& d, const GcOnePlan& p, const void* x, const void* y, void* o, void* part,
                  hipStream_t s) {
  const cplx<T>* X = (const cplx<T>*)x;
  const cplx<T>* Y = (const cplx<T>*)y;
  if (p.S > 1 && !part) {
    set_error("single hole contraction: a split over workgroups needs its partial tiles");
    return QTG_EARG;
  }
  const GcDesc* nd = nullptr;
  const GcBlockWg* nw = nullptr;
  if (p.S == 1 && (int64_t)d.bef * d.aft <= 128) {
    // short reductions: four wavefronts, the launch itself decides
    hipLaunchKernelGGL((gc_block<T, 1, 4>), dim3((unsigned)p.macro), dim3(256), 0, s, nd, nw, d, 1, X, Y, (cplx<T>*)o,
                       (cplx<T>*)nullptr);
  } else if (p.S == 1) {
    hipLaunchKernelGGL((gc_block<T, 1, 16>), dim3((unsigned)p.macro), dim3(1024), 0, s, nd, nw, d, 1, X, Y,
                       (cplx<T>*)o, (cplx<T>*)nullptr);
  } else {
    hipLaunchKernelGGL((gc_block<T, 2, 4>), dim3((unsigned)(p.macro * p.S)), dim3(256), 0, s, nd, nw, d, p.S, X, Y,
                       (cplx<T>*)o, (cplx<T>*)part);
    hipLaunchKernelGGL(gc_block_sum<T>, dim3((unsigned)(16 * p.macro)), dim3(1024), 0, s, nd, nw, d, p.S,
                       (const cplx<T>*)part, (cplx<T>*)o);
  }
  QTG_LAUNCH_CHECK();
  return QTG_OK;
}
template int launch_gc_one<double>(const GcDesc&, const GcOnePlan&, const void*, const void*, void*, void*,
                                   hipStream_t);
template int launch_gc_one<float>(const GcDesc&, const GcOnePlan&, const void*, const void*, void*, void*,
                                  hipStream_t);

}  // namespace qtg
