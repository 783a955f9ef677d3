// Register-blocked complex contractions for many or large tiles: the forms
// of the grouped mode product and hole contraction whose launch fills the
// card, where operand traffic and not latency decides.
//
// gc_block (hole contraction): a workgroup owns a macro tile of up to
// NT x NT output tiles of 16 x 16; every wavefront holds all of it in
// registers and walks its own share of the reduction, so each element of the
// bra and the ket is loaded once per macro tile, and the shares are summed in
// LDS in wavefront order.  One wavefront per 16 x 16 tile (gc_grouped) reads
// each operand once per tile of the other index, from workgroups that the
// dispatcher spreads over XCDs with L2s of their own.  S > 1 splits a
// reduction over S workgroups as well; their partial tiles are summed in
// order by gc_block_sum.
//
// Descriptors pass gc_lean_ok (32-bit offsets, see gemm_ops.hip).
#include <algorithm>

#include "gemm_dev.hpp"
#include "gemm_ops.hpp"

namespace qtg {

namespace {

// --------------------------------------------------------- hole contraction
// This wavefront's share [kbeg, kend) of the macro tile (nrb x ncb tiles at
// columns j0 of the bra, l0 of the ket), KS k-steps of four per stage, the
// next stage's operands in flight behind the current MFMAs (4 per tile and
// k-step, 64 cycles each in FP64).  Columns past the tensor are clamped into
// it (never stored); k past the share reads in range and counts zero.
template <typename T, int NT, int KS>
__device__ inline void gc_block_product(const GcDesc& d, int j0, int l0, int nrb, int ncb, int kbeg, int kend,
                                        const cplx<T>* __restrict__ X, const cplx<T>* __restrict__ Y,
                                        typename MF<T>::v4 (&cr)[NT][NT], typename MF<T>::v4 (&ci)[NT][NT]) {
  const int lane = threadIdx.x & 63, li = lane & 15, kk = lane >> 4;
  const uint32_t bef = (uint32_t)d.bef, aft = (uint32_t)d.aft;
  const uint32_t xs = bef * (uint32_t)d.nx, ys = bef * (uint32_t)d.ny;  // stride of a
  const uint32_t xmax = (bef - 1u) + (aft - 1u) * xs, ymax = (bef - 1u) + (aft - 1u) * ys;
  uint32_t xrow[NT], yrow[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    xrow[t] = (uint32_t)min(j0 + t * 16 + li, d.nx - 1) * bef;
    yrow[t] = (uint32_t)min(l0 + t * 16 + li, d.ny - 1) * bef;
  }
  const cplx<T>* xp = X + d.x;
  const cplx<T>* yp = Y + d.y;
  int kc = kbeg + kk;
  uint32_t b = (uint32_t)kc % bef;
  const uint32_t a0 = (uint32_t)kc / bef;
  uint32_t px = b + a0 * xs, py = b + a0 * ys;
  const uint32_t q4 = 4u / bef, r4 = 4u % bef;
  const uint32_t dx = r4 + q4 * xs, dy = r4 + q4 * ys;
  auto load = [&](cplx<T>(&xv)[KS][NT], cplx<T>(&yv)[KS][NT]) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const bool kv = kc < kend;
      const uint32_t ox = min(px, xmax), oy = min(py, ymax);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (t < nrb) {
          const cplx<T> x = ld32(xp, xrow[t] + ox);
          xv[u][t] = mk<T>(kv ? x.re : (T)0, kv ? x.im : (T)0);
        }
        if (t < ncb) {
          const cplx<T> y = ld32(yp, yrow[t] + oy);
          yv[u][t] = mk<T>(kv ? y.re : (T)0, kv ? y.im : (T)0);
        }
      }
      kc += 4;
      b += r4;
      px += dx;
      py += dy;
      if (b >= bef) {
        b -= bef;
        px += xs - bef;
        py += ys - bef;
      }
    }
  };
  // the k-steps of a stage that starts at k0
  auto steps = [&](int k0, const cplx<T>(&xv)[KS][NT], const cplx<T>(&yv)[KS][NT]) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (u > 0 && k0 + 4 * u >= kend) break;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (i >= nrb) break;
        const T nxi = -xv[u][i].im;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (j >= ncb) break;
          cr[i][j] = MF<T>::mma(xv[u][i].re, yv[u][j].re, cr[i][j]);
          ci[i][j] = MF<T>::mma(xv[u][i].re, yv[u][j].im, ci[i][j]);
          cr[i][j] = MF<T>::mma(xv[u][i].im, yv[u][j].im, cr[i][j]);
          ci[i][j] = MF<T>::mma(nxi, yv[u][j].re, ci[i][j]);
        }
      }
    }
  };
  if (kbeg >= kend) return;
  cplx<T> xa[KS][NT], ya[KS][NT], xb[KS][NT], yb[KS][NT];
  load(xa, ya);
  for (int k = kbeg; k < kend; k += 8 * KS) {
    const bool second = k + 4 * KS < kend;
    if (second) load(xb, yb);
    steps(k, xa, ya);
    if (!second) break;
    if (k + 8 * KS < kend) load(xa, ya);
    steps(k + 4 * KS, xb, yb);
  }
}

// W wavefronts per workgroup; S workgroups per macro tile.  descs null: the
// one descriptor `one`.  Otherwise wgdesc[blockIdx.x] names the workgroup's
// descriptor and tile0 its first workgroup (S = 1).
template <typename T, typename TO, int NT, int W>
__global__ void __launch_bounds__(64 * W)
    gc_block(const GcDesc* __restrict__ descs, const int32_t* __restrict__ wgdesc, GcDesc one, int S,
             const cplx<T>* __restrict__ X0, const cplx<T>* __restrict__ X1, cplx<TO>* O, cplx<TO>* part) {
  constexpr int NB = NT > 1 ? 2 : 1;  // LDS buffers: one barrier per tile
  __shared__ cplx<TO> red[NB * W * 256];
  typedef typename MF<T>::v4 v4;
  const GcDesc d = descs ? descs[wgdesc[blockIdx.x]] : one;
  unsigned t = blockIdx.x - (descs ? (unsigned)d.tile0 : 0u);
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
  gc_block_product<T, NT, (NT == 1 ? 4 : NT == 2 ? 2 : 1)>(d, j0, l0, nrb, ncb, kbeg, kend, xbase, ybase, cr, ci);
  const int TJ = (d.nx + 15) >> 4;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    if (i >= nrb) break;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (j >= ncb) break;
      cplx<TO>* buf = red + (NB > 1 ? ((i * NT + j) & 1) * W * 256 : 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) buf[wave * 256 + q * 64 + lane] = mk<TO>((TO)cr[i][j][q], (TO)ci[i][j][q]);
      __syncthreads();
      if (threadIdx.x < 256) {
        const int e = threadIdx.x, el = e & 63, q = e >> 6;
        cplx<TO> v = buf[e];
#pragma unroll
        for (int w = 1; w < W; ++w) v = cadd(v, buf[w * 256 + e]);
        const int row = j0 + i * 16 + MF<T>::drow(el, q), col = l0 + j * 16 + (el & 15);
        if (part) {
          const int64_t tile = (int64_t)((l0 >> 4) + j) * TJ + (j0 >> 4) + i;
          part[(tile * S + s) * 256 + e] = v;
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

// Sums the S partial tiles of every 16 x 16 output tile.  Four workgroups a
// tile, 64 elements each; a wavefront adds a sixteenth of the partials in
// order, then the first adds the wavefronts' sums.
template <typename T>
__global__ void __launch_bounds__(1024)
    gc_block_sum(GcDesc d, int S, const cplx<T>* __restrict__ part, cplx<T>* O) {
  __shared__ cplx<T> red[15 * 64];
  const int TJ = (d.nx + 15) >> 4;
  const unsigned tile = blockIdx.x >> 2;
  const int lt = (int)(tile / (unsigned)TJ), jt = (int)(tile - (unsigned)lt * TJ);
  const int lane = threadIdx.x & 63, e = (int)(blockIdx.x & 3) * 64 + lane, g = wave_id();
  const int per = (S + 15) >> 4, s0 = min(S, g * per), s1 = min(S, s0 + per);
  const cplx<T>* p = part + (int64_t)tile * S * 256 + e;
  cplx<T> v = czero<T>();
#pragma unroll 8
  for (int s = s0; s < s1; ++s) v = cadd(v, p[(int64_t)s * 256]);
  if (g > 0) red[(g - 1) * 64 + lane] = v;
  __syncthreads();
  if (g > 0) return;
#pragma unroll
  for (int k = 0; k < 15; ++k) v = cadd(v, red[k * 64 + lane]);
  const int row = jt * 16 + MF<T>::drow(lane, e >> 6), col = lt * 16 + (lane & 15);
  if (row < d.nx && col < d.ny) {
    const int64_t o = d.out + row + (int64_t)col * d.nx;
    if (d.acc) v = cadd(v, O[o]);
    O[o] = v;
  }
}

}  // namespace

// A reduction of up to kOneWgK elements stays in one workgroup per tile: its
// 16 wavefronts take 14 us at K = 576 (24 x 24 output), where two launches
// take at least 14; at K = 1024 (32 x 32) 18 against 17 us, at 2048 (64 x 64)
// 32 against 18.  Beyond it, K is split over workgroups toward 512 of them
// (two per CU), with shares of at least 32 elements per wavefront (K = 4096,
// 64 x 64: 18 us; shares of 64: 27) and the partial tiles within
// max_part_elems (0: no split over workgroups).  One wavefront per tile
// (gc_single) took 4891 us at K = 65536, 64 x 64 complex128; this takes 80,
// of which the operands' 134 MB at the card's copy rate are 28.
GcOnePlan plan_gc_one(const GcDesc& d, int64_t max_part_elems) {
  constexpr int64_t kOneWgK = 768;
  const int64_t K = (int64_t)d.bef * d.aft;
  GcOnePlan p{};
  p.tiles = (int64_t)((d.nx + 15) / 16) * ((d.ny + 15) / 16);
  p.S = 1;
  const int64_t m2 = (int64_t)((d.nx + 31) / 32) * ((d.ny + 31) / 32);
  if (K > kOneWgK) {
    int64_t S = std::min<int64_t>((512 + m2 - 1) / m2, K / 128);
    S = std::min<int64_t>(S, max_part_elems / (p.tiles * 256));
    if (S > 1) {
      p.nt = 2;
      p.S = (int)S;
      p.macro = m2;
      return p;
    }
  }
  p.nt = 1;
  p.macro = p.tiles;
  return p;
}

template <typename T>
int launch_gc_one(const GcDesc& d, const GcOnePlan& p, const void* x, const void* y, void* o, void* part,
                  hipStream_t s) {
  const cplx<T>* X = (const cplx<T>*)x;
  const cplx<T>* Y = (const cplx<T>*)y;
  if (p.nt == 1) {
    hipLaunchKernelGGL((gc_block<T, T, 1, 16>), dim3((unsigned)p.macro), dim3(1024), 0, s, (const GcDesc*)nullptr,
                       (const int32_t*)nullptr, d, 1, X, Y, (cplx<T>*)o, (cplx<T>*)nullptr);
  } else {
    const bool split = p.S > 1;
    if (split && !part) {
      set_error("single hole contraction: a split over workgroups needs its partial tiles");
      return QTG_EARG;
    }
    hipLaunchKernelGGL((gc_block<T, T, 2, 4>), dim3((unsigned)(p.macro * p.S)), dim3(256), 0, s,
                       (const GcDesc*)nullptr, (const int32_t*)nullptr, d, p.S, X, Y, (cplx<T>*)o,
                       split ? (cplx<T>*)part : (cplx<T>*)nullptr);
    if (split)
      hipLaunchKernelGGL(gc_block_sum<T>, dim3((unsigned)(4 * p.tiles)), dim3(1024), 0, s, d, p.S, (const cplx<T>*)part,
                         (cplx<T>*)o);
  }
  QTG_LAUNCH_CHECK();
  return QTG_OK;
}
template int launch_gc_one<double>(const GcDesc&, const GcOnePlan&, const void*, const void*, void*, void*,
                                   hipStream_t);
template int launch_gc_one<float>(const GcDesc&, const GcOnePlan&, const void*, const void*, void*, void*,
                                  hipStream_t);

}  // namespace qtg
