// Shared device/host helpers of the gfx950 engine: complex arithmetic on
// interleaved (re, im) pairs, status handling and launch checks.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/qutree_amd.h"

namespace qtg {

template <typename T>
struct alignas(2 * sizeof(T)) cplx {
  T re, im;
};

template <typename T>
__host__ __device__ inline cplx<T> mk(T r, T i) {
  cplx<T> c;
  c.re = r;
  c.im = i;
  return c;
}
template <typename T>
__host__ __device__ inline cplx<T> czero() {
  return mk<T>(T(0), T(0));
}
// acc += a * b
template <typename T>
__device__ inline void cfma(cplx<T>& acc, const cplx<T>& a, const cplx<T>& b) {
  acc.re = fma(a.re, b.re, acc.re);
  acc.re = fma(-a.im, b.im, acc.re);
  acc.im = fma(a.re, b.im, acc.im);
  acc.im = fma(a.im, b.re, acc.im);
}
// acc += conj(a) * b
template <typename T>
__device__ inline void cfmac(cplx<T>& acc, const cplx<T>& a, const cplx<T>& b) {
  acc.re = fma(a.re, b.re, acc.re);
  acc.re = fma(a.im, b.im, acc.re);
  acc.im = fma(a.re, b.im, acc.im);
  acc.im = fma(-a.im, b.re, acc.im);
}
template <typename T>
__host__ __device__ inline cplx<T> cmul(const cplx<T>& a, const cplx<T>& b) {
  return mk<T>(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
template <typename T>
__host__ __device__ inline cplx<T> cadd(const cplx<T>& a, const cplx<T>& b) {
  return mk<T>(a.re + b.re, a.im + b.im);
}
template <typename T>
__host__ __device__ inline cplx<T> cconj(const cplx<T>& a) {
  return mk<T>(a.re, -a.im);
}

// Sum over the 64 lanes, the same value in every lane, on the vector ALU
// alone: neighbours, quads, half rows and rows by lane permutations within a
// row of 16, then the row totals broadcast upward (row_bcast 15 and 31) and
// lane 63 read.  Six cross-lane steps through LDS (__shfl) take about five
// times as long, which is most of a serial chain of reductions.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
__device__ inline double wave_total(double v) {
  v = dpp_add<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v = dpp_add<0x141, 0xf>(v);  // row_half_mirror
  v = dpp_add<0x140, 0xf>(v);  // row_mirror: every lane its row's total
  v = dpp_add<0x142, 0xa>(v);  // row_bcast15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast31 into rows 2 and 3
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// The same sum in the order of a butterfly over lane distances 32, 16, ... 1,
// to the bit what v += __shfl_xor(v, 32), ... gives in every lane and
// __shfl_down in lane 0, without the LDS: halves and rows exchanged by
// permlane swaps, then rotations by 8 and by 4 within a row (whose values
// repeat every 8 lanes by then, so lane i - 4 holds what lane i ^ 4 does) and
// quad permutations.
__device__ inline double swap_add32(double v) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double swap_add16(double v) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double wave_butterfly(double v) {
  v = swap_add16(swap_add32(v));
  v = dpp_add<0x128, 0xf>(v);   // row_ror:8
  v = dpp_add<0x124, 0xf>(v);   // row_ror:4
  v = dpp_add<0x4E, 0xf>(v);    // quad_perm [2,3,0,1]
  return dpp_add<0xB1, 0xf>(v);  // quad_perm [1,0,3,2]
}

// per-thread last error of the C ABI
void set_error(const std::string& msg);
const char* get_error();

#define QTG_HIP_TRY(expr)                                                                  \
  do {                                                                                     \
    hipError_t _e = (expr);                                                                \
    if (_e != hipSuccess) {                                                                \
      ::qtg::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));                 \
      return QTG_EDEVICE;                                                                  \
    }                                                                                      \
  } while (0)

#define QTG_LAUNCH_CHECK()                                                                 \
  do {                                                                                     \
    hipError_t _e = hipGetLastError();                                                     \
    if (_e != hipSuccess) {                                                                \
      ::qtg::set_error(std::string("kernel launch: ") + hipGetErrorString(_e));            \
      return QTG_EDEVICE;                                                                  \
    }                                                                                      \
  } while (0)

inline hipStream_t S(qtg_stream s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace qtg
