// Device helpers shared by the MFMA contraction kernels (gemm_ops.hip,
// gemm_block.hip): the 16x16x4 complex k-step, wave-uniform indices and
// 32-bit addressing from a uniform base.
#pragma once
#include <hip/hip_ext.h>

#include "gemm_ops.hpp"

namespace qtg {

// Launches k; with kt set, through hipExtLaunchKernelGGL so that kt's events
// carry the kernel's own start and stop times (no marker packets around it).
template <typename K, typename... A>
void launch_timed(K k, dim3 grid, dim3 block, unsigned lds, hipStream_t s, const KernelTiming* kt, A... a) {
  if (kt) hipExtLaunchKernelGGL(k, grid, block, lds, s, kt->start, kt->stop, 0, a...);
  else hipLaunchKernelGGL(k, grid, block, lds, s, a...);
}

template <typename T>
struct MF;
template <>
struct MF<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ inline int drow(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct MF<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ inline int drow(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// (cr, ci) += a * b on one complex k-step (a is already conjugated if needed)
template <typename T>
__device__ inline void cmma(typename MF<T>::v4& cr, typename MF<T>::v4& ci, const cplx<T>& a, const cplx<T>& b) {
  cr = MF<T>::mma(a.re, b.re, cr);
  cr = MF<T>::mma(-a.im, b.im, cr);
  ci = MF<T>::mma(a.re, b.im, ci);
  ci = MF<T>::mma(a.im, b.re, ci);
}

// Wavefront index in the workgroup, as a wave-uniform (scalar) value, so that
// descriptor loads and address arithmetic stay on the scalar unit.
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// base[off] when ok, else zero.  The load itself is unconditional, from
// base[0] when !ok (base is the start of an operand, always in bounds): a
// guarded load would let the compiler select between the operand and a stack
// zero and fall back to generic (flat) loads.
template <typename T>
__device__ inline cplx<T> ldz(const cplx<T>* __restrict__ base, int64_t off, bool ok) {
  const cplx<T> v = base[ok ? off : 0];
  return ok ? v : czero<T>();
}

// base[idx] for idx < 2^27: a 32-bit byte offset from the base
template <typename V>
__device__ inline V ld32(const V* base, uint32_t idx) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + (idx * (uint32_t)sizeof(V)));
}
template <typename V>
__device__ inline V* at32(V* base, uint32_t idx) {
  return reinterpret_cast<V*>(reinterpret_cast<char*>(base) + (idx * (uint32_t)sizeof(V)));
}

}  // namespace qtg
