// Batched FP64 small-matrix kernels (smallmat.hip).
#pragma once
#include <cstdint>

#include "common.hpp"

namespace qtg {

// One matrix of a batch: input at a, output at q (complex-element offsets
// from the launch's base pointers), eigenvalues at e (heev), shape m x n
// (square ops use n).
struct SmItem {
  int64_t a, q, e, m;
  int32_t n, pad;
};

// Every launcher takes either a device item array (items) or, with items
// null, a uniform batch: item b is u with a, q, e advanced by b times st's.
// heev (U, ev; either may be null) and/or the regularised inverse R (eps)
int launch_heev_batch(const SmItem* items, const SmItem& u, const SmItem& st, int64_t count, int nmax,
                      const void* in, void* U, double* ev, void* R, double eps, hipStream_t s);
int launch_inverse_batch(const SmItem* items, const SmItem& u, const SmItem& st, int64_t count, int nmax,
                         const void* in, void* out, hipStream_t s);
// thin Q of every (m x n) item, n <= 64, m >= n, none larger than mmax x
// nmax; in and out may alias.  With R non-null, an item with e >= 0 also
// writes its n x n upper triangular R (A = Q R) at R + e.  positive: the Q
// whose R has a positive diagonal (R itself is not adjusted), for matrices
// that qr_in_registers.
int launch_qr_batch(const SmItem* items, const SmItem& u, const SmItem& st, int64_t count, int64_t mmax, int nmax,
                    const void* in, void* out, hipStream_t s, void* R = nullptr, bool positive = false);
// thin Q of one matrix by the kernel of the larger matrices, whatever its
// size: for matrices of nearly dependent columns whose Q, the rounding's own
// choice in the directions they leave open, is to stay what it is
int launch_qr_in_place(const SmItem& u, const void* in, void* out, hipStream_t s);
inline bool qr_in_registers(int64_t m, int n) {
  return m <= 256 || (m <= 576 && n <= 24);
}

}  // namespace qtg
