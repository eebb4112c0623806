// One-dimensional operators along a line that a lane holds in registers, the
// matrix uniform over the wavefront (device code).
#pragma once
#include <hip/hip_runtime.h>

#include "fold.hpp"

namespace bpx {
namespace {

// rows of a uniform R x C row-major matrix through scalar registers, row
// n + 1 requested while row n is in use: body(n, row) for n = 0..R-1. The
// opaque update of the pointer before each row keeps the compiler from
// holding the whole matrix in scalar registers.
template <int R, int C, typename T, typename F>
__device__ inline void uniform_rows(const T* M, F&& body) {
  typedef const __attribute__((address_space(4))) T* cptr;
  cptr Mc = (cptr)M;
  T d[2][C];
  asm volatile("" : "+s"(Mc));
#pragma unroll
  for (int m = 0; m < C; ++m) d[0][m] = Mc[m];
#pragma unroll
  for (int n = 0; n < R; ++n) {
    if (n + 1 < R) {
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" : "+s"(Mc));
#pragma unroll
      for (int m = 0; m < C; ++m) d[(n + 1) & 1][m] = Mc[(n + 1) * C + m];
    }
    body(n, d[n & 1]);
  }
}

// Even-odd form of y = A x for a 1D operator A (N x M) with A[N-1-n][M-1-m]
// = SIGN * A[n][m] (the interpolation matrix between symmetric point sets
// and its transpose: SIGN = 1; the derivative on symmetric points and its
// transpose: SIGN = -1). With xe[m] = x[m] + x[M-1-m], xo[m] = x[m] -
// x[M-1-m] (m < M/2) and Ae = (A[n][m] + A[n][M-1-m]) / 2, Ao = (A[n][m] -
// A[n][M-1-m]) / 2: ye[n] = Ae xe (+ A[n][M/2] x[M/2] for odd M), yo[n] =
// Ao xo, y[n] = ye + yo and y[N-1-n] = SIGN (ye - yo), which halves the
// multiply-adds (Kopriva's even-odd decomposition). Table row n (n <=
// (N-1)/2): Ae[n][0..M/2-1], A[n][M/2] (odd M), Ao[n][0..M/2-1]; in the
// middle row of an odd N only the part that does not vanish is used.
template <int N, int M>
struct EoShape {
  static constexpr int hM = M / 2, oM = M & 1, LE = hM + oM, RL = LE + hM;
  static constexpr int hN = N / 2, oN = N & 1, rows = hN + oN, size = rows * RL;
};

template <int N, int M, int SIGN, typename T, typename P>
__device__ inline void eo_apply(const T* tab, const T (&x)[M], P&& put) {  // put(n, y[n])
  using E = EoShape<N, M>;
  T xe[E::hM > 0 ? E::hM : 1], xo[E::hM > 0 ? E::hM : 1];
#pragma unroll
  for (int m = 0; m < E::hM; ++m) {
    xe[m] = x[m] + x[M - 1 - m];
    xo[m] = x[m] - x[M - 1 - m];
  }
  uniform_rows<E::rows, E::RL>(tab, [&](int n, const T* r) {
    const bool mid = E::oN && n == E::hN;
    T ye = 0, yo = 0;
    if (!mid || SIGN > 0) {
#pragma unroll
      for (int m = 0; m < E::hM; ++m) ye = fmad(r[m], xe[m], ye);
      if constexpr (E::oM) ye = fmad(r[E::hM], x[E::hM], ye);
    }
    if (!mid || SIGN < 0) {
#pragma unroll
      for (int m = 0; m < E::hM; ++m) yo = fmad(r[E::LE + m], xo[m], yo);
    }
    if (mid) {
      put(n, SIGN > 0 ? ye : yo);
    } else {
      put(n, ye + yo);
      put(N - 1 - n, SIGN > 0 ? ye - yo : yo - ye);
    }
  });
}

// offsets of the four tables in the kernel's even-odd array: I (MQ x NQ),
// I^T, D (MQ x MQ, the cubature derivative) and D^T; then D by rows
template <int NQ>
struct EoTables {
  static constexpr int MQ = NQ + 1;
  static constexpr int I = 0, IT = I + EoShape<MQ, NQ>::size, D = IT + EoShape<NQ, MQ>::size,
                       DT = D + EoShape<MQ, MQ>::size, ROWS = DT + EoShape<MQ, MQ>::size;
};

}  // namespace
}  // namespace bpx
