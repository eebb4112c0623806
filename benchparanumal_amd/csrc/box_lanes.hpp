// Pieces that the structured-box operators (box_ax_body.hpp, box_cub.hip)
// share: the rows of a lane's pencil, the start of a CG iteration, and the
// factors of a trilinear element along a line of nodes.
#pragma once
#include <hip/hip_runtime.h>

#include "box_common.hpp"
#include "buffer_rsrc.hpp"
#include "fold.hpp"

namespace bpx {
namespace {

// 1/x by Newton steps on the hardware's (1 ulp in FP32)
__device__ inline float reciprocal(float x) {
  const float y = __builtin_amdgcn_rcpf(x);
  return fmad(fmad(-x, y, 1.0f), y, y);
}
__device__ inline double reciprocal(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fmad(fmad(-x, y, 1.0), y, y);
  return fmad(fmad(-x, y, 1.0), y, y);
}

// MODE_FOLD: the direction update of a CG iteration and the x update of the
// one before inside the Ax. Every element forms the new direction of all its
// nodes from r and the old one (neighbours form the same bits), the owner
// writes it, to another vector. An iteration is then this kernel and
// k_box_update_r: at 24^3, p = 7 FP32 76 -> 54 us against four kernels with
// k_bp5_ax, at 10^3, p = 4 affine FP64 23 -> 13 us.
enum { MODE_PLAIN = 0, MODE_DOT = 1, MODE_FOLD = 2 };

// Byte offsets of the rows of the nodes (ai, bj, k), k = 0..NQ-1, of field f
// of an element: row0 at k = 0 (owned one layer down), then row1 + (k-1)*stride;
// masked ones beyond the resource's range
template <typename T, int NQ>
__device__ inline void box_pencil_offsets(const BoxGrid& g, int F, int f, int ex, int ey, int ez, int ai, int bj,
                                          bool active, unsigned (&off)[NQ]) {
  constexpr int N = NQ - 1, S = (int)sizeof(T);
  const int ox = ex - (ai == 0), oy = ey - (bj == 0);
  const bool on = active && ox >= 0 && oy >= 0 && !(ai == N && ex == g.nx - 1) && !(bj == N && ey == g.ny - 1);
  const int Nx = BoxGrid::owned<N>(ox, g.nx), Ny = BoxGrid::owned<N>(oy, g.ny);
  const int stride = Nx * Ny;
  const int at = ((bj == 0 ? N : bj) - 1) * Nx + (ai == 0 ? N : ai) - 1;
  const int Nz = BoxGrid::owned<N>(ez, g.nz);
  const unsigned row1 = (unsigned)(g.template base<N>(F, ox, oy, ez) + f * stride * Nz + at);
  const unsigned row0 = (unsigned)(g.template base<N>(F, ox, oy, ez - 1) + (f * N + N - 1) * stride + at);
  off[0] = on && ez > 0 ? row0 * S : kBoxMasked;
#pragma unroll
  for (int k = 1; k < NQ; ++k) off[k] = on && k <= Nz ? (row1 + (k - 1) * stride) * S : kBoxMasked;
}

// MODE_FOLD: the new direction of the pencil in rq, written where the lane
// owns it, and x of the iteration before; true (uniform over the problem) if
// the iteration stops here. s_f: 33 doubles.
template <typename T, int NQ, bool BATCH>
__device__ inline bool box_direction(const BoxAxArgs<T>& a, BatchState* bs, int it, int grp, bool own,
                                     const unsigned (&off)[NQ], T (&rq)[NQ], double* s_f) {
  const int t = threadIdx.x;
  const __amdgpu_buffer_rsrc_t rr_ = box_rsrc(a.r), rp = box_rsrc(a.q), rx = box_rsrc(a.x), ro = box_rsrc(a.p);
  T pv[NQ], xv[NQ];
  const bool first = it == 0, apply = (BATCH || a.pending) && !first;
#pragma unroll
  for (int k = 0; k < NQ; ++k) rq[k] = buffer_load<T>(rr_, off[k]);
  if (!first) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) pv[k] = buffer_load<T>(rp, off[k]);
  }
  if (apply) {
#pragma unroll
    for (int k = 1; k < NQ; ++k) xv[k] = buffer_load<T>(rx, own ? off[k] : kBoxMasked);
  }
  if (t < 64) {
    const double v = wave_fold(a.part_rr, a.nrr);
    if (t == 0) s_f[32] = v;
  }
  __syncthreads();
  double rr = s_f[32], tol2;
  const double tol = BATCH ? bs->tol : a.tol;
  if (first) {
    const double nrm = sqrt(rr);  // rdotr = norm2(r)^2 (linearSolverCG.cpp:84-85)
    rr = nrm * nrm;
    tol2 = fmax(tol * tol * rr, tol * tol);
  } else {
    tol2 = BATCH ? bs->tol2 : a.st->tol2;
  }
  bool stop = !(rr > tol2) || !isfinite(rr);
  if constexpr (BATCH) {
    stop = stop || it >= bs->maxit;
    if (grp == 0 && t == 0) {
      bs->rr_k = rr;
      if (first) bs->tol2 = tol2;
      if (stop) {
        bs->rnorm = sqrt(rr);
        if (!isfinite(rr)) bs->breakdown = 1;
        bs->stop_at = it + 1;
      }
    }
  } else if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) {
    a.hist_rr[a.k] = rr;
    if (first) {
      a.st->tol2 = tol2;
      a.st->breakdown = 0;
      a.st->done = 0;
      a.st->stop_at = 0;
    }
    if (stop) {
      a.st->iter = a.k;
      if (!isfinite(rr)) a.st->breakdown = 1;
      a.st->stop_at = a.k + 1;
    }
  }
  if (apply) {
    const T al = (T)(BATCH ? bs->alpha : a.hist_alpha[it - 1]);
#pragma unroll
    for (int k = 1; k < NQ; ++k) buffer_store<T>(fmad(al, pv[k], xv[k]), rx, own ? off[k] : kBoxMasked);
  }
  if (stop) return true;
  if (!first) {
    const T beta = (T)(rr / (BATCH ? bs->rr_prev : a.hist_rr[it - 1]));
#pragma unroll
    for (int k = 0; k < NQ; ++k) rq[k] = fmad(beta, pv[k], rq[k]);
  }
#pragma unroll
  for (int k = 1; k < NQ; ++k) buffer_store<T>(rq[k], ro, own ? off[k] : kBoxMasked);
  return false;
}

// A trilinear element along the line (r, s) = const: x_r = Ar + Br t, x_s =
// As + Bs t and x_t = Ct, so the adjugate's rows J grad r = x_s x x_t = Pr +
// Qr t and J grad s = x_t x x_r = Ps + Qs t are linear in t, and J grad t =
// x_r x x_s = T0 + T1 t + T2 t^2 and J = x_t . (J grad t) are quadratic.
template <typename T>
struct TrilinearLine {
  T Pr[3], Qr[3], Ps[3], Qs[3], T0[3], T1[3], T2[3], jt[3];

  // ce: the element's 24 map coefficients; formed in C and then rounded
  template <typename C, typename P>
  __device__ inline void set(P ce, C r, C sn) {
    C Ar[3], Br[3], As[3], Bs[3], Ct[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const C c_r = ce[8 * d + 0], c_s = ce[8 * d + 1], c_t = ce[8 * d + 2], c_rs = ce[8 * d + 3];
      const C c_rt = ce[8 * d + 4], c_st = ce[8 * d + 5], c_rst = ce[8 * d + 6];
      Ar[d] = fmad(c_rs, sn, c_r);
      Br[d] = fmad(c_rst, sn, c_rt);
      As[d] = fmad(c_rs, r, c_s);
      Bs[d] = fmad(c_rst, r, c_st);
      Ct[d] = fmad(Br[d], r, fmad(c_st, sn, c_t));
      if constexpr (sizeof(C) != sizeof(T)) __builtin_amdgcn_sched_barrier(0);
    }
    auto cross = [](const C* u, const C* v, int d) {
      const int d1 = (d + 1) % 3, d2 = (d + 2) % 3;
      return fmad(u[d1], v[d2], -(u[d2] * v[d1]));
    };
    C j0 = 0, j1 = 0, j2 = 0;
#pragma unroll
    for (int d = 2; d >= 0; --d) {
      Pr[d] = (T)cross(As, Ct, d);
      Qr[d] = (T)cross(Bs, Ct, d);
      Ps[d] = (T)cross(Ct, Ar, d);
      Qs[d] = (T)cross(Ct, Br, d);
      const C t0 = cross(Ar, As, d), t1 = cross(Ar, Bs, d) + cross(Br, As, d), t2 = cross(Br, Bs, d);
      T0[d] = (T)t0;
      T1[d] = (T)t1;
      T2[d] = (T)t2;
      j0 = d == 2 ? Ct[d] * t0 : fmad(Ct[d], t0, j0);
      j1 = d == 2 ? Ct[d] * t1 : fmad(Ct[d], t1, j1);
      j2 = d == 2 ? Ct[d] * t2 : fmad(Ct[d], t2, j2);
    }
    jt[0] = (T)j0;
    jt[1] = (T)j1;
    jt[2] = (T)j2;
  }

  // before each node of the line: without it the compiler forms every node's
  // values before the first is used and spills
  __device__ inline void pin() {
#pragma unroll
    for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(Pr[d]), "+v"(Ps[d]), "+v"(T0[d]), "+v"(jt[d]));
  }

  __device__ inline T jacobian(T tk) const { return fmad(fmad(jt[2], tk, jt[1]), tk, jt[0]); }

  // (Gr, Gs, Gt) = w J G (qr, qs, qt) and W = w J at t, as adj (w/J) adj^T
  // applied to the gradient, G itself not formed
  template <bool KAPPA>
  __device__ inline void flux(T tk, T w, T kap, T qr, T qs, T qt, T& Gr, T& Gs, T& Gt, T& W) const {
    T ar[3], as[3], av[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      ar[d] = fmad(Qr[d], tk, Pr[d]);
      as[d] = fmad(Qs[d], tk, Ps[d]);
      av[d] = fmad(fmad(T2[d], tk, T1[d]), tk, T0[d]);
    }
    const T J = jacobian(tk);
    T sc = w * reciprocal(J);
    W = J * w;
    if constexpr (KAPPA) sc *= kap;
    T gx[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) gx[d] = sc * fmad(av[d], qt, fmad(as[d], qs, ar[d] * qr));
    Gr = fmad(ar[2], gx[2], fmad(ar[1], gx[1], ar[0] * gx[0]));
    Gs = fmad(as[2], gx[2], fmad(as[1], gx[1], as[0] * gx[0]));
    Gt = fmad(av[2], gx[2], fmad(av[1], gx[1], av[0] * gx[0]));
  }
};

}  // namespace
}  // namespace bpx
