// BP5 / BP6 Ax on the structured hex box, FP64 and FP32: the operator of
// okl/bp5AxHex3D.okl:415-569 (and bp6AxHex3D.okl) with the geometry formed
// in the kernel and the rows of box.hpp in place of GlobalToLocal.
//
// What it leaves out of memory. The box's elements are trilinear maps of
// their 8 vertices, so the 7 factors of a node (56 bytes in FP64, 340 of the
// 518 MB that the stored-factor kernel moves at 24^3, p = 7) follow from 24
// numbers per element, and the row of a node from its place in the box. A
// node then costs its q (read), its result (written) and nothing else:
// 94 MB. The factors are the exact derivatives of the map; the stored ones
// are derivatives by D, whose rounding the operator magnifies (relative
// error against exact arithmetic at 24^3, p = 7: 8e-14 stored, 2e-15 here).
// Measured there, FP64: Ax 97 -> 38 us, operator 127 -> 55 us; BP6 (three
// fields, the geometry formed for each) 255 -> 166 us. Of the 38 us the vector
// ALU issues for 21 and LDS for 9; 103 MB move.
//
// Layout (the pencil form of ax_bp5.hip): a lane owns the nodes (k, b, a),
// k = 0..Nq-1, of its element; one-dimensional contractions run along a
// pencil that one lane holds, with the matrix uniform over the wavefront,
// and values move between directions through two LDS buffers, 16 accesses
// per node (the sheet form reads 4 Nq). D is antisymmetric about the middle
// of the GLL points in both indices, so each contraction works on the even
// and odd parts of its pencil: Nq^2/2 + 2 Nq operations in place of Nq^2,
// and D and its transpose share one table of Nq^2/2 values.
//
// At Nq = 8 an element is one wavefront, whose LDS traffic needs no
// workgroup barrier (a wavefront's LDS operations execute in order).
#pragma once
#include <hip/hip_runtime.h>

#include "box_lanes.hpp"

namespace bpx {
namespace {

// y = D x (or D^T x) from the even-odd table: row n <= (NQ-1)/2 holds
// S[n][m] = (D[n][m] + D[n][NQ-1-m])/2 for m < NQ/2, D[n][NQ/2] for odd NQ,
// A[n][m] = (D[n][m] - D[n][NQ-1-m])/2 for m < NQ/2. Rows come through
// scalar loads. Up to Nq = 8 the table (64 scalar registers in FP64) may
// stay in registers; beyond, each row is requested where it is used.
//
// BY_ROWS: D itself, which follows the table, in sums of Nq terms in order.
template <typename T, int NQ, bool BY_ROWS>
struct EvenOdd {
  static constexpr int H = NQ / 2, ODD = NQ & 1, ROWS = H + ODD;
  typedef const __attribute__((address_space(4))) T* cptr;
  static constexpr bool HOLD = NQ <= 8;

  template <typename F>
  __device__ static inline void rows(cptr tab, F&& body) {
    if constexpr (HOLD) {
#pragma unroll
      for (int n = 0; n < ROWS; ++n) {
        T r[NQ];
#pragma unroll
        for (int m = 0; m < NQ; ++m) r[m] = tab[n * NQ + m];
        body(n, r);
      }
    } else {  // row n + 1 on its way while row n is in use
      T r[2][NQ];
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" : "+s"(tab));
#pragma unroll
      for (int m = 0; m < NQ; ++m) r[0][m] = tab[m];
#pragma unroll
      for (int n = 0; n < ROWS; ++n) {
        if (n + 1 < ROWS) {
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" : "+s"(tab));
#pragma unroll
          for (int m = 0; m < NQ; ++m) r[(n + 1) & 1][m] = tab[(n + 1) * NQ + m];
        }
        body(n, r[n & 1]);
      }
    }
  }

  __device__ static inline void apply(cptr tab, const T (&x)[NQ], T (&y)[NQ]) {
    if constexpr (BY_ROWS) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        T a = 0;
#pragma unroll
        for (int m = 0; m < NQ; ++m) a = fmad(tab[(ROWS + n) * NQ + m], x[m], a);
        y[n] = a;
      }
      return;
    }
    T xe[H], xo[H];
#pragma unroll
    for (int m = 0; m < H; ++m) {
      xe[m] = x[m] + x[NQ - 1 - m];
      xo[m] = x[m] - x[NQ - 1 - m];
    }
    const T xm = x[H];  // the middle value (odd NQ)
    rows(tab, [&](int n, const T* r) {
      T ye = 0, yo = 0;
#pragma unroll
      for (int m = 0; m < H; ++m) {
        ye = fmad(r[H + ODD + m], xo[m], ye);
        if (n < H) yo = fmad(r[m], xe[m], yo);
      }
      if (n == H) {
        y[n] = ye;
      } else {
        if constexpr (ODD) yo = fmad(r[H], xm, yo);
        y[n] = ye + yo;
        y[NQ - 1 - n] = ye - yo;
      }
    });
  }

  __device__ static inline void apply_transposed(cptr tab, const T (&x)[NQ], T (&y)[NQ]) {
    if constexpr (BY_ROWS) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) y[n] = T(0);
#pragma unroll
      for (int m = 0; m < NQ; ++m)
#pragma unroll
        for (int n = 0; n < NQ; ++n) y[n] = fmad(tab[(ROWS + m) * NQ + n], x[m], y[n]);
      return;
    }
    T ye[H], yo[H], ym = 0;
#pragma unroll
    for (int n = 0; n < H; ++n) ye[n] = yo[n] = T(0);
    rows(tab, [&](int m, const T* r) {
      if (m < H) {
        const T xe = x[m] + x[NQ - 1 - m], xo = x[m] - x[NQ - 1 - m];
#pragma unroll
        for (int n = 0; n < H; ++n) {
          ye[n] = fmad(r[n], xo, ye[n]);
          yo[n] = fmad(r[H + ODD + n], xe, yo[n]);
        }
        if constexpr (ODD) ym = fmad(r[H], xo, ym);
      } else {  // the middle row: D[mid][n], antisymmetric in n
#pragma unroll
        for (int n = 0; n < H; ++n) yo[n] = fmad(r[H + ODD + n], x[H], yo[n]);
      }
    });
#pragma unroll
    for (int n = 0; n < H; ++n) {
      y[n] = ye[n] + yo[n];
      y[NQ - 1 - n] = ye[n] - yo[n];
    }
    if constexpr (ODD) y[H] = ym;
  }
};

// occupancy handed to the register allocator: what the pencils, the map's
// 25 constants and the temporaries fit without spilling
template <typename T, int NQ>
constexpr int box_waves() {
  return sizeof(T) == 4 ? (NQ <= 8 ? 7 : NQ <= 12 ? 5 : 4) : (NQ <= 8 ? 4 : NQ <= 12 ? 3 : 2);
}

template <int NQ>
__device__ inline void element_sync() {
  if constexpr (NQ == 8) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    asm volatile("" ::: "memory");
  } else {
    __syncthreads();
  }
  __builtin_amdgcn_sched_barrier(0);
}

// GEO: where the factors come from
enum { GEO_TRILINEAR = 0, GEO_AFFINE = 1, GEO_STORED = 2 };

// D by rows where the even-odd parts cost bits: up to Nq = 6 they take a
// tenth off the operations, but rounded to FP32 they leave the operator up to
// 20% (Nq = 6, affine) farther from exact arithmetic than rows do, from Nq = 7
// on 5 to 25% closer. In FP64, where the formed factors are far closer than
// the stored ones, only affine elements (whose factors are the stored ones)
// show it, 6% at Nq = 6.
template <typename T, int NQ, int GEO>
constexpr bool box_by_rows() {
  return sizeof(T) == 4 ? NQ <= 6 : GEO == GEO_AFFINE && NQ == 6;
}

// LDS of one workgroup: the two pencil buffers and the sums
template <typename T, int NQ, int MODE>
struct BoxAxLds {
  static constexpr int LE = NQ * (NQ * NQ + 8);  // an element's pencils
  T b[box_epb(NQ) * LE];                         // pencils along i
  T c[box_epb(NQ) * LE];                         // pencils along j
  // sums; f[32] hands the folded r.r out
  double f[MODE == MODE_PLAIN ? 1 : NQ * NQ * box_epb(NQ)];
};

template <typename T, int NQ, int GEO, bool KAPPA, int MODE, bool BATCH>
__device__ inline void box_ax_body(BoxAxArgs<T> a, int per_xcd, BoxAxLds<T, NQ, MODE>& lds) {
  constexpr int N = NQ - 1, NQ2 = NQ * NQ, NP = NQ2 * NQ, EPB = box_epb(NQ);
  constexpr int LK = NQ2 + 8, LE = NQ * LK, S = (int)sizeof(T);
  using EO = EvenOdd<T, NQ, box_by_rows<T, NQ, GEO>()>;
  typedef typename EO::cptr cptr;
  T* const s_b = lds.b;
  T* const s_c = lds.c;
  double* const s_f = lds.f;

  const int t = threadIdx.x;
  BoxGrid g;
  int grp = 0, it = a.k;  // element group, iteration
  long long row0v = 0;    // first row of the problem in the vectors
  BatchState* bs = nullptr;
  if constexpr (BATCH) {
    // (items and problems through the constant address space: scalar loads,
    // so what follows from them stays uniform)
    typedef const __attribute__((address_space(4))) BoxBatchItem* iptr;
    typedef const __attribute__((address_space(4))) BoxBatchProb* pptr;
    const iptr item = (iptr)a.items + blockIdx.x;
    const int pid = item->pid;
    const pptr pr = (pptr)a.probs + pid;
    bs = a.bst + pid;
    if (bs->done) return;
    g.nx = pr->g.nx;
    g.ny = pr->g.ny;
    g.nz = pr->g.nz;
    g.dx.m = pr->g.dx.m;
    g.dx.s1 = pr->g.dx.s1;
    g.dx.s2 = pr->g.dx.s2;
    g.dy.m = pr->g.dy.m;
    g.dy.s1 = pr->g.dy.s1;
    g.dy.s2 = pr->g.dy.s2;
    grp = item->e0 / EPB;
    row0v = pr->off;
    a.z = a.tab + pr->tab;
    a.w64 = a.z + NQ;
    a.eo = a.w64 + NQ;
    a.geo += 24 * pr->el0;
    a.AqL += pr->loc;
    if constexpr (MODE == MODE_FOLD) {
      it = __builtin_amdgcn_readfirstlane(bs->iter);
      if (bs->stop_at != 0 && bs->stop_at <= it) return;
      if ((it & 1) == 0) {  // the direction of iteration k is in p for odd k
        const T* q = a.p;
        a.p = const_cast<T*>(a.q);
        a.q = q;
      }
      a.r += row0v;
      a.p += row0v;
      a.x += row0v;
      a.part_rr += pr->rr0;
      a.nrr = it == 0 ? pr->ninit : pr->nrr;
      a.part += pr->pAp0;
    }
    a.q += row0v;
  } else {
    g = a.g;
    grp = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if constexpr (MODE == MODE_FOLD) {
      if (a.k > 0 && (a.st->done || (a.st->stop_at != 0 && a.st->stop_at <= a.k))) return;
    }
  }
  const int nel = g.elements();
  if (grp * EPB >= nel) return;  // uniform
  int es = t / NQ2;
  if constexpr (NQ == 8) es = __builtin_amdgcn_readfirstlane(es);
  const int tl = t - es * NQ2;
  const int ai = tl % NQ, bj = tl / NQ;
  const bool active = grp * EPB + es < nel;
  const int e = active ? grp * EPB + es : 0;
  const int f = blockIdx.y;

  int ex, ey, ez;
  g.element(e, ex, ey, ez);
  unsigned off[NQ];
  box_pencil_offsets<T, NQ>(g, a.F, f, ex, ey, ez, ai, bj, active, off);
  T rq[NQ];
  if constexpr (MODE == MODE_FOLD) {
    if (box_direction<T, NQ, BATCH>(a, bs, it, grp, ai > 0 && bj > 0, off, rq, s_f)) return;  // uniform
  } else {
    const __amdgpu_buffer_rsrc_t rs = box_rsrc(a.q + (size_t)blockIdx.z * a.ldq);
#pragma unroll
    for (int k = 0; k < NQ; ++k) rq[k] = buffer_load<T>(rs, off[k]);
  }

  // LDS slots. Along k (node (k, b, a)): kb + k*LK in s_b, kc + k*LK in s_c;
  // along i (node (b, a, m)): oi[m] in s_b; along j (node (b, m, a)):
  // jc + m*NQ in s_c. (oi[m] = ib + (m + a) mod NQ.) The rotation in s_b keeps its three access patterns
  // free of bank conflicts.
  const int kb = es * LE + bj * NQ + (ai + bj) % NQ;
  const int kc = es * LE + bj * NQ + ai;
  const int jc = es * LE + bj * LK + ai;
  const int ib = es * LE + bj * LK + ai * NQ;
  // formed where they are used (an opaque copy of the lane's a each time),
  // not held in NQ registers across the node loop
  auto slots_i = [&](int (&oi)[NQ]) {
    int r = ai;
    asm volatile("" : "+v"(r));
#pragma unroll
    for (int m = 0; m < NQ; ++m) oi[m] = ib + (m + r < NQ ? m + r : m + r - NQ);
  };
  cptr tab = (cptr)a.eo;

#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    s_b[k * LK + kb] = rq[k];
    s_c[k * LK + kc] = rq[k];
  }
  element_sync<NQ>();
  // r derivative at (j, k) = (a, b), s derivative at (i, k) = (a, b); each
  // lane overwrites only its own pencil
  {
    int oi[NQ];
    slots_i(oi);
    T v[NQ], y[NQ];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = s_b[oi[m]];
    EO::apply(tab, v, y);
#pragma unroll
    for (int m = 0; m < NQ; ++m) s_b[oi[m]] = y[m];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = s_c[jc + m * NQ];
    EO::apply(tab, v, y);
#pragma unroll
    for (int m = 0; m < NQ; ++m) s_c[jc + m * NQ] = y[m];
  }
  element_sync<NQ>();

  // along k: t derivative, the factors, the mass term; Gr and Gs out, Gt kept
  T gt[NQ], rA[NQ];
  double dot = 0;
  EO::apply(tab, rq, gt);
  __builtin_amdgcn_sched_barrier(0);
  {
    TrilinearLine<T> map;
    T ga[6], gw = 0;
    if constexpr (GEO == GEO_TRILINEAR) {
      map.set((cptr)a.geo + (size_t)24 * e, a.z[ai], a.z[bj]);
    } else if constexpr (GEO == GEO_AFFINE) {
#pragma unroll
      for (int c = 0; c < 6; ++c) ga[c] = a.geo[6 * (size_t)e + c];
      gw = a.wJ[e];
    }
    // a node's weight is formed in FP64 and, in FP32, rounded once: rounded
    // 1D weights shift all nodes of a kind at once (N = 2, 1/3 and 4/3: half of
    // the FP32 operator's error; N = 7, affine: a third), for 0.5% of its time
    typedef const __attribute__((address_space(4))) double* wptr;
    const double wij = GEO == GEO_STORED ? 0.0 : a.w64[ai] * a.w64[bj];
    T zk[NQ];  // uniform: scalar loads
    double wk[NQ];
    if constexpr (GEO != GEO_STORED) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        if constexpr (GEO == GEO_TRILINEAR) zk[k] = ((cptr)a.z)[k];
        wk[k] = ((wptr)a.w64)[k];
      }
    }
    const T* kap = nullptr;
    int kstep = 0;
    if constexpr (KAPPA) {
      const int LX = g.nx * N + 1, LY = g.ny * N + 1;
      kap = a.kappa + (size_t)(ez * N) * ((size_t)LX * LY) + (size_t)(ey * N + bj) * LX + (ex * N + ai);
      kstep = LX * LY;
    }
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      // one node at a time: without these the compiler forms every node's
      // map values before the first is used and spills
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (GEO == GEO_TRILINEAR) map.pin();
      const T qr = s_b[k * LK + kb], qs = s_c[k * LK + kc], qt = gt[k];
      T Gr, Gs, Gt, W;
      if constexpr (GEO == GEO_TRILINEAR) {
        T kv = T(1);
        if constexpr (KAPPA) kv = kap[(size_t)k * kstep];
        map.template flux<KAPPA>(zk[k], (T)(wij * wk[k]), kv, qr, qs, qt, Gr, Gs, Gt, W);
      } else {
        T g[6];
        if constexpr (GEO == GEO_AFFINE) {
          const T w = (T)(wij * wk[k]);
          T wg = w;
          if constexpr (KAPPA) wg *= kap[(size_t)k * kstep];
#pragma unroll
          for (int c = 0; c < 6; ++c) g[c] = ga[c] * wg;
          W = gw * w;
        } else {
          const size_t n = (size_t)e * NP + k * NQ2 + tl;
#pragma unroll
          for (int c = 0; c < 6; ++c) g[c] = a.geo[6 * n + c];
          W = a.wJ[n];
        }
        Gr = fmad(g[2], qt, fmad(g[1], qs, g[0] * qr));
        Gs = fmad(g[4], qt, fmad(g[3], qs, g[1] * qr));
        Gt = fmad(g[5], qt, fmad(g[4], qs, g[2] * qr));
      }
      s_b[k * LK + kb] = Gr;
      s_c[k * LK + kc] = Gs;
      gt[k] = Gt;
      rA[k] = (a.lambda * W) * rq[k];
      if constexpr (MODE != MODE_PLAIN && sizeof(T) == 8) {
        // q.Aq node by node: grad q . G grad q + lambda W q^2
        dot = fmad(rA[k], rq[k], fmad(Gt, qt, fmad(Gs, qs, fmad(Gr, qr, dot))));
        asm volatile("" : "+v"(dot));
      }
      asm volatile("" : "+v"(gt[k]), "+v"(rA[k]));
    }
  }
  // (the table is requested again: held across the nodes it would take the
  // scalar registers of their coordinates and weights)
  asm volatile("" : "+s"(tab));
  {
    T y[NQ];
    EO::apply_transposed(tab, gt, y);
#pragma unroll
    for (int k = 0; k < NQ; ++k) rA[k] += y[k];
  }
  element_sync<NQ>();
  // the divergence's r part along i, its s part along j
  {
    int oi[NQ];
    slots_i(oi);
    T v[NQ], y[NQ];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = s_b[oi[m]];
    EO::apply_transposed(tab, v, y);
#pragma unroll
    for (int m = 0; m < NQ; ++m) s_b[oi[m]] = y[m];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = s_c[jc + m * NQ];
    EO::apply_transposed(tab, v, y);
#pragma unroll
    for (int m = 0; m < NQ; ++m) s_c[jc + m * NQ] = y[m];
  }
  element_sync<NQ>();
#pragma unroll
  for (int k = 0; k < NQ; ++k) rA[k] += s_b[k * LK + kb] + s_c[k * LK + kc];
  if constexpr (MODE != MODE_PLAIN) {
    if constexpr (sizeof(T) == 4) {  // q.Aq from the rounded results, as the rows see them
#pragma unroll
      for (int k = 0; k < NQ; ++k) dot = fmad((double)rq[k], (double)rA[k], dot);
    }
    const double v = block_sum<NQ2 * EPB>(dot, s_f);
    if (t == 0) a.part[(size_t)blockIdx.y * ((nel + EPB - 1) / EPB) + grp] = v;
  }
  if (active) {
    T* out = a.AqL + (size_t)blockIdx.z * a.ldAq + ((size_t)e * a.F + f) * NP + tl;
#pragma unroll
    for (int k = 0; k < NQ; ++k) out[k * NQ2] = rA[k];
  }
}

}  // namespace
}  // namespace bpx
