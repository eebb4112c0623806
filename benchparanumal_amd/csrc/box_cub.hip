// BP1/BP2 (mass) and BP3/BP4 (over-integrated stiffness + lambda*mass) Ax on
// the structured hex box, FP64 and FP32: the operators of
// okl/bp1AxHex3D.okl:61-325 and okl/bp3AxHex3D.okl:369-712 with cubwJ and
// cubggeo formed in the kernel from the elements' trilinear maps
// (TrilinearLine) and the rows of box.hpp in place of GlobalToLocal.
// Compiled once per Nq.
//
// A node costs its q and its result: the stored-factor kernels (ax_cub.hip)
// also read 7 factors per cubature point (56 bytes, 564 MB of 793 at 24^3,
// p = 7, for one BP3 field) and a row number per node.
//
// A workgroup holds box_epb(MQ) elements of one field, MQ = Nq + 1 cubature
// points a direction. Every one-dimensional operator runs along a line that
// one lane holds, in even-odd form (even_odd.hpp), and values move between
// directions through LDS, a line rewritten in place by the lane that read it:
//   k-lines (j,i):  q from memory (neighbouring lanes on neighbouring rows),
//                   x = I q along k                              -> A
//   j-lines (g,i):  I along j, in place                          -> A
//   i-lines (g,b):  u = I along i
//     mass:         times w J, back along i                      -> A
//     stiffness:    u -> A, ur = D u -> B
//   t-lines (b,a):  u into registers, ut = D u
//   s-lines (g,a):  us = D u, in place                           -> A
//   t-lines (b,a):  the fluxes: Gr -> B, Gs -> A; res = lambda W u + D^T Gt
//   s-lines (g,a):  D^T Gs, in place (A); r-lines (g,b): D^T Gr (B), kept
//   t-lines (b,a):  A += res
//   i-lines (g,b):  A + D^T Gr, back along i, in place           -> A
//   j-lines (g,i):  back along j, in place                       -> A
//   k-lines (j,i):  back along k                                 -> Aq
// 23 LDS accesses per point (mass: 8); odd line strides keep
// all but the k, j and s lines free of bank conflicts.
//
// Measured at 24^3, p = 7: BP4 operator 319 -> 245 us, BP3 mixed solve 150 ->
// 86 ms; BP1 on 23 x 21 x 19, p = 6, operator 41 -> 24 us. Of the 200 us of
// BP4's Ax the vector ALU issues for 117 (1295 instructions per wavefront, 500
// of them the factors) and LDS for 50, a third as much again lost to bank
// conflicts; 323 MB move.
#include "box_lanes.hpp"
#include "even_odd.hpp"

#ifndef BPX_NQ
#error "compile with -DBPX_NQ=<Nq>"
#endif

namespace bpx {
namespace {

// tiles of one workgroup and the sums (f[32] hands the folded r.r out)
template <typename T, int NQ, bool STIFF, int MODE>
struct BoxCubLds {
  // (at MQ = 7 and 16 a longer slab leaves a third fewer conflicts)
  static constexpr int MQ = NQ + 1, PR = MQ | 1, PS = MQ * PR + (MQ == 7 ? 5 : MQ == 16 ? 15 : 0), TILE = MQ * PS, EPB = box_epb(MQ);
  T a[EPB * TILE];
  T b[STIFF ? EPB * TILE : 1];
  double map[EPB * 24], z[MQ], w[MQ];  // the elements' maps, the points and weights
  double f[MODE == MODE_PLAIN ? 1 : MQ * MQ * EPB];
};

// occupancy handed to the register allocator
template <typename T, int NQ, bool STIFF>
constexpr int box_cub_waves() {
  if (!STIFF) return sizeof(T) == 4 ? (NQ <= 8 ? 6 : 4) : (NQ <= 8 ? 5 : 3);
  return sizeof(T) == 4 ? (NQ <= 8 ? 5 : NQ <= 11 ? 4 : 3) : (NQ <= 8 ? 4 : 2);
}

template <typename T, int NQ, bool STIFF, int MODE>
__global__ __launch_bounds__((NQ + 1) * (NQ + 1) * box_epb(NQ + 1))
    __attribute__((amdgpu_waves_per_eu(box_cub_waves<T, NQ, STIFF>()))) void k_box_cub(BoxAxArgs<T> a, int per_xcd) {
  constexpr int N = NQ - 1, NQ2 = NQ * NQ, NP = NQ2 * NQ, MQ = NQ + 1, MQ2 = MQ * MQ, EPB = box_epb(MQ);
  using Lds = BoxCubLds<T, NQ, STIFF, MODE>;
  constexpr int PR = Lds::PR, PS = Lds::PS, TILE = Lds::TILE, NT = MQ2 * EPB;
  using ET = EoTables<NQ>;
  typedef const __attribute__((address_space(4))) double* cptr;
  __shared__ Lds lds;

  const int t = threadIdx.x;
  const BoxGrid g = a.g;
  const int grp = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if constexpr (MODE == MODE_FOLD) {
    if (a.k > 0 && (a.st->done || (a.st->stop_at != 0 && a.st->stop_at <= a.k))) return;
  }
  const int nel = g.elements();
  if (grp * EPB >= nel) return;  // uniform
  const int f = blockIdx.y;
  // The maps, points and weights are FP64 (FP32 too, where the factors are
  // rounded as formed: rounded data would shift a whole element's at once).
  // Through LDS: lanes of a wavefront belong to several elements, and loads
  // at the use are waited for (BP3 mixed solve at 24^3, p = 7: 101 -> 85 ms).
  for (int i = t; i < EPB * 24; i += NT) lds.map[i] = a.geo64[min(grp * EPB * 24 + i, nel * 24 - 1)];
  if (t < MQ) {
    lds.z[t] = a.z64[t];
    lds.w[t] = a.w64[t];
  }

  // k-lines: line (j, i) = (kj, ki) of slot ks
  const int ks = t / NQ2, kl = t - ks * NQ2;
  const int ki = kl % NQ, kj = kl / NQ;
  const bool onk = ks < EPB, active = onk && grp * EPB + ks < nel;
  const int ke = active ? grp * EPB + ks : 0;
  T rq[NQ];
  {
    int ex, ey, ez;
    g.element(ke, ex, ey, ez);
    unsigned off[NQ];
    box_pencil_offsets<T, NQ>(g, a.F, f, ex, ey, ez, ki, kj, active, off);
    if constexpr (MODE == MODE_FOLD) {
      const bool stop = box_direction<T, NQ, false>(a, nullptr, a.k, grp, ki > 0 && kj > 0, off, rq, lds.f);
      if (__builtin_amdgcn_readfirstlane((int)stop)) return;  // uniform
    } else {
      const __amdgpu_buffer_rsrc_t rs = box_rsrc(a.q);
#pragma unroll
      for (int k = 0; k < NQ; ++k) rq[k] = buffer_load<T>(rs, off[k]);
    }
  }
  // point (g, b, a) of a tile: g*PS + b*PR + a
  // (idle lanes read a live line and store nothing; a wavefront of idle lanes
  // skips the line: the matrix pointer must stay uniform)
  const int t0 = __builtin_amdgcn_readfirstlane(t);
  const bool wk = t0 < EPB * NQ2, wj = t0 < EPB * NQ * MQ;
  T* const Ak = lds.a + (onk ? ks * TILE + kj * PR + ki : 0);
  const int js = t / (NQ * MQ), jl = t - js * (NQ * MQ);  // j-lines (g, i)
  const bool onj = js < EPB;
  T* const Aj = lds.a + (onj ? js * TILE + (jl / NQ) * PS + jl % NQ : 0);
  const int ls = t / MQ2, ll = t - ls * MQ2;  // t-lines (b, a), i-lines (g, b), s-lines (g, a)
  const int lh = ll / MQ, lw = ll - lh * MQ;
  const int el = grp * EPB + ls;
  const cptr zc = (cptr)a.z64, wc = (cptr)a.w64;
  const double* const ce = lds.map + 24 * ls;
  const int io = ls * TILE + lh * PS + lw * PR;  // i-line, step 1
  const int so = ls * TILE + lh * PS + lw;       // s-line, step PR
  const int to = ls * TILE + lh * PR + lw;       // t-line, step PS
  const T* const eo = a.eo;
  const double* const eo64 = a.eo64;

  auto interp = [&](const T(&x)[NQ], T(&y)[MQ]) { eo_apply<MQ, NQ, 1>(eo + ET::I, x, [&](int n, T v) { y[n] = v; }); };
  auto project = [&](const T(&x)[MQ], T(&y)[NQ]) { eo_apply<NQ, MQ, 1>(eo + ET::IT, x, [&](int n, T v) { y[n] = v; }); };
  auto diff = [&](const T(&x)[MQ], T(&y)[MQ]) { eo_apply<MQ, MQ, -1>(eo + ET::D, x, [&](int n, T v) { y[n] = v; }); };
  auto diff_t = [&](const T(&x)[MQ], T(&y)[MQ]) { eo_apply<MQ, MQ, -1>(eo + ET::DT, x, [&](int n, T v) { y[n] = v; }); };

  // Along t, FP32 up to Nq = 6: D by rows. Its even-odd parts round
  // differently, which at p = 5 makes the operator's error 9% larger (2.22e-7
  // against 2.04e-7; this way 2.00e-7); at p = 6 and 7 they are as close and
  // faster (24^3, p = 7: mixed solve 88 -> 85.5 ms).
  constexpr bool ROWS = sizeof(T) == 4 && NQ <= 6;
  auto diff_line = [&](const T(&x)[MQ], T(&y)[MQ]) {
    if constexpr (ROWS) {
      uniform_rows<MQ, MQ>(eo + ET::ROWS, [&](int n, const T* r) {
        T acc = 0;
#pragma unroll
        for (int m = 0; m < MQ; ++m) acc = fmad(r[m], x[m], acc);
        y[n] = acc;
      });
    } else {
      diff(x, y);
    }
  };
  auto add_diff_t = [&](const T(&x)[MQ], T(&y)[MQ]) {  // y += D^T x
    if constexpr (ROWS) {
      uniform_rows<MQ, MQ>(eo + ET::ROWS, [&](int m, const T* r) {
#pragma unroll
        for (int n = 0; n < MQ; ++n) y[n] = fmad(r[n], x[m], y[n]);
      });
    } else {
      T v[MQ];
      diff_t(x, v);
#pragma unroll
      for (int m = 0; m < MQ; ++m) y[m] += v[m];
    }
  };

  // FP32 up to Nq = 8: the last projection in FP64 (which issues at the same
  // rate), its result rounded once. It pays for the factors, whose 7 values a
  // point are formed in FP32 instead of rounded from FP64 ones: without it the
  // operator's error is up to 3.5% larger than with stored factors (p = 7),
  // with it smaller at every degree.
  constexpr bool END64 = sizeof(T) == 4 && NQ <= 8;
  auto project_last = [&](const T(&x)[MQ], T(&y)[NQ]) {
    if constexpr (END64) {
      double xd[MQ];
#pragma unroll
      for (int m = 0; m < MQ; ++m) xd[m] = x[m];
      eo_apply<NQ, MQ, 1>(eo64 + ET::IT, xd, [&](int n, double v) { y[n] = (T)v; });
    } else {
      project(x, y);
    }
  };

  {
    T y[MQ];
    interp(rq, y);
    if (onk)
#pragma unroll
      for (int m = 0; m < MQ; ++m) Ak[m * PS] = y[m];
  }
  __syncthreads();
  if (wj) {
    T v[NQ], y[MQ];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = Aj[m * PR];
    interp(v, y);
    if (onj)
#pragma unroll
      for (int m = 0; m < MQ; ++m) Aj[m * PR] = y[m];
  }
  __syncthreads();

  double dot = 0;
  if constexpr (!STIFF) {
    T v[NQ], u[MQ];
#pragma unroll
    for (int m = 0; m < NQ; ++m) v[m] = lds.a[io + m];
    interp(v, u);
    // J along the line (s, t) = (z[lw], z[lh]): the map with its directions
    // turned (s, t, r) for (r, s, t), x_s = Ar + Br r, x_t = As + Bs r, x_r = Ct
    double jt[3];
    {
      const double sn = lds.z[lw], tn = lds.z[lh];
      double Ar[3], Br[3], As[3], Bs[3], Ct[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double* const c = ce + 8 * d;
        Ar[d] = fmad(c[5], tn, c[1]);
        Br[d] = fmad(c[6], tn, c[3]);
        As[d] = fmad(c[5], sn, c[2]);
        Bs[d] = fmad(c[6], sn, c[4]);
        Ct[d] = fmad(Br[d], sn, fmad(c[4], tn, c[0]));
      }
      jt[0] = jt[1] = jt[2] = 0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int d1 = (d + 1) % 3, d2 = (d + 2) % 3;
        const double c0 = fmad(Ar[d1], As[d2], -(Ar[d2] * As[d1]));
        const double c1 = fmad(Ar[d1], Bs[d2], -(Ar[d2] * Bs[d1])) + fmad(Br[d1], As[d2], -(Br[d2] * As[d1]));
        const double c2 = fmad(Br[d1], Bs[d2], -(Br[d2] * Bs[d1]));
        jt[0] = fmad(Ct[d], c0, jt[0]);
        jt[1] = fmad(Ct[d], c1, jt[1]);
        jt[2] = fmad(Ct[d], c2, jt[2]);
      }
    }
    const double wst = lds.w[lw] * lds.w[lh];
#pragma unroll
    for (int m = 0; m < MQ; ++m) {
      const double zm = zc[m], wm = wc[m];
      const T Wu = (T)(fmad(fmad(jt[2], zm, jt[1]), zm, jt[0]) * (wst * wm)) * u[m];
      if constexpr (MODE != MODE_PLAIN && sizeof(T) == 8) {
        if (el < nel) dot = fmad(Wu, u[m], dot);
      }
      u[m] = Wu;
    }
    project(u, v);
#pragma unroll
    for (int m = 0; m < NQ; ++m) lds.a[io + m] = v[m];
  } else {
    {
      T v[NQ], u[MQ], ur[MQ];
#pragma unroll
      for (int m = 0; m < NQ; ++m) v[m] = lds.a[io + m];
      interp(v, u);
#pragma unroll
      for (int m = 0; m < MQ; ++m) lds.a[io + m] = u[m];
      diff(u, ur);
#pragma unroll
      for (int m = 0; m < MQ; ++m) lds.b[io + m] = ur[m];
    }
    __syncthreads();
    T u[MQ], gt[MQ];
#pragma unroll
    for (int m = 0; m < MQ; ++m) u[m] = lds.a[to + m * PS];
    __syncthreads();
    {
      T v[MQ], us[MQ];
#pragma unroll
      for (int m = 0; m < MQ; ++m) v[m] = lds.a[so + m * PR];
      diff(v, us);
#pragma unroll
      for (int m = 0; m < MQ; ++m) lds.a[so + m * PR] = us[m];
    }
    diff_line(u, gt);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    {
      TrilinearLine<T> map;
      map.set(ce, lds.z[lw], lds.z[lh]);
      const double wij = lds.w[lw] * lds.w[lh];
#pragma unroll
      for (int k = 0; k < MQ; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        map.pin();
        const T qr = lds.b[to + k * PS], qs = lds.a[to + k * PS], qt = gt[k];
        T Gr, Gs, Gt, W;
        map.template flux<false>((T)zc[k], (T)(wij * wc[k]), T(1), qr, qs, qt, Gr, Gs, Gt, W);
        lds.b[to + k * PS] = Gr;
        lds.a[to + k * PS] = Gs;
        const T m = (a.lambda * W) * u[k];
        if constexpr (MODE != MODE_PLAIN && sizeof(T) == 8) {
          if (el < nel) dot = fmad(m, u[k], fmad(Gt, qt, fmad(Gs, qs, fmad(Gr, qr, dot))));
          asm volatile("" : "+v"(dot));
        }
        gt[k] = Gt;
        u[k] = m;
        asm volatile("" : "+v"(gt[k]), "+v"(u[k]));
      }
    }
    __syncthreads();
    add_diff_t(gt, u);
    T rr[MQ];
    {
      T v[MQ], y[MQ];
#pragma unroll
      for (int m = 0; m < MQ; ++m) v[m] = lds.a[so + m * PR];
      diff_t(v, y);
#pragma unroll
      for (int m = 0; m < MQ; ++m) lds.a[so + m * PR] = y[m];
#pragma unroll
      for (int m = 0; m < MQ; ++m) v[m] = lds.b[io + m];
      diff_t(v, rr);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MQ; ++m) lds.a[to + m * PS] += u[m];
    __syncthreads();
    {
      T v[MQ], y[NQ];
#pragma unroll
      for (int m = 0; m < MQ; ++m) v[m] = rr[m] + lds.a[io + m];
      project(v, y);
#pragma unroll
      for (int m = 0; m < NQ; ++m) lds.a[io + m] = y[m];
    }
  }
  __syncthreads();
  if (wj) {
    T v[MQ], y[NQ];
#pragma unroll
    for (int m = 0; m < MQ; ++m) v[m] = Aj[m * PR];
    project(v, y);
    if (onj)
#pragma unroll
      for (int m = 0; m < NQ; ++m) Aj[m * PR] = y[m];
  }
  __syncthreads();
  if (wk) {
    T v[MQ], y[NQ];
#pragma unroll
    for (int m = 0; m < MQ; ++m) v[m] = Ak[m * PS];
    project_last(v, y);
    if constexpr (MODE != MODE_PLAIN && sizeof(T) == 4) {  // q.Aq from the rounded results, as the rows see them
      if (active)
#pragma unroll
        for (int k = 0; k < NQ; ++k) dot = fmad((double)rq[k], (double)y[k], dot);
    }
    if (active) {
      T* const out = a.AqL + ((size_t)ke * a.F + f) * NP + kl;
#pragma unroll
      for (int k = 0; k < NQ; ++k) out[k * NQ2] = y[k];
    }
  }
  if constexpr (MODE != MODE_PLAIN) {
    const double v = block_sum<NT>(dot, lds.f);
    if (t == 0) a.part[(size_t)blockIdx.y * ((nel + EPB - 1) / EPB) + grp] = v;
  }
}

template <typename T, int NQ, bool STIFF, int MODE>
int launch_mode(hipStream_t s, const BoxAxArgs<T>& a) {
  constexpr int EPB = box_epb(NQ + 1);
  const int per = ((a.g.elements() + EPB - 1) / EPB + 7) / 8;
  launch_stamped(k_box_cub<T, NQ, STIFF, MODE>, dim3((unsigned)per * 8, a.F), dim3((NQ + 1) * (NQ + 1) * EPB), s,
                 a.evStart, a.evStop, a, per);
  BPX_HIP(hipGetLastError());
  return BPX_OK;
}

template <typename T, int NQ, bool STIFF>
int launch_form(hipStream_t s, const BoxAxArgs<T>& a) {
  if (a.fold) return launch_mode<T, NQ, STIFF, MODE_FOLD>(s, a);
  if (a.part) return launch_mode<T, NQ, STIFF, MODE_DOT>(s, a);
  return launch_mode<T, NQ, STIFF, MODE_PLAIN>(s, a);
}

}  // namespace

template <typename T, int NQ>
int launch_box_cub_nq(hipStream_t s, const BoxAxArgs<T>& a) {
  return a.op == BOX_OP_MASS ? launch_form<T, NQ, false>(s, a) : launch_form<T, NQ, true>(s, a);
}

template int launch_box_cub_nq<double, BPX_NQ>(hipStream_t, const BoxAxArgs<double>&);
template int launch_box_cub_nq<float, BPX_NQ>(hipStream_t, const BoxAxArgs<float>&);

}  // namespace bpx
