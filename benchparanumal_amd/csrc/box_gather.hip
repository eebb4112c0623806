// Gather of local values onto the rows of a structured hex box, without maps.
//
// The sums of libs/ogs/okl/ogsKernels.okl:86-122 (each row from 0, its
// copies in ascending local order) with the row numbering of box.hpp: a lane
// holds a column (i, j) of an element's owned nodes and walks k. A node's
// copies are its own element's value and, on the faces i = N, j = N and
// k = N, those of the up to 7 elements above it; own, +x, +y, +x+y, then the
// same four one layer up is ascending local order, so the result is the map
// gather's bit for bit.
//
// Bound by memory: 8 bytes read per local node and 8 written per row, where
// the map gather (k_gather) also reads a column id per local node and a row
// start per row (a third of its bytes). Copies that do not exist are loads at an
// offset beyond the buffer resource, which read 0 without touching memory:
// no load sits under a branch, so all of a lane's loads are in flight
// together. Each XCD (block mod 8) takes a contiguous eighth of the
// elements, so a face read again by its neighbour is found in that L2.
// Measured at 24^3, p = 7 (operator minus Ax, FP64): one field 32 -> 27 us,
// three fields 102 -> 70 us, and 16 right-hand sides at 20^3 in one launch
// 288 -> 210 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "box_common.hpp"
#include "buffer_rsrc.hpp"
#include "fold.hpp"

#ifndef BPX_NQ
#error "compile with -DBPX_NQ=<Nq>"
#endif

namespace bpx {
namespace {

constexpr int GT = 256;  // lanes per workgroup

__device__ inline double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <int NQ>
constexpr int box_gather_slots() {
  return GT / ((NQ - 1) * (NQ - 1));
}

// One column of owned nodes: sums for k = k0 .. k0+KC-1 (owned k from 1)
template <typename T, int NQ>
struct BoxColumn {
  static constexpr int N = NQ - 1, NQ2 = NQ * NQ, NP = NQ2 * NQ;
  int row, stride, nk;         // row of k = 1, rows per layer, owned layers (0: idle lane)
  unsigned own, ox, oy, oxy;   // byte offsets of the copies at k = 0
  unsigned zown, zx, zy, zxy;  // one layer of elements up, their k = 0 plane

  __device__ inline void set(const BoxGrid& g, int F, int f, int e, int c, bool on) {
    int ex, ey, ez;
    g.element(e, ex, ey, ez);
    const int i = c % N + 1, j = c / N + 1;
    const int Nx = BoxGrid::owned<N>(ex, g.nx), Ny = BoxGrid::owned<N>(ey, g.ny), Nz = BoxGrid::owned<N>(ez, g.nz);
    on = on && i <= Nx && j <= Ny;
    stride = Nx * Ny;
    nk = on ? Nz : 0;
    row = g.base<N>(F, ex, ey, ez) + f * stride * Nz + (j - 1) * Nx + i - 1;
    constexpr unsigned S = sizeof(T);
    const unsigned ES = F * NP * S;  // bytes of an element
    const unsigned at = e * ES + f * NP * S;
    const bool fx = i == N, fy = j == N, fz = Nz == N;
    own = on ? at + (j * NQ + i) * S : kBoxMasked;
    ox = on && fx ? at + ES + j * NQ * S : kBoxMasked;
    oy = on && fy ? at + g.nx * ES + i * S : kBoxMasked;
    oxy = on && fx && fy ? at + (g.nx + 1) * ES : kBoxMasked;
    const unsigned up = g.nx * g.ny * ES;
    zown = on && fz ? own + up : kBoxMasked;
    zx = on && fz && fx ? ox + up : kBoxMasked;
    zy = on && fz && fy ? oy + up : kBoxMasked;
    zxy = on && fz && fx && fy ? oxy + up : kBoxMasked;
  }
};

template <typename T, int NQ, typename Put>
__device__ inline void box_column_sums(const BoxColumn<T, NQ>& b, __amdgpu_buffer_rsrc_t rs, Put&& put) {
  constexpr int N = NQ - 1, NQ2 = NQ * NQ, S = (int)sizeof(T);
  constexpr int KC = 8;  // layers in flight
#pragma unroll
  for (int k0 = 1; k0 <= N; k0 += KC) {
    constexpr int M = KC < N ? KC : N;
    T v[M][4], z[4];
#pragma unroll
    for (int u = 0; u < M; ++u) {
      const int k = k0 + u;
      if (k > N) continue;
      v[u][0] = buffer_load<T>(rs, b.own + k * NQ2 * S);
      v[u][1] = buffer_load<T>(rs, b.ox + k * NQ2 * S);
      v[u][2] = buffer_load<T>(rs, b.oy + k * NQ2 * S);
      v[u][3] = buffer_load<T>(rs, b.oxy + k * NQ2 * S);
      if (k == N) {
        z[0] = buffer_load<T>(rs, b.zown);
        z[1] = buffer_load<T>(rs, b.zx);
        z[2] = buffer_load<T>(rs, b.zy);
        z[3] = buffer_load<T>(rs, b.zxy);
      }
    }
#pragma unroll
    for (int u = 0; u < M; ++u) {
      const int k = k0 + u;
      if (k > N) continue;
      T acc = T(0) + v[u][0];
      acc += v[u][1];
      acc += v[u][2];
      acc += v[u][3];
      if (k == N) {
        acc += z[0];
        acc += z[1];
        acc += z[2];
        acc += z[3];
      }
      put(k, acc);
    }
  }
}

// rows of one vector (grid.y: the field, grid.z: the vector)
template <typename T, int NQ>
__global__ __launch_bounds__(GT) void k_box_gather(BoxGrid g, int F, int per_xcd, const T* __restrict__ AqL,
                                                   long long ldL, T* __restrict__ out, long long ldo) {
  constexpr int N = NQ - 1, N2 = N * N, SL = box_gather_slots<NQ>();
  const int grp = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  const int es = (int)threadIdx.x / N2;
  const int e = grp * SL + es;
  BoxColumn<T, NQ> b;
  b.set(g, F, blockIdx.y, e, (int)threadIdx.x - es * N2, es < SL && e < g.elements());
  T* o = out + (size_t)blockIdx.z * ldo;
  box_column_sums<T, NQ>(b, box_rsrc(AqL + (size_t)blockIdx.z * ldL), [&](int k, T v) {
    if (k <= b.nk) o[b.row + (k - 1) * b.stride] = v;
  });
}

// The end of a CG iteration on the box: the gather of Ap with
// cg::UpdateCG's r -= alpha Ap (libs/core/linearSolverCG.cpp:131-156), Ap
// itself never stored. alpha = r.r / p.Ap from the Ax kernel's partials;
// one partial of the new r.r per workgroup. The arithmetic per row and the
// breakdown test are k_cg_update_r's. A workgroup walks items (element
// group, field) of its XCD's eighth; its first item's loads are issued
// before the partials are folded.
template <typename T, int NQ>
__global__ __launch_bounds__(GT) void k_box_update_r(BoxGrid g, int F, int items, BoxUpdateR<T> u) {
  constexpr int N = NQ - 1, N2 = N * N, SL = box_gather_slots<NQ>();
  __shared__ double s_f[GT + 1];
  if (u.st->done || u.st->stop_at) return;
  const int es = (int)threadIdx.x / N2, c = (int)threadIdx.x - es * N2;
  const int per = (items + 7) / 8, x = blockIdx.x & 7;
  const int end = min((x + 1) * per, items), step = (int)(gridDim.x >> 3);
  const __amdgpu_buffer_rsrc_t rs = box_rsrc(u.AqL);
  T alpha = T(0);
  double rr = 0;
  bool folded = false;
  for (int it = x * per + (int)(blockIdx.x >> 3);; it += step) {
    const bool have = it < end;
    if (folded && !have) break;  // (a workgroup without items still folds once: uniform)
    const int grp = it / F, e = grp * SL + es;
    BoxColumn<T, NQ> b;
    b.set(g, F, it - grp * F, e, c, have && es < SL && e < g.elements());
    T Ap[N], r[N];
#pragma unroll
    for (int k = 0; k < N; ++k) r[k] = u.r[b.nk > k ? b.row + k * b.stride : 0];
    box_column_sums<T, NQ>(b, rs, [&](int k, T v) { Ap[k - 1] = v; });
    if (!folded) {
      const double pAp = block_fold<GT>(u.part_pAp, u.npAp, s_f);
      const double al = u.hist_rr[u.k] / pAp;
      if (!isfinite(al) || !(pAp > 0.0)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
          u.st->breakdown = 1;
          u.st->done = 1;
          u.st->iter = u.k;
        }
        return;
      }
      if (blockIdx.x == 0 && threadIdx.x == 0) u.hist_alpha[u.k] = al;
      alpha = (T)al;
      folded = true;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if (k < b.nk) {
        const T rn = fmad(-alpha, Ap[k], r[k]);
        u.r[b.row + k * b.stride] = rn;
        rr += (double)rn * (double)rn;
      }
    }
  }
  const double t = block_sum<GT>(rr, s_f);
  if (threadIdx.x == 0) u.part_rr[blockIdx.x] = t;
}

}  // namespace

template <typename T, int NQ>
int launch_box_update_r_nq(hipStream_t s, const BoxGrid& g, int F, const BoxUpdateR<T>& u, int* nrr) {
  constexpr int SL = box_gather_slots<NQ>();
  const int items = (g.elements() + SL - 1) / SL * F;
  const int grid = std::min((items + 7) / 8 * 8, kBoxRrParts);
  hipLaunchKernelGGL((k_box_update_r<T, NQ>), dim3(grid), dim3(GT), 0, s, g, F, items, u);
  BPX_HIP(hipGetLastError());
  *nrr = grid;
  return BPX_OK;
}

template int launch_box_update_r_nq<double, BPX_NQ>(hipStream_t, const BoxGrid&, int, const BoxUpdateR<double>&, int*);
template int launch_box_update_r_nq<float, BPX_NQ>(hipStream_t, const BoxGrid&, int, const BoxUpdateR<float>&, int*);

template <typename T, int NQ>
int launch_box_gather_nq(hipStream_t s, const BoxGrid& g, int F, int K, const T* AqL, long long ldL, T* out,
                         long long ldo) {
  constexpr int SL = box_gather_slots<NQ>();
  const int groups = (g.elements() + SL - 1) / SL;
  const int per = (groups + 7) / 8;
  hipLaunchKernelGGL((k_box_gather<T, NQ>), dim3((unsigned)per * 8, F, K), dim3(GT), 0, s, g, F, per, AqL, ldL, out,
                     ldo);
  BPX_HIP(hipGetLastError());
  return BPX_OK;
}

template int launch_box_gather_nq<double, BPX_NQ>(hipStream_t, const BoxGrid&, int, int, const double*, long long,
                                                  double*, long long);
template int launch_box_gather_nq<float, BPX_NQ>(hipStream_t, const BoxGrid&, int, int, const float*, long long,
                                                 float*, long long);

}  // namespace bpx
