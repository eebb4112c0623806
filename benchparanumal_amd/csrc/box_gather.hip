// The gathers of box_gather_body.hpp, one problem per launch. Compiled once
// per Nq.
#include <algorithm>

#include "box_gather_body.hpp"

#ifndef BPX_NQ
#error "compile with -DBPX_NQ=<Nq>"
#endif

namespace bpx {
namespace {

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
