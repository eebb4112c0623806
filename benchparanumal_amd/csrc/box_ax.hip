// The Ax of box_ax_body.hpp, one problem per launch. Compiled once per Nq.
#include "box_ax_body.hpp"

#ifndef BPX_NQ
#error "compile with -DBPX_NQ=<Nq>"
#endif

namespace bpx {
namespace {

template <typename T, int NQ, int GEO, bool KAPPA, int MODE>
__global__ __launch_bounds__(NQ* NQ* box_epb(NQ)) __attribute__((amdgpu_waves_per_eu(box_waves<T, NQ>()))) void k_box_ax(
    BoxAxArgs<T> a, int per_xcd) {
  __shared__ BoxAxLds<T, NQ, MODE> lds;
  box_ax_body<T, NQ, GEO, KAPPA, MODE, false>(a, per_xcd, lds);
}

template <typename T, int NQ, int GEO, bool KAPPA, int MODE>
int launch_mode(hipStream_t s, const BoxAxArgs<T>& a) {
  constexpr int EPB = box_epb(NQ);
  const int per = ((a.g.elements() + EPB - 1) / EPB + 7) / 8;
  launch_stamped(k_box_ax<T, NQ, GEO, KAPPA, MODE>, dim3((unsigned)per * 8, a.F, a.K), dim3(NQ * NQ * EPB), s, a.evStart,
                 a.evStop, a, per);
  BPX_HIP(hipGetLastError());
  return BPX_OK;
}

template <typename T, int NQ, int GEO, bool KAPPA>
int launch_geo(hipStream_t s, const BoxAxArgs<T>& a) {
  if (a.fold) return launch_mode<T, NQ, GEO, KAPPA, MODE_FOLD>(s, a);
  if (a.part) return launch_mode<T, NQ, GEO, KAPPA, MODE_DOT>(s, a);
  return launch_mode<T, NQ, GEO, KAPPA, MODE_PLAIN>(s, a);
}

}  // namespace

template <typename T, int NQ>
int launch_box_ax_nq(hipStream_t s, const BoxAxArgs<T>& a) {
  if constexpr (sizeof(T) == 8) {  // the variable coefficient is an FP64 operator
    if (a.kappa)
      return a.geoKind == BOX_GEO_AFFINE ? launch_geo<T, NQ, GEO_AFFINE, true>(s, a)
                                         : launch_geo<T, NQ, GEO_TRILINEAR, true>(s, a);
  } else {
    if (a.geoKind == BOX_GEO_STORED) return launch_geo<T, NQ, GEO_STORED, false>(s, a);
  }
  return a.geoKind == BOX_GEO_AFFINE ? launch_geo<T, NQ, GEO_AFFINE, false>(s, a)
                                     : launch_geo<T, NQ, GEO_TRILINEAR, false>(s, a);
}

template int launch_box_ax_nq<double, BPX_NQ>(hipStream_t, const BoxAxArgs<double>&);
template int launch_box_ax_nq<float, BPX_NQ>(hipStream_t, const BoxAxArgs<float>&);

}  // namespace bpx
