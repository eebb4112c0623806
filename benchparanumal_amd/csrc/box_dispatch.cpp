// Run-time degree -> compiled Nq instantiation of the structured-box kernels.
#include "box_common.hpp"

namespace bpx {

#define BPX_BOX_SWITCH(CALL)                                                                       \
  switch (g.N + 1) {                                                                               \
    CALL(2) CALL(3) CALL(4) CALL(5) CALL(6) CALL(7) CALL(8) CALL(9) CALL(10) CALL(11) CALL(12)     \
    CALL(13) CALL(14) CALL(15) CALL(16)                                                            \
    default: return set_error(BPX_ERR_UNSUPPORTED, "box: degree N must be in 1..15");              \
  }

template <typename T>
int launch_box_gather(hipStream_t s, const BoxGrid& g, int F, int K, const T* AqL, long long ldL, T* out,
                      long long ldo) {
  if (!AqL || !out) return set_error(BPX_ERR_INVALID_ARGUMENT, "box gather: null device pointer");
  if (K < 1 || K > kBoxMaxRhs) return set_error(BPX_ERR_INVALID_ARGUMENT, "box gather: K outside 1..65535");
#define BPX_CALL(NQ) case NQ: return launch_box_gather_nq<T, NQ>(s, g, F, K, AqL, ldL, out, ldo);
  BPX_BOX_SWITCH(BPX_CALL)
#undef BPX_CALL
}

template <typename T>
int launch_box_ax(hipStream_t s, const BoxAxArgs<T>& a) {
  const BoxGrid& g = a.g;
  if (!a.q || !a.AqL) return set_error(BPX_ERR_INVALID_ARGUMENT, "box Ax: null device pointer");
  if (a.K < 1 || a.K > kBoxMaxRhs) return set_error(BPX_ERR_INVALID_ARGUMENT, "box Ax: K outside 1..65535");
  const bool gll = a.op == BOX_OP_GLL;
  const bool geo = gll ? a.geo && (a.geoKind == BOX_GEO_TRILINEAR ? a.z : a.wJ) && (a.geoKind == BOX_GEO_STORED || a.w64)
                       : a.geo64 && a.z64 && a.w64 && (sizeof(T) == 8 || a.eo64);
  if (!a.eo || !geo)
    return set_error(BPX_ERR_INVALID_ARGUMENT, "box Ax: null geometry/operator pointer");
  if (!gll && (a.geoKind != BOX_GEO_TRILINEAR || a.kappa || a.K != 1))
    return set_error(BPX_ERR_UNSUPPORTED, "box Ax: the cubature operators have constant coefficients and one right-hand side");
  if (a.fold && (!a.part || !a.r || !a.p || !a.x || !a.part_rr || !a.hist_rr || !a.hist_alpha || !a.st || a.p == a.q))
    return set_error(BPX_ERR_INVALID_ARGUMENT, "box Ax: incomplete CG arguments");
#define BPX_CALL(NQ) case NQ: return gll ? launch_box_ax_nq<T, NQ>(s, a) : launch_box_cub_nq<T, NQ>(s, a);
  BPX_BOX_SWITCH(BPX_CALL)
#undef BPX_CALL
}

int box_gather_elements(int Nq) { return box_gather_epb(Nq); }

int box_ax_elements(int Nq) { return box_epb(Nq); }

int box_ax_partials(const BoxGrid& g, int F, int op) {
  const int epb = box_epb(g.N + (op == BOX_OP_GLL ? 1 : 2));
  return (g.elements() + epb - 1) / epb * F;
}

template <typename T>
int launch_box_update_r(hipStream_t s, const BoxGrid& g, int F, const BoxUpdateR<T>& u, int* nrr) {
  if (!u.AqL || !u.r || !u.part_pAp || !u.part_rr || !u.st || !u.hist_rr || !u.hist_alpha)
    return set_error(BPX_ERR_INVALID_ARGUMENT, "box update: null device pointer");
#define BPX_CALL(NQ) case NQ: return launch_box_update_r_nq<T, NQ>(s, g, F, u, nrr);
  BPX_BOX_SWITCH(BPX_CALL)
#undef BPX_CALL
}

template int launch_box_update_r<double>(hipStream_t, const BoxGrid&, int, const BoxUpdateR<double>&, int*);
template int launch_box_update_r<float>(hipStream_t, const BoxGrid&, int, const BoxUpdateR<float>&, int*);
template int launch_box_ax<double>(hipStream_t, const BoxAxArgs<double>&);
template int launch_box_ax<float>(hipStream_t, const BoxAxArgs<float>&);
template int launch_box_gather<double>(hipStream_t, const BoxGrid&, int, int, const double*, long long, double*,
                                       long long);
template int launch_box_gather<float>(hipStream_t, const BoxGrid&, int, int, const float*, long long, float*,
                                      long long);

}  // namespace bpx
