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
  if (K < 1 || K > 65535) return set_error(BPX_ERR_INVALID_ARGUMENT, "box gather: K outside 1..65535");
#define BPX_CALL(NQ) case NQ: return launch_box_gather_nq<T, NQ>(s, g, F, K, AqL, ldL, out, ldo);
  BPX_BOX_SWITCH(BPX_CALL)
#undef BPX_CALL
}

template int launch_box_gather<double>(hipStream_t, const BoxGrid&, int, int, const double*, long long, double*,
                                       long long);
template int launch_box_gather<float>(hipStream_t, const BoxGrid&, int, int, const float*, long long, float*,
                                      long long);

}  // namespace bpx
