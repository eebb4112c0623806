// The CG iteration of a ragged batch (batch.hip): the Ax and the gather of
// the box kernels over the problems of every degree, two launches in all. A
// launch per degree left the chip idle (64 problems of degrees 3 to 8: 12
// launches of 2 to 16 us one after another, also as parallel branches of a
// graph, whose nodes the host still queues one by one, 4 us each). Here a
// workgroup takes an item of any degree and jumps to that degree's body; the
// registers are those of the largest body, so degrees up to 8 and above have
// a kernel each. 64 problems, 1.07 million unknowns, to 1e-8: 29.2 -> 12.5 ms
// (an iteration 70 -> 27 us; bound by one workgroup's chain of loads, sums
// and LDS passes, which the small problems do not fill the chip to hide).
#include "box_ax_body.hpp"
#include "box_gather_body.hpp"

namespace bpx {
namespace {

// The largest Nq of the first kernel. A batch with degrees on both sides pays
// for two launch pairs, one with only low degrees in the second kernel for
// that one's registers. us per iteration with 6 / 7 / 9 / 12 (24 to 64 boxes):
// degrees 3-8 47.1 / 46.5 / 34.7 / 35.8, 1-4 17.0 / 17.0 / 17.2 / 17.3, 5-12
// 55.6 / 55.1 / 57.3 / 55.6, 6-9 31.3 / 41.4 / 42.1 / 28.0, 8-15 42.8 / 42.1 /
// 52.0 / 52.2, 1-15 49.3 / 49.4 / 50.4 / 52.6 (one kernel for all degrees does
// not compile): 9 keeps the common degrees, up to 8, in one.
constexpr int kLow = 9;

template <int LO, int HI, typename F>
__device__ inline void dispatch(int nq, F&& f) {
  if constexpr (LO <= HI) {
    if (nq == LO)
      f(std::integral_constant<int, LO>());
    else
      dispatch<LO + 1, HI>(nq, f);
  }
}

template <int LO, int HI>
constexpr size_t lds_bytes() {
  size_t m = 0;
  if constexpr (LO <= HI) {
    m = lds_bytes<LO + 1, HI>();
    if (sizeof(BoxAxLds<double, LO, MODE_FOLD>) > m) m = sizeof(BoxAxLds<double, LO, MODE_FOLD>);
  }
  return m;
}

// LO..HI: the degrees' Nq. Lanes past a degree's workgroup leave at once.
template <int LO, int HI, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HI <= kLow ? 3 : 2))) void k_box_batch_ax(
    BoxAxArgs<double> a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef const __attribute__((address_space(4))) BoxBatchItem* iptr;
  typedef const __attribute__((address_space(4))) BoxBatchProb* pptr;
  const int nq = ((pptr)a.probs)[((iptr)a.items)[blockIdx.x].pid].g.N + 1;
  dispatch<LO, HI>(nq, [&](auto c) {
    constexpr int NQ = decltype(c)::value;
    if (threadIdx.x < NQ * NQ * box_epb(NQ))
      box_ax_body<double, NQ, GEO_TRILINEAR, false, MODE, true>(a, 0, *reinterpret_cast<BoxAxLds<double, NQ, MODE>*>(smem));
  });
}

// k_box_update_r for one degree's problems of a batch: a workgroup per item,
// the scalars in the problem's state. Fields are split between the two
// kernels of an iteration (see batch.hip): this one reads rr_k and stop_at,
// and the first workgroup writes alpha, rr_prev and iter, or done once the
// Ax kernel has recorded a stop.
template <int NQ>
__device__ inline void update_body(const BoxBatchUpdate& u, double* s_f) {
  constexpr int N = NQ - 1, N2 = N * N, SL = box_gather_slots<NQ>();
  const BoxBatchItem item = u.items[blockIdx.x];
  const BoxBatchProb pr = u.probs[item.pid];
  BatchState* st = u.st + item.pid;
  const bool lead = item.e0 == 0 && threadIdx.x == 0;
  if (st->done) return;
  if (st->stop_at) {
    if (lead) st->done = 1;
    return;
  }
  const int es = (int)threadIdx.x / N2, e = item.e0 + es;
  BoxColumn<double, NQ> b;
  b.set(pr.g, 1, 0, e, (int)threadIdx.x - es * N2, es < SL && e < pr.g.elements());
  double* rv = u.r + pr.off;
  double Ap[N], r[N];
#pragma unroll
  for (int k = 0; k < N; ++k) r[k] = u.r[k < b.nk ? pr.off + b.row + k * b.stride : 0];
  box_column_sums<double, NQ>(b, box_rsrc(u.AqL + pr.loc), [&](int k, double v) { Ap[k - 1] = v; });
  const double pAp = block_fold<GT>(u.part_pAp + pr.pAp0, pr.npAp, s_f);
  const double rr = st->rr_k, alpha = rr / pAp;
  if (!isfinite(alpha) || !(pAp > 0.0)) {
    if (lead) {
      st->breakdown = 1;
      st->done = 1;
      st->rnorm = sqrt(rr);
    }
    return;
  }
  double v = 0;
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (k < b.nk) {
      const double rn = fmad(-alpha, Ap[k], r[k]);
      rv[b.row + k * b.stride] = rn;
      v += rn * rn;
    }
  const double t = block_sum<GT>(v, s_f);
  if (threadIdx.x == 0) u.part_rr[pr.rr0 + item.e0 / SL] = t;
  if (lead) {
    st->alpha = alpha;
    st->rr_prev = rr;
    st->iter = st->iter + 1;
  }
}


template <int LO, int HI>
__global__ __launch_bounds__(GT) void k_box_batch_update_r(BoxBatchUpdate u) {
  __shared__ double s_f[GT + 1];
  const int nq = __builtin_amdgcn_readfirstlane(u.probs[u.items[blockIdx.x].pid].g.N) + 1;
  dispatch<LO, HI>(nq, [&](auto c) { update_body<decltype(c)::value>(u, s_f); });
}

template <int LO, int HI, int MODE>
int launch_ax(hipStream_t s, const BoxAxArgs<double>& a) {
  constexpr size_t lds = lds_bytes<LO, HI>();
  hipLaunchKernelGGL((k_box_batch_ax<LO, HI, MODE>), dim3((unsigned)a.nitems), dim3(256), lds, s, a);
  BPX_HIP(hipGetLastError());
  return BPX_OK;
}

// more than 64 KB of LDS has to be granted to a kernel
template <int LO, int HI, int MODE>
int grant_lds() {
  constexpr size_t lds = lds_bytes<LO, HI>();
  if constexpr (lds > 65536)
    BPX_HIP(hipFuncSetAttribute((const void*)k_box_batch_ax<LO, HI, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  return BPX_OK;
}

}  // namespace

int prepare_box_batch() {
  if (int st = grant_lds<2, kLow, MODE_PLAIN>()) return st;
  if (int st = grant_lds<2, kLow, MODE_FOLD>()) return st;
  if (int st = grant_lds<kLow + 1, 16, MODE_PLAIN>()) return st;
  return grant_lds<kLow + 1, 16, MODE_FOLD>();
}

int box_batch_class(int N) { return N + 1 <= kLow ? 0 : 1; }

int launch_box_batch_ax(hipStream_t s, int cls, const BoxAxArgs<double>& a) {
  if (a.nitems == 0) return BPX_OK;
  if (!a.q || !a.AqL || !a.geo || !a.tab || !a.items || !a.probs || !a.bst ||
      (a.fold && (!a.part || !a.r || !a.p || !a.x || !a.part_rr)))
    return set_error(BPX_ERR_INVALID_ARGUMENT, "batch Ax: null pointer");
  if (a.fold) return cls == 0 ? launch_ax<2, kLow, MODE_FOLD>(s, a) : launch_ax<kLow + 1, 16, MODE_FOLD>(s, a);
  return cls == 0 ? launch_ax<2, kLow, MODE_PLAIN>(s, a) : launch_ax<kLow + 1, 16, MODE_PLAIN>(s, a);
}

int launch_box_batch_update_r(hipStream_t s, int cls, const BoxBatchUpdate& u) {
  if (u.nitems == 0) return BPX_OK;
  if (cls == 0)
    hipLaunchKernelGGL((k_box_batch_update_r<2, kLow>), dim3((unsigned)u.nitems), dim3(GT), 0, s, u);
  else
    hipLaunchKernelGGL((k_box_batch_update_r<kLow + 1, 16>), dim3((unsigned)u.nitems), dim3(GT), 0, s, u);
  BPX_HIP(hipGetLastError());
  return BPX_OK;
}

}  // namespace bpx
