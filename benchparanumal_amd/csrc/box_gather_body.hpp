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
#pragma once
#include <hip/hip_runtime.h>

#include "box_common.hpp"
#include "buffer_rsrc.hpp"
#include "fold.hpp"

namespace bpx {
namespace {

constexpr int GT = kBoxGatherLanes;

template <int NQ>
constexpr int box_gather_slots() {
  return box_gather_epb(NQ);
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

}  // namespace
}  // namespace bpx
