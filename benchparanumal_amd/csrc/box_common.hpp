// Per-degree launchers of the structured-box kernels (box_*.hip, compiled
// once per Nq); box_dispatch.cpp maps the run-time degree onto them.
#pragma once
#include "box.hpp"
#include "bpx_internal.hpp"

namespace bpx {

template <typename T, int NQ>
int launch_box_gather_nq(hipStream_t s, const BoxGrid& g, int F, int K, const T* AqL, long long ldL, T* out,
                         long long ldo);

template <typename T, int NQ>
int launch_box_ax_nq(hipStream_t s, const BoxAxArgs<T>& a);
template <typename T, int NQ>
int launch_box_cub_nq(hipStream_t s, const BoxAxArgs<T>& a);
template <typename T, int NQ>
int launch_box_update_r_nq(hipStream_t s, const BoxGrid& g, int F, const BoxUpdateR<T>& u, int* nrr);

// lanes and elements per workgroup of the gathers: a lane per owned column
constexpr int kBoxGatherLanes = 256;
constexpr int box_gather_epb(int Nq) { return kBoxGatherLanes / ((Nq - 1) * (Nq - 1)); }

// elements per workgroup of the Ax, by the points per direction: about 256 lanes
constexpr int box_epb(int Nq) { return Nq * Nq >= 144 ? 1 : 256 / (Nq * Nq); }

}  // namespace bpx
