// Rows of a structured hex box in closed form (host and device code).
//
// On the nx x ny x nz box with its boundary masked, rows are numbered by
// their first local copy (libs/ogs/ogsSetup.cpp:87-290), elements x fastest.
// A lattice node therefore belongs to the lowest element that holds it, and
// element (ex, ey, ez) owns its nodes i = 1..Nx, j = 1..Ny, k = 1..Nz, where
// Nx is N, or N - 1 in the last element along x, whose node i = N is masked
// (likewise y, z). Its rows are one run, in local order, field after field:
// node (i, j, k) of field f is row
//   base + ((f*Nz + k - 1)*Ny + j - 1)*Nx + i - 1
// with base = F*(ez*N*TX*TY + Nz*(ey*N*TX + Ny*ex*N)), TX = nx*N - 1 and
// TY = ny*N - 1. Kernels that use this form read no index maps.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define BPX_BOX_FN __host__ __device__ inline
#else
#define BPX_BOX_FN inline
#endif

namespace bpx {

// n / d for 32-bit unsigned n by a multiply and two shifts (Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994,
// figure 4.1)
struct FastDiv {
  uint32_t m = 0, s1 = 0, s2 = 0;
  void set(uint32_t d) {
    uint32_t l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    m = (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
    s1 = l < 1 ? l : 1;
    s2 = l > 1 ? l - 1 : 0;
  }
  BPX_BOX_FN uint32_t div(uint32_t n) const {
    const uint32_t t = (uint32_t)(((uint64_t)m * n) >> 32);
    return (t + ((n - t) >> s1)) >> s2;
  }
};

// largest vector of the box kernels (bytes): offsets are unsigned 32-bit
constexpr unsigned kBoxRange = 0xFFF00000u;

struct BoxGrid {
  int nx = 0, ny = 0, nz = 0, N = 0;
  FastDiv dx, dy;
  void set(int nx_, int ny_, int nz_, int N_) {
    nx = nx_;
    ny = ny_;
    nz = nz_;
    N = N_;
    dx.set((uint32_t)nx);
    dy.set((uint32_t)ny);
  }
  BPX_BOX_FN int elements() const { return nx * ny * nz; }
  BPX_BOX_FN void element(int e, int& ex, int& ey, int& ez) const {
    const int r = (int)dx.div((uint32_t)e);
    ez = (int)dy.div((uint32_t)r);
    ex = e - r * nx;
    ey = r - ez * ny;
  }
  // owned nodes along one direction of element `at` of `n`
  template <int N_>
  BPX_BOX_FN static int owned(int at, int n) {
    return at == n - 1 ? N_ - 1 : N_;
  }
  // first row of element (ex, ey, ez), F fields
  template <int N_>
  BPX_BOX_FN int base(int F, int ex, int ey, int ez) const {
    const int TX = nx * N_ - 1, TY = ny * N_ - 1;
    return F * (ez * N_ * TX * TY + owned<N_>(ez, nz) * (ey * N_ * TX + owned<N_>(ey, ny) * ex * N_));
  }
};

}  // namespace bpx
