// Geometric factors at one point from the 9 coordinate derivatives, shared
// by the host setup (host/mesh.cpp) and the device setup (setup.hip) so that
// both evaluate the same expressions in the same order; with floating-point
// contraction off in both builds the two give the same bits.
//
// Reference: libs/mesh/meshGeometricFactorsHex3D.cpp:116-135 (J by cofactor
// expansion, the inverse Jacobian's rows by cofactors over J, and the six
// entries of J (grad r)(grad r)^T); the formula is the textbook one.
#pragma once

#if defined(__HIPCC__)
#define BPX_HD __host__ __device__
#else
#define BPX_HD
#endif

namespace bpx {

struct Geo9 {
  double xr, xs, xt, yr, ys, yt, zr, zs, zt;
};

// J and the 6 symmetric entries of J (grad r)(grad r)^T
BPX_HD inline void metric(const Geo9& d, double& J, double g[6]) {
  J = d.xr * (d.ys * d.zt - d.zs * d.yt) - d.yr * (d.xs * d.zt - d.zs * d.xt) +
      d.zr * (d.xs * d.yt - d.ys * d.xt);
  const double rx = (d.ys * d.zt - d.zs * d.yt) / J, ry = -(d.xs * d.zt - d.zs * d.xt) / J,
               rz = (d.xs * d.yt - d.ys * d.xt) / J;
  const double sx = -(d.yr * d.zt - d.zr * d.yt) / J, sy = (d.xr * d.zt - d.zr * d.xt) / J,
               sz = -(d.xr * d.yt - d.yr * d.xt) / J;
  const double tx = (d.yr * d.zs - d.zr * d.ys) / J, ty = -(d.xr * d.zs - d.zr * d.xs) / J,
               tz = (d.xr * d.ys - d.yr * d.xs) / J;
  g[0] = J * (rx * rx + ry * ry + rz * rz);
  g[1] = J * (rx * sx + ry * sy + rz * sz);
  g[2] = J * (rx * tx + ry * ty + rz * tz);
  g[3] = J * (sx * sx + sy * sy + sz * sz);
  g[4] = J * (sx * tx + sy * ty + sz * tz);
  g[5] = J * (tx * tx + ty * ty + tz * tz);
}

// sign (+1 / -1) of the reference coordinates r, s, t of vertex v (0..7) in
// the reference's vertex order (libs/mesh/meshSetElementType.cpp)
BPX_HD constexpr double vertex_r(int v) { return ((v ^ (v >> 1)) & 1) ? 1.0 : -1.0; }
BPX_HD constexpr double vertex_s(int v) { return ((v >> 1) & 1) ? 1.0 : -1.0; }
BPX_HD constexpr double vertex_t(int v) { return ((v >> 2) & 1) ? 1.0 : -1.0; }

// the trilinear map's weight of vertex v at (r, s, t)
BPX_HD inline double vertex_weight(int v, double r, double s, double t) {
  return 0.125 * (1 + vertex_r(v) * r) * (1 + vertex_s(v) * s) * (1 + vertex_t(v) * t);
}

// The coefficients of r, s, t, rs, rt, st and rst of the trilinear map whose
// values at the 8 vertices are V, and one pad. Differences along the edges
// come first: they are exact, or rounded relative to themselves, where sums
// of coordinates would be rounded relative to the distance from the origin
// (which left the operator of N = 1 on 15 elements a side twice as far from
// exact arithmetic as its stored factors are).
BPX_HD inline void trilinear_coefficients(const double* V, double* c) {
  const double r0 = V[1] - V[0], r1 = V[2] - V[3], r2 = V[5] - V[4], r3 = V[6] - V[7];  // edges along r
  const double s0 = V[3] - V[0], s1 = V[2] - V[1], s2 = V[7] - V[4], s3 = V[6] - V[5];
  const double t0 = V[4] - V[0], t1 = V[5] - V[1], t2 = V[6] - V[2], t3 = V[7] - V[3];
  c[0] = 0.125 * ((r0 + r1) + (r2 + r3));
  c[1] = 0.125 * ((s0 + s1) + (s2 + s3));
  c[2] = 0.125 * ((t0 + t1) + (t2 + t3));
  c[3] = 0.125 * ((r1 - r0) + (r3 - r2));  // rs
  c[4] = 0.125 * ((r2 - r0) + (r3 - r1));  // rt
  c[5] = 0.125 * ((s2 - s0) + (s3 - s1));  // st
  c[6] = 0.125 * ((r3 - r2) - (r1 - r0));  // rst
  c[7] = 0.0;
}

}  // namespace bpx
