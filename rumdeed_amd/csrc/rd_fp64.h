// The FP64 pair terms.
//
// What bounds the FP64 pair kernels is the VALU time of one square root and
// one division per image partner.  Pair distances of a diode are far from
// every range limit, so the kernels test the coordinates once per staged chunk
// (f64_ordinary) and take the sequences of rd_ops64.h; a chunk that holds an
// extreme, infinite or NaN coordinate takes the general operations, with the
// same results.  Measured, ten image terms: accelerations of 16 384 electrons
// 14.69 -> 11.16 ms; the field on 256 x 256 cathode points over 4096
// electrons, with the paired distances of surface_pair64, 14.65 -> 6.04 ms.
#pragma once

#include <hip/hip_runtime.h>

#include "rd_internal.h"
#include "rd_ops64.h"

namespace rd {

// 1 / r^3 of the softened distance r = sqrt(r2) + es.
template <class M>
__device__ __forceinline__ double inv_r3_64(double r2, double es) {
  const double r = M::sqrt(r2) + es;
  return M::rcp(r * r * r);
}

// Direct and planar image factors of one pair (acc_ic_planar_series.inc:19-63):
// i0 = 1 / r^3 of the direct term, (ix, iy, iz) the image series (g.ic).  za, zb:
// the heights of the pair's first and second particle; (dx, dy, dz): target -
// source.  For the source as the target, i0 and iz are the same and ix, iy
// change sign.
template <class M>
__device__ __forceinline__ void planar_series64(const DevGeom& g, double dx, double dy, double dz,
                                                double za, double zb, double& i0, double& ix,
                                                double& iy, double& iz) {
  const double dxy2 = M::lift(dx * dx + dy * dy);
  i0 = inv_r3_64<M>(dxy2 + dz * dz, g.es);
  ix = iy = iz = 0.0;
  if (!g.ic) return;
  auto partner = [&](double z_ic, double& diff) {
    diff = za - z_ic;
    return inv_r3_64<M>(dxy2 + diff * diff, g.es);
  };
  double diff;
  double inv = partner(-1.0 * zb, diff);
  ix = -dx * inv;
  iy = -dy * inv;
  iz = -diff * inv;
  for (int n = 1; n <= g.nic; ++n) {
    const double tnd = 2.0 * n * g.d;
    inv = partner(tnd - zb, diff);
    ix = ix - dx * inv;
    iy = iy - dy * inv;
    iz = iz - diff * inv;
    inv = partner(-tnd - zb, diff);
    ix = ix - dx * inv;
    iy = iy - dy * inv;
    iz = iz - diff * inv;
    inv = partner(tnd + zb, diff);
    ix = ix + dx * inv;
    iy = iy + dy * inv;
    iz = iz + diff * inv;
    inv = partner(-tnd + zb, diff);
    ix = ix + dx * inv;
    iy = iy + dy * inv;
    iz = iz + diff * inv;
  }
}

// Direct and image terms of one pair with the charge product pre.
template <class M>
__device__ __forceinline__ void planar_pair64(const DevGeom& g, double pre, double dx, double dy,
                                              double dz, double za, double zb, double& ax,
                                              double& ay, double& az) {
  double i0, ix, iy, iz;
  planar_series64<M>(g, dx, dy, dz, za, zb, i0, ix, iy, iz);
  const double p0 = pre * i0;
  ax = p0 * dx;
  ay = p0 * dy;
  az = p0 * dz;
  if (!g.ic) return;
  ax = ax + pre * ix;
  ay = ay + pre * iy;
  az = az + pre * iz;
}

// planar_pair64 with image charges for a target on the cathode, za = 0.  The
// direct term and the n = 0 image are at the same distance, and so are the
// opposite partner at tnd - zb with the same-charge one at -tnd + zb, and the
// one at -tnd - zb with the one at tnd + zb: their z differences are exact
// negations, so the 2 + 4 nic distances of the series are 1 + 2 nic square
// roots and divisions; the additions are those of planar_pair64, in its
// order.  Z: the z component alone (a flat cathode's emission needs no other).
template <class M, bool Z>
__device__ __forceinline__ void surface_pair64(const DevGeom& g, double pre, double dx, double dy,
                                               double zb, double& ax, double& ay, double& az) {
  const double dxy2 = M::lift(dx * dx + dy * dy);
  const double i0 = inv_r3_64<M>(dxy2 + zb * zb, g.es);
  const double p0 = pre * i0;
  double ix = 0.0, iy = 0.0, iz = -zb * i0;
  if (!Z) {
    ix = -dx * i0;
    iy = -dy * i0;
  }
  for (int n = 1; n <= g.nic; ++n) {
    const double tnd = 2.0 * n * g.d;
    const double u = tnd - zb, w = tnd + zb;
    const double ia = inv_r3_64<M>(dxy2 + u * u, g.es);
    const double ib = inv_r3_64<M>(dxy2 + w * w, g.es);
    const double pa = u * ia, pb = w * ib;
    iz = (((iz + pa) - pb) - pb) + pa;
    if (!Z) {
      const double xa = dx * ia, xb = dx * ib, ya = dy * ia, yb = dy * ib;
      ix = (((ix - xa) - xb) + xb) + xa;
      iy = (((iy - ya) - yb) + yb) + ya;
    }
  }
  az = p0 * -zb + pre * iz;
  if (!Z) {
    ax = p0 * dx + pre * ix;
    ay = p0 * dy + pre * iy;
  }
}

// Sphere image force of the pair (a, b) at b's offset d = a - b with |d|^2 = r2
// and its root s (acc_tip_ic_force.inc:17-22, t**1.5 = t * sqrt(t)); the image
// (x_im, y_im, z_im) and the distance dis_a from the sphere's centre are a's.
template <class M>
__device__ __forceinline__ void tip_ic64(double dx, double dy, double dz, double r2, double s,
                                         double ex, double ey, double ez, double dis_a, double R,
                                         double kt, double& icx, double& icy, double& icz) {
  const double tb = (-ex) * (-ex) + (-ey) * (-ey) + (-ez) * (-ez);
  const typename M::Div da(r2 * s), db(dis_a * (tb * M::sqrt(tb)));
  icx = kt * (da(dx) - db(R * ex));
  icy = kt * (da(dy) - db(R * ey));
  icz = kt * (da(dz) - db(R * ez));
}

}  // namespace rd
