// FP64 sums with the lanes on the pair terms.
//
// The canonical order adds the 256 terms of a source chunk in sequence.  With a
// lane per target (k_accel64, k_field64) that chain of additions and its terms
// run in one lane: a call on few targets has fewer wavefronts than the chip
// has SIMDs, and each issues an FP64 instruction every eight cycles at best.
// Here the lanes form the terms, LDS holds them, and a few lanes add them in
// the canonical order, so the results are the same bits.  What bounds a light
// term (no image series) is that chain, 256 additions of 8 cycles: three
// workgroups share a CU, so that the others' terms fill it.
//   k_rows64     few targets: a workgroup takes kRowT targets and a source
//                chunk, a lane per source.  A field point over 431 electrons, one
//                image term: 139 -> 9 us; 853 electrons, ten terms: 820 -> 101 us
//                a call.
//   k_accel64sym many particles: a workgroup takes two chunks of particles and
//                evaluates each of their pairs once, for both particles.  16 384
//                electrons, ten image terms: 10.96 -> 6.18 ms; 6000: 2.26 -> 1.10.
#pragma once

#include "rd_field.h"
#include "rd_fp64.h"
#include "rd_internal.h"

namespace rd {

constexpr int kRowT = 8;  // targets of a k_rows64 workgroup

// One chunk's terms, added in sequence from +0 (terms of +0 beyond the chunk's
// end leave the sum as it is: it is never -0).  One half is read while the
// other is added.
__device__ __forceinline__ double sum_chunk(const double* terms) {
  const double2* row = reinterpret_cast<const double2*>(terms);
  constexpr int H = 8, G = kChunk / (2 * H), D = 3;  // 16 terms a group, two groups in flight
  double v = 0.0;
  double2 r[D][H];
#pragma unroll
  for (int g = 0; g < D - 1; ++g)
#pragma unroll
    for (int k = 0; k < H; ++k) r[g][k] = row[g * H + k];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (g + D - 1 < G) {
#pragma unroll
      for (int k = 0; k < H; ++k) r[(g + D - 1) % D][k] = row[(g + D - 1) * H + k];
    }
#pragma unroll
    for (int k = 0; k < H; ++k) v = (v + r[g % D][k].x) + r[g % D][k].y;
    // keeps the reads in their place: all moved up, they would be spilled
    asm volatile("" : "+v"(v) : : "memory");
  }
  return v;
}

// k_accel64 (POINTS: k_field64) for few targets; the same partials.
template <int KIND, bool POINTS>
__global__ __launch_bounds__(kBlock, 3) void k_rows64(
    const Ent* tab, int ne, const SimDesc* desc, const SimState* st,
    const double* __restrict__ TX, const double* __restrict__ TY, const double* __restrict__ TZ,
    const double* __restrict__ X, const double* __restrict__ Y, const double* __restrict__ Z,
    const double* __restrict__ Q, const int32_t* __restrict__ SP, const double* __restrict__ img,
    double* __restrict__ part) {
  constexpr bool kTip = KIND == RD_GEOM_TIP;
  __shared__ __align__(16) double term[3 * kRowT][kChunk + 2];
  __shared__ double tgt[8][kRowT];  // x, y, z, charge factor; tip: image distance and point
  __shared__ int tsp[kRowT];
  __shared__ int s_surf;
  const Tile tl = tile_of(tab, ne, POINTS, kRowT);
  const Ent& e = tl.e;
  const int n = st[e.slot].n;
  const int targets = POINTS ? e.m : n;
  const int i0 = tl.bx * kRowT;
  if (i0 >= targets) return;
  const int nchunks = min((n + kChunk - 1) / kChunk, e.band1);
  const int c0 = e.band0 + tl.by * e.cps;
  if (c0 >= nchunks) return;
  const int c1 = min(nchunks, c0 + e.cps);
  const DevGeom g = desc[e.slot].g;
  if (g.kind != KIND) return;
  const int t = threadIdx.x;
  const int nt = min(kRowT, targets - i0);
  const bool tts = !POINTS && e.tts > 0;
  const size_t S = (size_t)e.pslots * (POINTS ? e.m : e.n_ub);
  const int ld = POINTS ? e.m : e.n_ub;
  double* P = part + e.part_off;
  bool ord = kTip || f64_ordinary(g.d);
  if (t == 0) s_surf = !kTip && g.ic;
  __syncthreads();
  if (t < nt) {
    const int gi = (POINTS ? e.pbase : e.base) + i0 + t;
    const double x = TX[gi], y = TY[gi], z = TZ[gi];
    tgt[0][t] = x;
    tgt[1][t] = y;
    tgt[2][t] = z;
    tgt[3][t] = POINTS ? g.dfc : Q[gi] * g.dfc;
    ord = ord && f64_ordinary(x) && f64_ordinary(y) && f64_ordinary(z);
    if (POINTS && z != 0.0) s_surf = 0;
    if (tts) tsp[t] = SP[gi];
    if (kTip && g.ic) {
      double da, xi, yi, zi;
      if (POINTS) {
        tip_image_point64(x, y, z, g.z0, g.R, da, xi, yi, zi);
      } else {
        da = img[4 * (size_t)gi];
        xi = img[4 * (size_t)gi + 1];
        yi = img[4 * (size_t)gi + 2];
        zi = img[4 * (size_t)gi + 3];
      }
      tgt[4][t] = da;
      tgt[5][t] = xi;
      tgt[6][t] = yi;
      tgt[7][t] = zi;
      ord = ord && f64_ordinary(da) && f64_ordinary(xi) && f64_ordinary(yi) && f64_ordinary(zi);
    }
  }
  for (int c = c0; c < c1; ++c) {
    const int j = c * kChunk + t;
    const bool in_n = j < n;
    const int gj = e.base + min(j, n - 1);
    const double x2 = X[gj], y2 = Y[gj], z2 = Z[gj], q2 = Q[gj];
    bool so = f64_ordinary(x2) && f64_ordinary(y2) && f64_ordinary(z2);
    double da2 = 0, xi2 = 0, yi2 = 0, zi2 = 0;
    if (!POINTS && kTip && g.ic) {
      da2 = img[4 * (size_t)gj];
      xi2 = img[4 * (size_t)gj + 1];
      yi2 = img[4 * (size_t)gj + 2];
      zi2 = img[4 * (size_t)gj + 3];
      so = so && f64_ordinary(da2) && f64_ordinary(xi2) && f64_ordinary(yi2) && f64_ordinary(zi2);
    }
    const int sp2 = tts ? SP[gj] : 0;
    const bool fast = __syncthreads_and(ord && so);
    auto terms = [&](auto m, auto on_cathode) {
      using M = decltype(m);
#pragma unroll 1
      for (int u = 0; u < nt; ++u) {
        const double x1 = tgt[0][u], y1 = tgt[1][u], z1 = tgt[2][u];
        const double pre = POINTS ? q2 * tgt[3][u] : tgt[3][u] * q2;
        const double dx = x1 - x2, dy = y1 - y2, dz = z1 - z2;
        const int i = i0 + u;
        bool first = POINTS || j > i;
        bool take = in_n;
        if (!POINTS) {
          take = take && j != i;
          if (tts) {
            TtsRole role;
            role.sp1 = tsp[u];
            role.ion_only_e = role.sp1 == RD_SPECIES_ION && (e.step % e.tts) != 0;
            take = tts_pair(role, i, j, sp2, first) && take;
          }
        }
        double ax, ay, az;
        if (decltype(on_cathode)::value) {
          surface_pair64<M, false>(g, pre, dx, dy, z2, ax, ay, az);
        } else if (!kTip) {
          planar_pair64<M>(g, pre, dx, dy, dz, first ? z1 : z2, first ? z2 : z1, ax, ay, az);
        } else {
          const double r2 = M::lift(dx * dx + dy * dy) + dz * dz;
          const double rt = M::sqrt(r2);
          const double r = rt + g.es;
          const double p0 = pre * M::rcp(r * r * r);
          ax = p0 * dx;
          ay = p0 * dy;
          az = p0 * dz;
          if (g.ic) {
            // the image is the first particle's, the offset first - second
            const double sg = first ? 1.0 : -1.0;
            double icx, icy, icz;
            tip_ic64<M>(sg * dx, sg * dy, sg * dz, r2, rt,
                        first ? tgt[5][u] - x2 : xi2 - x1, first ? tgt[6][u] - y2 : yi2 - y1,
                        first ? tgt[7][u] - z2 : zi2 - z1, first ? tgt[4][u] : da2, g.R, g.ktip,
                        icx, icy, icz);
            ax = ax + sg * pre * icx;
            ay = ay + sg * pre * icy;
            az = az + pre * icz;
          }
        }
        term[3 * u][t] = take ? ax : 0.0;
        term[3 * u + 1][t] = take ? ay : 0.0;
        term[3 * u + 2][t] = take ? az : 0.0;
      }
    };
    if (!fast)
      terms(Ieee64{}, std::false_type{});
    else if (POINTS && s_surf)
      terms(Fast64{}, std::bool_constant<POINTS && !kTip>{});
    else
      terms(Fast64{}, std::false_type{});
    __syncthreads();
    if (t < 3 * nt) P[(t % 3) * S + (size_t)(c - e.band0) * ld + i0 + t / 3] = sum_chunk(term[t]);
    // the next chunk's vote is the barrier between these sums and its terms
  }
}

// ---- pairs of chunks ------------------------------------------------------------

constexpr int kSymI = 8;  // rows of a tile

// The workgroups of an entry of nc chunks: first `both` pairs of chunks I < J,
// each for the particles of both; then quarters of a chunk's rows over one
// chunk, for the rows alone: the chunks over themselves and, both ways round,
// the pairs that are left.  The small ones even out the CUs at the launch's
// end: pairs beyond a multiple of the CUs are left where they are few, less than
// a third of a round (ten image terms, ms, all pairs once / some left: 12 000
// electrons, 57 pairs beyond 4 x 256: 3.85 / 3.52; 7000, 122 beyond 256: 1.57 / 1.74).
constexpr int kSymParts = 4;
constexpr int kSymRound = 256;
__host__ __device__ inline int sym_pairs(int nc) { return nc * (nc - 1) / 2; }
__host__ __device__ inline int sym_groups(int nc, int both) {
  return both + kSymParts * (nc + 2 * (sym_pairs(nc) - both));
}
struct SymTask {
  int I, J, part;  // part < 0: all rows, for both chunks
};
__device__ __forceinline__ SymTask sym_task(int local, int nc, int both) {
  SymTask s;
  int k = local;
  bool swap = false;
  s.part = -1;
  if (local >= both) {
    s.part = (local - both) % kSymParts;
    const int u = (local - both) / kSymParts;
    if (u < nc) {
      s.I = s.J = u;
      return s;
    }
    k = both + (u - nc) / 2;
    swap = (u - nc) & 1;
  }
  int J = (int)((sqrtf(8.0f * (float)k + 1.0f) + 1.0f) * 0.5f);  // J (J - 1) / 2 <= k
  while (J * (J + 1) / 2 <= k) ++J;
  while (J * (J - 1) / 2 > k) --J;
  const int I = k - J * (J - 1) / 2;
  s.I = swap ? J : I;
  s.J = swap ? I : J;
  return s;
}

// Accelerations, each pair of particles evaluated once.  The terms of the pair
// for its two particles differ in the charge product's rounding and in sign
// alone: the offsets are exact negations, and the image terms are those of the
// lower index for both.  A lane holds a particle of chunk J and adds its terms
// in the rows' order; the rows' terms go through LDS, kSymI rows at a time, to
// a lane per row and component.
template <int KIND>
__global__ __launch_bounds__(kBlock, 3) void k_accel64sym(
    const Ent* tab, int ne, const SimDesc* desc, const SimState* st, const double* __restrict__ X,
    const double* __restrict__ Y, const double* __restrict__ Z, const double* __restrict__ Q,
    const double* __restrict__ img, double* __restrict__ part) {
  constexpr bool kTip = KIND == RD_GEOM_TIP;
  __shared__ __align__(16) double term[3 * kSymI][kChunk + 2];
  const Ent& e = tab[find_entry(tab, ne, blockIdx.x, true)];
  const int n = st[e.slot].n;
  const SymTask task = sym_task(blockIdx.x - e.wg1, e.nchunks_ub, e.segs);
  const int I = task.I, J = task.J;
  if (max(I, J) * kChunk >= n) return;
  const DevGeom g = desc[e.slot].g;
  if (g.kind != KIND) return;
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool both = task.part < 0;
  const double* x = X + e.base;
  const double* y = Y + e.base;
  const double* z = Z + e.base;
  const double* q = Q + e.base;
  const double* im = img + 4 * (size_t)e.base;
  const int n_ub = e.n_ub;
  const size_t S = (size_t)e.pslots * n_ub;
  double* P = part + e.part_off;
  const int i0 = I * kChunk, cnti = min(kChunk, n - i0);
  const int r0 = both ? 0 : task.part * (kChunk / kSymParts);
  const int r1 = both ? cnti : min(cnti, r0 + kChunk / kSymParts);
  if (r0 >= r1) return;
  const int j = J * kChunk + t;
  const bool in_n = j < n;
  const int jc = min(j, n - 1);
  const double x2 = x[jc], y2 = y[jc], z2 = z[jc], q2 = q[jc], qd2 = q2 * g.dfc;
  double da2 = 0, xi2 = 0, yi2 = 0, zi2 = 0;
  bool ord = (kTip || f64_ordinary(g.d)) && f64_ordinary(x2) && f64_ordinary(y2) && f64_ordinary(z2);
  {
    const int k = min(i0 + t, n - 1);
    ord = ord && f64_ordinary(x[k]) && f64_ordinary(y[k]) && f64_ordinary(z[k]);
    if (kTip && g.ic) {
      for (int v = 0; v < 4; ++v) ord = ord && f64_ordinary(im[4 * (size_t)k + v]);
      da2 = im[4 * (size_t)jc];
      xi2 = im[4 * (size_t)jc + 1];
      yi2 = im[4 * (size_t)jc + 2];
      zi2 = im[4 * (size_t)jc + 3];
      ord = ord && f64_ordinary(da2) && f64_ordinary(xi2) && f64_ordinary(yi2) && f64_ordinary(zi2);
    }
  }
  const bool fast = __syncthreads_and(ord);
  double cx = 0.0, cy = 0.0, cz = 0.0;  // the column's sums
  // a row's values are uniform and go through the scalar cache, one row ahead
  double xn = x[i0 + r0], yn = y[i0 + r0], zn = z[i0 + r0], qn = q[i0 + r0];
  auto rows = [&](auto m) {
    using M = decltype(m);
#pragma unroll 1
    for (int ib = r0; ib < r1; ib += kSymI) {
#pragma unroll 2
      for (int r = 0; r < kSymI; ++r) {
        const int i = i0 + ib + r;
        const double x1 = xn, y1 = yn, z1 = zn, q1 = qn;
        const int in = min(i + 1, n - 1);
        xn = x[in];
        yn = y[in];
        zn = z[in];
        qn = q[in];
        const bool first = j > i;
        const bool take = in_n && i < n && j != i;
        const double dx = x1 - x2, dy = y1 - y2, dz = z1 - z2;
        const double pre = (q1 * g.dfc) * q2;  // at the row's particle
        double i3, fx, fy, fz;  // direct and image factors of the charge products
        if (!kTip) {
          planar_series64<M>(g, dx, dy, dz, first ? z1 : z2, first ? z2 : z1, i3, fx, fy, fz);
        } else {
          const double r2 = M::lift(dx * dx + dy * dy) + dz * dz;
          const double rt = M::sqrt(r2);
          const double rd = rt + g.es;
          i3 = M::rcp(rd * rd * rd);
          if (g.ic) {
            const double sg = first ? 1.0 : -1.0;
            const size_t o = 4 * (size_t)min(i, n - 1);
            const double da1 = im[o], xi1 = im[o + 1], yi1 = im[o + 2], zi1 = im[o + 3];
            tip_ic64<M>(sg * dx, sg * dy, sg * dz, r2, rt, first ? xi1 - x2 : xi2 - x1,
                        first ? yi1 - y2 : yi2 - y1, first ? zi1 - z2 : zi2 - z1,
                        first ? da1 : da2, g.R, g.ktip, fx, fy, fz);
            fx = sg * fx;
            fy = sg * fy;
          }
        }
        const double p0 = pre * i3;
        double ax = p0 * dx, ay = p0 * dy, az = p0 * dz;
        if (g.ic) {
          ax = ax + pre * fx;
          ay = ay + pre * fy;
          az = az + pre * fz;
        }
        term[3 * r][t] = take ? ax : 0.0;
        term[3 * r + 1][t] = take ? ay : 0.0;
        term[3 * r + 2][t] = take ? az : 0.0;
        if (both) {  // I < J: every row is a particle, only the last chunk is ragged
          const double pre2 = qd2 * q1, p2 = pre2 * i3;  // at the column's particle
          ax = p2 * -dx;
          ay = p2 * -dy;
          az = p2 * -dz;
          if (g.ic) {
            ax = ax - pre2 * fx;
            ay = ay - pre2 * fy;
            az = az + pre2 * fz;
          }
          cx = cx + ax;
          cy = cy + ay;
          cz = cz + az;
        }
      }
      __syncthreads();
      // one wavefront adds the rows' terms, the next one those of the next tile
      if (wv == ((ib / kSymI) & 3) && lane < 3 * min(kSymI, r1 - ib))
        P[(lane % 3) * S + (size_t)J * n_ub + i0 + ib + lane / 3] = sum_chunk(term[lane]);
      __syncthreads();
    }
  };
  if (fast)
    rows(Fast64{});
  else
    rows(Ieee64{});
  if (both && in_n) {
    const size_t o = (size_t)I * n_ub + j;
    P[o] = cx;
    P[S + o] = cy;
    P[2 * S + o] = cz;
  }
}

}  // namespace rd
