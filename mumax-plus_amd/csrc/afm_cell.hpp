// The two sublattices of an antiferromagnet with uniform parameters: field and
// torque of one cell of both.
//
// The general sublattice kernel evaluates one sublattice per thread with every
// rule of the reference (per-cell parameters, masks, regions, open boundaries):
// some 1500 vector instructions a cell, most of them address arithmetic,
// divisions and rules that a uniform magnet does not need, and each
// sublattice's thread loads the neighbours of both.  Here one thread does both
// sublattices of a cell from one set of loads, all divisions are folded into
// host-side coefficients, and missing neighbours (free boundaries) are a
// branch that only boundary cells take.  A single layer with free surfaces
// needs no z neighbours: its two exchange terms cancel and its two DMI terms
// are the same linear form of the boundary vector.
#pragma once

#include "field_cell.hpp"

namespace mpa {

// Coefficients of one sublattice (s: sister).
struct AfmUniform {
  float kex[3];    // 2 A / (Ms c^2)
  float knn[3];    // A_nn / (Ms_s c^2)
  float kd[3][3];  // own DMI (xy, xz, yz) of each axis / (Ms c)
  float ki[3][3];  // inter-sublattice DMI / (Ms c)
  float D[D_COUNT];  // own tensor (J/m2), for the boundary vector
  float cz[3];     // cell sizes
  float ic[3];     // 1 / cell size
  float h2a, an;   // 1 / (2 A), A_nn
  float site;      // 4 A_c / (a^2 Ms_s)
  float u[3], ku1, ku2;  // 2 K1 / Ms, 4 K2 / Ms
  float hext[3];
  float b1, b2;    // -2 B / Ms
  float alpha;
};

struct AfmPair {
  int nx, ny, nz, ncell;
  int ox, oy, oz, mgx, mgy, mgz, mox, moy, moz;
  AfmUniform c[2];
  const float* m[2];
  const float* hd;      // demag field of both, nullptr without
  const float* strain;  // 6 N, nullptr without dynamic strain
  float rigid[6];       // uniform applied strain (me_rigid)
  int ex, dmi, nn, uni, me, flatz;
};

__device__ __forceinline__ float3 afm_dmi(const float (&k)[3], float3 v) {
  return f3(k[0] * v.y + k[1] * v.z, -k[0] * v.x + k[2] * v.z, -k[1] * v.x - k[2] * v.y);
}
// the reference's inter-sublattice form (dmi.cu:229-231), as subtracted
__device__ __forceinline__ float3 afm_inter(const float (&k)[3], float3 v) {
  return f3(-k[0] * v.y + k[1] * v.z, k[0] * v.x + k[2] * v.z, k[1] * v.x - k[2] * v.y);
}

// Adds the exchange, DMI and neighbour terms of the pair of directions -/+ of
// `axis` to h (one sublattice: m its value, s the sister's; mn, sn at the
// neighbours, ok whether they exist).
__device__ __forceinline__ void afm_axis(const AfmPair& P, const AfmUniform& c, int axis, float3 m, float3 s,
                                         const float3 (&mn)[2], const float3 (&sn)[2], const bool (&ok)[2],
                                         float3& hex, float3& hdm, float3& hnn) {
  float3 me[2] = {mn[0], mn[1]}, sd[2] = {sn[0], sn[1]}, se[2] = {sn[0], sn[1]};
  if (!(ok[0] && ok[1])) {
    // Neumann boundary with the DMI term and the sister's normal derivative on
    // the bulk side (exchange.cu:176-189, dmi.cu:200-222, afmexchange.cu:122-132)
    const float3 g1 = dmi_gamma(c.D, axis, m), g2 = dmi_gamma(c.D, axis, s);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (ok[k]) continue;
      const float delta = k ? c.cz[axis] : -c.cz[axis], idelta = k ? c.ic[axis] : -c.ic[axis];
      const float3 zero = f3(0.f, 0.f, 0.f);
      const float3 ds = ok[k ^ 1] ? idelta * (s - sn[k ^ 1]) : zero;
      const float3 dm = ok[k ^ 1] ? idelta * (m - mn[k ^ 1]) : zero;
      me[k] = m + (delta * c.h2a) * (c.an * cross3(cross3(ds, m), m) + g1);
      sd[k] = s + (delta * c.h2a) * (c.an * cross3(cross3(idelta * (me[k] - m), s), s) + g2);
      se[k] = s + (delta * c.h2a) * (c.an * cross3(cross3(dm, s), s) + g2);
    }
  }
  if (P.ex) hex = hex + c.kex[axis] * (me[0] + me[1] - 2.f * m);
  if (P.dmi) hdm = hdm + afm_dmi(c.kd[axis], me[1] - me[0]) + afm_inter(c.ki[axis], sd[1] - sd[0]);
  if (P.nn) hnn = hnn + c.knn[axis] * (se[0] + se[1] - 2.f * s);
}

// Field of one sublattice at cell idx.
__device__ __forceinline__ float3 afm_field(const AfmPair& P, const AfmUniform& c, float3 m, float3 s,
                                            const float3 (&mn)[6], const float3 (&sn)[6], const bool (&ok)[6],
                                            const float (&e)[6], float3 hd) {
  float3 hex = f3(0.f, 0.f, 0.f), hdm = hex, hnn = hex;
#pragma unroll
  for (int axis = 0; axis < 3; ++axis) {
    if (axis == 2 && P.flatz) {
      if (P.dmi) {
        // free surfaces above and below: m +- c/(2A) X, their difference alone
        const float3 g1 = c.h2a * dmi_gamma(c.D, 2, m);
        const float3 x2 = c.h2a * (c.an * cross3(cross3(g1, s), s) + dmi_gamma(c.D, 2, s));
        hdm = hdm + (2.f * c.cz[2]) * (afm_dmi(c.kd[2], g1) + afm_inter(c.ki[2], x2));
      }
      continue;
    }
    const float3 a[2] = {mn[2 * axis], mn[2 * axis + 1]}, b[2] = {sn[2 * axis], sn[2 * axis + 1]};
    const bool o[2] = {ok[2 * axis], ok[2 * axis + 1]};
    afm_axis(P, c, axis, m, s, a, b, o, hex, hdm, hnn);
  }
  float3 h = hex;
  if (P.uni) {
    const float3 u = f3(c.u[0], c.u[1], c.u[2]);
    const float mu = dot3(m, u);
    h = h + (c.ku1 * mu + c.ku2 * mu * mu * mu) * u;
  }
  h = h + f3(c.hext[0], c.hext[1], c.hext[2]);
  h = h + hdm;
  if (P.me)
    h = h + f3(c.b1 * e[0] * m.x + c.b2 * (e[3] * m.y + e[4] * m.z), c.b1 * e[1] * m.y + c.b2 * (e[5] * m.z + e[3] * m.x),
               c.b1 * e[2] * m.z + c.b2 * (e[4] * m.x + e[5] * m.y));
  h = h + hnn;
  h = h + c.site * s;
  return h + hd;  // last, so that a field without demag plus the demag field is this sum
}

}  // namespace mpa
