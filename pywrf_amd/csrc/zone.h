// The specified-zone updates of an acoustic substep (pywrf/wrf_boundary.py:188-405)
// as device functions of one point with their host-side setup, shared by the
// zone kernels and by the acoustic kernels that apply them to what they write.
#pragma once
#include "common.h"

#define ZONE_AT(p, k, j, i) at_b((p), D.ob((k), (j), (i)))
#define ZONE_AT2(p, j, i) at_b((p), D.ob2((j), (i)))

// staggering of the relax/spec routines (wrf_boundary.py:_bounds logic)
static inline void bounds_of(char v, const pywrf_grid_t* g, int& ibe, int& jbe, int& ktf) {
  ibe = g->ide - 1;
  jbe = g->jde - 1;
  ktf = g->kde - 1;
  if (v == 'u') ibe = g->ide;
  if (v == 'v') jbe = g->jde;
  if (v == 'm' || v == 'h') ktf = g->kte;
}

// ---------------------------------------------------------------- spec_bdyupdate
struct UpdJob {
  Box all;
  Dims D;
  float* f;
  const float* t;
  float dt;
  int jts, jtf, its, itf, jbs, jbe;
};

// how many of the reference's statements update (j, i): the start and end rows and columns
__device__ inline int spec_upd_times(const UpdJob& b, int j, int i) {
  bool ic = i >= b.its && i < b.itf, jc = j >= b.jbs + 1 && j < b.jbe - 1;
  return (j == b.jts && ic) + (j == b.jtf - 1 && ic) + (i == b.its && jc) + (i == b.itf - 1 && jc);
}

// the value v of point (k, j, i), tendency tv, after the update (v itself outside the zone)
__device__ inline float spec_upd_value(const UpdJob& b, int k, int j, int i, float v, float tv) {
  const int n = b.all.has(k, j, i) ? spec_upd_times(b, j, i) : 0;
  for (int m = 0; m < n; ++m) v = v + b.dt * tv;
  return v;
}

__device__ inline void spec_upd_point(const UpdJob& b, int k, int j, int i) {
  const Dims& D = b.D;
  const int n = spec_upd_times(b, j, i);
  if (!n) return;
  long q = D.ix(k, j, i);
  float v = b.f[q], tv = b.t[q];
  for (int m = 0; m < n; ++m) v = v + b.dt * tv;
  b.f[q] = v;
}

// Host side of spec_bdyupdate: the job and its edge-band width (1 when the
// updated rows jts, jtf-1 and columns its, itf-1 are the box's sides, else 0).
static inline int spec_upd_job(const pywrf_grid_t* g, float* field, const float* field_tend, double dt, char variable,
                        UpdJob& b, int& w) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  char v = variable;
  if (v == 'U') v = 'u'; else if (v == 'V') v = 'v'; else if (v == 'M') v = 'm'; else if (v == 'H') v = 'h';
  int itf = imin(g->ite, g->ide - 1), jtf = imin(g->jte, g->jde - 1), ktf = g->kde - 1, jbe = g->jde - 1;
  if (v == 'u') itf = imin(g->ite, g->ide);
  if (v == 'v') { jbe = g->jde; jtf = imin(g->jte, g->jde); }
  if (v == 'm' || v == 'h') ktf = g->kte;
  int nz = g->nz;
  if (g->kds == 0 && g->kde == 0) { ktf = 1; nz = 1; }  // 2-D field (the reference's unsqueeze path)
  if (itf > g->nx || jbe > g->ny || jtf > g->ny || ktf > nz || g->its < 0 || g->jts < 0) return PYWRF_E_RANGE;
  pywrf_grid_t g2 = *g;
  g2.nz = nz;
  b.all = mkbox(g->kts, ktf, imin(g->jts, g->jds), imax(jtf, jbe), g->its, itf);
  b.D = dims_of(&g2);
  b.f = field; b.t = field_tend; b.dt = F(dt);
  b.jts = g->jts; b.jtf = jtf; b.its = g->its; b.itf = itf; b.jbs = g->jds; b.jbe = jbe;
  w = (g->jts == b.all.j0 && jtf == b.all.j1) ? 1 : 0;
  return 0;
}

// Whether the job's updated points are the ring around a box that lies inside it,
// so that a kernel that computes the box can update the ring as it passes the
// other points through.
static inline bool spec_upd_rings(const UpdJob& b, const Box& in) {
  return in.j0 > b.jts && in.j1 <= b.jtf - 1 && in.i0 > b.its && in.i1 <= b.itf - 1;
}

// ---------------------------------------------------------------- spec_bdyupdate_ph
struct PhStrip {
  Box all;
  int w;
  const float *ph_save, *ft, *mu_tend, *muts;
  float* f;
  float dt;
  int jts, ibs, ibe, jbs, jbe;
};

__device__ inline void ph_strip_point(const Dims& D, const PhStrip& a, int k, int j, int i) {
  bool ir = i >= a.ibs && i < a.ibe, jc = j >= a.jbs + 1 && j < a.jbe - 1;
  int n = (j == a.jts && ir) + (j == a.jbe - 1 && ir) + (i == a.ibs && jc) + (i == a.ibe - 1 && jc);
  if (!n) return;
  long q = D.ix(k, j, i);
  float mt = ZONE_AT2(a.muts, j, i);
  float mo = mt - a.dt * ZONE_AT2(a.mu_tend, j, i);
  float v = a.f[q];
  for (int m = 0; m < n; ++m) v = v * mo / mt + a.dt * a.ft[q] / mt + a.ph_save[q] * (mo / mt - 1.0f);
  a.f[q] = v;
}

static inline int ph_strip_setup(const pywrf_grid_t* g, const float* ph_save, float* field, const float* field_tend,
                          const float* mu_tend, const float* muts, double dt, char variable_in, PhStrip& a) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  char v = variable_in;
  if (v == 'U') v = 'u'; else if (v == 'V') v = 'v'; else if (v == 'M') v = 'm'; else if (v == 'H') v = 'h';
  int ibe, jbe, ktf;
  bounds_of(v, g, ibe, jbe, ktf);
  if (ibe > g->nx || jbe > g->ny || ktf > g->nz || g->ids < 0 || g->jds < 0) return PYWRF_E_RANGE;
  a.all = mkbox(g->kts, ktf, imin(g->jts, g->jds), imax(jbe, g->jts + 1), g->ids, ibe);
  a.w = (g->jts == a.all.j0 && jbe == a.all.j1) ? 1 : 0;
  a.ph_save = ph_save; a.f = field; a.ft = field_tend; a.mu_tend = mu_tend; a.muts = muts; a.dt = F(dt);
  a.jts = g->jts; a.ibs = g->ids; a.ibe = ibe; a.jbs = g->jds; a.jbe = jbe;
  return 0;
}

// ---------------------------------------------------------------- zero_grad_bdy
struct ZgStrip {
  Box all;
  float* f;
  int ibs, ibe, jbs, jbe;
};

__device__ inline void zero_grad_point(const Dims& D, const ZgStrip& a, int k, int j, int i) {
  bool ring = (j == a.jbs || j == a.jbe - 1) || (i == a.ibs || i == a.ibe - 1);
  if (!ring) return;
  int sj = j < a.jbs + 1 ? a.jbs + 1 : (j > a.jbe - 2 ? a.jbe - 2 : j);
  int si = i < a.ibs + 1 ? a.ibs + 1 : (i > a.ibe - 2 ? a.ibe - 2 : i);
  ZONE_AT(a.f, k, j, i) = ZONE_AT(a.f, k, sj, si);
}

static inline int zero_grad_setup(const pywrf_grid_t* g, float* field, char variable_in, ZgStrip& a) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  char v = variable_in;
  if (v == 'U') v = 'u'; else if (v == 'V') v = 'v';
  int ibe = g->ide - 1, jbe = g->jde - 1, ktf = g->kde - 1;
  if (v == 'u') ibe = g->ide;
  if (v == 'v') jbe = g->jde;
  if (v == 'w') ktf = g->kde;
  if (ibe > g->nx || jbe > g->ny || ktf > g->nz || g->ids < 0 || g->jds < 0) return PYWRF_E_RANGE;
  a.all = mkbox(g->kts, ktf, g->jds, jbe, g->ids, ibe);
  a.f = field; a.ibs = g->ids; a.ibe = ibe; a.jbs = g->jds; a.jbe = jbe;
  return 0;
}
