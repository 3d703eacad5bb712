// Acoustic small-step machinery (pywrf/wrf_dynamics.py:3152-3930):
// small_step_prep, calc_p_rho, calc_coef_w, advance_uv, advance_mu_t,
// advance_w, sumflux, calc_mu_uv_1, small_step_finish.
//
// Where the reference clones an argument and updates a box of the clone, the
// kernel writes the whole output array (box points computed, the rest copied)
// in the same pass.  Column recurrences (eta velocity, Thomas solve) run one
// thread per (j, i) column with k marching; the output buffer doubles as the
// column scratch, so no full-grid temporaries are allocated.
#include "common.h"

#ifndef PW_COL_XCD
#define PW_COL_XCD 1
#endif
#include "consts.h"
#include "openbc.h"
#include "zone.h"

#define AT(p, k, j, i) at_b((p), D.ob((k), (j), (i)))
#define AT2(p, j, i) at_b((p), D.ob2((j), (i)))

int pw_check_grid(const pywrf_grid_t* g, int r);
#define CHECK(g, r) do { int _e = pw_check_grid((g), (r)); if (_e) return _e; } while (0)

static Box plane(const pywrf_grid_t* g) { return mkbox(0, 1, 0, g->ny, 0, g->nx); }

// ------------------------------------------------------------------ small_step_prep
struct SsPrep2 {
  const float *mub, *muu, *muv;
  float *mu_1, *mu_2, *muus, *muvs, *muts, *mudf, *mu_save;
  int rk1, j0, j1, i0, i1, i1u, j1v;
};

__global__ void k_ssprep_2d(Box b, Dims D, SsPrep2 a) {
  int j, i;
  if (!box_column(b, j, i)) return;
  bool h = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  bool hu = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1u;
  long q = D.ix2(j, i);
  if (a.rk1) {
    bool hv = j >= a.j0 && j < a.j1v && i >= a.i0 && i < a.i1;
    float m2 = a.mu_2[q];
    if (h) {
      a.mu_1[q] = m2 + 0.0f;
      a.mudf[q] = 0.0f;
      a.muts[q] = a.mub[q] + m2;
      a.mu_save[q] = m2 + 0.0f;
      a.mu_2[q] = 0.0f;
    }
    if (hu) a.muus[q] = a.muu[q] + 0.0f;
    if (hv) a.muvs[q] = a.muv[q] + 0.0f;
  } else {
    bool hv = j >= a.j0 && j < a.j1v && i >= a.i0 && i < a.i1u;  // i-range i1u as in the reference
    if (h) a.muts[q] = a.mub[q] + a.mu_1[q];
    if (hu) a.muus[q] = 0.5f * (a.mub[q] + a.mu_1[q] + AT2(a.mub, j, i - 1) + AT2(a.mu_1, j, i - 1));
    if (hv) a.muvs[q] = 0.5f * (a.mub[q] + a.mu_1[q] + AT2(a.mub, j - 1, i) + AT2(a.mu_1, j - 1, i));
    if (h) {
      float m2 = a.mu_2[q];
      a.mu_save[q] = m2 + 0.0f;
      a.mu_2[q] = a.mu_1[q] - m2;
    }
  }
}

struct SsPrep3 {
  float *u_1, *v_1, *w_1, *t_1, *ph_1;
  const float *u_2, *v_2, *w_2, *t_2, *ph_2;
  float *u_save, *v_save, *w_save, *t_save, *ph_save, *ww_save, *c2a;
  const float *ww, *pb, *p, *alt, *muu, *muus, *muv, *muvs, *mut, *muts, *msfuy, *msfvx_inv, *msfty;
  float *u_out, *v_out, *w_out, *t_out, *ph_out;
  int rk1, k1, kde, j0, j1, i0, i1, i1u, j1v;
};

__global__ void k_ssprep_3d(Box all, Dims D, SsPrep3 a) {
  int k, j, i;
  if (!box_point(all, k, j, i)) return;
  long q = D.ix(k, j, i);
  long q2 = D.ix2(j, i);
  bool hcol = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  bool bm = k < a.k1 && hcol;
  bool bu = k < a.k1 && j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1u;
  bool bv = k < a.k1 && j >= a.j0 && j < a.j1v && i >= a.i0 && i < a.i1;
  bool bw = k < a.kde && hcol;
  // every value is formed first and stored last, so that no load waits on a
  // store, and every operand (all at this point) is loaded before the
  // branches, so that no branch waits on its loads
  const float u2 = a.u_2[q], v2 = a.v_2[q], t2 = a.t_2[q], w2 = a.w_2[q], p2 = a.ph_2[q];
  // the *_1 fields are read only past the first stage (rk1 is uniform)
  const float u1l = a.rk1 ? 0.0f : a.u_1[q], v1l = a.rk1 ? 0.0f : a.v_1[q], t1l = a.rk1 ? 0.0f : a.t_1[q];
  const float w1l = a.rk1 ? 0.0f : a.w_1[q], p1l = a.rk1 ? 0.0f : a.ph_1[q];
  const float pbq = a.pb[q], pq = a.p[q], altq = a.alt[q], wwq = a.ww[q];
  const float muus = a.muus[q2], muu = a.muu[q2], msfuy = a.msfuy[q2], muvs = a.muvs[q2], muv = a.muv[q2];
  const float msfvx_inv = a.msfvx_inv[q2], muts = a.muts[q2], mut = a.mut[q2], msfty = a.msfty[q2];
  float uo = u2, u1 = 0.0f;
  if (bu) {
    u1 = a.rk1 ? u2 + 0.0f : u1l;
    uo = (muus * u1 - muu * u2) / msfuy;
  }
  float vo = v2, v1 = 0.0f;
  if (bv) {
    v1 = a.rk1 ? v2 + 0.0f : v1l;
    vo = (muvs * v1 - muv * v2) * msfvx_inv;
  }
  float to = t2, t1 = 0.0f, c2 = 0.0f;
  if (bm) {
    t1 = a.rk1 ? t2 + 0.0f : t1l;
    c2 = F(pw::cpovcv) * (pbq + pq) / altq;
    to = muts * t1 - mut * t2;
  }
  float wo = w2, po = p2, w1 = 0.0f, p1 = 0.0f, wws = 0.0f;
  const bool wwz = !bw && hcol && (k == 0 || k == a.kde - 1);
  if (bw) {
    w1 = a.rk1 ? w2 + 0.0f : w1l;
    p1 = a.rk1 ? p2 + 0.0f : p1l;
    wo = (muts * w1 - mut * w2) / msfty;
    po = p1 - p2;
    wws = wwq;
  }
  if (bu) {
    if (a.rk1) a.u_1[q] = u1;
    a.u_save[q] = u2 + 0.0f;
  }
  a.u_out[q] = uo;
  if (bv) {
    if (a.rk1) a.v_1[q] = v1;
    a.v_save[q] = v2 + 0.0f;
  }
  a.v_out[q] = vo;
  if (bm) {
    if (a.rk1) a.t_1[q] = t1;
    a.c2a[q] = c2;
    a.t_save[q] = t2 + 0.0f;
  }
  a.t_out[q] = to;
  if (bw) {
    if (a.rk1) {
      a.w_1[q] = w1;
      a.ph_1[q] = p1;
    }
    a.w_save[q] = w2 + 0.0f;
    a.ph_save[q] = p2 + 0.0f;
    a.ww_save[q] = wws;
  } else if (wwz) {
    a.ww_save[q] = 0.0f;
  }
  a.w_out[q] = wo;
  a.ph_out[q] = po;
}

extern "C" int pywrf_small_step_prep(const pywrf_grid_t* g, float* u_1, const float* u_2, float* v_1,
                                     const float* v_2, float* w_1, const float* w_2, float* t_1, const float* t_2,
                                     float* ph_1, const float* ph_2, const float* mub, float* mu_1, float* mu_2,
                                     const float* muu, float* muus, const float* muv, float* muvs, const float* mut,
                                     float* muts, float* mudf, float* u_save, float* v_save, float* w_save,
                                     float* t_save, float* ph_save, float* mu_save, const float* ww,
                                     float* ww_save, float* c2a, const float* pb, const float* p, const float* alt,
                                     const float* msfuy, const float* msfvx_inv, const float* msfty, int rk_step,
                                     float* u_out, float* v_out, float* w_out, float* t_out, float* ph_out,
                                     pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kde > g->nz || g->kts != 0) return PYWRF_E_RANGE;
  int j0 = g->jts, j1 = imin(g->jte, g->jde - 1), i0 = g->its, i1 = imin(g->ite, g->ide - 1);
  int k1 = imin(g->kte, g->kde - 1), i1u = g->ite, j1v = g->jte;
  SsPrep2 a2 = {mub, muu, muv, mu_1, mu_2, muus, muvs, muts, mudf, mu_save, rk_step == 1, j0, j1, i0, i1, i1u, j1v};
  Dims D = dims_of(g);
  Box b2 = mkbox(0, 1, j0, imax(j1, j1v), i0, imax(i1, i1u));
  PW_LAUNCH_COLS(k_ssprep_2d, b2, s, D, a2);
  SsPrep3 a3 = {u_1, v_1, w_1, t_1, ph_1, u_2, v_2, w_2, t_2, ph_2, u_save, v_save, w_save, t_save, ph_save,
                ww_save, c2a, ww, pb, p, alt, muu, muus, muv, muvs, mut, muts, msfuy, msfvx_inv, msfty,
                u_out, v_out, w_out, t_out, ph_out, rk_step == 1, k1, g->kde, j0, j1, i0, i1, i1u, j1v};
  PW_LAUNCH_BOX(k_ssprep_3d, whole(g), s, D, a3);
  PW_RET();
}

// ------------------------------------------------------------------ calc_p_rho
struct PRho {
  const float *al_in, *p_in, *ph, *alt, *t_2, *t_1, *c2a, *mu, *mut, *rdnw;
  float *al, *p, *pm1;
  float t0, smdiv;
  int step;
  const float* pm_in;   // pm1 on entry, where it is not updated in place
};

__global__ void k_calc_p_rho(Box all, Dims D, Box b, PRho a) {
  int k, j, i;
  if (!box_point(all, k, j, i)) return;
  long q = D.ix(k, j, i);
  // the box's operands are loaded before the branch (a load under a branch is
  // waited for before the branch ends); the level above is clamped into the
  // array, its value being used only inside the box, where k + 1 is a level.
  // The incoming al and p are read only outside the box (a wave inside it
  // skips them as one), pm1 only past step 0 (uniform)
  const bool in = b.has(k, j, i);
  const float al_in = in ? 0.0f : a.al_in[q], p_in = in ? 0.0f : a.p_in[q];
  const float ph0 = a.ph[q], ph1 = AT(a.ph, imin(k + 1, D.nz - 1), j, i);
  const float altq = a.alt[q], t1 = a.t_1[q], t2 = a.t_2[q], c2 = a.c2a[q], pm = a.step != 0 ? a.pm1[q] : 0.0f;
  const float mut = AT2(a.mut, j, i), mu = AT2(a.mu, j, i), rd = a.rdnw[k];
  float al = al_in, p = p_in, pmo = 0.0f;
  if (in) {
    al = -1.0f / mut * (altq * mu + rd * (ph1 - ph0));
    p = c2 * (altq * (t2 - mu * t1) / (mut * (a.t0 + t1)) - al);
    if (a.step != 0) {
      pmo = p + 0.0f;
      p = p + a.smdiv * (p - pm);
    }
  }
  a.al[q] = al;
  a.p[q] = p;
  if (a.step == 0) a.pm1[q] = p + 0.0f;
  else if (in) a.pm1[q] = pmo;
}

extern "C" int pywrf_calc_p_rho(const pywrf_grid_t* g, const float* al_in, const float* p_in, const float* ph,
                                const float* alt, const float* t_2, const float* t_1, const float* c2a, float* pm1,
                                const float* mu, const float* mut, double t0, const float* rdnw, double smdiv,
                                int step, float* al_out, float* p_out, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  Box b = mkbox(g->kts, imin(g->kte, g->kde - 1), g->jts, imin(g->jte, g->jde - 1), g->its,
                imin(g->ite, g->ide - 1));
  if (b.k1 + 1 > g->nz) return PYWRF_E_RANGE;
  PRho a = {al_in, p_in, ph, alt, t_2, t_1, c2a, mu, mut, rdnw, al_out, p_out, pm1, F(t0), F(smdiv), step, pm1};
  PW_LAUNCH_BOX(k_calc_p_rho, whole(g), s, dims_of(g), b, a);
  PW_RET();
}

// calc_p_rho past step 0 and the open-boundary fills that follow it in a
// substep, of al, p, ph, muts, mu and mudf.  A halo cell of al and p is formed
// from the operands of the cell its fill copies; the fills of the others
// (whose halos the formula reads nowhere) are the first blocks.  us at
// 240 x 240 x 41 and 40 x 40 x 41: 24.7 and 4.9, against 28.1 and 8.3 in two launches.
struct PRhoBc {
  PRho r;
  Box b;
  BcSpec c;                        // al's and p's fill, on levels [k0, k1)
  int k0, k1;
  BcJob job[4];                    // ph, muts, mu, mudf
  int nph, nfill, ntx, nty;        // ph's blocks, all fills'; tiles along i and j
};
#define PB_ROWS (BC_THREADS / PW_TX)

__global__ void __launch_bounds__(BC_THREADS) k_calc_p_rho_bc(Dims D, PRhoBc a) {
  if ((int)blockIdx.x < a.nfill) {
    const int t = (int)blockIdx.x;
    const BcJob& f = a.job[t < a.nph ? 0 : t - a.nph + 1];
    open_bc_plane(f.p + (long)(f.k0 + (t < a.nph ? t : 0)) * D.plane(), D.nx, f.c);
    return;
  }
  const int t = (int)blockIdx.x - a.nfill;
  const int i = t % a.ntx * PW_TX + (int)threadIdx.x % PW_TX, j = t / a.ntx % a.nty * PB_ROWS + (int)threadIdx.x / PW_TX,
            k = t / a.ntx / a.nty;
  if (i >= D.nx || j >= D.ny) return;
  int js = j, is = i;
  if (k >= a.k0 && k < a.k1) open_bc_source(a.c, js, is);
  const PRho& r = a.r;
  const long q = D.ix(k, j, i), qs = D.ix(k, js, is);
  const bool in = a.b.has(k, js, is), own = a.b.has(k, j, i);
  const float al_in = in ? 0.0f : r.al_in[qs], p_in = in ? 0.0f : r.p_in[qs];
  const float ph0 = r.ph[qs], ph1 = AT(r.ph, imin(k + 1, D.nz - 1), js, is);
  const float altq = r.alt[qs], t1 = r.t_1[qs], t2 = r.t_2[qs], c2 = r.c2a[qs];
  const float pm = r.pm_in[qs];
  const float mut = AT2(r.mut, js, is), mu = AT2(r.mu, js, is), rd = r.rdnw[k];
  float al = al_in, p = p_in, pmo = 0.0f;
  if (in) {
    al = -1.0f / mut * (altq * mu + rd * (ph1 - ph0));
    p = c2 * (altq * (t2 - mu * t1) / (mut * (r.t0 + t1)) - al);
    pmo = p + 0.0f;
    p = p + r.smdiv * (p - pm);
  }
  r.al[q] = al;
  r.p[q] = p;
  r.pm1[q] = own ? pmo : r.pm_in[q];
}

extern "C" int pywrf_calc_p_rho_bc(const pywrf_grid_t* g, const pywrf_grid_t* g3, const pywrf_grid_t* g2,
                                   const float* al_in, const float* p_in, float* ph, const float* alt, const float* t_2,
                                   const float* t_1, const float* c2a, const float* pm1_in, float* mu, float* mut, double t0,
                                   const float* rdnw, double smdiv, int step, float* mudf, const char* variables,
                                   float* al_out, float* p_out, float* pm1_out, pywrf_stream_t s) {
  if (!pw_size_ok(g) || !pw_size_ok(g3) || !pw_size_ok(g2)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  // variables: of ph, al, p, muts, mu, mudf
  if (step == 0 || variables[1] != variables[2] || g3->nz != g->nz || g3->ny != g->ny || g3->nx != g->nx ||
      g2->ny != g->ny || g2->nx != g->nx || mu == mut || mu == mudf || mut == mudf || pm1_in == pm1_out ||
      al_in == al_out || p_in == p_out)
    return PYWRF_E_ARG;
  PRhoBc a;
  a.b = mkbox(g->kts, imin(g->kte, g->kde - 1), g->jts, imin(g->jte, g->jde - 1), g->its, imin(g->ite, g->ide - 1));
  if (a.b.k1 + 1 > g->nz) return PYWRF_E_RANGE;
  a.r = {al_in, p_in, ph, alt, t_2, t_1, c2a, mu, mut, rdnw, al_out, p_out, pm1_out, F(t0), F(smdiv), step, pm1_in};
  a.k0 = g3->kts;
  int e = bc_spec3(g3, variables[1], a.c, a.k1), kph = 0;
  if (!e && !bc_spec_ok(g->ny, g->nx, g->nz, a.k0, a.k1, a.c)) e = PYWRF_E_RANGE;
  if (!e) e = bc_spec3(g3, variables[0], a.job[0].c, kph);
  if (!e && !bc_spec_ok(g->ny, g->nx, g->nz, g3->kts, kph, a.job[0].c)) e = PYWRF_E_RANGE;
  a.job[0].p = ph; a.job[0].k0 = g3->kts;
  a.nph = a.job[0].nk = imax(kph - g3->kts, 0);
  float* plane[3] = {mut, mu, mudf};
  for (int f = 0; f < 3 && !e; ++f) {
    BcJob& jb = a.job[f + 1];
    jb.p = plane[f]; jb.k0 = 0; jb.nk = 1;
    e = bc_spec2(g2, variables[f + 3], jb.c);
    if (!e && !bc_spec_ok(g2->ny, g2->nx, 1, 0, 1, jb.c)) e = PYWRF_E_RANGE;
  }
  if (e) return e;
  // the fills' targets must lie outside what the formula reads
  for (int f = 0; f < 4; ++f) {
    const BcSpec& c = a.job[f].c;
    if (a.b.j0 < c.jds || a.b.i0 < c.ids || a.b.j1 > (c.vstag ? c.jde : c.jde - 1) ||
        a.b.i1 > (c.ustag ? c.ide : c.ide - 1))
      return PYWRF_E_RANGE;
  }
  a.nfill = a.nph + 3;
  a.ntx = (g->nx + PW_TX - 1) / PW_TX;
  a.nty = (g->ny + PB_ROWS - 1) / PB_ROWS;
  const long blocks = a.nfill + (long)a.ntx * a.nty * g->nz;
  hipLaunchKernelGGL(k_calc_p_rho_bc, dim3((unsigned)blocks), dim3(BC_THREADS), 0, (hipStream_t)s, dims_of(g), a);
  PW_RET();
}

// ------------------------------------------------------------------ calc_coef_w
// Column block (a 512-thread workgroup owns 64 i-columns of one row j): the
// tridiagonal coefficients of every level are formed level-parallel (a written
// out, the diagonal and upper coefficients staged in LDS); one wave then runs
// the forward elimination alpha/gamma per column from LDS.
#define CW_TI 64
#define CW_TB 512
#define CW_TG (CW_TB / CW_TI)
struct CoefW {
  float *a, *alpha, *gamma;
  const float *mut, *cqw, *rdn, *rdnw, *c2a;
  float C, m2C, p2C, lid;
  int kde;
};

__global__ void __launch_bounds__(CW_TB) k_calc_coef_w(Box b, Dims D, CoefW p) {
  extern __shared__ float sm[];
  float* s_a = sm;                  // [nz][CW_TI] sub-diagonal
  float* s_b = sm + D.nz * CW_TI;   // diagonal
  float* s_c = sm + 2 * D.nz * CW_TI;   // super-diagonal
  const int lane = threadIdx.x % CW_TI, grp = threadIdx.x / CW_TI;
  int bx, by;
  xcd_block_2d(bx, by);   // rows of one XCD contiguous (neighbouring rows share an L2)
  const int j = b.j0 + by, i = b.i0 + bx * CW_TI + lane;
  const bool ok = i < b.i1;
  const int kde = p.kde;
  float m = 0.0f;
  if (ok) {
    m = AT2(p.mut, j, i);
    for (int k = 1 + grp; k < kde - 1; k += CW_TG) {
      float cq = AT(p.cqw, k, j, i), c2 = AT(p.c2a, k, j, i), c2m = AT(p.c2a, k - 1, j, i);
      float ak = 0.0f;
      if (k >= 2) {
        ak = -cq * p.C * p.rdn[k] * p.rdnw[k - 1] * c2m / (m * m);
        AT(p.a, k, j, i) = ak;
      }
      s_a[k * CW_TI + lane] = ak;
      s_b[k * CW_TI + lane] = 1.0f + cq * p.C * p.rdn[k] * (p.rdnw[k] * c2 / (m * m) + p.rdnw[k - 1] * c2m / (m * m));
      s_c[k * CW_TI + lane] = -cq * p.C * p.rdn[k] * p.rdnw[k] * c2 / (m * m);
    }
  }
  __syncthreads();
  if (!ok || grp != 0) return;
  float r2 = p.rdnw[kde - 2] * p.rdnw[kde - 2];
  AT(p.a, 1, j, i) = 0.0f;
  float atop = p.m2C * r2 * AT(p.c2a, kde - 2, j, i) * p.lid / (m * m);
  AT(p.a, kde - 1, j, i) = atop;
  AT(p.gamma, 0, j, i) = 0.0f;
  float gm = 0.0f;
  for (int k = 1; k < kde - 1; ++k) {
    float al = 1.0f / (s_b[k * CW_TI + lane] - s_a[k * CW_TI + lane] * gm);
    gm = s_c[k * CW_TI + lane] * al;
    AT(p.alpha, k, j, i) = al;
    AT(p.gamma, k, j, i) = gm;
  }
  float bb = 1.0f + p.p2C * r2 * AT(p.c2a, kde - 2, j, i) / (m * m);
  AT(p.alpha, kde - 1, j, i) = 1.0f / (bb - atop * gm);
  AT(p.gamma, kde - 1, j, i) = 0.0f;
}

extern "C" int pywrf_calc_coef_w(const pywrf_grid_t* g, float* a, float* alpha, float* gamma, const float* mut,
                                 const float* cqw, const float* rdn, const float* rdnw, const float* c2a,
                                 double dts, double g_, double epssm, int top_lid, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kde > g->nz || g->kde < 3) return PYWRF_E_RANGE;
  double C = (0.5 * dts * g_ * (1. + epssm));
  C = C * C;
  Box b = mkbox(0, 1, g->jts, imin(g->jte, g->jde - 1), g->its, imin(g->ite, g->ide - 1));
  const size_t lds = 3 * (size_t)g->nz * CW_TI * sizeof(float);
  if (lds > 64 * 1024) return PYWRF_E_RANGE;
  if (b.nj() <= 0 || b.ni() <= 0) PW_RET();
  CoefW p = {a, alpha, gamma, mut, cqw, rdn, rdnw, c2a, F(C), F(-2. * C), F(2. * C), top_lid ? 0.0f : 1.0f, g->kde};
  hipLaunchKernelGGL(k_calc_coef_w, dim3((unsigned)((b.ni() + CW_TI - 1) / CW_TI), (unsigned)b.nj()), dim3(CW_TB),
                     lds, (hipStream_t)s, b, dims_of(g), p);
  PW_RET();
}

// ------------------------------------------------------------------ advance_uv
struct AdvUV {
  const float *u_in, *ru_tend, *v_in, *rv_tend, *p, *pb, *ph, *php, *alt, *al, *mu, *muu, *cqu, *muv, *cqv, *mudf;
  const float *msfux, *msfuy, *msfvx, *msfvx_inv, *msfvy, *cf, *fnm, *fnp, *rdnw;
  float *u, *v;
  float rdx, rdy, dts, dfx, dfy;
  int kde;
};

// A thread marches up kc levels of its column, the values of the plane formed
// once, p, ph and the pressure on w levels taken over from level to level, all
// loads before the branches (neighbours clamped into the plane; what lies
// outside a box is not used).
//
// ZONE: the specified zone's update of u and v (zu, zv: the ring around bu, bv)
// on the points the boxes leave out.  240 x 240 x 41: 33.7 us, one
// point a thread 46.2; the zone's update adds 0.5 us, as a launch of its own 5.2.
template <bool ZONE>
__global__ void __launch_bounds__(PW_BLOCK) k_advance_uv(Box all, Dims D, AdvUV a, Box bu, Box bv, UpdJob zu, UpdJob zv,
                                                         int kc) {
  const int i = all.i0 + (int)(blockIdx.x * PW_TX + threadIdx.x), j = all.j0 + (int)(blockIdx.y * PW_TY + threadIdx.y);
  if (i >= all.i1 || j >= all.j1) return;
  const int ka = all.k0 + (int)blockIdx.z * kc, kb = imin(ka + kc, all.k1);
  const unsigned C = D.ob2(j, i), W = D.ob2(j, imax(i - 1, 0)), S = D.ob2(imax(j - 1, 0), i);
  const unsigned plane = (unsigned)D.plane() * 4u;
  const bool u2 = bu.has2(j, i), v2 = bv.has2(j, i);
  const float msfuy = at_b(a.msfuy, C), muc = at_b(a.mu, C), dfc = at_b(a.mudf, C);
  const float rx = at_b(a.msfux, C) / msfuy, ry = at_b(a.msfvy, C) / at_b(a.msfvx, C);
  const float Au = rx * 0.5f * a.rdx * at_b(a.muu, C), Bu = rx * a.rdx, Mu = 0.5f * (at_b(a.mu, W) + muc);
  const float Av = ry * 0.5f * a.rdy * at_b(a.muv, C), Bv = ry * a.rdy, Mv = 0.5f * (at_b(a.mu, S) + muc);
  const float mxu = a.dfx * (dfc - at_b(a.mudf, W)) / msfuy, mxv = a.dfy * (dfc - at_b(a.mudf, S)) * at_b(a.msfvx_inv, C);
  unsigned o = (unsigned)ka * plane;
  float pc = at_b(a.p, o + C), pw = at_b(a.p, o + W), ps = at_b(a.p, o + S);
  float phc = at_b(a.ph, o + C), phw = at_b(a.ph, o + W), phs = at_b(a.ph, o + S);
  float du = 0.0f, dv = 0.0f;   // the pressure on w level k at the u and v faces
  if (ka == 0) {
    const unsigned p1 = imin(1, D.nz - 1) * plane, p2 = imin(2, D.nz - 1) * plane;
    const float c1 = at_b(a.p, p1 + C), c2 = at_b(a.p, p2 + C);
    const float f0 = level(a.cf, 0), f1 = level(a.cf, 1), f2 = level(a.cf, 2);
    du = 0.5f * (f0 * (pc + pw) + f1 * (c1 + at_b(a.p, p1 + W)) + f2 * (c2 + at_b(a.p, p2 + W)));
    dv = 0.5f * (f0 * (pc + ps) + f1 * (c1 + at_b(a.p, p1 + S)) + f2 * (c2 + at_b(a.p, p2 + S)));
  } else if (ka < a.kde - 1) {
    const unsigned m = o - plane;
    const float fm = level(a.fnm, ka), fp = level(a.fnp, ka), pmc = at_b(a.p, m + C);
    du = 0.5f * (fm * (pc + pw) + fp * (pmc + at_b(a.p, m + W)));
    dv = 0.5f * (fm * (pc + ps) + fp * (pmc + at_b(a.p, m + S)));
  }
  for (int k = ka; k < kb; ++k) {
    const unsigned t = o + C, up = k + 1 < D.nz ? o + plane : o;
    float u = at_b(a.u_in, t), v = at_b(a.v_in, t);
    const float tu = at_b(a.ru_tend, t), tv = at_b(a.rv_tend, t);
    if (k < bu.k1) {   // bu, bv: the same levels
      const bool lev = k >= bu.k0, inu = u2 && lev, inv = v2 && lev;
      const float cqu = at_b(a.cqu, t), cqv = at_b(a.cqv, t);
      const float pnc = at_b(a.p, up + C), pnw = at_b(a.p, up + W), pns = at_b(a.p, up + S);
      const float pcc = at_b(a.ph, up + C), pcw = at_b(a.ph, up + W), pcs = at_b(a.ph, up + S);
      const float ac = at_b(a.alt, t), aw = at_b(a.alt, o + W), as = at_b(a.alt, o + S);
      const float lc = at_b(a.al, t), lw = at_b(a.al, o + W), ls = at_b(a.al, o + S);
      const float bc = at_b(a.pb, t), bw = at_b(a.pb, o + W), bs = at_b(a.pb, o + S);
      const float hc = at_b(a.php, t), hw = at_b(a.php, o + W), hs = at_b(a.php, o + S);
      float dun = 0.0f, dvn = 0.0f;
      if (k + 1 != a.kde - 1) {
        const float fm = level(a.fnm, k + 1), fp = level(a.fnp, k + 1);
        dun = 0.5f * (fm * (pnc + pnw) + fp * (pc + pw));
        dvn = 0.5f * (fm * (pnc + pns) + fp * (pc + ps));
      }
      const float rd = level(a.rdnw, k);
      const float xu = Au * (((pcc - pcw) + (phc - phw)) + (ac + aw) * (pc - pw) + (lc + lw) * (bc - bw)) +
                       Bu * (hc - hw) * (rd * (dun - du) - Mu);
      const float xv = Av * (((pcc - pcs) + (phc - phs)) + (ac + as) * (pc - ps) + (lc + ls) * (bc - bs)) +
                       Bv * (hc - hs) * (rd * (dvn - dv) - Mv);
      if (inu) u = (u + a.dts * tu) - a.dts * cqu * xu + mxu;
      else if (ZONE) u = spec_upd_value(zu, k, j, i, u, tu);
      if (inv) v = (v + a.dts * tv) - a.dts * cqv * xv + mxv;
      else if (ZONE) v = spec_upd_value(zv, k, j, i, v, tv);
      du = dun; dv = dvn;
      pc = pnc; pw = pnw; ps = pns;
      phc = pcc; phw = pcw; phs = pcs;
    } else if (ZONE) {
      u = spec_upd_value(zu, k, j, i, u, tu);
      v = spec_upd_value(zv, k, j, i, v, tv);
    }
    at_b(a.u, t) = u;
    at_b(a.v, t) = v;
    o += plane;
  }
}

// gz non-null: also spec_bdyupdate of u with ru_tend and of v with rv_tend, step zdt
static int advance_uv(const pywrf_grid_t* g, const float* u_in, const float* ru_tend, const float* v_in,
                                const float* rv_tend, const float* p, const float* pb, const float* ph,
                                const float* php, const float* alt, const float* al, const float* mu,
                                const float* muu, const float* cqu, const float* muv, const float* cqv,
                                const float* mudf, const float* msfux, const float* msfuy, const float* msfvx,
                                const float* msfvx_inv, const float* msfvy, double rdx, double rdy, double dts,
                                const float* cf, const float* fnm, const float* fnp, double emdiv,
                                const float* rdnw, int spec_zone, float* u_out, float* v_out,
                                const pywrf_grid_t* gz, double zdt, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  int k1 = imin(g->kte, g->kde - 1);
  if (k1 + 1 > g->nz || g->kde > g->nz) return PYWRF_E_RANGE;
  int i0 = imax(g->its, g->ids + spec_zone), i1 = imin(g->ite, g->ide - spec_zone - 1);
  int j0 = imax(g->jts, g->jds + spec_zone), j1 = imin(g->jte, g->jde - spec_zone - 1);
  int i1u = imin(g->ite, g->ide - spec_zone), j1v = imin(g->jte, g->jde - spec_zone);
  double dx = 1. / rdx, dy = 1. / rdy;
  AdvUV a = {u_in, ru_tend, v_in, rv_tend, p, pb, ph, php, alt, al, mu, muu, cqu, muv, cqv, mudf, msfux, msfuy,
             msfvx, msfvx_inv, msfvy, cf, fnm, fnp, rdnw, u_out, v_out, F(rdx), F(rdy), F(dts), F(-emdiv * dx),
             F(-emdiv * dy), g->kde};
  Box bu = mkbox(g->kts, k1, j0, j1, i0, i1u);
  Box bv = mkbox(g->kts, k1, j0, j1v, i0, i1);
  UpdJob zu = {}, zv = {};
  bool ring = false;
  if (gz) {
    int wu, wv, e = spec_upd_job(gz, u_out, ru_tend, zdt, 'u', zu, wu);
    if (!e) e = spec_upd_job(gz, v_out, rv_tend, zdt, 'v', zv, wv);
    if (e) return e;
    ring = spec_upd_rings(zu, bu) && spec_upd_rings(zv, bv);
  }
  const Box all = whole(g);
  const int kc = march_levels(all);
  dim3 grid((unsigned)((all.ni() + PW_TX - 1) / PW_TX), (unsigned)((all.nj() + PW_TY - 1) / PW_TY),
            (unsigned)((all.nk() + kc - 1) / kc));
  hipLaunchKernelGGL(ring ? k_advance_uv<true> : k_advance_uv<false>, grid, dim3(PW_TX, PW_TY), 0, (hipStream_t)s, all,
                     dims_of(g), a, bu, bv, zu, zv, kc);
  if (gz && !ring) {
    int e = pywrf_spec_bdyupdate(gz, u_out, ru_tend, zdt, 'u', s);
    return e ? e : pywrf_spec_bdyupdate(gz, v_out, rv_tend, zdt, 'v', s);
  }
  PW_RET();
}

#define UV_ARGS                                                                                                      \
  const float *u_in, const float *ru_tend, const float *v_in, const float *rv_tend, const float *p, const float *pb, \
      const float *ph, const float *php, const float *alt, const float *al, const float *mu, const float *muu,       \
      const float *cqu, const float *muv, const float *cqv, const float *mudf, const float *msfux,                   \
      const float *msfuy, const float *msfvx, const float *msfvx_inv, const float *msfvy, double rdx, double rdy,    \
      double dts, const float *cf, const float *fnm, const float *fnp, double emdiv, const float *rdnw,              \
      int spec_zone, float *u_out, float *v_out
#define UV_PASS                                                                                                     \
  u_in, ru_tend, v_in, rv_tend, p, pb, ph, php, alt, al, mu, muu, cqu, muv, cqv, mudf, msfux, msfuy, msfvx,         \
      msfvx_inv, msfvy, rdx, rdy, dts, cf, fnm, fnp, emdiv, rdnw, spec_zone, u_out, v_out

extern "C" int pywrf_advance_uv(const pywrf_grid_t* g, UV_ARGS, pywrf_stream_t s) {
  return advance_uv(g, UV_PASS, nullptr, 0.0, s);
}

extern "C" int pywrf_advance_uv_zone(const pywrf_grid_t* g, const pywrf_grid_t* gz, UV_ARGS, double zone_dt,
                                     pywrf_stream_t s) {
  if (!pw_size_ok(gz) || !pw_size_ok(g) || gz->nz != g->nz || gz->ny != g->ny || gz->nx != g->nx) return PYWRF_E_RANGE;
  return advance_uv(g, UV_PASS, gz, zone_dt, s);
}

// ------------------------------------------------------------------ advance_mu_t
struct AdvMuT {
  const float *ww_in, *ww_1, *u, *u_1, *v, *v_1, *mu_in, *mut, *muave_in, *muts_in, *muu, *muv, *mudf_in;
  const float *t_in, *t_1, *t_ave_in, *ft, *mu_tend, *dnw, *fnm, *fnp, *rdnw;
  const float *msfuy, *msfvx_inv, *msftx, *msfty;
  float *ww, *t, *t_ave, *muave, *muts, *mudf, *mu;
  float rdx, rdy, dts, ep1, em1, hrdx, hrdy;
  int k1, kde, j0, j1, i0, i1;
};

// Column block: a 512-thread workgroup owns TI consecutive i-columns of one
// row j and all levels; wave `grp` takes levels grp, grp + TG, ...  The
// divergence dvdxi of every (k, i) is computed by all waves and staged in LDS;
// the column sum, the column-mass update and the eta-velocity recurrence
// follow from LDS; all waves finally apply the theta update.  Columns outside
// the update box copy their inputs (clone semantics).
//
// What bounds it is memory latency: the grid's blocks are all resident at once
// and reach each phase together, so every phase that loads costs a full
// round trip.  Each wave therefore loads everything it will need, for all of
// its LPT levels, before the first barrier (no load is under a branch; level
// indices are clamped to k1 - 1), and keeps five values a level in registers
// across the serial part; after it there are only stores.  Each level's
// vertical theta flux is formed once and passed to the level below in LDS.
#define TI 64
#define TB 512
#define TG (TB / TI)

#define CB_MAXNZ 128   // column blocks hold at most 64 KB of per-level LDS, so nz <= 128

// the wave's number, known to the compiler to be the same in all its lanes
__device__ __forceinline__ int wave_of_block() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x / TI); }

//
// ZONE: the specified zone's update of t, mu and muts (zt, zm, zs: the ring
// around the box) on the columns it passes through.  Those columns' loads all
// precede their stores: level by level, each behind the stores of the one
// before, they were what the waves at the sides of the domain took longest for.
// 35.6 us at 240 x 240 x 41 (11.0 at 40 x 40) with the zone's update, against
// 35.7 (11.4) and a further launch of 5.2 (3.3) us.
template <int LPT, bool ZONE>
__global__ void __launch_bounds__(TB) k_advance_mu_t(Dims D, AdvMuT a, UpdJob zt, UpdJob zm, UpdJob zs) {
  extern __shared__ float sm[];
  __shared__ float s_part[(CB_MAXNZ / 16 + 1) * TI];
  const int nz = D.nz, k1 = a.k1;
  float* s_dv = sm;             // [nz][TI] dvdxi, then the eta-velocity decrements, then the theta fluxes
  float* s_ww = sm + nz * TI;   // [nz][TI] eta velocity before subtracting ww_1
  const int lane = threadIdx.x % TI, grp = wave_of_block();
  int bx, by;
#if PW_COL_XCD
  xcd_block_2d(bx, by);
#else
  bx = (int)blockIdx.x; by = (int)blockIdx.y;
#endif
  const int j = by, i = bx * TI + lane;
  const bool vi = i < D.nx;
  const bool row = j >= a.j0 && j < a.j1 && a.i0 < a.i1;
  const bool h = vi && row && i >= a.i0 && i < a.i1;
  if (vi && !h) {   // all loads before the first store
    float x[LPT + 1], y[LPT + 1], z[LPT + 1], t[LPT + 1];
#pragma unroll
    for (int m = 0; m <= LPT; ++m) {
      const long q = D.ix(imin(grp + m * TG, nz - 1), j, i);
      x[m] = a.ww_in[q]; y[m] = a.t_in[q]; z[m] = a.t_ave_in[q];
      t[m] = ZONE ? a.ft[q] : 0.0f;
    }
    if (grp == 0) {
      const long q = D.ix2(j, i);
      const float ma = a.muave_in[q], ms = a.muts_in[q], mf = a.mudf_in[q], mi = a.mu_in[q];
      const float mt = ZONE ? a.mu_tend[q] : 0.0f;
      a.muave[q] = ma;
      a.muts[q] = ZONE ? spec_upd_value(zs, 0, j, i, ms, mt) : ms;
      a.mudf[q] = mf;
      a.mu[q] = ZONE ? spec_upd_value(zm, 0, j, i, mi, mt) : mi;
    }
#pragma unroll
    for (int m = 0; m <= LPT; ++m) {
      const int k = grp + m * TG;
      if (k >= nz) break;
      const long q = D.ix(k, j, i);
      a.ww[q] = x[m];
      a.t[q] = ZONE ? spec_upd_value(zt, k, j, i, y[m], t[m]) : y[m];
      a.t_ave[q] = z[m];
    }
    // LPT is chosen for the kte - 1 levels of the box; the arrays may hold more
    for (int k = grp + (LPT + 1) * TG; k < nz; k += TG) {
      const long q = D.ix(k, j, i);
      const float wk = a.ww_in[q], tk = a.t_in[q], ak = a.t_ave_in[q];
      a.ww[q] = wk;
      a.t[q] = ZONE ? spec_upd_value(zt, k, j, i, tk, a.ft[q]) : tk;
      a.t_ave[q] = ak;
    }
  }
  if (!row) return;   // the whole block
  const int ic = imin(imax(i, a.i0), a.i1 - 1);   // lanes outside the box load (and drop) its edge column's values
  const long q2 = D.ix2(j, ic);
  const float mvn = AT2(a.muv, j + 1, ic), xn = AT2(a.msfvx_inv, j + 1, ic), mvs = a.muv[q2], xs = a.msfvx_inv[q2];
  const float mue = AT2(a.muu, j, ic + 1), ye = AT2(a.msfuy, j, ic + 1), muw = a.muu[q2], yw = a.msfuy[q2];
  const float mx = a.msftx[q2], my = a.msfty[q2], mt = a.mu_tend[q2], mu_old = a.mu_in[q2], mut = a.mut[q2];
  const float ww0 = AT(a.ww_in, 0, j, ic);
  float r_t[LPT], r_p[LPT], r_h[LPT], r_c[LPT], r_w1[LPT];
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = imin(grp + m * TG, k1 - 1), kd = imax(k - 1, 0);
    const float vn = AT(a.v, k, j + 1, ic), v1n = AT(a.v_1, k, j + 1, ic), vs = AT(a.v, k, j, ic), v1s = AT(a.v_1, k, j, ic);
    const float ue = AT(a.u, k, j, ic + 1), u1e = AT(a.u_1, k, j, ic + 1), uw = AT(a.u, k, j, ic), u1w = AT(a.u_1, k, j, ic);
    const float tin = AT(a.t_in, k, j, ic), ftq = AT(a.ft, k, j, ic), t1 = AT(a.t_1, k, j, ic), t1d = AT(a.t_1, kd, j, ic);
    const float tn = AT(a.t_1, k, j + 1, ic), ts = AT(a.t_1, k, j - 1, ic);
    const float te = AT(a.t_1, k, j, ic + 1), tw = AT(a.t_1, k, j, ic - 1);
    r_w1[m] = AT(a.ww_1, k, j, ic);
    const float vy = (vn + mvn * v1n * xn) - (vs + mvs * v1s * xs);
    const float ux = (ue + mue * u1e / ye) - (uw + muw * u1w / yw);
    const float dv = mx * my * (a.rdy * vy + a.rdx * ux);
    if (grp + m * TG < k1) s_dv[k * TI + lane] = dv;
    const float yterm = a.hrdy * (vn * (tn + t1) - vs * (t1 + ts));
    const float xterm = a.hrdx * (ue * (te + t1) - uw * (t1 + tw));
    r_t[m] = tin + 0.0f;
    r_p[m] = tin + my * a.dts * ftq;
    r_h[m] = mx * (yterm + xterm);
    r_c[m] = level(a.fnm, k) * t1 + level(a.fnp, k) * t1d;
  }
  __syncthreads();
  // The column sum dmdt in torch's order (torch_outer_sum with nz <= 128:
  // blocks of 16 levels summed from +0 one after the other, the tail from +0,
  // tail + (sum of the block sums) + 0 + 0; levels from k1 on add +0, which
  // changes no partial sum): each block's chain and the tail's are
  // independent, so the waves form them side by side.
  const int nb = nz >> 4;
  for (int c = grp; c <= nb; c += TG) {
    const int k0 = c << 4, ke = imin(imin(k0 + 16, nz), k1);
    float acc = 0.0f;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const int k = imin(k0 + m, k1 - 1);
      const float x = level(a.dnw, k) * s_dv[k * TI + lane];
      acc += k0 + m < ke ? x : 0.0f;
    }
    s_part[c * TI + lane] = acc;
  }
  __syncthreads();
  // every wave forms the column's dmdt from the block sums (the same floats)
  float blocks = 0.0f;
  for (int c = 0; c < nb; ++c) blocks += s_part[c * TI + lane];
  float dmdt = s_part[nb * TI + lane] + blocks;
  dmdt = dmdt + 0.0f;
  dmdt = dmdt + 0.0f;
  if (grp == 0 && h) {
    const float mu = mu_old + a.dts * (dmdt + mt);
    a.mu[q2] = mu;
    a.mudf[q2] = dmdt + mt;
    a.muts[q2] = mut + mu;
    a.muave[q2] = 0.5f * (a.ep1 * mu + a.em1 * (mu_old + 0.0f));
  }
  // the eta-velocity decrements dnw(k) (dmdt + dvdxi(k) + mu_tend) / msfty of
  // every level at once, in place of dvdxi(k) (this wave's own entries)
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = grp + m * TG;
    if (k < k1) s_dv[k * TI + lane] = level(a.dnw, k) * (dmdt + s_dv[k * TI + lane] + mt) / my;
  }
  __syncthreads();
  if (grp == 0) {
    // the decrements 8 levels at a time into registers first (s_dv and s_ww
    // share one LDS buffer, so a read after a store to s_ww would wait for it)
    float wk = ww0;
    s_ww[lane] = wk;
    int k = 1;
    for (; k + 7 < k1; k += 8) {
      float dv[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) dv[m] = s_dv[(k - 1 + m) * TI + lane];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        wk = wk - dv[m];
        s_ww[(k + m) * TI + lane] = wk;
      }
    }
    for (; k < k1; ++k) {
      wk = wk - s_dv[(k - 1) * TI + lane];
      s_ww[k * TI + lane] = wk;
    }
  }
  __syncthreads();
  // the vertical theta flux wdtn(k) of each level (zero at k = 0) into s_dv
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = grp + m * TG;
    if (k < k1) {
      const float wwk = s_ww[k * TI + lane] - r_w1[m];
      r_w1[m] = wwk;
      r_c[m] = k > 0 ? wwk * r_c[m] : 0.0f;
      s_dv[k * TI + lane] = r_c[m];
    }
  }
  __syncthreads();
  if (!h) return;
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = grp + m * TG;
    if (k >= k1) continue;
    const float wdu = k + 1 < k1 ? s_dv[(k + 1) * TI + lane] : 0.0f;
    AT(a.ww, k, j, i) = r_w1[m];
    AT(a.t_ave, k, j, i) = r_t[m];
    AT(a.t, k, j, i) = r_p[m] - a.dts * my * (r_h[m] + level(a.rdnw, k) * (wdu - r_c[m]));
  }
  for (int k = k1 + grp; k < nz; k += TG) {   // levels at and above k1 copy their inputs
    const long q = D.ix(k, j, i);
    const float x = a.ww_in[q], y = a.t_in[q], z = a.t_ave_in[q];
    a.ww[q] = x;
    a.t[q] = y;
    a.t_ave[q] = z;
  }
}

static int column_block_launch_check(const pywrf_grid_t* g, int narrays) {
  size_t bytes = (size_t)narrays * g->nz * TI * sizeof(float);
  return bytes <= 64 * 1024 ? 0 : PYWRF_E_RANGE;
}

#define MUT_ARGS                                                                                                       \
  const float *ww_in, const float *ww_1, const float *u, const float *u_1, const float *v, const float *v_1,           \
      const float *mu_in, const float *mut, const float *muave_in, const float *muts_in, const float *muu,             \
      const float *muv, const float *mudf_in, const float *t_in, const float *t_1, const float *t_ave_in,              \
      const float *ft, const float *mu_tend, double rdx, double rdy, double dts, double epssm, const float *dnw,       \
      const float *fnm, const float *fnp, const float *rdnw, const float *msfuy, const float *msfvx_inv,               \
      const float *msftx, const float *msfty, float *ww_out, float *t_out, float *t_ave_out, float *muave_out,         \
      float *muts_out, float *mudf_out, float *mu_out
#define MUT_PASS                                                                                                       \
  ww_in, ww_1, u, u_1, v, v_1, mu_in, mut, muave_in, muts_in, muu, muv, mudf_in, t_in, t_1, t_ave_in, ft, mu_tend,     \
      rdx, rdy, dts, epssm, dnw, fnm, fnp, rdnw, msfuy, msfvx_inv, msftx, msfty, ww_out, t_out, t_ave_out,             \
      muave_out, muts_out, mudf_out, mu_out

// gz non-null: also spec_bdyupdate of t with ft (gz) and of mu and muts with mu_tend (gz2, 2-D), step zdt
static int advance_mu_t(const pywrf_grid_t* g, MUT_ARGS, const pywrf_grid_t* gz, const pywrf_grid_t* gz2, double zdt,
                        pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kte > g->nz || g->kte < 2) return PYWRF_E_RANGE;
  AdvMuT a = {ww_in, ww_1, u, u_1, v, v_1, mu_in, mut, muave_in, muts_in, muu, muv, mudf_in, t_in, t_1, t_ave_in,
              ft, mu_tend, dnw, fnm, fnp, rdnw, msfuy, msfvx_inv, msftx, msfty, ww_out, t_out, t_ave_out,
              muave_out, muts_out, mudf_out, mu_out, F(rdx), F(rdy), F(dts), F(1. + epssm), F(1. - epssm),
              F(0.5 * rdx), F(0.5 * rdy), g->kte - 1, g->kde, imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2),
              imax(g->its, g->ids + 1), imin(g->ite, g->ide - 2)};
  if (column_block_launch_check(g, 2)) return PYWRF_E_RANGE;
  UpdJob zt = {}, zm = {}, zs = {};
  bool ring = false;
  if (gz) {
    int w, e = spec_upd_job(gz, t_out, ft, zdt, 't', zt, w);
    if (!e) e = spec_upd_job(gz2, mu_out, mu_tend, zdt, 'm', zm, w);
    if (!e) e = spec_upd_job(gz2, muts_out, mu_tend, zdt, 'm', zs, w);
    if (e) return e;
    const Box in = mkbox(0, g->nz, a.j0, a.j1, a.i0, a.i1);
    ring = spec_upd_rings(zt, in) && spec_upd_rings(zm, in) && spec_upd_rings(zs, in);
  }
  dim3 grid((g->nx + TI - 1) / TI, g->ny);
  // levels a wave keeps in registers: 5 covers the model's 40 mass levels
  auto kern = a.k1 <= 5 * TG ? (ring ? k_advance_mu_t<5, true> : k_advance_mu_t<5, false>)
              : a.k1 <= 8 * TG ? (ring ? k_advance_mu_t<8, true> : k_advance_mu_t<8, false>)
                               : (ring ? k_advance_mu_t<16, true> : k_advance_mu_t<16, false>);
  hipLaunchKernelGGL(kern, grid, dim3(TB), 2 * g->nz * TI * sizeof(float), (hipStream_t)s, dims_of(g), a, zt, zm, zs);
  if (gz && !ring) {
    int e = pywrf_spec_bdyupdate(gz, t_out, ft, zdt, 't', s);
    if (!e) e = pywrf_spec_bdyupdate(gz2, mu_out, mu_tend, zdt, 'm', s);
    return e ? e : pywrf_spec_bdyupdate(gz2, muts_out, mu_tend, zdt, 'm', s);
  }
  PW_RET();
}

extern "C" int pywrf_advance_mu_t(const pywrf_grid_t* g, MUT_ARGS, pywrf_stream_t s) {
  return advance_mu_t(g, MUT_PASS, nullptr, nullptr, 0.0, s);
}

extern "C" int pywrf_advance_mu_t_zone(const pywrf_grid_t* g, const pywrf_grid_t* gz, const pywrf_grid_t* gz2, MUT_ARGS,
                                       double zone_dt, pywrf_stream_t s) {
  if (!pw_size_ok(g) || !pw_size_ok(gz) || !pw_size_ok(gz2) || gz->nz != g->nz || gz->ny != g->ny || gz->nx != g->nx ||
      gz2->ny != g->ny || gz2->nx != g->nx)
    return PYWRF_E_RANGE;
  return advance_mu_t(g, MUT_PASS, gz, gz2, zone_dt, s);
}

// ------------------------------------------------------------------ advance_w
struct AdvW {
  const float *w_in, *rw_tend, *ww, *w_save, *u, *v, *mut, *muave, *muts, *t_2ave_in, *t_2, *t_1, *ph_in, *ph_1;
  const float *phb, *ph_tend, *ht, *c2a, *cqw, *alt, *a, *alpha, *gamma, *fnm, *fnp, *rdnw, *rdn, *cf;
  const float *msftx, *msfty;
  float *t_2ave, *w, *ph;
  float dts, t0, ep1, em1, hgem1, rdx, rdy, hdtsg, dtsg, mhdtsg, dampmag, hpi, hdepth;
  int k1, j0, j1, i0, i1;
};

// Column block as in advance_mu_t, bound the same way: every operand of a
// wave's LPT levels (1 + grp, 1 + grp + TG, ... up to k1) is loaded before the
// first barrier and what the later phases need of it stays in registers (ten
// values a level; the outputs may be the inputs' own arrays); level 0, whose w is the surface condition, belongs to one
// wave.  Four LDS arrays are used in turn: wd holds the geopotential
// advection wdwn, then the pressure term of each half level, then a; rhs the
// phi right-hand side, then w; yp the buoyancy term c2a alt t_2ave of each half
// level, then gamma; al alpha.  Each term is formed once and read by the two
// levels that difference it.  One wave then runs the Thomas sweeps out of
// LDS, and all waves apply the Rayleigh damping (its weights formed before the
// first barrier) and store.
template <int LPT>
__global__ void __launch_bounds__(TB) k_advance_w(Dims D, AdvW a) {
  extern __shared__ float sm[];
  const int nz = D.nz, k1 = a.k1;
  float* s_wd = sm;
  float* s_rhs = sm + 1 * nz * TI;
  float* s_yp = sm + 2 * nz * TI;
  float* s_al = sm + 3 * nz * TI;
  const int lane = threadIdx.x % TI, grp = wave_of_block();
  int bx, by;
#if PW_COL_XCD
  xcd_block_2d(bx, by);
#else
  bx = (int)blockIdx.x; by = (int)blockIdx.y;
#endif
  const int j = by, i = bx * TI + lane;
  const bool vi = i < D.nx;
  const bool row = j >= a.j0 && j < a.j1 && a.i0 < a.i1;
  const bool h = vi && row && i >= a.i0 && i < a.i1;
  if (vi && !h) {   // all loads before the first store
    float x[LPT + 1], y[LPT + 1], z[LPT + 1];
#pragma unroll
    for (int m = 0; m <= LPT; ++m) {
      const long q = D.ix(imin(grp + m * TG, nz - 1), j, i);
      x[m] = a.t_2ave_in[q]; y[m] = a.w_in[q]; z[m] = a.ph_in[q];
    }
#pragma unroll
    for (int m = 0; m <= LPT; ++m) {
      const int k = grp + m * TG;
      if (k >= nz) break;
      const long q = D.ix(k, j, i);
      a.t_2ave[q] = x[m];
      a.w[q] = y[m];
      a.ph[q] = z[m];
    }
  }
  if (!row) return;   // the whole block
  const int ic = imin(imax(i, a.i0), a.i1 - 1);   // lanes outside the box load (and drop) its edge column's values
  const long q2 = D.ix2(j, ic);
  const float G = F(pw::g);
  const float mut = a.mut[q2], muts = a.muts[q2], muave = a.muave[q2], my = a.msfty[q2], mx = a.msftx[q2];
  const float mi = 1.0f / my;
  auto theta_ave = [&](float t2i, float t2, float t1) -> float {
    const float t = 0.5f * (a.ep1 * t2 + a.em1 * t2i);
    return (t + muave * a.t0) / (muts * (a.t0 + t1));
  };
  const float htop = (AT(a.ph_1, k1, j, ic) + AT(a.phb, k1, j, ic)) / G;
  const float hbot = htop - a.hdepth;
  const int ktw = (k1 - 1) % TG, k0w = ktw == TG - 2 ? TG - 3 : TG - 2;   // the waves that own the top level and level 0
  float r_a[LPT], r_ga[LPT], r_w[LPT], r_cq[LPT], r_cb[LPT], r_e[LPT], r_rhs[LPT], r_phi[LPT], r_hk[LPT];
  float r_ws[LPT], r_t2a[LPT], t2a_sfc = 0.0f, z_a = 0.0f, z_e = 0.0f, z_b = 0.0f;
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = imin(1 + grp + m * TG, k1), kl = imin(k, k1 - 1);   // kl: the half level above k, where there is one
    const float t2i = AT(a.t_2ave_in, k, j, ic), t2 = AT(a.t_2, kl, j, ic), t1 = AT(a.t_1, kl, j, ic);
    const float pht = AT(a.ph_tend, k, j, ic), win = AT(a.w_in, k, j, ic);
    const float phi = AT(a.ph_in, k, j, ic), php = AT(a.ph_in, kl + 1, j, ic);
    const float ww0 = AT(a.ww, k, j, ic), wwm = AT(a.ww, k - 1, j, ic);
    const float p10 = AT(a.ph_1, k, j, ic), p1m = AT(a.ph_1, k - 1, j, ic);
    const float pb0 = AT(a.phb, k, j, ic), pbm = AT(a.phb, k - 1, j, ic);
    const float c2 = AT(a.c2a, kl, j, ic), alt = AT(a.alt, kl, j, ic), cq = AT(a.cqw, kl, j, ic);
    const float rwt = AT(a.rw_tend, k, j, ic);
    r_ws[m] = AT(a.w_save, k, j, ic);
    r_a[m] = AT(a.a, k, j, ic);
    const float al = AT(a.alpha, k, j, ic);
    r_ga[m] = AT(a.gamma, k, j, ic);
    // wdwn(k) = 0.5 (ww[k] + ww[k-1]) rdnw[k-1] (ph_1[k] - ph_1[k-1] + phb[k] - phb[k-1])
    const float wd = 0.5f * (ww0 + wwm) * level(a.rdnw, k - 1) * (p10 - p1m + pb0 - pbm);
    const float t2a = k < k1 ? theta_ave(t2i, t2, t1) : t2i;
    if (1 + grp + m * TG <= k1) {
      s_wd[k * TI + lane] = wd;
      s_yp[k * TI + lane] = c2 * alt * t2a;   // read below k1 only
      s_al[k * TI + lane] = al;
    }
    r_t2a[m] = t2a;
    r_w[m] = win + a.dts * rwt;
    r_cq[m] = mi * cq;
    r_cb[m] = c2 * level(a.rdnw, kl) / mut;
    r_e[m] = a.em1 * (php - phi);
    r_rhs[m] = a.dts * (pht + a.hgem1 * win);
    r_phi[m] = phi;
    r_hk[m] = (p10 + pb0) / G;
  }
  if (grp == ktw) {
    const float c2m = AT(a.c2a, k1 - 1, j, ic), alm = AT(a.alt, k1 - 1, j, ic);
    const float ph0 = AT(a.ph_in, k1, j, ic), phm = AT(a.ph_in, k1 - 1, j, ic), rn = level(a.rdnw, k1 - 1);
    const float t2a = theta_ave(AT(a.t_2ave_in, k1 - 1, j, ic), AT(a.t_2, k1 - 1, j, ic), AT(a.t_1, k1 - 1, j, ic));
    z_a = a.mhdtsg / mut * (rn * rn) * 2.0f * c2m;
    z_e = a.em1 * (ph0 - phm);
    z_b = a.dtsg * (2.0f * rn * c2m * alm * t2a + muave);
  }
  float z_cb = 0.0f, w_sfc = 0.0f, ph_sfc = 0.0f;
  if (grp == k0w) {
    const float cf1 = level(a.cf, 0), cf2 = level(a.cf, 1), cf3 = level(a.cf, 2);
    auto V3 = [&](int jj, int ii) {
      return cf1 * AT(a.v, 0, jj, ii) + cf2 * AT(a.v, 1, jj, ii) + cf3 * AT(a.v, 2, jj, ii);
    };
    auto U3 = [&](int jj, int ii) {
      return cf1 * AT(a.u, 0, jj, ii) + cf2 * AT(a.u, 1, jj, ii) + cf3 * AT(a.u, 2, jj, ii);
    };
    const float c2 = AT(a.c2a, 0, j, ic), alt = AT(a.alt, 0, j, ic), php = AT(a.ph_in, 1, j, ic);
    const float t2i = AT(a.t_2ave_in, 0, j, ic), t2 = AT(a.t_2, 0, j, ic), t1 = AT(a.t_1, 0, j, ic);
    ph_sfc = AT(a.ph_in, 0, j, ic);
    const float htc = AT2(a.ht, j, ic);
    const float ty = (AT2(a.ht, j + 1, ic) - htc) * V3(j + 1, ic) + (htc - AT2(a.ht, j - 1, ic)) * V3(j, ic);
    const float tx = (AT2(a.ht, j, ic + 1) - htc) * U3(j, ic + 1) + (htc - AT2(a.ht, j, ic - 1)) * U3(j, ic);
    w_sfc = my * 0.5f * a.rdy * ty + mx * 0.5f * a.rdx * tx;
    t2a_sfc = theta_ave(t2i, t2, t1);
    s_yp[lane] = c2 * alt * t2a_sfc;
    z_cb = c2 * level(a.rdnw, 0) / mut;
    z_e = a.em1 * (php - ph_sfc);
    s_rhs[lane] = 0.0f;
  }
  __syncthreads();
  // the phi right-hand side
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = 1 + grp + m * TG;
    if (k > k1) continue;
    float r = r_rhs[m];
    if (k < k1) r = r - a.dts * (level(a.fnm, k) * s_wd[(k + 1) * TI + lane] + level(a.fnp, k) * s_wd[k * TI + lane]);
    r = r_phi[m] + my * r / mut;
    r_rhs[m] = r;
    s_rhs[k * TI + lane] = r;
  }
  __syncthreads();
  // the pressure term of each half level, and the top level's w
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = 1 + grp + m * TG;
    if (k < k1) {
      s_wd[k * TI + lane] = r_cb[m] * (a.ep1 * (s_rhs[(k + 1) * TI + lane] - r_rhs[m]) + r_e[m]);
    } else if (k == k1) {
      r_w[m] = r_w[m] + mi * (z_a * (a.ep1 * (r_rhs[m] - s_rhs[(k1 - 1) * TI + lane]) + z_e) - z_b);
    }
  }
  if (grp == k0w) s_wd[lane] = z_cb * (a.ep1 * (s_rhs[TI + lane] - 0.0f) + z_e);
  __syncthreads();
  // the explicit w predictor
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = 1 + grp + m * TG;
    if (k > k1) continue;
    float w = r_w[m];
    if (k < k1) {
      const float X = a.hdtsg * level(a.rdn, k) * (s_wd[k * TI + lane] - s_wd[(k - 1) * TI + lane]);
      const float Y = level(a.rdn, k) * (s_yp[k * TI + lane] - s_yp[(k - 1) * TI + lane]) - muave;
      w = w + r_cq[m] * X + a.dtsg * mi * Y;
    }
    s_rhs[k * TI + lane] = w;
  }
  if (grp == k0w) s_rhs[lane] = w_sfc;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = 1 + grp + m * TG;
    if (k > k1) continue;
    s_wd[k * TI + lane] = r_a[m];
    s_yp[k * TI + lane] = r_ga[m];
  }
  __syncthreads();
  // The sweeps take their operands 8 levels at a time into registers before
  // the dependent arithmetic: the LDS arrays are runtime offsets into one
  // buffer, so a read placed after a store to s_rhs would be made to wait for
  // it.  The other waves form their damping weights meanwhile.
  if (grp == 0) {
    float* s_w = s_rhs;
    const float *s_a = s_wd, *s_ga = s_yp;
    float wm = s_w[lane];
    int k = 1;
    for (; k + 7 <= k1; k += 8) {
      float wv[8], av[8], lv[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        wv[m] = s_w[(k + m) * TI + lane]; av[m] = s_a[(k + m) * TI + lane]; lv[m] = s_al[(k + m) * TI + lane];
      }
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        wm = (wv[m] - av[m] * wm) * lv[m];
        s_w[(k + m) * TI + lane] = wm;
      }
    }
    for (; k <= k1; ++k) {
      wm = (s_w[k * TI + lane] - s_a[k * TI + lane] * wm) * s_al[k * TI + lane];
      s_w[k * TI + lane] = wm;
    }
    float wp = wm;
    k = k1 - 1;
    for (; k - 7 >= 1; k -= 8) {
      float wv[8], gv[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) { wv[m] = s_w[(k - m) * TI + lane]; gv[m] = s_ga[(k - m) * TI + lane]; }
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        wp = wv[m] - gv[m] * wp;
        s_w[(k - m) * TI + lane] = wp;
      }
    }
    for (; k >= 1; --k) {
      wp = s_w[k * TI + lane] - s_ga[k * TI + lane] * wp;
      s_w[k * TI + lane] = wp;
    }
  }
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    float dw = 0.0f;
    if (r_hk[m] >= hbot) {
      const float sn = sinf(a.hpi * (r_hk[m] - hbot) / a.hdepth);
      dw = a.dampmag * (sn * sn);
    }
    r_ws[m] = dw * mut * r_ws[m];
    r_hk[m] = 1.0f + dw;
  }
  __syncthreads();
  if (!h) return;
#pragma unroll
  for (int m = 0; m < LPT; ++m) {
    const int k = 1 + grp + m * TG;
    if (k > k1) continue;
    const float w = (s_rhs[k * TI + lane] - r_ws[m]) / r_hk[m];
    AT(a.t_2ave, k, j, i) = r_t2a[m];
    AT(a.w, k, j, i) = w;
    AT(a.ph, k, j, i) = r_rhs[m] + my * 0.5f * a.dts * G * a.ep1 * w / muts;
  }
  if (grp == k0w) {
    AT(a.t_2ave, 0, j, i) = t2a_sfc;
    AT(a.w, 0, j, i) = w_sfc;
    AT(a.ph, 0, j, i) = ph_sfc;
  }
  for (int k = k1 + 1 + grp; k < nz; k += TG) {   // levels above k1 copy their inputs
    const long q = D.ix(k, j, i);
    const float x = a.t_2ave_in[q], y = a.w_in[q], z = a.ph_in[q];
    a.t_2ave[q] = x;
    a.w[q] = y;
    a.ph[q] = z;
  }
}

extern "C" int pywrf_advance_w(const pywrf_grid_t* g, const float* w_in, const float* rw_tend, const float* ww,
                               const float* w_save, const float* u, const float* v, const float* mut,
                               const float* muave, const float* muts, const float* t_2ave_in, const float* t_2,
                               const float* t_1, const float* ph_in, const float* ph_1, const float* phb,
                               const float* ph_tend, const float* ht, const float* c2a, const float* cqw,
                               const float* alt, const float* a, const float* alpha, const float* gamma,
                               double rdx, double rdy, double dts, double t0, double epssm, const float* fnm,
                               const float* fnp, const float* rdnw, const float* rdn, const float* cf,
                               const float* msftx, const float* msfty, float* t_2ave_out, float* w_out,
                               float* ph_out, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kte > g->nz || g->kte < 3) return PYWRF_E_RANGE;
  const double pi_ = 3.14159265359, G = pw::g;
  AdvW p = {w_in, rw_tend, ww, w_save, u, v, mut, muave, muts, t_2ave_in, t_2, t_1, ph_in, ph_1, phb, ph_tend, ht,
            c2a, cqw, alt, a, alpha, gamma, fnm, fnp, rdnw, rdn, cf, msftx, msfty, t_2ave_out, w_out, ph_out,
            F(dts), F(t0), F(1. + epssm), F(1. - epssm), F(0.5 * G * (1. - epssm)), F(rdx), F(rdy),
            F(0.5 * dts * G), F(dts * G), F(-0.5 * dts * G), F(dts * 0.2), F(0.5 * pi_), F(5000.), g->kte - 1,
            imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2), imax(g->its, g->ids + 1), imin(g->ite, g->ide - 2)};
  if (column_block_launch_check(g, 6)) return PYWRF_E_RANGE;   // the LDS of nz levels the entry point has always taken
  dim3 grid((g->nx + TI - 1) / TI, g->ny);
  auto kern = k_advance_w<5>;   // nz <= 42 (column_block_launch_check), so 5 levels a wave hold levels 1 .. 40
  if (p.k1 > 5 * TG) kern = k_advance_w<6>;
  hipLaunchKernelGGL(kern, grid, dim3(TB), 4 * g->nz * TI * sizeof(float), (hipStream_t)s, dims_of(g), p);
  PW_RET();
}

// ------------------------------------------------------------------ sumflux
struct SumFlux {
  const float *ru, *rv, *ww, *u_lin, *v_lin, *ww_lin, *muu, *muv, *msfuy, *msfvx_inv;
  float *ru_m, *rv_m, *ww_m;
  Box all, bu, bv, bw;
  int first, last;
  float n;
};

__device__ inline void sumflux_point(const Dims& D, const SumFlux& a, int k, int j, int i) {
  long q = D.ix(k, j, i);
  // every operand is at this point, so all loads are issued before the
  // branches (a load inside a divergent branch is waited for before the
  // branch ends); `first` and `last` are uniform
  float rm = a.first ? 0.0f : a.ru_m[q], vm = a.first ? 0.0f : a.rv_m[q], wm = a.first ? 0.0f : a.ww_m[q];
  const float rq = a.ru[q], vq = a.rv[q], wq = a.ww[q];
  float ul = 0.0f, vl = 0.0f, wl = 0.0f, mu = 0.0f, my = 0.0f, mv = 0.0f, mx = 0.0f;
  if (a.last) {
    ul = a.u_lin[q]; vl = a.v_lin[q]; wl = a.ww_lin[q];
    mu = AT2(a.muu, j, i); my = AT2(a.msfuy, j, i); mv = AT2(a.muv, j, i); mx = AT2(a.msfvx_inv, j, i);
  }
  if (a.bu.has(k, j, i)) {
    rm = rm + rq;
    if (a.last) rm = rm / a.n + mu * ul / my;
  }
  if (a.bv.has(k, j, i)) {
    vm = vm + vq;
    if (a.last) vm = vm / a.n + mv * vl * mx;
  }
  if (a.bw.has(k, j, i)) {
    wm = wm + wq;
    if (a.last) wm = wm / a.n + wl;
  }
  a.ru_m[q] = rm;
  a.rv_m[q] = vm;
  a.ww_m[q] = wm;
}

__global__ void k_sumflux(Box b, Dims D, SumFlux a) {
  int k, j, i;
  if (box_point(b, k, j, i)) sumflux_point(D, a, k, j, i);
}

// sumflux, and beside it spec_bdyupdate_ph and zero_grad_bdy on the one-cell
// rings of two other arrays: the grid's first nr z-slabs hold the rings' blocks
// (ne of them for each ring and level), so that their chains of strided loads
// run beside the other blocks and not after them.  23.0 us at 240 x 240 x 41
// against 20.3 and 7.5 us for two launches; 26.5 with the rings last.
__global__ void k_sumflux_zone(Box b, Dims D, SumFlux a, PhStrip p, ZgStrip z, int ne, int nr) {
  int j, i;
  if ((int)blockIdx.z >= nr) {
    const int k = b.k0 + (int)blockIdx.z - nr;
    j = b.j0 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
    i = b.i0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (j < b.j1 && i < b.i1) sumflux_point(D, a, k, j, i);
    return;
  }
  int t = ((int)blockIdx.z * (int)gridDim.y + (int)blockIdx.y) * (int)gridDim.x + (int)blockIdx.x;
  const int e = t % ne * PW_EDGE_BLOCK + (int)(threadIdx.y * PW_TX + threadIdx.x);
  t /= ne;
  if (t < p.all.nk()) {
    if (edge_at(p.all, 1, e, j, i)) ph_strip_point(D, p, p.all.k0 + t, j, i);
  } else if (t - p.all.nk() < z.all.nk()) {
    if (edge_at(z.all, 1, e, j, i)) zero_grad_point(D, z, z.all.k0 + t - p.all.nk(), j, i);
  }
}

static int sumflux_setup(const pywrf_grid_t* g, SumFlux& a, int iteration, int number_of_small_timesteps) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kte > g->nz || number_of_small_timesteps == 0) return PYWRF_E_RANGE;
  int mini = imin(g->ide - 1, g->ite), minj = imin(g->jde - 1, g->jte), mink = imin(g->kde - 1, g->kte);
  a.bu = mkbox(g->kts, mink, g->jts, minj, g->its, g->ite);
  a.bv = mkbox(g->kts, mink, g->jts, g->jte, g->its, mini);
  a.bw = mkbox(g->kts, g->kte, g->jts, minj, g->its, mini);
  a.all = mkbox(g->kts, g->kte, g->jts, g->jte, g->its, g->ite);
  a.first = iteration == 1; a.last = iteration == number_of_small_timesteps; a.n = (float)number_of_small_timesteps;
  return 0;
}

extern "C" int pywrf_sumflux(const pywrf_grid_t* g, const float* ru, const float* rv, const float* ww,
                             const float* u_lin, const float* v_lin, const float* ww_lin, const float* muu,
                             const float* muv, float* ru_m, float* rv_m, float* ww_m, const float* msfuy,
                             const float* msfvx_inv, int iteration, int number_of_small_timesteps,
                             pywrf_stream_t s) {
  SumFlux a = {ru, rv, ww, u_lin, v_lin, ww_lin, muu, muv, msfuy, msfvx_inv, ru_m, rv_m, ww_m};
  if (int e = sumflux_setup(g, a, iteration, number_of_small_timesteps)) return e;
  PW_LAUNCH_BOX(k_sumflux, a.all, s, dims_of(g), a);
  PW_RET();
}

extern "C" int pywrf_sumflux_zone(const pywrf_grid_t* g, const pywrf_grid_t* gz, const float* ru, const float* rv,
                                  const float* ww, const float* u_lin, const float* v_lin, const float* ww_lin,
                                  const float* muu, const float* muv, float* ru_m, float* rv_m, float* ww_m,
                                  const float* msfuy, const float* msfvx_inv, int iteration,
                                  int number_of_small_timesteps, const float* ph_save, float* ph,
                                  const float* ph_tend, const float* mu_tend, const float* muts, double dt,
                                  char variable_in, float* zg_field, char zg_variable, pywrf_stream_t s) {
  SumFlux a = {ru, rv, ww, u_lin, v_lin, ww_lin, muu, muv, msfuy, msfvx_inv, ru_m, rv_m, ww_m};
  if (int e = sumflux_setup(g, a, iteration, number_of_small_timesteps)) return e;
  if (!pw_size_ok(gz) || gz->nz != g->nz || gz->ny != g->ny || gz->nx != g->nx) return PYWRF_E_RANGE;
  for (const void* f : {(const void*)ph, (const void*)zg_field})
    for (const void* o : {(const void*)ru, (const void*)rv, (const void*)ww, (const void*)ru_m, (const void*)rv_m,
                          (const void*)ww_m, (const void*)u_lin, (const void*)v_lin, (const void*)ww_lin})
      if (f == o) return PYWRF_E_ARG;
  if (ph == zg_field) return PYWRF_E_ARG;
  PhStrip p;
  ZgStrip z;
  if (int e = ph_strip_setup(gz, ph_save, ph, ph_tend, mu_tend, muts, dt, variable_in, p)) return e;
  if (int e = zero_grad_setup(gz, zg_field, zg_variable, z)) return e;
  const bool band = p.w == 1 && 2 <= p.all.nj() && 2 <= p.all.ni() && 2 <= z.all.nj() && 2 <= z.all.ni();
  if (!band || p.all.size() <= 0 || z.all.size() <= 0 || a.all.size() <= 0) {   // as the calls
    PW_LAUNCH_BOX(k_sumflux, a.all, s, dims_of(g), a);
    return pywrf_spec_bdyupdate_ph_zero_grad(gz, ph_save, ph, ph_tend, mu_tend, muts, dt, variable_in, zg_field,
                                             zg_variable, s);
  }
  const long n = imax((int)edge_count(p.all, 1), (int)edge_count(z.all, 1));
  const int ne = (int)((n + PW_EDGE_BLOCK - 1) / PW_EDGE_BLOCK);
  dim3 grid((unsigned)((a.all.ni() + PW_TX - 1) / PW_TX), (unsigned)((a.all.nj() + PW_TY - 1) / PW_TY), 1);
  const long slab = (long)grid.x * grid.y, rings = (long)ne * (p.all.nk() + z.all.nk());
  const int nr = (int)((rings + slab - 1) / slab);
  grid.z = (unsigned)(a.all.nk() + nr);
  hipLaunchKernelGGL(k_sumflux_zone, grid, dim3(PW_TX, PW_TY), 0, (hipStream_t)s, a.all, dims_of(g), a, p, z, ne, nr);
  PW_RET();
}

// ------------------------------------------------------------------ calc_mu_uv_1
__global__ void k_calc_mu_uv_1(Box b, Dims D, const float* mu, float* muu, float* muv, int jts, int jtf, int jte,
                               int its, int itf, int ite) {
  int j, i;
  if (!box_column(b, j, i)) return;
  if (j < jtf) {
    if (i >= its + 1 && i < ite - 1) AT2(muu, j, i) = 0.5f * (AT2(mu, j, i) + AT2(mu, j, i - 1));
    else if (i == its) AT2(muu, j, i) = AT2(mu, j, i);
    if (i == ite - 1) AT2(muu, j, i) = AT2(mu, j, ite - 2);
  }
  if (i < itf) {
    if (j >= jts + 1 && j < jte - 1) AT2(muv, j, i) = 0.5f * (AT2(mu, j, i) + AT2(mu, j - 1, i));
    else if (j == jts) AT2(muv, j, i) = AT2(mu, j, i);
    if (j == jte - 1) AT2(muv, j, i) = AT2(mu, jte - 2, i);
  }
}

extern "C" int pywrf_calc_mu_uv_1(const pywrf_grid_t* g, const float* mu, float* muu, float* muv, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  int jtf = imin(g->jte, g->jde - 1), itf = imin(g->ite, g->ide - 1);
  Box b = mkbox(0, 1, g->jts, g->jte, g->its, g->ite);
  PW_LAUNCH_COLS(k_calc_mu_uv_1, b, s, dims_of(g), mu, muu, muv, g->jts, jtf, g->jte, g->its, itf, g->ite);
  PW_RET();
}

// ------------------------------------------------------------------ small_step_finish
struct SsFin {
  const float *u_2, *v_2, *w_2, *t_2, *ph_2, *ww1, *mut, *muts, *muu, *muus, *muv, *muvs;
  const float *u_save, *v_save, *w_save, *t_save, *ph_save, *mu_save, *msfuy, *msfvx, *msfty, *h_diabatic;
  float *ww, *mu_2, *u, *v, *w, *ph, *t;
  float dtsn;
  int last, kde, j0, j1, i0, i1, jte, ite;
};

__global__ void k_ssfinish(Box all, Dims D, SsFin a) {
  int k, j, i;
  if (!box_point(all, k, j, i)) return;
  long q = D.ix(k, j, i), q2 = D.ix2(j, i);
  bool hcol = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  // every value is formed first and stored last, so that no load waits on a
  // store, and every operand (all at this point) is loaded before the
  // branches, so that no branch waits on its loads
  const float v2 = a.v_2[q], vs = a.v_save[q], u2 = a.u_2[q], us = a.u_save[q];
  const float w2 = a.w_2[q], ws = a.w_save[q], p2 = a.ph_2[q], ps = a.ph_save[q], wwq = a.ww[q], ww1 = a.ww1[q];
  const float t2 = a.t_2[q], ts = a.t_save[q], hd = a.last ? a.h_diabatic[q] : 0.0f;
  const float msfvx = a.msfvx[q2], muv = a.muv[q2], muvs = a.muvs[q2], msfuy = a.msfuy[q2], muu = a.muu[q2];
  const float muus = a.muus[q2], msfty = a.msfty[q2], mut = a.mut[q2], muts = a.muts[q2];
  const float mu2 = a.mu_2[q2], musv = a.mu_save[q2];
  float v = v2;
  if (k < a.kde - 1 && j >= a.j0 && j < a.jte && i >= a.i0 && i < a.i1) v = (msfvx * v + vs * muv) / muvs;
  float u = u2;
  if (k < a.kde - 1 && j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.ite) u = (msfuy * u + us * muu) / muus;
  float w = w2, ph = p2, wwn = 0.0f;
  const bool hw = k < a.kde && hcol;
  if (hw) {
    w = (msfty * w + ws * mut) / muts;
    ph = ph + ps;
    wwn = wwq + ww1;
  }
  float t = t2;
  if (k < a.kde - 1 && hcol) {
    if (!a.last) t = (t + ts * mut) / muts;
    else t = (t - a.dtsn * mut * hd + ts * mut) / muts;
  }
  const bool hm = k == 0 && hcol;
  const float mu = hm ? mu2 + musv : 0.0f;
  a.v[q] = v;
  a.u[q] = u;
  if (hw) a.ww[q] = wwn;
  a.w[q] = w;
  a.ph[q] = ph;
  a.t[q] = t;
  if (hm) a.mu_2[q2] = mu;
}

extern "C" int pywrf_small_step_finish(const pywrf_grid_t* g, const float* u_2, const float* v_2, const float* w_2,
                                       const float* t_2, const float* ph_2, float* ww, const float* ww1,
                                       float* mu_2, const float* mut, const float* muts, const float* muu,
                                       const float* muus, const float* muv, const float* muvs,
                                       const float* u_save, const float* v_save, const float* w_save,
                                       const float* t_save, const float* ph_save, const float* mu_save,
                                       const float* msfuy, const float* msfvx, const float* msfty,
                                       const float* h_diabatic, int number_of_small_timesteps, double dts,
                                       int rk_step, int rk_order, float* u_out, float* v_out, float* w_out,
                                       float* ph_out, float* t_out, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kde > g->nz || g->kds != 0) return PYWRF_E_RANGE;
  SsFin a = {u_2, v_2, w_2, t_2, ph_2, ww1, mut, muts, muu, muus, muv, muvs, u_save, v_save, w_save, t_save,
             ph_save, mu_save, msfuy, msfvx, msfty, h_diabatic, ww, mu_2, u_out, v_out, w_out, ph_out, t_out,
             F(dts * number_of_small_timesteps), rk_step >= rk_order, g->kde, g->jts, imin(g->jte, g->jde - 1),
             g->its, imin(g->ite, g->ide - 1), g->jte, g->ite};
  PW_LAUNCH_BOX(k_ssfinish, whole(g), s, dims_of(g), a);
  PW_RET();
}
