// Adjoints (transposes) of linear parts of the step, for gradients through it.
//
// (the advection tendencies' are in adv_adj.hip)
//
// * rk_update_scalar (wrf_dynamics.py:4055-4119): pointwise.
// * The column tridiagonal solve of advance_w (wrf_dynamics.py:3758-3765):
//   forward elimination w[k] = (w[k] - a[k] w[k-1]) alpha[k], k = 1..K, then
//   back substitution w[k] = w[k] - gamma[k] w[k+1], k = K-1..1.  The
//   adjoint runs the transposed sweeps in the opposite order (the back
//   substitution's transpose upwards, the elimination's downwards) and also
//   gives the sensitivities to a, alpha and gamma.
#include "common.h"
#include "consts.h"
#include "diff.h"
#include "openbc.h"

int pw_check_grid(const pywrf_grid_t* g, int r);
#define CHECK(g, r) do { int _e = pw_check_grid((g), (r)); if (_e) return _e; } while (0)

// ------------------------------------------------------------------ rk_update_scalar^T
struct AdjU {
  const float *lam, *msfty, *mu_old, *mu_new, *mu_base;
  float *lam_n, *lam_adv, *lam_sc, *lam_prev;
  float dt;
  Box bf, bi, bs;   // the updated box, the advection box (spec zone excluded), the sc_tend box
};

__global__ void k_rk_update_scalar_adj(Box all, Dims D, AdjU a) {
  int k, j, i;
  if (!box_point(all, k, j, i)) return;
  const float l = AT(a.lam, k, j, i);
  if (a.bf.has(k, j, i)) {
    const float muold = AT2(a.mu_old, j, i) + AT2(a.mu_base, j, i);
    const float munew = AT2(a.mu_new, j, i) + AT2(a.mu_base, j, i);
    const float lt = (a.dt * l) / munew;        // d q_new / d tendency
    AT(a.lam_n, k, j, i) += (muold * l) / munew;
    AT(a.lam_adv, k, j, i) = a.bi.has(k, j, i) ? lt * AT2(a.msfty, j, i) : 0.0f;
    if (a.lam_sc) AT(a.lam_sc, k, j, i) = a.bs.has(k, j, i) ? lt : 0.0f;
    AT(a.lam_prev, k, j, i) = 0.0f;
  } else {
    AT(a.lam_adv, k, j, i) = 0.0f;
    if (a.lam_sc) AT(a.lam_sc, k, j, i) = 0.0f;
    AT(a.lam_prev, k, j, i) = l;                // points the update leaves alone
  }
}

extern "C" int pywrf_rk_update_scalar_adjoint(const pywrf_grid_t* g, const float* lam_new, const float* msfty,
                                              const float* mu_old, const float* mu_new, const float* mu_base,
                                              double dt, int spec_zone, float* lam_n, float* lam_adv, float* lam_sc,
                                              float* lam_prev, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kde - 1 > g->nz || g->jde - 1 > g->ny || g->ide - 1 > g->nx) return PYWRF_E_RANGE;
  AdjU a;
  a.lam = lam_new; a.msfty = msfty; a.mu_old = mu_old; a.mu_new = mu_new; a.mu_base = mu_base;
  a.lam_n = lam_n; a.lam_adv = lam_adv; a.lam_sc = lam_sc; a.lam_prev = lam_prev;
  a.dt = F(dt);
  a.bf = mkbox(g->kts, g->kde - 1, g->jts, g->jde - 1, g->its, g->ide - 1);
  a.bi = mkbox(g->kts, imin(g->kte, g->kde - 1), imax(g->jts, g->jds + spec_zone), imin(g->jte, g->jde - spec_zone - 1),
               imax(g->its, g->ids + spec_zone), imin(g->ite, g->ide - spec_zone - 1));
  a.bs = mkbox(g->kts, g->kte - 1, g->jts, imin(g->jte, g->jde - 1), g->its, imin(g->ite, g->ide - 1));
  Box all = whole(g);
  PW_LAUNCH_BOX(k_rk_update_scalar_adj, all, s, dims_of(g), a);
  PW_RET();
}

// ------------------------------------------------------------------ tridiagonal solve and its adjoint
// One thread per column of advance_w's box; consecutive threads take
// consecutive i, so every level's access is a contiguous row segment.
struct Tri {
  const float *a, *alpha, *gamma;
  float* w;
  int K;   // levels 1..K are solved; level 0 holds the lower boundary value
};

__global__ void k_tridiag_solve(Box b, Dims D, Tri t) {
  int j, i;
  if (!box_column(b, j, i)) return;
  float prev = AT(t.w, 0, j, i);
  for (int k = 1; k <= t.K; ++k) {
    const float y = (AT(t.w, k, j, i) - AT(t.a, k, j, i) * prev) * AT(t.alpha, k, j, i);
    AT(t.w, k, j, i) = y;
    prev = y;
  }
  float next = prev;   // w[K]
  for (int k = t.K - 1; k >= 1; --k) {
    const float x = AT(t.w, k, j, i) - AT(t.gamma, k, j, i) * next;
    AT(t.w, k, j, i) = x;
    next = x;
  }
}

static bool tri_box(const pywrf_grid_t* g, Box& b, int& K) {
  K = g->kte - 1;
  b = mkbox(0, K + 1, imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2), imax(g->its, g->ids + 1),
            imin(g->ite, g->ide - 2));
  return g->kts == 0 && K >= 1 && K < g->nz;
}

extern "C" int pywrf_tridiag_solve(const pywrf_grid_t* g, const float* a, const float* alpha, const float* gamma,
                                   float* w, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  Box b;
  Tri t;
  if (!tri_box(g, b, t.K)) return PYWRF_E_RANGE;
  t.a = a; t.alpha = alpha; t.gamma = gamma; t.w = w;
  PW_LAUNCH_COLS(k_tridiag_solve, b, s, dims_of(g), t);
  PW_RET();
}

// Adjoint of the solve: given the right-hand side r (the input of the
// solve), the solution x and the sensitivity lam of x, writes the
// sensitivities of r (over lam, in place), a, alpha and gamma.  The forward
// elimination's intermediate y is recomputed from r.
struct TriAdj {
  const float *a, *alpha, *gamma, *r, *x;
  float *lam, *ga, *galpha, *ggamma, *y;
  int K;
};

__global__ void k_tridiag_adj(Box b, Dims D, TriAdj t) {
  int j, i;
  if (!box_column(b, j, i)) return;
  // recompute y (the elimination's output) into t.y
  float prev = AT(t.r, 0, j, i);
  AT(t.y, 0, j, i) = prev;
  for (int k = 1; k <= t.K; ++k) {
    const float y = (AT(t.r, k, j, i) - AT(t.a, k, j, i) * prev) * AT(t.alpha, k, j, i);
    AT(t.y, k, j, i) = y;
    prev = y;
  }
  // back substitution x[k] = y[k] - gamma[k] x[k+1], run for k = K-1..1:
  // transposed upwards; lam becomes the sensitivity of y
  AT(t.ggamma, 0, j, i) = 0.0f;
  AT(t.ggamma, t.K, j, i) = 0.0f;
  for (int k = 1; k <= t.K - 1; ++k) {
    const float lk = AT(t.lam, k, j, i);
    AT(t.ggamma, k, j, i) = -lk * AT(t.x, k + 1, j, i);
    AT(t.lam, k + 1, j, i) -= AT(t.gamma, k, j, i) * lk;
  }
  // elimination y[k] = (r[k] - a[k] y[k-1]) alpha[k], k = 1..K: transposed
  // downwards; lam becomes the sensitivity of r
  AT(t.ga, 0, j, i) = 0.0f;
  AT(t.galpha, 0, j, i) = 0.0f;
  for (int k = t.K; k >= 1; --k) {
    const float ly = AT(t.lam, k, j, i);
    const float al = AT(t.alpha, k, j, i);
    const float ym = AT(t.y, k - 1, j, i);
    const float lr = ly * al;
    AT(t.galpha, k, j, i) = ly * (AT(t.r, k, j, i) - AT(t.a, k, j, i) * ym);
    AT(t.ga, k, j, i) = -lr * ym;
    AT(t.lam, k, j, i) = lr;
    AT(t.lam, k - 1, j, i) -= AT(t.a, k, j, i) * lr;
  }
}

extern "C" int pywrf_tridiag_solve_adjoint(const pywrf_grid_t* g, const float* a, const float* alpha,
                                           const float* gamma, const float* r, const float* x, float* lam,
                                           float* grad_a, float* grad_alpha, float* grad_gamma, float* work,
                                           pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  TriAdj t;
  Box b;
  if (!tri_box(g, b, t.K)) return PYWRF_E_RANGE;
  t.a = a; t.alpha = alpha; t.gamma = gamma; t.r = r; t.x = x; t.lam = lam;
  t.ga = grad_a; t.galpha = grad_alpha; t.ggamma = grad_gamma; t.y = work;
  PW_LAUNCH_COLS(k_tridiag_adj, b, s, dims_of(g), t);
  PW_RET();
}

// adds v to *p (atomically: neighbouring columns share points); zero adds are skipped
__device__ inline void atomic_add(float* p, float v) { if (v != 0.0f) atomicAdd(p, v); }

__global__ void k_zero_n(float* p, long n) {
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) p[q] = 0.0f;
}

__global__ void k_zero_2(float* x, float* y, long n) {
  float* p = blockIdx.y ? y : x;
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) p[q] = 0.0f;
}

// ------------------------------------------------------------------ advance_w^T
// advance_w (wrf_dynamics.py:3641-3796) with respect to w, ph, t_2, t_2ave,
// u, v, ww, muts and muave (the coefficients -- mut, c2a, cqw, alt, the
// tridiagonal factors, the damping weights from ph_1 -- fixed).  It is linear
// in all but muts, whose derivatives take the forward's outputs t_2ave and w:
//   t2a[k]  = (0.5 ((1+e) t_2[k] + (1-e) t2a_in[k]) + muave t0) / (muts (t0 + t_1[k])),  k < K
//   rhs[k]  = ph[k] + msfty dts (ph_tend[k] + 0.5 g (1-e) w[k] - ...) / mut,            1 <= k <= K
//   wp[k]   = w[k] + ... (rhs, ph at k-1, k, k+1; t2a at k-1, k),                      1 <= k <= K
//   ws      = the column solve of wp (w[0] from the terrain slopes and u, v),
//   w_out   = (ws - dampwt mut w_save) / (1 + dampwt),
//   ph_out  = rhs + msfty 0.5 dts g (1+e) w_out / muts,
// with K = kte - 1, on the columns [jds+1, jde-2) x [ids+1, ide-2); every
// other point passes w, ph and t_2ave through.  w[0] is formed from the
// terrain slopes and u, v at levels 0..2 (cf1..cf3), and muave enters
// t2a's numerator and wp[k] as - dts g muave / msfty.  work, work2: 3-D
// scratch.
struct AdjW {
  const float *lT, *lW, *lP;                      // sensitivities of the outputs t_2ave, w, ph
  const float *mut, *muts, *t_1, *ph_1, *phb, *c2a, *cqw, *alt, *a, *alpha, *gamma, *rdnw, *rdn, *msfty;
  const float *t2a_out, *w_out, *ht, *msftx, *cf;  // the forward's outputs t_2ave, w; terrain, map factor, cf1..3
  const float *fnm, *fnp;
  float *lw_in, *lph_in, *lt2, *lt2a_in, *work, *work2;
  float *lu, *lv, *lmuts, *lmuave, *lww;           // u, v: zeroed by the caller, atomic adds
  float *lrw, *lpht, *lws;                         // rw_tend, ph_tend, w_save
  float* lt1;                                      // t_1
  const float *ww, *wsave;                         // the call's ww and w_save
  float* lph1;                                     // ph_1: vertical advection and damping
  float dts, t0, ep1, em1, dampmag, hpi, hdepth, rdx, rdy;
  int K, j0, j1, i0, i1;
};

// The column kernels below take 64 columns of a row to a block of 8 waves and
// deal the levels out to the waves: a thread that walks all the levels of a
// column waits for memory at each of them, and a plane has too few columns
// (225 waves at 120 x 120, on 1024 SIMDs) to hide it.
#define CA_COLS 64
#define CA_WAVES 8
#define CA_THREADS (CA_COLS * CA_WAVES)

// the wave's number, known to the compiler to be the same in all its lanes
__device__ __forceinline__ int ca_wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x / CA_COLS); }

// The sum over the block's waves of each lane's v, in every wave.
__device__ inline float ca_sum(float (*red)[CA_COLS], int g, int lane, float v) {
  red[g][lane] = v;
  __syncthreads();
  float t = 0.0f;
#pragma unroll
  for (int n = 0; n < CA_WAVES; ++n) t += red[n][lane];
  return t;
}

static inline dim3 ca_grid(const pywrf_grid_t* g, int cols) {
  return dim3((unsigned)((g->nx + cols - 1) / cols), (unsigned)g->ny);
}

// Wave g takes levels g, g + 8, ...  Four per-level arrays pass values between
// the waves: W the sensitivity of the solved w, A1 gamma and then each half
// level's H = P (S[k+1] - S[k]), S[k] = mi cqw 0.5 dts g rdn W[k] (the two
// neighbours of a half level both read it), A2 alpha, A3 a and then that of rhs.
// One wave runs the sweeps.  The arrays lie in LDS; BIG (beyond 58 levels, where
// they would pass 64 KB with the sums') keeps them in the block's own columns of the scratch and
// of outputs that a later phase writes.  At
// 120 x 120 x 41 35 us, where one thread a column took 375 (and 10 launches zeroed
// its outputs).
template <bool BIG>
__global__ void __launch_bounds__(CA_THREADS) k_advance_w_adj(Dims D, AdjW a) {
  extern __shared__ float sm[];
  __shared__ float s_d[CA_WAVES][CA_COLS], s_m[CA_WAVES][CA_COLS], s_s[CA_WAVES][CA_COLS];
  constexpr int LV = 6;   // levels whose loads are issued together
  const int nz = D.nz, K = a.K;
  const int lane = threadIdx.x % CA_COLS, g = ca_wave();
  const int j = (int)blockIdx.y, i = (int)blockIdx.x * CA_COLS + lane;
  const bool row = j >= a.j0 && j < a.j1 && a.i0 < a.i1;
  const bool h = row && i >= a.i0 && i < a.i1;
  if (i < D.nx && !h) {
    for (int k = g; k < nz; k += CA_WAVES) {
      const long q = D.ix(k, j, i);
      const float x = a.lW[q], y = a.lP[q], z = a.lT[q];
      a.lw_in[q] = x; a.lph_in[q] = y; a.lt2a_in[q] = z;
      a.lt2[q] = 0.0f; a.lww[q] = 0.0f; a.lrw[q] = 0.0f; a.lpht[q] = 0.0f; a.lws[q] = 0.0f; a.lt1[q] = 0.0f;
      a.lph1[q] = 0.0f;
    }
    if (g == 0) { AT2(a.lmuts, j, i) = 0.0f; AT2(a.lmuave, j, i) = 0.0f; }
  }
  if (!row) return;   // the whole block
  const int ic = imin(imax(i, a.i0), a.i1 - 1);   // lanes outside the box run its edge column and store nothing
  const long q0 = D.ix2(j, ic), plane = D.plane();
  float* W = BIG ? a.work + q0 : sm + lane;
  float* A1 = BIG ? a.lww + q0 : sm + 1 * nz * CA_COLS + lane;
  float* A2 = BIG ? a.lrw + q0 : sm + 2 * nz * CA_COLS + lane;
  float* A3 = BIG ? a.work2 + q0 : sm + 3 * nz * CA_COLS + lane;
  const long st = BIG ? plane : CA_COLS;
  const bool own = !BIG || h;                     // may write the per-level arrays
  const float G = F(pw::g);
  const float my = a.msfty[q0], mi = 1.0f / my, mut = a.mut[q0], muts = a.muts[q0];
  // the damping weights (as the forward forms them) and the sensitivity of the solved w
  const float htop = (AT(a.ph_1, K, j, ic) + AT(a.phb, K, j, ic)) / G, hbot = htop - a.hdepth;
  float dsum = 0.0f;
  for (int kb = g; kb < nz; kb += CA_WAVES * LV) {
    float lW[LV], lP[LV], p1[LV], pb[LV], wsv[LV], wo[LV], ga[LV], al[LV], av[LV];
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const long q = q0 + imin(kb + m * CA_WAVES, nz - 1) * plane;
      lW[m] = a.lW[q]; lP[m] = a.lP[q]; p1[m] = a.ph_1[q]; pb[m] = a.phb[q]; wsv[m] = a.wsave[q]; wo[m] = a.w_out[q];
      ga[m] = a.gamma[q]; al[m] = a.alpha[q]; av[m] = a.a[q];
    }
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const int k = kb + m * CA_WAVES;
      if (k >= nz) break;
      const bool upd = k >= 1 && k <= K;
      const float hk = (p1[m] + pb[m]) / G, lwd = lW[m] + my * 0.5f * a.dts * G * a.ep1 / muts * lP[m];
      float dw = 0.0f, dd = 0.0f;
      if (upd && hk >= hbot) {
        const float th = a.hpi * (hk - hbot) / a.hdepth, sn = sinf(th);
        dw = a.dampmag * (sn * sn);
        // the weight's dependence on ph_1: through hk at this level and hbot (from level K); at level K the two cancel
        if (k < K)
          dd = lwd * (-mut * wsv[m] - wo[m]) / (1.0f + dw) *
               (a.dampmag * 2.0f * sn * cosf(th) * a.hpi / a.hdepth) / G;
      }
      dsum += dd;
      if (own) { W[k * st] = lwd / (1.0f + dw); A1[k * st] = ga[m]; A2[k * st] = al[m]; A3[k * st] = av[m]; }
      if (h) {
        const long q = q0 + k * plane;
        a.lws[q] = upd ? -dw * mut / (1.0f + dw) * lwd : 0.0f;   // the damping's pull towards w_save
        a.lph1[q] = dd;                                          // completed below by this thread
      }
    }
  }
  s_d[g][lane] = dsum;
  __syncthreads();
  // the column solve, transposed: back substitution upwards, elimination downwards.  Eight levels' operands at a
  // time are read before the dependent arithmetic.
  const float a_1 = A3[1 * st];
  if (g == 0 && own) {
    float w = W[1 * st];
    for (int kb = 1; kb < K; kb += 8) {
      float n[8], c[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) { const int k = imin(kb + m, K - 1); n[m] = W[(k + 1) * st]; c[m] = A1[k * st]; }
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        if (kb + m >= K) break;
        w = n[m] - c[m] * w;
        W[(kb + m + 1) * st] = w;
      }
    }
    for (int kb = K; kb >= 1; kb -= 8) {
      float n[8], c[8], e[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int k = imax(kb - m, 1);
        n[m] = W[imax(k - 1, 1) * st]; c[m] = A2[k * st]; e[m] = A3[k * st];
      }
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int k = kb - m;
        if (k < 1) break;
        w = w * c[m];
        W[k * st] = w;
        w = n[m] - e[m] * w;
      }
    }
  }
  __syncthreads();
  auto S = [&](int k, float cq) { return mi * cq * (0.5f * a.dts * G * level(a.rdn, k)) * W[k * st]; };
  // H of each half level (between k and k + 1); the top one also takes the top level's predictor
  for (int kb = g; kb < K; kb += CA_WAVES * LV) {
    float c2[LV], cq[LV], cqp[LV];
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const long q = q0 + imin(kb + m * CA_WAVES, K - 1) * plane;
      c2[m] = a.c2a[q]; cq[m] = a.cqw[q]; cqp[m] = a.cqw[q + plane];
    }
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const int k = kb + m * CA_WAVES;
      if (k >= K) break;
      const float rw = level(a.rdnw, k), P = c2[m] * rw / mut;
      const float lo = k >= 1 ? S(k, cq[m]) : 0.0f;
      float H;
      if (k < K - 1) H = P * (S(k + 1, cqp[m]) - lo);
      else H = -P * lo - mi * (-0.5f * a.dts * G / mut * rw * rw * 2.0f * c2[m]) * W[K * st];
      if (own) A1[k * st] = H;
    }
  }
  __syncthreads();
  // rhs, ph, w and the forcings; t2a[k] for k < K from t_2, t2a_in, muave and muts
  const float gam = my * a.dts * 0.5f * G * a.em1 / mut, cp = my * 0.5f * a.dts * G * a.ep1;
  float smu = 0.0f, sms = 0.0f;
  for (int kb = g; kb < nz; kb += CA_WAVES * LV) {
    float lP[LV], lT[LV], c2[LV], alt[LV], t1[LV], to[LV], wo[LV];
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const long q = q0 + imin(kb + m * CA_WAVES, nz - 1) * plane;
      lP[m] = a.lP[q]; lT[m] = a.lT[q]; c2[m] = a.c2a[q]; alt[m] = a.alt[q]; t1[m] = a.t_1[q]; to[m] = a.t2a_out[q];
      wo[m] = a.w_out[q];
    }
#pragma unroll
    for (int m = 0; m < LV; ++m) {
      const int k = kb + m * CA_WAVES;
      if (k >= nz) break;
      const long q = q0 + k * plane;
      const bool upd = k >= 1 && k <= K;
      const float L = upd ? W[k * st] : 0.0f;
      const float dH = (k < K ? A1[k * st] : 0.0f) - (upd ? A1[(k - 1) * st] : 0.0f);
      const float r = upd ? lP[m] + a.ep1 * dH : 0.0f;
      if (upd) {
        smu -= a.dts * G * mi * L;
        sms -= cp * wo[m] / (muts * muts) * lP[m];
      }
      float l = lT[m];
      if (k < K) {
        const float tg = a.dts * G * mi, ca = c2[m] * alt[m];
        if (k >= 1) l += tg * level(a.rdn, k) * ca * L;
        if (k + 1 < K) l -= tg * level(a.rdn, k + 1) * ca * W[(k + 1) * st];
        else l -= tg * 2.0f * level(a.rdnw, k) * ca * W[K * st];
        const float den = muts * (a.t0 + t1[m]);
        smu += a.t0 / den * l;
        sms -= to[m] / muts * l;
        if (h) {
          a.lt2[q] = 0.5f * a.ep1 / den * l;
          a.lt2a_in[q] = 0.5f * a.em1 / den * l;
          a.lt1[q] = -to[m] / (a.t0 + t1[m]) * l;
        }
      } else if (h) {
        a.lt2[q] = 0.0f;
        a.lt2a_in[q] = l;
        a.lt1[q] = 0.0f;
      }
      if (h) {
        a.lph_in[q] = upd ? a.em1 * dH + r : k < 1 ? lP[m] + a.em1 * dH : lP[m];
        a.lw_in[q] = upd ? L + gam * r : 0.0f;             // w[0] is overwritten from the terrain
        a.lpht[q] = upd ? my * a.dts / mut * r : 0.0f;     // rhs holds msfty dts ph_tend / mut
        a.lrw[q] = upd ? a.dts * L : 0.0f;                 // rw_tend enters the predictor as dts rw_tend
      }
      if (own) A3[k * st] = r;
    }
  }
  // the surface w (from the terrain and u, v at levels 0..2) enters the solve at level 1 and is an output itself
  if (g == CA_WAVES - 1 && h) {
    const float lw0 = AT(a.lW, 0, j, i) - a_1 * W[1 * st];
    const float htc = AT2(a.ht, j, i), mx = AT2(a.msftx, j, i);
    const float cy = my * 0.5f * a.rdy * lw0, cx = mx * 0.5f * a.rdx * lw0;
    const float vn = cy * (AT2(a.ht, j + 1, i) - htc), vs = cy * (htc - AT2(a.ht, j - 1, i));
    const float ue = cx * (AT2(a.ht, j, i + 1) - htc), uw = cx * (htc - AT2(a.ht, j, i - 1));
    for (int c = 0; c < 3; ++c) {
      const float cf = level(a.cf, c);
      atomic_add(&AT(a.lv, c, j + 1, i), cf * vn);
      atomic_add(&AT(a.lv, c, j, i), cf * vs);
      atomic_add(&AT(a.lu, c, j, i + 1), cf * ue);
      atomic_add(&AT(a.lu, c, j, i), cf * uw);
    }
  }
  s_m[g][lane] = smu;
  s_s[g][lane] = sms;
  __syncthreads();
  if (!h) return;
  // rhs[k] = ph[k] + msfty dts 0.5 g (1-e) w[k] / mut - msfty dts (fnm[k] wup[k] + fnp[k] wdn[k]) / mut
  // + (terms without w, ph, ww), wup / wdn = 0.5 (ww[k+1] + ww[k]) / (ww[k] + ww[k-1]) times rdnw and the
  // ph_1 + phb differences above / below level k (k < K): each half level's term is in the two levels beside it
  auto Fh = [&](int k) {
    const float c = -a.dts * my / mut;
    return (k >= 1 ? level(a.fnm, k) * (c * A3[k * st]) : 0.0f) +
           (k + 1 < K ? level(a.fnp, k + 1) * (c * A3[(k + 1) * st]) : 0.0f);
  };
  for (int k = g; k < nz; k += CA_WAVES) {
    const long q = q0 + k * plane;
    const long qm = q0 + imax(k - 1, 0) * plane, qp = q0 + imin(k + 1, nz - 1) * plane;
    const float p0 = a.ph_1[q], pm = a.ph_1[qm], pp = a.ph_1[qp], b0 = a.phb[q], bm = a.phb[qm], bp = a.phb[qp];
    const float w0 = a.ww[q], wm = a.ww[qm], wp = a.ww[qp];
    float lww = 0.0f, l1 = a.lph1[q];
    if (k < K) {
      const float f = 0.5f * level(a.rdnw, k) * Fh(k);
      lww += (pp - p0 + bp - b0) * f;
      l1 -= (wp + w0) * f;
    }
    if (k >= 1 && k <= K) {
      const float f = 0.5f * level(a.rdnw, k - 1) * Fh(k - 1);
      lww += (p0 - pm + b0 - bm) * f;
      l1 += (w0 + wm) * f;
    }
    if (k == K)
      for (int n = 0; n < CA_WAVES; ++n) l1 -= s_d[n][lane];
    a.lww[q] = lww;
    a.lph1[q] = l1;
  }
  if (g == 0) {
    float x = 0.0f, y = 0.0f;
    for (int n = 0; n < CA_WAVES; ++n) { x += s_m[n][lane]; y += s_s[n][lane]; }
    a.lmuave[q0] = x;
    a.lmuts[q0] = y;
  }
}

extern "C" int pywrf_advance_w_adjoint(const pywrf_grid_t* g, const float* lam_t2ave_out, const float* lam_w_out,
                                       const float* lam_ph_out, const float* mut, const float* muts,
                                       const float* t_1, const float* ph_1, const float* phb, const float* c2a,
                                       const float* cqw, const float* alt, const float* a, const float* alpha,
                                       const float* gamma, double dts, double t0, double epssm, const float* rdnw,
                                       const float* rdn, const float* msfty, const float* t2ave_out,
                                       const float* w_out, const float* ht, const float* msftx, const float* cf,
                                       double rdx, double rdy, const float* fnm, const float* fnp, float* lam_w,
                                       float* lam_ph, float* lam_t_2, float* lam_t2ave, float* lam_u,
                                       float* lam_v, float* lam_muts, float* lam_muave, float* lam_ww,
                                       float* lam_rw_tend, float* lam_ph_tend, float* lam_w_save, float* lam_t_1,
                                       const float* ww, const float* w_save, float* lam_ph_1, float* work,
                                       float* work2, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kts != 0 || g->kte > g->nz || g->kte < 3) return PYWRF_E_RANGE;
  AdjW p;
  p.lT = lam_t2ave_out; p.lW = lam_w_out; p.lP = lam_ph_out;
  p.mut = mut; p.muts = muts; p.t_1 = t_1; p.ph_1 = ph_1; p.phb = phb; p.c2a = c2a; p.cqw = cqw; p.alt = alt;
  p.a = a; p.alpha = alpha; p.gamma = gamma; p.rdnw = rdnw; p.rdn = rdn; p.msfty = msfty;
  p.lw_in = lam_w; p.lph_in = lam_ph; p.lt2 = lam_t_2; p.lt2a_in = lam_t2ave; p.work = work; p.work2 = work2;
  p.t2a_out = t2ave_out; p.w_out = w_out; p.ht = ht; p.msftx = msftx; p.cf = cf;
  p.lu = lam_u; p.lv = lam_v; p.lmuts = lam_muts; p.lmuave = lam_muave; p.lww = lam_ww;
  p.lrw = lam_rw_tend; p.lpht = lam_ph_tend; p.lws = lam_w_save; p.lt1 = lam_t_1;
  p.ww = ww; p.wsave = w_save; p.lph1 = lam_ph_1;
  p.fnm = fnm; p.fnp = fnp;
  p.rdx = F(rdx); p.rdy = F(rdy);
  p.dts = F(dts); p.t0 = F(t0); p.ep1 = F(1. + epssm); p.em1 = F(1. - epssm);
  p.dampmag = F(dts * 0.2); p.hpi = F(0.5 * 3.14159265359); p.hdepth = 5000.0f;
  p.K = g->kte - 1;
  p.j0 = imax(g->jts, g->jds + 1); p.j1 = imin(g->jte, g->jde - 2);
  p.i0 = imax(g->its, g->ids + 1); p.i1 = imin(g->ite, g->ide - 2);
  if (p.j0 < 1 || p.i0 < 1 || p.j1 + 1 > g->ny || p.i1 + 1 > g->nx || g->nz < 3) return PYWRF_E_RANGE;
  const long n3 = (long)g->nz * g->ny * g->nx;
  hipLaunchKernelGGL(k_zero_2, dim3(512, 2), dim3(256), 0, (hipStream_t)s, lam_u, lam_v, n3);
  const size_t lds = 4 * sizeof(float) * CA_COLS * (size_t)g->nz;
  if (lds + 3 * sizeof(float) * CA_THREADS <= 64 * 1024)
    hipLaunchKernelGGL(k_advance_w_adj<false>, ca_grid(g, CA_COLS), dim3(CA_THREADS), lds, (hipStream_t)s, dims_of(g), p);
  else
    hipLaunchKernelGGL(k_advance_w_adj<true>, ca_grid(g, CA_COLS), dim3(CA_THREADS), 0, (hipStream_t)s, dims_of(g), p);
  PW_RET();
}

// ------------------------------------------------------------------ advance_uv^T
// advance_uv (wrf_dynamics.py:3391-3525) is linear in u, v, ru_tend, rv_tend,
// p, ph, al, mu and mudf once alt, pb, php, cqu / cqv, the column masses
// muu / muv and the map factors are fixed.  For a u point (k, j, i) of its box
//   u += dts ru_tend - dts cqu dpx + mudf_x,
//   dpx = A (ph[k+1,i] - ph[k+1,i-1] + ph[k,i] - ph[k,i-1]
//            + (alt[k,i] + alt[k,i-1]) (p[k,i] - p[k,i-1]) + (al[k,i] + al[k,i-1]) (pb[k,i] - pb[k,i-1]))
//       + B[k] (rdnw[k] (dpn[k+1] - dpn[k]) - 0.5 (mu[i-1] + mu[i])),
//   A = msfux / msfuy 0.5 rdx muu,  B[k] = msfux / msfuy rdx (php[k,i] - php[k,i-1]),
//   dpn[0] from p[0..2] with cf1..cf3, dpn[k] = 0.5 (fnm[k] (p[k,i] + p[k,i-1]) + fnp[k] (p[k-1,i] + p[k-1,i-1])),
//   dpn[kde-1] = 0,  mudf_x = -emdiv dx (mudf[i] - mudf[i-1]) / msfuy;
// v the same along j; u, v pass through.
struct AdjUV {
  const float *lu, *lv, *alt, *pb, *php, *cqu, *cqv, *muu, *muv, *msfux, *msfuy, *msfvx, *msfvy, *msfvx_inv;
  const float *fnm, *fnp, *rdnw, *cf;
  float *gp, *gph, *gal, *gmu, *gmudf, *grut, *grvt, *glu, *glv;
  float dts, rdx, rdy, emdiv, dx, dy;
  int k0, k1, kde1;              // levels [k0, k1) of the box; dpn is zero at kde1 = kde - 1
  Box bu, bv;                    // the u and v boxes (j, i ranges)
};


// In gather form: each column reads the two u and two v points around it (its
// own, where it is the upper side of the difference, and the next one, where it
// is the lower).  Wave g takes the run of levels [g L, (g + 1) L) of 64 columns
// and walks it with the levels below and above at hand (a run evaluates two
// levels more than it writes), the next level's 23 values loaded before this
// one's stores; the plane's sums go over the waves in LDS.  At 120 x 120 x 41
// 16 us, where one thread a column with atomic adds took 113 + 107 (u, v).
struct UVLevel { float l[4], cq[4], php[5], alt[5], pb[5]; };   // faces: u here, u east, v here, v north; c, w, e, s, n
struct UVSum { float ph, p, al, c; };                           // the level's shares of ph, p (alt term), al; rdnw BG

__global__ void __launch_bounds__(CA_THREADS) k_advance_uv_adj(Dims D, AdjUV a) {
  __shared__ float s_mu[CA_WAVES][CA_COLS], s_df[CA_WAVES][CA_COLS];
  const int lane = threadIdx.x % CA_COLS, g = ca_wave(), L = (D.nz + CA_WAVES - 1) / CA_WAVES;
  const int j = (int)blockIdx.y, i = (int)blockIdx.x * CA_COLS + lane, ic = imin(i, D.nx - 1);
  const bool w = i < D.nx;
  const int ie = imin(ic + 1, D.nx - 1), iw = imax(ic - 1, 0), jn = imin(j + 1, D.ny - 1), js = imax(j - 1, 0);
  const bool on[4] = {a.bu.has2(j, ic), ic + 1 < D.nx && a.bu.has2(j, ic + 1), a.bv.has2(j, ic),
                      j + 1 < D.ny && a.bv.has2(j + 1, ic)};
  // per face: map factor times 1 / dx, times half the mass, and the divergence damping's weight with its sign
  const float mf[4] = {AT2(a.msfux, j, ic) / AT2(a.msfuy, j, ic) * a.rdx, AT2(a.msfux, j, ie) / AT2(a.msfuy, j, ie) * a.rdx,
                       AT2(a.msfvy, j, ic) / AT2(a.msfvx, j, ic) * a.rdy, AT2(a.msfvy, jn, ic) / AT2(a.msfvx, jn, ic) * a.rdy};
  const float A[4] = {mf[0] * 0.5f * AT2(a.muu, j, ic), mf[1] * 0.5f * AT2(a.muu, j, ie),
                      mf[2] * 0.5f * AT2(a.muv, j, ic), mf[3] * 0.5f * AT2(a.muv, jn, ic)};
  const float dd[4] = {-a.emdiv * a.dx / AT2(a.msfuy, j, ic), a.emdiv * a.dx / AT2(a.msfuy, j, ie),
                       -a.emdiv * a.dy * AT2(a.msfvx_inv, j, ic), a.emdiv * a.dy * AT2(a.msfvx_inv, jn, ic)};
  auto load = [&](int k) {
    k = imin(imax(k, 0), D.nz - 1);
    const unsigned c = D.ob(k, j, ic), e = D.ob(k, j, ie), v = D.ob(k, jn, ic), s = D.ob(k, js, ic), x = D.ob(k, j, iw);
    UVLevel r;
    r.l[0] = at_b(a.lu, c); r.l[1] = at_b(a.lu, e); r.l[2] = at_b(a.lv, c); r.l[3] = at_b(a.lv, v);
    r.cq[0] = at_b(a.cqu, c); r.cq[1] = at_b(a.cqu, e); r.cq[2] = at_b(a.cqv, c); r.cq[3] = at_b(a.cqv, v);
    r.php[0] = at_b(a.php, c); r.php[1] = at_b(a.php, x); r.php[2] = at_b(a.php, e); r.php[3] = at_b(a.php, s); r.php[4] = at_b(a.php, v);
    r.alt[0] = at_b(a.alt, c); r.alt[1] = at_b(a.alt, x); r.alt[2] = at_b(a.alt, e); r.alt[3] = at_b(a.alt, s); r.alt[4] = at_b(a.alt, v);
    r.pb[0] = at_b(a.pb, c); r.pb[1] = at_b(a.pb, x); r.pb[2] = at_b(a.pb, e); r.pb[3] = at_b(a.pb, s); r.pb[4] = at_b(a.pb, v);
    return r;
  };
  auto sums = [&](const UVLevel& r, int k) {
    UVSum t = {0.0f, 0.0f, 0.0f, 0.0f};
    if (k < a.k0 || k >= a.k1) return t;
    // the face's difference is upper minus lower; the column is the upper side of faces 0 and 2
    const float dphp[4] = {r.php[0] - r.php[1], r.php[2] - r.php[0], r.php[0] - r.php[3], r.php[4] - r.php[0]};
    const float salt[4] = {r.alt[0] + r.alt[1], r.alt[2] + r.alt[0], r.alt[0] + r.alt[3], r.alt[4] + r.alt[0]};
    const float dpb[4] = {r.pb[0] - r.pb[1], r.pb[2] - r.pb[0], r.pb[0] - r.pb[3], r.pb[4] - r.pb[0]};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (!on[f]) continue;
      const float G = -a.dts * r.cq[f] * r.l[f], AG = A[f] * G;   // sensitivity of dp at the face
      const float sg = f % 2 ? -AG : AG;
      t.ph += sg;
      t.p += sg * salt[f];
      t.al += AG * dpb[f];
      t.c += mf[f] * dphp[f] * G;
    }
    return t;
  };
  const int ka = g * L, kb = imin(ka + L, D.nz);
  float smu = 0.0f, sdf = 0.0f;
  if (ka < kb) {
    UVLevel cur = load(ka), nxt = load(ka + 1);
    UVSum below = sums(load(ka - 1), ka - 1), here = sums(cur, ka), above;
    // dpn[0], from p[0..2] with cf1..cf3, has c[0] alone
    const float c0 = ka < 3 ? level(a.rdnw, 0) * sums(load(0), 0).c : 0.0f;
    auto dpn = [&](int k, float lo, float hi) {   // the sensitivity of dpn[k], 1 <= k < k1, below the model's top
      return k >= 1 && k < a.k1 && k < a.kde1 ? level(a.rdnw, k - 1) * lo - level(a.rdnw, k) * hi : 0.0f;
    };
    for (int k = ka; k < kb; ++k) {
      above = sums(nxt, k + 1);
      const UVLevel far = load(k + 2);
      const long q = D.ix(k, j, ic);
      float p = here.p;
      if (k < 3 && a.k1 > 0) p += 0.5f * level(a.cf, k) * -c0;
      p += 0.5f * level(a.fnm, k) * dpn(k, below.c, here.c);
      if (k + 1 < a.k1) p += 0.5f * level(a.fnp, k + 1) * dpn(k + 1, here.c, above.c);
      const bool lv = k >= a.k0 && k < a.k1;
      if (lv) {
        smu += -0.5f * here.c;
#pragma unroll
        for (int f = 0; f < 4; ++f) sdf += on[f] ? dd[f] * cur.l[f] : 0.0f;
      }
      if (w) {
        a.gp[q] = p;
        a.gph[q] = here.ph + below.ph;
        a.gal[q] = here.al;
        a.glu[q] = cur.l[0];
        a.glv[q] = cur.l[2];
        a.grut[q] = lv && on[0] ? a.dts * cur.l[0] : 0.0f;
        a.grvt[q] = lv && on[2] ? a.dts * cur.l[2] : 0.0f;
      }
      below = here; here = above; cur = nxt; nxt = far;
    }
  }
  const float mu = ca_sum(s_mu, g, lane, smu), df = ca_sum(s_df, g, lane, sdf);
  if (g == 0 && w) {
    AT2(a.gmu, j, i) = mu;
    AT2(a.gmudf, j, i) = df;
  }
}

// Outputs: lam_u / lam_v (= the sensitivities of the outputs: u and v pass
// through), lam_p, lam_ph, lam_al, lam_mu, lam_mudf, lam_ru_tend,
// lam_rv_tend, each written in full.

extern "C" int pywrf_advance_uv_adjoint(const pywrf_grid_t* g, const float* lam_u_out, const float* lam_v_out,
                                        const float* pb, const float* php, const float* alt, const float* muu,
                                        const float* cqu, const float* muv, const float* cqv, const float* msfux,
                                        const float* msfuy, const float* msfvx, const float* msfvx_inv,
                                        const float* msfvy, double rdx, double rdy, double dts, const float* cf,
                                        const float* fnm, const float* fnp, double emdiv, const float* rdnw,
                                        int spec_zone, float* lam_u, float* lam_v, float* lam_p, float* lam_ph,
                                        float* lam_al, float* lam_mu, float* lam_mudf, float* lam_ru_tend,
                                        float* lam_rv_tend, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kts != 0 || g->nz < 3 || g->kde > g->nz || g->kte > g->nz) return PYWRF_E_RANGE;
  AdjUV a;
  a.lu = lam_u_out; a.lv = lam_v_out; a.alt = alt; a.pb = pb; a.php = php; a.cqu = cqu; a.cqv = cqv;
  a.muu = muu; a.muv = muv; a.msfux = msfux; a.msfuy = msfuy; a.msfvx = msfvx; a.msfvy = msfvy;
  a.msfvx_inv = msfvx_inv; a.fnm = fnm; a.fnp = fnp; a.rdnw = rdnw; a.cf = cf;
  a.gp = lam_p; a.gph = lam_ph; a.gal = lam_al; a.gmu = lam_mu; a.gmudf = lam_mudf;
  a.grut = lam_ru_tend; a.grvt = lam_rv_tend; a.glu = lam_u; a.glv = lam_v;
  a.dts = F(dts); a.rdx = F(rdx); a.rdy = F(rdy); a.emdiv = F(emdiv); a.dx = F(1.0 / rdx); a.dy = F(1.0 / rdy);
  a.k0 = g->kts; a.k1 = imin(g->kte, g->kde - 1); a.kde1 = g->kde - 1;
  const int i0 = imax(g->its, g->ids + spec_zone), i1 = imin(g->ite, g->ide - spec_zone - 1);
  const int j0 = imax(g->jts, g->jds + spec_zone), j1 = imin(g->jte, g->jde - spec_zone - 1);
  const int iu1 = imin(g->ite, g->ide - spec_zone), jv1 = imin(g->jte, g->jde - spec_zone);
  if (i0 < 1 || j0 < 1 || iu1 > g->nx || jv1 > g->ny || a.k1 + 1 > g->nz) return PYWRF_E_RANGE;
  a.bu = mkbox(0, 1, j0, j1, i0, iu1);
  a.bv = mkbox(0, 1, j0, jv1, i0, i1);
  hipLaunchKernelGGL(k_advance_uv_adj, ca_grid(g, CA_COLS), dim3(CA_THREADS), 0, (hipStream_t)s, dims_of(g), a);
  PW_RET();
}

// ------------------------------------------------------------ advance_mu_t adjoint
// The transpose of advance_mu_t (wrf_dynamics.py:3528-3638) with respect to u,
// v, ww, mu, muave, muts, mudf, t, t_ave, ft and mu_tend, with t_1 and the
// map factors held fixed (u_1, v_1 and ww_1 enter additively).  On a column
// (j, i) of the box, levels k < k1 = kte - 1:
//   dvdxi[k] = msftx msfty (rdy (v[k,j+1] - v[k,j]) + rdx (u[k,i+1] - u[k,i]) + terms in u_1, v_1),
//   S = sum_k dnw[k] dvdxi[k] + mu_tend,  mu' = mu + dts S,  mudf' = S,  muts' = mut + mu',
//   muave' = 0.5 ((1 + epssm) mu' + (1 - epssm) mu),
//   ww'[0] = ww[0] - ww_1[0],  ww'[k] = ww[0] - sum_{m<k} dnw[m] (S + dvdxi[m]) / msfty - ww_1[k],
//   wdtn[k] = ww'[k] (fnm[k] t_1[k] + fnp[k] t_1[k-1]) (0 < k < k1; 0 at 0 and k1),
//   t_ave' = t,  t' = t + msfty dts ft - dts msfty (msftx (0.5 rdy (v[k,j+1] (t_1[j+1] + t_1) - v (t_1 + t_1[j-1]))
//                    + 0.5 rdx (u[i+1] (t_1[i+1] + t_1) - u (t_1 + t_1[i-1]))) + rdnw[k] (wdtn[k+1] - wdtn[k])).
// Outside the box every output is its input.  The sensitivity of dvdxi takes
// the suffix sums of the ww sensitivities (their own and, through wdtn, t's)
// and the total sensitivity of S.
struct AdjMuT {
  const float *lww, *lt, *ltave, *lmuave, *lmuts, *lmudf, *lmu;
  const float *t1, *msftx, *msfty, *dnw, *fnm, *fnp, *rdnw;
  float *gww, *gu, *gv, *gmu, *gmuave, *gmuts, *gmudf, *gt, *gtave, *gft, *gmut;
  // the large-step fields: u_1, v_1 in the divergence (times muu / msfuy, muv msfvx_inv), ww_1
  // subtracted from ww, t_1 in the theta fluxes (with u, v and the forward's ww)
  const float *u, *v, *wwo, *muu, *muv, *msfuy, *msfvx_inv;
  float *gu1, *gv1, *gww1, *gt1;
  float rdx, rdy, dts, epssm;
  int k1;
};

// In gather form: the faces' shares of a column come from it and from its
// western and southern neighbours.  A block's 64 lanes are 63 columns and, in
// lane 0, the one west of them, whose shares reach lane 1 by a lane shift; of
// the row to the south the block forms the sums again (three more arrays read,
// where a second kernel would write and read the sensitivity of dvdxi).  Wave g takes a
// run of levels: a first pass down it gives the run's sum of the ww
// sensitivities, and, with the sums of the runs above, a second pass
// everything else.  At 120 x 120 x 41 21 us, where one thread
// a column with atomic adds took 227 (and 15 launches prepared its outputs).
struct MuTLevel { float lww, lt, t1, lwws, lts, t1s, lte, ltn, t1w, ltave, wwo, u, ue, v, vn; };

__global__ void __launch_bounds__(CA_THREADS) k_advance_mu_t_adj(Box b, Dims D, AdjMuT a) {
  __shared__ float s_r[2][CA_WAVES][CA_COLS], s_a[2][CA_WAVES][CA_COLS], s_dn[CA_WAVES];
  const int lane = threadIdx.x % CA_COLS, g = ca_wave(), L = (D.nz + CA_WAVES - 1) / CA_WAVES;
  const int j = (int)blockIdx.y, i = (int)blockIdx.x * (CA_COLS - 1) - 1 + lane;
  const int ic = imin(imax(i, 0), D.nx - 1);
  const int ie = imin(ic + 1, D.nx - 1), iw = imax(ic - 1, 0), jn = imin(j + 1, D.ny - 1), js = imax(j - 1, 0);
  const bool own = lane > 0 && i < D.nx;
  const bool in = i >= 0 && b.has2(j, i), ins = b.has2(j - 1, i), inn = b.has2(j + 1, i), ine = b.has2(j, i + 1);
  const float mfx = AT2(a.msftx, j, ic), mfy = AT2(a.msfty, j, ic);
  const float mfxs = AT2(a.msftx, js, ic), mfys = AT2(a.msfty, js, ic);
  const float e = a.epssm, c = a.dts * mfy, cs = a.dts * mfys;
  auto lmn_of = [&](int jj) {
    return AT2(a.lmu, jj, ic) + AT2(a.lmuts, jj, ic) + 0.5f * (1.0f + e) * AT2(a.lmuave, jj, ic);
  };
  const float lmn = lmn_of(j), lmns = lmn_of(js);
  const int ka = g * L, kb = imin(ka + L, a.k1);
  // the sensitivity of wdtn[k] (0 < k < k1), and with it that of ww'[k]: its own and t's
  auto wdtn = [&](int k, float cc, float lt, float ltm) {
    return k >= 1 ? cc * (level(a.rdnw, k) * lt - level(a.rdnw, k - 1) * ltm) : 0.0f;
  };
  auto lw_of = [&](int k, float lww, float lwdtn, float t1, float t1m) {
    return k >= 1 ? lww + lwdtn * (level(a.fnm, k) * t1 + level(a.fnp, k) * t1m) : lww;
  };
  float R = 0.0f, A = 0.0f, Rs = 0.0f, As = 0.0f, dns = 0.0f;
#pragma unroll 3
  for (int k = kb - 1; k >= ka; --k) {
    const int km = imax(k - 1, 0);
    const float lt = AT(a.lt, k, j, ic), ltm = AT(a.lt, km, j, ic), t1 = AT(a.t1, k, j, ic), t1m = AT(a.t1, km, j, ic);
    const float ls = AT(a.lt, k, js, ic), lsm = AT(a.lt, km, js, ic), t1s = AT(a.t1, k, js, ic), t1sm = AT(a.t1, km, js, ic);
    const float dn = level(a.dnw, k);
    dns += dn;
    A += dn * R;
    As += dn * Rs;
    R += lw_of(k, AT(a.lww, k, j, ic), wdtn(k, c, lt, ltm), t1, t1m);
    Rs += lw_of(k, AT(a.lww, k, js, ic), wdtn(k, cs, ls, lsm), t1s, t1sm);
  }
  s_r[0][g][lane] = R; s_a[0][g][lane] = A;
  s_r[1][g][lane] = Rs; s_a[1][g][lane] = As;
  if (lane == 0) s_dn[g] = dns;
  __syncthreads();
  // R: the sum over the runs above; A: over all levels, dnw times the sum above the level
  R = 0.0f; Rs = 0.0f;
  float T = 0.0f, Ts = 0.0f;
  A = 0.0f; As = 0.0f;
  for (int n = CA_WAVES - 1; n >= 0; --n) {
    if (n == g) { R = T; Rs = Ts; }
    const float dn = s_dn[n];
    A += s_a[0][n][lane] + dn * T;
    As += s_a[1][n][lane] + dn * Ts;
    T += s_r[0][n][lane];
    Ts += s_r[1][n][lane];
  }
  const float lS = a.dts * lmn + AT2(a.lmudf, j, ic) - A / mfy;
  const float lSs = a.dts * lmns + AT2(a.lmudf, js, ic) - As / mfys;
  if (g == 0 && own) {
    const float lmuave = AT2(a.lmuave, j, i);
    AT2(a.gmu, j, i) = in ? lmn + 0.5f * (1.0f - e) * lmuave : AT2(a.lmu, j, i);
    AT2(a.gmuave, j, i) = in ? 0.0f : lmuave;
    AT2(a.gmuts, j, i) = in ? 0.0f : AT2(a.lmuts, j, i);
    AT2(a.gmudf, j, i) = in ? 0.0f : AT2(a.lmudf, j, i);
    AT2(a.gmut, j, i) = in ? lS : 0.0f;
  }
  const float uc = AT2(a.muu, j, ic) / AT2(a.msfuy, j, ic), vc = AT2(a.muv, j, ic) * AT2(a.msfvx_inv, j, ic);
  const float ce = a.dts * AT2(a.msfty, j, ie) * AT2(a.msftx, j, ie), cn = a.dts * AT2(a.msfty, jn, ic) * AT2(a.msftx, jn, ic);
  auto load = [&](int k) {
    k = imin(imax(k, 0), D.nz - 1);
    const unsigned o = D.ob(k, j, ic), os = D.ob(k, js, ic), oe = D.ob(k, j, ie), on = D.ob(k, jn, ic);
    MuTLevel r;
    r.lww = at_b(a.lww, o); r.lt = at_b(a.lt, o); r.t1 = at_b(a.t1, o); r.lwws = at_b(a.lww, os);
    r.lts = at_b(a.lt, os); r.t1s = at_b(a.t1, os); r.lte = at_b(a.lt, oe); r.ltn = at_b(a.lt, on);
    r.t1w = AT(a.t1, k, j, iw); r.ltave = at_b(a.ltave, o); r.wwo = at_b(a.wwo, o);
    r.u = at_b(a.u, o); r.ue = at_b(a.u, oe); r.v = at_b(a.v, o); r.vn = at_b(a.v, on);
    return r;
  };
  // a share of nothing, whatever the other factor holds: the forward does not read it there
  auto times = [](float share, float x) { return share != 0.0f ? share * x : 0.0f; };
  const int kt = imin(ka + L, D.nz);   // the run's top, above the mass levels too
  if (ka >= kt) return;
  MuTLevel x = load(kt - 1), y = load(kt - 2);
  float up = 0.0f;   // from the level above, through t_1[k-1]: lwdtn[k+1] ww'[k+1] fnp[k+1]
  if (kt < a.k1) {
    const float lt = AT(a.lt, kt, j, ic);
    up = wdtn(kt, c, lt, x.lt) * AT(a.wwo, kt, j, ic) * level(a.fnp, kt);
  }
  for (int k = kt - 1; k >= ka; --k) {
    const MuTLevel z = load(k - 2);
    const bool lev = k < a.k1, inl = in && lev;
    const float dn = lev ? level(a.dnw, k) : 0.0f;
    const float ldv = dn * lS - dn / mfy * R, ldvs = dn * lSs - dn / mfys * Rs;
    const float lwd = lev ? wdtn(k, c, x.lt, y.lt) : 0.0f, lwds = lev ? wdtn(k, cs, x.lts, y.lts) : 0.0f;
    const float lwk = lev ? lw_of(k, x.lww, lwd, x.t1, y.t1) : 0.0f;
    R += lwk;
    if (lev) Rs += lw_of(k, x.lwws, lwds, x.t1s, y.t1s);
    const float q = inl ? -a.dts * mfy * mfx * x.lt : 0.0f, qs = ins && lev ? -a.dts * mfys * mfxs * x.lts : 0.0f;
    const float qe = ine && lev ? -ce * x.lte : 0.0f, qn = inn && lev ? -cn * x.ltn : 0.0f;
    const float du = inl ? mfx * mfy * a.rdx * ldv : 0.0f, dv = inl ? mfx * mfy * a.rdy * ldv : 0.0f;
    const float dvs = ins && lev ? mfxs * mfys * a.rdy * ldvs : 0.0f;
    const float duw = lane_below(du), qw = lane_below(q);
    const float hx = 0.5f * a.rdx, hy = 0.5f * a.rdy;
    // t_1 in the horizontal theta fluxes, and in the vertical flux wdtn[k] = ww'[k] (fnm[k] t_1[k] + fnp[k] t_1[k-1])
    float gt1 = hx * (times(qw - q, x.u) + times(q - qe, x.ue)) + hy * (times(qs - q, x.v) + times(q - qn, x.vn));
    const float wl = lwd * x.wwo;
    if (inl) gt1 += (k >= 1 ? wl * level(a.fnm, k) : 0.0f) + up;
    up = k >= 1 ? wl * level(a.fnp, k) : 0.0f;
    if (own) {
      const long p = D.ix(k, j, i);
      a.gu[p] = (duw - du) + times((qw - q) * hx, x.t1 + x.t1w);
      a.gv[p] = (dvs - dv) + times((qs - q) * hy, x.t1 + x.t1s);
      a.gu1[p] = times(duw - du, uc);
      a.gv1[p] = times(dvs - dv, vc);
      a.gt1[p] = gt1;
      a.gww[p] = inl ? (k == 0 ? R : 0.0f) : x.lww;
      a.gww1[p] = inl ? -lwk : 0.0f;             // ww' = ww - ww_1
      a.gt[p] = inl ? x.lt + x.ltave : x.lt;
      a.gtave[p] = inl ? 0.0f : x.ltave;
      a.gft[p] = inl ? mfy * a.dts * x.lt : 0.0f;
    }
    x = y; y = z;
  }
}

extern "C" int pywrf_advance_mu_t_adjoint(const pywrf_grid_t* g, const float* lam_ww, const float* lam_t,
                                          const float* lam_t_ave, const float* lam_muave, const float* lam_muts,
                                          const float* lam_mudf, const float* lam_mu, const float* t_1,
                                          const float* msftx, const float* msfty, const float* dnw,
                                          const float* fnm, const float* fnp, const float* rdnw, double rdx,
                                          double rdy, double dts, double epssm, float* lam_ww_ori, float* lam_u,
                                          float* lam_v, float* lam_mu_ori, float* lam_muave_ori,
                                          float* lam_muts_ori, float* lam_mudf_ori, float* lam_t_ori,
                                          float* lam_t_ave_ori, float* lam_ft, float* lam_mu_tend,
                                          const float* ww_out, const float* u, const float* v, const float* muu,
                                          const float* muv, const float* msfuy, const float* msfvx_inv,
                                          float* lam_u_1, float* lam_v_1, float* lam_ww_1, float* lam_t_1,
                                          pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (g->kts != 0 || g->kte > g->nz || g->kte < 2) return PYWRF_E_RANGE;
  AdjMuT a;
  a.lww = lam_ww; a.lt = lam_t; a.ltave = lam_t_ave; a.lmuave = lam_muave; a.lmuts = lam_muts;
  a.lmudf = lam_mudf; a.lmu = lam_mu; a.t1 = t_1; a.msftx = msftx; a.msfty = msfty; a.dnw = dnw;
  a.fnm = fnm; a.fnp = fnp; a.rdnw = rdnw;
  a.gww = lam_ww_ori; a.gu = lam_u; a.gv = lam_v; a.gmu = lam_mu_ori; a.gmuave = lam_muave_ori;
  a.gmuts = lam_muts_ori; a.gmudf = lam_mudf_ori; a.gt = lam_t_ori; a.gtave = lam_t_ave_ori; a.gft = lam_ft;
  a.gmut = lam_mu_tend;
  a.u = u; a.v = v; a.wwo = ww_out; a.muu = muu; a.muv = muv; a.msfuy = msfuy; a.msfvx_inv = msfvx_inv;
  a.gu1 = lam_u_1; a.gv1 = lam_v_1; a.gww1 = lam_ww_1; a.gt1 = lam_t_1;
  a.rdx = F(rdx); a.rdy = F(rdy); a.dts = F(dts); a.epssm = F(epssm);
  a.k1 = g->kte - 1;
  const int j0 = imax(g->jts, g->jds + 1), j1 = imin(g->jte, g->jde - 2);
  const int i0 = imax(g->its, g->ids + 1), i1 = imin(g->ite, g->ide - 2);
  if (j0 < 1 || i0 < 1 || j1 + 1 > g->ny || i1 + 1 > g->nx) return PYWRF_E_RANGE;
  Box b = mkbox(0, 1, j0, j1, i0, i1);
  hipLaunchKernelGGL(k_advance_mu_t_adj, ca_grid(g, CA_COLS - 1), dim3(CA_THREADS), 0, (hipStream_t)s, b, dims_of(g), a);
  PW_RET();
}

// ------------------------------------------------------------------ calc_p_rho^T
// calc_p_rho (wrf_dynamics.py:3269-3313) in its box (levels kts..min(kte,
// kde-1), the interior columns):
//   al = -(alt mu + rdnw[k] (ph[k+1] - ph[k])) / mut,
//   p  = c2a (alt (t_2 - mu t_1) / (mut (t0 + t_1)) - al),
// then, on a call with step != 0, p' = p + smdiv (p - pm1) and pm1' = p (in
// the box); at step 0 pm1' is a copy of the whole of p.  Outside the box al and
// p keep their incoming values.  alt, t_1 and c2a are held fixed.  ph[k]'s
// sensitivity gathers al[k]'s and al[k-1]'s, those of mu and mut are summed
// down the column.
struct AdjPRho {
  const float *lal, *lp, *lpm1;                          // sensitivities of the results
  const float *ph, *alt, *t_2, *t_1, *c2a, *mu, *mut, *rdnw;
  float *gal, *gp, *gpm1, *gph, *gt2, *gmu, *gmut;     // sensitivities of the inputs
  float* gt1;                                           // t_1 (null: not wanted)
  float t0, smdiv;
  int step;
};

// Wave g takes a run of levels of 64 columns (and the level below it again,
// for its share of ph), the next level's ten values loaded before this one's
// stores.  At 120 x 120 x 41
// 12.5 us, 50.7 with one thread a column.
struct PRhoLevel { float lal, lp, lpm, ph0, ph1, alt, t2, t1, c2; };

__global__ void __launch_bounds__(CA_THREADS) k_calc_p_rho_adj(Dims D, Box b, AdjPRho a) {
  __shared__ float s_mu[CA_WAVES][CA_COLS], s_mt[CA_WAVES][CA_COLS];
  const int lane = threadIdx.x % CA_COLS, g = ca_wave(), L = (D.nz + CA_WAVES - 1) / CA_WAVES;
  const int j = (int)blockIdx.y, i = (int)blockIdx.x * CA_COLS + lane, ic = imin(i, D.nx - 1);
  const bool w = i < D.nx, col = w && b.has2(j, i);
  const float mut = col ? AT2(a.mut, j, ic) : 1.0f, mu = col ? AT2(a.mu, j, ic) : 0.0f;
  float gmu = 0.0f, gmut = 0.0f;
  const long plane = D.plane(), q0 = D.ix2(j, ic);
  auto load = [&](int k) {
    k = imin(imax(k, 0), D.nz - 1);
    const long q = q0 + k * plane;
    PRhoLevel r = {a.lal[q], a.lp[q], a.lpm1[q], a.ph[q], a.ph[q0 + imin(k + 1, D.nz - 1) * plane], a.alt[q], a.t_2[q],
                   a.t_1[q], a.c2a[q]};
    return r;
  };
  // lpr: the sensitivity of p before the damping; the result is that of al, through p as well
  auto lal_of = [&](const PRhoLevel& r, float& cl) {
    const float lpr = a.step != 0 ? r.lp * (1.0f + a.smdiv) + r.lpm : r.lp + r.lpm;
    cl = r.c2 * lpr;
    return r.lal - cl;
  };
  const int ka = g * L, kb = imin(ka + L, D.nz);
  if (ka < kb) {
    float cl, prev = 0.0f;   // prev: rdnw[k-1] (al[k-1]'s sensitivity) / mut
    if (col && ka - 1 >= b.k0 && ka - 1 < b.k1) prev = level(a.rdnw, ka - 1) * lal_of(load(ka - 1), cl) / mut;
    PRhoLevel x = load(ka);
    for (int k = ka; k < kb; ++k) {
      const PRhoLevel y = load(k + 1);
      float r = 0.0f, gal = x.lal, gp = a.step != 0 ? x.lp : x.lp + x.lpm, gpm = a.step != 0 ? x.lpm : 0.0f;
      float gt2 = 0.0f, gt1 = 0.0f;
      if (col && k >= b.k0 && k < b.k1) {
        const float rd = level(a.rdnw, k);
        const float al = -1.0f / mut * (x.alt * mu + rd * (x.ph1 - x.ph0));
        const float den = mut * (a.t0 + x.t1);
        const float pa = x.alt * (x.t2 - mu * x.t1) / den;
        const float l = lal_of(x, cl);
        gpm = a.step != 0 ? -a.smdiv * x.lp : 0.0f;
        gt2 = cl * x.alt / den;
        gt1 = cl * (-x.alt * mu / den - pa / (a.t0 + x.t1));
        gmu += cl * (-(x.alt * x.t1) / den) + l * (-x.alt / mut);
        gmut += cl * (-pa / mut) + l * (-al / mut);
        r = rd * l / mut;
        gal = 0.0f;
        gp = 0.0f;
      }
      if (w) {
        const long q = q0 + k * plane;
        a.gal[q] = gal;
        a.gp[q] = gp;
        a.gpm1[q] = gpm;
        a.gt2[q] = gt2;
        if (a.gt1) a.gt1[q] = gt1;
        a.gph[q] = r - prev;
      }
      prev = r;
      x = y;
    }
  }
  const float sm = ca_sum(s_mu, g, lane, gmu), st = ca_sum(s_mt, g, lane, gmut);
  if (g == 0 && w) {
    AT2(a.gmu, j, i) = sm;
    AT2(a.gmut, j, i) = st;
  }
}

extern "C" int pywrf_calc_p_rho_adjoint(const pywrf_grid_t* g, const float* lam_al, const float* lam_p,
                                        const float* lam_pm1, const float* ph, const float* alt, const float* t_2,
                                        const float* t_1, const float* c2a, const float* mu, const float* mut,
                                        double t0, const float* rdnw, double smdiv, int step, float* lam_al_ori,
                                        float* lam_p_ori, float* lam_pm1_in, float* lam_ph, float* lam_t_2,
                                        float* lam_mu, float* lam_mut, float* lam_t_1, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  Box b = mkbox(g->kts, imin(g->kte, g->kde - 1), g->jts, imin(g->jte, g->jde - 1), g->its,
                imin(g->ite, g->ide - 1));
  if (b.k1 + 1 > g->nz) return PYWRF_E_RANGE;
  AdjPRho a = {lam_al, lam_p, lam_pm1, ph, alt, t_2, t_1, c2a, mu, mut, rdnw,
               lam_al_ori, lam_p_ori, lam_pm1_in, lam_ph, lam_t_2, lam_mu, lam_mut, lam_t_1, F(t0), F(smdiv),
               step};
  hipLaunchKernelGGL(k_calc_p_rho_adj, ca_grid(g, CA_COLS), dim3(CA_THREADS), 0, (hipStream_t)s, dims_of(g), b, a);
  PW_RET();
}

// ------------------------------------------------------------------ sumflux^T
// sumflux (wrf_dynamics.py:3799-3839) is linear: on its first call the three
// accumulators are zeroed over the tile, each then adds its flux over its box,
// and on the last call the sum is divided by the number of calls (the u_lin
// terms are fixed).  One thread per point.
struct SumLin {
  const float *muu, *muv, *msfuy, *msfvx_inv;
  float *gul, *gvl, *gwl;                               // u_lin, v_lin, ww_lin (null: not wanted)
};

__global__ void k_sumflux_adj(Box all, Dims D, const float* lru_m, const float* lrv_m, const float* lww_m,
                              float* gru, float* grv, float* gww, float* gru_m, float* grv_m, float* gww_m, Box b,
                              Box bu, Box bv, Box bw, int first, int last, float n, SumLin sl) {
  int k, j, i;
  if (!box_point(all, k, j, i)) return;
  const long q = D.ix(k, j, i);
  const bool zeroed = first && b.has(k, j, i);
  const float* lam[3] = {lru_m, lrv_m, lww_m};
  float* gf[3] = {gru, grv, gww};
  float* ga[3] = {gru_m, grv_m, gww_m};
  const Box* bx[3] = {&bu, &bv, &bw};
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    const float l = lam[f][q];
    const bool in = bx[f]->has(k, j, i);
    const float s = last ? l / n : l;
    gf[f][q] = in ? s : 0.0f;
    ga[f][q] = zeroed ? 0.0f : (in ? s : l);
  }
  // the last call adds muu u_lin / msfuy, muv v_lin msfvx_inv and ww_lin
  if (sl.gul) {
    const bool iu = last && bu.has(k, j, i), iv = last && bv.has(k, j, i), iw = last && bw.has(k, j, i);
    sl.gul[q] = iu ? lru_m[q] * (AT2(sl.muu, j, i) / AT2(sl.msfuy, j, i)) : 0.0f;
    sl.gvl[q] = iv ? lrv_m[q] * (AT2(sl.muv, j, i) * AT2(sl.msfvx_inv, j, i)) : 0.0f;
    sl.gwl[q] = iw ? lww_m[q] : 0.0f;
  }
}

extern "C" int pywrf_sumflux_adjoint(const pywrf_grid_t* g, const float* lam_ru_m, const float* lam_rv_m,
                                     const float* lam_ww_m, int iteration, int number_of_small_timesteps,
                                     float* lam_ru, float* lam_rv, float* lam_ww, float* lam_ru_m_in,
                                     float* lam_rv_m_in, float* lam_ww_m_in, const float* muu, const float* muv,
                                     const float* msfuy, const float* msfvx_inv, float* lam_u_lin,
                                     float* lam_v_lin, float* lam_ww_lin, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kte > g->nz || number_of_small_timesteps == 0) return PYWRF_E_RANGE;
  int mini = imin(g->ide - 1, g->ite), minj = imin(g->jde - 1, g->jte), mink = imin(g->kde - 1, g->kte);
  Box bu = mkbox(g->kts, mink, g->jts, minj, g->its, g->ite);
  Box bv = mkbox(g->kts, mink, g->jts, g->jte, g->its, mini);
  Box bw = mkbox(g->kts, g->kte, g->jts, minj, g->its, mini);
  Box b = mkbox(g->kts, g->kte, g->jts, g->jte, g->its, g->ite);
  if (lam_u_lin && (!lam_v_lin || !lam_ww_lin || !muu || !muv || !msfuy || !msfvx_inv)) return PYWRF_E_ARG;
  SumLin sl = {muu, muv, msfuy, msfvx_inv, lam_u_lin, lam_v_lin, lam_ww_lin};
  PW_LAUNCH_BOX(k_sumflux_adj, whole(g), s, dims_of(g), lam_ru_m, lam_rv_m, lam_ww_m, lam_ru, lam_rv, lam_ww,
                lam_ru_m_in, lam_rv_m_in, lam_ww_m_in, b, bu, bv, bw, iteration == 1,
                iteration == number_of_small_timesteps, (float)number_of_small_timesteps, sl);
  PW_RET();
}

// ------------------------------------------------------------------ open-boundary fill^T
// The fill of one plane (set_physical_bc3d / bc2d, wrf_dynamics.py:164-278) is
// a run of copies: the x-halos from the first / last interior column (over
// rows that include the y-halos), then the y-halos from the first / last
// interior row.  Its transpose runs the two in the opposite order, each copy
// target handing its sensitivity to its source and keeping none: first the
// y-copies (one thread per column and side, its three targets in turn), a
// barrier, then the x-copies (one thread per row and side).  No two threads
// of one phase share a source or a target, so no atomics are needed; an
// x-copy's source in a y-halo row then receives the sensitivity of the value
// it held before the y-copies, which is what the x-copies read.
__device__ inline void open_bc_plane_adj(float* a, int nx, const BcSpec& c) {
  const int ny_items = 2 * (c.yc1 - c.yc0);
  for (int t = (int)threadIdx.x; t < ny_items; t += (int)blockDim.x) {
    const int col = c.yc0 + t / 2, side = t & 1;
    int srow, d0;
    if (side == 0) { srow = c.jds; d0 = c.jds - 3; }
    else if (c.vstag) { srow = c.jde - 1; d0 = c.jde; }
    else { srow = c.jde - 2; d0 = c.jde - 1; }
    float sum = 0.0f;
    for (int h = 0; h < 3; ++h) {
      float* p = a + (long)(d0 + h) * nx + col;
      sum += *p;
      *p = 0.0f;
    }
    a[(long)srow * nx + col] += sum;
  }
  __syncthreads();
  const int r0 = c.ustag ? c.ur0 : c.xr0, r1 = c.ustag ? c.ur1 : c.xr1;
  const int nstart = c.xr1 - c.xr0, nx_items = nstart + (r1 - r0);
  for (int t = (int)threadIdx.x; t < nx_items; t += (int)blockDim.x) {
    int row, src, d0;
    if (t < nstart) { row = c.xr0 + t; src = c.ids; d0 = c.ids - 3; }
    else { row = r0 + (t - nstart); src = c.ustag ? c.ide - 1 : c.ide - 2; d0 = c.ustag ? c.ide : c.ide - 1; }
    float* base = a + (long)row * nx;
    float sum = 0.0f;
    for (int h = 0; h < 3; ++h) {
      sum += base[d0 + h];
      base[d0 + h] = 0.0f;
    }
    base[src] += sum;
  }
}

#define PW_BC_ADJ_MAX 32
struct BcAdjJobs {
  int n;
  BcJob job[PW_BC_ADJ_MAX];
};

__global__ void k_open_bc_adj_group(long plane, int nx, BcAdjJobs J) {
  if ((int)blockIdx.y >= J.n) return;
  const BcJob& jb = J.job[blockIdx.y];
  if ((int)blockIdx.x >= jb.nk) return;
  open_bc_plane_adj(jb.p + (long)(jb.k0 + (int)blockIdx.x) * plane, nx, jb.c);
}

extern "C" int pywrf_set_physical_bc_group_adjoint(const pywrf_grid_t* g3, const pywrf_grid_t* g2, int n,
                                                   void* const* lam_fields, const char* variables,
                                                   const int* is2d, pywrf_stream_t s) {
  if (!pw_size_ok(g3) || !pw_size_ok(g2)) return PYWRF_E_RANGE;
  if (n < 0 || n > PW_BC_ADJ_MAX || g3->ny != g2->ny || g3->nx != g2->nx) return PYWRF_E_ARG;
  BcAdjJobs J;
  J.n = n;
  int maxk = 1;
  for (int f = 0; f < n; ++f) {
    BcJob& jb = J.job[f];
    jb.p = (float*)lam_fields[f];
    int e, k1 = 1;
    if (is2d[f]) {
      e = bc_spec2(g2, variables[f], jb.c);
      jb.k0 = 0;
      if (!e && !bc_spec_ok(g2->ny, g2->nx, 1, 0, 1, jb.c)) e = PYWRF_E_RANGE;
    } else {
      e = bc_spec3(g3, variables[f], jb.c, k1);
      jb.k0 = g3->kts;
      if (!e && !bc_spec_ok(g3->ny, g3->nx, g3->nz, g3->kts, k1, jb.c)) e = PYWRF_E_RANGE;
    }
    if (e) return e;
    // the copies' sources must lie outside their targets (interior rows and columns)
    if (jb.c.jde - 2 <= jb.c.jds || jb.c.ide - 2 <= jb.c.ids) return PYWRF_E_RANGE;
    jb.nk = k1 - jb.k0 > 0 ? k1 - jb.k0 : 0;
    maxk = imax(maxk, jb.nk);
  }
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_open_bc_adj_group, dim3(maxk, n), dim3(BC_THREADS), 0, (hipStream_t)s,
                     (long)g3->ny * g3->nx, g3->nx, J);
  PW_RET();
}

// ------------------------------------------------------------------ small_step_prep^T (past the first stage)
// small_step_prep (wrf_dynamics.py:3152-3266) past the first RK stage, with
// pb, p, alt (so c2a) held fixed: on its boxes it saves u_2 .. ph_2 and ww,
// and forms the acoustic variables
//   u = (muus u_1 - muu u_2) / msfuy,  v = (muvs v_1 - muv v_2) msfvx_inv,
//   t = muts t_1 - mut t_2,  w = (muts w_1 - mut w_2) / msfty,  ph = ph_1 - ph_2,
// with muts = mub + mu_1, muus / muvs the averages of mub + mu_1 onto the u / v
// points, mu_save = mu_2 and mu_2' = mu_1 - mu_2.  Pass 1 (column blocks, wave g on levels g, g + 8, ...; 32 us
// at 120 x 120 x 41, 156 with one thread a column) gives the 3-D sensitivities and sums down the column those of
// muus, muvs and muts; pass 2 (one thread per point of the plane) gathers
// the averages' and the masses' shares into mu_1 and mu_2.
struct PrepAdj {
  const float *lus, *lvs, *lws, *lts, *lps, *lwws, *luo, *lvo, *lwo, *lto, *lpo;   // 3-D results
  const float *lmu2, *lmuts, *lmuus, *lmuvs, *lmusave;                             // plane results
  const float *u_1, *v_1, *w_1, *t_1, *muus, *muvs, *muts, *muu, *muv, *mut, *msfuy, *msfvx_inv, *msfty;
  float *gu2, *gv2, *gw2, *gt2, *gph2, *gu1, *gv1, *gw1, *gt1, *gph1, *gww;
  float *smuus, *smuvs, *smuts;                                                    // plane scratch
  float *gmu1, *gmu2;
  int k1, kde, j0, j1, i0, i1, i1u, j1v;
};

__global__ void __launch_bounds__(CA_THREADS) k_ssprep_adj(Dims D, PrepAdj a) {
  __shared__ float s_u[CA_WAVES][CA_COLS], s_v[CA_WAVES][CA_COLS], s_t[CA_WAVES][CA_COLS];
  const int lane = threadIdx.x % CA_COLS, g = ca_wave();
  const int j = (int)blockIdx.y, i = imin((int)blockIdx.x * CA_COLS + lane, D.nx - 1);
  const bool w = (int)blockIdx.x * CA_COLS + lane < D.nx;   // the lanes beyond the row have no levels
  const bool h = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  const bool ur = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1u;
  const bool vr = j >= a.j0 && j < a.j1v && i >= a.i0 && i < a.i1;
  const bool vsr = j >= a.j0 && j < a.j1v && i >= a.i0 && i < a.i1u;   // the muvs box (i-range i1u)
  const float muus = AT2(a.muus, j, i), muvs = AT2(a.muvs, j, i), muts = AT2(a.muts, j, i);
  const float muu = AT2(a.muu, j, i), muv = AT2(a.muv, j, i), mut = AT2(a.mut, j, i);
  const float my = AT2(a.msfuy, j, i), mvx = AT2(a.msfvx_inv, j, i), mty = AT2(a.msfty, j, i);
  float su = 0.0f, sv = 0.0f, st = 0.0f;
  for (int k = w ? g : D.nz; k < D.nz; k += CA_WAVES) {
    const long q = D.ix(k, j, i);
    const bool bu = k < a.k1 && ur, bv = k < a.k1 && vr, bm = k < a.k1 && h, bw = k < a.kde && h;
    const float luo = a.luo[q], lvo = a.lvo[q], lwo = a.lwo[q], lto = a.lto[q], lpo = a.lpo[q];
    if (bu) {
      a.gu2[q] = a.lus[q] - luo * muu / my;
      a.gu1[q] = luo * muus / my;
      su += luo * a.u_1[q] / my;
    } else {
      a.gu2[q] = luo;
      a.gu1[q] = 0.0f;
    }
    if (bv) {
      a.gv2[q] = a.lvs[q] - lvo * muv * mvx;
      a.gv1[q] = lvo * muvs * mvx;
      sv += lvo * a.v_1[q] * mvx;
    } else {
      a.gv2[q] = lvo;
      a.gv1[q] = 0.0f;
    }
    if (bm) {
      a.gt2[q] = a.lts[q] - lto * mut;
      a.gt1[q] = lto * muts;
      st += lto * a.t_1[q];
    } else {
      a.gt2[q] = lto;
      a.gt1[q] = 0.0f;
    }
    if (bw) {
      a.gw2[q] = a.lws[q] - lwo * mut / mty;
      a.gw1[q] = lwo * muts / mty;
      st += lwo * a.w_1[q] / mty;
      a.gph2[q] = a.lps[q] - lpo;
      a.gph1[q] = lpo;
      a.gww[q] = a.lwws[q];
    } else {
      a.gw2[q] = lwo;
      a.gw1[q] = 0.0f;
      a.gph2[q] = lpo;
      a.gph1[q] = 0.0f;
      a.gww[q] = 0.0f;
    }
  }
  su = ca_sum(s_u, g, lane, su);
  sv = ca_sum(s_v, g, lane, sv);
  st = ca_sum(s_t, g, lane, st);
  if (g != 0 || !w) return;
  AT2(a.smuus, j, i) = ur ? AT2(a.lmuus, j, i) + su : 0.0f;
  AT2(a.smuvs, j, i) = vsr ? AT2(a.lmuvs, j, i) + sv : 0.0f;
  AT2(a.smuts, j, i) = h ? AT2(a.lmuts, j, i) + st : 0.0f;
}

__global__ void k_ssprep_adj_2d(Box all, Dims D, PrepAdj a) {
  int j, i;
  if (!box_column(all, j, i)) return;
  const bool h = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  const float lmu2 = AT2(a.lmu2, j, i);
  // muus[j][i] and muus[j][i+1] average mu_1[j][i]; muvs[j][i] and muvs[j+1][i] too
  float g1 = 0.5f * (AT2(a.smuus, j, i) + (i + 1 < D.nx ? AT2(a.smuus, j, i + 1) : 0.0f)) +
             0.5f * (AT2(a.smuvs, j, i) + (j + 1 < D.ny ? AT2(a.smuvs, j + 1, i) : 0.0f));
  float g2 = lmu2;                                        // outside the box mu_2 passes through
  if (h) {
    g1 += AT2(a.smuts, j, i) + lmu2;                      // muts = mub + mu_1, mu_2' = mu_1 - mu_2
    g2 = AT2(a.lmusave, j, i) - lmu2;
  }
  AT2(a.gmu1, j, i) = g1;
  AT2(a.gmu2, j, i) = g2;
}

extern "C" int pywrf_small_step_prep_adjoint(
    const pywrf_grid_t* g, int rk_step, const float* lam_u_save, const float* lam_v_save, const float* lam_w_save,
    const float* lam_t_save, const float* lam_ph_save, const float* lam_ww_save, const float* lam_u,
    const float* lam_v, const float* lam_w, const float* lam_t, const float* lam_ph, const float* lam_mu_2,
    const float* lam_muts, const float* lam_muus, const float* lam_muvs, const float* lam_mu_save,
    const float* u_1, const float* v_1, const float* w_1, const float* t_1, const float* muus, const float* muvs,
    const float* muts, const float* muu, const float* muv, const float* mut, const float* msfuy,
    const float* msfvx_inv, const float* msfty, float* lam_u_2_in, float* lam_v_2_in, float* lam_w_2_in,
    float* lam_t_2_in, float* lam_ph_2_in, float* lam_u_1, float* lam_v_1, float* lam_w_1, float* lam_t_1,
    float* lam_ph_1, float* lam_ww, float* lam_mu_1, float* lam_mu_2_in, float* work2d, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  if (rk_step == 1) return PYWRF_E_ARG;            // the first stage copies: not differentiated here
  if (g->kde > g->nz || g->kts != 0) return PYWRF_E_RANGE;
  PrepAdj a = {lam_u_save, lam_v_save, lam_w_save, lam_t_save, lam_ph_save, lam_ww_save, lam_u, lam_v, lam_w,
               lam_t, lam_ph, lam_mu_2, lam_muts, lam_muus, lam_muvs, lam_mu_save, u_1, v_1, w_1, t_1, muus, muvs,
               muts, muu, muv, mut, msfuy, msfvx_inv, msfty, lam_u_2_in, lam_v_2_in, lam_w_2_in, lam_t_2_in,
               lam_ph_2_in, lam_u_1, lam_v_1, lam_w_1, lam_t_1, lam_ph_1, lam_ww, nullptr, nullptr, nullptr,
               lam_mu_1, lam_mu_2_in, imin(g->kte, g->kde - 1), g->kde, g->jts, imin(g->jte, g->jde - 1), g->its,
               imin(g->ite, g->ide - 1), g->ite, g->jte};
  const long n2 = (long)g->ny * g->nx;
  a.smuus = work2d; a.smuvs = work2d + n2; a.smuts = work2d + 2 * n2;
  if (a.j0 < 1 || a.i0 < 1) return PYWRF_E_RANGE;   // the averages read j-1 / i-1
  Box pl = mkbox(0, 1, 0, g->ny, 0, g->nx);
  hipLaunchKernelGGL(k_ssprep_adj, ca_grid(g, CA_COLS), dim3(CA_THREADS), 0, (hipStream_t)s, dims_of(g), a);
  PW_LAUNCH_COLS(k_ssprep_adj_2d, pl, s, dims_of(g), a);
  PW_RET();
}

// ------------------------------------------------------------------ calc_mu_uv_1^T
// calc_mu_uv_1 (wrf_dynamics.py:3844-3860) sets muu / muv from mu: the
// two-point average inside, mu itself on the first row / column and the
// second last point's value on the last; elsewhere muu / muv keep theirs.
// Transpose: each written point hands its sensitivity to the mu points it
// read (atomic adds onto the zeroed lam_mu) and keeps none.
__global__ void k_calc_mu_uv_1_adj(Box b, Dims D, const float* lmuu, const float* lmuv, float* gmu, float* gmuu,
                                   float* gmuv, int jts, int jtf, int jte, int its, int itf, int ite) {
  int j, i;
  if (!box_column(b, j, i)) return;
  float lu = AT2(lmuu, j, i), lv = AT2(lmuv, j, i);
  bool wu = false, wv = false;
  if (j < jtf) {
    if (i == ite - 1) { atomic_add(&AT2(gmu, j, ite - 2), lu); wu = true; }
    else if (i >= its + 1) { atomic_add(&AT2(gmu, j, i), 0.5f * lu); atomic_add(&AT2(gmu, j, i - 1), 0.5f * lu); wu = true; }
    else if (i == its) { atomic_add(&AT2(gmu, j, its), lu); wu = true; }
  }
  if (i < itf) {
    if (j == jte - 1) { atomic_add(&AT2(gmu, jte - 2, i), lv); wv = true; }
    else if (j >= jts + 1) { atomic_add(&AT2(gmu, j, i), 0.5f * lv); atomic_add(&AT2(gmu, j - 1, i), 0.5f * lv); wv = true; }
    else if (j == jts) { atomic_add(&AT2(gmu, jts, i), lv); wv = true; }
  }
  AT2(gmuu, j, i) = wu ? 0.0f : lu;
  AT2(gmuv, j, i) = wv ? 0.0f : lv;
}

__global__ void k_copy_n(const float* src, float* dst, long n) {
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) dst[t] = src[t];
}

extern "C" int pywrf_calc_mu_uv_1_adjoint(const pywrf_grid_t* g, const float* lam_muu, const float* lam_muv,
                                          float* lam_mu, float* lam_muu_in, float* lam_muv_in, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 1);
  const int jtf = imin(g->jte, g->jde - 1), itf = imin(g->ite, g->ide - 1);
  if (g->ite - 2 < 0 || g->jte - 2 < 0) return PYWRF_E_RANGE;
  const long n2 = (long)g->ny * g->nx;
  hipLaunchKernelGGL(k_zero_n, dim3(256), dim3(256), 0, (hipStream_t)s, lam_mu, n2);
  // outside the box muu / muv pass through
  hipLaunchKernelGGL(k_copy_n, dim3(256), dim3(256), 0, (hipStream_t)s, lam_muu, lam_muu_in, n2);
  hipLaunchKernelGGL(k_copy_n, dim3(256), dim3(256), 0, (hipStream_t)s, lam_muv, lam_muv_in, n2);
  Box b = mkbox(0, 1, g->jts, g->jte, g->its, g->ite);
  PW_LAUNCH_COLS(k_calc_mu_uv_1_adj, b, s, dims_of(g), lam_muu, lam_muv, lam_mu, lam_muu_in, lam_muv_in, g->jts, jtf,
                 g->jte, g->its, itf, g->ite);
  PW_RET();
}

// ------------------------------------------------------------------ small_step_finish^T
// small_step_finish (wrf_dynamics.py:3863-3978) couples the acoustic
// variables back on its boxes:
//   u = (msfuy u + u_save muu) / muus,  v = (msfvx v + v_save muv) / muvs,
//   w = (msfty w + w_save mut) / muts,  ph = ph + ph_save,  ww = ww + ww1,
//   t = (t [- dts n mut h_diabatic] + t_save mut) / muts,  mu_2 = mu_2 + mu_save;
// elsewhere the fields pass.  mut, muu, muv, the map factors and h_diabatic
// are held fixed.  Column blocks, wave g on levels g, g + 8, ... (23 us at
// 120 x 120 x 41, 102 with one thread a column); the
// sensitivities of muus, muvs and muts are summed down the column (muts by division: the results are inputs).
struct FinAdj {
  const float *lu, *lv, *lw, *lph, *lww, *lt, *lmu;                                // results
  const float *uo, *vo, *wo, *to;                                                  // forward results
  const float *muu, *muus, *muv, *muvs, *mut, *muts, *msfuy, *msfvx, *msfty;
  float *gu, *gv, *gw, *gph, *gww, *gt, *gus, *gvs, *gws, *gps, *gww1, *gts;
  float *gmuus, *gmuvs, *gmuts, *gmu2, *gmusave;
  int kde, j0, j1, i0, i1, jte, ite;
};

__global__ void __launch_bounds__(CA_THREADS) k_ssfinish_adj(Dims D, FinAdj a) {
  __shared__ float s_u[CA_WAVES][CA_COLS], s_v[CA_WAVES][CA_COLS], s_t[CA_WAVES][CA_COLS];
  const int lane = threadIdx.x % CA_COLS, g = ca_wave();
  const int j = (int)blockIdx.y, i = imin((int)blockIdx.x * CA_COLS + lane, D.nx - 1);
  const bool w = (int)blockIdx.x * CA_COLS + lane < D.nx;   // the lanes beyond the row have no levels
  const bool h = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.i1;
  const bool vr = j >= a.j0 && j < a.jte && i >= a.i0 && i < a.i1;
  const bool ur = j >= a.j0 && j < a.j1 && i >= a.i0 && i < a.ite;
  const float muus = AT2(a.muus, j, i), muvs = AT2(a.muvs, j, i), muts = AT2(a.muts, j, i);
  const float muu = AT2(a.muu, j, i), muv = AT2(a.muv, j, i), mut = AT2(a.mut, j, i);
  const float my = AT2(a.msfuy, j, i), mx = AT2(a.msfvx, j, i), mty = AT2(a.msfty, j, i);
  float su = 0.0f, sv = 0.0f, st = 0.0f;
  for (int k = w ? g : D.nz; k < D.nz; k += CA_WAVES) {
    const long q = D.ix(k, j, i);
    const float lv = a.lv[q], lu = a.lu[q], lw = a.lw[q], lph = a.lph[q], lww = a.lww[q], lt = a.lt[q];
    if (k < a.kde - 1 && vr) {
      a.gv[q] = lv * mx / muvs;
      a.gvs[q] = lv * muv / muvs;
      sv -= lv * a.vo[q] / muvs;
    } else {
      a.gv[q] = lv;
      a.gvs[q] = 0.0f;
    }
    if (k < a.kde - 1 && ur) {
      a.gu[q] = lu * my / muus;
      a.gus[q] = lu * muu / muus;
      su -= lu * a.uo[q] / muus;
    } else {
      a.gu[q] = lu;
      a.gus[q] = 0.0f;
    }
    if (k < a.kde && h) {
      a.gw[q] = lw * mty / muts;
      a.gws[q] = lw * mut / muts;
      st -= lw * a.wo[q] / muts;
      a.gps[q] = lph;
      a.gww1[q] = lww;
    } else {
      a.gw[q] = lw;
      a.gws[q] = 0.0f;
      a.gps[q] = 0.0f;
      a.gww1[q] = 0.0f;
    }
    a.gph[q] = lph;
    a.gww[q] = lww;
    if (k < a.kde - 1 && h) {
      a.gt[q] = lt / muts;
      a.gts[q] = lt * mut / muts;
      st -= lt * a.to[q] / muts;
    } else {
      a.gt[q] = lt;
      a.gts[q] = 0.0f;
    }
  }
  su = ca_sum(s_u, g, lane, su);
  sv = ca_sum(s_v, g, lane, sv);
  st = ca_sum(s_t, g, lane, st);
  if (g != 0 || !w) return;
  AT2(a.gmuus, j, i) = su;
  AT2(a.gmuvs, j, i) = sv;
  AT2(a.gmuts, j, i) = st;
  const float lmu = AT2(a.lmu, j, i);
  AT2(a.gmu2, j, i) = lmu;
  AT2(a.gmusave, j, i) = h ? lmu : 0.0f;
}

extern "C" int pywrf_small_step_finish_adjoint(
    const pywrf_grid_t* g, const float* lam_u, const float* lam_v, const float* lam_w, const float* lam_ph,
    const float* lam_ww, const float* lam_t, const float* lam_mu_2, const float* u_out, const float* v_out,
    const float* w_out, const float* t_out, const float* muu, const float* muus, const float* muv,
    const float* muvs, const float* mut, const float* muts, const float* msfuy, const float* msfvx,
    const float* msfty, float* lam_u_2, float* lam_v_2, float* lam_w_2, float* lam_ph_2, float* lam_ww_in,
    float* lam_t_2, float* lam_u_save, float* lam_v_save, float* lam_w_save, float* lam_ph_save, float* lam_ww1,
    float* lam_t_save, float* lam_muus, float* lam_muvs, float* lam_muts, float* lam_mu_2_in, float* lam_mu_save,
    pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 0);
  if (g->kde > g->nz || g->kds != 0) return PYWRF_E_RANGE;
  FinAdj a = {lam_u, lam_v, lam_w, lam_ph, lam_ww, lam_t, lam_mu_2, u_out, v_out, w_out, t_out, muu, muus, muv,
              muvs, mut, muts, msfuy, msfvx, msfty, lam_u_2, lam_v_2, lam_w_2, lam_ph_2, lam_ww_in, lam_t_2,
              lam_u_save, lam_v_save, lam_w_save, lam_ph_save, lam_ww1, lam_t_save, lam_muus, lam_muvs, lam_muts,
              lam_mu_2_in, lam_mu_save, g->kde, g->jts, imin(g->jte, g->jde - 1), g->its, imin(g->ite, g->ide - 1),
              g->jte, g->ite};
  hipLaunchKernelGGL(k_ssfinish_adj, ca_grid(g, CA_COLS), dim3(CA_THREADS), 0, (hipStream_t)s, dims_of(g), a);
  PW_RET();
}
