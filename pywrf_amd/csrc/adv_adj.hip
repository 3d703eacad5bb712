// Adjoints of the advection tendencies (wrf_dynamics.py:1112-2028): with the
// mass fluxes fixed the tendency of u, v, w or a scalar q is linear in q (for u
// and v but for the two faces at the domain's ends, whose upwind value is
// chosen by the sign of u or v itself: the forward's branch is taken), each
// face value being vel * sum_o c_o(face, sign) q(face + o).
//
// Gather form: every point sums, over the six faces of each direction whose
// stencils hold it, the face's sensitivity (formed from the adjoint tendencies
// of the two points it separates) times its coefficient.  No atomics; every
// output point is written once.
//
// One wave owns 58 columns of a row and marches up the levels, as the forward
// scalar transport does: lane l holds column i0 - 3 + l, the x-faces are formed
// once by their own lane and read by DPP lane shifts, the six y-faces around
// the row are formed from its neighbours, and the six z-faces around a level
// slide up in registers.  A face is held as two numbers, its weighted
// sensitivity under the upwind choice it took and zero under the other, so a
// 5th-order face costs a point two multiply-adds.  Scattering the shares with
// atomic adds instead (up to 21 a point) was bound by the L2's atomics: u, v, w
// at 120x120x41 52, 47 and 59 us with the zeroing beside them, here 13, 15 and
// 15 us (32, 36 and 35 at 240x240x41); the scalar form that gathered with one
// thread a point 94.5 us at 240x240x41, here 28 us (2.0 TB/s of its six arrays):
// what is left is each level's load latency with 3 to 5 waves a SIMD.
#include "common.h"
#include "consts.h"

#define AT(p, k, j, i) at_b((p), D.ob((k), (j), (i)))
#define AT2(p, j, i) at_b((p), D.ob2((j), (i)))

int pw_check_grid(const pywrf_grid_t* g, int r);
#define CHECK(g, r) do { int _e = pw_check_grid((g), (r)); if (_e) return _e; } while (0)

// rows a wave (2 at 240x240x41: 31 us a scalar call against 28; the waves are too few to hide each other's latency)
#define AA_R 1

namespace {

enum Kind { SCALAR, WIND_U, WIND_V, WIND_W };

struct AdvAdj {
  // q: u or v (its sign picks the end faces' side); mA: the map factor of the
  // horizontal terms; mB: msfvx (v's vertical term is scaled by mA / mB)
  const float *lam, *q, *ru, *rv, *rom, *mA, *mB, *fzm, *fzp, *rdz;
  float* out;
  float rdx, rdy;
  int ids, ide, jds, jde, ktf, accumulate;
  Box b, by, bx;           // the forward's boxes: all terms, the y-term, the x-term
  int j0, j1, i0, i1;      // rows and columns a stencil can reach
};

// How a face weighs its stencil.  END_LO / END_HI: the end faces of u along x
// and v along y; FZ: the interpolated face below the first or above the last
// full level.
enum Rule { NONE, FIFTH, THIRD, MEAN, FZ, END_LO, END_HI };

// rule of face f of a direction with domain [d0, d1); own: the wind component's own direction
__device__ inline int hrule(int f, int d0, int d1, bool own) {
  const int e = own ? d1 : d1 - 1;   // one past the last face
  if (f >= d0 + 3 && f < e - 2) return FIFTH;
  if (f == d0 + 1) return own ? END_LO : MEAN;
  if (!own && f == e - 1) return MEAN;
  if (f == d0 + 2 || f == e - 2) return THIRD;
  if (own && f == e - 1) return END_HI;
  return NONE;
}

template <int KIND>
__device__ inline int zrule(int kf, int ktf) {
  if (KIND == WIND_W) {
    if (kf < 1 || kf > ktf) return NONE;
    if (kf == 1 || kf == ktf) return MEAN;
    return kf >= 3 && kf < ktf - 1 ? FIFTH : THIRD;
  }
  if (kf < 1 || kf >= ktf) return NONE;
  if (kf >= 3 && kf < ktf - 2) return FIFTH;
  return kf == 1 || kf == ktf - 1 ? FZ : THIRD;
}

// Weights of the points at face - 3 .. face + 2 in the face value, by rule:
// under the positive upwind choice, then under the negative one (FZ's are the
// level's fzm and fzp).
__constant__ const float kWeights[7][12] = {
    {},
    {2.0f / 60, -13.0f / 60, 47.0f / 60, 27.0f / 60, -3.0f / 60, 0, 0, -3.0f / 60, 27.0f / 60, 47.0f / 60, -13.0f / 60, 2.0f / 60},
    {0, -2.0f / 12, 10.0f / 12, 4.0f / 12, 0, 0, 0, 0, 4.0f / 12, 10.0f / 12, -2.0f / 12, 0},
    {0, 0, 0.5f, 0.5f, 0, 0, 0, 0, 0.5f, 0.5f, 0, 0},
    {},
    {0, 0, 0, 1.0f, 0, 0, 0, 0, 0.5f, 0.5f, 0, 0},
    {0, 0, 1.0f, 0, 0, 0, 0, 0, 0.5f, 0.5f, 0, 0}};

// acc plus the share of the point at face + o, for the face's weighted
// sensitivity P under the positive upwind choice, N under the negative one
__device__ __forceinline__ float fifth(int o, float P, float N, float acc) {
  const float cp[6] = {2.0f / 60, -13.0f / 60, 47.0f / 60, 27.0f / 60, -3.0f / 60, 0.0f};
  if (o < 2) acc = __builtin_fmaf(cp[o + 3], P, acc);
  if (o > -3) acc = __builtin_fmaf(cp[2 - o], N, acc);   // the mirrored weights: cn(o) = cp(-1 - o)
  return acc;
}
// the same for any rule; a point outside the stencil takes nothing, not 0 times the face
__device__ __forceinline__ float share(int rule, int o, float P, float N, float fm, float fp, float acc) {
  float cp = kWeights[rule][o + 3], cn = kWeights[rule][o + 9];
  if (o == 0 || o == -1) {
    if (rule == FZ) cp = cn = o == 0 ? fm : fp;
  }
  if (cp != 0.0f) acc = __builtin_fmaf(cp, P, acc);
  if (cn != 0.0f) acc = __builtin_fmaf(cn, N, acc);
  return acc;
}

// a face with sensitivity gF and mass flux vel; a face no point takes carries
// nothing, whatever the flux there holds
__device__ __forceinline__ void split(float gF, float vel, bool pos, float& P, float& N) {
  const float x = gF == 0.0f ? 0.0f : gF * vel;
  P = pos ? x : 0.0f;
  N = pos ? 0.0f : x;
}

template <int KIND>
__global__ void __launch_bounds__(PW_TX * PW_TY) k_adv_adj(Dims D, AdvAdj a, int kc_len) {
  constexpr int R = AA_R;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y), lane = (int)threadIdx.x;
  const int k0 = (int)blockIdx.z * kc_len, k1 = imin(k0 + kc_len, D.nz);
  const int c0 = a.i0 + (int)blockIdx.x * 58, i = c0 - 3 + lane;
  const int j0 = a.j0 + ((int)blockIdx.y * PW_TY + wave) * R;
  const Box& b = a.b;
  if (!a.accumulate) {   // points no stencil reaches
    for (int k = k0; k < k1; ++k)
      for (int j = (int)blockIdx.y * PW_TY + wave; j < D.ny; j += (int)gridDim.y * PW_TY)
        for (int ii = (int)blockIdx.x * PW_TX + lane; ii < D.nx; ii += (int)gridDim.x * PW_TX)
          if (j < a.j0 || j >= a.j1 || ii < a.i0 || ii >= a.i1) AT(a.out, k, j, ii) = 0.0f;
  }
  if (j0 >= a.j1) return;
  // indices clamped into the array so that every load is unconditional; what
  // is taken at a clamped index is masked
  const int ic = imin(imax(i, 0), D.nx - 1);
  auto row = [&](int j) { return imin(imax(j, 0), D.ny - 1); };
  auto lev = [&](int k) { return imin(imax(k, 0), D.nz - 1); };
  const bool own = lane >= 3 && lane < 61 && i < a.i1;
  const bool inb = i >= b.i0 && i < b.i1, inx = i >= a.bx.i0 && i < a.bx.i1;
  const bool xin = c0 - 2 >= a.ids + 3 && c0 + 60 < (KIND == WIND_U ? a.ide - 2 : a.ide - 3);   // 5th-order x-faces only
  float wy[R + 6], wx[R], wz[R];   // weights of a point's y-, x- and z-terms
#pragma unroll
  for (int o = 0; o < R + 6; ++o) {
    const int j = j0 - 3 + o;
    const float m = AT2(a.mA, row(j), ic);
    wy[o] = inb && j >= a.by.j0 && j < a.by.j1 ? m * a.rdy : 0.0f;
    if (o >= 3 && o < R + 3) {
      wx[o - 3] = inx && j >= a.bx.j0 && j < a.bx.j1 ? m * a.rdx : 0.0f;
      const bool in = inb && j >= b.j0 && j < b.j1;
      wz[o - 3] = in ? (KIND == WIND_V ? m / AT2(a.mB, row(j), ic) : 1.0f) : 0.0f;
    }
  }
  const int xrule = hrule(i, a.ids, a.ide, KIND == WIND_U);
  float xw[12];   // the weights of the lane's own x-face
  if (!xin) {
#pragma unroll
    for (int o = 0; o < 12; ++o) xw[o] = kWeights[xrule][o];
  }
  auto masked = [](float w, float x) { return w != 0.0f ? w * x : 0.0f; };
  // mass flux along z at face kf of row j, from x = rom there and y = the other value it is the mean of
  auto zother = [&](int kf, int j) -> float {
    if (KIND == WIND_V) return AT(a.rom, lev(kf), row(j - 1), ic);
    if (KIND == WIND_W) return AT(a.rom, lev(kf - 1), row(j), ic);
    return 0.0f;
  };
  auto zvel = [&](float x, float y) -> float {
    if (KIND == WIND_U) return 0.5f * (lane_below(x) + x);
    return KIND == SCALAR ? x : 0.5f * (x + y);
  };
  // the two values a horizontal flux f (ru or rv) of row j at level k is interpolated from (w; else the first)
  auto hload = [&](const float* f, int k, int j, float& x, float& y) {
    const bool top = KIND == WIND_W && k >= a.ktf;
    x = AT(f, top ? a.ktf - 1 : k, row(j), ic);
    y = KIND == WIND_W ? AT(f, imax(top ? a.ktf - 2 : k - 1, 0), row(j), ic) : 0.0f;
  };
  auto hlevel = [&](int k, float x, float y) -> float {
    if (KIND != WIND_W) return x;
    const bool top = k >= a.ktf;
    const float m = level(a.fzm, top ? a.ktf - 1 : k), p = level(a.fzp, top ? a.ktf - 1 : k);
    return top ? (2.0f - m) * x - p * y : m * x + p * y;
  };
  // weight of the tendency at level k in its low z-face (of its high one: the same below the top)
  auto zlow = [&](int k) -> float {
    const bool top = KIND == WIND_W && k == a.ktf;
    const float x = level(a.rdz, top ? a.ktf - 1 : lev(k));
    return k < b.k0 || k >= b.k1 ? 0.0f : top ? 2.0f * x : x;
  };
  auto zhigh = [&](int k) -> float {
    const float x = level(a.rdz, lev(k));
    return k < b.k0 || k >= b.k1 || (KIND == WIND_W && k == a.ktf) ? 0.0f : x;
  };
  // the z-face kf of row j0 + r from the adjoint tendencies below and above it
  auto zface = [&](int kf, int r, float vel, float lo, float hi, float& P, float& N) {
    const int rule = zrule<KIND>(kf, a.ktf);
    const float gF = rule == NONE ? 0.0f : masked(wz[r] * zlow(kf), hi) - masked(wz[r] * zhigh(kf - 1), lo);
    // the reference's sign at the 3rd-order face below the top of v and w
    const bool flip = (KIND == WIND_V && rule == THIRD && kf != 2) || (KIND == WIND_W && rule == THIRD && kf != 2);
    split(gF, vel, flip ? vel >= 0.0f : -vel >= 0.0f, P, N);
  };
  float zp[R][6], zn[R][6], zl[R];   // faces k-2 .. k+3 around level k, and the adjoint tendency at the last one's level
  {
    float l[R][6], v[R][5];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int m = 0; m < 6; ++m) l[r][m] = AT(a.lam, lev(k0 - 3 + m), row(j0 + r), ic);
#pragma unroll
      for (int m = 0; m < 5; ++m) v[r][m] = zvel(AT(a.rom, lev(k0 - 2 + m), row(j0 + r), ic), zother(k0 - 2 + m, j0 + r));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int m = 0; m < 5; ++m)   // the march's first step adds the sixth
        zface(k0 - 2 + m, r, v[r][m], l[r][m], l[r][m + 1], zp[r][m + 1], zn[r][m + 1]);
      zl[r] = l[r][5];
    }
  }
  // what a level loads, all before its arithmetic (fetching the next level's too: no faster)
  struct Level { float L[R + 6], y0[R + 6], y1[R + 6], qy[R + 6], x0[R], x1[R], qx[R], lz[R], z0[R], z1[R], told[R]; };
  auto fetch = [&](int k, Level& v) {
#pragma unroll
    for (int o = 0; o < R + 6; ++o) {
      v.L[o] = AT(a.lam, k, row(j0 - 3 + o), ic);
      if (KIND == WIND_V || o > 0) hload(a.rv, k, j0 - 3 + o, v.y0[o], v.y1[o]);   // at the face below row j0 - 3 + o
      if (KIND == WIND_V) v.qy[o] = AT(a.q, k, row(j0 - 3 + o), ic);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      hload(a.ru, k, j0 + r, v.x0[r], v.x1[r]);
      if (KIND == WIND_V) v.x1[r] = AT(a.ru, k, row(j0 + r - 1), ic);
      if (KIND == WIND_U) v.qx[r] = AT(a.q, k, row(j0 + r), ic);
      v.lz[r] = AT(a.lam, lev(k + 3), row(j0 + r), ic);
      v.z0[r] = AT(a.rom, lev(k + 3), row(j0 + r), ic);
      v.z1[r] = zother(k + 3, j0 + r);
      v.told[r] = a.accumulate ? AT(a.out, k, row(j0 + r), ic) : 0.0f;
    }
  };
#pragma unroll 1
  for (int k = k0; k < k1; ++k) {
    const bool kin = k >= b.k0 && k < b.k1;
    Level v;
    fetch(k, v);
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    if (kin) {
      // y: the faces j0 - 2 .. j0 + R + 2, each handed to the rows it weighs
      const bool yin = j0 - 2 >= a.jds + 3 && j0 + R + 2 < (KIND == WIND_V ? a.jde - 2 : a.jde - 3);
      float A = masked(wy[0], v.L[0]);
#pragma unroll
      for (int m = 0; m < R + 5; ++m) {
        const int jf = j0 - 2 + m;
        const float B = masked(wy[m + 1], v.L[m + 1]);
        float vel = hlevel(k, v.y0[m + 1], v.y1[m + 1]);
        if (KIND == WIND_U) vel = 0.5f * (vel + lane_below(vel));
        if (KIND == WIND_V) vel = 0.5f * (vel + v.y0[m]);
        float P, N;
        if (yin) {
          split(B - A, vel, vel >= 0.0f, P, N);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (r + 2 - m >= -3 && r + 2 - m <= 2) acc[r] = fifth(r + 2 - m, P, N, acc[r]);
        } else {
          const int rule = hrule(jf, a.jds, a.jde, KIND == WIND_V);
          bool pos = vel >= 0.0f;
          if (KIND == WIND_U && jf == a.jde - 3) pos = true;   // the sign the forward takes there
          if (KIND == WIND_V && rule == END_LO) pos = v.qy[m + 1] < 0.0f;
          if (KIND == WIND_V && rule == END_HI) pos = v.qy[m] > 0.0f;
          split(rule == NONE ? 0.0f : B - A, vel, pos, P, N);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (r + 2 - m >= -3 && r + 2 - m <= 2) acc[r] = share(rule, r + 2 - m, P, N, 0.0f, 0.0f, acc[r]);
        }
        A = B;
      }
      // x: each lane forms the face below its column; a point reads those of lanes -2 .. +3
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float ax = masked(wx[r], v.L[r + 3]);
        float vel = hlevel(k, v.x0[r], v.x1[r]);
        if (KIND == WIND_U) vel = 0.5f * (vel + lane_below(vel));
        if (KIND == WIND_V) vel = 0.5f * (vel + v.x1[r]);
        const float gF = ax - lane_below(ax);
        if (xin) {
          float P[6], N[6];
          split(gF, vel, vel >= 0.0f, P[2], N[2]);
          P[1] = lane_below(P[2]); P[0] = lane_below(P[1]);
          N[1] = lane_below(N[2]); N[0] = lane_below(N[1]);
          P[3] = lane_above(P[2]); P[4] = lane_above(P[3]); P[5] = lane_above(P[4]);
          N[3] = lane_above(N[2]); N[4] = lane_above(N[3]); N[5] = lane_above(N[4]);
#pragma unroll
          for (int m = 0; m < 6; ++m) acc[r] = fifth(2 - m, P[m], N[m], acc[r]);
        } else {   // the face's own lane weighs it for the six points, which then read their shares
          const float vnext = lane_above(vel), qw = KIND == WIND_U ? lane_below(v.qx[r]) : 0.0f;
          bool pos = vel >= 0.0f;
          if (KIND == SCALAR && i == a.ide - 3) pos = vnext >= 0.0f;   // sign from ru at ide - 2
          if (KIND == WIND_U && xrule == END_LO) pos = v.qx[r] < 0.0f;
          if (KIND == WIND_U && xrule == END_HI) pos = qw > 0.0f;
          const float x = xrule == NONE || gF == 0.0f ? 0.0f : gF * vel;
          float S[6];
#pragma unroll
          for (int o = 0; o < 6; ++o) {
            const float c = pos ? xw[o] : xw[o + 6];
            S[o] = c != 0.0f ? c * x : 0.0f;
          }
          acc[r] += S[3] + lane_above(S[2]) + lane_above(lane_above(S[1])) + lane_above(lane_above(lane_above(S[0]))) +
                    lane_below(S[4]) + lane_below(lane_below(S[5]));
        }
      }
    }
    // z: slide the window up and add the face k + 3
    const bool zin = k - 2 >= 3 && k + 3 < (KIND == WIND_W ? a.ktf - 1 : a.ktf - 2);
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int m = 0; m < 5; ++m) { zp[r][m] = zp[r][m + 1]; zn[r][m] = zn[r][m + 1]; }
      zface(k + 3, r, zvel(v.z0[r], v.z1[r]), zl[r], v.lz[r], zp[r][5], zn[r][5]);
      zl[r] = v.lz[r];
#pragma unroll
      for (int m = 0; m < 6; ++m) {
        if (zin) {
          acc[r] = fifth(2 - m, zp[r][m], zn[r][m], acc[r]);
        } else {
          const int kf = k - 2 + m, kl = lev(kf);
          acc[r] = share(zrule<KIND>(kf, a.ktf), 2 - m, zp[r][m], zn[r][m], level(a.fzm, kl), level(a.fzp, kl), acc[r]);
        }
      }
      if (own && j0 + r < a.j1) AT(a.out, k, j0 + r, i) = v.told[r] + acc[r];
    }
  }
}

template <int KIND>
int launch(const pywrf_grid_t* g, AdvAdj& a, pywrf_stream_t s) {
  a.j0 = imax(g->jts - 3, g->jds); a.j1 = imin(g->jte + 3, g->jde);
  a.i0 = imax(g->its - 3, g->ids); a.i1 = imin(g->ite + 3, g->ide);
  const int gx = imax(1, (a.i1 - a.i0 + 57) / 58);
  // levels a wave: a short march where eight levels would leave fewer than four
  // waves for each of the 1024 SIMDs (120x120x41: 16.1 us a call with 3, 19.9
  // with 4, 27.6 with 8; the scalar at 240x240x41: 28.4, 29.0, 27.8)
  const int kc = (long)gx * ((a.j1 - a.j0 + AA_R - 1) / AA_R) * ((g->nz + 7) / 8) >= 4096 ? 8 : 3;
  const int gy = imax(1, (a.j1 - a.j0 + AA_R * PW_TY - 1) / (AA_R * PW_TY));
  auto kern = k_adv_adj<KIND>;
  hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)gy, (unsigned)((g->nz + kc - 1) / kc)), dim3(PW_TX, PW_TY), 0,
                     (hipStream_t)s, dims_of(g), a, kc);
  PW_RET();
}

// the common fields; the boxes' common columns and rows are [i0, i1) x [j0, j1)
AdvAdj common(const pywrf_grid_t* g, const float* lam, const float* ru, const float* rv, const float* rom,
              const float* mA, const float* fzm, const float* fzp, const float* rdz, double rdx, double rdy,
              float* out) {
  AdvAdj a = {};
  a.lam = lam; a.ru = ru; a.rv = rv; a.rom = rom; a.mA = mA; a.mB = mA; a.fzm = fzm; a.fzp = fzp; a.rdz = rdz;
  a.out = out; a.rdx = F(rdx); a.rdy = F(rdy);
  a.ids = g->ids; a.ide = g->ide; a.jds = g->jds; a.jde = g->jde; a.ktf = imin(g->kte, g->kde - 1);
  return a;
}

}  // namespace

extern "C" int pywrf_advect_scalar_adjoint(const pywrf_grid_t* g, const float* lam_tend, const float* ru,
                                           const float* rv, const float* rom, const float* msftx, const float* fzm,
                                           const float* fzp, double rdx, double rdy, const float* rdzw,
                                           float* lam_field, int accumulate, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 4);
  AdvAdj a = common(g, lam_tend, ru, rv, rom, msftx, fzm, fzp, rdzw, rdx, rdy, lam_field);
  a.accumulate = accumulate;
  if (g->kts != 0 || a.ktf + 1 > g->nz || g->kte > g->nz) return PYWRF_E_RANGE;
  const int i0 = g->its, i1 = imin(g->ite, g->ide - 1), j0 = g->jts, j1 = imin(g->jte, g->jde - 1);
  a.b = mkbox(g->kts, a.ktf, j0, j1, i0, i1);
  a.by = mkbox(g->kts, a.ktf, imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2), i0, i1);
  a.bx = mkbox(g->kts, a.ktf, j0, j1, imax(g->ids + 1, g->its), imin(g->ide - 2, g->ite));
  return launch<SCALAR>(g, a, s);
}

extern "C" int pywrf_advect_u_adjoint(const pywrf_grid_t* g, const float* lam_tendency, const float* u,
                                      const float* ru, const float* rv, const float* rom, const float* msfux,
                                      const float* fzm, const float* fzp, double rdx, double rdy,
                                      const float* rdzw, float* lam_u, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 4);
  AdvAdj a = common(g, lam_tendency, ru, rv, rom, msfux, fzm, fzp, rdzw, rdx, rdy, lam_u);
  a.q = u;
  if (g->kts != 0 || a.ktf + 1 > g->nz) return PYWRF_E_RANGE;
  const int i0 = imax(g->ids + 1, g->its), i1 = imin(g->ide - 1, g->ite);
  const int j0 = g->jts, j1 = imin(g->jte, g->jde - 1);
  a.b = a.bx = mkbox(g->kts, a.ktf, j0, j1, i0, i1);
  a.by = mkbox(g->kts, a.ktf, imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2), i0, i1);
  return launch<WIND_U>(g, a, s);
}

extern "C" int pywrf_advect_v_adjoint(const pywrf_grid_t* g, const float* lam_tendency, const float* v,
                                      const float* ru, const float* rv, const float* rom, const float* msfvx,
                                      const float* msfvy, const float* fzm, const float* fzp, double rdx, double rdy,
                                      const float* rdzw, float* lam_v, pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 4);
  AdvAdj a = common(g, lam_tendency, ru, rv, rom, msfvy, fzm, fzp, rdzw, rdx, rdy, lam_v);
  a.q = v;
  a.mB = msfvx;
  if (g->kts != 0 || a.ktf + 1 > g->nz) return PYWRF_E_RANGE;
  const int i0 = g->its, i1 = imin(g->ite, g->ide - 1);
  const int j0 = imax(g->jts, g->jds + 1), j1 = imin(g->jte, g->jde - 1);
  a.b = a.by = mkbox(g->kts, a.ktf, j0, j1, i0, i1);
  a.bx = mkbox(g->kts, a.ktf, j0, j1, imax(g->ids + 1, g->its), imin(g->ide - 2, g->ite));
  return launch<WIND_V>(g, a, s);
}

extern "C" int pywrf_advect_w_adjoint(const pywrf_grid_t* g, const float* lam_tendency, const float* ru,
                                      const float* rv, const float* rom, const float* msftx, const float* fzm,
                                      const float* fzp, double rdx, double rdy, const float* rdzu, float* lam_w,
                                      pywrf_stream_t s) {
  if (!pw_size_ok(g)) return PYWRF_E_RANGE;
  CHECK(g, 4);
  AdvAdj a = common(g, lam_tendency, ru, rv, rom, msftx, fzm, fzp, rdzu, rdx, rdy, lam_w);
  if (g->kts != 0 || a.ktf + 1 > g->nz || a.ktf < 3) return PYWRF_E_RANGE;
  const int i0 = g->its, i1 = imin(g->ite, g->ide - 1);
  const int j0 = g->jts, j1 = imin(g->jte, g->jde - 1);
  a.b = mkbox(g->kts + 1, a.ktf + 1, j0, j1, i0, i1);
  a.by = mkbox(g->kts + 1, a.ktf + 1, imax(g->jts, g->jds + 1), imin(g->jte, g->jde - 2), i0, i1);
  a.bx = mkbox(g->kts + 1, a.ktf + 1, j0, j1, imax(g->ids + 1, g->its), imin(g->ide - 2, g->ite));
  return launch<WIND_W>(g, a, s);
}
