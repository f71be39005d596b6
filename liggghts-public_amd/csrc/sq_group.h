// Superquadric contact-point solve by eight lanes per pair: the arithmetic and
// control flow of the reference's calc_contact_point
// (math_extra_liggghts_superquadric.cpp:778-1022) and of the homotopy
// calc_contact_point_if_no_previous_point_avaialable (:1390-1430), the same
// operations in the same order but for the rounding of the powers (sq_pow.h),
// spread so that one Newton iteration is a short chain instead of a long one.
//
// What bounds it: a pair's solve is sequential, and of 100,000 random pairs the
// slowest takes thousands of iterations, so a launch lasts as long as one
// pair's chain. One thread per pair took 18 us for each of its iterations:
// four shape functions (five powers each, issued one after another) and a 4 x 4
// inverse, its arrays in scratch memory. Here
//   - four lanes (a quad) hold one particle: lane c raises local coordinate c
//     to its power, and lanes 0 and 1 the two powers of x^n2 + y^n2, so a shape
//     function is two powers deep; the other particle's quad does the same
//     beside it;
//   - every evaluation also forms the Hessian, lane c its column c: when the
//     point is accepted (nearly always) the next iteration's Jacobian is there
//     without another pair of shape functions;
//   - lane c owns column c of the Jacobian and forms the four cofactors of
//     row c of its inverse.
// Values move inside a row of 16 lanes by DPP (quad_perm, row_ror:8), not
// through LDS, which holds the power's tables and what a lane touches rarely.
// The 880 B of scratch that remain are the GMRES of a nearly singular Jacobian,
// kept out of line. An iteration takes 2.7 us. 100k fresh pairs: 126 -> 21 ms to
// 228 -> 33 ms by the slowest pair drawn; the pair kernels of 50k superquadrics
// (k_pair_start, k_pair_solve, k_pair_finish) 43 -> 7.4 ms a step.
#pragma once

#include "sq_device.h"
#include "sq_pow.h"

namespace sqd {

// lane layout in a row of 16: bits 0-1 column c, bit 2 which of the row's two
// pairs, bit 3 the particle (0: A, 1: B)
constexpr int kGroupLanes = 8;
constexpr int kGroupBlock = 64;                      // threads per block: one wavefront
constexpr int kGroupsPerBlock = kGroupBlock / kGroupLanes;

template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// lane K of the quad
template <int K> __device__ __forceinline__ double quad_bcast(double v) { return dpp_mov<K * 0x55>(v); }
// lane (c + K) % 4 of the quad
template <int K> __device__ __forceinline__ double quad_rot(double v) {
  return dpp_mov<((0 + K) % 4) | (((1 + K) % 4) << 2) | (((2 + K) % 4) << 4) | (((3 + K) % 4) << 6)>(v);
}
// the same lane of the other particle's quad (row_ror:8)
__device__ __forceinline__ double other_quad(double v) { return dpp_mov<0x128>(v); }

__device__ __forceinline__ double sel3(int c, double a, double b, double d) { return c == 0 ? a : (c == 1 ? b : d); }

// one particle of a pair on one lane of its quad
struct QSq {
  int c, isb;       // column (0-3; 3 repeats coordinate 2), particle
  double center[3];
  double rc[3], rr[3];  // column c and row c of the rotation
  double vinv;          // reciprocal half-axis of coordinate c
  double n1, n2;
  double e1, e2;        // this lane's exponents: of its coordinate, and of x^n2 + y^n2
                        // (even lanes n1 / n2, odd lanes that less 2)
  int i1, i2;           // the same as integers where the reference multiplies them out, else kNoInt
  double koef, minshape;  // minshape: the smallest half-axis (of both, once a stage is set)
};
constexpr int kNoInt = -1000;

__device__ __forceinline__ void q_set(const PowTab &t, QSq &s, double a, double b, double d, double n1, double n2) {
  s.vinv = 1.0 / sel3(s.c, a, b, d);
  s.minshape = fmin(fmin(a, b), d);
  s.n1 = n1;
  s.n2 = n2;
  s.koef = q_pow(t, 0.5, (n1 > n2 ? n1 : n2) - 2.0);
  const int ellipsoid = comp_double(n1, 2.0, 1e-2) && comp_double(n2, 2.0, 1e-2);
  const int int_blk = ellipsoid || (is_integer(n1) && is_integer(n2));
  const double ec = s.c < 2 ? n2 : n1;
  s.e1 = ec - 2.0;
  s.i1 = int_blk ? (int)floor(ec + 1e-2) - 2 : kNoInt;
  const double q = n1 / n2;
  const bool odd = (s.c & 1) != 0;
  s.e2 = odd ? q - 2.0 : q;
  s.i2 = odd && is_integer(q) ? (int)((double)(int)floor(q + 1e-2) - 2.0) : kNoInt;
}

// pose: center[3], quat[4] (w,i,j,k), shape[3], blockiness[2]
__device__ __forceinline__ void q_init(QSq &s, const double *pose) {
  Sq t;
  init(t, pose);
  const int lane = threadIdx.x & 15;
  s.c = lane & 3;
  s.isb = (lane >> 3) & 1;
  for (int k = 0; k < 3; k++) s.center[k] = t.center[k];
  for (int k = 0; k < 3; k++) {
    s.rc[k] = sel3(s.c, t.rot[3 * k], t.rot[3 * k + 1], t.rot[3 * k + 2]);
    s.rr[k] = sel3(s.c, t.rot[k], t.rot[3 + k], t.rot[6 + k]);
  }
}

// shape functions, gradients (both particles, on every lane) and this lane's
// column of its particle's Hessian at x
struct QEval {
  double f1, f2, gA[3], gB[3], h[3];
};

__device__ __forceinline__ void q_eval(const PowTab &t, const QSq &s, const double *x, QEval &e) {
  const double d[3] = {x[0] - s.center[0], x[1] - s.center[1], x[2] - s.center[2]};
  const double v = (s.rc[0] * d[0] + s.rc[1] * d[1] + s.rc[2] * d[2]) * s.vinv;
  const double av = fabs(v);
  double p22;
  if (s.i1 != kNoInt)
    p22 = pow_abs_int_sel(v, s.i1);
  else
    p22 = q_pow(t, av, s.e1);
  const double p21 = p22 * av, p2 = p21 * av;
  const double v0 = quad_bcast<0>(v), v1 = quad_bcast<1>(v);
  const double p210 = quad_bcast<0>(p21), p211 = quad_bcast<1>(p21);
  const double p20 = quad_bcast<0>(p2), p21_ = quad_bcast<1>(p2), zcn1 = quad_bcast<2>(p2);
  const double n1 = s.n1, n2 = s.n2, k = s.koef;
  const double ka = k * s.vinv;
  const int same = comp_double(n1, n2, 1e-2);
  const bool lat = s.c < 2;  // x or y
  double f, gl = ka * n1 * sgn(v) * p21, hd = n1 * ((lat ? n2 : n1) - 1.0) * p22, h01 = 0.0;
  if (same) {
    f = k * (p20 + p21_ + zcn1 - 1.0);
  } else {
    const double xy = p210 * fabs(v0) + p211 * fabs(v1);
    // lanes 0 and 2: (x^n2 + y^n2)^(n1/n2); lanes 1 and 3: the power less two
    double pw;
    if (s.i2 != kNoInt)
      pw = pow_abs_int(xy, s.i2);
    else
      pw = q_pow(t, fabs(xy), s.e2);
    const double xyp2 = quad_bcast<1>(pw);
    const double xyp1 = xyp2 * xy;
    f = k * (quad_bcast<0>(pw) + zcn1 - 1.0);
    if (lat) {
      gl *= xyp1;
      hd = hd * xyp1 + (n1 - n2) * n1 * p21 * p21 * xyp2;
    }
    const double pv = p21 * s.vinv;
    h01 = k * (n1 - n2) * n1 * sgn(v0) * sgn(v1) * quad_bcast<0>(pv) * quad_bcast<1>(pv) * xyp2;
  }
  hd = ka * hd * s.vinv;
  const double gl0 = quad_bcast<0>(gl), gl1 = quad_bcast<1>(gl), gl2 = quad_bcast<2>(gl);
  const double h00 = quad_bcast<0>(hd), h11 = quad_bcast<1>(hd), h22 = quad_bcast<2>(hd);
  // component c of the gradient and row c of rotation x local Hessian, then
  // every lane its column of (rotation x local Hessian) x rotation^T
  const double gc = s.rr[0] * gl0 + s.rr[1] * gl1 + s.rr[2] * gl2;
  const double t0 = s.rr[0] * h00 + s.rr[1] * h01;
  const double t1 = s.rr[0] * h01 + s.rr[1] * h11;
  const double t2 = s.rr[2] * h22;
  const double g[3] = {quad_bcast<0>(gc), quad_bcast<1>(gc), quad_bcast<2>(gc)};
  e.h[0] = quad_bcast<0>(t0) * s.rr[0] + quad_bcast<0>(t1) * s.rr[1] + quad_bcast<0>(t2) * s.rr[2];
  e.h[1] = quad_bcast<1>(t0) * s.rr[0] + quad_bcast<1>(t1) * s.rr[1] + quad_bcast<1>(t2) * s.rr[2];
  e.h[2] = quad_bcast<2>(t0) * s.rr[0] + quad_bcast<2>(t1) * s.rr[1] + quad_bcast<2>(t2) * s.rr[2];
  const double fo = other_quad(f);
  e.f1 = s.isb ? fo : f;
  e.f2 = s.isb ? f : fo;
  for (int i = 0; i < 3; i++) {
    const double go = other_quad(g[i]);
    e.gA[i] = s.isb ? go : g[i];
    e.gB[i] = s.isb ? g[i] : go;
  }
}

// the residual vector F of calc_F at a given mu, its square and the merit
__device__ __forceinline__ double q_residual(const QEval &e, double mu_sq, double *F, double &merit) {
  for (int k = 0; k < 3; k++) F[k] = e.gA[k] + mu_sq * e.gB[k];
  F[3] = e.f1 - e.f2;
  merit = merit_of(e.gA, e.gB, e.f1, e.f2);
  return F[0] * F[0] + F[1] * F[1] + F[2] * F[2] + F[3] * F[3];
}

// the point between the centres that splits their distance in `ratio`
__device__ __forceinline__ void q_between(const QSq &s, double ratio, double *p) {
  for (int k = 0; k < 3; k++) {
    const double o = other_quad(s.center[k]);
    const double ca = s.isb ? o : s.center[k], cb = s.isb ? s.center[k] : o;
    p[k] = ratio * cb + (1.0 - ratio) * ca;
  }
}

// out of line: a nearly singular Jacobian is rare, and its 100 values kept in
// registers would halve the wavefronts in flight
__device__ __noinline__ void gmres44_cold(const double *A, const double *b, const double *x0, double *x) {
  gmres44(A, b, x0, x);
}

// delta = J^-1 F where |det J| > 1, else GMRES from the last delta. jc is this
// lane's column of J. The reference decides by its own expansion of the
// determinant; where the cofactor expansion is beyond 1 by far more than
// either one's rounding error (below 1e-13 of the product of the column sums)
// the decision is known without it.
__device__ __forceinline__ void q_direction(int c, const double *jc, const double *F, double *delta) {
  // columns c, c+1, c+2, c+3 (mod 4)
  double m[4][4];
  for (int r = 0; r < 4; r++) {
    m[r][0] = jc[r];
    m[r][1] = quad_rot<1>(jc[r]);
    m[r][2] = quad_rot<2>(jc[r]);
    m[r][3] = quad_rot<3>(jc[r]);
  }
  // inv[4 c + i] of inv4: cofactor4(i, c) with the columns counted from c
  double inv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
#define SQG_E(a, b) m[(i + 6 + (b)) % 4][(6 + (a)) % 4]
    const double t = +SQG_E(+1, -1) * SQG_E(+0, +0) * SQG_E(-1, +1) + SQG_E(+1, +1) * SQG_E(+0, -1) * SQG_E(-1, +0) +
                     SQG_E(-1, -1) * SQG_E(+1, +0) * SQG_E(+0, +1) - SQG_E(-1, -1) * SQG_E(+0, +0) * SQG_E(+1, +1) -
                     SQG_E(-1, +1) * SQG_E(+0, -1) * SQG_E(+1, +0) - SQG_E(+1, -1) * SQG_E(-1, +0) * SQG_E(+0, +1);
#undef SQG_E
    inv[i] = ((c - i) & 1) ? t : -t;
  }
  const double part = jc[0] * inv[0];
  double D = 0;
  D += quad_bcast<0>(part);
  D += quad_bcast<1>(part);
  D += quad_bcast<2>(part);
  D += quad_bcast<3>(part);
  const double cs = fabs(jc[0]) + fabs(jc[1]) + fabs(jc[2]) + fabs(jc[3]);
  const double bound = (quad_bcast<0>(cs) * quad_bcast<1>(cs)) * (quad_bcast<2>(cs) * quad_bcast<3>(cs));
  bool invert = fabs(D) > 2.0 + 1e-12 * bound;
  if (!invert) {
    double J4[16];
    for (int r = 0; r < 4; r++) {
      J4[4 * r] = quad_bcast<0>(jc[r]);
      J4[4 * r + 1] = quad_bcast<1>(jc[r]);
      J4[4 * r + 2] = quad_bcast<2>(jc[r]);
      J4[4 * r + 3] = quad_bcast<3>(jc[r]);
    }
    invert = fabs(det4(J4)) > 1.0;
    if (!invert) {
      // copies: arrays whose address leaves the function live in scratch memory
      double Fc[4], d0[4], d1[4];
      cp4(Fc, F);
      cp4(d0, delta);
      gmres44_cold(J4, Fc, d0, d1);
      cp4(delta, d1);
    }
  }
  if (invert) {
    if (D != 0) {
      const double Di = 1.0 / D;
      for (int i = 0; i < 4; i++) inv[i] = inv[i] * Di;
    }
    double dc = 0.0;
    for (int j = 0; j < 4; j++)
      if (inv[j] != 0.0 && F[j] != 0.0) dc += inv[j] * F[j];
    delta[0] = quad_bcast<0>(dc);
    delta[1] = quad_bcast<1>(dc);
    delta[2] = quad_bcast<2>(dc);
    delta[3] = quad_bcast<3>(dc);
  }
}

// What a pair's solve starts from: the homotopy from volume-equivalent
// spheres; a given point, the homotopy when that solve fails or misses the
// merit tolerance; a given point only.
enum { kStartFresh = 0, kStartGiven = 1, kStartOnly = 2 };

// One pair as it is handed to the solve: the start, its point, and the point
// that stays when a given start breaks off.
struct QTask {
  double est[3], cp[3];
  int start;
};

struct QResult {
  double fi, fj, gA[3], gB[3];
  int iters, fail, fallback;
};

// What a lane touches rarely, in LDS instead of registers (each lane its own
// column): the stage's result so far, the pair's homotopy constants, the
// golden-section interval.
enum { kColdCp = 0, kColdRad = 3, kColdRatio, kColdNinv, kColdA, kColdB, kColdRes, kColdSize };
struct QCold {
  double v[kColdSize][kGroupBlock];
};
struct GroupLds {
  PowTab tab;
  QCold cold;
};

// Pairs from `src` until it has no more, solved by the groups of a wavefront
// side by side, as one loop over evaluations: groups at different places of
// their solves (a stage's two starts, a Newton step, a golden-section point)
// evaluate together, and a group that is done takes its next pair while the
// others go on. src.next(task), src.pose(pose) (this lane's particle of the pair: center,
// quat, shape, blockiness; read again at each stage, which is cheaper than 24
// registers) and src.put(result) are called by a group's eight lanes.
// Every iteration of the loop evaluates one point of each group's pair; a
// solve has at most max_iter iterations a stage, so the loop ends.
template <typename Source>
__device__ __forceinline__ void q_solve_all(Source &src, const int max_iter, GroupLds &shared) {
  QCold &lds = shared.cold;
  load_pow_tab(shared.tab);
  const int ln = threadIdx.x & 63;
#define SQG_COLD(k) lds.v[k][ln]
  const double tol1 = 1e-10, tol2 = 1e-12;
  enum { kInit1, kInit2, kTrial, kGoldA, kGoldB, kGoldEnd };
  int start;
  double x[3], mt = 0;  // the point to evaluate and its mu
  QSq s;
  QResult r;
  int N = 0, stage = 0;
  // the stage's solve: accepted point, its gradients, Hessian column, residual vector
  double point[3], mu = 0, F[4], h[3], delta[4] = {0, 0, 0, 0};
  double res1 = 0, merit1 = 0, alpha = 0;
  int iter = 0, phase = kInit1;
  bool fresh_pair = true, new_stage = true;
  for (;;) {
    if (fresh_pair) {
      QTask t;
      if (!src.next(t)) return;
      start = t.start;
      cp3(x, t.est);
      double pose[12];
      src.pose(pose);
      q_init(s, pose);
      const double rad = cbrt(pose[7] * pose[8] * pose[9]);
      const double rado = other_quad(rad);
      const double ri = s.isb ? rado : rad, rj = s.isb ? rad : rado;
      SQG_COLD(kColdRad) = rad;
      SQG_COLD(kColdRatio) = ri / (ri + rj);
      const double nown = fmax(pose[10], pose[11]), nmax = fmax(nown, other_quad(nown));
      const int N1 = (int)((nmax - 2.0) / 1.0 + 1);
      N = N1 > 10 ? N1 : 10;
      SQG_COLD(kColdNinv) = 1.0 / (double)N;
      r.iters = r.fail = r.fallback = 0;
      r.fi = r.fj = 0.0;
      for (int k = 0; k < 3; k++) SQG_COLD(kColdCp + k) = t.cp[k];
      stage = start == kStartFresh ? 0 : -1;
      fresh_pair = false;
    }
    if (new_stage) {
      double pose[12];
      src.pose(pose);
      const double n1 = pose[10], n2 = pose[11];
      double sh[3], m1 = n1, m2 = n2;
      for (int k = 0; k < 3; k++) sh[k] = pose[7 + k];
      if (stage >= 0) {
        const double rad = SQG_COLD(kColdRad), Ninv = SQG_COLD(kColdNinv);
        for (int k = 0; k < 3; k++) sh[k] = rad + (sh[k] - rad) * (double)stage * Ninv;
        m1 = 2.0 + (n1 - 2.0) * (double)stage * Ninv;
        m2 = 2.0 + (n2 - 2.0) * (double)stage * Ninv;
      }
      q_set(shared.tab, s, sh[0], sh[1], sh[2], m1, m2);
      s.minshape = fmin(s.minshape, other_quad(s.minshape));
      if (stage == 0) {
        q_between(s, SQG_COLD(kColdRatio), x);
        for (int k = 0; k < 3; k++) SQG_COLD(kColdCp + k) = x[k];
      } else if (stage > 0) {
        for (int k = 0; k < 3; k++) x[k] = SQG_COLD(kColdCp + k);
      }
      r.fail = 0;
      phase = kInit1;
      new_stage = false;
    }
    QEval e;
    q_eval(shared.tab, s, x, e);
    double mu_sq = mt * mt;
    if (phase <= kInit2) {
      mu_sq = -dot3(e.gA, e.gB) / dot3(e.gB, e.gB);
      mt = sqrt(fabs(mu_sq));
    }
    double Fe[4], merit;
    const double res = q_residual(e, mu_sq, Fe, merit);
    // whether this point becomes the solve's point, the iteration is over, the stage is over
    bool take = false, newton = false, over = false;
    if (phase == kInit1) {
      take = true;
      over = merit < tol1;
    } else if (phase == kInit2) {
      take = !(res1 < res);
      over = (take ? merit : merit1) < tol1;
      newton = !over;
    } else if (phase == kTrial) {
      const double deltax = fmax(fmax(fabs(delta[0]), fabs(delta[1])), fabs(delta[2]));
      take = res < res1 || merit < tol1 || deltax < tol2 * s.minshape;
      if (take) {
        over = merit < tol1 || deltax < tol2 * s.minshape;
      } else {
        SQG_COLD(kColdA) = 0.0;
        SQG_COLD(kColdB) = 1.0;
        phase = kGoldA;
      }
    } else if (phase == kGoldA) {
      SQG_COLD(kColdRes) = res;
      phase = kGoldB;
    } else if (phase == kGoldB) {
      // golden-section step; the point the search ends at is evaluated once
      // more, which spares keeping both candidates whole
      const double a = SQG_COLD(kColdA), b = SQG_COLD(kColdB), resa = SQG_COLD(kColdRes);
      const double alpha1 = b - (b - a) * kPhiInv;
      phase = kGoldA;
      if ((resa < res ? resa : res) < res1) {
        if (resa < res) alpha = alpha1;
        phase = kGoldEnd;
      } else {
        const double na = resa > res ? alpha1 : a, nb = resa > res ? b : alpha;
        SQG_COLD(kColdA) = na;
        SQG_COLD(kColdB) = nb;
        if (!(fabs(nb - na) > 1e-8)) phase = kGoldEnd;
      }
    } else {
      take = true;
      over = merit < tol1;
    }
    if (take) {
      if (phase >= kTrial) {
        if (fabs(res1 - res) / fmax(res1, res) < 1e-3) over = true;
        if (iter >= max_iter - 1) r.fail = 1;
        iter++;
        if (r.fail) over = true;
        newton = !over;
      }
      res1 = res;
      merit1 = merit;
      mu = mt;
      cp3(point, x);
      cp4(F, Fe);
      cp3(h, e.h);
      cp3(r.gA, e.gA);
      cp3(r.gB, e.gB);
      r.fi = e.f1;
      r.fj = e.f2;
    }
    bool keep_cp = false;  // the solve broke off: its result stays what it was
    if (phase == kInit1) {
      iter = 0;
      q_between(s, SQG_COLD(kColdRatio), x);
      phase = kInit2;
      for (int k = 0; k < 4; k++) delta[k] = 0.0;
    }
    if (newton) {
      double jc[4];
      const double msq = mu * mu;
      for (int i = 0; i < 3; i++) {
        const double ho = other_quad(h[i]);
        const double ha = s.isb ? ho : h[i], hb = s.isb ? h[i] : ho;
        const double col = ha + msq * hb;
        jc[i] = s.c < 3 ? col : 2.0 * mu * r.gB[i];
      }
      jc[3] = s.c < 3 ? sel3(s.c, r.gA[0] - r.gB[0], r.gA[1] - r.gB[1], r.gA[2] - r.gB[2]) : 0.0;
      q_direction(s.c, jc, F, delta);
      const bool nan = isnan(delta[0]) || isnan(delta[1]) || isnan(delta[2]) || isnan(delta[3]);
      const double deltax = fmax(fmax(fabs(delta[0]), fabs(delta[1])), fabs(delta[2]));
      if (nan) r.fail = 1;
      if (deltax == 0.0 || nan) {
        if (deltax == 0.0 && iter >= max_iter - 1) r.fail = 1;
        iter++;
        over = true;
        keep_cp = deltax != 0.0;
      }
      alpha = 1.0;
      phase = kTrial;
    }
    if (over) {
      if (!keep_cp)
        for (int k = 0; k < 3; k++) SQG_COLD(kColdCp + k) = point[k];
      r.iters += iter;
      iter = 0;
      bool done;
      if (stage < 0) {
        const double m = merit_of(r.gA, r.gB, r.fi, r.fj);
        done = start == kStartOnly || (!r.fail && m < 1e-10);
        if (!done) r.fallback = 1;
      } else {
        done = stage == N;
      }
      new_stage = true;
      stage++;
      if (done) {
        const double cp[3] = {SQG_COLD(kColdCp), SQG_COLD(kColdCp + 1), SQG_COLD(kColdCp + 2)};
        src.put(r, cp);
        fresh_pair = true;
      }
    } else if (phase >= kTrial) {
      // the next point along the step: the whole step, the two golden-section
      // points of [a, b], or the point the search ended at
      if (phase == kGoldA || phase == kGoldB) {
        const double a = SQG_COLD(kColdA), b = SQG_COLD(kColdB);
        alpha = phase == kGoldA ? b - (b - a) * kPhiInv : a + (b - a) * kPhiInv;
      }
      if (phase == kTrial) {
        for (int k = 0; k < 3; k++) x[k] = point[k] - delta[k];
        mt = mu - delta[3];
      } else {
        for (int k = 0; k < 3; k++) x[k] = point[k] + (-alpha) * delta[k];
        mt = mu - alpha * delta[3];
      }
    }
  }
#undef SQG_COLD
}

// the next free index below n of a queue shared by all groups (one atomic per
// group), or -1
__device__ __forceinline__ int64_t q_take(unsigned *queue, int64_t n) {
  const int lane = threadIdx.x & 15;
  int k = 0;
  if ((lane & 11) == 0) k = (int)atomicAdd(queue, 1u);
  k = __builtin_amdgcn_mov_dpp(k, 0x00, 0xf, 0xf, true);              // lane 0 of the quad
  const int o = __builtin_amdgcn_mov_dpp(k, 0x128, 0xf, 0xf, true);   // the other particle's quad
  k = (lane & 8) ? o : k;
  return (int64_t)(unsigned)k < n ? (int64_t)(unsigned)k : -1;
}

// whether this lane writes its group's results
__device__ __forceinline__ bool q_leader() { return (threadIdx.x & 11) == 0; }

}  // namespace sqd
