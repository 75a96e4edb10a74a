// Trees of one shape: a free root link with four equal legs (serial hinge
// chains of K links), one lane per leg.
//
// One thread per env makes a substep of such a robot one dependent chain of
// some 14,000 instructions without contacts, on a wavefront that has its SIMD
// to itself (the tree's arrays fill the register file), so a call takes as
// long for one robot as for 65,536.  Here an env is a quad of lanes: lane b
// holds leg b, and every lane holds the root.  The legs' work goes on side by
// side, the root's is repeated on the four lanes, and what the legs add to
// the root (subtree forces, composite inertias, the factor's update, the
// solver's dot products) are sums over the quad, two DPP additions each with
// no LDS and no wait.  16 envs share a wavefront.
//
// What bounds it: the chain of one wavefront (378 registers and 36 KB of LDS
// for the quadruped: one wavefront per SIMD).  One thread per env against this
// kernel: 27 -> 6.3 us a substep off the ground for 8,192 quadrupeds, 72 -> 21
// us for one quadruped on the floor, 140 -> 26 us for 4,096 ants, 146 -> 109 us
// for 65,536 quadrupeds with their frames.
//
// The constrained products need no tree pass: with M = L^T L the rows
// L^-T J^T of a lane's contacts and limits are formed once per substep (they
// live on the lane's leg and the root: K + 6 numbers), and
// A v = (L^-T J^T)^T (L^-T J^T) v + diag v is two dot products per row and
// one quad sum of six.  Every candidate keeps a slot on its lane, so there is
// no second path for many contacts; a slot that no lane of the wavefront
// uses is skipped.  The step is the reference's (pipeline.py:64-94) as
// bgx_step.h restates it.
//
// The four lanes of an env must agree bit for bit on the root and on every
// decision: quad_sum adds commutatively and keeps the compiler from fusing
// its additions with the lane's own products.
#pragma once

#include <hip/hip_runtime.h>

#include "bgx_launch.h"
#include "bgx_batch.h"
#include "bgx_step.h"

namespace bgx {

constexpr int STAR_ENVS = WAVE / STAR_LEGS;  // envs per wavefront

template <class T>
struct Star {
  static constexpr int K = (T::L - 1) / STAR_LEGS;
  static constexpr int NCL = [] {
    int j = 0;
    while (star_leg_cand<T>(0, j) >= 0) ++j;
    return j;
  }();
  static constexpr int NCR = T::NCAND - STAR_LEGS * NCL;  // on the root, lane j holds the j-th
  static constexpr int S = NCL + (NCR > 0 ? 1 : 0);       // slots of a lane
  static constexpr int SN = S > 0 ? S : 1;
  static constexpr int CSTEP = NCL > 0 ? star_leg_cand<T>(1, 0) - star_leg_cand<T>(0, 0) : 0;
  // last leg link whose dofs move slot s's link (-1: the root)
  static constexpr int link(int s) {
    return s < NCL ? T::CAND_LINK[star_leg_cand<T>(0, s)] - 1 : -1;
  }
  static constexpr int cand0(int s) {
    return s < NCL ? star_leg_cand<T>(0, s) : star_root_cand<T>(0);
  }
};

// the sum of x over the env's quad, the same bits on its four lanes; every
// lane of the quad must be active
BGX_D float quad_sum(float x) {
#pragma clang fp contract(off)
  asm("" : "+v"(x));
  const float y =
      x + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1,
                                                             0xf, 0xf, true));
  return y + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, y), 0x4E,
                                                                0xf, 0xf, true));
}
BGX_D V3 quad_sum(V3 v) { return V3{quad_sum(v.x), quad_sum(v.y), quad_sum(v.z)}; }
// the lanes of this lane's quad for which p holds
BGX_D unsigned quad_ballot(bool p) {
  return (unsigned)(__ballot(p) >> (threadIdx.x & (WAVE - STAR_LEGS))) & 0xfu;
}
template <class X>
BGX_D X by_leg(int b, X x0, X x1, X x2, X x3) {
  const X lo = (b & 1) ? x1 : x0, hi = (b & 1) ? x3 : x2;
  return (b & 2) ? hi : lo;
}
// the actuator of leg b's k-th hinge
template <class T>
BGX_D int star_act_of_leg(int b, int k) {
  constexpr int K = Star<T>::K;
  return by_leg(b, star_act<T>(6 + k), star_act<T>(6 + K + k), star_act<T>(6 + 2 * K + k),
                star_act<T>(6 + 3 * K + k));
}

// the limit row of leg b's k-th hinge
template <class T>
constexpr int star_lim_row(int d) {
  for (int i = 0; i < T::NLIM; ++i)
    if (T::LIM_D[i] == d) return i;
  return 0;
}
template <class T>
BGX_D int star_lim_of_leg(int b, int k) {
  constexpr int K = Star<T>::K;
  return by_leg(b, star_lim_row<T>(6 + k), star_lim_row<T>(6 + K + k),
                star_lim_row<T>(6 + 2 * K + k), star_lim_row<T>(6 + 3 * K + k));
}

template <class T>
struct StarState {
  static constexpr int K = Star<T>::K;
  float rq[7], rv[6];  // root, the same on the four lanes
  float q[K], qd[K];   // this lane's leg
};

// the state from / to an env's rows; the root's entries are spread over the
// quad, so that a wavefront's stores cover whole rows
template <class T>
BGX_D void star_load(StarState<T>& s, int b, const float* qp, const float* qdp) {
  constexpr int K = Star<T>::K;
#pragma unroll
  for (int k = 0; k < 7; ++k) s.rq[k] = qp[k];
#pragma unroll
  for (int k = 0; k < 6; ++k) s.rv[k] = qdp[k];
#pragma unroll
  for (int k = 0; k < K; ++k) s.q[k] = qp[7 + b * K + k], s.qd[k] = qdp[6 + b * K + k];
}
template <class T>
BGX_D void star_store_q(const StarState<T>& s, int b, float* qp) {
  constexpr int K = Star<T>::K;
  qp[b] = by_leg(b, s.rq[0], s.rq[1], s.rq[2], s.rq[3]);
  if (b < 3) qp[4 + b] = by_leg(b, s.rq[4], s.rq[5], s.rq[6], 0.f);
#pragma unroll
  for (int k = 0; k < K; ++k) qp[7 + b * K + k] = s.q[k];
}
template <class T>
BGX_D void star_store_qd(const StarState<T>& s, int b, float* qdp) {
  constexpr int K = Star<T>::K;
  qdp[b] = by_leg(b, s.rv[0], s.rv[1], s.rv[2], s.rv[3]);
  if (b < 2) qdp[4 + b] = by_leg(b, s.rv[4], s.rv[5], 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < K; ++k) qdp[6 + b * K + k] = s.qd[k];
}

// world frames of the root and of this lane's leg (kinematics.py:31-108);
// XD: also the frames' velocities
template <class T, bool XD, class S>
BGX_D void star_frames(const float* ml, int b, const S* rq, const S* q, const float* rv,
                       const float* qd, V3T<S>& xp0, Q4T<S>& xr0, V3T<S>* xp, Q4T<S>* xr,
                       V3T<S>* xa0, V3T<S>* xa, V3T<S>* xv) {
  constexpr int K = Star<T>::K;
  const float* lk = ml + T::OFF_LINK;
  {
    V3T<S> p{rq[0], rq[1], rq[2]};
    const Q4T<S> r{rq[3], rq[4], rq[5], rq[6]};
    const V3T<S> jpos = lift3<S>(ldv3(lk + LK_JPOS));
    p = (p + jpos) - rotate(jpos, r);
    const Q4T<S> trot = lift4<S>(ldq4(lk + LK_TROT));
    xp0 = lift3<S>(ldv3(lk + LK_TPOS)) + rotate(p, trot);
    xr0 = qmul(trot, r);
  }
  if constexpr (XD) *xa0 = rotate(lift3<S>(v3(rv[3], rv[4], rv[5])), xr0);
  lk += LINK_STRIDE * (1 + b * K);
  const float* df = ml + T::OFF_DOF + DOF_STRIDE * (6 + b * K);
#pragma unroll
  for (int k = 0; k < K; ++k, lk += LINK_STRIDE, df += DOF_STRIDE) {
    const V3T<S> ang = lift3<S>(ldv3(df + DF_ANG));
    const Q4T<S> rk = qnormalize(qrot_axis(ang, q[k]));
    const V3T<S> jpos = lift3<S>(ldv3(lk + LK_JPOS));
    const Q4T<S> trot = lift4<S>(ldq4(lk + LK_TROT));
    const V3T<S> p = lift3<S>(ldv3(lk + LK_TPOS)) + rotate(jpos - rotate(jpos, rk), trot);
    const V3T<S> pp = k == 0 ? xp0 : xp[k - 1];
    const Q4T<S> pr = k == 0 ? xr0 : xr[k - 1];
    xp[k] = pp + rotate(p, pr);
    xr[k] = qmul(pr, qmul(trot, rk));
    if constexpr (XD) {
      const V3T<S> pa = k == 0 ? *xa0 : xa[k - 1];
      const V3T<S> pv = k == 0 ? lift3<S>(v3(rv[0], rv[1], rv[2])) : xv[k - 1];
      xv[k] = pv + cross(pa, xp[k] - pp);
      xa[k] = pa + rotate(ang * qd[k], xr[k]);
    }
  }
  xr0 = qnormalize(xr0);
#pragma unroll
  for (int k = 0; k < K; ++k) xr[k] = qnormalize(xr[k]);
}

// mass-weighted COM offset and rotational inertia of one link about rc
// (dynamics.py:44-55)
template <class S>
BGX_D void star_inertia(const float* lk, V3T<S> xp, Q4T<S> xr, V3T<S> rc, V3T<S>& cc,
                        Sym3T<S>& ci) {
  const V3T<S> p = (xp + rotate(lift3<S>(ldv3(lk + LK_IPOS)), xr)) - rc;
  const float m = lk[LK_MASS];
  S R[3][3], RI[3][3];
  quat_to_3x3(qmul(xr, lift4<S>(ldq4(lk + LK_IROT))), R);
  const float* i0 = lk + LK_I;
  const Sym3T<S> I0{lift<S>(i0[0]), lift<S>(i0[1]), lift<S>(i0[2]),
                    lift<S>(i0[3]), lift<S>(i0[4]), lift<S>(i0[5])};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const V3T<S> c = symmul(I0, V3T<S>{R[i][0], R[i][1], R[i][2]});
    RI[i][0] = c.x, RI[i][1] = c.y, RI[i][2] = c.z;
  }
  auto rir = [&](int i, int j) {
    return RI[i][0] * R[j][0] + RI[i][1] * R[j][1] + RI[i][2] * R[j][2];
  };
  const S pp = dot(p, p);
  ci = Sym3T<S>{rir(0, 0) + (pp - p.x * p.x) * m, rir(1, 1) + (pp - p.y * p.y) * m,
                rir(2, 2) + (pp - p.z * p.z) * m, rir(0, 1) - p.x * p.y * m,
                rir(0, 2) - p.x * p.z * m, rir(1, 2) - p.y * p.z * m};
  cc = p * m;
}

// M = L^T L of the env: this leg's block and its columns at the root, and
// the root's block (the same on the four lanes); inv: 1 / diagonal of L
template <int K>
struct StarFactor {
  float leg[K][K], col[K][6], root[6][6], inv[K], inv0[6];

  // z = L^-T z, a vector that lives on this leg and the root alone
  BGX_D void lt_own(float* z, float* zr) const {
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      z[k] *= inv[k];
#pragma unroll
      for (int j = 0; j < k; ++j) z[j] -= leg[k][j] * z[k];
#pragma unroll
      for (int j = 0; j < 6; ++j) zr[j] -= col[k][j] * z[k];
    }
    lt_root(zr);
  }
  BGX_D void lt_root(float* zr) const {
#pragma unroll
    for (int i = 5; i >= 0; --i) {
      zr[i] *= inv0[i];
#pragma unroll
      for (int j = 0; j < i; ++j) zr[j] -= root[i][j] * zr[i];
    }
  }
  // z = L^-T z of a whole env's vector
  BGX_D void lt(float* z, float* zr) const {
    float p[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      z[k] *= inv[k];
#pragma unroll
      for (int j = 0; j < k; ++j) z[j] -= leg[k][j] * z[k];
#pragma unroll
      for (int j = 0; j < 6; ++j) p[j] += col[k][j] * z[k];
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) zr[j] -= quad_sum(p[j]);
    lt_root(zr);
  }
  // z = L^-1 z of a whole env's vector
  BGX_D void l(float* z, float* zr) const {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
#pragma unroll
      for (int j = 0; j < i; ++j) zr[i] -= root[i][j] * zr[j];
      zr[i] *= inv0[i];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
      for (int j = 0; j < 6; ++j) z[k] -= col[k][j] * zr[j];
#pragma unroll
      for (int j = 0; j < k; ++j) z[k] -= leg[k][j] * z[j];
      z[k] *= inv[k];
    }
  }
};

// The contact rows of a lane: slot i's row x = L^-T J^T along n, mu t1 or
// mu t2, K + 6 numbers (leg, then root).  Up to two slots stay in registers;
// more would push the solver's vectors into accumulation registers, a move
// for every use, so they live in LDS: float4 q of a row at
// base[(q WAVE + lane) 4], read without bank conflicts.
template <class T>
struct StarRows {
  static constexpr int K = Star<T>::K, W = (K + 6 + 3) / 4 * 4, Q = W / 4;
  static constexpr bool LDS = Star<T>::S > 2;
  static constexpr int FLOATS = LDS ? Star<T>::S * 3 * W * WAVE : 0;
  float4* base;
  float r[LDS ? 1 : Star<T>::SN][3][W];
  BGX_D void put(int i, int x, const float* v) {
    if constexpr (LDS) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
        base[((i * 3 + x) * Q + q) * WAVE] =
            float4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    } else {
#pragma unroll
      for (int k = 0; k < W; ++k) r[i][x][k] = v[k];
    }
  }
  BGX_D void get(int i, float (*v)[W]) const {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      if constexpr (LDS) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const float4 f = base[((i * 3 + x) * Q + q) * WAVE];
          v[x][4 * q] = f.x, v[x][4 * q + 1] = f.y, v[x][4 * q + 2] = f.z, v[x][4 * q + 3] = f.w;
        }
      } else {
#pragma unroll
        for (int k = 0; k < W; ++k) v[x][k] = r[i][x][k];
      }
    }
  }
  // fn(i, rows of slot i) for the slots that are on.  The next slot's rows are
  // read before, on or not (an unused slot's are never looked at): behind its
  // branch, they would be waited for with nothing else to do.
  template <class Fn>
  BGX_D void each(const bool* on, Fn fn) const {
    float next[3][W];
    if (Star<T>::S > 0) get(0, next);
#pragma unroll
    for (int i = 0; i < Star<T>::S; ++i) {
      float j[3][W];
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int k = 0; k < W; ++k) j[x][k] = next[x][k];
      if (i + 1 < Star<T>::S) get(i + 1, next);
      if (on[i]) fn(i, j);
    }
  }
};

// LDS of a wavefront (floats): the model table, then the contact rows
template <class T>
constexpr int star_table_floats() { return (T::SIZE + 3) / 4 * 4; }
template <class T>
constexpr int star_lds_floats() { return star_table_floats<T>() + StarRows<T>::FLOATS; }

// one substep (pipeline.step, pipeline.py:64-94).  ml: the model table in
// LDS; probe (or null): the env's probe row.  Returns the active contacts.
template <class T>
BGX_D int star_substep(float* ml, int b, StarState<T>& s, const float* act,
                       float* probe) {
  using SR = Star<T>;
  constexpr int K = SR::K, S = SR::S, SN = SR::SN, NV = T::NV;
  const float* lk0 = ml + T::OFF_LINK;
  const float* lkb = lk0 + LINK_STRIDE * (1 + b * K);
  const float* df0 = ml + T::OFF_DOF;
  const float* dfb = df0 + DOF_STRIDE * (6 + b * K);

  V3 xp0, xp[K];
  Q4 xr0, xr[K];
  star_frames<T, false, float>(ml, b, s.rq, s.q, nullptr, nullptr, xp0, xr0, xp, xr, nullptr,
                               nullptr, nullptr);

  // ---- root COM (dynamics.py:37-43), cinr (:44-55)
  const float m0 = lk0[LK_MASS];
  V3 rc;
  {
    V3 sm = v3zero();
    float ms = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const float* lk = lkb + LINK_STRIDE * k;
      sm = sm + (xp[k] + rotate(ldv3(lk + LK_IPOS), xr[k])) * lk[LK_MASS];
      ms = ms + lk[LK_MASS];
    }
    sm = (xp0 + rotate(ldv3(lk0 + LK_IPOS), xr0)) * m0 + quad_sum(sm);
    const float ims = rcp(m0 + quad_sum(ms));
    rc = V3{sm.x * ims, sm.y * ims, sm.z * ims};
  }
  V3 cc0, cc[K];
  Sym3 ci0, ci[K];
  float km[K];
  star_inertia(lk0, xp0, xr0, rc, cc0, ci0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    star_inertia(lkb + LINK_STRIDE * k, xp[k], xr[k], rc, cc[k], ci[k]);
    km[k] = lkb[LINK_STRIDE * k + LK_MASS];
  }

  // ---- cdof (dynamics.py:56-89): the root's translations are the world's
  // axes, its rotations (ra, rv); the leg's hinges (ca, cv)
  V3 ra[3], rv[3], ca[K], cv[K];
  {
    const Q4 jr = qmul(xr0, ldq4(lk0 + LK_TROT));
    const V3 jp = (xp0 + rotate(ldv3(lk0 + LK_TPOS), xr0)) + rotate(ldv3(lk0 + LK_JPOS), jr);
    const V3 off = rc - jp;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      ra[k] = rotate(unit3(k), jr);
      rv[k] = cross(ra[k], off);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float* lk = lkb + LINK_STRIDE * k;
    const V3 pp = k == 0 ? xp0 : xp[k - 1];
    const Q4 pr = k == 0 ? xr0 : xr[k - 1];
    const Q4 jr = qmul(pr, ldq4(lk + LK_TROT));
    const V3 jp = (pp + rotate(ldv3(lk + LK_TPOS), pr)) + rotate(ldv3(lk + LK_JPOS), jr);
    ca[k] = rotate(ldv3(dfb + DOF_STRIDE * k + DF_ANG), jr);
    cv[k] = cross(ca[k], rc - jp);
  }

  // ---- link velocities (dynamics.py:90-103)
  const V3 rlin = v3(s.rv[0], s.rv[1], s.rv[2]);
  const V3 va0 = ra[0] * s.rv[3] + ra[1] * s.rv[4] + ra[2] * s.rv[5];
  const V3 vv0 = rlin + (rv[0] * s.rv[3] + rv[1] * s.rv[4] + rv[2] * s.rv[5]);
  V3 va[K], vv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    va[k] = (k == 0 ? va0 : va[k - 1]) + ca[k] * s.qd[k];
    vv[k] = (k == 0 ? vv0 : vv[k - 1]) + cv[k] * s.qd[k];
  }

  // ---- RNEA bias (dynamics.py:105-184), passive and actuator forces
  // (:187-236, actuator.py:23-57)
  float z[K], zr[6];  // qf_smooth
  {
    const V3 acc0 = cross(rlin, va0) - ldv3(ml + H_GRAVITY);  // linear; no angular part
    V3 f2a, f2v, f3a, f3v;
    inertia_mul(cc0, ci0, m0, va0, vv0, f2a, f2v);
    cross_force(va0, vv0, f2a, f2v, f3a, f3v);
    const V3 fa0 = cross(cc0, acc0) + f3a, fv0 = acc0 * m0 + f3v;
    V3 aa = v3zero(), av = acc0, fa[K], fv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      V3 oa, ov, f1a, f1v;
      cross_motion(k == 0 ? va0 : va[k - 1], k == 0 ? vv0 : vv[k - 1], ca[k], cv[k], oa, ov);
      aa = aa + oa * s.qd[k], av = av + ov * s.qd[k];
      inertia_mul(cc[k], ci[k], km[k], aa, av, f1a, f1v);
      inertia_mul(cc[k], ci[k], km[k], va[k], vv[k], f2a, f2v);
      cross_force(va[k], vv[k], f2a, f2v, f3a, f3v);
      fa[k] = f1a + f3a, fv[k] = f1v + f3v;
    }
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      if (k + 1 < K) fa[k] = fa[k] + fa[k + 1], fv[k] = fv[k] + fv[k + 1];
      const float* df = dfb + DOF_STRIDE * k;
      float p = -df[DF_DAMPING] * s.qd[k];
      p = -s.q[k] * df[DF_STIFFNESS] + p;
      z[k] = p - (dot(cv[k], fv[k]) + dot(ca[k], fa[k]));
      if (star_act<T>(6 + k) >= 0) {
        const float* ac = ml + T::OFF_ACT + star_act_of_leg<T>(b, k) * ACT_STRIDE;
        const float ctl = clipf(act[k], ac[AC_CTRL_LO], ac[AC_CTRL_HI]);
        const float bias = ac[AC_GEAR] * (s.q[k] * ac[AC_BIAS_Q] + s.qd[k] * ac[AC_BIAS_QD]);
        z[k] += clipf(ac[AC_GAIN] * ctl + bias, ac[AC_FORCE_LO], ac[AC_FORCE_HI]) * ac[AC_GEAR];
      }
    }
    const V3 Fa = fa0 + quad_sum(fa[0]), Fv = fv0 + quad_sum(fv[0]);
    zr[0] = Fv.x, zr[1] = Fv.y, zr[2] = Fv.z;
#pragma unroll
    for (int k = 0; k < 3; ++k) zr[3 + k] = dot(rv[k], Fv) + dot(ra[k], Fa);
#pragma unroll
    for (int k = 0; k < 6; ++k) zr[k] = -df0[DOF_STRIDE * k + DF_DAMPING] * s.rv[k] - zr[k];
  }
  if (probe) {
#pragma unroll
    for (int k = 0; k < K; ++k) probe[6 + b * K + k] = z[k];
    if (b == 0)
#pragma unroll
      for (int k = 0; k < 6; ++k) probe[k] = zr[k];
  }

  // ---- mass.matrix (mass.py:27-83) and its factor, leaves first
  StarFactor<K> F;
  {
#pragma unroll
    for (int k = K - 1; k > 0; --k) {
      cc[k - 1] = cc[k - 1] + cc[k];
      ci[k - 1] = symadd(ci[k - 1], ci[k]);
      km[k - 1] = km[k - 1] + km[k];
    }
    float up[6][6];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      V3 fa, fv;
      inertia_mul(cc[k], ci[k], km[k], ca[k], cv[k], fa, fv);
      F.leg[k][k] = dot(cv[k], fv) + dot(ca[k], fa) + dfb[DOF_STRIDE * k + DF_ARMATURE];
#pragma unroll
      for (int j = 0; j < k; ++j) F.leg[k][j] = dot(cv[j], fv) + dot(ca[j], fa);
      F.col[k][0] = fv.x, F.col[k][1] = fv.y, F.col[k][2] = fv.z;
#pragma unroll
      for (int j = 0; j < 3; ++j) F.col[k][3 + j] = dot(rv[j], fv) + dot(ra[j], fa);
    }
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      const float lkk = fsqrt(F.leg[k][k]);
      F.inv[k] = rcp(lkk);
#pragma unroll
      for (int j = 0; j < k; ++j) F.leg[k][j] *= F.inv[k];
#pragma unroll
      for (int j = 0; j < 6; ++j) F.col[k][j] *= F.inv[k];
#pragma unroll
      for (int i = 0; i < k; ++i) {
        const float a = F.leg[k][i];
#pragma unroll
        for (int j = 0; j <= i; ++j) F.leg[i][j] -= a * F.leg[k][j];
#pragma unroll
        for (int j = 0; j < 6; ++j) F.col[i][j] -= a * F.col[k][j];
      }
#pragma unroll
      for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j)
          up[i][j] = (k == K - 1 ? 0.f : up[i][j]) + F.col[k][i] * F.col[k][j];
    }
    const V3 tc = cc0 + quad_sum(cc[0]);
    const Sym3 ti{ci0.xx + quad_sum(ci[0].xx), ci0.yy + quad_sum(ci[0].yy),
                  ci0.zz + quad_sum(ci[0].zz), ci0.xy + quad_sum(ci[0].xy),
                  ci0.xz + quad_sum(ci[0].xz), ci0.yz + quad_sum(ci[0].yz)};
    const float tm = m0 + quad_sum(km[0]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      V3 fa, fv;
      inertia_mul(tc, ti, tm, ra[i], rv[i], fa, fv);
      F.root[3 + i][0] = fv.x, F.root[3 + i][1] = fv.y, F.root[3 + i][2] = fv.z;
#pragma unroll
      for (int j = 0; j <= i; ++j) F.root[3 + i][3 + j] = dot(rv[j], fv) + dot(ra[j], fa);
#pragma unroll
      for (int j = 0; j <= i; ++j) F.root[i][j] = j == i ? tm : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) F.root[i][i] += df0[DOF_STRIDE * i + DF_ARMATURE];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) F.root[i][j] -= quad_sum(up[i][j]);
#pragma unroll
    for (int k = 5; k >= 0; --k) {
      F.inv0[k] = rcp(fsqrt(F.root[k][k]));
#pragma unroll
      for (int j = 0; j < k; ++j) F.root[k][j] *= F.inv0[k];
#pragma unroll
      for (int i = 0; i < k; ++i) {
        const float a = F.root[k][i];
#pragma unroll
        for (int j = 0; j <= i; ++j) F.root[i][j] -= a * F.root[k][j];
      }
    }
  }

  // ---- w = L^-T qf_smooth; the unconstrained acceleration is L^-1 w
  float w[K], wr[6];
#pragma unroll
  for (int k = 0; k < K; ++k) w[k] = z[k];
#pragma unroll
  for (int k = 0; k < 6; ++k) wr[k] = zr[k];
  F.lt(w, wr);

  // ---- contact rows (contact.py + MJX plane collisions, constraint.py):
  // slot s has three rows of L^-T J^T, along n, mu t1 and mu t2 (its pyramid
  // rows are n + mu t, n - mu t), on the leg jl and the root jr
  using SRows = StarRows<T>;
  SRows J;
  J.base = (float4*)(ml + star_table_floats<T>()) + threadIdx.x % WAVE;
  float diag[SN], sb[SN][4];
  bool on[SN];  // slots that any lane of the wavefront uses
  bool active[SN];
  int n_c = 0;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    constexpr int NCL = SR::NCL;
    const bool leg = i < NCL;
    const int kk = SR::link(i);
    const int c0 = SR::cand0(i);
    const bool held = leg || b < SR::NCR;
    const float* cd = ml + T::OFF_CAND +
                      CAND_STRIDE * (c0 + (leg ? b * SR::CSTEP : (held ? b : 0)));
    const V3 xpl = leg ? xp[kk >= 0 ? kk : 0] : xp0;
    const Q4 xrl = leg ? xr[kk >= 0 ? kk : 0] : xr0;
    V3 ctr = xpl + rotate(ldv3(cd + CD_GPOS), xrl);
    V3 axis = v3zero();
    if (T::CAND_KIND[c0] == KIND_CAPSULE) {
      axis = quat_zaxis(qmul(xrl, ldq4(cd + CD_GQUAT)));
      ctr = ctr + axis * (cd[CD_HALFLEN] * cd[CD_SIGN]);
    }
    const float radius = cd[CD_RADIUS];
    const float dist = (ctr.z - cd[CD_PPOS + 2]) - radius;
    active[i] = held && dist < 0.f;
    on[i] = __ballot(active[i]) != 0ull;
    n_c += __builtin_popcount(quad_ballot(active[i]));
    diag[i] = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) sb[i][k] = 0.f;
    if (on[i]) {
      float j[3][SRows::W];  // this slot's rows
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int k = 0; k < SRows::W; ++k) j[x][k] = 0.f;
      V3 t1 = ldv3(cd + CD_T1);
      if (T::CAND_KIND[c0] == KIND_CAPSULE) {
        // along the capsule where it lies, y where it stands
        float bn;
        const V3 bt = vnormalize(v3(axis.x, axis.y, 0.f), &bn);
        t1 = bn < 0.5f ? v3(0.f, 1.f, 0.f) : bt;
      }
      const float mu = cd[CD_MU], tw = cd[CD_TW];
      const float* im = cd + CD_IMP;
      const float imp = impedance(im, dist);
      const V3 r = v3(ctr.x, ctr.y, ctr.z - (radius + 0.5f * dist)) - rc;
      const float az = active[i] ? 1.f : 0.f;
      const float ax = active[i] ? t1.x * mu : 0.f, ay = active[i] ? t1.y * mu : 0.f;
      diag[i] = active[i] ? (tw + mu * mu * tw) * (2.f * mu * mu * imp_ratio(imp)) : 0.f;
      auto rows = [&](V3 v, float& e0, float& e1, float& e2) {
        e0 = az * v.z;
        e1 = ax * v.x + ay * v.y;
        e2 = ax * v.y - ay * v.x;
      };
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (k <= kk) rows(cv[k] + cross(ca[k], r), j[0][k], j[1][k], j[2][k]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        rows(unit3(k), j[0][K + k], j[1][K + k], j[2][K + k]);
        rows(rv[k] + cross(ra[k], r), j[0][K + 3 + k], j[1][K + 3 + k], j[2][K + 3 + k]);
      }
      // velocity of the contact point at qd
      const V3 ka = leg ? va[kk >= 0 ? kk : 0] : va0, kv = leg ? vv[kk >= 0 ? kk : 0] : vv0;
      float q0, q1, q2, e[3];
      rows(kv + cross(ka, r), q0, q1, q2);
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        F.lt_own(j[x], j[x] + K);
        J.put(i, x, j[x]);
        e[x] = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) e[x] += j[x][k] * w[k];
#pragma unroll
        for (int k = 0; k < 6; ++k) e[x] += j[x][K + k] * wr[k];
      }
      const float kt = active[i] ? im[IM_K] * imp * dist : 0.f, bq = im[IM_B];
      sb[i][0] = (e[0] + e[1]) + (bq * (q0 + q1) + kt);
      sb[i][1] = (e[0] - e[1]) + (bq * (q0 - q1) + kt);
      sb[i][2] = (e[0] + e[2]) + (bq * (q0 + q2) + kt);
      sb[i][3] = (e[0] - e[2]) + (bq * (q0 - q2) + kt);
    }
  }

  // ---- u = M^-1 qf_smooth
  float u[K], ur[6];
#pragma unroll
  for (int k = 0; k < K; ++k) u[k] = w[k];
#pragma unroll
  for (int k = 0; k < 6; ++k) ur[k] = wr[k];
  F.l(u, ur);

  // ---- limit rows (constraint.py:101-132): side times a row of L^-T
  float ll[K][K], lr[K][6], ldiag[K], lb[K];
  bool act_l[K];
  bool any_l = false;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    act_l[k] = false, ldiag[k] = 0.f, lb[k] = 0.f;
    if (!star_lim<T>(6 + k)) continue;
    const float* df = dfb + DOF_STRIDE * k;
    const float pmin = s.q[k] - df[DF_LO], pmax = df[DF_HI] - s.q[k];
    const float pos = fminf(fminf(pmin, pmax), 0.f);
    act_l[k] = pos < 0.f;
    const float side = act_l[k] ? (pmin < pmax ? 1.f : -1.f) : 0.f;
    const float* im = df + DF_IMP;
    const float imp = impedance(im, pos);
    const float aref = act_l[k] ? (-im[IM_B] * (side * s.qd[k]) - im[IM_K] * imp * pos) : 0.f;
    ldiag[k] = act_l[k] ? df[DF_INVWEIGHT] * imp_ratio(imp) : 0.f;
    lb[k] = side * u[k] - aref;
#pragma unroll
    for (int j = 0; j < K; ++j) ll[k][j] = j == k ? side : 0.f;
#pragma unroll
    for (int j = 0; j < 6; ++j) lr[k][j] = 0.f;
    any_l = any_l || act_l[k];
  }
  const bool on_l = __ballot(any_l) != 0ull;
  if (on_l) {
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (star_lim<T>(6 + k)) F.lt_own(ll[k], lr[k]);
  }

  bool mine = any_l;
#pragma unroll
  for (int i = 0; i < S; ++i) mine = mine || active[i];
  const bool has_rows = quad_ballot(mine) != 0u;
  int iters = 0, trials = 0;
  if (__ballot(has_rows) != 0ull) {
    // ---- jaxopt.ProjectedGradient: FISTA + backtracking line search from 0;
    // an env's control is the same on its four lanes
    float X[SN][4], Y[SN][4], G[SN][4], R[SN][4];
    float xl[K], yl[K], gl[K], rl[K];
#pragma unroll
    for (int i = 0; i < SN; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) X[i][k] = Y[i][k] = G[i][k] = R[i][k] = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) xl[k] = yl[k] = gl[k] = rl[k] = 0.f;
    // products with A = P^T P + diag, P = L^-T J^T.  A sweep over the rows ends
    // one product and begins the next, t being P in of the product that ends:
    // out receives A in, then nxt gives the next input of the same row, summed
    // into t.  So a product reads its rows once, where summing and applying in
    // turn reads them twice, and where rows live in LDS those reads (1 KB an
    // instruction) are the solver's longest stretch.  65,536 quadrupeds, us a
    // substep, the same bits: 130 -> 94 over 40 env steps from a standing
    // start, 166 -> 117 once settled on the floor.
    float t[K], tr[6], p[6];
    auto add_slot = [&](int i, const float (*j)[SRows::W], auto nxt) {
      const float v0 = nxt(i, 0), v1 = nxt(i, 1), v2 = nxt(i, 2), v3_ = nxt(i, 3);
      const float a[3] = {(v0 + v1) + (v2 + v3_), v0 - v1, v2 - v3_};
#pragma unroll
      for (int x = 0; x < 3; ++x) {
#pragma unroll
        for (int k = 0; k < K; ++k)
          if (k <= SR::link(i)) t[k] += a[x] * j[x][k];
#pragma unroll
        for (int k = 0; k < 6; ++k) p[k] += a[x] * j[x][K + k];
      }
    };
    auto add_limit = [&](int k, float v) {
#pragma unroll
      for (int j = 0; j <= k; ++j) t[j] += v * ll[k][j];
#pragma unroll
      for (int j = 0; j < 6; ++j) p[j] += v * lr[k][j];
    };
    auto clear = [&]() {
#pragma unroll
      for (int k = 0; k < K; ++k) t[k] = 0.f;
#pragma unroll
      for (int k = 0; k < 6; ++k) p[k] = 0.f;
    };
    auto sum_root = [&]() {
#pragma unroll
      for (int k = 0; k < 6; ++k) tr[k] = quad_sum(p[k]);
    };
    // t = P nxt
    auto gather = [&](auto nxt, auto nxt_l) {
      clear();
      J.each(on, [&](int i, const float (*j)[SRows::W]) { add_slot(i, j, nxt); });
      if (on_l) {
#pragma unroll
        for (int k = 0; k < K; ++k)
          if (star_lim<T>(6 + k)) add_limit(k, nxt_l(k));
      }
      sum_root();
    };
    // out = A in (t = P in), then t = P nxt where next says so
    auto sweep = [&](auto in, auto in_l, auto out, auto out_l, auto next, auto nxt, auto nxt_l) {
      constexpr bool NEXT = decltype(next)::value;
      float u_[K];
#pragma unroll
      for (int k = 0; k < K; ++k) u_[k] = t[k];
      if constexpr (NEXT) clear();
      J.each(on, [&](int i, const float (*j)[SRows::W]) {
        float e[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          e[x] = 0.f;
#pragma unroll
          for (int k = 0; k < 6; ++k) e[x] += j[x][K + k] * tr[k];
#pragma unroll
          for (int k = 0; k < K; ++k)
            if (k <= SR::link(i)) e[x] += j[x][k] * u_[k];
        }
        out(i, 0, e[0] + e[1] + diag[i] * in(i, 0));
        out(i, 1, e[0] - e[1] + diag[i] * in(i, 1));
        out(i, 2, e[0] + e[2] + diag[i] * in(i, 2));
        out(i, 3, e[0] - e[2] + diag[i] * in(i, 3));
        if constexpr (NEXT) add_slot(i, j, nxt);
      });
      if (on_l) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (!star_lim<T>(6 + k)) continue;
          float e = 0.f;
#pragma unroll
          for (int j = 0; j < 6; ++j) e += lr[k][j] * tr[j];
#pragma unroll
          for (int j = 0; j <= k; ++j) e += ll[k][j] * u_[j];
          out_l(k, e + ldiag[k] * in_l(k));
          if constexpr (NEXT) add_limit(k, nxt_l(k));
        }
      }
      if constexpr (NEXT) sum_root();
    };
    // A product that may not be wanted (after a rejected or a last step) begins
    // in the sweep before it only where that saves reads of LDS.  Ants, whose
    // rows are in registers, take 18.4 us a substep at 4,096 without and 20.6
    // with it.
    constexpr std::true_type always{};
    constexpr std::bool_constant<SRows::LDS> if_lds{};
    const int maxiter = (int)ml[H_MAXITER], maxls = (int)ml[H_MAXLS];
    const float tol = ml[H_TOL], lseps = ml[H_LSEPS];
    float tk = 1.f, eta = 1.f, err;
    auto y_ = [&](int i, int k) { return Y[i][k]; };
    auto y_l = [&](int k) { return yl[k]; };
    auto r_ = [&](int i, int k) { return R[i][k]; };
    auto r_l = [&](int k) { return rl[k]; };
    // x+ = relu(y - eta g) and d = x+ - y
    auto x_ = [&](int i, int k) { return fmaxf(Y[i][k] - eta * G[i][k], 0.f); };
    auto x_l = [&](int k) { return fmaxf(yl[k] - eta * gl[k], 0.f); };
    auto d_ = [&](int i, int k) { return x_(i, k) - Y[i][k]; };
    auto d_l = [&](int k) { return x_l(k) - yl[k]; };
    // the residual at y = 0
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) R[i][k] = sb[i][k];
#pragma unroll
    for (int k = 0; k < K; ++k) rl[k] = lb[k];
    bool running = has_rows && maxiter > 0;
    if (running) gather(r_, r_l);
    for (int it = 0; running; ++it) {
      // R is the residual r = A y + b: the gradient at y is g = A^T r
      float dd = 0.f;
      auto next_d = [&](int i, int k) {
        const float d = d_(i, k);
        dd += d * d;
        return d;
      };
      auto next_dl = [&](int k) {
        const float d = d_l(k);
        dd += d * d;
        return d;
      };
      sweep(r_, r_l, [&](int i, int k, float o) { G[i][k] = o; },
            [&](int k, float o) { gl[k] = o; }, always, next_d, next_dl);
      // line search over x+ = relu(y - eta g).  f is quadratic, so with
      // d = x+ - y its test f(x+) - f(y) > g.d + |d|^2 / (2 eta) is
      // |A d|^2 / 2 > |d|^2 / (2 eta), without the difference of two nearly
      // equal sums: fewer steps are decided by rounding (a tie still is), and
      // the taped substep decides by the same test (bgx_step.h).  R becomes
      // A d, the next input if the step is taken.
      for (int ls = 0;; ++ls) {
        float ad = 0.f;
        sweep(d_, d_l,
              [&](int i, int k, float o) {
                R[i][k] = o;
                ad += o * o;
              },
              [&](int k, float o) {
                rl[k] = o;
                ad += o * o;
              },
              if_lds, r_, r_l);
        trials += 1;
        if (!(eta * (0.5f * quad_sum(ad)) > 0.5f * quad_sum(dd) + lseps) || ls >= maxls) break;
        eta *= 0.5f;
        dd = 0.f;
        gather(next_d, next_dl);
      }
      if constexpr (!if_lds) gather(r_, r_l);
      // error at x+: |relu(x+ - grad f(x+)) - x+|, grad f(x+) = g + A^T A d;
      // and the next y, x+ + beta (x+ - x)
      const float tn = 0.5f * (1.f + fsqrt(1.f + 4.f * tk * tk));
      const float beta = (tk - 1.f) * rcp(tn);
      float e2 = 0.f;
      sweep(r_, r_l,
            [&](int i, int k, float o) {
              const float xn = x_(i, k);
              const float dv = fmaxf(xn - (G[i][k] + o), 0.f) - xn;
              e2 += dv * dv;
              Y[i][k] = xn + beta * (xn - X[i][k]);
              X[i][k] = xn;
            },
            [&](int k, float o) {
              const float xn = x_l(k);
              const float dv = fmaxf(xn - (gl[k] + o), 0.f) - xn;
              e2 += dv * dv;
              yl[k] = xn + beta * (xn - xl[k]);
              xl[k] = xn;
            },
            if_lds, y_, y_l);
      err = fsqrt(quad_sum(e2));
      eta = eta <= 1e-6f ? 1.f : eta * 2.f;
      tk = tn;
      iters += 1;
      running = err > tol && it + 1 < maxiter;
      if (running) {
        if constexpr (!if_lds) gather(y_, y_l);
        sweep(y_, y_l, [&](int i, int k, float o) { R[i][k] = o + sb[i][k]; },
              [&](int k, float o) { rl[k] = o + lb[k]; }, always, r_, r_l);
      }
    }
    // ---- qdd = u + L^-1 (L^-T J^T) x (integrator.py:58-64)
    gather([&](int i, int k) { return X[i][k]; }, [&](int k) { return xl[k]; });
    F.l(t, tr);
#pragma unroll
    for (int k = 0; k < K; ++k) u[k] = has_rows ? u[k] + t[k] : u[k];
#pragma unroll
    for (int k = 0; k < 6; ++k) ur[k] = has_rows ? ur[k] + tr[k] : ur[k];
  }
  if (probe) {
#pragma unroll
    for (int k = 0; k < K; ++k) probe[NV + 6 + b * K + k] = u[k];
    if (b == 0) {
#pragma unroll
      for (int k = 0; k < 6; ++k) probe[NV + k] = ur[k];
      probe[2 * NV] = (float)n_c;
      probe[2 * NV + 1] = (float)iters;
      probe[2 * NV + 2] = (float)trials;
    }
  }

  // ---- semi-implicit Euler (integrator.py:26-84)
  const float dt = ml[H_DT];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    s.qd[k] = s.qd[k] + u[k] * dt;
    s.q[k] = s.q[k] + s.qd[k] * dt;
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) s.rv[k] = s.rv[k] + ur[k] * dt;
  const Q4 rot = integrate_rot(Q4{s.rq[3], s.rq[4], s.rq[5], s.rq[6]},
                               v3(s.rv[3], s.rv[4], s.rv[5]), dt);
  s.rq[3] = rot.w, s.rq[4] = rot.x, s.rq[5] = rot.y, s.rq[6] = rot.z;
#pragma unroll
  for (int k = 0; k < 3; ++k) s.rq[k] = s.rq[k] + s.rv[k] * dt;
  return n_c;
}

// a pointer known to be LDS again after a call that is not inlined
BGX_D float* star_lds(float* p) { return (float*)(__attribute__((address_space(3))) float*)p; }

// The frames of an env's state (pipeline.init's x, xd).  A function of its
// own, so that a step's frames and init's are the same code: bitwise equal.
template <class T>
BGX_ITEM void star_write_frames(const Launch& a, long long env, int b, float* lds,
                                StarState<T> s, bool live) {
  constexpr int K = Star<T>::K;
  const float* ml = star_lds(lds);
  V3 xp0, xp[K], xa0, xa[K], xv[K];
  Q4 xr0, xr[K];
  star_frames<T, true, float>(ml, b, s.rq, s.q, s.rv, s.qd, xp0, xr0, xp, xr, &xa0, xa, xv);
  if (!live) return;
  const long long o = env * T::L, ol = o + 1 + b * K;
  auto put3 = [&](float* base, V3 root, const V3* leg) {
    if (!base) return;
    if (b < 3) base[3 * o + b] = by_leg(b, root.x, root.y, root.z, 0.f);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float* p = base + 3 * (ol + k);
      p[0] = leg[k].x, p[1] = leg[k].y, p[2] = leg[k].z;
    }
  };
  put3(a.x_pos, xp0, xp);
  if (a.x_rot) {
    a.x_rot[4 * o + b] = by_leg(b, xr0.w, xr0.x, xr0.y, xr0.z);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float* p = a.x_rot + 4 * (ol + k);
      p[0] = xr[k].w, p[1] = xr[k].x, p[2] = xr[k].y, p[3] = xr[k].z;
    }
  }
  put3(a.xd_ang, xa0, xa);
  put3(a.xd_vel, v3(s.rv[0], s.rv[1], s.rv[2]), xv);
}

// the model table at M into LDS (a wavefront's workgroup)
template <class T>
BGX_D void star_stage(const float* M, float* lds) {
  for (int i = threadIdx.x; i < T::SIZE; i += WAVE) lds[i] = M[i];
  __syncthreads();
}

// The LDS of a wavefront in star_item: one object for every kernel that calls
// it, so that its address is a constant there.  Behind a pointer from two
// callers the same substep took 512 registers and 640 bytes of scratch a lane
// instead of 378 and 400 (65,536 quadrupeds, one substep with its frames: 147
// us instead of 109).
template <class T>
BGX_D float* star_smem() {
  constexpr int N = star_lds_floats<T>();
  __shared__ __align__(16) float mem[T::BATCH && CHAIN_LDS_FLOATS > N ? CHAIN_LDS_FLOATS : N];
  return mem;
}

// The envs of one item (up to STAR_ENVS), n_steps x n_frames substeps.  An
// env past the item's count computes on the item's last env and writes
// nothing.  A function of its own (as chain_item): the homogeneous kernel and
// the batch kernel call the same code.
template <class T>
BGX_ITEM void star_item(const Launch& a, const BatchItem& it) {
  constexpr int K = Star<T>::K, NQ = T::NQ, NV = T::NV, NU = T::NU;
  float* lds = star_smem<T>();
  const int b = threadIdx.x % STAR_LEGS, e = threadIdx.x / STAR_LEGS;
  const bool live = e < it.n;
  const int ec = live ? e : it.n - 1;
  const long long env = it.env + ec;
  star_stage<T>(a.M + it.m_off, lds);
  float* qp = a.q + it.q + (long long)ec * NQ;
  float* qdp = a.qd + it.qd + (long long)ec * NV;
  const float* actp = (NU > 0 && a.act) ? a.act + it.act + (long long)ec * NU : nullptr;
  const long long n_sub = (long long)a.n_steps * a.n_frames, seg = blockIdx.y;
  float* subq = (live && a.sub_q) ? a.sub_q + (seg * n_sub * a.n + env) * NQ : nullptr;
  float* subqd = (live && a.sub_qd) ? a.sub_qd + (seg * n_sub * a.n + env) * NV : nullptr;
  float* probe = (live && a.probe) ? a.probe + env * (2 * NV + 3) : nullptr;
  StarState<T> s;
  star_load(s, b, a.q_in ? a.q_in + it.q + (long long)ec * NQ : qp,
            a.qd_in ? a.qd_in + it.qd + (long long)ec * NV : qdp);
  const int n_steps = a.n_steps, n_frames = a.n_frames;
  int st = 0;
  for (int t = 0; t < n_steps; ++t) {
    float act[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      act[k] = 0.f;
      if (star_act<T>(6 + k) >= 0) {
        if (actp) act[k] = actp[t * a.act_stride + star_act_of_leg<T>(b, k)];
      }
    }
    for (int f = 0; f < n_frames; ++f) {
      if (subq) {
        const long long o = ((long long)t * n_frames + f) * a.n;
        star_store_q(s, b, subq + o * NQ);
        star_store_qd(s, b, subqd + o * NV);
      }
      // the status of the one-thread kernel: more contacts than its slots
      if (star_substep<T>(lds, b, s, act, probe) > T::KC) st |= ST_SLOW_PATH;
    }
    if (live && a.q_traj) star_store_q(s, b, a.q_traj + t * a.q_step + it.q + (long long)e * NQ);
    if (live && a.qd_traj)
      star_store_qd(s, b, a.qd_traj + t * a.qd_step + it.qd + (long long)e * NV);
  }
  bool finite = true;
#pragma unroll
  for (int k = 0; k < 7; ++k) finite = finite && isfinite(s.rq[k]);
#pragma unroll
  for (int k = 0; k < 6; ++k) finite = finite && isfinite(s.rv[k]);
#pragma unroll
  for (int k = 0; k < K; ++k) finite = finite && isfinite(s.q[k]) && isfinite(s.qd[k]);
  if (quad_ballot(!finite) != 0u) st |= ST_NONFINITE;
  if (live) {
    star_store_q(s, b, qp);
    star_store_qd(s, b, qdp);
    if (a.status && b == 0) {
      if (a.n_seg > 1) atomicOr(a.status + env, st);
      else a.status[env] = a.status_or ? (a.status[env] | st) : st;
    }
  }
  if (a.x_pos || a.x_rot || a.xd_ang || a.xd_vel)
    star_write_frames<T>(a, env, b, lds, s, live);
}

// the item of a homogeneous launch's workgroup (checkpoint segment blockIdx.y)
template <class T>
BGX_D BatchItem star_home_item(const Launch& a) {
  BatchItem it{};
  const long long seg = blockIdx.y, env0 = (long long)blockIdx.x * STAR_ENVS;
  it.kind = BATCH_TREE;
  it.n = (int)(a.n - env0 < STAR_ENVS ? a.n - env0 : STAR_ENVS);
  it.env = env0;
  it.q = (seg * a.n + env0) * T::NQ, it.qd = (seg * a.n + env0) * T::NV;
  it.act = seg * a.seg_act_stride + env0 * T::NU;
  return it;
}

template <class T>
__global__ __launch_bounds__(WAVE) void k_star(Launch a) {
  star_item<T>(a, star_home_item<T>(a));
}

// the batch kernel (bgx_batch.h) of a topology of this shape
template <class T>
__global__ __launch_bounds__(WAVE) void k_star_batch(Launch a) {
  for (;;) {
    const int i = next_item(a);
    if (i < 0) break;
    const BatchItem it = a.items[i];
    if (it.kind == BATCH_CHAIN) run_chain_item(a, it, star_smem<T>());
    else star_item<T>(a, it);
    __syncthreads();  // the next item reuses the LDS
  }
  batch_done(a);
}

template <class T>
__global__ __launch_bounds__(WAVE) void k_star_init(Launch a) {
  __shared__ float lds[T::SIZE];
  const int b = threadIdx.x % STAR_LEGS;
  const long long env = (long long)blockIdx.x * STAR_ENVS + threadIdx.x / STAR_LEGS;
  const long long ec = env < a.n ? env : a.n - 1;
  star_stage<T>(a.M, lds);
  StarState<T> s;
  star_load(s, b, (a.q_in ? a.q_in : a.q) + ec * T::NQ, (a.qd_in ? a.qd_in : a.qd) + ec * T::NV);
  if (env < a.n) {
    if (a.q_in) star_store_q(s, b, a.q + env * T::NQ);
    if (a.qd_in) star_store_qd(s, b, a.qd + env * T::NV);
  }
  star_write_frames<T>(a, ec, b, lds, s, env < a.n);
}

}  // namespace bgx
