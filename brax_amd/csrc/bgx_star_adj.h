// Stage B of the adjoint (bgx_adjoint.h) along the q coordinates, a lane per
// leg (bgx_star.h): one quad of lanes per (env, q coordinate).
//
// The one-thread kernel runs the step's position terms for the whole robot in
// dual numbers as one dependent chain; a small batch fills a quarter of the
// SIMDs with it.  Here a lane carries one leg and the root, and the sums over
// the legs are the step's quad sums on values and tangents.  Contractions
// with the cotangents are summed a leg per lane; the root's are the same on
// the four lanes and counted once.
#pragma once

#include "bgx_adjoint.h"
#include "bgx_star.h"

namespace bgx {

BGX_D Dual quad_sum(Dual x) { return Dual{quad_sum(x.v), quad_sum(x.d)}; }
BGX_D V3T<Dual> quad_sum(V3T<Dual> v) {
  return V3T<Dual>{quad_sum(v.x), quad_sum(v.y), quad_sum(v.z)};
}

// d/de <cotangents, ingredients(q + e dq_dir, qd)> (adjoint_b_q); every lane
// of the quad returns it
template <class T>
BGX_D float star_adjoint_q(const float* ml, int b, const float* q_in, const float* qd_in,
                           const float* act, RecPtr rec, int dir) {
  using R = AdjRec<T>;
  using S = Dual;
  using V = V3T<S>;
  using SR = Star<T>;
  constexpr int K = SR::K, D0 = 6, NRC = R::NRC;
  const int d_leg = D0 + b * K;
  // the cotangent of M: the root's rows, then each leg's (7 + k entries for
  // its k-th dof: the root's columns, the leg's, the diagonal)
  constexpr int MROOT = 21, MLEG = K * 7 + K * (K - 1) / 2;
  const float* lk0 = ml + T::OFF_LINK;
  const float* lkb = lk0 + LINK_STRIDE * (1 + b * K);
  const float* dfb = ml + T::OFF_DOF + DOF_STRIDE * d_leg;

  S rq[7], q[K];
  float qr[6], ql[K];
#pragma unroll
  for (int k = 0; k < 7; ++k) rq[k] = dual(q_in[k], k == dir ? 1.f : 0.f);
#pragma unroll
  for (int k = 0; k < 6; ++k) qr[k] = qd_in[k];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    q[k] = dual(q_in[7 + b * K + k], 7 + b * K + k == dir ? 1.f : 0.f);
    ql[k] = qd_in[d_leg + k];
  }
  float phi = 0.f, phr = 0.f;  // this leg's part, the root's

  V xp0, xp[K];
  Q4T<S> xr0, xr[K];
  star_frames<T, false, S>(ml, b, rq, q, nullptr, nullptr, xp0, xr0, xp, xr, (V*)nullptr,
                        (V*)nullptr, (V*)nullptr);
  const float m0 = lk0[LK_MASS];
  V rc;
  {
    const S zero = lift<S>(0.f);
    V sm{zero, zero, zero};
    float ms = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const float* lk = lkb + LINK_STRIDE * k;
      sm = sm + (xp[k] + rotate(lift3<S>(ldv3(lk + LK_IPOS)), xr[k])) * lk[LK_MASS];
      ms = ms + lk[LK_MASS];
    }
    sm = (xp0 + rotate(lift3<S>(ldv3(lk0 + LK_IPOS)), xr0)) * m0 + quad_sum(sm);
    rc = sm * rcp(m0 + quad_sum(ms));
  }
  V cc0, cc[K];
  Sym3T<S> ci0, ci[K];
  float km[K];
  star_inertia(lk0, xp0, xr0, rc, cc0, ci0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    star_inertia(lkb + LINK_STRIDE * k, xp[k], xr[k], rc, cc[k], ci[k]);
    km[k] = lkb[LINK_STRIDE * k + LK_MASS];
  }
  V ra[3], rv[3], ca[K], cv[K];
  {
    const Q4T<S> jr = qmul(xr0, lift4<S>(ldq4(lk0 + LK_TROT)));
    const V jp = (xp0 + rotate(lift3<S>(ldv3(lk0 + LK_TPOS)), xr0)) +
                 rotate(lift3<S>(ldv3(lk0 + LK_JPOS)), jr);
    const V off = rc - jp;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      ra[k] = rotate(lift3<S>(unit3(k)), jr);
      rv[k] = cross(ra[k], off);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float* lk = lkb + LINK_STRIDE * k;
    const V pp = k == 0 ? xp0 : xp[k - 1];
    const Q4T<S> pr = k == 0 ? xr0 : xr[k - 1];
    const Q4T<S> jr = qmul(pr, lift4<S>(ldq4(lk + LK_TROT)));
    const V jp = (pp + rotate(lift3<S>(ldv3(lk + LK_TPOS)), pr)) +
                 rotate(lift3<S>(ldv3(lk + LK_JPOS)), jr);
    ca[k] = rotate(lift3<S>(ldv3(dfb + DOF_STRIDE * k + DF_ANG)), jr);
    cv[k] = cross(ca[k], rc - jp);
  }
  // the cdof part of J's cotangent
  auto put3 = [&](int f, V v) { return rec[f] * v.x.d + rec[f + 1] * v.y.d + rec[f + 2] * v.z.d; };
#pragma unroll
  for (int k = 0; k < 3; ++k)
    phr += put3(R::CAB + 3 * (3 + k), ra[k]) + put3(R::CVB + 3 * (3 + k), rv[k]);
#pragma unroll
  for (int k = 0; k < K; ++k)
    phi += put3(R::CAB + 3 * (d_leg + k), ca[k]) + put3(R::CVB + 3 * (d_leg + k), cv[k]);

  const V rlin = lift3<S>(v3(qr[0], qr[1], qr[2]));
  const V va0 = ra[0] * qr[3] + ra[1] * qr[4] + ra[2] * qr[5];
  const V vv0 = rlin + (rv[0] * qr[3] + rv[1] * qr[4] + rv[2] * qr[5]);
  V va[K], vv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    va[k] = (k == 0 ? va0 : va[k - 1]) + ca[k] * ql[k];
    vv[k] = (k == 0 ? vv0 : vv[k - 1]) + cv[k] * ql[k];
  }
  // ---- qf_smooth = passive - bias + tau
  {
    const V acc0 = cross(rlin, va0) - lift3<S>(ldv3(ml + H_GRAVITY));
    V f2a, f2v, f3a, f3v;
    inertia_mul(cc0, ci0, m0, va0, vv0, f2a, f2v);
    cross_force(va0, vv0, f2a, f2v, f3a, f3v);
    const V fa0 = cross(cc0, acc0) + f3a, fv0 = acc0 * m0 + f3v;
    const S zero = lift<S>(0.f);
    V aa{zero, zero, zero}, av = acc0, fa[K], fv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      V oa, ov, f1a, f1v;
      cross_motion(k == 0 ? va0 : va[k - 1], k == 0 ? vv0 : vv[k - 1], ca[k], cv[k], oa, ov);
      aa = aa + oa * ql[k], av = av + ov * ql[k];
      inertia_mul(cc[k], ci[k], km[k], aa, av, f1a, f1v);
      inertia_mul(cc[k], ci[k], km[k], va[k], vv[k], f2a, f2v);
      cross_force(va[k], vv[k], f2a, f2v, f3a, f3v);
      fa[k] = f1a + f3a, fv[k] = f1v + f3v;
    }
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      if (k + 1 < K) fa[k] = fa[k] + fa[k + 1], fv[k] = fv[k] + fv[k + 1];
      const float* df = dfb + DOF_STRIDE * k;
      float t = -q[k].d * df[DF_STIFFNESS] - (dot(cv[k], fv[k]) + dot(ca[k], fa[k])).d;
      if (star_act<T>(D0 + k) >= 0) {
        const int u = star_act_of_leg<T>(b, k);
        const float* ac = ml + T::OFF_ACT + u * ACT_STRIDE;
        const float ctl = clipf(act ? act[u] : 0.f, ac[AC_CTRL_LO], ac[AC_CTRL_HI]);
        const float f = ac[AC_GAIN] * ctl +
                        ac[AC_GEAR] * (q[k].v * ac[AC_BIAS_Q] + ql[k] * ac[AC_BIAS_QD]);
        if (!(f < ac[AC_FORCE_LO]) && !(f > ac[AC_FORCE_HI]))
          t += ac[AC_GEAR] * (q[k].d * ac[AC_BIAS_Q]) * ac[AC_GEAR];
      }
      phi += rec[R::QFB + d_leg + k] * t;
    }
    const V Fa = fa0 + quad_sum(fa[0]), Fv = fv0 + quad_sum(fv[0]);
    phr -= rec[R::QFB] * Fv.x.d + rec[R::QFB + 1] * Fv.y.d + rec[R::QFB + 2] * Fv.z.d;
#pragma unroll
    for (int k = 0; k < 3; ++k) phr -= rec[R::QFB + 3 + k] * (dot(rv[k], Fv) + dot(ra[k], Fa)).d;
  }
  // ---- M, entry by entry
  {
#pragma unroll
    for (int k = K - 1; k > 0; --k) {
      cc[k - 1] = cc[k - 1] + cc[k];
      ci[k - 1] = symadd(ci[k - 1], ci[k]);
      km[k - 1] = km[k - 1] + km[k];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      V fa, fv;
      inertia_mul(cc[k], ci[k], km[k], ca[k], cv[k], fa, fv);
      const int row = R::MB + MROOT + b * MLEG + k * 7 + k * (k - 1) / 2;
      phi += put3(row, fv);
#pragma unroll
      for (int j = 0; j < 3; ++j) phi += rec[row + 3 + j] * (dot(rv[j], fv) + dot(ra[j], fa)).d;
#pragma unroll
      for (int j = 0; j <= k; ++j) phi += rec[row + 6 + j] * (dot(cv[j], fv) + dot(ca[j], fa)).d;
    }
    const V tc = cc0 + quad_sum(cc[0]);
    const Sym3T<S> ti{ci0.xx + quad_sum(ci[0].xx), ci0.yy + quad_sum(ci[0].yy),
                      ci0.zz + quad_sum(ci[0].zz), ci0.xy + quad_sum(ci[0].xy),
                      ci0.xz + quad_sum(ci[0].xz), ci0.yz + quad_sum(ci[0].yz)};
    const float tm = m0 + quad_sum(km[0]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      V fa, fv;
      inertia_mul(tc, ti, tm, ra[i], rv[i], fa, fv);
      const int row = R::MB + (3 + i) * (4 + i) / 2;
      phr += put3(row, fv);
#pragma unroll
      for (int j = 0; j <= i; ++j) phr += rec[row + 3 + j] * (dot(rv[j], fv) + dot(ra[j], fa)).d;
    }
  }
  // ---- contact rows of this lane's active candidates
#pragma unroll
  for (int i = 0; i < SR::S; ++i) {
    const bool leg = i < SR::NCL;
    const int kk = SR::link(i), c0 = SR::cand0(i);
    const bool held = leg || b < SR::NCR;
    const int c = c0 + (leg ? b * SR::CSTEP : (held ? b : 0));
    const int s = held ? tape_int(rec[R::CSLOT + c], -1, R::KS - 1) : -1;
    if (s >= 0) {
      const float* cd = ml + T::OFF_CAND + CAND_STRIDE * c;
      const V xpl = leg ? xp[kk >= 0 ? kk : 0] : xp0;
      const Q4T<S> xrl = leg ? xr[kk >= 0 ? kk : 0] : xr0;
      V ctr = xpl + rotate(lift3<S>(ldv3(cd + CD_GPOS)), xrl);
      V t1 = lift3<S>(ldv3(cd + CD_T1));
      if (T::CAND_KIND[c0] == KIND_CAPSULE) {
        const V axis = quat_zaxis(qmul(xrl, lift4<S>(ldq4(cd + CD_GQUAT))));
        ctr = ctr + axis * (cd[CD_HALFLEN] * cd[CD_SIGN]);
        const V bt = vnormalize(V{axis.x, axis.y, lift<S>(0.f)}, (S*)nullptr);
        t1 = tape_int(rec[R::CFB + c], 0, 1) ? lift3<S>(v3(0.f, 1.f, 0.f)) : bt;
      }
      const float radius = cd[CD_RADIUS], mu = cd[CD_MU], tw = cd[CD_TW];
      const S dist = (ctr.z - cd[CD_PPOS + 2]) - radius;
      const V r = V{ctr.x, ctr.y, ctr.z - (radius + 0.5f * dist)} - rc;
      const float* im = cd + CD_IMP;
      const S imp = impedance(im, dist);
      const S diag = (tw + mu * mu * tw) * (2.f * mu * mu * imp_ratio(imp));
      const S kt = im[IM_K] * imp * dist;
      const float bq = im[IM_B];
      const V ka = leg ? va[kk >= 0 ? kk : 0] : va0, kv = leg ? vv[kk >= 0 ? kk : 0] : vv0;
      const V vq = kv + cross(ka, r);
      const float e0 = vq.z.d, e1 = (mu * (t1.x * vq.x + t1.y * vq.y)).d,
                  e2 = (mu * (t1.x * vq.y - t1.y * vq.x)).d;
      const int r0 = 4 * s;
      phi += rec[R::AB + r0] * -(bq * (e0 + e1) + kt.d);
      phi += rec[R::AB + r0 + 1] * -(bq * (e0 - e1) + kt.d);
      phi += rec[R::AB + r0 + 2] * -(bq * (e0 + e2) + kt.d);
      phi += rec[R::AB + r0 + 3] * -(bq * (e0 - e2) + kt.d);
      phi += ((rec[R::DB + r0] + rec[R::DB + r0 + 1]) +
              (rec[R::DB + r0 + 2] + rec[R::DB + r0 + 3])) * diag.d;
      // mu t1 = (x, y, 0), mu t2 = (-y, x, 0)
      const int g = R::SLB + R::SBW * s;
      const float tx = mu * t1.x.d, ty = mu * t1.y.d;
      phi += rec[g + 3] * tx + rec[g + 4] * ty;
      phi += rec[g + 7] * tx - rec[g + 6] * ty;
      phi += put3(g + 9, r);
    }
  }
  // ---- limit rows
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (!star_lim<T>(D0 + k)) continue;
    const int i = star_lim_of_leg<T>(b, k);
    const float* df = dfb + DOF_STRIDE * k;
    const S pmin = q[k] - df[DF_LO], pmax = df[DF_HI] - q[k];
    const S pos = min_(min_(pmin, pmax), lift<S>(0.f));
    if (pos.v < 0.f) {
      const float* im = df + DF_IMP;
      const S imp = impedance(im, pos);
      phi += rec[R::DB + NRC + i] * (df[DF_INVWEIGHT] * imp_ratio(imp)).d -
             rec[R::AB + NRC + i] * (im[IM_K] * imp * pos).d;
    }
  }
  // ---- q' = f(q, qd') at fixed qd'
#pragma unroll
  for (int k = 0; k < 3; ++k) phr += rec[R::GQ1 + k] * rq[k].d;
  {
    const V ang = lift3<S>(v3(rec[R::QD1 + 3], rec[R::QD1 + 4], rec[R::QD1 + 5]));
    const Q4T<S> r1 = integrate_rot(Q4T<S>{rq[3], rq[4], rq[5], rq[6]}, ang, ml[H_DT]);
    phr += rec[R::GQ1 + 3] * r1.w.d + rec[R::GQ1 + 4] * r1.x.d + rec[R::GQ1 + 5] * r1.y.d +
           rec[R::GQ1 + 6] * r1.z.d;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) phi += rec[R::GQ1 + 7 + b * K + k] * q[k].d;
  return quad_sum(phi) + phr;
}

}  // namespace bgx
