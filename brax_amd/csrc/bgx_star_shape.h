// The shape that the lane-per-leg kernels take (bgx_star.h): a free root link
// with four equal legs, serial chains of hinges.  Compile-time only.
#pragma once

namespace bgx {

constexpr int STAR_LEGS = 4;

// candidate index of the j-th candidate on leg b (-1: none), and of the j-th
// on the root
template <class T>
constexpr int star_leg_cand(int b, int j) {
  const int K = (T::L - 1) / STAR_LEGS;
  for (int c = 0; c < T::NCAND; ++c) {
    const int l = T::CAND_LINK[c];
    if (l >= 1 + b * K && l < 1 + (b + 1) * K && j-- == 0) return c;
  }
  return -1;
}
template <class T>
constexpr int star_root_cand(int j) {
  for (int c = 0; c < T::NCAND; ++c)
    if (T::CAND_LINK[c] == 0 && j-- == 0) return c;
  return -1;
}
// the actuator / limit row of dof d, or -1
template <class T>
constexpr int star_act(int d) {
  for (int u = 0; u < T::NU; ++u)
    if (T::ACT_D[u] == d) return u;
  return -1;
}
template <class T>
constexpr bool star_lim(int d) {
  for (int i = 0; i < T::NLIM; ++i)
    if (T::LIM_D[i] == d) return true;
  return false;
}

// whether topology T has this shape, leg by leg the same structure
template <class T>
constexpr bool star_ok() {
  if (T::PER_ENV || T::PAIRS || !T::PLANE_Z || T::MLANE) return false;
  if (T::L < 1 + STAR_LEGS || (T::L - 1) % STAR_LEGS != 0 || T::LTYPE[0] != 0) return false;
  const int K = (T::L - 1) / STAR_LEGS;
  if (K > 3 || T::PARENT[0] >= 0 || T::QADR[0] != 0 || T::DADR[0] != 0) return false;
  for (int l = 1; l < T::L; ++l) {
    const int k = (l - 1) % K, d = 5 + l;
    if (T::LTYPE[l] != 1 || T::PARENT[l] != (k == 0 ? 0 : l - 1)) return false;
    if (T::DADR[l] != d || T::QADR[l] != d + 1 || !T::DOF_HINGE[d]) return false;
    if ((star_act<T>(d) >= 0) != (star_act<T>(6 + k) >= 0)) return false;
    if (star_lim<T>(d) != star_lim<T>(6 + k)) return false;
  }
  for (int u = 0; u < T::NU; ++u) {
    if (T::ACT_D[u] < 6 || T::ACT_Q[u] != T::ACT_D[u] + 1) return false;
    if (star_act<T>(T::ACT_D[u]) != u) return false;  // one actuator per dof
  }
  for (int i = 0; i < T::NLIM; ++i)
    if (T::LIM_D[i] < 6 || T::LIM_Q[i] != T::LIM_D[i] + 1) return false;
  int per_leg = 0, on_root = 0;
  while (star_leg_cand<T>(0, per_leg) >= 0) ++per_leg;
  while (star_root_cand<T>(on_root) >= 0) ++on_root;
  if (per_leg * STAR_LEGS + on_root != T::NCAND || per_leg > 4 || on_root > STAR_LEGS) return false;
  for (int b = 0; b < STAR_LEGS; ++b) {
    if (star_leg_cand<T>(b, per_leg) >= 0) return false;
    for (int j = 0; j < per_leg; ++j) {
      const int c0 = star_leg_cand<T>(0, j), c = star_leg_cand<T>(b, j);
      if (c < 0 || T::CAND_KIND[c] != T::CAND_KIND[c0]) return false;
      if (T::CAND_LINK[c] - b * K != T::CAND_LINK[c0]) return false;
      // leg b's candidates at one distance from leg 0's
      if (c - c0 != b * (star_leg_cand<T>(1, 0) - star_leg_cand<T>(0, 0))) return false;
    }
  }
  // the root's candidates: one kind, consecutive
  for (int j = 1; j < on_root; ++j) {
    const int c = star_root_cand<T>(j), p = star_root_cand<T>(j - 1);
    if (c < 1 || p != c - 1 || T::CAND_KIND[c] != T::CAND_KIND[c - 1]) return false;
  }
  return true;
}

}  // namespace bgx
