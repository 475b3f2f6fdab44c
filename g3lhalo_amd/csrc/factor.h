// factor.h -- compile-time structure of the Genz-Malik point set, used to
// evaluate each distinct sub-expression of an integrand once per region.
//
// Along every dimension the points of one region take only seven
// coordinates: the centre, c -/+ lambda2 h, c -/+ lambda4 h, c -/+ lambda5 h
// (src/hcubature.cpp:343-414).  A quantity that depends on a subset S of the
// dimensions (u_NFW(k1, m, z) depends on l1, m, z) therefore takes at most
// as many distinct values as there are distinct projections of the points
// onto S -- 33 of the 93 points of a 5-D region for a 3-dimensional S.
// Proj<D, MASK> lists those projection classes: cls[q] is the class of
// point q, rep[c] the first point of class c (its representative).  Every
// point of a class has bit-identical coordinates on S, so a value computed
// at the representative is the value the point itself would compute.
#pragma once
#include <stdint.h>

#include "layout.h"

namespace g3l {

// Coordinate code of point q along dimension d, in the point order of
// rule_point: 0 centre, 1 c - l2 h, 2 c + l2 h, 3 c - l4 h, 4 c + l4 h,
// 5 c - l5 h, 6 c + l5 h.
constexpr int gm_code(int D, int q, int d) {
  if (q == 0) return 0;
  int t = q - 1;
  if (t < 4 * D) {
    int k = t >> 2, s = t & 3;
    return k != d ? 0 : 1 + s;
  }
  t -= 4 * D;
  if (t < 2 * D * (D - 1)) {
    int p = t >> 2, s = t & 3;
    int i = 0, rem = p;
    while (rem >= D - 1 - i) {
      rem -= D - 1 - i;
      ++i;
    }
    int j = i + 1 + rem;
    if (d == i) return (s == 1 || s == 2) ? 4 : 3;
    if (d == j) return s >= 2 ? 4 : 3;
    return 0;
  }
  t -= 2 * D * (D - 1);
  unsigned signs = (unsigned)t ^ ((unsigned)t >> 1);
  return ((signs >> d) & 1u) ? 5 : 6;
}

constexpr unsigned bit(int d) { return 1u << d; }

template <int D, unsigned MASK>
struct Proj {
  static constexpr int NP = rule_points(D);
  int n = 0;
  uint8_t cls[NP] = {};
  uint8_t rep[NP] = {};
};

// Key of point q on the dimensions of MASK: three bits per dimension.
constexpr unsigned gm_key(int D, int q, unsigned mask) {
  unsigned k = 0;
  for (int d = 0; d < D; ++d)
    if ((mask >> d) & 1u) k |= (unsigned)gm_code(D, q, d) << (3 * d);
  return k;
}

template <int D, unsigned MASK>
constexpr Proj<D, MASK> make_proj() {
  Proj<D, MASK> p{};
  unsigned key[Proj<D, MASK>::NP] = {};
  unsigned ckey[Proj<D, MASK>::NP] = {};
  for (int q = 0; q < Proj<D, MASK>::NP; ++q) key[q] = gm_key(D, q, MASK);
  for (int q = 0; q < Proj<D, MASK>::NP; ++q) {
    int found = -1;
    for (int c = 0; c < p.n; ++c)
      if (ckey[c] == key[q]) {
        found = c;
        break;
      }
    if (found < 0) {
      p.rep[p.n] = (uint8_t)q;
      ckey[p.n] = key[q];
      found = p.n++;
    }
    p.cls[q] = (uint8_t)found;
  }
  return p;
}

// Number of classes, and the table itself on the host side.
template <int D, unsigned MASK>
struct ProjTab {
  static constexpr Proj<D, MASK> host = make_proj<D, MASK>();
  static constexpr int n = host.n;
};
// Packed per-class (or per-point) look-ups: one word from constant memory and
// a few bit extracts instead of a byte load, with its address, per index.
template <int N, class W = uint16_t>
struct Packed {
  W w[N] = {};
};

// Coordinate codes of the classes of (A, last dimension), then (B, last), then
// (C, last): A's, B's or C's code in bits 0-2, the last dimension's in bits 4-6.
template <int D, int A, int B, int C>
constexpr Packed<3 * make_proj<D, bit(A) | bit(D - 1)>().n, uint8_t> make_codes() {
  constexpr int n = make_proj<D, bit(A) | bit(D - 1)>().n;
  Packed<3 * n, uint8_t> t{};
  const Proj<D, bit(A) | bit(D - 1)> a = make_proj<D, bit(A) | bit(D - 1)>();
  const Proj<D, bit(B) | bit(D - 1)> b = make_proj<D, bit(B) | bit(D - 1)>();
  const Proj<D, bit(C) | bit(D - 1)> c = make_proj<D, bit(C) | bit(D - 1)>();
  for (int i = 0; i < n; ++i) {
    t.w[i] = (uint8_t)(gm_code(D, a.rep[i], A) | gm_code(D, a.rep[i], D - 1) << 4);
    t.w[n + i] = (uint8_t)(gm_code(D, b.rep[i], B) | gm_code(D, b.rep[i], D - 1) << 4);
    t.w[2 * n + i] = (uint8_t)(gm_code(D, c.rep[i], C) | gm_code(D, c.rep[i], D - 1) << 4);
  }
  return t;
}
// The code of class c of one dimension: the centre, then the axis points'
// codes 1-4, then the last group's (all upper, 6, first).
template <int D, int A>
constexpr bool single_codes() {
  constexpr Proj<D, bit(A)> p = make_proj<D, bit(A)>();
  for (int c = 0; c < p.n; ++c)
    if (gm_code(D, p.rep[c], A) != (c < 5 ? c : 11 - c)) return false;
  return p.n == 7;
}
constexpr __host__ __device__ int single_code(int c) { return c < 5 ? c : 11 - c; }

}  // namespace g3l
