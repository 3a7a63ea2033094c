// Two GSRB iterations of a merged level in one z march (device side): the pair form of
// zmarch.hpp with four half sweeps in flight, red and black of the first iteration and red and
// black of the second, each one plane behind the one before.  The field is read and written once
// where two launches of zmarch.hpp do so twice, which is what bounds those on levels that do not
// fit the caches.
//
// - The owned pairs cover the column FX x FY grown by 4 in x and y.  Half sweep h is right on
//   the column grown by 3 - h; a lane outside computes values that nothing stored depends on.
// - Step k: barrier; plane k+4's old values into LDS buffer (k+4) mod 6; red of plane k+3, black
//   of plane k+2, red of plane k+1, black of plane k, each from its own plane's LDS buffer (x, y
//   neighbours, written in the step before or earlier) and this thread's registers (z neighbours,
//   the half sweep before having just passed the plane above); store plane k.  A half sweep
//   reads one colour of its plane and writes the other, and no two of a step share a plane.  Five
//   buffers would do; six make the march's unrolled period 6 steps.
// - All four cells of a step have the same index in the pair.
// - With old values known to be zero (ZSRC) the first red pass is lambda (0 - rhs) without
//   neighbours, and old values are neither loaded nor put into LDS (only that pass would read
//   them).
#pragma once
#include <type_traits>

#include "zmarch.hpp"

namespace amrmg {
namespace ops {

template <class T, int FX, int FY>
__device__ __forceinline__ T (*zmarch2_lds())[(FX + 8) * (FY + 8)] {
  __shared__ __align__(16) T S[6][(FX + 8) * (FY + 8)];
  return S;
}

template <class T, bool LAP, int FX, int FY, int NT, int DEPTH, bool ZSRC>
__device__ __forceinline__ void zmarch2_body(const FusedArgs& a, int w, T* __restrict__ dst,
                                             const T* __restrict__ src, const T* __restrict__ rhs, T dxinv,
                                             T lambda, T alpha, T beta, T c1, T c2) {
  constexpr int PX = FX / 2 + 4, PY = FY + 8, NP = PX * PY;
  constexpr int LW = 2 * PX, LPL = LW * PY;
  static_assert(FX % 2 == 0 && NP <= NT, "two-iteration tile does not fit the workgroup");
  static_assert(DEPTH >= 1 && DEPTH <= 2, "loads run 1 or 2 steps ahead");
  T(*S)[LPL] = zmarch2_lds<T, FX, FY>();
  using P2 = Pair<T>;

  // threads beyond the tile take the position of thread 0, as in zmarch_body
  const bool act = threadIdx.x < NP;
  const int tid = act ? (int)threadIdx.x : 0;
  const int px = tid % PX, py = tid / PX;
  const int tx = w % a.ntx, ty = (w / a.ntx) % a.nty, ch = w / (a.ntx * a.nty);
  const int x0 = a.lo[0] + tx * FX, y0 = a.lo[1] + ty * FY;
  const int k0 = a.lo[2] + ch * a.kc;
  const int k1 = min(k0 + a.kc, a.hi[2] + 1);
  const int i0 = x0 - 4 + 2 * px, j = y0 - 4 + py;
  const int pmax = a.lo[0] + 2 * ((a.hi[0] - a.lo[0]) / 2);
  const long long xy = a.off + (clampi(i0, a.lo[0], pmax) - a.lo[0] + 1) +
                       (long long)(clampi(j, a.lo[1], a.hi[1]) - a.lo[1] + 1) * a.sy;
  auto zoff = [&](int p) { return (long long)(clampi(p, a.lo[2], a.hi[2]) - a.lo[2] + 1) * a.sz; };
  const int rb = py * LW + 2 * px;

  // in step k every half sweep updates the pair's cell of index s = (i0 + j + k + 1) & 1 = sA ^ P
  const int sA = (i0 + j + k0 + 1) & 1;
  int o_own[2], o_far[2], o_yp[2], o_ym[2];
  bool sodd[2];
#pragma unroll
  for (int P = 0; P < 2; P++) {
    const int s = sA ^ P;
    sodd[P] = s == 1;
    o_own[P] = rb + s;
    o_far[P] = clampi(rb + (s ? 2 : -1), 0, LPL - 1);
    o_yp[P] = min(rb + LW + s, LPL - 1);
    o_ym[P] = max(rb - LW + s, 0);
  }
  const bool tile_face = x0 - 3 <= a.lo[0] || x0 + FX + 2 >= a.hi[0] || y0 - 3 <= a.lo[1] || y0 + FY + 2 >= a.hi[1];
  const bool st_ok = act && px >= 2 && px <= PX - 3 && i0 <= a.hi[0] && j >= y0 && j <= min(y0 + FY - 1, a.hi[1]);
  const bool odd_tile = ((a.hi[0] - a.lo[0]) & 1) == 0 && x0 + FX > a.hi[0];
  const bool st_pair = i0 + 1 <= a.hi[0];

  // 6 plane slots, plane p in slot (p - (k0 - 6)) mod 6
  P2 ph[6], rr[6];
  RB<T> v[6], f[6];
  auto load_phi = [&](P2& d, int p) {
    if (!ZSRC) d = *reinterpret_cast<const P2*>(src + xy + zoff(p));
  };
  auto load_rhs = [&](P2& d, int p) { d = *reinterpret_cast<const P2*>(rhs + xy + zoff(p)); };
  auto to_rb = [&](const P2& d, bool first) { return first ? RB<T>{d.x, d.y} : RB<T>{d.y, d.x}; };
  auto update = [&](auto ZFc, const T* L, int P, int q, T own, T oth, T zp, T zm, T r) {
    constexpr bool ZF = decltype(ZFc)::value;
    const T far = L[o_far[P]], yp = L[o_yp[P]], ym = L[o_ym[P]];
    T sx = oth + far, yp2 = yp, ym2 = ym;
    if (tile_face) {
      const int i = i0 + (sA ^ P);
      const T vxp = sodd[P] ? far : oth, vxm = sodd[P] ? oth : far;
      const T xp = (i == a.hi[0]) ? face_ghost(a.kind[0][1], own, vxm, c1, c2) : vxp;
      const T xm = (i == a.lo[0]) ? face_ghost(a.kind[0][0], own, vxp, c1, c2) : vxm;
      sx = xp + xm;
      yp2 = (j == a.hi[1]) ? face_ghost(a.kind[1][1], own, ym, c1, c2) : yp;
      ym2 = (j == a.lo[1]) ? face_ghost(a.kind[1][0], own, yp, c1, c2) : ym;
    }
    T zp2 = zp, zm2 = zm;
    if (ZF) {
      zp2 = (q == a.hi[2]) ? face_ghost(a.kind[2][1], own, zm, c1, c2) : zp;
      zm2 = (q == a.lo[2]) ? face_ghost(a.kind[2][0], own, zp, c1, c2) : zm;
    }
    return zm_new<T, LAP>(sx, yp2, ym2, zp2, zm2, own, r, dxinv, lambda, alpha, beta);
  };
  const unsigned nz1 = (unsigned)(a.hi[2] - a.lo[2]);
  auto in_rect = [&](int q) { return (unsigned)(q - a.lo[2]) <= nz1; };
  auto inside = [&](int q) { return (unsigned)(q - a.lo[2] - 1) < nz1 - 1u; };

  // step k = k0 - 6 + 6 m + U with its first H half sweeps (the steps before k0 start the pipeline)
  auto step = [&](auto Uc, auto Hc, int k) {
    constexpr int U = decltype(Uc)::value, H = decltype(Hc)::value;
    constexpr int P = U & 1;
    constexpr int S4 = (U + 4) % 6, S3 = (U + 3) % 6, SPH = (U + 4 + DEPTH) % 6, SRH = (U + 3 + DEPTH) % 6;
    lds_barrier();
    if constexpr (ZSRC) {
      v[S4] = RB<T>{T(0.0), T(0.0)};
    } else {
      reinterpret_cast<P2*>(S[S4])[rb / 2] = ph[S4];
      v[S4] = to_rb(ph[S4], sodd[P]);
    }
    f[S3] = to_rb(rr[S3], !sodd[P]);
    load_phi(ph[SPH], k + 4 + DEPTH);
    load_rhs(rr[SRH], k + 3 + DEPTH);
    auto half = [&](auto hc) {
      constexpr int h = decltype(hc)::value;
      constexpr int C = (U + 9 - h) % 6, Cp = (U + 10 - h) % 6, Cm = (U + 8 - h) % 6;
      const int q = k + 3 - h;
      if (h < 3 && !in_rect(q)) return;
      T nv;
      if constexpr (h == 0 && ZSRC) {
        // zm_new with zeros
        nv = LAP ? lambda * f[C].r : lambda * (T(0.0) - f[C].r);
      } else if constexpr (h % 2 == 0) {
        if (inside(q))
          nv = update(std::false_type{}, S[C], P, q, v[C].r, v[C].b, v[Cp].b, v[Cm].b, f[C].r);
        else
          nv = update(std::true_type{}, S[C], P, q, v[C].r, v[C].b, v[Cp].b, v[Cm].b, f[C].r);
      } else {
        if (inside(q))
          nv = update(std::false_type{}, S[C], P, q, v[C].b, v[C].r, v[Cp].r, v[Cm].r, f[C].b);
        else
          nv = update(std::true_type{}, S[C], P, q, v[C].b, v[C].r, v[Cp].r, v[Cm].r, f[C].b);
      }
      if constexpr (h % 2 == 0) v[C].r = nv;
      else v[C].b = nv;
      if constexpr (h < 3) S[C][o_own[P]] = nv;
    };
    half(std::integral_constant<int, 0>{});
    if constexpr (H > 1) half(std::integral_constant<int, 1>{});
    if constexpr (H > 2) half(std::integral_constant<int, 2>{});
    if constexpr (H > 3) {
      half(std::integral_constant<int, 3>{});
      const P2 o = sodd[P] ? P2{v[U % 6].r, v[U % 6].b} : P2{v[U % 6].b, v[U % 6].r};
      T* d = dst + xy + zoff(k);
      if (odd_tile) {
        if (st_ok) {
          if (st_pair) *reinterpret_cast<P2*>(d) = o;
          else *d = o.x;
        }
      } else if (st_ok) {
        *reinterpret_cast<P2*>(d) = o;
      }
    }
  };

  // prologue of step k0-6: old values of planes k0-4 .. k0-3+DEPTH, rhs of planes k0-3 ..
  // k0-4+DEPTH; planes k0-4 and k0-3 into registers (their red cells have index 1 - sA and sA),
  // plane k0-3 into its buffer
#pragma unroll
  for (int d = 2; d < 4 + DEPTH; d++) load_phi(ph[d], k0 - 6 + d);
#pragma unroll
  for (int d = 3; d < 3 + DEPTH; d++) load_rhs(rr[d], k0 - 6 + d);
  if constexpr (ZSRC) {
    v[2] = v[3] = RB<T>{T(0.0), T(0.0)};
  } else {
    v[2] = to_rb(ph[2], sA == 1);
    v[3] = to_rb(ph[3], sA == 0);
    reinterpret_cast<P2*>(S[3])[rb / 2] = ph[3];
  }
#define ZM2_STEP(U, H, k) step(std::integral_constant<int, U>{}, std::integral_constant<int, H>{}, k)
  ZM2_STEP(0, 1, k0 - 6);
  ZM2_STEP(1, 1, k0 - 5);
  ZM2_STEP(2, 2, k0 - 4);
  ZM2_STEP(3, 2, k0 - 3);
  ZM2_STEP(4, 3, k0 - 2);
  ZM2_STEP(5, 3, k0 - 1);
  for (int kb = k0; kb < k1; kb += 6) {
    ZM2_STEP(0, 4, kb);
    if (kb + 1 >= k1) break;
    ZM2_STEP(1, 4, kb + 1);
    if (kb + 2 >= k1) break;
    ZM2_STEP(2, 4, kb + 2);
    if (kb + 3 >= k1) break;
    ZM2_STEP(3, 4, kb + 3);
    if (kb + 4 >= k1) break;
    ZM2_STEP(4, 4, kb + 4);
    if (kb + 5 >= k1) break;
    ZM2_STEP(5, 4, kb + 5);
  }
#undef ZM2_STEP
}

}  // namespace ops
}  // namespace amrmg
