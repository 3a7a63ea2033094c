// One GSRB iteration of a merged level with variable coefficients, marching in z with x pairs
// (device side): the schedule of zmarch_body (zmarch.hpp), red of plane k+1 and black of plane k
// in step k, with the update of vc_fused_new.
//
// What bounds it: the operands, seven values a cell against three with constant coefficients
// (phi read and written, rhs, aCoef, one face value per direction), 56 bytes in FP64.  Each pair's
// operands are loaded once, a step ahead, and serve its red and its black update; the column
// grown by 2 that the workgroup needs is what it reads too much.  The face arrays have rows of nx + 1 or
// nx values without padding, so faces are loaded singly; rhs, aCoef and phi as pairs.
#pragma once
#include <type_traits>

#include "zmarch.hpp"

namespace amrmg {
namespace {

// coefficient operands of a rectangle
template <class T>
struct VCFused {
  const T* a;
  const T* b0;
  const T* b1;
  const T* b2;
  long long foff[3];  // face index of the rectangle's low corner, per direction
  int fsy[3], fsz[3];
};

// rhs, aCoef, x faces and y faces of a pair
template <class T>
struct VCPair {
  ops::Pair<T> r, a;
  T x0, x1, x2, ym0, ym1, yp0, yp1;
};

// the same of one cell, with its lower z face
template <class T>
struct VCOne {
  T r, a, b0m, b0p, b1m, b1p, b2m;
};

template <class T, int FX, int FY, int NT, bool ZSRC>
__device__ __forceinline__ void vc_zmarch_body(const ops::FusedArgs& a, const VCFused<T>& vc, int w,
                                               T* __restrict__ dst, const T* __restrict__ src,
                                               const T* __restrict__ rhs, T dxinv, T scale, T alpha, T beta, T c1,
                                               T c2) {
  using ops::clampi;
  using ops::face_ghost;
  using P2 = ops::Pair<T>;
  using RB = ops::RB<T>;
  constexpr int PX = FX / 2 + 2, PY = FY + 4, NP = PX * PY;
  constexpr int LW = 2 * PX, LPL = LW * PY;
  static_assert(FX % 2 == 0 && NP <= NT, "z-march tile does not fit the workgroup");
  constexpr int DEPTH = 1;  // steps that loads run ahead; 2 takes more registers: 35.0 for 32.8 us a launch
  T(*S)[LPL] = ops::zmarch_lds<T, FX, FY>();

  const bool act = threadIdx.x < NP;
  const int tid = act ? (int)threadIdx.x : 0;
  const int px = tid % PX, py = tid / PX;
  const int tx = w % a.ntx, ty = (w / a.ntx) % a.nty, ch = w / (a.ntx * a.nty);
  const int x0 = a.lo[0] + tx * FX, y0 = a.lo[1] + ty * FY;
  const int k0 = a.lo[2] + ch * a.kc;
  const int k1 = min(k0 + a.kc, a.hi[2] + 1);
  const int i0 = x0 - 2 + 2 * px, j = y0 - 2 + py;
  const int pmax = a.lo[0] + 2 * ((a.hi[0] - a.lo[0]) / 2);
  // every load is from an address clamped into the rectangle's cells or faces; what it returns
  // outside is never used by a stored value
  const int di = clampi(i0, a.lo[0], pmax) - a.lo[0], dj = clampi(j, a.lo[1], a.hi[1]) - a.lo[1];
  const int nx = a.hi[0] - a.lo[0] + 1;
  const int d1 = min(di + 1, nx - 1) - di, d2 = min(di + 2, nx) - di;  // second cell and third x face
  // a lane's place in a plane in bytes: with the plane's address uniform, each access is a scalar
  // base and a 32-bit offset (the launcher takes this march only where a plane has less than 2^31 bytes)
  const unsigned oc = (unsigned)(di + 1 + (dj + 1) * a.sy) * (unsigned)sizeof(T);
  const unsigned of0 = (unsigned)(di + dj * vc.fsy[0]) * (unsigned)sizeof(T), of02 = of0 + d2 * (unsigned)sizeof(T);
  const unsigned of1 = (unsigned)(di + dj * vc.fsy[1]) * (unsigned)sizeof(T), of11 = of1 + d1 * (unsigned)sizeof(T);
  const unsigned of2 = (unsigned)(di + dj * vc.fsy[2]) * (unsigned)sizeof(T), of21 = of2 + d1 * (unsigned)sizeof(T);
  auto at = [](const T* base, unsigned o) { return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o); };
  auto at2 = [](const T* base, unsigned o) {
    return reinterpret_cast<const P2*>(reinterpret_cast<const char*>(base) + o);
  };
  auto zc = [&](int p) { return (long long)(clampi(p, a.lo[2], a.hi[2]) - a.lo[2]); };
  const int rb = py * LW + 2 * px;

  // the red cell of plane k+1 and the black cell of plane k have index s = sA ^ P in the pair
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
  const bool tile_face = x0 - 1 <= a.lo[0] || x0 + FX >= a.hi[0] || y0 - 1 <= a.lo[1] || y0 + FY >= a.hi[1];
  const bool st_ok = act && px >= 1 && px <= PX - 2 && i0 <= a.hi[0] && j >= y0 && j <= min(y0 + FY - 1, a.hi[1]);
  const bool odd_tile = ((a.hi[0] - a.lo[0]) & 1) == 0 && x0 + FX > a.hi[0];
  const bool st_pair = i0 + 1 <= a.hi[0];

  // 6 slots: plane p (and z face plane p, below plane p) in slot (p - (k0 - 2)) mod 6
  P2 ph[6], zf[6];
  VCPair<T> q[6];
  RB v[6];
  VCOne<T> black{};  // operands of the black cell of the step's plane k, kept from the step before
  auto load_phi = [&](P2& d, int p) {
    if (ZSRC) d = P2{T(0.0), T(0.0)};
    else d = *at2(src + a.off + (zc(p) + 1) * a.sz, oc);
  };
  auto load_ops = [&](VCPair<T>& d, int p) {
    const long long z = zc(p);
    d.r = *at2(rhs + a.off + (z + 1) * a.sz, oc);
    d.a = *at2(vc.a + a.off + (z + 1) * a.sz, oc);
    const T* b0 = vc.b0 + vc.foff[0] + z * vc.fsz[0];
    const T* b1 = vc.b1 + vc.foff[1] + z * vc.fsz[1];
    d.x0 = *at(b0, of0);
    d.x1 = *at(b0 + 1, of0);
    d.x2 = *at(b0, of02);
    d.ym0 = *at(b1, of1);
    d.ym1 = *at(b1, of11);
    d.yp0 = *at(b1 + vc.fsy[1], of1);
    d.yp1 = *at(b1 + vc.fsy[1], of11);
  };
  auto load_zf = [&](P2& d, int p) {
    const T* b2 = vc.b2 + vc.foff[2] + (long long)(clampi(p, a.lo[2], a.hi[2] + 1) - a.lo[2]) * vc.fsz[2];
    d.x = *at(b2, of2);
    d.y = *at(b2, of21);
  };
  auto to_rb = [&](const P2& d, bool first) { return first ? RB{d.x, d.y} : RB{d.y, d.x}; };
  auto sel = [&](bool s, T x, T y) { return s ? y : x; };

  auto pick = [&](const VCPair<T>& o, const P2& zlo, bool s) {
    return VCOne<T>{sel(s, o.r.x, o.r.y), sel(s, o.a.x, o.a.y), sel(s, o.x0, o.x1),    sel(s, o.x1, o.x2),
                    sel(s, o.ym0, o.ym1), sel(s, o.yp0, o.yp1), sel(s, zlo.x, zlo.y)};
  };
  auto update = [&](const T* L, int P, int p, const VCOne<T>& o, const P2& zhi, T own, T oth, T vzp, T vzm) {
    const bool s = sodd[P];
    const T far = L[o_far[P]], vyp = L[o_yp[P]], vym = L[o_ym[P]];
    const T vxp = s ? far : oth, vxm = s ? oth : far;
    T xp = vxp, xm = vxm, yp = vyp, ym = vym, zp = vzp, zm = vzm;
    if (tile_face) {
      const int i = i0 + (sA ^ P);
      xp = (i == a.hi[0]) ? face_ghost(a.kind[0][1], own, vxm, c1, c2) : vxp;
      xm = (i == a.lo[0]) ? face_ghost(a.kind[0][0], own, vxp, c1, c2) : vxm;
      yp = (j == a.hi[1]) ? face_ghost(a.kind[1][1], own, vym, c1, c2) : vyp;
      ym = (j == a.lo[1]) ? face_ghost(a.kind[1][0], own, vyp, c1, c2) : vym;
    }
    if (p == a.hi[2]) zp = face_ghost(a.kind[2][1], own, vzm, c1, c2);  // uniform
    if (p == a.lo[2]) zm = face_ghost(a.kind[2][0], own, vzp, c1, c2);
    const T b0m = o.b0m, b0p = o.b0p, b1m = o.b1m, b1p = o.b1p, b2m = o.b2m, b2p = sel(s, zhi.x, zhi.y), ac = o.a;
    // lambda (k_vc_lambda's expression)
    T l = ac * alpha;
    T sumVal = b0p + b0m;
    l = l + scale * beta * sumVal;
    sumVal = b1p + b1m;
    l = l + scale * beta * sumVal;
    sumVal = b2p + b2m;
    l = l + scale * beta * sumVal;
    const T lam = T(1.0) / l;
    // GSRBHELMHOLTZVC (vc_lofphi's expression)
    const T sum = b0p * (xp - own) - b0m * (own - xm) + b1p * (yp - own) - b1m * (own - ym) + b2p * (zp - own) -
                  b2m * (own - zm);
    const T lofphi = alpha * ac * own - beta * sum * dxinv;
    return own - lam * (lofphi - o.r);
  };
  const unsigned nz1 = (unsigned)(a.hi[2] - a.lo[2]);
  auto in_rect = [&](int p) { return (unsigned)(p - a.lo[2]) <= nz1; };

  // step k = k0 - 2 + 6 m + U (FULL: with its black pass, k >= k0)
  auto step = [&](auto Uc, auto FULLc, int k) {
    constexpr int U = decltype(Uc)::value;
    constexpr bool FULL = decltype(FULLc)::value;
    constexpr int Sm1 = (U + 5) % 6, S0 = U % 6, S1 = (U + 1) % 6, S2 = (U + 2) % 6;
    constexpr int SPH = (U + 2 + DEPTH) % 6, SQ = (U + 1 + DEPTH) % 6;
    constexpr int P = U & 1;
    ops::lds_barrier();
    reinterpret_cast<P2*>(S[S2 % 3])[rb / 2] = ph[S2];
    v[S2] = to_rb(ph[S2], sodd[P]);
    load_phi(ph[SPH], k + 2 + DEPTH);
    load_ops(q[SQ], k + 1 + DEPTH);
    load_zf(zf[SPH], k + 2 + DEPTH);
    if (in_rect(k + 1)) {
      T* L = S[S1 % 3];
      const T nv = update(L, P, k + 1, pick(q[S1], zf[S1], sodd[P]), zf[S2], v[S1].r, v[S1].b, v[S2].b, v[S0].b);
      v[S1].r = nv;
      L[o_own[P]] = nv;
    }
    if (FULL) {
      v[S0].b = update(S[S0 % 3], P, k, black, zf[S1], v[S0].b, v[S0].r, v[S1].r, v[Sm1].r);
      const P2 o = sodd[P] ? P2{v[S0].r, v[S0].b} : P2{v[S0].b, v[S0].r};
      T* d = reinterpret_cast<T*>(reinterpret_cast<char*>(dst + a.off + (zc(k) + 1) * a.sz) + oc);
      if (odd_tile) {
        if (st_ok) {
          if (st_pair) *reinterpret_cast<P2*>(d) = o;
          else *d = o.x;
        }
      } else if (st_ok) {
        *reinterpret_cast<P2*>(d) = o;
      }
    }
    black = pick(q[S1], zf[S1], !sodd[P]);
  };

  // prologue of step k0-2: phi of planes k0-2 .. k0-1+DEPTH, operands of planes k0-1 ..
  // k0-2+DEPTH, z faces k0-1 .. k0-1+DEPTH
#pragma unroll
  for (int d = 0; d < DEPTH + 2; d++) load_phi(ph[d], k0 - 2 + d);
#pragma unroll
  for (int d = 1; d <= DEPTH; d++) load_ops(q[d], k0 - 2 + d);
#pragma unroll
  for (int d = 1; d < DEPTH + 2; d++) load_zf(zf[d], k0 - 2 + d);
  v[0] = to_rb(ph[0], sA == 1);
  v[1] = to_rb(ph[1], sA == 0);
  reinterpret_cast<P2*>(S[1])[rb / 2] = ph[1];
#define VCZ_STEP(U, F, k) step(std::integral_constant<int, U>{}, std::integral_constant<bool, F>{}, k)
  VCZ_STEP(0, false, k0 - 2);
  VCZ_STEP(1, false, k0 - 1);
  for (int kb = k0 - 2; kb + 2 < k1; kb += 6) {
    VCZ_STEP(2, true, kb + 2);
    if (kb + 3 >= k1) break;
    VCZ_STEP(3, true, kb + 3);
    if (kb + 4 >= k1) break;
    VCZ_STEP(4, true, kb + 4);
    if (kb + 5 >= k1) break;
    VCZ_STEP(5, true, kb + 5);
    if (kb + 6 >= k1) break;
    VCZ_STEP(0, true, kb + 6);
    if (kb + 7 >= k1) break;
    VCZ_STEP(1, true, kb + 7);
  }
#undef VCZ_STEP
}

}  // namespace
}  // namespace amrmg
