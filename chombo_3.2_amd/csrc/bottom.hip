// One workgroup solves one level's BiCGStab bottom.
//
// What bounds it: the solve is a chain of short dependent passes over at most 32 thousand
// cells (per BiCGStab iteration: eight colour sweeps, two operator applications, four dot
// products and two norms whose terms the reference adds serially), so it is bound by the
// latency of each pass, not by bytes.  Hence the layout:
// - A slot is an x-adjacent pair of cells of one row, one cell of each colour.  Thread t owns
//   slots t, t + NT, ...; every vector is an array of (red, black) pairs, moved 16 bytes a lane
//   without index arithmetic or ghost cells, and an elementwise step needs no barrier.
// - During a relaxation each colour is an array in LDS.  A cell's six neighbours have the other
//   colour: slot q's own other cell and the cells at q +- 1, q +- nxh, q +- plane of that array,
//   so a colour sweep reads one array and writes the other.  Levels whose two colours do not fit
//   LDS keep there only the colour that is read, and the vector itself in memory.  Face ghosts are
//   formed from the cell itself (the reference's fill-then-read).
// - The loop's code is executed once per pass by every wave, so its size counts: at 61 to 115 KB
//   (every sweep inlined where it is used, W = 2 unrolled) an iteration spent most of its time
//   fetching instructions past the 64 KB instruction cache.  So each kind of pass appears once:
//   a BiCGStab iteration is two halves of the same form, and one reduction routine serves all.
// - The terms of a dot product or norm are formed by the owners and put into LDS in each
//   box's Fortran order; one thread per box (dot product) or box column (norm) then adds them
//   in the reference's order (FArrayBox::dotProduct, FArrayBox::sumPow, boxes in layout
//   order), so the results are bitwise the reference's.  Levels with more terms than LDS
//   holds split every box's rows evenly over several stages.
//
// Measured (MI355X, FP64, whole solves; before: the general kernel of batch.hip or, per box, for
// several components, the host-driven BiCGStab): 64^3 3.41 -> 2.60 ms, 120x88x104 (bottom
// 30x22x26) 91.5 -> 30.4 ms, 96^3 + one level with three components 66.3 -> 20.1 ms, a batch of
// 96 problems 93.4 -> 55.9 ms.  Per BiCGStab iteration on 17 thousand cells: 130 us, of which
// colour sweeps 38, operator 13, vector updates 32, terms into LDS 26, serial sums 15.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <type_traits>

#include "bottom.hpp"

namespace amrmg {

// ---------------------------------------------------------------------------
// host tables
// ---------------------------------------------------------------------------
namespace {
// an entry's word: its slot number (16 bits), these, and whether it is empty
enum : unsigned {
  kSlotMask = 0xffff,
  kGeoRedFirst = 1 << 16,   // the red cell is the slot's first cell (i = 2a)
  kGeoPair = 1 << 17,       // the second cell exists (2a + 1 < nx)
  kGeoXlo = 1 << 18,        // a == 0
  kGeoXhi = 1 << 19,        // a == nxh - 1
  kGeoYlo = 1 << 20, kGeoYhi = 1 << 21, kGeoZlo = 1 << 22, kGeoZhi = 1 << 23,
  kEmpty = 1u << 31
};
// doubles from one box's terms to the next's: 16-byte aligned, and 2 modulo 4 so that the boxes'
// serial sums start in different banks
long long stage_pitch(long long n) { return (n + 1) / 4 * 4 + 2; }
constexpr int kLdsBytes = 160 * 1024 - 512;  // LDS a workgroup may hold on gfx950, less a margin
}  // namespace

bool BottomTables::build(const std::vector<Box>& boxes, const Box& rect, const int kind[3][2], int nc, long long cs,
                         const std::function<long long(int, int, int, int)>& offset) {
  plan = BottomPlan{};
  word.clear(); cell.clear(); term.clear(); col.clear(); box.clear();
  const int n[3] = {rect.len(0), rect.len(1), rect.len(2)};
  for (int d = 0; d < 3; d++) {
    if (n[d] < 1) return false;
    if (kind[d][0] == 3 && (n[d] & 1)) return false;  // the two ends would have one colour
    for (int s = 0; s < 2; s++)
      if (kind[d][s] != 0 && kind[d][s] != 1 && kind[d][s] != 3) return false;
  }
  const int nxh = (n[0] + 1) / 2;
  const long long per = (long long)nxh * n[1] * n[2], slots = per * nc;
  if (slots > kBottomMaxSlots) return false;
  long long cells = 0, ncol = 0;
  for (const Box& b : boxes) {
    cells += b.npts();
    ncol += b.len(0);
  }
  if (cells != rect.npts()) return false;  // the boxes do not tile the level
  const int nbox = (int)boxes.size();
  // sums region: per box two dot products and a norm, per box column one, and 16 results
  const long long sums = ncol + 3LL * nbox + 16;
  const long long room = kLdsBytes / 8 - sums;
  if (room < slots) return false;
  plan.two = 2 * slots <= room ? 1 : 0;
  // reduction stages: every box's rows split evenly, two dot products side by side
  int nst = 1;
  for (;; nst++) {
    if (nst > 64) return false;
    long long off = 0;
    for (const Box& b : boxes) {
      const int rows = nc * b.len(1) * b.len(2);
      off += stage_pitch((long long)b.len(0) * ((rows + nst - 1) / nst));
    }
    if (2 * off <= room) {
      plan.stage = (int)off;
      break;
    }
  }
  plan.nst = nst;
  plan.mainDoubles = (int)std::max<long long>((plan.two ? 2 : 1) * slots, 2LL * plan.stage);
  plan.sumDoubles = (int)sums;
  plan.nslot = (int)slots;
  plan.ncell = (int)cells;
  plan.nxh = nxh;
  plan.plane = nxh * n[1];
  plan.wrap[0] = nxh - 1;
  plan.wrap[1] = (n[1] - 1) * nxh;
  plan.wrap[2] = (n[2] - 1) * plan.plane;
  plan.nbox = nbox;
  plan.ncol = (int)ncol;
  const int lo3 = rect.lo[0] + rect.lo[1] + rect.lo[2];
  std::vector<unsigned> inner, outer;
  for (int c = 0; c < nc; c++)
    for (int k = 0; k < n[2]; k++)
      for (int j = 0; j < n[1]; j++)
        for (int a = 0; a < nxh; a++) {
          unsigned g = 0;
          if (((2 * a + j + k + lo3) & 1) == 0) g |= kGeoRedFirst;
          if (2 * a + 1 < n[0]) g |= kGeoPair;
          if (a == 0) g |= kGeoXlo;
          if (a == nxh - 1) g |= kGeoXhi;
          if (j == 0) g |= kGeoYlo;
          if (j == n[1] - 1) g |= kGeoYhi;
          if (k == 0) g |= kGeoZlo;
          if (k == n[2] - 1) g |= kGeoZhi;
          const bool in = !(g & (kGeoXlo | kGeoXhi | kGeoYlo | kGeoYhi | kGeoZlo | kGeoZhi));
          (in ? inner : outer).push_back(g | (unsigned)(c * per + (long long)(k * n[1] + j) * nxh + a));
        }
  // a short list of inner slots does not pay for its own pass
  if (inner.size() < 256) {
    outer.insert(outer.end(), inner.begin(), inner.end());
    std::sort(outer.begin(), outer.end(), [](unsigned a, unsigned b) { return (a & kSlotMask) < (b & kSlotMask); });
    inner.clear();
  }
  while (inner.size() % 64) inner.push_back(inner.back() | kEmpty);
  plan.nint = (int)inner.size();
  word = inner;
  word.insert(word.end(), outer.begin(), outer.end());
  plan.nlist = (int)word.size();
  cell.assign(word.size(), int2{-1, -1});
  term.assign(word.size(), int2{-1, -1});
  std::vector<int> entry((size_t)slots, -1);
  for (size_t t = 0; t < word.size(); t++)
    if (!(word[t] & kEmpty)) entry[word[t] & kSlotMask] = (int)t;
  long long off = 0, seen = 0;
  for (int b = 0; b < nbox; b++) {
    const Box& bx = boxes[b];
    BottomBox t;
    t.off = (int)off;
    t.nx = bx.len(0);
    t.rows = nc * bx.len(1) * bx.len(2);
    t.rp = (t.rows + nst - 1) / nst;
    t.col0 = (int)col.size();
    off += stage_pitch((long long)t.nx * t.rp);
    box.push_back(t);
    for (int i = 0; i < t.nx; i++) col.push_back(int2{b, i});
    int row = 0;
    for (int c = 0; c < nc; c++)
      for (int k = bx.lo[2]; k <= bx.hi[2]; k++)
        for (int j = bx.lo[1]; j <= bx.hi[1]; j++, row++)
          for (int i = bx.lo[0]; i <= bx.hi[0]; i++) {
            const int i0 = i - rect.lo[0], j0 = j - rect.lo[1], k0 = k - rect.lo[2];
            if (i0 < 0 || i0 >= n[0] || j0 < 0 || j0 >= n[1] || k0 < 0 || k0 >= n[2]) return false;
            const size_t q = (size_t)entry[(size_t)(c * per + (long long)(k0 * n[1] + j0) * nxh + (i0 >> 1))];
            const long long o = offset(b, i, j, k) + c * cs;
            if (o < 0 || o > INT32_MAX) return false;
            const int pos = (row / t.rp) * plan.stage + t.off + (row % t.rp) * t.nx + (i - bx.lo[0]);
            const bool red = ((i + j + k) & 1) == 0;
            int& ce = red ? cell[q].x : cell[q].y;
            if (ce >= 0) return false;  // two boxes hold the cell
            ce = (int)o;
            (red ? term[q].x : term[q].y) = pos;
            seen++;
          }
  }
  return seen == cells * nc;
}
void* BottomTables::upload(Context* ctx, const std::vector<BottomTables*>& all, long long* bytes) {
  if (ctx->dry) return nullptr;
  auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
  std::vector<char> host;
  std::vector<size_t> at;
  auto put = [&](const void* src, size_t n) {
    at.push_back(host.size());
    host.resize(host.size() + pad(n));
    std::memcpy(host.data() + at.back(), src, n);
  };
  for (BottomTables* t : all) {
    if (t->plan.nslot == 0) continue;
    put(t->word.data(), sizeof(unsigned) * t->word.size());
    put(t->cell.data(), sizeof(int2) * t->cell.size());
    put(t->term.data(), sizeof(int2) * t->term.size());
    put(t->box.data(), sizeof(BottomBox) * t->box.size());
    put(t->col.data(), sizeof(int2) * t->col.size());
  }
  if (host.empty()) return nullptr;
  void* mem = nullptr;
  dev_alloc(ctx, &mem, host.size(), "hipMalloc bottom tables");
  dev_h2d(ctx, mem, host.data(), host.size(), "copy bottom tables");
  *bytes += (long long)host.size();
  size_t q = 0;
  for (BottomTables* t : all) {
    if (t->plan.nslot == 0) continue;
    char* d = (char*)mem;
    t->plan.word = (const unsigned*)(d + at[q]);
    t->plan.cell = (const int2*)(d + at[q + 1]);
    t->plan.term = (const int2*)(d + at[q + 2]);
    t->plan.box = (const BottomBox*)(d + at[q + 3]);
    t->plan.col = (const int2*)(d + at[q + 4]);
    q += 5;
  }
  return mem;
}

// ---------------------------------------------------------------------------
// device
// ---------------------------------------------------------------------------
namespace {

template <class V>
struct alignas(2 * sizeof(V)) RBPair {
  V r, b;
};

struct BottomLev {
  double dxinv, lambda, alpha, beta;
  int lap;
  int kxl, kxh, kyl, kyh, kzl, kzh;  // face rules
  int nxh, plane, wx, wy, wz;
};

// homogeneous ghost of a face cell: k_fill_ghosts' Dirichlet 2 * 0 - near, Neumann near
template <class V>
__device__ __forceinline__ V face_value(int kind, V own) {
  return kind == 1 ? V(2) * V(0.0) - own : own;
}
// the sum of the six neighbours of slot q's cell of one colour, in the reference's order
// (xp + xm first, whose sum commutes): own value, the slot's other cell, Lo = the other
// colour's values in LDS
template <class V>
__device__ __forceinline__ V six_sum(const BottomLev& L, unsigned g, int q, bool first, V own, V oth, const V* Lo) {
  const bool xout = (g & (first ? kGeoXlo : kGeoXhi)) != 0;
  const bool ylo = (g & kGeoYlo) != 0, yhi = (g & kGeoYhi) != 0, zlo = (g & kGeoZlo) != 0, zhi = (g & kGeoZhi) != 0;
  const bool px = L.kxl == 3, py = L.kyl == 3, pz = L.kzl == 3;
  // addresses stay inside the level's slots: a neighbour outside it is its periodic image, or
  // (replaced below) the slot itself
  const int ox = xout ? (px ? (first ? L.wx : -L.wx) : 0) : (first ? -1 : 1);
  const int oyp = yhi ? (py ? -L.wy : 0) : L.nxh, oym = ylo ? (py ? L.wy : 0) : -L.nxh;
  const int ozp = zhi ? (pz ? -L.wz : 0) : L.plane, ozm = zlo ? (pz ? L.wz : 0) : -L.plane;
  V far = Lo[q + ox], yp = Lo[q + oyp], ym = Lo[q + oym], zp = Lo[q + ozp], zm = Lo[q + ozm];
  if (xout && !px) far = face_value(first ? L.kxl : L.kxh, own);
  const V in = (first && !(g & kGeoPair)) ? face_value(L.kxh, own) : oth;
  if (yhi && !py) yp = face_value(L.kyh, own);
  if (ylo && !py) ym = face_value(L.kyl, own);
  if (zhi && !pz) zp = face_value(L.kzh, own);
  if (zlo && !pz) zm = face_value(L.kzl, own);
  return in + far + yp + ym + zp + zm;
}
// the same for a slot whose neighbours are all inside the level
template <class V>
__device__ __forceinline__ V six_sum_in(const BottomLev& L, int q, bool first, V oth, const V* Lo) {
  const V far = Lo[first ? q - 1 : q + 1], yp = Lo[q + L.nxh], ym = Lo[q - L.nxh], zp = Lo[q + L.plane],
          zm = Lo[q - L.plane];
  return oth + far + yp + ym + zp + zm;
}
// GSRBLAPLACIAN / GSRBHELMHOLTZ
template <class V>
__device__ __forceinline__ V gsrb_new(const BottomLev& L, V s6, V own, V r) {
  const V dxinv = V(L.dxinv), lambda = V(L.lambda);
  if (L.lap) {
    const V lphi = s6 * dxinv;
    return lambda * (r - lphi);
  }
  const V lphi = (s6 - V(6.0) * own) * dxinv;
  const V helmop = V(L.alpha) * own + V(L.beta) * lphi;
  return own + lambda * (helmop - r);
}

template <class T, int NT, bool TREE>
__global__ void __launch_bounds__(NT) k_bottom(BottomLaunch<T> A) {
  const int prob = blockIdx.x, tid = threadIdx.x;
  if (A.active && !A.active[prob]) return;
  const BottomPlan P = A.plans[prob];
  const int S = P.nslot;
  if (S == 0) return;  // another kernel's problem
  extern __shared__ double lds[];
  double* sums = lds + P.mainDoubles;
  double* boxsum = sums + P.ncol;    // two dot products and a norm per box
  double* result = boxsum + 3 * P.nbox;  // 16 entries, used in turn
  int turn = 0;

  BottomLev L;
  const BatchCoef& cf = A.coef ? A.coef[prob] : A.cf;
  L.dxinv = cf.dxinv;
  L.lambda = cf.lambda;
  L.alpha = cf.alpha;
  L.beta = cf.beta;
  L.lap = cf.lap;
  L.kxl = cf.kind[0][0];
  L.kxh = cf.kind[0][1];
  L.kyl = cf.kind[1][0];
  L.kyh = cf.kind[1][1];
  L.kzl = cf.kind[2][0];
  L.kzh = cf.kind[2][1];
  // preCond's factor (AMRPoissonOp.cpp:304-329)
  const double mult = 1.0 / (cf.alpha - 2.0 * 3 * cf.beta / (cf.dx * cf.dx));
  L.nxh = P.nxh;
  L.plane = P.plane;
  L.wx = P.wrap[0];
  L.wy = P.wrap[1];
  L.wz = P.wrap[2];
  T* corr = (A.corr ? A.corr[prob] : A.corr1) + P.base;
  const T* res = (A.res ? A.res[prob] : A.res1) + P.base;
  using D2 = RBPair<double>;
  D2* vec = (D2*)A.vecs + P.vec;
  const int N = P.nlist;  // vectors list the entries of the plan
  D2 *x = vec, *b = vec + N, *r = vec + 2 * N, *r_tilde = vec + 3 * N, *e = vec + 4 * N, *pp = vec + 5 * N,
     *tilde = vec + 6 * N, *t = vec + 7 * N, *v = vec + 8 * N;
  const bool two = P.two != 0;

  // Entry i belongs to thread i mod NT in every pass, so passes that touch only an entry's own
  // values need no barrier.  each: one entry at a time.
  auto each = [&](auto f) {
    for (int i = tid; i < N; i += NT) f(i);
  };
  // M entries at a time of [i0, i1): all their loads ld(i), then st(i, loaded)
  auto batch = [&](auto Mc, int i1, int i0, auto ld, auto st) {
    constexpr int M = decltype(Mc)::value;
    for (; i0 < i1; i0 += M * NT) {
      decltype(ld(0)) w[M];
#pragma unroll
      for (int u = 0; u < M; u++) w[u] = ld(min(i0 + u * NT, i1 - 1));
#pragma unroll
      for (int u = 0; u < M; u++)
        if (i0 + u * NT < i1) st(i0 + u * NT, w[u]);
    }
  };
  using M2 = std::integral_constant<int, NT <= 256 ? 1 : 2>;
  using M4 = std::integral_constant<int, NT <= 256 ? 1 : 4>;
  // the entries inside the level and the others apart (nint is a multiple of 64: a wave's
  // entries are of one kind)
  auto kinds = [&](auto ld, auto st) {
    batch(M2{}, P.nint, tid, [&](int i) { return ld(std::true_type{}, i); }, st);
    const int i = P.nint > tid ? tid + (P.nint - tid + NT - 1) / NT * NT : tid;
    batch(std::integral_constant<int, 1>{}, N, i, [&](int i) { return ld(std::false_type{}, i); }, st);
  };
  // A relaxed vector: its two colours in LDS (V values, by slot) when both fit, else the colour
  // to be read in LDS and the pairs themselves in memory at m (by entry)
  auto colours = [&](auto V0, int c) {
    using V = decltype(V0);
    return (V*)lds + ((two && c) ? S : 0);
  };
  // colour c of the pairs in m into LDS (not `two`)
  auto publish = [&](int c, auto* m) {
    using V = decltype(m->r);
    __syncthreads();  // the other colour's readers are done
    V* B = colours(V(0), 0);
    struct In {
      V v;
      unsigned g;
    };
    batch(M4{}, N, tid, [&](int i) { return In{c ? m[i].b : m[i].r, P.word[i]}; },
          [&](int, const In& w) {
            if (!(w.g & kEmpty)) B[w.g & kSlotMask] = w.v;
          });
    __syncthreads();
  };
  // one colour of a GSRB iteration; a barrier follows before that colour is read
  auto colour = [&](int c, auto* m, const auto* rhs) {
    using V = std::remove_const_t<decltype(rhs->r)>;
    if (!two) publish(1 - c, m);
    const V* Lo = colours(V(0), 1 - c);
    V* Lc = colours(V(0), c);
    struct In {
      V own, s6, f;
      unsigned g;
    };
    kinds(
        [&](auto inner, int i) {
          In w;
          w.g = P.word[i];
          const RBPair<V> f = rhs[i];
          const int q = w.g & kSlotMask;
          const bool first = ((w.g & kGeoRedFirst) != 0) == (c == 0);
          V oth;
          if (two) {
            w.own = Lc[q];
            oth = Lo[q];
          } else {
            const RBPair<V> p = m[i];
            w.own = c ? p.b : p.r;
            oth = c ? p.r : p.b;
          }
          w.f = c ? f.b : f.r;
          if constexpr (decltype(inner)::value) {
            w.s6 = six_sum_in<V>(L, q, first, oth, Lo);
          } else {
            w.s6 = six_sum<V>(L, w.g, q, first, w.own, oth, Lo);
            if (!first && !(w.g & kGeoPair)) w.g |= kEmpty;  // the last slot of a row may have one cell
          }
          return w;
        },
        [&](int i, const In& w) {
          if (w.g & kEmpty) return;
          const V nv = gsrb_new<V>(L, w.s6, w.own, w.f);
          if (two) Lc[w.g & kSlotMask] = nv;
          else if (c) m[i].b = nv;
          else m[i].r = nv;
        });
    if (two) __syncthreads();
  };
  // the pairs of a vector to relax: into LDS (`two`; the barrier makes them visible) or memory
  auto put_pair = [&](int i, unsigned g, auto* m, auto w) {
    using V = decltype(w.r);
    if (two) {
      if (g & kEmpty) return;
      colours(V(0), 0)[g & kSlotMask] = w.r;
      colours(V(0), 1)[g & kSlotMask] = w.b;
    } else {
      m[i] = w;
    }
  };
  auto get_pair = [&](int i, unsigned g, auto* m) {
    using P2 = std::remove_const_t<std::remove_reference_t<decltype(*m)>>;
    using V = decltype(m->r);
    if (two) return P2{colours(V(0), 0)[g & kSlotMask], colours(V(0), 1)[g & kSlotMask]};
    return *(P2*)(m + i);
  };

  // ---- bottom of MultiGrid::cycle: the correction is zero on entry, relax in T ----
  {
    using T2 = RBPair<T>;
    T2 *em = (T2*)tilde, *fm = (T2*)t;  // FP32 levels use the first half of each vector
    each([&](int i) {
      const int2 c = P.cell[i];
      fm[i] = T2{c.x >= 0 ? res[c.x] : T(0), c.y >= 0 ? res[c.y] : T(0)};
      T2 w{T(0), T(0)};
      if (!A.par.relaxFirst) w = T2{c.x >= 0 ? corr[c.x] : T(0), c.y >= 0 ? corr[c.y] : T(0)};
      put_pair(i, P.word[i], em, w);
    });
    __syncthreads();
    if (A.par.relaxFirst) {
#pragma unroll 1
      for (int it = 0; it < 2 * A.par.nbottom; it++) colour(it & 1, em, (const T2*)fm);
      if (P.ncell == 1) {
        each([&](int i) {
          const int2 c = P.cell[i];
          const T2 w = get_pair(i, P.word[i], em);
          if (c.x >= 0) corr[c.x] = w.r;
          if (c.y >= 0) corr[c.y] = w.b;
        });
        return;
      }
    }
    // PromotedBottomSolver: widen the correction and the residual
    each([&](int i) {
      const T2 w = get_pair(i, P.word[i], em), f = fm[i];
      x[i] = D2{(double)w.r, (double)w.b};
      b[i] = D2{(double)f.r, (double)f.b};
    });
  }

  // One pass of the operator.  First (sweeps) preCond (AMRPoissonOp.cpp:304-329): tilde = src *
  // scale, then `sweeps` colours of GSRB with right-hand side src; or (no sweeps) tilde = src *
  // 1.0.  Then out = applyOp(tilde), or with rhs the residual of tilde, lap as OPERATORLAP forms it.
  D2* hold = x + kBottomVectors * (size_t)N;  // a tenth vector, for levels that are not `two`
  auto level_pass = [&](D2* out, const D2* src, double scale, int sweeps, const D2* rhs) {
    __syncthreads();  // LDS is free (a reduction may still read its stage)
    struct Src {
      D2 w;
      unsigned g;
    };
    batch(M4{}, N, tid, [&](int i) { return Src{src[i], P.word[i]}; },
          [&](int i, const Src& s) { put_pair(i, s.g, tilde, D2{s.w.r * scale, s.w.b * scale}); });
    __syncthreads();
#pragma unroll 1
    for (int it = 0; it < sweeps; it++) colour(it & 1, tilde, src);
    auto emit = [&](int i, D2 p, double lr, double lb) {
      const D2 l{(lr - 6.0 * p.r) * L.dxinv, (lb - 6.0 * p.b) * L.dxinv};
      if (rhs) {
        const D2 f = rhs[i];
        out[i] = D2{-(L.alpha * p.r) - L.beta * l.r + f.r, -(L.alpha * p.b) - L.beta * l.b + f.b};
      } else {
        out[i] = D2{L.alpha * p.r + L.beta * l.r, L.alpha * p.b + L.beta * l.b};
      }
    };
    if (two) {
      const double *Lr = colours(0.0, 0), *Lb = colours(0.0, 1);
      struct In {
        D2 p;
        double sr, sb;
      };
      kinds(
          [&](auto inner, int i) {
            const unsigned g = P.word[i];
            const int q = g & kSlotMask;
            const bool rf = (g & kGeoRedFirst) != 0;
            In w;
            w.p = D2{Lr[q], Lb[q]};
            if constexpr (decltype(inner)::value) {
              w.sr = six_sum_in<double>(L, q, rf, w.p.b, Lb);
              w.sb = six_sum_in<double>(L, q, !rf, w.p.r, Lr);
            } else {
              w.sr = six_sum<double>(L, g, q, rf, w.p.r, w.p.b, Lb);
              w.sb = six_sum<double>(L, g, q, !rf, w.p.b, w.p.r, Lr);
            }
            return w;
          },
          [&](int i, const In& w) {
            tilde[i] = w.p;
            emit(i, w.p, w.sr, w.sb);
          });
      return;
    }
    // one colour at a time: the red cells' sums wait in the tenth vector
#pragma unroll 1
    for (int c = 0; c < 2; c++) {
      publish(1 - c, tilde);
      const double* Lo = colours(0.0, 0);
      struct In {
        D2 p;
        double s6, sr;
      };
      kinds(
          [&](auto inner, int i) {
            const unsigned g = P.word[i];
            In w;
            w.p = tilde[i];
            w.sr = c ? hold[i].r : 0.0;
            const int q = g & kSlotMask;
            const bool first = ((g & kGeoRedFirst) != 0) == (c == 0);
            const double own = c ? w.p.b : w.p.r, oth = c ? w.p.r : w.p.b;
            if constexpr (decltype(inner)::value) w.s6 = six_sum_in<double>(L, q, first, oth, Lo);
            else w.s6 = six_sum<double>(L, g, q, first, own, oth, Lo);
            return w;
          },
          [&](int i, const In& w) {
            if (c == 0) hold[i].r = w.s6;
            else emit(i, w.p, w.sr, w.s6);
          });
    }
  };

  // ---- reductions ----
  // A serial sum of n terms st[0], st[1], ... in order onto acc: one chain of dependent adds
  // (2.5 ns each on registers) fed by 16-byte reads, the next four of them in flight while
  // these are added (4.2 ns per term; 6.6 with 8-byte reads, 7.4 without the overlap, which the
  // scheduling barriers keep).  st is 16-byte aligned.
  auto serial = [&](const double* st, int n, double acc) {
    constexpr int K = 4;
    using W2 = RBPair<double>;
    const W2* p = (const W2*)st;
    const int h = n / 2;
    W2 pa[K], pb[K];
    auto get = [&](W2(&w)[K], int at) {
#pragma unroll
      for (int u = 0; u < K; u++) w[u] = p[at + u];
    };
    auto add = [&](const W2(&w)[K]) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < K; u++) {
        acc += w[u].r;
        acc += w[u].b;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    int m = 0;
    if (K <= h) {
      get(pa, 0);
      for (; m + 3 * K <= h; m += 2 * K) {
        get(pb, m + K);
        add(pa);
        get(pa, m + 2 * K);
        add(pb);
      }
      add(pa);
      m += K;
    }
    for (m = 2 * m; m < n; m++) acc += st[m];
    return acc;
  };
  // the terms st[0], st[stride], ... of a box column's rows in this stage: as many as LDS holds, serially
  // in one thread (a box of 2 x 90 x 90 cells has 8100 rows in one stage, and two threads add them)
  auto column_sum = [&](const double* st, int n, int stride, double acc, bool assign) {
    constexpr int K = 4;
    if (assign && n > 0) {
      acc = *st;
      st += stride;
      n--;
    }
    for (; n >= K; n -= K, st += K * stride) {
      double w[K];
#pragma unroll
      for (int u = 0; u < K; u++) w[u] = st[u * stride];
#pragma unroll
      for (int u = 0; u < K; u++) acc += w[u];
    }
    for (; n > 0; n--, st += stride) acc += *st;
    return acc;
  };
  // the terms of one pass into LDS: w * u of stage s (dot), u * u of stage s2 (square; in the
  // second half of the region), and w * u of stage s2 there instead (dot2)
  auto fill = [&](const D2* u, const D2* w, bool dot, bool square, bool dot2, int s, int s2) {
    const int p0 = s * P.stage, p2 = s2 * P.stage;
    double* at2 = lds + P.stage;
    struct In {
      D2 u, w;
      int2 c;
    };
    batch(M2{}, N, tid, [&](int i) { return In{u[i], w[i], P.term[i]}; },
          [&](int, const In& x) {
            auto cell = [&](int c, double a, double b) {
              if (c < 0) return;
              const unsigned q = (unsigned)(c - p0), q2 = (unsigned)(c - p2);
              const double ab = b * a;
              if (dot && q < (unsigned)P.stage) lds[q] = ab;
              if ((square || dot2) && q2 < (unsigned)P.stage) at2[q2] = square ? a * a : ab;
            };
            cell(x.c.x, x.u.r, x.w.r);
            cell(x.c.y, x.u.b, x.w.b);
          });
  };
  // Tree order: each thread adds its entries' terms (red, then black), the 64 threads of a wave are
  // added pairwise, and the 16 waves' sums in order; the result depends only on the level
  auto tree_sum = [&](const D2* a1, const D2* b1) {
    double acc = 0.0;
    each([&](int i) {
      const D2 u = a1[i], w = b1[i];
      const int2 c = P.cell[i];
      if (c.x >= 0) acc += u.r * w.r;
      if (c.y >= 0) acc += u.b * w.b;
    });
    for (int o = 32; o > 0; o >>= 1) acc = acc + __shfl_down(acc, o, 64);
    __syncthreads();
    if ((tid & 63) == 0) lds[tid >> 6] = acc;
    __syncthreads();
    double total = lds[0];
    for (int w = 1; w < NT / 64; w++) total = total + lds[w];
    return total;
  };
  // red[0] = the dot product (w, u) (dot), red[1] = the dot product (u, u) (square) or the
  // square of norm(u, 2) (square and norms).  A dot product: per box a serial sum in Fortran
  // order from 0.0 (FArrayBox::dotProduct, components outermost), the boxes added in layout
  // order from 0.0.  The norm: FArrayBox::sumPow(2) per box (column sums over rows, the first
  // square assigned, then the columns in i order), the boxes added in order from 0.0.
  // Two reductions share each stage's pass; a dot product alone takes two stages a pass.
  double red[2];
  auto reduce = [&](const D2* u, const D2* w, bool dot, bool square, bool norms) {
    if constexpr (TREE) {
#pragma unroll 1
      for (int m = 0; m < 2; m++) {
        const double t2 = (m ? square : dot) ? tree_sum(u, m ? u : w) : 0.0;
        if (m) red[1] = t2;
        else red[0] = t2;
      }
      return;
    }
    const int step = square ? 1 : 2;
    const int nd = dot + (square && !norms);  // serial sums per box
    for (int s = 0; s < P.nst; s += step) {
      const int s2 = square ? s : s + 1;
      __syncthreads();
      fill(u, w, dot, square, !square, s, s2);
      __syncthreads();
      for (int c = tid; c < nd * P.nbox; c += NT) {
        const int m = c >= P.nbox ? 1 : 0;
        const BottomBox bx = P.box[c - m * P.nbox];
        auto rows = [&](int s) { return max(min(bx.rp, bx.rows - s * bx.rp), 0); };
        double acc = s ? boxsum[c] : 0.0;
        for (int h = 0; h < step; h++)
          acc = serial(lds + (m + h) * P.stage + bx.off, s + h < P.nst ? rows(s + h) * bx.nx : 0, acc);
        boxsum[c] = acc;
      }
      // (the last threads, so that these run beside the serial sums of the first)
      if (norms)
        for (int c = NT - 1 - tid; c < P.ncol; c += NT) {
          const int2 bc = P.col[c];
          const BottomBox bx = P.box[bc.x];
          const int rows = max(min(bx.rp, bx.rows - s * bx.rp), 0);
          sums[c] = column_sum(lds + P.stage + bx.off + bc.y, rows, bx.nx, s ? sums[c] : 0.0, s == 0);
        }
    }
    __syncthreads();
    if (norms) {
      for (int q = tid; q < P.nbox; q += NT) {
        const BottomBox bx = P.box[q];
        double sum = sums[bx.col0];
        for (int i = 1; i < bx.nx; i++) sum += sums[bx.col0 + i];
        boxsum[2 * P.nbox + q] = sum;
      }
      __syncthreads();
    }
    if (tid < 2) {
      const double* p = boxsum + (tid == 0 ? 0 : (norms ? 2 : 1)) * P.nbox;
      double val = 0.0;
      if (tid == 0 ? dot : square)
        for (int q = 0; q < P.nbox; q++) val += p[q];
      result[(turn + tid) & 15] = val;
    }
    __syncthreads();
    red[0] = result[turn & 15];
    red[1] = result[(turn + 1) & 15];
    turn += 2;
  };

  // ---- BiCGStabSolver::solve ----
  const double eps = A.metric ? A.metric[2 * prob + 1] : A.eps1;
  const double convergenceMetric = A.metric ? A.metric[2 * prob] : A.metric1;
  auto add_e = [&]() {  // incr(x, e, 1.0)
    each([&](int i) {
      const D2 w = x[i], z = e[i];
      x[i] = D2{w.r + z.r * 1.0, w.b + z.b * 1.0};
    });
  };
  int recount = 0, iter = 0, restarts = 0;
  double rho[4] = {0, 0, 0, 0}, nrm[2] = {0, 0};
  double alpha[2] = {0, 0}, beta[2] = {0, 0}, omega[2] = {0, 0};
  double initial_norm = 0, initial_residual = 0;
  bool init = true;
  // Each turn of the loop is one operator pass and its reductions: the residual that starts
  // or restarts the solve (RESIDUAL), the first half of an iteration (p_tilde, v and alpha) or
  // the second (s_tilde, t and omega).  The norm of r after the residual and after the second
  // half comes with the dot product (r_tilde, r) that the next iteration starts with.
  enum { RESIDUAL, FIRST, SECOND };
  int stage = RESIDUAL;
  bool begun = false, apply_e = true;
#pragma unroll 1
  for (;;) {
    const bool second = stage == SECOND;
    if (stage == RESIDUAL) {
      level_pass(r, x, 1.0, 0, b);
    } else {
      if (stage == FIRST) {
        if (init) {
          each([&](int i) { pp[i] = r[i]; });
          init = false;
        } else {
          // scale(p, beta); incr(p, v, -beta*omega); incr(p, r, 1.0)
          beta[1] = (rho[1] / rho[2]) * (alpha[1] / omega[1]);
          const double bw = -beta[1] * omega[1], bt1 = beta[1];
          auto upd = [&](double p0, double v0, double r0) {
            const double s1 = p0 * bt1;
            const double s2 = s1 + v0 * bw;
            return s2 + r0 * 1.0;
          };
          struct In {
            D2 p, v, r;
          };
          batch(M2{}, N, tid, [&](int i) { return In{pp[i], v[i], r[i]}; },
                [&](int i, const In& w) {
                  pp[i] = D2{upd(w.p.r, w.v.r, w.r.r), upd(w.p.b, w.v.b, w.r.b)};
                });
        }
      }
      level_pass(second ? t : v, second ? r : pp, mult, 4, nullptr);
    }
    // the reductions of this turn: `part` 0 the half's dot products, 1 the norm of r
#pragma unroll 1
    for (int part = stage == RESIDUAL ? 1 : 0; part < 2; part++) {
      if (part == 1) {
        if (stage == RESIDUAL)
          each([&](int i) {
            r_tilde[i] = r[i];
            e[i] = D2{0.0, 0.0};
          });
        reduce(r, r_tilde, stage != FIRST, true, true);
        nrm[0] = std::sqrt(red[1]);
        if (stage != FIRST) rho[0] = red[0];  // (r_tilde, r)
        break;
      }
      if (second) {
        reduce(t, r, true, true, false);
        omega[0] = red[0] / red[1];
      } else {
        reduce(v, r_tilde, true, false, false);
        const double m = red[0];
        alpha[0] = rho[1] / m;
        if (!(fabs(m) > A.par.small * fabs(rho[1]))) {
          each([&](int i) { r[i] = D2{0.0, 0.0}; });
          nrm[0] = 0.0;
          break;
        }
      }
      // r += y * m, e += tilde * w
      const D2* y = second ? t : v;
      const double w0 = second ? omega[0] : alpha[0], wm = -w0;
      struct In {
        D2 r, y, e, s;
      };
      batch(M2{}, N, tid, [&](int i) { return In{r[i], y[i], e[i], tilde[i]}; },
            [&](int i, const In& w) {
              r[i] = D2{w.r.r + w.y.r * wm, w.r.b + w.y.b * wm};
              e[i] = D2{w.e.r + w.s.r * w0, w.e.b + w.s.b * w0};
            });
    }
    if (stage == RESIDUAL) {
      if (!begun) {
        begun = true;
        initial_norm = initial_residual = nrm[1] = nrm[0];
        if (convergenceMetric > 0) initial_norm = convergenceMetric;
      } else {
        rho[1] = 0.0; rho[2] = 0.0; rho[3] = 0.0;
        alpha[0] = 0; beta[0] = 0; omega[0] = 0;
        restarts++;
        init = true;
      }
    } else {
      if (stage == FIRST && nrm[0] > eps * initial_norm && nrm[0] > A.par.reps * initial_residual) {
        stage = SECOND;
        continue;
      }
      if (nrm[0] <= eps * initial_norm || nrm[0] <= A.par.reps * initial_residual) break;  // exit status 1
      if (omega[0] == 0.0 || nrm[0] > (1 - A.par.hang) * nrm[1]) {
        if (recount == 0) {
          recount = 1;
        } else {
          recount = 0;
          add_e();
          if (restarts == A.par.numRestarts) {  // exit status 3
            apply_e = false;
            break;
          }
          stage = RESIDUAL;
          continue;
        }
      }
    }
    // the next iteration
    if (!((iter < A.par.imax && nrm[0] > eps * nrm[1]) && (nrm[1] > 0))) break;
    iter++;
    nrm[1] = nrm[0]; alpha[1] = alpha[0]; beta[1] = beta[0]; omega[1] = omega[0];
    rho[3] = rho[2]; rho[2] = rho[1];
    rho[1] = rho[0];
    if (rho[1] == 0.0) break;  // exit status 2
    stage = FIRST;
  }
  if (tid == 0 && A.stats) A.stats[prob] += iter;
  // incr(x, e, 1.0), rounded back into the V-cycle's precision
  each([&](int i) {
    D2 w = x[i];
    const D2 z = e[i];
    if (apply_e) w = D2{w.r + z.r * 1.0, w.b + z.b * 1.0};
    const int2 c = P.cell[i];
    if (c.x >= 0) corr[c.x] = (T)w.r;
    if (c.y >= 0) corr[c.y] = (T)w.b;
  });
}

template <class T, int NT, bool TREE>
void run_bottom(Context* ctx, const BottomLaunch<T>& a, int nprob, size_t bytes) {
  if (bytes > (size_t)kLdsBytes) throw std::runtime_error("bottom solve: LDS exceeded");
  auto* k = &k_bottom<T, NT, TREE>;
  if (bytes > 64 * 1024)
    hip_check(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes),
              "bottom LDS size");
  hipLaunchKernelGGL(k, dim3(nprob), dim3(NT), bytes, ctx->stream, a);
  hip_check(hipGetLastError(), "k_bottom");
}

}  // namespace

template <class T>
void launch_bottom(Context* ctx, const BottomLaunch<T>& a, int nprob, int maxSlots, size_t ldsBytes, bool tree) {
  if (nprob <= 0 || ctx->dry) return;
  if (maxSlots > kBottomMaxSlots) throw std::runtime_error("bottom solve: level too large");
  if (tree) run_bottom<T, 1024, true>(ctx, a, nprob, ldsBytes);
  else if (maxSlots <= 64) run_bottom<T, 64, false>(ctx, a, nprob, ldsBytes);
  else if (maxSlots <= 256) run_bottom<T, 256, false>(ctx, a, nprob, ldsBytes);
  else run_bottom<T, 1024, false>(ctx, a, nprob, ldsBytes);
}
template void launch_bottom<double>(Context*, const BottomLaunch<double>&, int, int, size_t, bool);
template void launch_bottom<float>(Context*, const BottomLaunch<float>&, int, int, size_t, bool);

}  // namespace amrmg
