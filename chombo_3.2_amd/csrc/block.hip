// A smoothing visit of a small merged level in one launch.
//
// What bounds it: on levels of up to about a million cells the V-cycle is a chain of launches, each
// a few microseconds of dependent latency (a z march of six planes takes 6.5 us however small
// the level), with all data in L2.  So a workgroup takes a block of BX x BY x BZ cells with a halo
// wide enough for the whole visit into LDS in one go, all loads in flight together, and runs
// every half sweep there: the red cells of the block grown by 2 s - 1, the black ones of the block
// grown by 2 s - 2, ... (the halo is recomputed by the neighbouring blocks, which read old values
// only, as in the one-launch relaxation of kernels.hip, whose face rules and expressions these
// are).  The price is the halo: a two-sweep visit reads (8 + 8)^3 / 8^3 = 8 times its cells, from L2.
//
// Measured at 64^3, FP64 (8 x 8 x 8 blocks, 512 threads): the visit down 12.1 us (marching: two
// relaxations of 6.6 us, ghosts 3.6, restriction 5), the visit up 8.7 us (prolongation 5, two of
// 6.6); a 64^3 solve 2.60 -> 1.39 ms together with the shorter march.
//
// PROLONG enters with the loads (phi + coarse(i >> 1) for every cell of the halo); RESTRICTRES
// runs on the finished block grown by one.  Per level a V-cycle then has two launches in place of
// eight: relax, relax, ghost fill, restrict and prolong, relax, relax.
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "block.hpp"
#include "fused.hpp"

namespace amrmg {
namespace ops {

namespace {

struct BlockArgs {
  int lo[3], hi[3];
  long long off;  // slab index of (lo-1, lo-1, lo-1)
  int sy, sz;
  int ntx, nty, nwork;
  int kind[3][2];
  // the coarsened level
  int clo[3];
  long long coff;
  int csy, csz;
};

// x neighbour sums in the reference's order with the face rules of fused_new
template <class T>
__device__ __forceinline__ T block_six(const BlockArgs& a, const T* S, int c, int W, int P, int i, int j, int k, T own,
                                       T c1, T c2) {
  const T vxp = S[c + 1], vxm = S[c - 1], vyp = S[c + W], vym = S[c - W], vzp = S[c + P], vzm = S[c - P];
  const T xp = (i == a.hi[0]) ? face_ghost(a.kind[0][1], own, vxm, c1, c2) : vxp;
  const T xm = (i == a.lo[0]) ? face_ghost(a.kind[0][0], own, vxp, c1, c2) : vxm;
  const T yp = (j == a.hi[1]) ? face_ghost(a.kind[1][1], own, vym, c1, c2) : vyp;
  const T ym = (j == a.lo[1]) ? face_ghost(a.kind[1][0], own, vyp, c1, c2) : vym;
  const T zp = (k == a.hi[2]) ? face_ghost(a.kind[2][1], own, vzm, c1, c2) : vzp;
  const T zm = (k == a.lo[2]) ? face_ghost(a.kind[2][0], own, vzp, c1, c2) : vzm;
  return xp + xm + yp + ym + zp + zm;
}

template <class T, bool LAP, int BX, int BY, int BZ, int NS, bool REST, int NT>
__global__ void __launch_bounds__(NT) k_block_visit(BlockArgs a, T* __restrict__ dst, const T* __restrict__ src,
                                                    const T* __restrict__ rhs, const T* __restrict__ coarse,
                                                    T* __restrict__ resc, T dxinv, T lambda, T alpha, T beta, T c1,
                                                    T c2) {
  constexpr int G = 2 * NS + (REST ? 1 : 0);  // halo of phi; rhs needs one less
  constexpr int EX = BX + 2 * G, EY = BY + 2 * G, EZ = BZ + 2 * G, EP = EX * EY, EN = EP * EZ;
  constexpr int RX = EX - 2, RY = EY - 2, RZ = EZ - 2, RN = RX * RY * RZ;
  constexpr int NL = (EN + NT - 1) / NT, NR = (RN + NT - 1) / NT;
  __shared__ T S[EN];
  __shared__ T R[RN];
  const int w = xcd_contiguous_block();
  if (w >= a.nwork) return;
  const int tid = threadIdx.x;
  const int tx = w % a.ntx, ty = (w / a.ntx) % a.nty, tz = w / (a.ntx * a.nty);
  const int x0 = a.lo[0] + tx * BX, y0 = a.lo[1] + ty * BY, z0 = a.lo[2] + tz * BZ;
  auto gidx = [&](int i, int j, int k) {
    return a.off + (i - a.lo[0] + 1) + (long long)(j - a.lo[1] + 1) * a.sy + (long long)(k - a.lo[2] + 1) * a.sz;
  };
  // every load is from an address clamped into the rectangle; values outside it are never used
  {
    T p[NL], r[NR];
    if (src) {
#pragma unroll
      for (int u = 0; u < NL; u++) {
        const int q = min(tid + NT * u, EN - 1);
        const int i = clampi(x0 - G + q % EX, a.lo[0], a.hi[0]), j = clampi(y0 - G + (q / EX) % EY, a.lo[1], a.hi[1]),
                  k = clampi(z0 - G + q / EP, a.lo[2], a.hi[2]);
        p[u] = src[gidx(i, j, k)];
      }
    } else {
#pragma unroll
      for (int u = 0; u < NL; u++) p[u] = T(0.0);
    }
#pragma unroll
    for (int u = 0; u < NR; u++) {
      const int q = min(tid + NT * u, RN - 1);
      const int i = clampi(x0 - G + 1 + q % RX, a.lo[0], a.hi[0]),
                j = clampi(y0 - G + 1 + (q / RX) % RY, a.lo[1], a.hi[1]),
                k = clampi(z0 - G + 1 + q / (RX * RY), a.lo[2], a.hi[2]);
      r[u] = rhs[gidx(i, j, k)];
    }
    if (coarse) {
#pragma unroll
      for (int u = 0; u < NL; u++) {
        const int q = min(tid + NT * u, EN - 1);
        const int i = clampi(x0 - G + q % EX, a.lo[0], a.hi[0]), j = clampi(y0 - G + (q / EX) % EY, a.lo[1], a.hi[1]),
                  k = clampi(z0 - G + q / EP, a.lo[2], a.hi[2]);
        p[u] = p[u] + coarse[a.coff + ((i >> 1) - a.clo[0] + 1) + (long long)((j >> 1) - a.clo[1] + 1) * a.csy +
                             (long long)((k >> 1) - a.clo[2] + 1) * a.csz];
      }
    }
#pragma unroll
    for (int u = 0; u < NL; u++)
      if (tid + NT * u < EN) S[tid + NT * u] = p[u];
#pragma unroll
    for (int u = 0; u < NR; u++)
      if (tid + NT * u < RN) R[tid + NT * u] = r[u];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2 * NS; h++) {
    const int colour = h & 1;
    const int g = 2 * NS - 1 - h + (REST ? 1 : 0);  // this half sweep covers the block grown by g
    const int HX = (BX + 2 * g) / 2, HY = BY + 2 * g, HN = HX * HY * (BZ + 2 * g);
    for (int q = tid; q < HN; q += NT) {
      const int j = y0 - g + (q / HX) % HY, k = z0 - g + q / (HX * HY);
      const int i = x0 - g + 2 * (q % HX) + ((x0 - g + j + k + colour) & 1);
      if (i < a.lo[0] || i > a.hi[0] || j < a.lo[1] || j > a.hi[1] || k < a.lo[2] || k > a.hi[2]) continue;
      const int c = (i - x0 + G) + (j - y0 + G) * EX + (k - z0 + G) * EP;
      const T own = S[c];
      const T f = R[(i - x0 + G - 1) + (j - y0 + G - 1) * RX + (k - z0 + G - 1) * (RX * RY)];
      const T s6 = block_six<T>(a, S, c, EX, EP, i, j, k, own, c1, c2);
      if (LAP) {
        const T lphi = s6 * dxinv;
        S[c] = lambda * (f - lphi);
      } else {
        const T lphi = (s6 - T(6.0) * own) * dxinv;
        const T helmop = alpha * own + beta * lphi;
        S[c] = own + lambda * (helmop - f);
      }
    }
    __syncthreads();
  }
  for (int q = tid; q < BX * BY * BZ; q += NT) {
    const int i = x0 + q % BX, j = y0 + (q / BX) % BY, k = z0 + q / (BX * BY);
    if (i <= a.hi[0] && j <= a.hi[1] && k <= a.hi[2])
      dst[gidx(i, j, k)] = S[(i - x0 + G) + (j - y0 + G) * EX + (k - z0 + G) * EP];
  }
  if constexpr (REST) {
    // RESTRICTRES (AMRPoissonOpF.ChF:394-438): a coarse cell's eight children in the Fortran
    // loop order; the block starts on even cells and the rectangle's extents are even
    for (int q = tid; q < BX * BY * BZ / 8; q += NT) {
      const int I = q % (BX / 2), J = (q / (BX / 2)) % (BY / 2), K = q / (BX * BY / 4);
      const int i0 = x0 + 2 * I, j0 = y0 + 2 * J, k0 = z0 + 2 * K;
      if (i0 > a.hi[0] || j0 > a.hi[1] || k0 > a.hi[2]) continue;
      T acc = T(0.0);
      for (int kk = 0; kk < 2; kk++)
        for (int jj = 0; jj < 2; jj++)
#pragma unroll
          for (int ii = 0; ii < 2; ii++) {
            const int i = i0 + ii, j = j0 + jj, k = k0 + kk;
            const int c = (i - x0 + G) + (j - y0 + G) * EX + (k - z0 + G) * EP;
            const T p = S[c];
            const T f = R[(i - x0 + G - 1) + (j - y0 + G - 1) * RX + (k - z0 + G - 1) * (RX * RY)];
            const T lofphi =
                alpha * p + beta * (block_six<T>(a, S, c, EX, EP, i, j, k, p, c1, c2) - p * T(2.0) * T(3.0)) * dxinv;
            acc = acc + (f - lofphi) / T(8.0);
          }
      resc[a.coff + ((i0 >> 1) - a.clo[0] + 1) + (long long)((j0 >> 1) - a.clo[1] + 1) * a.csy +
           (long long)((k0 >> 1) - a.clo[2] + 1) * a.csz] = acc;
    }
  }
}

constexpr int kBX = 8, kBY = 8, kBZ = 8, kBT = 512;

}  // namespace

template <class T>
void block_visit(const DeviceLayout& L, const FaceRules& fr, const DeviceLayout* Lc, T* dst, const T* src,
                 const T* rhs, const T* coarse, T* resc, double dx, double alpha, double beta, int sweeps,
                 bool zero_src) {
  if (!block_visit_ok(L)) throw std::runtime_error("block_visit: level does not qualify");
  if (sweeps != 1 && sweeps != 2) throw std::runtime_error("block_visit: one or two sweeps");
  if (dst == src || dst == rhs) throw std::runtime_error("block_visit: dst must be a separate field");
  if ((coarse || resc) && (!Lc || !Lc->merged)) throw std::runtime_error("block_visit: no merged coarser level");
  if (coarse && zero_src) throw std::runtime_error("block_visit: prolongation onto a field that is not read");
  const DBox& R = L.h_boxes[L.nbox];
  BlockArgs a{};
  for (int q = 0; q < 3; q++) {
    a.lo[q] = R.lo[q];
    a.hi[q] = R.hi[q];
  }
  for (int d = 0; d < 3; d++)
    for (int s = 0; s < 2; s++) {
      if (fr.kind[d][s] < 0 || fr.kind[d][s] > 2) throw std::runtime_error("block_visit: bad face rule");
      a.kind[d][s] = fr.kind[d][s];
    }
  a.off = R.off;
  a.sy = R.sy;
  a.sz = R.sz;
  if (coarse || resc) {
    const DBox& C = Lc->h_boxes[Lc->nbox];
    for (int q = 0; q < 3; q++) {
      if (R.lo[q] % 2 != 0 || (R.hi[q] + 1) % 2 != 0 || R.lo[q] / 2 != C.lo[q] || (R.hi[q] + 1) / 2 - 1 != C.hi[q])
        throw std::runtime_error("block_visit: the coarser level is not the level coarsened by 2");
      a.clo[q] = C.lo[q];
    }
    a.coff = C.off;
    a.csy = C.sy;
    a.csz = C.sz;
  }
  a.ntx = (L.rect.len(0) + kBX - 1) / kBX;
  a.nty = (L.rect.len(1) + kBY - 1) / kBY;
  a.nwork = a.ntx * a.nty * ((L.rect.len(2) + kBZ - 1) / kBZ);
  const int grid = (a.nwork + 7) / 8 * 8;
  const double dxinv = 1.0 / (dx * dx);
  double sum_b = 0.0;
  for (int d = 0; d < 3; d++) sum_b = sum_b + 2.0 * dxinv;
  const bool lap = (alpha == 0.0 && beta == 1.0);
  const double lambda = lap ? -1.0 / sum_b : -1.0 / (alpha - beta * sum_b);
  const T* s = zero_src ? nullptr : src;
  // algorithmic bytes of the visit: read phi (not when it is known zero), read rhs, write phi; the
  // coarse field
  const double bytes = ((zero_src ? 16.0 : 24.0) + (coarse || resc ? 1.0 : 0.0)) * sizeof(T) / 8.0 * L.valid_cells;
  hipEvent_t ev = profile_begin(L.ctx, KC_GSRB);
#define BLOCK_LAUNCH(LAPV, NS, RESTV)                                                                            \
  hipLaunchKernelGGL((k_block_visit<T, LAPV, kBX, kBY, kBZ, NS, RESTV, kBT>), dim3(grid), dim3(kBT), 0,         \
                     L.ctx->stream, a, dst, s, rhs, coarse, resc, T(dxinv), T(lambda), T(alpha), T(beta), T(fr.c1), \
                     T(fr.c2))
#define BLOCK_PICK(LAPV)                                      \
  do {                                                        \
    if (sweeps == 2 && resc) BLOCK_LAUNCH(LAPV, 2, true);     \
    else if (sweeps == 2) BLOCK_LAUNCH(LAPV, 2, false);       \
    else if (resc) BLOCK_LAUNCH(LAPV, 1, true);               \
    else BLOCK_LAUNCH(LAPV, 1, false);                        \
  } while (0)
  if (lap) BLOCK_PICK(true);
  else BLOCK_PICK(false);
#undef BLOCK_PICK
#undef BLOCK_LAUNCH
  hip_check(hipGetLastError(), "k_block_visit");
  profile_end(L.ctx, ev, KC_GSRB, bytes, (double)L.valid_cells * sweeps);
}
template void block_visit<double>(const DeviceLayout&, const FaceRules&, const DeviceLayout*, double*, const double*,
                                  const double*, const double*, double*, double, double, double, int, bool);
template void block_visit<float>(const DeviceLayout&, const FaceRules&, const DeviceLayout*, float*, const float*,
                                 const float*, const float*, float*, double, double, double, int, bool);

}  // namespace ops
}  // namespace amrmg
