// Smoothing visits of small merged levels as one launch each (block.hip): one or two GSRB
// iterations, optionally with the prolongation before them or the restriction of the residual
// after them.
#pragma once
#include "ops.hpp"

namespace amrmg {
namespace ops {

// Whether the block visits apply to a level: merged, with the one-launch relaxation's face
// rules, and of at most kBlockCells cells.  Above that the marching kernels, which read each cell
// about 1.5 times per iteration and not 8 times per visit, are ahead (a V-cycle of n^3 cells
// over its coarser levels, microseconds, blocks and marching launches: 16^3 111 and 166, 64^3 176
// and 225, 80^3 293 and 329, 96^3 455 and 463, 112^3 680 and 650, 128^3 945 and 865; FP32 64^3 175
// and 230, 96^3 428 and 455, 112^3 625 and 635, 128^3 862 and 846).
constexpr long long kBlockCells = 1LL << 20;
inline bool block_visit_ok(const DeviceLayout& L) { return L.merged && L.valid_cells <= kBlockCells; }

// dst <- `sweeps` (1 or 2) GSRB iterations of src (+ prolonged coarse) with right-hand side rhs;
// zero_src: src is known to be zero and not read (then coarse must be null); coarse not null:
// PROLONG first, src + coarse(i >> 1); resc not null: RESTRICTRES of the result onto the
// coarsened level.  Lc: the coarsened level (null when neither is given).  Bitwise the
// sequence of prolong, gsrb_fused (sweeps times) and restrict_res.
template <class T>
void block_visit(const DeviceLayout& L, const FaceRules& fr, const DeviceLayout* Lc, T* dst, const T* src,
                 const T* rhs, const T* coarse, T* resc, double dx, double alpha, double beta, int sweeps,
                 bool zero_src);

}  // namespace ops
}  // namespace amrmg
