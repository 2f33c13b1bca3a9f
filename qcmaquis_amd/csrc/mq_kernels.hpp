// Launch wrappers of the device kernels (mq_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "mq_plan.hpp"

namespace mq {

// Pipeline stage of a launch: each stage gets its own kernel instantiation so
// that profiles attribute time per stage.
enum Stage { ST_SIGMA = 0, ST_SIGMA_OUT = 1, ST_STEP = 2, ST_STEP_OUT = 3, ST_FUSE = 4, ST_MISC = 5 };

// sigma: the instantiation of the sigma's psi reshape (its own kernel name in profiles)
hipError_t launch_copy2d(const Copy2D *tasks, int n, const double *src, double *dst, hipStream_t s,
                         bool sigma = false);
hipError_t launch_copy2d(const Copy2D *tasks, int n, const double *src, float *dst, hipStream_t s,
                         bool sigma = false);
hipError_t launch_to_f32(const double *src, float *dst, int64_t n, hipStream_t s);
// one workgroup per pack of strips (StripList::packs)
// nvec > 1: the same task list for nvec vectors, vector v at T + v * src_stride and
// C + v * dst_stride
hipError_t launch_wapply(const Strip *strips, const Pack *packs, int npacks, const Src *srcs, const double *T,
                         double *C, int stage, hipStream_t s, int nvec = 1, int64_t src_stride = 0,
                         int64_t dst_stride = 0);
hipError_t launch_wapply(const Strip *strips, const Pack *packs, int npacks, const Src *srcs, const float *T, float *C,
                         int stage, hipStream_t s, int nvec = 1, int64_t src_stride = 0, int64_t dst_stride = 0);
// grouped GEMM over a plan's tile list (FP64; FP32 operands with FP32 or FP64 output,
// multiplied in FP32 or, with bf16x3, as three bf16 products accumulated in FP32);
// split_gids, nsplit: the groups with split-K partials; rblocks: workgroups of 256 that
// cover the largest one's elements (GemmList::reduce_blocks);
// rowmap: the row placements of groups with rowmap > 0 (may be null when none has)
hipError_t launch_gemm(const GemmGroup *groups, const GemmTile *tiles, int ntiles, const int *split_gids, int nsplit, int rblocks,
                       const double *A, const double *B, double *C, double *W, const RowMap *rowmap, int stage,
                       hipStream_t s);
hipError_t launch_gemm(const GemmGroup *groups, const GemmTile *tiles, int ntiles, const int *split_gids, int nsplit, int rblocks,
                       const float *A, const float *B, float *C, float *W, const RowMap *rowmap, int stage,
                       hipStream_t s, bool bf16x3 = false);
hipError_t launch_gemm(const GemmGroup *groups, const GemmTile *tiles, int ntiles, const int *split_gids, int nsplit, int rblocks,
                       const float *A, const float *B, double *C, float *W, const RowMap *rowmap, int stage,
                       hipStream_t s, bool bf16x3 = false);
// the sigma's output GEMM of plans with a gathered A operand (HostPlan::gather)
hipError_t launch_gemm_gather(const GemmGroup *groups, const GemmTile *tiles, int ntiles, const int *split_gids,
                              int nsplit, int rblocks, const double *A, const double *B, double *C, double *W,
                              const GatherSrc *src, const GatherQuad *quad, const GatherRow *row, hipStream_t s,
                              bool bf16x3 = false);
hipError_t launch_gemm_gather(const GemmGroup *groups, const GemmTile *tiles, int ntiles, const int *split_gids,
                              int nsplit, int rblocks, const float *A, const float *B, double *C, float *W,
                              const GatherSrc *src, const GatherQuad *quad, const GatherRow *row, hipStream_t s,
                              bool bf16x3);
// Davidson vector operations.  Vector pairs and coefficients are kernel arguments, at
// most kCombMax per launch.
constexpr int kCombMax = 48;
struct PairArgs {
    const double *x[kCombMax], *y[kCombMax];
};
struct CombArgs {
    const double *v[kCombMax];
    double c[kCombMax];
};
struct RitzArgs {
    double c[kCombMax];
};
// partial[p * nblocks + block] of x_p . y_p (device or pinned host memory)
hipError_t launch_multidot(const PairArgs &a, int npairs, int64_t n, int nblocks, double *partial, hipStream_t s);
// one step of an orthonormalisation against V (m vectors, one after another); partials
// are [row][block], row 0 t.t (when self), then V_i.t; see k_orth
enum OrthMode { ORTH_DOTS = 0, ORTH_CORRECTION = 1, ORTH_UPDATE = 2 };
hipError_t launch_orth(OrthMode mode, const double *V, int64_t n, int m, double *t, const double *u, const double *r,
                       const double *w, const double *pin, const double *ptau, bool self, int nblocks, double *pout,
                       hipStream_t s);
hipError_t launch_normalise(double *t, int64_t n, int nblocks, const double *p0, const double *p1, const double *p2,
                            hipStream_t s);
// Ritz vector u, residual r and the partials of r.r, r.u, u.u; see k_ritz
hipError_t launch_ritz(const RitzArgs &c, int nv, const double *V, const double *VA, int64_t n, double theta,
                       bool first, bool last, double *u, double *r, int nblocks, double *pdev, double *phost,
                       hipStream_t s);
// out = (x - f u) / (theta - D), elementwise, leaving the elements where theta == D
// undivided (MultDiagonal::mult_diag); out may alias x
hipError_t launch_diag_scale(const double *x, const double *u, double f, const double *D, double theta, double *out,
                             int64_t n, hipStream_t s);
hipError_t launch_lincomb(const CombArgs &a, int nv, int64_t n, double beta, double *out, hipStream_t s);
// two-site split: gather psi into the SVD working matrices (X must be zeroed
// first) and the assembly of the two site tensors
hipError_t launch_split_gather(const SplitSlab *slabs, int n, const double *psi, double *X, hipStream_t s);
// Jacobi SVD of every block: init (V = I, flags), one launch per round of a sweep
// (one wave per column pair of every block), the end-of-sweep flag update, and
// the sorted singular values with their permutation
hipError_t launch_jacobi_init(const SvdBlk *blks, int nblk, double *V, int32_t *done, int32_t *rot, int32_t *sweeps,
                              hipStream_t s);
hipError_t launch_jacobi_round(const SvdBlk *blks, const int32_t *slot_blk, const int32_t *slot_k, int nslots, int t,
                               double *X, double *V, const int32_t *done, int32_t *rot, hipStream_t s);
hipError_t launch_jacobi_sweep_end(int nblk, int sweep, int32_t *done, int32_t *rot, int32_t *sweeps,
                                   hipStream_t s);
hipError_t launch_jacobi_finish(const SvdBlk *blks, int nblk, int max_c, const double *X, double *S, int32_t *perm,
                                const int32_t *done, int32_t *sweeps, hipStream_t s);
hipError_t launch_split_assemble(const SvdBlk *blks, int nblk, int max_keep, const int32_t *keep,
                                 const int64_t *a_off, const int64_t *b_off, int l2r, const double *X,
                                 const double *V, const double *S, const int32_t *perm, double *A, double *B,
                                 hipStream_t s);

}  // namespace mq
