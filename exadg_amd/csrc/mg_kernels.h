// Multigrid kernels: polynomial (p) transfer between DG levels on the same mesh and the
// continuous Q1 operator (the c-transfer and the other continuous levels are in cg_kernels.h).
//
// Reference: MultigridTransfer (solvers_and_preconditioners/multigrid/transfer.cpp:28-96) ->
// MGTwoLevelTransfer::reinit_polynomial_transfer; the continuous coarse level of the hybrid
// multigrid (multigrid_preconditioner_base.cpp:191-226) with Dirichlet constraints
// (multigrid/constraints.h:109-194) acting as identity rows (operator_base.cpp:299-309).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "topology.h"

namespace ExaDG
{
// Q1 node numbering of the structured box: (n_d + 1) nodes per non-periodic direction,
// n_d nodes per periodic direction (node n_d is node 0).
struct Q1Topology
{
  int nc[3];
  int nn[3];        // nodes per direction
  int periodic[3];
  int dirichlet[6]; // side constrained (Dirichlet, non-periodic)
};

// dst_f += (P x P x P) src_c per cell, P = nf x nc interpolation matrix (row-major)
template<typename Number>
hipError_t launch_p_prolongate_add(Number * dst_f, Number const * src_c, Number const * P, int nf,
                                   int nc, int64_t n_cells, hipStream_t s);
// dst_c += (P^T x P^T x P^T) src_f per cell
template<typename Number>
hipError_t launch_p_restrict_add(Number * dst_c, Number const * src_f, Number const * P, int nf,
                                 int nc, int64_t n_cells, hipStream_t s);
// The rows of an assembled 27-point stencil, entry j for the neighbour offset
// (j%3-1, (j/3)%3-1, j/9-1). Per node: 27 planes of n_nodes weights. Where all cells are alike (an
// affine box) a row depends only on how far its node is from the mesh's ends: per direction 2 if
// periodic, else the coordinate c if c < 2 or there are fewer than 5 nodes, c + 5 - m for the last
// two of m nodes, 2 between; class kx + 5 (ky + 5 kz), whose row starts at kQ1ClassStride entries
// times it. `classes` is used if it is not null.
//
// Planes of kQ1ClassBytes and more are replaced by classes: they are read in full by every step, the
// classes from cache, but with their loads behind the node's class. V-cycles with 100 - 130 steps,
// planes / classes in us: FP64 on 28 x 27 x 26 nodes (4 MB) 338 / 355, 35 x 34 x 33 (8 MB) 460 / 467,
// 50 x 49 x 48 (25 MB) 961 / 911, 61^3 (49 MB) 2014 / 1628, 67^3 (65 MB) 2906 / 2301, periodic in x
// and y 66 x 66 x 67 3647 / 2442; FP32 35 x 34 x 33 (4 MB) 352 / 357, 50 x 49 x 48 (13 MB)
// 612 / 620, 61^3 (25 MB) 1195 / 1003, 67^3 (32 MB) 1737 / 1326.
constexpr int     kQ1Classes = 125, kQ1ClassStride = 28;
constexpr int64_t kQ1ClassBytes = 20000000;
template<typename Number>
struct Q1Weights
{
  Number const *planes, *classes;
};
// Q1 operator as an assembled 27-point stencil (periodic wrap; constrained rows identity)
template<typename Number>
hipError_t launch_q1_stencil(Number * dst, Number const * src, Q1Weights<Number> const & W,
                             Q1Topology const & q, hipStream_t s);
// one Chebyshev-Jacobi step with the stencil application fused:
// x_new = (1+f1) x - f1 x_old (if has_old) + f2 dinv (b - A x)
template<typename Number>
hipError_t launch_q1_chebyshev(Number * x_new, Number const * x, Number const * x_old,
                               Number const * b, Number const * dinv, Q1Weights<Number> const & W,
                               Q1Topology const & q, Number f1, Number f2, bool has_old,
                               hipStream_t s);

// PCG with point Jacobi on a Q1 level of at most kQ1PcgMaxNodes nodes, in one workgroup: x from zero
// to |r| <= max(1e-12, rel_tol |b|), with the mean of b and of every residual removed if singular. r
// and v: n entries of workspace each; result: iterations, then 1 if a residual was not
// finite. The line lies where one workgroup's pass over the stencil takes as long as an iteration
// driven from the host, host-driven / here: whole solves with the FP32 V-cycle 729 nodes 9.2 / 3.7 ms,
// 1296 nodes 33 / 11.5 ms, 9261 nodes 21.8 / 15.6 ms, 17576 nodes 34.5 / 39.2 ms; one V-cycle at 9261
// nodes FP32 1401 / 999 us, FP64, which reads twice the bytes, 1441 / 1289 us.
constexpr int kQ1PcgMaxNodes = 10000;
template<typename Number>
struct Q1PcgArgs
{
  Number *       x, *r, *v;
  Number const * b, *dinv, *W;
  Q1Topology     q;
  int            n, max_iter, singular;
  double         rel_tol;
  double *       result;
};
template<typename Number>
hipError_t launch_q1_pcg(Q1PcgArgs<Number> const & args, hipStream_t s);

}  // namespace ExaDG
