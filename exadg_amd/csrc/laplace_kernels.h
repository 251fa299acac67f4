// Launch interface of the SIPG Laplace kernels (host-callable, no HIP types beyond streams).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "topology.h"

namespace ExaDG
{
enum class ApplyMode : int
{
  vmult     = 0,  // dst = A src
  vmult_add = 1,  // dst += A src
  diagonal  = 2,  // dst[cell, i] = (A_KK)_{ii}: unit-vector probing of the cell-local block
  // Chebyshev-Jacobi step fused into the epilogue (src = x, dst = x_new):
  // x_new = (1 + f1) x - f1 x_old (if has_old) + f2 dinv (b - A x); x_old may alias dst
  chebyshev = 3,
  // residual in the epilogue: dst = rhs - A src (dst may alias rhs, not src)
  residual = 4,
  // residual and p-restriction in the epilogue: per cell
  // dst_coarse += (R x R x R)(rhs - A src), R = P^T with P the n x nc prolongation matrix;
  // dst is the coarse DG vector of the same cells (nc^3 values per cell)
  residual_restrict = 5
};

// Centrosymmetric n x n matrices (A_ij = A_{n-1-i,n-1-j}, such as the 1D mass and stiffness
// on symmetric nodes) are stored in even-odd form, which needs ~n^2/2 products per
// application instead of n^2: with m = n/2 and m_e = m + n%2,
//   Ae (m x m_e): (A_ij + A_{i,n-1-j})/2 for j < m, A_im for j = m (odd n),
//   Ao (m x m):   (A_ij - A_{i,n-1-j})/2,
//   Am (m_e, odd n only): the middle row A_mj, j <= m.
// The Cartesian kernel packs at every n (its line Laplacian shares the even and odd parts with the
// end derivatives and the flux terms); the general kernel for n >= 6 (at n = 5 its saving
// is 4% of the instructions and the FP32 instantiation measured slower with it).
constexpr int  eo_size(int n, bool packed)
{
  return packed ? (n / 2) * (n / 2 + n % 2) + (n / 2) * (n / 2) + (n % 2 ? n / 2 + 1 : 0) : n * n;
}
constexpr int  cs_size(int n) { return eo_size(n, true); }
constexpr bool gen_packed(int n) { return n >= 6; }
constexpr int  gen_size(int n) { return eo_size(n, gen_packed(n)); }
// Offsets in the Cartesian kernel's table: the unit-interval mass M in even-odd form, the end
// derivative d0, d0 in even-odd form (DE_j = (d0_j + d0_{n-1-j})/2 for j < n/2 and d0_m in the
// middle for odd n, DO_j = (d0_j - d0_{n-1-j})/2; the other end mirrors it, d1_j = -d0_{n-1-j}),
// then per direction the stiffness times c/h and DE, DO times c/(2h), c the scale of the
// direction's Kronecker term
template<int N>
struct CartTable
{
  static constexpr int M = 0, D0 = cs_size(N), DE = D0 + N, DO = DE + N / 2 + N % 2, L = D0 + 2 * N;
  static constexpr int line(int d) { return L + d * (cs_size(N) + N); }
};

// Offsets in the general kernel's table: S n*n, Dq n*n, d0 n, d1 n; l(0), l(1), l'(0), l'(1) of the
// Lagrange polynomials on the Gauss points, n each; and the four sweep matrices S, Dq, S^T, Dq^T in
// even-odd form. S is centrosymmetric and Dq skew-centrosymmetric (A_ij = -A_{n-1-i,n-1-j}) on the
// symmetric Gauss points; the skew form stores Ae and Ao as above and, for odd n, the middle row's
// coefficients of the odd part, A_mj for j < m, padded to m_e entries.
template<int N>
struct GenTable
{
  static constexpr int S = 0, DQ = N * N, D0 = 2 * N * N, D1 = D0 + N, L0 = D1 + N, L1 = L0 + N,
                       G0 = L1 + N, G1 = G0 + N, SE = G1 + N, DE = SE + gen_size(N),
                       STE = DE + gen_size(N), DTE = STE + gen_size(N), SIZE = DTE + gen_size(N);
};
template<typename Number>
struct SipgArgs
{
  // 1D tables (CartTable, GenTable) in device memory: as a by-value copy in the kernel arguments each
  // launch wrote them anew and read them past the L2 cache
  Number const * tables;
  // Cartesian kernel: the scales c_x = h_y h_z, ... of the three Kronecker terms, and c_d/(2 h_d)
  Number         scale[3], half[3];
  Number const * src;
  Number *       dst;
  Number const * cell_metric;  // general kernel only
  Number const * face_data;    // general kernel only
  Number const * tau_face;
  BoxTopology    topo;
  int64_t        n_cells;
  int            probe;      // diagonal mode: local index of the unit vector
  // diagonal mode: 0 stores (A_KK)_{probe,probe} at dst[cell n^3 + probe]; 1 stores the whole
  // response A_KK e_probe as column `probe` of the cell's n^3 x n^3 block,
  // dst[(cell n^3 + probe) n^3 + e] (the block is symmetric, so this is also row `probe`)
  int            block = 0;
  int            tile_rows;  // traversal: y-rows per tile (one tile per XCD)
  // Cartesian layered kernel: the penalty of a cell inside the mesh and what each boundary face
  // normal to a direction adds; the lane assignment (cartesian_line_map, device memory) and the
  // tiling, set by the launch
  double         tau_base, tau_step[3];
  int const *    line_map = nullptr;
  int            row_length = 0, tiles = 0, layers_per_segment = 0;
  // chebyshev and residual modes
  Number const * x_old   = nullptr;
  Number const * rhs     = nullptr;
  Number const * dinv    = nullptr;
  Number         f1      = 0;
  Number         f2      = 0;
  int            has_old = 0;
  // residual_restrict mode: P (n x nc, row-major) and nc
  Number const * restrict_P  = nullptr;
  int            restrict_nc = 0;
};

// degree 1..8; mode as above. Returns hipError of the launch.
template<typename Number>
hipError_t launch_sipg_general(int degree, ApplyMode mode, SipgArgs<Number> const & args,
                               hipStream_t stream);
// Diagonal of the affine SIPG operator in closed form, one thread per DoF: the cell block is
// L_x (x) h_y M (x) h_z M + h_x M (x) L_y (x) h_z M + h_x M (x) h_y M (x) L_z with the 1D
// cell-local line operators L_d (the cell's own face terms, neighbours zero, or the cell's own
// values across a periodic face of a one-cell direction), so its diagonal is a sum of three
// products of 1D diagonals. diag1d: [M_ii | K_ii | d0 | d1] of the unit interval (4n doubles).
template<typename Number>
hipError_t launch_cartesian_diagonal(Number * diag, double const * diag1d, Number const * tau_face,
                                     BoxTopology const & topo, double const (&h)[3], int n,
                                     int64_t n_cells, hipStream_t stream);

// Diagonal of the curved SIPG operator, sum-factorized, one group of n^2 lanes per cell:
// the cell term sum_q G_ab(q) d_a phi_i d_b phi_i as six three-sweep contractions of the metric
// with products of the 1D tables, plus the own-side face terms of the face-layer DoFs,
// c w (tau phi_i^2 - phi_i a.grad phi_i) with c = 1 (interior, neighbour zero), 2 (Dirichlet
// mirror), 0 (Neumann). tab1d: [SS | DD | SD] (n x n each, [q][i]: S^2, D^2, S D with S the
// Gauss interpolation and D = Dq S) then [l'(0) of node 0, l'(1) of node n-1]. Meshes with a
// one-cell periodic direction are not handled (the cell is its own neighbour).
template<typename Number>
hipError_t launch_general_diagonal(Number * diag, double const * tab1d, SipgArgs<Number> const & a,
                                   int degree, hipStream_t stream);

// The lane assignment of the layered Cartesian kernel's x- and y-lines: per direction one entry per
// lane, its LDS base | line << 16 (the two other coordinates, lower fastest) | the cell's column
// and row in the tile << 23 and << 26, or -1; empty for degrees without that kernel
template<typename Number>
std::vector<int> cartesian_line_map(int degree);

// The kernel that vmult and vmult_add launch for these arguments
template<typename Number>
char const * cartesian_vmult_kernel(int degree, SipgArgs<Number> const & args);

template<typename Number>
hipError_t launch_sipg_cartesian(int degree, ApplyMode mode, SipgArgs<Number> const & args,
                                 hipStream_t stream);

}  // namespace ExaDG
