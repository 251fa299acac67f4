// SIPG Laplace operator kernels for CDNA4 (gfx950): curved meshes, and the diagonals (the affine
// operator is in cartesian_kernels.hip).
//
// The operator kernels are element-centric: one group of (k+1)^2 lanes owns one cell, computes the
// cell integral and all six face integrals seen from that cell (reading the neighbour's
// lines from global memory / L2), and writes each dst entry exactly once -- no atomics.
// A workgroup packs floor(256/(k+1)^2) cells; each cell gets its own LDS slice.
//
// Reference semantics: LaplaceOperator::do_cell_integral / do_face_integral /
// do_boundary_integral (poisson/spatial_discretization/laplace_operator.cpp:129-265),
// LaplaceKernel::calculate_{gradient,value}_flux (laplace_operator.h:180-197) and the
// homogeneous mirror BCs of weak_boundary_conditions.h:39-47,142-160.
#include <hip/hip_runtime.h>

#include <atomic>

#include "../../include/exadg_amd.h"
#include "laplace_kernels.h"
#include "sipg_lines.h"

namespace ExaDG
{
namespace
{
constexpr int cells_per_block(int n) { return (256 / (n * n)) > 0 ? 256 / (n * n) : 1; }

// Base offset and stride of the line along direction d through lane (p,q) of an N^3 block with
// strides 1, PX, PY; (p,q) index the two other directions in increasing order.
template<int N, int PX = N, int PY = N * N>
__device__ __forceinline__ void line_geometry(int d, int p, int q, int & base, int & stride)
{
  if(d == 0)
  {
    base   = PX * p + PY * q;
    stride = 1;
  }
  else if(d == 1)
  {
    base   = p + PY * q;
    stride = PX;
  }
  else
  {
    base   = p + PX * q;
    stride = PY;
  }
}

// face type (kInterior or the boundary type) of side (d, s) of a cell, all six in two bits each, and
// the face's index. 32 bits number the faces of a curved mesh: its 6 n^3 metric values per cell and
// 7 n^2 values for each of three faces (528 bytes at n = 2 in FP32) end at 5.5e8 cells in 288 GB
__device__ __forceinline__ int face_types(BoxTopology const & t, int const (&cc)[3])
{
  int types = 0;
#pragma unroll
  for(int d = 0; d < 3; ++d)
  {
    types |= (cc[d] > 0 || t.periodic[d] ? kInterior : t.bc[2 * d]) << (4 * d);
    types |= (cc[d] < t.nc[d] - 1 || t.periodic[d] ? kInterior : t.bc[2 * d + 1]) << (4 * d + 2);
  }
  return types;
}

__device__ __forceinline__ int face_index(BoxTopology const & t, int const (&cc)[3], int d, int side)
{
  int const t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
  int const fl = cc[d] + side == t.layers[d] ? 0 : cc[d] + side;
  return (int)t.face_base[d] + fl + t.layers[d] * (cc[t1] + t.nc[t1] * cc[t2]);
}

// the cell's unit vector in diagonal (probing) mode, else the src line
template<int N, typename Number, ApplyMode mode>
__device__ __forceinline__ void source_line(Number const * __restrict__ src, int64_t cell, int base,
                                            int stride, int probe, Number (&v)[N])
{
  constexpr int N3 = N * N * N;
  if constexpr(mode == ApplyMode::diagonal)
  {
#pragma unroll
    for(int i = 0; i < N; ++i)
      v[i] = (base + i * stride == probe) ? Number(1) : Number(0);
  }
  else
    load_line<N>(src + cell * N3 + base, stride, v);
}

// ================================================================ general (curved) kernel
//
// Cell term by collocation at the Gauss points: u_q = (S x S x S) u, reference gradient
// by the Gauss collocation derivative Dq, symmetric metric G = JxW J^{-1} J^{-T} per point,
// then the transposed sweeps. Face terms between the two: the own traces from the Gauss
// values, the neighbour traces interpolated from the face nodes, flux with the per-point
// normal-derivative vectors a = J^{-1} n of both sides, and the face tests added to the
// Gauss-level residual before the transposed interpolation back to the nodes.
//
// What bounds it: LDS passes (busy 62% of the cycles in FP64 at k = 5, 66% in FP32 at k = 3), the
// vector-memory address unit (52% / 31%) and the vector instructions (36% / 58%), each waiting on the
// others between barriers; the address unit had been busy 65 - 70%. x-neighbours of the workgroup's row are therefore read from LDS (their strided
// x-lines cost some 48 address cycles per load), the lanes' rows and columns of Dq come from LDS,
// the face types and indices are 32-bit and the types taken once, and the LDS strides avoid bank
// conflicts (GenLayout): FP64 k = 5 on 48^3 cells 651 -> 569 us (3.4 -> 3.9 TB/s of the 2.2 GB it
// cannot do without), k = 2 on 61 x 47 x 53 167 -> 151 us, FP32 k = 3 on 43 x 37 x 51 89 -> 86 us,
// the FP32 V-cycle of the k = 5 mesh 7.05 -> 6.37 ms, the same bits.

// FP64 at n = 2, 4, 5, 6: one face direction per round, so that the smaller workspace admits another
// workgroup per CU (n = 4 on 64^3 cells 502 -> 449 us, n = 2 on 80^3 185 -> 181; n = 3 818 -> 797 on
// 96^3 but 158 -> 161 on 61 x 47 x 53 and a spill, so it stays)
template<int N, typename Number>
constexpr bool general_single_rounds()
{
  return sizeof(Number) == 8 && N <= 6 && N != 3;
}

// The z derivative of the Gauss values taken after the face phase, so that it is not held
// across the face rounds: it removes the spills of FP32 n = 6 and FP64 n = 6 and lowers the
// register counts (FP64 n = 9 173 -> 132 VGPRs, three waves per SIMD instead of two), 4% for
// the V-cycles of the curved k = 5 hierarchy and 6% for the FP64 k = 5 vmult. FP64 at n = 8
// stays at three waves per SIMD either way and only pays the extra LDS reads (7%), except the
// Chebyshev step, which it brings from two waves to three (k = 7 V-cycle 8% faster).
template<int N, typename Number, ApplyMode mode>
constexpr bool general_late_gz()
{
  return !(sizeof(Number) == 8 && N == 8 && mode != ApplyMode::chebyshev);
}

// LDS strides of a cell: along y (PX) and z (PY) in its tensors, FS from one face array to the
// next, and S from cell to cell. A group of 16 FP64 (32 FP32) lanes is served in one pass if its
// addresses differ modulo 16 (32) entries; these are the strides with the fewest passes over the
// sweeps of the three directions and the face lines that leave the number of workgroups per CU as it
// is (modeled passes per access 1.4 - 2.3, dense 1.4 - 4.3; at FP64 k = 5 27% and at FP32 34% of
// the LDS cycles had been conflicts).
template<int N, typename Number>
struct GenLayout
{
  static constexpr bool dp = sizeof(Number) == 8;
  static constexpr int  PX = N == 4 && !dp ? 5 : N;
  static constexpr int  PY = N == 2 ? 6 : N == 3 ? (dp ? 9 : 13) : N == 4 ? (dp ? 19 : 24) : N == 5 ? 25 :
                             N == 6 ? (dp ? 39 : 37) : N == 7 ? (dp ? 55 : 49) : N == 8 ? (dp ? 65 : 69) : 81;
  static constexpr int  FS = N == 4 ? 17 : N == 5 ? (dp ? 25 : 26) : N == 6 ? (dp ? 39 : 36) :
                             N == 7 ? (dp ? 50 : 49) : N == 8 ? (dp ? 65 : 67) : N == 9 ? 83 : N * N;
  static constexpr int  S  = N == 2 ? (dp ? 44 : 76) : N == 3 ? (dp ? 171 : 181) : N == 4 ? (dp ? 219 : 364) :
                             N == 5 ? (dp ? 377 : 569) : N == 6 ? (dp ? 708 : 804) : N == 7 ? (dp ? 1185 : 1137) :
                             N == 8 ? (dp ? 1559 : 1641) : 2193;
  static constexpr int  PC = (N - 1) * (PX + PY) + N;
  // cell phase: the x and y gradients (the z one stays in registers); face phases: 8 trace
  // arrays per direction, two directions per round (x and y, then z) or one
  static constexpr int faces = (general_single_rounds<N, Number>() ? 8 : 16) * FS;
  static_assert(S >= PC + (2 * PC > faces ? 2 * PC : faces), "cell tensor and workspace");
  // then the table Dq, whose rows and columns the lanes of the face phases index
  static constexpr int size = cells_per_block(N) * S + N * N;
};

// Face terms from the cell's values at the Gauss points. The own traces at the
// face Gauss points are one dot product per end of the lane's d-line of U (the Gauss values, in
// A at this point): u = sum_q l_q(0) U_q, du/dxi_d = sum_q l_q'(0) U_q with l_q the Lagrange
// polynomials on the Gauss points; only the neighbour traces (at the face nodes) need the 2D
// interpolation (S x S). The flux: per face point the traces and normal derivatives of both
// sides (a = J^{-1} n from the per-face data), laplace_operator.h:180-197 with the mirror
// values of weak_boundary_conditions.h on boundary faces; the tangential-gradient tests are
// folded into the value test by Dq^T along the face lines.
// The results end in four scalars per direction for the lane's d-line at Gauss indices (p, q):
// fr[d] = (value test, normal-derivative test) at the lower end, then at the upper end; the
// transposed derivative sweeps add l(0) fr[0] + l'(0) fr[1] + l(1) fr[2] + l'(1) fr[3] to that
// line of the Gauss-level residual. Compared with face rounds after the cell phase on nodal
// traces, this drops the 2D interpolation of the own-side traces and all transposed face
// interpolations; the face arrays of direction j live at W + 8 j N^2.
template<int N, typename Number, ApplyMode mode, int ND>
__device__ __forceinline__ void gauss_faces(int const (&dirs)[ND], SipgArgs<Number> const & a,
                                            int64_t cell, int const (&cc)[3], int types, bool active,
                                            int lt, Number const * U, Number * W, Number const * Dq,
                                            Number const (&nbw)[3][2], Number const (&nbdw)[3][2],
                                            Number (&fr)[3][4])
{
  using L           = GenLayout<N, Number>;
  constexpr int  N2 = N * N, FS = L::FS;
  using T           = GenTable<N>;
  Number const * d0 = a.tables + T::D0;
  Number const * d1 = a.tables + T::D1;
  Number const * SE = a.tables + T::SE;
  Number const * L0 = a.tables + T::L0;
  Number const * L1 = a.tables + T::L1;
  Number const * G0 = a.tables + T::G0;
  Number const * G1 = a.tables + T::G1;
  int const      p = lt % N, q = lt / N;
  auto type = [&](int j, int side) { return (types >> (4 * dirs[j] + 2 * side)) & 3; };
  // F1: own traces at the face Gauss points, neighbour traces at the face nodes
  if(active)
#pragma unroll
    for(int j = 0; j < ND; ++j)
    {
      int const d = dirs[j];
      Number *  E = W + 8 * j * FS;
      int       base, stride;
      line_geometry<N, L::PX, L::PY>(d, p, q, base, stride);
      Number v[N];
      load_line<N>(U + base, stride, v);
      E[0 * FS + lt] = dot_line<N>(L0, v);
      E[1 * FS + lt] = dot_line<N>(G0, v);
      E[4 * FS + lt] = dot_line<N>(L1, v);
      E[5 * FS + lt] = dot_line<N>(G1, v);
      Number nl = 0, dnl = 0, nr = 0, dnr = 0;
      if constexpr(mode != ApplyMode::diagonal)
      {
        if(type(j, 0) == kInterior)
          nl = nbw[d][0], dnl = nbdw[d][0];
        if(type(j, 1) == kInterior)
          nr = nbw[d][1], dnr = nbdw[d][1];
      }
      else
      {
        // probing the cell-local block: neighbours contribute zero, except a cell that is its
        // own periodic neighbour (one cell along d), whose other end then acts as neighbour
        Number u[N];
        line_geometry<N>(d, p, q, base, stride);
        source_line<N, Number, mode>(a.src, cell, base, stride, a.probe, u);
        if(neighbor_id(a.topo, cc, d, 0) == cell)
          nl = u[N - 1], dnl = dot_line<N>(d1, u);
        if(neighbor_id(a.topo, cc, d, 1) == cell)
          nr = u[0], dnr = dot_line<N>(d0, u);
      }
      E[2 * FS + lt] = nl;
      E[3 * FS + lt] = dnl;
      E[6 * FS + lt] = nr;
      E[7 * FS + lt] = dnr;
    }
  __syncthreads();
  // F2/F3: the neighbour arrays (slots 2, 3 of each side) to the face Gauss points
  if(active)
    for(int task = lt; task < 4 * ND * N; task += N2)
    {
      int const which = task / N, r = task % N;
      Number *  arr   = W + (8 * (which >> 2) + 4 * ((which >> 1) & 1) + 2 + (which & 1)) * FS;
      Number    v[N], o[N];
      load_line<N>(arr + N * r, 1, v);
      gen_apply<N, false>(SE, v, o);
      store_line<N>(arr + N * r, 1, o);
    }
  __syncthreads();
  if(active)
    for(int task = lt; task < 4 * ND * N; task += N2)
    {
      int const which = task / N, r = task % N;
      Number *  arr   = W + (8 * (which >> 2) + 4 * ((which >> 1) & 1) + 2 + (which & 1)) * FS;
      Number    v[N], o[N];
      load_line<N>(arr + r, N, v);
      gen_apply<N, false>(SE, v, o);
      store_line<N>(arr + r, N, o);
    }
  __syncthreads();
  // F4: fluxes at the face quadrature points (side s, point lt), held in registers until
  // every lane has read E
  Number res[ND][2][4];
  Number D1[N], D2[N];  // the lane's rows of Dq, then its columns
  load_line<N>(Dq + N * p, 1, D1);
  load_line<N>(Dq + N * q, 1, D2);
  if(active)
#pragma unroll
    for(int j = 0; j < ND; ++j)
#pragma unroll
      for(int s = 0; s < 2; ++s)
      {
        int const d = dirs[j];
        int const t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
        int const qq = lt, q1 = qq % N, q2 = qq / N;
        if(type(j, s) == EXADG_BC_NEUMANN)
        {  // homogeneous Neumann: u+ = u-, du+/dn = -du-/dn -> no contribution
          res[j][s][0] = res[j][s][1] = res[j][s][2] = res[j][s][3] = Number(0);
          continue;
        }
        int const      f  = face_index(a.topo, cc, d, s);
        Number const * fd = a.face_data + (size_t)f * (7 * N2);
        Number         aK[3], aN[3];
#pragma unroll
        for(int c = 0; c < 3; ++c)
        {
          Number const am = fd[c * N2 + qq], ap = fd[(3 + c) * N2 + qq];
          aK[c]           = s ? am : -ap;
          aN[c]           = s ? ap : -am;
        }
        Number const   w   = fd[6 * N2 + qq];
        Number const * Es  = W + 8 * j * FS + s * 4 * FS;
        Number         gt1 = 0, gt2 = 0;
#pragma unroll
        for(int m = 0; m < N; ++m)
        {
          gt1 += D1[m] * Es[m + N * q2];
          gt2 += D2[m] * Es[q1 + N * m];
        }
        Number const u      = Es[qq];
        Number const dudn_K = aK[d] * Es[FS + qq] + aK[t1] * gt1 + aK[t2] * gt2;
        Number       uN, dudn_N;
        if(type(j, s) == kInterior)
        {
          Number g1 = 0, g2 = 0;
#pragma unroll
          for(int m = 0; m < N; ++m)
          {
            g1 += D1[m] * Es[2 * FS + m + N * q2];
            g2 += D2[m] * Es[2 * FS + q1 + N * m];
          }
          uN     = Es[2 * FS + qq];
          dudn_N = aN[d] * Es[3 * FS + qq] + aN[t1] * g1 + aN[t2] * g2;
        }
        else
        {  // homogeneous Dirichlet: u+ = -u-, du+/dn = du-/dn
          uN     = -u;
          dudn_N = dudn_K;
        }
        Number const tau   = a.tau_face[f];
        Number const jump  = u - uN;
        Number const sigma = Number(-0.5) * jump * w;
        res[j][s][0]       = -(Number(0.5) * (dudn_K + dudn_N) - tau * jump) * w;
        res[j][s][1]       = sigma * aK[t1];
        res[j][s][2]       = sigma * aK[t2];
        res[j][s][3]       = sigma * aK[d];
      }
  __syncthreads();
  if(active)
#pragma unroll
    for(int j = 0; j < ND; ++j)
#pragma unroll
      for(int s = 0; s < 2; ++s)
#pragma unroll
        for(int c = 0; c < 4; ++c)
          W[(8 * j + 4 * s + c) * FS + lt] = res[j][s][c];
  __syncthreads();
  // F5: tangential gradient tests folded into the value test (Dq^T); this lane's results
  load_line<N>(Dq + p, N, D1);
  load_line<N>(Dq + q, N, D2);
  if(active)
#pragma unroll
    for(int j = 0; j < ND; ++j)
#pragma unroll
      for(int s = 0; s < 2; ++s)
      {
        int const      qq = lt, q1 = qq % N, q2 = qq / N;
        Number const * R  = W + (8 * j + 4 * s) * FS;
        Number         acc = R[qq];
#pragma unroll
        for(int m = 0; m < N; ++m)
          acc += D1[m] * R[FS + m + N * q2] + D2[m] * R[2 * FS + q1 + N * m];
        fr[dirs[j]][2 * s]     = acc;
        fr[dirs[j]][2 * s + 1] = R[3 * FS + qq];
      }
  __syncthreads();  // W is reused next
}

// Minimum waves per SIMD asked of the compiler for the general kernel, matched to what the
// LDS allows: FP64 at n = 2 five, at n = 3..6 four (n = 5, 6 with one face direction per round, whose
// smaller workspace admits a fourth workgroup per CU: n = 5 8% faster, n = 6 4%); FP32 at n = 3
// eight (<= 64 VGPRs, 19 KB of LDS per workgroup), at n = 4..6 seven (<= 72 VGPRs), at n = 7 six
template<int N, typename Number>
constexpr int general_min_waves()
{
  if constexpr(sizeof(Number) == 8)
    return N == 2 ? 5 : N <= 6 ? 4 : 1;
  else
    return N == 3 ? 8 : (N >= 4 && N <= 6) ? 7 : N == 7 ? 6 : 1;
}

template<int N, typename Number, ApplyMode mode>
__global__ void __launch_bounds__(256)
  __attribute__((amdgpu_waves_per_eu(general_min_waves<N, Number>()))) sipg_general_kernel(SipgArgs<Number> a)
{
  using L           = GenLayout<N, Number>;
  constexpr int  N2 = N * N, N3 = N * N * N, PX = L::PX, PY = L::PY;
  constexpr int  CPB = cells_per_block(N);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Number *       smem = reinterpret_cast<Number *>(smem_raw);
  int const      slot = threadIdx.x / N2;
  int const      lt   = threadIdx.x - slot * N2;
  int const      pos0 = (int)xcd_logical_block(blockIdx.x, gridDim.x) * CPB;
  bool const     active = slot < CPB && pos0 + slot < (int)a.n_cells;
  Number *       A      = smem + (active ? slot : 0) * L::S;
  Number *       W      = A + L::PC;
  Number *       Gx = W, *Gy = W + L::PC;
  Number *       Dq = smem + CPB * L::S;
  Number const * SE  = a.tables + GenTable<N>::SE;
  Number const * DE  = a.tables + GenTable<N>::DE;
  Number const * STE = a.tables + GenTable<N>::STE;
  Number const * DTE = a.tables + GenTable<N>::DTE;
  int const      p = lt % N, q = lt / N;
  // LDS bases of the lane's x-, y- and z-line
  int const      bx = PX * p + PY * q, by = p + PY * q, bz = p + PX * q;
  int            cc[3] = {0, 0, 0};
  if(active)
    traversal_coords(a.topo, a.tile_rows, pos0, slot, cc);
  int64_t const cell  = active ? cell_id(a.topo, cc) : 0;
  int const     types = face_types(a.topo, cc);
  if(threadIdx.x < N2)
    Dq[threadIdx.x] = a.tables[GenTable<N>::DQ + threadIdx.x];
  // x-neighbours in the same workgroup are read from its LDS
  bool const in_block_l = slot > 0 && cc[0] > 0;
  bool const in_block_r = slot + 1 < CPB && cc[0] + 1 < a.topo.nc[0] && pos0 + slot + 1 < (int)a.n_cells;

  // neighbour traces of this lane's line in every direction: value and derivative at the
  // shared face, read up front so that the loads overlap the cell phases
  Number nbw[3][2] = {}, nbdw[3][2] = {};
  auto   load_traces = [&](int d) {
    if constexpr(mode != ApplyMode::diagonal)
      if(active)
      {
        Number const * d0 = a.tables + GenTable<N>::D0;
        Number const * d1 = a.tables + GenTable<N>::D1;
        int            base, stride;
        line_geometry<N>(d, p, q, base, stride);
#pragma unroll
        for(int sd = 0; sd < 2; ++sd)
        {
          int const n_d = a.topo.nc[d], stride_c = d == 0 ? 1 : d == 1 ? a.topo.nc[0] : a.topo.nc[0] * a.topo.nc[1];
          bool const wrap = sd ? cc[d] == n_d - 1 : cc[d] == 0;
          int const  nbc  = (int)cell + (sd ? stride_c : -stride_c) * (wrap ? 1 - n_d : 1);
          bool const read = ((types >> (4 * d + 2 * sd)) & 3) == kInterior &&
                            !(d == 0 && (sd ? in_block_r : in_block_l));
          if(read)
          {
            Number w[N];
            load_line<N>(a.src + (size_t)nbc * N3 + base, stride, w);
            nbw[d][sd]  = sd ? w[0] : w[N - 1];
            nbdw[d][sd] = dot_line<N>(sd ? d0 : d1, w);
          }
        }
      }
  };
  load_traces(0);
  load_traces(1);
  load_traces(2);

  // load the cell values: z-lines of consecutive lanes, consecutive addresses
  if(active)
#pragma unroll
    for(int m = 0; m < N; ++m)
      if constexpr(mode == ApplyMode::diagonal)
        A[bz + PY * m] = (lt + N2 * m == a.probe) ? Number(1) : Number(0);
      else
        A[bz + PY * m] = a.src[cell * N3 + lt + N2 * m];
  __syncthreads();
  // nodal -> Gauss values: x, y sweeps in place; the x-neighbours' traces from their nodal lines
  // before these are overwritten
  {
    Number v[N], o[N];
    if(active)
    {
      if constexpr(mode != ApplyMode::diagonal)
      {
        Number w[N];
        if(in_block_l)
        {
          load_line<N>(A - L::S + bx, 1, w);
          nbw[0][0]  = w[N - 1];
          nbdw[0][0] = dot_line<N>(a.tables + GenTable<N>::D1, w);
        }
        if(in_block_r)
        {
          load_line<N>(A + L::S + bx, 1, w);
          nbw[0][1]  = w[0];
          nbdw[0][1] = dot_line<N>(a.tables + GenTable<N>::D0, w);
        }
      }
      load_line<N>(A + bx, 1, v);
      gen_apply<N, false>(SE, v, o);
    }
    if constexpr(mode != ApplyMode::diagonal)
      __syncthreads();
    if(active)
      store_line<N>(A + bx, 1, o);
  }
  __syncthreads();
  if(active)
  {
    Number v[N], o[N];
    load_line<N>(A + by, PX, v);
    gen_apply<N, false>(SE, v, o);
    store_line<N>(A + by, PX, o);
  }
  __syncthreads();
  // z sweep, then the z derivative at the Gauss points: this lane's z-line (points lt + m N2),
  // kept in registers -- the same lane applies the metric at those points below. With
  // late_gz the derivative is taken after the face phase from the z-line in A instead, so that
  // it is not live across the face rounds (the same values)
  constexpr bool late_gz = general_late_gz<N, Number, mode>();
  Number         gz_line[N];
  if(active)
  {
    Number v[N], o[N];
    load_line<N>(A + bz, PY, v);
    gen_apply<N, false>(SE, v, o);
    store_line<N>(A + bz, PY, o);
    if constexpr(!late_gz)
      gen_apply<N, true>(DE, o, gz_line);
  }
  __syncthreads();
  // the face terms from the Gauss values in A: four result scalars per direction per lane, added
  // by the transposed derivative sweeps below
  Number fr[3][4] = {};
  {
    if constexpr(general_single_rounds<N, Number>())
    {
      int const x[1] = {0}, y[1] = {1}, z[1] = {2};
      gauss_faces<N, Number, mode, 1>(x, a, cell, cc, types, active, lt, A, W, Dq, nbw, nbdw, fr);
      gauss_faces<N, Number, mode, 1>(y, a, cell, cc, types, active, lt, A, W, Dq, nbw, nbdw, fr);
      gauss_faces<N, Number, mode, 1>(z, a, cell, cc, types, active, lt, A, W, Dq, nbw, nbdw, fr);
    }
    else
    {
      int const xy[2] = {0, 1}, z[1] = {2};
      gauss_faces<N, Number, mode, 2>(xy, a, cell, cc, types, active, lt, A, W, Dq, nbw, nbdw, fr);
      gauss_faces<N, Number, mode, 1>(z, a, cell, cc, types, active, lt, A, W, Dq, nbw, nbdw, fr);
    }
  }
  Number const * L0 = a.tables + GenTable<N>::L0;
  Number const * L1 = a.tables + GenTable<N>::L1;
  Number const * G0 = a.tables + GenTable<N>::G0;
  Number const * G1 = a.tables + GenTable<N>::G1;
  // line o of the Gauss-level residual += the face tests of the lane's d-line
  auto add_face_tests = [&](Number(&o)[N], Number const(&f)[4]) {
#pragma unroll
    for(int i = 0; i < N; ++i)
      o[i] += L0[i] * f[0] + G0[i] * f[1] + L1[i] * f[2] + G1[i] * f[3];
  };
  if(active)
  {
    Number v[N], g[N];
    load_line<N>(A + bx, 1, v);
    gen_apply<N, true>(DE, v, g);
    store_line<N>(Gx + bx, 1, g);
    load_line<N>(A + by, PX, v);
    gen_apply<N, true>(DE, v, g);
    store_line<N>(Gy + by, PX, g);
    if constexpr(late_gz)
    {
      load_line<N>(A + bz, PY, v);
      gen_apply<N, true>(DE, v, gz_line);
    }
  }
  __syncthreads();
  // metric: (fx,fy,fz) = G (gx,gy,gz), G symmetric per quadrature point
  if(active)
  {
    Number const * G = a.cell_metric + cell * 6 * N3;
#pragma unroll
    for(int m = 0; m < N; ++m)
    {
      int const    e  = lt + m * N2, l = bz + m * PY;
      Number const gx = Gx[l], gy = Gy[l], gz = gz_line[m];
      Number const g00 = G[e], g11 = G[N3 + e], g22 = G[2 * N3 + e];
      Number const g01 = G[3 * N3 + e], g02 = G[4 * N3 + e], g12 = G[5 * N3 + e];
      Gx[l]            = g00 * gx + g01 * gy + g02 * gz;
      Gy[l]            = g01 * gx + g11 * gy + g12 * gz;
      gz_line[m]       = g02 * gx + g12 * gy + g22 * gz;
    }
  }
  __syncthreads();
  // transposed derivative sweeps summed into A, then S^T back to nodal values
  if(active)
  {
    Number v[N], o[N];
    load_line<N>(Gx + bx, 1, v);
    gen_apply<N, true>(DTE, v, o);
    add_face_tests(o, fr[0]);
    store_line<N>(A + bx, 1, o);
  }
  __syncthreads();
  if(active)
  {
    Number v[N], o[N], w[N];
    load_line<N>(Gy + by, PX, v);
    gen_apply<N, true>(DTE, v, o);
    add_face_tests(o, fr[1]);
    load_line<N>(A + by, PX, w);
#pragma unroll
    for(int i = 0; i < N; ++i)
      w[i] += o[i];
    store_line<N>(A + by, PX, w);
  }
  __syncthreads();
  if(active)
  {
    Number o[N], w[N];
    gen_apply<N, true>(DTE, gz_line, o);
    add_face_tests(o, fr[2]);
    load_line<N>(A + bz, PY, w);
#pragma unroll
    for(int i = 0; i < N; ++i)
      w[i] += o[i];
    gen_apply<N, false>(STE, w, o);
    store_line<N>(A + bz, PY, o);
  }
  __syncthreads();
  if(active)
  {
    Number v[N], o[N];
    load_line<N>(A + by, PX, v);
    gen_apply<N, false>(STE, v, o);
    store_line<N>(A + by, PX, o);
  }
  __syncthreads();
  if(active)
  {
    Number v[N], o[N];
    load_line<N>(A + bx, 1, v);
    gen_apply<N, false>(STE, v, o);
    store_line<N>(A + bx, 1, o);
  }
  __syncthreads();

  if constexpr(mode == ApplyMode::residual_restrict)
  {
    // r = rhs - A u in A, then the three transposed interpolation sweeps x, y, z of the
    // restriction through the workspace; the coarse cell's values are added to dst
    int const      nc = a.restrict_nc;
    Number const * P  = a.restrict_P;  // P[i nc + c]: fine node i, coarse node c
    Number *       W1 = W;             // nc x N x N
    Number *       W2 = W + L::PC;     // nc x nc x N
    if(active)
#pragma unroll
      for(int m = 0; m < N; ++m)
        A[bz + PY * m] = a.rhs[cell * N3 + lt + N2 * m] - A[bz + PY * m];
    __syncthreads();
    if(active)
    {
      int const j = lt % N, k = lt / N;  // x-line (j, k)
      for(int c = 0; c < nc; ++c)
      {
        Number s = 0;
#pragma unroll
        for(int i = 0; i < N; ++i)
          s += P[i * nc + c] * A[i + PX * j + PY * k];
        W1[c + nc * (j + N * k)] = s;
      }
    }
    __syncthreads();
    if(active && lt < nc * N)
    {
      int const c0 = lt % nc, k = lt / nc;  // y-line (c0, k)
      for(int c1 = 0; c1 < nc; ++c1)
      {
        Number s = 0;
#pragma unroll
        for(int j = 0; j < N; ++j)
          s += P[j * nc + c1] * W1[c0 + nc * (j + N * k)];
        W2[c0 + nc * (c1 + nc * k)] = s;
      }
    }
    __syncthreads();
    if(active && lt < nc * nc)
    {
      int const     c0 = lt % nc, c1 = lt / nc;  // z-line (c0, c1)
      int64_t const nc3 = (int64_t)nc * nc * nc;
      for(int c2 = 0; c2 < nc; ++c2)
      {
        Number s = 0;
#pragma unroll
        for(int k = 0; k < N; ++k)
          s += P[k * nc + c2] * W2[c0 + nc * (c1 + nc * k)];
        a.dst[cell * nc3 + c0 + nc * (c1 + nc * c2)] += s;
      }
    }
    return;
  }
  if(active)
#pragma unroll
    for(int m = 0; m < N; ++m)
    {
      int const     e  = lt + N2 * m;
      size_t const  g  = (size_t)cell * N3 + e;
      Number const  ax = A[bz + PY * m];
      if constexpr(mode == ApplyMode::diagonal)
      {
        if(a.block)
          a.dst[((size_t)cell * N3 + a.probe) * N3 + e] = ax;
        else if(e == a.probe)
          a.dst[g] = ax;
      }
      else if constexpr(mode == ApplyMode::vmult_add)
        a.dst[g] += ax;
      else if constexpr(mode == ApplyMode::residual)
        a.dst[g] = a.rhs[g] - ax;
      else if constexpr(mode == ApplyMode::chebyshev)
      {
        Number v = (Number(1) + a.f1) * a.src[g] + a.f2 * a.dinv[g] * (a.rhs[g] - ax);
        if(a.has_old)
          v -= a.f1 * a.x_old[g];
        a.dst[g] = v;
      }
      else
        a.dst[g] = ax;
    }
}

template<int N, typename Number, ApplyMode mode>
hipError_t launch_general_n(SipgArgs<Number> const & a, hipStream_t stream)
{
  constexpr int CPB    = cells_per_block(N);
  int const     blocks = (int)((a.n_cells + CPB - 1) / CPB);
  size_t const  lds    = sizeof(Number) * GenLayout<N, Number>::size;
  // set once per instantiation; concurrent first calls may both set it, which is harmless
  static std::atomic<bool> attr{false};
  if(lds > 65536 && !attr.load(std::memory_order_acquire))
  {
    hipError_t e = hipFuncSetAttribute((void const *)sipg_general_kernel<N, Number, mode>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if(e != hipSuccess)
      return e;
    attr.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL((sipg_general_kernel<N, Number, mode>), dim3(blocks), dim3(256), lds, stream, a);
  return hipGetLastError();
}

template<typename Number, ApplyMode mode>
hipError_t dispatch_general(int degree, SipgArgs<Number> const & a, hipStream_t s)
{
  switch(degree)
  {
    case 1: return launch_general_n<2, Number, mode>(a, s);
    case 2: return launch_general_n<3, Number, mode>(a, s);
    case 3: return launch_general_n<4, Number, mode>(a, s);
    case 4: return launch_general_n<5, Number, mode>(a, s);
    case 5: return launch_general_n<6, Number, mode>(a, s);
    case 6: return launch_general_n<7, Number, mode>(a, s);
    case 7: return launch_general_n<8, Number, mode>(a, s);
    case 8: return launch_general_n<9, Number, mode>(a, s);
    default: return hipErrorInvalidValue;
  }
}

// diagonal entry i of the 1D cell-local line operator along a direction of width h: the line
// Laplacian of the Cartesian kernel applied to the unit vector e_i, with the exterior trace of
// weak_boundary_conditions.h on boundary faces (type_l/type_r EXADG_BC_*), zero across interior
// faces, or the cell's own opposite end across the periodic faces of a one-cell direction (self)
__device__ inline double line_diagonal(double const * t, int n, int i, double h, int type_l,
                                       int type_r, bool self, double tau_l, double tau_r)
{
  double const * M = t;
  double const * K = t + n;
  double const * d0 = t + 2 * n;
  double const * d1 = t + 3 * n;
  (void)M;
  double const u0 = i == 0 ? 1.0 : 0.0, un = i == n - 1 ? 1.0 : 0.0;
  double const du0 = d0[i], du1 = d1[i];
  double       wl = 0, dwl = 0, wr = 0, dwr = 0;
  if(type_l == EXADG_BC_DIRICHLET)
    wl = -u0, dwl = du0;
  else if(type_l == EXADG_BC_NEUMANN)
    wl = u0, dwl = -du0;
  else if(self)
    wl = un, dwl = du1;
  if(type_r == EXADG_BC_DIRICHLET)
    wr = -un, dwr = du1;
  else if(type_r == EXADG_BC_NEUMANN)
    wr = un, dwr = -du1;
  else if(self)
    wr = u0, dwr = du0;
  double const jl = 0.5 * (u0 - wl), jr = 0.5 * (un - wr);
  double       o  = (K[i] + d0[i] * jl - d1[i] * jr) / h;
  if(i == 0)
    o += 0.5 * (du0 + dwl) / h + 2.0 * tau_l * jl;
  if(i == n - 1)
    o += 2.0 * tau_r * jr - 0.5 * (du1 + dwr) / h;
  return o;
}

template<typename Number>
__global__ void __launch_bounds__(256)
  cartesian_diagonal_kernel(Number * diag, double const * t, Number const * tau_face,
                            BoxTopology topo, double h0, double h1, double h2, int n,
                            int64_t n_dofs)
{
  int64_t const g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(g >= n_dofs)
    return;
  int const     n3   = n * n * n;
  int64_t const cell = g / n3;
  int const     e    = (int)(g - cell * n3);
  int const     id[3] = {e % n, (e / n) % n, e / (n * n)};
  int           cc[3];
  cell_coords(topo, cell, cc);
  double const h[3] = {h0, h1, h2};
  double       L[3], m[3];
#pragma unroll
  for(int d = 0; d < 3; ++d)
  {
    int const  n_d = topo.nc[d], per = topo.periodic[d];
    int const  t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
    bool const has_l = cc[d] > 0 || per, has_r = cc[d] < n_d - 1 || per;
    bool const self  = per && n_d == 1;
    int64_t const fbase = topo.face_base[d] + (int64_t)topo.layers[d] * (cc[t1] + (int64_t)topo.nc[t1] * cc[t2]);
    int const     fr    = (per && cc[d] + 1 == n_d) ? 0 : cc[d] + 1;
    int const     tl = has_l ? -1 : topo.bc[2 * d], tr = has_r ? -1 : topo.bc[2 * d + 1];
    L[d] = line_diagonal(t, n, id[d], h[d], tl, tr, self, (double)tau_face[fbase + cc[d]],
                         (double)tau_face[fbase + fr]);
    m[d] = h[d] * t[id[d]];
  }
  diag[g] = (Number)(L[0] * m[1] * m[2] + m[0] * L[1] * m[2] + m[0] * m[1] * L[2]);
}
template<int N, typename Number>
__global__ void __launch_bounds__(256)
  general_diagonal_kernel(Number * diag, double const * __restrict__ t1d, SipgArgs<Number> a)
{
  constexpr int  N2 = N * N, N3 = N * N * N;
  constexpr int  CPB = cells_per_block(N);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *       smem   = reinterpret_cast<double *>(smem_raw);
  int const      slot   = threadIdx.x / N2;
  int const      lt     = threadIdx.x - slot * N2;
  int const      pos0   = (int)xcd_logical_block(blockIdx.x, gridDim.x) * CPB;
  bool const     active = slot < CPB && pos0 + slot < (int)a.n_cells;
  double *       W1     = smem + (active ? slot : 0) * 2 * N3;
  double *       W2     = W1 + N3;
  double const * SS = t1d, *DD = t1d + N2, *SD = t1d + 2 * N2;
  int const      p = lt % N, q = lt / N;
  int            cc[3] = {0, 0, 0};
  if(active)
    traversal_coords(a.topo, a.tile_rows, pos0, slot, cc);
  int64_t const cell = active ? cell_id(a.topo, cc) : 0;
  double        acc[N];
#pragma unroll
  for(int m = 0; m < N; ++m)
    acc[m] = 0;
  // cell term: component c of G (g00, g11, g22, g01, g02, g12) against tables per direction
  for(int term = 0; term < 6; ++term)
  {
    int const      c  = term;
    double const * T0 = term == 0 ? DD : (term == 3 || term == 4) ? SD : SS;
    double const * T1 = term == 1 ? DD : (term == 3 || term == 5) ? SD : SS;
    double const * T2 = term == 2 ? DD : (term == 4 || term == 5) ? SD : SS;
    double const   f  = term < 3 ? 1.0 : 2.0;
    if(active)
    {
      Number const * G = a.cell_metric + cell * 6 * N3 + (int64_t)c * N3 + N * (p + N * q);
      double         g[N];
#pragma unroll
      for(int q0 = 0; q0 < N; ++q0)
        g[q0] = (double)G[q0];
#pragma unroll
      for(int i0 = 0; i0 < N; ++i0)
      {
        double s = 0;
#pragma unroll
        for(int q0 = 0; q0 < N; ++q0)
          s += T0[q0 * N + i0] * g[q0];
        W1[i0 + N * (p + N * q)] = s;  // (i0, q1 = p, q2 = q)
      }
    }
    __syncthreads();
    if(active)
    {
      double v[N];
#pragma unroll
      for(int q1 = 0; q1 < N; ++q1)
        v[q1] = W1[p + N * (q1 + N * q)];  // (i0 = p, q1, q2 = q)
#pragma unroll
      for(int i1 = 0; i1 < N; ++i1)
      {
        double s = 0;
#pragma unroll
        for(int q1 = 0; q1 < N; ++q1)
          s += T1[q1 * N + i1] * v[q1];
        W2[p + N * (i1 + N * q)] = s;
      }
    }
    __syncthreads();
    if(active)
    {
      double v[N];
#pragma unroll
      for(int q2 = 0; q2 < N; ++q2)
        v[q2] = W2[p + N * (q + N * q2)];  // (i0 = p, i1 = q, q2)
#pragma unroll
      for(int i2 = 0; i2 < N; ++i2)
      {
        double s = 0;
#pragma unroll
        for(int q2 = 0; q2 < N; ++q2)
          s += T2[q2 * N + i2] * v[q2];
        acc[i2] += f * s;
      }
    }
  }
  // face terms of the face-layer DoFs
  if(active)
  {
    double const lp[2] = {t1d[3 * N2], t1d[3 * N2 + 1]};  // l'(0) of node 0, l'(1) of node N-1
#pragma unroll
    for(int d = 0; d < 3; ++d)
#pragma unroll
      for(int s = 0; s < 2; ++s)
      {
        int const end = s ? N - 1 : 0;
        // this lane's DoFs on the face: (i_t1, i_t2) and the slot m of its z-line
        int it1, it2, mfix = -1;
        if(d == 0)
        {
          if(p != end)
            continue;
          it1 = q;  // i1, and i2 runs over m
          it2 = -1;
        }
        else if(d == 1)
        {
          if(q != end)
            continue;
          it1 = p;  // i0, and i2 runs over m
          it2 = -1;
        }
        else
        {
          it1  = p;
          it2  = q;
          mfix = end;
        }
        int64_t const nb = neighbor_id(a.topo, cc, d, s);
        int const     type = nb >= 0 ? kInterior : a.topo.bc[2 * d + s];
        double const  cf   = type == kInterior ? 1.0 : type == EXADG_BC_DIRICHLET ? 2.0 : 0.0;
        if(cf == 0.0)
          continue;
        int const      t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
        int64_t const  fid = face_id(a.topo, cc, d, s);
        Number const * fd  = a.face_data + fid * 7 * N2;
        double const   tau = (double)a.tau_face[fid];
        // out(i_t1, i_t2) = sum_{q1,q2} CA SS SS + CB SD SS + CC SS SD
        double out[N];
#pragma unroll
        for(int m = 0; m < N; ++m)
          out[m] = 0;
        for(int q2 = 0; q2 < N; ++q2)
        {
          double rA = 0, rB = 0, rC = 0;  // sum over q1 with the it1 tables
#pragma unroll
          for(int q1 = 0; q1 < N; ++q1)
          {
            int const    qq = q1 + N * q2;
            double const am_d = (double)fd[d * N2 + qq], ap_d = (double)fd[(3 + d) * N2 + qq];
            double const am_1 = (double)fd[t1 * N2 + qq], ap_1 = (double)fd[(3 + t1) * N2 + qq];
            double const am_2 = (double)fd[t2 * N2 + qq], ap_2 = (double)fd[(3 + t2) * N2 + qq];
            double const ad = s ? am_d : -ap_d, a1 = s ? am_1 : -ap_1, a2 = s ? am_2 : -ap_2;
            double const w  = (double)fd[6 * N2 + qq];
            double const CA = cf * w * (tau - ad * lp[s]);
            double const CB = -cf * w * a1;
            double const CC = -cf * w * a2;
            rA += CA * SS[q1 * N + it1];
            rB += CB * SD[q1 * N + it1];
            rC += CC * SS[q1 * N + it1];
          }
          if(mfix >= 0)
            out[mfix] += (rA + rB) * SS[q2 * N + it2] + rC * SD[q2 * N + it2];
          else
#pragma unroll
            for(int m = 0; m < N; ++m)
              out[m] += (rA + rB) * SS[q2 * N + m] + rC * SD[q2 * N + m];
        }
#pragma unroll
        for(int m = 0; m < N; ++m)
          acc[m] += out[m];
      }
#pragma unroll
    for(int m = 0; m < N; ++m)
      diag[cell * N3 + p + N * q + N2 * m] = (Number)acc[m];
  }
}

template<int N, typename Number>
hipError_t launch_general_diagonal_n(Number * diag, double const * t1d, SipgArgs<Number> const & a,
                                     hipStream_t stream)
{
  constexpr int CPB    = cells_per_block(N);
  int const     blocks = (int)((a.n_cells + CPB - 1) / CPB);
  size_t const  lds    = sizeof(double) * CPB * 2 * N * N * N;
  static std::atomic<bool> attr{false};
  if(lds > 65536 && !attr.load(std::memory_order_acquire))
  {
    hipError_t e = hipFuncSetAttribute((void const *)general_diagonal_kernel<N, Number>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if(e != hipSuccess)
      return e;
    attr.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL((general_diagonal_kernel<N, Number>), dim3(blocks), dim3(256), lds, stream,
                     diag, t1d, a);
  return hipGetLastError();
}
}  // namespace

template<typename Number>
hipError_t launch_sipg_general(int degree, ApplyMode mode, SipgArgs<Number> const & a,
                               hipStream_t s)
{
  switch(mode)
  {
    case ApplyMode::vmult: return dispatch_general<Number, ApplyMode::vmult>(degree, a, s);
    case ApplyMode::vmult_add: return dispatch_general<Number, ApplyMode::vmult_add>(degree, a, s);
    case ApplyMode::diagonal: return dispatch_general<Number, ApplyMode::diagonal>(degree, a, s);
    case ApplyMode::chebyshev: return dispatch_general<Number, ApplyMode::chebyshev>(degree, a, s);
    case ApplyMode::residual: return dispatch_general<Number, ApplyMode::residual>(degree, a, s);
    case ApplyMode::residual_restrict:
      if(a.restrict_P == nullptr || a.restrict_nc < 1 || a.restrict_nc > degree + 1)
        return hipErrorInvalidValue;
      return dispatch_general<Number, ApplyMode::residual_restrict>(degree, a, s);
  }
  return hipErrorInvalidValue;
}

template<typename Number>
hipError_t launch_cartesian_diagonal(Number * diag, double const * diag1d, Number const * tau_face,
                                     BoxTopology const & topo, double const (&h)[3], int n,
                                     int64_t n_cells, hipStream_t stream)
{
  int64_t const n_dofs = n_cells * n * n * n;
  if(n_dofs == 0)
    return hipSuccess;
  int64_t const blocks = (n_dofs + 255) / 256;
  hipLaunchKernelGGL((cartesian_diagonal_kernel<Number>), dim3((unsigned)blocks), dim3(256), 0,
                     stream, diag, diag1d, tau_face, topo, h[0], h[1], h[2], n, n_dofs);
  return hipGetLastError();
}

template<typename Number>
hipError_t launch_general_diagonal(Number * diag, double const * tab1d, SipgArgs<Number> const & a,
                                   int degree, hipStream_t stream)
{
  switch(degree)
  {
    case 1: return launch_general_diagonal_n<2, Number>(diag, tab1d, a, stream);
    case 2: return launch_general_diagonal_n<3, Number>(diag, tab1d, a, stream);
    case 3: return launch_general_diagonal_n<4, Number>(diag, tab1d, a, stream);
    case 4: return launch_general_diagonal_n<5, Number>(diag, tab1d, a, stream);
    case 5: return launch_general_diagonal_n<6, Number>(diag, tab1d, a, stream);
    case 6: return launch_general_diagonal_n<7, Number>(diag, tab1d, a, stream);
    case 7: return launch_general_diagonal_n<8, Number>(diag, tab1d, a, stream);
    case 8: return launch_general_diagonal_n<9, Number>(diag, tab1d, a, stream);
    default: return hipErrorInvalidValue;
  }
}

template hipError_t launch_general_diagonal<double>(double *, double const *,
                                                    SipgArgs<double> const &, int, hipStream_t);
template hipError_t launch_general_diagonal<float>(float *, double const *,
                                                   SipgArgs<float> const &, int, hipStream_t);
template hipError_t launch_cartesian_diagonal<double>(double *, double const *, double const *,
                                                      BoxTopology const &, double const (&)[3], int,
                                                      int64_t, hipStream_t);
template hipError_t launch_cartesian_diagonal<float>(float *, double const *, float const *,
                                                     BoxTopology const &, double const (&)[3], int,
                                                     int64_t, hipStream_t);
template hipError_t launch_sipg_general<double>(int, ApplyMode, SipgArgs<double> const &, hipStream_t);
template hipError_t launch_sipg_general<float>(int, ApplyMode, SipgArgs<float> const &, hipStream_t);

}  // namespace ExaDG
