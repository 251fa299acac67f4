// Weak DG divergence of a discrete velocity, one workgroup per cell (divergence_operator.cpp
// :168-298, weak form). The velocity goes to the Gauss points of QGauss(k_u+1) by three S
// sweeps per component in LDS, the reference-gradient data -C u (C = JxW J^{-1}) is tested with
// the pressure basis at those points, and each face adds the central flux of the own end node
// layer and the neighbour's opposite layer, interpolated to the face points. Element-centric:
// every face is evaluated from both cells and every pressure entry is written once.
#include <hip/hip_runtime.h>

#include "../../include/exadg_amd.h"
#include "divergence_kernels.h"

namespace ExaDG
{
namespace
{
constexpr int kThreads = 256;

// out[i + m0 (j + m1 k)] for in[a + n0 (b + n1 c)] with one matrix along one direction:
// along direction `dir` apply M (rows: output index, m_out x m_in, M[o * m_in + a]), the
// other two directions copied
__device__ __forceinline__ void sweep(double const * M, int m_out, int m_in, int dir, int const (&ext_in)[3],
                      double const * in, double * out, bool transpose)
{
  int ext_out[3] = {ext_in[0], ext_in[1], ext_in[2]};
  ext_out[dir]   = m_out;
  int const total = ext_out[0] * ext_out[1] * ext_out[2];
  for(int e = threadIdx.x; e < total; e += kThreads)
  {
    int idx[3] = {e % ext_out[0], (e / ext_out[0]) % ext_out[1], e / (ext_out[0] * ext_out[1])};
    int const o = idx[dir];
    double    s = 0;
    for(int a = 0; a < m_in; ++a)
    {
      idx[dir]       = a;
      double const m = transpose ? M[a * m_out + o] : M[o * m_in + a];
      s += m * in[idx[0] + ext_in[0] * (idx[1] + ext_in[1] * idx[2])];
    }
    out[e] = s;
  }
}

// NU, NP: nodes per direction of velocity and pressure, or 0 to take them from the arguments. With
// the sizes known the index arithmetic of the sweeps (a dozen divisions per entry otherwise) folds
// away.
template<int NU, int NP>
__global__ void __launch_bounds__(kThreads) divergence_apply_kernel(DivergenceArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int const      nu = NU ? NU : a.n_u, np = NP ? NP : a.n_p;
  int const      nu2 = nu * nu, nu3 = nu2 * nu, np3 = np * np * np;
  double *       U   = reinterpret_cast<double *>(smem_raw);  // 3 nu^3 velocity, then Gauss data
  double *       T0  = U + 3 * nu3;                            // nu^3
  double *       T1  = T0 + nu3;                               // nu^3
  double *       O   = T1 + nu3;                               // np^3 result
  double *       Fm  = O + np3;                                // 3 nu^2 own face values
  double *       Fp  = Fm + 3 * nu2;                           // 3 nu^2 neighbour face values
  double *       Ft  = Fp + 3 * nu2;                           // nu^2 face flux
  double *       Fs  = Ft + nu2;                               // 6 nu^2 face scratch
  double const * Su  = a.tables;
  double const * Sp  = Su + nu2;
  double const * Sdp = Sp + nu * np;
  int64_t const  c   = blockIdx.x;
  int            cc[3];
  cell_coords(a.topo, c, cc);

  for(int e = threadIdx.x; e < 3 * nu3; e += kThreads)
    U[e] = a.src[c * 3 * nu3 + e];
  __syncthreads();
  int const full[3] = {nu, nu, nu};
  // velocity at the Gauss points, component by component (in place through T0, T1)
  for(int k = 0; k < 3; ++k)
  {
    sweep(Su, nu, nu, 0, full, U + k * nu3, T0, false);
    __syncthreads();
    sweep(Su, nu, nu, 1, full, T0, T1, false);
    __syncthreads();
    sweep(Su, nu, nu, 2, full, T1, T0, false);
    __syncthreads();
    for(int e = threadIdx.x; e < nu3; e += kThreads)
      U[k * nu3 + e] = T0[e];
    __syncthreads();
  }
  // F_j = -sum_k C[j][k] u_k (reference-gradient data), overwriting U
  double const * cg = a.cell_geo + c * 12 * nu3;
  for(int q = threadIdx.x; q < nu3; q += kThreads)
  {
    double const u0 = U[q], u1 = U[nu3 + q], u2 = U[2 * nu3 + q];
    double       f[3];
    for(int j = 0; j < 3; ++j)
      f[j] = -(cg[(3 + 3 * j) * nu3 + q] * u0 + cg[(4 + 3 * j) * nu3 + q] * u1 +
               cg[(5 + 3 * j) * nu3 + q] * u2);
    U[q] = f[0], U[nu3 + q] = f[1], U[2 * nu3 + q] = f[2];
  }
  for(int e = threadIdx.x; e < np3; e += kThreads)
    O[e] = 0.0;
  __syncthreads();
  // O += sum_j (D_j)^T F_j: along direction j the derivative table, otherwise values
  for(int j = 0; j < 3; ++j)
  {
    int       ext[3] = {nu, nu, nu};
    double *  in     = U + j * nu3;
    double *  bufs[2] = {T0, T1};
    double *  cur    = in;
    for(int d = 0; d < 3; ++d)
    {
      double * out = (d == 2) ? T0 : bufs[(d + 1) % 2];
      if(d == 2 && cur == T0)
        out = T1;
      sweep(d == j ? Sdp : Sp, np, nu, d, ext, cur, out, true);
      ext[d] = np;
      __syncthreads();
      cur = out;
    }
    for(int e = threadIdx.x; e < np3; e += kThreads)
      O[e] += cur[e];
    __syncthreads();
  }

  // faces
  for(int d = 0; d < 3; ++d)
    for(int sd = 0; sd < 2; ++sd)
    {
      int64_t const nb = neighbor_id(a.topo, cc, d, sd);
      bool const    interior = nb >= 0;
      if(!interior && a.topo.bc[2 * d + sd] != EXADG_BC_DIRICHLET)
        continue;  // wall at rest: u+ = -u-, the central flux vanishes
      int const t1 = tangent1(d), t2 = tangent2(d);
      // end node layers: own at sd, neighbour at 1 - sd; indices (t1 fastest) -> Fm / Fp
      for(int e = threadIdx.x; e < 3 * nu2; e += kThreads)
      {
        int const k = e / nu2, r = e % nu2, i1 = r % nu, i2 = r / nu;
        int       idx[3];
        idx[t1]   = i1;
        idx[t2]   = i2;
        idx[d]    = sd ? nu - 1 : 0;
        int const own = idx[0] + nu * (idx[1] + nu * idx[2]);
        Fm[e]     = a.src[c * 3 * nu3 + k * nu3 + own];
        if(interior)
        {
          idx[d]      = sd ? 0 : nu - 1;
          int const o2 = idx[0] + nu * (idx[1] + nu * idx[2]);
          Fp[e]        = a.src[nb * 3 * nu3 + k * nu3 + o2];
        }
      }
      __syncthreads();
      // tangential interpolation of the 3 (or 6) layers: along t1, then t2
      int const nl = interior ? 6 : 3;
      for(int e = threadIdx.x; e < nl * nu2; e += kThreads)
      {
        int const  l = e / nu2, r = e % nu2, q1 = r % nu, i2 = r / nu;
        double *   L = (l < 3 ? Fm + l * nu2 : Fp + (l - 3) * nu2);
        double     s = 0;
        for(int i1 = 0; i1 < nu; ++i1)
          s += Su[q1 * nu + i1] * L[i1 + nu * i2];
        Fs[e] = s;
      }
      __syncthreads();
      for(int e = threadIdx.x; e < nl * nu2; e += kThreads)
      {
        int const l = e / nu2, r = e % nu2, q1 = r % nu, q2 = r / nu;
        double    s = 0;
        for(int i2 = 0; i2 < nu; ++i2)
          s += Su[q2 * nu + i2] * Fs[l * nu2 + q1 + nu * i2];
        (l < 3 ? Fm + l * nu2 : Fp + (l - 3) * nu2)[q1 + nu * q2] = s;
      }
      __syncthreads();
      double const * fg = a.face_geo + face_id(a.topo, cc, d, sd) * 6 * nu2;
      double const   sg = sd ? 1.0 : -1.0;  // own outward normal = sg n
      for(int q = threadIdx.x; q < nu2; q += kThreads)
      {
        double f = 0;
        for(int k = 0; k < 3; ++k)
        {
          double const v = interior ? 0.5 * (Fm[k * nu2 + q] + Fp[k * nu2 + q]) : Fm[k * nu2 + q];
          f += v * fg[(3 + k) * nu2 + q];
        }
        Ft[q] = sg * f;
      }
      __syncthreads();
      // pressure test: the end node layer along d, Sp tangentially
      for(int e = threadIdx.x; e < np * np; e += kThreads)
      {
        int const i1 = e % np, i2 = e / np;
        double    s  = 0;
        for(int q2 = 0; q2 < nu; ++q2)
        {
          double t = 0;
          for(int q1 = 0; q1 < nu; ++q1)
            t += Sp[q1 * np + i1] * Ft[q1 + nu * q2];
          s += Sp[q2 * np + i2] * t;
        }
        int idx[3];
        idx[d]  = sd ? np - 1 : 0;
        idx[t1] = i1;
        idx[t2] = i2;
        O[idx[0] + np * (idx[1] + np * idx[2])] += s;
      }
      __syncthreads();
    }
  for(int e = threadIdx.x; e < np3; e += kThreads)
    a.dst[c * np3 + e] = O[e];
}

// Affine boxes: the weak divergence is a sum of Kronecker products, one per velocity component,
//   b = M_z M_y (G_x u_x) + M_x (M_z (G_y u_y) + M_y (G_z u_z)),
// M_d = h_d M the rectangular mass matrix of pressure and velocity and G_d along the component's own
// direction: -int phi_i' psi_j and the central flux at both ends, half of the own end value and
// half of the neighbour's (all of the own one at an outflow, none at a wall). One group of n_u^2
// lanes per cell, a line per lane; lines are contracted in place (a buffer line holds n_u or n_p
// entries): G along x, y and z; M along y and z; M along z and x; the sum. No geometry is read.
// Bound by HBM (the velocity in, the pressure out) and the LDS passes of the eight sweeps: k_u = 5,
// k_p = 4 on 32^3 cells 56 us (3.7 TB/s of the 203 MB), the general kernel with its 0.9 GB of point
// data 855 us.
template<int NU, int NP>
__global__ void __launch_bounds__(kThreads) divergence_affine_kernel(DivergenceAffineArgs a)
{
  constexpr int NU2 = NU * NU, NU3 = NU2 * NU, NP3 = NP * NP * NP;
  constexpr int M  = NU > NP ? NU : NP;
  constexpr int PY = M, PZ = M * M | 1, PC = PZ * (M - 1) + M * M;  // odd plane stride
  constexpr int CPB = kThreads / NU2;
  __shared__ double smem[CPB * 3 * PC];
  int const         slot = threadIdx.x / NU2, lt = threadIdx.x - slot * NU2;
  int64_t const     c      = xcd_logical_block(blockIdx.x, gridDim.x) * CPB + slot;
  bool const        active = slot < CPB && c < a.n_cells;
  double *          T[3];
#pragma unroll
  for(int k = 0; k < 3; ++k)
    T[k] = smem + ((active ? slot : 0) * 3 + k) * PC;
  double ends[3][2], we[3][2];  // neighbour's end value of this lane's line; weight of the own one
  if(active)
  {
    double const * u = a.src + c * 3 * NU3;
#pragma unroll
    for(int k = 0; k < 3; ++k)
#pragma unroll
      for(int z = 0; z < NU; ++z)
        T[k][lt % NU + PY * (lt / NU) + PZ * z] = u[k * NU3 + lt + NU2 * z];
    int cc[3];
    cell_coords(a.topo, c, cc);
#pragma unroll
    for(int d = 0; d < 3; ++d)
#pragma unroll
      for(int s = 0; s < 2; ++s)
      {
        int64_t const nb   = neighbor_id(a.topo, cc, d, s);
        int const     p = lt % NU, q = lt / NU, end = s ? 0 : NU - 1;
        int const     at = d == 0 ? end + NU * lt : d == 1 ? p + NU * end + NU2 * q : lt + NU2 * end;
        ends[d][s] = nb >= 0 ? 0.5 * a.src[(nb * 3 + d) * NU3 + at] : 0.0;
        we[d][s]   = nb >= 0 ? 0.5 : a.topo.bc[2 * d + s] == EXADG_BC_DIRICHLET ? 1.0 : 0.0;
      }
  }
  __syncthreads();
  if(active)
  {
    int const p = lt % NU, q = lt / NU;
#pragma unroll
    for(int d = 0; d < 3; ++d)
    {
      int const base = d == 0 ? PY * p + PZ * q : d == 1 ? p + PZ * q : p + PY * q;
      int const st   = d == 0 ? 1 : d == 1 ? PY : PZ;
      double    v[NU];
#pragma unroll
      for(int i = 0; i < NU; ++i)
        v[i] = T[d][base + i * st];
      double const lo = we[d][0] * v[0] + ends[d][0], up = we[d][1] * v[NU - 1] + ends[d][1];
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        double s = 0;
#pragma unroll
        for(int j = 0; j < NU; ++j)
          s += a.G[i * NU + j] * v[j];
        if(i == 0)
          s -= lo;
        if(i == NP - 1)
          s += up;
        T[d][base + i * st] = a.area[d] * s;
      }
    }
  }
  __syncthreads();
  // T <- M T along one direction, for the lines of e0 x e1 entries of the two others
  auto mass = [&](double const * in, double const * in2, double * out, int d, int e0, int e1) {
    for(int t = lt; t < e0 * e1; t += NU2)
    {
      int const p = t % e0, q = t / e0;
      int const base = d == 0 ? PY * p + PZ * q : d == 1 ? p + PZ * q : p + PY * q;
      int const st   = d == 0 ? 1 : d == 1 ? PY : PZ;
      double    v[NU];
#pragma unroll
      for(int i = 0; i < NU; ++i)
        v[i] = in2 ? in[base + i * st] + in2[base + i * st] : in[base + i * st];
#pragma unroll
      for(int i = 0; i < NP; ++i)
      {
        double s = 0;
#pragma unroll
        for(int j = 0; j < NU; ++j)
          s += a.M[i * NU + j] * v[j];
        out[base + i * st] = s;
      }
    }
  };
  if(active)
  {
    mass(T[0], nullptr, T[0], 1, NP, NU);  // (i0, z)
    mass(T[2], nullptr, T[2], 1, NU, NP);  // (x, i2)
    mass(T[1], nullptr, T[1], 2, NU, NP);  // (x, i1)
  }
  __syncthreads();
  if(active)
  {
    mass(T[0], nullptr, T[0], 2, NP, NP);
    mass(T[1], T[2], T[1], 0, NP, NP);
  }
  __syncthreads();
  if(active)
    for(int e = lt; e < NP3; e += NU2)
    {
      int const at          = e % NP + PY * (e / NP % NP) + PZ * (e / (NP * NP));
      a.dst[c * NP3 + e] = T[0][at] + T[1][at];
    }
}

template<int NU, int NP>
hipError_t launch_affine(DivergenceAffineArgs const & a, hipStream_t s)
{
  constexpr int CPB = kThreads / (NU * NU);
  hipLaunchKernelGGL((divergence_affine_kernel<NU, NP>), dim3((unsigned)((a.n_cells + CPB - 1) / CPB)),
                     dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

template<int NU, int NP>
hipError_t launch_general(DivergenceArgs const & a, hipStream_t s)
{
  int const    nu = a.n_u, np = a.n_p;
  size_t const lds = sizeof(double) * (5 * nu * nu * nu + np * np * np + 13 * nu * nu);
  if(lds > 65536)
    return hipErrorInvalidValue;  // at most 5 * 729 + 729 + 1053 doubles = 43.6 KB for n <= 9
  hipLaunchKernelGGL((divergence_apply_kernel<NU, NP>), dim3((unsigned)a.n_cells), dim3(kThreads), lds, s,
                     a);
  return hipGetLastError();
}

// one thread per node; per-thread tables e^{2 pi i m x_d}, m = 0..K, in LDS
constexpr int kInterpThreads = 128;

__global__ void __launch_bounds__(kInterpThreads)
  fourier_interpolate_kernel(double * u, double const * __restrict__ x, double const * __restrict__ md,
                             int n_modes, int K, int n3, int64_t n_points)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int const     nk = K + 1;
  double *      E  = reinterpret_cast<double *>(smem_raw) + threadIdx.x * 6 * nk;
  int64_t const p  = (int64_t)blockIdx.x * kInterpThreads + threadIdx.x;
  if(p >= n_points)
    return;
  for(int d = 0; d < 3; ++d)
  {
    double sn, cs;
    sincos(2.0 * M_PI * x[d * n_points + p], &sn, &cs);
    double * e = E + d * 2 * nk;
    e[0]       = 1.0;
    e[1]       = 0.0;
    for(int m = 1; m <= K; ++m)
    {
      e[2 * m]     = e[2 * m - 2] * cs - e[2 * m - 1] * sn;
      e[2 * m + 1] = e[2 * m - 2] * sn + e[2 * m - 1] * cs;
    }
  }
  double v[3] = {0, 0, 0};
  for(int m = 0; m < n_modes; ++m)
  {
    double const * q = md + 8 * m;
    int const      a0 = (int)q[0], a1 = (int)q[1], a2 = (int)q[2];
    double const * ex = E + 2 * (a0 < 0 ? -a0 : a0);
    double const * ey = E + 2 * nk + 2 * (a1 < 0 ? -a1 : a1);
    double const * ez = E + 4 * nk + 2 * (a2 < 0 ? -a2 : a2);
    double const   xr = ex[0], xi = a0 < 0 ? -ex[1] : ex[1];
    double const   yr = ey[0], yi = a1 < 0 ? -ey[1] : ey[1];
    double const   zr0 = ez[0], zi0 = a2 < 0 ? -ez[1] : ez[1];
    double const   ar = xr * yr - xi * yi, ai = xr * yi + xi * yr;
    double const   zr = ar * zr0 - ai * zi0, zi = ar * zi0 + ai * zr0;
    double const   w  = q[6] * zr - q[7] * zi;
    v[0] += w * q[3];
    v[1] += w * q[4];
    v[2] += w * q[5];
  }
  int64_t const c = p / n3, i = p % n3;
  for(int k = 0; k < 3; ++k)
    u[(c * 3 + k) * n3 + i] = v[k];
}
}  // namespace

hipError_t launch_divergence_apply(DivergenceArgs const & a, hipStream_t s)
{
  int const nu = a.n_u, np = a.n_p;
  if(nu < 2 || nu > 9 || np < 2 || np > 9 || a.n_cells < 1 || !a.dst || !a.src || !a.cell_geo ||
     !a.face_geo || !a.tables)
    return hipErrorInvalidValue;
  // the pairs of degrees in use: velocity of one degree more than the pressure, or equal
#define EXADG_CASE(NU, NP)      \
  if(nu == NU && np == NP)      \
    return launch_general<NU, NP>(a, s);
  EXADG_CASE(3, 2) EXADG_CASE(4, 3) EXADG_CASE(5, 4) EXADG_CASE(6, 5) EXADG_CASE(7, 6) EXADG_CASE(8, 7)
  EXADG_CASE(9, 8)
  EXADG_CASE(2, 2) EXADG_CASE(3, 3) EXADG_CASE(4, 4) EXADG_CASE(5, 5) EXADG_CASE(6, 6) EXADG_CASE(7, 7)
  EXADG_CASE(8, 8) EXADG_CASE(9, 9)
#undef EXADG_CASE
  return launch_general<0, 0>(a, s);
}

bool has_divergence_affine(int nu, int np) { return nu >= 2 && nu <= 9 && np >= 2 && (np == nu || np == nu - 1); }

hipError_t launch_divergence_affine(DivergenceAffineArgs const & a, int nu, int np, hipStream_t s)
{
  if(!has_divergence_affine(nu, np) || a.n_cells < 1 || !a.dst || !a.src)
    return hipErrorInvalidValue;
#define EXADG_CASE(NU, NP)      \
  if(nu == NU && np == NP)      \
    return launch_affine<NU, NP>(a, s);
  EXADG_CASE(3, 2) EXADG_CASE(4, 3) EXADG_CASE(5, 4) EXADG_CASE(6, 5) EXADG_CASE(7, 6) EXADG_CASE(8, 7)
  EXADG_CASE(9, 8)
  EXADG_CASE(2, 2) EXADG_CASE(3, 3) EXADG_CASE(4, 4) EXADG_CASE(5, 5) EXADG_CASE(6, 6) EXADG_CASE(7, 7)
  EXADG_CASE(8, 8) EXADG_CASE(9, 9)
#undef EXADG_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_fourier_interpolate(double * u, double const * x_nodes, double const * mode_data,
                                      int n_modes, int K, int n3, int64_t n_cells, hipStream_t s)
{
  if(!u || !x_nodes || !mode_data || n_modes < 1 || K < 0 || K > 8 || n3 < 1 || n_cells < 1)
    return hipErrorInvalidValue;
  int64_t const n_points = n_cells * n3;
  size_t const  lds      = sizeof(double) * kInterpThreads * 6 * (K + 1);  // <= 55.3 KB
  int64_t const blocks   = (n_points + kInterpThreads - 1) / kInterpThreads;
  hipLaunchKernelGGL(fourier_interpolate_kernel, dim3((unsigned)blocks), dim3(kInterpThreads), lds, s,
                     u, x_nodes, mode_data, n_modes, K, n3, n_points);
  return hipGetLastError();
}
}  // namespace ExaDG
