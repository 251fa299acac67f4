// Multigrid transfer and coarse-level kernels (see mg_kernels.h).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/exadg_amd.h"
#include "mg_kernels.h"

namespace ExaDG
{
namespace
{
// ---------------------------------------------------------------- p-transfer
//
// One cell per group of nf^2 lanes, three sum-factorized 1D interpolation sweeps through LDS.
// PROLONG: input nc^3 -> output nf^3 with M = P; else input nf^3 -> output nc^3 with M = P^T.
template<typename Number, bool PROLONG>
__global__ void __launch_bounds__(256)
  p_transfer_kernel(Number * dst, Number const * src, Number const * P, int nf, int nc,
                    int64_t n_cells, int cpb)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Number *      sm     = reinterpret_cast<Number *>(smem_raw);
  int const     nf3    = nf * nf * nf;
  int const     tpc    = nf * nf;
  int const     slot   = threadIdx.x / tpc;
  int const     lt     = threadIdx.x - slot * tpc;
  int64_t const cell   = (int64_t)blockIdx.x * cpb + slot;
  bool const    active = slot < cpb && cell < n_cells;
  Number *      b0     = sm + (active ? slot : 0) * 2 * nf3;
  Number *      b1     = b0 + nf3;
  int const     nin = PROLONG ? nc : nf, nout = PROLONG ? nf : nc;
  int const     nin3 = nin * nin * nin, nout3 = nout * nout * nout;
  auto          M = [&](int a, int i) { return PROLONG ? P[a * nc + i] : P[i * nc + a]; };

  if(active)
    for(int e = lt; e < nin3; e += tpc)
      b0[e] = src[cell * nin3 + e];
  __syncthreads();
  if(active)
    for(int task = lt; task < nin * nin; task += tpc)
    {
      int const j = task % nin, k = task / nin;
      for(int a = 0; a < nout; ++a)
      {
        Number s = 0;
        for(int i = 0; i < nin; ++i)
          s += M(a, i) * b0[i + nin * (j + nin * k)];
        b1[a + nout * (j + nin * k)] = s;
      }
    }
  __syncthreads();
  if(active)
    for(int task = lt; task < nout * nin; task += tpc)
    {
      int const a = task % nout, k = task / nout;
      for(int b = 0; b < nout; ++b)
      {
        Number s = 0;
        for(int j = 0; j < nin; ++j)
          s += M(b, j) * b1[a + nout * (j + nin * k)];
        b0[a + nout * (b + nout * k)] = s;
      }
    }
  __syncthreads();
  if(active)
    for(int task = lt; task < nout * nout; task += tpc)
    {
      int const a = task % nout, b = task / nout;
      for(int c = 0; c < nout; ++c)
      {
        Number s = 0;
        for(int k = 0; k < nin; ++k)
          s += M(c, k) * b0[a + nout * (b + nout * k)];
        dst[cell * nout3 + a + nout * (b + nout * c)] += s;
      }
    }
}

// Q1 operator as an assembled 27-point stencil: W[j * n + node] couples node with its
// neighbour at offset (j % 3 - 1, (j / 3) % 3 - 1, j / 9 - 1) (periodic wrap). Weights to
// constrained or missing neighbours are zero and those reads are clamped in bounds; a
// constrained node's row is the identity. One thread per node, W read plane by plane
// (consecutive nodes, consecutive addresses), or, on affine boxes, from the 125 node classes' rows
// (Q1Weights). The levels are small, a wave or two per SIMD, so
// what a thread issues before its loads counts: with the node's coordinates and the 27 addresses in
// 32 bits (Index, below 2^31 nodes) a V-cycle with 80 of these steps at 33 x 32 x 32 nodes takes 669
// instead of 764 us (FP64 966 instead of 1017), at 17 x 16 x 16 nodes 372 instead of 401. (Three
// steps per launch on overlapping blocks of 6^3 nodes, with the weights in registers: no faster at
// 33 x 32 x 32 nodes, 8% at 17 x 16 x 16, and 1.8 times slower at 61 x 60 x 60.)
template<bool classed, typename Number, typename Index>
__device__ __forceinline__ Number q1_stencil_row(Number const * __restrict__ W,
                                                 Number const * __restrict__ src,
                                                 Q1Topology const & q, Index node, Index n)
{
  Index const n0 = (Index)q.nn[0], n1 = (Index)q.nn[1], n2 = (Index)q.nn[2];
  Index const r = node / n0, z = r / n1, x = node - r * n0, y = r - z * n1;
  // offsets of the three neighbours per direction
  auto neighbours = [](Index c, Index m, int periodic, Index stride, Index (&o)[3]) {
    o[0] = (c > 0 ? c - 1 : (periodic ? m - 1 : 0)) * stride;
    o[1] = c * stride;
    o[2] = (c < m - 1 ? c + 1 : (periodic ? 0 : m - 1)) * stride;
  };
  Index ox[3], oy[3], oz[3];
  neighbours(x, n0, q.periodic[0], 1, ox);
  neighbours(y, n1, q.periodic[1], n0, oy);
  neighbours(z, n2, q.periodic[2], n0 * n1, oz);
  auto   value = [&](int j) { return src[ox[j % 3] + (oy[(j / 3) % 3] + oz[j / 9])]; };
  Number acc   = 0;
  if constexpr(classed)
  {
    auto kind = [](Index c, Index m, int periodic) {
      return periodic ? 2 : m < 5 || c < 2 ? (int)c : c >= m - 2 ? (int)(c + 5 - m) : 2;
    };
    int const c = kind(x, n0, q.periodic[0]) +
                  5 * (kind(y, n1, q.periodic[1]) + 5 * kind(z, n2, q.periodic[2]));
    int const c0 = __builtin_amdgcn_readfirstlane(c);
    // the values first: their loads do not wait for the class
    Number u[27];
#pragma unroll
    for(int j = 0; j < 27; ++j)
      u[j] = value(j);
    // a wave of one class (most of them where x is periodic) takes its row by scalar loads
    if(__builtin_amdgcn_ballot_w64(c != c0) == 0)
    {
      auto const w = (Number const __attribute__((address_space(4))) *)W + kQ1ClassStride * c0;
#pragma unroll
      for(int j = 0; j < 27; ++j)
        acc += w[j] * u[j];
    }
    else
    {
      constexpr int V = 16 / sizeof(Number);
      struct alignas(16) Pack
      {
        Number w[V];
      };
      Pack const * const p = reinterpret_cast<Pack const *>(W + kQ1ClassStride * c);
      Pack               w[kQ1ClassStride / V];
#pragma unroll
      for(int i = 0; i < kQ1ClassStride / V; ++i)
        w[i] = p[i];
#pragma unroll
      for(int j = 0; j < 27; ++j)
        acc += w[j / V].w[j % V] * u[j];
    }
  }
  else
  {
#pragma unroll
    for(int j = 0; j < 27; ++j)
      acc += (W + (int64_t)j * n)[node] * value(j);
  }
  return acc;
}

template<bool classed, typename Number, typename Index>
__global__ void __launch_bounds__(256)
  q1_stencil_kernel(Number * __restrict__ dst, Number const * __restrict__ src,
                    Number const * __restrict__ W, Q1Topology q, Index n)
{
  Index const node = (Index)blockIdx.x * blockDim.x + threadIdx.x;
  if(node < n)
    dst[node] = q1_stencil_row<classed, Number, Index>(W, src, q, node, n);
}

// one Chebyshev step on the Q1 level with the operator application fused in:
//   x_new = (1 + f1) x - f1 x_old + f2 D^{-1} (b - A x)     (variant 2)
//   x_new = (1 + f1) x + f2 D^{-1} (b - A x)                (variant 1)
template<bool classed, typename Number, typename Index>
__global__ void __launch_bounds__(256)
  q1_chebyshev_kernel(Number * __restrict__ x_new, Number const * __restrict__ x,
                      Number const * x_old, Number const * __restrict__ b,
                      Number const * __restrict__ dinv, Number const * __restrict__ W,
                      Q1Topology q, Number f1, Number f2, int variant, Index n)
{
  Index const node = (Index)blockIdx.x * blockDim.x + threadIdx.x;
  if(node >= n)
    return;
  Number const t = q1_stencil_row<classed, Number, Index>(W, x, q, node, n);
  Number       v = (Number(1) + f1) * x[node] + f2 * dinv[node] * (b[node] - t);
  if(variant == 2)
    v -= f1 * x_old[node];
  x_new[node] = v;
}

inline int blocks_for(int64_t n) { return (int)((n + 255) / 256); }
}  // namespace

template<typename Number>
hipError_t launch_p_prolongate_add(Number * dst_f, Number const * src_c, Number const * P, int nf,
                                   int nc, int64_t n_cells, hipStream_t s)
{
  int const    cpb = 256 / (nf * nf);
  size_t const lds = sizeof(Number) * cpb * 2 * nf * nf * nf;
  hipLaunchKernelGGL((p_transfer_kernel<Number, true>), dim3((n_cells + cpb - 1) / cpb), dim3(256),
                     lds, s, dst_f, src_c, P, nf, nc, n_cells, cpb);
  return hipGetLastError();
}

template<typename Number>
hipError_t launch_p_restrict_add(Number * dst_c, Number const * src_f, Number const * P, int nf,
                                 int nc, int64_t n_cells, hipStream_t s)
{
  int const    cpb = 256 / (nf * nf);
  size_t const lds = sizeof(Number) * cpb * 2 * nf * nf * nf;
  hipLaunchKernelGGL((p_transfer_kernel<Number, false>), dim3((n_cells + cpb - 1) / cpb), dim3(256),
                     lds, s, dst_c, src_f, P, nf, nc, n_cells, cpb);
  return hipGetLastError();
}

template<typename Number>
hipError_t launch_q1_stencil(Number * dst, Number const * src, Q1Weights<Number> const & W,
                             Q1Topology const & q, hipStream_t s)
{
  int64_t const n     = (int64_t)q.nn[0] * q.nn[1] * q.nn[2];
  auto          apply = [&](auto classed, auto nodes) {
    using Index = decltype(nodes);
    hipLaunchKernelGGL((q1_stencil_kernel<decltype(classed)::value, Number, Index>),
                       dim3((n + 127) / 128), dim3(128), 0, s, dst, src,
                       classed ? W.classes : W.planes, q, nodes);
  };
  if(W.classes)
    n < INT32_MAX ? apply(std::true_type(), (uint32_t)n) : apply(std::true_type(), n);
  else
    n < INT32_MAX ? apply(std::false_type(), (uint32_t)n) : apply(std::false_type(), n);
  return hipGetLastError();
}

template<typename Number>
hipError_t launch_q1_chebyshev(Number * x_new, Number const * x, Number const * x_old,
                               Number const * b, Number const * dinv, Q1Weights<Number> const & W,
                               Q1Topology const & q, Number f1, Number f2, bool has_old,
                               hipStream_t s)
{
  int64_t const n    = (int64_t)q.nn[0] * q.nn[1] * q.nn[2];
  auto          step = [&](auto classed, auto nodes) {
    using Index = decltype(nodes);
    hipLaunchKernelGGL((q1_chebyshev_kernel<decltype(classed)::value, Number, Index>),
                       dim3((n + 127) / 128), dim3(128), 0, s, x_new, x, x_old, b, dinv,
                       classed ? W.classes : W.planes, q, f1, f2, has_old ? 2 : 1, nodes);
  };
  if(W.classes)
    n < INT32_MAX ? step(std::true_type(), (uint32_t)n) : step(std::true_type(), n);
  else
    n < INT32_MAX ? step(std::false_type(), (uint32_t)n) : step(std::false_type(), n);
  return hipGetLastError();
}

#define EXADG_INST(T)                                                                              \
  template hipError_t launch_p_prolongate_add<T>(T *, T const *, T const *, int, int, int64_t,     \
                                                 hipStream_t);                                     \
  template hipError_t launch_p_restrict_add<T>(T *, T const *, T const *, int, int, int64_t,       \
                                               hipStream_t);                                       \
  template hipError_t launch_q1_stencil<T>(T *, T const *, Q1Weights<T> const &, Q1Topology const &, \
                                           hipStream_t);                                           \
  template hipError_t launch_q1_chebyshev<T>(T *, T const *, T const *, T const *, T const *,      \
                                             Q1Weights<T> const &, Q1Topology const &, T, T, bool,  \
                                             hipStream_t);
EXADG_INST(double)
EXADG_INST(float)
#undef EXADG_INST

}  // namespace ExaDG
