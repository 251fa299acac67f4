// Line helpers of the SIPG kernels: a lane holds one line of an n^3 tensor in registers and
// applies the 1D matrices to it (device code).
#pragma once
#include <hip/hip_runtime.h>

#include "laplace_kernels.h"

namespace ExaDG
{
namespace
{
constexpr int kInterior = 2;  // face type besides EXADG_BC_DIRICHLET / EXADG_BC_NEUMANN

// out[i] = sum_j M[i*N+j] in[j]
template<int N, typename Number, typename Table>
__device__ __forceinline__ void mat_apply(Table const M, Number const (&in)[N],
                                          Number (&out)[N])
{
#pragma unroll
  for(int i = 0; i < N; ++i)
  {
    Number s = 0;
#pragma unroll
    for(int j = 0; j < N; ++j)
      s += M[i * N + j] * in[j];
    out[i] = s;
  }
}

// out = A in for a centrosymmetric (Skew = false) or skew-centrosymmetric (Skew = true) A,
// stored in even-odd form when Packed (always in the Cartesian kernel, else see gen_packed), else as the plain row-major
// matrix. Centro: out_i = E_i + O_i, out_{n-1-i} = E_i - O_i, middle output (odd n) from the
// even part; skew: out_{n-1-i} = O_i - E_i and the middle output from the odd part.
template<int N, bool Packed, bool Skew, typename Number, typename Table>
__device__ __forceinline__ void eo_apply(Table const T, Number const (&in)[N],
                                         Number (&out)[N])
{
  if constexpr(!Packed)
    mat_apply<N>(T, in, out);
  else
  {
    constexpr int  m = N / 2, me = m + N % 2;
    Table const    Ae = T;
    Table const    Ao = T + m * me;
    Table const    Am = Ao + m * m;
    Number         e[me], o[m];
#pragma unroll
    for(int j = 0; j < m; ++j)
    {
      e[j] = in[j] + in[N - 1 - j];
      o[j] = in[j] - in[N - 1 - j];
    }
    if constexpr(N % 2 == 1)
      e[m] = in[m];
#pragma unroll
    for(int i = 0; i < m; ++i)
    {
      Number E = 0, O = 0;
#pragma unroll
      for(int j = 0; j < me; ++j)
        E += Ae[i * me + j] * e[j];
#pragma unroll
      for(int j = 0; j < m; ++j)
        O += Ao[i * m + j] * o[j];
      out[i]         = E + O;
      out[N - 1 - i] = Skew ? O - E : E - O;
    }
    if constexpr(N % 2 == 1)
    {
      Number s = 0;
      if constexpr(Skew)
      {
#pragma unroll
        for(int j = 0; j < m; ++j)
          s += Am[j] * o[j];
      }
      else
      {
#pragma unroll
        for(int j = 0; j < me; ++j)
          s += Am[j] * e[j];
      }
      out[m] = s;
    }
  }
}

// the Cartesian kernel's centrosymmetric 1D products (CartTable)
template<int N, typename Number, typename Table>
__device__ __forceinline__ void cs_apply(Table const T, Number const (&in)[N],
                                         Number (&out)[N])
{
  eo_apply<N, true, false>(T, in, out);
}

// the general kernel's sweeps (GenTable): S and S^T centrosymmetric, Dq and Dq^T skew
template<int N, bool Skew, typename Number>
__device__ __forceinline__ void gen_apply(Number const * __restrict__ T, Number const (&in)[N],
                                          Number (&out)[N])
{
  eo_apply<N, gen_packed(N), Skew>(T, in, out);
}

template<int N, typename Number>
__device__ __forceinline__ void load_line(Number const * p, int stride, Number (&v)[N])
{
#pragma unroll
  for(int i = 0; i < N; ++i)
    v[i] = p[i * stride];
}

template<int N, typename Number>
__device__ __forceinline__ void store_line(Number * p, int stride, Number const (&v)[N])
{
#pragma unroll
  for(int i = 0; i < N; ++i)
    p[i * stride] = v[i];
}

template<int N, typename Number, typename Table>
__device__ __forceinline__ Number dot_line(Table const a, Number const (&v)[N])
{
  Number s = 0;
#pragma unroll
  for(int i = 0; i < N; ++i)
    s += a[i] * v[i];
  return s;
}
}  // namespace
}  // namespace ExaDG
