// The coarse PCG solve of a small Q1 level in one workgroup.
//
// Driven from the host, a CG iteration is some ten launches and two waits for its scalars, about
// 90 us whatever the level's size; here it is one pass of 1024 threads over the stencil with the
// direction in LDS and three workgroup sums, bound by the latency of the stencil reads of one CU:
// 2 us at 9^3 nodes, 8 us per 1000 nodes beyond (one CU reads the weights, 108 bytes a node in FP32,
// from L2 in every iteration).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "../../include/exadg_amd.h"
#include "mg_kernels.h"

namespace ExaDG
{
namespace
{
constexpr int kPcgThreads = 1024;

// sums over the workgroup of K values per thread, the same on every thread (wave sums by
// butterflies, the waves' sums in order: deterministic)
template<int K>
__device__ __forceinline__ void block_sums(double (&v)[K], double * scratch)
{
#pragma unroll
  for(int k = 0; k < K; ++k)
#pragma unroll
    for(int m = 32; m > 0; m >>= 1)
      v[k] += __shfl_xor(v[k], m);
  __syncthreads();  // the scratch is free
  if((threadIdx.x & 63) == 0)
#pragma unroll
    for(int k = 0; k < K; ++k)
      scratch[k * (kPcgThreads / 64) + (threadIdx.x >> 6)] = v[k];
  __syncthreads();
#pragma unroll
  for(int k = 0; k < K; ++k)
  {
    double s = 0;
    for(int w = 0; w < kPcgThreads / 64; ++w)
      s += scratch[k * (kPcgThreads / 64) + w];
    v[k] = s;
  }
}

// PCG with point Jacobi from a zero initial guess to |r| <= max(1e-12, rel_tol |b|), the direction
// in LDS. PER > 0: up to PER nodes per thread with r, v and x in registers; PER = 0: any number, r
// and v in global memory (a.r, a.v). FP64 dot products as in the host-driven solve.
template<typename Number, int PER>
__global__ void __launch_bounds__(kPcgThreads) q1_pcg_kernel(Q1PcgArgs<Number> a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *  scratch = reinterpret_cast<double *>(smem_raw);  // 3 sums of 16 waves
  Number *  p       = reinterpret_cast<Number *>(scratch + 3 * (kPcgThreads / 64));
  int const n = a.n, tid = threadIdx.x;
  int const n0 = a.q.nn[0], n1 = a.q.nn[1], n2 = a.q.nn[2];
  Number    r_[PER > 0 ? PER : 1], v_[PER > 0 ? PER : 1], x_[PER > 0 ? PER : 1];
  auto      each = [&](auto && f) {  // f(node, slot) over this thread's nodes
    if constexpr(PER > 0)
    {
#pragma unroll
      for(int k = 0; k < PER; ++k)
        if(tid + k * kPcgThreads < n)
          f(tid + k * kPcgThreads, k);
    }
    else
      for(int e = tid; e < n; e += kPcgThreads)
        f(e, 0);
  };
  auto r = [&](int e, int k) -> Number & {
    if constexpr(PER > 0)
      return r_[k];
    else
      return a.r[e];
  };
  auto v = [&](int e, int k) -> Number & {
    if constexpr(PER > 0)
      return v_[k];
    else
      return a.v[e];
  };
  auto x = [&](int e, int k) -> Number & {
    if constexpr(PER > 0)
      return x_[k];
    else
      return a.x[e];
  };
  auto subtract_mean = [&]() {
    double s[1] = {0};
    each([&](int e, int k) { s[0] += (double)r(e, k); });
    block_sums<1>(s, scratch);
    Number const mean = (Number)(s[0] / (double)n);
    each([&](int e, int k) { r(e, k) -= mean; });
  };
  auto norm_and_dot = [&](double (&s)[2]) {  // r.r and r.z with z = D^-1 r
    s[0] = s[1] = 0;
    each([&](int e, int k) {
      Number const re = r(e, k), ze = a.dinv[e] * re;
      s[0] += (double)re * (double)re;
      s[1] += (double)re * (double)ze;
    });
    block_sums<2>(s, scratch);
  };
  each([&](int e, int k) {
    r(e, k) = a.b[e];
    x(e, k) = Number(0);
  });
  if(a.singular)
    subtract_mean();
  double s[2];
  norm_and_dot(s);
  double const wanted = a.rel_tol * sqrt(s[0]), tol = 1e-12 < wanted ? wanted : 1e-12;
  double       rho = s[1];
  int          it = 0, status = 0;
  if(!(sqrt(s[0]) <= tol))
  {
    each([&](int e, int k) { p[e] = a.dinv[e] * r(e, k); });
    for(it = 1; it <= a.max_iter; ++it)
    {
      __syncthreads();  // p
      Number const * W = a.W;
      // the weights are read anew in every iteration, not kept in registers
      if constexpr(PER != 1)
        asm volatile("" : "+s"(W));
      double pv[1] = {0};
      each([&](int e, int k) {
        unsigned const t = (unsigned)e / (unsigned)n0;
        int const      nz = t / (unsigned)n1, ny = t - nz * n1, nx = e - t * n0;
        int            ix[3], iy[3], iz[3];
#pragma unroll
        for(int o = 0; o < 3; ++o)
        {
          auto side = [o](int c, int m, int periodic) {
            c += o - 1;
            return c < 0 ? (periodic ? m - 1 : 0) : c >= m ? (periodic ? 0 : m - 1) : c;
          };
          ix[o] = side(nx, n0, a.q.periodic[0]);
          iy[o] = side(ny, n1, a.q.periodic[1]) * n0;
          iz[o] = side(nz, n2, a.q.periodic[2]) * n0 * n1;
        }
        Number sum = 0;
#pragma unroll
        for(int m = 0; m < 27; ++m)
          sum += (W + (int64_t)m * n)[(unsigned)e] * p[ix[m % 3] + iy[(m / 3) % 3] + iz[m / 9]];
        v(e, k) = sum;
        pv[0] += (double)p[e] * (double)sum;
      });
      block_sums<1>(pv, scratch);
      double const alpha = rho / pv[0];
      each([&](int e, int k) {
        x(e, k) += (Number)alpha * p[e];
        r(e, k) += (Number)(-alpha) * v(e, k);
      });
      if(a.singular)
        subtract_mean();
      norm_and_dot(s);
      double const rn = sqrt(s[0]);
      if(!isfinite(rn))
      {
        status = 1;
        break;
      }
      if(rn <= tol)
        break;
      double const beta = s[1] / rho;
      rho               = s[1];
      each([&](int e, int k) { p[e] = a.dinv[e] * r(e, k) + (Number)beta * p[e]; });
    }
  }
  if constexpr(PER > 0)
    each([&](int e, int k) { a.x[e] = x_[k]; });
  if(tid == 0)
  {
    a.result[0] = min(it, a.max_iter);
    a.result[1] = status;
  }
}

template<typename Number, int PER>
hipError_t launch_pcg(Q1PcgArgs<Number> const & a, hipStream_t s)
{
  size_t const lds = 3 * (kPcgThreads / 64) * sizeof(double) + a.n * sizeof(Number);
  int const    lds_max = 3 * (kPcgThreads / 64) * sizeof(double) + kQ1PcgMaxNodes * sizeof(Number);
  static std::atomic<bool> attr{false};
  if(lds > 65536 && !attr.load(std::memory_order_acquire))
  {
    hipError_t e = hipFuncSetAttribute((void const *)q1_pcg_kernel<Number, PER>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    if(e != hipSuccess)
      return e;
    attr.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL((q1_pcg_kernel<Number, PER>), dim3(1), dim3(kPcgThreads), lds, s, a);
  return hipGetLastError();
}
}  // namespace

template<typename Number>
hipError_t launch_q1_pcg(Q1PcgArgs<Number> const & a, hipStream_t s)
{
  if(a.n < 1 || a.n > kQ1PcgMaxNodes)
    return hipErrorInvalidValue;
  int const per = (a.n + kPcgThreads - 1) / kPcgThreads;
  if(per <= 1)
    return launch_pcg<Number, 1>(a, s);
  if(per <= 2)
    return launch_pcg<Number, 2>(a, s);
  return launch_pcg<Number, 0>(a, s);
}

template hipError_t launch_q1_pcg<double>(Q1PcgArgs<double> const &, hipStream_t);
template hipError_t launch_q1_pcg<float>(Q1PcgArgs<float> const &, hipStream_t);
}  // namespace ExaDG
