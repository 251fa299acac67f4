// FP32 GEMM of the learned guess's network on the matrix cores, with strided operands.
//
//   C(i,j) = epilogue(sum_k A(i,k) B(k,j)), A(i,k) = A[i a_i + k a_k], B(k,j) = B[k b_k + j b_j]
//
// A workgroup of four waves computes a TM x TN tile, each wave a quadrant of (TM/32) x (TN/32)
// blocks of v_mfma_f32_16x16x4f32 (FP32 operands and accumulation). Lane l supplies A(l%16, l/16)
// and B(l/16, l%16) of a 16 x 4 / 4 x 16 step and holds D(4 (l/16) + r, l%16), r = 0..3. The order
// of the sum over k is free as long as A and B agree, so a lane takes four consecutive k for the
// four steps of a stage of 16: an operand that is contiguous along k lies in LDS as rows of 16
// (stride 20, one 16-byte read per row and stage), one that is contiguous along i or j as
// columns (stride T + 4, bank-free 4-byte reads). The next stage travels to registers while the
// current one is multiplied and then to the other of two LDS buffers: one barrier per stage.
//
// What bounds it: the matrix cores (157 TFLOP/s FP32) for the large batches, the length of one
// tile's chain of stages for minibatches. The three products of a prediction (32768 x 128 x 500, x 128,
// 32768 x 125 x 128, 6.3 GFLOP) take 104 us (61 TFLOP/s), 199 us with 64 x 64 tiles, one LDS buffer
// and 4-byte loads; a gradient of 4096 samples with its eight products 189 us instead of 358, of
// which 100 us are the products, 30 us the split sums (from 64 to 16 parts and fewer).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "guess_kernels.h"

namespace ExaDG
{
namespace
{
constexpr int TK = 16, kChain = 4;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One operand's T x 16 stage: rows r (i or j), depth k. KU: contiguous along k, else along the rows.
template<int T, bool KU>
struct Operand
{
  static constexpr int ld = KU ? TK + 4 : T + 4, size = KU ? T * ld : TK * ld;
  static constexpr int quads = T * TK / 4, per = (quads + 255) / 256;
  f32x4                q[per];

  // rows r0.. of `rows` valid ones, depths k0.. below ke; vec: 16-byte aligned quads
  __device__ __forceinline__ void load(float const * __restrict__ P, int64_t s_r, int64_t s_k, int r0,
                                       int rows, int k0, int ke, bool vec)
  {
#pragma unroll
    for(int p = 0; p < per; ++p)
    {
      int const e = threadIdx.x + 256 * p;
      q[p]        = f32x4{0.f, 0.f, 0.f, 0.f};
      if(quads % 256 != 0 && e >= quads)
        continue;
      int const     r = r0 + (KU ? e / (TK / 4) : 4 * (e % (T / 4)));
      int const     k = k0 + (KU ? 4 * (e % (TK / 4)) : e / (T / 4));
      float const * at = P + r * s_r + k * s_k;
      if(r >= rows || k >= ke)
        continue;
      int const n = KU ? ke - k : rows - r;
      if(vec && n >= 4)
        q[p] = *reinterpret_cast<f32x4 const *>(at);
      else
#pragma unroll
        for(int t = 0; t < 4; ++t)
          if(t < n)
            q[p][t] = at[t];
    }
  }
  __device__ __forceinline__ void store(float * S) const
  {
#pragma unroll
    for(int p = 0; p < per; ++p)
    {
      int const e = threadIdx.x + 256 * p;
      if(quads % 256 != 0 && e >= quads)
        continue;
      int const at = KU ? (e / (TK / 4)) * ld + 4 * (e % (TK / 4)) : (e / (T / 4)) * ld + 4 * (e % (T / 4));
      *reinterpret_cast<f32x4 *>(S + at) = q[p];
    }
  }
  // the four depths 4 lk .. 4 lk + 3 of row r
  static __device__ __forceinline__ f32x4 read(float const * S, int r, int lk)
  {
    if constexpr(KU)
      return *reinterpret_cast<f32x4 const *>(S + r * ld + 4 * lk);
    else
      return f32x4{S[(4 * lk) * ld + r], S[(4 * lk + 1) * ld + r], S[(4 * lk + 2) * ld + r],
                   S[(4 * lk + 3) * ld + r]};
  }
  static __device__ __forceinline__ float at(float const * S, int r, int k)
  {
    return S[KU ? r * ld + k : k * ld + r];
  }
};

__device__ __forceinline__ float epilogue(SgemmArgs const & a, float v, int64_t i, int j)
{
  if(a.bias)
    v += a.bias[j];
  if(a.relu)
    v = v > 0.f ? v : 0.f;
  if(a.mask && a.mask[i * a.ldc + j] <= 0.f)
    v = 0.f;
  return v;
}

// With gridDim.z > 1 (split K), block z covers k in [z kc, min(K, (z+1) kc)) and writes its raw
// partial product to partial + z M N, and the row sums of A to partial + gridDim.z M N + z M;
// splitk_reduce_kernel adds the parts and applies the epilogue.
// Short (gradients, whose sums over the batch are long): the products of kChain stages are summed
// from zero and then added to `total`, so that a chain of rounding has 64 products and then one
// term per 64, and the row sums and the parts are added in FP64. With one chain per part (128 and more
// products) gradients take 1 - 4% less time (4096 samples 183 us, now 189) but have errors that grow
// with the batch: first layer's weights 1.1 - 1.3 times, biases 1.2 - 2.4 times the ones here.
template<int TM, int TN, bool AK, bool BK, bool Short>
__global__ void __launch_bounds__(256) sgemm_kernel(SgemmArgs a, float * partial, int kc, bool va, bool vb)
{
  using OA         = Operand<TM, AK>;
  using OB         = Operand<TN, BK>;
  constexpr int RB = TM / 32, CB = TN / 32;
  __shared__ __align__(16) float As[2][OA::size];
  __shared__ __align__(16) float Bs[2][OB::size];
  int const tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int const i0 = blockIdx.y * TM, j0 = blockIdx.x * TN;
  int const kb = blockIdx.z * kc, ke = min(a.K, kb + kc);
  int const wr = (wave >> 1) * (TM / 2), wc = (wave & 1) * (TN / 2);  // this wave's quadrant
  int const li = lane & 15, lk = lane >> 4;
  bool const row_sum = a.row_sum && blockIdx.x == 0;
  f32x4      acc[RB][CB], total[RB][CB];  // total: of the whole part, if Short
#pragma unroll
  for(int rb = 0; rb < RB; ++rb)
#pragma unroll
    for(int cb = 0; cb < CB; ++cb)
      acc[rb][cb] = total[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int PARTS = 256 / TM, DEPTH = TK / PARTS;
  double        sum   = 0;  // of row tid % TM over this thread's depths
  OA            qa;
  OB            qb;
  qa.load(a.A, a.a_i, a.a_k, i0, a.M, kb, ke, va);
  qb.load(a.B, a.b_j, a.b_k, j0, a.N, kb, ke, vb);
  qa.store(As[0]);
  qb.store(Bs[0]);
  __syncthreads();
  int buf = 0;
  for(int k0 = kb; k0 < ke; k0 += TK, buf ^= 1)
  {
    bool const more = k0 + TK < ke;
    if(more)
    {
      qa.load(a.A, a.a_i, a.a_k, i0, a.M, k0 + TK, ke, va);
      qb.load(a.B, a.b_j, a.b_k, j0, a.N, k0 + TK, ke, vb);
    }
    f32x4 x[RB], y[CB];
#pragma unroll
    for(int rb = 0; rb < RB; ++rb)
      x[rb] = OA::read(As[buf], wr + 16 * rb + li, lk);
#pragma unroll
    for(int cb = 0; cb < CB; ++cb)
      y[cb] = OB::read(Bs[buf], wc + 16 * cb + li, lk);
#pragma unroll
    for(int t = 0; t < 4; ++t)
#pragma unroll
      for(int rb = 0; rb < RB; ++rb)
#pragma unroll
        for(int cb = 0; cb < CB; ++cb)
          acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[rb][t], y[cb][t], acc[rb][cb], 0, 0, 0);
    if(row_sum)
#pragma unroll
      for(int t = 0; t < DEPTH; ++t)
        sum += OA::at(As[buf], tid % TM, tid / TM * DEPTH + t);
    if(more)
    {
      qa.store(As[buf ^ 1]);
      qb.store(Bs[buf ^ 1]);
    }
    if constexpr(Short)
      if(!more || (k0 - kb) % (kChain * TK) == (kChain - 1) * TK)
      {
#pragma unroll
        for(int rb = 0; rb < RB; ++rb)
#pragma unroll
          for(int cb = 0; cb < CB; ++cb)
          {
            total[rb][cb] += acc[rb][cb];
            acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
    __syncthreads();
  }
  bool const split = gridDim.z > 1;
  if(row_sum)
  {
    double * const parts = reinterpret_cast<double *>(As[0]);
    static_assert(2 * 256 <= OA::size, "the parts of the row sums in the operand's buffer");
    parts[tid] = sum;
    __syncthreads();
    if(tid < TM && i0 + tid < a.M)
    {
      for(int p = 1; p < PARTS; ++p)
        sum += parts[tid + p * TM];
      (split ? partial + (int64_t)gridDim.z * a.M * a.N + (int64_t)blockIdx.z * a.M : a.row_sum)[i0 + tid] = (float)sum;
    }
  }
#pragma unroll
  for(int rb = 0; rb < RB; ++rb)
#pragma unroll
    for(int cb = 0; cb < CB; ++cb)
#pragma unroll
      for(int r = 0; r < 4; ++r)
      {
        int const i = i0 + wr + 16 * rb + 4 * lk + r, j = j0 + wc + 16 * cb + li;
        if(i >= a.M || j >= a.N)
          continue;
        if(split)
          partial[((int64_t)blockIdx.z * a.M + i) * a.N + j] = (Short ? total : acc)[rb][cb][r];
        else
          a.C[i * a.ldc + j] = epilogue(a, (Short ? total : acc)[rb][cb][r], i, j);
      }
}

__global__ void __launch_bounds__(256) splitk_reduce_kernel(SgemmArgs a, float const * __restrict__ part, int splits)
{
  int64_t const total = (int64_t)a.M * a.N, rows = a.row_sum ? a.M : 0;
  for(int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total + rows; e += (int64_t)gridDim.x * 256)
  {
    bool const    sum = e >= total;
    float const * p   = part + (sum ? splits * total + (e - total) : e);
    double        d   = 0;
    for(int z = 0; z < splits; ++z)
      d += p[z * (sum ? rows : total)];
    float const v = (float)d;
    if(sum)
      a.row_sum[e - total] = v;
    else
    {
      int const i = (int)(e / a.N), j = (int)(e - (int64_t)i * a.N);
      a.C[i * a.ldc + j] = epilogue(a, v, i, j);
    }
  }
}

template<int TM, int TN>
hipError_t launch_tile(SgemmArgs const & a, float * workspace, int64_t workspace_floats, hipStream_t s)
{
  int const tiles = ((a.N + TN - 1) / TN) * ((a.M + TM - 1) / TM);
  // split K when the tiles alone cannot fill the card (weight gradients: K = batch), into parts
  // of at least eight stages
  int splits = 1;
  if(workspace != nullptr && tiles < 256 && a.K >= 16 * TK)
  {
    splits = std::min((256 + tiles - 1) / tiles, a.K / (8 * TK));
    splits = (int)std::min<int64_t>(splits, workspace_floats / ((int64_t)a.M * (a.N + 1)));
    splits = std::max(splits, 1);
  }
  int const kc = splits > 1 ? ((a.K + splits - 1) / splits + TK - 1) / TK * TK : a.K;
  splits       = (a.K + kc - 1) / kc;
  // quads are read as such where every row of them is 16-byte aligned
  auto aligned = [](float const * p, int64_t stride) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 4 == 0;
  };
  bool const ak = a.a_k == 1, bk = a.b_j != 1;
  bool const va = aligned(a.A, ak ? a.a_i : a.a_k), vb = aligned(a.B, bk ? a.b_j : a.b_k);
  dim3 const grid((a.N + TN - 1) / TN, (a.M + TM - 1) / TM, splits);
  auto launch = [&](auto a_k, auto b_k, auto chains) {
    hipLaunchKernelGGL((sgemm_kernel<TM, TN, decltype(a_k)::value, decltype(b_k)::value, decltype(chains)::value>),
                       grid, dim3(256), 0, s, a, workspace, kc, va, vb);
  };
  using Yes = std::true_type;
  using No  = std::false_type;
  // gradients in short chains, except for the large tiles: their results are long and their sums, over
  // the width or the outputs, short
  if constexpr(TN == 64)
  {
    if(workspace != nullptr)
      ak ? (bk ? launch(Yes(), Yes(), Yes()) : launch(Yes(), No(), Yes())) : launch(No(), No(), Yes());
    else
      ak ? (bk ? launch(Yes(), Yes(), No()) : launch(Yes(), No(), No())) : launch(No(), No(), No());
  }
  else
    ak ? (bk ? launch(Yes(), Yes(), No()) : launch(Yes(), No(), No())) : launch(No(), No(), No());
  hipError_t const e = hipGetLastError();
  if(e != hipSuccess || splits == 1)
    return e;
  int64_t const total = (int64_t)a.M * (a.N + 1);
  int const     g     = (int)std::min<int64_t>((total + 255) / 256, 2048);
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3(g), dim3(256), 0, s, a, workspace, splits);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_sgemm(SgemmArgs const & a, float * workspace, int64_t workspace_floats, hipStream_t s)
{
  // each operand contiguous along one of its indices, and not A along i with B along k
  if(a.M < 1 || a.N < 1 || a.K < 1 || (a.a_i != 1 && a.a_k != 1) || (a.b_k != 1 && a.b_j != 1) ||
     (a.a_k != 1 && a.b_j != 1))
    return hipErrorInvalidValue;
  // the largest tile that still gives every CU one; splitting K (long sums only) counts as tiles
  auto tiles = [&](int tm, int tn) { return (int64_t)((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn); };
  if(tiles(64, 128) >= 256)
    return launch_tile<64, 128>(a, workspace, workspace_floats, s);
  if(tiles(64, 64) >= 256 || (workspace != nullptr && a.K >= 1024))
    return launch_tile<64, 64>(a, workspace, workspace_floats, s);
  return launch_tile<32, 64>(a, workspace, workspace_floats, s);
}
}  // namespace ExaDG
