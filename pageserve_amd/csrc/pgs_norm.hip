// RMSNorm of the activations feeding the q|k|v and gate|up projections
// (engine/model.py:29-34, called at engine/model.py:166 and :187), as one
// kernel instead of the reference's chain of elementwise and reduction ops:
//
//   var  = mean_j x[i, j]^2           (fp32)
//   r    = 1 / sqrt(var + eps)         (torch.rsqrt; IEEE sqrt and divide here)
//   h    = bf16( w[j] * bf16( x[i, j] * r ) )
//
// The two bf16 roundings are the reference's: x * r is cast back to the model
// dtype before the multiply by the bf16 norm weight.  One workgroup per row;
// the sum of squares is reduced in a fixed order (per-thread strided sums,
// then a fixed butterfly inside each wave, then the waves in order), so
// results do not depend on timing.  2 B read and 2 B written per element; at
// decode and prefill-chunk sizes the time is the launch and its one memory
// round trip, so a row of whole 16-byte pieces is read once, with its norm
// weights beside it, into registers (NV pieces per thread, K <= 2048 NV):
// [6, 2048] 3.3 -> 2.4 us against reading it twice.
#include "pgs_linear.h"

namespace pgs {
namespace {

constexpr int kNormThreads = 256;

__device__ __forceinline__ float bf16_round(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

// The row's sum of squares from each thread's share: a butterfly whose lanes
// all end with the same value, then the waves in order.
__device__ __forceinline__ float row_total(float ss) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
  __shared__ float part[kNormThreads / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < kNormThreads / 64; ++i) total += part[i];
  return total;
}

__device__ __forceinline__ void add_squares(u32x4 v, float& ss) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float lo = bf16_bits_to_f32(static_cast<uint16_t>(v[e])), hi = bf16_bits_to_f32(static_cast<uint16_t>(v[e] >> 16));
    ss += lo * lo;
    ss += hi * hi;
  }
}

__device__ __forceinline__ u32x4 scaled(u32x4 v, u32x4 g, float r) {
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x0 = bf16_bits_to_f32(static_cast<uint16_t>(v[e])), x1 = bf16_bits_to_f32(static_cast<uint16_t>(v[e] >> 16));
    const float g0 = bf16_bits_to_f32(static_cast<uint16_t>(g[e])), g1 = bf16_bits_to_f32(static_cast<uint16_t>(g[e] >> 16));
    o[e] = pack_bf16x2(g0 * bf16_round(x0 * r), g1 * bf16_round(x1 * r));
  }
  return o;
}

// NV > 0: rows of at most NV * 2048 values in whole aligned 16-byte pieces;
// 0: longer rows of such pieces, read twice; -1: any row, by element.
template <int NV>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(const uint16_t* __restrict__ x,
                                                               const uint16_t* __restrict__ w, float eps,
                                                               uint16_t* __restrict__ h, int K) {
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * K;
  uint16_t* hr = h + row * K;
  const int tid = threadIdx.x;

  float ss = 0.f;
  if constexpr (NV > 0) {
    // (a piece past K reads the row's last one and is not counted)
    u32x4 v[NV], g[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = ld16(xr + min((i * kNormThreads + tid) * 8, K - 8));
#pragma unroll
    for (int i = 0; i < NV; ++i) g[i] = ld16(w + min((i * kNormThreads + tid) * 8, K - 8));
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if ((i * kNormThreads + tid) * 8 < K) add_squares(v[i], ss);
    const float r = 1.0f / sqrtf(row_total(ss) / static_cast<float>(K) + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (const int j = (i * kNormThreads + tid) * 8; j < K) *reinterpret_cast<u32x4*>(hr + j) = scaled(v[i], g[i], r);
  } else if constexpr (NV == 0) {
    for (int j = tid * 8; j < K; j += kNormThreads * 8) add_squares(ld16(xr + j), ss);
    const float r = 1.0f / sqrtf(row_total(ss) / static_cast<float>(K) + eps);
    for (int j = tid * 8; j < K; j += kNormThreads * 8)
      *reinterpret_cast<u32x4*>(hr + j) = scaled(ld16(xr + j), ld16(w + j), r);
  } else {
    for (int j = tid; j < K; j += kNormThreads) {
      const float f = bf16_bits_to_f32(xr[j]);
      ss += f * f;
    }
    const float r = 1.0f / sqrtf(row_total(ss) / static_cast<float>(K) + eps);
    for (int j = tid; j < K; j += kNormThreads)
      hr[j] = f32_to_bf16_bits(bf16_bits_to_f32(w[j]) * bf16_round(bf16_bits_to_f32(xr[j]) * r));
  }
}

}  // namespace
}  // namespace pgs

using namespace pgs;

extern "C" int pgs_rmsnorm(const void* x, const void* weight, float eps, void* h, int64_t m, int64_t k, void* stream) {
  if (m < 0 || k < 0 || m > 0x7fffffff || k > 0x7fffffff)
    return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_rmsnorm: bad size m=%lld k=%lld", (long long)m, (long long)k);
  if (m == 0) return PGS_OK;
  if (k == 0) return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_rmsnorm: hidden size k=0");
  if (!x || !weight || !h) return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_rmsnorm: null pointer");
  if (!aligned(x, 2) || !aligned(weight, 2) || !aligned(h, 2)) return fail(PGS_ERR_MISALIGNED, "pgs_rmsnorm: misaligned");
  if (!(eps >= 0.f)) return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_rmsnorm: eps must be >= 0");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (int rc = require_device("pgs_rmsnorm", st)) return rc;
  const bool vec = k % 8 == 0 && aligned(x, 16) && aligned(weight, 16) && aligned(h, 16);
  const auto* xp = reinterpret_cast<const uint16_t*>(x);
  const auto* wp = reinterpret_cast<const uint16_t*>(weight);
  auto* hp = reinterpret_cast<uint16_t*>(h);
  const int kk = static_cast<int>(k);
  const dim3 grid(static_cast<unsigned>(m)), block(kNormThreads);
  if (!vec) hipLaunchKernelGGL(rmsnorm_kernel<-1>, grid, block, 0, st, xp, wp, eps, hp, kk);
  else if (k <= 2048) hipLaunchKernelGGL(rmsnorm_kernel<1>, grid, block, 0, st, xp, wp, eps, hp, kk);
  else if (k <= 4096) hipLaunchKernelGGL(rmsnorm_kernel<2>, grid, block, 0, st, xp, wp, eps, hp, kk);
  else if (k <= 8192) hipLaunchKernelGGL(rmsnorm_kernel<4>, grid, block, 0, st, xp, wp, eps, hp, kk);
  else hipLaunchKernelGGL(rmsnorm_kernel<0>, grid, block, 0, st, xp, wp, eps, hp, kk);
  return check_launch("rmsnorm kernel");
}
