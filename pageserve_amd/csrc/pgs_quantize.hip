// Per-output-row symmetric INT8 quantizer and dequantizer (gfx950).
//
// quantize_per_channel: engine/quantization.py:16-23.  Per row: max|w| (exact:
// a max is order independent), the scale absmax / 127 with a correctly rounded
// IEEE divide, then round-half-to-even of the correctly rounded quotient
// w / scale (quantize_bits below), which is what the reference's CPU
// arithmetic does; the results are bit-identical.  quantize_tile_kernel holds
// eight rows in registers and reads the weight once; quantize_rows_kernel (one
// row per workgroup, the row read twice) takes what does not fit it.
//
// dequantize: engine/quantization.py:26-27.  fp32 product q * scale, then one
// round-to-nearest-even conversion to the output type.
#include "pgs_linear.h"

namespace pgs {
namespace {

constexpr int kQuantThreads = 256;
constexpr int kTileMaxK = 12288;  // columns quantize_tile_kernel holds (96 registers of fp32 per thread, 96 KiB of LDS)

template <bool BF16, int VEC>
__device__ __forceinline__ void load_row_vec(const void* __restrict__ base, int64_t elem, float (&f)[VEC]) {
  if constexpr (BF16) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(base) + elem;
    if constexpr (VEC == 8) {
      u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(v[i] << 16);
        f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) f[i] = bf16_bits_to_f32(p[i]);
    }
  } else {
    const float* p = reinterpret_cast<const float*>(base) + elem;
    if constexpr (VEC == 4) {
      f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] = v[i];
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) f[i] = p[i];
    }
  }
}

// |w| as ordered bits: the unsigned maximum over a row is the bits of max|w|,
// with an infinity above every finite value and any NaN above that, so a row
// holding a NaN gets a NaN scale, as torch's amax gives in the reference
__device__ __forceinline__ uint32_t abs_bits(float f) { return __float_as_uint(f) & 0x7fffffffu; }

constexpr uint32_t kInfBits = 0x7f800000u;

// :20 clamp(min=1e-8) (a NaN stays NaN, as torch's clamp keeps it), :21 / 127.0
__device__ __forceinline__ float row_scale(uint32_t bits) {
  const float amax = __uint_as_float(bits);
  return (bits > kInfBits ? amax : fmaxf(amax, 1e-8f)) / 127.0f;
}

// A word whose low byte is int8(rint(w / s)), y = 1 / s (IEEE divide).  The
// quotient is correctly rounded without a division: two residual corrections
// of w * y, the residuals exact in the fused multiply-add (Markstein's
// theorem: with y the correctly rounded reciprocal and q within an ulp of
// w / s, q + y * (w - q s) rounds to the correctly rounded quotient; the first
// correction brings q within that ulp; s lies in [7.8e-11, 2.7e36], so
// nothing but a quotient far below 1/2 can underflow).  Adding 1.5 * 2^23
// then rounds half to even to an integer and leaves it in the low bits
// (|w / s| <= 127 (1 + 2^-23), so no clamp is needed).  A row whose scale is
// infinite or NaN is all zero (0 for a finite / infinite quotient, and what
// the reference's int8 conversion of NaN gives): the caller masks it.
// A dozen instructions fewer than the IEEE division per weight.
__device__ __forceinline__ uint32_t quantize_bits(float w, float s, float y) {
  const float q0 = __fmul_rn(w, y);
  const float q1 = __fmaf_rn(__fmaf_rn(-q0, s, w), y, q0);
  const float q2 = __fmaf_rn(__fmaf_rn(-q1, s, w), y, q1);
  return __float_as_uint(__fadd_rn(q2, 12582912.0f));
}

// the low bytes of four words in one
__device__ __forceinline__ uint32_t low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu);
}

// Eight rows per workgroup of 1024 threads, two waves per row.  Bound by
// memory: each weight is read once, into registers (NV 16-byte pieces per
// thread), where the one-row kernel reads every row twice.  Eight rows
// because eight rows' 16-byte lane segments are one 128-byte line of the
// packed layout: the quantized tile goes through LDS and out as whole lines,
// where a workgroup per row writes 16-byte parts of lines that eight
// workgroups on eight XCDs share.  Padding rows and columns of the packed
// layout are written as zeros here (no separate fill).
template <bool BF16, int NV, bool PACKED>
__global__ __launch_bounds__(1024) void quantize_tile_kernel(const void* __restrict__ w, int64_t n, int k, int kb,
                                                             int8_t* __restrict__ q, float* __restrict__ scale) {
  constexpr int VEC = BF16 ? 8 : 4, TPR = 128;
  constexpr int LD = NV * VEC * TPR + 16;  // (16: the eight rows on distinct banks)
  const int r = uniform(static_cast<int>(threadIdx.x >> 7)), t = threadIdx.x & (TPR - 1);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * 8;
  const int64_t row = row0 + r;
  const bool live = row < n;
  // (buffer resources of exactly this row: a piece past k, or of a row past
  // n, reads zeros and quantizes to zeros, and a store there is dropped)
  const int64_t first = (live ? row : 0) * k;
  const __amdgpu_buffer_rsrc_t wres = make_rsrc(static_cast<const char*>(w) + first * (BF16 ? 2 : 4), live ? k * (BF16 ? 2 : 4) : 0);
  const __amdgpu_buffer_rsrc_t qres = make_rsrc(q + first, live ? k : 0);
  __shared__ uint32_t red[16];
  __shared__ __attribute__((aligned(16))) char tile[PACKED ? 8 * LD : 16];

  u32x4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(wres, t * 16, i * TPR * 16, kLoadNT);
  uint32_t mx = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (BF16) mx = max(mx, max((v[i][c] << 16) & 0x7fffffffu, v[i][c] & 0x7fff0000u));
      else mx = max(mx, v[i][c] & 0x7fffffffu);
    }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), off)));
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = max(red[2 * r], red[2 * r + 1]);
  const float s = row_scale(mx);
  if (t == 0 && live) scale[row] = s;
  const float y = 1.0f / s;
  const uint32_t keep = mx < kInfBits ? 0xffffffffu : 0u;

#pragma unroll
  for (int i = 0; i < NV; ++i) {
    uint32_t o[VEC / 4];
#pragma unroll
    for (int c = 0; c < VEC / 4; ++c) {
      float f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        f[j] = BF16 ? __uint_as_float((j & 1) ? v[i][2 * c + (j >> 1)] & 0xffff0000u : v[i][2 * c + (j >> 1)] << 16)
                    : __uint_as_float(v[i][j]);
      o[c] = low_bytes(quantize_bits(f[0], s, y), quantize_bits(f[1], s, y), quantize_bits(f[2], s, y),
                       quantize_bits(f[3], s, y)) & keep;
    }
    if constexpr (PACKED) {
      const int e = (i * TPR + t) * VEC;
      if constexpr (BF16) *reinterpret_cast<u32x2*>(tile + r * LD + e) = u32x2{o[0], o[1]};
      else *reinterpret_cast<uint32_t*>(tile + r * LD + e) = o[0];
    } else {
      if constexpr (BF16) __builtin_amdgcn_raw_buffer_store_b64(u32x2{o[0], o[1]}, qres, t * VEC, i * TPR * VEC, 0);
      else __builtin_amdgcn_raw_buffer_store_b32(o[0], qres, t * VEC, i * TPR * VEC, 0);
    }
  }
  if constexpr (PACKED) {
    __syncthreads();
    // segment sg (16 columns) of row rr: eight rows side by side in memory
    int8_t* dst = q + (row0 >> 4) * kb * 1024 + (row0 & 8) * 16;
    for (int i = threadIdx.x; i < kb * 32; i += 1024) {
      const int rr = i & 7, sg = i >> 3;
      *reinterpret_cast<u32x4*>(dst + static_cast<int64_t>(sg >> 2) * 1024 + (sg & 3) * 256 + rr * 16) =
          *reinterpret_cast<const u32x4*>(tile + rr * LD + sg * 16);
    }
  }
}

// PACKED: write q in the packed tile layout (kb = packed_kblocks(k)) instead
// of row-major; a VEC-element group never straddles a 16-byte lane segment.
template <bool BF16, int VEC, bool PACKED>
__global__ __launch_bounds__(kQuantThreads) void quantize_rows_kernel(
    const void* __restrict__ w, int64_t k, int64_t kb, int8_t* __restrict__ q, float* __restrict__ scale) {
  const int64_t row = blockIdx.x;
  const int64_t nvec = k / VEC;
  const int64_t base = row * k;
  __shared__ uint32_t red[kQuantThreads / kWave];

  uint32_t mx = 0;
  for (int64_t v = threadIdx.x; v < nvec; v += kQuantThreads) {
    float f[VEC];
    load_row_vec<BF16, VEC>(w, base + v * VEC, f);
#pragma unroll
    for (int i = 0; i < VEC; ++i) mx = max(mx, abs_bits(f[i]));
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), off)));
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = mx;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kQuantThreads / kWave; ++i) mx = max(mx, red[i]);

  const float s = row_scale(mx);
  if (threadIdx.x == 0) scale[row] = s;
  const float y = 1.0f / s;
  const uint32_t keep = mx < kInfBits ? 0xffffffffu : 0u;

  for (int64_t v = threadIdx.x; v < nvec; v += kQuantThreads) {
    float f[VEC];
    load_row_vec<BF16, VEC>(w, base + v * VEC, f);
    const int64_t dst = PACKED ? packed_offset(row, v * VEC, kb) : base + v * VEC;
    if constexpr (VEC == 8) {
      uint32_t o[2];
#pragma unroll
      for (int c = 0; c < 2; ++c)
        o[c] = low_bytes(quantize_bits(f[4 * c], s, y), quantize_bits(f[4 * c + 1], s, y),
                         quantize_bits(f[4 * c + 2], s, y), quantize_bits(f[4 * c + 3], s, y)) & keep;
      *reinterpret_cast<u32x2*>(q + dst) = u32x2{o[0], o[1]};
    } else if constexpr (VEC == 4) {
      *reinterpret_cast<uint32_t*>(q + dst) =
          low_bytes(quantize_bits(f[0], s, y), quantize_bits(f[1], s, y), quantize_bits(f[2], s, y),
                    quantize_bits(f[3], s, y)) & keep;
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const int64_t d = PACKED ? packed_offset(row, v * VEC + i, kb) : base + v * VEC + i;
        q[d] = static_cast<int8_t>(quantize_bits(f[i], s, y) & keep);
      }
    }
  }
}

// q and out taken as flat arrays, so that any k reads and writes whole
// vectors (16 bytes of output per thread and item, consecutive threads side by
// side: full lines both ways): the E weights of an item lie in one row or, for
// k >= E, at most two.  IDX: 32-bit index arithmetic where the element count
// allows (one division per item).  Quantizing and dequantizing a [16000, 8000]
// fp32 weight row-major: 329 -> 244 us (5.2 TB/s).  ITEMS: one for up to 4 Mi
// weights, whose time is one thread's chain (bf16 of [976, 2048], with 1 / 2 / 4
// items 2.80 / 2.91 / 3.47 us), else two ([31250, 2048] 33.9 / 30.9 / 31.2).
template <int OUT, typename IDX, int ITEMS>
__global__ __launch_bounds__(256) void dequantize_flat_kernel(const int8_t* __restrict__ q,
                                                              const float* __restrict__ scale, IDX n, IDX k,
                                                              IDX total, void* __restrict__ out) {
  constexpr int E = OUT == PGS_DTYPE_F32 ? 4 : 8;
  const IDX first = (static_cast<IDX>(blockIdx.x) * (256 * ITEMS) + threadIdx.x) * E;
  uint32_t wv[ITEMS][E / 4];
  float s0[ITEMS], s1[ITEMS];
  int cut[ITEMS];  // weights of the item in its first row
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    IDX e = first + static_cast<IDX>(i) * 256 * E;
    e = e + E <= total ? e : 0;  // (in bounds: total >= k >= E)
    if constexpr (E == 8) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(q + e);
      wv[i][0] = v[0];
      wv[i][1] = v[1];
    } else {
      wv[i][0] = *reinterpret_cast<const uint32_t*>(q + e);
    }
    const IDX r = e / k, left = k - (e - r * k);
    cut[i] = left < E ? static_cast<int>(left) : E;
    s0[i] = scale[r];
    s1[i] = scale[r + 1 < n ? r + 1 : r];
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const IDX e = first + static_cast<IDX>(i) * 256 * E;
    if (e >= total) return;
    if (e + E > total) {  // the last, shorter item
      for (IDX j = e; j < total; ++j) store_dequant<OUT>(out, j, static_cast<float>(q[j]) * scale[j / k]);
      return;
    }
    float f[E];
#pragma unroll
    for (int c = 0; c < E / 4; ++c) {
      f[4 * c] = sbyte_to_f32<0>(wv[i][c]);
      f[4 * c + 1] = sbyte_to_f32<1>(wv[i][c]);
      f[4 * c + 2] = sbyte_to_f32<2>(wv[i][c]);
      f[4 * c + 3] = sbyte_to_f32<3>(wv[i][c]);
    }
#pragma unroll
    for (int j = 0; j < E; ++j) f[j] *= j < cut[i] ? s0[i] : s1[i];
    store_dequant16<OUT>(out, e, f);
  }
}

template <int OUT>
__global__ __launch_bounds__(256) void dequantize1_kernel(const int8_t* __restrict__ q,
                                                          const float* __restrict__ scale, int64_t k,
                                                          int64_t total, void* __restrict__ out) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= total) return;
  store_dequant<OUT>(out, e, static_cast<float>(q[e]) * scale[e / k]);
}

template <int OUT>
int launch_dequant(const int8_t* q, const float* scale, int64_t n, int64_t k, void* out, hipStream_t st) {
  const int64_t total = n * k;
  constexpr int E = OUT == PGS_DTYPE_F32 ? 4 : 8;
  // (up to 512 Ki weights of rows of no whole 16: by element, without the second
  // scale and the short last piece of the others: bf16 [97, 2047] 2.15 against 2.6 us)
  if (k >= E && aligned(q, 8) && aligned(out, 16) && (k % 16 == 0 || total > (1 << 19))) {
    const int64_t per = 256 * E * (total <= (4 << 20) ? 1 : 2);
    const unsigned blocks = static_cast<unsigned>((total + per - 1) / per);
    const dim3 grid(blocks), block(256);
    const uint32_t n32 = static_cast<uint32_t>(n), k32 = static_cast<uint32_t>(k), t32 = static_cast<uint32_t>(total);
    if (total <= (4 << 20))
      hipLaunchKernelGGL((dequantize_flat_kernel<OUT, uint32_t, 1>), grid, block, 0, st, q, scale, n32, k32, t32, out);
    else if (total + per < (1ll << 32))
      hipLaunchKernelGGL((dequantize_flat_kernel<OUT, uint32_t, 2>), grid, block, 0, st, q, scale, n32, k32, t32, out);
    else
      hipLaunchKernelGGL((dequantize_flat_kernel<OUT, int64_t, 2>), grid, block, 0, st, q, scale, n, k, total, out);
  } else {
    const int64_t blocks = (total + 255) / 256;
    hipLaunchKernelGGL(dequantize1_kernel<OUT>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, q, scale,
                       k, total, out);
  }
  return check_launch("pgs_dequantize");
}

// Whether the eight-row kernel is the faster one.  Its workgroups hold eight rows
// and wait for all of a row's loads, so it needs about one per CU; below that the
// n workgroups of the one-row kernel, small and read from L2 the second time, end
// sooner (one-row -> eight-row kernel, us).  Row-major fp32 [n, 2048] at n = 256 /
// 1024 / 1536 / 4096: 3.0 -> 4.2, 4.4 -> 4.7, 5.3 -> 5.3, 10.9 -> 9.0, and [n, 12288]
// at 256 / 512 / 1024: 9.0 -> 12.3, 12.9 -> 13.5, 18.7 -> 16.1; bf16 [n, 2048] at
// 1024 / 2048 / 4096: 3.8 -> 4.2, 5.0 -> 5.1, 7.6 -> 7.1.  Packed, whose one-row kernel
// writes parts of lines: fp32 [n, 2048] at 256 / 1024: 3.4 -> 4.4, 5.4 -> 4.9, [n,
// 12288] at 256 / 512: 10.7 -> 12.8, 16.6 -> 14.1.  Where padding is to be cleared the
// one-row kernel needs a fill launch: [150, 2048] 4.7 -> 4.1, only longer rows are
// sooner done with it ([150 | 600, 12288] 11.6 -> 12.4, 21.6 -> 14.6).
bool tile_quantizer(bool packed, bool f32, int64_t n, int64_t k) {
  if (packed && (n % 16 != 0 || k % 64 != 0)) return k <= 5120 || n >= 512;
  if (packed) return n >= 1024 || n * k >= 6 << 20;
  return f32 ? n >= 1536 || n * k >= 9 << 20 : n >= 2048;
}

template <bool PACKED>
int launch_quantize(const char* fn, const void* w, int w_dtype, int64_t n, int64_t k, int8_t* q, float* scale,
                    void* stream) {
  if (n < 0 || k < 0)
    return fail(PGS_ERR_INVALID_ARGUMENT, "%s: negative size n=%lld k=%lld", fn, (long long)n, (long long)k);
  if (w_dtype != PGS_DTYPE_F32 && w_dtype != PGS_DTYPE_BF16)
    return fail(PGS_ERR_INVALID_ARGUMENT, "%s: weight dtype code %d not fp32/bf16", fn, w_dtype);
  if (n == 0) return PGS_OK;
  if (n > 0x7fffffff) return fail(PGS_ERR_INVALID_ARGUMENT, "%s: n=%lld too large", fn, (long long)n);
  if (!scale || (k > 0 && (!w || !q))) return fail(PGS_ERR_INVALID_ARGUMENT, "%s: null pointer", fn);
  const size_t esz = (w_dtype == PGS_DTYPE_F32) ? 4 : 2;
  if (!aligned(w, esz) || !aligned(scale, 4))
    return fail(PGS_ERR_MISALIGNED, "%s: weight/scale not aligned to element size", fn);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (int rc = require_device(fn, st)) return rc;
  const int64_t kb = packed_kblocks(k);
  // rows of whole, aligned 16-byte pieces that fit the tile kernel's registers
  // and LDS: up to 12288 columns, in steps whose unused loads are few (the step at
  // 8192: fp32 [11008, 5128] row-major / packed 59.0 / 66.8 us, 74.3 / 76.8 in the
  // loads of 12288; 65.6 KB of LDS leave room for a second packed workgroup)
  const int vec = w_dtype == PGS_DTYPE_F32 ? 4 : 8;
  if (k > 0 && k % vec == 0 && k <= kTileMaxK && aligned(w, 16) && aligned(q, PACKED ? 16 : vec) &&
      tile_quantizer(PACKED, w_dtype == PGS_DTYPE_F32, n, k)) {
    const dim3 grid(static_cast<unsigned>(PACKED ? (n + 15) / 16 * 2 : (n + 7) / 8));
    const int kk = static_cast<int>(k), kbb = static_cast<int>(kb);
#define PGS_QUANT_TILE(BF, NV)                                                                                   \
  hipLaunchKernelGGL((quantize_tile_kernel<BF, NV, PACKED>), grid, dim3(1024), 0, st, w, n, kk, kbb, q, scale)
    if (w_dtype == PGS_DTYPE_F32) {
      if (k <= 1024) PGS_QUANT_TILE(false, 2);
      else if (k <= 2048) PGS_QUANT_TILE(false, 4);
      else if (k <= 5120) PGS_QUANT_TILE(false, 10);
      else if (k <= 8192) PGS_QUANT_TILE(false, 16);
      else PGS_QUANT_TILE(false, 24);
    } else {
      if (k <= 1024) PGS_QUANT_TILE(true, 1);
      else if (k <= 2048) PGS_QUANT_TILE(true, 2);
      else if (k <= 5120) PGS_QUANT_TILE(true, 5);
      else if (k <= 8192) PGS_QUANT_TILE(true, 8);
      else PGS_QUANT_TILE(true, 12);
    }
#undef PGS_QUANT_TILE
    return check_launch(fn);
  }
  if (PACKED && k > 0 && (n % 16 != 0 || k % 64 != 0)) {
    // padding rows/columns of the packed buffer must read as zero
    int rc = fill_zero(q, packed_bytes(n, k), st);
    if (rc) return rc;
  }
  dim3 grid(static_cast<unsigned>(n)), block(kQuantThreads);
  if (w_dtype == PGS_DTYPE_F32) {
    if (k % 4 == 0 && aligned(w, 16) && aligned(q, 4))
      hipLaunchKernelGGL((quantize_rows_kernel<false, 4, PACKED>), grid, block, 0, st, w, k, kb, q, scale);
    else
      hipLaunchKernelGGL((quantize_rows_kernel<false, 1, PACKED>), grid, block, 0, st, w, k, kb, q, scale);
  } else {
    if (k % 8 == 0 && aligned(w, 16) && aligned(q, 8))
      hipLaunchKernelGGL((quantize_rows_kernel<true, 8, PACKED>), grid, block, 0, st, w, k, kb, q, scale);
    else
      hipLaunchKernelGGL((quantize_rows_kernel<true, 1, PACKED>), grid, block, 0, st, w, k, kb, q, scale);
  }
  return check_launch(fn);
}

}  // namespace
}  // namespace pgs

using namespace pgs;

extern "C" int pgs_quantize_per_channel(const void* w, int w_dtype, int64_t n, int64_t k, int8_t* q,
                                        float* scale, void* stream) {
  return launch_quantize<false>("pgs_quantize_per_channel", w, w_dtype, n, k, q, scale, stream);
}

extern "C" int pgs_quantize_per_channel_packed(const void* w, int w_dtype, int64_t n, int64_t k, int8_t* packed,
                                               float* scale, void* stream) {
  return launch_quantize<true>("pgs_quantize_per_channel_packed", w, w_dtype, n, k, packed, scale, stream);
}

extern "C" int pgs_dequantize(const int8_t* q, const float* scale, int64_t n, int64_t k, void* out, int out_dtype,
                              void* stream) {
  if (n < 0 || k < 0)
    return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_dequantize: negative size n=%lld k=%lld", (long long)n, (long long)k);
  if (n == 0 || k == 0) return PGS_OK;
  if (!q || !scale || !out) return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_dequantize: null pointer");
  if (!aligned(scale, 4)) return fail(PGS_ERR_MISALIGNED, "pgs_dequantize: scale not 4-byte aligned");
  if (n * k / 16 > 0x7fffffffLL * 256LL)
    return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_dequantize: tensor too large");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (out_dtype != PGS_DTYPE_F32 && out_dtype != PGS_DTYPE_BF16 && out_dtype != PGS_DTYPE_F16)
    return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_dequantize: output dtype code %d not supported", out_dtype);
  if (int rc = require_device("pgs_dequantize", st)) return rc;
  switch (out_dtype) {
    case PGS_DTYPE_F32:
      if (!aligned(out, 4)) return fail(PGS_ERR_MISALIGNED, "pgs_dequantize: fp32 output not 4-byte aligned");
      return launch_dequant<PGS_DTYPE_F32>(q, scale, n, k, out, st);
    case PGS_DTYPE_BF16:
      if (!aligned(out, 2)) return fail(PGS_ERR_MISALIGNED, "pgs_dequantize: bf16 output not 2-byte aligned");
      return launch_dequant<PGS_DTYPE_BF16>(q, scale, n, k, out, st);
    case PGS_DTYPE_F16:
      if (!aligned(out, 2)) return fail(PGS_ERR_MISALIGNED, "pgs_dequantize: fp16 output not 2-byte aligned");
      return launch_dequant<PGS_DTYPE_F16>(q, scale, n, k, out, st);
    default:
      return fail(PGS_ERR_INVALID_ARGUMENT, "pgs_dequantize: output dtype code %d not supported", out_dtype);
  }
}
