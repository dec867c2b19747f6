// NF4 quantisation of a dense weight (the format step of loading a model):
// quant.py's torch steps in one pass over the weight, with their bits. Per
// block of bs elements of the flattened weight absmax = max |w| in fp32, each
// w * (1 / absmax) goes to the nearest code point (a value on a midpoint takes
// the lower one), two codes a byte, the even element in the high nibble.
//
// Bound by the read of the weight (9728 x 2560 bf16: 50 MB in, 14 MB out, 20
// us) and, in a whole call, by the host's allocations (53 us); the torch steps
// went over fp32 copies of it in 35 launches (587 us). A block's 8 elements a
// lane keep the absmax inside a wave, so the weight is read once.
#include "ttsp_common.h"

namespace ttsp {

namespace {

// The nearest code of v: torch.bucketize(v, mids, right=False) is the number
// of midpoints below v (all 15 for NaN). QBINS equal bins over [-1, 1] hold at
// most one midpoint each and none within 1e-3 of an edge (a CPU test checks
// both), so bin t's entry - the midpoints below it, and the next one - decides
// v with one comparison, whichever side of an edge v's rounded bin falls.
constexpr int QBINS = 64;

__device__ __forceinline__ uint32_t nearest(float v, const float2* tab) {
  const float t = fminf(fmaxf(__builtin_fmaf(v, QBINS / 2, QBINS / 2), 0.0f), (float)(QBINS - 1));
  const float2 e = tab[(int)t];
  const uint32_t q = __float_as_uint(e.x) + (e.y >= v ? 0u : 1u);
  return v != v ? 15u : q;
}

template <int DT>
__device__ __forceinline__ void load8(const void* A, long long i, float (&v)[8]) {
  if constexpr (DT == DT_F32) {
    const f32x4* p = reinterpret_cast<const f32x4*>((const float*)A + i);
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = a[j], v[4 + j] = b[j];
  } else {
    const u32x4 a = *reinterpret_cast<const u32x4*>((const uint16_t*)A + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[2 * j] = Elem<DT>::load(a[j]), v[2 * j + 1] = Elem<DT>::load(a[j] >> 16);
  }
}

constexpr int Q_CH = 4;  // 8-element chunks a lane takes, their loads in flight together

// Lane l of a wave holds 8 consecutive elements of each 512-element chunk: a
// block is bs / 8 neighbouring lanes (8 to 64). |w| is compared as its bit
// pattern, so a NaN (the largest pattern) is the block's absmax, as in torch.
template <int DT>
__global__ __launch_bounds__(256) void nf4_quantize_kernel(const void* __restrict__ A, long long n, int bs_shift,
                                                           const float* __restrict__ LUT, uint8_t* __restrict__ W,
                                                           float* __restrict__ AMAX) {
  __shared__ float2 tab[QBINS];
  const int lane = threadIdx.x & 63;
  const long long c0 = ((long long)blockIdx.x * 4 + (threadIdx.x >> 6)) * Q_CH;
  float v[Q_CH][8];
#pragma unroll
  for (int c = 0; c < Q_CH; ++c) {
    const long long i = (c0 + c) * 512 + 8 * lane;
    if (i + 8 <= n) {
      load8<DT>(A, i, v[c]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[c][j] = i + j < n ? load_elem(A, i + j, DT) : 0.0f;
    }
  }
  if (threadIdx.x < QBINS) {
    const float edge = (float)threadIdx.x * (2.0f / QBINS) - 1.0f;
    uint32_t below = 0;
    float next = __uint_as_float(0x7f800000u);
    for (int k = 14; k >= 0; --k) {
      const float mid = __fmul_rn(__fadd_rn(LUT[k], LUT[k + 1]), 0.5f);
      if (mid < edge) ++below;
      else next = mid;
    }
    tab[threadIdx.x] = make_float2(__uint_as_float(below), next);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < Q_CH; ++c) {
    const long long i = (c0 + c) * 512 + 8 * lane;
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) m = max(m, __float_as_uint(v[c][j]) & 0x7fffffffu);
    for (int d = 1; d < (1 << (bs_shift - 3)); d *= 2) m = max(m, (uint32_t)__shfl_xor((int)m, d));
    const float am = __uint_as_float(m);
    const float inv = am > 0.0f ? __fdiv_rn(1.0f, am) : 0.0f;
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= nearest(__fmul_rn(v[c][j], inv), tab) << (8 * (j >> 1) + (j & 1 ? 0 : 4));
    if (i >= n) continue;
    if ((i & ((1ll << bs_shift) - 1)) == 0) AMAX[i >> bs_shift] = am;
    if (i + 8 <= n) {
      *reinterpret_cast<uint32_t*>(W + i / 2) = w;
    } else {
      for (int j = 0; 2 * j < n - i; ++j) W[i / 2 + j] = (uint8_t)(w >> (8 * j));
    }
  }
}

// Blocks of 256 values (X - *OFFSET) to the nearest of 256 ascending code
// points: one workgroup a block, one value a thread, the midpoint count by
// bisection over the 255 midpoints in LDS.
__global__ __launch_bounds__(256) void quantize_scales_kernel(const float* __restrict__ X, long long n,
                                                              const float* __restrict__ OFFSET,
                                                              const float* __restrict__ CODE, uint8_t* __restrict__ Q,
                                                              float* __restrict__ AMAX) {
  __shared__ float mids[256];
  __shared__ uint32_t part[4];
  const int tid = threadIdx.x;
  const long long i = (long long)blockIdx.x * 256 + tid;
  const float x = i < n ? __fsub_rn(X[i], OFFSET[0]) : 0.0f;
  if (tid < 255) mids[tid] = __fmul_rn(__fadd_rn(CODE[tid], CODE[tid + 1]), 0.5f);
  uint32_t m = __float_as_uint(x) & 0x7fffffffu;
  for (int d = 1; d < 64; d *= 2) m = max(m, (uint32_t)__shfl_xor((int)m, d));
  if ((tid & 63) == 0) part[tid >> 6] = m;
  __syncthreads();
  const float am = __uint_as_float(max(max(part[0], part[1]), max(part[2], part[3])));
  if (tid == 0) AMAX[blockIdx.x] = am;
  if (i >= n) return;
  const float v = __fmul_rn(x, am > 0.0f ? __fdiv_rn(1.0f, am) : 0.0f);
  int q = 0;
#pragma unroll
  for (int s = 128; s; s >>= 1)
    if (!(mids[q + s - 1] >= v)) q += s;
  Q[i] = (uint8_t)q;
}

}  // namespace
}  // namespace ttsp

using namespace ttsp;

// A (16-byte aligned, n elements of fp16 / bf16 / fp32, n even) to packed
// codes W (4-byte aligned, n / 2 bytes) and fp32 AMAX; blocksize 64 to 512.
extern "C" int ttsp_nf4_quantize(const void* A, int dtype, long long n, int blocksize, const float* LUT, uint8_t* W,
                                 float* AMAX, hipStream_t stream) {
  int bs = 6;
  while (bs < 9 && (1 << bs) < blocksize) ++bs;
  if ((1 << bs) != blocksize || n < 0 || n % 2 || !LUT) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  if (!A || !W || !AMAX || (uintptr_t)A % 16 || (uintptr_t)W % 4) return (int)hipErrorInvalidValue;
  const long long per = 4ll * Q_CH * 512, blocks = (n + per - 1) / per;
  if (blocks > 0x7fffffffll) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks);
  if (dtype == DT_BF16)
    hipLaunchKernelGGL(nf4_quantize_kernel<DT_BF16>, grid, dim3(256), 0, stream, A, n, bs, LUT, W, AMAX);
  else if (dtype == DT_F16)
    hipLaunchKernelGGL(nf4_quantize_kernel<DT_F16>, grid, dim3(256), 0, stream, A, n, bs, LUT, W, AMAX);
  else if (dtype == DT_F32)
    hipLaunchKernelGGL(nf4_quantize_kernel<DT_F32>, grid, dim3(256), 0, stream, A, n, bs, LUT, W, AMAX);
  else
    return (int)hipErrorInvalidValue;
  TTSP_RETURN_LAUNCH();
}

// The second level: X - *OFFSET in blocks of 256 to indices into the 256
// ascending points of CODE, with fp32 AMAX per block.
extern "C" int ttsp_quantize_scales(const float* X, long long n, const float* OFFSET, const float* CODE, uint8_t* Q,
                                    float* AMAX, hipStream_t stream) {
  if (n < 0 || n > 0x7fffffffll * 256) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  if (!X || !OFFSET || !CODE || !Q || !AMAX) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(quantize_scales_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, X, n, OFFSET,
                     CODE, Q, AMAX);
  TTSP_RETURN_LAUNCH();
}
