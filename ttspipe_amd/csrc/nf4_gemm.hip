// The launch plans of the NF4 matrix products, the reduce kernels of their K
// splits and the C entry points. The products themselves: nf4_gemv.hip (one
// and two rows), nf4_skinny.hip (to 16), nf4_gemm_few.hip (9 to 64),
// nf4_gemm_tile.hip (65 to 512) and nf4_gemm_dense.hip (more).
#include "gemv_common.h"

namespace ttsp {

constexpr int KT = 64;  // codes per K-step

// Y[n][m] = epilogue(round(sum over z of YP[z][n][m])), the sum in z order;
// 8 consecutive m per thread (16-byte stores when vec).
template <int DT>
__global__ __launch_bounds__(256) void nf4_gemm_reduce_kernel(const float* __restrict__ YP, int splits,
                                                              uint16_t* __restrict__ Y,
                                                              const uint16_t* __restrict__ R, int epi, int M,
                                                              int N) {
  const int chunks = (M + 7) / 8;
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= (long long)chunks * N) return;
  const int n = (int)(c / chunks), m = (int)(c % chunks) * 8;
  const bool vec = (epi & 4) != 0;
  const int ep = epi & 3;
  const size_t o = (size_t)n * M + m;
  float acc[8];
  if (vec && m + 8 <= M) {
    const float4* p = reinterpret_cast<const float4*>(YP + o);
    float4 a = p[0], b = p[1];
    for (int z = 1; z < splits; ++z) {
      const float4* q = reinterpret_cast<const float4*>(YP + (size_t)z * N * M + o);
      const float4 u = q[0], v = q[1];
      a.x += u.x, a.y += u.y, a.z += u.z, a.w += u.w;
      b.x += v.x, b.y += v.y, b.z += v.z, b.w += v.w;
    }
    acc[0] = a.x, acc[1] = a.y, acc[2] = a.z, acc[3] = a.w, acc[4] = b.x, acc[5] = b.y, acc[6] = b.z, acc[7] = b.w;
    uint32_t rw[4] = {0u, 0u, 0u, 0u};
    if (ep) {
      const uint4 rv = *reinterpret_cast<const uint4*>(R + o);
      rw[0] = rv.x, rw[1] = rv.y, rw[2] = rv.z, rw[3] = rv.w;
    }
    uint32_t ow[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t h2[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float y = Elem<DT>::load(Elem<DT>::store(acc[2 * q + u]));
        const float r = Elem<DT>::load(rw[q] >> (16 * u));
        float v = y;
        if (ep == 1) v = __fadd_rn(r, y);
        else if (ep == 2) v = __fmul_rn(Elem<DT>::load(Elem<DT>::store(silu_rn(r))), y);
        h2[u] = Elem<DT>::store(v);
      }
      ow[q] = h2[0] | (h2[1] << 16);
    }
    *reinterpret_cast<uint4*>(Y + o) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
  } else {
    for (int u = 0; u < 8 && m + u < M; ++u) {
      float a = YP[o + u];
      for (int z = 1; z < splits; ++z) a += YP[(size_t)z * N * M + o + u];
      const float y = Elem<DT>::load(Elem<DT>::store(a));
      float v = y;
      if (ep == 1) v = __fadd_rn(Elem<DT>::load(R[o + u]), y);
      else if (ep == 2) v = __fmul_rn(Elem<DT>::load(Elem<DT>::store(silu_rn(Elem<DT>::load(R[o + u])))), y);
      Y[o + u] = Elem<DT>::store(v);
    }
  }
}

// The split-K reduce, its epilogue and the fork's RMSNorm of each output row
// in one launch: Y is nf4_gemm_reduce_kernel's output, YN = rms_norm(Y, G, eps)
// with rms_norm_kernel's order (chunk c of 8 values by lane c % 64 in step
// c / 64, each chunk an fma chain of squares, DPP sums, steps left to right).
// One workgroup per output row with a wave per step (64 * ceil(M / 512)
// threads, at most 8 waves): each wave issues all of its loads - the splits'
// partials, the residual and the norm weight - before using any, so the row
// costs one memory round trip; the step sums meet in LDS.
// M % 8 == 0, M <= 64 * 8 * NRM_CH.
constexpr int NRM_CH = 8;
template <int DT, int S>
__global__ __launch_bounds__(64 * NRM_CH) void nf4_gemm_reduce_norm_kernel(const float* __restrict__ YP,
                                                                          uint16_t* __restrict__ Y,
                                                                          const uint16_t* __restrict__ R, int epi,
                                                                          int M, int N,
                                                                          const uint16_t* __restrict__ G, float eps,
                                                                          uint16_t* __restrict__ YN) {
  __shared__ float step_sum[NRM_CH];
  const int lane = threadIdx.x & 63, j = threadIdx.x >> 6;  // this wave's step
  const int n = blockIdx.x;
  const int nc = M >> 3, ep = epi & 3, nsteps = (nc + 63) >> 6;
  const int c = min(lane + 64 * j, nc - 1);
  const size_t o = (size_t)n * M + 8 * (size_t)c;
  float4 p[S][2];
#pragma unroll
  for (int z = 0; z < S; ++z) {
    const float4* q = reinterpret_cast<const float4*>(YP + (size_t)z * N * M + o);
    p[z][0] = q[0];
    p[z][1] = q[1];
  }
  const uint4 rv = ep ? *reinterpret_cast<const uint4*>(R + o) : make_uint4(0, 0, 0, 0);
  const uint4 gv = *reinterpret_cast<const uint4*>(G + 8 * (size_t)c);
  const uint32_t rw[4] = {rv.x, rv.y, rv.z, rv.w};
  uint32_t ow[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t h2[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = 2 * q + u;  // element of the chunk, in the reduce kernel's order
      float a = e < 4 ? (&p[0][0].x)[e] : (&p[0][1].x)[e - 4];
#pragma unroll
      for (int z = 1; z < S; ++z) a += e < 4 ? (&p[z][0].x)[e] : (&p[z][1].x)[e - 4];
      const float y = Elem<DT>::load(Elem<DT>::store(a));
      const float r = Elem<DT>::load(rw[q] >> (16 * u));
      float v = y;
      if (ep == 1) v = __fadd_rn(r, y);
      else if (ep == 2) v = __fmul_rn(Elem<DT>::load(Elem<DT>::store(silu_rn(r))), y);
      h2[u] = Elem<DT>::store(v);
    }
    ow[q] = h2[0] | (h2[1] << 16);
  }
  const uint4 h = make_uint4(ow[0], ow[1], ow[2], ow[3]);
  const bool own = lane + 64 * j < nc;
  if (own) *reinterpret_cast<uint4*>(Y + o) = h;
  const float part = wave_sum_dpp(own ? sumsq8<DT>(h, 0.0f) : 0.0f);
  if (lane == 0) step_sum[j] = part;
  __syncthreads();
  float ss = step_sum[0];
  for (int k = 1; k < nsteps; ++k) ss = __fadd_rn(ss, step_sum[k]);
  const float rr = rsqrt_rn(__fadd_rn(__fdiv_rn(ss, (float)M), eps));
  if (own) *reinterpret_cast<uint4*>(YN + o) = norm8<DT>(h, gv, rr);
}

// K splits of the split entry (ttsp_nf4_gemm_split and the forms that leave or
// add its sums): none where 64 x 128 tiles give every CU a workgroup; up to
// 128 tiles the largest split (2, 4, 8; each an even number of at least 8
// K-steps) whose workgroups fit one to a CU: a split's fp32 partial sums cost
// a write and a read of splits x N x M floats, so a second pass of workgroups
// only pays where each split keeps a long K run. Between 128 and 256 tiles 4
// splits pay only past 16 K-steps each. 256 to 512 rows: span_plan below. 33 to
// 64 rows: 4 ways where each split keeps 8 or more K-steps, else 2 (callers
// with a choice take ttsp_nf4_gemm_few's plan, which is faster). Up to 32 rows
// the few-row or the skinny kernel unsplit, but for K past their longest rows.
constexpr int SKINNY_MAX_N = 16;
int skinny_max_k();
bool few_unsplit(int M, int K, int N);
int few_splits(int M, int K, int N);
bool few_pair(int M, int K, int N);
// Up to 64 rows, unsplit: the few-row kernel, or up to 16 the skinny one.
static bool skinny(int K, int N) { return N <= SKINNY_MAX_N && K <= skinny_max_k(); }

static long long gemm_tiles(int M, int N, int bm, int bn) {
  return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

constexpr int SPLIT_SMALL_N = 32;

int gemm_tile(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
              float offset, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int bs_shift,
              int bs2_shift, int splits, float* YP, hipStream_t st);

// 256 to 512 rows: 4 K-splits where K has 64 or more steps and there are at
// least 75 64 x 128 tiles; with fewer steps none from 512 tiles and 2 from 300.
// 0: no rule here.
constexpr int SPAN_MIN_N = 256, SPAN_MAX_N = 512;
static int span_plan(int M, int K, int N) {
  if (N < SPAN_MIN_N || N > SPAN_MAX_N) return 0;
  const int steps = K / KT;
  const long long t = gemm_tiles(M, N, 64, 128);
  if (steps >= 64) return t >= 75 && steps % 8 == 0 && steps / 4 <= 64 ? 4 : 0;
  if (t >= 512) return 1;
  return t >= 300 && steps % 4 == 0 ? 2 : 0;
}

static int gemm_plan(int M, int K, int N) {
  const int steps = K / KT;
  if (N > SPLIT_SMALL_N && N <= 64)
    for (int sp = 4; sp >= 2; sp /= 2)
      if (steps % (2 * sp) == 0 && steps / sp >= 8) return sp;
  if (skinny(K, N) || few_unsplit(M, K, N)) return 1;
  if (const int span = span_plan(M, K, N)) return span;
  const long long t = gemm_tiles(M, N, 64, 128);
  if (t >= 256) return 1;
  int splits = 1;
  if (t > 128) {
    if (steps % 8 == 0 && steps / 4 > 16) splits = 4;
  } else {
    for (int sp = 2; sp <= 8; sp *= 2) {
      if (steps % (2 * sp) || steps / sp < 8 || t * sp > 256) break;
      splits = sp;
    }
  }
  return splits;
}

int gemm_few(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
             float offset, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int bs_shift,
             int bs2_shift, int splits, float* YP, hipStream_t st);
bool few_takes(int M, int K, int N);

// Y = epilogue(round(sum of the splits' partials)) (epi bit 2: vectorised)
int gemm_reduce(int dt, const float* YP, int splits, void* Y, const void* R, int epi, int M, int N, hipStream_t st) {
  const long long chunks = (long long)((M + 7) / 8) * N;
  const dim3 rg((unsigned)((chunks + 255) / 256));
  if (dt == DT_BF16)
    hipLaunchKernelGGL(nf4_gemm_reduce_kernel<DT_BF16>, rg, dim3(256), 0, st, YP, splits, (uint16_t*)Y,
                       (const uint16_t*)R, epi, M, N);
  else
    hipLaunchKernelGGL(nf4_gemm_reduce_kernel<DT_F16>, rg, dim3(256), 0, st, YP, splits, (uint16_t*)Y,
                       (const uint16_t*)R, epi, M, N);
  TTSP_RETURN_LAUNCH();
}

// gemm_reduce with the fork's RMSNorm of each row to YN (2, 4 or 8 splits; M
// and the pointers as nf4_gemm_reduce_norm_kernel takes them, checked by the caller)
static int gemm_reduce_norm(int x_dtype, const float* work, int splits, void* Y, const void* R, int epi, int M, int N,
                            const void* G, float eps, void* YN, hipStream_t stream) {
  const dim3 grid((unsigned)N), block((unsigned)(64 * ((M / 8 + 63) / 64)));
#define TTSP_RN(DTV, SV)                                                                                      \
  hipLaunchKernelGGL((nf4_gemm_reduce_norm_kernel<DTV, SV>), grid, block, 0, stream, work, (uint16_t*)Y, \
                     (const uint16_t*)R, epi, M, N, (const uint16_t*)G, eps, (uint16_t*)YN)
#define TTSP_RS(DTV)                  \
  if (splits == 2) TTSP_RN(DTV, 2);   \
  else if (splits == 4) TTSP_RN(DTV, 4); \
  else TTSP_RN(DTV, 8);
  if (x_dtype == DT_BF16) {
    TTSP_RS(DT_BF16)
  } else {
    TTSP_RS(DT_F16)
  }
#undef TTSP_RS
#undef TTSP_RN
  TTSP_RETURN_LAUNCH();
}

// A product in `splits` K splits: the few-row kernel where it takes the rows,
// else the tiles. splits > 1 leaves the sums in YP, and with reduce adds them
// (epi bit 2: vectorised output).
int gemm_mfma(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
              float offset, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int bs_shift,
              int bs2_shift, int splits, float* YP, hipStream_t st, bool reduce = true) {
  if (K % (2 * KT)) return (int)hipErrorInvalidValue;
  if (splits > 1 && (!YP || (K / KT) % (2 * splits))) return (int)hipErrorInvalidValue;
  const bool few = few_takes(M, K, N);
  if (int rc = few ? gemm_few(X, dt, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits,
                              YP, st)
                   : gemm_tile(X, dt, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits,
                               YP, st))
    return rc;
  if (splits > 1 && reduce) return gemm_reduce(dt, YP, splits, Y, R, epi, M, N, st);
  return 0;
}

bool gemv_fits(int M, int K, int blocksize, int N);
int gemv_rows(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX,
              const float* CODE2, float offset, const float* LUT, void* Y, const void* R, int epi,
              int M, int K, int N, int blocksize, int blocksize2, hipStream_t st);
// Up to this many activation rows take the GEMV (each weight byte looked up
// once, one fp32 chain per row) rather than the few-row MFMA kernel: two rows
// cost 1.0-1.3x one row that way (gate 9728 x 2560: 7.5 against 9.4 us).
constexpr int GEMV_ROWS_N = 2;
int gemm_skinny(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
                float offset, const float* LUT, void* Y, const void* RES, int epi, int M, int K, int N, int bs_shift,
                int bs2_shift, hipStream_t st);
int gemm_tile_swiglu(const void* X, int dt, const uint8_t* W1, const uint8_t* A8_1, const float* AMAX_1,
                     const float* CODE2_1, float offset_1, const uint8_t* W3, const uint8_t* A8_3, const float* AMAX_3,
                     const float* CODE2_3, float offset_3, const float* LUT, void* Y, int M, int K, int N, int bs_shift,
                     int bs2_shift, hipStream_t st);
int gemm_skinny_pair(const void* X, int dt, const uint8_t* W1, const uint8_t* A8_1, const float* AMAX_1,
                     const float* CODE2_1, float offset_1, const uint8_t* W3, const uint8_t* A8_3, const float* AMAX_3,
                     const float* CODE2_3, float offset_3, const float* LUT, void* Y, int M, int K, int N, int bs_shift,
                     int bs2_shift, hipStream_t st);
bool skinny_pair_fits(int K, int N);
int gemm_few_pair(const void* X, int dt, const uint8_t* W1, const uint8_t* A8_1, const float* AMAX_1,
                  const float* CODE2_1, float offset_1, const uint8_t* W3, const uint8_t* A8_3, const float* AMAX_3,
                  const float* CODE2_3, float offset_3, const float* LUT, void* Y, int M, int K, int N, int bs_shift,
                  int bs2_shift, hipStream_t st);

// Whether the SwiGLU pair takes the few-row or the skinny kernel's pair form:
// where each of its two GEMMs would run that kernel (3 to 32 rows, unsplit;
// two rows take the GEMV, whose one-launch pair is ttsp_nf4_gemv_fused_rows).
static bool swiglu_skinny(int M, int K, int N) {
  if (M <= 0 || K <= 0 || K % 128 || N <= GEMV_ROWS_N) return false;
  return few_unsplit(M, K, N) ? few_pair(M, K, N) : skinny_pair_fits(K, N);
}

// Whether the SwiGLU pair fits one launch of the tile kernel: where each of
// its two GEMMs runs that kernel unsplit and over whole K (256 to 512 rows of
// at least 512 64 x 128 tiles and K below 4096), so that the one launch gives
// their bits. One launch against w1 and then w3 with the gate: 9728 x 2560 at
// 385 rows 74 / 78 us, at 512 73.5 / 76. (Second-level groups shorter than K take
// two launches; the kernel would serve them.)
static bool swiglu_fits(int M, int K, int N, int bs_shift, int bs2_shift, bool nested) {
  if (M <= 0 || K <= 0 || K % 128 || N <= 64 || span_plan(M, K, N) != 1) return false;
  return !(nested && (long long)K > (1LL << (bs_shift + bs2_shift)));
}

}  // namespace ttsp

using namespace ttsp;

// Argument checks shared by the entry points; fills the scale shifts.
static int gemm_args(const void* X, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
                     const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int blocksize,
                     int blocksize2, int* bs_shift, int* bs2_shift) {
  if (N <= 0 || M <= 0 || K <= 0 || !X || !W || !AMAX || !LUT || !Y) return (int)hipErrorInvalidValue;
  if (A8 && !CODE2) return (int)hipErrorInvalidValue;
  *bs_shift = 0, *bs2_shift = 0;
  while ((1 << *bs_shift) < blocksize) ++*bs_shift;
  if (A8)
    while ((1 << *bs2_shift) < blocksize2) ++*bs2_shift;
  if ((1 << *bs_shift) != blocksize || *bs_shift < 6 || (A8 && (1 << *bs2_shift) != blocksize2))
    return (int)hipErrorInvalidValue;
  if (K % 128 || K % blocksize || epi < 0 || epi > 2 || (epi && !R)) return (int)hipErrorInvalidValue;
  return 0;
}

// One entry for every row count: up to GEMV_ROWS_N rows take the
// bandwidth-bound GEMV (or, past the rows it holds, the kernels below), up
// to 64 rows the skinny or the few-row MFMA kernel (weights streamed once),
// more rows the tile kernel (weights read once per 128 rows), unsplit.
extern "C" int ttsp_nf4_gemm(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8,
                             const float* AMAX, const float* CODE2, float offset, const float* LUT,
                             void* Y, const void* R, int epi, int M, int K, int N, int blocksize,
                             int blocksize2, hipStream_t stream) {
  if (N >= 1 && N <= GEMV_ROWS_N && M > 0 && K > 0 && X && W && AMAX && LUT && Y && (!A8 || CODE2) &&
      gemv_fits(M, K, blocksize, N))
    return gemv_rows(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, blocksize, blocksize2,
                     stream);
  int bs_shift, bs2_shift;
  if (int rc = gemm_args(X, W, A8, AMAX, CODE2, LUT, Y, R, epi, M, K, N, blocksize, blocksize2, &bs_shift,
                         &bs2_shift))
    return rc;
  // (one row whose K the GEMV cannot hold, K > 32768, takes the tiled kernel below)
  if (few_unsplit(M, K, N))
    return gemm_few(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, 1, nullptr,
                    stream);
  if (N >= 2 && skinny(K, N))
    return gemm_skinny(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, stream);
  return gemm_mfma(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, 1, nullptr,
                   stream);
}

extern "C" int ttsp_nf4_gemm_splits(int M, int K, int N) {
  if (M <= 0 || K <= 0 || N <= 1 || K % 128) return 1;
  return gemm_plan(M, K, N);
}

// The splits a caller with a workspace should take from 65 rows:
// ttsp_nf4_gemm_splits', but from 256 rows unsplit instead of 2 ways where no
// norm follows in the reduce (M past its widest row; with the reduce, us, 1
// split against 2: 9728 x 2560 at 256 rows 27.6 / 31.8, 6144 x 2560 at 512 27.9
// / 33.7, 7168 x 2048 at 385 24.8 / 31.7; sums that another kernel adds keep
// the two splits); and 2 instead of 4 where a split still has 32 K-steps or
// more but fewer than 64: half the sums to reduce, which a wide weight feels (2
// splits against 4: 2560 x 4096 at 256 rows 22.9 / 22.5, at 385 26.9 / 25.6, at
// 512 27.6 / 27.4; 5120 x 5120 at 512 45.2 / 57.4, 14336 x 4096 88.6 / 111.7).
namespace ttsp {

int tile_splits(int M, int K, int N) {
  if (M <= 0 || K <= 0 || N <= 1 || K % 128) return 1;
  const int span = span_plan(M, K, N), plan = gemm_plan(M, K, N);
  if (N <= 64 || !span) return plan;
  if (M > 64 * 8 * NRM_CH && span == 2) return 1;
  return span == 4 && K / KT < 128 && K / KT % 4 == 0 ? 2 : plan;
}

// Estimated us of the tile kernel from 65 rows: rounds of 256 workgroups, each
// its K-steps (measured a step: 0.75 us with both K halves in a workgroup,
// 0.95 of 256 weight rows, 0.66 of 128) and ~5 us of first loads and epilogue;
// a split's sums and reduce as the dense plan prices them. The forms follow
// nf4_gemm_tile.hip's choice.
double tile_estimate(int M, int K, int N) {
  const int z = tile_splits(M, K, N), steps = K / KT / z;
  const long long t64 = gemm_tiles(M, N, 64, 128) * z, t128 = gemm_tiles(M, N, 128, 128) * z,
                  t256 = gemm_tiles(M, N, 256, 128) * z;
  double us = t64 <= 256 ? steps / 2 * 0.75 + 5.0
              : t256 > 128 ? (double)((t256 + 255) / 256) * (steps * 0.95 + 5.0)
                            : (double)((t128 + 255) / 256) * (steps * 0.66 + 5.0);
  if (z > 1) us += 4.0 + (double)z * N * M * 8.0 / 4e6;
  return us;
}

}  // namespace ttsp

extern "C" int ttsp_nf4_gemm_tile_splits(int M, int K, int N) { return tile_splits(M, K, N); }

extern "C" int ttsp_nf4_gemm_split(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8,
                                   const float* AMAX, const float* CODE2, float offset, const float* LUT,
                                   void* Y, const void* R, int epi, int M, int K, int N, int blocksize,
                                   int blocksize2, float* work, int splits, hipStream_t stream) {
  if (N <= 1 || splits < 1 || (splits != ttsp_nf4_gemm_splits(M, K, N) && splits != tile_splits(M, K, N)))
    return (int)hipErrorInvalidValue;
  if (splits == 1)
    return ttsp_nf4_gemm(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, blocksize,
                         blocksize2, stream);
  int bs_shift, bs2_shift;
  if (int rc = gemm_args(X, W, A8, AMAX, CODE2, LUT, Y, R, epi, M, K, N, blocksize, blocksize2, &bs_shift,
                         &bs2_shift))
    return rc;
  if (!work || (uintptr_t)work % 16) return (int)hipErrorInvalidValue;
  const bool vec = M % 8 == 0 && (uintptr_t)Y % 16 == 0 && (!epi || (uintptr_t)R % 16 == 0);
  return gemm_mfma(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi | (vec ? 4 : 0), M, K, N, bs_shift,
                   bs2_shift, splits, work, stream);
}

static int log2_of(int v) {
  int sh = 0;
  while (sh < 30 && (1 << sh) < v) ++sh;
  return (1 << sh) == v ? sh : -1;
}

extern "C" int ttsp_nf4_gemm_swiglu_fits(int M, int K, int N, int blocksize, int blocksize2, int nested) {
  const int bs = log2_of(blocksize), bs2 = nested ? log2_of(blocksize2) : 0;
  if (bs < 6 || bs2 < 0 || K % blocksize) return 0;
  return swiglu_skinny(M, K, N) || swiglu_fits(M, K, N, bs, bs2, nested != 0) ? 1 : 0;
}

extern "C" int ttsp_nf4_gemm_swiglu(const void* X, int x_dtype, const uint8_t* W1, const uint8_t* A8_1,
                                    const float* AMAX_1, const float* CODE2_1, float offset_1, const uint8_t* W3,
                                    const uint8_t* A8_3, const float* AMAX_3, const float* CODE2_3,
                                    float offset_3, const float* LUT, void* Y, int M, int K, int N, int blocksize,
                                    int blocksize2, hipStream_t stream) {
  int bs_shift, bs2_shift;
  if (int rc = gemm_args(X, W1, A8_1, AMAX_1, CODE2_1, LUT, Y, nullptr, 0, M, K, N, blocksize, blocksize2,
                         &bs_shift, &bs2_shift))
    return rc;
  if (!W3 || !AMAX_3 || (A8_3 != nullptr) != (A8_1 != nullptr) || (A8_3 && !CODE2_3))
    return (int)hipErrorInvalidValue;
  if ((uintptr_t)X % 16 || (uintptr_t)W1 % 16 || (uintptr_t)W3 % 16) return (int)hipErrorInvalidValue;
  if (few_pair(M, K, N))
    return gemm_few_pair(X, x_dtype, W1, A8_1, AMAX_1, CODE2_1, offset_1, W3, A8_3, AMAX_3, CODE2_3, offset_3, LUT, Y,
                         M, K, N, bs_shift, bs2_shift, stream);
  if (swiglu_skinny(M, K, N))
    return gemm_skinny_pair(X, x_dtype, W1, A8_1, AMAX_1, CODE2_1, offset_1, W3, A8_3, AMAX_3, CODE2_3, offset_3, LUT,
                            Y, M, K, N, bs_shift, bs2_shift, stream);
  if (!swiglu_fits(M, K, N, bs_shift, bs2_shift, A8_1 != nullptr)) return (int)hipErrorInvalidValue;
  return gemm_tile_swiglu(X, x_dtype, W1, A8_1, AMAX_1, CODE2_1, offset_1, W3, A8_3, AMAX_3, CODE2_3, offset_3, LUT, Y,
                        M, K, N, bs_shift, bs2_shift, stream);
}

extern "C" int ttsp_nf4_gemm_partials(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8,
                                      const float* AMAX, const float* CODE2, float offset, const float* LUT, int M,
                                      int K, int N, int blocksize, int blocksize2, float* work, int splits,
                                      hipStream_t stream) {
  if (N <= 1 || splits < 2 || splits != ttsp_nf4_gemm_splits(M, K, N) || !work || (uintptr_t)work % 16)
    return (int)hipErrorInvalidValue;
  int bs_shift, bs2_shift;
  // (Y is not written: the split launch stops at its partial sums)
  if (int rc = gemm_args(X, W, A8, AMAX, CODE2, LUT, work, nullptr, 0, M, K, N, blocksize, blocksize2, &bs_shift,
                         &bs2_shift))
    return rc;
  return gemm_mfma(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, nullptr, nullptr, 0, M, K, N, bs_shift, bs2_shift,
                   gemm_plan(M, K, N), work, stream, false);
}

extern "C" int ttsp_nf4_gemm_split_norm(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8,
                                        const float* AMAX, const float* CODE2, float offset, const float* LUT,
                                        void* Y, const void* R, int epi, int M, int K, int N, int blocksize,
                                        int blocksize2, float* work, int splits, const void* G, float eps, void* YN,
                                        hipStream_t stream) {
  if (N <= 1 || (splits != 2 && splits != 4 && splits != 8) ||
      (splits != ttsp_nf4_gemm_splits(M, K, N) && splits != tile_splits(M, K, N)))
    return (int)hipErrorInvalidValue;
  if (M % 8 || M > 64 * 8 * NRM_CH || !G || !YN || !work) return (int)hipErrorInvalidValue;
  if ((uintptr_t)Y % 16 || (uintptr_t)YN % 16 || (uintptr_t)G % 16 || (uintptr_t)work % 16 ||
      (epi && (uintptr_t)R % 16))
    return (int)hipErrorInvalidValue;
  if (x_dtype != DT_BF16 && x_dtype != DT_F16) return (int)hipErrorInvalidValue;
  int bs_shift, bs2_shift;
  if (int rc = gemm_args(X, W, A8, AMAX, CODE2, LUT, Y, R, epi, M, K, N, blocksize, blocksize2, &bs_shift,
                         &bs2_shift))
    return rc;
  if (int rc = gemm_mfma(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift,
                         splits, work, stream, false))
    return rc;
  return gemm_reduce_norm(x_dtype, work, splits, Y, R, epi, M, N, G, eps, YN, stream);
}

// ---- 9 to 64 rows with the sums of K splits in a caller's workspace

extern "C" int ttsp_nf4_gemm_few_splits(int M, int K, int N) { return few_splits(M, K, N); }

extern "C" int ttsp_nf4_gemm_few(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8, const float* AMAX,
                                 const float* CODE2, float offset, const float* LUT, void* Y, const void* R, int epi,
                                 int M, int K, int N, int blocksize, int blocksize2, float* work, const void* G,
                                 float eps, void* YN, hipStream_t stream) {
  const int splits = few_splits(M, K, N);
  if (splits < 1 || (splits > 1 && (!work || (uintptr_t)work % 16)) || (!Y && (splits == 1 || G)))
    return (int)hipErrorInvalidValue;
  int bs_shift, bs2_shift;
  if (int rc = gemm_args(X, W, A8, AMAX, CODE2, LUT, Y ? Y : work, R, epi, M, K, N, blocksize, blocksize2, &bs_shift,
                         &bs2_shift))
    return rc;
  if (G) {
    if (splits == 1 || M % 8 || M > 64 * 8 * NRM_CH || !YN) return (int)hipErrorInvalidValue;
    if ((uintptr_t)Y % 16 || (uintptr_t)YN % 16 || (uintptr_t)G % 16 || (epi && (uintptr_t)R % 16))
      return (int)hipErrorInvalidValue;
  }
  if (x_dtype != DT_BF16 && x_dtype != DT_F16) return (int)hipErrorInvalidValue;
  if (int rc = gemm_few(X, x_dtype, W, A8, AMAX, CODE2, offset, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits,
                        work, stream))
    return rc;
  if (splits == 1 || !Y) return 0;
  if (G) return gemm_reduce_norm(x_dtype, work, splits, Y, R, epi, M, N, G, eps, YN, stream);
  const bool vec = M % 8 == 0 && (uintptr_t)Y % 16 == 0 && (!epi || (uintptr_t)R % 16 == 0);
  return gemm_reduce(x_dtype, work, splits, Y, R, epi | (vec ? 4 : 0), M, N, stream);
}
