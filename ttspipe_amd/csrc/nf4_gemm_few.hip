// NF4 matrix product for 9 to 64 activation rows: Y[N][M] = X[N][K] . W^T, the
// weight in the bitsandbytes NF4 layout (nf4_gemv.hip gives it), each
// dequantised weight the exact round(code * scale) of bitsandbytes'
// dequantize_4bit.
//
// With this few rows a launch is bound by latency and by the lookups and
// multiplies of the dequantisation, not by the matrix cores or the memory, so
// the kernel is a set of waves that never wait for each other in the K loop:
//
//   * A workgroup owns 32 weight rows; its four waves (and gridDim.z
//     workgroups) each take a run of the 64-code K-steps for all of them, so a
//     wave's sums are one or two 32 x 32 MFMA blocks. The waves' sums are added
//     in wave order at the end, the workgroups' by a reduce launch.
//   * Each wave has a ring of its own in LDS: a step's activations (8 rows of
//     128 bytes a load, as many loads as there are rows) and codes (1 KB)
//     arrive by buffer_load ... lds two steps ahead, waited for by count: no
//     barrier and no registers. Inside a row's LDS copy 16-byte segment s of row t sits at
//     slot s ^ ((t >> 1) & 7), so fragment reads touch every bank once.
//   * A lane's codes of a step are 32 of one row's 64: both codes of a byte
//     from one lookup in a table of code pairs, fp32 products with the block's
//     scale, one pack-convert a pair. The lookups run two slices ahead of the
//     products that use them (scheduling barriers: left alone the compiler
//     issues four, waits, multiplies, and pays the LDS latency four times a step).
//   * Scales are resolved to fp32 in LDS, per wave, before the loop (and every
//     SC steps of a longer run), whatever the block sizes.
//
// Measured (graph replay over rotated weights, bf16, nested), the kernels it
// replaces against it, us: 9728 x 2560 12.7 -> 9.4 at 16 rows, 16.4 -> 10.9 at
// 32, 23.0 -> 18.0 at 64; 6144 x 2560 9.4 -> 6.5, 16.4 -> 7.1, 16.9 -> 9.9;
// with the sums left to a reduce that also writes the next norm, 2560 x 9728
// 15.5 -> 8.7, 24.9 -> 9.9, 24.9 -> 13.0 and 2560 x 4096 7.7 -> 5.3, 12.2 ->
// 5.9, 14.8 -> 7.8. Eight waves a workgroup instead of more workgroups were
// slower (9728 x 2560 at 16 rows 12.9 us: one workgroup a CU, two rounds).
#include "nf4_mfma.h"

namespace ttsp {

namespace {

constexpr int KT = 64;   // codes per K-step
constexpr int CH = 1024; // bytes of one wave-wide load
constexpr int KS = 4;    // waves a workgroup, each a run of the K-steps
constexpr int SP = 33;   // pitch of a step's 32 scales

struct FewMat {
  const uint8_t* W;
  const uint8_t* A8;
  const float* AMAX;
  const float* CODE2;
  float offset;
};

// XL: 8-row activation loads a step; MATS: 2 for the SwiGLU pair
template <int XL, int MATS>
struct FewCfg {
  // the pair at 32 rows: two stages, so that two workgroups fit a CU (9728 rows: 304 workgroups)
  static constexpr int TN = XL > 4 ? 2 : 1;
  static constexpr int ST = MATS == 2 && XL == 4 ? 2 : 3;
  static constexpr int SC = 5 * ST;  // steps whose scales a wave resolves at once (at most 16: lanes)
  static constexpr int STAGE = (XL + MATS) * CH;
  static constexpr int L = XL + MATS;
  static constexpr int PART = TN * 16 * 64 * 4;  // a wave's partial sums of one matrix
};

template <int XL, int MATS, typename RS>
__device__ __forceinline__ void few_load(uint8_t* __restrict__ dst, RS xr, const RS (&wr)[MATS],
                                         const uint32_t (&xoff)[XL], uint32_t woff, int k0) {
#pragma unroll
  for (int j = 0; j < XL; ++j)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr_t)(dst + j * CH), 16, xoff[j], k0 * 2, 0, 0);
#pragma unroll
  for (int t = 0; t < MATS; ++t)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr[t], (lds_ptr_t)(dst + (XL + t) * CH), 16, woff, k0 / 2, 0, 0);
}

template <int DT, int XL, int MATS, typename RS>
__device__ __forceinline__ void few_step(const uint8_t* __restrict__ rd, uint8_t* __restrict__ dst,
                                         const float2* __restrict__ lut, const float* __restrict__ sc, RS xr,
                                         const RS (&wr)[MATS], const uint32_t (&xoff)[XL], uint32_t woff, int k0n,
                                         int lane, f32x16_v (&acc)[MATS][FewCfg<XL, MATS>::TN]) {
  using C = FewCfg<XL, MATS>;
  u32x4 codes[MATS];
  float sv[MATS];
#pragma unroll
  for (int t = 0; t < MATS; ++t) {
    codes[t] = *reinterpret_cast<const u32x4*>(rd + (XL + t) * CH + lane * 16);
    sv[t] = sc[t * C::SC * SP];
  }
  u32x4 bf[4][C::TN];
  auto read_x = [&](int kk) {
#pragma unroll
    for (int b = 0; b < C::TN; ++b) {
      const int t = (32 * b + (lane & 31)) & (8 * XL - 1), sg = 4 * (lane >> 5) + kk;
      bf[kk][b] = *reinterpret_cast<const u32x4*>(rd + t * 128 + ((sg ^ ((t >> 1) & 7)) << 4));
    }
  };
  // slice i is quarter kk = i / MATS of matrix i % MATS; the lookups of slice
  // i + 2 are issued before slice i's are used
  constexpr int NS = 4 * MATS;
  float2 pc[3][4];
  auto look = [&](int i) {
    const uint32_t wv = codes[i % MATS][i / MATS];
#pragma unroll
    for (int j = 0; j < 4; ++j) pc[i % 3][j] = lut[(wv >> (8 * j)) & 0xffu];
  };
  __builtin_amdgcn_sched_barrier(0);
  few_load<XL, MATS>(dst, xr, wr, xoff, woff, k0n);
  look(0);
  read_x(0);
  look(1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int t = i % MATS, kk = i / MATS;
    if (i + 2 < NS) look(i + 2);
    if (t == MATS - 1 && kk < 3) read_x(kk + 1);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 af;
#pragma unroll
    for (int e = 0; e < 4; ++e) af[e] = pack2<DT>(__fmul_rn(pc[i % 3][e].x, sv[t]), __fmul_rn(pc[i % 3][e].y, sv[t]));
#pragma unroll
    for (int b = 0; b < C::TN; ++b) acc[t][b] = mfma32<DT>(af, bf[kk][b], acc[t][b]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int DT, int XL, int MATS, bool NESTED>
__global__ __launch_bounds__(64 * KS, 2) void nf4_gemm_few_kernel(
    const uint16_t* __restrict__ X, FewMat m0, FewMat m1, const float* __restrict__ LUT, uint16_t* __restrict__ Y,
    const uint16_t* __restrict__ R, int epi, int M, int K, int N, int bs_shift, int bs2_shift, float* __restrict__ YP) {
#if defined(__HIP_DEVICE_COMPILE__)
  using C = FewCfg<XL, MATS>;
  __shared__ __align__(16) uint8_t ring0[KS][C::STAGE];
  __shared__ __align__(16) uint8_t ring1[KS][C::STAGE];
  __shared__ __align__(16) uint8_t ring2[KS][C::ST > 2 ? C::STAGE : 16];
  __shared__ __align__(16) uint8_t own[C::STAGE >= C::PART ? 16 : KS * C::PART];
  __shared__ float2 lut2_s[256];
  __shared__ float code2_s[NESTED ? 256 * MATS : 1];
  __shared__ float sc_s[KS][MATS * C::SC * SP];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mb = blockIdx.x * 32;
  // this wave's K-steps: run w of the KS * gridDim.z runs
  const int steps = K / KT, runs = KS * gridDim.z, run = blockIdx.z * KS + wave;
  const int s_lo = (int)((long long)steps * run / runs), s_hi = (int)((long long)steps * (run + 1) / runs);
  const int ns = s_hi - s_lo;

  const float lutv0 = LUT[tid >> 4], lutv1 = LUT[tid & 15];
  float c2v[MATS];
  if constexpr (NESTED) {
    c2v[0] = m0.CODE2[tid];
    if constexpr (MATS == 2) c2v[1] = m1.CODE2[tid];
  }
  // scale entry i of this lane: row 4 i + lane / 16 of the 32, step base + lane % 16
  uint32_t a8v[MATS][8];
  float amv[MATS][8];
  auto load_scales = [&](int base) {
#pragma unroll
    for (int t = 0; t < MATS; ++t) {
      const FewMat& m = t ? m1 : m0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = min(mb + 4 * i + (lane >> 4), M - 1), s = min(base + (lane & 15), steps - 1);
        const uint32_t b = (uint32_t)row * (uint32_t)(K >> bs_shift) + ((uint32_t)(s * KT) >> bs_shift);
        if constexpr (NESTED) {
          a8v[t][i] = m.A8[b];
          amv[t][i] = m.AMAX[b >> bs2_shift];
        } else {
          amv[t][i] = m.AMAX[b];
        }
      }
    }
  };
  auto store_scales = [&]() {
#pragma unroll
    for (int t = 0; t < MATS; ++t)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float s = amv[t][i];
        if constexpr (NESTED)
          s = __fadd_rn(__fmul_rn(code2_s[256 * t + a8v[t][i]], s), t ? m1.offset : m0.offset);
        if ((lane & 15) < C::SC) sc_s[wave][t * C::SC * SP + (lane & 15) * SP + 4 * i + (lane >> 4)] = s;
      }
  };
  load_scales(s_lo);

  typedef __amdgpu_buffer_rsrc_t RS;
  const RS xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, (int)((size_t)N * K * 2),
                                                  0x00020000);
  RS wr[MATS];
  wr[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m0.W), (short)0, (int)((size_t)M * K / 2), 0x00020000);
  if constexpr (MATS == 2)
    wr[1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m1.W), (short)0, (int)((size_t)M * K / 2),
                                              0x00020000);
  uint32_t xoff[XL];
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const int t = 8 * j + (lane >> 3), sg = (lane & 7) ^ ((t >> 1) & 7);
    xoff[j] = (uint32_t)min(t, N - 1) * (uint32_t)K * 2u + (uint32_t)sg * 16u;
  }
  const uint32_t woff = (uint32_t)min(mb + (lane & 31), M - 1) * (uint32_t)(K / 2) + 16u * (lane >> 5);
  auto koff = [&](int s) { return min(s_lo + s, steps - 1) * KT; };
  few_load<XL, MATS>(ring0[wave], xr, wr, xoff, woff, koff(0));
  if constexpr (C::ST > 2) few_load<XL, MATS>(ring1[wave], xr, wr, xoff, woff, koff(1));

  lut2_s[tid] = make_float2(lutv0, lutv1);
  if constexpr (NESTED) {
    code2_s[tid] = c2v[0];
    if constexpr (MATS == 2) code2_s[256 + tid] = c2v[1];
  }
  TTSP_WAIT_LGKM0();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  store_scales();

  f32x16_v acc[MATS][C::TN];
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][b][r] = 0.0f;

  // step s reads stage s % 3; its loads were issued two steps before. The
  // stage step s + 2 refills was read in step s - 1.
  for (int base = 0; base < ns; base += C::SC) {
    if (base) {  // the next steps' scales
      load_scales(s_lo + base);
      store_scales();
    }
    auto one = [&](int s, const uint8_t* rd, uint8_t* dst) {
      TTSP_WAIT_VM_LGKM0((C::ST - 2) * C::L);
      asm volatile("" ::: "memory");
      few_step<DT, XL, MATS>(rd, dst, lut2_s, &sc_s[wave][(s - base) * SP + (lane & 31)], xr, wr, xoff, woff,
                             koff(s + C::ST - 1), lane, acc);
    };
    const int end = min(ns, base + C::SC);
    int s = base;
    if constexpr (C::ST == 3) {
      for (; s + 3 <= end; s += 3) {
        one(s, ring0[wave], ring2[wave]);
        one(s + 1, ring1[wave], ring0[wave]);
        one(s + 2, ring2[wave], ring1[wave]);
      }
      if (s < end) one(s, ring0[wave], ring2[wave]);
      if (s + 1 < end) one(s + 1, ring1[wave], ring0[wave]);
    } else {
      for (; s + 2 <= end; s += 2) {
        one(s, ring0[wave], ring1[wave]);
        one(s + 1, ring1[wave], ring0[wave]);
      }
      if (s < end) one(s, ring0[wave], ring1[wave]);
    }
  }
  TTSP_WAIT_VM_LGKM0(0);

  // the waves' sums, added in wave order
  float* const part0 = reinterpret_cast<float*>(C::STAGE >= C::PART ? &ring0[0][0] : own);
  constexpr int PW = (C::STAGE >= C::PART ? C::STAGE : C::PART) / 4;
  asm volatile("" ::: "memory");
  // thread (g, lane) of a 32-column block: 4 consecutive weight rows of one activation row
  const int g = wave, n_l = lane & 31, m = mb + 8 * g + 4 * (lane >> 5);
  float v[C::TN][MATS][4];
#pragma unroll
  for (int t = 0; t < MATS; ++t) {
    if (t) __syncthreads();
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) part0[wave * PW + (b * 16 + r) * 64 + lane] = acc[t][b][r];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float* p = part0 + (b * 16 + 4 * g + c) * 64 + lane;
        v[b][t][c] = p[0];
#pragma unroll
        for (int k = 1; k < KS; ++k) v[b][t][c] = __fadd_rn(v[b][t][c], p[k * PW]);
      }
  }
  const bool v4 = (M & 3) == 0 && (epi & 8);
  const int ep = epi & 3;
#pragma unroll
  for (int b = 0; b < C::TN; ++b) {
    const int n = 32 * b + n_l;
    if (n >= N || m >= M) continue;
    const size_t o = (size_t)n * M + m;
    if (YP) {
      float* yp = YP + (size_t)blockIdx.z * N * M + o;
      if ((M & 3) == 0) {
        *reinterpret_cast<float4*>(yp) = make_float4(v[b][0][0], v[b][0][1], v[b][0][2], v[b][0][3]);
      } else {
        for (int c = 0; c < 4; ++c)
          if (m + c < M) yp[c] = v[b][0][c];
      }
      continue;
    }
    uint16_t ov[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (MATS == 2)
        ov[c] = mm_epi<DT>(Elem<DT>::load(Elem<DT>::store(v[b][1][c])), Elem<DT>::store(v[b][0][c]), 2);
      else
        ov[c] = mm_epi<DT>(Elem<DT>::load(Elem<DT>::store(v[b][0][c])), ep && m + c < M ? R[o + c] : (uint16_t)0, ep);
    }
    if (v4) {
      *reinterpret_cast<uint2*>(Y + o) =
          make_uint2((uint32_t)ov[0] | ((uint32_t)ov[1] << 16), (uint32_t)ov[2] | ((uint32_t)ov[3] << 16));
    } else {
      for (int c = 0; c < 4; ++c)
        if (m + c < M) Y[o + c] = ov[c];
    }
  }
#endif
}

template <int DT, int XL, int MATS>
void launch_few(const void* X, const FewMat& a, const FewMat& b, const float* LUT, void* Y, const void* R, int epi,
                int M, int K, int N, int bs_shift, int bs2_shift, int splits, float* YP, hipStream_t st) {
  const dim3 grid((M + 31) / 32, 1, splits);
  if (a.A8)
    hipLaunchKernelGGL((nf4_gemm_few_kernel<DT, XL, MATS, true>), grid, dim3(64 * KS), 0, st, (const uint16_t*)X, a, b,
                       LUT, (uint16_t*)Y, (const uint16_t*)R, epi, M, K, N, bs_shift, bs2_shift, YP);
  else
    hipLaunchKernelGGL((nf4_gemm_few_kernel<DT, XL, MATS, false>), grid, dim3(64 * KS), 0, st, (const uint16_t*)X, a,
                       b, LUT, (uint16_t*)Y, (const uint16_t*)R, epi, M, K, N, bs_shift, bs2_shift, YP);
}

template <int DT, int MATS>
int few_rows(const void* X, const FewMat& a, const FewMat& b, const float* LUT, void* Y, const void* R, int epi, int M,
             int K, int N, int bs_shift, int bs2_shift, int splits, float* YP, hipStream_t st) {
  if (N <= 16) {
    launch_few<DT, 2, MATS>(X, a, b, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
  } else if (N <= 32) {
    launch_few<DT, 4, MATS>(X, a, b, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
  } else {
    if constexpr (MATS == 1)
      launch_few<DT, 8, MATS>(X, a, b, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
    else
      return (int)hipErrorInvalidValue;
  }
  TTSP_RETURN_LAUNCH();
}

}  // namespace

constexpr int FEW_MIN_N = 9, FEW_MAX_N = 64, FEW_PAIR_MAX_N = 32;
// The longest row of an unsplit product of 17 to 32 rows; longer ones take the
// plan's K splits.
constexpr int FEW_UNSPLIT_MAX_K = 10240;

// Whether the kernel takes the shape: byte offsets of X and W and the scale
// indices below 2^31.
bool few_takes(int M, int K, int N) {
  if (M <= 0 || K <= 0 || K % 128 || N < FEW_MIN_N || N > FEW_MAX_N) return false;
  return (long long)N * K * 2 < (1ll << 31) && (long long)M * K / 2 < (1ll << 31);
}

// Whether an unsplit product of N rows runs here: from 17 rows always, but at
// 17 to 32 of a longer K than FEW_UNSPLIT_MAX_K, whose four waves a workgroup
// would each add a long run (256 x 40960 at 32 rows 57.9 us, 20.3 in 4 splits;
// 1024 x 16384 25.7 and 12.9; at 2560 x 4096 the two are within 0.6 us); at 9 to
// 16 the skinny kernel's 16-row tiles make more workgroups of a small matrix.
// Measured at 16 rows, skinny against this kernel, us: 1024 x 2560 6.5 / 6.7,
// 2560 x 4096 8.4 / 8.7, 4096 x 2560 6.9 / 6.9; past 4096 rows the skinny one
// takes a second round: 5120 x 2560 9.7 / 6.9, 6144 x 2560 9.9 / 7.0, 9728 x
// 2560 12.3 / 9.8, 6144 x 9728 29.0 / 15.5. (The line here, 6144 rows and K up
// to 4096, is on the safe side of that.)
bool few_unsplit(int M, int K, int N) {
  if (!few_takes(M, K, N)) return false;
  return N > 16 ? N > 32 || K <= FEW_UNSPLIT_MAX_K : (M + 31) / 32 >= 192 && K <= 4096;
}

// K splits where the sums' reduce costs nothing extra (it also writes the next
// norm, or another kernel adds the sums): the most, up to 4, whose workgroups
// fit one to a CU and leave every wave two K-steps.
int few_splits(int M, int K, int N) {
  if (!few_takes(M, K, N)) return 0;
  const int tiles = (M + 31) / 32, steps = K / KT;
  int sp = 1;
  while (sp < 4 && tiles * sp * 2 <= 256 && steps / (KS * sp * 2) >= 2) sp *= 2;
  return sp;
}

bool few_pair(int M, int K, int N) { return N <= FEW_PAIR_MAX_N && few_unsplit(M, K, N); }

// splits > 1: the sums of each split to YP [splits][N][M]; else Y with the
// epilogue. Alignment of Y for the 8-byte stores is checked here.
int gemm_few(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
             float offset, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int bs_shift,
             int bs2_shift, int splits, float* YP, hipStream_t st) {
  if (!few_takes(M, K, N) || splits < 1 || (splits > 1 && !YP) || (uintptr_t)X % 16 || (uintptr_t)W % 16)
    return (int)hipErrorInvalidValue;
  const FewMat a{W, A8, AMAX, CODE2, offset};
  const int e = (epi & 3) | ((uintptr_t)Y % 8 == 0 ? 8 : 0);
  float* yp = splits > 1 ? YP : nullptr;
  if (dt == DT_BF16) return few_rows<DT_BF16, 1>(X, a, a, LUT, Y, R, e, M, K, N, bs_shift, bs2_shift, splits, yp, st);
  if (dt == DT_F16) return few_rows<DT_F16, 1>(X, a, a, LUT, Y, R, e, M, K, N, bs_shift, bs2_shift, splits, yp, st);
  return (int)hipErrorInvalidValue;
}

// Y = round(round(silu(X . W1^T)) * round(X . W3^T)), with the bits of gemm_few
// unsplit on each: every wave takes its K run of both weights.
int gemm_few_pair(const void* X, int dt, const uint8_t* W1, const uint8_t* A8_1, const float* AMAX_1,
                  const float* CODE2_1, float offset_1, const uint8_t* W3, const uint8_t* A8_3, const float* AMAX_3,
                  const float* CODE2_3, float offset_3, const float* LUT, void* Y, int M, int K, int N, int bs_shift,
                  int bs2_shift, hipStream_t st) {
  if (!few_pair(M, K, N) || (uintptr_t)X % 16 || (uintptr_t)W1 % 16 || (uintptr_t)W3 % 16)
    return (int)hipErrorInvalidValue;
  const FewMat a{W1, A8_1, AMAX_1, CODE2_1, offset_1}, b{W3, A8_3, AMAX_3, CODE2_3, offset_3};
  const int e = (uintptr_t)Y % 8 == 0 ? 8 : 0;
  if (dt == DT_BF16)
    return few_rows<DT_BF16, 2>(X, a, b, LUT, Y, nullptr, e, M, K, N, bs_shift, bs2_shift, 1, nullptr, st);
  if (dt == DT_F16)
    return few_rows<DT_F16, 2>(X, a, b, LUT, Y, nullptr, e, M, K, N, bs_shift, bs2_shift, 1, nullptr, st);
  return (int)hipErrorInvalidValue;
}

}  // namespace ttsp
