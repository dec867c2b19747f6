// NF4 matrix product for long prompts (more than 512 activation rows):
// Y[N][M] = X[N][K] . W^T in two launches. The weight's codes become
// round(code * scale) in the activation type once (the values bitsandbytes'
// dequantize_4bit gives) in a workspace of the call, and a bf16 / fp16 matrix
// kernel multiplies them.
//
// Why two launches: fused tiles dequantise each weight once per activation
// tile (16 times at 2048 rows) through LDS table lookups, in the same waves
// that feed the matrix cores: 9728 x 2560 at 2048 rows ran 216 us (472
// TFLOP/s). Writing the 50 MB of dense weights costs ~13 us, and a kernel
// with nothing but loads and MFMAs in its K loop runs at twice the rate.
//
// The matrix kernel. Operands reach an LDS ring by buffer_load ... lds (no
// register staging), a whole number of steps ahead. A wave's fragments of
// slice kk + 1 are read while slice kk multiplies, across the step's barrier
// too: the last slice of a step is multiplied after it. Scheduling barriers
// hold that order (left alone the compiler sinks the fragment reads to their
// use and the ring's loads to the end of the step: 256 x 128 tiles, 9728 x
// 2560 at 2048 rows, 137 -> 107 us with the epilogue below).
// The epilogue is small on purpose. Outputs pass through the (free) ring, a
// padded row at a time per wave, and leave as 16-byte pieces of whole rows in
// a rolled loop. Stored from the accumulators with every residual form
// unrolled it was 45 KB of straight-line code, fetched cold by every launch:
// 256 x 256 tiles took 40 us a launch longer.
// Tiles: 256 x 128 with three stages (one workgroup a CU), or 192 x 256 with
// two where that takes fewer rounds of workgroups (6144 x 2560 at 2048 rows:
// 57 against 70 us). 128 x 128 and 160 x 128 with two workgroups a CU were
// within 5 % at 2048 rows and up to 20 % behind at 700; 256 x 256 leaves too
// few tiles. Sums run along K in the same order in every tile shape, so the
// shape does not change a bit of the result; see dense_plan for the order.
#include "nf4_mfma.h"

namespace ttsp {

namespace {

// A workgroup's tile: BM weight rows x BN activation rows, WM x WN waves, a
// ring of ST stages of KT elements of K.
template <int BM_, int BN_, int WM_, int WN_, int ST_>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KT = 64, ST = ST_;
  static constexpr int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;
  static constexpr int ROWB = KT * 2;                      // bytes of a tile row
  static constexpr int RPL = 1024 / ROWB;                  // rows a wave-wide load moves
  static constexpr int LA = BM / RPL / NW, LB = BN / RPL / NW;  // loads a wave and step
  static constexpr int STAGE = (BM + BN) * ROWB;
  static constexpr int SL = KT / 16;                       // K-slices of a step
  // a step's loads are issued in LP parts: one to a slice where the ring holds
  // a step more than is being read, all at once where they must land in one step
  static constexpr int LP = ST > 2 ? SL : 1;
  static_assert(BM % (RPL * NW) == 0 && BN % (RPL * NW) == 0, "loads split evenly over the waves");
  // segment s of tile row t sits at 16-byte slot s ^ swz(t) of the row: the 16
  // rows of a fragment read's lanes then cover all 64 banks once
  __device__ static __forceinline__ int swz(int t) { return (t >> 1) & 7; }
};

template <int DT, typename C, typename RS>
struct Ctx {
  RS wr, xr;
  uint32_t aoff[C::LA], boff[C::LB];
  uint32_t afrag[C::SL], bfrag[C::SL];  // LDS byte offsets of this lane's fragments of slice kk
  int wave;
};

// the loads of a stage, or (P parts) part p of them
template <typename C, int P, typename X>
__device__ __forceinline__ void load_stage(const X& c, uint8_t* __restrict__ dst, int koff, int p = 0) {
#pragma unroll
  for (int j = 0; j < C::LA + C::LB; ++j) {
    if (j % P != p) continue;
    if (j < C::LA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(c.wr, (lds_ptr_t)(dst + (c.wave * C::LA + j) * 1024), 16, c.aoff[j], koff,
                                               0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          c.xr, (lds_ptr_t)(dst + C::BM * C::ROWB + (c.wave * C::LB + j - C::LA) * 1024), 16, c.boff[j - C::LA], koff, 0,
          0);
  }
}

template <typename C>
__device__ __forceinline__ void read_slice(const uint8_t* rd, uint32_t ao, uint32_t bo, u32x4 (&af)[C::TM],
                                           u32x4 (&bf)[C::TN]) {
#pragma unroll
  for (int b = 0; b < C::TN; ++b) bf[b] = *reinterpret_cast<const u32x4*>(rd + bo + b * 32 * C::ROWB);
#pragma unroll
  for (int a = 0; a < C::TM; ++a) af[a] = *reinterpret_cast<const u32x4*>(rd + ao + a * 32 * C::ROWB);
}

template <int DT, typename C>
__device__ __forceinline__ void mul_slice(const u32x4 (&af)[C::TM], const u32x4 (&bf)[C::TN],
                                          f32x16_v (&acc)[C::TM][C::TN]) {
#pragma unroll
  for (int a = 0; a < C::TM; ++a)
#pragma unroll
    for (int b = 0; b < C::TN; ++b) acc[a][b] = mfma32<DT>(af[a], bf[b], acc[a][b]);
}

// The end of a run of K-steps: its sums join those of the runs before (fold 1:
// the first run), as a K split's reduce adds its splits.
template <typename C>
__device__ __forceinline__ void end_run(f32x16_v (&acc)[C::TM][C::TN], f32x16_v (&sum)[C::TM][C::TN], int fold) {
#pragma unroll
  for (int a = 0; a < C::TM; ++a)
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sum[a][b][r] = fold == 1 ? acc[a][b][r] : __fadd_rn(sum[a][b][r], acc[a][b][r]);
        acc[a][b][r] = 0.0f;
      }
}

// One step: stage rd has landed for every wave; the stage dst, which every
// wave has finished reading, takes the operands at K byte offset koff. The
// last slice's fragments are read here and multiplied in the next call.
template <int DT, typename C, bool FIRST, bool RUNS, typename X>
__device__ __forceinline__ void step(const X& c, const uint8_t* __restrict__ rd, uint8_t* __restrict__ dst, int koff,
                                     u32x4 (&af)[2][C::TM], u32x4 (&bf)[2][C::TN], f32x16_v (&acc)[C::TM][C::TN],
                                     f32x16_v (&sum)[RUNS ? C::TM : 1][RUNS ? C::TN : 1], int fold) {
  // (SL is even: slice kk's fragments are in set kk & 1, the pending ones in set 1)
  read_slice<C>(rd, c.afrag[0], c.bfrag[0], af[0], bf[0]);
  if constexpr (!FIRST) load_stage<C, C::LP>(c, dst, koff, 0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!FIRST) mul_slice<DT, C>(af[1], bf[1], acc);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (RUNS && !FIRST)
    if (fold) end_run<C>(acc, sum, fold);
#pragma unroll
  for (int kk = 0; kk + 1 < C::SL; ++kk) {
    read_slice<C>(rd, c.afrag[kk + 1], c.bfrag[kk + 1], af[(kk + 1) & 1], bf[(kk + 1) & 1]);
    if constexpr (!FIRST && C::LP > 1) load_stage<C, C::LP>(c, dst, koff, kk + 1);
    __builtin_amdgcn_sched_barrier(0);
    mul_slice<DT, C>(af[kk & 1], bf[kk & 1], acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int DT, typename C, bool SW, bool RUNS>
__global__ __launch_bounds__(64 * C::NW) void nf4_gemm_dense_kernel(
    const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, uint16_t* __restrict__ Y,
    const uint16_t* __restrict__ R, int epi, int M, int K, int N, int runs, float* __restrict__ YP) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __align__(16) uint8_t ring0[C::STAGE];
  __shared__ __align__(16) uint8_t ring1[C::STAGE];
  __shared__ __align__(16) uint8_t ring2[C::ST > 2 ? C::STAGE : 16];
  static_assert(C::ST == 2 || C::ST == 3, "ring of two or three stages");
  constexpr int BMO = SW ? C::BM / 2 : C::BM;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  // XCD x takes a contiguous run of tiles (workgroup b runs on XCD b % 8), the
  // activation tiles innermost
  const int tn = (N + C::BN - 1) / C::BN;
  const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int tile = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
  const int n0 = (tile % tn) * C::BN, m0 = (tile / tn) * BMO;
  const int nsteps = K / C::KT / gridDim.z, kbase = blockIdx.z * nsteps * C::KT * 2;  // bytes

  typedef __amdgpu_buffer_rsrc_t RS;
  Ctx<DT, C, RS> c;
  c.wave = wave;
  c.xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, (int)((size_t)N * K * 2), 0x00020000);
  c.wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W), (short)0,
                                           (int)((size_t)M * K * (SW ? 4 : 2)), 0x00020000);
  {
    const int lr = lane / (C::ROWB / 16), ls = lane % (C::ROWB / 16);
#pragma unroll
    for (int j = 0; j < C::LA; ++j) {
      const int t = (wave * C::LA + j) * C::RPL + lr;
      int row = m0 + t;
      if constexpr (SW) row = m0 + 32 * (t >> 6) + (t & 31);
      row = min(row, M - 1) + (SW && (t & 32) ? M : 0);
      c.aoff[j] = (uint32_t)row * (uint32_t)K * 2u + (uint32_t)((ls ^ C::swz(t)) * 16 + kbase);
    }
#pragma unroll
    for (int j = 0; j < C::LB; ++j) {
      const int t = (wave * C::LB + j) * C::RPL + lr;
      c.boff[j] = (uint32_t)min(n0 + t, N - 1) * (uint32_t)K * 2u + (uint32_t)((ls ^ C::swz(t)) * 16 + kbase);
    }
#pragma unroll
    for (int kk = 0; kk < C::SL; ++kk) {
      const int r = lane & 31, sg = 4 * (lane >> 5) + kk;  // (the tile kernel's order of a step's products)
      const uint32_t o = r * C::ROWB + ((sg ^ C::swz(r)) << 4);
      c.afrag[kk] = o + wm * C::TM * 32 * C::ROWB;
      c.bfrag[kk] = o + wn * C::TN * 32 * C::ROWB + C::BM * C::ROWB;
    }
  }
  f32x16_v acc[C::TM][C::TN];
#pragma unroll
  for (int a = 0; a < C::TM; ++a)
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;
  f32x16_v sum[RUNS ? C::TM : 1][RUNS ? C::TN : 1];
  u32x4 af[2][C::TM], bf[2][C::TN];
  constexpr int L = C::LA + C::LB, SB = C::KT * 2;
  const int last = (nsteps - 1) * SB;

  load_stage<C, 1>(c, ring0, 0);
  load_stage<C, 1>(c, ring1, min(SB, last));
  if constexpr (C::ST > 2) load_stage<C, 1>(c, ring2, min(2 * SB, last));
  // between steps: this wave's reads of the stage are done and its loads of
  // the next have landed; past the barrier, every wave's
  auto meet = [&]() {
    TTSP_WAIT_VM_LGKM0((C::ST - 2) * L);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  TTSP_WAIT_VM_LGKM0((C::ST - 1) * L);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  step<DT, C, true, RUNS>(c, ring0, ring0, 0, af, bf, acc, sum, 0);
  // RUNS: the steps left of this run, and the fold its end takes
  int left = RUNS ? nsteps / runs : 0, fold = 1;
  // step s reads stage s % ST and refills stage (s - 1) % ST with step s - 1 + ST
  auto one = [&](int s, const uint8_t* rd, uint8_t* dst) {
    meet();
    int f = 0;
    if constexpr (RUNS)
      if (--left == 0) f = fold, fold = 2, left = nsteps / runs;
    step<DT, C, false, RUNS>(c, rd, dst, min((s - 1 + C::ST) * SB, last), af, bf, acc, sum, f);
  };
  int s = 1;
  if constexpr (C::ST == 2) {
    for (; s + 2 <= nsteps; s += 2) {
      one(s, ring1, ring0);
      one(s + 1, ring0, ring1);
    }
    if (s < nsteps) one(s, ring1, ring0);
  } else {
    for (; s + 3 <= nsteps; s += 3) {
      one(s, ring1, ring0);
      one(s + 1, ring2, ring1);
      one(s + 2, ring0, ring2);
    }
    if (s < nsteps) one(s, ring1, ring0);
    if (s + 1 < nsteps) one(s + 1, ring2, ring1);
  }
  mul_slice<DT, C>(af[1], bf[1], acc);
  if constexpr (RUNS) {
#pragma unroll
    for (int a = 0; a < C::TM; ++a)
#pragma unroll
      for (int b = 0; b < C::TN; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = __fadd_rn(sum[a][b][r], acc[a][b][r]);
  }

  // accumulator r of lane l is (weight row 8 (r / 4) + 4 (l / 32) + r % 4, activation row l % 32)
  TTSP_WAIT_VM_LGKM0(0);
  __syncthreads();
  constexpr int PITCH = C::TM * 64 + 16, WB = 32 * PITCH, PERST = C::STAGE / WB;
  static_assert(C::NW <= 2 * PERST, "output staging exceeds the ring");
  uint8_t* const stg = wave < PERST ? ring0 + wave * WB : ring1 + (wave - PERST) * WB;
  if (YP) {  // (M % 4 == 0: the plan)
    // each 32 x 32 block through the wave's own LDS, so that a store writes
    // whole 128-byte pieces of 8 rows, not 32 bytes of 32 (with the reduce, us:
    // 2560 x 9728 in 4 splits at 1500 rows 104.2 -> 100.4, 1024 x 3072 at 1200
    // 26.7 -> 24.2, 2560 x 4096 at 1024 44.9 -> 42.6)
    constexpr int PP = 36;  // floats a staged row
    static_assert(32 * PP * 4 <= WB, "a block exceeds the wave's staging");
    float* const ws = reinterpret_cast<float*>(stg);
    float* yp = YP + (size_t)blockIdx.z * N * M;
#pragma unroll
    for (int b = 0; b < C::TN; ++b)
#pragma unroll
      for (int a = 0; a < C::TM; ++a) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<float4*>(ws + (lane & 31) * PP + 8 * g + 4 * (lane >> 5)) =
              make_float4(acc[a][b][4 * g], acc[a][b][4 * g + 1], acc[a][b][4 * g + 2], acc[a][b][4 * g + 3]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int nl = 8 * j + (lane >> 3), n = n0 + (wn * C::TN + b) * 32 + nl;
          const int m = m0 + (wm * C::TM + a) * 32 + 4 * (lane & 7);
          const float4 v = *reinterpret_cast<const float4*>(ws + nl * PP + 4 * (lane & 7));
          if (n < N && m < M) *reinterpret_cast<float4*>(yp + (size_t)n * M + m) = v;
        }
      }
    return;
  }
  const int ep = SW ? 2 : epi & 3;
  const bool vec = (M & 7) == 0 && (epi & 8);
  constexpr int CPR = C::TM * (SW ? 2 : 4);  // 16-byte output chunks of a row
#pragma unroll
  for (int b = 0; b < C::TN; ++b) {
    // the block's rows are written and read by different lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int a = 0; a < C::TM; ++a)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2*>(stg + (lane & 31) * PITCH + a * 64 + g * 16 + (lane >> 5) * 8) =
            make_uint2(pack2<DT>(acc[a][b][4 * g], acc[a][b][4 * g + 1]),
                       pack2<DT>(acc[a][b][4 * g + 2], acc[a][b][4 * g + 3]));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
    for (int e = lane; e < 32 * CPR; e += 64) {
      const int nl = e / CPR, ch = e % CPR;
      const int n = n0 + (wn * C::TN + b) * 32 + nl;
      const int m = m0 + wm * (SW ? C::TM / 2 : C::TM) * 32 + ch * 8;
      if (n >= N || m >= M) continue;
      const size_t o = (size_t)n * M + m;
      const bool full = vec && m + 8 <= M;
      u32x4 y, r = {0, 0, 0, 0};
      if constexpr (SW) {
        const uint8_t* src = stg + nl * PITCH + (ch >> 2) * 128 + (ch & 3) * 16;
        r = *reinterpret_cast<const u32x4*>(src);
        y = *reinterpret_cast<const u32x4*>(src + 64);
      } else {
        y = *reinterpret_cast<const u32x4*>(stg + nl * PITCH + ch * 16);
      }
      mm_store8<DT>(Y, R, o, m, M, full, ep, y, SW, r);
    }
  }
#endif
}

// Weights of one or two matrices (grid.y) to dense 16-bit rows: 8 codes (a
// dword) a lane and chunk, so a wave reads 256 and writes 1024 contiguous
// bytes an instruction, DQ_CH chunks of loads in flight before the first use.
// Bound by the 16-bit stores.
struct DqMat {
  const uint32_t* W;
  const uint8_t* A8;
  const float* AMAX;
  const float* CODE2;
  float offset;
};

constexpr int DQ_CH = 8;

template <int DT, bool NESTED>
__global__ __launch_bounds__(256) void nf4_dequant16_kernel(DqMat m0, DqMat m1, const float* __restrict__ LUT,
                                                            uint16_t* __restrict__ OUT, long long nd, int bs_shift,
                                                            int bs2_shift) {
  __shared__ float2 lut2_s[256];
  __shared__ float code2_s[NESTED ? 256 : 1];
  const bool second = blockIdx.y != 0;
  const uint32_t* __restrict__ W = second ? m1.W : m0.W;
  const uint8_t* __restrict__ A8 = second ? m1.A8 : m0.A8;
  const float* __restrict__ AMAX = second ? m1.AMAX : m0.AMAX;
  const float* CODE2 = second ? m1.CODE2 : m0.CODE2;
  const float offset = second ? m1.offset : m0.offset;
  u32x4* out = reinterpret_cast<u32x4*>(OUT) + (second ? nd : 0);
  const int tid = threadIdx.x;
  const long long d0 = ((long long)blockIdx.x * 4 + (tid >> 6)) * (64 * DQ_CH) + (tid & 63);
  uint32_t w[DQ_CH], a8[DQ_CH];
  float am[DQ_CH];
#pragma unroll
  for (int i = 0; i < DQ_CH; ++i) {
    const long long d = min(d0 + 64 * i, nd - 1);
    w[i] = __builtin_nontemporal_load(W + d);
    const long long b = (8 * d) >> bs_shift;
    if constexpr (NESTED) {
      a8[i] = A8[b];
      am[i] = AMAX[b >> bs2_shift];
    } else {
      am[i] = AMAX[b];
    }
  }
  lut2_s[tid] = make_float2(LUT[tid >> 4], LUT[tid & 15]);
  if constexpr (NESTED) code2_s[tid] = CODE2[tid];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < DQ_CH; ++i) {
    const long long d = d0 + 64 * i;
    if (d >= nd) break;
    float s = am[i];
    if constexpr (NESTED) s = __fadd_rn(__fmul_rn(code2_s[a8[i]], s), offset);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float2 pc = lut2_s[(w[i] >> (8 * j)) & 0xffu];
      o[j] = pack2<DT>(__fmul_rn(pc.x, s), __fmul_rn(pc.y, s));
    }
    out[d] = o;
  }
}

template <int DT>
int launch_dequant16(const DqMat& a, const DqMat& b, int mats, const float* LUT, uint16_t* out, long long nd,
                     int bs_shift, int bs2_shift, hipStream_t st) {
  const dim3 grid((unsigned)((nd + 256 * DQ_CH - 1) / (256 * DQ_CH)), mats);
  if (a.A8)
    hipLaunchKernelGGL((nf4_dequant16_kernel<DT, true>), grid, dim3(256), 0, st, a, b, LUT, out, nd, bs_shift,
                       bs2_shift);
  else
    hipLaunchKernelGGL((nf4_dequant16_kernel<DT, false>), grid, dim3(256), 0, st, a, b, LUT, out, nd, bs_shift,
                       bs2_shift);
  TTSP_RETURN_LAUNCH();
}

typedef Cfg<256, 128, 4, 2, 3> Tall;
typedef Cfg<192, 256, 2, 4, 2> Wide;

template <int DT, typename C, bool SW, bool RUNS>
int launch_dense(const void* X, const uint16_t* W, void* Y, const void* R, int epi, int M, int K, int N, int splits,
                 int runs, float* YP, hipStream_t st) {
  constexpr int BMO = SW ? C::BM / 2 : C::BM;
  const dim3 grid(((M + BMO - 1) / BMO) * ((N + C::BN - 1) / C::BN), 1, splits);
  hipLaunchKernelGGL((nf4_gemm_dense_kernel<DT, C, SW, RUNS>), grid, dim3(64 * C::NW), 0, st, (const uint16_t*)X, W,
                     (uint16_t*)Y, (const uint16_t*)R, epi, M, K, N, runs, YP);
  TTSP_RETURN_LAUNCH();
}

}  // namespace
}  // namespace ttsp

extern "C" int ttsp_nf4_gemm_splits(int M, int K, int N);

namespace ttsp {
namespace {

struct DensePlan {
  bool wide;
  int splits;  // 0: not served
  int runs;    // of each split's K-steps
};

long long tiles(int M, int N, int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

// The sums' order: the K splits ttsp_nf4_gemm_splits gives at 512 rows, each
// summed along K and then added in order, whether as splits here or as runs
// inside a workgroup. Where the 512-row product adds that way too
// (ttsp_nf4_gemm_span_splits), a prompt's spans give the same bits run together
// as one by one. Estimated us: rounds of 256 workgroups, each its K-steps (measured 0.72
// us a 256 x 128 step, 1.05 a 192 x 256 step) and ~5 us of first loads and
// epilogue; splits add the partial sums' traffic and a launch. The least wins.
DensePlan dense_plan(int M, int K, int N, double* us_out = nullptr) {
  const int steps = K / 64, parts = ttsp_nf4_gemm_splits(M, K, 512);
  DensePlan best{false, 0, 1};
  double least = 0.0;
  for (int wide = 0; wide < 2; ++wide)
    for (int sp = 1; sp <= parts; sp += parts - 1) {
      if (sp > 1 && M % 4) break;
      const long long t = (wide ? tiles(M, N, Wide::BM, Wide::BN) : tiles(M, N, Tall::BM, Tall::BN)) * sp;
      double us = (double)((t + 255) / 256) * (steps / sp * (wide ? 1.05 : 0.72) + 5.0);
      if (sp > 1) us += 4.0 + (double)sp * N * M * 8.0 / 4e6;
      if (!best.splits || us < least) best = DensePlan{wide != 0, sp, parts / sp}, least = us;
      if (parts == 1) break;
    }
  if (us_out) *us_out = least;
  return best;
}

template <int DT>
int dense_form(const DensePlan& p, const void* X, const uint16_t* W, void* Y, const void* R, int epi, int M, int K,
               int N, float* YP, hipStream_t st) {
  if (p.runs > 1)
    return p.wide ? launch_dense<DT, Wide, false, true>(X, W, Y, R, epi, M, K, N, p.splits, p.runs, YP, st)
                  : launch_dense<DT, Tall, false, true>(X, W, Y, R, epi, M, K, N, p.splits, p.runs, YP, st);
  return p.wide ? launch_dense<DT, Wide, false, false>(X, W, Y, R, epi, M, K, N, p.splits, 1, YP, st)
                : launch_dense<DT, Tall, false, false>(X, W, Y, R, epi, M, K, N, p.splits, 1, YP, st);
}

}  // namespace

double tile_estimate(int M, int K, int N);
bool tile_halves(int M, int N, int splits);
int gemm_reduce(int dt, const float* YP, int splits, void* Y, const void* R, int epi, int M, int N, hipStream_t st);

constexpr int DENSE_MIN_N = 513;

static int pow2_shift(int v) {
  int sh = 0;
  while (sh < 30 && (1 << sh) < v) ++sh;
  return v > 0 && (1 << sh) == v ? sh : -1;
}

static bool dense_fits(int M, int K, int N, int mats) {
  if (M <= 0 || K <= 0 || N < DENSE_MIN_N || K % 128) return false;
  return (long long)N * K * 2 < (1ll << 31) && (long long)M * K * 2 * mats < (1ll << 31);
}

}  // namespace ttsp

using namespace ttsp;

// Whether the dense form is faster than the tile kernel by their estimates,
// counting here the dequantisation's bytes at ~5.2 TB/s and its launch (us,
// dense against tiles: 9728 x 2560 at 700 rows 50 / 43, at 1024 64 / 79, at
// 2048 113 / 128; 2048 x 2560 at 1024 29.5 / 22.2, at 2048 35.7 / 35.9; 1024 x
// 3072 at 2048 37.8 / 26.2). Over 48 weights of 1024 x 2048 to 9728 x 9728 at
// 1024 to 2048 rows the estimates' choice was within 1 % of the faster form in
// all but a few, and 8 % off at the worst.
static bool dense_pays(int M, int K, int N) {
  double us = 0.0;
  dense_plan(M, K, N, &us);
  return us + 3.0 + (double)M * K * 2.5 / 5.2e6 < tile_estimate(M, K, N);
}

// The K splits `ttsp_nf4_gemm_dense` takes a product in, 0 where it does not
// serve it: small products, and below 1024 rows where it does not pay. From
// 1024 rows a prompt's merged spans take it for its order of sums
// (ttsp_nf4_gemm_span_splits), other callers where ttsp_nf4_gemm_dense_pays.
extern "C" int ttsp_nf4_gemm_dense_splits(int M, int K, int N) {
  if (!dense_fits(M, K, N, 1) || (long long)M * K < (1ll << 21) || (double)M * K * N < 2.5e9) return 0;
  return N >= 1024 || dense_pays(M, K, N) ? dense_plan(M, K, N).splits : 0;
}

extern "C" int ttsp_nf4_gemm_dense_pays(int M, int K, int N) {
  return ttsp_nf4_gemm_dense_splits(M, K, N) && dense_pays(M, K, N) ? 1 : 0;
}

// The K splits of a 512-row product whose bits the dense form keeps at every
// run of 512-row spans (1024, 1536 and 2048 rows); 0 where there are none: a
// weight it does not serve at all of them, or one whose 512-row product adds
// its K in halves (nf4_gemm_tile.hip's two-group form: few tiles, such as 4096
// x 2560 or 1024 x 3072).
extern "C" int ttsp_nf4_gemm_span_splits(int M, int K) {
  for (int n = 1024; n <= 2048; n += 512)
    if (!ttsp_nf4_gemm_dense_splits(M, K, n)) return 0;
  const int parts = ttsp_nf4_gemm_splits(M, K, 512);
  return tile_halves(M, 512, parts) ? 0 : parts;
}

// Y = epilogue(X . W^T). `work` (16-byte aligned) holds M * K dense weights,
// then, with K splits, splits * N * M fp32 partial sums.
extern "C" int ttsp_nf4_gemm_dense(const void* X, int x_dtype, const uint8_t* W, const uint8_t* A8, const float* AMAX,
                                   const float* CODE2, float offset, const float* LUT, void* Y, const void* R, int epi,
                                   int M, int K, int N, int blocksize, int blocksize2, void* work, hipStream_t stream) {
  const int bs = pow2_shift(blocksize), bs2 = A8 ? pow2_shift(blocksize2) : 0;
  const int splits = ttsp_nf4_gemm_dense_splits(M, K, N);
  if (!splits || !X || !W || !AMAX || !LUT || !Y || !work || (A8 && !CODE2) || bs < 6 || bs2 < 0 || K % blocksize ||
      epi < 0 || epi > 2 || (epi && !R) || (x_dtype != DT_BF16 && x_dtype != DT_F16))
    return (int)hipErrorInvalidValue;
  if ((uintptr_t)X % 16 || (uintptr_t)W % 4 || (uintptr_t)work % 16) return (int)hipErrorInvalidValue;
  const DensePlan plan = dense_plan(M, K, N);
  const DqMat m{(const uint32_t*)W, A8, AMAX, CODE2, offset};
  uint16_t* wd = (uint16_t*)work;
  float* yp = splits > 1 ? (float*)(wd + (size_t)M * K) : nullptr;
  const bool al16 = (uintptr_t)Y % 16 == 0 && (!epi || (uintptr_t)R % 16 == 0);
  const int e = epi | (al16 ? 8 : 0);
  const long long nd = (long long)M * K / 8;
#define TTSP_DENSE(DTV)                                                                                        \
  do {                                                                                                         \
    if (int rc = launch_dequant16<DTV>(m, m, 1, LUT, wd, nd, bs, bs2, stream)) return rc;                      \
    if (int rc = dense_form<DTV>(plan, X, wd, Y, R, e, M, K, N, yp, stream)) return rc;                        \
  } while (0)
  if (x_dtype == DT_BF16) TTSP_DENSE(DT_BF16);
  else TTSP_DENSE(DT_F16);
#undef TTSP_DENSE
  if (splits > 1)
    return gemm_reduce(x_dtype, yp, splits, Y, R, epi | (M % 8 == 0 && al16 ? 4 : 0), M, N, stream);
  return 0;
}

// Whether the SwiGLU pair is served as one matrix launch with the bits of two:
// where each weight's own product is served unsplit and in one run.
extern "C" int ttsp_nf4_gemm_dense_swiglu_fits(int M, int K, int N) {
  if (!dense_fits(M, K, N, 2) || ttsp_nf4_gemm_dense_splits(M, K, N) != 1) return 0;
  return dense_plan(M, K, N).runs == 1 ? 1 : 0;
}

// Y = round(round(silu(X . W1^T)) * round(X . W3^T)); `work` holds 2 * M * K
// dense weights. A tile takes alternate 32-row groups of the two weights, so a
// wave holds the gate and the up output of the same element.
extern "C" int ttsp_nf4_gemm_dense_swiglu(const void* X, int x_dtype, const uint8_t* W1, const uint8_t* A8_1,
                                          const float* AMAX_1, const float* CODE2_1, float offset_1, const uint8_t* W3,
                                          const uint8_t* A8_3, const float* AMAX_3, const float* CODE2_3,
                                          float offset_3, const float* LUT, void* Y, int M, int K, int N,
                                          int blocksize, int blocksize2, void* work, hipStream_t stream) {
  const int bs = pow2_shift(blocksize), bs2 = A8_1 ? pow2_shift(blocksize2) : 0;
  if (!ttsp_nf4_gemm_dense_swiglu_fits(M, K, N) || !X || !W1 || !W3 || !AMAX_1 || !AMAX_3 || !LUT || !Y || !work ||
      (A8_1 != nullptr) != (A8_3 != nullptr) || (A8_1 && (!CODE2_1 || !CODE2_3)) || bs < 6 || bs2 < 0 ||
      K % blocksize || (x_dtype != DT_BF16 && x_dtype != DT_F16))
    return (int)hipErrorInvalidValue;
  if ((uintptr_t)X % 16 || (uintptr_t)W1 % 4 || (uintptr_t)W3 % 4 || (uintptr_t)work % 16)
    return (int)hipErrorInvalidValue;
  const DqMat a{(const uint32_t*)W1, A8_1, AMAX_1, CODE2_1, offset_1};
  const DqMat b{(const uint32_t*)W3, A8_3, AMAX_3, CODE2_3, offset_3};
  uint16_t* wd = (uint16_t*)work;
  const long long nd = (long long)M * K / 8;
  const int e = (uintptr_t)Y % 16 == 0 ? 8 : 0;
  if (x_dtype == DT_BF16) {
    if (int rc = launch_dequant16<DT_BF16>(a, b, 2, LUT, wd, nd, bs, bs2, stream)) return rc;
    return launch_dense<DT_BF16, Tall, true, false>(X, wd, Y, nullptr, e, M, K, N, 1, 1, nullptr, stream);
  }
  if (int rc = launch_dequant16<DT_F16>(a, b, 2, LUT, wd, nd, bs, bs2, stream)) return rc;
  return launch_dense<DT_F16, Tall, true, false>(X, wd, Y, nullptr, e, M, K, N, 1, 1, nullptr, stream);
}
