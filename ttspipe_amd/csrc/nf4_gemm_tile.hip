// NF4 matrix product for 65 to 512 activation rows (and the shapes the other
// kernels leave): Y[N][M] = X[N][K] . W^T, the weight in the bitsandbytes NF4
// layout (nf4_gemv.hip gives it), each dequantised weight the exact
// round(code * scale) of bitsandbytes' dequantize_4bit.
//
// A wave owns 32 weight rows x 128 activation rows (four 32x32 MFMA blocks); a
// workgroup is W such waves, on KG halves of its K-steps. Activations (shared
// by a half's waves) and each wave's own codes reach a three-stage LDS ring by
// buffer_load ... lds, so nothing is staged in registers. Inside a row's LDS
// copy 16-byte segment s of row t sits at slot s ^ ((t >> 1) & 7).
//
// The loop is one long pipeline. Dequantisation (lookups in a table of code
// pairs, fp32 products with the scale, one pack-convert a pair) takes about as
// many issue slots as the products take matrix-core time, so each slice's
// products are woven with the next slice's arithmetic, the lookups of the one
// after and its activation reads, across steps too: the next step's codes are
// the wave's own loads and need no barrier, and the last slice is multiplied
// past the barrier, under the next step's first reads. Without the weaving a
// step of one 256-row workgroup took 0.94 us, with it 0.74 (9728 x 2560 at 512
// rows 43 -> 36 us; the kernel before, two-stage and unwoven, 51).
//
// Forms (bf16, nested, us, the kernels replaced against this):
// * 64 rows a workgroup with both K halves (W 2, KG 2), where those tiles fit
//   one to a CU: 9728 x 2560 at 100 rows 27.0 -> 19.6, 6144 x 2560 at 256
//   26.6 -> 19.1, 2560 x 9728 at 100 (4 splits) 28.2 -> 22.8. One copy of the
//   code table: its few waves gain less from 16 copies than writing them costs
//   (at 16 copies 19.8, 19.5 and 23.2; 1024 x 1024 at 256 rows, where a short K
//   leaves the prologue most of the launch, 10.9 against 10.4, and in 2 splits
//   slower than the kernel before).
// * 256 rows (W 8) where more than half the CUs get one: one code table serves
//   eight waves, so it can hold 32 copies (64 KB: a lookup's 64 lanes then
//   touch every bank the minimum number of times), -5 % against one copy.
// * 128 rows (W 4) between: 9728 x 2560 at 256 rows 34.1 -> 28.0. At 128 of the
//   256-row tiles, where 128-row ones still fit one to a CU, they are the
//   faster: 8192 x 2560 at 512 rows 33.4 -> 29.3, with a gate 42.6 -> 35.7; 4096 x
//   1024 at 1000 rows with a gate 27.2 -> 21.7 (24.5 in the kernel before).
// The SwiGLU form takes W 4 with one copy, so that two workgroups fit a CU
// (9728 x 2560 at 512 rows 86 -> 73; W 8 with 32 copies was slower).
#include "nf4_mfma.h"

namespace ttsp {

namespace {

constexpr int KT = 64;            // codes per K-step
constexpr int CH = 1024;          // bytes of one wave-wide load
constexpr int BN = 128;           // activation rows per workgroup
constexpr int BSTAGE = BN * 128;  // activation bytes per step
constexpr int ST = 3;             // ring stages
constexpr int SC = 15;            // steps whose scales a wave resolves at once (a multiple of ST, at most 16)
constexpr int SP = 33;            // pitch of a step's 32 scales

struct TileMat {
  const uint8_t* W;
  const uint8_t* A8;
  const float* AMAX;
  const float* CODE2;
  float offset;
};

template <int W, typename RS>
__device__ __forceinline__ void tile_load(uint8_t* __restrict__ dst, RS xr, RS wr, const uint32_t (&xoff)[16 / W],
                                          uint32_t woff, int k0, int wave) {
#pragma unroll
  for (int j = 0; j < 16 / W; ++j)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr_t)(dst + (wave * (16 / W) + j) * CH), 16, xoff[j], k0 * 2, 0,
                                             0);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr_t)(dst + BSTAGE + wave * CH), 16, woff, k0 / 2, 0, 0);
}

// What a wave carries between calls of tile_step: the dequantised fragment and
// the X fragments of the step's slice 0, the codes of the step, the code pairs
// of slices 0 (used) and 1, and the block scale.
struct TileRegs {
  u32x4 codes, af;
  u32x4 bf[2][4];
  float2 pc[2][4];
  float s;
};

template <int DT>
__device__ __forceinline__ u32x4 dequant8(const float2 (&pc)[4], float s) {
  u32x4 af;
#pragma unroll
  for (int e = 0; e < 4; ++e) af[e] = pack2<DT>(__fmul_rn(pc[e].x, s), __fmul_rn(pc[e].y, s));
  return af;
}

template <int REP>
__device__ __forceinline__ void lookup(const float2* __restrict__ lut, uint32_t lane8, uint32_t w, float2 (&pc)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t a;
    if constexpr (REP == 32) a = __builtin_amdgcn_perm(w, lane8, 0x0C0C0400u + ((uint32_t)j << 8));
    else a = ((w >> (8 * j)) & 0xffu) * (8 * REP) + lane8;
    pc[j] = *reinterpret_cast<const float2*>(reinterpret_cast<const uint8_t*>(lut) + a);
  }
}

__device__ __forceinline__ void read_x(const uint8_t* rd, int lane, int kk, u32x4 (&bf)[4]) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int t = 32 * b + (lane & 31), sg = 4 * (lane >> 5) + kk;
    bf[b] = *reinterpret_cast<const u32x4*>(rd + t * 128 + ((sg ^ ((t >> 1) & 7)) << 4));
  }
}

// the region's instruction order: each product followed by a share of the
// other slices' reads and arithmetic, which run under it
__device__ __forceinline__ void weave() {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS reads
    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // VALU
  }
  __builtin_amdgcn_sched_barrier(0);
}

// One step. rd: its stage, landed for every wave; nx: the next step's, whose
// loads the caller's wave has waited for when wait() returns (its own codes)
// and all waves' past the barrier; dst (= rd) then takes the step after the
// ring's.
template <int DT, int W, int REP, int VM, bool LAST, typename RS>
__device__ __forceinline__ void tile_step(const uint8_t* __restrict__ rd, const uint8_t* __restrict__ nx,
                                          uint8_t* __restrict__ dst, const float2* __restrict__ lut,
                                          const float* __restrict__ scn, RS xr, RS wr, const uint32_t (&xoff)[16 / W],
                                          uint32_t woff, int k0n, int wave, int lane, uint32_t lane8, TileRegs& g,
                                          f32x16_v (&acc)[4]) {
  u32x4 an;
  // slice 0's products; slice 1's fragments, slice 2's lookups
  read_x(rd, lane, 1, g.bf[1]);
  an = dequant8<DT>(g.pc[1], g.s);
  lookup<REP>(lut, lane8, g.codes[2], g.pc[0]);
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = mfma32<DT>(g.af, g.bf[0][b], acc[b]);
  weave();
  g.af = an;
  read_x(rd, lane, 2, g.bf[0]);
  an = dequant8<DT>(g.pc[0], g.s);
  lookup<REP>(lut, lane8, g.codes[3], g.pc[1]);
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = mfma32<DT>(g.af, g.bf[1][b], acc[b]);
  weave();
  g.af = an;
  // the next step's codes: this wave's own loads
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
  u32x4 cn;
  float sn;
  if constexpr (!LAST) {
    cn = *reinterpret_cast<const u32x4*>(nx + BSTAGE + wave * CH + lane * 16);
    sn = *scn;
  }
  read_x(rd, lane, 3, g.bf[1]);
  an = dequant8<DT>(g.pc[1], g.s);
  if constexpr (!LAST) lookup<REP>(lut, lane8, cn[0], g.pc[0]);
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = mfma32<DT>(g.af, g.bf[0][b], acc[b]);
  weave();
  g.af = an;
  if constexpr (LAST) {
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = mfma32<DT>(g.af, g.bf[1][b], acc[b]);
  } else {
    TTSP_WAIT_LGKM0();  // this wave is done reading the stage, and (above) its loads of the next have landed
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    g.codes = cn;
    g.s = sn;
    read_x(nx, lane, 0, g.bf[0]);
    tile_load<W>(dst, xr, wr, xoff, woff, k0n, wave);
    an = dequant8<DT>(g.pc[0], g.s);
    lookup<REP>(lut, lane8, g.codes[1], g.pc[1]);
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = mfma32<DT>(g.af, g.bf[1][b], acc[b]);
    weave();
    g.af = an;
  }
}

// W waves of 32 weight rows each, KG groups of them over the workgroup's
// K-steps. SW: the SwiGLU form, waves 0 .. W / 2 - 1 take rows of the first
// weight (the gate), the others the same rows of the second.
template <int DT, bool NESTED, int W, int KG, int REP, bool SW>
__global__ __launch_bounds__(64 * W * KG) void nf4_gemm_tile_kernel(
    const uint16_t* __restrict__ X, TileMat m1, TileMat m3, const float* __restrict__ LUT, uint16_t* __restrict__ Y,
    const uint16_t* __restrict__ R, int epi, int M, int K, int N, int bs_shift, int bs2_shift, float* __restrict__ YP) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NT = 64 * W * KG, BM = 32 * W, BMO = SW ? BM / 2 : BM;
  constexpr int STAGE = BSTAGE + W * CH, L = 16 / W + 1;
  __shared__ __align__(16) uint8_t ring0[KG][STAGE];
  __shared__ __align__(16) uint8_t ring1[KG][STAGE];
  __shared__ __align__(16) uint8_t ring2[KG][STAGE];
  __shared__ __align__(16) float2 lut2_s[256 * REP];
  __shared__ float code2_s[NESTED ? (SW ? 512 : 256) : 1];
  __shared__ float sc_s[W * KG][SC * SP];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wid % W, kg = wid / W;
  // XCD x takes a contiguous run of tiles (workgroup b runs on XCD b % 8), the
  // activation tiles innermost: their workgroups share the weight's codes
  const int tn = (N + BN - 1) / BN, total = gridDim.x, xcd = blockIdx.x & 7;
  const int tile = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  const int n0 = (tile % tn) * BN, m0 = (tile / tn) * BMO;
  const bool second = SW && wave >= W / 2;
  const uint8_t* const Wm = second ? m3.W : m1.W;
  const uint8_t* const A8m = second ? m3.A8 : m1.A8;
  const float* const AMm = second ? m3.AMAX : m1.AMAX;
  const float offm = second ? m3.offset : m1.offset;
  // this group's K-steps: run z KG + kg of gridDim.z KG equal ones
  const int steps = K / KT, ns = steps / (int)(gridDim.z * KG), s_lo = (blockIdx.z * KG + kg) * ns;

  const float lutl = LUT[lane & 15];
  const float lutv0 = LUT[(tid & 255) >> 4], lutv1 = LUT[tid & 15];
  float c2v[SW ? 2 : 1];
  if constexpr (NESTED) {
    c2v[0] = m1.CODE2[tid & 255];
    if constexpr (SW) c2v[1] = m3.CODE2[tid & 255];
  }
  const int mw = m0 + 32 * (second ? wave - W / 2 : wave);  // this wave's first weight row
  const uint32_t rowblk = (uint32_t)(K >> bs_shift);
  uint32_t a8v[8];
  float amv[8];
  auto load_scales = [&](int base) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = min(mw + 4 * i + (lane >> 4), M - 1), s = min(base + (lane & 15), steps - 1);
      const size_t b = (size_t)row * rowblk + ((uint32_t)(s * KT) >> bs_shift);
      if constexpr (NESTED) {
        a8v[i] = A8m[b];
        amv[i] = AMm[b >> bs2_shift];
      } else {
        amv[i] = AMm[b];
      }
    }
  };
  auto store_scales = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float s = amv[i];
      if constexpr (NESTED) s = __fadd_rn(__fmul_rn(code2_s[(second ? 256 : 0) + a8v[i]], s), offm);
      if ((lane & 15) < SC) sc_s[wid][(lane & 15) * SP + 4 * i + (lane >> 4)] = s;
    }
  };
  load_scales(s_lo);

  // buffers that start at the tile's first rows: offsets stay below 2^31 for any M and N
  const size_t rowbytes = (size_t)K / 2;
  const size_t xbytes = (size_t)min(BN, N - n0) * K * 2, wbytes = (size_t)min(BMO, M - m0) * rowbytes;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(X) + (size_t)n0 * K, (short)0, (int)xbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(Wm) + (size_t)m0 * rowbytes, (short)0, (int)wbytes, 0x00020000);
  uint32_t xoff[16 / W];
#pragma unroll
  for (int j = 0; j < 16 / W; ++j) {
    const int t = 8 * (wave * (16 / W) + j) + (lane >> 3), sg = (lane & 7) ^ ((t >> 1) & 7);
    xoff[j] = (uint32_t)min(t, N - 1 - n0) * (uint32_t)K * 2u + (uint32_t)sg * 16u;
  }
  const uint32_t woff = (uint32_t)(min(mw + (lane & 31), M - 1) - m0) * (uint32_t)rowbytes + 16u * (lane >> 5);
  auto koff = [&](int s) { return (s_lo + min(s, ns - 1)) * KT; };
  tile_load<W>(ring0[kg], xr, wr, xoff, woff, koff(0), wave);
  tile_load<W>(ring1[kg], xr, wr, xoff, woff, koff(1), wave);
  if constexpr (REP == 1) {
    lut2_s[tid & 255] = make_float2(lutv0, lutv1);
  } else {
    // thread t writes copies of entry t / (REP / 2) + ..: two 8-byte copies a store
    constexpr int PER = REP / 2;
#pragma unroll
    for (int i = 0; i < 256 * PER / NT; ++i) {
      const int q = i * NT + tid, e = q / PER;
      const float hi = __shfl(lutl, e >> 4), lo = __shfl(lutl, e & 15);
      *reinterpret_cast<float4*>(&lut2_s[e * REP + 2 * (q % PER)]) = make_float4(hi, lo, hi, lo);
    }
  }
  if constexpr (NESTED) {
    code2_s[tid & 255] = c2v[0];
    if constexpr (SW) code2_s[256 + (tid & 255)] = c2v[1];
  }
  TTSP_WAIT_LGKM0();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  store_scales();

  f32x16_v acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.0f;

  tile_load<W>(ring2[kg], xr, wr, xoff, woff, koff(2), wave);
  TTSP_WAIT_VM_LGKM0((ST - 1) * L);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const uint32_t lane8 = 8u * (lane & (REP - 1));
  const float* const scl = &sc_s[wid][lane & 31];
  TileRegs g;
  g.codes = *reinterpret_cast<const u32x4*>(ring0[kg] + BSTAGE + wave * CH + lane * 16);
  g.s = scl[0];
  read_x(ring0[kg], lane, 0, g.bf[0]);
  lookup<REP>(lut2_s, lane8, g.codes[0], g.pc[0]);
  lookup<REP>(lut2_s, lane8, g.codes[1], g.pc[1]);
  g.af = dequant8<DT>(g.pc[0], g.s);
  // c: the next step's index in the chunk of resolved scales
  auto one = [&](int s, int c, const uint8_t* rd, const uint8_t* nx, uint8_t* dst) {
    tile_step<DT, W, REP, (ST - 2) * L, false>(rd, nx, dst, lut2_s, scl + c * SP, xr, wr, xoff, woff, koff(s + ST),
                                               wave, lane, lane8, g, acc);
  };
  int c = 0;
  int s = 0;
  for (; s + 3 < ns; s += 3) {
    one(s, c + 1, ring0[kg], ring1[kg], ring0[kg]);
    one(s + 1, c + 2, ring1[kg], ring2[kg], ring1[kg]);
    c += 3;
    if (c == SC) {  // the next steps' scales (the chunk's own have all been read; SC is a multiple of 3)
      load_scales(s_lo + s + 3);
      store_scales();
      c = 0;
    }
    one(s + 2, c, ring2[kg], ring0[kg], ring2[kg]);
  }
  const uint8_t* lastst = ring0[kg];
  if (s + 1 < ns) {
    one(s, c + 1, ring0[kg], ring1[kg], ring0[kg]);
    lastst = ring1[kg];
  }
  if (s + 2 < ns) {
    one(s + 1, c + 2, ring1[kg], ring2[kg], ring1[kg]);
    lastst = ring2[kg];
  }
  tile_step<DT, W, REP, 0, true>(lastst, lastst, ring0[kg], lut2_s, scl, xr, wr, xoff, woff, 0, wave, lane, lane8, g, acc);
  TTSP_WAIT_VM_LGKM0(0);
  __syncthreads();  // the ring is free

  if constexpr (KG == 2) {  // the second group's sums join the first's
    static_assert(W * 4 * 16 * 64 * 4 <= KG * STAGE, "the sums exceed a ring stage");
    float* p = reinterpret_cast<float*>(&ring0[0][0]) + wave * 4096 + lane;
    if (kg == 1) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) p[(b * 16 + r) * 64] = acc[b][r];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = __fadd_rn(acc[b][r], p[(b * 16 + r) * 64]);
    }
  }
  if (YP) {
    if (kg) return;
    // each wave's 32 x 32 blocks through LDS of its own, so that a store writes
    // whole 128-byte pieces of 8 rows, not 32 bytes of 32 (512 rows, traced:
    // 6144 x 2560 in 2 splits 30.1 -> 27.3 us, 2560 x 4096 in 4 26.3 -> 22.4,
    // 2560 x 9728 in 4 42.2 -> 40.6)
    constexpr int PP = 36;  // floats a staged row
    static_assert(4 * 32 * PP * 4 <= KG * STAGE, "four waves' blocks exceed a ring stage");
    float* const ws = reinterpret_cast<float*>((wave & 4 ? &ring2[0][0] : &ring1[0][0]) + (wave & 3) * (32 * PP * 4));
    float* yp = YP + (size_t)blockIdx.z * N * M;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(ws + (lane & 31) * PP + 8 * g + 4 * (lane >> 5)) =
            make_float4(acc[b][4 * g], acc[b][4 * g + 1], acc[b][4 * g + 2], acc[b][4 * g + 3]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int nl = 8 * j + (lane >> 3), n = n0 + 32 * b + nl, m = mw + 4 * (lane & 7);
        const float4 v = *reinterpret_cast<const float4*>(ws + nl * PP + 4 * (lane & 7));
        if (n >= N || m >= M) continue;
        const size_t o = (size_t)n * M + m;
        if ((M & 3) == 0) {
          *reinterpret_cast<float4*>(yp + o) = v;
        } else {
          for (int c = 0; c < 4; ++c)
            if (m + c < M) yp[o + c] = c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
        }
      }
    }
    return;
  }
  // the rounded tile through the ring's three stages, stored as 16-byte pieces
  // of whole rows. The epilogue's operands are requested before the staging
  // (read piece by piece in the loop they cost a memory round trip a turn) and
  // the gate's eight silus run interleaved; what is left of the gate is its
  // arithmetic, 64 silus a thread. us, plain / residual / gate: 9728 x 2560 at
  // 256 rows 25.7 / 31.2 / 37.0 before, 25.4 / 27.8 / 31.3; 3072 x 1024 at 512
  // 11.2 / 13.2 / 16.5 before, 10.5 / 11.7 / 13.5.
  constexpr int PITCH = BM * 2 + 16, CPR = BMO / 8, STEP = NT / CPR, IT = BN / STEP;
  constexpr int RPS = KG * STAGE / PITCH;  // rows a stage holds
  static_assert(3 * RPS >= BN && NT % CPR == 0 && BN % STEP == 0, "the tile exceeds the ring");
  static_assert(KG == 1 || RPS >= BN, "ring0 may still be read (the second group's sums)");
  auto row_at = [&](int n) {
    if (RPS >= BN || n < RPS) return &ring1[0][0] + n * PITCH;
    return n < 2 * RPS ? &ring2[0][0] + (n - RPS) * PITCH : &ring0[0][0] + (n - 2 * RPS) * PITCH;
  };
  const int ep = SW ? 2 : epi & 3;
  const int ch = tid % CPR, m = m0 + ch * 8;
  const bool full = (M & 7) == 0 && (epi & 8) && m + 8 <= M;
  constexpr int IR = SW ? 1 : IT;
  u32x4 rr[IR];
#pragma unroll
  for (int i = 0; i < IR; ++i) rr[i] = u32x4{0, 0, 0, 0};
  if (!SW && ep && full) {
#pragma unroll
    for (int i = 0; i < IR; ++i)
      rr[i] = *reinterpret_cast<const u32x4*>(R + (size_t)min(n0 + tid / CPR + i * STEP, N - 1) * M + m);
  }
  if (kg == 0) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      uint8_t* const row = row_at(32 * b + (lane & 31)) + wave * 64 + (lane >> 5) * 8;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2*>(row + g * 16) = make_uint2(pack2<DT>(acc[b][4 * g], acc[b][4 * g + 1]),
                                                             pack2<DT>(acc[b][4 * g + 2], acc[b][4 * g + 3]));
    }
  }
  __syncthreads();
  if (!SW && !ep && full) {  // nothing to compute: all reads, then all stores
    u32x4 y[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) y[i] = *reinterpret_cast<const u32x4*>(row_at(tid / CPR + i * STEP) + ch * 16);
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int n = n0 + tid / CPR + i * STEP;
      if (n < N) *reinterpret_cast<u32x4*>(Y + (size_t)n * M + m) = y[i];
    }
    return;
  }
#pragma unroll 1
  for (int i = 0; i < IT; ++i) {
    const int nl = tid / CPR + i * STEP, n = n0 + nl;
    const uint8_t* const src = row_at(nl) + ch * 16;
    u32x4 r = rr[0];
#pragma unroll
    for (int k = 0; k + 1 < IR; ++k) rr[k] = rr[k + 1];
    if (n >= N || m >= M) continue;
    const u32x4 y = *reinterpret_cast<const u32x4*>(src + (SW ? BMO * 2 : 0));
    if constexpr (SW) r = *reinterpret_cast<const u32x4*>(src);
    mm_store8<DT>(Y, R, (size_t)n * M + m, m, M, full, ep, y, SW || full, r);
  }
#endif
}

template <int DT, int W, int KG, int REP, bool SW>
int launch_tile(const void* X, const TileMat& a, const TileMat& b, const float* LUT, void* Y, const void* R, int epi,
                int M, int K, int N, int bs_shift, int bs2_shift, int splits, float* YP, hipStream_t st) {
  constexpr int BMO = SW ? 16 * W : 32 * W;
  const long long tiles = (long long)((M + BMO - 1) / BMO) * ((N + BN - 1) / BN);
  if (tiles > 0x7fffffffll) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)tiles, 1, splits), block(64 * W * KG);
  if (a.A8)
    hipLaunchKernelGGL((nf4_gemm_tile_kernel<DT, true, W, KG, REP, SW>), grid, block, 0, st, (const uint16_t*)X, a, b,
                       LUT, (uint16_t*)Y, (const uint16_t*)R, epi, M, K, N, bs_shift, bs2_shift, YP);
  else
    hipLaunchKernelGGL((nf4_gemm_tile_kernel<DT, false, W, KG, REP, SW>), grid, block, 0, st, (const uint16_t*)X, a, b,
                       LUT, (uint16_t*)Y, (const uint16_t*)R, epi, M, K, N, bs_shift, bs2_shift, YP);
  TTSP_RETURN_LAUNCH();
}

}  // namespace

bool tile_halves(int M, int N, int splits);

namespace {

template <int DT>
int tile_form(const void* X, const TileMat& a, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N,
              int bs_shift, int bs2_shift, int splits, float* YP, hipStream_t st) {
  const long long nt = (long long)((N + BN - 1) / BN) * splits;
  if (tile_halves(M, N, splits))
    return launch_tile<DT, 2, 2, 1, false>(X, a, a, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
  if ((M + 255) / 256 * nt > 128)
    return launch_tile<DT, 8, 1, 32, false>(X, a, a, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
  return launch_tile<DT, 4, 1, 32, false>(X, a, a, LUT, Y, R, epi, M, K, N, bs_shift, bs2_shift, splits, YP, st);
}

}  // namespace

// Whether gemm_tile adds a split's sums as two K halves (tile_form's first
// form) instead of in one run along K.
bool tile_halves(int M, int N, int splits) {
  return (long long)((M + 63) / 64) * ((N + BN - 1) / BN) * splits <= 256;
}

// splits > 1 writes fp32 partials to YP [splits][N][M] (the caller reduces
// them and applies the epilogue), each split a whole even number of K-steps;
// else Y with epilogue epi & 3. 16-byte alignment of Y and R is checked here.
int gemm_tile(const void* X, int dt, const uint8_t* W, const uint8_t* A8, const float* AMAX, const float* CODE2,
              float offset, const float* LUT, void* Y, const void* R, int epi, int M, int K, int N, int bs_shift,
              int bs2_shift, int splits, float* YP, hipStream_t st) {
  if (splits < 1 || K % (2 * KT * splits) || (splits > 1 && !YP)) return (int)hipErrorInvalidValue;
  if ((uintptr_t)X % 16 || (uintptr_t)W % 16) return (int)hipErrorInvalidValue;  // 16-byte loads to LDS
  const TileMat a{W, A8, AMAX, CODE2, offset};
  const bool al16 = (uintptr_t)Y % 16 == 0 && (!(epi & 3) || (uintptr_t)R % 16 == 0);
  const int e = (epi & 3) | (al16 ? 8 : 0);
  float* yp = splits > 1 ? YP : nullptr;
  if (dt == DT_BF16) return tile_form<DT_BF16>(X, a, LUT, Y, R, e, M, K, N, bs_shift, bs2_shift, splits, yp, st);
  if (dt == DT_F16) return tile_form<DT_F16>(X, a, LUT, Y, R, e, M, K, N, bs_shift, bs2_shift, splits, yp, st);
  return (int)hipErrorInvalidValue;
}

// Y = round(round(silu(X . W1^T)) * round(X . W3^T)) in one unsplit launch,
// with the two launches' bits where they run unsplit on whole K (the caller
// checks the plan). Both weights share blocksize and nesting.
int gemm_tile_swiglu(const void* X, int dt, const uint8_t* W1, const uint8_t* A8_1, const float* AMAX_1,
                     const float* CODE2_1, float offset_1, const uint8_t* W3, const uint8_t* A8_3, const float* AMAX_3,
                     const float* CODE2_3, float offset_3, const float* LUT, void* Y, int M, int K, int N, int bs_shift,
                     int bs2_shift, hipStream_t st) {
  if ((uintptr_t)X % 16 || (uintptr_t)W1 % 16 || (uintptr_t)W3 % 16) return (int)hipErrorInvalidValue;
  const TileMat a{W1, A8_1, AMAX_1, CODE2_1, offset_1}, b{W3, A8_3, AMAX_3, CODE2_3, offset_3};
  const int e = (uintptr_t)Y % 16 == 0 ? 8 : 0;
  if (dt == DT_BF16)
    return launch_tile<DT_BF16, 4, 1, 1, true>(X, a, b, LUT, Y, nullptr, e, M, K, N, bs_shift, bs2_shift, 1, nullptr, st);
  if (dt == DT_F16)
    return launch_tile<DT_F16, 4, 1, 1, true>(X, a, b, LUT, Y, nullptr, e, M, K, N, bs_shift, bs2_shift, 1, nullptr, st);
  return (int)hipErrorInvalidValue;
}

}  // namespace ttsp
