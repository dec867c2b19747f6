// Top-k / top-p / temperature draw of one logit row in one workgroup.
//
// Result (what the reference's fused sampler returns, app/engine/
// fusedsample.py:1-19): take the k = min(max(TOPK, 1), 64, V) largest logits,
// ties to the lowest index, in descending order; keep the first and every one
// whose inclusive cumulative probability under softmax(row) is <= TOPP; draw
// argmax over the kept of l / max(T, 1e-5) - log(-log(max(u, 1e-20))), with u
// the caller's uniform number of that vocabulary index (the Gumbel form of the
// fork's argmax(probs / Exp(1))), ties to the lowest index.
//
// Design (one workgroup of 4 waves; thread t holds elements t, t + 256, ...):
//   1. Every element is requested before the first is used, and becomes an
//      order-preserving 16-bit key in a register (a float's bit pattern with
//      the sign bit flipped, all bits flipped for negative values: unsigned
//      key order is float order). The block max M and the softmax normaliser
//      Z = sum exp(l - M) follow (fixed order: thread, wave, then the four
//      waves in turn; the sum reads the row from LDS in a rolled loop, since
//      an exp per register would be tens of KB of code fetched cold).
//   2. The k-th largest key t is built bit by bit from the top: a candidate
//      prefix survives when at least k keys are >= it. Counting is by wave
//      ballots - one compare and popcount per key register, summed in scalar
//      registers - and the four wave counts meet in LDS; 16 rounds, one
//      barrier each.
//   3. Every key > t (fewer than k) and the first k - #(> t) keys equal to t in
//      index order become the k candidates: the ballots' counts per (slot,
//      wave), which are in index order, get an exclusive prefix sum in LDS, and
//      a lane's place is that plus the ballot's bits below it.
//   4. One wave orders the candidates by rank counting: candidate c's rank is
//      the number of candidates that beat it (larger key, or equal key and
//      lower index), so ranks are a permutation and no sorting network is
//      needed; the others' keys come by readlane.
//   5. It finishes: lane j holds the j-th candidate's probability, an inclusive
//      scan gives the cumulative mass, the top-p cut and the scores follow, and
//      a butterfly over (score, index) picks the draw.
// Bound by the serial chain of these steps. With the keys in LDS (read again
// in each of the 16 rounds, and by index for the candidates) a 4096-entry row
// took 38 us; now 12 (500 entries 11.3 -> 7.4, 8193 70.5 -> 30.9, 32768 264 -> 82).
#include "ttsp_common.h"

namespace ttsp {

constexpr int SMP_THREADS = 256;
constexpr int SMP_WAVES = SMP_THREADS / 64;
constexpr int SMP_MAX_K = 64;
constexpr int SMP_MAX_V = 32768;  // 128 key registers a thread, the row in 64 KB of LDS

__device__ __forceinline__ uint32_t key_of(uint32_t h) { return (h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u); }
__device__ __forceinline__ uint32_t bits_of(uint32_t k) { return (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu); }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) v = fmaxf(v, __shfl_xor(v, d));
  return v;
}

// Inclusive prefix sum over the 64 lanes (Hillis-Steele, fixed order).
template <typename T>
__device__ __forceinline__ T wave_scan(T v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T o = __shfl_up(v, d);
    if (lane >= d) v = v + o;
  }
  return v;
}

// SL: key registers a thread (V <= 256 SL). A register past the row costs its
// share of every count, so there are five: 64 entries took 9.2 us with 16 and
// take 6.3 with 2 (7.6 before), 8193 took 71.4 with 128 and take 29.5 with 64.
template <int DT, int SL>
__global__ __launch_bounds__(SMP_THREADS) void sample_topk_kernel(const uint16_t* __restrict__ L, int V,
                                                                  const uint16_t* __restrict__ TEMP,
                                                                  const uint16_t* __restrict__ TOPP,
                                                                  const long long* __restrict__ TOPK,
                                                                  const float* __restrict__ U, int* __restrict__ OUT) {
  constexpr int NC = SL * SMP_WAVES;  // (slot, wave) counts, in index order
  __shared__ uint16_t row[SL * SMP_THREADS];
  __shared__ float red[SMP_WAVES];
  __shared__ int cnt[2][SMP_WAVES];
  __shared__ int cgt[NC], ceq[NC], total_s;
  __shared__ int cand[SMP_MAX_K], candk[SMP_MAX_K];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = (int)min(min(max(TOPK[0], 1LL), (long long)SMP_MAX_K), (long long)V);
  const uint32_t temp = TEMP[0], topp = TOPP[0];

  // 1. keys, block max, normaliser
  uint32_t key[SL];
#pragma unroll
  for (int j = 0; j < SL; ++j) key[j] = L[min(tid + SMP_THREADS * j, V - 1)];
  float mx = -__builtin_inff();
#pragma unroll
  for (int j = 0; j < SL; ++j) {
    const int i = tid + SMP_THREADS * j;
    if (i < V) mx = fmaxf(mx, Elem<DT>::load(key[j]));
    row[i] = (uint16_t)key[j];
    key[j] = i < V ? key_of(key[j]) : 0u;  // (past the row: below every candidate prefix)
  }
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  float M = red[0];
#pragma unroll
  for (int w = 1; w < SMP_WAVES; ++w) M = fmaxf(M, red[w]);
  float z = 0.0f;
#pragma unroll 4
  for (int i = tid; i < V; i += SMP_THREADS) z = __fadd_rn(z, exp_cw(__fsub_rn(Elem<DT>::load(row[i]), M)));
  z = wave_sum_dpp(z);
  __syncthreads();  // every wave has read red[] as maxima
  if (lane == 0) red[wave] = z;

  // 2. the k-th largest key
  uint32_t t = 0;
#pragma unroll 1
  for (int bit = 15; bit >= 0; --bit) {
    const uint32_t c = t | (1u << bit);
    int n = 0;  // wave-uniform: the wave's keys >= c
#pragma unroll
    for (int j = 0; j < SL; ++j) n += __popcll(__ballot(key[j] >= c));
    if (lane == 0) cnt[bit & 1][wave] = n;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int w = 0; w < SMP_WAVES; ++w) total += cnt[bit & 1][w];
    if (total >= k) t = c;
  }
  float Z = red[0];
#pragma unroll
  for (int w = 1; w < SMP_WAVES; ++w) Z = __fadd_rn(Z, red[w]);

  // 3. index-ordered places: all keys > t, then the first `need` keys == t
#pragma unroll
  for (int j = 0; j < SL; ++j) {
    const int ngt = __popcll(__ballot(key[j] > t));
    const int neq = __popcll(__ballot(key[j] == t && tid + SMP_THREADS * j < V));
    if (lane == 0) cgt[j * SMP_WAVES + wave] = ngt, ceq[j * SMP_WAVES + wave] = neq;
  }
  __syncthreads();
  if (wave < 2) {  // one wave a list: lane l sums its NC / 64 entries
    int* const list = wave ? ceq : cgt;
    constexpr int PER = NC > 64 ? NC / 64 : 1;
    int v[PER], s = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) v[e] = NC >= 64 || lane < NC ? list[lane * PER + e] : 0, s += v[e];
    const int inc = wave_scan(s, lane);
    int at = inc - s;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      if (NC >= 64 || lane < NC) list[lane * PER + e] = at;
      at += v[e];
    }
    if (wave == 0 && lane == 63) total_s = inc;
  }
  __syncthreads();
  const int total_gt = total_s, need = k - total_gt;  // need >= 1 by the choice of t
  const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
  for (int j = 0; j < SL; ++j) {
    const int i = tid + SMP_THREADS * j;
    const bool gt = key[j] > t, eq = key[j] == t && i < V;
    const unsigned long long bg = __ballot(gt), be = __ballot(eq);
    if (bg | be) {
      int at = -1;
      if (gt) at = cgt[j * SMP_WAVES + wave] + __popcll(bg & below);
      if (eq) {
        const int r = ceq[j * SMP_WAVES + wave] + __popcll(be & below);
        if (r < need) at = total_gt + r;
      }
      if (at >= 0) cand[at] = i, candk[at] = (int)key[j];
    }
  }
  __syncthreads();
  if (wave != 0) return;

  // 4. rank counting (one wave from here on): key and index in one word, which
  // is larger for the larger key or the lower index (V <= 2^15)
  const int me = lane < k ? cand[lane] : 0, mk = lane < k ? candk[lane] : 0;
  const uint32_t word = ((uint32_t)mk << 16) | (0xffffu - (uint32_t)me);
  int rank = 0;
#pragma unroll 4
  for (int j = 0; j < k; ++j) rank += (uint32_t)__builtin_amdgcn_readlane((int)word, j) > word;
  __builtin_amdgcn_wave_barrier();
  if (lane < k) cand[rank] = me, candk[rank] = mk;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  // 5. cumulative mass, top-p cut, draw
  const float T = fmaxf(Elem<DT>::load(temp), 1e-5f);
  const float P = Elem<DT>::load(topp);
  int idx = 0x7fffffff;
  float p = 0.0f, l = 0.0f;
  if (lane < k) {
    idx = cand[lane];
    l = Elem<DT>::load(bits_of((uint32_t)candk[lane]));
    p = __fdiv_rn(exp_cw(__fsub_rn(l, M)), Z);
  }
  const float c = wave_scan(p, lane);
  const bool keep = lane < k && (lane == 0 || c <= P);
  float score = -__builtin_inff();
  if (keep) {
    const float g = -logf(-logf(fmaxf(U[idx], 1e-20f)));
    score = __fadd_rn(__fdiv_rn(l, T), g);
  } else {
    idx = 0x7fffffff;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float os = __shfl_xor(score, d);
    const int oi = __shfl_xor(idx, d);
    if (os > score || (os == score && oi < idx)) score = os, idx = oi;
  }
  if (lane == 0) OUT[0] = idx;
}

template <int DT>
void launch_sample(const uint16_t* L, int V, const uint16_t* TEMP, const uint16_t* TOPP, const long long* TOPK,
                   const float* U, int* OUT, hipStream_t st) {
#define TTSP_SMP(SLV) \
  hipLaunchKernelGGL((sample_topk_kernel<DT, SLV>), dim3(1), dim3(SMP_THREADS), 0, st, L, V, TEMP, TOPP, TOPK, U, OUT)
  if (V <= 2 * SMP_THREADS) TTSP_SMP(2);
  else if (V <= 16 * SMP_THREADS) TTSP_SMP(16);
  else if (V <= 32 * SMP_THREADS) TTSP_SMP(32);
  else if (V <= 64 * SMP_THREADS) TTSP_SMP(64);
  else TTSP_SMP(128);
#undef TTSP_SMP
}

}  // namespace ttsp

using namespace ttsp;

extern "C" int ttsp_sample_max_top_k(void) { return SMP_MAX_K; }

extern "C" int ttsp_sample_max_vocab(void) { return SMP_MAX_V; }

extern "C" int ttsp_sample_topk(const void* L, int V, int dtype, const void* TEMP, const void* TOPP,
                                const long long* TOPK, const float* U, int* OUT, void* stream) {
  if (!L || !TEMP || !TOPP || !TOPK || !U || !OUT || V <= 0 || V > SMP_MAX_V) return (int)hipErrorInvalidValue;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DT_BF16)
    launch_sample<DT_BF16>((const uint16_t*)L, V, (const uint16_t*)TEMP, (const uint16_t*)TOPP, TOPK, U, OUT, st);
  else if (dtype == DT_F16)
    launch_sample<DT_F16>((const uint16_t*)L, V, (const uint16_t*)TEMP, (const uint16_t*)TOPP, TOPK, U, OUT, st);
  else
    return (int)hipErrorInvalidValue;
  TTSP_RETURN_LAUNCH();
}
