// Sparse attention forward for calls with a handful of query rows (decode steps): one workgroup per (query row, head)
// streams the keys and values of the chunks the row selected, eight waves side by side, and merges their results in
// LDS.  Reads the selection bits, or picks the chunks itself from the scores that the pooling pass left (which spares the gate's launch),
// leaves no partial result in memory and needs no second launch.
//
// Bound by memory: with one row per sequence nothing is shared, every selected chunk is read once.  Each wave has a
// whole unit of 64 keys in flight (K and V, 32 KB at head dimension 128), one 16-byte piece per lane and load, LPR
// consecutive lanes on the same key, so every load instruction reads whole lines.  There is nothing for the matrix cores:
// a product with one row uses 1/32 of them, and the vector arithmetic (about 600 instructions per unit) hides under the
// loads.  16 requests against 512 to 32768 keys, 32 over 8 heads of 128, top-k 8 of 128-key chunks: 44 us, where the
// column form takes 113 us, its combine 6 and the lists it walks another 10.  (Held to 128 registers, for two workgroups per unit, it spills: 105.9 ->
// 107.0 us for the whole call, 8 requests, heads of 256 27.6 -> 30.0.)
#include "fmoba_common.h"

namespace fmoba {

constexpr int kFewWaves = 8;

// sum over the LPR consecutive lanes that share a key, in all of them
template <int LPR>
__device__ __forceinline__ float sum_lpr(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
#define FMOBA_ROR(N) x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x120 + N, 0xf, 0xf, true))
  if constexpr (LPR == 8) {
    // rotations work on 16 lanes: quads first, then the half-row mirror pairs the two quads of eight lanes
    x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0xb1, 0xf, 0xf, true));   // quad_perm 1 0 3 2
    x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x4e, 0xf, 0xf, true));   // quad_perm 2 3 0 1
    x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x141, 0xf, 0xf, true));  // row_half_mirror
  } else {
    FMOBA_ROR(8);
    FMOBA_ROR(4);
    FMOBA_ROR(2);
    FMOBA_ROR(1);
    if constexpr (LPR == 32) {
      const UPair p = swap16(__float_as_uint(x));
      x = __uint_as_float(p.a) + __uint_as_float(p.b);
    }
  }
#undef FMOBA_ROR
#endif
  return x;
}

// The best kp of a row's nc scores and behind them chunk `self` (the row's own; below 0: none), ascending in `chunks`; returns how many.
// One wave, a chunk per lane and place, a count is a ballot; the order is that of topk_gate_few_kernel (score descending, chunk
// descending; a candidate needs a score above -inf), so is the selection.  The places are registers for up to 64 NJ chunks, NJ = 0: `keys` in LDS
// (registers for 4096 chunks were 167 of them, and 72 scalars spilled, in every decode call).
template <int NJ>
__device__ __forceinline__ int pick_chunks(const float *scores, int64_t stride, int nc, int kp, int self, int lane, uint32_t *keys, int *chunks) {
  // in the order of the scores; 0: no candidate
  auto order = [&](int c, float x) { return c < nc && x + 0.f > -INFINITY ? float_order_key(x + 0.f) : 0u; };  // (-0 is +0)
  constexpr int GRP = NJ > 0 ? NJ : 8;  // places at a time
  const int ngrp = NJ > 0 ? 1 : (nc + GRP * 64 - 1) / (GRP * 64);
  uint32_t key[GRP];
  for (int g = 0; g < ngrp; ++g) {
    float x[GRP];
#pragma unroll
    for (int j = 0; j < GRP; ++j) {
      const int c = (g * GRP + j) * 64 + lane;
      x[j] = c < nc ? scores[(int64_t)c * stride] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < GRP; ++j) {
      key[j] = order((g * GRP + j) * 64 + lane, x[j]);
      if constexpr (NJ == 0) keys[(g * GRP + j) * 64 + lane] = key[j];
    }
  }
  auto place = [&](int g, int j) { return NJ > 0 ? key[j] : keys[(g * GRP + j) * 64 + lane]; };  // (its own lane wrote it)
  auto count_ge = [&](uint32_t v) {
    int n = 0;
    for (int g = 0; g < ngrp; ++g)
#pragma unroll
      for (int j = 0; j < GRP; ++j) n += __popcll(__ballot(place(g, j) >= v));
    return n;
  };
  // the largest cut with at least kp keys at or above it, or one with exactly kp (1: all of them, if there are no more)
  uint32_t cut = 1u;
  const int all = kp > 0 ? count_ge(1u) : 0;
  if (all > kp) {
    cut = 0u;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t trial = cut | (1u << bit);
      const int n = count_ge(trial);
      if (n >= kp) cut = trial;
      if (n == kp) break;
    }
  }
  int excess = all > kp ? count_ge(cut) - kp : 0;  // of the keys equal to the cut, the lowest chunks go
  int total = 0;
  for (int g = 0; g < (all > 0 ? ngrp : 0); ++g)
#pragma unroll
    for (int j = 0; j < GRP; ++j) {
      const uint32_t k = place(g, j);
      unsigned long long eq = __ballot(k == cut);
      const unsigned long long gt = __ballot(k > cut);
      while (excess > 0 && eq != 0ull) {
        eq &= eq - 1ull;
        --excess;
      }
      const unsigned long long m = gt | eq;
      if ((m >> lane) & 1ull) chunks[total + __popcll(m & ((1ull << lane) - 1ull))] = (g * GRP + j) * 64 + lane;
      total += __popcll(m);
    }
  if (self >= 0) {
    if (lane == 0) chunks[total] = self;
    ++total;
  }
  return total;
}

// SCORED: the row's chunks come from the scores that the pooling pass left (FewGate), else from the gate's selection bits.
template <typename T, int HD, bool SCORED>
__global__ __launch_bounds__(64 * kFewWaves, 2) void attn_fwd_few_kernel(fmoba_attn_fwd_args a, const uint32_t *bm, int nw, FewGate few) {
  constexpr int LPR = HD / 8, KPI = 64 / LPR;  // lanes per key, keys per load instruction
  constexpr int NIN = HD == 64 ? 8 : 16;       // load instructions per unit and operand
  constexpr int BK = NIN * KPI;                // keys per unit
  __shared__ int sChunk[SCORED ? 128 : kFewChunks];        // (top-k is at most 64)
  __shared__ uint32_t sKeys[SCORED ? kFewChunks : 1];
  __shared__ int sCount;
  __shared__ float sAcc[kFewWaves][HD], sM[kFewWaves], sL[kFewWaves];
  const int h = blockIdx.x, t = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the row's sequence: the sequences that end at or before it (empty ones included) come first
  int b = 0;
  for (int b0 = 0; b0 < a.batch; b0 += 64) b += __popcll(__ballot(b0 + lane < a.batch && a.cu_seqlens_q[b0 + lane + 1] <= t));
  if (b >= a.batch) return;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  const int D = a.head_dim, Bn = a.lg_block_n;
  const int hk = h / (a.heads / a.heads_k);
  const int kend = max(0, a.is_causal ? min(Lk, t - q0 + (Lk - Lq) + 1) : Lk);  // keys [0, kend) are visible
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;

  // ---- the chunks of the row ----
  if constexpr (SCORED) {
    if (wave == 0) {
      const int row = t - q0, rp = row + Lk - Lq;  // rp: the row's place among the keys
      const int own = few.is_causal && rp >= 0 ? rp / Bn : -1, self = row < few.rows && own < a.max_cols ? own : -1;
      const int nc = row >= few.rows ? 0 : min(few.is_causal ? max(own, 0) : (Lk + Bn - 1) / Bn, a.max_cols);
      const int kp = few.is_causal ? few.topk - 1 : few.topk;
      const int64_t stride = (int64_t)few.heads * few.rows;
      const float *sc = few.scores + ((int64_t)few.cu_seqlens_km[b] * few.heads + h) * few.rows + row;
      const int total = nc <= 256 ? pick_chunks<4>(sc, stride, nc, kp, self, lane, sKeys, sChunk) : pick_chunks<0>(sc, stride, nc, kp, self, lane, sKeys, sChunk);
      if (lane == 0) sCount = total;
    }
  } else if (wave == 0) {
    const int nwu = min(((kend + Bn - 1) / Bn + 31) >> 5, nw);
    int total = 0;
    for (int w0 = 0; w0 < nwu; w0 += 64) {
      uint32_t x = w0 + lane < nwu ? bm[((int64_t)h * nw + w0 + lane) * a.total_q + t] : 0u;
      int incl = __popc(x);
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(incl, o, 64);
        incl += lane >= o ? up : 0;
      }
      int at = total + incl - __popc(x);
      while (x) {
        const int c = (w0 + lane) * 32 + __ffs(x) - 1;
        sChunk[at++] = c;
        x &= x - 1;
      }
      total += __builtin_amdgcn_readlane(incl, 63);
    }
    if (lane == 0) sCount = total;
  }
  // this lane's features of the query row
  const int e = (lane % LPR) * 8;
  const int ec = min(e, D - 8);
  float q[8];
  {
    const Pack8 x = ld_global16(reinterpret_cast<const uint16_t *>(a.q) + (int64_t)t * a.q_row_stride + (int64_t)h * a.q_head_stride + ec);
    unpack8<T>(x, q);
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = e < D ? q[i] : 0.f;
  }
  const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)k0 * a.k_row_stride + (int64_t)hk * a.k_head_stride + ec;
  const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)k0 * a.v_row_stride + (int64_t)hk * a.v_head_stride + ec;
  __syncthreads();
  const int upc = Bn / BK, nunit = sCount * upc;

  float m = -INFINITY, l = 0.f, acc[8];  // l and acc: over this lane's keys (every KPI-th)
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  for (int u = wave; u < nunit; u += kFewWaves) {
    const int key0 = sChunk[u / upc] * Bn + (u % upc) * BK;
    if (key0 >= kend) continue;
    Pack8 kx[NIN], vx[NIN];
    const int kr = key0 + lane / LPR;
#pragma unroll
    for (int i = 0; i < NIN; ++i) kx[i] = ld_global16(kg + (int64_t)min(kr + i * KPI, Lk - 1) * a.k_row_stride);
#pragma unroll
    for (int i = 0; i < NIN; ++i) vx[i] = ld_global16(vg + (int64_t)min(kr + i * KPI, Lk - 1) * a.v_row_stride);
    float s[NIN], mu = -INFINITY;
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      float f[8];
      unpack8<T>(kx[i], f);
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) d = fmaf(q[j], f[j], d);
      d = sum_lpr<LPR>(d) * scale_log2;
      s[i] = kr + i * KPI < kend ? d : -INFINITY;
      mu = fmaxf(mu, s[i]);
    }
#pragma unroll
    for (int o = LPR; o < 64; o <<= 1) mu = fmaxf(mu, __shfl_xor(mu, o, 64));
    const float mn = fmaxf(m, mu), mref = mn == -INFINITY ? 0.f : mn;
    const float resc = __builtin_amdgcn_exp2f(m - mref);
    m = mn;
    l *= resc;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] *= resc;
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      const float p = __builtin_amdgcn_exp2f(s[i] - mref);
      float f[8];
      unpack8<T>(vx[i], f);
      l += p;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(p, f[j], acc[j]);
    }
  }
  // ---- the lanes' sums, then the waves' ----
#pragma unroll
  for (int o = LPR; o < 64; o <<= 1) {
    l += __shfl_xor(l, o, 64);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += __shfl_xor(acc[j], o, 64);
  }
  if (lane < LPR) {
#pragma unroll
    for (int j = 0; j < 8; ++j) sAcc[wave][e + j] = acc[j];
  }
  if (lane == 0) {
    sM[wave] = m;
    sL[wave] = l;
  }
  __syncthreads();
  if (tid >= HD) return;
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < kFewWaves; ++w) M = fmaxf(M, sM[w]);
  const float Mref = M == -INFINITY ? 0.f : M;
  float L = 0.f, o = 0.f;
#pragma unroll
  for (int w = 0; w < kFewWaves; ++w) {
    const float f = __builtin_amdgcn_exp2f(sM[w] - Mref);
    L = fmaf(f, sL[w], L);
    o = fmaf(f, sAcc[w][tid], o);
  }
  const bool empty = !(L > 0.f);
  if (tid < D)
    reinterpret_cast<uint16_t *>(a.out)[(int64_t)t * a.o_row_stride + (int64_t)h * a.o_head_stride + tid] = float_to_elem_bits<T>(empty ? 0.f : o / L);
  if (tid == 0) a.softmax_lse[(int64_t)h * a.total_q + t] = empty ? INFINITY : (M + __builtin_amdgcn_logf(L)) * 0.6931471805599453f;
}

// Where this form is the one to take.  It reads the chunks of every (row, head) anew, so it wants calls whose rows share
// little: at most eight query rows per sequence, and no more to read than the keys and values of the call are (twice, if
// a row's bound counts chunks it does not have).
bool fwd_few_rows(const fmoba_attn_fwd_args &a) {
  if (a.max_seqlen_q > kFewRows || a.max_cols > kFewChunks || a.max_cols < 1 || a.lg_block_n % 64 != 0 || a.total_q > 65535) return false;
  const int64_t unit = a.lg_block_n % 128 == 0 ? 128 : 64;
  const int64_t chunk_rows = (int64_t)a.max_visits_per_row * unit;  // keys a row may select
  const int64_t per_row = chunk_rows < a.max_seqlen_k ? chunk_rows : a.max_seqlen_k;
  return (int64_t)a.total_q * a.heads * per_row <= 4 * (int64_t)a.total_k * a.heads_k;
}

template <typename T, bool SCORED>
static void launch_few(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, const FewGate &few, hipStream_t s) {
  const dim3 grid(a.heads, a.total_q), block(64 * kFewWaves);
  if (a.head_dim <= 64)
    hipLaunchKernelGGL((attn_fwd_few_kernel<T, 64, SCORED>), grid, block, 0, s, a, bm, nw, few);
  else if (a.head_dim <= 128)
    hipLaunchKernelGGL((attn_fwd_few_kernel<T, 128, SCORED>), grid, block, 0, s, a, bm, nw, few);
  else
    hipLaunchKernelGGL((attn_fwd_few_kernel<T, 256, SCORED>), grid, block, 0, s, a, bm, nw, few);
}
void run_fwd_few(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, hipStream_t s) {
  if (a.dtype == FMOBA_DTYPE_BF16)
    launch_few<bf16_t, false>(a, bm, nw, FewGate{}, s);
  else
    launch_few<f16_t, false>(a, bm, nw, FewGate{}, s);
}
void run_fwd_few_scored(const fmoba_attn_fwd_args &a, const FewGate &few, hipStream_t s) {
  if (a.dtype == FMOBA_DTYPE_BF16)
    launch_few<bf16_t, true>(a, nullptr, 0, few, s);
  else
    launch_few<f16_t, true>(a, nullptr, 0, few, s);
}

}  // namespace fmoba
