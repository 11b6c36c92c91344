// The choice of a row's chunks from the scores of up to 32 NT of them, one lane pair per query row: what the gate (topk_csc.hip) and the row-block forward that does the
// gate's work itself (attn_fwd_rows.hip) have in common.
#pragma once

#include "fmoba_common.h"

namespace fmoba {

// n + (x0 > y) + (x1 > y) + (x2 > y) + (x3 > y): four compares into four scalar register pairs, then four adds with
// carry, so that no add follows its compare at once (a vector instruction that reads a scalar register written by the
// one before it has to wait; left alone, the compiler pairs every compare with its consumer and pads with idle slots)
__device__ __forceinline__ int count4_gt(int n, float x0, float x1, float x2, float x3, float y) {
#if defined(__HIP_DEVICE_COMPILE__)
  unsigned long long m0, m1, m2, m3;
  asm("v_cmp_gt_f32_e64 %1, %5, %9\n\t"
      "v_cmp_gt_f32_e64 %2, %6, %9\n\t"
      "v_cmp_gt_f32_e64 %3, %7, %9\n\t"
      "v_cmp_gt_f32_e64 %4, %8, %9\n\t"
      "v_addc_co_u32_e64 %0, vcc, 0, %0, %1\n\t"
      "v_addc_co_u32_e64 %0, vcc, 0, %0, %2\n\t"
      "v_addc_co_u32_e64 %0, vcc, 0, %0, %3\n\t"
      "v_addc_co_u32_e64 %0, vcc, 0, %0, %4"
      : "+v"(n), "=&s"(m0), "=&s"(m1), "=&s"(m2), "=&s"(m3)
      : "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(y)
      : "vcc");
  return n;
#else
  return n + (x0 > y) + (x1 > y) + (x2 > y) + (x3 > y);
#endif
}

// x >= y in two halves: four compares into four scalar register pairs first, then an add with carry per flag
// where it is needed (a vector instruction that reads a scalar register written by the one before it has to
// wait two slots: with the compares of four scores ahead of their adds nothing waits; left alone, the compiler
// materialises every flag as 0 / 1 first).  Volatile, so that the compares stay ahead of the adds.
struct Flags4 {
  unsigned long long m[4];
};
__device__ __forceinline__ Flags4 flags4_ge(float x0, float x1, float x2, float x3, float y) {
  Flags4 f;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_cmp_ge_f32_e64 %0, %4, %8\n\t"
               "v_cmp_ge_f32_e64 %1, %5, %8\n\t"
               "v_cmp_ge_f32_e64 %2, %6, %8\n\t"
               "v_cmp_ge_f32_e64 %3, %7, %8"
               : "=&s"(f.m[0]), "=&s"(f.m[1]), "=&s"(f.m[2]), "=&s"(f.m[3])
               : "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(y));
#else
  f.m[0] = x0 >= y;
  f.m[1] = x1 >= y;
  f.m[2] = x2 >= y;
  f.m[3] = x3 >= y;
#endif
  return f;
}
// the same with x > y
__device__ __forceinline__ Flags4 flags4_gt(float x0, float x1, float x2, float x3, float y) {
  Flags4 f;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_cmp_gt_f32_e64 %0, %4, %8\n\t"
               "v_cmp_gt_f32_e64 %1, %5, %8\n\t"
               "v_cmp_gt_f32_e64 %2, %6, %8\n\t"
               "v_cmp_gt_f32_e64 %3, %7, %8"
               : "=&s"(f.m[0]), "=&s"(f.m[1]), "=&s"(f.m[2]), "=&s"(f.m[3])
               : "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(y));
#else
  f.m[0] = x0 > y;
  f.m[1] = x1 > y;
  f.m[2] = x2 > y;
  f.m[3] = x3 > y;
#endif
  return f;
}
// (w << 1) | flag of the lane: one add with carry
__device__ __forceinline__ uint32_t shift_in_flag(uint32_t w, unsigned long long flag) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_addc_co_u32_e64 %0, vcc, %0, %0, %1" : "+v"(w) : "s"(flag) : "vcc");
  return w;
#else
  return (w << 1) | (uint32_t)(flag & 1);
#endif
}

// Up to this many winners a row's cut is found by taking its best scores off one by one (two and a half instructions per score and winner), beyond by bisection
// (about ten passes of two): both are bound by vector instructions.  Gate of 16 heads, bisection and this: 8192 tokens, 64 chunks, heads of 64 3 winners 14.3 -> 10.6 us, 8 14.2 -> 12.1,
// 10 14.1 -> 13.6, 12 14.7 -> 15.4, heads of 128 8 16.3 -> 13.9, 10 16.4 -> 15.0, 12 17.7 -> 18.1; 12800 tokens, 100 chunks, heads of 64 8 23.0 -> 19.9, 10 23.6 -> 21.5, 12 23.7 -> 23.9,
// heads of 128 8 28.6 -> 25.2, 10 30.7 -> 30.2, heads of 256 8 48.2 -> 43.9, 10 48.3 -> 45.3.
constexpr int kGatePeels = 10;
// The wave's 32 rows, lane (row l % 32): qf holds the row's slices as the B operand, the chunk means lie in the LDS tile from ldsTile on (rows of HD elements, piece c
// of row r at c ^ tile_swz<HD>(r)), n_tiles * 32 of them.  The row's candidates are the chunks [0, nc); it keeps the best kp and its own chunk (own; below 0: none).
// emit(t, w): word t of the row's selection, t < words, the same in both halves of the wave.
// PEEL: the best scores are taken off one by one, up to kGatePeels of them: the gate's own launch (an instance without serves more winners: with both searches it took 0.2 to 0.9 us of 13 to 35
// more), and the row-block forward where several sets of waves wait for the choice (1024 + 2048 tokens, 8 heads of 64, call 30.4 -> 28.6 us).  In the workgroups of one set, which overlap each
// other's choices, the second search of the cut only made the code longer (8191 tokens of short documents 123.6 -> 124.7 us).  One chain of comparisons: four side by side are no faster where
// a wave has its SIMD to itself (1024 + 2048 tokens, 8 heads of 64 24.4 us either way) and cost the gate's launch 12.1 -> 12.8 (64 chunks, heads of 64, 8 winners), 13.9 -> 14.8 (of 128).
template <typename T, int HD, int NT, bool PEEL, typename Emit>
__device__ __forceinline__ void gate_select(uint32_t ldsTile, const Pack8 (&qf)[HD / 16], int lane, int n_tiles, int nc, int kp, int own, bool valid, int words, const Emit &emit) {
  constexpr int KS = HD / 16, RB = HD * 2;
  const int hh = lane >> 5;
  // scores: lane (query l%32) gets chunk t*32 + acc_row(i, hh) in register i of tile t;
  // chunks that are not candidates of the row hold -inf
  float sc[NT][16];
  float vmin = INFINITY, vmax = -INFINITY;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (t < n_tiles) {
      f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const Pack8 af = lds_read16(ldsTile + (uint32_t)((t * 32 + (lane & 31)) * RB) + (uint32_t)(((hh * KS + ks) ^ tile_swz<HD>(lane & 31)) * 16));
        acc = mfma32<T>(af, qf[ks], acc);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int c = t * 32 + acc_row(i, hh);
        const bool cand = c < nc;
        const float x = acc[i];
        sc[t][i] = cand ? x : -INFINITY;
        vmin = fminf(vmin, cand ? x : INFINITY);
        vmax = fmaxf(vmax, sc[t][i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[t][i] = -INFINITY;
    }
  }
  vmin = min_xor32_f(vmin);
  vmax = max_xor32_f(vmax);

  // K' = number of scored chunks to keep (the own chunk takes one slot in causal mode).
  // A row keeps every candidate x with x > tau, plus, among the candidates equal to tau_eq,
  // those with chunk index >= iota.  tau is found below the K'-th of the best scores (PEEL), or by bisection between the row's smallest
  // and largest score and the search stops as soon as exactly K' scores lie above the probe.
  // The bracket is kept as order-preserving integer keys (lo_k, hi_k]; the first probes
  // bisect the VALUE range (few steps for ordinary score distributions), later ones the key
  // range (at most 32 more steps whatever the values).  If the bracket closes first, the
  // scores inside it are all equal and tie across the cut: the highest chunk indices win.
  const bool need = (nc > kp) && (kp > 0);
  float tau = -INFINITY;    // nc <= K': every candidate with a score above -inf
  float tau_eq = INFINITY;  // no tie group by default
  int n_eq = 0;
  uint32_t iota = 0u;
  uint32_t lo_k = float_order_key(vmin) - 1u;  // count(x > lo) = nc > K'
  uint32_t hi_k = float_order_key(vmax);       // count(x > hi) = 0  < K'
  int c_lo = nc, c_hi = 0;
  bool open = need;
  // A row whose bracket holds exactly one score too many, or one too few, needs no more probes: the cut lies right
  // below the largest score of the bracket, or right at its smallest.  When every open row of the wave is in that state
  // (about eight probes in, where the search of the slowest row takes twelve or thirteen), one pass over the scores
  // finds that score for all of them, the largest of -x for the rows that want the smallest.  The cut it gives is
  // exact unless the score occurs twice; such rows are found by their count below and searched to the end.
  bool guessed = false;
  auto bisect = [&](bool may_finish) {
    for (int iter = 0;; ++iter) {
      if (open && hi_k - lo_k <= 1u) {
        // nothing representable strictly inside: every score in (lo, hi] equals hi
        tau = order_key_float(hi_k);
        if (tau != -INFINITY) {
          tau_eq = tau;
          n_eq = kp - c_hi;
        }
        open = false;
      }
      if (!__any(open)) break;
      if (may_finish) {
        const bool up = kp - c_hi == 1, dn = c_lo - kp == 1;
        if (__all(!open || up || dn)) {
          const bool want_min = open && !up;
          const uint32_t flip = want_min ? 0x80000000u : 0u;
          // (x > lo for a score x is x >= the next float above lo, which after -0 is the smallest positive number)
          const uint32_t above_lo = lo_k + (lo_k == 0x7fffffffu ? 2u : 1u);
          const float bound = want_min ? -order_key_float(above_lo) : order_key_float(hi_k);
          float best = -INFINITY;
#pragma unroll
          for (int t = 0; t < NT; ++t)
            if (t < n_tiles) {
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const float y = __uint_as_float(__float_as_uint(sc[t][i]) ^ flip);
                best = fmaxf(best, y <= bound ? y : -INFINITY);
              }
            }
          best = max_xor32_f(best);
          if (open) {
            const float v = __uint_as_float(__float_as_uint(best) ^ flip);
            uint32_t below = float_order_key(v) - 1u;  // (the float below +0 that compares below it is not -0)
            if (below == 0x7fffffffu) below -= 1u;
            tau = up ? order_key_float(below) : v;
            guessed = true;
            open = false;
          }
          break;
        }
      }
      uint32_t pk = lo_k + ((hi_k - lo_k) >> 1);
      if (iter < 12) {
        const float mf = 0.5f * order_key_float(lo_k + 1u) + 0.5f * order_key_float(hi_k);
        const uint32_t mk = float_order_key(mf);
        if (mk > lo_k && mk < hi_k) pk = mk;
      }
      const float probe = order_key_float(pk);
      int cnt = 0;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < n_tiles) {
#pragma unroll
          for (int i = 0; i < 16; i += 4) cnt = count4_gt(cnt, sc[t][i], sc[t][i + 1], sc[t][i + 2], sc[t][i + 3], probe);
        }
      cnt = sum_xor32_i(cnt);
      if (open) {
        if (cnt == kp) {
          tau = probe;
          open = false;
        } else if (cnt > kp) {
          lo_k = pk;
          c_lo = cnt;
        } else {
          hi_k = pk;
          c_hi = cnt;
        }
      }
    }
  };
  if (PEEL && kp <= kGatePeels && __any(open && nc - kp > 1)) {
    // The largest score, the largest below it, .., kp of them: the cut lies right below the last.  Exact unless a score of those occurs twice, which
    // the count below shows.
    float last = INFINITY;
    for (int n = 0; n < kp; ++n) {
      float best = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < n_tiles) {
#pragma unroll
          for (int i = 0; i < 16; ++i) best = fmaxf(best, sc[t][i] < last ? sc[t][i] : -INFINITY);
        }
      last = max_xor32_f(best);
    }
    if (open) {
      uint32_t below = float_order_key(last) - 1u;  // (the float below +0 that compares below it is not -0)
      if (below == 0x7fffffffu) below -= 1u;
      tau = order_key_float(below);
      guessed = true;
      open = false;
    }
  } else {
    bisect(true);
  }
  bool any_tie = __any(n_eq > 0);  // some row of the wave has a tie across its cut
  // Without a tie in the wave a score is selected iff it lies above tau: the flags of the lane's 16 scores of a tile,
  // shifted in one by one (w + w + flag: one add with carry each), highest first.
  uint32_t bits[NT];
  auto flags_above_tau = [&]() {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bits[t] = 0u;
      if (t < n_tiles) {
#pragma unroll
        for (int i4 = 3; i4 >= 0; --i4) {
          const Flags4 f = flags4_gt(sc[t][4 * i4 + 3], sc[t][4 * i4 + 2], sc[t][4 * i4 + 1], sc[t][4 * i4], tau);
#pragma unroll
          for (int j = 0; j < 4; ++j) bits[t] = shift_in_flag(bits[t], f.m[j]);
        }
      }
    }
  };
  if (!any_tie) flags_above_tau();
  if (__any(guessed)) {
    int above = 0;
    if (!any_tie) {
#pragma unroll
      for (int t = 0; t < NT; ++t) above += __popc(bits[t]);
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < n_tiles) {
#pragma unroll
          for (int i = 0; i < 16; i += 4) above = count4_gt(above, sc[t][i], sc[t][i + 1], sc[t][i + 2], sc[t][i + 3], tau);
        }
    }
    above = sum_xor32_i(above);
    const bool again = guessed && above != kp;
    if (__any(again)) {
      open = again;
      bisect(false);
      any_tie = __any(n_eq > 0);
      if (!any_tie) flags_above_tau();
    }
  }
  // a tie group keeps its n_eq highest chunk indices
  if (any_tie) {
    const bool tie = n_eq > 0;
    int ceq = 0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t < n_tiles) {
#pragma unroll
        for (int i = 0; i < 16; ++i) ceq += (sc[t][i] == tau_eq) ? 1 : 0;
      }
    ceq = sum_xor32_i(ceq);
    const bool split = tie && ceq > n_eq;
    if (__any(split)) {
      uint32_t i_acc = 0u;
      constexpr int IB = (NT * 32 <= 64) ? 6 : (NT * 32 <= 128 ? 7 : 8);
      for (int bit = IB - 1; bit >= 0; --bit) {
        const uint32_t trial = i_acc | (1u << bit);
        // (Made anew in every turn: the flags of 128 and 256 scores, the same in all of them, were kept in scalar registers beside the loop, which took them
        // from the whole kernel: 79 and 223 scalars spilled, in a path that next to no row takes.  Gate of 32384 tokens, 16 heads, 256 chunks 138 -> 124 us for
        // heads of 64 and 152 -> 138 of 128, 128 chunks 80 -> 75.5.)
        float eq = tau_eq;
#if defined(__HIP_DEVICE_COMPILE__)
        if constexpr (NT > 2) asm volatile("" : "+v"(eq));
#endif
        int cnt = 0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (t < n_tiles) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const uint32_t c = (uint32_t)(t * 32 + acc_row(i, hh));
              cnt += ((sc[t][i] == eq) & (c >= trial)) ? 1 : 0;
            }
          }
        cnt = sum_xor32_i(cnt);
        if (cnt >= n_eq) i_acc = trial;
      }
      if (split) iota = i_acc;
    }
  }

  // selection words (32 chunks each), own chunk forced in causal mode
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (t < words) {
      uint32_t w = 0u;
      if (t < n_tiles && kp > 0) {
        if (!any_tie) {
          // the four nibbles of the flags move to the places of the lane's chunks (4 hh + 8 g .. + 3)
          const uint32_t b = bits[t];
          w = ((b & 0xfu) | ((b & 0xf0u) << 4) | ((b & 0xf00u) << 8) | ((b & 0xf000u) << 12)) << (4 * hh);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const uint32_t c = (uint32_t)(t * 32 + acc_row(i, hh));
            const float x = sc[t][i];
            const bool s = (x > tau) | ((x == tau_eq) & (c >= iota));
            w |= s ? (1u << ((8 * (i >> 2) + (i & 3)) + 4 * hh)) : 0u;
          }
        }
      }
      {
        const UPair wp = swap32(w);
        w = wp.a | wp.b;
      }
      if (own >= 0 && (own >> 5) == t) w |= 1u << (own & 31);
      if (!valid) w = 0u;
      emit(t, w);
    }
  }
}

// The gate of a row block, by the workgroup that is about to walk its keys (SPLIT sets of RW waves of 32 rows each; the first set chooses): candidates of some
// row of the block, their means into LDS, scores, choice, as topk_gate_kernel does it.  Q is asked for and not awaited when it begins, arranged when it ends.
// The rows' words go to sBits (word w of row r at w * 32 RW + r), and if column lists follow to memory with their counts, by way of sHist (kRowGateChunks words).
// km0, Cb: the sequence's first mean and how many it has.  Takes row_gate_lds bytes of `smem`, which are free when it ends.
template <int HD>
constexpr size_t row_gate_lds() { return (size_t)kRowGateChunks * HD * 2; }
template <typename T, int HD, int RW, int SPLIT>
__device__ __forceinline__ void gate_row_block(const fmoba_attn_fwd_args &a, const RowGate &gate, uint8_t *smem, uint32_t *sBits, int *sHist, Pack8 (&qb)[HD / 16], int b, int h, int hk,
                                               int q0, int r0, int rlast, int Lq, int off, int nw, int km0, int Cb) {
  constexpr int NT = kRowGateChunks / 32, VPR = HD / 8, RPI = 64 / VPR, NTHR = SPLIT * RW * 64, KS = HD / 16;
  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5, wave = wave_all % RW, set = wave_all / RW;
  const int Bn = a.lg_block_n, D = a.head_dim, row = r0 + wave * 32 + (lane & 31);
  const bool causal = a.is_causal != 0, valid = row < Lq;
  const int rmax = rlast + off;
  const int nsc = min(causal ? (rmax < 0 ? 0 : min(Cb, rmax / Bn)) : Cb, min(a.max_cols, kRowGateChunks));
  const int n_tiles = (nsc + 31) >> 5;
  const uint32_t ldsTile = (uint32_t)(uintptr_t)smem;
  const uint16_t *kmp = gate.km + (int64_t)hk * gate.km_head_stride;
  for (int v = wave_all; v < n_tiles * 32 / RPI; v += SPLIT * RW) {
    const int c = v * RPI + lane / VPR, pc = lane % VPR;
    const int e = min((pc ^ tile_swz<HD>(c)) * 8, D - 8);
    global_to_lds16(kmp + (int64_t)(km0 + min(c, nsc - 1)) * gate.km_row_stride + e, ldsTile + (uint32_t)v * 1024u);
  }
  for (int v = tid; v < NT * 32; v += NTHR) sHist[v] = 0;
  wait_all_loads();
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qb[ks].w[0]), "+v"(qb[ks].w[1]), "+v"(qb[ks].w[2]), "+v"(qb[ks].w[3]));
#endif
  __syncthreads();
  q_rows_arrange<HD>(qb, hh, D);
  if (set == 0) {
    const int rp = row + off, own = causal && valid && rp >= 0 ? rp / Bn : -1;
    const int nc = min(causal ? min(max(own, 0), Cb) : valid ? Cb : 0, nsc);
    uint32_t *selp = gate.sel + (int64_t)h * gate.W * a.total_q + q0 + row;
    gate_select<T, HD, NT, (SPLIT > 1)>(ldsTile, qb, lane, n_tiles, nc, causal ? gate.topk - 1 : gate.topk, own, valid, nw, [&](int t, uint32_t w) {
      if (hh == 0) sBits[t * 32 * RW + wave * 32 + lane] = w;
      if (gate.sel != nullptr) {
        if (valid && hh == 0) selp[(int64_t)t * a.total_q] = w;
        if (__any(w != 0u)) {
          const int mycnt = bit_column_count32(w, lane);
          if (lane < 32 && mycnt) atomicAdd(&sHist[t * 32 + lane], mycnt);
        }
      }
    });
  }
  __syncthreads();
  if (gate.sel != nullptr) {
    for (int c = tid; c < nw * 32 && c < a.max_cols; c += NTHR) {
      const int v = sHist[c];
      if (v) atomicAdd(&gate.segcnt[(((int64_t)b * a.heads + h) * gate.nseg + r0 / gate.seg_rows) * a.max_cols + c], v);
    }
  }
}

}  // namespace fmoba
