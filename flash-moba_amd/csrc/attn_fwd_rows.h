// What the row-block kernels of the forward (attn_fwd_rows.hip, attn_fwd_rows_wide.hip) have in common: the layout of a workgroup's LDS
// and the list of its steps.
#pragma once

#include "fmoba_common.h"

namespace fmoba {

constexpr int kRowsStepCap = 4096;  // 64-key steps of one row block (its step list lives in LDS)
constexpr int kRowsWordCap = 128;   // bitmap words per row (32 chunks each)
constexpr int kRowsWords = 16;  // selection words per row that the workgroup keeps in LDS (512 chunks)

template <int HD, int RW, int SPLIT>
struct FwdRowsDirectSmem {
  static constexpr int ROWS = 32 * RW;  // rows of a workgroup: 32 for each wave of a set
  static constexpr int LDO = HD + 8;   // elements, per-wave output tile [32 rows][LDO]
  static constexpr size_t tile = (size_t)64 * HD * 2;       // one 64-key tile of K or V
  static constexpr size_t ring = 4 * tile;                    // K, K, V, V: the rings of one set of waves
  static constexpr size_t oStep = SPLIT * ring;               // int[step_cap]: key block | chunk << 16
  static constexpr int UPW = ROWS / 64;                       // unions of 64 rows' selection words per word
  // behind the steps, sized by the call: uint32[nw][UPW] unions, uint32[nw][ROWS] the rows' selection words, int[kRowGateChunks] counts of those that choose their chunks
  static size_t bytes(int step_cap, int nw) { return oStep + ((size_t)step_cap + (size_t)nw * (UPW + ROWS) + kRowGateChunks) * 4; }
  static_assert((size_t)RW * 32 * LDO * 2 <= ring && (size_t)RW * HD * 128 <= ring, "output tiles must fit the K/V rings");
};

// IN_LDS: the rows' words are in sBits already, visible to every thread.
// The steps of a row block: the selection words of its rows go to sBits (word w of row r at w * ROWS + r), the 64-key blocks of every chunk that
// a row of it selected to sStep in ascending order (key block | chunk << 16).  `words` points to word 0 of the block's first row, `stride`
// words lie between two words of a row, `nrow` rows exist, keys [0, kend) are visible to some row.  Returns the number of steps, of which at most step_cap are listed.
// Every thread of the workgroup takes part; ends with the lists visible to all of them.
template <int ROWS, int NTHR, bool IN_LDS = false>
__device__ __forceinline__ int row_block_steps(const uint32_t *words, int64_t stride, int nrow, int kend, int Bn, int nw, int step_cap, int *sStep,
                                               uint32_t *sUnion, uint32_t *sBits) {
  constexpr int UPW = ROWS / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), sub = Bn >> 6;
  const int nchunk = kend > 0 ? (kend + Bn - 1) / Bn : 0;
  const int nwu = min((nchunk + 31) >> 5, nw);
  // (the words stay in LDS for the walk: a load from global memory inside the step loop would make the compiler
  // wait for every outstanding load of the wave, the tile loads included, at every step)
  for (int it = wave; it < nwu * UPW; it += NTHR / 64) {  // one word of 64 rows per wave
    const int w = it / UPW, rw = (it % UPW) * 64 + lane;
    uint32_t x;
    if constexpr (IN_LDS) {
      x = sBits[w * ROWS + rw];
    } else {
      x = rw < nrow ? words[w * stride + rw] : 0u;
      sBits[w * ROWS + rw] = x;
    }
    const uint32_t u = or_wave(x);
    if (lane == 0) sUnion[it] = u;
  }
  __syncthreads();
  // One thread per chunk: a chunk of the union contributes its 64-key blocks that hold a visible key.  All but the last visible
  // chunk have all of theirs, so a chunk's first step is the number of chunks of the union before it times the blocks of one: no
  // scan over the workgroup, and no atomics for the unions (1024 tokens, 8 heads of 64: 14.7 -> 14.3 us).
  const int nchunk_u = min(nchunk, nwu * 32);
  int nstep_all = 0;
  if (nchunk_u > 0) {
    auto word = [&](int w) {
      uint32_t u = sUnion[w * UPW];
      if constexpr (UPW == 2) u |= sUnion[w * 2 + 1];
      return u;
    };
    for (int c = tid; c < nchunk_u; c += NTHR) {
      int before = 0;
      for (int w = 0; w < (c >> 5); ++w) before += __popc(word(w));
      const uint32_t u = word(c >> 5);
      if ((u >> (c & 31)) & 1u) {
        int pos = (before + __popc(u & ((1u << (c & 31)) - 1u))) * sub;
        const int cnt = min(sub, (kend - c * Bn + 63) >> 6);
        for (int jb = 0; jb < cnt; ++jb, ++pos)
          if (pos < step_cap) sStep[pos] = (c * sub + jb) | (c << 16);
      }
    }
    const int last = nchunk_u - 1;
    const uint32_t ul = word(last >> 5) & (0xffffffffu >> (31 - (last & 31)));
    int nsel = __popc(ul);
    for (int w = 0; w < (last >> 5); ++w) nsel += __popc(word(w));
    nstep_all = nsel * sub - (((ul >> (last & 31)) & 1u) ? sub - min(sub, (kend - last * Bn + 63) >> 6) : 0);
    nstep_all = __builtin_amdgcn_readfirstlane(nstep_all);
  }
  __syncthreads();
  return nstep_all;
}

// The same steps where the rows' words are in sBits and the chunks no more than kRowGateChunks, by every wave for itself: all write the same list and none waits for
// another (two barriers and the LDS reads behind them were 1800 clocks in front of a workgroup's first loads, 700 are left).  Ends with the list visible to the wave.
template <int ROWS>
__device__ __forceinline__ int gated_row_block_steps(int kend, int Bn, int nw, int step_cap, int *sStep, const uint32_t *sBits) {
  static_assert(kRowGateChunks == 64, "a chunk per lane");
  const int lane = threadIdx.x & 63, sub = Bn >> 6;
  const int nchunk = kend > 0 ? min((kend + Bn - 1) / Bn, nw * 32) : 0;
  uint32_t x[2] = {0u, 0u};
#pragma unroll
  for (int w = 0; w < 2; ++w)
    if (w < nw) {
#pragma unroll
      for (int r = 0; r < ROWS; r += 64) x[w] |= sBits[w * ROWS + r + lane];
    }
  const uint32_t lo = __builtin_amdgcn_readfirstlane(or_wave(x[0])), hi = __builtin_amdgcn_readfirstlane(or_wave(x[1]));
  unsigned long long u = ((unsigned long long)hi << 32) | lo;
  if (nchunk < 64) u &= (1ull << nchunk) - 1ull;
  if ((u >> lane) & 1ull) {
    int pos = (int)__popcll(u & ((1ull << lane) - 1ull)) * sub;
    const int cnt = min(sub, (kend - lane * Bn + 63) >> 6);
    for (int jb = 0; jb < cnt; ++jb, ++pos)
      if (pos < step_cap) sStep[pos] = (lane * sub + jb) | (lane << 16);
  }
  wave_lds_fence();
  const int last = nchunk - 1;
  return u == 0ull ? 0 : (int)__popcll(u) * sub - (((u >> last) & 1ull) ? sub - min(sub, (kend - last * Bn + 63) >> 6) : 0);
}

}  // namespace fmoba
