// Sparse attention forward over a CSC pattern: the entry points, and the column-stationary form in two
// launches (sparse patterns; the row-block form for dense ones is in attn_fwd_rows.hip).
//
//   attn_fwd_col_kernel     : one workgroup per (key block of KB = 64 or 128 keys, KEY head,
//                             sequence).  K and V of the block lie in LDS; the ascending row lists
//                             of the query heads that share the key head are walked in gathered
//                             32-row tiles, each wave taking tiles of its own:
//                             S^T = K Q^T (one lane owns one query row, so the softmax
//                             reductions over the block's keys stay in registers), P^T goes from
//                             the accumulators straight into the operand registers of
//                             O^T = V^T P^T (V^T through transposing LDS reads).  Every visit of
//                             a (row, key block) pair leaves a PARTIAL result: the block-local
//                             maximum m, the sum l of exp2(s - m) and the output row (bf16 or fp32:
//                             unnormalised; fp16: divided by l).  Over ranked lists (the gated path)
//                             its slot is that of the key block among the row's, made of the list
//                             entry's rank; over plain lists the row hands it out from a counter.
//   attn_fwd_combine_kernel : sixteen lanes per (row, head) merge the row's partials in ascending
//                             key-block order: that of the slots over ranked lists, else found by
//                             sorting the block ids, so the result does not depend on which slot a
//                             visit happened to get.  Out, log-sum-exp.
//
// Work and traffic are proportional to the number of (row, key block) visits whatever the number of
// chunks per sequence; a row-stationary formulation degenerates when every 128-row block touches
// thousands of chunks with one or two rows each.
#include "fmoba_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace fmoba {

// row-block form when a row selects at least 10/50 (64-key blocks) resp. 10/27 (128-key blocks) of the chunks it may see:
// break-even points measured at 8192 to 32768 tokens (columns against rows: 64-key blocks, 32768 tokens 0.20 of the chunks 4128
// against 4200 us; 128-key blocks, 4 x 4096 tokens 0.31 250 against 291, 0.44 312 against 295).  With grouped heads the
// columns are level with 128-key blocks only at 0.45 (16384 tokens, 16 over 4 heads, 0.30 719 against 1051 us, 0.45 1041 against 1073); the
// line stays at 10/27 for them too, as rows that the row-block form adds up in fp32 are not moved to 16-bit partial rows
// (8192 tokens, 0.41 of the chunks: error of the output against 64 bits 2.17e-3 in row blocks, 2.63e-3 in columns).
constexpr int kFwdRowsDensity64 = 50, kFwdRowsDensity128 = 27;
// The same above head dimension 128 (fp32 partial rows in the column form; whole prefill, 8 heads of 256, columns against rows): 64-key blocks,
// 2 x 4096 tokens 0.12 of the chunks 170 against 178 us, 0.24 249 against 181, 16384 tokens 0.12 897 against 1168, 0.25 1691 against 1220; 128-key
// blocks, 2 x 4096 tokens 0.24 176 against 188, 0.48 252 against 190, 8 x 2048 tokens 0.38 481 against 451, 16384 tokens 0.25 874 against 1169, 0.5 1552
// against 1200.  From one 128-row block per compute unit on: fewer of them leave units idle for the length of a walk.
constexpr int kFwdRowsDensityWide64 = 57, kFwdRowsDensityWide128 = 28, kFwdRowsWideBlocks = 256;
// Partial results of wide heads that a call may ask for, counted without the padding of part_row_elems (up to 6 % more is allocated), as the line lay
// before rows were padded: no call changes its form by it.
constexpr int64_t kWidePartialBytes = (int64_t)16 << 30;

struct FwdWs {
  int32_t *cnt;      // [total_q * heads] visits handed out per (row, head)
  float4 *hdr;       // [total_q * heads * cap] {m (log2 domain), l, key block id, -}; ranked: float2 {m, l}
  void *part;        // [total_q * heads * cap][part_row_elems] partial outputs (fwd_part_size bytes per element)
  int32_t cap;
  const uint32_t *visits;  // per (head, row), with ranked lists: the form whose slots are in key-block order (null: the other one)
};

// Bytes per element of a partial row: the 16-bit type of the call, fp32 at head dimensions above 128.  There this form serves
// dense patterns too, whose rows the row-block form adds up in fp32 from end to end, and the two agree in precision.
constexpr size_t fwd_part_size(int head_dim) { return head_dim > 128 ? 4 : 2; }

// fp16 partial rows are divided by their sum of probabilities first: as they leave the products they are up to 64 or 128 times
// the values, beyond the range of the type from values of about 500 on.
// (8192 tokens, heads of 128, top-k 8 of 128-key chunks: error of the output against 64 bits 3.33e-4 -> 3.16e-4, 175 us with and
// without; 32768 tokens, 32 heads, top-k 16 3040 -> 3054 us, the runs of one side differ by 16.)
template <typename T, int HD>
constexpr bool kFwdNormalisedParts = std::is_same_v<T, f16_t> && fwd_part_size(HD) == 2;

template <int HD, int KB>
struct FwdColSmem {
  static constexpr size_t tile = (size_t)KB * HD * 2;  // K or V of the block: rows of exactly HD elements, swizzled
  static constexpr size_t oOut = 2 * tile;             // [NW waves][32 rows][128 bytes]: a part of a tile's partial rows on its way out
  // Two workgroups of four waves per compute unit; 128 keys of 256 features fill the unit's LDS: one workgroup of eight.
  static constexpr int NW = 2 * (oOut + 4 * 4096) <= 160 * 1024 ? 4 : 8;
  static constexpr size_t bytes = oOut + NW * 4096;
  static_assert(bytes * (8 / NW) <= 160 * 1024, "eight waves per compute unit");
};

// The blocks that exist alone, by length or by pairs (one pair at a time is for sequences far beyond these).  Pair by pair only where they are at most half:
// the look-up is one more load in front of the lists' bounds (parts of prompts against 9216, 33000 and 20000 keys, 0.63 of the blocks 241.5 -> 243.3 us; six of
// 300 rows against 3000 to 60000, 0.4 202.9 -> 195.2).
static ItemOrder col_order(const fmoba_attn_fwd_args &a, int ngrp, int hd, int kb) {
  const bool longest_first = longest_items_first(std::max(a.total_q, a.total_k), a.heads, hd * 2);
  const bool listed = lists_blocks(a.total_k, a.max_seqlen_k, a.batch, ngrp, kb, true) && (int64_t)a.max_seqlen_q * hd * 4 < kOnePairBytes;
  if (listed && longest_first) return kListedLongestFirst;
  if (listed && (int64_t)a.batch * ceil_div(a.max_seqlen_k, kb) >= 2 * listed_blocks(a.total_k, a.batch, kb)) return kListedPairs;
  return longest_first ? kLongestFirst : kPairOrder;
}

// Two workgroups per compute unit, two waves per SIMD, no barrier after the block's K and V have arrived.  What bounds it
// depends on the lists.  Long ones (32768 tokens, 32 heads, top-k 16 of 256 chunks: 2000 rows per list): the partial
// results on their way out and the gathered Q rows, together about 4 TB/s.  Short ones (a part of a prompt against the
// keys so far, 1000 query rows: 28 rows per list): the three dependent loads before a workgroup's first product, hence
// small workgroups that share a unit and serve all heads of a group.  The kernel this one replaces had one workgroup of
// 512-register waves per unit and head and walked 128 rows between barriers: on those two shapes 2.32 -> 2.17 ms and
// 530 -> 162 us, 8192 tokens with top-k 8 148 -> 132 us, 262144 tokens 9.99 -> 9.12 ms, and one row per sequence against
// 16 sequences of up to 32768 keys 651 -> 113 us.  Since then, with the Q rows in runs of 64 bytes, the row ids ahead of the block and
// no registers spilled: 2.08 -> 1.94 ms, 164 -> 154 us, 114 -> 109 us, 9.35 -> 8.53 ms, and 2 x 4096 tokens, 8 heads of 256, 175 -> 158 us.
// Head dimensions above 128: an fp32 partial row per 128 keys is as many bytes as a 16-bit one per 64, and 128 keys are what one
// workgroup of eight waves finds room for (2 x 4096 tokens, 8 heads of 256, top-k 8 of 128-key chunks, forward: 16-bit rows
// per 64 keys 273 us, fp32 rows per 64 keys 450, per 128 keys 269).  Chunks that 128 does not divide pay for the wider rows:
// top-k 16 of 64-key chunks 259 -> 439 us.
// FULL: the head dimension is HD.  RANKED: a visit's slot is the place of its key block among the row's, made of the list entry's rank;
// otherwise the row hands out slots from a counter.  The counters (a returning atomic on a line of its own per visit) and the ids
// that the combine then needs to find the order are a tenth of the kernel (32 heads, top-k 16 of 128-key chunks, 32768 tokens: 1950 -> 1766 us,
// 16 heads, 262144 tokens: 8.55 -> 7.43 ms), and the launch that clears them 5.5 us.
template <typename T, int HD, int KB, bool FULL, bool RANKED>
__global__ __launch_bounds__((64 * FwdColSmem<HD, KB>::NW), 2) void attn_fwd_col_kernel(fmoba_attn_fwd_args a, FwdWs ws, int grp, ItemOrder order) {
  typedef FwdColSmem<HD, KB> SM;
  constexpr int KS = HD / 16, NDT = HD / 32, VPR = HD / 8, KT = KB / 32, RB = HD * 2, NW = SM::NW;
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  const bool one_pair = (int64_t)a.max_seqlen_q * HD * 4 >= kOnePairBytes;
  const int ngrp = a.heads / grp;
  int nb, b, h0;
  if (order >= kListedLongestFirst) {
    const BlockItem item = order == kListedPairs ? listed_pair_item<KB>(blockIdx.x, a.batch, ngrp, a.max_seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k)
                                                 : listed_item<KB, false>(blockIdx.x, a.batch, ngrp, a.max_seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    nb = item.idx, b = item.b, h0 = item.h * grp;
  } else {
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * ngrp, (a.max_seqlen_k + KB - 1) / KB, one_pair, order == kLongestFirst);
    nb = item.idx, b = item.pair / ngrp, h0 = (item.pair - b * ngrp) * grp;
  }
  const int hk = h0 / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  const int key0 = nb * KB;
  const int c = key0 / a.lg_block_n;
  // lane j: the list of head h0 + j (at most 64 of them: fwd_col_heads), asked for together with the sequence's bounds: neither needs
  // the other
  int nnz = 0;
  int64_t lbase = 0;
  if (c < a.max_cols && lane < grp) {
    const int64_t ci = ((int64_t)b * a.heads + h0 + lane) * a.max_cols + c;
    nnz = a.col_nnz[ci];
    lbase = a.col_offsets[ci];
  }
  const int k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  if (key0 >= Lk || c >= a.max_cols) return;
  const int off = Lk - Lq;
  const int D = FULL ? HD : a.head_dim;
  const bool causal = a.is_causal != 0;
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;
  const uint32_t ldsK = (uint32_t)(uintptr_t)smem, ldsV = ldsK + (uint32_t)SM::tile, ldsOut = ldsK + (uint32_t)(SM::oOut + wave * 4096);

  // k-step ks takes piece 4 (ks / 2) + ks % 2 + 2 hh of a row (the order in which Q arrives, see fetch)
  const uint32_t rowoff = (uint32_t)((lane & 31) * RB + (((2 * hh) ^ tile_swz<HD>(lane & 31)) * 16));
  const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
  const uint32_t troff = (uint32_t)(r0t * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
  int incl = (nnz + 31) >> 5;  // tiles of the lists up to this one
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(incl, o, 64);
    incl += lane >= o ? up : 0;
  }
  const int ntile = __builtin_amdgcn_readlane(incl, 63);
  if (ntile == 0) return;
  // The wave's tiles: tile t + 2 NW is picked (its row ids are asked for) and the rows of tile t + NW are fetched while tile t
  // is worked on, and all of these loads are awaited at one place, before the stores of tile t: one counter covers
  // loads and stores alike, and a load issued after the stores would be waited for together with them.
  int g = 0, rem = 0, ridn = 0;
  Pack8 qb[KS];
  int slot = 0;
  const int sub = a.lg_block_n / KB, jb = (key0 - c * a.lg_block_n) / KB;  // key blocks of a column, this one's number
  // (no branch around the loads: where two paths join, the compiler copies what was loaded, and waits for it there)
  auto pick = [&](auto to_lds, int t) {
    t = min(t, ntile - 1);
    g = __popcll(__ballot(incl <= t));
    const int first = t - (g ? __builtin_amdgcn_readlane(incl, g - 1) : 0);
    const int n = __builtin_amdgcn_readlane(nnz, g);
    const uint32_t blo = __builtin_amdgcn_readlane((uint32_t)lbase, g), bhi = __builtin_amdgcn_readlane((uint32_t)(lbase >> 32), g);
    const int64_t at = (int64_t)(((uint64_t)bhi << 32) | blo) + first * 32;
    rem = n - first * 32;
    const int32_t *p = a.row_indices + at + min(lane & 31, rem - 1);
    if constexpr (decltype(to_lds)::value)
      global_to_lds4(p, ldsOut);
    else
      ridn = *p;
  };
  int rid = -1, hcur = 0;
  auto fetch = [&](int t) {  // Q rows and partial slots of the picked tile
    rid = tile_row_code(RANKED ? ridn & kListRowMask : ridn, (lane & 31) < rem, Lq);
    hcur = h0 + g;
    // Four lanes fetch 64 bytes of a row together: load 2 j brings pieces 4 j .. 4 j + 3 of the tile's first sixteen rows, load 2 j + 1 those
    // of the other sixteen, and an exchange of 16-lane rows then gives every lane pieces of its own row.  (A lane that fetched its own
    // row's pieces touched a line of its own in every load, 64 lines a load where it is sixteen now: 32768 tokens, 32 heads, top-k 16
    // 2089 -> 1924 us, 262144 tokens 9200 -> 8561.)
    const UPair rr = swap16((uint32_t)rid & 0x7fffffffu);
    const uint16_t *qh = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)hcur * a.q_head_stride;
    const uint16_t *qa = qh + (uint64_t)rr.a * (uint32_t)a.q_row_stride, *qo = qh + (uint64_t)rr.b * (uint32_t)a.q_row_stride;
#pragma unroll
    for (int j = 0; j < KS / 2; ++j) {
      const int e = min((4 * j + (lane >> 4)) * 8, D - 8);  // (features past D: zeroed in arrived())
      qb[2 * j] = ld_global16(qa + e);
      qb[2 * j + 1] = ld_global16(qo + e);
    }
    if constexpr (RANKED)
      slot = (ridn >> kListRowBits) * sub + jb;
    else
      slot = take_slot(ws.cnt + ((int64_t)(q0 + (rid & 0x7fffffff)) * a.heads + hcur), rid >= 0 && hh == 0 && t < ntile);
  };
  auto arrived = [&]() {
    wait_all_loads();
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qb[ks].w[0]), "+v"(qb[ks].w[1]), "+v"(qb[ks].w[2]), "+v"(qb[ks].w[3]));
    asm volatile("" : "+v"(slot), "+v"(ridn));
#pragma unroll
    for (int j = 0; j < KS / 2; ++j)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        auto x = __builtin_amdgcn_permlane16_swap(qb[2 * j].w[w], qb[2 * j + 1].w[w], false, false);
        qb[2 * j].w[w] = x[0];
        qb[2 * j + 1].w[w] = x[1];
      }
#endif
    if (D < HD) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int w = 0; w < 4; ++w) qb[ks].w[w] = (4 * (ks >> 1) + (ks & 1) + 2 * hh) * 8 < D ? qb[ks].w[w] : 0u;
    }
  };
  // The row ids of the first tile before the block's K and V, and waited for without them: the counter of a wave's loads counts in
  // order, and the Q rows are the longest chain of a workgroup with few tiles (column bounds, row ids, rows: parts of prompts of 1024 rows
  // against 9000 to 33000 keys 160 -> 154 us).  They come by way of the wave's part of LDS for the partial rows.
  pick(std::true_type{}, wave);
  constexpr int RPI = 64 / VPR, NI = KB / RPI / NW;
  {
    const int rl = lane / VPR, pc = lane % VPR;
    const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)(k0 + key0) * a.k_row_stride + (int64_t)hk * a.k_head_stride;
    const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)(k0 + key0) * a.v_row_stride + (int64_t)hk * a.v_head_stride;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int key = (wave * NI + i) * RPI + rl;
      const int e = min((pc ^ tile_swz<HD>(key)) * 8, D - 8);
      const int64_t kc = min(key, Lk - 1 - key0);
      global_to_lds16(kg + kc * a.k_row_stride + e, ldsK + (uint32_t)((wave * NI + i) * 1024));
      global_to_lds16(vg + kc * a.v_row_stride + e, ldsV + (uint32_t)((wave * NI + i) * 1024));
    }
  }
  wait_loads_but<2 * NI>();
  ridn = lds_read_vec<int>(ldsOut + (uint32_t)(lane * 4));
  fetch(wave);
  pick(std::false_type{}, wave + NW);
  arrived();
  __syncthreads();
  for (int t = wave; t < ntile; t += NW) {
    const int r = rid, h = hcur;
    const int s0 = RANKED ? slot : __shfl(slot, lane & 31, 64);
    const int pidx = (r >= 0 && s0 < ws.cap) ? ((q0 + r) * a.heads + h) * ws.cap + s0 : -1;
    // keys beyond lim are masked
    const int lim = r < 0 ? -1 : min(causal ? r + off : 0x7fffffff, Lk - 1) - key0;
    f32x16 st[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) st[kt][i] = 0.f;
    uint32_t ak = ldsK + rowoff;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(ak));
#endif
    // (the K operands of a k-step are read while the step before it is on the matrix cores; the fences keep the compiler
    // from moving every read next to its product)
    Pack8 kf[2][KT];
    auto k_read = [&](auto kc) {
      constexpr int ks = decltype(kc)::value;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) kf[ks & 1][kt] = lds_read16((ak ^ (uint32_t)((4 * (ks >> 1) + (ks & 1)) * 16)) + (uint32_t)(kt * 32 * RB));
    };
    k_read(std::integral_constant<int, 0>{});
    static_for<KS>([&](auto kc) {
      constexpr int ks = decltype(kc)::value;
      if constexpr (ks + 1 < KS) k_read(std::integral_constant<int, ks + 1>{});
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) st[kt] = mfma32<T>(kf[ks & 1][kt], qb[ks], st[kt]);
      __builtin_amdgcn_sched_barrier(0);
    });
    fetch(t + NW);
    pick(std::false_type{}, t + 2 * NW);
    if (!__all(lim >= KB - 1)) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int jrel = kt * 32 + 8 * (i >> 2) + (i & 3) + 4 * hh;
          st[kt][i] = jrel <= lim ? st[kt][i] : -INFINITY;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) m = fmaxf(m, st[kt][i]);
    m = max_xor32_f(m) * scale_log2;
    const float m_use = m == -INFINITY ? 0.f : m;
    float l = 0.f;
    Pack8 pf[KT][2];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(st[kt][8 * s2 + 2 * w], scale_log2, -m_use));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(st[kt][8 * s2 + 2 * w + 1], scale_log2, -m_use));
          l += p0 + p1;
          pf[kt][s2].w[w] = pack2<T>(p0, p1);
        }
    l = sum_xor32_f(l);
    constexpr bool NORM = kFwdNormalisedParts<T, HD>;
    const float inv = NORM && l > 0.f ? 1.f / l : 0.f;
    constexpr bool F32 = fwd_part_size(HD) == 4;
    // a tile's partial rows, 128 bytes of every row at a time: 64 features in 16 bits, 32 features in fp32
    constexpr int HELD = F32 ? NDT / KT : NDT;  // feature tiles that are kept until the next tile's loads are in
    Pack8 x[F32 ? HELD : NDT / 2][4];
    uint32_t tv = ldsV + troff;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(tv));
#endif
    // V^T operands: those of the next KT products are read while KT products run
    Pack8 vt[2][KT];
    auto v_read = [&](auto hc) {  // half hc & 1 of feature tile hc / 2
      constexpr int hb = decltype(hc)::value, dt = hb >> 1;
      const uint32_t xlo = (uint32_t)(dt * 4 * 16), xhi = (uint32_t)(((dt * 4) ^ TileSwz<HD>::kRow8) * 16);
#pragma unroll
      for (int u = 0; u < KT; ++u) {
        const int q = (hb & 1) * KT + u;  // key tile q / 2, half q & 1
        const uint32_t olo = (uint32_t)(q * 16 * RB), ohi = olo + (uint32_t)(8 * RB);
        vt[hb & 1][u] = lds_tr8((tv ^ xlo) + olo, (tv ^ xhi) + ohi);
      }
    };
    v_read(std::integral_constant<int, 0>{});
    // Rows leave through LDS, 128 bytes of each at a time, so that eight lanes store the 128 bytes of a row together: stored
    // from where the products leave them (16 bytes per lane, 32 per row and instruction) every line went to memory
    // in pieces, and the kernel took nearly twice as long (275 against 146 us at 8192 tokens).  Piece p of row r lies at piece p ^ (r & 7).
    auto flush = [&](const Pack8(&piece)[4], int part) {
#pragma unroll
      for (int e = 0; e < 4; ++e) lds_write_vec<u32x4_t>(ldsOut + (uint32_t)((lane & 31) * 128 + (((2 * e + hh) ^ (lane & 7)) * 16)), pack8_vec(piece[e]));
      wave_lds_fence();
      Pack8 y[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = lds_read16(ldsOut + (uint32_t)((8 * k + (lane >> 3)) * 128 + (((lane & 7) ^ ((lane >> 3) & 7)) * 16)));
      wave_lds_fence();
      typedef std::conditional_t<F32, float, uint16_t> E;
      const int f = (part * 8 + (lane & 7)) * (int)(16 / sizeof(E)), PD = part_row_elems(D, (int)sizeof(E));
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int p2 = __shfl(pidx, 8 * k + (lane >> 3), 64);
        if (p2 >= 0 && f < PD) st_stream16(reinterpret_cast<E *>(ws.part) + ((uint64_t)(uint32_t)p2 * (uint32_t)PD + (uint32_t)f), y[k]);
      }
    };
    // once the next tile's loads are in, what is held of this one leaves
    auto flush_held = [&]() {
      arrived();
      if (pidx >= 0 && hh == 0) {
        // The headers of a row share a line.  Where a pair's blocks run on one XCD its L2 collects them (32768 tokens 1975 -> 1789 us, 8192
        // tokens 106 -> 103); where all XCDs work on one pair they go past the caches (262144 tokens 8.04 -> 7.51 ms).
        if constexpr (RANKED) {
          if (one_pair)
            st_stream8(reinterpret_cast<float2 *>(ws.hdr) + pidx, __float_as_uint(m), __float_as_uint(l));
          else
            reinterpret_cast<float2 *>(ws.hdr)[pidx] = make_float2(m, l);
        } else
          st_stream16(ws.hdr + pidx, Pack8{{__float_as_uint(m), __float_as_uint(l), (uint32_t)nb, 0u}});
      }
      // (the header past the caches, as the rows: written the ordinary way it cost 6 to 8 % of the kernel)
#pragma unroll
      for (int part = 0; part < (int)(sizeof(x) / sizeof(x[0])); ++part) flush(x[part], part);
    };
    f32x16 o;
    static_for<2 * NDT>([&](auto hc) {
      constexpr int hb = decltype(hc)::value, dt = hb >> 1;
      if constexpr (hb + 1 < 2 * NDT) v_read(std::integral_constant<int, hb + 1>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr ((hb & 1) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < KT; ++u) {
        const int q = (hb & 1) * KT + u;
        o = mfma32<T>(vt[hb & 1][u], pf[q >> 1][q & 1], o);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr ((hb & 1) == 0) return;
      if constexpr (F32) {
        Pack8 y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int w = 0; w < 4; ++w) y[e].w[w] = __float_as_uint(o[4 * e + w]);
        if constexpr (dt < HELD) {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[dt][e] = y[e];
          if constexpr (dt == HELD - 1) flush_held();
        } else {
          flush(y, dt);
        }
      } else {
        if constexpr (NORM) {
#pragma unroll
          for (int i = 0; i < 16; ++i) o[i] *= inv;
        }
        // four features per lane and group of eight: the two halves of the wave exchange, so that a lane stores eight
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const uint32_t ev = pack2<T>(o[8 * j + 2 * w], o[8 * j + 2 * w + 1]), od = pack2<T>(o[8 * j + 4 + 2 * w], o[8 * j + 4 + 2 * w + 1]);
            Pack8 &y = x[dt >> 1][2 * (dt & 1) + j];
#if defined(__HIP_DEVICE_COMPILE__)
            auto sw = __builtin_amdgcn_permlane32_swap(ev, od, false, false);
            y.w[w] = sw[0];
            y.w[2 + w] = sw[1];
#else
            y.w[w] = ev, y.w[2 + w] = od;
#endif
          }
        }
        if constexpr (dt == NDT - 1) flush_held();
      }
    });
  }
}

// One 16-lane group per (row, head), four per wave, sixteen per block of 256: a row's chain of dependent steps (count,
// headers, order, rows) is mostly waiting, so a wave runs four of them side by side.  Lane li of a group owns the
// 16-byte pieces li, li + 16, .. (NP of them) of the row, whose elements are of type E
// (NORM: divided by the visit's sum of probabilities).
// RANKED: the slots are in key-block order and none of the first `visits` is empty.  The headers and the first rows are asked for beside the count, whole groups of U together without
// branches, and what U does not divide together under them: a row of few visits was a chain of loads (16-bit rows, pass alone: 8192 tokens, 16 heads of 128, top-k 8 52.2 -> 50.2 us; parts of prompts
// 38.4 -> 36.7; 24000 tokens, 8 heads of 128, top-k 5 61.1 -> 54.2; of 96, top-k 7 70.0 -> 57.5; 16 and 22 visits as before, 792 and 750).  Whole groups under the branches of the remainder hold each
// other up where few workgroups wait for their rows: 137 rows, 8 heads of 128, 16 visits 5.9 -> 6.7, without 6.0; 300 rows of 64, 12 visits 5.3 -> 5.8, without 5.3.
// Rows of fp32 (heads above 128) are awaited: short sequences have rows of fewer visits, and what is read in vain is four times as much (seven sequences of 21 to 652 tokens, 8 heads of 256, top-k 4
// 11.8 -> 15.0 us with early rows, 11.5 without; 9000 tokens, top-k 7 96.5 -> 94.4 and 92.7).
// What bounds rows of many visits is the memory: their reads alone, by this pattern, reach 7.1 TB/s, with the output rows
// written between them (a sixteenth of the bytes) 5.7.  The next rows on their way while rows are added: 22 visits 750 -> 820, for the registers.  Over plain lists the rows' places come from LDS: nothing is early, and whole
// groups of U and single rows take 60 us where groups with branches take 67 (12182 tokens, 16 heads of 64, top-k 4).
template <typename T, typename E, int NP, bool NORM, bool RANKED>
__global__ __launch_bounds__(256) void attn_fwd_combine_kernel(fmoba_attn_fwd_args a, FwdWs ws, int capl) {
  extern __shared__ __attribute__((aligned(16))) int sOrdAll[];  // [16 groups][capl]: slot of the partial of rank r
  __shared__ float sWgt[16][16], sWl[16][16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, grp = lane >> 4, li = lane & 15;
  const int sg = wv * 4 + grp;  // group of the block
  int *sOrd = sOrdAll + (size_t)sg * capl;
  const int64_t total = (int64_t)a.total_q * a.heads;
  const int64_t rh_raw = (int64_t)blockIdx.x * 16 + sg;  // (global row) * heads + head
  const bool valid = rh_raw < total;
  const int64_t rh = valid ? rh_raw : total - 1;
  const int64_t row = rh / a.heads;
  const int h = (int)(rh - row * a.heads);
  const int D = a.head_dim;
  const int nall = !valid ? 0 : RANKED ? (int)(ws.visits[(int64_t)h * a.total_q + row] & 0xffffu) : ws.cnt[rh];
  const int n = min(nall, ws.cap);
  if (nall > ws.cap && li == 0 && a.visits_overflow != nullptr) atomicMax(a.visits_overflow, nall);  // visits were dropped
  int nmax = max(n, __shfl_xor(n, 16, 64));
  nmax = max(nmax, __shfl_xor(nmax, 32, 64));  // the wave walks the longest of its four rows
  constexpr int PE = 16 / sizeof(E);  // elements of a piece
  const int c0 = li * PE;             // the lane's pieces begin at features c0, c0 + 16 * PE, ..
  const bool mine = c0 < D;
  float acc[PE * NP];
#pragma unroll
  for (int i = 0; i < PE * NP; ++i) acc[i] = 0.f;
  float L = 0.f, M = -INFINITY;
  const float4 *hdr = ws.hdr + rh * ws.cap;
  const float2 *hdr2 = reinterpret_cast<const float2 *>(ws.hdr) + rh * ws.cap;
  const int PD = part_row_elems(D, (int)sizeof(E));
  const E *part = reinterpret_cast<const E *>(ws.part) + rh * ws.cap * PD;
  // The slot a visit got is arbitrary (a counter handed it out), the sum must not depend on it: every partial gets
  // its rank in ascending key-block order over the WHOLE row (equal ids, a malformed pattern, are ordered by slot),
  // and the partials are merged in rank order, 16 at a time.
  if constexpr (!RANKED) group_rank_order(reinterpret_cast<const int *>(hdr) + 2, 4, n, nmax, sOrd, lane);
  auto load = [&](Pack8(&y)[NP], int slot) {
    const E *from = part + (int64_t)slot * PD + c0;
#pragma unroll
    for (int p = 0; p < NP; ++p) y[p] = ld_stream16(c0 + p * 16 * PE < D ? from + p * 16 * PE : from);
  };
  // rows i0 .. of a ranked row, as far as there are `have` of them
  constexpr int U = 4;
  auto fetch = [&](Pack8(&y)[U][NP], int i0, int have) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i0 + u >= have) break;
      load(y[u], i0 + u);
    }
  };
  constexpr bool kEarly = NP == 1;  // (rows of 16 bits)
  Pack8 x[U][NP];  // (of ranked rows)
  float2 head = {-INFINITY, 0.f};
  if constexpr (RANKED) {  // asked for beside the count: what lies behind it is not used
    if (li < ws.cap) head = hdr2[li];
    if (kEarly && mine) fetch(x, 0, ws.cap);
  }
  for (int base = 0; base < nmax; base += 16) {
    const int cntb = min(16, max(n - base, 0));
    float mj = -INFINITY, lj = 0.f;
    if (li < cntb) {
      if constexpr (RANKED) {
        mj = head.x, lj = head.y;
        if (base + 16 + li < n) head = hdr2[base + 16 + li];
      } else {
        const float4 hd = hdr[sOrd[base + li]];
        mj = hd.x, lj = hd.y;
      }
    }
    float mb = mj;
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) mb = fmaxf(mb, __shfl_xor(mb, o, 64));
    const float Mn = fmaxf(M, mb);
    const float Mu = Mn == -INFINITY ? 0.f : Mn;
    const float resc = __builtin_amdgcn_exp2f(M - Mu);  // M = -inf: nothing accumulated yet, factor 0 on zeros
#pragma unroll
    for (int i = 0; i < PE * NP; ++i) acc[i] *= resc;
    L *= resc;
    M = Mn;
    const float wj = (li < cntb) ? __builtin_amdgcn_exp2f(mj - Mu) : 0.f;
    wave_lds_fence();
    if (li < cntb) {
      sWgt[sg][li] = NORM ? wj * lj : wj;
      sWl[sg][li] = wj * lj;
    }
    wave_lds_fence();
    // sums in rank order: every lane of the group adds the same sequence
    for (int t = 0; t < cntb; ++t) L += sWl[sg][t];
    if (mine) {
      auto add = [&](const Pack8(&x)[NP], float w) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if constexpr (sizeof(E) == 4) {
              acc[4 * p + k] = fmaf(w, __uint_as_float(x[p].w[k]), acc[4 * p + k]);
            } else {
              acc[8 * p + 2 * k] = fmaf(w, elem_to_float<T>((uint16_t)(x[p].w[k] & 0xffffu)), acc[8 * p + 2 * k]);
              acc[8 * p + 2 * k + 1] = fmaf(w, elem_to_float<T>((uint16_t)(x[p].w[k] >> 16)), acc[8 * p + 2 * k + 1]);
            }
          }
      };
      if constexpr (RANKED) {
        int t = 0;
        for (; t + U <= cntb; t += U) {
          if (!kEarly || base + t > 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) load(x[u], base + t + u);
          }
#pragma unroll
          for (int u = 0; u < U; ++u) add(x[u], sWgt[sg][t + u]);
        }
        if (t < cntb) {
          if (!kEarly || base + t > 0) fetch(x, base + t, n);
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (t + u < cntb) add(x[u], sWgt[sg][t + u]);
        }
      } else {
        int t = 0;
        for (; t + U <= cntb; t += U) {  // independent loads, four in flight
          Pack8 y[U][NP];
          float w[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            load(y[u], sOrd[base + t + u]);
            w[u] = sWgt[sg][t + u];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) add(y[u], w[u]);
        }
        for (; t < cntb; ++t) {
          Pack8 y[NP];
          load(y, sOrd[base + t]);
          add(y, sWgt[sg][t]);
        }
      }
    }
  }
  if (!valid) return;
  const bool empty = !(L > 0.f);
  const float inv = empty ? 0.f : 1.f / L;
  uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + row * a.o_row_stride + (int64_t)h * a.o_head_stride + c0;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    struct alignas(2 * PE) {
      uint32_t w[PE / 2];
    } o;
#pragma unroll
    for (int k = 0; k < PE / 2; ++k) o.w[k] = pack2<T>(acc[PE * p + 2 * k] * inv, acc[PE * p + 2 * k + 1] * inv);
    if (c0 + p * 16 * PE < D) *reinterpret_cast<decltype(o) *>(op + p * 16 * PE) = o;
  }
  if (li == 0) a.softmax_lse[(int64_t)h * a.total_q + row] = empty ? INFINITY : (M + __builtin_amdgcn_logf(L)) * 0.6931471805599453f;
}

__global__ void fwd_empty_kernel(void *out, float *lse, int64_t n_out_words, int64_t n_lse) {
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, st = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = i0; i < n_out_words; i += st) reinterpret_cast<uint32_t *>(out)[i] = 0u;
  for (int64_t i = i0; i < n_lse; i += st) lse[i] = INFINITY;
}

__global__ void fwd_zero_i32_kernel(int32_t *p, int64_t n, int32_t *one_more) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0;
  if (one_more != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *one_more = 0;
}

// visits per (row, head) of a pattern: grid over list entries is not possible without the segment of each
// entry, so one workgroup walks one column list
__global__ __launch_bounds__(256) void csc_row_visits_kernel(fmoba_attn_fwd_args a, int32_t *cnt, int kb) {
  const int c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int64_t bh = (int64_t)b * a.heads + h;
  const int nnz = a.col_nnz[bh * a.max_cols + c];
  const int32_t *list = a.row_indices + a.col_offsets[bh * a.max_cols + c];
  // key blocks of this column that exist in the sequence
  const int key_lo = c * a.lg_block_n, key_hi = min(Lk, key_lo + a.lg_block_n);
  const int nblk = key_hi > key_lo ? (key_hi - key_lo + kb - 1) / kb : 0;
  if (nblk == 0) return;
  for (int i = threadIdx.x; i < nnz; i += 256) {
    const int r = list[i];
    if (r >= 0 && r < Lq) atomicAdd(&cnt[(int64_t)(q0 + r) * a.heads + h], nblk);
  }
}
// The same with the counts of a range of rows of one (sequence, head) in LDS: no atomics in memory, the maximum on the way out.  Every workgroup
// reads all lists of the pair (in any order) and counts what falls into its rows; a wave takes 512 entries of two lists at a time.
// Bound by the latency of those loads, which go out together, past a list's end from its last entry: each under a branch of its own with a wait (entries that exist alone
// were asked for) took 90 us where this takes 30 (30039 tokens, 8 heads, top-k 14; 12182 tokens, 16 heads, top-k 4 27 -> 12).
// grid (row ranges, heads, batch); `range` rows in LDS, `max_out` cleared before.
__global__ __launch_bounds__(1024) void csc_row_visits_lds_kernel(fmoba_attn_fwd_args a, int32_t *cnt, int32_t *max_out, int kb, int range) {
  extern __shared__ int32_t visits[];
  constexpr int kCols = 512;
  __shared__ int64_t first[kCols];
  __shared__ int32_t len[kCols], blocks[kCols], most;
  const int h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int64_t bh = (int64_t)b * a.heads + h;
  const int ncols = min(a.max_cols, (Lk + a.lg_block_n - 1) / a.lg_block_n);
  if (tid == 0) most = 0;
  for (int r0 = blockIdx.x * range; r0 < Lq; r0 += gridDim.x * range) {
    const int rows = min(range, Lq - r0);
    for (int i = tid; i < rows; i += blockDim.x) visits[i] = 0;
    for (int c0 = 0; c0 < ncols; c0 += kCols) {
      const int nc = min(kCols, ncols - c0);
      __syncthreads();
      for (int i = tid; i < nc; i += blockDim.x) {
        const int key_lo = (c0 + i) * a.lg_block_n, key_hi = min(Lk, key_lo + a.lg_block_n);
        first[i] = a.col_offsets[bh * a.max_cols + c0 + i];
        len[i] = a.col_nnz[bh * a.max_cols + c0 + i];
        blocks[i] = (key_hi - key_lo + kb - 1) / kb;  // key blocks of the column that exist in the sequence
      }
      __syncthreads();
      for (int c = 2 * wave; c < nc; c += 2 * waves) {
        const bool two = c + 1 < nc;
        const int32_t *list[2] = {a.row_indices + first[c], a.row_indices + first[two ? c + 1 : c]};
        const int n[2] = {len[c], two ? len[c + 1] : 0};
        for (int p = 0; p < max(n[0], n[1]); p += 512) {
          int r[2][8];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            if (p >= n[u]) continue;  // (entries past a list's end are not read, not even where the list is empty)
#pragma unroll
            for (int i = 0; i < 8; ++i) r[u][i] = list[u][min(p + i * 64 + lane, n[u] - 1)];
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int add = blocks[u && two ? c + 1 : c];
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (p + i * 64 + lane < n[u] && (uint32_t)(r[u][i] - r0) < (uint32_t)rows) atomicAdd(&visits[r[u][i] - r0], add);
          }
        }
      }
    }
    __syncthreads();
    int m = 0;
    for (int i = tid; i < rows; i += blockDim.x) {
      const int v = visits[i];
      cnt[(int64_t)(q0 + r0 + i) * a.heads + h] = v;
      m = max(m, v);
    }
    for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    if (lane == 0 && m > 0) atomicMax(&most, m);
    __syncthreads();  // (the next range takes the places)
  }
  __syncthreads();
  if (tid == 0 && most > 0) atomicMax(max_out, most);  // (one per workgroup: atomics on one address go one after the other, some 15 ns each)
}
__global__ __launch_bounds__(256) void max_i32_kernel(const int32_t *p, int64_t n, int32_t *out) {
  int m = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) m = max(m, p[i]);
  for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  __shared__ int most[4];
  if ((threadIdx.x & 63) == 0) most[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = max(max(most[0], most[1]), max(most[2], most[3]));
    if (m > 0) atomicMax(out, m);
  }
}

static inline size_t fwd_align256(size_t x) { return (x + 255) & ~(size_t)255; }
static inline int fwd_key_block(int lg_block_n) { return lg_block_n % 128 == 0 ? 128 : 64; }
// partial slots per (row, head): above head dimension 128, where dense patterns come here too, no more than a sequence has key blocks
// (top-k times the chunk can be far beyond the keys of a short sequence)
static inline int64_t fwd_partial_cap(const fmoba_attn_fwd_args &a) {
  const int64_t visits = a.max_visits_per_row;
  return a.head_dim > 128 ? std::min(visits, std::max<int64_t>(1, ceil_div64(a.max_seqlen_k, fwd_key_block(a.lg_block_n)))) : visits;
}
// the combine keeps the order of sixteen rows' partial results in LDS, beside two 16 x 16 tables
constexpr int kCombineStaticLds = 2 * 16 * 16 * 4;
static inline bool fwd_combine_fits(const fmoba_attn_fwd_args &a) {
  return (fwd_partial_cap(a) + 15) / 16 * 16 * 64 + kCombineStaticLds <= 160 * 1024;
}

// the row-block form (attn_fwd_rows.hip)
bool fwd_rows_feasible(const fmoba_attn_fwd_args &a);
bool fwd_rows_direct(const fmoba_attn_fwd_args &a);  // without loader waves
bool fwd_few_rows(const fmoba_attn_fwd_args &a);  // its variant for calls with a handful of rows (attn_fwd_few.hip)
size_t fwd_rows_workspace_bytes(const fmoba_attn_fwd_args &a);
int run_fwd_rows(const fmoba_attn_fwd_args &a, int phases, hipStream_t s);

// Mean length of the sequence that a row belongs to, of `batch` sequences of `total` rows whose longest has `longest` and the others as many as each other (the
// least that it can be).
static int64_t row_mean_length(int64_t total, int64_t longest, int64_t batch) {
  longest = std::min(longest, total);
  if (batch <= 1 || longest <= 0) return longest;
  const double rest = (double)(total - longest);
  return (int64_t)(((double)longest * (double)longest + rest * rest / (double)(batch - 1)) / (double)total);
}

// Which form runs.  The row-block form multiplies every row of a 128-row block with every chunk that
// any of its rows selected, the column form only the selected pairs but pays a partial result per
// visit: the first wins while a row selects more than about a fifth of the chunks it may see (64-key blocks) or
// more than about three eighths of them (128-key blocks, whose visits cost the column form less per key).
static bool fwd_use_rows(const fmoba_attn_fwd_args &a) {
  if (a.fwd_mode == 1) return false;
  if (!fwd_rows_feasible(a)) return false;
  if (a.fwd_mode == 2 || fwd_few_rows(a)) return true;
  const int64_t chunks_per_seq = std::max<int64_t>(1, ceil_div64(ceil_div64(std::max(a.total_k, 1), a.batch), a.lg_block_n));
  const int64_t seen = a.is_causal ? (chunks_per_seq + 1) / 2 : chunks_per_seq;
  const int64_t chunks_per_row = std::max<int64_t>(1, (int64_t)a.max_visits_per_row * fwd_key_block(a.lg_block_n) / a.lg_block_n);
  const bool wide_keys = fwd_key_block(a.lg_block_n) == 128;
  if (a.head_dim > 128) {
    const int64_t partials = (int64_t)a.total_q * a.heads * fwd_partial_cap(a);
    if (!fwd_combine_fits(a) || partials >= ((int64_t)1 << 31) || partials * (int64_t)(a.head_dim * fwd_part_size(a.head_dim) + 16) > kWidePartialBytes) return true;
    // (What a row may see goes by its own sequence's length, of which the longest is known, and by where its queries lie in it.  By the mean length and as
    // if every call were a whole prompt, columns against rows: one sequence of 25592 tokens with five short ones, 8 heads, top-k 3 of 256-key chunks 1452
    // against 2956 us, parts of prompts of 1451 rows against 11481 keys, 32 over 4 heads, top-k 7 of 64-key chunks 259 against 670.)
    const int64_t kl = row_mean_length(a.total_k, a.max_seqlen_k, a.batch), ql = std::min(kl, row_mean_length(a.total_q, a.max_seqlen_q, a.batch));
    const int64_t seen_wide = std::max<int64_t>(1, (a.is_causal ? kl - ql / 2 : kl) / a.lg_block_n);
    return fwd_rows_direct(a) && (int64_t)a.heads * (a.total_q / 128 + a.batch) >= kFwdRowsWideBlocks && chunks_per_row * (wide_keys ? kFwdRowsDensityWide128 : kFwdRowsDensityWide64) >= seen_wide * 10;
  }
  return chunks_per_row * (wide_keys ? kFwdRowsDensity128 : kFwdRowsDensity64) >= seen * 10;
}

// Query heads per workgroup.  All heads of a group share the block's K and V and a workgroup's first loads, which is most of the
// time of a call with short lists (1000-row parts of prompts against 9000 to 33000 keys: 164 us, 325 with a head each).  Long
// lists make few long workgroups of it, so the group is divided until there are three rounds of them for the chip's 512
// places, as long as each of the four waves keeps two tiles (32 over 8 heads, top-k 4 of 128-key chunks: 4096 tokens
// 131 -> 68 us, 8192 tokens 190 -> 127, 16384 tokens 292 -> 231; with one head each 24576 tokens take 462 us instead of 419).
static int fwd_col_heads(const fmoba_attn_fwd_args &a, int kb) {
  const int grp = a.heads / a.heads_k;
  const int64_t blocks = (int64_t)a.total_k / kb + a.batch;
  const int64_t tiles = (int64_t)a.total_q * fwd_partial_cap(a) / 32 / blocks;  // of one head's lists, on average
  int best = grp;
  while (best > 64 || grp % best != 0) --best;  // (a lane of the kernel's waves per list)
  for (int gs = best - 1; gs >= 1 && blocks * (a.heads / best) < 1536 && tiles * gs >= 8; --gs)
    if (grp % gs == 0) best = gs;
  return best;
}
template <typename T, int HD, int KB>
static int launch_fwd_col(const fmoba_attn_fwd_args &a, const FwdWs &ws, hipStream_t s) {
  const bool ranked = ws.visits != nullptr;
  const int grp = fwd_col_heads(a, KB);
  const ItemOrder order = col_order(a, a.heads / grp, HD, KB);
  auto kern = a.head_dim == HD ? (ranked ? attn_fwd_col_kernel<T, HD, KB, true, true> : attn_fwd_col_kernel<T, HD, KB, true, false>)
                               : (ranked ? attn_fwd_col_kernel<T, HD, KB, false, true> : attn_fwd_col_kernel<T, HD, KB, false, false>);
  const size_t smem = FwdColSmem<HD, KB>::bytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_fwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const int64_t items = (a.heads / grp) * (order >= kListedLongestFirst ? listed_blocks(a.total_k, a.batch, KB) : (int64_t)a.batch * ceil_div(a.max_seqlen_k, KB));
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_fwd: too many (sequence, head, key block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(64 * FwdColSmem<HD, KB>::NW), smem, s, a, ws, grp, order);
  return 0;
}
template <typename T>
static int run_fwd(const fmoba_attn_fwd_args &a, const FwdWs &ws, int phases, hipStream_t s) {
  const int64_t rows = (int64_t)a.total_q * a.heads;
  if (phases & FMOBA_FWD_COLUMNS) {
    if (ws.visits == nullptr) hipLaunchKernelGGL(fwd_zero_i32_kernel, dim3(512), dim3(256), 0, s, ws.cnt, rows, (int32_t *)nullptr);
    const int kb = fwd_key_block(a.lg_block_n);
    int rc;
    if (a.head_dim > 128)
      rc = kb == 128 ? launch_fwd_col<T, 256, 128>(a, ws, s) : launch_fwd_col<T, 256, 64>(a, ws, s);
    else if (a.head_dim <= 64)
      rc = kb == 128 ? launch_fwd_col<T, 64, 128>(a, ws, s) : launch_fwd_col<T, 64, 64>(a, ws, s);
    else
      rc = kb == 128 ? launch_fwd_col<T, 128, 128>(a, ws, s) : launch_fwd_col<T, 128, 64>(a, ws, s);
    if (rc) return rc;
  }
  if (phases & FMOBA_FWD_COMBINE) {
    const int capl = combine_order_entries(ws.cap);
    const bool ranked = ws.visits != nullptr;
    const size_t smem = ranked ? 0 : (size_t)16 * capl * 4;
    constexpr bool NORM = kFwdNormalisedParts<T, 128>;
    auto kern = a.head_dim > 128 ? (ranked ? attn_fwd_combine_kernel<T, float, 4, false, true> : attn_fwd_combine_kernel<T, float, 4, false, false>)
                                 : (ranked ? attn_fwd_combine_kernel<T, uint16_t, 1, NORM, true> : attn_fwd_combine_kernel<T, uint16_t, 1, NORM, false>);
    if (smem > 32 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
      set_error("attn_fwd: a row with up to %d visits needs %zu bytes of LDS for the order of its partial results", ws.cap, smem);
      return 2;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 15) / 16)), dim3(256), smem, s, a, ws, capl);
  }
  return 0;
}

}  // namespace fmoba

extern "C" int32_t fmoba_attn_fwd_key_block(int32_t lg_block_n) { return fmoba::fwd_key_block(lg_block_n); }

static size_t fwd_cols_workspace_bytes(const fmoba_attn_fwd_args &a) {
  using namespace fmoba;
  if (a.max_visits_per_row <= 0) return 256;
  const size_t rows = (size_t)a.total_q * a.heads, cap = (size_t)fwd_partial_cap(a);
  return fwd_align256((rows + 1) * 4) + fwd_align256(rows * cap * 16) + fwd_align256(rows * cap * part_row_elems(a.head_dim, (int)fwd_part_size(a.head_dim)) * fwd_part_size(a.head_dim)) + 256;
}

extern "C" size_t fmoba_attn_fwd_workspace_bytes(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  if (a == nullptr || a->total_q <= 0 || a->heads <= 0 || a->head_dim <= 0 || a->batch <= 0 || a->lg_block_n <= 0) return 256;
  if (fwd_use_rows(*a)) return fwd_rows_workspace_bytes(*a);
  return fwd_cols_workspace_bytes(*a);
}

extern "C" int32_t fmoba_attn_fwd_uses_row_blocks(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  if (a == nullptr || a->total_q <= 0 || a->heads <= 0 || a->head_dim <= 0 || a->batch <= 0 || a->lg_block_n <= 0) return 0;
  return fwd_use_rows(*a) ? 1 : 0;
}

static int fwd_check_common(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  FMOBA_REQUIRE(a != nullptr, "attn_fwd: null args");
  FMOBA_REQUIRE(a->dtype == FMOBA_DTYPE_F16 || a->dtype == FMOBA_DTYPE_BF16, "FlashMoBA only support fp16 and bf16 data type");
  FMOBA_REQUIRE(a->batch > 0, "batch size must be positive");
  FMOBA_REQUIRE(a->head_dim > 0 && a->head_dim <= 256, "FlashMoBA forward only supports head dimension at most 256");
  FMOBA_REQUIRE(a->head_dim % 8 == 0, "query, key, value, and out_ must have a head_size that is a multiple of 8");
  FMOBA_REQUIRE(a->heads > 0 && a->heads_k > 0 && a->heads % a->heads_k == 0, "Number of heads in key/value must divide number of heads in query");
  FMOBA_REQUIRE(a->lg_block_m >= 128 && a->lg_block_m <= 1024, "m_lg_block_dim must be at least 128 and at most 1024");
  FMOBA_REQUIRE(a->lg_block_m % 64 == 0, "m_lg_block_dim must be a multiple of 64");
  FMOBA_REQUIRE(a->lg_block_n > 0 && a->lg_block_n % 64 == 0, "n_lg_block_dim must be a multiple of 64");
  FMOBA_REQUIRE(a->total_q >= 0 && a->total_k >= 0 && a->max_seqlen_q >= 0 && a->max_seqlen_k >= 0 && a->max_cols >= 0, "negative size");
  FMOBA_REQUIRE(a->cu_seqlens_q && a->cu_seqlens_k, "attn_fwd: null cu_seqlens pointer");
  FMOBA_REQUIRE(a->batch <= 65535 && a->heads <= 65535, "attn_fwd: batch/heads too large for the launch grid");
  return 0;
}

// Counts in LDS or by atomics in memory.  In LDS a workgroup reads all lists of its (sequence, head), some 10 entries per ns, so the longest sequence is the
// call; the whole chip does 27 atomics per ns, up to 60 where the counters of few heads lie close together.  So LDS where a call is worth
// many heads of its longest sequence.  Atomics and LDS, us: 262144 tokens, top-k 16 of 128-key chunks, 1 head 141 and 408, 8 heads 1204 and 436;
// 90000 tokens, top-k 8, 2 heads 55 and 85, 16 heads 446 and 94; 20000 tokens, 2 heads 16.5 and 19.5, 16 heads 106 and 25; sequences of 20000, 4 x 1 head 21.3 and 20.3, 16 x 2
// heads 128 and 32; one of 200000 with seven of 2048, 1 head 59 and 186.  And where the longest lists are so short that their reading takes less than the two more launches: 8 heads of
// 1000 tokens 8.3 and 7.3.  (The line is the one of a pass that read 2.4 entries per ns; LDS has since been the faster from four heads of the longest sequence on.)
static bool csc_visits_in_lds(const fmoba_attn_fwd_args &a) {
  const int64_t longest = std::max(1, a.max_seqlen_q), alike = (int64_t)a.heads * a.total_q / longest;
  return alike >= std::max(12, 64 / a.heads) || (alike >= 8 && longest * a.max_cols <= 32768);
}
extern "C" int32_t fmoba_csc_row_visits_in_lds(const fmoba_attn_fwd_args *a) { return a != nullptr && a->heads > 0 && csc_visits_in_lds(*a) ? 1 : 0; }

extern "C" int fmoba_csc_max_row_visits(const fmoba_attn_fwd_args *a, int32_t *counts, int32_t *max_out, void *stream) {
  using namespace fmoba;
  if (int rc = fwd_check_common(a)) return rc;
  FMOBA_REQUIRE(counts && max_out, "csc_max_row_visits: null output pointer");
  hipStream_t s = (hipStream_t)stream;
  const int64_t rows = (int64_t)a->total_q * a->heads;
  hipLaunchKernelGGL(fwd_zero_i32_kernel, dim3(256), dim3(256), 0, s, counts, rows, max_out);
  if (rows > 0 && a->max_cols > 0 && a->total_k > 0) {
    FMOBA_REQUIRE(a->col_offsets && a->col_nnz && a->row_indices, "csc_max_row_visits: null CSC pointer");
    // Row ranges: enough of them for a workgroup per compute unit, 1024 to 32768 rows.
    const int64_t pairs = (int64_t)a->batch * a->heads;
    const int per = ceil_div(a->max_seqlen_q, (int)std::max<int64_t>(1, 256 / pairs));
    const int range = std::min(32768, std::max(1024, (per + 255) & ~255)), nrange = std::max(1, ceil_div(a->max_seqlen_q, range));
    const size_t smem = (size_t)range * 4;
    auto kern = csc_row_visits_lds_kernel;
    if (csc_visits_in_lds(*a) &&
        (smem <= 32 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess)) {
      hipLaunchKernelGGL(kern, dim3(nrange, a->heads, a->batch), dim3(1024), smem, s, *a, counts, max_out, fwd_key_block(a->lg_block_n), range);
    } else {
      hipLaunchKernelGGL(csc_row_visits_kernel, dim3(a->max_cols, a->heads, a->batch), dim3(256), 0, s, *a, counts, fwd_key_block(a->lg_block_n));
      hipLaunchKernelGGL(max_i32_kernel, dim3(256), dim3(256), 0, s, counts, rows, max_out);
    }
  }
  FMOBA_LAUNCH_CHECK("csc_max_row_visits");
  return 0;
}

// the tensors and strides of a call that has keys
static int fwd_check_tensors(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  FMOBA_REQUIRE(a->k && a->v, "attn_fwd: null k/v pointer");
  const int64_t st[] = {a->q_row_stride, a->q_head_stride, a->k_row_stride, a->k_head_stride,
                        a->v_row_stride, a->v_head_stride, a->o_row_stride, a->o_head_stride};
  for (int64_t x : st) FMOBA_REQUIRE(x % 8 == 0, "attn_fwd: strides must be multiples of 8 elements");
  FMOBA_REQUIRE(a->q_row_stride < ((int64_t)1 << 31), "attn_fwd: q_row_stride must be below 2^31 elements");
  FMOBA_REQUIRE(((uintptr_t)a->q % 16) == 0 && ((uintptr_t)a->k % 16) == 0 && ((uintptr_t)a->v % 16) == 0 && ((uintptr_t)a->out % 16) == 0,
                "attn_fwd: q, k, v and out must be 16-byte aligned");
  FMOBA_REQUIRE(a->max_visits_per_row > 0, "attn_fwd: max_visits_per_row must be positive");
  return 0;
}

extern "C" int fmoba_attn_fwd(const fmoba_attn_fwd_args *a, void *stream) { return fmoba_attn_fwd_phases(a, 3, stream); }

extern "C" int fmoba_attn_fwd_phases(const fmoba_attn_fwd_args *a, int32_t phases, void *stream) { return fmoba_attn_fwd_ranked(a, nullptr, phases, stream); }

extern "C" int fmoba_attn_fwd_ranked(const fmoba_attn_fwd_args *a, const uint32_t *visits, int32_t phases, void *stream) {
  using namespace fmoba;
  if (int rc = fwd_check_common(a)) return rc;
  FMOBA_REQUIRE(phases > 0 && phases <= 3, "attn_fwd: phases must be a mask of bits 1, 2");
  hipStream_t s = (hipStream_t)stream;
  if (a->total_q == 0 || a->max_seqlen_q == 0) return 0;
  FMOBA_REQUIRE(a->q && a->out && a->softmax_lse, "attn_fwd: null q/out/lse pointer");
  if (a->max_seqlen_k == 0 || a->total_k == 0 || a->max_cols == 0) {
    // no keys: out = 0, lse = +inf (csrc/flash_moba/flash_moba_api.cpp:589-593); needs a dense out
    FMOBA_REQUIRE(a->o_head_stride == a->head_dim && a->o_row_stride == (int64_t)a->heads * a->head_dim,
                  "attn_fwd: out must be contiguous when there are no keys");
    hipLaunchKernelGGL(fwd_empty_kernel, dim3(512), dim3(256), 0, s, a->out, a->softmax_lse,
                       (int64_t)a->total_q * a->heads * a->head_dim / 2, (int64_t)a->total_q * a->heads);
    FMOBA_LAUNCH_CHECK("attn_fwd(empty)");
    return 0;
  }
  FMOBA_REQUIRE((a->col_offsets && a->col_nnz && a->row_indices) || (a->selection_bits && fwd_use_rows(*a)), "attn_fwd: null CSC pointer");
  if (int rc = fwd_check_tensors(a)) return rc;
  FMOBA_REQUIRE(a->fwd_mode >= 0 && a->fwd_mode <= 2, "attn_fwd: fwd_mode must be 0 (automatic), 1 (columns) or 2 (row blocks)");
  FMOBA_REQUIRE(a->fwd_mode != 2 || fwd_rows_feasible(*a), "attn_fwd: the row-block form does not take this shape (more than %d chunks or %d keys per sequence)",
                32 * 128, 64 * 4096);
  const size_t need = fmoba_attn_fwd_workspace_bytes(a);
  FMOBA_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= need, "attn_fwd: workspace too small (%zu < %zu)", a->workspace_bytes, need);
  if (fwd_use_rows(*a)) {
    FMOBA_REQUIRE(visits == nullptr || a->selection_bits != nullptr, "attn_fwd: the row-block form reads plain lists or selection bits");
    if (int rc = run_fwd_rows(*a, phases, s)) return rc;
    FMOBA_LAUNCH_CHECK("attn_fwd");
    return 0;
  }
  const size_t rows = (size_t)a->total_q * a->heads;
  FMOBA_REQUIRE(rows * (size_t)fwd_partial_cap(*a) < ((size_t)1 << 31),
                "attn_fwd: %zu partial rows exceed the 2^31 the column form indexes (their workspace would not fit any device either)",
                rows * (size_t)fwd_partial_cap(*a));
  uintptr_t p = ((uintptr_t)a->workspace + 255) & ~(uintptr_t)255;
  FwdWs ws;
  ws.cap = (int32_t)fwd_partial_cap(*a);
  ws.cnt = reinterpret_cast<int32_t *>(p);
  p += fwd_align256((rows + 1) * 4);
  ws.hdr = reinterpret_cast<float4 *>(p);
  p += fwd_align256(rows * ws.cap * 16);
  ws.part = reinterpret_cast<void *>(p);
  ws.visits = visits;
  int rc = a->dtype == FMOBA_DTYPE_BF16 ? run_fwd<bf16_t>(*a, ws, phases, s) : run_fwd<f16_t>(*a, ws, phases, s);
  if (rc) return rc;
  FMOBA_LAUNCH_CHECK("attn_fwd");
  return 0;
}

namespace fmoba {
bool fwd_rows_gated(const fmoba_attn_fwd_args &a);  // attn_fwd_rows.hip
// the checks of a forward call whose gate is part of it (topk_csc.hip)
int fwd_check_gated(const fmoba_attn_fwd_args *a) {
  if (int rc = fwd_check_common(a)) return rc;
  FMOBA_REQUIRE(a->total_q > 0 && a->max_seqlen_q > 0 && a->total_k > 0 && a->max_seqlen_k > 0, "attn_fwd: empty problem");
  FMOBA_REQUIRE(a->q && a->out && a->softmax_lse, "attn_fwd: null q/out/lse pointer");
  if (int rc = fwd_check_tensors(a)) return rc;
  FMOBA_REQUIRE(fmoba_attn_fwd_gates_rows(a) != 0, "attn_fwd_gated_rows: not a call of this form (fmoba_attn_fwd_gates_rows tells)");
  return 0;
}
bool pool_scores_feasible(int head_dim, int group, int rows, int batch);                                       // mean_pool.hip
int mean_pool_with_scores(const fmoba_mean_pool_args *a, const FewGate &few, int64_t total_k, void *stream);
void run_fwd_few_scored(const fmoba_attn_fwd_args &a, const FewGate &few, hipStream_t s);                      // attn_fwd_few.hip
}  // namespace fmoba

extern "C" int32_t fmoba_attn_fwd_gates_rows(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  return fmoba_attn_fwd_uses_row_blocks(a) && a->fwd_mode == 0 && fwd_rows_gated(*a) ? 1 : 0;
}

extern "C" size_t fmoba_attn_fwd_gated_few_bytes(const fmoba_attn_fwd_args *a) {
  using namespace fmoba;
  if (a == nullptr || a->total_q <= 0 || a->total_k <= 0 || a->heads <= 0 || a->heads_k <= 0 || a->batch <= 0 || a->max_seqlen_q <= 0 || a->lg_block_n <= 0) return 0;
  if (a->fwd_mode != 0 || !fwd_rows_feasible(*a) || !fwd_few_rows(*a) || !pool_scores_feasible(a->head_dim, a->heads / a->heads_k, a->max_seqlen_q, a->batch)) return 0;
  return fwd_align256((size_t)(a->total_k / a->lg_block_n + a->batch) * a->heads * a->max_seqlen_q * 4);
}

extern "C" int fmoba_attn_fwd_gated_few(const fmoba_mean_pool_args *m, const fmoba_attn_fwd_args *a, int32_t topk, int32_t gate_is_causal, float *scores, void *stream) {
  using namespace fmoba;
  if (int rc = fwd_check_common(a)) return rc;
  FMOBA_REQUIRE(m != nullptr && scores != nullptr && m->cu_seqlens_km != nullptr, "attn_fwd_gated_few: null pointer");
  FMOBA_REQUIRE(fmoba_attn_fwd_gated_few_bytes(a) > 0, "attn_fwd_gated_few: not a call of this form (fmoba_attn_fwd_gated_few_bytes tells)");
  FMOBA_REQUIRE(topk >= 1 && topk <= 64, "moba_topk must be in [1, 64]");
  FMOBA_REQUIRE(m->k == a->k && m->cu_seqlens_k == a->cu_seqlens_k && m->batch == a->batch && m->heads_k == a->heads_k && m->head_dim == a->head_dim &&
                    m->chunk == a->lg_block_n && m->dtype == a->dtype && m->k_row_stride == a->k_row_stride && m->k_head_stride == a->k_head_stride,
                "attn_fwd_gated_few: the two argument structs describe different problems");
  FMOBA_REQUIRE(m->max_chunks == a->max_cols && a->max_cols == ceil_div(a->max_seqlen_k, a->lg_block_n), "attn_fwd_gated_few: max_cols is ceil(max_seqlen_k / lg_block_n)");
  FMOBA_REQUIRE(a->q && a->out && a->softmax_lse, "attn_fwd: null q/out/lse pointer");
  if (int rc = fwd_check_tensors(a)) return rc;
  FewGate few;
  few.q = reinterpret_cast<const uint16_t *>(a->q), few.cu_seqlens_q = a->cu_seqlens_q, few.cu_seqlens_km = m->cu_seqlens_km, few.scores = scores;
  few.q_row_stride = a->q_row_stride, few.q_head_stride = a->q_head_stride;
  few.heads = a->heads, few.group = a->heads / a->heads_k, few.rows = a->max_seqlen_q, few.topk = topk, few.is_causal = gate_is_causal;
  if (int rc = mean_pool_with_scores(m, few, a->total_k, stream)) return rc;
  run_fwd_few_scored(*a, few, (hipStream_t)stream);
  FMOBA_LAUNCH_CHECK("attn_fwd_gated_few");
  return 0;
}
