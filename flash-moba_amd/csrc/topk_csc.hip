// Fused top-k block gating and deterministic CSC build.
//
//   topk_gate_kernel : scores S^T = KM * Q^T on MFMA, per-row exact top-k by the best scores one by one or by bisection on
//                      order-preserving keys, scores held in registers (no score matrix, no sorted
//                      list and no per-row index list ever reaches HBM); emits one selection
//                      BIT per (row, chunk) and per-(2048-row segment, chunk) counts.
//   csc_scan_kernel  : per (sequence, head) scan of the counts -> col_nnz, col_offsets
//                      (int64) and per-segment start offsets; clears the unused tail of
//                      the row-list buffer.
//   csc_fill_kernel  : walks the bit columns in row order and writes each chunk's row list
//                      ascending, so no sort pass is needed afterwards.
//   csc_lists_kernel : the two in one launch, for calls with few counts per (sequence, head).
#include "gate_select.h"

#include <algorithm>
#include <mutex>

namespace fmoba {

constexpr int kGateRows = 128;   // query rows per workgroup (4 waves x 32)
constexpr int kSegRows = 2048;   // rows per counting segment (fewer for small problems, see csc_seg_rows)

struct TopkParams {
  fmoba_fused_topk_args a;
  uint32_t *sel;      // [heads][W][total_q] selection bits, word w covers chunks 32w..32w+31
  int32_t *segcnt;    // [batch][heads][nseg][max_cols], null if no lists are wanted
  int32_t W, nseg, max_cols, seg_rows;
  fmoba_csc_ranks ranks;       // all null: not wanted
  int32_t rows_in_x;           // the gate's grid, see gate_item
  int32_t sub_fwd, sub_bwd;    // key blocks of the attention's forward and backward (partials) per chunk
};

// Rows per counting segment.  A wave of the fill kernel walks one segment of one 32-chunk word column, 64 rows at a
// time, one step after the other, and a step is a chain (load the words, 32 ballots, a store per chunk) that only
// other waves can cover: segments of 2048 rows keep the counts small, but the fill wants many thousands of waves,
// so segments shrink (down to 256 rows, a multiple of the gate's 128-row blocks) until there are 16384 of them.  The
// headline batch (eight sequences, 65536 tokens) gets 512-row segments: fill 116 -> 63 us against 6272 waves of 2048
// rows (256-row segments: 56 us, but twice the counts to clear, scan and keep); a single sequence of 8192 tokens
// 86 -> 15 us against its 128 waves.  Beyond that the fill does not gain (262144 tokens: 131072 waves of 2048 rows
// 1.55 ms, twice as many of 1024 rows 1.62 ms and the scan of the counts four times as long).
static inline int csc_seg_rows(int64_t batch, int64_t heads, int64_t max_seqlen_q, int64_t W) {
  int seg_rows = kSegRows;
  const int64_t lq = max_seqlen_q > 0 ? max_seqlen_q : 1;
  while (seg_rows > 256 && batch * heads * W * ((lq + seg_rows - 1) / seg_rows) < 16384) seg_rows >>= 1;
  return seg_rows;
}

// The gates' workgroups, block of rows mb of query head h: grid (heads, blocks of rows, batch), from the last rows, which have the most
// chunks, to the first.  The heads of a row lie side by side in memory and start side by side, and an XCD (workgroup number mod 8) sees
// the chunk means of every eighth head only.  Against all blocks of a head, first to last: 32768 tokens, 32 heads 251 -> 229 us, 8192
// tokens, 16 heads 19.8 -> 17.2, 12037 tokens in five sequences 31.7 -> 27.5, 262144 tokens 2909 -> 2845.  More blocks of rows than the
// second dimension of a grid takes: (blocks of rows, heads, batch).
constexpr int kMaxGridY = 65535;
struct GateItem {
  int mb, h;
};
__device__ __forceinline__ GateItem gate_item(const TopkParams &p) {
  if (p.rows_in_x) return GateItem{(int)(gridDim.x - 1 - blockIdx.x), (int)blockIdx.y};
  return GateItem{(int)(gridDim.y - 1 - blockIdx.y), (int)blockIdx.x};
}

// PEEL: how a row's cut is found (kGatePeels)
template <typename T, int HD, bool PEEL, int NT>
__global__ __launch_bounds__(256, (NT == 8 || HD > 128) ? 2 : 4) void topk_gate_kernel(TopkParams p) {
  constexpr int KS = HD / 16;
  constexpr int VPR = HD / 8;    // 16-byte pieces of a row of chunk means
  constexpr int RPI = 64 / VPR;  // tile rows one load instruction brings (64 lanes x 16 bytes)
  constexpr int RB = HD * 2;     // bytes of a tile row: exactly HD elements, swizzled instead of padded
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int *sHist = reinterpret_cast<int *>(smem + (size_t)NT * 32 * RB);

  const fmoba_fused_topk_args &a = p.a;
  const GateItem item = gate_item(p);
  const int mb = item.mb, h = item.h, b = blockIdx.z;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int m0 = mb * kGateRows;
  if (m0 >= Lq) return;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int km0 = a.cu_seqlens_km[b];
  const int Cb = a.cu_seqlens_km[b + 1] - km0;
  const int off = Lk - Lq;
  const int B = a.chunk;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = lane >> 5;

  // chunks [0, nsc) can be candidates of some row of this block
  int nsc;
  if (a.is_causal) {
    const int rmax = min(m0 + kGateRows - 1, Lq - 1) + off;
    nsc = rmax < 0 ? 0 : min(Cb, rmax / B);
  } else {
    nsc = Cb;
  }
  nsc = min(nsc, min(p.max_cols, NT * 32));  // never beyond the LDS tile, whatever max_seqlen_k the caller gave
  const int n_tiles = (nsc + 31) >> 5;

  // The chunk means of this (sequence, kv head) go from global memory straight into LDS (global_load_lds, all loads
  // of a wave in flight at once): piece c of tile row r lies at piece c ^ tile_swz<HD>(r).  Rows past the last chunk
  // that can be a candidate and features past head_dim are fetched from a row / piece that exists: such scores are
  // masked below, such features meet zeros of q.
  const uint32_t ldsTile = (uint32_t)(uintptr_t)smem;
  if (nsc > 0) {
    const uint16_t *kmp = reinterpret_cast<const uint16_t *>(a.km) + (int64_t)hk * a.km_head_stride;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int ninstr = n_tiles * 32 / RPI;
    for (int v = wave_u; v < ninstr; v += 4) {
      const int c = v * RPI + lane / VPR, pc = lane % VPR;
      const int e = min((pc ^ tile_swz<HD>(c)) * 8, D - 8);
      global_to_lds16(kmp + (int64_t)(km0 + min(c, nsc - 1)) * a.km_row_stride + e, ldsTile + (uint32_t)v * 1024u);
    }
  }
  for (int v = tid; v < NT * 32; v += 256) sHist[v] = 0;

  // this lane's query row and its operand slices (contraction index permuted so that each
  // half-wave reads one contiguous half of the row)
  const int r = m0 + wave * 32 + (lane & 31);
  const bool valid = r < Lq;
  Pack8 qf[KS];
  {
    const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride;
    q_rows_load<HD>(qf, qp, a.q_row_stride, m0 + wave * 32, Lq, lane, D);
  }
  wait_all_loads();
  __syncthreads();
  q_rows_arrange<HD>(qf, hh, D);

  const int rp = r + off;
  int nc;  // number of candidate chunks of this row: chunks strictly before its own chunk
  if (a.is_causal)
    nc = (valid && rp >= 0) ? min(rp / B, Cb) : 0;
  else
    nc = valid ? Cb : 0;
  nc = min(nc, nsc);
  const int kp = a.is_causal ? a.topk - 1 : a.topk;
  const int own = a.is_causal && valid && rp >= 0 ? rp / B : -1;
  const int seg = m0 / p.seg_rows;
  uint32_t *selp = p.sel + (int64_t)h * p.W * a.total_q + q0 + r;
  gate_select<T, HD, NT, PEEL>(ldsTile, qf, lane, n_tiles, nc, kp, own, valid, p.W, [&](int t, uint32_t w) {
    if (valid && hh == 0) selp[(int64_t)t * a.total_q] = w;
    // per-chunk counts of this wave's 32 rows (both halves of the wave hold the rows' words)
    if (p.segcnt != nullptr && __any(w != 0u)) {
      const int mycnt = bit_column_count32(w, lane);
      if (lane < 32 && mycnt) atomicAdd(&sHist[t * 32 + lane], mycnt);
    }
  });
  __syncthreads();
  for (int c = tid; c < p.W * 32 && c < p.max_cols; c += 256) {
    const int v = sHist[c];
    if (v && p.segcnt != nullptr) atomicAdd(&p.segcnt[(((int64_t)b * a.heads + h) * p.nseg + seg) * p.max_cols + c], v);
  }
}

// ------------------------------------------------------------------------------------
// The same gate for sequences with more key chunks than one set of register tiles holds, and for few winners among more than 128.  Chunks are
// scored in groups of 64; every row keeps the K' best (score, chunk) pairs seen so far, and the next group competes against
// them.  The total order (score descending, chunk index descending) is strict, so the running winners after the last group are
// exactly the global top-K'.  PL places per lane, two lanes per row: 8, 16 or 32 for top-k up to 17, 33 and 64 (one more than the places
// where the own chunk takes no place).
//  * a row's winners stay in REGISTERS across the groups, sorted: the weaker half of its places in the lane with
//    chunks 0..3 of every eight, the stronger half in its partner.  A new winner is offered to the strong half, which
//    passes on what it gives up, and goes in with one pass of minimum / maximum: no compare, no choice between the lanes
//    (shares sorted per lane needed both: which lane holds the weakest was two exchanges and six selects per winner);
//  * the chunk means of the next group are fetched into the LDS tile while the current group is worked on;
//  * the scores of a group lie in LDS, a row of 64 floats, and a mask of 64 bits per row says which of them reach the row's
//    weakest winner ("entrants", two instructions per score): the row takes them from the lowest bit up.  (A list of entrants
//    with their chunks, built score by score, cost five instructions and two LDS stores per score.)
//  * the first group has no winners yet: a few probes find a score that at least K' and, as a rule, no more than K' + kGateSlack
//    of the group reach, and those are its entrants.  The order does the rest, ties and all.
// 262144 tokens, 16 heads, top-k 16 of 128-key chunks 3859 -> 2921 us; 1024-row parts of prompts with 9000 to 33000 keys, 32
// heads, top-k 8 51 -> 29 us (before: winners shared out by lane, lists of entrants, the whole cut of the first group searched).  Bound by
// the vector instructions (87 % of the clocks at 262144 tokens), most of them the pass of a new winner.  Above 16 winners: 126187 tokens, 16 heads, top-k
// 28 of 64-key chunks, gating and lists 9514 -> 2340 us, 54437 tokens, 32 heads, top-k 27 2603 -> 1007, 40000 tokens, 16 heads, top-k 50 1748 -> 846 (before:
// winners in two lists in LDS, an entrant looked for the weakest of all, one workgroup per compute unit).
// ------------------------------------------------------------------------------------
// A winner is ONE double between 1 and 2: order key of its score and chunk are 48 bits of its fraction, so that the order "score
// descending, chunk descending" is the order of the doubles and minimum / maximum are single instructions.
constexpr double kSlotFiller = INFINITY;  // place beyond the K'-th: above every winner
constexpr double kSlotEmpty = 0.5;        // place of a winner still to come: below every winner
constexpr uint32_t kNoEntrant = 0x3fd00000u;  // upper word of a double below kSlotEmpty

__device__ __forceinline__ double double_of(uint32_t hi, uint32_t lo) { return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo)); }
// the winner of a score and its chunk, or a double below all places
__device__ __forceinline__ double winner_word(float score, int chunk, bool has) {
  // (x + 0 turns -0 into +0: the order keys must agree with the float compares of the search)
  const uint32_t u = __float_as_uint(score + 0.f);
  const uint32_t key = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);  // (float_order_key, an instruction less)
  return double_of(has ? 0x3ff00000u | (key >> 16) : kNoEntrant, (key << 16) | (uint32_t)chunk);
}
__device__ __forceinline__ bool winner_real(double w) { return w >= 1.0 && w < (double)INFINITY; }
__device__ __forceinline__ uint32_t winner_key(double w) { return (uint32_t)((uint64_t)__double_as_longlong(w) >> 16); }
__device__ __forceinline__ int winner_chunk(double w) { return (int)((uint32_t)__double_as_longlong(w) & 0xffffu); }
// the lesser of two winners as one instruction (fmin first brings every operand that comes round a
// loop into canonical form, one more instruction per operand and turn; winners are never NaN)
__device__ __forceinline__ double min_winner(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  double d;
  asm("v_min_f64 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
  return d;
#else
  return a < b ? a : b;
#endif
}
__device__ __forceinline__ double max_winner(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  double d;
  asm("v_max_f64 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
  return d;
#else
  return a > b ? a : b;
#endif
}
// in lanes 0..31 the word of lane + 32, in the others +infinity
__device__ __forceinline__ double upper_half_or_inf(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
#if defined(__HIP_DEVICE_COMPILE__)
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, 0u, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), 0x7ff00000u, false, false);
  return double_of(hi[1], lo[1]);
#else
  return v;
#endif
}
// A winner word x goes up the ascending places w, all but the smallest of them and x stay: and while it goes up the last eight, the float at lds_addr is on
// its way, which is the result.  One statement from the request to the wait: the compiler waits for an LDS read of its own where it issues it when
// the address comes round a loop, and a register whose value has yet to arrive must not be one that it may copy or spill.  (Nothing
// else of the wave may be on its way from LDS.)
template <int PL>
__device__ __forceinline__ float insert_winner(double (&places)[PL], double x, uint32_t lds_addr) {
  float score;
#pragma unroll
  for (int j = 0; j < PL - 8; ++j) places[j] = min_winner(max_winner(places[j], x), places[j + 1]);
  double *w = places + PL - 8;
#if defined(__HIP_DEVICE_COMPILE__)
  double t;
  asm volatile("ds_read_b32 %0, %10\n\t"
               "v_max_f64 %9, %1, %11\n\t"
               "v_min_f64 %1, %9, %2\n\t"
               "v_max_f64 %9, %2, %11\n\t"
               "v_min_f64 %2, %9, %3\n\t"
               "v_max_f64 %9, %3, %11\n\t"
               "v_min_f64 %3, %9, %4\n\t"
               "v_max_f64 %9, %4, %11\n\t"
               "v_min_f64 %4, %9, %5\n\t"
               "v_max_f64 %9, %5, %11\n\t"
               "v_min_f64 %5, %9, %6\n\t"
               "v_max_f64 %9, %6, %11\n\t"
               "v_min_f64 %6, %9, %7\n\t"
               "v_max_f64 %9, %7, %11\n\t"
               "v_min_f64 %7, %9, %8\n\t"
               "v_max_f64 %8, %8, %11\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(score), "+&v"(w[0]), "+&v"(w[1]), "+&v"(w[2]), "+&v"(w[3]), "+&v"(w[4]), "+&v"(w[5]), "+&v"(w[6]), "+&v"(w[7]), "=&v"(t)
               : "v"(lds_addr), "v"(x)
               : "memory");
#else
  w[7] = x;
  score = (float)lds_addr;
#endif
  return score;
}

constexpr int kStreamGroup = 64;            // chunks per group: the bits of a row's mask
constexpr int kStreamRowBytes = 64 * 4 + 16;  // a row's scores in LDS (16 bytes more: eight rows apart in banks)
constexpr int kGateSlack = 3;               // (1, 3, 5 too many: 262144 tokens 2970, 2921, 2912 us, 32768 tokens 260, 250, 254)
template <int HD>
static constexpr size_t gate_stream_smem() {
  return (size_t)kStreamGroup * HD * 2 + (size_t)kGateRows * kStreamRowBytes;  // tile and scores; later the selection words of a pass
}
template <typename T, int HD, int PL>  // PL: winners' places per lane
__global__ __launch_bounds__(256, HD > 128 || PL > 16 ? 2 : 3) void topk_gate_stream_kernel(TopkParams p) {
  constexpr int KS = HD / 16;
  constexpr int GC = kStreamGroup, NT = GC / 32;
  constexpr int VPR = HD / 8;             // 16-byte pieces of a row of chunk means
  constexpr int RPI = 64 / VPR;           // tile rows one load instruction brings (64 lanes x 16 bytes)
  constexpr int NV = GC / RPI / 4;        // load instructions per wave and tile
  static_assert(NV >= 1 && NV * RPI * 4 == GC, "the four waves share a tile evenly");
  constexpr int RB = HD * 2;              // bytes of a tile row: exactly HD elements, swizzled instead of padded
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // after the last group the words and counts of WP word columns at a time: [WP][128], [WP][32]
  uint32_t *sSel = reinterpret_cast<uint32_t *>(smem);

  const fmoba_fused_topk_args &a = p.a;
  const GateItem item = gate_item(p);
  const int mb = item.mb, h = item.h, b = blockIdx.z;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int m0 = mb * kGateRows;
  if (m0 >= Lq) return;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int km0 = a.cu_seqlens_km[b];
  const int Cb = min(a.cu_seqlens_km[b + 1] - km0, p.max_cols);
  const int off = Lk - Lq;
  const int B = a.chunk;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = lane >> 5;
  const int rs = wave * 32 + (lane & 31);  // row slot inside the block

  int nsc;  // chunks [0, nsc) can be candidates of some row of this block
  if (a.is_causal) {
    const int rmax = min(m0 + kGateRows - 1, Lq - 1) + off;
    nsc = rmax < 0 ? 0 : min(Cb, rmax / B);
  } else {
    nsc = Cb;
  }
  const int ngroups = (nsc + GC - 1) / GC;

  const int r = m0 + rs;
  const bool valid = r < Lq;
  Pack8 qf[KS];
  {
    const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride;
    q_rows_load<HD>(qf, qp, a.q_row_stride, m0 + wave * 32, Lq, lane, D);
  }
  const int rp = r + off;
  int nc;  // candidate chunks of this row: chunks strictly before its own chunk
  if (a.is_causal)
    nc = (valid && rp >= 0) ? min(rp / B, Cb) : 0;
  else
    nc = valid ? Cb : 0;
  const int kp = a.is_causal ? a.topk - 1 : a.topk;

  const uint16_t *kmp = reinterpret_cast<const uint16_t *>(a.km) + (int64_t)hk * a.km_head_stride;
  // The chunk means of a group go from global memory straight into the LDS tile (global_load_lds: no registers hold
  // them on the way), every wave a quarter of the rows, issued as soon as the scores of the group before have been
  // formed and awaited at the top of the next group: the rest of a group's work runs under them.  Piece c of tile row
  // r lies at piece c ^ tile_swz<HD>(r).  Rows past the last chunk that can be a candidate and features past head_dim
  // are fetched from a row / piece that exists: such scores are masked, such features meet zeros of q.
  const uint32_t ldsTile = (uint32_t)(uintptr_t)smem;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto tile_issue = [&](int g) {
    const int c0 = g * GC, gsc = min(GC, nsc - c0);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = (wave_u * NV + v) * RPI + lane / VPR, pc = lane % VPR;
      const int e = min((pc ^ tile_swz<HD>(c)) * 8, D - 8);
      global_to_lds16(kmp + (int64_t)(km0 + c0 + min(c, gsc - 1)) * a.km_row_stride + e, ldsTile + (uint32_t)((wave_u * NV + v) * 1024));
    }
  };
  // this lane's operand row of a 32-chunk tile: row lane % 32, pieces hh * KS ..
  const uint32_t a_row = ldsTile + (uint32_t)((lane & 31) * RB);
  const int a_swz = tile_swz<HD>(lane & 31);
  static_assert(PL % 8 == 0, "insert_winner");
  double win[PL];  // places hh * PL .. of the row's winners, ascending
#pragma unroll
  for (int j = 0; j < PL; ++j) win[j] = hh * PL + j < kp ? kSlotEmpty : kSlotFiller;
  const uint32_t row_b = ldsTile + (uint32_t)(GC * RB + rs * kStreamRowBytes);  // the row's scores

  if (ngroups > 0) tile_issue(0);
  q_rows_arrange<HD>(qf, hh, D);
#pragma nounroll
  for (int g = 0; g < ngroups; ++g) {
    const int c0 = g * GC;
    const int gsc = min(GC, nsc - c0);
    const int n_tiles = (gsc + 31) >> 5;
    wait_all_loads();
    __syncthreads();  // this group's tile is in LDS

    // this group's scores; chunks that are no candidates of the row (its own chunk and later ones) count as -inf
    float sc[NT][16];
    const bool all_cand = __all(nc >= c0 + GC);
    {
      // The tiles of the group side by side, and the operands of contraction step ks + 1 on their way from LDS while
      // the products of step ks run: one tile after the other, every read awaited by its product, a wave spent a
      // group's worth of LDS latencies in a single chain.  (A tile past the group's last chunk holds copies of
      // chunks that exist, see tile_issue; its scores are masked like those of every chunk that is no candidate.)
      f32x16 acc[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
      auto operand = [&](int t, int ks) { return lds_read16(a_row + (uint32_t)(t * 32 * RB) + (uint32_t)(((hh * KS + ks) ^ a_swz) * 16)); };
      Pack8 af[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) af[t] = operand(t, 0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        Pack8 nx[NT];
        if (ks + 1 < KS) {
#pragma unroll
          for (int t = 0; t < NT; ++t) nx[t] = operand(t, ks + 1);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = mfma32<T>(af[t], qf[ks], acc[t]);
        if (ks + 1 < KS) {
#pragma unroll
          for (int t = 0; t < NT; ++t) af[t] = nx[t];
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (all_cand) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[t][i] = acc[t][i];
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[t][i] = (c0 + t * 32 + acc_row(i, hh) < nc) ? acc[t][i] : -INFINITY;
        }
      }
    }
    __syncthreads();  // everyone has read the tile: the next group's chunk means may land in it
    if (g + 1 < ngroups) tile_issue(g + 1);

    // scores from `bound` on are the group's entrants
    float bound;
    if (g == 0) {
      // No winners yet: bisection between the smallest and the largest score (as in topk_gate_kernel: first the range of values,
      // then the range of order keys) until no more than kGateSlack scores too many lie above the lower end.  The lower end
      // always has at least K' above it, or all there are; scores of minus infinity and NaN are never among them.
      float vmin = INFINITY, vmax = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          vmin = fminf(vmin, sc[t][i] == -INFINITY ? INFINITY : sc[t][i]);  // (no candidates, or never chosen)
          vmax = fmaxf(vmax, sc[t][i]);
        }
      vmin = min_xor32_f(vmin);
      vmax = max_xor32_f(vmax);
      const int ntot = max(0, min(nc - c0, GC));
      bool open = ntot > kp + kGateSlack && kp > 0 && vmin < vmax;
      const uint32_t lowest = float_order_key(-INFINITY);
      uint32_t lo_k = open ? max(float_order_key(vmin) - 1u, lowest) : lowest;
      if (lo_k == 0x7fffffffu) lo_k -= 1u;  // (-0 is not below a vmin of +0)
      uint32_t hi_k = float_order_key(vmax);
#pragma nounroll
      for (int iter = 0;; ++iter) {
        open = open && hi_k - lo_k > 1u;
        if (!__any(open)) break;
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
#pragma unroll
          for (int i = 0; i < 16; i += 4) cnt = count4_gt(cnt, sc[t][i], sc[t][i + 1], sc[t][i + 2], sc[t][i + 3], probe);
        cnt = sum_xor32_i(cnt);
        if (open) {
          if (cnt >= kp) {
            lo_k = pk;
            open = cnt > kp + kGateSlack;
          } else {
            hi_k = pk;
          }
        }
      }
      // (the next float above lo, which after -0 is the smallest positive number)
      bound = kp > 0 ? order_key_float(lo_k + (lo_k == 0x7fffffffu ? 2u : 1u)) : INFINITY;
    } else {
      // Scores that reach the row's weakest winner (a new chunk has a higher index than every earlier one, so an equal score
      // wins the tie); every finite score while places are empty; none if the row keeps none
      double weakest = win[0];
      {
        const uint64_t u = (uint64_t)__double_as_longlong(weakest);
        weakest = double_of(swap32((uint32_t)(u >> 32)).a, swap32((uint32_t)u).a);
      }
      bound = winner_real(weakest) ? order_key_float(winner_key(weakest)) : weakest < 1.0 ? order_key_float(float_order_key(-INFINITY) + 1u) : INFINITY;
    }

    // the scores to LDS, the row's mask of entrants (both lanes of the row hold it)
    uint64_t mask = 0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint32_t m16 = 0u;
#pragma unroll
      for (int i4 = 3; i4 >= 0; --i4) {
        const Flags4 f = flags4_ge(sc[t][4 * i4 + 3], sc[t][4 * i4 + 2], sc[t][4 * i4 + 1], sc[t][4 * i4], bound);
#pragma unroll
        for (int j = 0; j < 4; ++j) m16 = shift_in_flag(m16, f.m[j]);
        const f32x4 quad = {sc[t][4 * i4], sc[t][4 * i4 + 1], sc[t][4 * i4 + 2], sc[t][4 * i4 + 3]};
        lds_write_vec<f32x4>(row_b + (uint32_t)((t * 32 + 8 * i4) * 4 + 16 * hh), quad);
      }
      // the four nibbles of the flags move to the places of the lane's chunks (4 hh + 8 g .. + 3)
      const uint32_t w = ((m16 & 0xfu) | ((m16 & 0xf0u) << 4) | ((m16 & 0xf00u) << 8) | ((m16 & 0xf000u) << 12)) << (4 * hh);
      const UPair wp = swap32(w);
      mask |= (uint64_t)(wp.a | wp.b) << (32 * t);
    }
    wave_lds_fence();

    auto stream = [&](auto two) {
      // (entrant e + 1 is on its way from LDS while entrant e goes up the winners)
      auto next_bit = [&]() { return (int)__builtin_ctzll(mask | (1ull << 63)); };
      int xc = next_bit();
      bool has = mask != 0;
      float xv = lds_read_vec<float>(row_b + 4u * (uint32_t)xc);
      mask &= mask - 1;
#pragma nounroll
      while (__any(has)) {
        double x = winner_word(xv, c0 + xc, has);
        has = mask != 0;
        xc = next_bit();
        mask &= mask - 1;
        if constexpr (decltype(two)::value) x = min_winner(x, upper_half_or_inf(win[0]));  // what the strong half does not keep
        xv = insert_winner(win, x, row_b + 4u * (uint32_t)xc);
      }
    };
    // (up to eight winners have their places in the weak half alone; 16 and 32 places per lane serve more winners than that)
    if (PL == 8 && kp <= PL)
      stream(std::integral_constant<bool, false>{});
    else
      stream(std::integral_constant<bool, true>{});
    wave_lds_fence();  // (the row takes the next group's scores)
  }
  __syncthreads();

  // selection words and per-chunk counts of the block, assembled in LDS and written out in passes of WP word columns
  // (what the tile and the lists hold), so that a sequence may have any number of chunks
  constexpr int kPassWords = (int)(gate_stream_smem<HD>() / ((kGateRows + 32) * 4));
  const int WP = min(p.W, kPassWords);
  int *sHist = reinterpret_cast<int *>(sSel + WP * kGateRows);
  const int seg = m0 / p.seg_rows;
  for (int w0 = 0; w0 < p.W; w0 += WP) {
    const int wn = min(WP, p.W - w0);
    __syncthreads();  // the pass before has been written out
    for (int v = tid; v < wn * kGateRows; v += 256) sSel[v] = 0u;
    for (int c = tid; c < wn * 32; c += 256) sHist[c] = 0;
    __syncthreads();
    if (valid) {
#pragma unroll
      for (int j = 0; j < PL; ++j) {
        if (winner_real(win[j])) {
          const int c = winner_chunk(win[j]);
          const int cw = (c >> 5) - w0;
          if ((uint32_t)cw < (uint32_t)wn) {
            atomicOr(&sSel[cw * kGateRows + rs], 1u << (c & 31));
            atomicAdd(&sHist[c - 32 * w0], 1);
          }
        }
      }
      if (hh == 0 && a.is_causal && rp >= 0) {
        const int c = rp / B;  // the own chunk is always selected
        const int cw = (c >> 5) - w0;
        if (c < p.max_cols && (uint32_t)cw < (uint32_t)wn) {
          atomicOr(&sSel[cw * kGateRows + rs], 1u << (c & 31));
          atomicAdd(&sHist[c - 32 * w0], 1);
        }
      }
    }
    __syncthreads();
    for (int v = tid; v < wn * kGateRows; v += 256) {
      const int t = v / kGateRows, slot_r = v - t * kGateRows;
      if (m0 + slot_r < Lq) p.sel[((int64_t)h * p.W + w0 + t) * a.total_q + q0 + m0 + slot_r] = sSel[v];
    }
    for (int c = tid; c < wn * 32; c += 256) {
      const int v = sHist[c];
      if (v && p.segcnt != nullptr) atomicAdd(&p.segcnt[(((int64_t)b * a.heads + h) * p.nseg + seg) * p.max_cols + 32 * w0 + c], v);
    }
  }
}

// ------------------------------------------------------------------------------------
// The gate for calls with at most eight query rows per sequence (decode steps).  The kernels above give a row to a pair
// of lanes and let four waves work on 128 rows; with one row three of the waves and 63 of 64 lanes idle through a chain of
// LDS reads, products and a dozen probes (20 us for 16 requests of up to 256 chunks, 32 heads).  Here the eight waves share the
// chunks (their means straight from memory as the A operand: nothing is read twice), the scores of the few rows meet in
// LDS, and a whole wave searches the cut of a row: a chunk per lane and register, a count is a ballot.  The products are
// the same as above, so are the scores, and the order (score descending, chunk descending) is total: the same selection.
// 20 -> 13.6 us there.
// ------------------------------------------------------------------------------------
// NJ: chunks per lane of a row's wave
template <typename T, int HD, int NJ>
__global__ __launch_bounds__(512) void topk_gate_few_kernel(TopkParams p) {
  constexpr int KS = HD / 16;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float *sScore = reinterpret_cast<float *>(smem);  // [rows][NJ * 64]
  const fmoba_fused_topk_args &a = p.a;
  const int h = blockIdx.x, b = blockIdx.y;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = min(a.cu_seqlens_q[b + 1] - q0, a.max_seqlen_q);  // (at most kFewRows)
  if (Lq <= 0) return;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int km0 = a.cu_seqlens_km[b];
  const int Cb = min(min(a.cu_seqlens_km[b + 1] - km0, p.max_cols), NJ * 64);
  const int off = Lk - (a.cu_seqlens_q[b + 1] - q0);
  const int B = a.chunk, D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  int nsc = Cb;  // chunks that are candidates of the last row
  if (a.is_causal) {
    const int rmax = Lq - 1 + off;
    nsc = rmax < 0 ? 0 : min(Cb, rmax / B);
  }
  const int r = lane & 31;
  Pack8 qf[KS];
  {
    const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)(q0 + min(r, Lq - 1)) * a.q_row_stride + (int64_t)h * a.q_head_stride;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int e = (hh * KS + ks) * 8;
      qf[ks] = (r < Lq && e < D) ? ld_global16(qp + e) : zero_pack8();
    }
  }
  const uint16_t *kmp = reinterpret_cast<const uint16_t *>(a.km) + (int64_t)km0 * a.km_row_stride + (int64_t)hk * a.km_head_stride;
  for (int t = wave; t * 32 < nsc; t += 8) {
    const uint16_t *row = kmp + (int64_t)min(t * 32 + (lane & 31), nsc - 1) * a.km_row_stride;
    Pack8 af[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) af[ks] = ld_global16(row + min((hh * KS + ks) * 8, D - 8));
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = mfma32<T>(af[ks], qf[ks], s);
    if (r < Lq) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4 *>(sScore + r * (NJ * 64) + t * 32 + 8 * g + 4 * hh) = f32x4{s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
    }
  }
  __syncthreads();
  if (wave >= Lq) return;
  {
    const int row = wave, rp = row + off;
    const bool self = a.is_causal && rp >= 0;
    const int nc = a.is_causal ? (rp >= 0 ? min(min(rp / B, Cb), nsc) : 0) : Cb;
    const int kp = a.is_causal ? a.topk - 1 : a.topk;
    const int pself = self ? rp / B : -1;
    // keys in the order of the scores; 0: no candidate, or a score that no cut lies below (-inf, not a number)
    uint32_t key[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c = j * 64 + lane;
      key[j] = 0u;
      if (j * 64 < nc) {
        const float x = sScore[row * (NJ * 64) + c] + 0.f;  // (-0 is +0)
        key[j] = (c < nc && x > -INFINITY) ? float_order_key(x) : 0u;
      }
    }
    auto count_ge = [&](uint32_t v) {
      int n = 0;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (j * 64 < nc) n += __popcll(__ballot(key[j] >= v));
      return n;
    };
    // the largest cut with at least K' keys at or above it (1: all of them, if there are no more than K')
    uint32_t cut = 1u;
    if (kp > 0 && count_ge(1u) > kp) {
      cut = 0u;
      for (int bit = 31; bit >= 0; --bit) {
        const uint32_t trial = cut | (1u << bit);
        if (count_ge(trial) >= kp) cut = trial;
      }
    }
    int spare = kp - (cut == 0xffffffffu ? 0 : count_ge(cut + 1u));  // places left for the keys equal to the cut: the highest chunks
    uint32_t w_lo = 0u, w_hi = 0u;                                  // lane w: words w and 64 + w of the row
#pragma unroll
    for (int j = NJ - 1; j >= 0; --j) {
      if (j * 64 >= p.max_cols) continue;
      unsigned long long m = 0ull;
      if (kp > 0 && j * 64 < nc) {
        m = __ballot(key[j] > cut);
        unsigned long long eq = __ballot(key[j] == cut);
        int n = __popcll(eq);
        while (n > spare) {
          eq &= eq - 1ull;  // the lowest chunk goes
          --n;
        }
        spare -= n;
        m |= eq;
      }
      if (self && (pself >> 6) == j) m |= 1ull << (pself & 63);
      if (p.segcnt != nullptr && ((m >> lane) & 1ull) && j * 64 + lane < p.max_cols)
        atomicAdd(&p.segcnt[((int64_t)b * a.heads + h) * p.nseg * p.max_cols + j * 64 + lane], 1);
      const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
      uint32_t &w = j < 32 ? w_lo : w_hi;
      const int at = (2 * j) & 63;
      w = lane == at ? lo : lane == at + 1 ? hi : w;
    }
    uint32_t *selp = p.sel + (int64_t)h * p.W * a.total_q + q0 + row;
    if (lane < p.W) selp[(int64_t)lane * a.total_q] = w_lo;
    if (64 + lane < p.W) selp[(int64_t)(64 + lane) * a.total_q] = w_hi;
  }
}

// How many chunks a row selected below each word of its selection (PREFIX), and its visits, for rows first, first + step, .. of `rows` rows of sequence b from `row0` on;
// with them, shared out among `nblk` blocks, the rows before the first sequence and after the last one (a buffer longer than its batch), which have no visits:
// the combine kernels look at every row.
template <bool PREFIX>
__device__ __forceinline__ void rank_rows(const TopkParams &p, int h, int b, int blk, int nblk, int row0, int rows) {
  const fmoba_fused_topk_args &a = p.a;
  constexpr int nthr = 256;
  const int tid = threadIdx.x;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b], last = (Lk + a.chunk - 1) / a.chunk - 1;  // the sequence's last chunk
  {
    uint32_t *vh = p.ranks.visits + (int64_t)h * a.total_q;
    const int64_t first = (int64_t)blk * nthr + tid, step = (int64_t)nblk * nthr;
    if (b == 0)
      for (int64_t i = first; i < q0; i += step) vh[i] = 0u;
    if (b == a.batch - 1)
      for (int64_t i = (int64_t)q0 + Lq + first; i < a.total_q; i += step) vh[i] = 0u;
  }
  for (int k = 0; k < rows; k += nthr) {
    const int r = row0 + k + tid;
    if (r >= Lq) return;
    const int rp = r + Lk - Lq, own = rp >= 0 ? rp / a.chunk : -1;
    const int nw = a.is_causal ? (own < 0 ? 0 : min(p.W, (own >> 5) + 1)) : p.W;
    const uint32_t *words = p.sel + (int64_t)h * p.W * a.total_q + q0 + r;
    uint8_t *pre = PREFIX ? p.ranks.prefix + (int64_t)h * p.W * a.total_q + q0 + r : nullptr;
    int n = 0, has_last = 0;
    for (int w0 = 0; w0 < nw; w0 += 8) {
      uint32_t x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = w0 + i < nw ? words[(int64_t)(w0 + i) * a.total_q] : 0u;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (PREFIX && w0 + i > 0 && w0 + i < nw) pre[(int64_t)(w0 + i) * a.total_q] = (uint8_t)n;
        n += __popc(x[i]);
        if (w0 + i == (last >> 5)) has_last = (x[i] >> (last & 31)) & 1;
      }
    }
    // Forward: all key blocks of a selected chunk that exist.  Backward: under the causal rule those of the row's own chunk, its
    // last one, that begin at or before the row.
    auto blocks = [&](int sub, int keys) {
      const int kb = a.chunk / sub;
      return (keys + kb - 1) / kb;
    };
    const int nf = n * p.sub_fwd - has_last * (p.sub_fwd - blocks(p.sub_fwd, Lk - last * a.chunk));
    const int nb = n == 0         ? 0
                   : a.is_causal ? (n - 1) * p.sub_bwd + blocks(p.sub_bwd, rp - own * a.chunk + 1)
                                 : n * p.sub_bwd - has_last * (p.sub_bwd - blocks(p.sub_bwd, Lk - last * a.chunk));
    p.ranks.visits[(int64_t)h * a.total_q + q0 + r] = (uint32_t)nf | ((uint32_t)nb << 16);
  }
}

// grid (heads, batch, 1 + blocks of kRankRows rows if ranks are wanted), block 256.
// RANKS: with the blocks of the ranks, a kernel of its own: in one with both, the scan of plain lists was 4073 instructions with 36 scalars
// spilled, 571 and none without (8192 tokens, 16 heads 5.4 -> 4.9 us, 32768 tokens, 32 heads 13.3 -> 12.6).  The ranks' loops stay
// unrolled, spilled scalars and all: rolled up they keep fewer loads in flight (262144 tokens 254 -> 264 us).
constexpr int kRankRows = 1024;
template <bool RANKS>
__global__ __launch_bounds__(256) void csc_scan_kernel(TopkParams p) {
  const fmoba_fused_topk_args &a = p.a;
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  // (independent of the scan, whose few workgroups mostly wait: scan without and with the ranks, 8192 tokens, 16 heads 6.0 and 6.8 us; 262144 tokens 122 and
  // 250 us)
  if (RANKS && blockIdx.z > 0) {
    rank_rows<true>(p, h, b, blockIdx.z - 1, gridDim.z - 1, (int)(blockIdx.z - 1) * kRankRows, kRankRows);
    return;
  }
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int nseg_b = (Lq + p.seg_rows - 1) / p.seg_rows;
  const int64_t bh = (int64_t)b * a.heads + h;
  int32_t *segc = p.segcnt + bh * p.nseg * p.max_cols;
  const int64_t base = ((int64_t)q0 * a.heads + (int64_t)Lq * h) * a.topk;
  __shared__ int sscan[256];
  __shared__ int64_t stotal;
  if (tid == 0) stotal = 0;
  __syncthreads();
  for (int c0 = 0; c0 < p.max_cols; c0 += 256) {
    const int c = c0 + tid;
    int nnz = 0;
    if (c < p.max_cols) {
      // eight counts in flight at a time (a long sequence has over a hundred segments, and a load that waits for
      // the store before it costs a round trip each)
      for (int s0 = 0; s0 < nseg_b; s0 += 8) {
        int v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = s0 + i < nseg_b ? segc[(int64_t)(s0 + i) * p.max_cols + c] : 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (s0 + i < nseg_b) segc[(int64_t)(s0 + i) * p.max_cols + c] = nnz;
          nnz += v[i];
        }
      }
    }
    sscan[tid] = nnz;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int v = (tid >= d) ? sscan[tid - d] : 0;
      __syncthreads();
      sscan[tid] += v;
      __syncthreads();
    }
    const int64_t run = stotal;
    if (c < p.max_cols) {
      a.col_nnz[bh * p.max_cols + c] = nnz;
      a.col_offsets[bh * p.max_cols + c] = base + run + (int64_t)(sscan[tid] - nnz);
    }
    __syncthreads();
    if (tid == 255) stotal = run + sscan[255];
    __syncthreads();
  }
  // slots of this (sequence, head) region that no list uses stay 0
  const int64_t start = base + stotal, end = base + (int64_t)Lq * a.topk;
  for (int64_t i = start + tid; i < end; i += 256) a.flat_indices[i] = 0;
}

// x with the value of lane `lane` (the same in every lane) replaced by v (the same in every lane)
template <int LANE>
__device__ __forceinline__ uint32_t write_lane(uint32_t x, uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_writelane_b32 %0, %1, %2" : "+v"(x) : "s"(v), "n"(LANE));
#else
  (void)v;
#endif
  return x;
}
// base[byte_offset] = value in the lanes of `lanes`, all others do nothing (base: the same in every lane)
__device__ __forceinline__ void store_i32_in_lanes(int32_t *base, uint32_t byte_offset, int value, unsigned long long lanes) {
#if defined(__HIP_DEVICE_COMPILE__)
  unsigned long long saved;
  asm volatile("s_mov_b64 %0, exec\n\t"
               "s_mov_b64 exec, %1\n\t"
               "global_store_dword %2, %3, %4\n\t"
               "s_mov_b64 exec, %0"
               : "=&s"(saved)
               : "s"(lanes), "v"(byte_offset), "v"(value), "s"(base)
               : "memory");
#else
  (void)base, (void)byte_offset, (void)value, (void)lanes;
#endif
}

// n + 1 in the lanes of `lanes`
__device__ __forceinline__ uint32_t count_lanes(uint32_t n, unsigned long long lanes) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_addc_co_u32_e64 %0, vcc, 0, %0, %1" : "+v"(n) : "s"(lanes) : "vcc");
#else
  (void)lanes;
#endif
  return n;
}

// Rows r (lane by lane) with words w of a word column: every row goes to the lists of the chunks it selected.  rel: lane j's is the place of the
// next row of chunk j, counted from `lists`.
template <bool RANKED>
__device__ __forceinline__ void fill_step(int32_t *lists, uint32_t &rel, int r, uint32_t w, uint32_t nth) {
  // the chunks that some row of the step selects (a scalar, so that the others cost no vector instruction)
  const uint32_t present = __builtin_amdgcn_readfirstlane(__ockl_wfred_or_u32(w));
  if (present == 0u) return;
  static_for<32>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if (present & (1u << j)) {
      const unsigned long long m = __ballot((w & (1u << j)) != 0u);
      const uint32_t at = __builtin_amdgcn_readlane(rel, j);
      const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      if constexpr (RANKED) {
        store_i32_in_lanes(lists, (at + rank) << 2, (int)((nth << kListRowBits) | (uint32_t)r), m);
        nth = count_lanes(nth, m);
      } else {
        store_i32_in_lanes(lists, (at + rank) << 2, r, m);
      }
      rel = write_lane<j>(rel, at + (uint32_t)__popcll(m));
    }
  });
}

// grid (nseg * W, heads, batch), block 64: one wave walks the rows of one segment of one 32-chunk word column
// RANKED: with every row id its chunk's place among the chunks of the row, in the bits from kListRowBits on (in an array of their own,
// a byte per entry, the ranks cost a second store per chunk and step: 262144 tokens 789 -> 1723 us, 874 this way)
template <bool RANKED>
__global__ __launch_bounds__(64) void csc_fill_kernel(TopkParams p) {
  const fmoba_fused_topk_args &a = p.a;
  // consecutive workgroups: consecutive segments of one word column, i.e. consecutive memory.  (With the word column
  // as the fast index the waves that run at the same time read addresses a whole word column apart -- total_q words,
  // a power of two more often than not -- and meet in the same memory channel.)
  const int wc = blockIdx.x / p.nseg, seg = blockIdx.x - wc * p.nseg;
  const int h = blockIdx.y, b = blockIdx.z, lane = threadIdx.x;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int r0 = seg * p.seg_rows;
  if (r0 >= Lq) return;
  const int r1 = min(Lq, r0 + p.seg_rows);
  // with the causal rule a row selects no chunk beyond its own: the rows before the word column's first chunk hold zeros
  int rb0 = r0;
  if (a.is_causal) {
    const int64_t off = (int64_t)(a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b]) - Lq;
    const int64_t first_row = (int64_t)wc * 32 * a.chunk - off;
    if (first_row >= r1) return;
    if (first_row > r0) rb0 = r0 + (int)((first_row - r0) / 64 * 64);
  }
  const int64_t bh = (int64_t)b * a.heads + h;
  // Where the next rows of chunk wc * 32 + j go: lane j keeps the position relative to the start of the word column's
  // first list (the 32 lists follow each other, far less than 2^30 entries), the start itself is a scalar.  A step
  // costs vector instructions and nothing else (the vector pipes are busy 85 % of the kernel's time), so a chunk that
  // some row of the step selects takes five: the lane's rank among the rows (mbcnt), the slot, the store in the lanes
  // of the ballot (the ballot itself is the exec mask), and the new position written back into lane j.
  const int64_t first = a.col_offsets[bh * p.max_cols + wc * 32];
  int32_t *const lists = a.flat_indices + first;
  uint32_t rel = 0u;
  {
    const int c = wc * 32 + lane;
    if (lane < 32 && c < p.max_cols)
      rel = (uint32_t)(a.col_offsets[bh * p.max_cols + c] - first) + (uint32_t)p.segcnt[(bh * p.nseg + seg) * p.max_cols + c];
  }
  const uint32_t *words = p.sel + ((int64_t)h * p.W + wc) * a.total_q + q0;
  const uint8_t *pre = RANKED ? p.ranks.prefix + ((int64_t)h * p.W + wc) * a.total_q + q0 : nullptr;
  for (int rb = rb0; rb < r1; rb += 64) {
    const int r = rb + lane;
    const uint32_t w = (r < r1) ? words[r] : 0u;
    const uint32_t nth = RANKED && wc > 0 && r < r1 ? pre[r] : 0u;  // chunks that the row selected so far
    fill_step<RANKED>(lists, rel, r, w, nth);
  }
}

// Scan and fill in one launch, for calls with few counts per (sequence, head): every workgroup adds up the counts it needs itself (no more than kListCounts of them,
// each wave a quarter, all loads in flight at once), a segment's rows are asked for together with them, and with ranks the chunks of a row below the word column are
// counted from its words, of which there are few.  grid (nseg * W, + nseg for the visits if ranks are wanted; heads, batch), a wave for each 64 rows of a segment.
// What bounds it is a chain: launch, counts, 32 ballots and stores.  The scan before it was a launch and a chain of its own whose few workgroups left the chip
// empty, and one wave per segment walks four times as far: 8192 tokens, 16 heads, ranked lists of 128-key chunks, scan and fill 17.6 us, one wave per segment
// 15.1, this 10.0 (four waves of eight chunks each, which read the words below four times: 10.9, and 23 where this takes 19); parts of prompts of 1024 rows
// against 9000 to 33000 keys, 32 heads 22.0 -> 19.4; 8191 tokens of short documents, plain lists 10.7 -> 4.8.  More counts, or longer segments (which calls of
// many waves have), go to the two launches: there the scan is a small part of the time and the counts of a workgroup would be a large one.  So do calls of many
// workgroups, each of which counts for itself, earlier where ranks are made beside the lists: ranked, 9856 of them 28.2 us against 21.4 and 5120 of them 22.7
// against 18.7, while 3840 win (above); plain, 4800 of them (12037 tokens, 16 heads) 11.8 against 18.0, and 11200 (24571 tokens, 32 heads) as long as the two
// launches.
constexpr int kListCounts = 4096, kListWords = 16, kListSegRows = 256, kListGroups = 8192, kListRankedGroups = 4096;
template <bool RANKED>
__global__ __launch_bounds__(256) void csc_lists_kernel(TopkParams p) {
  const fmoba_fused_topk_args &a = p.a;
  __shared__ int sBefore[4], sAll[4][32], sMine[4][32], sStep[4][32];
  const int h = blockIdx.y, b = blockIdx.z, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31;
  if (RANKED && (int)blockIdx.x >= p.nseg * p.W) {
    const int blk = blockIdx.x - p.nseg * p.W;
    rank_rows<false>(p, h, b, blk, p.nseg, blk * p.seg_rows, p.seg_rows);
    return;
  }
  const int wc = blockIdx.x / p.nseg, seg = blockIdx.x - wc * p.nseg;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int r0 = seg * kListSegRows;
  if (r0 >= Lq && seg > 0) return;
  const int r1 = min(Lq, r0 + kListSegRows), nseg_b = (Lq + kListSegRows - 1) / kListSegRows;
  // with the causal rule a row selects no chunk beyond its own: the rows before the word column's first chunk hold zeros
  bool rows = r0 < r1;
  if (a.is_causal) rows = rows && (int64_t)wc * 32 * a.chunk - ((int64_t)(a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b]) - Lq) < r1;
  // (the first segment's workgroup tells where the lists of its word column are, those of the last word column clear what no list uses)
  if (!rows && seg > 0 && wc < p.W - 1) return;
  const int64_t bh = (int64_t)b * a.heads + h;
  const int32_t *cnt = p.segcnt + bh * p.nseg * p.max_cols;
  const int cols = p.max_cols, c = wc * 32 + j;
  const int r = r0 + wave * 64 + lane;
  const uint32_t *below = p.sel + (int64_t)h * p.W * a.total_q + q0 + r;
  const uint32_t w = rows && r < r1 ? below[(int64_t)wc * a.total_q] : 0u;
  uint32_t nth = 0u;
  if constexpr (RANKED) {
    for (int v0 = 0; v0 < (rows ? wc : 0); v0 += 8) {
      uint32_t x[8];
#pragma unroll
      for (int v = 0; v < 8; ++v) x[v] = v0 + v < wc && r < r1 ? below[(int64_t)(v0 + v) * a.total_q] : 0u;
#pragma unroll
      for (int v = 0; v < 8; ++v) nth += __popc(x[v]);
    }
  }
  // counts of this column (lanes j and 32 + j: column j, two segments at a time), all of them and those of the segments before this one; and of the columns
  // before the word column
  int before = 0, all = 0, mine = 0;
  for (int s0 = 0; s0 < nseg_b; s0 += 32) {
    int y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = s0 + 8 * i + 2 * wave + (lane >> 5);
      y[i] = c < cols && s < nseg_b ? cnt[s * cols + c] : 0;
    }
    for (int c0 = lane; c0 < wc * 32; c0 += 128) {
      int x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int s = s0 + 4 * (i >> 1) + wave, c1 = c0 + 64 * (i & 1);
        x[i] = c1 < wc * 32 && s < nseg_b ? cnt[s * cols + c1] : 0;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) before += x[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      all += y[i];
      mine += s0 + 8 * i + 2 * wave + (lane >> 5) < seg ? y[i] : 0;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o, 64);
  all = sum_xor32_i(all);
  mine = sum_xor32_i(mine);
  const int step = sum_xor32_i(bit_column_count32(w, lane));  // rows of this wave in column j
  if (lane < 32) sAll[wave][lane] = all, sMine[wave][lane] = mine, sStep[wave][lane] = step;
  if (lane == 0) sBefore[wave] = before;
  __syncthreads();
  before = __builtin_amdgcn_readfirstlane((sBefore[0] + sBefore[1]) + (sBefore[2] + sBefore[3]));
  all = (sAll[0][j] + sAll[1][j]) + (sAll[2][j] + sAll[3][j]);
  mine = (sMine[0][j] + sMine[1][j]) + (sMine[2][j] + sMine[3][j]);
#pragma unroll
  for (int i = 0; i < 3; ++i) mine += i < wave ? sStep[i][j] : 0;
  int incl = all;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const int up = __shfl_up(incl, o, 32);
    incl += j >= o ? up : 0;
  }
  const int64_t base = ((int64_t)q0 * a.heads + (int64_t)Lq * h) * a.topk;
  if (seg == 0 && threadIdx.x < 32 && c < cols) {
    a.col_nnz[bh * cols + c] = all;
    a.col_offsets[bh * cols + c] = base + before + incl - all;
  }
  if (wc == p.W - 1) {
    const int64_t end = base + (int64_t)Lq * a.topk;
    for (int64_t i = base + before + __builtin_amdgcn_readlane(incl, 31) + seg * 256 + threadIdx.x; i < end; i += nseg_b * 256) a.flat_indices[i] = 0;
  }
  uint32_t rel = (uint32_t)(incl - all + mine);
  if (rows) fill_step<RANKED>(a.flat_indices + base + before, rel, r, w, nth);
}

// ------------------------------------------------------------------------------------
// ordered per-row lists (indices / values), only produced on request: one wave per
// (row, head).  The SET of chunks is the gate's own (its selection bits: the lists name
// exactly the chunks whose columns hold the row, also where two scores are so close that
// another summation order would rank them the other way round); the scores that order the
// set are plain FMA sums, then rounds of wave-wide arg-max under the total order (score
// desc, chunk desc).
// ------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(64) void topk_raw_kernel(fmoba_fused_topk_args a, int kr, const uint32_t *sel, int W) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float *sScore = reinterpret_cast<float *>(smem);  // [Cpad]
  const int row_g = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  // locate the sequence of this row
  int b = 0;
  while (b + 1 < a.batch && a.cu_seqlens_q[b + 1] <= row_g) ++b;
  const int q0 = a.cu_seqlens_q[b];
  const int Lq = a.cu_seqlens_q[b + 1] - q0;
  const int r = row_g - q0;
  int32_t *oi = a.raw_indices + ((int64_t)row_g * a.heads + h) * kr;
  float *ov = a.raw_values + ((int64_t)row_g * a.heads + h) * kr;
  for (int s = lane; s < kr; s += 64) {
    oi[s] = -1;
    ov[s] = -INFINITY;
  }
  if (r < 0 || r >= Lq) return;
  const int Lk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
  const int km0 = a.cu_seqlens_km[b];
  const int Cb = a.cu_seqlens_km[b + 1] - km0;
  const int rp = r + Lk - Lq;
  const int hk = h / (a.heads / a.heads_k);
  int nc = a.is_causal ? (rp >= 0 ? min(rp / a.chunk, Cb) : 0) : Cb;
  const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)row_g * a.q_row_stride + (int64_t)h * a.q_head_stride;
  const uint16_t *kmp = reinterpret_cast<const uint16_t *>(a.km) + (int64_t)hk * a.km_head_stride;
  const uint32_t *selrow = sel + (int64_t)h * W * a.total_q + row_g;
  for (int c = lane; c < nc; c += 64) {
    float s = -INFINITY;  // (chunks the gate did not select never enter the lists)
    if ((c >> 5) < W && ((selrow[(int64_t)(c >> 5) * a.total_q] >> (c & 31)) & 1u)) {
      s = 0.f;
      const uint16_t *kr_ = kmp + (int64_t)(km0 + c) * a.km_row_stride;
      for (int d = 0; d < a.head_dim; ++d) s = fmaf(elem_to_float<T>(qp[d]), elem_to_float<T>(kr_[d]), s);
      if (s == -INFINITY) s = -3.4028234663852886e38f;  // a selected chunk keeps its place in the list
    }
    sScore[c] = s;
  }
  __syncthreads();
  int slot = 0;
  if (a.is_causal && rp >= 0) {
    if (lane == 0) {
      oi[0] = rp / a.chunk;
      ov[0] = INFINITY;
    }
    slot = 1;
  }
  // previous winner (score key, chunk) bounds the next search from above
  uint32_t pk = 0xffffffffu;
  int pc = 0x7fffffff;
  for (; slot < a.topk; ++slot) {
    uint32_t bk = 0u;
    int bc = -1;
    for (int c = lane; c < nc; c += 64) {
      const float s = sScore[c];
      if (s == -INFINITY) continue;  // never inserted by a strict '>' against -inf
      const uint32_t k = float_order_key(s);
      const bool below_prev = (k < pk) || (k == pk && c < pc);
      const bool better = (k > bk) || (k == bk && c > bc);
      if (below_prev && better) {
        bk = k;
        bc = c;
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const uint32_t ok = (uint32_t)__shfl_xor((int)bk, o, 64);
      const int oc = __shfl_xor(bc, o, 64);
      if (ok > bk || (ok == bk && oc > bc)) {
        bk = ok;
        bc = oc;
      }
    }
    if (bc < 0) break;
    if (lane == 0) {
      oi[slot] = bc;
      ov[slot] = sScore[bc];
    }
    pk = bk;
    pc = bc;
  }
}

__global__ void fill_i32_kernel(int32_t *p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

static inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace fmoba

extern "C" size_t fmoba_fused_topk_workspace_bytes(int32_t batch, int32_t total_q, int32_t heads, int32_t max_seqlen_q,
                                                   int32_t max_seqlen_k, int32_t chunk) {
  using namespace fmoba;
  if (batch <= 0 || heads <= 0 || chunk <= 0 || total_q < 0) return 0;
  const int64_t max_cols = ceil_div64(max_seqlen_k, chunk);
  const int64_t W = ceil_div64(max_cols, 32);
  const int64_t nseg = ceil_div64(max_seqlen_q > 0 ? max_seqlen_q : 1, csc_seg_rows(batch, heads, max_seqlen_q, W));
  return align256((size_t)heads * W * total_q * 4) + align256((size_t)batch * heads * nseg * max_cols * 4) + 256;
}

namespace fmoba {
// chunks that a row keeps besides its own
static int gate_winners(const TopkParams &p) { return p.a.is_causal ? p.a.topk - 1 : p.a.topk; }
template <typename T, int HD, int NT>
static int launch_gate(const TopkParams &p, dim3 grid, hipStream_t s) {
  const size_t smem = (size_t)NT * 32 * HD * 2 + (size_t)NT * 32 * 4;
  auto kern = topk_gate_kernel<T, HD, false, NT>;
  if constexpr (NT < 8)  // (with more chunks so few winners are the stream's)
    if (gate_winners(p) <= kGatePeels) kern = topk_gate_kernel<T, HD, true, NT>;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("fused_topk: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  hipLaunchKernelGGL(kern, grid, dim3(256), smem, s, p);
  return 0;
}
// chunk indices are 16-bit fields of the running winners (topk_gate_stream_kernel) and the forward's step lists
constexpr int kMaxChunksPerSequence = 65535;
template <typename T, int HD>
static int launch_gate_stream(const TopkParams &p, dim3 grid, hipStream_t s) {
  const size_t smem = gate_stream_smem<HD>();
  const int kp = gate_winners(p);
  auto kern = kp <= 16 ? topk_gate_stream_kernel<T, HD, 8> : kp <= 32 ? topk_gate_stream_kernel<T, HD, 16> : topk_gate_stream_kernel<T, HD, 32>;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("fused_topk: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  hipLaunchKernelGGL(kern, grid, dim3(256), smem, s, p);
  return 0;
}
template <typename T>
static int launch_gate_stream_hd(const TopkParams &p, dim3 grid, hipStream_t s) {
  // (groups of 64 chunks, three workgroups per compute unit; with groups of 128 and two workgroups 6.4 ms instead of 5.1 at 262144 tokens)
  if (p.a.head_dim <= 64) return launch_gate_stream<T, 64>(p, grid, s);
  if (p.a.head_dim <= 128) return launch_gate_stream<T, 128>(p, grid, s);
  return launch_gate_stream<T, 256>(p, grid, s);
}
template <typename T, int HD, int NJ>
static int launch_gate_few_nj(const TopkParams &p, hipStream_t s) {
  const size_t smem = (size_t)std::min(p.a.max_seqlen_q, kFewRows) * NJ * 64 * 4;
  auto kern = topk_gate_few_kernel<T, HD, NJ>;
  if (smem > 32 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("fused_topk: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  hipLaunchKernelGGL(kern, dim3(p.a.heads, p.a.batch), dim3(512), smem, s, p);
  return 0;
}
template <typename T, int HD>
static int launch_gate_few(const TopkParams &p, hipStream_t s) {
  if (p.max_cols <= 256) return launch_gate_few_nj<T, HD, 4>(p, s);
  if (p.max_cols <= 1024) return launch_gate_few_nj<T, HD, 16>(p, s);
  return launch_gate_few_nj<T, HD, 64>(p, s);
}
template <typename T>
static int launch_gate_few_hd(const TopkParams &p, hipStream_t s) {
  if (p.a.head_dim <= 64) return launch_gate_few<T, 64>(p, s);
  if (p.a.head_dim <= 128) return launch_gate_few<T, 128>(p, s);
  return launch_gate_few<T, 256>(p, s);
}
template <typename T, int HD>
static int launch_gate_nt(const TopkParams &p, dim3 grid, hipStream_t s) {
  if (p.W <= 2) return launch_gate<T, HD, 2>(p, grid, s);
  if (p.W <= 4) return launch_gate<T, HD, 4>(p, grid, s);
  // more than 128 chunks and no more than 16 winners: in groups.  (Gating and lists, in groups and with all scores in registers: 32768 tokens, 32 heads, 128-key
  // chunks, top-k 16 333 and 384 us, top-k 4 246 and 335; 10000 tokens, 16 heads of 64, 157 chunks, top-k 16 55.7 and 59.5.  With up
  // to 128 chunks registers are the faster form: 21000 tokens in two sequences, top-k 12 55 against 64 us, 16384 tokens, top-k 8 41 against 43.)
  if (gate_winners(p) <= 16) return launch_gate_stream<T, HD>(p, grid, s);
  return launch_gate<T, HD, 8>(p, grid, s);
}
template <typename T>
static int launch_gate_hd(const TopkParams &p, dim3 grid, hipStream_t s) {
  if (p.a.head_dim <= 64) return launch_gate_nt<T, 64>(p, grid, s);
  if (p.a.head_dim <= 128) return launch_gate_nt<T, 128>(p, grid, s);
  return launch_gate_nt<T, 256>(p, grid, s);
}
}  // namespace fmoba

namespace fmoba {
int mean_pool_with_offsets(const fmoba_mean_pool_args *a, int32_t *clear, int64_t clear_vec16, void *stream);
int fwd_check_gated(const fmoba_attn_fwd_args *a);                                                  // attn_fwd.hip
int run_fwd_rows_gated(const fmoba_attn_fwd_args &a, const RowGate &gate, hipStream_t s);           // attn_fwd_rows.hip
}
// The call behind the entry points: everything of `a` except its workspace fields, which come as arguments.  `pool`: the
// pooling pass that comes first and clears the segment counts; null: the chunk means are there already.  `attn`: the forward that takes the gate's place.
static int fused_topk_run(const fmoba_fused_topk_args *a, void *workspace, size_t workspace_bytes, const fmoba_mean_pool_args *pool, bool lists,
                          const fmoba_csc_ranks *ranks, void *stream, const fmoba_attn_fwd_args *attn = nullptr) {
  using namespace fmoba;
  FMOBA_REQUIRE(a != nullptr, "fused_topk: null args");
  FMOBA_REQUIRE(a->dtype == FMOBA_DTYPE_F16 || a->dtype == FMOBA_DTYPE_BF16, "FlashMoBA only supports fp16 and bf16 data types");
  FMOBA_REQUIRE(a->topk >= 1 && a->topk <= 64, "moba_topk must be in [1, 64]");
  FMOBA_REQUIRE(a->batch > 0, "batch size must be positive");
  FMOBA_REQUIRE(a->head_dim > 0 && a->head_dim <= 256, "head_size must be <= 256");
  FMOBA_REQUIRE(a->head_dim % 8 == 0, "head_size must be multiple of 8");
  FMOBA_REQUIRE(a->heads > 0 && a->heads_k > 0 && a->heads % a->heads_k == 0, "#heads in key/value must divide #heads in query");
  FMOBA_REQUIRE(a->chunk > 0, "moba_chunk_size must be positive");
  FMOBA_REQUIRE(a->total_q >= 0 && a->max_seqlen_q >= 0 && a->max_seqlen_k >= 0, "negative size");
  FMOBA_REQUIRE(a->cu_seqlens_q && a->cu_seqlens_k && a->cu_seqlens_km, "fused_topk: null cu_seqlens pointer");
  FMOBA_REQUIRE((a->col_offsets && a->col_nnz) || a->max_seqlen_k == 0 || !lists, "fused_topk: null col_offsets/col_nnz pointer");
  FMOBA_REQUIRE(a->flat_indices || (int64_t)a->total_q * a->heads * a->topk == 0 || !lists, "fused_topk: null flat_indices pointer");
  FMOBA_REQUIRE((a->raw_indices == nullptr) == (a->raw_values == nullptr), "fused_topk: raw_indices and raw_values go together");
  hipStream_t s = (hipStream_t)stream;
  const int max_cols = ceil_div(a->max_seqlen_k, a->chunk);
  const int64_t nslots = (int64_t)a->total_q * a->heads * a->topk;
  const int kr = (a->topk + 15) / 16 * 16;

  if (max_cols == 0 || a->max_seqlen_k == 0) {
    // no keys: lists stay empty; the reference fills the row list with -1 here
    // (csrc/flash_topk/flash_topk_api.cpp:250-255)
    if (nslots) hipLaunchKernelGGL(fill_i32_kernel, dim3(1024), dim3(256), 0, s, a->flat_indices, nslots, -1);
    if (a->raw_indices && a->total_q) {
      hipLaunchKernelGGL(fill_i32_kernel, dim3(1024), dim3(256), 0, s, a->raw_indices, (int64_t)a->total_q * a->heads * kr, -1);
      hipLaunchKernelGGL(fill_i32_kernel, dim3(1024), dim3(256), 0, s, reinterpret_cast<int32_t *>(a->raw_values),
                         (int64_t)a->total_q * a->heads * kr, (int32_t)0xff800000);
    }
    FMOBA_LAUNCH_CHECK("fused_topk(empty)");
    return 0;
  }
  const bool big = max_cols > 256;  // more chunks than the register-resident gate holds: grouped gate
  FMOBA_REQUIRE(max_cols <= kMaxChunksPerSequence, "fused_topk: %d key chunks per sequence; at most %d are supported", max_cols, kMaxChunksPerSequence);
  // (the fill keeps list positions as 32-bit byte offsets from the first of the 32 lists of a word column)
  FMOBA_REQUIRE(a->max_seqlen_q < (1 << 24), "fused_topk: max_seqlen_q = %d; sequences of up to %d query rows are supported", a->max_seqlen_q,
                (1 << 24) - 1);
  FMOBA_REQUIRE(a->q && a->km, "fused_topk: null q/km pointer");
  FMOBA_REQUIRE(a->q_row_stride % 8 == 0 && a->q_head_stride % 8 == 0 && a->km_row_stride % 8 == 0 && a->km_head_stride % 8 == 0,
                "fused_topk: strides must be multiples of 8 elements");
  FMOBA_REQUIRE(((uintptr_t)a->q % 16) == 0 && ((uintptr_t)a->km % 16) == 0, "fused_topk: q and km must be 16-byte aligned");
  FMOBA_REQUIRE(a->batch <= 65535 && a->heads <= 65535, "fused_topk: batch/heads too large for the launch grid");

  TopkParams p;
  p.a = *a;
  p.max_cols = max_cols;
  p.W = ceil_div(max_cols, 32);
  p.seg_rows = csc_seg_rows(a->batch, a->heads, a->max_seqlen_q, p.W);
  p.nseg = ceil_div(a->max_seqlen_q > 0 ? a->max_seqlen_q : 1, p.seg_rows);
  p.ranks = ranks != nullptr ? *ranks : fmoba_csc_ranks{nullptr, nullptr};
  p.sub_fwd = p.sub_bwd = 1;
  if (ranks != nullptr) {
    FMOBA_REQUIRE(ranks->visits && (ranks->prefix || p.W == 1), "pool_and_gate_ranked: null pointer");
    FMOBA_REQUIRE(a->chunk % 64 == 0, "pool_and_gate_ranked: the attention takes chunks of a multiple of 64 keys");
    p.sub_fwd = a->chunk % 128 == 0 ? a->chunk / 128 : a->chunk / 64;                       // (fmoba_attn_fwd_key_block)
    p.sub_bwd = a->chunk % 128 == 0 && a->head_dim > 64 ? a->chunk / 128 : a->chunk / 64;
    FMOBA_REQUIRE((int64_t)a->topk * p.sub_bwd < 65536, "pool_and_gate_ranked: more than 65535 visits per row");
  }
  const size_t sel_bytes = align256((size_t)a->heads * p.W * a->total_q * 4);
  const size_t seg_bytes = align256((size_t)a->batch * a->heads * p.nseg * max_cols * 4);
  FMOBA_REQUIRE(workspace != nullptr && workspace_bytes >= sel_bytes + seg_bytes, "fused_topk: workspace too small (%zu < %zu)",
                workspace_bytes, sel_bytes + seg_bytes);
  uintptr_t wsp = ((uintptr_t)workspace + 255) & ~(uintptr_t)255;
  FMOBA_REQUIRE(wsp + sel_bytes + seg_bytes <= (uintptr_t)workspace + workspace_bytes, "fused_topk: workspace too small after alignment");
  p.sel = reinterpret_cast<uint32_t *>(wsp);
  p.segcnt = reinterpret_cast<int32_t *>(wsp + sel_bytes);

  if (a->total_q == 0 || a->max_seqlen_q == 0) {
    // no query rows: every column is empty, offsets are the (constant) region bases
    const int64_t n = (int64_t)a->batch * a->heads * max_cols;
    hipLaunchKernelGGL(fill_i32_kernel, dim3(256), dim3(256), 0, s, p.segcnt, (int64_t)(seg_bytes / 4), 0);
    hipLaunchKernelGGL(csc_scan_kernel<false>, dim3(a->heads, a->batch), dim3(256), 0, s, p);
    (void)n;
    FMOBA_LAUNCH_CHECK("fused_topk(no rows)");
    return 0;
  }

  if (pool != nullptr) {
    if (int rc = mean_pool_with_offsets(pool, p.segcnt, lists ? (int64_t)(seg_bytes / 16) : 0, stream)) return rc;
  } else {
    hipLaunchKernelGGL(fill_i32_kernel, dim3(512), dim3(256), 0, s, p.segcnt, (int64_t)(seg_bytes / 4), 0);
  }
  if (!lists) p.segcnt = nullptr;
  const int row_blocks = ceil_div(a->max_seqlen_q, kGateRows);
  p.rows_in_x = row_blocks > kMaxGridY;
  const dim3 ggrid = p.rows_in_x ? dim3(row_blocks, a->heads, a->batch) : dim3(a->heads, row_blocks, a->batch);
  int rc;
  if (attn != nullptr)
    rc = run_fwd_rows_gated(*attn, RowGate{reinterpret_cast<const uint16_t *>(a->km), a->cu_seqlens_km, a->km_row_stride, a->km_head_stride, a->topk, lists ? p.sel : nullptr, p.segcnt, p.W,
                                           p.nseg, p.seg_rows}, s);
  else if (a->max_seqlen_q <= kFewRows && max_cols <= kFewChunks)
    rc = (a->dtype == FMOBA_DTYPE_BF16) ? launch_gate_few_hd<bf16_t>(p, s) : launch_gate_few_hd<f16_t>(p, s);
  else if (big)
    rc = (a->dtype == FMOBA_DTYPE_BF16) ? launch_gate_stream_hd<bf16_t>(p, ggrid, s) : launch_gate_stream_hd<f16_t>(p, ggrid, s);
  else
    rc = (a->dtype == FMOBA_DTYPE_BF16) ? launch_gate_hd<bf16_t>(p, ggrid, s) : launch_gate_hd<f16_t>(p, ggrid, s);
  if (rc) return rc;
  FMOBA_LAUNCH_CHECK(attn != nullptr ? "attn_fwd_rows_kernel (gated)" : "topk_gate_kernel");
  if (!lists) return 0;
  const int64_t list_groups = (int64_t)p.nseg * (p.W + (ranks ? 1 : 0)) * a->heads * a->batch;
  if ((int64_t)p.nseg * max_cols <= kListCounts && p.W <= kListWords && p.seg_rows == kListSegRows && list_groups <= (ranks ? kListRankedGroups : kListGroups)) {
    hipLaunchKernelGGL(ranks ? csc_lists_kernel<true> : csc_lists_kernel<false>, dim3(p.nseg * p.W + (ranks ? p.nseg : 0), a->heads, a->batch), dim3(256), 0, s, p);
    FMOBA_LAUNCH_CHECK("csc_lists_kernel");
  } else {
    if (ranks)
      hipLaunchKernelGGL(csc_scan_kernel<true>, dim3(a->heads, a->batch, 1 + ceil_div(a->max_seqlen_q, kRankRows)), dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL(csc_scan_kernel<false>, dim3(a->heads, a->batch), dim3(256), 0, s, p);
    FMOBA_LAUNCH_CHECK("csc_scan_kernel");
    hipLaunchKernelGGL(ranks ? csc_fill_kernel<true> : csc_fill_kernel<false>, dim3(p.nseg * p.W, a->heads, a->batch), dim3(64), 0, s, p);
    FMOBA_LAUNCH_CHECK("csc_fill_kernel");
  }
  if (a->raw_indices) {
    const size_t smem = (size_t)(max_cols + 64) * 4;
    dim3 rgrid(a->total_q, a->heads);
    if (a->dtype == FMOBA_DTYPE_BF16)
      hipLaunchKernelGGL(topk_raw_kernel<bf16_t>, rgrid, dim3(64), smem, s, *a, kr, p.sel, p.W);
    else
      hipLaunchKernelGGL(topk_raw_kernel<f16_t>, rgrid, dim3(64), smem, s, *a, kr, p.sel, p.W);
    FMOBA_LAUNCH_CHECK("topk_raw_kernel");
  }
  return 0;
}

extern "C" int fmoba_fused_topk(const fmoba_fused_topk_args *a, void *stream) {
  FMOBA_REQUIRE(a != nullptr, "fused_topk: null args");
  return fused_topk_run(a, a->workspace, a->workspace_bytes, nullptr, true, nullptr, stream);
}

static int pool_and_gate(const fmoba_mean_pool_args *m, const fmoba_fused_topk_args *g, bool want_lists, const fmoba_csc_ranks *r, void *stream, const fmoba_attn_fwd_args *attn = nullptr) {
  FMOBA_REQUIRE(m != nullptr && g != nullptr, "pool_and_gate: null args");
  FMOBA_REQUIRE(m->km == g->km && m->cu_seqlens_km == g->cu_seqlens_km && m->cu_seqlens_k == g->cu_seqlens_k && m->batch == g->batch &&
                    m->heads_k == g->heads_k && m->head_dim == g->head_dim && m->chunk == g->chunk && m->dtype == g->dtype,
                "pool_and_gate: the two argument structs describe different problems");
  FMOBA_REQUIRE(g->total_q > 0 && g->max_seqlen_q > 0 && g->max_seqlen_k > 0, "pool_and_gate: empty problem");
  FMOBA_REQUIRE(m->max_chunks == fmoba::ceil_div(g->max_seqlen_k, g->chunk), "pool_and_gate: max_chunks is ceil(max_seqlen_k / chunk)");
  FMOBA_REQUIRE(want_lists || g->raw_indices == nullptr, "pool_and_gate: the ordered lists come with the column lists only");
  return fused_topk_run(g, g->workspace, g->workspace_bytes, m, want_lists, r, stream, attn);
}

extern "C" int fmoba_pool_and_gate(const fmoba_mean_pool_args *m, const fmoba_fused_topk_args *g, int32_t want_lists, void *stream) {
  return pool_and_gate(m, g, want_lists != 0, nullptr, stream);
}

extern "C" int fmoba_attn_fwd_gated_rows(const fmoba_mean_pool_args *m, const fmoba_fused_topk_args *g, const fmoba_attn_fwd_args *a, int32_t want_lists, void *stream) {
  if (int rc = fmoba::fwd_check_gated(a)) return rc;
  FMOBA_REQUIRE(m != nullptr && g != nullptr, "attn_fwd_gated_rows: null args");
  FMOBA_REQUIRE(g->q == a->q && g->q_row_stride == a->q_row_stride && g->q_head_stride == a->q_head_stride && g->cu_seqlens_q == a->cu_seqlens_q && m->k == a->k &&
                    g->cu_seqlens_k == a->cu_seqlens_k && g->batch == a->batch && g->total_q == a->total_q && g->heads == a->heads && g->heads_k == a->heads_k &&
                    g->head_dim == a->head_dim && g->max_seqlen_q == a->max_seqlen_q && g->max_seqlen_k == a->max_seqlen_k && g->chunk == a->lg_block_n &&
                    g->dtype == a->dtype && (g->is_causal != 0) == (a->is_causal != 0) && a->max_cols == fmoba::ceil_div(a->max_seqlen_k, a->lg_block_n),
                "attn_fwd_gated_rows: the argument structs describe different problems");
  return pool_and_gate(m, g, want_lists != 0, nullptr, stream, a);
}

extern "C" int fmoba_pool_and_gate_ranked(const fmoba_mean_pool_args *m, const fmoba_fused_topk_args *g, const fmoba_csc_ranks *r, void *stream) {
  FMOBA_REQUIRE(r != nullptr, "pool_and_gate_ranked: null ranks");
  return pool_and_gate(m, g, true, r, stream);
}

// ------------------------------------------------------------------------------------
// The same call for callers that cannot allocate device memory (HIP graph capture, serving loops): selection bits and
// segment counts live in a fixed array of the code object instead of a caller's workspace.  Every device that loads
// the library holds its own copy of the array at its own address, which the runtime tells once per device.
// ------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[FMOBA_STATIC_SCRATCH_BYTES];

namespace fmoba {
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` per device, null until asked for
}  // namespace fmoba

extern "C" int fmoba_fused_topk_static(const fmoba_fused_topk_args *a, void *stream) {
  using namespace fmoba;
  FMOBA_REQUIRE(a != nullptr, "fused_topk_static: null args");
  const size_t need = fmoba_fused_topk_workspace_bytes(a->batch, a->total_q, a->heads, a->max_seqlen_q, a->max_seqlen_k, a->chunk);
  FMOBA_REQUIRE(need <= (size_t)FMOBA_STATIC_SCRATCH_BYTES,
                "fused_topk_static: this call needs %zu bytes of scratch memory, the library's fixed buffer holds %zu; use fmoba_fused_topk with a workspace",
                need, (size_t)FMOBA_STATIC_SCRATCH_BYTES);
  int dev = -1;
  FMOBA_REQUIRE(hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices, "fused_topk_static: no current HIP device (or its index is above %d)", kMaxDevices - 1);
  void *ptr = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
      void *p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      FMOBA_REQUIRE(e == hipSuccess && p != nullptr, "fused_topk_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
      g_scratch_ptr[dev] = p;
    }
    ptr = g_scratch_ptr[dev];
  }
  return fused_topk_run(a, ptr, (size_t)FMOBA_STATIC_SCRATCH_BYTES, nullptr, true, nullptr, stream);
}
