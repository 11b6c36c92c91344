// Sparse attention backward over a CSC pattern, without a single global atomic.
//
//   bwd_prep_kernel      : delta[row] = sum_d dO*O (fp32).
//   attn_bwd_dkdv_kernel : COLUMN-stationary.  One workgroup per (64-key block, query heads that share it,
//                          sequence) keeps K and V of the block in registers and walks the block's
//                          ascending row lists in rounds of 64 gathered rows (head dimensions up to
//                          128; above: attn_bwd_wide.hip):
//                            S = Q K^T, dP = dO V^T
//                            P = exp2(S*scale*log2e - LSE*log2e), dS = P o (dP - delta)
//                            dV^T += dO^T P, dK^T += Q^T dS     (transposing LDS reads)
//                            dQ^T_partial = K^T dS^T            (per visit of a (row, key block) pair)
//                          dK/dV live in registers for the whole list and are written
//                          once.  For dQ the kernel leaves either its dS tiles (16-bit, indexed by
//                          row-list position) or, per visit, a dQ partial row (16-bit; fp16: scaled) in a
//                          slot that the row hands out from a counter.
//   attn_bwd_dkdv_partials_kernel : the same for the long calls, dQ partials at head dimension 128.
//   attn_bwd_dq_kernel   : dQ from the dS tiles, one workgroup per 256 query rows, dQ in registers
//                          (patterns in which a row block meets a dozen rows or more per step).
//   attn_bwd_dq_combine_kernel : dQ from the partials, sixteen lanes per (row, head) add them in ascending
//                          key-block order and scales.  Work and traffic are proportional to
//                          the number of visits, whatever the number of chunks per sequence.
// In the dK/dV kernels nothing moves data through registers: the gathered Q / dO rows go from global
// memory straight to LDS (global_load_lds), one round ahead.
#include "fmoba_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace fmoba {

constexpr int kBwdRoundRows = 128;  // rows of a column list the workgroup takes per round: two 32-row tiles per wave pair

template <int HD>
struct BwdSmem {
  // The gathered Q / dO tiles have rows of exactly HD elements (the loads that fill them write 64 lanes x 16 bytes
  // to consecutive addresses) and are swizzled instead of padded: the 16-byte piece c of tile row r lies at piece
  // c ^ tile_swz<HD>(r).  With that, the 16-byte row reads (lane -> row lane % 32) and the transposing 8-byte
  // reads both spread over all banks.
  static constexpr int LDQ = HD + 16;  // elements, K and V while they are read into registers (plain padded rows)
  static constexpr int LDS_ = 32 + 8;  // elements, dS^T tile rows [key][32 rows]
  static constexpr size_t tileBytes = (size_t)32 * HD * 2;
  static constexpr size_t oQ = 0;                                   // [2 buffers][4 tiles][32][HD]
  static constexpr size_t odO = oQ + 8 * tileBytes;
  static constexpr size_t odS = odO + 8 * tileBytes;               // [2 pairs][2 tile slots][64 keys][LDS_] or [2 tile slots][128 keys][LDS_]
  static constexpr size_t oRid = odS + (size_t)2 * 2 * 64 * LDS_ * 2;  // int[2 buffers][128]: row ids, one round before the rest
  static constexpr size_t oRow = oRid + 2 * kBwdRoundRows * 4;     // int[2 buffers][128]
  static constexpr size_t oSlot = oRow + 2 * kBwdRoundRows * 4;
  static constexpr size_t oLse = oSlot + 2 * kBwdRoundRows * 4;    // LSE * log2(e)
  static constexpr size_t oDelta = oLse + 2 * kBwdRoundRows * 4;
  static constexpr size_t bytes = oDelta + 2 * kBwdRoundRows * 4;
  static constexpr int LDR = HD + 4;  // floats, output transpose buffer [2][64 or 128 keys][LDR]
  static_assert((size_t)2 * 128 * LDQ * 2 <= 16 * tileBytes, "K and V pass through the tiles");
  static_assert(bytes <= 160 * 1024, "LDS of one compute unit");
};

struct BwdWs {
  int32_t dkv_heads;  // heads of dK / dV (of the kernels that sum query heads)
  int32_t *cnt;    // [total_q * heads] visits handed out per (row, head)
  int32_t *pid;    // [total_q * heads * cap] key block id of each partial
  uint16_t *part;  // [total_q * heads * cap][part_row_elems] dQ partials (times dq_part_scale)
  int32_t cap;
  const uint32_t *visits;  // as in the forward pass (null: slots from the counters)
  int32_t row_mask;        // of list entries: kListRowMask for ranked lists, else -1
  int32_t *tab;    // dS form: first list position of every column in every block of kDqRows query rows (RunTable)
  uint16_t *ds;    // dS tiles (row-stationary dQ form): [row list position / 32][key of the column / 8][position % 32][8 keys]
};

// Where the lists of the columns enter the row blocks of the dQ pass: [head][column][row block, and one past the last], the columns
// of sequence b from number cu_seqlens_k[b] / Bn + b on (which leaves every sequence room for its own).  The delta pass looks the places
// up, a wave per column, in front of its rows; found by every workgroup of the dQ pass for its own row block, two searches of
// a dozen dependent loads per column, they were a quarter of that pass on short sequences.  Delta and dQ pass, and the clearing of the
// padded delta that was a launch of its own: 8191 tokens of short documents 43.4 -> 36.6 us, 24571 tokens, 32 over 8 heads 728 -> 697,
// 65536 tokens in eight sequences 1675 -> 1656 (its places take 25 us of the delta pass; with those looked up that no row block reads, past a
// sequence's end or before a column's first row, 27, and beside 256 sequences of 512 tokens one of 65536 took 842 us instead of 788).
constexpr int kDqRows = 256;
struct RunTable {
  int cols, blocks;  // columns of all sequences, row blocks + 1
  __host__ __device__ __forceinline__ int64_t at(int h, int col) const { return ((int64_t)h * cols + col) * blocks; }
};
static inline RunTable bwd_run_table(const fmoba_attn_bwd_args &a) {
  return RunTable{a.total_k / a.lg_block_n + a.batch, ceil_div(a.max_seqlen_q, kDqRows) + 1};
}

// Softmax scale of dQ in the partials form: fp16 partial rows carry it (as far as it makes them smaller), the sums of bf16 ones get it.
// Without it the rows are sqrt(head_dim) times the gradient they add up to, and fp16 rows overflow where the gradient does not.
// (8192 tokens, heads of 128, top-k 8 of 128-key chunks, error of dQ against 64 bits: 3.69e-4 -> 3.59e-4, with dout 100 times
// smaller 3.75e-4 -> 3.70e-4; 1000 times smaller, where the gradient itself is mostly below the normal numbers of the type, 0.85e-3 ->
// 1.09e-3.  dK/dV and dQ of 32768 tokens, 32 heads, top-k 16: 5060 us before and after.)
template <typename T>
__device__ __forceinline__ float dq_part_scale(float softmax_scale) {
  return std::is_same_v<T, f16_t> ? fminf(softmax_scale, 1.f) : 1.f;
}
template <typename T>
__device__ __forceinline__ float dq_sum_scale(float softmax_scale) {
  return std::is_same_v<T, f16_t> ? fmaxf(softmax_scale, 1.f) : softmax_scale;
}
template <typename T>
__device__ __forceinline__ uint2 pack4_scaled(float x, float y, float z, float w, float scale) {
  if constexpr (std::is_same_v<T, f16_t>)
    return make_uint2(pack2<T>(x * scale, y * scale), pack2<T>(z * scale, w * scale));
  else
    return make_uint2(pack2<T>(x, y), pack2<T>(z, w));
}

// ------------------------------------------------------------------------------------
// dK / dV.  One workgroup per (64 keys, query heads that share them, sequence) walks the row lists of its heads, 64
// gathered rows a round.  S^T and dP^T of a (32 keys, 32 rows) tile are one wave's (A = K / V in registers, B = the rows: one
// lane owns one row, so LSE and delta are one register each); P and dS go to LDS, [row][key], 16-bit; then every wave adds
// up dV^T or dK^T of half of the features and all keys over the round's 64 rows (both operands through transposing
// reads).  Four waves of 256 registers, two workgroups per compute unit: what one waits for (two barriers a round, the next
// round's rows, which come straight into LDS a round ahead) the other covers.
// dQ: the dS form leaves dS, by position in the row lists (attn_bwd_dq_kernel); the partials form, built for head
// dimensions up to 64, multiplies it with K^T (in registers) and leaves a part row per visit in the slot that the row hands
// out (attn_bwd_dq_combine_kernel).
// Measured against one workgroup of four 512-register waves per unit, products and softmax interleaved by hand (which stays
// for the partials form at head dimension 128, attn_bwd_dkdv_partials_kernel): 8191 tokens of short documents, heads of 64
// 100 -> 49 us; 12037 tokens, heads of 96 227 -> 177 us; 2 x 4096 tokens 223 -> 214 us; 65536-token batch 2.94 -> 2.65 ms.
// One workgroup of eight waves per 128 keys (half of the gathers, three buffers): 256 us where two of 64 keys take 214.
// Head dimensions 65 to 96: tiles of 96 features against 128 before, 12037 tokens, 16 heads of 96 180 -> 159 us, 2 x 4096 tokens,
// heads of 80 202 -> 164.
// ------------------------------------------------------------------------------------
template <int HD, bool DQP>
struct DkdvSmem {
  static constexpr int NBUF = 2;
  static constexpr int PRB = 128;                        // bytes of a P / dS row
  static constexpr size_t tile = (size_t)64 * HD * 2;        // 64 gathered rows of Q or dO, swizzled (tile_swz)
  static constexpr size_t oQ = 0;                             // [NBUF]
  static constexpr size_t odO = oQ + NBUF * tile;             // [NBUF]
  static constexpr size_t oP = odO + NBUF * tile;             // [64 rows][64 keys], piece p (8 keys) of row r at p ^ tile_swz<64>(r)
  static constexpr size_t odS = oP + 64 * PRB;
  static constexpr size_t oOut = odS + 64 * PRB;              // partials form: [64 rows][HD], dQ part rows on their way out
  static constexpr size_t oSlot = oOut + (DQP ? (size_t)64 * HD * 2 : 0);  // int[2][64]: places of the part rows
  static constexpr size_t bytes_loop = oSlot + (DQP ? 2 * 64 * 4 : 0);
  static constexpr int LDR = HD + 4;                          // floats, output staging [2][64 keys][LDR]
  static constexpr size_t bytes_out = (size_t)2 * 64 * LDR * 4;
  static constexpr size_t bytes = bytes_loop > bytes_out ? bytes_loop : bytes_out;
  static_assert(bytes <= 160 * 1024 && (size_t)64 * HD * 2 <= NBUF * tile, "LDS of one compute unit; K and V pass through the tiles");
};

// RANKED (partials form): part rows go to the place of the block among the row's, which the rank of the list entry gives
// NEAR: a gathered row's place is a 32-bit byte offset from the sequence's first row that one 24-bit multiply makes (rows_near).
// Three waves per SIMD for the dS form of heads up to 64, whose LDS takes three workgroups to a unit: the compiler's own choice for rows far apart was 182
// registers (166 now) and two waves, backward of 8191 tokens, 16 heads 248 us against 236, of 16384, 32 heads 1264 against 1223.
template <typename T, int HD, bool DQP, bool RANKED, bool NEAR>
__global__ __launch_bounds__(256, HD <= 64 && !DQP ? 3 : 2) void attn_bwd_dkdv_kernel(fmoba_attn_bwd_args a, BwdWs ws, ItemOrder order) {
  typedef DkdvSmem<HD, DQP> SM;
  constexpr int KS = HD / 16, NDT = HD / 32, VPR = HD / 8, RB = HD * 2, LDR = SM::LDR, PRB = SM::PRB;
  constexpr int NKEY = 64;   // keys of the workgroup
  // tiles of dV or dK that a wave adds up: half of the features and all keys, or all three feature tiles and half of the keys
  constexpr int NDW = NDT % 2 == 0 ? NDT / 2 : NDT, NKW = NDT % 2 == 0 ? 2 : 1;
  static_assert(!DQP || NDT % 2 == 0, "the partials form divides the features");
  constexpr float kLog2e = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  const int gh = ws.dkv_heads, gs = a.heads / gh;  // heads of dK / dV, query heads that are added up in one
  int nb, b, hg;
  if (order == kListedLongestFirst) {
    const BlockItem item = listed_item<NKEY, false>(blockIdx.x, a.batch, gh, a.max_seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    nb = item.idx, b = item.b, hg = item.h;
  } else {
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * gh, (a.max_seqlen_k + NKEY - 1) / NKEY, (int64_t)a.max_seqlen_q * HD * 4 >= kOnePairBytes, order == kLongestFirst);
    nb = item.idx, b = item.pair / gh, hg = item.pair - b * gh;
  }
  const int h0 = hg * gs;
  const int key0 = nb * NKEY;
  const int Bn = a.lg_block_n, c = key0 / Bn;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  // lane j: the row list of head h0 + j (a group larger than a wave is split by the caller)
  int nnz = 0;
  int64_t lbase = 0;
  if (c < a.max_cols && lane < gs) {
    const int64_t ci = ((int64_t)b * a.heads + h0 + lane) * a.max_cols + c;
    nnz = a.col_nnz[ci];
    lbase = a.col_offsets[ci];
  }
  const int k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  if (key0 >= Lk) return;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int off = Lk - Lq;
  const int D = a.head_dim;
  const int PD = part_row_elems(D, 2);
  (void)PD;
  const int hk = h0 / (a.heads / a.heads_k);
  const int kq = wave & 1, rt = wave >> 1;   // S and dP: this wave's 32 keys and 32 rows
  const int sel = wave >> 1, fw = wave & 1;  // sums: dV (0) or dK (1), half fw of the features or of the keys
  const int d0 = NKW == 2 ? fw * NDW : 0, kk0 = NKW == 2 ? 0 : fw;  // first feature tile, first key tile
  const bool causal = a.is_causal != 0;
  const float scale_log2 = a.softmax_scale * kLog2e;
  const uint32_t lds = (uint32_t)(uintptr_t)smem, ldsQ = lds + (uint32_t)SM::oQ, ldsdO = lds + (uint32_t)SM::odO, ldsP = lds + (uint32_t)SM::oP, ldsdS = lds + (uint32_t)SM::odS;
  constexpr uint32_t TILE = (uint32_t)SM::tile;
  constexpr int NI = VPR / 4;                // load instructions per wave, operand and round: 16 rows

  // K and V of the block pass through the tiles on their way to registers
  {
    const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)(k0 + key0) * a.k_row_stride + (int64_t)hk * a.k_head_stride;
    const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)(k0 + key0) * a.v_row_stride + (int64_t)hk * a.v_head_stride;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int v = (wave * NI + i) * 64 + lane, key = v / VPR, pc = v - key * VPR;
      const int e = min((pc ^ tile_swz<HD>(key)) * 8, D - 8);
      const int64_t kc = min(key, Lk - 1 - key0);
      global_to_lds16(kg + kc * a.k_row_stride + e, ldsQ + (uint32_t)((wave * NI + i) * 1024));
      global_to_lds16(vg + kc * a.v_row_stride + e, ldsdO + (uint32_t)((wave * NI + i) * 1024));
    }
  }
  // Rows that lie before the block see none of its keys; only a block that is not its column's first has any in its lists
  // (of a gated pattern; others are masked), so only there the lists are searched for their first row.
  int start = 0;
  if (causal && key0 != c * Bn) {
    for (int g = 0; g < gs; ++g) {
      const int n = __builtin_amdgcn_readlane(nnz, g);
      const uint32_t blo = __builtin_amdgcn_readlane((uint32_t)lbase, g), bhi = __builtin_amdgcn_readlane((uint32_t)(lbase >> 32), g);
      const int st = n > 0 ? lower_bound_wave_i32(a.row_indices + (int64_t)(((uint64_t)bhi << 32) | blo), n, key0 - off, ws.row_mask) : 0;
      start = lane == g ? st : start;
    }
  }
  nnz -= start;
  lbase += start;
  int incl = (nnz + 63) >> 6;  // rounds of the lists up to this lane's
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(incl, o, 64);
    incl += lane >= o ? up : 0;
  }
  const int nround = __builtin_amdgcn_readlane(incl, 63);
  const int koff = key0 - c * Bn;  // offset of the block inside its column

  // a round: its head, the place of its first entry in the row lists and how many it has
  struct Round {
    int h, n;
    int64_t pos;
  };
  auto round_at = [&](int r) {  // (past the end: the last round again)
    r = min(r, nround - 1);
    const int g = __popcll(__ballot(incl <= r));
    const int j = (r - (g ? __builtin_amdgcn_readlane(incl, g - 1) : 0)) * 64;
    const uint32_t blo = __builtin_amdgcn_readlane((uint32_t)lbase, g), bhi = __builtin_amdgcn_readlane((uint32_t)(lbase >> 32), g);
    return Round{h0 + g, __builtin_amdgcn_readlane(nnz, g) - j, (int64_t)(((uint64_t)bhi << 32) | blo) + j};
  };
  const int64_t dstride = (int64_t)a.total_q + 128 * (int64_t)a.batch;
  const uint16_t *qg = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride;
  const uint16_t *dog = reinterpret_cast<const uint16_t *>(a.dout) + (int64_t)q0 * a.do_row_stride;

  f32x16 acc[NDW][NKW];  // register i of tile [d][kk] <-> feature (d0 + d) * 32 + acc_row(i, hh), key (kk0 + kk) * 32 + lane % 32
#pragma unroll
  for (int d = 0; d < NDW; ++d)
#pragma unroll
    for (int kk = 0; kk < NKW; ++kk)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[d][kk][i] = 0.f;

  const int myrow = rt * 32 + (lane & 31);  // this lane's row of a round
  const uint32_t rowoff = (uint32_t)((lane & 31) * RB + ((tile_frag_piece<HD>(hh, 0) ^ tile_swz<HD>(lane & 31)) * 16));
  const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
  const uint32_t troff = (uint32_t)(r0t * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
  auto entry_at = [&](const Round &w) { return a.row_indices + w.pos + min(myrow, w.n - 1); };
  const int nsub = Bn / NKEY, jsub = koff / NKEY;  // key blocks of the column, this one's number
  auto code = [&](int raw, const Round &w) { return tile_row_code(raw & ws.row_mask, myrow < w.n, Lq); };
  Round w0{}, w1{};  // the round at hand and the one after it
  int raw0 = 0, raw_nx = 0;
  if (nround > 0) {
    w0 = round_at(0), w1 = round_at(1);
    raw0 = *entry_at(w0), raw_nx = *entry_at(w1);
  }
  wait_all_loads();
  __syncthreads();
  Pack8 kf[KS], vf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    kf[ks] = lds_read16(tile_frag_addr<HD>(ldsQ + (uint32_t)(kq * 32 * RB) + rowoff, ks));
    vf[ks] = lds_read16(tile_frag_addr<HD>(ldsdO + (uint32_t)(kq * 32 * RB) + rowoff, ks));
    if (D < HD && tile_frag_piece<HD>(hh, ks) * 8 >= D) kf[ks] = vf[ks] = zero_pack8();
  }
  // partials form: K^T of this wave's features, the A operand of dQ^T = K^T dS^T (keys 16 s4 + 8 hh .. + 7)
  Pack8 ktf[DQP ? NDW : 1][4];
  if constexpr (DQP) {
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int d = 0; d < NDW; ++d) {
        uint32_t ad[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int key = 16 * s4 + 8 * hh + 4 * u + (li >> 2);
          ad[u] = ldsQ + (uint32_t)(key * RB + ((((kq * NDW + d) * 4 + ((lane >> 4) & 1) * 2 + ((li & 3) >> 1)) ^ tile_swz<HD>(key)) * 16) + (li & 1) * 8);
        }
        ktf[d][s4] = lds_tr8(ad[0], ad[1]);
      }
  }
  __syncthreads();
  if (nround > 0) {
    // rows of a round (ids `rid`): Q and dO into the buffer, 16 rows per wave, of its own 32
    int ft = tid;  // thread index for the code around the products, re-made opaque in every round: what is derived from it is not kept in registers
    // What a round's head has of its own: changes when the walk goes on to the next head of the group.
    struct Head {
      int h;
      const uint16_t *q, *dout;
      const float *lse, *del;
    };
    auto head_at = [&](int h) {
      return Head{h, qg + (int64_t)h * a.q_head_stride, dog + (int64_t)h * a.do_head_stride, a.softmax_lse + (int64_t)h * a.total_q + q0,
                  a.softmax_d + (int64_t)h * dstride + q0 + 128 * b};
    };
    Head hd = head_at(w0.h);
    uint32_t fsrc[NI];  // the rows this lane fetches pieces of
    auto feed_rows = [&](int rid) {  // (all exchanges at once: one wait for them)
#pragma unroll
      for (int i = 0; i < NI; ++i) fsrc[i] = (uint32_t)__shfl(rid, kq * 16 + (i * 64 + (ft & 63)) / VPR, 64);
    };
    auto feed = [&](auto ic, uint32_t buf) {  // load ic of Q and of dO
      constexpr int I = decltype(ic)::value;
      const int v = I * 64 + (ft & 63), r16 = v / VPR, pc = v - r16 * VPR, tr = kq * 16 + r16;  // row of the tile of 32, piece
      const uint32_t src = fsrc[I] & 0x7fffffffu;
      const uint32_t e = (uint32_t)min((pc ^ tile_swz<HD>(tr)) * 8, D - 8);
      const uint32_t dst = buf + (uint32_t)((rt * 32 + kq * 16) * RB + I * 1024);
      if constexpr (NEAR) {
        global_to_lds16_sbase(mul24_u32(src, (uint32_t)a.q_row_stride * 2u) + e * 2u, hd.q, ldsQ + dst);
        global_to_lds16_sbase(mul24_u32(src, (uint32_t)a.do_row_stride * 2u) + e * 2u, hd.dout, ldsdO + dst);
      } else {
        global_to_lds16(hd.q + ((uint64_t)src * (uint32_t)a.q_row_stride + e), ldsQ + dst);
        global_to_lds16(hd.dout + ((uint64_t)src * (uint32_t)a.do_row_stride + e), ldsdO + dst);
      }
    };
    int rid0 = code(raw0, w0), rid1 = code(raw_nx, w1);
    feed_rows(rid0);
    static_for<NI>([&](auto ic) { feed(ic, 0u); });
    float lse = 0.f, del = 0.f;
    int slot = 0;
    int *sSlot = reinterpret_cast<int *>(smem + SM::oSlot);
    const int trash = a.total_q * a.heads * ws.cap;  // a spare part row: takes what absent rows and visits beyond the caller's bound write
    // LSE, delta and (partials form, handed out by the waves of key quarter 0) the part row of a round's rows
    auto scalars = [&](int rid, int rank, const Round &w, bool counted) {
      const int rc = rid & 0x7fffffff;
      if constexpr (NEAR) {  // (offsets of 32 bits)
        lse = *reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(hd.lse) + (uint32_t)rc * 4u);
        del = *reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(hd.del) + (uint32_t)rc * 4u);
      } else {
        lse = hd.lse[rc];
        del = hd.del[rc];
      }
      if constexpr (DQP && RANKED)
        slot = rank * nsub + jsub;
      else if constexpr (DQP)
        slot = take_slot(ws.cnt + ((int64_t)(q0 + rc) * a.heads + w.h), rid >= 0 && hh == 0 && kq == 0 && counted);
    };
    auto arrived = [&]() {
      wait_all_loads();
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(lse), "+v"(del), "+v"(raw_nx), "+v"(slot));
#endif
    };
    int rank1 = raw_nx >> kListRowBits;  // (of ranked lists)
    scalars(rid0, raw0 >> kListRowBits, w0, true);
    arrived();
    __syncthreads();
    uint32_t buf = 0u;
    for (int r = 0; r < nround; ++r) {
#if defined(__HIP_DEVICE_COMPILE__)
      if constexpr (DQP) asm volatile("" : "+v"(ft));
#endif
      // places of this lane in the P and dS rows (and of its row in a round)
      const int fl = ft & 63, fh = fl >> 5, fli = fl & 15, frow = rt * 32 + (fl & 31), fr = (fli >> 2) + 4 * fh;
      const uint32_t pw = (uint32_t)(frow * PRB + fh * 8), psw = (uint32_t)tile_swz<64>(frow);
      const uint32_t pread = (uint32_t)(fr * PRB + (((((fl >> 4) & 1) * 2 + ((fli & 3) >> 1)) ^ tile_swz<64>(fr)) * 16) + (fli & 1) * 8);
      const Round w2 = round_at(r + 2);
      const float lse2 = rid0 >= 0 ? lse * kLog2e : INFINITY, delta = del;
      if constexpr (DQP) {
        if (kq == 0 && fh == 0) sSlot[(r & 1) * 64 + frow] = (rid0 >= 0 && slot < ws.cap) ? ((q0 + rid0) * a.heads + w0.h) * ws.cap + slot : trash;
      }
      // The next round's rows and scalars, the row ids of the one after it.  The rows are asked for between the products of S and dP, a
      // load of Q and one of dO after every four, by 32-bit offsets.  Before the products, one after the other with an exchange, a wait for it and a
      // 64-bit product each, and with the head's addresses made anew every round: 65536 tokens in eight sequences, training step 7543
      // us against 7430 now, 24571 tokens, 32 over 8 heads 2782 -> 2720, 12037 tokens, heads of 96 479 -> 473, 2 x 4096 tokens 482 -> 477.
      if (w1.h != hd.h) hd = head_at(w1.h);
      feed_rows(rid1);
      scalars(rid1, rank1, w1, r + 1 < nround);
      raw_nx = *entry_at(w2);
      // S^T and dP^T: lane -> row, register i -> key kq * 32 + acc_row(i, hh)
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.f;
      const uint32_t aq = ldsQ + buf + (uint32_t)(rt * 32 * RB) + rowoff, ad = ldsdO + buf + (uint32_t)(rt * 32 * RB) + rowoff;
      constexpr int NB = DQP ? 1 : 2;  // k-steps per batch of reads
      Pack8 qf[2][NB], df[2][NB];
      auto rd = [&](auto bc) {
        constexpr int B = decltype(bc)::value;
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          qf[B & 1][u] = lds_read16(tile_frag_addr<HD>(aq, B * NB + u));
          df[B & 1][u] = lds_read16(tile_frag_addr<HD>(ad, B * NB + u));
        }
      };
      rd(std::integral_constant<int, 0>{});
      static_for<KS / NB>([&](auto bc) {
        constexpr int B = decltype(bc)::value;
        if constexpr (B + 1 < KS / NB) rd(std::integral_constant<int, B + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          s = mfma32<T>(kf[B * NB + u], qf[B & 1][u], s);
          dp = mfma32<T>(vf[B * NB + u], df[B & 1][u], dp);
        }
        if constexpr (B < NI) {
          if (r + 1 < nround) feed(bc, buf ^ TILE);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      const int lim = rid0 < 0 ? -1 : min(causal ? rid0 + off : 0x7fffffff, Lk - 1) - key0 - kq * 32;  // last visible key of this wave's 32
      if (!__all(lim >= 31)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + (i & 3) + 4 * hh <= lim ? s[i] : -INFINITY;
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float p[4], d[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          p[j] = __builtin_amdgcn_exp2f(fmaf(s[4 * g + j], scale_log2, -lse2));
          d[j] = p[j] * (dp[4 * g + j] - delta);
        }
        const uint32_t at = pw + (((uint32_t)(kq * 4 + g) ^ psw) * 16u);
        lds_write_vec<uint2>(ldsP + at, make_uint2(pack2<T>(p[0], p[1]), pack2<T>(p[2], p[3])));
        lds_write_vec<uint2>(ldsdS + at, make_uint2(pack2<T>(d[0], d[1]), pack2<T>(d[2], d[3])));
      }
      __syncthreads();  // P and dS of the round are in LDS
      // dV^T[f][key] += dO^T[f][row] P[row][key], dK^T[f][key] += Q^T[f][row] dS[row][key]
      const uint32_t tx = (sel ? ldsQ : ldsdO) + buf + troff, px = (sel ? ldsdS : ldsP) + pread;
      Pack8 pb[2][NKW], xa[2][NDW];
      auto rd2 = [&](auto sc) {
        constexpr int S4 = decltype(sc)::value;
#pragma unroll
        for (int kk = 0; kk < NKW; ++kk) {
          const uint32_t o = (uint32_t)(S4 * 16 * PRB);
          pb[S4 & 1][kk] = lds_tr8(tile_tr_addr<64>(px, kk0 + kk) + o, tile_tr_addr8<64>(px, kk0 + kk) + o);
        }
#pragma unroll
        for (int d = 0; d < NDW; ++d) {
          const uint32_t o = (uint32_t)(S4 * 16 * RB);
          xa[S4 & 1][d] = lds_tr8(tile_tr_addr<HD>(tx, d0 + d) + o, tile_tr_addr8<HD>(tx, d0 + d) + o);
        }
      };
      rd2(std::integral_constant<int, 0>{});
      static_for<4>([&](auto sc) {
        constexpr int S4 = decltype(sc)::value;
        if constexpr (S4 < 3) rd2(std::integral_constant<int, S4 + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < NDW; ++d)
#pragma unroll
          for (int kk = 0; kk < NKW; ++kk) acc[d][kk] = mfma32<T>(xa[S4 & 1][d], pb[S4 & 1][kk], acc[d][kk]);
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (DQP) {
        // dQ^T[f][row] of this wave's 32 rows and its share of the features, over all keys of the block
        f32x16 dq[NDW];
#pragma unroll
        for (int d = 0; d < NDW; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) dq[d][i] = 0.f;
        Pack8 sf[2][2];
        auto rd3 = [&](auto sc) {
          constexpr int S = decltype(sc)::value;
#pragma unroll
          for (int u = 0; u < 2; ++u) sf[S & 1][u] = lds_read16(ldsdS + (uint32_t)(frow * PRB) + (((uint32_t)(2 * (2 * S + u) + fh) ^ psw) * 16u));
        };
        rd3(std::integral_constant<int, 0>{});
        static_for<2>([&](auto sc) {
          constexpr int S = decltype(sc)::value;
          if constexpr (S + 1 < 2) rd3(std::integral_constant<int, S + 1>{});
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int d = 0; d < NDW; ++d) dq[d] = mfma32<T>(ktf[d][2 * S + u], sf[S & 1][u], dq[d]);
          __builtin_amdgcn_sched_barrier(0);
        });
        // rows through LDS, so that a row's 16-byte pieces leave together (piece p of row r at p ^ tile_swz<64>(r))
        const uint32_t ldsOut = lds + (uint32_t)SM::oOut;
#pragma unroll
        for (int d = 0; d < NDW; ++d)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            lds_write_vec<uint2>(ldsOut + (uint32_t)(frow * RB + fh * 8) + (((uint32_t)((kq * NDW + d) * 4 + g) ^ psw) * 16u),
                                 pack4_scaled<T>(dq[d][4 * g], dq[d][4 * g + 1], dq[d][4 * g + 2], dq[d][4 * g + 3], dq_part_scale<T>(a.softmax_scale)));
        arrived();
        __syncthreads();  // the part rows are there; the next round's rows are, and this one's are no longer read
#pragma unroll
        for (int v0 = 0; v0 < 64 * VPR; v0 += 256) {
          const int v = v0 + ft, row = v / VPR, pcs = v - row * VPR;
          const uint32_t p = (uint32_t)sSlot[(r & 1) * 64 + row];
          const Pack8 x = lds_read16(ldsOut + (uint32_t)(row * RB) + (((uint32_t)pcs ^ (uint32_t)tile_swz<64>(row)) * 16u));
          if (pcs * 8 < PD) st_stream16(ws.part + ((uint64_t)p * (uint32_t)PD + (uint32_t)(pcs * 8)), x);
          if (!RANKED && pcs == 0) ws.pid[p] = nb;
        }
      } else {
        // dS of row `lane`, key groups 2 wave and 2 wave + 1: consecutive lanes write consecutive pieces of the dS tile
        Pack8 x[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) x[u] = lds_read16(ldsdS + (uint32_t)(lane * PRB) + (((uint32_t)(2 * wave + u) ^ (uint32_t)tile_swz<64>(lane)) * 16u));
        arrived();
        if (lane < w0.n) {
          uint16_t *dst = ds_piece(ws.ds, w0.pos, lane, (koff >> 3) + 2 * wave, Bn >> 3);
#pragma unroll
          for (int u = 0; u < 2; ++u) *reinterpret_cast<Pack8 *>(dst + 256 * u) = x[u];
        }
        __syncthreads();  // the next round's rows are in LDS, this one's are no longer read
      }
      w0 = w1, rid0 = rid1;
      w1 = w2, rid1 = code(raw_nx, w2), rank1 = raw_nx >> kListRowBits;
      buf ^= TILE;
    }
    __syncthreads();  // (the last part rows have left LDS)
  }

  // ---- dK^T / dV^T leave as rows, once ----
  float *red = reinterpret_cast<float *>(smem);  // [dV, dK][keys][LDR]
#pragma unroll
  for (int d = 0; d < NDW; ++d)
#pragma unroll
    for (int kk = 0; kk < NKW; ++kk)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4 *>(red + (size_t)(sel * NKEY + (kk0 + kk) * 32 + (lane & 31)) * LDR + (d0 + d) * 32 + 8 * g + 4 * hh) =
            f32x4{acc[d][kk][4 * g], acc[d][kk][4 * g + 1], acc[d][kk][4 * g + 2], acc[d][kk][4 * g + 3]};
  __syncthreads();
  uint16_t *dkg = reinterpret_cast<uint16_t *>(a.dk) + (int64_t)(k0 + key0) * a.dk_row_stride + (int64_t)hg * a.dk_head_stride;
  uint16_t *dvg = reinterpret_cast<uint16_t *>(a.dv) + (int64_t)(k0 + key0) * a.dv_row_stride + (int64_t)hg * a.dv_head_stride;
  for (int v = tid; v < NKEY * VPR; v += 256) {
    const int key = v / VPR, e = (v - key * VPR) * 8;
    if (key0 + key >= Lk || e >= D) continue;
    const float *s0 = red + (size_t)key * LDR + e, *s1 = s0 + NKEY * LDR;
    Pack8 ov, ok;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      ov.w[w] = pack2<T>(s0[2 * w], s0[2 * w + 1]);
      ok.w[w] = pack2<T>(s1[2 * w] * a.softmax_scale, s1[2 * w + 1] * a.softmax_scale);
    }
    *reinterpret_cast<Pack8 *>(dvg + (int64_t)key * a.dv_row_stride + e) = ov;
    *reinterpret_cast<Pack8 *>(dkg + (int64_t)key * a.dk_row_stride + e) = ok;
  }
}

// dK / dV and dQ partials at head dimension 128 (the long calls).  Four waves of 512 registers, one per SIMD, all of which
// compute: each keeps 32 keys x head_dim of dK^T and dV^T and its K and V operands in registers, and runs the softmax
// arithmetic of one tile between the products of another.
// KB = 1: the workgroup owns 64 keys, wave pair px takes tiles 2 px, 2 px + 1 of a round and wave kq of the pair the
// key half kq.  KB = 2 (columns of a multiple of 128 keys, whose two 64-key blocks share one row list): it owns 128
// keys, every wave takes all four tiles for its key quarter kq, so a gathered row serves twice the keys and a visit
// leaves one dQ partial instead of two.
// NEAR: the host has checked that a gathered row's place in q and dout is a 32-bit byte offset from the sequence's first
// row that one 24-bit multiply makes (launch_dkdv); otherwise the loads take 64-bit addresses per lane.
// LISTED: the block is looked up (listed_item).  An instance of its own, for ranked lists with NEAR: with the look-up as a branch beside the other decoding
// every launch was slower (256 and 237 registers either way; 32768 tokens, 32 heads: 3.77 ms against 3.54).
template <typename T, int HD, int KB, bool NEAR, bool RANKED, bool LISTED>
__global__ __launch_bounds__(256) void attn_bwd_dkdv_partials_kernel(fmoba_attn_bwd_args a, BwdWs ws, ItemOrder order) {
  typedef BwdSmem<HD> SM;
  constexpr int KS = HD / 16, LDQ = SM::LDQ, LDS_ = SM::LDS_, NDT = HD / 32, VPR = HD / 8, LDR = SM::LDR;
  constexpr int NKEY = 64 * KB;         // keys of the workgroup
  constexpr int NDH = NDT / (2 * KB);   // feature tiles of dQ per wave
  constexpr int LDH = NDH * 32 + 8;     // elements, per-wave dQ part-row tile [32][LDH]
  static_assert(NDH >= 1, "128-key workgroups need head_dim 128");
  static_assert((size_t)KB * 32 * LDH * 2 <= SM::tileBytes, "the dQ part rows of KB waves pass through a tile");
  constexpr uint32_t TB = (uint32_t)SM::tileBytes;
  constexpr int RB = HD * 2;    // bytes of a tile row
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int *sRid = reinterpret_cast<int *>(smem + SM::oRid);
  int *sRow = reinterpret_cast<int *>(smem + SM::oRow);
  int *sSlot = reinterpret_cast<int *>(smem + SM::oSlot);
  float *sLse = reinterpret_cast<float *>(smem + SM::oLse);
  float *sDelta = reinterpret_cast<float *>(smem + SM::oDelta);

  int nb, b, h;
  if constexpr (LISTED) {
    const BlockItem item = listed_item<NKEY, false>(blockIdx.x, a.batch, a.heads, a.max_seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    nb = item.idx, b = item.b, h = item.h;
  } else {
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * a.heads, (a.max_seqlen_k + NKEY - 1) / NKEY, (int64_t)a.max_seqlen_q * HD * 4 >= kOnePairBytes, order == kLongestFirst);
    nb = item.idx, b = item.pair / a.heads, h = item.pair - b * a.heads;
  }
  const int key0 = nb * NKEY;
  // One workgroup per compute unit: nothing covers the dependent loads before the first round, so their chain is kept
  // short.  Where the block's column list lies depends on nothing that is loaded (but for a block that is looked up): asked for together with the
  // sequence bounds.
  const int Bn = a.lg_block_n;
  const int c = key0 / Bn;
  const int64_t bh = (int64_t)b * a.heads + h;
  int nnz = 0;
  int64_t lbase = 0;
  if (c < a.max_cols) {
    nnz = a.col_nnz[bh * a.max_cols + c];
    lbase = a.col_offsets[bh * a.max_cols + c];
  }
  const int k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  if (key0 >= Lk) return;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int off = Lk - Lq;
  const int D = a.head_dim, PD = part_row_elems(a.head_dim, 2);
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = lane >> 5;
  const int kq = KB == 1 ? (wave & 1) : wave;  // this wave's 32 keys of the block, and its share of the dQ features
  const int px = KB == 1 ? (wave >> 1) : 0;    // KB = 1: wave pair, takes tiles 2 px and 2 px + 1 of every round
  const bool causal = a.is_causal != 0;
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;
  constexpr float kLog2e = 1.4426950408889634f;

  // ---- the key block: through LDS into registers.  The loads are issued first and stored after the look-up of
  // the column list below, so that the two chains of dependent loads wait together (one workgroup per compute
  // unit: nothing else covers them) ----------------------------------------------
  constexpr int NKV = NKEY * VPR / 256;
  Pack8 xk[NKV], xv[NKV];
  {
    const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)(k0 + key0) * a.k_row_stride + (int64_t)hk * a.k_head_stride;
    const uint16_t *vp = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)(k0 + key0) * a.v_row_stride + (int64_t)hk * a.v_head_stride;
#pragma unroll
    for (int i = 0; i < NKV; ++i) {
      const int v = tid + 256 * i;
      const int key = v / VPR, e = (v - key * VPR) * 8;
      xk[i] = zero_pack8();
      xv[i] = zero_pack8();
      if (key0 + key < Lk && e < D) {
        xk[i] = ld_global16(kp + (int64_t)key * a.k_row_stride + e);
        xv[i] = ld_global16(vp + (int64_t)key * a.v_row_stride + e);
      }
    }
  }

  // ---- this block's column list --------------------------------------------------------------
  // The rows of the first two rounds are asked for together with the probes of the search below, as if the walk
  // began at the head of the list (it does unless rows of the list lie before the block); otherwise they are
  // fetched again.
  int spec01[2] = {0, 0};
  const int nsub = Bn / NKEY, jsub = (key0 - c * Bn) / NKEY;  // key blocks of the column, this one's number
  if (tid < kBwdRoundRows && nnz > 0) {
#pragma unroll
    for (int sr = 0; sr < 2; ++sr) spec01[sr] = a.row_indices[lbase + min(sr * kBwdRoundRows + tid, nnz - 1)];
  }
  int start = 0;
  // rows r with r + off < key0 see no key of this block
  constexpr int row_mask = RANKED ? kListRowMask : -1;
  if (causal && nnz > 0) start = lower_bound_wave_i32(a.row_indices + lbase, nnz, key0 - off, row_mask);
  const int32_t *list = a.row_indices + lbase + start;
  const int n = nnz - start;               // rows of the list that the block walks
  const int nround = (n + kBwdRoundRows - 1) / kBwdRoundRows;
  int rid01[2] = {-1, -1};         // threads 0..127: row ids of rounds 0 and 1
  int rank01[2] = {0, 0};
  if (tid < kBwdRoundRows && n > 0) {
#pragma unroll
    for (int sr = 0; sr < 2; ++sr) {
      const int j = sr * kBwdRoundRows + tid;
      const int r = start == 0 ? spec01[sr] : list[min(j, n - 1)];
      rid01[sr] = tile_row_code(r & row_mask, j < n, Lq);
      rank01[sr] = r >> kListRowBits;
    }
  }

  {
    uint16_t *sK = reinterpret_cast<uint16_t *>(smem), *sV = sK + NKEY * LDQ;
#pragma unroll
    for (int i = 0; i < NKV; ++i) {
      const int v = tid + 256 * i;
      const int key = v / VPR, e = (v - key * VPR) * 8;
      *reinterpret_cast<Pack8 *>(sK + key * LDQ + e) = xk[i];
      *reinterpret_cast<Pack8 *>(sV + key * LDQ + e) = xv[i];
    }
  }
  __syncthreads();
  // B operands of S and dP: this lane's key, its half of the head dim; K^T of this wave's half of the features for
  // the dQ products.  They never change, so they stay in registers.
  u32x4_t kb[KS], vb[KS];  // (in accumulation registers)
  u32x4_t kt[NDH][4 * KB];  // (in accumulation registers)
  {
    const uint16_t *sK = reinterpret_cast<const uint16_t *>(smem), *sV = sK + NKEY * LDQ;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      kb[t] = pack8_vec(*reinterpret_cast<const Pack8 *>(sK + (kq * 32 + (lane & 31)) * LDQ + (hh * KS + t) * 8));
      vb[t] = pack8_vec(*reinterpret_cast<const Pack8 *>(sV + (kq * 32 + (lane & 31)) * LDQ + (hh * KS + t) * 8));
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+a"(kb[t]), "+a"(vb[t]));
#endif
    }
    lds_cu16 *trK = tr_lane_base(sK, LDQ, lane) + 8 * hh * LDQ;
#pragma unroll
    for (int s4 = 0; s4 < 4 * KB; ++s4)
#pragma unroll
      for (int d2 = 0; d2 < NDH; ++d2) {
        const int lo = 16 * s4 * LDQ + (kq * NDH + d2) * 32;
        kt[d2][s4] = pack8_vec(tr_frag8_at(trK, lo, lo + 4 * LDQ));
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+a"(kt[d2][s4]));
#endif
      }
  }

  const uint16_t *qg = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride;
  const uint16_t *dog = reinterpret_cast<const uint16_t *>(a.dout) + (int64_t)q0 * a.do_row_stride + (int64_t)h * a.do_head_stride;
  const float *lseg = a.softmax_lse + (int64_t)h * a.total_q + q0;
  const float *delg = a.softmax_d + (int64_t)h * ((int64_t)a.total_q + 128 * (int64_t)a.batch) + q0 + 128 * b;
  int32_t *cntg = ws.cnt + (int64_t)q0 * a.heads + h;  // counter of local row r: cntg[r * heads]
  float *red = reinterpret_cast<float *>(smem);  // [2][NKEY][LDR]: dV^T, dK^T on their way out

  f32x16 dv[NDT], dk[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dv[dt][i] = 0.f;
      dk[dt][i] = 0.f;
    }

  if (nround > 0) {
    // ---- feeding the tiles --------------------------------------------------------------------------
    // Nothing passes through registers: every wave fetches one of the four tiles of the NEXT round with loads that
    // write straight to LDS, issued in the first half of a round and awaited at its end.  Threads 0..127 carry the
    // per-row scalars: the row id of round s+2 (it has to be in LDS one round before the tile loads that use it),
    // and LSE, delta and the dQ-partial slot of round s+1.
    const uint32_t ldsQ = (uint32_t)(uintptr_t)(smem + SM::oQ), ldsdO = (uint32_t)(uintptr_t)(smem + SM::odO);
    int v_rank = rank01[1];  // RANKED: the rank of the entry of v_rid
    int n_rid = -1, v_rid = rid01[1], m_rid = -1, m_slot = 0;  // v_rid: the checked row id that was stored last = the one of the next round
    float m_lse = 0.f, m_del = 0.f;
    int ft = tid;  // thread index for the feeding code, re-made opaque in every round (see below)
    auto rid_issue = [&](int sr) {
      if (tid < kBwdRoundRows) {
        n_rid = list[min(sr * kBwdRoundRows + ft, n - 1)];  // used (and checked) only when it is stored: no wait for it here
      }
    };
    auto rid_store = [&](int sr) {
      if (tid < kBwdRoundRows) {
        const int j = sr * kBwdRoundRows + ft;
        v_rid = tile_row_code(n_rid & row_mask, j < n, Lq);
        v_rank = n_rid >> kListRowBits;
        sRid[(sr & 1) * kBwdRoundRows + ft] = v_rid;
      }
    };
    auto meta_issue = [&](int rid, int rank) {  // rid: this thread's row of the round after the current one
      if (tid < kBwdRoundRows) {
        m_rid = rid;
        const int rc = max(m_rid, 0);
        m_lse = lseg[rc];
        m_del = delg[rc];
        // every visit of a (row, key block) pair takes one dQ-partial slot of the row
        if constexpr (RANKED)
          m_slot = rank * nsub + jsub;
        else if (m_rid >= 0)
          m_slot = atomicAdd(cntg + (int64_t)m_rid * a.heads, 1);
      }
    };
    const int64_t trash = (int64_t)a.total_q * a.heads * ws.cap;  // spare row: takes the writes of absent rows, no branch
    auto meta_store = [&](int sr) {
      if (tid < kBwdRoundRows) {
        const int i = (sr & 1) * kBwdRoundRows + ft;
        const bool ok = m_rid >= 0;
        sRow[i] = m_rid;
        // where the visit's dQ partial goes, as an index of partial rows (2^31 of them would be half a terabyte): the
        // row's slot, or the spare row for an absent row and for a visit beyond the caller's bound
        sSlot[i] = (ok && m_slot < ws.cap) ? (int)((((int64_t)(q0 + m_rid)) * a.heads + h) * ws.cap + m_slot) : (int)trash;
        sLse[i] = ok ? m_lse * kLog2e : INFINITY;  // absent rows: exp2(x - inf) = 0
        sDelta[i] = ok ? m_del : 0.f;
      }
    };
    auto tile_issue = [&](int sr) {  // tile `wave` of round sr
      constexpr int RPI = 64 / VPR, NI = 32 / RPI;  // tile rows per instruction, instructions per tile
      const int fl = ft & 63, rl = fl / VPR, p = fl - rl * VPR;
      const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane(((sr & 1) * 4 + wave) * (int)TB);
      const uint32_t qs = (uint32_t)a.q_row_stride, dos = (uint32_t)a.do_row_stride;  // (32 x 32 -> 64-bit products: one instruction each)
      // Absent rows and features past head_dim are fetched from a row and a piece that exist (tile_row_code): every
      // load is unconditional, and what such data meets is an exact zero (probabilities of absent rows, K / V features
      // past head_dim) or is never written out.
      int src[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) src[i] = sRid[(sr & 1) * kBwdRoundRows + wave * 32 + i * RPI + rl] & 0x7fffffff;
      if constexpr (NEAR) {
        // the sequence's rows lie within 4 GB of its first one: a 32-bit byte offset per lane from a wave-uniform base,
        // one full-rate multiply (the 64-bit products take four times as long, and an address takes two more additions)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const uint32_t e2 = (uint32_t)min((p ^ tile_swz<HD>(i * RPI + rl)) * 8, D - 8) * 2u;
          global_to_lds16_sbase(mul24_u32((uint32_t)src[i], qs * 2u) + e2, qg, ldsQ + dst + (uint32_t)(i * RPI * RB));
          global_to_lds16_sbase(mul24_u32((uint32_t)src[i], dos * 2u) + e2, dog, ldsdO + dst + (uint32_t)(i * RPI * RB));
        }
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const uint32_t e = (uint32_t)min((p ^ tile_swz<HD>(i * RPI + rl)) * 8, D - 8);
          global_to_lds16(qg + ((uint64_t)(uint32_t)src[i] * qs + e), ldsQ + dst + (uint32_t)(i * RPI * RB));
          global_to_lds16(dog + ((uint64_t)(uint32_t)src[i] * dos + e), ldsdO + dst + (uint32_t)(i * RPI * RB));
        }
      }
    };

    // The same loads one at a time, for rows near the base.  A load instruction of a kilobyte holds the wave for about
    // 70 clocks while the unit's four waves issue theirs together (the unit's vector memory path takes 64 bytes per
    // clock: a round's 64 KB are a thousand clocks of it), and a wave that waits there issues no products either.  So
    // the Q loads go between the products of the round's first stage, one per two products, and the dO loads between
    // those of the second, instead of all at the start of the round; the offsets stay in registers until then.  (With
    // a test per load of whether the rows are near, that gain was lost: hence the NEAR instantiations.)
    constexpr bool kSpreadLoads = NEAR;
    constexpr int NTI = 32 / (64 / VPR);  // load instructions per tile and operand
    static_assert(NTI == KS, "one pair of tile loads per k-step of the first stage");
    uint32_t t_q[kSpreadLoads ? NTI : 1], t_do[kSpreadLoads ? NTI : 1], t_dst = 0;  // byte offsets of this lane's pieces
    auto tile_rows = [&](int sr) {
      constexpr int RPI = 64 / VPR;
      const int fl = ft & 63, rl = fl / VPR, p = fl - rl * VPR;
      t_dst = (uint32_t)__builtin_amdgcn_readfirstlane(((sr & 1) * 4 + wave) * (int)TB);
      const uint32_t qs = (uint32_t)a.q_row_stride, dos = (uint32_t)a.do_row_stride;
#pragma unroll
      for (int i = 0; i < (kSpreadLoads ? NTI : 0); ++i) {
        const uint32_t src = (uint32_t)(sRid[(sr & 1) * kBwdRoundRows + wave * 32 + i * RPI + rl] & 0x7fffffff);
        const uint32_t e2 = (uint32_t)min((p ^ tile_swz<HD>(i * RPI + rl)) * 8, D - 8) * 2u;
        t_q[i] = mul24_u32(src, qs * 2u) + e2;
        t_do[i] = mul24_u32(src, dos * 2u) + e2;
      }
    };
    auto tile_issue_q = [&](auto ic) {
      constexpr int I = decltype(ic)::value, RPI = 64 / VPR;
      if constexpr (kSpreadLoads) global_to_lds16_sbase(t_q[I], qg, ldsQ + t_dst + (uint32_t)(I * RPI * RB));
    };
    auto tile_issue_do = [&](auto ic) {
      constexpr int I = decltype(ic)::value, RPI = 64 / VPR;
      if constexpr (kSpreadLoads) global_to_lds16_sbase(t_do[I], dog, ldsdO + t_dst + (uint32_t)(I * RPI * RB));
    };

    if (tid < kBwdRoundRows) {
      sRid[tid] = rid01[0];
      sRid[kBwdRoundRows + tid] = rid01[1];
    }
    __syncthreads();  // K, V are in registers; the row ids of rounds 0 and 1 are in LDS
    meta_issue(rid01[0], rank01[0]);
    tile_issue(0);
    meta_store(0);
    wait_all_loads();
    __syncthreads();

    // ---- compute-wave stages ---------------------------------------------------------------------
    // A wave is alone on its SIMD, so the MFMA pipe only stays busy if the softmax arithmetic
    // of one tile runs between the products of the other tile of the round.  Every stage is cut into
    // four chunks (a quarter of the products + a quarter of the softmax rows); the operands of chunk
    // g+1 are read from LDS while chunk g computes, and the scheduler is fenced between chunks: left
    // alone, the compiler sinks every read next to the MFMA that uses it and waits for it there.
    typedef std::integral_constant<int, 0> C0;
    typedef std::integral_constant<int, 1> C1;
    constexpr int KC = KS / 4;       // k-steps of S / dP per chunk
    constexpr int BC = NDT / 2;      // (d-tile, row-half) operand pairs of dV / dK per chunk
    // byte addresses of this lane's pieces in tile 0 of the pair, buffer 0: row reads (row lane % 32, pieces
    // hh * KS ..) and transposing reads (row (lane % 16) / 4 + 4 hh, feature tile 0); every other operand is an
    // exclusive-or on the piece bits plus a constant
    const uint32_t pairQ = ldsQ + (uint32_t)(px * 2) * TB, pairdO = ldsdO + (uint32_t)(px * 2) * TB;
    const uint32_t rowoff = (uint32_t)((lane & 31) * RB + (((hh * KS) ^ tile_swz<HD>(lane & 31)) * 16));
    const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
    const uint32_t troff = (uint32_t)(r0t * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
    // (no registers to spare for those: the bases are re-made opaque wherever they are used, so that nothing derived from
    // them is kept from one use to the next)
    uint32_t aQ = pairQ + rowoff, adO = pairdO + rowoff, tQ = pairQ + troff, tdO = pairdO + troff;
    auto opaque = [](uint32_t &x, uint32_t &y) {
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(x), "+v"(y));
#else
      (void)x, (void)y;
#endif
    };
    auto opaque1 = [](uint32_t &x) {
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(x));
#else
      (void)x;
#endif
    };
    uint16_t *sdS = reinterpret_cast<uint16_t *>(smem + SM::odS) + (size_t)px * 2 * 64 * LDS_;  // (px = 0 with 128 keys)
    lds_cu16 *trdS = tr_lane_base(sdS, LDS_, lane) + 8 * hh * LDS_;  // dS^T tile: 8 consecutive keys per read
    // the dQ part rows of a tile leave through the first tile of the pair, which nobody reads after the barrier in
    // the middle of the round: Q's for even waves, dO's for odd ones, one half of it each with four key quarters
    uint16_t *sdQ0 = reinterpret_cast<uint16_t *>(smem + ((kq & 1) ? SM::odO : SM::oQ) + (size_t)(px * 2) * TB + (size_t)(kq >> 1) * (TB / 2));
    const int *pRow = sRow + px * 64;
    uint32_t smx0 = (uint32_t)(uintptr_t)(smem + SM::oRow) + (uint32_t)(px * 64 * 4 + hh * 16);  // softmax inputs of this lane's rows
    Pack8 qa[2][KC], doa[2][KC];     // A operands of S and dP (this lane's row, its half of the head dim), double-buffered by chunk
    Pack8 dot[2][BC], qt[2][BC];     // dO^T / Q^T operands of the dV / dK products, double-buffered by chunk
    f32x4 lse4[2], del4[2];          // softmax inputs of a chunk's four rows
    Pack8 pf[2][2], dsf[2][2];       // P and dS of both tiles of the round as MFMA operands
    Pack8 dsx[4 * KB];               // dS^T of all keys of the block as the B operand of the dQ products
    f32x16 dqa[NDH];
    f32x16 s[2], dp[2];
    auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
    // pc: buffer of the round; pp: tile pair (always 0 with KB = 1, where the pair is part of the addresses); tsc: tile of the pair
    auto ld_a = [&](auto pc, auto pp, auto tsc, auto gc) {
      constexpr uint32_t TO = (uint32_t)(decltype(pc)::value * 4 + decltype(pp)::value * 2 + decltype(tsc)::value) * TB;
      constexpr int G = decltype(gc)::value;
      opaque(aQ, adO);
#pragma unroll
      for (int t = 0; t < KC; ++t) {
        qa[G & 1][t] = lds_read16((aQ ^ (uint32_t)((G * KC + t) * 16)) + TO);
        doa[G & 1][t] = lds_read16((adO ^ (uint32_t)((G * KC + t) * 16)) + TO);
      }
    };
    // this lane's key; key j is visible to row r iff r >= row_thr (rows that do not exist are stored as -1)
    const int j = key0 + kq * 32 + (lane & 31);
    const int row_thr = j >= Lk ? 0x7fffffff : (causal ? max(0, j - off) : 0);
    // rows from this one on see every key of the block (no row does if the block reaches past the sequence)
    const int all_visible_from = key0 + NKEY > Lk ? 0x7fffffff : (causal ? max(0, key0 + NKEY - 1 - off) : 0);
    // The causal rule and the end of the sequence enter S as its starting value: 0 where row and key see each other,
    // -inf elsewhere (the products then leave -inf there and the exponential gives 0), and only in rounds that have
    // such pairs at all (`masked`, the same for the whole wave): the rows of a list come in ascending order, so
    // from the first row that sees every key of the block on, S starts from nothing and no comparison is made.
    auto mm_a = [&](auto pc, auto pp, auto tsc, auto gc, bool masked, auto &&after_step, auto &&after_product) {
      constexpr int TS = decltype(tsc)::value, G = decltype(gc)::value;
      static_for<KC>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        if (G == 0 && t == 0) {
          if (masked) {
            constexpr int TSG = decltype(pc)::value * 4 + decltype(pp)::value * 2 + TS;
            opaque1(smx0);
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
              const int4 r4 = lds_read_vec<int4>(smx0 + (uint32_t)(TSG * 32 + 8 * g4) * 4);
              s[TS][4 * g4] = r4.x >= row_thr ? 0.f : -INFINITY;
              s[TS][4 * g4 + 1] = r4.y >= row_thr ? 0.f : -INFINITY;
              s[TS][4 * g4 + 2] = r4.z >= row_thr ? 0.f : -INFINITY;
              s[TS][4 * g4 + 3] = r4.w >= row_thr ? 0.f : -INFINITY;
            }
            mfma32_b_acc<T, false>(s[TS], qa[G & 1][t], kb[G * KC + t]);
          } else {
            mfma32_b_acc<T, true>(s[TS], qa[G & 1][t], kb[G * KC + t]);
          }
          after_product(std::integral_constant<int, 2 * t>{});
          mfma32_b_acc<T, true>(dp[TS], doa[G & 1][t], vb[G * KC + t]);
        } else {
          mfma32_b_acc<T, false>(s[TS], qa[G & 1][t], kb[G * KC + t]);
          after_product(std::integral_constant<int, 2 * t>{});
          mfma32_b_acc<T, false>(dp[TS], doa[G & 1][t], vb[G * KC + t]);
        }
        after_step(std::integral_constant<int, G * KC + t>{});
        after_product(std::integral_constant<int, 2 * t + 1>{});
      });
      if constexpr (G == 3) mfma_results_ready(s[TS], dp[TS]);
    };
    auto ld_b = [&](auto pc, auto pp, auto tsc, auto gc) {
      constexpr uint32_t TO = (uint32_t)(decltype(pc)::value * 4 + decltype(pp)::value * 2 + decltype(tsc)::value) * TB;
      constexpr int G = decltype(gc)::value;
      opaque(tQ, tdO);
#pragma unroll
      for (int t = 0; t < BC; ++t) {
        const int pi = G * BC + t, dt = pi >> 1, s2 = pi & 1;
        // rows 16 s2 + (0..3) + 4 hh and the same + 8, features dt * 32 ..
        const uint32_t olo = TO + (uint32_t)(16 * s2 * RB), ohi = olo + (uint32_t)(8 * RB);
        const uint32_t xlo = (uint32_t)(dt * 4 * 16), xhi = (uint32_t)(((dt * 4) ^ TileSwz<HD>::kRow8) * 16);
        dot[G & 1][t] = lds_tr8((tdO ^ xlo) + olo, (tdO ^ xhi) + ohi);
        qt[G & 1][t] = lds_tr8((tQ ^ xlo) + olo, (tQ ^ xhi) + ohi);
      }
    };
    auto mm_b = [&](auto tsc, auto gc, auto &&after_product) {
      constexpr int TS = decltype(tsc)::value, G = decltype(gc)::value;
      // dV^T[d][key] += dO^T[d][row] P[row][key];  dK^T[d][key] += Q^T[d][row] dS[row][key]
      static_for<BC>([&](auto tc) {
        constexpr int t = decltype(tc)::value, pi = G * BC + t, DT = pi >> 1, s2 = pi & 1;
        mfma32_c_acc<T, 2 * DT>(dv[DT], dot[G & 1][t], pf[TS][s2]);
        after_product(std::integral_constant<int, 2 * t>{});
        mfma32_c_acc<T, 2 * DT + 1>(dk[DT], qt[G & 1][t], dsf[TS][s2]);
        after_product(std::integral_constant<int, 2 * t + 1>{});
      });
    };
    auto ld_s = [&](auto pc, auto pp, auto tsc, auto gc) {
      constexpr int TS = decltype(pc)::value * 4 + decltype(pp)::value * 2 + decltype(tsc)::value, G = decltype(gc)::value;
      // accumulator registers 4G..4G+3 hold rows TS * 32 + 8 G + 4 hh + (0..3); one address register, the rest
      // are offsets in the instructions
      constexpr uint32_t O = (uint32_t)(TS * 32 + 8 * G) * 4;
      opaque1(smx0);
      lse4[G & 1] = lds_read_vec<f32x4>(smx0 + O + (uint32_t)(SM::oLse - SM::oRow));
      del4[G & 1] = lds_read_vec<f32x4>(smx0 + O + (uint32_t)(SM::oDelta - SM::oRow));
    };
    // The softmax of a chunk's four rows in four parts, one behind each of the chunk's four products: a wave issues in order, so what is to
    // run under a product has to stand right behind it.
    static_assert(KC == 2 && BC == 2, "four products per chunk");
    float pr[4], ds[4];
    auto smx = [&](auto tsc, auto gc, auto ic) {
      constexpr int TS = decltype(tsc)::value, G = decltype(gc)::value, I = decltype(ic)::value;
      pr[I] = __builtin_amdgcn_exp2f(fmaf(s[TS][4 * G + I], scale_log2, -lse4[G & 1][I]));  // (-inf for a masked pair, see mm_a)
      auto grad = [&](int jj) { ds[jj] = pr[jj] * (dp[TS][4 * G + jj] - del4[G & 1][jj]); };
      // operand register s2 = G/2 holds rows 16*s2 + 8*(w/2) + 4*hh + ..: words 2*(G%2), 2*(G%2)+1
      auto pack = [&](int w) {
        pf[TS][G >> 1].w[2 * (G & 1) + w] = pack2<T>(pr[2 * w], pr[2 * w + 1]);
        dsf[TS][G >> 1].w[2 * (G & 1) + w] = pack2<T>(ds[2 * w], ds[2 * w + 1]);
      };
      if constexpr (I > 0) grad(I - 1);
      if constexpr (I == 2) pack(0);
      if constexpr (I == 3) {
        grad(3);
        pack(1);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // dQ of the tile: both waves of a pair put dS^T of their 32 keys into one LDS tile [64 keys][32 rows]; after a
    // barrier each wave computes dQ^T = K^T dS^T over all 64 keys for ITS half of the features.  The
    // half rows (16-bit) go to the partial slot that the row handed out for this visit.
    auto ds_write = [&](auto tsc) {
      constexpr int TS = decltype(tsc)::value;
      // tile slot TS of the pair, rows of all keys of the block
      uint16_t *t = sdS + (size_t)(TS * NKEY + kq * 32 + (lane & 31)) * LDS_;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        *reinterpret_cast<uint2 *>(t + 16 * s2 + 4 * hh) = make_uint2(dsf[TS][s2].w[0], dsf[TS][s2].w[1]);
        *reinterpret_cast<uint2 *>(t + 16 * s2 + 8 + 4 * hh) = make_uint2(dsf[TS][s2].w[2], dsf[TS][s2].w[3]);
      }
    };
    auto dq_load = [&](auto tsc) {
      constexpr int TS = decltype(tsc)::value;
#pragma unroll
      for (int s4 = 0; s4 < 4 * KB; ++s4) dsx[s4] = tr_frag8_at(trdS, (TS * NKEY + 16 * s4) * LDS_, (TS * NKEY + 16 * s4 + 4) * LDS_);
    };
    auto dq_mma = [&](auto gc) {  // a quarter of the products per chunk
      constexpr int G = decltype(gc)::value;
#pragma unroll
      for (int d2 = 0; d2 < NDH; ++d2) {
#pragma unroll
        for (int t = 0; t < KB; ++t) {
          if (G == 0 && t == 0)
            mfma32_a_acc<T, true>(dqa[d2], kt[d2][G * KB + t], dsx[G * KB + t]);
          else
            mfma32_a_acc<T, false>(dqa[d2], kt[d2][G * KB + t], dsx[G * KB + t]);
        }
      }
      if constexpr (G == 3) {
        static_assert(NDH <= 2, "one or two feature tiles of dQ per wave");
        if constexpr (NDH == 1)
          mfma_results_ready(dqa[0]);
        else
          mfma_results_ready(dqa[0], dqa[1]);
      }
    };
    auto dq_store = [&](auto pc, auto pp, auto tsc) {
      constexpr int TS = decltype(pc)::value * 4 + decltype(pp)::value * 2 + decltype(tsc)::value;
      constexpr uint32_t SO = (uint32_t)(decltype(pc)::value * 4 + decltype(pp)::value * 2) * TB;  // the tile that serves as staging
      // register i of feature tile d2 <-> feature d2*32 + acc_row(i, hh) of this wave's half, this lane's row
      uint32_t bw = (uint32_t)(uintptr_t)sdQ0 + (uint32_t)(((lane & 31) * LDH + 4 * hh) * 2), unused_w = 0;
      opaque(bw, unused_w);
#pragma unroll
      for (int d2 = 0; d2 < NDH; ++d2)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          lds_write_vec<uint2>(bw + SO + (uint32_t)((d2 * 32 + 8 * g) * 2),
                               pack4_scaled<T>(dqa[d2][4 * g], dqa[d2][4 * g + 1], dqa[d2][4 * g + 2], dqa[d2][4 * g + 3], dq_part_scale<T>(a.softmax_scale)));
      wave_lds_fence();
      constexpr int LPR = NDH * 4;        // lanes per part row (16 bytes each)
      constexpr int RPP = 64 / LPR;       // rows per pass
      const int col = (lane % LPR) * 8;
      uint32_t bs = (uint32_t)(uintptr_t)(smem + SM::oRow) + (uint32_t)((px * 64 + lane / LPR) * 4);
      uint32_t bx = (uint32_t)(uintptr_t)sdQ0 + (uint32_t)(((lane / LPR) * LDH + col) * 2);
      opaque(bs, bx);
      // (one test around all rows of the tile rather than one per store: a lane either has a piece of the part
      // row or it has not)
      uint32_t pidx[32 / RPP];
#pragma unroll
      for (int k = 0; k < 32 / RPP; ++k) pidx[k] = (uint32_t)lds_read_vec<int>(bs + (uint32_t)(TS * 32 + k * RPP) * 4 + (uint32_t)(SM::oSlot - SM::oRow));
      if (kq * (NDH * 32) + col < PD) {
#pragma unroll
        for (int k = 0; k < 32 / RPP; ++k) {
          const Pack8 x = lds_read16(bx + SO + (uint32_t)(k * RPP * LDH * 2));
          st_stream16(ws.part + ((uint64_t)pidx[k] * (uint32_t)PD + (uint32_t)(kq * (NDH * 32) + col)), x);
        }
      }
      if (!RANKED && kq == 0 && col == 0) {
#pragma unroll
        for (int k = 0; k < 32 / RPP; ++k) ws.pid[pidx[k]] = nb;
      }
      wave_lds_fence();
    };
    // One round of a pair = its tiles 2 px and 2 px + 1, both already in LDS.  Tiles past the end of the list hold
    // absent rows (row id -1, zero data): they run through the same code and add nothing.
    auto process_round = [&](auto pc, auto pp, int r) {  // pc: parity of r = the LDS buffer that holds the round
      // (the first row of the pair's first tile is its earliest; -1 if the pair has no row)
      const bool masked = __builtin_amdgcn_readfirstlane(pRow[(decltype(pc)::value * 4 + decltype(pp)::value * 2) * 32]) < all_visible_from;
      // S, dP of the first tile
      ld_a(pc, pp, C0{}, C0{});
      fence();
      static_for<4>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        if constexpr (G < 3) {
          ld_a(pc, pp, C0{}, std::integral_constant<int, G + 1>{});
        } else {  // the first operands of the next stage: a stage that began with its own reads began with their latency
          ld_a(pc, pp, C1{}, C0{});
          ld_s(pc, pp, C0{}, C0{});
        }
        mm_a(pc, pp, C0{}, gc, masked, [&](auto ic) {
          if constexpr (kSpreadLoads && decltype(pp)::value == 0) tile_issue_q(ic);
        }, [](auto) {});
        fence();
      });
      // S, dP of the second tile between the softmax rows of the first
      static_for<4>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        if constexpr (G < 3) {
          ld_a(pc, pp, C1{}, std::integral_constant<int, G + 1>{});
          ld_s(pc, pp, C0{}, std::integral_constant<int, G + 1>{});
        } else {
          ld_b(pc, pp, C0{}, C0{});
          ld_s(pc, pp, C1{}, C0{});
        }
        mm_a(pc, pp, C1{}, gc, masked, [&](auto ic) {
          if constexpr (kSpreadLoads && decltype(pp)::value == 0) tile_issue_do(ic);
        }, [&](auto ic) { smx(C0{}, gc, ic); });
        fence();
      });
      // dV, dK of the first tile between the softmax rows of the second
      // (a second pair of the same waves reuses the dS^T tiles of the first: its readers have to be done)
      if constexpr (decltype(pp)::value == 1) __syncthreads();
      ds_write(C0{});
      fence();
      static_for<4>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        if constexpr (G < 3) {
          ld_b(pc, pp, C0{}, std::integral_constant<int, G + 1>{});
          ld_s(pc, pp, C1{}, std::integral_constant<int, G + 1>{});
        } else {
          ld_b(pc, pp, C1{}, C0{});
        }
        mm_b(C0{}, gc, [&](auto ic) { smx(C1{}, gc, ic); });
        fence();
      });
      // dV, dK of the second tile; dQ of the first one runs between them: by now all key
      // groups have put dS^T of both tiles into LDS, so the one barrier the exchange needs hardly ever waits
      ds_write(C1{});
      __syncthreads();
      dq_load(C0{});
      fence();
      static_for<4>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        if constexpr (G < 3) ld_b(pc, pp, C1{}, std::integral_constant<int, G + 1>{});
        mm_b(C1{}, gc, [](auto) {});
        dq_mma(gc);
        fence();
      });
      dq_store(pc, pp, C0{});
      // dQ of the second tile
      dq_load(C1{});
      fence();
      static_for<4>([&](auto gc) {
        dq_mma(gc);
        fence();
      });
      // The tiles of the next round must be in LDS before the barrier that ends this one, and one counter covers
      // loads and stores alike: the round's last partial rows are issued after that wait, so that they complete
      // under the next round instead of being waited for.
      if constexpr (KB == 1 || decltype(pp)::value == 1) {
        wait_all_loads();
        meta_store(r + 1);
        rid_store(r + 2);
      }
      dq_store(pc, pp, C1{});
    };
    auto round = [&](auto pc, int r) {
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(ft));
#endif
      rid_issue(r + 2);
      meta_issue(v_rid, v_rank);
      if constexpr (kSpreadLoads)
        tile_rows(r + 1);
      else
        tile_issue(r + 1);
      process_round(pc, C0{}, r);
      if constexpr (KB == 2) process_round(pc, C1{}, r);
      __syncthreads();  // round r + 1 is in LDS; everyone is done with round r
    };
    for (int r = 0; r < nround; r += 2) {
      round(C0{}, r);
      if (r + 1 < nround) round(C1{}, r + 1);
    }
  }

  // ---- dK^T / dV^T: every wave puts its sums into LDS (one copy per pair); with two pairs the rows add them on their way out
  __syncthreads();  // K and V have left LDS (lists without rows come here directly)
  constexpr int NCOPY = KB == 1 ? 2 : 1;
  constexpr size_t kCopy = (size_t)2 * NKEY * LDR;  // floats of one copy: dV^T then dK^T
  static_assert(NCOPY * kCopy * 4 <= SM::bytes, "the output buffers reuse the tiles");
  {
    float *mine = red + (size_t)px * kCopy;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float *rp = mine + (size_t)(kq * 32 + (lane & 31)) * LDR + dt * 32 + 8 * g + 4 * hh;
        f32x4 v4, k4;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          v4[jj] = dv[dt][4 * g + jj];
          k4[jj] = dk[dt][4 * g + jj];
        }
        *reinterpret_cast<f32x4 *>(rp) = v4;
        *reinterpret_cast<f32x4 *>(rp + NKEY * LDR) = k4;
      }
  }
  __syncthreads();

  // ---- dK^T / dV^T leave as rows, once ----------------------------------------------------------------
  uint16_t *dkg = reinterpret_cast<uint16_t *>(a.dk) + (int64_t)(k0 + key0) * a.dk_row_stride + (int64_t)h * a.dk_head_stride;
  uint16_t *dvg = reinterpret_cast<uint16_t *>(a.dv) + (int64_t)(k0 + key0) * a.dv_row_stride + (int64_t)h * a.dv_head_stride;
  for (int v = tid; v < NKEY * VPR; v += 256) {
    const int key = v / VPR, e = (v - key * VPR) * 8;
    if (key0 + key >= Lk || e >= D) continue;
    const float *s0 = red + (size_t)key * LDR + e, *s1 = s0 + NKEY * LDR;
    float fv[8], fk[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      fv[w] = s0[w];
      fk[w] = s1[w];
      if constexpr (NCOPY == 2) {
        fv[w] += s0[kCopy + w];
        fk[w] += s1[kCopy + w];
      }
    }
    Pack8 ov, ok;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      ov.w[w] = pack2<T>(fv[2 * w], fv[2 * w + 1]);
      ok.w[w] = pack2<T>(fk[2 * w] * a.softmax_scale, fk[2 * w + 1] * a.softmax_scale);
    }
    *reinterpret_cast<Pack8 *>(dvg + (int64_t)key * a.dv_row_stride + e) = ov;
    *reinterpret_cast<Pack8 *>(dkg + (int64_t)key * a.dk_row_stride + e) = ok;
  }
}

// ------------------------------------------------------------------------------------
// dQ, first form: row blocks.  One workgroup owns 256 consecutive query rows of one (sequence, head) and
// walks the 64-key blocks of every column in which one of its rows appears.  The dS rows of a step (written by the
// dK/dV pass in list order) go from global memory straight into the registers of the lane that owns the query row;
// rows that are absent contribute zeros, so every wave multiplies its own 32-row tiles and keeps dQ in registers
// for the whole walk.  All waves compute, two per SIMD (four at head dimensions up to 64), and nothing only moves data.  What a
// step needs from other threads -- its K tile (global memory straight into LDS, global_load_lds, every wave a share
// of the tile, swizzled rows of exactly head_dim elements) and the list positions of its rows (scattered into LDS by
// the thread whose index is the row's place in the step's run) -- is prepared for a whole group of G steps at once,
// one group ahead, so the workgroup meets at a barrier once per group: inside a group every wave runs at its own
// pace, and a wave's chain of dependent steps (where are my rows in this column's list -> fetch them -> multiply)
// is covered by the products of the other wave of its SIMD.
//
// What bounds it: the misses a unit can have in flight (dS pieces of 64 to 512 bytes at scattered places), and in calls of few
// workgroups the longest walk.  Head dimensions 65 to 128: four waves with two row tiles each, two workgroups per unit and
// groups of two steps; from 97 on eight waves of one tile where the walks are few and long (run_bwd draws the line).  One workgroup of eight
// waves of two tiles per unit (groups of four steps, 512 rows) read half of the K tiles
// but met at one barrier and left no unit a second walk: 65536 tokens in eight sequences, top-k 32 of 64-key chunks
// 1634 -> 1556 us, 24571 tokens, 32 over 8 heads 691 -> 624, 12037 tokens, heads of 96 182 -> 124 (with the order of the items
// below; tiles of 96 features instead of 128: 129 -> 115), 2 x 4096 tokens 143 -> 125.  Up to 64: eight waves of one tile (with two tiles in four waves 4096
// tokens 58 -> 67 us). Above 128: eight waves of one tile, one workgroup per unit (its K tiles take 128 KB).
// ------------------------------------------------------------------------------------
constexpr int kDqColBatch = 256;
constexpr int kDqMaxSteps = 512;

template <int HD, int RT, int NW>
struct DqSmem {
  static constexpr int ROWS = NW * 32 * RT;
  static constexpr int G = 2;  // steps per group (one workgroup barrier per group)
  static constexpr int NS = 2 * G;              // K tiles / position slots in LDS: the group in use and the next one
  static constexpr int LDO = HD + 8;   // elements, per-wave output tile [32 rows][LDO] (reuses the K tiles at the end)
  static constexpr size_t tileBytes = (size_t)64 * HD * 2;
  static constexpr size_t outBytes = (size_t)NW * 32 * LDO * 2;
  static constexpr size_t prepBytes = (size_t)kDqColBatch * 16 + (size_t)kDqMaxSteps * 4;
  static constexpr size_t oK = 0;                                   // [NS][64 keys][HD], swizzled; later the output tiles
  static constexpr size_t ringBytes = NS * tileBytes > outBytes ? NS * tileBytes : outBytes;
  static_assert(prepBytes <= ringBytes, "the preparation arrays lie over the K tiles");
  static constexpr size_t oTag = oK + ringBytes;                   // int[NS][ROWS]: (step tag << 10) | list position of the row in that step
  static constexpr size_t oInfo = oTag + (size_t)NS * ROWS * 4;    // int4[kDqMaxSteps]: key0, rows, list position (lo, hi)
  static constexpr size_t oMisc = oInfo + (size_t)kDqMaxSteps * 16;
  static constexpr size_t bytes = oMisc + 64;
  // what only the preparation of a batch of columns uses (no tile is in use or on its way then)
  static constexpr size_t oOff = oK;                                // int64[kDqColBatch]
  static constexpr size_t oLo = oOff + kDqColBatch * 8;
  static constexpr size_t oCnt = oLo + kDqColBatch * 4;
  static constexpr size_t oStep = oCnt + kDqColBatch * 4;
  static_assert(bytes <= 160 * 1024, "LDS of one compute unit");
};

struct DqItem {
  int pair, sb;
};
__device__ __forceinline__ DqItem dq_decode_item(int id, int npairs, int nsb_max, bool longest_first) {
  // One workgroup each for the slots of the chip (32 units per XCD, two to a unit) start all at once: the second half in
  // reverse, so that the longest walks share a unit with the shortest (4096 tokens, 32 over 8 heads: 113 -> 104 us, 8192
  // tokens, 16 heads: 198 -> 186).
  const int n = npairs % 8 == 0 ? npairs / 8 * nsb_max : 0;
  if (longest_first && n > 32 && n <= 64 && (id >> 3) >= 32) id = ((n + 31 - (id >> 3)) << 3) | (id & 7);
  // late row blocks (the longest walks) first
  const PairItem item = xcd_pair_item(id, npairs, nsb_max, false, longest_first);
  DqItem w;
  w.pair = item.pair < npairs ? item.pair : -1;
  w.sb = nsb_max - 1 - item.idx;
  return w;
}

// A buffer of (almost) 2^32 bytes from a wave-uniform address on, and 16 bytes of it at a byte offset per lane plus a constant: zeros from offset
// kRowBufferBytes on, without an access.
constexpr uint32_t kRowBufferBytes = 0xfffff000u;
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t RowBuffer;
__device__ __forceinline__ RowBuffer row_buffer(const uint16_t *p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p), 0, (int)kRowBufferBytes, 0x00020000);
}
__device__ __forceinline__ Pack8 row_buffer_load16(RowBuffer b, uint32_t lane_bytes, int offset) {
  const auto x = __builtin_amdgcn_raw_buffer_load_b128(b, (int)lane_bytes + offset, 0, 0);
  return Pack8{{x[0], x[1], x[2], x[3]}};
}
#else
typedef const uint16_t *RowBuffer;
__device__ __forceinline__ RowBuffer row_buffer(const uint16_t *p) { return p; }
__device__ __forceinline__ Pack8 row_buffer_load16(RowBuffer, uint32_t, int) { return Pack8{{0u, 0u, 0u, 0u}}; }
#endif

// RT: 32-row tiles per wave (with two, every K^T operand read from LDS feeds two MFMAs).  NW: waves.
template <typename T, int HD, int RT, int NW>
__global__ __launch_bounds__(64 * NW, HD > 64 ? 2 : 4) void attn_bwd_dq_kernel(fmoba_attn_bwd_args a, const uint16_t *ds_ws, const int32_t *tab, RunTable rt_, int row_mask, int nsb_max, ItemOrder order) {
  typedef DqSmem<HD, RT, NW> SM;
  constexpr int ROWS = SM::ROWS;  // query rows of the workgroup
  constexpr int LDO = SM::LDO, NDT = HD / 32, VPR = HD / 8;
  constexpr int RB = HD * 2;                       // bytes of a K tile row
  constexpr uint32_t TB = (uint32_t)SM::tileBytes;
  constexpr int NKI = VPR / NW;              // K load instructions per wave and tile
  static_assert(NKI >= 1 && NKI * NW == VPR, "the waves share a K tile evenly");
  constexpr int NS = SM::NS, G = SM::G;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int *sPos = reinterpret_cast<int *>(smem + SM::oTag);
  int *sLo = reinterpret_cast<int *>(smem + SM::oLo);
  int *sCnt = reinterpret_cast<int *>(smem + SM::oCnt);
  int *sStep = reinterpret_cast<int *>(smem + SM::oStep);
  int64_t *sOff = reinterpret_cast<int64_t *>(smem + SM::oOff);
  int4 *sInfo = reinterpret_cast<int4 *>(smem + SM::oInfo);
  int *sMisc = reinterpret_cast<int *>(smem + SM::oMisc);
  const uint32_t ldsK = (uint32_t)(uintptr_t)(smem + SM::oK);

  int b, h, sb, q0, Lq, k0, Lk;
  if (order == kListedLongestFirst) {
    const BlockItem item = listed_item<ROWS, true>(blockIdx.x, a.batch, a.heads, a.max_seqlen_q, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    b = item.b, h = item.h, sb = item.idx, q0 = item.q0, Lq = item.Lq, k0 = item.k0, Lk = item.Lk;
  } else {
    const DqItem wi = dq_decode_item(blockIdx.x, a.heads * a.batch, nsb_max, order == kLongestFirst);
    if (wi.pair < 0) return;
    b = wi.pair / a.heads, h = wi.pair - b * a.heads, sb = wi.sb;
    q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
    k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  }
  const int m0 = sb * ROWS;
  if (m0 >= Lq) return;
  const int rows_sb = min(ROWS, Lq - m0);
  const int off = Lk - Lq;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int Bn = a.lg_block_n, nsub = Bn / 64;
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool causal = a.is_causal != 0;

  for (int v = tid; v < NS * ROWS; v += 64 * NW) sPos[v] = 0;  // step tags start at 1

  int ncols = min((Lk + Bn - 1) / Bn, a.max_cols);
  const int last_rowpos = m0 + rows_sb - 1 + off;
  if (causal) ncols = last_rowpos < 0 ? 0 : min(ncols, last_rowpos / Bn + 1);
  const int64_t bh = (int64_t)b * a.heads + h;
  const int64_t *coff = a.col_offsets + bh * a.max_cols;
  static_assert(ROWS == kDqRows, "the row blocks of the table");
  const int32_t *runs = tab + rt_.at(h, k0 / Bn + b) + sb;  // of column 0; column c: rt_.blocks further on each
  const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)k0 * a.k_row_stride + (int64_t)hk * a.k_head_stride;
  const int cols_per_batch = min(kDqColBatch, kDqMaxSteps / nsub);

  // The steps of one batch of columns: for every column the part of its list that falls into this row block, then
  // one record per (column, 64-key block) that has rows and visible keys.  Its scratch arrays lie over the K tiles:
  // no tile is in use or on its way when the workgroup comes here.
  auto prepare_batch = [&](int cb, int cend) {
    __syncthreads();
    for (int c = cb + tid; c < cend; c += 64 * NW) {
      const int nnz = a.col_nnz[bh * a.max_cols + c];
      int lo = 0, cnt = 0;
      int64_t base = 0;
      if (nnz > 0) {
        base = coff[c];
        const int32_t *run = runs + (int64_t)c * rt_.blocks;
        lo = min(max(run[0], 0), nnz);
        cnt = min(min(max(run[1], lo), nnz) - lo, ROWS);
      }
      sLo[c - cb] = lo;
      sCnt[c - cb] = cnt;
      sOff[c - cb] = base + lo;
    }
    __syncthreads();
    if (wave == 0) {
      int nst = 0;
      for (int base = 0; base < (cend - cb) * nsub; base += 64) {
        const int idx = base + lane;
        const int cl = idx / nsub, kb = idx - cl * nsub;
        bool act = false;
        if (cl < cend - cb) {
          const int key0 = (cb + cl) * Bn + kb * 64;
          act = sCnt[cl] > 0 && key0 < Lk && !(causal && key0 > last_rowpos);
        }
        const unsigned long long m = __ballot(act);
        if (act) sStep[nst + __popcll(m & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))))] = (cl << 8) | kb;
        nst += __popcll(m);
      }
      if (lane == 0) sMisc[0] = nst;
    }
    __syncthreads();
    const int nsteps = __builtin_amdgcn_readfirstlane(sMisc[0]);
    // one record per step
    for (int st = tid; st < nsteps; st += 64 * NW) {
      const int code = sStep[st];
      const int cl = code >> 8, kb = code & 255;
      const int64_t pos0 = sOff[cl];
      // (y: rows of the run, at most ROWS, and above them the 64-key block's number inside its column)
      sInfo[st] = make_int4((cb + cl) * Bn + kb * 64, sCnt[cl] | (kb << 16), (int)(uint32_t)(pos0 & 0xffffffffll), (int)(pos0 >> 32));
    }
    __syncthreads();  // (also: everyone has read the scratch arrays before the first tile loads overwrite them)
    return nsteps;
  };

  f32x16 acc[RT][NDT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rt][dt][i] = 0.f;
  // Which rows a wave owns.  With eight waves w and w + 4 share a SIMD, and under the causal rule the later rows of the block
  // take part in more steps, so a SIMD gets the row tiles w and 7 - w: the four SIMDs then have the same number of products
  // to do.  With four waves each has a SIMD of its own (and shares it with a wave of another workgroup): tiles in order.
  const int wtile = wave < 4 ? wave : 11 - wave;
  int myrow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) myrow[rt] = (wtile * RT + rt) * 32 + (lane & 31);

  // K tile loads of this wave: lane l of instruction i brings number (wave * NKI + i) * 64 + l of the tile's pieces as they lie
  // in LDS; piece c of tile row r is stored at piece c ^ tile_swz<HD>(r)
  uint32_t ksrc[NKI];  // element offset of this lane's piece inside a tile that exists completely
#pragma unroll
  for (int i = 0; i < NKI; ++i) {
    const int v = (wave * NKI + i) * 64 + lane, r = v / VPR, kpp = v - r * VPR;
    ksrc[i] = (uint32_t)(r * (int)a.k_row_stride + min((kpp ^ tile_swz<HD>(r)) * 8, D - 8));
  }
  // K^T operands (transposing reads): lane l (i = l % 16) supplies the address of key 8 hh + i / 4 (+ 4 for the
  // second read) of a 16-key group, features 16 ((l / 16) % 2) + 4 (i % 4) .. of a 32-feature tile
  const int li = lane & 15;
  const int kk0 = 8 * hh + (li >> 2);
  const int low2 = ((lane >> 4) & 1) * 2 + ((li & 3) >> 1);
  const uint32_t tlo = (uint32_t)(kk0 * RB + ((low2 ^ tile_swz<HD>(kk0)) * 16) + (li & 1) * 8);
  const uint32_t thi = (uint32_t)((kk0 + 4) * RB + ((low2 ^ tile_swz<HD>(kk0 + 4)) * 16) + (li & 1) * 8);

  int tag_base = 0;
  Pack8 df[2][RT][4];  // this lane's dS rows of two consecutive steps (B operands)
  bool dfp[2][RT];
  int rid[G];
  for (int cb = 0; cb < ncols; cb += cols_per_batch) {
    const int nsteps = prepare_batch(cb, min(ncols, cb + cols_per_batch));
    if (nsteps == 0) continue;
    // The records of 64 steps from step wbase on, one per lane: what a step of the walk needs of them comes into scalar registers by a
    // lane read.  (Read from LDS where they are needed they were nine dependent LDS reads per group of two steps, and rows that are absent
    // were fetched from a place that exists and cleared before the products, a vector instruction per register.  Training steps without and
    // with the two: 65536 tokens in eight sequences 7393 -> 7311 us, 24571 tokens, 32 over 8 heads 2684 -> 2650, 12037 tokens, heads of 96
    // 474 -> 469, 2 x 4096 tokens, 8 heads of 256 509 -> 504, 8191 tokens of short documents 128.0 -> 126.7.)
    int4 rec = sInfo[min(lane, nsteps - 1)];
    int wbase = 0;
    struct Step {
      int key0, n, kb;  // first key, rows of the run, the 64-key block's number inside its column
      int64_t pos0;     // list position of the run
    };
    auto at = [&](int step) {
      const int l = min(step, nsteps - 1) - wbase;
      const int ny = __builtin_amdgcn_readlane(rec.y, l);
      return Step{__builtin_amdgcn_readlane(rec.x, l), ny & 0xffff, ny >> 16,
                  (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(rec.w, l) << 32) | (uint32_t)__builtin_amdgcn_readlane(rec.z, l))};
    };
    auto row_id = [&](int step) {  // row of list position tid of the step (clamped)
      const Step st = at(step);
      const uint32_t o = (uint32_t)min(tid & (ROWS - 1), st.n - 1) * 4u;
      return *reinterpret_cast<const int32_t *>(reinterpret_cast<const uint8_t *>(a.row_indices + st.pos0) + o) & row_mask;
    };
    auto put_pos = [&](int step, int rr) {  // thread t tells row rr, the t-th of the step's run, where it is
      if (step < nsteps && tid < ROWS) {
        const Step st = at(step);
        const int first_rel = causal ? st.key0 - off - m0 : -0x40000000;  // rows before it see no key of the block
        const int rel = rr - m0;
        if ((tid < st.n) & ((uint32_t)rel < (uint32_t)rows_sb) & (rel >= first_rel)) sPos[(step % NS) * ROWS + rel] = ((tag_base + step + 1) << 10) | tid;
      }
    };
    auto k_issue = [&](int step) {  // this wave's share of the K tile of `step`
      const int key0 = at(step).key0;
      const uint32_t dst = ldsK + (uint32_t)__builtin_amdgcn_readfirstlane(step % NS) * TB + (uint32_t)(wave * NKI) * 1024u;
      if (key0 + 64 <= Lk) {
        const uint16_t *kb0 = kp + (int64_t)key0 * a.k_row_stride;
#pragma unroll
        for (int i = 0; i < NKI; ++i) global_to_lds16_sbase(ksrc[i] * 2u, kb0, dst + (uint32_t)i * 1024u);
      } else {  // keys past the end of the sequence: the last key's data, which meets dS = 0
#pragma unroll
        for (int i = 0; i < NKI; ++i) {
          const int v = (wave * NKI + i) * 64 + lane, r = v / VPR, kpp = v - r * VPR;
          const int key = min(key0 + r, Lk - 1), e = min((kpp ^ tile_swz<HD>(r)) * 8, D - 8);
          global_to_lds16(kp + (int64_t)key * a.k_row_stride + e, dst + (uint32_t)i * 1024u);
        }
      }
    };
    // where this lane's rows are in the run of `step`
    auto row_pos = [&](int step, int (&v)[RT]) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) v[rt] = sPos[(min(step, nsteps - 1) % NS) * ROWS + myrow[rt]];
    };
    // Fetch this lane's dS rows of `step` (v: row_pos) into ring entry R.  A row that is absent reads past the end of the buffer that the
    // loads name, which gives zeros without an access: nothing to clear before the products.
    auto fetch = [&](auto rc, int step, const int (&v)[RT]) {
      constexpr int R = decltype(rc)::value;
      const Step st = at(step);
      const int tag = tag_base + min(step, nsteps - 1) + 1;
      // ds_piece_offset(pos0 + j, 8 kb + hh + 2 s4, Bn / 8) in two parts: what the step's run has in common (the tile of
      // its first position and the block's first piece: scalar arithmetic, 64 bits) and the lane's own part (at most
      // 9 tiles further on: 32 bits, no wide multiply among the vector instructions)
      const uint32_t kgs = (uint32_t)Bn >> 3, r0s = (uint32_t)st.pos0 & 31u;
      const RowBuffer buf = row_buffer(ds_ws + (((st.pos0 >> 5) * (int64_t)kgs + 8 * st.kb) << 8));
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const bool pres = (step < nsteps) & ((v[rt] >> 10) == tag);
        const uint32_t t = r0s + (uint32_t)(v[rt] & 1023);
        const uint32_t lane_bytes = ((mul24_u32(t >> 5, kgs) + (uint32_t)hh) << 9) + ((t & 31u) << 4);
        const uint32_t at_bytes = pres ? lane_bytes : kRowBufferBytes;
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) df[R][rt][s4] = row_buffer_load16(buf, at_bytes, 1024 * s4);
        dfp[R][rt] = pres;
      }
    };
    // the products of `step`; `between` runs after the first group of them (the tile loads of a later step: issued
    // there, they are younger than every load this step has waited for)
    auto compute = [&](auto rc, int step, auto &&between) {
      constexpr int R = decltype(rc)::value;
      bool anyp = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) anyp |= dfp[R][rt];
      if (!__any(anyp) || step >= nsteps) {
        between();
        return;
      }
      const uint32_t stage = ldsK + (uint32_t)__builtin_amdgcn_readfirstlane(step % NS) * TB;
      const uint32_t alo = tlo + stage, ahi = thi + stage;
      // K^T operands half a feature tile (two products per row tile) ahead of their use
      Pack8 kf[2][2];
      auto kread = [&](int u, Pack8 (&dst)[2]) {  // unit u: feature tile u / 2, keys 32 (u % 2) .. + 31
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const uint32_t o = (uint32_t)(16 * (2 * (u & 1) + s2) * RB);
          dst[s2] = lds_tr8(tile_tr_addr<HD>(alo, u >> 1) + o, tile_tr_addr<HD>(ahi, u >> 1) + o);
        }
      };
      kread(0, kf[0]);
#pragma unroll
      for (int u = 0; u < 2 * NDT; ++u) {
        if (u + 1 < 2 * NDT) kread(u + 1, kf[(u + 1) & 1]);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) acc[rt][u >> 1] = mfma32<T>(kf[u & 1][s2], df[R][rt][2 * (u & 1) + s2], acc[rt][u >> 1]);
        if (u == 0) between();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // before the loop: positions of steps 0 .. G, row ids of steps G + 1 .. 2 G, K tiles of steps 0 .. G - 1, dS rows of step 0
    {
      int r0[G + 1];
#pragma unroll
      for (int g = 0; g <= G; ++g) r0[g] = row_id(g);
#pragma unroll
      for (int g = 0; g < G; ++g) rid[g] = row_id(G + 1 + g);
#pragma unroll
      for (int g = 0; g <= G; ++g) put_pos(g, r0[g]);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) k_issue(g);
    __syncthreads();
    {
      int v[RT];
      row_pos(0, v);
      fetch(std::integral_constant<int, 0>{}, 0, v);
    }
    wait_all_loads();
    // group of steps s0 .. s0 + G - 1: positions of steps s0 + G + 1 .. s0 + 2 G into LDS, row ids of the G steps after
    // those, then per step the dS rows of the next step and the products of this one; the K tile loads of the next
    // group are issued among the products of the group's first step
    const int nsteps_pad = (nsteps + G - 1) / G * G;
    for (int s0 = 0; s0 < nsteps_pad; s0 += G) {
      if ((s0 & 31) == 0) {
        wbase = s0;
        rec = sInfo[min(s0 + lane, nsteps - 1)];
      }
      __syncthreads();  // the K tiles of this group and the positions up to step s0 + G are in LDS; everyone is done with the group before
#pragma unroll
      for (int g = 0; g < G; ++g) put_pos(s0 + G + 1 + g, rid[g]);
#pragma unroll
      for (int g = 0; g < G; ++g) rid[g] = row_id(s0 + 2 * G + 1 + g);
      static_for<G>([&](auto e) {
        constexpr int E = decltype(e)::value;
        const int s = s0 + E;
        int pos[RT];
        row_pos(s + 1, pos);
        fetch(std::integral_constant<int, (E + 1) & 1>{}, s + 1, pos);
        compute(std::integral_constant<int, E & 1>{}, s, [&]() {
          if constexpr (E == 0) {
#pragma unroll
            for (int g = 0; g < G; ++g) k_issue(s0 + G + g);
          }
        });
      });
      // this wave's share of the next group's K tiles has to be in LDS at the barrier: everything but the dS rows
      // fetched after it was issued
      wait_loads_but<(G - 1) * 4 * RT>();
    }
    tag_base += nsteps;
    wait_all_loads();
  }
  __syncthreads();  // every wave is done with the K tiles: they now hold the output tiles (one 32-row tile per wave)
  uint16_t *sOut = reinterpret_cast<uint16_t *>(smem + SM::oK) + (size_t)wave * 32 * LDO;
  uint16_t *op = reinterpret_cast<uint16_t *>(a.dq) + (int64_t)(q0 + m0) * a.dq_row_stride + (int64_t)h * a.dq_head_stride;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2 *>(sOut + (lane & 31) * LDO + dt * 32 + 8 * g + 4 * hh) =
            make_uint2(pack2<T>(acc[rt][dt][4 * g] * a.softmax_scale, acc[rt][dt][4 * g + 1] * a.softmax_scale),
                       pack2<T>(acc[rt][dt][4 * g + 2] * a.softmax_scale, acc[rt][dt][4 * g + 3] * a.softmax_scale));
    wave_lds_fence();
    // rows leave as 16-byte pieces, VPR of them per row, consecutive lanes taking consecutive pieces
#pragma unroll
    for (int v0 = 0; v0 < 32 * VPR; v0 += 64) {
      const int v = v0 + lane, rl = v / VPR, e = (v - rl * VPR) * 8;
      const int r2 = (wtile * RT + rt) * 32 + rl;
      if (r2 < rows_sb && e < D)
        *reinterpret_cast<Pack8 *>(op + (int64_t)r2 * a.dq_row_stride + e) = *reinterpret_cast<const Pack8 *>(sOut + rl * LDO + e);
    }
    wave_lds_fence();
  }
}

// ------------------------------------------------------------------------------------
// dQ, second form: the row's partials are added in ascending key-block order (sorted by block id: the slot a visit
// got is arbitrary, the sum must not depend on it) and scaled.  One 16-lane group per (row, head), four per wave,
// sixteen per block of 256: a row's chain of dependent steps (count, ids, order, rows) is mostly waiting, so a wave
// runs four of them side by side.  Lane li of a group owns the 16-byte piece li of the row.  Over ranked lists the first rows are asked for beside the count; the next four
// are on their way while four are added (36427 tokens, 32 heads of 64, top-k 4, training step 1408 -> 1359 us; 25298 tokens, 32 heads of 80, top-k 2 1344 -> 1297; plain lists,
// 82354 tokens, 16 heads of 64, top-k 4, pass alone 268 -> 251; 16 visits as before).  What it costs: rows at a sequence's beginning that have fewer visits read up to three too many (eleven
// sequences of 1048 to 8510 tokens, 8 heads of 128, top-k 5, pass alone 91.3 -> 94.3).
// ------------------------------------------------------------------------------------
template <typename T, bool RANKED>
__global__ __launch_bounds__(256) void attn_bwd_dq_combine_kernel(fmoba_attn_bwd_args a, BwdWs ws, int capl) {
  extern __shared__ __attribute__((aligned(16))) int sOrdAll[];  // [16 groups][capl]: slot of the partial of rank r
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
  const int c8 = li * 8;
  const bool mine = c8 < D;
  const int PD = part_row_elems(D, 2);
  const uint16_t *part = ws.part + rh * ws.cap * PD;
  // rows t .. of the row's order, as far as there are `have` of them
  auto fetch = [&](Pack8(&x)[4], int t, int have) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (t + u >= have) break;
      x[u] = ld_stream16(part + (int64_t)(RANKED ? t + u : sOrd[t + u]) * PD + c8);
    }
  };
  Pack8 x[4];
  if (RANKED && mine) fetch(x, 0, ws.cap);  // asked for beside the count: what lies behind it is not used
  const int nall = !valid ? 0 : RANKED ? (int)(ws.visits[(int64_t)h * a.total_q + row] >> 16) : ws.cnt[rh];
  const int n = min(nall, ws.cap);
  if (nall > ws.cap && li == 0 && a.visits_overflow != nullptr) atomicMax(a.visits_overflow, nall);  // visits were dropped
  int nmax = max(n, __shfl_xor(n, 16, 64));
  nmax = max(nmax, __shfl_xor(nmax, 32, 64));  // the wave walks the longest of its four rows
  const int32_t *pid = ws.pid + rh * ws.cap;
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  // ranks over the whole row: the order of the sum does not depend on which slot a visit got
  if constexpr (!RANKED) group_rank_order(pid, 1, n, nmax, sOrd, lane);
  if (mine) {
    auto add = [&](const Pack8 &x) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        acc[2 * k] += elem_to_float<T>((uint16_t)(x.w[k] & 0xffffu));
        acc[2 * k + 1] += elem_to_float<T>((uint16_t)(x.w[k] >> 16));
      }
    };
    if (!RANKED && n > 0) fetch(x, 0, n);
    for (int t = 0; t < n; t += 4) {  // the next rows are on their way while these are added
      Pack8 nx[4];
      if (t + 4 < n) fetch(nx, t + 4, n);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (t + u < n) add(x[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = nx[u];
    }
  }
  if (valid && mine) {
    const float scale = dq_sum_scale<T>(a.softmax_scale);
    Pack8 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o.w[k] = pack2<T>(acc[2 * k] * scale, acc[2 * k + 1] * scale);
    *reinterpret_cast<Pack8 *>(reinterpret_cast<uint16_t *>(a.dq) + row * a.dq_row_stride + (int64_t)h * a.dq_head_stride + c8) = o;
  }
}

// grid (ceil(max_seqlen_q / rows_per_block), heads, batch), block 256.
// LPR = 2^lg_lpr lanes cooperate on one row (LPR >= head_dim / 8).
constexpr int kPrepRows = 4;  // rows per thread: eight 16-byte loads in flight (with one row a thread had two, 4.7 TB/s)
// Output rows of 128 MB and more whose heads are whole cache lines are read past the caches (a line that two heads share would be read twice: 400 MB of rows, 16 heads of 80 198 -> 220 us, of 96
// 191 -> 204, of 112 194 -> 212, 32 heads of 40 267 -> 294).  Through them and past them, us: 16 heads of 128, 48 MB 19.6 and 25.0, 64 MB 25.0 and 26.9, 100 MB 36.5 and 38.0, 128 MB 50.4 and 48.3,
// 160 MB 69.6 and 60.7, 256 MB 138 and 120, 400 MB 208 and 199, 1 GB 414 and 392; 32 heads of 64, 64 MB 25.1 and 25.2, 100 MB 35.8 and 36.0, 128 MB 48.6 and 45.0, 256 MB 137 and 121.
// Consecutive rows in a thread, whose sums then leave in one store: 24 MB 11.6 -> 12.4, 160 MB 60.7 -> 63.7, 256 MB 120 -> 127, 1 GB 392 -> 404 (17 to 32 MB of heads of 64 11.9 -> 11.7, 15.9 -> 15.0).
constexpr int64_t kPrepStreamBytes = (int64_t)128 << 20;
template <typename T, bool STREAM>
__global__ __launch_bounds__(256) void bwd_prep_kernel(fmoba_attn_bwd_args a, int lg_lpr, int32_t *tab, RunTable rt, int row_mask, int ztab) {
  const int LPR = 1 << lg_lpr, rows_per_pass = 256 >> lg_lpr;
  // Uneven batches have up to millions of blocks past their sequence's end, each of which lives as long as its chain of loads: they leave
  // before anything else (65536 tokens and 256 sequences of 512: 764 -> 526 us)
  const int h = blockIdx.y, b = (int)blockIdx.z - ztab;
  const int q0 = a.cu_seqlens_q[max(b, 0)], Lq = a.cu_seqlens_q[max(b, 0) + 1] - q0;
  const int first = (int)blockIdx.x * rows_per_pass * kPrepRows;
  if (b >= 0 && blockIdx.x > 0 && first >= Lq) return;
  if (b < 0) {  // four columns of the run table, before everything else: a chain of loads that the rows cover
    const int lane = threadIdx.x & 63, Bn = a.lg_block_n;
    const int64_t col = ((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (col >= rt.cols) return;
    // the sequence: the last one whose columns begin at or before this one
    int lo = 0, hi = a.batch;  // columns of sequence lo begin at or before it, those of hi do not
    while (hi - lo > 1) {
      const int step = (hi - lo + 63) >> 6, q = lo + lane * step;
      const int below = max(1, (int)__popcll(__ballot(q < hi && a.cu_seqlens_k[q] / Bn + q <= col)));
      lo += (below - 1) * step;
      hi = min(lo + step, hi);
    }
    const int c = (int)col - (a.cu_seqlens_k[lo] / Bn + lo), Lk = a.cu_seqlens_k[lo + 1] - a.cu_seqlens_k[lo];
    if (c < 0 || c >= a.max_cols || c * Bn >= Lk) return;
    const int64_t ci = ((int64_t)lo * a.heads + h) * a.max_cols + c;
    const int nnz = a.col_nnz[ci];
    const int32_t *list = a.row_indices + a.col_offsets[ci];
    // The boundaries that the dQ pass reads: from the first row block that sees the column to the end of the sequence
    const int rows = a.cu_seqlens_q[lo + 1] - a.cu_seqlens_q[lo];
    const int first_row = a.is_causal ? max(c * Bn - (Lk - rows), 0) : 0;
    if (first_row >= rows) return;
    const int rb_first = first_row / kDqRows, rb_end = min((rows + kDqRows - 1) / kDqRows + 1, rt.blocks);
    // G lanes per boundary: a step of the search narrows it G + 1 times (short sequences have few boundaries and wait for the steps)
    int G = 64;
    while (G > 1 && G * (rb_end - rb_first) > 64) G >>= 1;
    const int li = lane % G;
    const unsigned long long mine = (G == 64 ? ~0ull : (1ull << G) - 1) << (lane - li);
    for (int rb0 = rb_first; rb0 < rb_end; rb0 += 64 / G) {
      const int rb = rb0 + lane / G, v = rb * kDqRows;
      int l = 0, r = nnz;
      while (__any(l < r)) {
        const int step = (r - l + G) / (G + 1), q = l + (li + 1) * step - 1;
        const int below = __popcll(__ballot(l < r && q < r && (list[q] & row_mask) < v) & mine);
        l += below * step;
        r = below < G ? min(l + step - 1, r) : r;
      }
      if (li == 0 && rb < rb_end) tab[rt.at(h, (int)col) + rb] = l;
    }
    return;
  }
  if (blockIdx.x == 0) {  // what lies between the sequences of the padded layout is zero
    float *dh = a.softmax_d + (int64_t)h * ((int64_t)a.total_q + 128 * (int64_t)a.batch);
    const int64_t end = b == a.batch - 1 ? (int64_t)a.total_q + 128 * (int64_t)a.batch : (int64_t)q0 + Lq + 128 * (int64_t)(b + 1);
    for (int64_t i = (int64_t)q0 + Lq + 128 * (int64_t)b + threadIdx.x; i < end; i += 256) dh[i] = 0.f;
    if (b == 0)
      for (int i = threadIdx.x; i < q0; i += 256) dh[i] = 0.f;
  }
  if (first >= Lq) return;
  const int r0 = first + (threadIdx.x >> lg_lpr), sub = threadIdx.x & (LPR - 1);
  const int e = sub * 8;
  const int D = a.head_dim;
  Pack8 o[kPrepRows], g[kPrepRows];
#pragma unroll
  for (int k = 0; k < kPrepRows; ++k) {
    const int r = r0 + k * rows_per_pass;
    o[k] = zero_pack8();
    g[k] = zero_pack8();
    if (r < Lq && e < D) {
      const uint16_t *from = reinterpret_cast<const uint16_t *>(a.out) + (int64_t)(q0 + r) * a.o_row_stride + (int64_t)h * a.o_head_stride + e;
      o[k] = STREAM ? ld_stream16(from) : ld_global16(from);
      g[k] = ld_global16(reinterpret_cast<const uint16_t *>(a.dout) + (int64_t)(q0 + r) * a.do_row_stride + (int64_t)h * a.do_head_stride + e);
    }
  }
#pragma unroll
  for (int k = 0; k < kPrepRows; ++k) {
    const int r = r0 + k * rows_per_pass;
    float fo[8], fg[8];
    unpack8<T>(o[k], fo);
    unpack8<T>(g[k], fg);
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = fmaf(fo[i], fg[i], acc);
    for (int w = LPR >> 1; w >= 1; w >>= 1) acc += __shfl_xor(acc, w, 64);
    if (r < Lq && sub == 0) a.softmax_d[(int64_t)h * ((int64_t)a.total_q + 128 * (int64_t)a.batch) + q0 + 128 * b + r] = acc;
  }
}

__global__ void zero_rows_kernel(void *p, int64_t rows, int64_t row_stride, int heads, int64_t head_stride, int D) {
  // zero a (rows, heads, D) 16-bit tensor with arbitrary row/head strides
  const int vpr = D / 8;
  const int64_t nvec = rows * heads * vpr;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nvec; v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t rh = v / vpr;
    const int e = (int)(v - rh * vpr) * 8;
    const int64_t row = rh / heads;
    const int h = (int)(rh - row * heads);
    *reinterpret_cast<Pack8 *>(reinterpret_cast<uint16_t *>(p) + row * row_stride + (int64_t)h * head_stride + e) = zero_pack8();
  }
}

// dK and dV (grid y) of query heads that were kept apart, added up over the group of a key head: src is (2, rows, heads_k, grp, D), packed.  fp32 sums from the first head
// to the last, eight features a lane.  Bound by its launch where such calls are
// small, by its bytes where they are long.  One launch for both, in place of a library's sum for each: training steps of 2178 tokens, 8 heads over 1 of 128 109.2 -> 98.2 us,
// 1663 tokens, 16 over 4 of 64 104.8 -> 97.5, 1786 tokens, 32 over 8 of 128 119.5 -> 110.7.
constexpr int kSumVecs = 256;
template <typename T>
__global__ __launch_bounds__(kSumVecs) void sum_heads_kernel(const uint16_t *__restrict__ src, uint16_t *__restrict__ dk, uint16_t *__restrict__ dv, int64_t rows, int heads_k, int grp,
                                                             int D, int64_t dk_row, int64_t dk_head, int64_t dv_row, int64_t dv_head) {
  const uint32_t vph = D / 8, vpr = vph * heads_k;
  const int64_t first = (int64_t)blockIdx.x * kSumVecs, row0 = first / vpr;  // (the 64-bit division is the workgroup's)
  const uint32_t t = (uint32_t)(first - row0 * vpr) + threadIdx.x;
  const uint32_t r = t / vpr, hv = t - r * vpr, h = hv / vph, e = (hv - h * vph) * 8;
  const int64_t row = row0 + r;
  if (row >= rows) return;
  const bool is_dv = blockIdx.y != 0;
  const uint16_t *from = src + (((is_dv ? rows : 0) + row) * heads_k + h) * (int64_t)grp * D + e;
  float sum[8] = {};
#pragma unroll 4
  for (int g = 0; g < grp; ++g) {
    float f[8];
    unpack8<T>(*reinterpret_cast<const Pack8 *>(from + (int64_t)g * D), f);
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] += f[i];
  }
  Pack8 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) out.w[i] = pack2<T>(sum[2 * i], sum[2 * i + 1]);
  *reinterpret_cast<Pack8 *>((is_dv ? dv + row * dv_row + h * dv_head : dk + row * dk_row + h * dk_head) + e) = out;
}

__global__ void zero_i32_kernel(int32_t *p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0;
}

__global__ void zero_f32_kernel(float *p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0.f;
}

template <typename K>
static int launch_dkdv_kernel(K kern, size_t smem, int heads, int keys, ItemOrder order, const fmoba_attn_bwd_args &a, const BwdWs &ws, hipStream_t s) {
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_bwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const int64_t items = heads * (order == kListedLongestFirst ? listed_blocks(a.total_k, a.batch, keys) : (int64_t)a.batch * ceil_div(a.max_seqlen_k, keys));
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_bwd: too many (sequence, head, key block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(256), smem, s, a, ws, order);
  return 0;
}
template <typename T, int HD, bool DQP>
static int launch_dkdv(const fmoba_attn_bwd_args &a, const BwdWs &ws, hipStream_t s) {
  // (one pair at a time is for sequences far beyond those that go longest first)
  const ItemOrder order = item_order(a.total_k, a.max_seqlen_k, a.batch, ws.dkv_heads, 64, longest_items_first(std::max(a.total_q, a.total_k), a.heads, HD * 4));
  const bool near_rows = rows_near(a);
  auto kern = near_rows ? attn_bwd_dkdv_kernel<T, HD, DQP, false, true> : attn_bwd_dkdv_kernel<T, HD, DQP, false, false>;
  if constexpr (DQP)
    if (ws.visits != nullptr) kern = near_rows ? attn_bwd_dkdv_kernel<T, HD, DQP, true, true> : attn_bwd_dkdv_kernel<T, HD, DQP, true, false>;
  return launch_dkdv_kernel(kern, DkdvSmem<HD, DQP>::bytes, ws.dkv_heads, 64, order, a, ws, s);
}
template <typename T, int HD, int KB>
static int launch_dkdv_partials(const fmoba_attn_bwd_args &a, const BwdWs &ws, hipStream_t s) {
  const bool near_rows = rows_near(a);
  const bool longest_first = longest_items_first(std::max(a.total_q, a.total_k), a.heads, HD * 4);
  // Workgroups of one to a unit, whose empty ones come last: looking blocks up pays where two thirds of them are empty (30000 tokens in twelve sequences, 8
  // heads, 4.5 times as many as there are blocks: step 440 -> 427 us; 1.5 to 2.2 times as many: 12846, 5768, 4917 and 6469 tokens 783 -> 790, 15400 in eight
  // 344.7 -> 347.2, 15004 in five and 8999 in eight, 16 heads, the same).
  const bool listed = near_rows && ws.visits != nullptr && lists_blocks(a.total_k, a.max_seqlen_k, a.batch, a.heads, 64 * KB, longest_first) &&
                      (int64_t)a.batch * ceil_div(a.max_seqlen_k, 64 * KB) >= 3 * listed_blocks(a.total_k, a.batch, 64 * KB);
  auto kern = listed                  ? attn_bwd_dkdv_partials_kernel<T, HD, KB, true, true, true>
              : ws.visits != nullptr ? (near_rows ? attn_bwd_dkdv_partials_kernel<T, HD, KB, true, true, false> : attn_bwd_dkdv_partials_kernel<T, HD, KB, false, true, false>)
                                     : (near_rows ? attn_bwd_dkdv_partials_kernel<T, HD, KB, true, false, false> : attn_bwd_dkdv_partials_kernel<T, HD, KB, false, false, false>);
  return launch_dkdv_kernel(kern, BwdSmem<HD>::bytes, a.heads, 64 * KB, listed ? kListedLongestFirst : longest_first ? kLongestFirst : kPairOrder, a, ws, s);
}

template <typename T, int HD, int RT, int NW>
static int launch_dq(const fmoba_attn_bwd_args &a, const BwdWs &ws, hipStream_t s) {
  auto kern = attn_bwd_dq_kernel<T, HD, RT, NW>;
  const size_t smem = DqSmem<HD, RT, NW>::bytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_bwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const int nsb_max = ceil_div(a.max_seqlen_q, DqSmem<HD, RT, NW>::ROWS);
  const ItemOrder order = item_order(a.total_q, a.max_seqlen_q, a.batch, a.heads, DqSmem<HD, RT, NW>::ROWS, longest_items_first(std::max(a.total_q, a.total_k), a.heads, HD * 2));
  const int64_t items = a.heads * (order == kListedLongestFirst ? listed_blocks(a.total_q, a.batch, DqSmem<HD, RT, NW>::ROWS) : (int64_t)a.batch * nsb_max);
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_bwd: too many (sequence, head, superblock) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(64 * NW), smem, s, a, ws.ds, ws.tab, bwd_run_table(a), ws.row_mask, nsb_max, order);
  return 0;
}

// head dimensions above 128 (attn_bwd_wide.hip)
int run_bwd_dkdv_wide(const fmoba_attn_bwd_args &a, uint16_t *ds_ws, int row_mask, hipStream_t s);

// columns of a multiple of 128 keys: one workgroup (and one dQ partial per visit) per 128 keys
static inline bool bwd_wide_blocks(const fmoba_attn_bwd_args &a) { return a.head_dim > 64 && a.lg_block_n % 128 == 0; }

// Which form of the dQ computation a call uses.  The row-stationary form works on (256-row block, key block) steps
// and is the faster one while a step has enough rows; with many chunks per sequence a step has one or two rows and
// only the per-visit partials scale.
//  - 128-key blocks at head dimensions 65 to 128 (a visit leaves one partial per 128 keys): partials below 0.37 of the chunks a
//    row may see (dK/dV and dQ together, partials against dS tiles: 32768 tokens, 0.30 of them 5130 against 5433 us, 0.45 7371 against 7048);
//  - 64-key blocks, and head dimensions up to 64: below a tenth.  That line is one of precision, not of time: dS tiles add a row's
//    visits up in fp32, a partial row is rounded to 16 bits (error of dQ against 64 bits, 8192 tokens, 0.12 of the chunks: 2.40e-3
//    with dS tiles, 2.93e-3 with partials), and calls that have had the fp32 sums keep them although partials are the faster form
//    further up (32768 tokens, 0.12 of the chunks, heads of 128 3142 against 3560 us, heads of 64 1999 against 2497).
static int bwd_dq_partials(const fmoba_attn_bwd_args &a) {
  if (a.head_dim > 128) return 0;  // head dimensions above 128: dS tiles and the row-block pass only
  if (a.dq_mode == 1) return 0;
  if (a.dq_mode == 2) return 1;
  const double chunks_per_seq = (double)a.total_k / a.batch / a.lg_block_n;
  const double chunks_per_row = (double)a.max_visits_per_row * 64.0 / a.lg_block_n;
  const double seen = a.is_causal ? 0.5 * chunks_per_seq : chunks_per_seq;
  return chunks_per_row < (bwd_wide_blocks(a) ? 0.37 : 0.10) * seen;
}
// Heads of dK / dV the call is best made with: heads / this many query heads are added up by one workgroup, in fp32, instead
// of in memory afterwards (24571 tokens, 32 over 8 heads: 1225 us and two sums of 48 us -> 1118 us).  All heads of a group, unless that
// leaves fewer than two rounds of workgroups for the chip's 512 (two per unit).  The long calls (partials at head dimension
// 128) have a kernel that takes one head at a time.
static bool bwd_sums_heads(const fmoba_attn_bwd_args &a) { return a.head_dim <= 64 || (a.head_dim <= 128 && !bwd_dq_partials(a)); }
static int bwd_dkv_heads(const fmoba_attn_bwd_args &a) {
  if (!bwd_sums_heads(a)) return a.heads;
  const int grp = a.heads / a.heads_k;
  const int64_t blocks = a.total_k / 64 + a.batch;
  for (int gs = grp < 64 ? grp : 64; gs > 1; --gs)
    if (grp % gs == 0 && blocks * (a.heads / gs) >= 1024) return a.heads / gs;
  return a.heads;
}
// partial slots per (row, head): max_visits_per_row counts 64-key blocks; with 128-key blocks a row has half as many
// visits (only the last column of a sequence can have an odd number of 64-key blocks)
static inline int32_t bwd_partial_cap(const fmoba_attn_bwd_args &a) {
  const int32_t mv = a.max_visits_per_row > 0 ? a.max_visits_per_row : 1;
  return bwd_wide_blocks(a) ? (mv + 1) / 2 : mv;
}

template <typename T>
static int run_bwd(const fmoba_attn_bwd_args &a, const BwdWs &ws, int phases, hipStream_t s) {
  const bool partials = bwd_dq_partials(a);
  if (phases & FMOBA_BWD_PREP) {
    int lg_lpr = 0;
    while ((8 << lg_lpr) < a.head_dim) ++lg_lpr;
    const int nx = ceil_div(a.max_seqlen_q, (256 >> lg_lpr) * kPrepRows);
    const RunTable rt = bwd_run_table(a);
    const int ztab = partials ? 0 : (int)ceil_div64(ceil_div(rt.cols, 4), nx);
    auto prep = a.head_dim % 64 == 0 && (int64_t)a.total_q * a.heads * a.head_dim * 2 >= kPrepStreamBytes ? bwd_prep_kernel<T, true> : bwd_prep_kernel<T, false>;
    if (a.batch + ztab <= 65535) {
      hipLaunchKernelGGL(prep, dim3(nx, a.heads, a.batch + ztab), dim3(256), 0, s, a, lg_lpr, ws.tab, rt, ws.row_mask, ztab);
    } else {  // (more planes than a launch has)
      if (ztab > 0) hipLaunchKernelGGL(prep, dim3(ceil_div(rt.cols, 4), a.heads, 1), dim3(256), 0, s, a, lg_lpr, ws.tab, rt, ws.row_mask, 1);
      hipLaunchKernelGGL(prep, dim3(nx, a.heads, a.batch), dim3(256), 0, s, a, lg_lpr, ws.tab, rt, ws.row_mask, 0);
    }
  }
  if (a.head_dim > 128) {
    // the plain feature-split dK/dV kernel (attn_bwd_wide.hip), then the row-block dQ pass over its dS tiles
    if (phases & FMOBA_BWD_DKDV)
      if (int rc = run_bwd_dkdv_wide(a, ws.ds, ws.row_mask, s)) return rc;
    if (phases & FMOBA_BWD_DQ)
      if (int rc = launch_dq<T, 256, 1, 8>(a, ws, s)) return rc;
    return 0;
  }
  if (phases & FMOBA_BWD_DKDV) {
    int rc;
    if (partials) {
      if (ws.visits == nullptr) hipLaunchKernelGGL(zero_i32_kernel, dim3(512), dim3(256), 0, s, ws.cnt, (int64_t)a.total_q * a.heads);
      rc = a.head_dim <= 64 ? launch_dkdv<T, 64, true>(a, ws, s) : (bwd_wide_blocks(a) ? launch_dkdv_partials<T, 128, 2>(a, ws, s) : launch_dkdv_partials<T, 128, 1>(a, ws, s));
    } else {
      rc = a.head_dim <= 64 ? launch_dkdv<T, 64, false>(a, ws, s) : a.head_dim <= 96 ? launch_dkdv<T, 96, false>(a, ws, s) : launch_dkdv<T, 128, false>(a, ws, s);
    }
    if (rc) return rc;
  }
  if (phases & FMOBA_BWD_DQ) {
    if (partials) {
      const int64_t rows = (int64_t)a.total_q * a.heads;
      const int capl = combine_order_entries(ws.cap);
      const size_t smem = ws.visits != nullptr ? 0 : (size_t)16 * capl * 4;
      auto kern = ws.visits != nullptr ? attn_bwd_dq_combine_kernel<T, true> : attn_bwd_dq_combine_kernel<T, false>;
      if (smem > 32 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
        set_error("attn_bwd: a row with up to %d visits needs %zu bytes of LDS for the order of its partial results", ws.cap, smem);
        return 2;
      }
      hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 15) / 16)), dim3(256), smem, s, a, ws, capl);
    } else {
      // Head dimensions 97 to 128: eight waves of one tile instead of four of two for few and long walks, each of which then has a unit (or
      // most of one) for itself and takes half the time for a step.  Training steps, four waves and eight: one sequence of 1531 tokens, 8 heads
      // 124.7 -> 120.6 us, 5000 tokens, 16 heads (320 row blocks) 356 -> 342, 8000 tokens, 8 heads 532 -> 518; 8192 tokens, 16 heads (512) 866 ->
      // 893; six sequences of 1010 (384 blocks of four to a sequence) 206 -> 209.
      const bool few = (int64_t)a.heads * ((a.total_q + (kDqRows - 1) * (int64_t)a.batch) / kDqRows) <= 400 && a.total_q >= 1500 * (int64_t)a.batch;
      int rc = a.head_dim <= 64   ? launch_dq<T, 64, 1, 8>(a, ws, s)
               : a.head_dim <= 96 ? (launch_dq<T, 96, 2, 4>(a, ws, s))
                                  : (few ? launch_dq<T, 128, 1, 8>(a, ws, s) : launch_dq<T, 128, 2, 4>(a, ws, s));
      if (rc) return rc;
    }
  }
  return 0;
}

static inline size_t bwd_align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace fmoba

extern "C" int32_t fmoba_attn_bwd_uses_partials(const fmoba_attn_bwd_args *a) {
  if (a == nullptr || a->batch <= 0 || a->lg_block_n <= 0) return 0;
  return fmoba::bwd_dq_partials(*a);
}

extern "C" int32_t fmoba_attn_bwd_dkv_heads(const fmoba_attn_bwd_args *a) {
  if (a == nullptr) return 0;
  if (a->heads_k <= 0 || a->heads % a->heads_k != 0 || a->batch <= 0 || a->lg_block_n <= 0) return a->heads;
  return fmoba::bwd_dkv_heads(*a);
}

extern "C" size_t fmoba_attn_bwd_workspace_bytes(const fmoba_attn_bwd_args *a) {
  using namespace fmoba;
  if (a == nullptr || a->total_q <= 0 || a->heads <= 0 || a->head_dim <= 0 || a->batch <= 0 || a->lg_block_n <= 0) return 256;
  if (!bwd_dq_partials(*a)) {
    const RunTable rt = bwd_run_table(*a);
    return ds_workspace_tiles(a->num_row_indices) * (size_t)a->lg_block_n * 64 + bwd_align256((size_t)rt.at(a->heads, 0) * 4) + 256;
  }
  const size_t rows = (size_t)a->total_q * a->heads, cap = (size_t)bwd_partial_cap(*a);
  // one spare partial row / block id at the end takes the writes of absent rows
  return bwd_align256(rows * 4) + bwd_align256((rows * cap + 1) * 4) + bwd_align256((rows * cap + 1) * part_row_elems(a->head_dim, 2) * 2) + 256;
}

extern "C" int fmoba_attn_bwd(const fmoba_attn_bwd_args *a, void *stream) { return fmoba_attn_bwd_phases(a, 7, stream); }

extern "C" int fmoba_attn_bwd_phases(const fmoba_attn_bwd_args *a, int32_t phases, void *stream) { return fmoba_attn_bwd_grouped(a, a ? a->heads : 0, phases, stream); }

extern "C" int fmoba_sum_grouped_heads(const void *apart, void *dk, void *dv, int64_t total_k, int32_t dkv_heads, int32_t heads_k, int32_t head_dim, int64_t dk_row_stride,
                                       int64_t dk_head_stride, int64_t dv_row_stride, int64_t dv_head_stride, int32_t dtype, void *stream) {
  using namespace fmoba;
  FMOBA_REQUIRE(dtype == FMOBA_DTYPE_F16 || dtype == FMOBA_DTYPE_BF16, "FlashMoBA only support fp16 and bf16 data type");
  FMOBA_REQUIRE(total_k >= 0 && heads_k > 0 && dkv_heads > 0 && dkv_heads % heads_k == 0, "sum_grouped_heads: dkv_heads must be a multiple of heads_k");
  FMOBA_REQUIRE(head_dim > 0 && head_dim % 8 == 0 && head_dim <= 256, "sum_grouped_heads: head_dim must be a multiple of 8 and at most 256");
  if (total_k == 0) return 0;
  for (const void *p : {apart, (const void *)dk, (const void *)dv}) FMOBA_REQUIRE(p != nullptr && (uintptr_t)p % 16 == 0, "sum_grouped_heads: tensors must be 16-byte aligned");
  for (int64_t x : {dk_row_stride, dk_head_stride, dv_row_stride, dv_head_stride}) FMOBA_REQUIRE(x % 8 == 0, "sum_grouped_heads: strides must be multiples of 8 elements");
  const int64_t blocks = ceil_div64(total_k * heads_k * (head_dim / 8), kSumVecs);
  FMOBA_REQUIRE(heads_k <= 65535 && blocks < ((int64_t)1 << 31), "sum_grouped_heads: more elements than a launch takes");
  auto kern = dtype == FMOBA_DTYPE_BF16 ? sum_heads_kernel<bf16_t> : sum_heads_kernel<f16_t>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 2), dim3(kSumVecs), 0, (hipStream_t)stream, (const uint16_t *)apart, (uint16_t *)dk, (uint16_t *)dv, total_k, heads_k, dkv_heads / heads_k,
                     head_dim, dk_row_stride, dk_head_stride, dv_row_stride, dv_head_stride);
  FMOBA_LAUNCH_CHECK("sum_grouped_heads");
  return 0;
}

extern "C" int fmoba_attn_bwd_grouped(const fmoba_attn_bwd_args *a, int32_t dkv_heads, int32_t phases, void *stream) {
  return fmoba_attn_bwd_ranked(a, nullptr, dkv_heads, phases, stream);
}

extern "C" int fmoba_attn_bwd_ranked(const fmoba_attn_bwd_args *a, const uint32_t *visits, int32_t dkv_heads, int32_t phases, void *stream) {
  using namespace fmoba;
  FMOBA_REQUIRE(a != nullptr, "attn_bwd: null args");
  FMOBA_REQUIRE(phases > 0 && phases <= 7, "attn_bwd: phases must be a mask of bits 1, 2, 4");
  FMOBA_REQUIRE(a->dtype == FMOBA_DTYPE_F16 || a->dtype == FMOBA_DTYPE_BF16, "FlashMoBA only support fp16 and bf16 data type");
  FMOBA_REQUIRE(a->batch > 0, "batch size must be positive");
  FMOBA_REQUIRE(a->head_dim > 0 && a->head_dim % 8 == 0, "head_size should be a multiple of 8");
  FMOBA_REQUIRE(a->head_dim <= 256, "FlashMoBA backward only supports head dimension at most 256");
  FMOBA_REQUIRE(a->heads > 0 && a->heads_k > 0 && a->heads % a->heads_k == 0, "Number of heads in key/value must divide number of heads in query");
  FMOBA_REQUIRE(dkv_heads == a->heads || (dkv_heads > 0 && dkv_heads % a->heads_k == 0 && a->heads % dkv_heads == 0 && a->heads / dkv_heads <= 64 && a->lg_block_n > 0 &&
                                          bwd_sums_heads(*a)),
                "attn_bwd: dkv_heads must be heads, or a multiple of heads_k that divides heads, at most 64 query heads each (not above head dimension 128, nor above 64 with dQ partials)");
  FMOBA_REQUIRE(a->lg_block_m % 64 == 0, "m_lg_block_dim must be a multiple of 64");
  FMOBA_REQUIRE(a->lg_block_n > 0 && a->lg_block_n % 64 == 0, "n_lg_block_dim must be a multiple of 64");
  FMOBA_REQUIRE(a->lg_block_n <= 64 * 256, "attn_bwd: n_lg_block_dim above 16384 is not supported");
  FMOBA_REQUIRE(a->total_q >= 0 && a->total_k >= 0 && a->max_seqlen_q >= 0 && a->max_seqlen_k >= 0 && a->max_cols >= 0 && a->max_visits_per_row >= 0 && a->num_row_indices >= 0,
                "negative size");
  FMOBA_REQUIRE(a->cu_seqlens_q && a->cu_seqlens_k, "attn_bwd: null cu_seqlens pointer");
  FMOBA_REQUIRE(a->batch <= 65535 && a->heads <= 65535, "attn_bwd: batch/heads too large for the launch grid");
  hipStream_t s = (hipStream_t)stream;
  const int64_t st[] = {a->q_row_stride,  a->q_head_stride,  a->k_row_stride,  a->k_head_stride,  a->v_row_stride,  a->v_head_stride,
                        a->o_row_stride,  a->o_head_stride,  a->do_row_stride, a->do_head_stride, a->dq_row_stride, a->dq_head_stride,
                        a->dk_row_stride, a->dk_head_stride, a->dv_row_stride, a->dv_head_stride};
  for (int64_t x : st) FMOBA_REQUIRE(x % 8 == 0, "attn_bwd: strides must be multiples of 8 elements");
  FMOBA_REQUIRE(a->k_row_stride < ((int64_t)1 << 24), "attn_bwd: k_row_stride must be below 2^24 elements");
  FMOBA_REQUIRE(a->q_row_stride < ((int64_t)1 << 31) && a->do_row_stride < ((int64_t)1 << 31), "attn_bwd: q / dout row strides must be below 2^31 elements");
  const void *ptrs[] = {a->dout, a->q, a->k, a->v, a->out, a->dq, a->dk, a->dv};
  for (const void *p : ptrs) FMOBA_REQUIRE(((uintptr_t)p % 16) == 0, "attn_bwd: tensors must be 16-byte aligned");

  if (a->total_k > 0) {
    FMOBA_REQUIRE(a->dk && a->dv, "attn_bwd: null dk/dv");
    if (a->max_seqlen_q == 0 || a->total_q == 0 || a->max_cols == 0) {
      // no query rows: dk = dv = 0 (csrc/flash_moba/flash_moba_api.cpp:834-839)
      hipLaunchKernelGGL(zero_rows_kernel, dim3(1024), dim3(256), 0, s, a->dk, (int64_t)a->total_k, a->dk_row_stride, dkv_heads, a->dk_head_stride, a->head_dim);
      hipLaunchKernelGGL(zero_rows_kernel, dim3(1024), dim3(256), 0, s, a->dv, (int64_t)a->total_k, a->dv_row_stride, dkv_heads, a->dv_head_stride, a->head_dim);
    }
  }
  if (a->total_q == 0 || a->max_seqlen_q == 0) {
    if (a->softmax_d) hipLaunchKernelGGL(zero_f32_kernel, dim3(64), dim3(256), 0, s, a->softmax_d, (int64_t)a->heads * ((int64_t)a->total_q + 128 * (int64_t)a->batch));
    FMOBA_LAUNCH_CHECK("attn_bwd(no rows)");
    return 0;
  }
  FMOBA_REQUIRE(a->dout && a->q && a->out && a->softmax_lse && a->dq && a->softmax_d, "attn_bwd: null pointer");
  if (a->total_k == 0 || a->max_seqlen_k == 0 || a->max_cols == 0) {
    // no keys: dq = 0
    if (phases & FMOBA_BWD_PREP)
      hipLaunchKernelGGL(zero_f32_kernel, dim3(256), dim3(256), 0, s, a->softmax_d, (int64_t)a->heads * ((int64_t)a->total_q + 128 * (int64_t)a->batch));
    hipLaunchKernelGGL(zero_rows_kernel, dim3(1024), dim3(256), 0, s, a->dq, (int64_t)a->total_q, a->dq_row_stride, a->heads, a->dq_head_stride, a->head_dim);
    FMOBA_LAUNCH_CHECK("attn_bwd(no keys)");
    return 0;
  }
  FMOBA_REQUIRE(a->k && a->v && a->col_offsets && a->col_nnz && a->row_indices, "attn_bwd: null k/v/CSC pointer");
  FMOBA_REQUIRE(a->max_visits_per_row > 0, "attn_bwd: max_visits_per_row must be positive");
  FMOBA_REQUIRE(a->dq_mode >= 0 && a->dq_mode <= 2, "attn_bwd: dq_mode must be 0 (automatic), 1 (row blocks) or 2 (partials)");
  FMOBA_REQUIRE(a->dq_mode != 2 || a->head_dim <= 128, "attn_bwd: head dimensions above 128 only have the row-block form of dQ");
  FMOBA_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= fmoba_attn_bwd_workspace_bytes(a), "attn_bwd: workspace too small");
  const size_t rows = (size_t)a->total_q * a->heads;
  uintptr_t wp = ((uintptr_t)a->workspace + 255) & ~(uintptr_t)255;
  BwdWs ws;
  ws.dkv_heads = dkv_heads;
  ws.cap = bwd_partial_cap(*a);
  ws.visits = visits;
  ws.row_mask = visits != nullptr ? kListRowMask : -1;
  // (the dK/dV pass keeps the place of a visit's dQ partial as a 32-bit index of partial rows)
  FMOBA_REQUIRE(!fmoba::bwd_dq_partials(*a) || rows * (size_t)ws.cap + 1 < ((size_t)1 << 31),
                "attn_bwd: %zu rows x heads with up to %d dQ partials each are more partial rows than the partials form addresses", rows, ws.cap);
  ws.tab = reinterpret_cast<int32_t *>(wp);
  ws.ds = reinterpret_cast<uint16_t *>(wp + bwd_align256((size_t)bwd_run_table(*a).at(a->heads, 0) * 4));
  ws.cnt = reinterpret_cast<int32_t *>(wp);
  wp += bwd_align256(rows * 4);
  ws.pid = reinterpret_cast<int32_t *>(wp);
  wp += bwd_align256((rows * ws.cap + 1) * 4);
  ws.part = reinterpret_cast<uint16_t *>(wp);
  int rc = a->dtype == FMOBA_DTYPE_BF16 ? run_bwd<bf16_t>(*a, ws, phases, s) : run_bwd<f16_t>(*a, ws, phases, s);
  if (rc) return rc;
  FMOBA_LAUNCH_CHECK("attn_bwd");
  return 0;
}
