// Sparse attention forward in row blocks for head dimensions above 128 (up to 256): the walk of attn_fwd_rows.hip with a
// loop of its own.
#include "attn_fwd_rows.h"
#include "gate_select.h"

#include <algorithm>

namespace fmoba {

// 128 rows per workgroup, four waves of 32 rows and 512 registers, one workgroup per compute unit: a wave's 256 features of O^T are half of the
// ordinary registers, its Q rows lie in accumulation registers, and the rings of two K and two V tiles take 128 KB.  With one wave per SIMD
// nothing runs under the softmax unless it stands there, so a step is two runs of 32 products: S of the next step, with the rescaling
// of O between them, and V^T P of this one, with the softmax of the next step between them.  Each run has the tile loads of a later step
// between its products, one per four (eight in a row at its start: 181 -> 171 us below).
// O is rescaled in every step, by a factor between 1/2 and 2 as a rule: that keeps a block's reference point at its maximum less
// a whole number, so that its largest probability is exact in 16 bits, and the whole number is chosen by the largest score of the walk so far: the
// reference point lies at most 1/2 above that score and 8 1/2 below it, however long the walk is.  (Chosen by the reference point before, it would go
// up to 1/2 further in every step: wrong fp16 results from 64 steps on, NaN in either type within a few hundred.)
// Error of the output against 64 bits, rows here and columns, whose blocks have their own maximum for reference: 2 x 4096 tokens, 8 heads, top-k 8 of
// 128-key chunks bf16 2.010e-3 and 2.047e-3, fp16 2.507e-4 and 2.554e-4; rows that see 64 steps 2.105e-3 and 2.106e-3, 2.632e-4 and 2.632e-4, 512 steps
// 2.108e-3 and 2.166e-3, 2.623e-4 and 2.694e-4, 2048 steps 2.094e-3 and 2.157e-3, 2.629e-4 and 2.699e-4.
// What bounds it: matrix products at the power limit (1.0 PFLOP/s executed at 16384 tokens; without the tile loads it would be 15 % faster, without
// the rescaling or the exponentials 3 to 5 %).  GATED as in attn_fwd_rows_kernel: forward of 2 x 4096 tokens, 8 heads, top-k 8 of 128-key chunks 178.7 -> 173.2
// us, of 2048 tokens, 16 heads 85.9 -> 80.4, 9000 tokens, 16 over 2 heads 343.6 -> 336.0.  The same call: columns 134 us and their combine 89 -> 171 us,
// training step 612 -> 530.
template <typename T, bool GATED>
__global__ __launch_bounds__(256, 1) void attn_fwd_rows_wide_kernel(fmoba_attn_fwd_args a, const uint32_t *bm, int nw, int step_cap, ItemOrder order, RowGate gate) {
  constexpr int HD = 256, RW = 4;
  typedef FwdRowsDirectSmem<HD, RW, 1> SM;
  constexpr int kRows = SM::ROWS, KS = HD / 16, LDO = SM::LDO, NDT = HD / 32, VPR = HD / 8, RB = HD * 2, NI = VPR / RW;
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  int *sStep = reinterpret_cast<int *>(smem + SM::oStep);
  uint32_t *sUnion = reinterpret_cast<uint32_t *>(sStep + step_cap);
  uint32_t *sBits = sUnion + nw * SM::UPW;
  int *sAgain = reinterpret_cast<int *>(sBits + nw * kRows);  // per wave: a sum is not finite

  // the longest walks (last rows of a causal sequence) start first
  int b, h, rb, q0, Lq, k0, Lk;
  if (order == kListedLongestFirst) {
    const BlockItem item = listed_item<kRows, true>(blockIdx.x, a.batch, a.heads, a.max_seqlen_q, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    b = item.b, h = item.h, rb = item.idx, q0 = item.q0, Lq = item.Lq, k0 = item.k0, Lk = item.Lk;
  } else {
    const int nrb = (a.max_seqlen_q + kRows - 1) / kRows;
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * a.heads, nrb, false, order == kLongestFirst);
    b = item.pair / a.heads, h = item.pair - b * a.heads, rb = nrb - 1 - item.idx;
    q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
    k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  }
  const int r0 = rb * kRows;
  if (r0 >= Lq) return;
  const int off = Lk - Lq;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  const bool causal = a.is_causal != 0;
  const int Bn = a.lg_block_n;
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;

  const int row = r0 + wave * 32 + (lane & 31);
  const bool valid = row < Lq;
  Pack8 qb[KS];
  q_rows_load<HD>(qb, reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride, a.q_row_stride,
                  r0 + wave * 32, Lq, lane, D);
  const int rlast = min(r0 + kRows - 1, Lq - 1);
  const int kend = min(Lk, causal ? rlast + off + 1 : Lk);  // keys [0, kend) are visible to some row
  int nstep;
  if constexpr (GATED) {
    static_assert(row_gate_lds<HD>() + kRowGateChunks * 4 <= SM::ring, "the chunk means and the counts lie where the K/V rings will");
    const int km0 = gate.cu_seqlens_km[b], Cm = gate.cu_seqlens_km[b + 1] - km0;
    gate_row_block<T, HD, RW, 1>(a, gate, smem, sBits, reinterpret_cast<int *>(smem + row_gate_lds<HD>()), qb, b, h, hk, q0, r0, rlast, Lq, off, nw, km0, Cm);
    nstep = row_block_steps<kRows, 256, true>(nullptr, 0, rlast - r0 + 1, kend, Bn, nw, step_cap, sStep, sUnion, sBits);
  } else {
    nstep = row_block_steps<kRows, 256>(bm + (int64_t)h * nw * a.total_q + q0 + r0, a.total_q, rlast - r0 + 1, kend, Bn, nw, step_cap, sStep, sUnion, sBits);
  }
  nstep = min(nstep, step_cap);
  if (nstep == 0) {  // no visible selected key: out = 0, lse = +inf for the rows of this block
    if (valid) {
      uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + row) * a.o_row_stride + (int64_t)h * a.o_head_stride;
      for (int e = hh * 8; e < D; e += 16) *reinterpret_cast<Pack8 *>(op + e) = zero_pack8();
      if (hh == 0) a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = INFINITY;
    }
    return;
  }
  auto entry_at = [&](int t) { return sStep[min(t, nstep - 1)]; };

  // ---- feeding the rings (attn_fwd_rows_kernel has the layout): every wave a quarter of a tile, eight loads of a kilobyte ----
  const uint32_t ldsK = (uint32_t)(uintptr_t)smem, ldsV = ldsK + (uint32_t)(2 * SM::tile);
  const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)k0 * a.k_row_stride + (int64_t)hk * a.k_head_stride;
  const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)k0 * a.v_row_stride + (int64_t)hk * a.v_head_stride;
  // A lane's piece in load i of a tile: row 2 (8 wave + i) + lane / 32.  Keys past the sequence are fetched from the last one.
  uint32_t piece[NI];  // its byte offset inside the row
#pragma unroll
  for (int i = 0; i < NI; ++i) piece[i] = (uint32_t)min(((lane & 31) ^ tile_swz<HD>((wave * NI + i) * 2 + (lane >> 5))) * 8, D - 8) * 2u;
  const uint32_t row2 = (uint32_t)(wave * NI * 4 + (lane >> 5) * 2);  // twice the row of load 0
  struct Tile {
    const uint16_t *base;
    uint32_t row_stride, dst, last2;
  };
  auto tile_at = [&](const uint16_t *g, int64_t row_stride, uint32_t ring, int slot, int entry) {
    const int key0 = (entry & 0xffff) << 6;
    return Tile{g + (uint64_t)(uint32_t)key0 * (uint32_t)row_stride, (uint32_t)row_stride, ring + (uint32_t)((slot & 1) * (int)SM::tile + wave * NI * 1024), (uint32_t)(Lk - 1 - key0) * 2u};
  };
  auto load_piece = [&](const Tile &x, int i) {
    global_to_lds16_sbase(mad24_u32(min(row2 + (uint32_t)(4 * i), x.last2), x.row_stride, piece[i]), x.base, x.dst + (uint32_t)(i * 1024));
  };
  auto tile_k = [&](int t, int entry) { return tile_at(kg, a.k_row_stride, ldsK, t, entry); };
  auto tile_v = [&](int t, int entry) { return tile_at(vg, a.v_row_stride, ldsV, t, entry); };
  auto feed = [&](const Tile &x) {
#pragma unroll
    for (int i = 0; i < NI; ++i) load_piece(x, i);
  };
  const int lim = valid ? min(causal ? row + off : 0x7fffffff, Lk - 1) : -1;  // last visible key
  // (Q is in registers before the first tile loads are issued: from here on the wave counts its outstanding loads)
  if constexpr (!GATED) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qb[ks].w[0]), "+v"(qb[ks].w[1]), "+v"(qb[ks].w[2]), "+v"(qb[ks].w[3]));
#endif
    q_rows_arrange<HD>(qb, hh, D);
  }
  // (Q stays in accumulation registers, which the products read as well as the others)
  u32x4_t qa[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qa[ks] = pack8_vec(qb[ks]);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+a"(qa[ks]));
#endif
  }
  wait_all_loads();

  f32x16 o[NDT];  // O^T: register i of feature tile dt <-> feature dt*32 + acc_row(i, hh), this lane's row
  f32x16 st[2];       // S^T: register i of tile kt <-> key kt*32 + acc_row(i, hh), this lane's row
  Pack8 pf[2][2], pn[2][2];  // P^T of step t and of step t + 1, as the B operand of O^T += V^T P^T
  float ref, top, l_run, alpha;  // reference point and largest score of the walk so far (log2)
  const uint32_t rowoff = (uint32_t)((lane & 31) * RB + ((tile_frag_piece<HD>(hh, 0) ^ tile_swz<HD>(lane & 31)) * 16));
  const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
  const uint32_t troff = (uint32_t)(r0t * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
  auto opaque = [](uint32_t &x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#else
    (void)x;
#endif
  };
  // ---- S^T of step t, the sums of the walk scaled by alpha meanwhile ----
  auto scores = [&](auto scaled, int t, const Tile &x) __attribute__((always_inline)) {
    uint32_t ak = ldsK + (uint32_t)((t & 1) * (int)SM::tile) + rowoff;
    opaque(ak);
    constexpr int AHEAD = 6;
    Pack8 kf[8];
    auto read = [&](int m) { kf[m & 7] = lds_read16(tile_frag_addr<HD>(ak, m % KS) + (uint32_t)((m / KS) * 32 * RB)); };
#pragma unroll
    for (int m = 0; m < AHEAD; ++m) read(m);
    auto scale = [&](int n0, int n1) {
      if constexpr (decltype(scaled)::value) {
#pragma unroll
        for (int n = n0; n < n1; ++n) o[n / 16][n % 16] *= alpha;
      }
    };
    scale(0, 32);
    __builtin_amdgcn_sched_barrier(0);
    static_for<2 * KS>([&](auto mc) {
      constexpr int m = decltype(mc)::value, kt = m / KS, ks = m % KS;
      if constexpr (ks == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kt][i] = 0.f;
      }
      st[kt] = mfma32<T>(kf[m & 7], Pack8{{qa[ks][0], qa[ks][1], qa[ks][2], qa[ks][3]}}, st[kt]);
      if constexpr (m + AHEAD < 2 * KS) read(m + AHEAD);
      scale(32 + 3 * m, 32 + 3 * m + 3);
      if constexpr (decltype(scaled)::value && m % 4 == 1) load_piece(x, m / 4);
      __builtin_amdgcn_sched_barrier(0);
    });
    // (the products would move to where they are used, behind the next branch)
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) asm volatile("" : "+v"(o[dt]));
#endif
  };
  // ---- the softmax of step t in slices: 0..3 row maximum, 4 reference point, 5..20 two exponentials each ----
  float mloc = 0.f, neg = 0.f, lsum = 0.f;
  bool active = false;
  uint32_t keep = 0u;  // nothing of a row that skips the step, whatever the scores are (one that takes part hands on its NaN scores)
  auto mask = [&](int key0, int c, uint32_t word) {
    active = valid && ((word >> (c & 31)) & 1u) != 0u && lim >= key0;
    const int lim_rel = active ? lim - key0 : -1;
    if (!__all(lim_rel >= 63 || lim_rel < 0)) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int jrel = kt * 32 + 8 * (i >> 2) + (i & 3) + 4 * hh;
          st[kt][i] = jrel <= lim_rel ? st[kt][i] : -INFINITY;
        }
    }
  };
  auto soft = [&](auto sc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    if constexpr (s < 4) {
      if constexpr (s == 0) mloc = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) mloc = fmaxf(mloc, st[s / 2][(s & 1) * 8 + i]);
    } else if constexpr (s == 4) {
      // The reference point of the exponentials is the block's maximum less a whole number (the largest p of the block is a
      // power of two, which the 16-bit P holds exactly) and within 1/2 of the walk's maximum so far, or below it by up to 8 1/2.
      const float x = max_xor32_f(mloc) * scale_log2;
      const bool seen = active && x > -INFINITY;
      const float k = x - top > 8.f ? 0.f : rintf(x - top);
      const float r = seen ? x - k : ref;
      top = seen ? fmaxf(top, x) : top;
      alpha = r == ref ? 1.f : __builtin_amdgcn_exp2f(ref - r);
      neg = seen ? -r : 0.f;  // (0: all scores are minus infinity or NaN)
      ref = r;
      lsum = 0.f;
      keep = active ? 0xffffffffu : 0u;
    } else if constexpr (s < 21) {
      constexpr int j = s - 5, kt = j / 8, w = j % 8;
      const float p0 = __builtin_amdgcn_exp2f(fmaf(st[kt][2 * w], scale_log2, neg));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(st[kt][2 * w + 1], scale_log2, neg));
      lsum += p0 + p1;
      pn[kt][w / 4].w[w % 4] = pack2<T>(p0, p1) & keep;
      if constexpr (j == 15) l_run = keep ? l_run * alpha + lsum : l_run;
    }
  };
  uint32_t took = 0u;  // keep of step t
  auto next = [&]() {
    took = keep;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) pf[kt][s2] = pn[kt][s2];
  };
  // ---- O^T += V^T P^T of step t, the softmax of step t + 1 meanwhile ----
  auto sums = [&](auto apart, int t, const Tile &x) __attribute__((always_inline)) {
    uint32_t tv = ldsV + (uint32_t)((t & 1) * (int)SM::tile) + troff;
    opaque(tv);
    Pack8 vt[2][4];
    auto read = [&](int m) {
      const uint32_t at = (uint32_t)((m & 3) * 16 * RB);
      vt[(m >> 2) & 1][m & 3] = lds_tr8(tile_tr_addr<HD>(tv, m >> 2) + at, tile_tr_addr8<HD>(tv, m >> 2) + at);
    };
    constexpr int AHEAD = 6;
#pragma unroll
    for (int m = 0; m < AHEAD; ++m) read(m);
    static_for<4>([&](auto sl) { soft(sl); });
    __builtin_amdgcn_sched_barrier(0);
    f32x16 with;
    static_for<4 * NDT>([&](auto mc) {
      constexpr int m = decltype(mc)::value, dt = m >> 2, u = m & 3;
      if constexpr (decltype(apart)::value) {
        if constexpr (u == 0) with = o[dt];
        with = mfma32<T>(vt[dt & 1][u], pf[u >> 1][u & 1], with);
        if constexpr (u == 3) {
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] = took ? with[i] : o[dt][i];
        }
      } else {
        o[dt] = mfma32<T>(vt[dt & 1][u], pf[u >> 1][u & 1], o[dt]);
      }
      if constexpr (m + AHEAD < 4 * NDT) read(m + AHEAD);
      if constexpr (m == 0) soft(std::integral_constant<int, 4>{});
      if constexpr (m % 4 == 3) load_piece(x, m / 4);
      if constexpr (m >= 2 && m < 18) soft(std::integral_constant<int, m + 3>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    next();
  };

  auto word_of = [&](int s) { return sBits[((s >> 16) >> 5) * kRows + wave * 32 + (lane & 31)]; };
  // A step's products take a row that skips it along with probabilities of zero, which leave NaN where V is infinite or NaN.  If
  // the block has any sum that is not finite, it is walked a second time with the sums of rows that skip a step set aside: as in the column form,
  // a row's output depends on the chunks that it selected alone.  (The look at the sums: training step of 2 x 4096 tokens, 8 heads 470.5 -> 472.7 us.)
  auto walk = [&](auto apart) __attribute__((always_inline)) {
    const int e0 = __builtin_amdgcn_readfirstlane(entry_at(0));
    int e1 = __builtin_amdgcn_readfirstlane(entry_at(1)), e2 = __builtin_amdgcn_readfirstlane(entry_at(2)), e3 = __builtin_amdgcn_readfirstlane(entry_at(3));  // of steps t + 1, t + 2, t + 3
    feed(tile_k(0, e0));
    feed(tile_k(1, e1));
    feed(tile_v(0, e0));
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    ref = -INFINITY, top = -INFINITY, l_run = 0.f, alpha = 1.f;
    wait_loads_but<2 * NI>();  // K(0)
    __syncthreads();
    scores(std::false_type{}, 0, Tile{});
    mask((e0 & 0xffff) << 6, e0 >> 16, word_of(e0));
    static_for<21>([&](auto sl) { soft(sl); });
    next();
    alpha = 1.f;
    __syncthreads();  // every wave has read K(0)
    feed(tile_k(2, e2));
    int e_nx = entry_at(4);
    // Two barriers per step: before S(t + 1) and before the products with V(t).  A tile of V is asked for behind the first, one of K behind the
    // second (among the products of that part), each one and a half steps ahead of its use; 2 NI loads are younger than the ones that a
    // barrier hands over.
    for (int t = 0; t < nstep; ++t) {
      wait_loads_but<2 * NI>();  // K(t + 1)
      __syncthreads();           // and every wave is done with V(t - 1)
      const uint32_t word = word_of(e1);
      scores(std::true_type{}, t + 1, tile_v(t + 1, e1));
      wait_loads_but<2 * NI>();  // V(t)
      __syncthreads();           // and every wave is done with K(t + 1)
      mask((e1 & 0xffff) << 6, e1 >> 16, t + 1 < nstep ? word : 0u);
      sums(apart, t, tile_k(t + 3, e3));
      e1 = e2, e2 = e3, e3 = __builtin_amdgcn_readfirstlane(e_nx);
      e_nx = entry_at(t + 5);
    }
    if constexpr (!decltype(apart)::value) {
      float x[4] = {0.f, 0.f, 0.f, 0.f};  // NaN if a sum is not finite
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i & 3] = fmaf(o[dt][i], 0.f, x[i & 3]);
      const bool mine = __any(valid && (x[0] + x[1]) + (x[2] + x[3]) != 0.f);
      if (lane == 0) sAgain[wave] = mine;
    }
    wait_all_loads();
    __syncthreads();  // every wave is done with the rings and nothing is in flight: they now hold the output tiles
  };
  walk(std::false_type{});
  if (__builtin_amdgcn_readfirstlane(sAgain[0] | sAgain[1] | sAgain[2] | sAgain[3]) != 0) walk(std::true_type{});

  const float l_tot = sum_xor32_f(l_run);
  const bool empty = !(l_tot > 0.f);
  const float inv = empty ? 0.f : 1.f / l_tot;
  uint16_t *sOut = reinterpret_cast<uint16_t *>(smem) + (size_t)wave * 32 * LDO;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2 *>(sOut + (lane & 31) * LDO + dt * 32 + 8 * g + 4 * hh) =
          make_uint2(pack2<T>(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv), pack2<T>(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv));
  if (valid && hh == 0)
    a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = empty ? INFINITY : (ref + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f;
  wave_lds_fence();
#pragma unroll
  for (int v0 = 0; v0 < 32 * VPR; v0 += 64) {
    const int v = v0 + lane, rl = v / VPR, e = (v - rl * VPR) * 8;
    const int r2 = r0 + wave * 32 + rl;
    if (r2 < Lq && e < D) {
      const Pack8 x = *reinterpret_cast<const Pack8 *>(sOut + rl * LDO + e);
      *reinterpret_cast<Pack8 *>(reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + r2) * a.o_row_stride + (int64_t)h * a.o_head_stride + e) = x;
    }
  }
}

int launch_rows_wide(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, const RowGate *gate, hipStream_t s) {
  typedef FwdRowsDirectSmem<256, 4, 1> SM;
  auto kern = a.dtype == FMOBA_DTYPE_BF16 ? (gate != nullptr ? attn_fwd_rows_wide_kernel<bf16_t, true> : attn_fwd_rows_wide_kernel<bf16_t, false>)
                                          : (gate != nullptr ? attn_fwd_rows_wide_kernel<f16_t, true> : attn_fwd_rows_wide_kernel<f16_t, false>);
  const int step_cap = ceil_div(a.max_seqlen_k, 64);  // (at most kRowsStepCap: fwd_rows_feasible)
  const size_t smem = SM::bytes(step_cap, nw) + 16;  // (and the four words of sAgain)
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_fwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const ItemOrder order = item_order(a.total_q, a.max_seqlen_q, a.batch, a.heads, SM::ROWS, longest_items_first(std::max(a.total_q, a.total_k), a.heads, 256 * 4));
  const int64_t items = a.heads * (order == kListedLongestFirst ? listed_blocks(a.total_q, a.batch, SM::ROWS) : (int64_t)a.batch * ceil_div(a.max_seqlen_q, SM::ROWS));
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_fwd: too many (sequence, head, row block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(256), smem, s, a, bm, nw, step_cap, order, gate != nullptr ? *gate : RowGate{});
  return 0;
}

}  // namespace fmoba
