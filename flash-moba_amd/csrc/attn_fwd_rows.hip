// Sparse attention forward, row-block form, for patterns dense enough that most row blocks
// touch most of the chunks they may see (flash_fwd_kernel.h:325-700 of the reference walks the
// same (row block, key block) grid through its CSC lists).
//
// One workgroup owns a block of consecutive query rows of one (sequence, head) and walks, in ascending
// key order, the 64-key blocks of every chunk that at least one of its rows selected; all rows take
// part in the matrix products of a step, and the rows that did not select the chunk are masked out
// of the softmax (their probabilities are exact zeros).  The running maximum, the running sum and
// the output accumulators stay in registers for the whole walk, so nothing but Q, K, V and the
// output moves.  Two kernels: attn_fwd_rows_kernel (128 rows and four waves per workgroup, or 64 rows and one, two or
// four sets of two, that fetch the K/V tiles straight into LDS themselves; head dimensions up to 128 and up to
// 512 chunks per sequence) and attn_fwd_rows_loader_kernel (128 rows, four compute and four loader waves; longer
// sequences).  Head dimensions above 128 have a loop of their own in attn_fwd_rows_wide.hip.  Calls with at most eight query rows per sequence have a
// kernel of their own (attn_fwd_few.hip).
//
// The selection of a row is one bit per chunk (the gating's own, or a bitmap built from the CSC lists by
// csc_bitmap_lds_kernel); the chunks a workgroup walks are the OR of its rows' bitmaps.
#include "attn_fwd_rows.h"
#include "gate_select.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace fmoba {

template <int HD>
struct FwdRowsSmem {
  static constexpr int LDQ = HD + 16;  // elements, K / V tiles (conflict-free for row reads and transposing reads)
  static constexpr int LDO = HD + 8;   // elements, per-wave output tile [32 rows][LDO]
  static constexpr size_t stage = (size_t)2 * 64 * LDQ * 2;  // K then V of one step
  static constexpr size_t oKV = 0;                            // [2 stages]; the output tiles reuse it at the end
  static constexpr size_t oStep = oKV + 2 * stage;            // int[kRowsStepCap]: key block | chunk << 16
  static constexpr size_t oUnion = oStep + (size_t)kRowsStepCap * 4;
  static constexpr size_t oOff = oUnion + (size_t)kRowsWordCap * 4;  // int[kRowsWordCap + 1]
  static constexpr size_t bytes = oOff + (size_t)(kRowsWordCap + 1) * 4 + 12;
  static_assert((size_t)4 * 32 * LDO * 2 <= 2 * stage, "output tiles must fit the K/V stages");
};

// one bit per (row, head, chunk): bm[(h * nw + c / 32) * total_q + q0 + r] bit c % 32 (the layout the gating
// leaves its selection in).  The lists may be in any order.
// A workgroup sets the words of a word column (32 lists) of one sequence in LDS and writes all of them: nothing to clear before, no atomics
// in memory (12037 tokens in five sequences, 16 heads, top-k 8 of 64-key chunks: 17.7 us and 4.9 to clear -> 8.5; 32000
// tokens, 8 heads, top-k 64 168 and 6 -> 37).  What is left
// is a chain of four loads.  A wave takes 1024 entries of a list at a time, sixteen loads in flight; sixteen waves, four where lists are
// of a few rows and workgroups many (decode of eight sequences, 32 heads: 9.0 us, 19.9 with sixteen).  grid (nw, heads, batch)
constexpr int kBitmapRows = 32768;  // rows of a sequence whose words fit a workgroup's LDS
__global__ __launch_bounds__(1024) void csc_bitmap_lds_kernel(fmoba_attn_fwd_args a, uint32_t *bm, int nw) {
  extern __shared__ uint32_t words[];
  __shared__ int64_t first[32];
  __shared__ int count[32];
  const int w = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int q0 = a.cu_seqlens_q[b], Lq = min(a.cu_seqlens_q[b + 1] - q0, a.max_seqlen_q);
  if (Lq <= 0) return;
  const int64_t bh = (int64_t)b * a.heads + h;
  if (tid < 32) {
    const int c = w * 32 + tid;
    first[tid] = c < a.max_cols ? a.col_offsets[bh * a.max_cols + c] : 0;
    count[tid] = c < a.max_cols ? a.col_nnz[bh * a.max_cols + c] : 0;
  }
  for (int i = tid; i < Lq; i += blockDim.x) words[i] = 0u;
  __syncthreads();
  for (int j = 0; j < 32; ++j) {
    const int n = __builtin_amdgcn_readfirstlane(count[j]);
    for (int p = ((wave - j) & (waves - 1)) * 1024; p < n; p += waves * 1024) {  // (short lists: a wave each)
      const int32_t *list = a.row_indices + first[j] + p;
      int r[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) r[i] = p + i * 64 + lane < n ? list[i * 64 + lane] : -1;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (r[i] >= 0 && r[i] < Lq) atomicOr(&words[r[i]], 1u << j);
    }
  }
  __syncthreads();
  uint32_t *out = bm + ((int64_t)h * nw + w) * a.total_q + q0;
  for (int i = tid; i < Lq; i += blockDim.x) out[i] = words[i];
}
// longer sequences
__global__ __launch_bounds__(256) void csc_bitmap_kernel(fmoba_attn_fwd_args a, uint32_t *bm, int nw) {
  const int c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int64_t bh = (int64_t)b * a.heads + h;
  const int nnz = a.col_nnz[bh * a.max_cols + c];
  const int32_t *list = a.row_indices + a.col_offsets[bh * a.max_cols + c];
  const uint32_t bit = 1u << (c & 31);
  for (int i = threadIdx.x; i < nnz; i += 256) {
    const int r = list[i];
    if (r >= 0 && r < Lq) atomicOr(&bm[((int64_t)h * nw + (c >> 5)) * a.total_q + q0 + r], bit);
  }
}

__global__ void fwd_zero_u32_kernel(uint32_t *p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0u;
}

template <typename T, int HD>
__global__ __launch_bounds__(512) void attn_fwd_rows_loader_kernel(fmoba_attn_fwd_args a, const uint32_t *bm, int nw) {
  typedef FwdRowsSmem<HD> SM;
  constexpr int KS = HD / 16, LDQ = SM::LDQ, LDO = SM::LDO, NDT = HD / 32, VPR = HD / 8;
  constexpr int NTHR = 512;
  constexpr int NV = 64 * VPR / 256;    // 16-byte vectors of one 64-key tile per loader thread
  constexpr int KSTEP = 256 / VPR;      // keys between two consecutive vectors of a loader thread
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int *sStep = reinterpret_cast<int *>(smem + SM::oStep);
  uint32_t *sUnion = reinterpret_cast<uint32_t *>(smem + SM::oUnion);
  int *sOff = reinterpret_cast<int *>(smem + SM::oOff);

  const int nrb = (a.max_seqlen_q + 127) / 128;
  const PairItem item = xcd_pair_item(blockIdx.x, a.batch * a.heads, nrb);
  const int b = item.pair / a.heads, h = item.pair - b * a.heads;
  const int q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
  const int rb = nrb - 1 - item.idx;  // the longest walks (last rows of a causal sequence) start first
  const int r0 = rb * 128;
  if (r0 >= Lq) return;
  const int k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
  const int off = Lk - Lq;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = lane >> 5;
  const bool is_loader = wave >= 4;
  const bool causal = a.is_causal != 0;
  const int Bn = a.lg_block_n, sub = Bn >> 6;
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;

  // ---- the steps of this row block -------------------------------------------------------------
  const int rlast = min(r0 + 127, Lq - 1);
  const int kend = min(Lk, causal ? rlast + off + 1 : Lk);  // keys [0, kend) are visible to some row
  const int nchunk = kend > 0 ? (kend + Bn - 1) / Bn : 0;
  const int nwu = min((nchunk + 31) >> 5, nw);
  for (int w = tid; w < nwu; w += NTHR) sUnion[w] = 0u;
  __syncthreads();
  {
    const int nrow = rlast - r0 + 1;
    const uint32_t *bp = bm + (int64_t)h * nw * a.total_q + q0 + r0;
    for (int i = tid; i < nrow * nwu; i += NTHR) {
      const int w = i / nrow, row = i - w * nrow;
      const uint32_t x = bp[(int64_t)w * a.total_q + row];
      if (x) atomicOr(&sUnion[w], x);
    }
  }
  __syncthreads();
  // One thread per chunk: a chunk of the union contributes its 64-key blocks that hold a visible key; a scan over the
  // workgroup gives every chunk the place of its first step (a thread per selection word walking its bits one after
  // the other took 6 of the 11 us that a workgroup spends outside its step loop).
  int nstep_all = 0;
  const int nchunk_u = min(nchunk, nwu * 32);
  for (int c0 = 0; c0 < nchunk_u; c0 += NTHR) {
    const int c = c0 + tid;
    int cnt = 0;
    if (c < nchunk_u && ((sUnion[c >> 5] >> (c & 31)) & 1u)) cnt = min(sub, (kend - c * Bn + 63) >> 6);
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(incl, o, 64);
      incl += lane >= o ? up : 0;
    }
    if (lane == 63) sOff[wave] = incl;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NTHR / 64; ++w) {
      const int v = sOff[w];
      before += w < wave ? v : 0;
      total += v;
    }
    int pos = nstep_all + before + incl - cnt;
    for (int jb = 0; jb < cnt; ++jb, ++pos)
      if (pos < kRowsStepCap) sStep[pos] = (c * sub + jb) | (c << 16);
    nstep_all += total;
    __syncthreads();
  }
  const int nstep = min(nstep_all, kRowsStepCap);

  typedef std::integral_constant<int, 0> C0;
  typedef std::integral_constant<int, 1> C1;
  const int nstep_pad = (nstep + 1) & ~1;
  if (nstep == 0) {  // no visible selected key: out = 0, lse = +inf for the rows of this block
    if (!is_loader) {
      const int row = r0 + wave * 32 + (lane & 31);
      if (row < Lq) {
        uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + row) * a.o_row_stride + (int64_t)h * a.o_head_stride;
        for (int e = hh * 8; e < D; e += 16) *reinterpret_cast<Pack8 *>(op + e) = zero_pack8();
        if (hh == 0) a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = INFINITY;
      }
    }
    return;
  }

  // K runs one step ahead of V: while the softmax of step t is evaluated the matrix cores already form
  // S of step t + 1.  Stage (t & 1) of each ring holds K(t) resp. V(t).
  uint16_t *const sKst = reinterpret_cast<uint16_t *>(smem + SM::oKV);
  uint16_t *const sVst = sKst + 2 * 64 * LDQ;

  if (is_loader) {
    const int lt = tid - 256;
    const int kb = lt / VPR, e = (lt - kb * VPR) * 8;
    const int ec = min(e, D - 8);
    const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)k0 * a.k_row_stride + (int64_t)hk * a.k_head_stride + ec;
    const uint16_t *vp = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)k0 * a.v_row_stride + (int64_t)hk * a.v_head_stride + ec;
    Pack8 rk[2][NV], rv[2][NV];
    // loads are unconditional (steps and keys clamped, the surplus zeroed when stored) so that the
    // outstanding loads are counted exactly
    const int64_t kstep_k = (int64_t)KSTEP * a.k_row_stride, kstep_v = (int64_t)KSTEP * a.v_row_stride;
    const bool whole_rows = D == HD;
    auto load_tile = [&](Pack8(&r)[NV], const uint16_t *base, int64_t row_stride, int64_t step_stride, int t) {
      const int key0 = (sStep[min(t, nstep - 1)] & 0xffff) << 6;
      if (key0 + 64 <= Lk) {  // every key of the tile exists: one multiplication, then additions
        const uint16_t *p0 = base + (int64_t)(key0 + kb) * row_stride;
#pragma unroll
        for (int i = 0; i < NV; ++i) r[i] = ld_global16(p0 + i * step_stride);
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i) r[i] = ld_global16(base + (int64_t)min(key0 + kb + i * KSTEP, Lk - 1) * row_stride);
      }
    };
    auto load_k = [&](auto par, int t) { load_tile(rk[decltype(par)::value], kp, a.k_row_stride, kstep_k, t); };
    auto load_v = [&](auto par, int t) { load_tile(rv[decltype(par)::value], vp, a.v_row_stride, kstep_v, t); };
    auto store_tile = [&](uint16_t *dst, const Pack8(&r)[NV], int t) {
      const int key0 = (sStep[t] & 0xffff) << 6;
      if (whole_rows && key0 + 64 <= Lk) {
#pragma unroll
        for (int i = 0; i < NV; ++i) *reinterpret_cast<Pack8 *>(dst + (kb + i * KSTEP) * LDQ + e) = r[i];
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int kl = kb + i * KSTEP;
          const bool ok = e < D && key0 + kl < Lk;
          Pack8 x = r[i];
#pragma unroll
          for (int w = 0; w < 4; ++w) x.w[w] = ok ? x.w[w] : 0u;
          *reinterpret_cast<Pack8 *>(dst + kl * LDQ + e) = x;
        }
      }
    };
    load_k(C0{}, 0);
    load_k(C1{}, 1);
    load_v(C0{}, 0);
    store_tile(sKst, rk[0], 0);
    load_k(C0{}, 2);
    load_v(C1{}, 1);
    __syncthreads();  // K(0) is in LDS
    if (1 < nstep) store_tile(sKst + 64 * LDQ, rk[1], 1);
    store_tile(sVst, rv[0], 0);
    load_k(C1{}, 3);
    load_v(C0{}, 2);
    auto loader_step = [&](auto par, int t) {  // par: parity of step t
      constexpr int P = decltype(par)::value;
      __syncthreads();  // K(t + 1) and V(t) are in LDS; the readers of K(t) and V(t - 1) are done
      if (t + 2 < nstep) store_tile(sKst + P * 64 * LDQ, rk[P], t + 2);
      if (t + 1 < nstep) store_tile(sVst + (P ^ 1) * 64 * LDQ, rv[P ^ 1], t + 1);
      load_k(par, t + 4);
      load_v(std::integral_constant<int, (P ^ 1)>{}, t + 3);
    };
    for (int t = 0; t < nstep_pad; t += 2) {
      loader_step(C0{}, t);
      loader_step(C1{}, t + 1);
    }
    __syncthreads();  // the compute waves are done with the stages
  } else {
    const int row = r0 + wave * 32 + (lane & 31);
    const bool valid = row < Lq;
    const int lim = valid ? min(causal ? row + off : 0x7fffffff, Lk - 1) : -1;  // last visible key
    const uint32_t *bmrow = bm + (int64_t)h * nw * a.total_q + q0 + min(row, Lq - 1);
    // this lane's query row as the B operand of S^T = K Q^T
    Pack8 qb[KS];
    {
      const uint16_t *qg = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)(q0 + min(row, Lq - 1)) * a.q_row_stride + (int64_t)h * a.q_head_stride;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int e = (hh * KS + ks) * 8;
        qb[ks] = (valid && e < D) ? ld_global16(qg + e) : zero_pack8();
      }
    }
    f32x16 o[NDT];  // O^T: register i of feature tile dt <-> feature dt*32 + acc_row(i, hh), this lane's row
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    f32x16 st[2][2];  // S^T of step t in st[t & 1]: register i of tile kt <-> key kt*32 + acc_row(i, hh), this lane's row
    float m_run = -INFINITY, l_run = 0.f;  // running maximum of the raw scores, running sum (this half of the wave)
    int cur_w = -1;
    uint32_t myword = 0u;
    const int kro = (lane & 31) * LDQ + hh * KS * 8;  // this lane's K row / feature slice within a 32-key tile

    auto k_frag = [&](const uint16_t *sK, int kt, int ks) { return *reinterpret_cast<const Pack8 *>(sK + kt * 32 * LDQ + kro + ks * 8); };
    // S of one step, not overlapped with anything (first step, and steps whose softmax the wave skips)
    auto s_plain = [&](const uint16_t *sK, f32x16(&sn)[2]) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        Pack8 kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[ks] = k_frag(sK, kt, ks);
#pragma unroll
        for (int i = 0; i < 16; ++i) sn[kt][i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sn[kt] = mfma32<T>(kf[ks], qb[ks], sn[kt]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };

    auto body = [&](auto par, int t) {
      constexpr int P = decltype(par)::value;
      const uint16_t *sKn = sKst + (P ^ 1) * 64 * LDQ;  // K(t + 1)
      const uint16_t *sV = sVst + P * 64 * LDQ;         // V(t)
      f32x16(&sc)[2] = st[P];
      f32x16(&sn)[2] = st[P ^ 1];
      const int s = sStep[t];
      const int key0 = (s & 0xffff) << 6, c = s >> 16;
      if ((c >> 5) != cur_w) {
        cur_w = c >> 5;
        myword = valid ? bmrow[(int64_t)cur_w * a.total_q] : 0u;
      }
      const bool active = ((myword >> (c & 31)) & 1u) != 0u && lim >= key0;
      // ---- part 0: operands of the first half of S(t + 1); row maximum of step t ----
      Pack8 kf[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = k_frag(sKn, 0, ks);
      const int lim_rel = active ? lim - key0 : -1;
      if (!__all(lim_rel >= 63 || lim_rel < 0)) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int jrel = kt * 32 + 8 * (i >> 2) + (i & 3) + 4 * hh;
            sc[kt][i] = jrel <= lim_rel ? sc[kt][i] : -INFINITY;
          }
      }
      float mloc = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, sc[kt][i]);
      mloc = max_xor32_f(mloc);
      // The reference point of the row's exponentials only moves when the block's maximum exceeds it by more than
      // 2^8 after scaling (always on the row's first block): p stays below 256, which the 16-bit P and the fp32 sums
      // hold easily, out and lse do not depend on the reference point, and O is rescaled a few times per row
      // instead of whenever one of the wave's 32 rows meets a new maximum.
      const bool grow = active & ((mloc - m_run) * scale_log2 > 8.f);
      const float m_new = grow ? mloc : m_run;
      const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);  // first visit: factor 0 on zeros
      const float neg_mc = active ? -m_new * scale_log2 : -INFINITY;  // rows that did not select the chunk: p = 0
      m_run = m_new;
      l_run *= alpha;
      if (!__all(alpha == 1.f)) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- part 1: S(t + 1) on the matrix cores under the exponentials of step t ----
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sn[kt][i] = 0.f;
      Pack8 pf[2][2];  // P^T as the B operand of O^T += V^T P^T, straight from the accumulators
      Pack8 vt[2][2];  // V^T operands of one feature tile
      lds_cu16 *trV = tr_lane_base(sV, LDQ, lane) + 4 * hh * LDQ;
      float lsum = 0.f;
      static_for<16>([&](auto gi) {
        constexpr int g = decltype(gi)::value;
        constexpr int M0 = g * (2 * KS) / 16, M1 = (g + 1) * (2 * KS) / 16;
#pragma unroll
        for (int mi = M0; mi < M1; ++mi) {
          const int kt = mi / KS, ks = mi % KS;
          sn[kt] = mfma32<T>(kf[ks], qb[ks], sn[kt]);
          if (kt == 0) kf[ks] = k_frag(sKn, 1, ks);  // the operand of the second key tile takes the register over
        }
        constexpr int kte = g / 8, j = g % 8;
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[kte][2 * j], scale_log2, neg_mc));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[kte][2 * j + 1], scale_log2, neg_mc));
        lsum += p0 + p1;
        pf[kte][j / 4].w[j % 4] = pack2<T>(p0, p1);
        if (g == 14) {  // V^T operands of the first feature tile
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
              const int lo = (kt * 32 + 16 * s2) * LDQ;
              vt[kt][s2] = tr_frag8_at(trV, lo, lo + 8 * LDQ);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      l_run += lsum;
      // ---- part 2: O^T += V^T P^T ----
      static_for<NDT>([&](auto di) {
        constexpr int dt = decltype(di)::value;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            o[dt] = mfma32<T>(vt[kt][s2], pf[kt][s2], o[dt]);
            if (dt + 1 < NDT) {  // the operand of the next feature tile takes the register over
              const int lo = (kt * 32 + 16 * s2) * LDQ + (dt + 1) * 32;
              vt[kt][s2] = tr_frag8_at(trV, lo, lo + 8 * LDQ);
            }
          }
        __builtin_amdgcn_sched_barrier(0);
      });
    };

    __syncthreads();  // K(0) is in LDS
    s_plain(sKst, st[0]);
    for (int t = 0; t < nstep_pad; t += 2) {
      __syncthreads();  // K(t + 1) and V(t) are in LDS
      body(C0{}, t);
      __syncthreads();
      if (t + 1 < nstep) body(C1{}, t + 1);
    }
    __syncthreads();  // every wave is done with the stages: they now hold the output tiles

    const float l_tot = sum_xor32_f(l_run);
    const bool empty = !(l_tot > 0.f);
    const float inv = empty ? 0.f : 1.f / l_tot;
    uint16_t *sOut = reinterpret_cast<uint16_t *>(smem + SM::oKV) + (size_t)wave * 32 * LDO;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2 *>(sOut + (lane & 31) * LDO + dt * 32 + 8 * g + 4 * hh) =
            make_uint2(pack2<T>(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv), pack2<T>(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv));
    if (valid && hh == 0)
      a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = empty ? INFINITY : (m_run * scale_log2 + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f;
    wave_lds_fence();
    // rows leave as 16-byte pieces, VPR of them per row, consecutive lanes taking consecutive pieces
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
}

// ------------------------------------------------------------------------------------
// The same walk without loader waves, for head dimensions up to 128: four (two) waves of 32 rows and 256 registers, two
// workgroups per compute unit, so that the matrix products of one run under the softmax arithmetic of the other whatever
// their steps wait for.  K and V tiles go from global memory straight into LDS (every wave issues a quarter of a tile's
// loads, one step ahead, rings of two stages each) in rows of exactly HD elements, swizzled instead of padded (piece c of row
// r lies at piece c ^ tile_swz(r)): the 16-byte row reads of the K operands and the transposing reads of the V^T operands
// both spread over all banks.  Keys past the sequence and features past head_dim are fetched from a key and a piece that
// exist: the scores of such keys are masked, Q is zero in such features and the corresponding output features are never
// stored.
// With eight waves of one workgroup in step (256 rows, the second four a part of a step late, rings two and three steps
// ahead), half of the tile loads but one barrier for all: 65536 tokens in eight sequences, top-k 32 of 64-key chunks 3.08 ms
// against 2.87 here, 2 x 4096 tokens 247 against 205 us, 12037 tokens in five sequences 290 against 253, 8191 tokens of short
// documents with heads of 64 51 against 40 (two workgroups cover each other's first loads, and 128 rows are less padding).
// Head dimensions 65 to 96 have tiles of 96 features (rows of 192 bytes): a quarter of the products of 128-feature tiles less
// (12037 tokens, 16 heads of 96, top-k 8 of 64-key chunks 208 -> 176 us; 2048 tokens, 8 heads 41 -> 29).
// With the products at a higher priority than the rest of a step, whole training steps: 65536 tokens in eight sequences 7681 -> 7549 us, 2 x 4096 tokens,
// top-k 8 of 128-key chunks 496 -> 484, 12037 tokens, 16 heads of 96 484 -> 481, 8191 tokens of short documents the same.
// GATED: the rows choose their chunks here (up to kRowGateChunks of them), while Q is in registers anyway, and the words of the selection go to memory only if
// column lists follow (with the counts these need).  The search for a row's cut is vector arithmetic of one wave beside the products of another workgroup's, where a gate
// launch in front leaves the matrix cores idle, reads Q once more and is a launch.  Whole calls: forward of 1024 + 2048 tokens, 8 heads of 64 33.5 -> 30.1 us,
// 1024 tokens 23.8 -> 20.6, 2048 tokens, 16 heads of 128 53.2 -> 50.3, parts of prompts of 512 and 1000 rows against 4000 and 7000 keys, 32 over 8 heads 172 ->
// 166; training step of 8191 tokens of short documents 122.2 -> 116.4, 5000 tokens, 8 heads of 112 216 -> 211, 8 x 4096 tokens, 32 over 8 heads, forward 1262
// -> 1234; nothing from 24571 tokens of training on.  (One to six scalars of these instances are spilled, none without the choice.)
// RW: waves of a set, which share its tiles.  SPLIT = 2 (4): two (four) sets of waves take turns at the steps of the same rows, with
// rings of their own; the results of a row meet in LDS at the end.  KH = 2: the tiles of a set are two waves', half kh of the keys each.  Which of them: launch_rows.
// ------------------------------------------------------------------------------------
template <typename T, int HD, int RW, int SPLIT, int KH, bool GATED>
__global__ __launch_bounds__(SPLIT * KH * RW * 64, 2) void attn_fwd_rows_kernel(fmoba_attn_fwd_args a, const uint32_t *bm, int nw, int step_cap, ItemOrder order, RowGate gate) {
  typedef FwdRowsDirectSmem<HD, RW, SPLIT> SM;
  constexpr int kRows = SM::ROWS;
  constexpr int KS = HD / 16, LDO = SM::LDO, NDT = HD / 32, VPR = HD / 8;
  constexpr int NSETS = SPLIT * KH, NTHR = NSETS * RW * 64;
  constexpr int NKT = 2 / KH;           // 32-key halves of a tile that a wave takes
  constexpr int RB = HD * 2;            // bytes of a tile row
  constexpr int FW = KH * RW;           // waves that share a ring
  constexpr int NI = VPR / FW;          // direct-to-LDS instructions (64 lanes x 16 bytes) per tile and wave
  static_assert(NI >= 1 && NI * FW == VPR, "the waves of a ring share the loads of a tile");
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  int *sStep = reinterpret_cast<int *>(smem + SM::oStep);
  uint32_t *sUnion = reinterpret_cast<uint32_t *>(sStep + step_cap);
  uint32_t *sBits = sUnion + nw * SM::UPW;

  // the longest walks (last rows of a causal sequence) start first
  int b, h, rb, q0, Lq, k0, Lk, km0 = 0, Cm = 0;  // km0, Cm: the sequence's first chunk mean and how many
  if (order == kListedLongestFirst) {
    const BlockItem item = listed_item<kRows, true>(blockIdx.x, a.batch, a.heads, a.max_seqlen_q, a.cu_seqlens_q, a.cu_seqlens_k, GATED ? gate.cu_seqlens_km : nullptr);
    if (item.b < 0) return;
    b = item.b, h = item.h, rb = item.idx, q0 = item.q0, Lq = item.Lq, k0 = item.k0, Lk = item.Lk, km0 = item.m0, Cm = item.Cm;
  } else {
    const int nrb = (a.max_seqlen_q + kRows - 1) / kRows;
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * a.heads, nrb, false, order == kLongestFirst);
    b = item.pair / a.heads, h = item.pair - b * a.heads, rb = nrb - 1 - item.idx;
    q0 = a.cu_seqlens_q[b], Lq = a.cu_seqlens_q[b + 1] - q0;
    k0 = a.cu_seqlens_k[b], Lk = a.cu_seqlens_k[b + 1] - k0;
    if constexpr (GATED) km0 = gate.cu_seqlens_km[b], Cm = gate.cu_seqlens_km[b + 1] - km0;
  }
  const int r0 = rb * kRows;
  if (r0 >= Lq) return;
  const int off = Lk - Lq;
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  const int wave = wave_all % RW, sid = wave_all / RW;    // rows 32 wave ..
  const int set = sid / KH, kh = sid % KH;                // steps set, set + SPLIT, .., half kh of the keys of a tile
  const int feeder = wave_all % FW;
  const bool causal = a.is_causal != 0;
  const int Bn = a.lg_block_n;
  const float scale_log2 = a.softmax_scale * 1.4426950408889634f;

  const int row = r0 + wave * 32 + (lane & 31);
  const bool valid = row < Lq;
  // this lane's query row as the B operand of S^T = K Q^T: asked for first, on its way while the steps are counted
  Pack8 qb[KS];
  {
    const uint16_t *qg = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride;
    q_rows_load<HD>(qb, qg, a.q_row_stride, r0 + wave * 32, Lq, lane, D);
  }

  // ---- the steps of this row block -------------------------------------------------------------
  const int rlast = min(r0 + kRows - 1, Lq - 1);
  const int kend = min(Lk, causal ? rlast + off + 1 : Lk);  // keys [0, kend) are visible to some row
  int nstep_all;
  if constexpr (GATED) {
    static_assert(row_gate_lds<HD>() <= SM::ring, "the chunk means lie where the K/V rings will");
    gate_row_block<T, HD, RW, NSETS>(a, gate, smem, sBits, reinterpret_cast<int *>(sBits + nw * kRows), qb, b, h, hk, q0, r0, rlast, Lq, off, nw, km0, Cm);
    nstep_all = gated_row_block_steps<kRows>(kend, Bn, nw, step_cap, sStep, sBits);
  } else {
    nstep_all = row_block_steps<kRows, NTHR>(bm + (int64_t)h * nw * a.total_q + q0 + r0, a.total_q, rlast - r0 + 1, kend, Bn, nw, step_cap, sStep, sUnion, sBits);
  }
  const int nstep_wg = min(nstep_all, step_cap);
  const int nstep = (nstep_wg - set + SPLIT - 1) / SPLIT, nturn = (nstep_wg + SPLIT - 1) / SPLIT;  // this set's steps, the turns of the loop
  // The entries of 64 turns from turn wbase on, one per lane: those of a step come into scalar registers by a lane read.  (Read from LDS in
  // front of a step's loads they were two dependent LDS reads at the start of every step: 65536 tokens in eight sequences, training step 7243 -> 7156 us,
  // 12037 tokens, heads of 96 465 -> 462, 2 x 4096 tokens 457.5 -> 455.7, forward of 3072 tokens, 8 heads of 64 34.7 -> 33.8.)
  int wbase = 0, ent = 0;
  auto entries_from = [&](int t) {
    wbase = t;
    ent = sStep[min((t + lane) * SPLIT + set, nstep_wg - 1)];
  };
  auto entry = [&](int t) { return __builtin_amdgcn_readlane(ent, t - wbase); };

  typedef std::integral_constant<int, 0> C0;
  typedef std::integral_constant<int, 1> C1;
  if (nstep_wg == 0) {  // no visible selected key: out = 0, lse = +inf for the rows of this block
    if (valid && sid == 0) {
      uint16_t *op = reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + row) * a.o_row_stride + (int64_t)h * a.o_head_stride;
      for (int e = hh * 8; e < D; e += 16) *reinterpret_cast<Pack8 *>(op + e) = zero_pack8();
      if (hh == 0) a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = INFINITY;
    }
    return;
  }

  // ---- feeding the rings: each wave of a set (two or four) fetches an equal run of a tile's 16-byte pieces, NI loads of 64 ----
  const uint32_t ldsK = (uint32_t)(uintptr_t)smem + (uint32_t)(set * (int)SM::ring), ldsV = ldsK + (uint32_t)(2 * SM::tile);
  const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)k0 * a.k_row_stride + (int64_t)hk * a.k_head_stride;
  const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)k0 * a.v_row_stride + (int64_t)hk * a.v_head_stride;
  // A lane's piece in load i, number (wave * NI + i) * 64 + lane of the tile: its byte offset from the tile's first key, for K
  // and for V.  A tile whose 64 keys all exist is fetched from a wave-uniform base plus these offsets (no vector
  // instruction per load); the last tile of a sequence clamps the keys per lane.
  uint32_t lofK[NI], lofV[NI];
  {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int v = (feeder * NI + i) * 64 + lane, tr = v / VPR, p = v - tr * VPR;
      const uint32_t e = (uint32_t)min((p ^ tile_swz<HD>(tr)) * 8, D - 8);
      lofK[i] = run_offset(((uint32_t)tr * (uint32_t)a.k_row_stride + e) * 2u, i % 4);
      lofV[i] = run_offset(((uint32_t)tr * (uint32_t)a.v_row_stride + e) * 2u, i % 4);
    }
  }
  auto feed = [&](const uint16_t *g, uint32_t row_stride, const uint32_t(&lof)[NI], uint32_t lds_ring, int stage, int t) {
    const int key0 = (entry(t) & 0xffff) << 6;
    const uint32_t dst = lds_ring + (uint32_t)__builtin_amdgcn_readfirstlane(stage * (int)SM::tile + feeder * NI * 1024);
    if (key0 + 64 <= Lk) {
      const uint16_t *base = g + (uint64_t)(uint32_t)key0 * row_stride;
      global_to_lds16_run<(NI < 4 ? NI : 4)>(lof, base, dst);
      if constexpr (NI > 4) global_to_lds16_run<NI - 4>(lof + 4, base, dst + 4096u);
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int v = (feeder * NI + i) * 64 + lane, tr = v / VPR, p = v - tr * VPR;  // row of the tile, piece
        const uint32_t e = (uint32_t)min((p ^ tile_swz<HD>(tr)) * 8, D - 8);
        const uint32_t key = (uint32_t)min(key0 + tr, Lk - 1);
        global_to_lds16(g + ((uint64_t)key * row_stride + e), dst + (uint32_t)(i * 1024));
      }
    }
  };
  auto feed_k = [&](int t) { feed(kg, (uint32_t)a.k_row_stride, lofK, ldsK, t & 1, t); };
  auto feed_v = [&](int t) { feed(vg, (uint32_t)a.v_row_stride, lofV, ldsV, t & 1, t); };
  const int lim = valid ? min(causal ? row + off : 0x7fffffff, Lk - 1) : -1;  // last visible key
  // (Q is in registers before the first tile loads are issued: from here on the wave counts its outstanding loads)
  if constexpr (!GATED) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qb[ks].w[0]), "+v"(qb[ks].w[1]), "+v"(qb[ks].w[2]), "+v"(qb[ks].w[3]));
#endif
    q_rows_arrange<HD>(qb, hh, D);
    wait_all_loads();
  }
  entries_from(0);
  feed_k(0);
  feed_k(1);
  feed_v(0);

  f32x16 o[NDT];  // O^T: register i of feature tile dt <-> feature dt*32 + acc_row(i, hh), this lane's row
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  f32x16 st[2][NKT];  // S^T of step t in st[t & 1]: register i of tile kt <-> key (kh + kt)*32 + acc_row(i, hh), this lane's row
  float m_run = -INFINITY, l_run = 0.f;  // running maximum of the raw scores, running sum (this half of the wave)
  // byte offsets of this lane's pieces inside a tile: row reads (key lane % 32 of a 32-key half, pieces hh * KS ..) and
  // transposing reads (key (lane % 16) / 4 + 4 hh, feature tile 0); every other operand is an exclusive-or on the piece
  // bits plus a constant
  const uint32_t rowoff = (uint32_t)((kh * 32 + (lane & 31)) * RB + ((tile_frag_piece<HD>(hh, 0) ^ tile_swz<HD>(lane & 31)) * 16));
  const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
  const uint32_t troff = (uint32_t)((kh * 32 + r0t) * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
  auto opaque = [](uint32_t &x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#else
    (void)x;
#endif
  };
  auto k_frag = [&](uint32_t ak, int kt, int ks) { return lds_read16(tile_frag_addr<HD>(ak, ks) + (uint32_t)(kt * 32 * RB)); };
  auto v_frag = [&](uint32_t tv, int dt, int kt, int s2) {
    const uint32_t o = (uint32_t)((kt * 32 + 16 * s2) * RB);
    return lds_tr8(tile_tr_addr<HD>(tv, dt) + o, tile_tr_addr8<HD>(tv, dt) + o);
  };
  // S of the first step, not overlapped with anything
  auto s_plain = [&](uint32_t ak, f32x16(&sn)[NKT]) {
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      Pack8 kf[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = k_frag(ak, kt, ks);
#pragma unroll
      for (int i = 0; i < 16; ++i) sn[kt][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) sn[kt] = mfma32<T>(kf[ks], qb[ks], sn[kt]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // A step in three parts.  part0: masks, row maximum and the reference point of step t (vector arithmetic); part1:
  // S(t + 1) on the matrix cores under the exponentials of step t; part2: O^T += V^T P^T of step t (matrix cores).
  // The other wave of the SIMD belongs to another workgroup (or set) and is in whatever part it is in.
  Pack8 pf[NKT][2];    // P^T as the B operand of O^T += V^T P^T, straight from the accumulators
  Pack8 kf[KS];        // K operands of S(t + 1): read at the start of part0, their latency runs under its arithmetic
  Pack8 vt[NKT][2];    // V^T operands of the first feature tile of step t: read at the end of part1
  float neg_mc = 0.f;  // minus the reference point of the row's exponentials, scaled; -inf for a row that skips the step
  int s_nx = entry(0);  // entry of the next step and this row's word of selection bits for its chunk
  uint32_t word_nx = sBits[((s_nx >> 16) >> 5) * kRows + wave * 32 + (lane & 31)];
  auto part0 = [&](auto par, int t) {
    constexpr int P = decltype(par)::value;
    f32x16(&sc)[NKT] = st[P];
    {
      uint32_t akn = ldsK + (uint32_t)(((t + 1) & 1) * (int)SM::tile) + rowoff;  // K(t + 1)
      opaque(akn);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = k_frag(akn, 0, ks);
    }
    // (the step's entry and this row's selection word were read during the step before: two dependent LDS reads at
    // this place would be waited for with nothing to do, by every wave at the start of every step)
    const int s = s_nx;
    const int key0 = ((s & 0xffff) << 6) + kh * 32, c = s >> 16;
    const uint32_t myword = word_nx;
    const bool active = valid && ((myword >> (c & 31)) & 1u) != 0u && lim >= key0;
    const int lim_rel = active ? lim - key0 : -1;
    if (!__all(lim_rel >= 32 * NKT - 1 || lim_rel < 0)) {
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int jrel = kt * 32 + 8 * (i >> 2) + (i & 3) + 4 * hh;
          sc[kt][i] = jrel <= lim_rel ? sc[kt][i] : -INFINITY;
        }
    }
    float mloc = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, sc[kt][i]);
    mloc = max_xor32_f(mloc);
    // The reference point of the row's exponentials only moves when the block's maximum exceeds it by more than 2^8
    // after scaling (always on the row's first block): p stays below 256, out and lse do not depend on the reference
    // point, and O is rescaled a few times per row instead of whenever one of the wave's 32 rows meets a new maximum.
    const bool grow = active & ((mloc - m_run) * scale_log2 > 8.f);
    const float m_new = grow ? mloc : m_run;
    const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);  // first visit: factor 0 on zeros
    neg_mc = active ? -m_new * scale_log2 : -INFINITY;  // rows that did not select the chunk: p = 0
    m_run = m_new;
    l_run *= alpha;
    if (!__all(alpha == 1.f)) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto part1 = [&](auto par, int t) {
    constexpr int P = decltype(par)::value;
    uint32_t akn = ldsK + (uint32_t)(((t + 1) & 1) * (int)SM::tile) + rowoff;  // K(t + 1)
    opaque(akn);
    f32x16(&sc)[NKT] = st[P];
    f32x16(&sn)[NKT] = st[P ^ 1];
    uint32_t tv = ldsV + (uint32_t)((t & 1) * (int)SM::tile) + troff;  // V(t)
    opaque(tv);
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) sn[kt][i] = 0.f;
    float lsum = 0.f;
    constexpr int NG = 8 * NKT;  // pairs of scores of a lane
    static_for<NG>([&](auto gi) {
      constexpr int g = decltype(gi)::value;
      constexpr int M0 = g * (NKT * KS) / NG, M1 = (g + 1) * (NKT * KS) / NG;
#pragma unroll
      for (int mi = M0; mi < M1; ++mi) {
        const int kt = mi / KS, ks = mi % KS;
        sn[kt] = mfma32<T>(kf[ks], qb[ks], sn[kt]);
        if (NKT == 2 && kt == 0) kf[ks] = k_frag(akn, 1, ks);  // the operand of the second key tile takes the register over
      }
      constexpr int kte = g / 8, j = g % 8;
      const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[kte][2 * j], scale_log2, neg_mc));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[kte][2 * j + 1], scale_log2, neg_mc));
      lsum += p0 + p1;
      pf[kte][j / 4].w[j % 4] = pack2<T>(p0, p1);
      if (g == NG / 8) s_nx = entry(t + 1);
      if (g == NG / 2) word_nx = sBits[((s_nx >> 16) >> 5) * kRows + wave * 32 + (lane & 31)];
      if (g == NG - 2) {  // V^T operands of the first feature tile
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) vt[kt][s2] = v_frag(tv, 0, kt, s2);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    l_run += lsum;
  };
  auto part2 = [&](int t) {
    uint32_t tv = ldsV + (uint32_t)((t & 1) * (int)SM::tile) + troff;  // V(t)
    opaque(tv);
    static_for<NDT>([&](auto di) {
      constexpr int dt = decltype(di)::value;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          o[dt] = mfma32<T>(vt[kt][s2], pf[kt][s2], o[dt]);
          if (dt + 1 < NDT) vt[kt][s2] = v_frag(tv, dt + 1, kt, s2);  // the operand of the next feature tile takes the register over
        }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  wait_all_loads();  // K(0), K(1), V(0)
  __syncthreads();
  {
    uint32_t ak0 = ldsK + rowoff;
    opaque(ak0);
    s_plain(ak0, st[0]);
  }
  __syncthreads();  // every wave has read K(0): K(2) takes its place
  auto step = [&](auto par, int t) {
    // K(t + 1) and V(t) are in LDS (the wait before the last barrier); the readers of K(t) and V(t - 1) are done
    feed_k(t + 2);
    feed_v(t + 1);
    if (t < nstep) {
      part0(par, t);
      // The wave that has products to issue goes first: an instruction of the other one's loads and masks, which takes an issue slot in front of
      // a product, leaves the matrix cores idle for it, and the other way round costs nothing.  (The two sets of a split workgroup are
      // in step and go the way they went: 34.8 us against 35.1, 3072 tokens, 8 heads of 64.)
      if constexpr (SPLIT == 1) __builtin_amdgcn_s_setprio(1);
      part1(par, t);
      part2(t);
      if constexpr (SPLIT == 1) __builtin_amdgcn_s_setprio(0);
    }
    wait_all_loads();
    __syncthreads();
  };
  for (int t = 0; t < nturn; t += 2) {
    if ((t & 31) == 0) entries_from(t);
    step(C0{}, t);
    if (t + 1 < nturn) step(C1{}, t + 1);
  }
  // (every wave is done with the rings and nothing is in flight: they now hold the sets' sums, then the output tiles)
  float l_tot = l_run;
  constexpr int NP = HD / 2 / NSETS;  // registers of O^T whose features a set takes to the end
  float share[NP];
  if constexpr (NSETS == 1) {
    static_for<NP>([&](auto rc) { share[decltype(rc)::value] = o[decltype(rc)::value / 16][decltype(rc)::value % 16]; });
  } else {
    static_assert(NP % 4 == 0 && (size_t)NSETS * RW * HD * 128 <= SPLIT * SM::ring, "whole groups of features; the sums fit the rings");
    // Sums as [set][wave][HD / 2 registers][64 lanes], m and l behind the lists.  Every set adds up an equal share of the features (the first set alone took 8100
    // clocks for four of them at head dimension 128, 4000 of 64, and all LDS reads).
    auto sums_of = [&](int st) { return reinterpret_cast<float *>(smem) + (size_t)(st * RW + wave) * (HD / 2) * 64 + lane; };
    float *ml = reinterpret_cast<float *>(sBits + nw * kRows + kRowGateChunks) + wave * 128 + lane;  // of set st: RW * 128 st further on
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) sums_of(sid)[(dt * 16 + i) * 64] = o[dt][i];
    ml[sid * RW * 128] = m_run;
    ml[sid * RW * 128 + 64] = l_run;
    __syncthreads();
    float f[NSETS], mn = -INFINITY;
#pragma unroll
    for (int st = 0; st < NSETS; ++st) f[st] = ml[st * RW * 128], mn = fmaxf(mn, f[st]);
    m_run = mn;
    const float mref = mn == -INFINITY ? 0.f : mn;
    l_tot = 0.f;
#pragma unroll
    for (int st = 0; st < NSETS; ++st) {
      f[st] = __builtin_amdgcn_exp2f((f[st] - mref) * scale_log2);
      l_tot += ml[st * RW * 128 + 64] * f[st];
    }
#pragma unroll
    for (int r = 0; r < NP; ++r) {
      share[r] = 0.f;
#pragma unroll
      for (int st = 0; st < NSETS; ++st) share[r] += sums_of(st)[(sid * NP + r) * 64] * f[st];
    }
    __syncthreads();  // (the output tiles lie where the sums did)
  }

  l_tot = sum_xor32_f(l_tot);
  const bool empty = !(l_tot > 0.f);
  const float inv = empty ? 0.f : 1.f / l_tot;
  uint16_t *sOut = reinterpret_cast<uint16_t *>(smem) + (size_t)wave * 32 * LDO;
#pragma unroll
  for (int g = 0; g < NP / 4; ++g)  // (features 2 NP sid .., eight to a group)
    *reinterpret_cast<uint2 *>(sOut + (lane & 31) * LDO + sid * 2 * NP + 8 * g + 4 * hh) =
        make_uint2(pack2<T>(share[4 * g] * inv, share[4 * g + 1] * inv), pack2<T>(share[4 * g + 2] * inv, share[4 * g + 3] * inv));
  if (valid && hh == 0 && sid == 0)
    a.softmax_lse[(int64_t)h * a.total_q + q0 + row] = empty ? INFINITY : (m_run * scale_log2 + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f;
  if constexpr (NSETS > 1)
    __syncthreads();
  else
    wave_lds_fence();
  // rows leave as 16-byte pieces, VPR of them per row, consecutive lanes taking consecutive pieces
#pragma unroll
  for (int v0 = 0; v0 < 32 * VPR; v0 += 64 * NSETS) {
    const int v = v0 + sid * 64 + lane, rl = v / VPR, e = (v - rl * VPR) * 8;
    const int r2 = r0 + wave * 32 + rl;
    if (rl < 32 && r2 < Lq && e < D) {
      const Pack8 x = *reinterpret_cast<const Pack8 *>(sOut + rl * LDO + e);
      *reinterpret_cast<Pack8 *>(reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + r2) * a.o_row_stride + (int64_t)h * a.o_head_stride + e) = x;
    }
  }
}

template <typename T, int HD, int RW, int SPLIT, int KH>
static int launch_rows_split(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, const RowGate *gate, hipStream_t s) {
  typedef FwdRowsDirectSmem<HD, RW, SPLIT> SM;
  auto kern = attn_fwd_rows_kernel<T, HD, RW, SPLIT, KH, false>;
  if constexpr (HD != 96)
    if (gate != nullptr) kern = attn_fwd_rows_kernel<T, HD, RW, SPLIT, KH, true>;
  const int step_cap = ceil_div(a.max_seqlen_k, 64);  // (at most kRowsStepCap: fwd_rows_feasible)
  const size_t smem = SM::bytes(step_cap, nw) + (SPLIT * KH > 1 ? SPLIT * KH * RW * 512 : 0);  // (m and l of the sets)
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_fwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const ItemOrder order = item_order(a.total_q, a.max_seqlen_q, a.batch, a.heads, SM::ROWS, longest_items_first(std::max(a.total_q, a.total_k), a.heads, HD * 4));
  const int64_t items = a.heads * (order == kListedLongestFirst ? listed_blocks(a.total_q, a.batch, SM::ROWS) : (int64_t)a.batch * ceil_div(a.max_seqlen_q, SM::ROWS));
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_fwd: too many (sequence, head, row block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(SPLIT * KH * RW * 64), smem, s, a, bm, nw, step_cap, order, gate != nullptr ? *gate : RowGate{});
  return 0;
}
// Four sets share a walk (head dimensions up to 64) where the workgroups of 64 rows are no more than the compute units, as their rings leave a unit
// room for one (two sets, of which two workgroups fit, take the calls above), and the longest walk is 16 steps or more: four sets take longer to start and to add
// up.  Forward, two sets and four: 2048 tokens, 8 heads (256 workgroups) 31.8 -> 30.2 us, 4096 tokens, 4 heads (256) 49.2 -> 45.3, 400 rows against 6000 keys,
// 8 heads (56) 64.7 -> 56.6, 632 rows against 24924 keys, 8 heads (88) 200 -> 164; 3072 tokens in two sequences, 8 heads (384) 33.8 -> 37.4.  Two sequences, 4
// heads, top-k 3 of 64-key chunks: of 1024 tokens 24.7 -> 24.2, 896 23.5 -> 23.8, 640 21.3 -> 22.5, 128 14.9 -> 16.5.
constexpr int kRowsFourSets = 256, kRowsFourSetsKeys = 1024;
// Which workgroup, by the 128-row blocks of the call and the mean length of its sequences:
// - two waves of 32 rows and two sets of them where 128-row blocks come to about one per compute unit (two at head dimensions up
//   to 64, where two such workgroups fit a unit): the walks are half as long and there are twice as many of them.  Against one
//   set of four waves (two sets of four, which served half of these calls before, lie between): heads of 64, 2048 tokens, 16 heads
//   38.4 -> 26.0 us, 4096 tokens 76 -> 66, 8192 tokens 206 -> 214 (beyond the line), c1 of two sequences, 8 heads 37 -> 25; heads of
//   128, 2048 tokens, 16 heads 50 -> 43, 2500 tokens 63 -> 66.
// - two waves and one set at head dimensions up to 64 for short sequences, whose workgroups spend half of their time on the way
//   to the first step: 64 rows are less padding and twice as many workgroups wait side by side.  8191 tokens of documents of 341
//   on average 34.8 -> 31.2 us, of 540 50 -> 43, of 1483 93.3 -> 89.7; one sequence of 8192 tokens 206 -> 206, 16384 765 -> 811.  (At
//   head dimension 128 the rings leave room for two workgroups of either kind, and the small ones have half of the waves: 73 -> 99.)
// - four waves and one set otherwise.
static int rows_sets(const fmoba_attn_fwd_args &a) {
  if (a.head_dim <= 64 && a.max_seqlen_k >= kRowsFourSetsKeys && a.heads * (((int64_t)a.total_q + 63 * a.batch) / 64) <= kRowsFourSets) return 4;
  return (int64_t)a.heads * (a.total_q / 128 + a.batch) <= (a.head_dim > 64 ? 288 : 544) ? 2 : 1;
}
// Two sets of waves whose tiles are shared by two waves each, which take a half of their keys (eight waves, the loads and the rings of four): half of a turn's arithmetic in front of a
// barrier.  Above head dimension 64, where the rings of two sets leave a unit room for one workgroup anyway, from sequences of 1024 keys on (shorter walks lose
// in the sums what they gain: heads of 128, two sequences of 128 tokens 13.9 -> 14.9 us, four of 512 19.7 -> 20.0).  The pass alone: 2048 tokens, 8 heads of 128 33.8 -> 32.1 us, not causal 33.9 ->
// 31.3, 16 heads 45.4 -> 43.9, 4096 tokens, 8 heads 75.1 -> 70.3, 3495 tokens, 8 heads of 96 45.3 -> 41.3, 3 x 1024 tokens, 8 heads of 128 28.3 -> 28.6, not causal 38.0 -> 36.2.
// Up to 64 a unit holds one such workgroup where it holds two of four waves, and what is more than there are units starts when the first are done.  That is no loss where the longest walk
// covers it, in causal calls whose items start longest first and whose heads fill the turns of the XCDs (each XCD has its share of every sequence).  A workgroup costs its walk and what ten to
// fourteen blocks of 64 keys take (start, choice, list, sums); if the sequences are about alike, the `later` workgroups are the rows' first `later` / (heads * batch) blocks, which start when walks
// of that length are done.  Workgroups that find no block count (a grid for the longest sequence has some in the others).  Calls of heads of 64, us, without and with: 1024 + 2048 tokens,
// 8 heads 27.7 and 26.6, 1700 + 900 25.5 and 24.3, 2500 + 500 31.2 and 29.5, 3000 35.3 and 33.9, 1100, 16 heads 21.0 and 20.2; refused: 2 x 1536, 8 heads 24.5 and 26.3, 3 x 1024 20.7 and
// 23.7, 1112 + 1512 25.6 and 28.3, 1400, 16 heads 23.5 and 24.0, 2 x 1200, 8 heads 22.3 and 21.9, 24 heads of 1024 21.0 and 24.1, four sequences of 407 to 2641, 4 heads 35.1 and 51.8, not causal
// (the pass alone) 1100, 16 heads 20.1 and 27.5, 1024 + 2048, 8 heads 29.9 and 39.6.  Beyond 400 workgroups of uneven sequences: 3000 + 600, 8 heads 35.9 and 37.7, 3500 + 300 + 200 39.1 and 42.8.
constexpr int kRowsHalves = 400, kRowsHalvesCost = 14;
static bool rows_halves(const fmoba_attn_fwd_args &a) {
  if (a.max_seqlen_k < kRowsFourSetsKeys) return false;
  if (a.head_dim > 64) return true;
  if (!a.is_causal || a.total_q != a.total_k || a.max_seqlen_q != a.max_seqlen_k || a.heads % 8 != 0) return false;
  const int nb = ceil_div(a.max_seqlen_q, 64);
  const bool listed = item_order(a.total_q, a.max_seqlen_q, a.batch, a.heads, 64, true) == kListedLongestFirst;
  const int64_t items = a.heads * (listed ? ((int64_t)a.total_q + 63 * a.batch) / 64 : (int64_t)a.batch * nb);
  return items <= kRowsHalves && 2 * (items - kRowsFourSets) <= (int64_t)(nb - kRowsHalvesCost) * a.heads * a.batch;
}
template <typename T, int HD>
static int launch_rows(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, hipStream_t s, const RowGate *gate = nullptr) {
  const int sets = rows_sets(a);
  if constexpr (HD <= 64)
    if (sets == 4) return launch_rows_split<T, HD, 2, 4, 1>(a, bm, nw, gate, s);
  if (sets == 2) return rows_halves(a) ? launch_rows_split<T, HD, 2, 2, 2>(a, bm, nw, gate, s) : launch_rows_split<T, HD, 2, 2, 1>(a, bm, nw, gate, s);
  if constexpr (HD <= 64)
    if (a.total_q <= (int64_t)1536 * a.batch) return launch_rows_split<T, HD, 2, 1, 1>(a, bm, nw, gate, s);
  return launch_rows_split<T, HD, 4, 1, 1>(a, bm, nw, gate, s);
}

template <typename T, int HD>
static int launch_rows_loader(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, hipStream_t s) {
  auto kern = attn_fwd_rows_loader_kernel<T, HD>;
  const size_t smem = FwdRowsSmem<HD>::bytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_fwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const int64_t items = (int64_t)a.batch * a.heads * ceil_div(a.max_seqlen_q, 128);
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_fwd: too many (sequence, head, row block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(512), smem, s, a, bm, nw);
  return 0;
}

// head dimensions above 128 (attn_fwd_rows_wide.hip)
int launch_rows_wide(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, const RowGate *gate, hipStream_t s);
// a call with a handful of rows (attn_fwd_few.hip)
bool fwd_few_rows(const fmoba_attn_fwd_args &a);
void run_fwd_few(const fmoba_attn_fwd_args &a, const uint32_t *bm, int nw, hipStream_t s);

bool fwd_rows_feasible(const fmoba_attn_fwd_args &a) {
  return a.head_dim <= 256 && ceil_div(a.max_cols, 32) <= kRowsWordCap && ceil_div(a.max_seqlen_k, 64) <= kRowsStepCap &&
         a.max_cols < 32768 && a.lg_block_n % 64 == 0;
}

// The kernels without loader waves: the rows' selection words fit the workgroup's LDS (512 chunks per sequence), the rows of a tile lie within 32-bit
// byte offsets of its first key.
bool fwd_rows_direct(const fmoba_attn_fwd_args &a) {
  return ceil_div(a.max_cols, 32) <= kRowsWords && a.k_row_stride < ((int64_t)1 << 24) && a.v_row_stride < ((int64_t)1 << 24);
}

size_t fwd_rows_workspace_bytes(const fmoba_attn_fwd_args &a) {
  if (a.selection_bits != nullptr) return 256;
  const size_t rows = (size_t)a.total_q * a.heads;
  return ((rows * (size_t)ceil_div(a.max_cols, 32) * 4 + 255) & ~(size_t)255) + 256;
}

// Calls whose rows can choose their chunks in attn_fwd_rows_kernel: the scores of a row are two tiles of products with the operands that Q already is; calls of
// a few rows have a gate of their own.  Heads of 72 to 96 keep the launch of the gate: in their tiles the operands' pieces lie in another order
// (tile_frag_piece<96>), which gate_select has no instance for.
bool fwd_rows_gated(const fmoba_attn_fwd_args &a) {
  return a.max_cols <= kRowGateChunks && a.max_seqlen_q > kFewRows && !fwd_few_rows(a) && fwd_rows_direct(a) &&
         (a.head_dim <= 64 || a.head_dim > 96);
}
int run_fwd_rows_gated(const fmoba_attn_fwd_args &a, const RowGate &gate, hipStream_t s) {
  const int nw = ceil_div(a.max_cols, 32);
  const bool bf = a.dtype == FMOBA_DTYPE_BF16;
  if (a.head_dim <= 64) return bf ? launch_rows<bf16_t, 64>(a, nullptr, nw, s, &gate) : launch_rows<f16_t, 64>(a, nullptr, nw, s, &gate);
  if (a.head_dim > 128) return launch_rows_wide(a, nullptr, nw, &gate, s);
  return bf ? launch_rows<bf16_t, 128>(a, nullptr, nw, s, &gate) : launch_rows<f16_t, 128>(a, nullptr, nw, s, &gate);
}

// bitmap build (phase 1) + the row-block pass (phase 2)
int run_fwd_rows(const fmoba_attn_fwd_args &a, int phases, hipStream_t s) {
  const int nw = ceil_div(a.max_cols, 32);
  const int64_t rows = (int64_t)a.total_q * a.heads;
  const uint32_t *bm = a.selection_bits;
  if (bm == nullptr) {
    uint32_t *own = reinterpret_cast<uint32_t *>(((uintptr_t)a.workspace + 255) & ~(uintptr_t)255);
    bm = own;
    if (phases & 1) {
      const size_t smem = (size_t)a.max_seqlen_q * 4;
      if (a.max_seqlen_q <= kBitmapRows &&
          (smem <= 32 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(csc_bitmap_lds_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess)) {
        hipLaunchKernelGGL(csc_bitmap_lds_kernel, dim3(nw, a.heads, a.batch), dim3(a.max_seqlen_q > 64 ? 1024 : 256), smem, s, a, own, nw);
      } else {
        hipLaunchKernelGGL(fwd_zero_u32_kernel, dim3(512), dim3(256), 0, s, own, rows * nw);
        hipLaunchKernelGGL(csc_bitmap_kernel, dim3(a.max_cols, a.heads, a.batch), dim3(256), 0, s, a, own, nw);
      }
    }
  }
  if ((phases & 2) && fwd_few_rows(a)) {
    run_fwd_few(a, bm, nw, s);
    return 0;
  }
  if (phases & 2) {
    const bool bf = a.dtype == FMOBA_DTYPE_BF16;
    int rc;
    const bool direct = fwd_rows_direct(a);
    if (a.head_dim <= 64)
      rc = direct ? (bf ? launch_rows<bf16_t, 64>(a, bm, nw, s) : launch_rows<f16_t, 64>(a, bm, nw, s))
                 : (bf ? launch_rows_loader<bf16_t, 64>(a, bm, nw, s) : launch_rows_loader<f16_t, 64>(a, bm, nw, s));
    else if (direct && a.head_dim <= 96)
      rc = bf ? launch_rows<bf16_t, 96>(a, bm, nw, s) : launch_rows<f16_t, 96>(a, bm, nw, s);
    else if (a.head_dim <= 128)
      rc = direct ? (bf ? launch_rows<bf16_t, 128>(a, bm, nw, s) : launch_rows<f16_t, 128>(a, bm, nw, s))
                 : (bf ? launch_rows_loader<bf16_t, 128>(a, bm, nw, s) : launch_rows_loader<f16_t, 128>(a, bm, nw, s));
    else
      rc = direct ? launch_rows_wide(a, bm, nw, nullptr, s) : (bf ? launch_rows_loader<bf16_t, 256>(a, bm, nw, s) : launch_rows_loader<f16_t, 256>(a, bm, nw, s));
    if (rc) return rc;
  }
  return 0;
}

}  // namespace fmoba

extern "C" int32_t fmoba_attn_fwd_row_sets(const fmoba_attn_fwd_args *a) { return a != nullptr && a->head_dim > 0 && a->head_dim <= 128 && fmoba::fwd_rows_direct(*a) ? fmoba::rows_sets(*a) : 1; }
extern "C" int32_t fmoba_attn_fwd_key_halves(const fmoba_attn_fwd_args *a) { return fmoba_attn_fwd_row_sets(a) == 2 && fmoba::rows_halves(*a) ? 1 : 0; }
