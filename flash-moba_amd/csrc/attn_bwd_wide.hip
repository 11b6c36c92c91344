// dK / dV and the dS tiles of the row-block dQ pass for head dimensions above 128, up to 256.
//
// The column-stationary scheme of attn_bwd_dkdv_kernel -- one workgroup per (64-key block, head, sequence) walks the
// block's ascending row list: S = Q K^T, dP = dO V^T, P = exp2(S*scale*log2e - LSE*log2e), dS = P o (dP - delta),
// dV^T += dO^T P, dK^T += Q^T dS -- cut so that a wave fits 256 registers and two waves share a SIMD.  dK^T and dV^T of 64
// keys x 256 features are 512 accumulator registers of one wave; here eight waves hold 64 each (a quarter of the
// features, all keys, of one of the two), and the four (key half, row half) tiles of S and the four of dP are one wave's
// each, with K resp. V of its key half in registers.  A round takes 64 gathered rows, which loads bring straight into LDS one
// round ahead; dP - delta goes to the wave that holds S of the same tile through LDS (fp32), P and dS to everybody (16 bits).
// 2 x 4096 tokens, 8 heads of 256, 8 of 128-key chunks: 1223 us with one 32-row tile at a time between two barriers and
// K and V as LDS operands, 235 us now.  What bounds it: one operand from LDS per product, and the two exchanges.
#include "fmoba_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace fmoba {

struct BwdWideSmem {
  static constexpr int HD = 256;
  static constexpr size_t tile = (size_t)64 * HD * 2;  // 64 gathered rows of Q or dO, swizzled (tile_swz)
  static constexpr size_t oQ = 0;                       // [2 buffers]
  static constexpr size_t odO = oQ + 2 * tile;          // [2 buffers]
  static constexpr size_t oP = odO + 2 * tile;          // [64 rows][64 keys], piece p (8 keys) of row r at p ^ (r & 7)
  static constexpr size_t odS = oP + 64 * 128;
  static constexpr size_t oX = odS + 64 * 128;          // dP - delta of the four tiles: [tile][4][64 lanes][4] fp32
  static constexpr size_t bytes = oX + 4 * 4096;
  static constexpr int LDR = HD + 4;                    // floats, output staging [64 keys][LDR], dV then dK
  static_assert(2 * (size_t)64 * LDR * 4 <= bytes, "the output staging reuses the tiles");
  static_assert(bytes <= 160 * 1024, "LDS of one compute unit");
};

// NEAR: as in attn_bwd_dkdv_kernel (attn_bwd.hip)
template <typename T, bool NEAR>
__global__ __launch_bounds__(512, 2) void attn_bwd_dkdv_wide_kernel(fmoba_attn_bwd_args a, uint16_t *ds_ws, int row_mask, ItemOrder order) {
  typedef BwdWideSmem SM;
  constexpr int HD = SM::HD, KS = HD / 16, VPR = HD / 8, RB = HD * 2, LDR = SM::LDR;
  constexpr float kLog2e = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  int nb, b, h;
  if (order == kListedLongestFirst) {
    const BlockItem item = listed_item<64, false>(blockIdx.x, a.batch, a.heads, a.max_seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k);
    if (item.b < 0) return;
    nb = item.idx, b = item.b, h = item.h;
  } else {
    const PairItem item = xcd_pair_item(blockIdx.x, a.batch * a.heads, (a.max_seqlen_k + 63) / 64, false, order == kLongestFirst);
    nb = item.idx, b = item.pair / a.heads, h = item.pair - b * a.heads;
  }
  const int key0 = nb * 64;
  const int Bn = a.lg_block_n, c = key0 / Bn;
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
  const int D = a.head_dim;
  const int hk = h / (a.heads / a.heads_k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hh = lane >> 5;
  const int rt = wave & 1, kq = (wave >> 1) & 1, is_s = wave >> 2;  // S (waves 4..7) or dP (0..3) of this wave's 32 rows and 32 keys
  const int fw = wave & 3, is_k = wave >> 2;                        // sums: dV (0..3) or dK (4..7), features 64 fw ..
  const bool causal = a.is_causal != 0;
  const float scale_log2 = a.softmax_scale * kLog2e;
  const uint32_t lds = (uint32_t)(uintptr_t)smem, ldsQ = lds + (uint32_t)SM::oQ, ldsdO = lds + (uint32_t)SM::odO, ldsP = lds + (uint32_t)SM::oP, ldsdS = lds + (uint32_t)SM::odS;
  const uint32_t ldsX = lds + (uint32_t)(SM::oX + (wave & 3) * 4096 + lane * 16);
  constexpr uint32_t TILE = (uint32_t)SM::tile;
  constexpr int RPI = 64 / VPR;  // tile rows per load instruction
  const int rl = lane / VPR, pc = lane % VPR;

  // K and V of the block pass through the tiles on their way to registers
  {
    const uint16_t *kg = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)(k0 + key0) * a.k_row_stride + (int64_t)hk * a.k_head_stride;
    const uint16_t *vg = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)(k0 + key0) * a.v_row_stride + (int64_t)hk * a.v_head_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = (wave * 4 + i) * RPI + rl;
      const int e = min((pc ^ tile_swz<HD>(key)) * 8, D - 8);
      const int64_t kc = min(key, Lk - 1 - key0);
      global_to_lds16(kg + kc * a.k_row_stride + e, ldsQ + (uint32_t)((wave * 4 + i) * 1024));
      global_to_lds16(vg + kc * a.v_row_stride + e, ldsdO + (uint32_t)((wave * 4 + i) * 1024));
    }
  }
  int start = 0;
  if (causal && nnz > 0 && Bn > 64) start = __builtin_amdgcn_readfirstlane(lower_bound_wave_i32(a.row_indices + lbase, nnz, key0 - off, row_mask));  // earlier rows see no key of the block
  const int32_t *list = a.row_indices + lbase + start;
  const int n = nnz - start;
  const int nround = (n + 63) >> 6;
  const int koff = key0 - c * Bn;  // offset of the block inside its column

  const uint16_t *qg = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)q0 * a.q_row_stride + (int64_t)h * a.q_head_stride;
  const uint16_t *dog = reinterpret_cast<const uint16_t *>(a.dout) + (int64_t)q0 * a.do_row_stride + (int64_t)h * a.do_head_stride;
  // the per-row scalar of this wave's part: LSE for S, delta for dP
  const float *sclg = is_s ? a.softmax_lse + (int64_t)h * a.total_q + q0 : a.softmax_d + (int64_t)h * ((int64_t)a.total_q + 128 * (int64_t)a.batch) + q0 + 128 * b;

  f32x16 acc[2][2];  // register i of tile [d][kk] <-> feature 64 fw + 32 d + acc_row(i, hh), key 32 kk + lane % 32
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[d][kk][i] = 0.f;

  const int myrow = rt * 32 + (lane & 31);  // this lane's row of a round
  int rid_nx = nround > 0 ? list[min(myrow, n - 1)] : 0;
  const uint32_t rowoff = (uint32_t)((lane & 31) * RB + (((hh * KS) ^ tile_swz<HD>(lane & 31)) * 16));
  const int li = lane & 15, r0t = (li >> 2) + 4 * hh;
  const uint32_t troff = (uint32_t)(r0t * RB + ((((((lane >> 4) & 1) * 2 + ((li & 3) >> 1))) ^ tile_swz<HD>(r0t)) * 16) + (li & 1) * 8);
  wait_all_loads();
  __syncthreads();
  Pack8 kf[KS];  // K or V of this wave's keys, the A operand
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    kf[ks] = lds_read16(((is_s ? ldsQ : ldsdO) + (uint32_t)(kq * 32 * RB) + rowoff) ^ (uint32_t)(ks * 16));
    if (D < HD && (hh * KS + ks) * 8 >= D) kf[ks] = zero_pack8();
  }
  __syncthreads();
  if (nround > 0) {
    auto code = [&](int raw, int r) { return tile_row_code(raw & row_mask, r * 64 + myrow < n, Lq); };
    uint32_t fsrc[4];  // the rows this lane fetches pieces of: eight per wave, of its own 32
    auto feed_rows = [&](int rid) {  // (all exchanges at once: one wait for them)
#pragma unroll
      for (int i = 0; i < 4; ++i) fsrc[i] = (uint32_t)__shfl(rid, (wave >> 1) * 8 + i * RPI + rl, 64);
    };
    auto feed = [&](auto ic, uint32_t buf) {  // load ic of Q and of dO
      constexpr int I = decltype(ic)::value;
      const int tr = (wave >> 1) * 8 + I * RPI + rl;
      const uint32_t src = fsrc[I] & 0x7fffffffu;
      const uint32_t e = (uint32_t)min((pc ^ tile_swz<HD>(tr)) * 8, D - 8);
      const uint32_t dst = buf + (uint32_t)((rt * 32 + (wave >> 1) * 8 + I * RPI) * RB);
      if constexpr (NEAR) {
        global_to_lds16_sbase(mul24_u32(src, (uint32_t)a.q_row_stride * 2u) + e * 2u, qg, ldsQ + dst);
        global_to_lds16_sbase(mul24_u32(src, (uint32_t)a.do_row_stride * 2u) + e * 2u, dog, ldsdO + dst);
      } else {
        global_to_lds16(qg + ((uint64_t)src * (uint32_t)a.q_row_stride + e), ldsQ + dst);
        global_to_lds16(dog + ((uint64_t)src * (uint32_t)a.do_row_stride + e), ldsdO + dst);
      }
    };
    int rid = code(rid_nx, 0);
    feed_rows(rid);
    static_for<4>([&](auto ic) { feed(ic, 0u); });
    float scl = sclg[rid & 0x7fffffff];
    rid_nx = list[min(64 + myrow, n - 1)];
    auto arrived = [&]() {
      wait_all_loads();
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("" : "+v"(scl), "+v"(rid_nx));
#endif
    };
    arrived();
    __syncthreads();
    const uint32_t pw = (uint32_t)(myrow * 128 + hh * 8), psw = (uint32_t)(myrow & 7);
    const uint32_t ptr0 = (is_k ? ldsdS : ldsP) + (uint32_t)(r0t * 128 + (((((lane >> 4) & 1) * 2 + ((li & 3) >> 1)) ^ (r0t & 7)) * 16) + (li & 1) * 8);
    for (int r = 0; r < nround; ++r) {
      const uint32_t buf = (r & 1) ? TILE : 0u;
      const int rcur = rid;
      const float x0 = is_s ? (rcur >= 0 ? scl * kLog2e : INFINITY) : scl;
      rid = code(rid_nx, r + 1);
      // (the rows by 32-bit offsets and between the products, as in attn_bwd_dkdv_kernel: 2 x 4096 tokens, 8 heads of 256, training step 506 -> 487 us)
      feed_rows(rid);
      scl = sclg[rid & 0x7fffffff];
      rid_nx = list[min((r + 2) * 64 + myrow, n - 1)];
      // S^T or dP^T: lane -> row, register i -> key 32 kq + acc_row(i, hh)
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
      const uint32_t aq = (is_s ? ldsQ : ldsdO) + buf + (uint32_t)(rt * 32 * RB) + rowoff;
      constexpr int NB = 4;  // k-steps per batch of reads
      Pack8 qf[2][NB];
      auto rd = [&](auto bc) {
        constexpr int B = decltype(bc)::value;
#pragma unroll
        for (int u = 0; u < NB; ++u) qf[B & 1][u] = lds_read16(aq ^ (uint32_t)((B * NB + u) * 16));
      };
      rd(std::integral_constant<int, 0>{});
      static_for<KS / NB>([&](auto bc) {
        constexpr int B = decltype(bc)::value;
        if constexpr (B + 1 < KS / NB) rd(std::integral_constant<int, B + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < NB; ++u) s = mfma32<T>(kf[B * NB + u], qf[B & 1][u], s);
        static_assert(KS / NB == 4, "a load of Q and one of dO after every batch of products");
        if (r + 1 < nround) feed(bc, buf ^ TILE);
        __builtin_amdgcn_sched_barrier(0);
      });
      const uint32_t at = pw + ((uint32_t)(kq * 4) ^ psw) * 16u;
      if (is_s) {
        const int lim = rcur < 0 ? -1 : min(causal ? rcur + off : 0x7fffffff, Lk - 1) - key0 - kq * 32;  // last visible key of this wave's 32
        if (!__all(lim >= 31)) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + (i & 3) + 4 * hh <= lim ? s[i] : -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], scale_log2, -x0));
#pragma unroll
        for (int g = 0; g < 4; ++g)
          lds_write_vec<uint2>(ldsP + (at ^ (uint32_t)(g * 16)), make_uint2(pack2<T>(s[4 * g], s[4 * g + 1]), pack2<T>(s[4 * g + 2], s[4 * g + 3])));
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          lds_write_vec<f32x4>(ldsX + (uint32_t)(g * 1024), f32x4{s[4 * g] - x0, s[4 * g + 1] - x0, s[4 * g + 2] - x0, s[4 * g + 3] - x0});
      }
      __syncthreads();  // dP - delta is there
      if (is_s) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 x = lds_read_vec<f32x4>(ldsX + (uint32_t)(g * 1024));
          lds_write_vec<uint2>(ldsdS + (at ^ (uint32_t)(g * 16)),
                               make_uint2(pack2<T>(s[4 * g] * x[0], s[4 * g + 1] * x[1]), pack2<T>(s[4 * g + 2] * x[2], s[4 * g + 3] * x[3])));
        }
      }
      __syncthreads();  // P and dS of the round are there
      // dV^T[f][key] += dO^T[f][row] P[row][key] or dK^T[f][key] += Q^T[f][row] dS[row][key]
      const uint32_t tx = (is_k ? ldsQ : ldsdO) + buf + troff;
      Pack8 pb[2][2], xa[2][2];
      auto rd2 = [&](auto sc) {
        constexpr int S4 = decltype(sc)::value;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const uint32_t po = (ptr0 ^ (uint32_t)(kk * 64)) + (uint32_t)(S4 * 16 * 128);
          pb[S4 & 1][kk] = lds_tr8(po, po + 8 * 128);
        }
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const uint32_t dt = (uint32_t)(fw * 2 + d), xlo = dt * 64u, xhi = ((dt * 4u) ^ (uint32_t)TileSwz<HD>::kRow8) * 16u;
          const uint32_t olo = (uint32_t)(S4 * 16 * RB), ohi = olo + (uint32_t)(8 * RB);
          xa[S4 & 1][d] = lds_tr8((tx ^ xlo) + olo, (tx ^ xhi) + ohi);
        }
      };
      rd2(std::integral_constant<int, 0>{});
      static_for<4>([&](auto sc) {
        constexpr int S4 = decltype(sc)::value;
        if constexpr (S4 < 3) rd2(std::integral_constant<int, S4 + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) acc[d][kk] = mfma32<T>(xa[S4 & 1][d], pb[S4 & 1][kk], acc[d][kk]);
        __builtin_amdgcn_sched_barrier(0);
      });
      // dS of row `lane`, key group `wave`: consecutive lanes write consecutive pieces of the dS tile
      {
        const Pack8 x = lds_read16(ldsdS + (uint32_t)(lane * 128) + (((uint32_t)wave ^ (uint32_t)(lane & 7)) * 16u));
        arrived();
        if (r * 64 + lane < n) *reinterpret_cast<Pack8 *>(ds_piece(ds_ws, lbase + start + r * 64, lane, (koff >> 3) + wave, Bn >> 3)) = x;
      }
      __syncthreads();  // the next round's rows are in LDS, this one's are no longer read
    }
  }

  // ---- dK^T / dV^T leave as rows, once ----
  float *red = reinterpret_cast<float *>(smem);  // [dV, dK][64 keys][LDR]
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4 *>(red + (size_t)(is_k * 64 + kk * 32 + (lane & 31)) * LDR + fw * 64 + d * 32 + 8 * g + 4 * hh) =
            f32x4{acc[d][kk][4 * g], acc[d][kk][4 * g + 1], acc[d][kk][4 * g + 2], acc[d][kk][4 * g + 3]};
  __syncthreads();
  uint16_t *dkg = reinterpret_cast<uint16_t *>(a.dk) + (int64_t)(k0 + key0) * a.dk_row_stride + (int64_t)h * a.dk_head_stride;
  uint16_t *dvg = reinterpret_cast<uint16_t *>(a.dv) + (int64_t)(k0 + key0) * a.dv_row_stride + (int64_t)h * a.dv_head_stride;
  for (int v = tid; v < 64 * VPR; v += 512) {
    const int key = v / VPR, e = (v - key * VPR) * 8;
    if (key0 + key >= Lk || e >= D) continue;
    const float *s0 = red + (size_t)key * LDR + e, *s1 = s0 + 64 * LDR;
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

template <typename T>
static int launch_dkdv_wide(const fmoba_attn_bwd_args &a, uint16_t *ds_ws, int row_mask, hipStream_t s) {
  auto kern = rows_near(a) ? attn_bwd_dkdv_wide_kernel<T, true> : attn_bwd_dkdv_wide_kernel<T, false>;
  const size_t smem = BwdWideSmem::bytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    set_error("attn_bwd: cannot reserve %zu bytes of LDS", smem);
    return 2;
  }
  const ItemOrder order = item_order(a.total_k, a.max_seqlen_k, a.batch, a.heads, 64, longest_items_first(std::max(a.total_q, a.total_k), a.heads, 1024));
  const int64_t items = a.heads * (order == kListedLongestFirst ? listed_blocks(a.total_k, a.batch, 64) : (int64_t)a.batch * ceil_div(a.max_seqlen_k, 64));
  if (items >= ((int64_t)1 << 31)) {
    set_error("attn_bwd: too many (sequence, head, key block) work items");
    return 1;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(512), smem, s, a, ds_ws, row_mask, order);
  return 0;
}

// dK / dV and the dS tiles for head dimensions above 128 (ds_ws: the dS workspace, laid out by ds_piece_offset)
int run_bwd_dkdv_wide(const fmoba_attn_bwd_args &a, uint16_t *ds_ws, int row_mask, hipStream_t s) {
  return a.dtype == FMOBA_DTYPE_BF16 ? launch_dkdv_wide<bf16_t>(a, ds_ws, row_mask, s) : launch_dkdv_wide<f16_t>(a, ds_ws, row_mask, s);
}

}  // namespace fmoba
