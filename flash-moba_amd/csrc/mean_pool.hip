// Per-chunk key mean-pool: km[c] = mean(K[c*B : (c+1)*B]) per (sequence, kv head).
// Pure streaming kernel: every 16-byte vector of K is read exactly once, coalesced along
// the (head, dim) axis, accumulated in fp32 and written once.
#include "fmoba_common.h"

namespace fmoba {

// What the first launch of the gated path does besides the pooling, so that it need not be a launch of its own (about
// five microseconds each on the device, and as much on the host): offsets of the pooled sequences, and counters of the
// gating that have to be zero.
struct PoolExtra {
  int32_t *cu_km;   // null: the offsets are an input (a.cu_seqlens_km)
  int32_t *clear;   // 16-byte aligned, clear_vec16 pieces of 16 bytes
  int64_t clear_vec16;
};

// grid (max_chunks, batch, ceil(vecs / 64)), block 256 = 4 waves.
// A wave owns 64 consecutive 16-byte vectors of the (heads_k*head_dim) axis; the four
// waves of the block split the rows of the chunk and reduce through LDS.
// HD > 0 (head_dim padded to 64, 128 or 256; blocks of whole heads): the means go nowhere, the block scores the sequence's few query rows with
// them while it has them.  Each wave takes key heads of the block; the query rows of a group's heads are the columns of one product (the one
// of topk_gate_few_kernel: the same scores to the last bit).  What it costs hides under the other blocks' loads, the gate is no launch any more, and the
// chunk of a lone row's own keys is not read.  Decode of 16 requests against 512 to 32768 keys, 32 over 8 heads of 128, top-k 8 of 128-key chunks 119 -> 106 us;
// one request of 3000 keys 21.3 -> 16.6, of 60000 48.5 -> 36.5; 20 of 256 to 65536, 32 over 32 heads 740 -> 694.  Heads of 256 too, though the query rows leave
// three waves per SIMD of eight: one request of 60000 keys, 8 heads 81.9 -> 62.4, eight of 1000 to 30000, 32 over 4 heads 61.4 -> 56.2, 32 of 512 to 32768, 32
// heads 907 -> 878.
// Keys that the chip's last cache (256 MB) cannot hold until the attention comes to them are read past the caches.  The pass alone, through them and past them: plain, 32 heads of 128, 160 MB of keys
// 39.9 and 33.1 us, 224 MB 55.4 and 40.8, 256 MB 62.2 and 45.4, 400 MB 99 and 71; with scores, 16 requests, 8 key heads of 128, 160 MB 30.5 and 29.0, 256 MB 45.9 and 43.9, 400 MB 70.4 and 65.8.
// Keys that it holds are read again from there: 67485 keys, 16 heads of 96 (207 MB) 40.7 us, past the caches 44.6, and the decode step after it 30.6 and 35.7.
constexpr int64_t kPoolStreamBytes = (int64_t)256 << 20;
// STREAM: with scores, read past the caches, known at the launch.  Plain pooling, whose arguments do not say how many keys there are: found out from the offsets; calls that are below the line
// even if every sequence is as long as the longest take the instance without (a third offset and a second loop: 8192 tokens, 16 heads of 128 7.4 -> 7.8 us, of 64 5.1 -> 5.5, 3072 tokens, 8 heads
// 5.1 -> 5.4, 24571 tokens, 8 heads 11.8 -> 12.1).
template <typename T, bool MANY, int HD, bool STREAM>
__global__ __launch_bounds__(256) void mean_pool_kernel(fmoba_mean_pool_args a, PoolExtra x, FewGate few) {
  const int c = blockIdx.x, b = blockIdx.y;
  const int seq_start = a.cu_seqlens_k[b], seq_end = a.cu_seqlens_k[b + 1];
  int total_k = 0;
  if constexpr (HD == 0 && STREAM) {
    total_k = a.cu_seqlens_k[a.batch];
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(total_k));  // awaited with the other two, not in front of the rows
#endif
  }
  const int row0 = seq_start + c * a.chunk;
  if (x.clear_vec16) {
    const int64_t nthr = (int64_t)gridDim.x * gridDim.y * gridDim.z * 256;
    int64_t i = (((int64_t)blockIdx.z * gridDim.y + b) * gridDim.x + c) * 256 + threadIdx.x;
    for (; i < x.clear_vec16; i += nthr) *reinterpret_cast<Pack8 *>(x.clear + 4 * i) = zero_pack8();
  }
  // first pooled row of the sequence: the chunks of the sequences before it, counted by the wave that writes the row
  const bool offsets = x.cu_km != nullptr;
  const bool tells = offsets && c == 0 && blockIdx.z == 0;
  int before = 0;
  if (offsets && threadIdx.x < 64 && (tells || row0 < seq_end)) {
    for (int i = threadIdx.x; i < b; i += 64) before += (a.cu_seqlens_k[i + 1] - a.cu_seqlens_k[i] + a.chunk - 1) / a.chunk;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o, 64);
    if (tells && threadIdx.x == 0) {
      x.cu_km[b] = before;
      if (b == a.batch - 1) x.cu_km[a.batch] = before + (seq_end - seq_start + a.chunk - 1) / a.chunk;
    }
  }
  if (row0 >= seq_end) return;
  int few_q0 = 0, few_rows = 0;
  if constexpr (HD > 0) {  // the chunks that are candidates of the last row (with the causal rule those before its own)
    few_q0 = few.cu_seqlens_q[b];
    const int lq = few.cu_seqlens_q[b + 1] - few_q0;
    few_rows = min(lq, few.rows);
    const int rmax = few_rows - 1 + (seq_end - seq_start) - lq;
    if (few_rows <= 0 || (few.is_causal && (rmax < 0 || c >= rmax / a.chunk))) return;
  }
  const int n = min(a.chunk, seq_end - row0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int vecs_per_head = a.head_dim >> 3;
  const int nvec = a.heads_k * vecs_per_head;
  const int block_heads = HD > 0 ? few.block_heads : 0;
  const int vec = HD > 0 ? blockIdx.z * block_heads * vecs_per_head + lane : blockIdx.z * 64 + lane;
  const bool active = vec < nvec && (HD == 0 || lane < block_heads * vecs_per_head);
  const int head = active ? vec / vecs_per_head : 0;
  const int d0 = active ? (vec - head * vecs_per_head) * 8 : 0;

  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  if (active) {
    const uint16_t *base = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)head * a.k_head_stride + d0;
    auto sum_rows = [&](auto stream) {
      auto load = [](const uint16_t *p) { return decltype(stream)::value ? ld_stream16(p) : ld_global16(p); };
      int r = wave;  // row of the chunk
      // Sixteen independent 16-byte loads in flight per lane, added up in the order of the loop of four below: with four, a chunk of 256 rows is
      // sixteen memory latencies one after the other.  For rows of up to 2 KB (forward of 3334 tokens, 8 heads, 256-key chunks 65.8 -> 62.0 us, decode of
      // 43 sequences of up to 59161 keys, 2 key heads of 64 102.9 -> 95.5, of 16 sequences, 8 key heads of 128 119.2 -> 118.6, 3072 tokens, 8 heads of 64, 128-key
      // chunks 34.2 -> 33.5); wider rows read fewer pages of memory at a time with four (decode of 8 sequences of 30000 keys, 32 key heads, 256-key
      // chunks 370 us, 392 with sixteen), and chunks of 64 rows gain nothing.
      for (; MANY && r + 60 < n; r += 64) {
        Pack8 p[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) p[j] = load(base + (int64_t)(row0 + r + 4 * j) * a.k_row_stride);
#pragma unroll
        for (int j = 0; j < 16; j += 4) {
          float f0[8], f1[8], f2[8], f3[8];
          unpack8<T>(p[j], f0);
          unpack8<T>(p[j + 1], f1);
          unpack8<T>(p[j + 2], f2);
          unpack8<T>(p[j + 3], f3);
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[i] += (f0[i] + f1[i]) + (f2[i] + f3[i]);
        }
      }
      // four in flight
      for (; r + 12 < n; r += 16) {
        Pack8 p0 = load(base + (int64_t)(row0 + r) * a.k_row_stride);
        Pack8 p1 = load(base + (int64_t)(row0 + r + 4) * a.k_row_stride);
        Pack8 p2 = load(base + (int64_t)(row0 + r + 8) * a.k_row_stride);
        Pack8 p3 = load(base + (int64_t)(row0 + r + 12) * a.k_row_stride);
        float f0[8], f1[8], f2[8], f3[8];
        unpack8<T>(p0, f0);
        unpack8<T>(p1, f1);
        unpack8<T>(p2, f2);
        unpack8<T>(p3, f3);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += (f0[i] + f1[i]) + (f2[i] + f3[i]);
      }
      for (; r < n; r += 4) {
        Pack8 p0 = load(base + (int64_t)(row0 + r) * a.k_row_stride);
        float f0[8];
        unpack8<T>(p0, f0);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += f0[i];
      }
    };
    if constexpr (HD > 0 || !STREAM) {
      sum_rows(std::integral_constant<bool, STREAM>{});
    } else {
      if ((int64_t)total_k * nvec * 16 >= kPoolStreamBytes)
        sum_rows(std::true_type{});
      else
        sum_rows(std::false_type{});
    }
  }
  // the query rows of this wave's first key head: on their way during the reduction
  constexpr int KS = HD > 0 ? HD / 16 : 1;
  const int r = lane & 31, hh = lane >> 5;
  Pack8 qf[KS];
  auto load_q = [&](int hk) {
    const int g = r / few.rows, row = r - g * few.rows;
    const bool mine = g < few.group && row < few_rows && hk < a.heads_k;
    const uint16_t *qp = few.q + (int64_t)(few_q0 + (mine ? row : 0)) * few.q_row_stride + (int64_t)(mine ? hk * few.group + g : 0) * few.q_head_stride;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = mine && hh * KS + ks < vecs_per_head ? ld_global16(qp + (hh * KS + ks) * 8) : zero_pack8();
  };
  if constexpr (HD > 0) load_q(blockIdx.z * block_heads + wave);
  __shared__ float red[4][64][9];
#pragma unroll
  for (int i = 0; i < 8; ++i) red[wave][lane][i] = acc[i];
  __syncthreads();
  __shared__ Pack8 mean[64];
  __shared__ int pooled_row;
  if (wave == 0 && active) {
    const float nf = (float)n;
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = ((red[0][lane][i] + red[1][lane][i]) + (red[2][lane][i] + red[3][lane][i])) / nf;
    Pack8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o.w[i] = pack2<T>(s[2 * i], s[2 * i + 1]);
    const int out_row = (offsets ? before : a.cu_seqlens_km[b]) + c;
    if constexpr (HD > 0) {
      mean[lane] = o;
      if (lane == 0) pooled_row = out_row;
    } else {
      uint16_t *dst = reinterpret_cast<uint16_t *>(a.km) + (int64_t)out_row * a.km_row_stride + (int64_t)head * a.km_head_stride + d0;
      *reinterpret_cast<Pack8 *>(dst) = o;
    }
  }
  if constexpr (HD > 0) {
    __syncthreads();
    for (int j = wave; j < block_heads; j += 4) {
      const int hk = blockIdx.z * block_heads + j;
      if (hk >= a.heads_k) break;
      if (j != wave) load_q(hk);
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mfma32<T>(mean[j * vecs_per_head + min(hh * KS + ks, vecs_per_head - 1)], qf[ks], s);  // (every row of the product is the chunk's)
      if (hh == 0 && r < few.group * few.rows) few.scores[((int64_t)pooled_row * few.heads + (int64_t)hk * few.group) * few.rows + r] = s[0];
    }
  }
}

// cu_km[b] = sum over b' < b of ceil(len_b' / chunk): one block, every thread a contiguous run of sequences.
__global__ __launch_bounds__(256) void chunk_offsets_kernel(const int32_t *cu, int32_t *cu_km, int batch, int chunk) {
  __shared__ int part[256];
  const int tid = threadIdx.x;
  const int per = (batch + 255) / 256;
  const int lo = min(batch, tid * per), hi = min(batch, lo + per);
  int s = 0;
  for (int b = lo; b < hi; ++b) s += (cu[b + 1] - cu[b] + chunk - 1) / chunk;
  part[tid] = s;
  __syncthreads();
  // inclusive scan over the 256 partial sums
  for (int d = 1; d < 256; d <<= 1) {
    const int v = tid >= d ? part[tid - d] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  int run = part[tid] - s;
  for (int b = lo; b < hi; ++b) {
    cu_km[b] = run;
    run += (cu[b + 1] - cu[b] + chunk - 1) / chunk;
  }
  if (tid == 255) cu_km[batch] = part[255];
}

}  // namespace fmoba

extern "C" int fmoba_chunk_offsets(const int32_t *cu_seqlens, int32_t *cu_seqlens_km, int32_t batch, int32_t chunk, void *stream) {
  using namespace fmoba;
  FMOBA_REQUIRE(batch > 0, "chunk_offsets: batch size must be positive");
  FMOBA_REQUIRE(chunk > 0, "chunk_offsets: chunk size must be positive");
  FMOBA_REQUIRE(cu_seqlens && cu_seqlens_km, "chunk_offsets: null pointer");
  hipLaunchKernelGGL(chunk_offsets_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, cu_seqlens, cu_seqlens_km, batch, chunk);
  FMOBA_LAUNCH_CHECK("chunk_offsets");
  return 0;
}

// `extra`: cu_km and clear_* of PoolExtra.  `few`: scores in place of the means (km and its strides are not looked at)
static int mean_pool_run(const fmoba_mean_pool_args *a, const fmoba::PoolExtra &extra, void *stream, const fmoba::FewGate *few = nullptr, int64_t total_k = 0) {
  using namespace fmoba;
  FMOBA_REQUIRE(a != nullptr, "mean_pool: null args");
  FMOBA_REQUIRE(a->dtype == FMOBA_DTYPE_F16 || a->dtype == FMOBA_DTYPE_BF16, "mean_pool: only fp16 and bf16 are supported");
  FMOBA_REQUIRE(a->batch > 0, "mean_pool: batch size must be positive");
  FMOBA_REQUIRE(a->chunk > 0, "mean_pool: chunk size must be positive");
  FMOBA_REQUIRE(a->head_dim > 0 && a->head_dim % 8 == 0, "mean_pool: head_dim must be a multiple of 8");
  FMOBA_REQUIRE(a->heads_k > 0, "mean_pool: heads_k must be positive");
  if (a->max_chunks <= 0) return 0;
  FMOBA_REQUIRE(a->k && (a->km || few != nullptr) && a->cu_seqlens_k && a->cu_seqlens_km, "mean_pool: null pointer");
  FMOBA_REQUIRE(a->k_row_stride % 8 == 0 && a->k_head_stride % 8 == 0 && (few != nullptr || (a->km_row_stride % 8 == 0 && a->km_head_stride % 8 == 0)),
                "mean_pool: strides must be multiples of 8 elements (16-byte vectors)");
  FMOBA_REQUIRE(((uintptr_t)a->k % 16) == 0 && (few != nullptr || ((uintptr_t)a->km % 16) == 0), "mean_pool: k and km must be 16-byte aligned");
  const int nvec = a->heads_k * (a->head_dim / 8);
  dim3 grid(a->max_chunks, a->batch, ceil_div(nvec, 64));
  FMOBA_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "mean_pool: batch or heads*dim too large for the launch grid");
  hipStream_t s = (hipStream_t)stream;
  const bool many = a->chunk > 64 && nvec <= 128;  // (the reasons stand at its loop)
  const int hd = few == nullptr ? 0 : a->head_dim <= 64 ? 64 : a->head_dim <= 128 ? 128 : 256;
  FewGate scored{};
  if (few != nullptr) {
    scored = *few;
    scored.block_heads = 64 / (a->head_dim / 8);
    grid.z = ceil_div(a->heads_k, scored.block_heads);
  }
  if (few == nullptr) total_k = (int64_t)a->batch * a->max_chunks * a->chunk;  // (no more than)
  // (narrow rows that share cache lines: 32 requests, 500 MB of keys of one head of 80 170.5 us, past the caches 174, of two of 40 166.4 and 170.9; two of 80 102.4 and 99.9)
  const bool stream_keys = (nvec % 8 == 0 || nvec >= 16) && total_k > (kPoolStreamBytes - 1) / (nvec * 16);
  auto pick = [&](auto t) {
    typedef decltype(t) T;
    auto instance = [&](auto hd_) {
      constexpr int HD = decltype(hd_)::value;
      if (stream_keys) return many ? mean_pool_kernel<T, true, HD, true> : mean_pool_kernel<T, false, HD, true>;
      return many ? mean_pool_kernel<T, true, HD, false> : mean_pool_kernel<T, false, HD, false>;
    };
    if (hd == 64) return instance(std::integral_constant<int, 64>{});
    if (hd == 128) return instance(std::integral_constant<int, 128>{});
    if (hd == 256) return instance(std::integral_constant<int, 256>{});
    return instance(std::integral_constant<int, 0>{});
  };
  hipLaunchKernelGGL(a->dtype == FMOBA_DTYPE_BF16 ? pick(bf16_t()) : pick(f16_t()), grid, dim3(256), 0, s, *a, extra, scored);
  FMOBA_LAUNCH_CHECK("mean_pool");
  return 0;
}

extern "C" int fmoba_mean_pool(const fmoba_mean_pool_args *a, void *stream) { return mean_pool_run(a, fmoba::PoolExtra{nullptr, nullptr, 0}, stream); }

namespace fmoba {
// every block counts the sequences before its own: up to this many it is no more than a handful of loads per lane
constexpr int kPoolOffsetsBatch = 1024;

int mean_pool_with_offsets(const fmoba_mean_pool_args *a, int32_t *clear, int64_t clear_vec16, void *stream) {
  int32_t *cu_km = const_cast<int32_t *>(a->cu_seqlens_km);
  if (a->batch > kPoolOffsetsBatch) {
    if (int rc = fmoba_chunk_offsets(a->cu_seqlens_k, cu_km, a->batch, a->chunk, stream)) return rc;
    cu_km = nullptr;
  }
  return mean_pool_run(a, PoolExtra{cu_km, clear, clear_vec16}, stream);
}

// Whether the pooling pass can score the rows of a call: a product has 32 columns.
bool pool_scores_feasible(int head_dim, int group, int rows, int batch) { return head_dim <= 256 && group * rows <= 32 && batch <= kPoolOffsetsBatch; }
int mean_pool_with_scores(const fmoba_mean_pool_args *a, const FewGate &few, int64_t total_k, void *stream) {
  return mean_pool_run(a, PoolExtra{const_cast<int32_t *>(a->cu_seqlens_km), nullptr, 0}, stream, &few, total_k);
}
}  // namespace fmoba
