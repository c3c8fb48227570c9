// Vision-token splice fused with the embedding gather, for gfx950.
//
// Semantics: SiQ_VLForCausalLM.forward (siq_vl/model/modeling.py:252-270):
//   token_embeddings = embed_tokens(input_ids)                      (:253)
//   positions = (input_ids == image_token_index).nonzero()         (:257)
//   check #positions == #vision rows (ValueError otherwise)         (:259-267)
//   token_embeddings[positions] = vision_flat (row-major order)    (:269-270)
// Here each output row is written once, from the vision rows for image
// tokens (in row-major order of their positions) or from the embedding table
// otherwise: no embedding row is gathered only to be overwritten, and the
// count needs no nonzero() on the host.
//
// Kernels:
//  * splice_fused_kernel (up to kFusedMaxTokens tokens): the whole forward
//    in one launch, each workgroup counting the image tokens before its own
//    (below); longer batches run the next two kernels;
//  * splice_scan_kernel (one workgroup; per round 16 chunks of 1024 tokens
//    loaded at once, wave ballots, one prefix over the 256 (chunk, wave)
//    counts): exclusive prefix count of image
//    tokens in token order -> rank[p] for every token, image_pos[r] = p for
//    image slot r < n_vision, counts[0] = image tokens found, counts[1] = ids
//    outside [0, vocab) (their rows are written as zeros; the reference's
//    embedding would raise a device-side assert);
//  * splice_gather_kernel: one wave per token row, 16 bytes per lane per
//    step (HBM-bound: read and write hidden * 2 bytes per token);
//  * gather_rows_kernel: dst[i] = src[rows[i]] (the backward's vision rows;
//    rows[i] < 0 gives a zero row);
//  * emb_prep_kernel, emb_sum_kernel, emb_hot_kernel: the embedding table's
//    gradient (below).
#include <algorithm>

#include "ids.h"
#include "splice.h"

namespace siq {

namespace {

constexpr int kScanThreads = 1024;
constexpr int kPer = 16;  // chunks of kScanThreads tokens per round of the scan

__global__ __launch_bounds__(kScanThreads) void splice_scan_kernel(const int64_t* __restrict__ ids, int64_t n,
                                                                   int64_t vocab, int64_t image_id,
                                                                   int64_t n_vision, int32_t* __restrict__ rank,
                                                                   int32_t* __restrict__ image_pos,
                                                                   int64_t* __restrict__ counts) {
  constexpr int NWV = kScanThreads / 64;
  static_assert(kPer * NWV == 256, "one (chunk, wave) count per lane quarter");
  __shared__ int cnt_sh[kPer * NWV];  // image tokens of (chunk i, wave w) at i * NWV + w, in token order
  __shared__ long long carry_sh;
  __shared__ unsigned long long bad_sh;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;  // lanes before this one
  if (tid == 0) {
    carry_sh = 0;
    bad_sh = 0;
  }
  __syncthreads();
  unsigned long long bad = 0;
  // rounds of kPer chunks of kScanThreads tokens; token c0 + i kScanThreads + tid goes to this thread, so
  // every load and store of a chunk is one contiguous run per wave
  for (int64_t c0 = 0; c0 < n; c0 += (int64_t)kScanThreads * kPer) {
    int64_t v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t pp = c0 + (int64_t)i * kScanThreads + tid;
      v[i] = pp < n ? ids[pp] : image_id - 1;
    }
    uint64_t m[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const bool inb = c0 + (int64_t)i * kScanThreads + tid < n;
      const bool img = inb && v[i] == image_id;
      bad += (inb && !img && (v[i] < 0 || v[i] >= vocab)) ? 1 : 0;
      m[i] = __ballot(img);
      if (lane == 0) cnt_sh[i * NWV + wv] = __popcll(m[i]);
    }
    __syncthreads();
    // every wave forms the exclusive prefix of the 256 counts in token order: lane l holds entries 4l .. 4l + 3
    const int a0 = cnt_sh[4 * lane], a1 = cnt_sh[4 * lane + 1], a2 = cnt_sh[4 * lane + 2], a3 = cnt_sh[4 * lane + 3];
    const int lsum = a0 + a1 + a2 + a3;
    int incl = lsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    const int total = __shfl(incl, 63);
    // entry i * NWV + wv sits in lane 4 i + wv / 4 at position wv % 4 (the same position for every i)
    const int k = wv & 3;
    const int mine = incl - lsum + (k > 0 ? a0 : 0) + (k > 1 ? a1 : 0) + (k > 2 ? a2 : 0);
    const long long carry = carry_sh;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t pp = c0 + (int64_t)i * kScanThreads + tid;
      const long long r = carry + __shfl(mine, 4 * i + (wv >> 2)) + __popcll(m[i] & below);
      if (pp < n) {
        rank[pp] = (int32_t)r;
        if (v[i] == image_id && r < n_vision) image_pos[r] = (int32_t)pp;
      }
    }
    __syncthreads();
    if (tid == 0) carry_sh += total;
    __syncthreads();
  }
  atomicAdd(&bad_sh, bad);
  __syncthreads();
  if (tid == 0) {
    counts[0] = carry_sh;
    counts[1] = (int64_t)bad_sh;
  }
  // fewer image tokens than vision rows (the count check fails, maybe only
  // later on the host): the slots no token filled hold -1, which the row
  // gather of the backward turns into zero rows instead of reading garbage
  for (long long r = carry_sh + tid; r < n_vision; r += kScanThreads) image_pos[r] = -1;
}

__global__ __launch_bounds__(256) void splice_gather_kernel(const SpliceArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t nvec = a.hidden / 8;
  for (int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); p < a.n; p += (int64_t)gridDim.x * 4) {
    const int64_t v = a.ids[p];
    const bf16* src = nullptr;
    if (v == a.image_id) {
      const int64_t r = a.rank[p];
      if (r < a.n_vision) src = a.vision + r * a.hidden;
    } else if (v >= 0 && v < a.vocab) {
      src = a.weight + v * a.hidden;
    }
    bf16* dst = a.out + p * a.hidden;
    for (int64_t c = lane; c < nvec; c += 64) st_bf16x8(dst + 8 * c, src ? ld_bf16x8(src + 8 * c) : zero_bf16x8());
  }
}

// One-kernel splice for batches of up to kFusedMaxTokens tokens (the scan
// kernel above is a single workgroup, and waiting for it costs more than
// counting again).  Workgroup w owns tokens [w R, w R + R), R = rpw (a
// multiple of 64): it counts the image tokens before its first token itself
// (every thread reads kFusedUnroll ids of the earlier tokens at a time; at
// most kFusedMaxTokens * 8 bytes, served by L2), ranks its own image tokens
// with wave ballots, records each row's source in LDS, then its eight waves
// copy the rows, kFusedUnroll 16-byte chunks per lane in flight.  The last
// workgroup reads every id, so it writes counts and fills the vision slots
// no token took with -1.  Outputs are those of splice_scan_kernel +
// splice_gather_kernel, bit for bit (the rank workspace is not used).
constexpr int kFusedThreads = 512;
constexpr int kFusedBlocks = 256;
constexpr int64_t kFusedMaxTokens = 32768;
constexpr int kFusedMaxRows = (int)(kFusedMaxTokens / kFusedBlocks);
constexpr int kFusedUnroll = 8;
static_assert(kFusedMaxRows % 64 == 0, "rows per workgroup come in waves of 64");

__global__ __launch_bounds__(kFusedThreads) void splice_fused_kernel(const SpliceArgs a, int32_t* __restrict__ image_pos,
                                                                     int64_t* __restrict__ counts, int rpw) {
  constexpr int NWV = kFusedThreads / 64;
  __shared__ const bf16* src_sh[kFusedMaxRows];
  __shared__ long long red_sh[2][NWV];
  __shared__ long long found_sh;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * rpw;
  const bool last = blockIdx.x == gridDim.x - 1;
  const int64_t image_id = a.image_id, vocab = a.vocab;

  // image tokens (and, in the last workgroup, ids outside [0, vocab)) before r0
  long long img = 0, bad = 0;
  for (int64_t base = tid; base < r0; base += (int64_t)kFusedThreads * kFusedUnroll) {
    int64_t v[kFusedUnroll];
#pragma unroll
    for (int u = 0; u < kFusedUnroll; ++u) {
      const int64_t p = base + (int64_t)u * kFusedThreads;
      v[u] = p < r0 ? a.ids[p] : image_id - 1;
    }
#pragma unroll
    for (int u = 0; u < kFusedUnroll; ++u) {
      const bool inb = base + (int64_t)u * kFusedThreads < r0;
      img += (inb && v[u] == image_id) ? 1 : 0;
      bad += (inb && v[u] != image_id && (v[u] < 0 || v[u] >= vocab)) ? 1 : 0;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    img += __shfl_xor(img, o);
    bad += __shfl_xor(bad, o);
  }
  if (lane == 0) {
    red_sh[0][wv] = img;
    red_sh[1][wv] = bad;
  }
  __syncthreads();
  if (wv == 0) {
    long long carry = 0, badt = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      carry += red_sh[0][w];
      badt += red_sh[1][w];
    }
    // this workgroup's tokens, 64 at a time in token order
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for (int j = 0; j < rpw; j += 64) {
      const int64_t p = r0 + j + lane;
      const bool inb = p < a.n;
      const int64_t v = inb ? a.ids[p] : image_id - 1;
      const bool isimg = inb && v == image_id;
      const uint64_t m = __ballot(isimg);
      const long long r = carry + __popcll(m & below);
      const bf16* src = nullptr;
      if (isimg) {
        if (r < a.n_vision) {
          src = a.vision + r * a.hidden;
          image_pos[r] = (int32_t)p;
        }
      } else if (v >= 0 && v < vocab) {
        src = a.weight + v * a.hidden;
      }
      src_sh[j + lane] = src;
      carry += __popcll(m);
      badt += __popcll(__ballot(inb && !isimg && (v < 0 || v >= vocab)));
    }
    if (last && lane == 0) {
      counts[0] = carry;
      counts[1] = badt;
      found_sh = carry;
    }
  }
  __syncthreads();
  if (last) {
    for (long long r = found_sh + tid; r < a.n_vision; r += kFusedThreads) image_pos[r] = -1;
  }

  // rows: wave wv copies rows wv, wv + NWV, ... of the workgroup's rows that exist, as one list of
  // (row, 16-byte chunk) pairs
  const int nvec = (int)(a.hidden / 8);
  const int nrows = (int)min<int64_t>(rpw, a.n - r0);
  const int my_rows = nrows > wv ? (nrows - wv + NWV - 1) / NWV : 0;
  const int total = my_rows * nvec;
  for (int base = lane; base < total; base += 64 * kFusedUnroll) {
    bf16x8 x[kFusedUnroll];
#pragma unroll
    for (int u = 0; u < kFusedUnroll; ++u) {
      const int idx = base + 64 * u;
      if (idx < total) {
        const int k = idx / nvec, c = idx - k * nvec;
        const bf16* src = src_sh[wv + NWV * k];
        x[u] = src ? ld_bf16x8(src + 8 * c) : zero_bf16x8();
      }
    }
#pragma unroll
    for (int u = 0; u < kFusedUnroll; ++u) {
      const int idx = base + 64 * u;
      if (idx < total) {
        const int k = idx / nvec, c = idx - k * nvec;
        st_bf16x8(a.out + (r0 + wv + NWV * k) * a.hidden + 8 * c, x[u]);
      }
    }
  }
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const bf16* __restrict__ src, const int32_t* __restrict__ rows,
                                                          int64_t n, int64_t hidden, bf16* __restrict__ dst) {
  const int lane = threadIdx.x & 63;
  const int64_t nvec = hidden / 8;
  for (int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); i < n; i += (int64_t)gridDim.x * 4) {
    const int32_t r = rows[i];
    const bf16* s = src + (int64_t)r * hidden;
    bf16* d = dst + i * hidden;
    for (int64_t c = lane; c < nvec; c += 64) st_bf16x8(d + 8 * c, r >= 0 ? ld_bf16x8(s + 8 * c) : zero_bf16x8());
  }
}

// ---------------------------------------------------------------- embedding-table gradient
// dW[v] = sum of grad[p] over the tokens p with ids[p] == v, for ids in
// [0, vocab) other than the skipped ones (the image token, whose rows the
// splice overwrote, and the table's padding index); rows that no token
// reaches are zero.  The sum runs in fp32 in the order of torch's sorted
// embedding backward (aten/src/ATen/native/cuda/EmbeddingBackwardKernel.cu:
// the ids sorted stably, so each id's tokens in position order, summed in
// partial sums of at most kRowsPerPartial rows that are then added in order)
// and is rounded to the table's dtype once.
//
//  * emb_prep_kernel: one workgroup per chunk of kEmbChunk tokens clears the
//    chunk's run table, sorts the 64-bit keys (id << 32 | position in the
//    chunk; skipped and invalid ids get all-ones keys, which sort last) with
//    a bitonic network in LDS, then records each id's run [begin, end) in the
//    run table (begin = end = 0: no run); the launch's other workgroups zero
//    the table gradient meanwhile (the HBM-bound bulk of the work: one
//    streaming pass of 16-byte stores);
//  * emb_sum_kernel: one wave per sorted key; the wave of the first key of an
//    id in the first chunk that holds the id sums the id's runs over that
//    chunk and the later ones (chunks are in position order, so the
//    concatenation is the stable order) and writes the row, if they are one
//    partial sum (at most kRowsPerPartial tokens); every other wave returns at
//    once, and the wave of an id with more tokens puts it on a list;
//  * emb_hot_kernel: the ids of the lists, a workgroup (or, for those of few
//    partial sums, some of its waves) per (id, column block).  The partial sums of an id are independent, so the sixteen waves
//    form one each, all its rows in flight, and the workgroup adds them in
//    order.  Token ids are Zipf-distributed (the commonest id of 12288 text
//    tokens comes about 700 times), and one wave adding those rows one after
//    the other waited for memory at each of them: 1065 us of the 1.24 ms that
//    the splice's forward and backward took at 16384 tokens x 1536; with the
//    lists emb_sum takes 27 us and emb_hot 36 us.
constexpr int kEmbChunk = kIdChunk;
constexpr int kRowsPerPartial = 10;
// Ids with more than one partial sum, by how many: up to 2, 4, 6 (tiers 0 to 2:
// as many waves) or more (tier 3: a workgroup).  A tier's list holds at most
// n / (tokens that its ids have at least) ids.
constexpr int kTiers = 4;
__host__ __device__ constexpr int tier_waves(int t) { return 2 * t + 2; }
__host__ __device__ constexpr int tier_tokens(int t) { return (t == 0 ? 1 : tier_waves(t - 1)) * kRowsPerPartial + 1; }
constexpr int kWarmTokens = tier_tokens(kTiers - 1) - 1;
static_assert(kWarmTokens <= 64, "a lane per token");

// Blocks [0, nch) sort one chunk each (after clearing that chunk's run
// table); the other blocks zero the table gradient meanwhile, so that the
// sort, which keeps only nch CUs busy, hides under the HBM-bound clear.
__global__ __launch_bounds__(1024) void emb_prep_kernel(const int64_t* __restrict__ ids, int64_t n, int64_t vocab,
                                                        int64_t skip0, int64_t skip1, uint64_t* __restrict__ keys,
                                                        int2* __restrict__ seg, int nch, u32x4* __restrict__ dw,
                                                        int64_t dw16, int* __restrict__ nhot) {
  __shared__ uint64_t sk[kEmbChunk];
  if (blockIdx.x == 0 && threadIdx.x < kTiers) nhot[threadIdx.x] = 0;
  const u32x4 z = {0u, 0u, 0u, 0u};
  if ((int)blockIdx.x >= nch) {
    const int64_t stride = (int64_t)(gridDim.x - nch) * 1024;
    for (int64_t i = (int64_t)(blockIdx.x - nch) * 1024 + threadIdx.x; i < dw16; i += stride) dw[i] = z;
    return;
  }
  int2* sg = seg + (int64_t)blockIdx.x * vocab;
  for (int64_t i = threadIdx.x; i < vocab; i += blockDim.x) sg[i] = make_int2(0, 0);
  const int64_t base = (int64_t)blockIdx.x * kEmbChunk;
  const int len = (int)min<int64_t>(kEmbChunk, n - base);
  int np2 = 64;
  while (np2 < len) np2 <<= 1;
  for (int i = threadIdx.x; i < np2; i += blockDim.x) {
    uint64_t k = kNoKey;
    if (i < len) {
      const int64_t v = ids[base + i];
      if (v >= 0 && v < vocab && v != skip0 && v != skip1) k = ((uint64_t)v << 32) | (uint32_t)i;
    }
    sk[i] = k;
  }
  __syncthreads();  // also orders the run table's clearing before its writes below
  sort_keys(sk, np2);
  // every key slot of the chunk is written (all-ones past the tokens), so the sum kernel reads no stale key
  uint64_t* kout = keys + base;
  for (int i = threadIdx.x; i < kEmbChunk; i += blockDim.x) {
    const uint64_t key = i < np2 ? sk[i] : kNoKey;
    kout[i] = key;
    if (key == kNoKey) continue;
    const uint32_t v = (uint32_t)(key >> 32);
    if (i == 0 || (uint32_t)(sk[i - 1] >> 32) != v) sg[v].x = i;
    if (i == len - 1 || (uint32_t)(sk[i + 1] >> 32) != v) sg[v].y = i + 1;
  }
}

template <typename T>
struct Vec16;
template <>
struct Vec16<bf16> {
  static constexpr int E = 8;
  typedef bf16x8 Raw;
  __device__ static void add(float (&x)[8], const Raw& v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] += (float)v[i];
  }
  __device__ static void store(bf16* p, const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (bf16)x[i];
    st_bf16x8(p, v);
  }
};
template <>
struct Vec16<float> {
  static constexpr int E = 4;
  typedef f32x4 Raw;
  __device__ static void add(float (&x)[4], const Raw& v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] += v[i];
  }
  __device__ static void store(float* p, const float (&x)[4]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{x[0], x[1], x[2], x[3]};
  }
};

// An id whose tokens make more than one partial sum: first chunk c that holds it.
struct HotId {
  uint32_t v;
  int c;
};
struct HotLists {
  HotId* ids[kTiers];
  int* n;  // [kTiers]
};

// The id's runs in chunks c .. c + 63 are read one per lane.  R rows x U
// 16-byte chunks per lane are in flight together.
template <typename T>
__global__ __launch_bounds__(256) void emb_sum_kernel(const T* __restrict__ grad, const uint64_t* __restrict__ keys,
                                                      const int2* __restrict__ seg, int nchunks, int64_t vocab,
                                                      int64_t hidden, T* __restrict__ dw, HotLists hot) {
  using V = Vec16<T>;
  constexpr int E = V::E, U = 4, R = 4;
  __shared__ uint32_t tok_sh[4][kRowsPerPartial];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t item = (int64_t)blockIdx.x * 4 + wv;
  if (item >= (int64_t)nchunks * kEmbChunk) return;
  const int c = (int)(item / kEmbChunk), i = (int)(item % kEmbChunk);
  const uint64_t key = keys[item];
  if (key == kNoKey) return;
  const uint32_t v = (uint32_t)(key >> 32);
  if (i > 0 && (uint32_t)(keys[item - 1] >> 32) == v) return;  // not the first key of its id in this chunk
  // an earlier chunk holding the id means its wave writes the row
  for (int c0 = 0; c0 < c; c0 += 64) {
    const int cc = c0 + lane;
    int2 r = make_int2(0, 0);
    if (cc < c) r = seg[(int64_t)cc * vocab + v];
    if (__ballot(r.y > r.x)) return;
  }
  // the id's tokens (a wave's own LDS row: its writes and reads run in order)
  int cnt = 0;
  for (int g0 = c; g0 < nchunks && cnt <= kWarmTokens; g0 += 64) {
    int2 mine = make_int2(0, 0);
    if (g0 + lane < nchunks) mine = seg[(int64_t)(g0 + lane) * vocab + v];
    const int len = mine.y - mine.x;
    int incl = len;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    const int at = cnt + incl - len;
    for (int t = 0; t < len && at + t < kRowsPerPartial; ++t)
      tok_sh[wv][at + t] = (uint32_t)((g0 + lane) * kEmbChunk) + (uint32_t)keys[(int64_t)(g0 + lane) * kEmbChunk + mine.x + t];
    cnt += __shfl(incl, 63);
  }
  if (cnt > kRowsPerPartial) {
#pragma unroll
    for (int t = 0; t < kTiers; ++t)
      if (lane == 0 && cnt >= tier_tokens(t) && (t == kTiers - 1 || cnt < tier_tokens(t + 1)))
        hot.ids[t][atomicAdd(hot.n + t, 1)] = HotId{v, c};
    return;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // the token list is in LDS
  const int64_t nvec = hidden / E;
  for (int64_t p0 = 0; p0 < nvec; p0 += 64 * U) {
    float part[U][E];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) part[u][e] = 0.f;
    for (int t0 = 0; t0 < cnt; t0 += R) {
      typename V::Raw x[R][U];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (t0 + r >= cnt) break;
        const T* src = grad + (int64_t)tok_sh[wv][t0 + r] * hidden;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t ch = p0 + 64 * u + lane;
          if (ch < nvec) x[r][u] = *reinterpret_cast<const typename V::Raw*>(src + ch * E);
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (t0 + r >= cnt) break;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (p0 + 64 * u + lane < nvec) V::add(part[u], x[r][u]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t ch = p0 + 64 * u + lane;
      if (ch < nvec) V::store(dw + (int64_t)v * hidden + ch * E, part[u]);
    }
  }
}

// One hot id and one block of 64 E columns per workgroup (ids strided over
// gridDim.x).  Rounds of kHotWaves partial sums: the workgroup lists the
// round's tokens in LDS (one thread per token), wave w sums rows
// kRowsPerPartial w .. of the round in order, and thread j adds the round's
// partial sums of column j in order to its running total.  Then the ids of few
// partial sums, as many to a workgroup as its waves are enough for, from the
// workgroups on that the lists before left without one.  (A workgroup to each of
// them: every id 11 times, 16384 tokens x 1536 230 us, where one wave had added
// the rows one by one in 146; 153 now; 40000 x 2048 553, 235 and 255.  In
// emb_sum's wave, one partial sum after the other, up to 40 rows held up the ids
// behind them: Zipf-distributed ids 163 -> 193 us.)
constexpr int kHotWaves = 16, kHotRound = kHotWaves * kRowsPerPartial;
struct HotShared {
  uint32_t* tok;  // [kHotRound]
  float* part;    // [kHotWaves][COLS]
  int* cnt;       // [kHotWaves]
};

// The ids of tier `t`, W = tier_waves(t) waves each; unit0: workgroups that the
// lists before took.
template <typename T, int TIER>
__device__ __forceinline__ void emb_warm(const T* __restrict__ grad, const uint64_t* __restrict__ keys,
                                         const int2* __restrict__ seg, int nchunks, int64_t vocab, int64_t hidden,
                                         T* __restrict__ dw, const HotId* __restrict__ ids, int n,
                                         const HotShared& sh, int& unit0) {
  if (n == 0) return;
  using V = Vec16<T>;
  constexpr int E = V::E, COLS = 64 * E, W = tier_waves(TIER), IDS = kHotWaves / W, NTOK = W * kRowsPerPartial;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, group = wv / W, wq = wv % W;
  const int64_t nvec = hidden / E, ch = (int64_t)blockIdx.y * 64 + lane, col0 = (int64_t)blockIdx.y * COLS;
  const int units = (n + IDS - 1) / IDS, G = (int)gridDim.x;
  for (int unit = ((int)blockIdx.x + G - unit0 % G) % G; unit < units; unit += G) {
    const bool mine = group < IDS && unit * IDS + group < n;
    const HotId id = ids[min(unit * IDS + group, n - 1)];
    if (mine && wq == 0) {
      int cnt = 0;
      for (int g0 = id.c; g0 < nchunks; g0 += 64) {
        int2 r = make_int2(0, 0);
        if (g0 + lane < nchunks) r = seg[(int64_t)(g0 + lane) * vocab + id.v];
        const int len = r.y - r.x;
        // lane cnt + rank: token `rank` of the chunks' runs, in the first chunk whose inclusive count exceeds it
        int q = -1, base = 0, upto = 0;
        for (uint64_t m = __ballot(len > 0); m != 0; m &= m - 1) {
          const int j = (int)__builtin_ctzll(m), l = __builtin_amdgcn_readlane(len, j);
          if (q < 0 && lane >= cnt && lane - cnt < upto + l) {
            q = j;
            base = upto;
          }
          upto += l;
        }
        const int at = __shfl(r.x, q & 63) + lane - cnt - base;
        if (q >= 0)
          sh.tok[group * NTOK + lane] =
              (uint32_t)((g0 + q) * kEmbChunk) + (uint32_t)keys[(int64_t)(g0 + q) * kEmbChunk + at];
        cnt += upto;
      }
      if (lane == 0) sh.cnt[group] = cnt;
    }
    __syncthreads();
    const int have = mine ? sh.cnt[group] : 0, r0 = wq * kRowsPerPartial, nr = min(kRowsPerPartial, have - r0);
    if (nr > 0 && ch < nvec) {
      typename V::Raw x[kRowsPerPartial];
      float part[E];
#pragma unroll
      for (int r = 0; r < kRowsPerPartial; ++r)  // rows past the last one re-read it
        x[r] = *reinterpret_cast<const typename V::Raw*>(
            grad + (int64_t)sh.tok[group * NTOK + r0 + min(r, nr - 1)] * hidden + ch * E);
#pragma unroll
      for (int e = 0; e < E; ++e) part[e] = 0.f;
#pragma unroll
      for (int r = 0; r < kRowsPerPartial; ++r)
        if (r < nr) V::add(part, x[r]);
#pragma unroll
      for (int e = 0; e < E; ++e) sh.part[wv * COLS + lane * E + e] = part[e];
    }
    __syncthreads();
    const int np = (have + kRowsPerPartial - 1) / kRowsPerPartial;
    if (mine) {
      for (int j = tid - group * W * 64; j < COLS && col0 + j < hidden; j += 64 * W) {
        float tot = 0.f;
        for (int w = 0; w < np; ++w) tot += sh.part[(group * W + w) * COLS + j];
        dw[(int64_t)id.v * hidden + col0 + j] = (T)tot;
      }
    }
    __syncthreads();  // the lists and sums are read no more
  }
  unit0 += units;
}

template <typename T>
__global__ __launch_bounds__(64 * kHotWaves) void emb_hot_kernel(const T* __restrict__ grad,
                                                                 const uint64_t* __restrict__ keys,
                                                                 const int2* __restrict__ seg, int nchunks,
                                                                 int64_t vocab, int64_t hidden, T* __restrict__ dw,
                                                                 HotLists hot) {
  using V = Vec16<T>;
  constexpr int E = V::E, COLS = 64 * E;
  static_assert(COLS <= 64 * kHotWaves, "a thread per column");
  __shared__ uint32_t tok_sh[kHotRound];
  __shared__ int cnt_sh[kHotWaves];
  __shared__ float part_sh[kHotWaves][COLS];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t nvec = hidden / E, ch = (int64_t)blockIdx.y * 64 + lane;
  const int64_t col = (int64_t)blockIdx.y * COLS + tid;
  static_assert(kTiers == 4, "the lists' lengths in one load");
  const int4 len = *reinterpret_cast<const int4*>(hot.n);
  const int n = len.w;
  for (int k = blockIdx.x; k < n; k += gridDim.x) {
    const uint32_t v = hot.ids[kTiers - 1][k].v;
    int g0 = hot.ids[kTiers - 1][k].c;  // chunks g0 .. g0 + 63: lane l holds chunk g0 + l's run, every wave alike
    int rank0 = 0;      // tokens of the group's runs listed so far
    int first, incl, total;
    auto group = [&]() {
      int2 mine = make_int2(0, 0);
      if (g0 + lane < nchunks) mine = seg[(int64_t)(g0 + lane) * vocab + v];
      first = mine.x;
      incl = mine.y - mine.x;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
      }
      total = __shfl(incl, 63);
    };
    group();
    float tot = 0.f;
    for (;;) {
      int have = 0;
      for (;;) {
        // token rank0 + tid of the group: in the first chunk whose inclusive count exceeds it
        const int take = min(total - rank0, kHotRound - have);
        const int rank = rank0 + tid;
        int q = 0, base = 0;
        for (int j = 0; j < 64 && g0 + j < nchunks; ++j) {
          const int upto = __builtin_amdgcn_readlane(incl, j);
          q = upto <= rank ? j + 1 : q;
          base = upto <= rank ? upto : base;
        }
        const int at = __shfl(first, q & 63) + rank - base;
        if (tid < take)
          tok_sh[have + tid] = (uint32_t)((g0 + q) * kEmbChunk) + (uint32_t)keys[(int64_t)(g0 + q) * kEmbChunk + at];
        have += take;
        rank0 += take;
        if (have == kHotRound || g0 + 64 >= nchunks) break;
        g0 += 64;
        rank0 = 0;
        group();
      }
      __syncthreads();
      if (have == 0) break;
      const int r0 = wv * kRowsPerPartial, nr = min(kRowsPerPartial, have - r0);
      if (nr > 0 && ch < nvec) {
        typename V::Raw x[kRowsPerPartial];
        float part[E];
#pragma unroll
        for (int r = 0; r < kRowsPerPartial; ++r)  // rows past the last one re-read it
          x[r] = *reinterpret_cast<const typename V::Raw*>(grad + (int64_t)tok_sh[r0 + min(r, nr - 1)] * hidden + ch * E);
#pragma unroll
        for (int e = 0; e < E; ++e) part[e] = 0.f;
#pragma unroll
        for (int r = 0; r < kRowsPerPartial; ++r)
          if (r < nr) V::add(part, x[r]);
#pragma unroll
        for (int e = 0; e < E; ++e) part_sh[wv][lane * E + e] = part[e];
      }
      __syncthreads();
      const int np = (have + kRowsPerPartial - 1) / kRowsPerPartial;
      if (tid < COLS && col < hidden)
        for (int w = 0; w < np; ++w) tot += part_sh[w][tid];
      // the next round's list does not touch part_sh, and its barrier comes before the next partial sums
    }
    if (tid < COLS && col < hidden) dw[(int64_t)v * hidden + col] = (T)tot;
    __syncthreads();  // part_sh and tok_sh are read no more
  }
  const HotShared sh{tok_sh, &part_sh[0][0], cnt_sh};
  int unit0 = n;
  emb_warm<T, 2>(grad, keys, seg, nchunks, vocab, hidden, dw, hot.ids[2], len.z, sh, unit0);
  emb_warm<T, 1>(grad, keys, seg, nchunks, vocab, hidden, dw, hot.ids[1], len.y, sh, unit0);
  emb_warm<T, 0>(grad, keys, seg, nchunks, vocab, hidden, dw, hot.ids[0], len.x, sh, unit0);
}

unsigned row_blocks(int64_t n) {
  int64_t b = (n + 3) / 4;
  if (b > 8192) b = 8192;
  return (unsigned)(b > 0 ? b : 1);
}

}  // namespace

hipError_t splice_fwd(const SpliceArgs& a, int32_t* image_pos, int64_t* counts, hipStream_t stream) {
  if (a.n > 0 && a.n <= kFusedMaxTokens) {
    // rows per workgroup: a multiple of 64 with at most kFusedBlocks workgroups
    const int64_t per = (a.n + kFusedBlocks - 1) / kFusedBlocks;
    const int rpw = (int)((per + 63) / 64 * 64);
    const unsigned blocks = (unsigned)((a.n + rpw - 1) / rpw);
    hipLaunchKernelGGL(splice_fused_kernel, dim3(blocks), dim3(kFusedThreads), 0, stream, a, image_pos, counts, rpw);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(splice_scan_kernel, dim3(1), dim3(kScanThreads), 0, stream, a.ids, a.n, a.vocab, a.image_id,
                     a.n_vision, a.rank, image_pos, counts);
  if (a.n > 0) hipLaunchKernelGGL(splice_gather_kernel, dim3(row_blocks(a.n)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

namespace {
// workspace of the table gradient: sorted keys, run table, the tiers' id lists and their lengths
struct EmbLayout {
  int64_t nch;
  size_t runs, hot[kTiers], nhot, total;
};
EmbLayout emb_layout(int64_t n, int64_t vocab) {
  EmbLayout L;
  L.nch = n > 0 ? (n + kEmbChunk - 1) / kEmbChunk : 0;
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  L.runs = al((size_t)L.nch * kEmbChunk * sizeof(uint64_t));
  size_t off = L.runs + al((size_t)L.nch * (size_t)vocab * sizeof(int2));
  for (int t = 0; t < kTiers; ++t) {
    L.hot[t] = off;
    off += al((size_t)((n > 0 ? n / tier_tokens(t) : 0) + 1) * sizeof(HotId));
  }
  L.nhot = off;
  L.total = off + 256;
  return L;
}

template <typename T>
void launch_emb_sums(const void* grad, const uint64_t* keys, const int2* seg, int64_t n, int nch, int64_t vocab,
                     int64_t hidden, void* dw, const HotLists& hot, hipStream_t stream) {
  const T* g = static_cast<const T*>(grad);
  T* out = static_cast<T*>(dw);
  const unsigned blocks = (unsigned)(((int64_t)nch * kEmbChunk + 3) / 4);
  hipLaunchKernelGGL(emb_sum_kernel<T>, dim3(blocks), dim3(256), 0, stream, g, keys, seg, nch, vocab, hidden, out, hot);
  // no more than one workgroup for every id that can be listed
  const unsigned ids = (unsigned)std::min<int64_t>(n / tier_tokens(0), 128);
  if (ids == 0) return;
  const unsigned cols = (unsigned)((hidden / Vec16<T>::E + 63) / 64);
  hipLaunchKernelGGL(emb_hot_kernel<T>, dim3(ids, cols), dim3(64 * kHotWaves), 0, stream, g, keys, seg, nch, vocab, hidden,
                     out, hot);
}
}  // namespace

size_t embedding_bwd_workspace_bytes(int64_t n, int64_t vocab) { return emb_layout(n, vocab).total; }

hipError_t embedding_bwd(const void* grad, const int64_t* ids, int64_t n, int64_t vocab, int64_t hidden, bool fp32,
                         int64_t skip0, int64_t skip1, void* dw, void* ws, hipStream_t stream) {
  const EmbLayout L = emb_layout(n, vocab);
  const int nch = (int)L.nch;
  char* base = static_cast<char*>(ws);
  uint64_t* keys = reinterpret_cast<uint64_t*>(base);
  int2* seg = reinterpret_cast<int2*>(base + L.runs);
  HotLists hot;
  for (int t = 0; t < kTiers; ++t) hot.ids[t] = reinterpret_cast<HotId*>(base + L.hot[t]);
  hot.n = reinterpret_cast<int*>(base + L.nhot);
  const int64_t dw16 = vocab * hidden * (fp32 ? 4 : 2) / 16;  // hidden % 8 == 0
  const int clear_blocks = (int)std::min<int64_t>((dw16 + 1023) / 1024, 512);
  hipLaunchKernelGGL(emb_prep_kernel, dim3((unsigned)(nch + std::max(clear_blocks, 1))), dim3(1024), 0, stream, ids, n,
                     vocab, skip0, skip1, keys, seg, nch, static_cast<u32x4*>(dw), dw16, hot.n);
  if (nch > 0) {
    if (fp32)
      launch_emb_sums<float>(grad, keys, seg, n, nch, vocab, hidden, dw, hot, stream);
    else
      launch_emb_sums<bf16>(grad, keys, seg, n, nch, vocab, hidden, dw, hot, stream);
  }
  return hipGetLastError();
}

hipError_t gather_rows(const bf16* src, const int32_t* rows, int64_t n, int64_t hidden, bf16* dst,
                       hipStream_t stream) {
  if (n > 0) hipLaunchKernelGGL(gather_rows_kernel, dim3(row_blocks(n)), dim3(256), 0, stream, src, rows, n, hidden, dst);
  return hipGetLastError();
}

}  // namespace siq
