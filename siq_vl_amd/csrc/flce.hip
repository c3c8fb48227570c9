// Fused lm_head linear + cross-entropy (forward and backward) for gfx950.
//
// Semantics: the reference computes logits = h W^T (transformers
// models/qwen2/modeling_qwen2.py:465), upcasts them to fp32 and calls
// F.cross_entropy(ignore_index=-100) with "mean" over non-ignored rows, or
// "sum" divided by num_items_in_batch (loss/loss_utils.py:32-71).  Here:
//   loss = sum_valid (lse_n - z_{n,y_n}) * inv_den,
//   dZ   = (softmax(z_n) - onehot(y_n)) * inv_den  (0 for ignored rows),
//   dH = dZ W,  dW = dZ^T H.
//
// Rows whose label is ignore_index (or out of range) contribute nothing: their
// dH row is zero and they add nothing to the loss or dW.  So the valid rows
// are first compacted, in order, into a contiguous buffer (padded with zero
// rows to the next 256-row tile), every stage below runs on the compacted rows
// only (each workgroup reads the valid count on the device and returns early
// past it), and dH rows are scattered back to their positions.
//
// Each row has a reference: its label logit in log2 units, from a dot product
// of its own (any value not far below the row's maximum does; every logit it
// can be exceeded by is caught below).  Softmax numerators are taken relative
// to it, so one factor per row turns them into probabilities, and the
// gradient products take them as they are.
//
// Pipeline per chunk of C compacted rows (the only logits-sized buffer is one
// chunk's softmax numerators):
//  1. logits GEMM  Z^T = W H_c^T (MFMA, 256x256 tiles, K = hdim).  The epilogue
//     never writes z: it writes E = exp2(z2 - ref) in bf16 (whose exponent
//     range is fp32's: full relative precision) and keeps, per (token,
//     256-column vocab tile), the sum of E (the chunked-vocab logsumexp), and
//     the label logit z_y.  A tile whose sum says that the reference is more
//     than 2^60 below some logit is redone relative to its own maximum, which
//     is recorded.
//  2. row pass over those sums: lse = ref + log2(sum), the row's loss, its
//     factor f = 2^(ref - lse) inv_den and its label weight w = (p_y - 1)
//     inv_den; E at the label is set to zero (the label's term is added in
//     fp32 instead); rows with redone tiles have their E brought to one
//     reference, the one that makes f a power of two; for dW, H's rows are
//     scaled by f and the rows sorted by label.
//  3. dH GEMM  dH_c^T = W^T E_c^T (split over the vocab), dH = f (sum over the
//     splits) + w W[y], and
//  4. dW GEMM  dW^T = (f H_c)^T E_c, plus the sums of w H over the rows of
//     each label.
// So dZ = (softmax - onehot) inv_den never exists: E is written once and read
// twice, where a pass between the products read it and wrote dZ (1.5 of 14.8
// ms at 16384 rows x 1536, V = 151936, 340 of 1970 us at 4099 x 896).  E is
// rounded once on its way into dH (dZ was twice); in dW one rounding of E and
// one of f H replace E's two (in rows with redone tiles E is rounded twice and f
// H not at all); the label terms, which dominate both gradients, are exact.
// With several chunks dW accumulates over them: in dW itself (bf16) when the
// valid rows span two chunks, in an fp32 workspace when they span more;
// whether a chunk starts, continues or finishes that sum is decided on the
// device from the valid-row count, so chunks past the valid rows cost nothing.  Every
// reduction has a fixed order, so results are bitwise reproducible.
//
// Loss only (no gradient wanted, e.g. evaluation under torch.no_grad): the
// logits epilogue keeps its tile sums and z_y but stores no E, the row pass
// stops at the loss, and neither gradient GEMM runs.
#include <algorithm>

#include "flce.h"
#include "gemm.h"
#include "ids.h"

namespace siq {

namespace {

using namespace gemm;

constexpr int kVT = BI;  // vocab columns per logits tile

// ---------------------------------------------------------------- logits
// A tile sum at or above this (or not a number) means the row's reference is
// too low for the tile.
constexpr float kRefLimit = 0x1p60f;

struct LogitsArgs {
  GOp W, H;               // W [V, hdim], H = hidden rows of the chunk [nc, hdim]
  const int64_t* y;       // chunk labels
  const float* ref;       // [nc] row references (log2 units)
  bf16* E;                // [nc, V]
  float* spart;           // [nvt, ldp] tile sum of exp2(z2 - ref); negated for a redone tile
  float* mpart;           // [nvt, ldp] a redone tile's own reference
  float* zy;              // [nc] label logit (natural units)
  const int64_t* nvalid;  // valid (compacted) rows in all chunks
  int64_t V, nc, c0, ldp;
  int nI, nJ;
  int store_e;            // 0: loss only, E is not needed
};

__global__ __launch_bounds__(NT) void flce_logits_kernel(const LogitsArgs p) {
  __shared__ __align__(16) bf16 smem[SMEM];
  int ti, tj;
  if (!tile_of(p.nI, p.nJ, 4, ti, tj)) return;
  const int64_t i0 = (int64_t)ti * BI, j0 = (int64_t)tj * BJ;
  if (j0 >= *p.nvalid - p.c0) return;  // token tile holds no valid row
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int wi = w & 1, wj = w >> 1;
  // accumulator (a, b, r) holds z for vocab row vbase + wave_row(a, wi) + 16 (r / 8) + (r % 8) and token
  // column j0 + wave_col(b, wj) + l32
  const int64_t vbase = i0 + 8 * h;
  // the tokens' references, and their labels' offsets from the tile (-1: elsewhere)
  float ref[2];
  int rel[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int64_t tok = min(j0 + wave_col(b, wj) + l32, p.nc - 1);
    ref[b] = p.ref[tok];
    const int64_t d = p.y[tok] - vbase;
    rel[b] = d >= 0 && d < 256 ? (int)d : -1;
  }
  f32x16 acc[4][2];
  gemm_core<true, true, false>(smem, p.W, p.H, i0, j0, 0, p.W.cols, acc);

  float* red = reinterpret_cast<float*>(smem);  // [2][256]
  // only the last vocab tile has rows past V: masked there alone
  if (i0 + BI > p.V) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (vbase + wave_row(a, wi) + 16 * (r >> 3) + (r & 7) >= p.V) acc[a][b][r] = -INFINITY;
  }
  // E of column b relative to m2 (stored where `store`), and its sum over the tile's rows of this wave
  auto numerators = [&](int b, float m2, bool store) {
    const int64_t tok = j0 + wave_col(b, wj) + l32;
    float sum = 0.f;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int64_t v0 = vbase + wave_row(a, wi) + 16 * jj;
        bf16x8 e8;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float e = exp2f_fast(__builtin_fmaf(acc[a][b][8 * jj + i], kLog2e, -m2));
          sum += e;
          e8[i] = (bf16)e;
        }
        if (store && v0 < p.V) st_bf16x8(p.E + tok * p.V + v0, e8);
      }
    }
    return half_sum(sum);
  };
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int col = wave_col(b, wj) + l32;
    const int64_t tok = j0 + col;
    const bool tv = tok < p.nc;
    // the label logit: held by at most one lane of the workgroup, for one
    // vocab tile in ~600 -- located with one range test per token
    const bool hit = tv && rel[b] >= 0 && ((rel[b] >> 6) & 1) == wi && ((rel[b] >> 3) & 1) == 0;
    if (__any(hit)) {
      const int r0 = rel[b] - 64 * wi;
      float zsel = 0.f;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (hit && r0 == wave_row(a, 0) + 16 * (r >> 3) + (r & 7)) zsel = acc[a][b][r];
      if (hit) p.zy[tok] = zsel;
    }
    const float sum = numerators(b, ref[b], p.store_e && tv);
    if (h == 0) red[wi * 256 + col] = sum;
  }
  __syncthreads();
  float tot[2];
  bool redo = false;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int col = wave_col(b, wj) + l32;
    const int64_t tok = j0 + col;
    tot[b] = red[col] + red[256 + col];
    redo |= tok < p.nc && !(tot[b] < kRefLimit);
    if (wi == 0 && h == 0 && tok < p.nc) p.spart[(int64_t)ti * p.ldp + tok] = tot[b];
  }
  if (!__syncthreads_or(redo)) return;
  // columns whose reference is too low: the same relative to the tile's maximum
  float mt[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float mx = -INFINITY;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, acc[a][b][r]);
    // log2 units (scaling by log2 e > 0 commutes with the max)
    mx = half_max(mx) * kLog2e;
    if (h == 0) red[wi * 256 + wave_col(b, wj) + l32] = mx;
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 2; ++b) mt[b] = fmaxf(red[wave_col(b, wj) + l32], red[256 + wave_col(b, wj) + l32]);
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int col = wave_col(b, wj) + l32;
    const bool bad = j0 + col < p.nc && !(tot[b] < kRefLimit);
    const float sum = numerators(b, mt[b], p.store_e && bad);
    if (h == 0) red[wi * 256 + col] = sum;
  }
  __syncthreads();
  if (wi == 0 && h == 0) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int col = wave_col(b, wj) + l32;
      const int64_t tok = j0 + col;
      if (tok < p.nc && !(tot[b] < kRefLimit)) {
        p.spart[(int64_t)ti * p.ldp + tok] = -(red[col] + red[256 + col]);
        p.mpart[(int64_t)ti * p.ldp + tok] = mt[b];
      }
    }
  }
}

// ---------------------------------------------------------------- row pass
struct RowArgs {
  const float* spart;    // [nvt, ldp] tile sums (negative: redone, relative to mpart)
  const float* mpart;
  const float* ref;      // [nc] row references (log2 units)
  const float* zy;
  const int64_t* y;      // chunk labels
  bf16* E;               // [nc, V]
  bf16* H;               // [nc, hdim] compacted rows: scaled by f (need_dw)
  float* f;              // [nc] factors of E
  float* wt;             // [nc] weights of the label terms
  float* loss_row;       // [nc] (chunk slice)
  const float* invden;
  const int64_t* nvalid;
  uint64_t* keys;        // [nsort, kIdChunk] rows sorted by label
  int32_t* slot;         // [V] cleared
  int64_t nc, nvt, V, hdim, c0, ldp;
  int nsort;             // sorting workgroups (0 without dW)
  int parts;             // workgroups per 64 rows
  int grads;             // 0: loss only (E was never stored)
};

// Workgroups [0, nsort) sort the chunk's labels; the others take 64 rows each,
// `parts` workgroups the same ones.  Sixteen waves read the rows' tile sums
// (lane = row, so each read is 256 contiguous bytes), added in a fixed order;
// that, and what is per row, every part does for itself.  What is per element
// (E of the rows with redone tiles, H scaled by f) is divided over the parts:
// few rows would otherwise leave it to a few CUs.  About as many workgroups as
// CUs (twice as many: up to 5% slower where rows are redone).  Measured, loss
// and dH, all rows redone, against one workgroup per 64 rows that took a row's
// tiles and its E one after the other: 512 x 1536 over 151936 columns 1.87 ->
// 0.58 ms, 2048 x 896 2.48 -> 1.17 ms, 16384 x 1536 13.5 -> 10.6 ms; no row
// redone: 0.52, 0.92 and 9.4 ms either way.
constexpr int kRowThreads = 1024, kRowRows = 64, kRowGroups = 256, kRowSeg = 64;
__global__ __launch_bounds__(kRowThreads) void flce_row_kernel(const RowArgs p) {
  constexpr int NWR = kRowThreads / 64, U = 8;
  __shared__ union {
    uint64_t sk[kIdChunk];
    struct {
      float sum[NWR][kRowRows], mx[NWR][kRowRows], redone[NWR][kRowRows], f[kRowRows], lse[kRowRows];
      int list[kRowRows], n;  // the rows with redone tiles
      float fac[kRowSeg][kRowRows];
    } r;
  } sh;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t nv = min(p.nc, *p.nvalid - p.c0);  // valid rows of the chunk
  if ((int)blockIdx.x < p.nsort) {
    const int64_t base = (int64_t)blockIdx.x * kIdChunk;
    const int len = (int)max((int64_t)0, min((int64_t)kIdChunk, nv - base));
    int np2 = 64;
    while (np2 < len) np2 <<= 1;
    for (int i = tid; i < np2; i += kRowThreads)
      sh.sk[i] = i < len ? ((uint64_t)p.y[base + i] << 32) | (uint32_t)i : kNoKey;
    __syncthreads();
    sort_keys(sh.sk, np2);
    for (int i = tid; i < kIdChunk; i += kRowThreads) p.keys[base + i] = i < np2 ? sh.sk[i] : kNoKey;
    return;
  }
  const int blk = (int)blockIdx.x - p.nsort, groups = ((int)gridDim.x - p.nsort) / p.parts;
  const int part = blk / groups;
  if (p.nsort > 0)
    for (int64_t v = (int64_t)blk * kRowThreads + tid; v < p.V; v += (int64_t)groups * p.parts * kRowThreads)
      p.slot[v] = 0;
  const int64_t r0 = (int64_t)(blk - part * groups) * kRowRows;
  if (r0 >= nv) return;
  const int64_t row = min(r0 + lane, nv - 1);
  const float rf = p.ref[row];
  float sum = 0.f;  // of the tiles relative to ref
  bool redone = false;
  for (int64_t t0 = w; t0 < p.nvt; t0 += NWR * U) {
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = t0 + NWR * u < p.nvt ? p.spart[(t0 + NWR * u) * p.ldp + row] : 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      redone |= s[u] < 0.f;
      sum += s[u] < 0.f ? 0.f : s[u];  // (a NaN too)
    }
  }
  sh.r.sum[w][lane] = sum;
  float top = rf;  // the reference of the sum
  if (__syncthreads_or(redone)) {
    // redone tiles: this wave's relative to their largest reference, then everything relative to the row's
    float mx = -INFINITY, s2 = 0.f;
    for (int64_t t0 = w; t0 < p.nvt; t0 += NWR * U) {
      float s[U], m[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t at = min(t0 + NWR * u, p.nvt - 1) * p.ldp + row;
        s[u] = p.spart[at];
        m[u] = p.mpart[at];
      }
      float top2 = mx;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        s[u] = t0 + NWR * u < p.nvt && s[u] < 0.f ? s[u] : 0.f;
        top2 = s[u] < 0.f ? fmaxf(top2, m[u]) : top2;
      }
      s2 = s2 > 0.f ? s2 * exp2f_fast(mx - top2) : 0.f;
      mx = top2;
#pragma unroll
      for (int u = 0; u < U; ++u) s2 -= s[u] < 0.f ? s[u] * exp2f_fast(m[u] - mx) : 0.f;
    }
    sh.r.mx[w][lane] = mx;
    sh.r.redone[w][lane] = s2;
    __syncthreads();
    mx = sh.r.mx[0][lane];
    for (int i = 1; i < NWR; ++i) mx = fmaxf(mx, sh.r.mx[i][lane]);
    redone = mx > -INFINITY;
    if (redone) top = fmaxf(rf, mx);
  }
  if (w == 0) {
    sum = sh.r.sum[0][lane];
    for (int i = 1; i < NWR; ++i) sum += sh.r.sum[i][lane];
    if (redone) {
      sum *= exp2f_fast(rf - top);
      for (int i = 0; i < NWR; ++i)
        if (sh.r.redone[i][lane] > 0.f) sum += sh.r.redone[i][lane] * exp2f_fast(sh.r.mx[i][lane] - top);
    }
    const float lse2 = top + __log2f(sum);
    const bool mine = r0 + lane < nv && part == 0;
    if (mine) p.loss_row[row] = lse2 * kLn2 - p.zy[row];
    if (p.grads) {
      // (a power of two in rows whose E is rounded once more below: then f H is exact)
      const float g = *p.invden;
      const float f = redone ? __builtin_ldexpf(1.f, __builtin_amdgcn_frexp_expf(g)) : exp2f_fast(top - lse2) * g;
      if (mine) {
        p.f[row] = f;
        p.wt[row] = (exp2f_fast(__builtin_fmaf(p.zy[row], kLog2e, -lse2)) - 1.f) * g;
        if (!redone) p.E[row * p.V + p.y[row]] = (bf16)0.f;
      }
      sh.r.f[lane] = f;
      sh.r.lse[lane] = lse2;
      const uint64_t m = __ballot(redone && r0 + lane < nv);
      if ((m >> lane) & 1) sh.r.list[__popcll(m & ((1ull << lane) - 1))] = lane;
      if (lane == 0) sh.r.n = __popcll(m);
    }
  }
  if (!p.grads) return;
  __syncthreads();
  // rows with redone tiles: E of every tile times what makes it the gradient over f (8 columns never straddle a
  // tile); this part's tiles, kRowSeg of them at a time, four rows at once
  constexpr int CT = 256, UE = 4;
  const float lse2 = sh.r.lse[lane], gm = __builtin_amdgcn_frexp_mantf(*p.invden);
  const int64_t tper = (p.nvt + p.parts - 1) / p.parts, te = min(p.nvt, (part + 1) * tper);
  for (int64_t tb = part * tper; sh.r.n > 0 && tb < te; tb += kRowSeg) {
    const int nt = (int)min((int64_t)kRowSeg, te - tb);
    float m[kRowSeg / NWR];
#pragma unroll
    for (int u = 0; u < kRowSeg / NWR; ++u) {
      const int64_t at = (tb + min(w + NWR * u, nt - 1)) * p.ldp + row;
      m[u] = p.mpart[at];
      m[u] = p.spart[at] < 0.f ? m[u] : rf;
    }
#pragma unroll
    for (int u = 0; u < kRowSeg / NWR; ++u) sh.r.fac[w + NWR * u][lane] = exp2f_fast(m[u] - lse2) * gm;
    __syncthreads();
    const int64_t c0 = tb * (kVT / 8);
    const int ne = (int)(min(p.V / 8, (tb + nt) * (kVT / 8)) - c0);
    for (int i = tid / CT; i < sh.r.n; i += kRowThreads / CT) {
      const int r = sh.r.list[i];
      const int64_t y = p.y[r0 + r] - 8 * c0;
      const int ych = y >= 0 && y < 8 * ne ? (int)y / 8 : -1, yq = (int)(y & 7);  // the label's place in the segment
      bf16* e = p.E + (r0 + r) * p.V + 8 * c0;
      for (int cc = tid % CT; cc < ne; cc += CT * UE) {
        bf16x8 x[UE];
#pragma unroll
        for (int u = 0; u < UE; ++u) x[u] = ld_bf16x8(e + 8 * min(cc + CT * u, ne - 1));
#pragma unroll
        for (int u = 0; u < UE; ++u) {
          const int c = cc + CT * u;
          if (c >= ne) break;
          const float k = sh.r.fac[c / (kVT / 8)][r];
#pragma unroll
          for (int q = 0; q < 8; ++q) x[u][q] = c == ych && q == yq ? (bf16)0.f : (bf16)((float)x[u][q] * k);
          st_bf16x8(e + 8 * c, x[u]);
        }
      }
    }
    __syncthreads();
  }
  if (p.nsort == 0) return;
  const int rows = (int)min((int64_t)kRowRows, nv - r0), gpr = (int)(p.hdim / 8);
  for (int i = part * kRowThreads + tid; i < rows * gpr; i += p.parts * kRowThreads) {
    const float f = sh.r.f[i / gpr];
    bf16* hp = p.H + r0 * p.hdim + 8 * (int64_t)i;
    bf16x8 x = ld_bf16x8(hp);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = (bf16)((float)x[k] * f);
    st_bf16x8(hp, x);
  }
}

// Label terms of dW: for each label of the chunk, the sums of w H over its
// rows in fp32, up to kLabelRound rows of one sorted run to a sum.  A sum lies
// in the slot of its first sorted key; a label's first one is in slot[label],
// the next one in next[its slot] (slots + 1; 0: none), so dW adds them in a
// fixed order.  One workgroup per key, of which those that start no sum return
// at once: a label that holds many rows has as many workgroups as sums.  (With
// one workgroup a label, loss, dH and dW of 16384 x 320 over 32008 columns, 11455
// rows of one label: 2.99 ms, 1.37 now; this kernel, labels Zipf-distributed,
// 6912 of 16384 rows x 1536 a call: 54 and 38 us.)  The sum's rows are listed
// one per thread; wave k adds rows k, k + 4, ..., eight in flight, and the
// waves' sums are added in order at the end.
constexpr int kLabelRound = 256;
struct LabelArgs {
  const uint64_t* keys;  // [nsort, kIdChunk]
  const bf16* H;         // [n, hdim] all rows, unscaled
  const int32_t* rows;   // chunk's compacted row -> row of H
  const float* wt;       // [nc]
  float* lsum;           // [nsort * kIdChunk (rows that exist), hdim]
  int32_t* slot;         // [V]
  int32_t* next;         // [nsort * kIdChunk]
  int64_t hdim;
  int nsort;
};
__global__ __launch_bounds__(256) void flce_label_kernel(const LabelArgs p) {
  constexpr int U = 3, R = 8, NWL = 4;
  static_assert(kLabelRound == 64 * NWL, "a thread per listed row");
  __shared__ int32_t row_sh[kLabelRound];
  __shared__ float wt_sh[kLabelRound];
  __shared__ __align__(16) float part_sh[NWL - 1][U * 64 * 8];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t item = blockIdx.x;
  const int c = (int)(item / kIdChunk), i = (int)(item % kIdChunk);
  const uint64_t* kc = p.keys + (int64_t)c * kIdChunk;
  const uint64_t key = kc[i];
  if (key == kNoKey) return;
  const uint32_t v = (uint32_t)(key >> 32);
  auto same = [&](int at) { return (uint32_t)(kc[at] >> 32) == v; };
  if (i > 0 && same(i - 1) && (i < kLabelRound || !same(i - kLabelRound))) return;  // inside the run's first round
  // the label's runs: this one, whether an earlier one exists, and the first key of the next later one
  int first = 0, end = 0;
  bool earlier = false;
  int32_t later = 0;
  for (int g0 = 0; g0 < p.nsort && later == 0; g0 += 64) {
    int2 r = make_int2(0, 0);
    if (g0 + lane < p.nsort) r = id_run(p.keys + (int64_t)(g0 + lane) * kIdChunk, v);
    const uint64_t has = __ballot(r.y > r.x);
    const int q = c - g0;  // this run's lane
    if (q >= 0 && q < 64) {
      first = __builtin_amdgcn_readlane(r.x, q);
      end = __builtin_amdgcn_readlane(r.y, q);
    }
    const uint64_t before = q >= 64 ? ~0ull : q > 0 ? (1ull << q) - 1 : 0ull;
    earlier |= (has & before) != 0;
    const uint64_t after = q < 0 ? has : q >= 63 ? 0ull : has & (~0ull << (q + 1));
    if (after != 0) {
      const int l = (int)__builtin_ctzll(after);
      later = (int32_t)((g0 + l) * kIdChunk + __builtin_amdgcn_readlane(r.x, l)) + 1;
    }
  }
  if ((i - first) % kLabelRound != 0) return;
  const int have = min(kLabelRound, end - i);
  if (tid == 0) {
    p.next[item] = i + kLabelRound < end ? (int32_t)item + kLabelRound + 1 : later;
    if (i == first && !earlier) p.slot[v] = (int32_t)item + 1;
  }
  if (tid < have) {
    const uint32_t k = (uint32_t)(c * kIdChunk) + (uint32_t)kc[i + tid];
    row_sh[tid] = p.rows[k];
    wt_sh[tid] = p.wt[k];
  }
  __syncthreads();
  const int64_t nvec = p.hdim / 8;
  for (int64_t p0 = 0; p0 < nvec; p0 += 64 * U) {
    float acc[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[u][e] = 0.f;
    for (int t0 = w; t0 < have; t0 += NWL * R) {
      bf16x8 x[R][U];
      float wr[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int t = min(t0 + NWL * r, have - 1);
        wr[r] = wt_sh[t];
        const bf16* src = p.H + (int64_t)row_sh[t] * p.hdim;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (p0 + 64 * u >= nvec) break;
          const int64_t ch = min(p0 + 64 * u + lane, nvec - 1);
          x[r][u] = ld_bf16x8(src + 8 * ch);
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (t0 + NWL * r >= have) break;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (p0 + 64 * u >= nvec) break;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[u][e] = __builtin_fmaf(wr[r], (float)x[r][u][e], acc[u][e]);
        }
      }
    }
    if (w > 0) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) part_sh[w - 1][(u * 64 + lane) * 8 + e] = acc[u][e];
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t ch = p0 + 64 * u + lane;
        if (ch >= nvec) continue;
#pragma unroll
        for (int k = 0; k < NWL - 1; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[u][e] += part_sh[k][(u * 64 + lane) * 8 + e];
        float* dst = p.lsum + item * p.hdim + 8 * ch;
        *reinterpret_cast<f32x4*>(dst) = f32x4{acc[u][0], acc[u][1], acc[u][2], acc[u][3]};
        *reinterpret_cast<f32x4*>(dst + 4) = f32x4{acc[u][4], acc[u][5], acc[u][6], acc[u][7]};
      }
    }
    __syncthreads();  // part_sh is read no more
  }
}

// ---------------------------------------------------------------- dH
struct DhArgs {
  GOp Wt;        // W [V, hdim] read as A[i = h][k = v]
  GOp E;         // [nc, V] read as B[j = tok][k = v]
  bf16* dh;      // dhidden [n, hdim]
  float* part;   // [slots][prow][hdim] partial sums (DhTiles; none when splits == 1)
  const float* f;         // [nc] row factors, label weights, labels
  const float* wt;
  const int64_t* y;
  const int32_t* rows;    // compacted row -> original row (whole batch)
  const int64_t* nvalid;
  int64_t hdim, nc, c0;
  int nI, splits, prow, run;  // hdim tiles; vocab ranges; rows of a slot; dh_run
};

// dH work: a unit is one (token tile, vocab range); its nI hdim tiles share
// the unit's E slab, so they run as consecutive blocks on one XCD (block b
// runs on XCD b % 8).  Units are dealt out over the XCDs in turn, ranges of a
// token tile on different XCDs.  With 8 ranges an XCD has one range of every
// token tile, and a last round of a few of its workgroups (32 run at a time)
// would leave the others idle: 27 token tiles x 6 hdim tiles are 5 rounds and
// 2 workgroups.  So the token tiles past the last whole round have their ranges
// cut into kDhSub parts.  With fewer ranges (more than 292 tiles: eight rounds
// or more) nothing is cut.  Measured, whole calls on one card: loss, dH and dW
// of 16384 rows, 11455 valid, x 1536 13.31 -> 13.05 ms; loss and dH of 4099
// rows, 2870 valid, x 896 1.57 -> 1.50 ms.
//
// A row's partial sums, and with them its last bits, must not depend on the
// caller's chunk.  So token tiles are those of the batch's counted rows, not of
// the chunk's (a chunk that starts inside one has the rest of it), and the
// "rounds" are those of runs of dh_run tiles, the default chunk: a tile is cut
// or not by its place in its run and by the batch's valid-row count, on the
// device.
constexpr int kDhSub = 4, kXcdSlots = 32;
// Splits of the dH vocab reduction: enough WGs to fill the chip several
// rounds over, bounded by the size of the fp32 partial sums.
int dh_splits(int64_t hdim, int64_t chunk) {
  const int64_t tiles = ((hdim + BI - 1) / BI) * ((chunk + BJ - 1) / BJ);
  int64_t s = (2048 + tiles - 1) / tiles;
  if (s < 1) s = 1;
  if (s > kXcds) s = kXcds;
  return (int)s;
}
// Token tiles whose E takes 2 GiB (the Python entry's default chunk).
int dh_run(int64_t V) { return (int)std::max<int64_t>((int64_t(1) << 31) / (2 * BJ * V), 1); }

// The token tiles of the rows [c0, c0 + nv), and where their partial sums lie:
// splits slots for a tile with whole ranges, kDhSub times 8 for one with cut
// ranges, in tile order.
struct DhTiles {
  int t0, t1;       // first tile, and past the last one
  int run, nj;      // tiles of a run; of the batch
  int full, last;   // cut tiles of a whole run, of the last one
  __device__ __forceinline__ int cut_before(int t) const {
    const int g = t / run, i = t - g * run, whole = nj / run;
    return g * full + max(0, g < whole ? i - (run - full) : i - (nj - whole * run - last));
  }
  // units of 8 slots before tile t (8 ranges)
  __device__ __forceinline__ int at(int t) const { return t - t0 + (kDhSub - 1) * (cut_before(t) - cut_before(t0)); }
  __device__ __forceinline__ bool cut(int t) const { return cut_before(t + 1) > cut_before(t); }
};
__device__ __forceinline__ DhTiles dh_tiles(int64_t nvalid, int64_t c0, int64_t nv, int nI, int splits, int run) {
  DhTiles T;
  T.t0 = (int)(c0 / BJ);
  T.t1 = nv > 0 ? (int)((c0 + nv + BJ - 1) / BJ) : T.t0;
  T.run = run;
  T.nj = (int)((nvalid + BJ - 1) / BJ);
  auto cut = [&](int n) {  // the tiles past the last whole round
    return splits == kXcds ? min(n, (int)(((int64_t)n * nI % kXcdSlots + nI - 1) / nI)) : 0;
  };
  T.full = cut(run);
  T.last = cut(T.nj % run);
  return T;
}
// Slots, also units, that the rows [c0, c0 + nc) can need.
int64_t dh_slots(int64_t c0, int64_t nc, int nI, int splits, int run) {
  const int64_t t0 = c0 / BJ, t1 = (c0 + nc + BJ - 1) / BJ, tiles = t1 - t0;
  if (splits < kXcds) return tiles * splits;
  const int64_t cut = std::min<int64_t>(run, (kXcdSlots - 1 + nI - 1) / nI) * ((t1 - 1) / run - t0 / run + 1);
  return kXcds * (tiles + (kDhSub - 1) * std::min(tiles, cut));
}

__global__ __launch_bounds__(NT) void flce_dh_kernel(const DhArgs p) {
  __shared__ __align__(16) bf16 smem[SMEM];
  const int64_t nv = min(p.nc, *p.nvalid - p.c0);
  const DhTiles T = dh_tiles(*p.nvalid, p.c0, nv, p.nI, p.splits, p.run);
  const int x = (int)(blockIdx.x % kXcds), k = (int)(blockIdx.x / kXcds);
  const int ti = k % p.nI, u = k / p.nI, unit = x + kXcds * u, slot = unit;
  // k-steps of the unit's range, or part of one
  const int64_t S = (p.E.cols + BK - 1) / BK, per = (S + p.splits - 1) / p.splits;
  int t;
  int64_t sb, se;
  if (p.splits < kXcds) {
    t = T.t0 + unit / p.splits;
    if (t >= T.t1) return;
    sb = (unit % p.splits) * per;
    se = min(S, sb + per);
  } else {
    if (T.t1 == T.t0 || u >= T.at(T.t1)) return;
    t = T.t0;  // the tile whose units u is among
    for (int end = T.t1; end - t > 1;) {
      const int mid = (t + end) / 2;
      if (T.at(mid) <= u)
        t = mid;
      else
        end = mid;
    }
    sb = x * per;
    se = min(S, sb + per);
    if (T.cut(t)) {
      const int64_t sub = (per + kDhSub - 1) / kDhSub;
      sb += (u - T.at(t)) * sub;
      se = min(se, sb + sub);
    }
  }
  const int64_t i0 = (int64_t)ti * BI, j0 = max((int64_t)t * BJ - p.c0, (int64_t)0);
  const int64_t j1 = min((int64_t)(t + 1) * BJ - p.c0, nv);  // the tile's rows of the chunk: j0 .. j1 - 1
  f32x16 acc[4][2];
  // (an empty range, of a vocabulary of few steps, leaves zeros)
  gemm_core<false, true, true>(smem, p.Wt, p.E, i0, j0, sb * BK, min(p.E.cols, se * BK), acc);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int wi = w & 1, wj = w >> 1;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int r = wave_col(b, wj) + l32;
    const int64_t tok = j0 + r;
    if (tok >= j1) continue;
    const int64_t orow = p.splits == 1 ? p.rows[p.c0 + tok] : 0;
    const float f = p.splits == 1 ? p.f[tok] : 0.f, wt = p.splits == 1 ? p.wt[tok] : 0.f;
    const bf16* wy = p.Wt.base + (p.splits == 1 ? p.y[tok] : 0) * p.hdim;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int64_t hh = i0 + wave_row(a, wi) + 16 * jj + 8 * h;
        if (hh >= p.hdim) continue;
        if (p.splits == 1) {
          const bf16x8 l = ld_bf16x8(wy + hh);
          bf16x8 o;
#pragma unroll
          for (int i = 0; i < 8; ++i) o[i] = (bf16)__builtin_fmaf(f, acc[a][b][8 * jj + i], wt * (float)l[i]);
          st_bf16x8(p.dh + orow * p.hdim + hh, o);
        } else {
          float* dst = p.part + ((int64_t)slot * p.prow + r) * p.hdim + hh;
          f32x4 lo, hi;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            lo[i] = acc[a][b][8 * jj + i];
            hi[i] = acc[a][b][8 * jj + 4 + i];
          }
          *reinterpret_cast<f32x4*>(dst) = lo;
          *reinterpret_cast<f32x4*>(dst + 4) = hi;
        }
      }
  }
}

// dH rows of the chunk: f times the fp32 partial sums of the row's token tile,
// added in slot order, plus the label term w W[y]; each compacted row written
// to its original row.
__global__ __launch_bounds__(256) void flce_dh_sum_kernel(const DhArgs p) {
  constexpr int U = 4;  // partial sums in flight
  const int64_t nv = min(p.nc, *p.nvalid - p.c0);
  const DhTiles T = dh_tiles(*p.nvalid, p.c0, nv, p.nI, p.splits, p.run);
  const int64_t gpr = p.hdim / 8, stride = p.prow * p.hdim;  // groups of 8 elements, hdim / 8 per row
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nv * gpr; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / gpr, col = 8 * (i - r * gpr);
    const int t = (int)((p.c0 + r) / BJ);
    const int64_t j0 = max((int64_t)t * BJ - p.c0, (int64_t)0);
    const int nslots = T.cut(t) ? kDhSub * kXcds : p.splits;
    const int64_t slot0 = p.splits < kXcds ? (t - T.t0) * p.splits : kXcds * T.at(t);
    const float* src = p.part + (r - j0) * p.hdim + col + stride * slot0;
    const bf16x8 l = ld_bf16x8(p.Wt.base + p.y[r] * p.hdim + col);
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    for (int s = 0; s < nslots; s += U, src += U * stride) {
      f32x4 lo[U], hi[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < nslots) {
          lo[u] = *reinterpret_cast<const f32x4*>(src + u * stride);
          hi[u] = *reinterpret_cast<const f32x4*>(src + u * stride + 4);
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < nslots) {
          a += lo[u];
          b += hi[u];
        }
    }
    const float f = p.f[r], wt = p.wt[r];
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o[k] = (bf16)__builtin_fmaf(f, a[k], wt * (float)l[k]);
      o[4 + k] = (bf16)__builtin_fmaf(f, b[k], wt * (float)l[4 + k]);
    }
    st_bf16x8(p.dh + (int64_t)p.rows[p.c0 + r] * p.hdim + col, o);
  }
}

// ---------------------------------------------------------------- dW
struct DwArgs {
  GOp Ht;        // hidden rows of the chunk [nc, hdim], scaled by f, read as A[i = h][k = tok]
  GOp Et;        // E [nc, V] read as B[j = v][k = tok]
  const int32_t* slot;   // [V] label terms: row of lsum + 1, or 0
  const int32_t* next;   // [rows] the label's next row of lsum + 1, or 0
  const float* lsum;     // [rows, hdim]
  bf16* dw;      // [V, hdim]
  float* acc32;  // [V, hdim] fp32 accumulator across chunks
  const int64_t* nvalid;
  int64_t hdim, V, c0, chunk;
  int nI, nJ;
};

__global__ __launch_bounds__(NT) void flce_dw_kernel(const DwArgs p) {
  __shared__ __align__(16) bf16 smem[SMEM];
  int ti, tj;
  if (!tile_of(p.nI, p.nJ, p.nI, ti, tj)) return;
  const int64_t i0 = (int64_t)ti * BI, j0 = (int64_t)tj * BJ;
  // The chunk's part in the sum over chunks, from the valid-row count: the
  // first chunk starts it, the one holding the last valid row finishes it
  // (bf16 store), chunks past it do nothing.  A single chunk (or no valid
  // row at all) stores bf16 directly.  Over two chunks the first one's sum is
  // kept in dW itself, in bf16, and the second adds to it: dW is rounded
  // twice, and the fp32 [V, hdim] round trip (twice dW's size, written and
  // read back) is saved.  Over more chunks the sum stays in fp32.
  // mode 0: bf16 store; 1: fp32 store; 2: fp32 add; 3: fp32 add + bf16
  // store; 4: bf16 add.
  const int64_t nvt_all = *p.nvalid;
  if (p.c0 > 0 && p.c0 >= nvt_all) return;
  const bool last = p.c0 + p.chunk >= nvt_all;
  const bool two = nvt_all <= 2 * p.chunk;
  const int mode = p.c0 == 0 ? (last || two ? 0 : 1) : (two ? 4 : (last ? 3 : 2));
  // tokens past the last 64-row step with a valid row are skipped (those up to
  // it are zero rows: flce_gather_kernel)
  const int64_t nv = nvt_all - p.c0;
  const int64_t ke = min(p.Ht.rows, nv > 0 ? ((nv + BK - 1) / BK) * BK : (int64_t)0);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int wi = w & 1, wj = w >> 1;
  int slot[2];  // of the columns' first label sum (loaded while there is a product to wait for)
#pragma unroll
  for (int b = 0; b < 2; ++b) slot[b] = nv > 0 ? p.slot[min(j0 + wave_col(b, wj) + l32, p.V - 1)] : 0;
  f32x16 acc[4][2];
  gemm_core<false, false, true>(smem, p.Ht, p.Et, i0, j0, 0, ke, acc);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int64_t v = j0 + wave_col(b, wj) + l32;
    if (v >= p.V) continue;
    for (int sl = slot[b]; sl > 0; sl = p.next[sl - 1]) {
      const float* lt = p.lsum + (int64_t)(sl - 1) * p.hdim + i0 + 8 * h;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const int64_t ho = wave_row(a, wi) + 16 * jj;
          if (i0 + 8 * h + ho >= p.hdim) continue;
          const f32x4 lo = *reinterpret_cast<const f32x4*>(lt + ho), hi = *reinterpret_cast<const f32x4*>(lt + ho + 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            acc[a][b][8 * jj + i] += lo[i];
            acc[a][b][8 * jj + 4 + i] += hi[i];
          }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int64_t hh = i0 + wave_row(a, wi) + 16 * jj + 8 * h;
        if (hh >= p.hdim) continue;
        f32x4 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lo[i] = acc[a][b][8 * jj + i];
          hi[i] = acc[a][b][8 * jj + 4 + i];
        }
        float* a32 = p.acc32 + v * p.hdim + hh;
        if (mode == 2 || mode == 3) {
          lo += *reinterpret_cast<const f32x4*>(a32);
          hi += *reinterpret_cast<const f32x4*>(a32 + 4);
        } else if (mode == 4) {
          const bf16x8 prev = ld_bf16x8(p.dw + v * p.hdim + hh);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            lo[i] += (float)prev[i];
            hi[i] += (float)prev[4 + i];
          }
        }
        if (mode == 1 || mode == 2) {
          *reinterpret_cast<f32x4*>(a32) = lo;
          *reinterpret_cast<f32x4*>(a32 + 4) = hi;
        } else {
          bf16x8 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            o[i] = (bf16)lo[i];
            o[4 + i] = (bf16)hi[i];
          }
          st_bf16x8(p.dw + v * p.hdim + hh, o);
        }
      }
  }
}

// ---------------------------------------------------------------- scalars
// Valid rows in order, compacted: rows[k] = the k-th row whose label counts,
// *nvalid = *count = their number; *bad = the labels out of range; *invden =
// what the loss is multiplied by.  One workgroup; per round 16 chunks of 1024
// labels are loaded at once, each wave ballots its valid lanes, and one prefix
// over the 256 (chunk, wave) counts places every valid row.  (The counts had a
// kernel of their own: one launch of a small call's ten, 5 us, and 12 us of
// kernel time at 16384 rows.)
__global__ __launch_bounds__(1024) void flce_compact_kernel(const int64_t* __restrict__ y, int64_t n, int64_t V,
                                                            int64_t ignore_index, int reduction,
                                                            const float* __restrict__ divisor,
                                                            int32_t* __restrict__ rows, int64_t* __restrict__ nvalid,
                                                            int64_t* __restrict__ count, int64_t* __restrict__ bad,
                                                            float* __restrict__ invden) {
  constexpr int CT = 1024, NWV = CT / 64, PER = 16;
  static_assert(PER * NWV == 256, "one (chunk, wave) count per lane quarter");
  __shared__ int cnt_sh[PER * NWV];  // valid rows of (chunk i, wave w) at i * NWV + w, in row order
  __shared__ long long carry_sh, bad_sh[NWV];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  long long nbad = 0;  // of this wave
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;  // lanes before this one
  if (tid == 0) carry_sh = 0;
  __syncthreads();
  for (int64_t c0 = 0; c0 < n; c0 += (int64_t)CT * PER) {
    int64_t v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int64_t r = c0 + (int64_t)i * CT + tid;
      v[i] = r < n ? y[r] : ignore_index;
    }
    uint64_t m[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      m[i] = __ballot(v[i] != ignore_index && v[i] >= 0 && v[i] < V);
      nbad += __popcll(__ballot(v[i] != ignore_index && !(v[i] >= 0 && v[i] < V)));
      if (lane == 0) cnt_sh[i * NWV + wv] = __popcll(m[i]);
    }
    __syncthreads();
    // exclusive prefix of the 256 counts in row order: lane l holds entries 4 l .. 4 l + 3
    const int a0 = cnt_sh[4 * lane], a1 = cnt_sh[4 * lane + 1], a2 = cnt_sh[4 * lane + 2], a3 = cnt_sh[4 * lane + 3];
    const int lsum = a0 + a1 + a2 + a3;
    int incl = lsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    const int total = __shfl(incl, 63);
    // entry i * NWV + wv sits in lane 4 i + wv / 4 at position wv % 4 (the same position for every i)
    const int k = wv & 3;
    const int mine = incl - lsum + (k > 0 ? a0 : 0) + (k > 1 ? a1 : 0) + (k > 2 ? a2 : 0);
    const long long carry = carry_sh;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const long long r = carry + __shfl(mine, 4 * i + (wv >> 2)) + __popcll(m[i] & below);
      if ((m[i] >> lane) & 1) rows[r] = (int32_t)(c0 + (int64_t)i * CT + tid);
    }
    __syncthreads();
    if (tid == 0) carry_sh += total;
    __syncthreads();
  }
  if (lane == 0) bad_sh[wv] = nbad;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < NWV; ++i) nbad += bad_sh[i];
    *nvalid = *count = carry_sh;
    *bad = nbad;
    *invden = reduction == 0 ? 1.f / (float)carry_sh : 1.f / *divisor;
  }
}

// The compacted operands: Hc[k] = H[rows[k]], yc[k] = y[rows[k]] and the row's
// reference, its label logit in log2 units, for k < nvalid; zero rows,
// ignore_index and 0 after them, up to the next multiple of 256 and at least
// BK - 1 of them: dW reduces over whole k-steps counted from the chunk's first
// row, wherever that lies, so its last one reads up to BK - 1 rows past the
// valid ones.  And dH = 0 on every row whose label does not count.  One wave
// per row, 16 bytes per lane per step.
__global__ __launch_bounds__(256) void flce_gather_kernel(const bf16* __restrict__ H, const bf16* __restrict__ W,
                                                          const int64_t* __restrict__ y,
                                                          const int32_t* __restrict__ rows,
                                                          const int64_t* __restrict__ nvalid, int64_t n, int64_t hdim,
                                                          int64_t V, int64_t ignore_index, bf16* __restrict__ Hc,
                                                          int64_t* __restrict__ yc, float* __restrict__ ref,
                                                          bf16* __restrict__ dh) {
  const int lane = threadIdx.x & 63;
  const int64_t nvec = hdim / 8, nv = *nvalid;
  const int64_t npad = min(((n + 255) / 256) * 256, max(((nv + 255) / 256) * 256, nv + BK - 1));
  const int64_t wstep = (int64_t)gridDim.x * 4;
  for (int64_t k = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); k < npad; k += wstep) {
    const bool real = k < nv;
    const int64_t src = real ? rows[k] : 0;
    const int64_t yk = real ? y[src] : ignore_index;
    float dot = 0.f;
    for (int64_t c = lane; c < nvec; c += 64) {
      const bf16x8 x = real ? ld_bf16x8(H + src * hdim + 8 * c) : zero_bf16x8();
      if (real) {
        const bf16x8 wy = ld_bf16x8(W + yk * hdim + 8 * c);
#pragma unroll
        for (int i = 0; i < 8; ++i) dot = __builtin_fmaf((float)x[i], (float)wy[i], dot);
      }
      st_bf16x8(Hc + k * hdim + 8 * c, x);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o);
    if (lane == 0) {
      yc[k] = yk;
      ref[k] = dot * kLog2e;
    }
  }
  if (dh == nullptr) return;  // loss only
  for (int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); t < n; t += wstep) {
    const int64_t v = y[t];
    if (v != ignore_index && v >= 0 && v < V) continue;
    for (int64_t c = lane; c < nvec; c += 64) st_bf16x8(dh + t * hdim + 8 * c, zero_bf16x8());
  }
}

__global__ __launch_bounds__(1024) void flce_loss_kernel(const float* __restrict__ loss_row, int64_t n,
                                                         const int64_t* __restrict__ nvalid,
                                                         const float* __restrict__ invden, float* loss) {
  __shared__ float sm[1024];
  float acc = 0.f;
  const int64_t nv = min(n, *nvalid);
  for (int64_t i = threadIdx.x; i < nv; i += 1024) acc += loss_row[i];
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 512; s >= 1; s >>= 1) {
    if ((int)threadIdx.x < s) sm[threadIdx.x] += sm[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = sm[0] * *invden;
}

// y = x * scalar in bf16 (rounded once from fp32).  x == y scales in place,
// and then an exact 1.0 returns at once; out of place it is a copy.
__global__ __launch_bounds__(256) void scale_bf16_kernel(const bf16* x, bf16* y, int64_t nvec, int64_t numel,
                                                         const float* __restrict__ scalar) {
  const float s = *scalar;
  if (s == 1.f && x == y) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * 256) {
    if (8 * i + 8 <= numel) {
      bf16x8 v = ld_bf16x8(x + 8 * i);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (bf16)((float)v[k] * s);
      st_bf16x8(y + 8 * i, v);
    } else {
      for (int64_t k = 8 * i; k < numel; ++k) y[k] = (bf16)((float)x[k] * s);
    }
  }
}

__global__ __launch_bounds__(256) void zero_bf16_kernel(bf16* __restrict__ x, int64_t nvec) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * 256)
    *reinterpret_cast<u32x4*>(x + 8 * i) = u32x4{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------- workspace
struct Layout {
  size_t invden, loss_row, mpart, spart, zy, f, wt, E, part, acc32, rows, hc, yc, ref, keys, slot, next, lsum, total;
  int64_t chunk, nvt;
  int splits, prow, run;  // of dH: vocab ranges, rows of a slot, dh_run
  int nsort;  // sorted runs of a chunk's labels (dW only)
};

size_t al(size_t x) { return (x + 255) & ~size_t(255); }

// need_dh false: loss only (no E, no gradient buffers); its chunks only bound
// the per-(row, vocab tile) sum buffers, so they are large.
constexpr int64_t kLossChunk = 32768;

Layout layout(int64_t n, int64_t hdim, int64_t V, int64_t chunk, bool need_dh, bool need_dw) {
  Layout L{};
  if (!need_dh) {
    need_dw = false;
    chunk = kLossChunk;
  }
  L.chunk = chunk < n ? chunk : (n > 0 ? n : 1);
  L.nvt = (V + kVT - 1) / kVT;
  const int64_t nchunks = n > 0 ? (n + L.chunk - 1) / L.chunk : 0;
  size_t off = 0;
  L.invden = off;
  off += 256;
  L.loss_row = off;
  off += al(sizeof(float) * (size_t)(n > 0 ? n : 1));
  L.mpart = off;
  off += al(sizeof(float) * (size_t)(L.chunk * L.nvt));
  L.spart = off;
  off += al(sizeof(float) * (size_t)(L.chunk * L.nvt));
  L.zy = off;
  off += al(sizeof(float) * (size_t)L.chunk);
  L.f = off;
  if (need_dh) off += al(sizeof(float) * (size_t)L.chunk);
  L.wt = off;
  if (need_dh) off += al(sizeof(float) * (size_t)L.chunk);
  L.E = off;
  if (need_dh) off += al(sizeof(bf16) * (size_t)(L.chunk * V));
  L.part = off;
  L.splits = dh_splits(hdim, L.chunk);
  L.prow = (int)std::min<int64_t>(L.chunk, BJ);
  L.run = dh_run(V);
  if (need_dh && L.splits > 1) {
    int64_t slots = 0;
    for (int64_t c0 = 0; c0 < nchunks * L.chunk; c0 += L.chunk)
      slots = std::max(slots, dh_slots(c0, std::min(L.chunk, n - c0), (int)((hdim + BI - 1) / BI), L.splits, L.run));
    off += al(sizeof(float) * (size_t)(slots * L.prow * hdim));
  }
  L.acc32 = off;
  // the fp32 dW sum: only when the valid rows may span more than two chunks
  // (over two, the first chunk's sum is kept in dW itself)
  if (need_dw && nchunks > 2) off += al(sizeof(float) * (size_t)(V * hdim));
  const int64_t npad = ((n > 0 ? n : 1) + 255) / 256 * 256;
  L.rows = off;
  off += al(sizeof(int32_t) * (size_t)npad);
  L.hc = off;
  off += al(sizeof(bf16) * (size_t)(npad * hdim));
  L.yc = off;
  off += al(sizeof(int64_t) * (size_t)npad);
  L.ref = off;
  off += al(sizeof(float) * (size_t)npad);
  L.nsort = need_dw ? (int)((L.chunk + kIdChunk - 1) / kIdChunk) : 0;
  L.keys = off;
  off += al(sizeof(uint64_t) * (size_t)L.nsort * kIdChunk);
  L.slot = off;
  if (need_dw) off += al(sizeof(int32_t) * (size_t)V);
  L.next = off;
  off += al(sizeof(int32_t) * (size_t)L.nsort * kIdChunk);
  L.lsum = off;  // the label terms' sums, one row for each row of the chunk
  if (need_dw) off += al(sizeof(float) * (size_t)(L.chunk * hdim));
  L.total = off;
  return L;
}

}  // namespace

size_t flce_workspace_bytes(int64_t n, int64_t hdim, int64_t vocab, int64_t chunk, bool need_dh, bool need_dw) {
  if (chunk <= 0) return 0;
  return layout(n, hdim, vocab, chunk, need_dh, need_dw).total;
}

hipError_t flce_run(const FlceArgs& a, hipStream_t stream) {
  const bool grads = a.grads;
  const Layout L = layout(a.n, a.hdim, a.vocab, a.chunk, grads, grads && a.dweight != nullptr);
  char* ws = static_cast<char*>(a.ws);
  float* invden = reinterpret_cast<float*>(ws + L.invden);
  float* loss_row = reinterpret_cast<float*>(ws + L.loss_row);
  float* mpart = reinterpret_cast<float*>(ws + L.mpart);
  float* spart = reinterpret_cast<float*>(ws + L.spart);
  float* zy = reinterpret_cast<float*>(ws + L.zy);
  bf16* E = reinterpret_cast<bf16*>(ws + L.E);
  float* part = reinterpret_cast<float*>(ws + L.part);
  float* acc32 = reinterpret_cast<float*>(ws + L.acc32);
  int64_t* nvalid = reinterpret_cast<int64_t*>(ws + L.invden) + 1;
  int32_t* rows = reinterpret_cast<int32_t*>(ws + L.rows);
  bf16* hcomp = reinterpret_cast<bf16*>(ws + L.hc);
  int64_t* ycomp = reinterpret_cast<int64_t*>(ws + L.yc);
  float* ref = reinterpret_cast<float*>(ws + L.ref);
  float* frow = reinterpret_cast<float*>(ws + L.f);
  float* wrow = reinterpret_cast<float*>(ws + L.wt);
  uint64_t* keys = reinterpret_cast<uint64_t*>(ws + L.keys);
  int32_t* slot = reinterpret_cast<int32_t*>(ws + L.slot);
  int32_t* next = reinterpret_cast<int32_t*>(ws + L.next);
  float* lsum = reinterpret_cast<float*>(ws + L.lsum);
  const int64_t V = a.vocab, Hd = a.hdim;

  hipLaunchKernelGGL(flce_compact_kernel, dim3(1), dim3(1024), 0, stream, a.labels, a.n, V, a.ignore_index,
                     a.reduction, a.divisor, rows, nvalid, a.count, a.bad_labels, invden);
  if (a.n > 0) {
    int64_t blocks = (a.n + 3) / 4;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(flce_gather_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a.hidden, a.weight, a.labels, rows,
                       nvalid, a.n, Hd, V, a.ignore_index, hcomp, ycomp, ref, grads ? a.dhidden : nullptr);
  }
  // chunks of compacted rows: the host sizes them for n rows; those past the
  // valid count return at once
  const int64_t nchunks = a.n > 0 ? (a.n + L.chunk - 1) / L.chunk : 0;
  for (int64_t ci = 0; ci < nchunks; ++ci) {
    const int64_t c0 = ci * L.chunk;
    const int64_t nc = (a.n - c0) < L.chunk ? (a.n - c0) : L.chunk;
    bf16* Hc = hcomp + c0 * Hd;
    const int64_t* yc = ycomp + c0;

    LogitsArgs lg{};
    lg.W = GOp{a.weight, Hd, V, Hd};
    lg.H = GOp{Hc, Hd, nc, Hd};
    lg.y = yc;
    lg.ref = ref + c0;
    lg.E = E;
    lg.mpart = mpart;
    lg.spart = spart;
    lg.zy = zy;
    lg.nvalid = nvalid;
    lg.c0 = c0;
    lg.V = V;
    lg.nc = nc;
    lg.ldp = L.chunk;
    lg.nI = (int)L.nvt;
    lg.nJ = (int)((nc + BJ - 1) / BJ);
    lg.store_e = grads ? 1 : 0;
    {
      const int total = lg.nI * lg.nJ;
      const int grid = ((total + kXcds - 1) / kXcds) * kXcds;
      hipLaunchKernelGGL(flce_logits_kernel, dim3(grid), dim3(NT), 0, stream, lg);
    }

    RowArgs rw{};
    rw.mpart = mpart;
    rw.spart = spart;
    rw.ref = ref + c0;
    rw.zy = zy;
    rw.y = yc;
    rw.E = E;
    rw.H = Hc;
    rw.f = frow;
    rw.wt = wrow;
    rw.loss_row = loss_row + c0;
    rw.invden = invden;
    rw.nvalid = nvalid;
    rw.keys = keys;
    rw.slot = slot;
    rw.c0 = c0;
    rw.nc = nc;
    rw.nvt = L.nvt;
    rw.V = V;
    rw.hdim = Hd;
    rw.ldp = L.chunk;
    rw.nsort = L.nsort;
    rw.grads = grads ? 1 : 0;
    const int64_t groups = (nc + kRowRows - 1) / kRowRows;
    rw.parts = grads ? (int)std::max<int64_t>(kRowGroups / groups, 1) : 1;
    hipLaunchKernelGGL(flce_row_kernel, dim3((unsigned)(L.nsort + groups * rw.parts)), dim3(kRowThreads), 0, stream, rw);
    if (!grads) continue;
    auto label_sums = [&]() {
      LabelArgs la{};
      la.keys = keys;
      la.H = a.hidden;
      la.rows = rows + c0;
      la.wt = wrow;
      la.lsum = lsum;
      la.slot = slot;
      la.next = next;
      la.hdim = Hd;
      la.nsort = L.nsort;
      hipLaunchKernelGGL(flce_label_kernel, dim3((unsigned)nc), dim3(256), 0, stream, la);
    };
    // dH may take the place of the hidden states: then they are read before it is written (otherwise right before
    // dW, which finds the sums in the caches: 300 x 4096 over 128256 columns 1134 us, 1153 in the other order)
    const bool in_place = a.dhidden < a.hidden + a.n * Hd && a.hidden < a.dhidden + a.n * Hd;
    if (a.dweight != nullptr && in_place) label_sums();

    DhArgs dh{};
    dh.Wt = GOp{a.weight, Hd, V, Hd};
    dh.E = GOp{E, V, nc, V};
    dh.dh = a.dhidden;
    dh.part = part;
    dh.f = frow;
    dh.wt = wrow;
    dh.y = yc;
    dh.rows = rows;
    dh.nvalid = nvalid;
    dh.c0 = c0;
    dh.hdim = Hd;
    dh.nc = nc;
    dh.nI = (int)((Hd + BI - 1) / BI);
    dh.splits = L.splits;
    dh.prow = L.prow;
    dh.run = L.run;
    {
      const int64_t units = dh_slots(c0, nc, dh.nI, L.splits, L.run);
      const int64_t grid = kXcds * dh.nI * ((units + kXcds - 1) / kXcds);
      hipLaunchKernelGGL(flce_dh_kernel, dim3((unsigned)grid), dim3(NT), 0, stream, dh);
    }
    if (L.splits > 1) {
      const int64_t nvec = nc * Hd / 8;
      int64_t blocks = (nvec + 255) / 256;
      if (blocks > 4096) blocks = 4096;
      hipLaunchKernelGGL(flce_dh_sum_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, dh);
    }

    if (a.dweight != nullptr) {
      if (!in_place) label_sums();
      DwArgs dw{};
      dw.Ht = GOp{Hc, Hd, nc, Hd};
      dw.Et = GOp{E, V, nc, V};
      dw.slot = slot;
      dw.next = next;
      dw.lsum = lsum;
      dw.dw = a.dweight;
      dw.acc32 = acc32;
      dw.nvalid = nvalid;
      dw.c0 = c0;
      dw.hdim = Hd;
      dw.V = V;
      dw.nI = (int)((Hd + BI - 1) / BI);
      dw.nJ = (int)L.nvt;
      dw.chunk = L.chunk;
      const int total = dw.nI * dw.nJ;
      const int grid = ((total + kXcds - 1) / kXcds) * kXcds;
      hipLaunchKernelGGL(flce_dw_kernel, dim3(grid), dim3(NT), 0, stream, dw);
    }
  }
  if (grads && a.n == 0 && a.dweight != nullptr) {
    // no rows: d loss / d W is zero (a fill kernel, so the call stays graph-capturable)
    const int64_t nvec = V * Hd / 8;
    int64_t blocks = (nvec + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(zero_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a.dweight, nvec);
  }
  hipLaunchKernelGGL(flce_loss_kernel, dim3(1), dim3(1024), 0, stream, loss_row, a.n, nvalid, invden, a.loss);
  return hipGetLastError();
}

hipError_t launch_scale_bf16(const bf16* src, bf16* dst, int64_t numel, const float* scalar, hipStream_t stream) {
  const int64_t nvec = (numel + 7) / 8;
  int64_t blocks = (nvec + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(scale_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, src, dst, nvec, numel, scalar);
  return hipGetLastError();
}

}  // namespace siq
