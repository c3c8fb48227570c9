// Tiled bf16 GEMM core for gfx950 shared by the fused CE and the projector:
// C[i][j] = sum_k A[i][k] B[j][k] over 256 x 256 tiles, 8 waves, k-steps of
// 64 staged in LDS by direct global->LDS loads, operand reads with
// ds_read_b128 / ds_read_b64_tr_b16, v_mfma_f32_32x32x16_bf16.  The two waves
// of a SIMD take turns: while one multiplies, the other reads its next
// operands and issues loads (gemm_core_l).
#pragma once
#include "lds.h"

namespace siq {
namespace gemm {

constexpr int BI = 256, BJ = 256, BK = 64, NT = 512;
constexpr int NW = NT / 64;         // 8 waves: 2 along I x 4 along J
constexpr int HALF = 128 * BK;      // bf16 elements of one staged operand half (16 KB)
constexpr int SMEM = 8 * HALF;      // A lo / hi, B lo / hi, two k-steps each (128 KB)
constexpr int kXcds = 8;

struct GOp {
  const bf16* base;
  int64_t ld, rows, cols;  // element (r, c) at base[r * ld + c]; 16-byte chunks along c
};

// Output index (inside the tile) of accumulator tile a / b of a wave: a wave
// owns 64 rows of each A half (tiles a = 0, 1: the lower half, 2, 3: the
// upper) and 32 columns of each B half (b = 0, 1).  acc[a][b][r] holds
// i = i0 + wave_row(a, wi) + drow(r, h), j = j0 + wave_col(b, wj) + l32.
__device__ __forceinline__ int wave_row(int a, int wi) { return 128 * (a >> 1) + 64 * wi + 32 * (a & 1); }
__device__ __forceinline__ int wave_col(int b, int wj) { return 128 * b + 32 * wj; }

// Operand halves (128 M or N indices, one k-step) live in LDS in one of two
// orientations, both XOR-swizzled at 16-byte granularity so the MFMA operand
// reads are bank-conflict free (64 banks of 4 bytes):
//  * KC ("k contiguous"): [128 rows][64 k], 128-byte rows; the rows are the
//    operand's M (or N) index.  Read as row operands (one chunk from each of
//    16 consecutive rows per quarter-wave): swz_kc spreads 16 rows over
//    distinct (bank half, chunk) pairs.
//  * NKC: [64 k][128 cols], 256-byte rows; the columns are the operand's M (or
//    N) index.  Read with ds_read_b64_tr_b16 (4 aligned chunks from each of 4
//    consecutive rows per half-wave): swz_nkc XORs the row into bits 2-3 of
//    the chunk index, so the 16 positions land in 16 distinct bank groups.
__device__ __forceinline__ int swz_kc(int r) { return (((r >> 1) & 3) << 1) | ((r >> 3) & 1); }
__device__ __forceinline__ int swz_nkc(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Direct global->LDS staging of an operand half: 16 instructions of 1 KB, two
// per wave (instruction 2 w + q; KC: rows 16 w + 8 q .. + 7, lane / 8 inside;
// NKC: k rows 8 w + 4 q .. + 3, lane / 16 inside).  A row-major operand whose
// tile starts at M / N index r0.  Rows (KC) or chunks (NKC) past the operand's
// extent re-read the last valid one (always in bounds; what that produces is
// never stored): the lane offsets are clamped once, so every k-step issues
// from a uniform base without address arithmetic.
template <bool KC>
struct OpLoad {
  GOp op;
  const bf16* base;
  uint32_t off[2][2];  // [half][q] byte offset of this lane's chunk from the k-step's base
  __device__ __forceinline__ void init(const GOp& o, int64_t r0, int lane, int w) {
    op = o;
    base = KC ? o.base + r0 * o.ld : o.base + r0;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (KC) {
          const int r = 16 * w + 8 * q + lane / 8;
          const int gr = min(128 * hf + r, (int)min(o.rows - 1 - r0, (int64_t)255));
          off[hf][q] = 2 * (uint32_t)(gr * (int)o.ld + 8 * ((lane % 8) ^ swz_kc(r)));
        } else {
          const int r = 8 * w + 4 * q + lane / 16;
          const int gc = min(128 * hf + 8 * ((lane % 16) ^ swz_nkc(r)), (int)min(o.cols - 8 - r0, (int64_t)248));
          off[hf][q] = 2 * (uint32_t)(r * (int)o.ld + gc);
        }
      }
  }
  // half hf of the k-step starting at k0 (64 valid k)
  __device__ __forceinline__ void issue(int hf, int64_t k0, bf16* lds, int wu) const {
    const bf16* b = KC ? base + k0 : base + k0 * op.ld;
#pragma unroll
    for (int q = 0; q < 2; ++q) dma16(b, off[hf][q], lds + (2 * wu + q) * 512);
  }
  // the same with only the first kval (< 64; KC: a multiple of 8) k valid: the
  // others re-read the last valid ones and are zeroed in the B operand (ztail)
  __device__ __forceinline__ void issue_tail(int hf, int64_t k0, int kval, bf16* lds, int wu, int lane) const {
    const bf16* b = KC ? base + k0 : base + k0 * op.ld;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      uint32_t o = off[hf][q];
      if (KC) {
        const int c = 8 * ((lane % 8) ^ swz_kc(16 * wu + 8 * q + lane / 8));
        o -= 2 * (uint32_t)max(0, c - (kval - 8));
      } else {
        const int r = 8 * wu + 4 * q + lane / 16;
        o -= 2 * (uint32_t)(max(0, r - (kval - 1)) * (int)op.ld);
      }
      dma16(b, o, lds + (2 * wu + q) * 512);
    }
  }
};

// MFMA operand reads of a wave's 32-row tiles of an operand half, the first
// at half row (KC) / column (NKC) `base`: returns for lane l the 8 k values
// (16 ks + 8 h + i, i = 0..7) of operand row base + 32 t + rowmap(l % 32), with
// rowmap = perm32 when PERM (A operands: the product's rows then come out as 8
// consecutive indices per accumulator group) and the identity otherwise (B
// operands).
template <bool KC, bool PERM, int NTL>
struct HalfRead {
  uint32_t off[4][2];  // KC: [ks][-]; NKC: [t][e]
  __device__ __forceinline__ void init(int lane, int base) {
    const int l32 = lane & 31, h = lane >> 5;
    if (KC) {
      const int r = base + (PERM ? perm32(l32) : l32);
      const int f = swz_kc(r);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) off[ks][0] = (uint32_t)(r * BK + (((2 * ks + h) ^ f) << 3));
    } else {
      const int G = lane >> 4, p = lane & 15, j = p >> 2, q = p & 3;
      const int cs = PERM ? 16 * (G & 1) + 8 * (q & 1) + 4 * (q >> 1) : 16 * (G & 1) + 4 * q;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int r = 8 * (G >> 1) + j + 4 * e;  // row within a 16-row k group
        const int f = swz_nkc(r);
#pragma unroll
        for (int t = 0; t < NTL; ++t) {
          const int col = base + 32 * t + cs;
          off[t][e] = (uint32_t)(r * 128 + (((col >> 3) ^ f) << 3) + (col & 7));
        }
      }
    }
  }
  __device__ __forceinline__ bf16x8 read(const bf16* S, int t, int ks) const {
    if (KC) return ld_bf16x8(S + off[ks][0] + t * 32 * BK);
    const bf16* b = S + ks * 16 * 128;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(b + off[t][0]));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(b + off[t][1]));
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
};

// Zeroes the k tail of a staged B half (k >= kval) once it has landed: the
// loader filled it by re-reading the last valid k, and the product must not
// see that.  KC [128][64]: thread t owns row t / 4, logical chunks 2 (t % 4),
// + 1; NKC [64][128]: row t / 8, the same two chunks of 8 t % 8.
template <bool KC>
__device__ __forceinline__ void ztail_pass(bf16* S, int kval, int tid) {
  const int r = KC ? tid >> 2 : tid >> 3;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = KC ? 2 * (tid & 3) + k : 2 * (tid & 7) + k;
    bf16* ptr = S + (KC ? r * BK + 8 * (c ^ swz_kc(r)) : r * 128 + 8 * (c ^ swz_nkc(r)));
    if (KC ? 8 * c >= kval : r >= kval) st_bf16x8(ptr, zero_bf16x8());
  }
}

// Maps a 1-D block id onto (I tile, J tile).  Block b is dispatched to XCD
// b % 8, so each XCD gets a contiguous run of the linear tile order; inside it
// tiles go in groups of GI I-tiles (I fastest), so the 32 workgroups running
// together on an XCD cover about GI I-tiles x 32/GI J-tiles and both operands'
// slabs are shared through that XCD's L2.
__device__ __forceinline__ bool tile_of(int nI, int nJ, int GI, int& ti, int& tj) {
  const int total = nI * nJ;
  const int per = (total + kXcds - 1) / kXcds;
  const int lin = (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
  if (lin >= total) return false;
  const int g = lin / (GI * nJ), within = lin - g * GI * nJ;
  const int gsize = min(GI, nI - g * GI);
  ti = g * GI + within % gsize;
  tj = within / gsize;
  return true;
}

// C[i][j] = sum_k A[i][k] B[j][k] over k in [kb, ke) (kb, ke multiples of BK
// except ke at the operand's end), accumulators as described at wave_row.
//
// A k-step is four phases, one per quarter of the wave's accumulators (64 x 32
// outputs, 8 MFMAs): lower A x lower B, lower A x upper B, upper A x upper B,
// upper A x lower B.  Each phase is a memory part (the operand reads that the
// phase needs and has not in registers yet: A lower, B upper, A upper and, in
// the last, the next step's B lower, so 8, 4, 8, 4 16-byte reads; and the
// loads of one operand half) and a compute part, each ended by a barrier.
// Waves 4-7 run one barrier behind waves 0-3, and waves w and w + 4 share a
// SIMD: while one multiplies, the other reads and loads.  With the whole
// workgroup in step (all waves read, then all multiply, one barrier and a
// drained load queue per k-step) the matrix cores stood idle during the reads
// and at the drain: busy 51-61% of the time, 66-76% now, at a lower clock (1.6
// GHz against 1.8: the card's power limit, which now bounds the long products,
// as it does the library's: 1.49 PFLOP/s on random operands, 2.1 on zeros).
// Kernel times of both builds on one card: cross-entropy of 16384 rows (11467
// counted) x 1536, V = 151936, logits 5.08 -> 4.52 ms, dH 5.30 -> 4.25 (its last
// round cut finer besides), dW 4.57 -> 4.42 (1.21 PFLOP/s); projector 4096 x 4096
// x 1536, forward 69.5 -> 62.7 us, dX 51.8 -> 48.0, dW 76.2 -> 68.1.
//
// Loads: a half is read in one phase (p) only; its buffer is loaded again, for
// two steps later, in phase p + 2 (by then every wave, also one a barrier
// behind, has passed the compute part of phase p, which ends with a wait for
// the wave's LDS reads: those of B lower, read a phase before it is multiplied,
// have no other; they are back by then, so it costs nothing), and read six
// phases after that.  A wave waits, at the end of each memory part, for the
// half that the next phase reads (all but the ten newest load instructions),
// so the queue is never drained before the last two steps.
//
// LA / LB: issue(half, k0, lds, wu) loads half `half` of the k-step at k0 (two
// instructions a wave), issue_tail the last, partial step (TAIL = false: there
// is none, k is a multiple of 64).
template <bool AKC, bool BKC, bool TAIL, class LA, class LB>
__device__ __forceinline__ void gemm_core_l(bf16* smem, LA& la, LB& lb, int64_t kb, int64_t ke,
                                            f32x16 (&acc)[4][2]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wi = w & 1, wj = w >> 1;
  const int wu = __builtin_amdgcn_readfirstlane(w);
  HalfRead<AKC, true, 2> ra;
  HalfRead<BKC, false, 1> rb;
  ra.init(lane, 64 * wi);
  rb.init(lane, 32 * wj);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = zero16();
  const int64_t span = ke > kb ? ke - kb : 0;
  const int n = (int)(span / BK), kval = (int)(span - (int64_t)n * BK);
  auto As = [&](int hf, int buf) { return smem + (2 * hf + buf) * HALF; };
  auto Bs = [&](int hf, int buf) { return smem + (4 + 2 * hf + buf) * HALF; };
  bf16x8 af[2][4], b0[4], b1[4];  // A half in use; B halves
  auto read_a = [&](int hf, int buf) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t) af[t][ks] = ra.read(As(hf, buf), t, ks);
  };
  auto read_b = [&](bf16x8 (&bf)[4], int hf, int buf) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) bf[ks] = rb.read(Bs(hf, buf), 0, ks);
  };
  auto multiply = [&](const bf16x8 (&bf)[4], int a, int b) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[a + t][b] = mfma32(af[t][ks], bf[ks], acc[a + t][b]);
  };
  if (n > 0) {
    // in the order in which they are read
    lb.issue(0, kb, Bs(0, 0), wu);
    la.issue(0, kb, As(0, 0), wu);
    lb.issue(1, kb, Bs(1, 0), wu);
    la.issue(1, kb, As(1, 0), wu);
    if (n > 1) {
      lb.issue(0, kb + BK, Bs(0, 1), wu);
      la.issue(0, kb + BK, As(0, 1), wu);
      lb.issue(1, kb + BK, Bs(1, 1), wu);
      wait_vmcnt<10>();
    } else {
      wait_vmcnt<4>();
    }
    phase_barrier();
    read_b(b0, 0, 0);
    wait_lds();
    if (wu >= NW / 2) phase_barrier();
    // one k-step from buffer `buf`; bl holds its lower B half on entry, bu the next step's on exit
    auto step = [&](int s, int buf, bf16x8 (&bl)[4], bf16x8 (&bu)[4]) {
      const int rem = n - 1 - s;  // steps after this one
      const int64_t k1 = kb + (int64_t)(s + 1) * BK, k2 = k1 + BK;
      auto compute = [&](const bf16x8 (&bf)[4], int a, int b) {
        phase_barrier();
        __builtin_amdgcn_s_setprio(1);
        multiply(bf, a, b);
        __builtin_amdgcn_s_setprio(0);
        wait_lds();
        phase_barrier();
      };
      read_a(0, buf);
      if (rem >= 1) {
        la.issue(1, k1, As(1, buf ^ 1), wu);
        wait_vmcnt<10>();
      } else {
        wait_vmcnt<2>();
      }
      compute(bl, 0, 0);
      read_b(bu, 1, buf);
      if (rem >= 2) {
        lb.issue(0, k2, Bs(0, buf), wu);
        wait_vmcnt<10>();
      } else if (rem == 1) {
        wait_vmcnt<8>();
      } else {
        wait_vmcnt<0>();
      }
      compute(bu, 0, 1);
      read_a(1, buf);
      if (rem >= 2) {
        la.issue(0, k2, As(0, buf), wu);
        wait_vmcnt<10>();
      } else if (rem == 1) {
        wait_vmcnt<6>();
      }
      compute(bu, 2, 1);
      if (rem >= 1) read_b(bu, 0, buf ^ 1);
      if (rem >= 2) {
        lb.issue(1, k2, Bs(1, buf), wu);
        wait_vmcnt<10>();
      } else if (rem == 1) {
        wait_vmcnt<4>();
      }
      compute(bl, 2, 0);
    };
    int s = 0;
    for (; s + 1 < n; s += 2) {
      step(s, 0, b0, b1);
      step(s + 1, 1, b1, b0);
    }
    if (s < n) step(s, 0, b0, b1);
    if (wu < NW / 2) phase_barrier();  // both groups have met the same number of barriers
  }
  __syncthreads();
  if constexpr (TAIL) {
    if (kval > 0) {
      const int64_t k0 = kb + (int64_t)n * BK;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        la.issue_tail(hf, k0, kval, As(hf, 0), wu, lane);
        lb.issue_tail(hf, k0, kval, Bs(hf, 0), wu, lane);
      }
      wait_vmcnt<0>();
      __syncthreads();
      ztail_pass<BKC>(Bs(0, 0), kval, tid);
      ztail_pass<BKC>(Bs(1, 0), kval, tid);
      __syncthreads();
      read_b(b0, 0, 0);
      read_b(b1, 1, 0);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        read_a(hf, 0);
        multiply(b0, 2 * hf, 0);
        multiply(b1, 2 * hf, 1);
      }
      __syncthreads();
    }
  }
}

// gemm_core_l over two row-major operands, tile (i0, j0).
template <bool AKC, bool BKC, bool TAIL>
__device__ __forceinline__ void gemm_core(bf16* smem, const GOp& A, const GOp& B, int64_t i0, int64_t j0, int64_t kb,
                                          int64_t ke, f32x16 (&acc)[4][2]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  OpLoad<AKC> la;
  OpLoad<BKC> lb;
  la.init(A, i0, lane, w);
  lb.init(B, j0, lane, w);
  gemm_core_l<AKC, BKC, TAIL>(smem, la, lb, kb, ke, acc);
}

}  // namespace gemm
}  // namespace siq
