// fp32 GEMM on the CDNA4 matrix cores (v_mfma_f32_32x32x2_f32) with a fused epilogue.
//
// Everything is column-major.  A workgroup of WM x WN x WK wavefronts owns a BM x BN tile of C and
// walks the concatenated K segments in slabs of BK.  The MFMA is issued "swapped" (its 32x2 operand
// comes from X, its 2x32 operand from A), which makes the 32 lanes of an accumulator register hold
// 32 consecutive m of one column n: stores to C are full 128-byte segments.
//
// The kernels:
//  * gemm_kernel (aligned operands, every tile configuration): 16-byte copies global -> registers
//    -> LDS with no shuffles for either memory order (Stage); software pipeline two slabs deep;
//    fragments read one group of 8 k ahead of the MFMAs that use them; the slab's staging work and
//    its handful of scalar bookkeeping instructions are issued between MFMA steps, never ahead of
//    them (a vector or scalar instruction that both wavefronts of a SIMD run behind the barrier is
//    time the matrix pipe stands still).  Products whose output has too few tiles split K across
//    workgroups through partial planes in a caller workspace (splitk_reduce_kernel, or a consumer
//    that adds the planes itself).  gate_gemm_cell_kernel is the same body with the LSTM cell as
//    its epilogue, gemm_kernel<..., true> (a ninth template argument) the same body for operands at any
//    float's address and with extents that are no multiple of 4.
//    Tiles of eight 32x32 blocks (products of few columns) run its streamed form, stream_body.
//    Tiles of 16 rows (narrow_body) and packed gate matrices (gate_gemm_packed_kernel, gate_gemm_narrow_kernel) are
//    for fewer columns still.
//  * gemm_generic_kernel (a ragged extent shorter than a copy or a tile, one slab of k): scalar loads, one
//    tile shape.
// WK > 1 splits every slab's k range over WK wavefront groups and reduces the partial
// accumulators through LDS in a fixed order; deep slabs (BK 64/128) let one workgroup per CU hide
// its own memory latency.  Workgroup ids are remapped so that each of the 8 XCDs (ids are dealt
// round-robin to XCDs) owns a contiguous range of tiles with n fastest: the tiles that share a
// slice of A (stacked gate weights, the V x H output embedding) meet in one XCD's L2.
// The tile configuration and the K split of a call come from a cost model over a measured table
// (gemm_tuning.inc, regenerated by tune_gemm.py on the target GPU).
#include "lh_common.h"

#include <climits>
#include <mutex>

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int PAD = 4;

struct GemmArgs {
  const float *A[LH_GEMM_MAX_SEGS];
  const float *X[LH_GEMM_MAX_SEGS];
  int lda[LH_GEMM_MAX_SEGS];
  int ldx[LH_GEMM_MAX_SEGS];
  int K[LH_GEMM_MAX_SEGS];
  int nseg;
  int M, N;
  float alpha, beta;
  const float *bias;
  int act;
  int act_rows;  // tanh applies to rows < act_rows
  const int *colmask;
  float *C;
  int ldc;
  int tiles_m, tiles_n;
  // K split across workgroups (main kernel only): workgroup (tile, split) takes slabs
  // [split * slabs_per_split, ...) of the concatenated segments and writes its raw partial tile
  // into plane `split` of the workspace (ws_ld x N floats each, column-major like C); a second
  // kernel adds the planes up in split order and applies the epilogue.
  int splits, slabs_per_split;
  float *ws_part;
  int ws_ld;
  // A (X) is contiguous along m (n) and that extent is no multiple of 4: the last row (column) of
  // tiles is moved back to end with the operand, see gemm_body
  int ragged_m, ragged_n;
  int leave_partial;  // host only: the caller sums the planes itself, no reduction launch
  // Gate product with the LSTM cell in its epilogue (gate_gemm_cell_kernel): M = 4 * cell_H rows
  // in gate order i, f, c', o; C (ldc) is a read-only addend to the pre-activations when beta = 1,
  // taken from column addend_col[n] when that is given; bias and colmask are the stacked gate bias
  // and the 0/1 column mask; the kernel writes c_out and h_out (cell_H x N) and nothing else.
  int cell_H;
  const float *c_prev;
  float *c_out, *h_out;
  float cell_clip;
  int sigmoid_f64;
  const int *addend_col;
  int addend_ncols;  // entries of addend_col are clamped to [0, addend_ncols)
  // gate_gemm_group_kernel: a problem whose pre-activations are not complete yet stores its
  // product here (4 * cell_H x N, leading dimension pre_ld) instead of running the cell
  float *pre_out;
  int pre_ld;
  // training form of the cell epilogue (both optional): the gate values i, f, g, o for the
  // backward pass (4 * cell_H x N, leading dimension 4 * cell_H), and the copy of h the layer
  // above reads through its dropout mask, h_drop = (drop_mask < keep) / keep * h (cell_H x N)
  float *gates_out;
  const float *drop_mask;
  float *h_drop;
  float keep;
};

// Stages one BK x BD operand slab: global -> registers (load), registers -> LDS [BK][BD+PAD] (store).
// KC = false: the operand is contiguous along the tile's outer dimension d (m or n);
// KC = true : the operand is contiguous along k (one run of BK floats per d).
// The loads are branch-free: an element outside the operand is fetched from a clamped (valid)
// address and replaced by zero when it is written to LDS.
template <int BD, int BK, int NT, bool KC, bool VEC>
struct SlabStage {
  static constexpr int kVecTotal = BD * BK / 4;
  static constexpr int kTotal = BD * BK;
  static constexpr int NV = (kVecTotal + NT - 1) / NT;
  static constexpr int NS = (kTotal + NT - 1) / NT;
  static_assert((VEC ? NV : NS) <= 32, "validity mask is 32 bits");
  float4 v[VEC ? NV : 1];
  float s[VEC ? 1 : NS];
  unsigned ok;  // bit i: element i of this thread lies inside the operand

  __device__ __forceinline__ void load(const float *__restrict__ base, int ld, int d0, int k0,
                                       int dlim, int klim, int tid) {
    ok = 0u;
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int f = tid + i * NT;
        int k, d;
        if constexpr (!KC) {
          k = k0 + f / (BD / 4);
          d = d0 + (f % (BD / 4)) * 4;
        } else {
          d = d0 + f / (BK / 4);
          k = k0 + (f % (BK / 4)) * 4;
        }
        const bool in = f < kVecTotal && k < klim && d < dlim;
        const size_t off = KC ? (size_t)d * ld + k : (size_t)k * ld + d;
        v[i] = *reinterpret_cast<const float4 *>(base + (in ? off : (size_t)0));
        ok |= in ? (1u << i) : 0u;
      }
    } else {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int e = tid + i * NT;
        int k, d;
        if constexpr (!KC) {
          k = k0 + e / BD;
          d = d0 + e % BD;
        } else {
          d = d0 + e / BK;
          k = k0 + e % BK;
        }
        const bool in = e < kTotal && k < klim && d < dlim;
        const size_t off = KC ? (size_t)d * ld + k : (size_t)k * ld + d;
        s[i] = base[in ? off : (size_t)0];
        ok |= in ? (1u << i) : 0u;
      }
    }
  }

  __device__ __forceinline__ void store(float *__restrict__ lds, int tid) const {
    constexpr int LD = BD + PAD;
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int f = tid + i * NT;
        if (f < kVecTotal) {
          const bool in = (ok >> i) & 1u;
          const float4 val = in ? v[i] : make_float4(0.f, 0.f, 0.f, 0.f);
          if constexpr (!KC) {
            const int k = f / (BD / 4);
            const int d = (f % (BD / 4)) * 4;
            *reinterpret_cast<float4 *>(lds + k * LD + d) = val;
          } else {
            const int d = f / (BK / 4);
            const int k = (f % (BK / 4)) * 4;
            lds[(k + 0) * LD + d] = val.x;
            lds[(k + 1) * LD + d] = val.y;
            lds[(k + 2) * LD + d] = val.z;
            lds[(k + 3) * LD + d] = val.w;
          }
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int e = tid + i * NT;
        if (e < kTotal) {
          int k, d;
          if constexpr (!KC) {
            k = e / BD;
            d = e % BD;
          } else {
            d = e / BK;
            k = e % BK;
          }
          lds[k * LD + d] = ((ok >> i) & 1u) ? s[i] : 0.f;
        }
      }
    }
  }
};

constexpr int cmax(int a, int b) { return a > b ? a : b; }

template <int BM, int BN, int WK, int BK>
constexpr int smem_floats() {
  return cmax(2 * BK * (BM + PAD + BN + PAD), (WK - 1) * BM * BN);
}

extern __shared__ __attribute__((aligned(16))) float smem[];

template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX, bool VEC>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_generic_kernel(const GemmArgs g) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 32, FN = TN / 32;
  static_assert(FM >= 1 && FN >= 1 && TM % 32 == 0 && TN % 32 == 0, "wave tile = 32x32 MFMA tiles");
  constexpr int KPW = BK / WK;  // k values one wavefront group consumes per slab
  static_assert(KPW >= 2 && KPW % 2 == 0 && BK % 4 == 0, "slab depth");
  constexpr int NSTEP = KPW / 2;
  constexpr int LDA = BM + PAD, LDX = BN + PAD;
  constexpr int kSlabFloats = BK * (LDA + LDX);
  static_assert(smem_floats<BM, BN, WK, BK>() * 4 <= 160 * 1024, "LDS capacity of a CU");

  float *const As0 = smem, *const Xs0 = smem + BK * LDA;
  float *const As1 = smem + kSlabFloats, *const Xs1 = As1 + BK * LDA;

  // XCD-aware tile assignment.
  const int nwg = gridDim.x, id = blockIdx.x;
  const int xcd = id % 8, within = id / 8;
  const int per = nwg / 8, rem = nwg % 8;
  const int logical = xcd * per + (xcd < rem ? xcd : rem) + within;
  const int m0 = (logical / g.tiles_n) * BM;
  const int n0 = (logical % g.tiles_n) * BN;

  const int tid = threadIdx.x;
  const int wave = tid / lh::kWave, lane = tid % lh::kWave;
  const int wk = wave / (WM * WN), wmn = wave % (WM * WN);
  const int wm = wmn % WM, wn = wmn / WM;
  const int l32 = lane % 32, lhi = lane / 32;

  floatx16 acc[FN][FM];
#pragma unroll
  for (int a = 0; a < FN; ++a)
#pragma unroll
    for (int b = 0; b < FM; ++b)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[a][b][j] = 0.f;

  SlabStage<BM, BK, NT, TA, VEC> sa;
  SlabStage<BN, BK, NT, !TX, VEC> sx;

  // segment descriptors live in scalar registers; the cursor selects among them without touching
  // the kernel-argument memory again inside the loop
  const float *const A0 = g.A[0], *const A1 = g.A[1], *const A2 = g.A[2];
  const float *const X0 = g.X[0], *const X1 = g.X[1], *const X2 = g.X[2];
  const int lda0 = g.lda[0], lda1 = g.lda[1], lda2 = g.lda[2];
  const int ldx0 = g.ldx[0], ldx1 = g.ldx[1], ldx2 = g.ldx[2];
  const int K0 = g.K[0], K1 = g.K[1], K2 = g.K[2];
  const int M = g.M, N = g.N;
  int total = (K0 + BK - 1) / BK;
  if (g.nseg > 1) total += (K1 + BK - 1) / BK;
  if (g.nseg > 2) total += (K2 + BK - 1) / BK;

  int lseg = 0, lk0 = 0;  // cursor of the next slab to load
#define LH_ISSUE()                                                  \
  do {                                                              \
    const float *Ab = lseg == 0 ? A0 : (lseg == 1 ? A1 : A2);       \
    const float *Xb = lseg == 0 ? X0 : (lseg == 1 ? X1 : X2);       \
    const int la = lseg == 0 ? lda0 : (lseg == 1 ? lda1 : lda2);    \
    const int lx = lseg == 0 ? ldx0 : (lseg == 1 ? ldx1 : ldx2);    \
    const int Ks = lseg == 0 ? K0 : (lseg == 1 ? K1 : K2);          \
    sa.load(Ab, la, m0, lk0, M, Ks, tid);                           \
    sx.load(Xb, lx, n0, lk0, N, Ks, tid);                           \
    lk0 += BK;                                                      \
    if (lk0 >= Ks) {                                                \
      ++lseg;                                                       \
      lk0 = 0;                                                      \
    }                                                               \
  } while (0)

  LH_ISSUE();
  sa.store(As0, tid);
  sx.store(Xs0, tid);
  __syncthreads();

  for (int s = 0; s < total; ++s) {
    const bool has_next = s + 1 < total;
    if (has_next) LH_ISSUE();
    const float *as = ((s & 1) ? As1 : As0) + (wk * KPW + lhi) * LDA + wm * TM + l32;
    const float *xs = ((s & 1) ? Xs1 : Xs0) + (wk * KPW + lhi) * LDX + wn * TN + l32;
    float fa[2][FM], fx[2][FN];
#pragma unroll
    for (int b = 0; b < FM; ++b) fa[0][b] = as[b * 32];
#pragma unroll
    for (int a = 0; a < FN; ++a) fx[0][a] = xs[a * 32];
#pragma unroll
    for (int i = 0; i < NSTEP; ++i) {
      const int cur = i & 1, nxt = cur ^ 1;
      if (i + 1 < NSTEP) {
#pragma unroll
        for (int b = 0; b < FM; ++b) fa[nxt][b] = as[(2 * (i + 1)) * LDA + b * 32];
#pragma unroll
        for (int a = 0; a < FN; ++a) fx[nxt][a] = xs[(2 * (i + 1)) * LDX + a * 32];
      }
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[cur][a], fa[cur][b], acc[a][b], 0, 0, 0);
    }
    if (has_next) {
      sa.store((s & 1) ? As0 : As1, tid);
      sx.store((s & 1) ? Xs0 : Xs1, tid);
    }
    __syncthreads();
  }
#undef LH_ISSUE

  if constexpr (WK > 1) {
    // Fixed-order reduction of the WK partial tiles through LDS (the slab buffers are dead now).
    constexpr int kPerWave = FN * FM * 16 * 64;
    if (wk > 0) {
      float *dst = smem + ((wk - 1) * (WM * WN) + wmn) * kPerWave + lane;
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
#pragma unroll
          for (int j = 0; j < 16; ++j) dst[((a * FM + b) * 16 + j) * 64] = acc[a][b][j];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int p = 0; p < WK - 1; ++p) {
      const float *src = smem + (p * (WM * WN) + wmn) * kPerWave + lane;
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
#pragma unroll
          for (int j = 0; j < 16; ++j) acc[a][b][j] += src[((a * FM + b) * 16 + j) * 64];
    }
  }

  // Epilogue: accumulator register j of lane l is C[m = .. + l%32][n = .. + 8*(j/4) + 4*(l/32) + j%4].
  // Everything the epilogue reads (old C for beta, the column mask, the bias) is fetched for a whole
  // 32x32 accumulator tile with independent loads before any of it is used, so the loads of one tile
  // overlap instead of costing one memory round trip each.
  const float alpha = g.alpha, beta = g.beta;
  const bool use_beta = beta != 0.f;
  const int *const colmask = g.colmask;
#pragma unroll
  for (int a = 0; a < FN; ++a) {
#pragma unroll
    for (int b = 0; b < FM; ++b) {
      const int m = m0 + wm * TM + b * 32 + l32;
      const bool m_ok = m < g.M;
      const int mc = m_ok ? m : 0;
      const float bv = g.bias ? g.bias[mc] : 0.f;
      const bool do_tanh = g.act == LH_ACT_TANH && m < g.act_rows;
      const int nb = n0 + wn * TN + a * 32 + lhi * 4;
      if constexpr (BM * BN <= 32 * 64) {
        // Small tiles run with few workgroups per CU, where a serial chain of loads in the epilogue
        // is a visible part of the launch: fetch four columns' worth before using any.
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float old[4], cm[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int n = nb + q * 8 + r;
            const int nc = n < g.N ? n : 0;
            old[r] = use_beta ? g.C[(size_t)nc * g.ldc + mc] : 0.f;
            cm[r] = colmask ? (float)colmask[nc] : 1.f;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int n = nb + q * 8 + r;
            float v = alpha * acc[a][b][q * 4 + r];
            if (use_beta) v += beta * old[r];
            v += bv;
            if (do_tanh) v = tanhf(v);
            if (colmask) v *= cm[r];
            if (m_ok && n < g.N) g.C[(size_t)n * g.ldc + m] = v;
          }
        }
      } else {
        // Large tiles: many workgroups share a CU and hide each other's epilogue; keep the register
        // footprint (and with it the number of resident workgroups) minimal.
        if (!m_ok) continue;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int n = nb + (j / 4) * 8 + (j % 4);
          if (n >= g.N) continue;
          float *cp = g.C + (size_t)n * g.ldc + m;
          float v = alpha * acc[a][b][j];
          if (use_beta) v += beta * *cp;
          v += bv;
          if (do_tanh) v = tanhf(v);
          if (colmask) v *= (float)colmask[n];
          *cp = v;
        }
      }
    }
  }
}


// =============================================================================================
// Main kernel.  What shapes it:
//   * On CDNA a VALU instruction and an MFMA do not overlap inside a SIMD: every non-MFMA vector
//     instruction in the loop costs about four cycles of matrix-pipe time.  The loop therefore
//     carries almost none.  Global addresses are a uniform base (scalar registers) plus
//     per-thread 32-bit byte offsets computed once per K segment; bounds along M / N are folded
//     into those offsets (out-of-range rows re-read the tile origin: they only feed rows and
//     columns of C that are never written); the K tail of a segment, one slab at most, is the only
//     place that masks data.  Staging is 16-byte copies global -> registers -> LDS with no
//     shuffling, for either memory order:
//   * an operand that is contiguous along k in memory lives in LDS as [k/4][d][4], and an MFMA
//     operand fragment for four k-steps is one ds_read_b128 per lane;
//   * an operand that is contiguous along d lives in LDS as [k][d], and a fragment is one
//     ds_read_b32 per k-step.
//     In both, lanes 0-31 take k = 8g+q and lanes 32-63 k = 8g+4+q for step q of group g: the K
//     order inside a slab is a fixed permutation applied to both operands, which leaves the dot
//     products unchanged.
// RAGGED: operands need no alignment beyond a float's.  A 16-byte global load from any dword address
// is one instruction here, and a wavefront's contiguous run only touches one more cache line.  What a
// 16-byte unit must not do is reach past the operand, so where the contiguous extent is no
// multiple of 4:
//   * along m or n, the last tile is moved back to end with the operand (rows that the tile before
//     it owns are computed again and not stored): the K loop knows nothing of it;
//   * along k, the segment's last unit is loaded from up to three floats earlier and shifted into
//     place on the masked path of the K tail, which the other slabs never take.
// An output projection of 30003 words (M = 30003, K = 1000) at 84 columns took 128 us on the scalar
// kernel and takes 64 us here, 48 columns 44 us, 12 columns 29 us.  Aligned operands keep kernels of their own: run through this
// form the 128x96 gate product (768 columns) took 119 us instead of 107.
typedef float unaligned_float4 __attribute__((ext_vector_type(4), aligned(4)));
template <bool RAGGED>
__device__ __forceinline__ float4 load4(const char *p) {
  if constexpr (!RAGGED) return *reinterpret_cast<const float4 *>(p);
  const unaligned_float4 t = *reinterpret_cast<const unaligned_float4 *>(p);
  return make_float4(t.x, t.y, t.z, t.w);
}

__device__ __forceinline__ float4 keep_if(float4 w, bool c) {
  // per component: a select between two float4 objects makes the compiler pick an address
  w.x = c ? w.x : 0.f;
  w.y = c ? w.y : 0.f;
  w.z = c ? w.z : 0.f;
  w.w = c ? w.w : 0.f;
  return w;
}

// The first `n` components of w, starting at its component 4 - n, and zeros (n <= 0: all zero).
__device__ __forceinline__ float4 keep_last(float4 w, int n) {
  float4 r;
  r.x = n >= 4 ? w.x : (n == 3 ? w.y : (n == 2 ? w.z : (n == 1 ? w.w : 0.f)));
  r.y = n >= 4 ? w.y : (n == 3 ? w.z : (n == 2 ? w.w : 0.f));
  r.z = n >= 4 ? w.z : (n == 3 ? w.w : 0.f);
  r.w = n >= 4 ? w.w : 0.f;
  return r;
}

template <int BD, int BK, int NT, bool KC, bool RAGGED>
struct Stage {
  static constexpr int KQ = BK / 4;
  // KC: 16-byte units per k-quad row.  A staging store walks k-quads first, and LDS takes 16-byte
  // stores eight lanes (128 bytes) at a time: the row stride keeps those eight on distinct
  // 16-byte bank groups (measured: 8 conflict cycles per store otherwise).
  static constexpr int LDQ = BD + (KQ == 4 ? 2 : 1);
  // !KC: floats per k row.  Stores are contiguous and fragment reads (32 consecutive floats per
  // lane half) are conflict-free for any stride; the pad only keeps rows 16-byte aligned.
  static constexpr int LDD = BD + 8;
  static constexpr int kFloats = KC ? KQ * LDQ * 4 : BK * LDD;
  static constexpr int kUnits = KQ * BD;  // 16-byte units in a slab
  static constexpr int NU = (kUnits + NT - 1) / NT;
  // every thread owns NU whole units: no per-unit guard (and no exec-mask bookkeeping in the K loop)
  static constexpr bool kExact = kUnits % NT == 0;
  static_assert(NU <= 32, "validity mask is 32 bits");
  static_assert(BD % 16 == 0 && BK % 16 == 0, "tile extents");

  float4 v[NU];
  unsigned goff[NU];  // byte offset of each unit from the slab origin
  unsigned ok;        // K-tail validity, one bit per unit
  int ktail;          // RAGGED: k values in the K tail

  // unit u of the slab: (d, k) of its first element and its float offset in LDS
  static __device__ __forceinline__ int unit_d(int u) { return KC ? u / KQ : (u % (BD / 4)) * 4; }
  static __device__ __forceinline__ int unit_k(int u) { return KC ? (u % KQ) * 4 : u / (BD / 4); }
  static __device__ __forceinline__ int unit_lds(int u) {
    return KC ? ((u % KQ) * LDQ + u / KQ) * 4 : (u / (BD / 4)) * LDD + (u % (BD / 4)) * 4;
  }
  // dn = rows/columns of the operand that exist from the tile origin on
  __device__ __forceinline__ void set_ld(int ld, int tid, int dn) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + i * NT;
      const int d = unit_d(u), k = unit_k(u);
      const unsigned off = KC ? (unsigned)(d * ld + k) * 4u : (unsigned)(k * ld + d) * 4u;
      goff[i] = d < dn ? off : 0u;
    }
  }
  // The same for a tile of a stacked gate matrix that holds BD/4 rows of each of the four gates:
  // tile row d is row (d % (BD/4)) of gate d / (BD/4); gates are H rows apart; rows_left = rows of
  // a gate that exist from the tile origin on.
  __device__ __forceinline__ void set_ld_gates(int ld, int tid, int H, int rows_left) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + i * NT;
      const int d = unit_d(u), k = unit_k(u);
      const int r = d % (BD / 4), row = (d / (BD / 4)) * H + r;
      const unsigned off = KC ? (unsigned)(row * ld + k) * 4u : (unsigned)(k * ld + row) * 4u;
      goff[i] = r < rows_left ? off : 0u;
    }
  }
  // kn (< BK) = k values left in the segment: units past it re-read the slab origin and are
  // zeroed before they reach LDS.  RAGGED: a unit along k that holds fewer than four of them is read
  // from that many floats earlier; when it is the slab's first one the whole tail is addressed from
  // four floats earlier (such a segment has at least four k values, so a slab lies before it).
  static __device__ __forceinline__ int tail_back(int kn) { return RAGGED && KC && kn < 4 ? 4 : 0; }
  __device__ __forceinline__ void clamp_tail(int tid, int kn) {
    if constexpr (RAGGED) {
      ktail = kn;
      const unsigned back = 4u * (unsigned)tail_back(kn);
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const int left = kn - unit_k(tid + i * NT);
        unsigned off = goff[i] + back;
        if (KC && left < 4) {
          // a unit of a row past the tile's bound sits at the origin and stays there
          const unsigned shift = 4u * (unsigned)(4 - left);
          off = off >= shift ? off - shift : 0u;
        }
        goff[i] = left > 0 ? off : 0u;
      }
    } else {
      ok = 0u;
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const bool in = unit_k(tid + i * NT) < kn;
        goff[i] = in ? goff[i] : 0u;
        ok |= in ? (1u << i) : 0u;
      }
    }
  }
  __device__ __forceinline__ void load(const float *__restrict__ base, int tid) {
    const char *b = reinterpret_cast<const char *>(base);
#pragma unroll
    for (int i = 0; i < NU; ++i)
      if (kExact || tid + i * NT < kUnits) v[i] = load4<RAGGED>(b + goff[i]);
  }
  __device__ __forceinline__ void zero_tail(int tid) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      if constexpr (RAGGED) {
        const int left = ktail - unit_k(tid + i * NT);
        v[i] = keep_last(v[i], KC ? left : (left > 0 ? 4 : 0));
      } else {
        v[i] = keep_if(v[i], (ok >> i) & 1u);
      }
    }
  }
  __device__ __forceinline__ void store(float *__restrict__ buf, int tid) const {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + i * NT;
      if (kExact || u < kUnits) *reinterpret_cast<float4 *>(buf + unit_lds(u)) = v[i];
    }
  }
  // Fragment reads.  origin = float offset for (first k of the wavefront's share, lane half, row d).
  static __device__ __forceinline__ int frag_origin(int k0, int lhi, int d) {
    return KC ? ((k0 / 4 + lhi) * LDQ + d) * 4 : (k0 + 4 * lhi) * LDD + d;
  }
  static __device__ __forceinline__ void read_frag(const float *__restrict__ origin, int grp,
                                                   int frag, float (&out)[4]) {
    if constexpr (KC) {
      const float4 t =
          *reinterpret_cast<const float4 *>(origin + (2 * grp * LDQ + frag * 32) * 4);
      out[0] = t.x, out[1] = t.y, out[2] = t.z, out[3] = t.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) out[q] = origin[(8 * grp + q) * LDD + frag * 32];
    }
  }
};

// ---- streamed form --------------------------------------------------------------------------
// One 32x32 block of C per wavefront, and every wavefront on its own: it reads the k it multiplies
// (CK of every slab) into a ring of LDS stages that no other wavefront touches, straight from
// memory (global_load_lds, no register and no LDS store of its own in between), and the K loop has
// no barrier.  All eight wavefronts share the sum over the partial blocks and the epilogue, and the cell's
// inputs are requested behind the first slabs.
// What bounds these products is not bandwidth but what a workgroup does between its loads and its MFMAs:
// with one workgroup per CU nothing else hides a staging store, a barrier or the wavefront that sums
// eight partial tiles alone.  4000 x 64, K = 1000 / 2000 (weights from HBM): 11.3 / 17.0 us staged, 9.4 / 14.3
// streamed; transposed 11.2 / 17.4 and 10.1 / 16.5.  A fixed part of 4.0 instead of 5.6 us (an empty launch:
// 2.8), and 0.63 us per slab of 128 k where the MFMAs alone take 0.47 at the 2.16 GHz the card runs here.
// Deeper rings (5 stages: 14.3), fragments read a slab ahead (15.2), 16 wavefronts (15.9) and four of 32 k each
// (15.6) gave nothing.  Shapes of 8 k per wavefront and slab stay staged except the 32x32 one: their 32-byte runs along k
// cost more than the stores (32x64, full CUs: 0.0108 us per k and workgroup against 0.0087).
constexpr int kRingStages = 4;
template <int BM, int BN, int WM, int WN, int WK, int BK>
constexpr bool streamed() {
  // eight wavefronts, a 32 x 32 block each, 16 k of every slab (8 where all of them share one block)
  return BM == 32 * WM && BN == 32 * WN && WK >= 4 && WM * WN * WK == 8 &&
         (BK == 16 * WK || (WK == 8 && BK == 64));
}
// Floats from one column to the next of a partial tile in LDS: a quarter of the rows (a gate's share
// of the tile) as padding puts the columns a wavefront reads at once on distinct banks.
template <int BM>
constexpr int spread_ld() {
  return BM + BM / 4;
}

template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX, bool RAGGED>
constexpr int smem2_floats() {
  constexpr int NT = 64 * WM * WN * WK;
  if constexpr (!RAGGED && streamed<BM, BN, WM, WN, WK, BK>())
    return cmax(kRingStages * WM * WN * BK * 64, WK * BN * spread_ld<BM>());
  return cmax(2 * (Stage<BM, BK, NT, TA, false>::kFloats + Stage<BN, BK, NT, !TX, false>::kFloats),
              (WK - 1) * BM * BN);
}

// A wavefront's CK x BD piece of one operand in its ring stage.  A load writes 64 consecutive
// 16-byte units, one per lane, so what the layout can choose is which unit a lane fetches:
//  * contiguous along d: rows of 32 floats, one per k; the k of a group of 8 in the order 0 4 2 6 1 5 3 7,
//    which puts the two k of one MFMA step (k and k + 4, lanes 0-31 and 32-63) into neighbouring rows:
//    a fragment read is 64 consecutive floats;
//  * contiguous along k: rows of CK floats, one per d, their units permuted (XOR with bits of d) so
//    that the 16 lanes of one phase of a 16-byte read meet all banks.
template <int CK, bool KC, int BD = 32>
struct Piece {
  static constexpr int U = CK / 4;       // KC: units per row
  static_assert(KC || BD == 32, "rows of k");
  static constexpr int kFloats = CK * BD;
  static constexpr int kLoads = kFloats / 256;  // wavefront loads per piece
  unsigned goff[kLoads];

  static __device__ __forceinline__ int swap02(int k) { return (k & ~5) | ((k & 1) << 2) | ((k >> 2) & 1); }
  static __device__ __forceinline__ int swizzle(int d) { return (d / (16 / U)) % U; }
  static __device__ __forceinline__ int unit_d(int u) { return KC ? u / U : (u % 8) * 4; }
  static __device__ __forceinline__ int unit_k(int u) {
    return KC ? ((u % U) ^ swizzle(u / U)) * 4 : swap02(u / 8);
  }
  // dn = rows/columns of the operand from the tile origin on, first = this wavefront's first of them
  __device__ __forceinline__ void set_ld(int ld, int lane, int first, int dn) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int u = lane + i * 64;
      const int d = first + unit_d(u), k = unit_k(u);
      const unsigned off = KC ? (unsigned)(d * ld + k) * 4u : (unsigned)(k * ld + d) * 4u;
      goff[i] = d < dn ? off : 0u;
    }
  }
  template <int GQ>
  __device__ __forceinline__ void set_ld_gates(int ld, int lane, int first, int H, int rows_left) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int u = lane + i * 64;
      const int d = first + unit_d(u), k = unit_k(u);
      const int r = d % GQ, row = (d / GQ) * H + r;
      const unsigned off = KC ? (unsigned)(row * ld + k) * 4u : (unsigned)(k * ld + row) * 4u;
      goff[i] = r < rows_left ? off : 0u;
    }
  }
  static __device__ __forceinline__ void load_unit(const float *base, unsigned off, unsigned lds) {
    // No register receives the data, so nothing the compiler allocates can meet the load in
    // flight; its addresses are read when it is issued.  Completion: wait_loads below.
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(off), "s"(base)
                 : "memory", "m0");
  }
  __device__ __forceinline__ void load(const float *base, unsigned lds) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load_unit(base, goff[i], lds + 1024u * i);
  }
  // The same where the segment ends behind the kn-th k: units past it fetch the first k's instead
  // (their fragments are zeroed).
  __device__ __forceinline__ void load_tail(const float *base, unsigned lds, int ld, int lane, int kn) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int k = unit_k(lane + i * 64);
      const unsigned back = (KC ? (unsigned)k : (unsigned)(k * ld)) * 4u;
      load_unit(base, k < kn ? goff[i] : (goff[i] >= back ? goff[i] - back : 0u), lds + 1024u * i);
    }
  }
  static __device__ __forceinline__ void read_frag(const float *piece, int grp, int l32, int lhi, float (&out)[4]) {
    if constexpr (KC) {
      const float4 t = *reinterpret_cast<const float4 *>(piece + (l32 * U + ((2 * grp + lhi) ^ swizzle(l32))) * 4);
      out[0] = t.x, out[1] = t.y, out[2] = t.z, out[3] = t.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) out[q] = piece[(8 * grp + swap02(q) + lhi) * 32 + l32];
    }
  }
};

// The cell of row r, column n from its pre-activations, and everything it leaves.
__device__ __forceinline__ void store_cell(const GemmArgs &g, float (&pre)[4], float c_prev, int colmask, int r, int n) {
  const int H = g.cell_H;
  float c, h;
  const float mask = (float)(colmask & 1);
  if (g.sigmoid_f64 && !(colmask & LH_MASK_F32_GATES))
    lh::lstm_cell_point<true>(pre[0], pre[1], pre[2], pre[3], c_prev, mask, g.cell_clip, c, h);
  else
    lh::lstm_cell_point<false>(pre[0], pre[1], pre[2], pre[3], c_prev, mask, g.cell_clip, c, h);
  const size_t o = (size_t)n * H + r;
  g.c_out[o] = c;
  g.h_out[o] = h;
  if (g.gates_out) {
    float *go = g.gates_out + (size_t)n * 4 * H + r;
#pragma unroll
    for (int q = 0; q < 4; ++q) go[(size_t)q * H] = pre[q];  // the cell left i, f, g, o there
  }
  if (g.h_drop) g.h_drop[o] = ((float)(g.drop_mask[o] < g.keep) * (1.0f / g.keep)) * h;
}

// At most N of this wavefront's loads still in flight; its LDS reads have returned.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX>
constexpr int smem2_floats() {
  return smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX, false>();
}

// The rare paths of the K loop (a new K segment, a short last slab) are a few dozen selects each.
// Left alone the compiler turns those branches into straight-line selects that every iteration
// executes, and vector ALU instructions take issue time from the matrix pipe; an empty statement
// the optimiser must keep makes each of them a real, normally untaken, branch.
#define LH_KEEP_BRANCH() asm volatile("" ::: "memory")

// CELL: the rows of a tile are BM/4 rows of each LSTM gate and the epilogue is the LSTM cell.
// Workgroups of a launch are dealt to the 8 XCDs round-robin; this gives every XCD a contiguous
// range of the launch's work items.
__device__ __forceinline__ int xcd_logical_id() {
  const int nwg = gridDim.x, id = blockIdx.x;
  const int xcd = id % 8, within = id / 8;
  const int per = nwg / 8, rem = nwg % 8;
  return xcd * per + (xcd < rem ? xcd : rem) + within;
}

// The streamed form of gemm_body.
// PACKED: A is a gate matrix as lh_gate_pack_f32 lays it out: for every 8 cells K rows of 32 floats, row k
// holding the four gates of each of the cells at that k.
constexpr int kPackCells = 8, kPackRows = 4 * kPackCells;
template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX, bool CELL, bool PACKED>
__device__ __forceinline__ void stream_body(const GemmArgs &g, const int m0, const int n0, const int split,
                                            const int splits) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int CK = BK / WK, NG = CK / 8;
  constexpr int NB = kRingStages;
  static_assert(NB == 4, "the waits of the K loop");
  using PA = Piece<CK, TA>;
  using PX = Piece<CK, !TX>;
  constexpr int kStage = PA::kFloats + PX::kFloats;  // floats of one wavefront's stage
  constexpr int kLoads = PA::kLoads + PX::kLoads;
  constexpr int GQ = BM / 4;

  const int tid = threadIdx.x, lane = tid % lh::kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / lh::kWave);
  const int wk = wave / (WM * WN), wmn = wave % (WM * WN);
  const int wm = wmn % WM, wn = wmn / WM;
  const int l32 = lane % 32, lhi = lane / 32;
  float *const ring = smem + wave * NB * kStage;
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)ring;

  const int M = g.M, N = g.N;
  const int slabs0 = (g.K[0] + BK - 1) / BK;
  const int slabs1 = g.nseg > 1 ? (g.K[1] + BK - 1) / BK : 0;
  const int slabs2 = g.nseg > 2 ? (g.K[2] + BK - 1) / BK : 0;
  const int first = split * g.slabs_per_split;
  const int total = min(g.slabs_per_split, slabs0 + slabs1 + slabs2 - first);
  int lseg = 0, k0 = first;  // segment and (below) k of the next slab to request
  if (k0 >= slabs0) {
    k0 -= slabs0;
    lseg = 1;
    if (k0 >= slabs1) {
      k0 -= slabs1;
      lseg = 2;
    }
  }
  k0 *= BK;
  int cseg = lseg, ck = k0;  // the same of the slab to multiply
  // (an array indexed by a variable would move the arguments to memory)
  auto pick = [](int seg, auto v0, auto v1, auto v2) __attribute__((always_inline)) {
    return seg == 0 ? v0 : (seg == 1 ? v1 : v2);
  };
#define LH_SEG(FIELD, SEG) pick(SEG, g.FIELD[0], g.FIELD[1], g.FIELD[2])

  PA pa;
  PX px;
  bool new_seg = true;
  const float *a = nullptr, *x = nullptr;  // this wavefront's first k of the next slab
  // PACKED: this wavefront's group of cells (a tile may reach past the last one)
  const int cells = PACKED ? min(m0 / kPackCells + wm, (g.cell_H - 1) / kPackCells) : 0;
  int step_a = 0, step_x = 0, lda = 0, ldx = 0, Ks = 0;
  unsigned put = ring_lds;  // stage the next slab goes to
  auto request = [&]() __attribute__((always_inline)) {
    if (new_seg) {
      LH_KEEP_BRANCH();
      Ks = LH_SEG(K, lseg);
      if (lda != LH_SEG(lda, lseg) || ldx != LH_SEG(ldx, lseg)) {
        LH_KEEP_BRANCH();
        lda = LH_SEG(lda, lseg), ldx = LH_SEG(ldx, lseg);
        if constexpr (PACKED) pa.set_ld(lda, lane, 0, kPackRows);
        else if constexpr (CELL) pa.template set_ld_gates<GQ>(lda, lane, 32 * wm, g.cell_H, g.cell_H - m0);
        else pa.set_ld(lda, lane, 32 * wm, M - m0);
        px.set_ld(ldx, lane, 32 * wn, N - n0);
      }
      const int k = k0 + wk * CK;
      if constexpr (PACKED) a = LH_SEG(A, lseg) + ((size_t)cells * Ks + k) * kPackRows;
      else a = LH_SEG(A, lseg) + (TA ? (size_t)m0 * lda + k : (size_t)k * lda + m0);
      x = LH_SEG(X, lseg) + (!TX ? (size_t)n0 * ldx + k : (size_t)k * ldx + n0);
      step_a = TA ? BK : BK * lda;
      step_x = !TX ? BK : BK * ldx;
    }
    const int kn = Ks - k0 - wk * CK;
    if (kn < CK) {
      LH_KEEP_BRANCH();
      if (kn <= 0) {  // nothing left for this wavefront: any valid address, nothing is multiplied
        a = LH_SEG(A, lseg) + (PACKED ? (size_t)cells * Ks * kPackRows : (TA ? (size_t)m0 * lda : (size_t)m0));
        x = LH_SEG(X, lseg) + (!TX ? (size_t)n0 * ldx : (size_t)n0);
      }
      pa.load_tail(a, put, lda, lane, kn);
      px.load_tail(x, put + PA::kFloats * 4u, ldx, lane, kn);
    } else {
      pa.load(a, put);
      px.load(x, put + PA::kFloats * 4u);
    }
    put = put + kStage * 4u == ring_lds + NB * kStage * 4u ? ring_lds : put + kStage * 4u;
    a += step_a;
    x += step_x;
    k0 += BK;
    new_seg = k0 >= Ks;
    if (new_seg) {
      ++lseg;
      k0 = 0;
    }
  };

  floatx16 acc;
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = 0.f;
  int issued = min(total, NB - 1);
  for (int i = 0; i < issued; ++i) request();

  // What the cell reads from memory, requested behind the first slabs: the epilogue would wait a
  // memory latency for it, two with addend_col.
  float ep_add[4] = {0.f, 0.f, 0.f, 0.f}, ep_bias[4] = {0.f, 0.f, 0.f, 0.f}, ep_c = 0.f;
  int ep_mask = 0;
  bool ep_ok = false;
  if constexpr (CELL) {
    static_assert(GQ * BN <= NT, "one cell per thread");
    const int r = m0 + tid % GQ, n = n0 + tid / GQ;
    ep_ok = tid < GQ * BN && r < g.cell_H && n < N;
    if (ep_ok && !g.pre_out) {
      int col = n;
      if (g.addend_col) col = min(max(g.addend_col[n], 0), g.addend_ncols - 1);
      const float *ad = g.C + (size_t)col * g.ldc + r;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (g.beta != 0.f) ep_add[q] = ad[(size_t)q * g.cell_H];
        ep_bias[q] = g.bias[q * g.cell_H + r];
      }
      ep_c = g.c_prev[(size_t)n * g.cell_H + r];
      ep_mask = g.colmask[n];
    }
  }

  const float *get = ring;
  int cK = LH_SEG(K, cseg);
  for (int s = 0; s < total; ++s) {
    const int behind = issued - 1 - s;  // slabs requested after this one
    if (behind >= 2) wait_loads<kLoads * 2>();
    else if (behind == 1) wait_loads<kLoads>();
    else wait_loads<0>();
    float fa[NG][4], fx[NG][4];
#pragma unroll
    for (int grp = 0; grp < NG; ++grp) {
      PA::read_frag(get, grp, l32, lhi, fa[grp]);
      PX::read_frag(get + PA::kFloats, grp, l32, lhi, fx[grp]);
    }
    // the stage this goes to was read in the last round, and those reads have returned
    if (issued < total) {
      request();
      ++issued;
    }
    const int kn = cK - ck - wk * CK;
    if (kn < CK) {
      LH_KEEP_BRANCH();
#pragma unroll
      for (int grp = 0; grp < NG; ++grp)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool in = 8 * grp + 4 * lhi + q < kn;
          fa[grp][q] = in ? fa[grp][q] : 0.f;
          fx[grp][q] = in ? fx[grp][q] : 0.f;
        }
    }
#pragma unroll
    for (int grp = 0; grp < NG; ++grp)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[grp][q], fa[grp][q], acc, 0, 0, 0);
    get = get + kStage == ring + NB * kStage ? ring : get + kStage;
    ck += BK;
    if (ck >= cK) {
      LH_KEEP_BRANCH();
      ck = 0;
      ++cseg;
      if (s + 1 < total) cK = LH_SEG(K, cseg);
    }
  }
#undef LH_SEG

  // Every wavefront puts its partial block into LDS as S[wk][n][m] once all of them have left
  // their rings, then every thread sums the WK values of its own elements, in the order of wk,
  // and takes them through the epilogue.
  constexpr int LDS_N = spread_ld<BM>();
  constexpr int kPlane = LDS_N * BN;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; ++j)
    smem[wk * kPlane + (wn * 32 + lhi * 4 + (j / 4) * 8 + (j % 4)) * LDS_N + wm * 32 + l32] = acc[j];
  __syncthreads();
  if constexpr (CELL) {
    if (!ep_ok) return;
    const int H = g.cell_H;
    const int rl = tid % GQ, nl = tid / GQ;
    const int r = m0 + rl, n = n0 + nl;
    float pre[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int ml = PACKED ? (rl / kPackCells) * kPackRows + (rl % kPackCells) * 4 + q : q * GQ + rl;
      const float *src = smem + nl * LDS_N + ml;
      pre[q] = src[0];
#pragma unroll
      for (int p = 1; p < WK; ++p) pre[q] += src[p * kPlane];
    }
    if (g.pre_out) {
      float *o = g.pre_out + (size_t)n * g.pre_ld + r;
#pragma unroll
      for (int q = 0; q < 4; ++q) o[(size_t)q * H] = pre[q];
      return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[q] = (g.beta != 0.f ? pre[q] + ep_add[q] : pre[q]) + ep_bias[q];
    store_cell(g, pre, ep_c, ep_mask, r, n);
  } else {
    // a split product stores the bare partial sums in its plane of the workspace
    const bool partial = splits > 1;
    const float alpha = partial ? 1.f : g.alpha, beta = partial ? 0.f : g.beta;
    const int *const colmask = partial ? nullptr : g.colmask;
    const float *const bias = partial ? nullptr : g.bias;
    const int act_rows = partial || g.act != LH_ACT_TANH ? 0 : g.act_rows;
    float *const Cb = partial ? g.ws_part + (size_t)split * g.ws_ld * N : g.C;
    const int ldc = partial ? g.ws_ld : g.ldc;
    static_assert(BM * BN % NT == 0, "whole elements per thread");
#pragma unroll
    for (int i = 0; i < BM * BN / NT; ++i) {
      const int idx = tid + i * NT;
      const int ml = idx % BM, nl = idx / BM;
      const int m = m0 + ml, n = n0 + nl;
      if (m >= M || n >= N) continue;
      const float *src = smem + nl * LDS_N + ml;
      float sum = src[0];
#pragma unroll
      for (int p = 1; p < WK; ++p) sum += src[p * kPlane];
      float *cp = Cb + (size_t)n * ldc + m;
      float v = alpha * sum;
      if (beta != 0.f) v += beta * *cp;
      if (bias) v += bias[m];
      if (m < act_rows) v = tanhf(v);
      if (colmask) v *= (float)colmask[n];
      *cp = v;
    }
  }
}

template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX, bool CELL, bool RAGGED>
__device__ __forceinline__ void gemm_body(const GemmArgs &g, const int logical) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 32, FN = TN / 32;
  static_assert(FM >= 1 && FN >= 1 && TM % 32 == 0 && TN % 32 == 0, "wave tile = 32x32 MFMA tiles");
  constexpr int KPW = BK / WK;  // k values one wavefront group consumes per slab
  static_assert(KPW % 8 == 0, "a fragment group covers 8 k (4 per lane half)");
  constexpr int NG = KPW / 8;
  constexpr bool kStream = !RAGGED && streamed<BM, BN, WM, WN, WK, BK>();
  using SA = Stage<BM, BK, NT, TA, RAGGED>;
  using SX = Stage<BN, BK, NT, !TX, RAGGED>;
  constexpr int kAF = SA::kFloats, kSlab = SA::kFloats + SX::kFloats;
  static_assert(smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX>() * 4 <= 160 * 1024,
                "LDS capacity of a CU");

  // XCD-aware tile assignment (logical): the splits of a tile are neighbours, same XCD, so the
  // partial tiles meet in its L2
  const int splits = g.splits;
  const int tile = splits == 1 ? logical : logical / splits;
  const int split = splits == 1 ? 0 : logical % splits;
  // CELL: m0 counts rows of ONE gate
  int m0 = (tile / g.tiles_n) * (CELL ? BM / 4 : BM);
  int n0 = (tile % g.tiles_n) * BN;
  // a tile that was moved back stores rows / columns from here on only (the host keeps the tile
  // extent within a ragged operand's)
  const int m_first = m0, n_first = n0;
  if constexpr (RAGGED) {
    if (!TA && g.ragged_m && m0 + BM > g.M) m0 = g.M - BM;
    if (TX && g.ragged_n && n0 + BN > g.N) n0 = g.N - BN;
  }

  const int tid = threadIdx.x;
  const int wave = tid / lh::kWave, lane = tid % lh::kWave;
  const int wk = wave / (WM * WN), wmn = wave % (WM * WN);
  const int wm = wmn % WM, wn = wmn / WM;
  const int l32 = lane % 32, lhi = lane / 32;

  floatx16 acc[FN][FM];
#pragma unroll
  for (int a = 0; a < FN; ++a)
#pragma unroll
    for (int b = 0; b < FM; ++b)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[a][b][j] = 0.f;

  if constexpr (kStream) {
    stream_body<BM, BN, WM, WN, WK, BK, TA, TX, CELL, false>(g, m0, n0, split, splits);
    return;
  }

  SA sa;
  SX sx;
  const int fa_off = SA::frag_origin(wk * KPW, lhi, wm * TM + l32);
  const int fx_off = kAF + SX::frag_origin(wk * KPW, lhi, wn * TN + l32);

  const float *const A0 = g.A[0], *const A1 = g.A[1], *const A2 = g.A[2];
  const float *const X0 = g.X[0], *const X1 = g.X[1], *const X2 = g.X[2];
  const int lda0 = g.lda[0], lda1 = g.lda[1], lda2 = g.lda[2];
  const int ldx0 = g.ldx[0], ldx1 = g.ldx[1], ldx2 = g.ldx[2];
  const int K0 = g.K[0], K1 = g.K[1], K2 = g.K[2];
  const int M = g.M, N = g.N;
  const int slabs0 = (K0 + BK - 1) / BK;
  const int slabs1 = g.nseg > 1 ? (K1 + BK - 1) / BK : 0;
  const int slabs2 = g.nseg > 2 ? (K2 + BK - 1) / BK : 0;
  // this workgroup's share of the slab sequence (the host never makes an empty share)
  const int first = split * g.slabs_per_split;
  const int total = min(g.slabs_per_split, slabs0 + slabs1 + slabs2 - first);
  int lseg = 0, lk0 = first;  // cursor of the next slab to load: segment, k offset inside it
  if (lk0 >= slabs0) {
    lk0 -= slabs0;
    lseg = 1;
    if (lk0 >= slabs1) {
      lk0 -= slabs1;
      lseg = 2;
    }
  }
  lk0 *= BK;
  // The K loop's scalar work is a few additions: the origin of the next slab in each operand
  // advances by a fixed step, and everything that depends on the segment (base pointers, leading
  // dimensions, the per-thread offsets) is set up only when a segment begins.  Both wavefronts of
  // a SIMD run this code at the same time, right behind the barrier, so every scalar instruction
  // here is time the matrix pipe stands still.
  bool new_seg = true;  // the next slab opens a segment (or the first one of this share)
  bool tail = false;    // the slab in the staging registers ends its segment short of BK
  const float *pa = nullptr, *px = nullptr;  // origin of the next slab inside A / X
  int step_a = 0, step_x = 0;                // floats from one slab to the next
  int kleft = 0;                             // k values of the segment not yet loaded
#define LH_ISSUE()                                                                 \
  do {                                                                             \
    if (new_seg) {                                                                 \
      LH_KEEP_BRANCH();                                                            \
      const float *Ab = lseg == 0 ? A0 : (lseg == 1 ? A1 : A2);                    \
      const float *Xb = lseg == 0 ? X0 : (lseg == 1 ? X1 : X2);                    \
      const int la = lseg == 0 ? lda0 : (lseg == 1 ? lda1 : lda2);                 \
      const int lx = lseg == 0 ? ldx0 : (lseg == 1 ? ldx1 : ldx2);                 \
      const int Ks = lseg == 0 ? K0 : (lseg == 1 ? K1 : K2);                       \
      if constexpr (CELL) sa.set_ld_gates(la, tid, g.cell_H, g.cell_H - m0);       \
      else sa.set_ld(la, tid, M - m0);                                             \
      sx.set_ld(lx, tid, N - n0);                                                  \
      pa = TA ? Ab + (size_t)m0 * la + lk0 : Ab + (size_t)lk0 * la + m0;           \
      px = !TX ? Xb + (size_t)n0 * lx + lk0 : Xb + (size_t)lk0 * lx + n0;          \
      step_a = TA ? BK : BK * la;                                                  \
      step_x = !TX ? BK : BK * lx;                                                 \
      kleft = Ks - lk0;                                                            \
    }                                                                              \
    tail = kleft < BK;                                                             \
    if (tail) {                                                                    \
      LH_KEEP_BRANCH();                                                            \
      sa.clamp_tail(tid, kleft);                                                   \
      sx.clamp_tail(tid, kleft);                                                   \
      if constexpr (RAGGED) {                                                      \
        pa -= SA::tail_back(kleft);                                                \
        px -= SX::tail_back(kleft);                                                \
      }                                                                            \
    }                                                                              \
    sa.load(pa, tid);                                                              \
    sx.load(px, tid);                                                              \
    pa += step_a;                                                                  \
    px += step_x;                                                                  \
    kleft -= BK;                                                                   \
    new_seg = kleft <= 0; /* a short last slab has clamped the offsets as well */  \
    if (new_seg) {                                                                 \
      ++lseg;                                                                      \
      lk0 = 0;                                                                     \
    }                                                                              \
  } while (0)
#define LH_STASH(BUF)         \
  do {                        \
    float *sb = (BUF);        \
    if (tail) {               \
      LH_KEEP_BRANCH();       \
      sa.zero_tail(tid);      \
      sx.zero_tail(tid);      \
    }                         \
    sa.store(sb, tid);        \
    sx.store(sb + kAF, tid);  \
  } while (0)

  // Software pipeline, two slabs deep: LDS holds slab s (being consumed) and slab s+1, the
  // staging registers hold slab s+2 in flight.  A slab goes to LDS at the START of the iteration
  // before it is consumed -- its buffer was released by the barrier that ended the previous
  // iteration -- so neither the global loads nor the LDS stores sit between two slabs of MFMAs.
  LH_ISSUE();
  LH_STASH(smem);
  if (total > 1) LH_ISSUE();
  __syncthreads();
  int cur = 0;  // float offset of the slab buffer being consumed
  // Fragments are read one group (8 k) ahead of the MFMAs that use them.  Deep slabs (one
  // workgroup per CU, nobody else to cover a stall) keep that up across slab boundaries: the
  // barrier that releases a slab sits BEFORE the MFMAs of its last group, whose fragments are in
  // registers by then, and the first group of the next slab is read right behind it, under those
  // MFMAs.  Shallow slabs run several workgroups per CU, which hide the one exposed read per slab
  // better than the dozen registers the carried fragments cost would (they lower the occupancy).
  constexpr bool kCarry = BK >= 64 && NG % 2 == 0;
  float fa[2][FM][4], fx[2][FN][4];
  if constexpr (kCarry) {
#pragma unroll
    for (int b = 0; b < FM; ++b) SA::read_frag(smem + fa_off, 0, b, fa[0][b]);
#pragma unroll
    for (int a = 0; a < FN; ++a) SX::read_frag(smem + fx_off, 0, a, fx[0][a]);
  }
  for (int s = 0; s < total; ++s) {
    const float *as = smem + cur + fa_off;
    const float *xs = smem + cur + fx_off;
    if constexpr (!kCarry) {
#pragma unroll
      for (int b = 0; b < FM; ++b) SA::read_frag(as, 0, b, fa[0][b]);
#pragma unroll
      for (int a = 0; a < FN; ++a) SX::read_frag(xs, 0, a, fx[0][a]);
    }
#pragma unroll
    for (int grp = 0; grp < NG; ++grp) {
      const int c = grp & 1, n = c ^ 1;
      if (grp + 1 < NG) {
#pragma unroll
        for (int b = 0; b < FM; ++b) SA::read_frag(as, grp + 1, b, fa[n][b]);
#pragma unroll
        for (int a = 0; a < FN; ++a) SX::read_frag(xs, grp + 1, a, fx[n][a]);
      } else if constexpr (kCarry) {
        // nothing moves across: the MFMAs of the groups before stay ahead of the barrier, where
        // they cover the latency of the fragment reads the barrier has to wait for
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        cur = kSlab - cur;
        if (s + 1 < total) {
#pragma unroll
          for (int b = 0; b < FM; ++b) SA::read_frag(smem + cur + fa_off, 0, b, fa[n][b]);
#pragma unroll
          for (int a = 0; a < FN; ++a) SX::read_frag(smem + cur + fx_off, 0, a, fx[n][a]);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int a = 0; a < FN; ++a)
#pragma unroll
          for (int b = 0; b < FM; ++b)
            // operands swapped on purpose: the transposed product puts consecutive m in
            // consecutive lanes of every accumulator register
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[c][a][q], fa[c][b][q],
                                                             acc[a][b], 0, 0, 0);
        // the staging work of the slab rides behind MFMAs that are already in the pipe instead
        // of standing between two groups of them
        if (grp == 0 && q == 0 && s + 1 < total) LH_STASH(smem + (kSlab - cur));
        if (grp == 0 && q == 1 && s + 2 < total) LH_ISSUE();
      }
    }
    if constexpr (!kCarry) {
      __syncthreads();
      cur = kSlab - cur;
    }
  }
#undef LH_ISSUE
#undef LH_STASH

  if constexpr (WK > 1) {
    // Fixed-order reduction of the WK partial tiles through LDS (the slab buffers are dead now).
    constexpr int kPerWave = FN * FM * 16 * 64;
    if (wk > 0) {
      float *dst = smem + ((wk - 1) * (WM * WN) + wmn) * kPerWave + lane;
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
#pragma unroll
          for (int j = 0; j < 16; ++j) dst[((a * FM + b) * 16 + j) * 64] = acc[a][b][j];
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
      for (int p = 0; p < WK - 1; ++p) {
        const float *src = smem + (p * (WM * WN) + wmn) * kPerWave + lane;
#pragma unroll
        for (int a = 0; a < FN; ++a)
#pragma unroll
          for (int b = 0; b < FM; ++b)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[a][b][j] += src[((a * FM + b) * 16 + j) * 64];
      }
    }
  }

  if constexpr (CELL) {
    // The four gates of a cell sit in different wavefronts: the tile goes through LDS as
    // S[n][m] (the slab buffers and the partial tiles are dead), then every thread of the
    // workgroup takes cells.
    constexpr int GQ = BM / 4;
    static_assert(smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX>() >= BM * BN, "tile does not fit LDS");
    if constexpr (WK > 1) __syncthreads();  // the partial tiles have been read
    if (wk == 0) {
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            smem[(wn * TN + a * 32 + lhi * 4 + (j / 4) * 8 + (j % 4)) * BM + wm * TM + b * 32 + l32] =
                acc[a][b][j];
    }
    __syncthreads();
    const int H = g.cell_H;
    const bool add = g.beta != 0.f;
    if (g.pre_out) {
      // the product alone, back in the stacked 4H x N layout
      constexpr int kCellsS = GQ * BN;
      for (int idx = tid; idx < kCellsS; idx += NT) {
        const int rl = idx % GQ, nl = idx / GQ;
        const int r = m0 + rl, n = n0 + nl;
        if (r < H && n < g.N) {
          float *o = g.pre_out + (size_t)n * g.pre_ld + r;
#pragma unroll
          for (int q = 0; q < 4; ++q) o[(size_t)q * H] = smem[nl * BM + q * GQ + rl];
        }
      }
      return;
    }
    // A thread's cells: everything they read from memory is fetched first, with independent
    // loads (the outputs may alias c_prev, so loads interleaved with the stores would wait for
    // one another, a memory latency per cell), then the arithmetic, then the stores.
    constexpr int kCells = GQ * BN, kPer = (kCells + NT - 1) / NT;
    float cprev[kPer], mask[kPer], pre[kPer][4];
    bool ok[kPer], f32_gates[kPer];  // f32_gates: bit 1 of the column's mask (see LH_MASK_F32_GATES)
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int idx = tid + i * NT;
      const int rl = idx % GQ, nl = idx / GQ;
      const int r = m0 + rl, n = n0 + nl;
      ok[i] = idx < kCells && r < H && n < g.N;
      cprev[i] = 0.f, mask[i] = 0.f, f32_gates[i] = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) pre[i][q] = 0.f;
      if (ok[i]) {
        int col = n;
        if (g.addend_col) col = min(max(g.addend_col[n], 0), g.addend_ncols - 1);
        const float *ad = g.C + (size_t)col * g.ldc + r;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float v = smem[nl * BM + q * GQ + rl];
          const float t = add ? ad[(size_t)q * H] : 0.f;
          pre[i][q] = (add ? v + t : v) + g.bias[q * H + r];
        }
        cprev[i] = g.c_prev[(size_t)n * H + r];
        const int cm = g.colmask[n];
        mask[i] = (float)(cm & 1);
        f32_gates[i] = (cm & LH_MASK_F32_GATES) != 0;
      }
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int idx = tid + i * NT;
      const int r = m0 + idx % GQ, n = n0 + idx / GQ;
      float c, h;
      if (g.sigmoid_f64 && !f32_gates[i])
        lh::lstm_cell_point<true>(pre[i][0], pre[i][1], pre[i][2], pre[i][3], cprev[i], mask[i],
                                  g.cell_clip, c, h);
      else
        lh::lstm_cell_point<false>(pre[i][0], pre[i][1], pre[i][2], pre[i][3], cprev[i], mask[i],
                                   g.cell_clip, c, h);
      if (ok[i]) {
        const size_t o = (size_t)n * H + r;
        g.c_out[o] = c;
        g.h_out[o] = h;
        if (g.gates_out) {
          float *go = g.gates_out + (size_t)n * 4 * H + r;
#pragma unroll
          for (int q = 0; q < 4; ++q) go[(size_t)q * H] = pre[i][q];  // the cell left i, f, g, o there
        }
        if (g.h_drop) g.h_drop[o] = ((float)(g.drop_mask[o] < g.keep) * (1.0f / g.keep)) * h;
      }
    }
    return;
  }

  if (wk > 0) return;

  // Epilogue: accumulator register j of lane l is C[m = .. + l%32][n = .. + 8*(j/4) + 4*(l/32) + j%4].
  // A split product stores the bare partial sums in its plane of the workspace instead.
  const bool partial = splits > 1;
  const float alpha = partial ? 1.f : g.alpha, beta = g.beta;
  const bool use_beta = !partial && beta != 0.f;
  const int *const colmask = partial ? nullptr : g.colmask;
  const float *const bias = partial ? nullptr : g.bias;
  const int act_rows = partial || g.act != LH_ACT_TANH ? 0 : g.act_rows;
  float *const Cb = partial ? g.ws_part + (size_t)split * g.ws_ld * g.N : g.C;
  const int ldc = partial ? g.ws_ld : g.ldc;
#pragma unroll
  for (int a = 0; a < FN; ++a) {
#pragma unroll
    for (int b = 0; b < FM; ++b) {
      const int m = m0 + wm * TM + b * 32 + l32;
      if (m >= g.M || (RAGGED && m < m_first)) continue;
      const float bv = bias ? bias[m] : 0.f;
      const bool do_tanh = m < act_rows;
      const int nb = n0 + wn * TN + a * 32 + lhi * 4;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int n = nb + (j / 4) * 8 + (j % 4);
        if (n >= g.N || (RAGGED && n < n_first)) continue;
        float *cp = Cb + (size_t)n * ldc + m;
        float v = alpha * acc[a][b][j];
        if (use_beta) v += beta * *cp;
        v += bv;
        if (do_tanh) v = tanhf(v);
        if (colmask) v *= (float)colmask[n];
        *cp = v;
      }
    }
  }
}

// ---- narrow form: products of at most a few 16-column blocks, packed gate products among them --------
// A tile of 16 rows (four cells) x 16 FC columns; the eight wavefronts share its k, 32 of every slab of 256
// each, streamed like stream_body's.  What bounds a gate product of few columns is reading the weights: 32-row
// tiles are 125 workgroups at 1000 hidden units, which leaves half the CUs idle, and the 32x32 MFMA multiplies
// 32 columns whatever there are; these are 250 workgroups with the 16x16x4 MFMA at the same rate per column.
// 1000 hidden units, K = 1000 / 2000, with cell: 12 columns 9.5 / 14.7 us on 32x32 tiles, 6.8 / 9.9 (16 and 32 MB of
// weights, 5.3 TB/s beyond the fixed part); 32 columns 10.1 / 15.3 and 8.6 / 12.3; 256 hidden units, 12 columns, K = 512
// 6.7 and 4.5.  From 1025 hidden units on it would be a second round of workgroups: at 1100 to 1800 units, 1 to 32 columns
// 32-row tiles on part of the CUs take 0.7 to 0.93 of its time (1200 units, 16 columns, K = 2400: 18.8 us and 23.2), at
// 2048 both read the weights at the same rate (16.8 us, K = 2048).
constexpr int kNarrowK = 32, kNarrowSlab = 8 * kNarrowK, kNarrowCells = 4;
constexpr int kNarrowLd = 20;  // floats between the columns of a partial block in LDS
template <int FC>
constexpr int narrow_stages() {
  return FC == 1 ? 4 : 3;
}
template <int FC>
constexpr int narrow_smem_floats() {
  return cmax(narrow_stages<FC>() * kNarrowSlab * 16 * (1 + FC), 8 * 16 * FC * kNarrowLd);
}
typedef float floatx4 __attribute__((ext_vector_type(4)));

// CELL: a packed gate product with its cell; otherwise a plain product with A as stored (TA: transposed), whose
// share of k may be split over workgroups.  1000 x 64 is 252 of these tiles and 64 of 32x32, which were either a
// quarter of the CUs or a split with a reduction behind it: K = 1000 / 2000 9.0 / 11.0 us there (a launch more of 4.5 us
// between other kernels at 2000), 5.9 / 8.9 here; transposed 8.1 / 10.7 and 5.2 / 7.6; 256 x 32, K = 1024 7.9 and 4.9.
template <int FC, bool TA, bool CELL>
__device__ __forceinline__ void narrow_body(const GemmArgs &g, const int logical) {
  constexpr int CK = kNarrowK, SLAB = kNarrowSlab, NB = narrow_stages<FC>(), BN = 16 * FC;
  using PX = Piece<CK, true, 16>;
  static_assert(!(TA && CELL), "packed gate matrices are read as stored");
  constexpr int kA = CK * 16, kStage = kA + FC * PX::kFloats;  // floats
  constexpr int kLoadsA = kA / 256, kLoads = kLoadsA + FC * PX::kLoads;
  const int splits = CELL ? 1 : g.splits, tile = logical / splits, split = logical % splits;
  const int m0 = (tile / g.tiles_n) * 16, n0 = (tile % g.tiles_n) * BN;
  const int cell0 = m0 / 4;  // CELL
  const int tid = threadIdx.x, lane = tid % lh::kWave;
  const int wk = __builtin_amdgcn_readfirstlane(tid / lh::kWave);
  const int l16 = lane % 16, lq = lane / 16;
  float *const ring = smem + wk * NB * kStage;
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)ring;
  const int M = g.M, N = g.N, H = g.cell_H;
  auto pick = [](int seg, auto v0, auto v1, auto v2) __attribute__((always_inline)) {
    return seg == 0 ? v0 : (seg == 1 ? v1 : v2);
  };
#define LH_SEG(FIELD, SEG) pick(SEG, g.FIELD[0], g.FIELD[1], g.FIELD[2])

  // A unit of the ring's A rows: row `pos` of 16 floats is k = 16 (pos / 16) + 4 (pos % 4) + pos / 4 % 4, so that the
  // four k of one MFMA step (4 apart, one per quarter of the wavefront) are neighbouring rows.
  auto a_k = [](int u) __attribute__((always_inline)) { return (u / 64) * 16 + 4 * (u / 4 % 4) + u / 16 % 4; };
  unsigned aoff[kLoadsA];
  PX pa, px[FC];  // pa: TA only
  const int slabs0 = (g.K[0] + SLAB - 1) / SLAB;
  const int slabs1 = g.nseg > 1 ? (g.K[1] + SLAB - 1) / SLAB : 0;
  const int slabs2 = g.nseg > 2 ? (g.K[2] + SLAB - 1) / SLAB : 0;
  const int first = split * g.slabs_per_split;
  const int total = min(g.slabs_per_split, slabs0 + slabs1 + slabs2 - first);
  int lseg = 0, k0 = first, Ks = 0, lda = 0, ldx = 0;
  if (k0 >= slabs0) {
    k0 -= slabs0;
    lseg = 1;
    if (k0 >= slabs1) {
      k0 -= slabs1;
      lseg = 2;
    }
  }
  k0 *= SLAB;
  int cseg = lseg, ck = k0, step_a = 0;
  bool new_seg = true;
  const float *a = nullptr, *x = nullptr;
  unsigned put = ring_lds;
  auto request = [&]() __attribute__((always_inline)) {
    if (new_seg) {
      LH_KEEP_BRANCH();
      Ks = LH_SEG(K, lseg);
      if (lda != LH_SEG(lda, lseg) || ldx != LH_SEG(ldx, lseg)) {
        LH_KEEP_BRANCH();
        lda = LH_SEG(lda, lseg), ldx = LH_SEG(ldx, lseg);
        if constexpr (TA) {
          pa.set_ld(lda, lane, 0, M - m0);
        } else {
#pragma unroll
          for (int i = 0; i < kLoadsA; ++i) {
            const int u = lane + i * 64;
            const unsigned off = (unsigned)(a_k(u) * lda + (u % 4) * 4) * 4u;
            aoff[i] = CELL || (u % 4) * 4 < M - m0 ? off : 0u;  // (a packed block is padded)
          }
        }
        step_a = TA ? SLAB : SLAB * lda;
#pragma unroll
        for (int c = 0; c < FC; ++c) px[c].set_ld(ldx, lane, 16 * c, N - n0);
      }
      const int k = k0 + wk * CK;
      if constexpr (CELL)
        a = LH_SEG(A, lseg) + ((size_t)(cell0 / kPackCells) * Ks + k) * kPackRows + cell0 % kPackCells * 4;
      else a = LH_SEG(A, lseg) + (TA ? (size_t)m0 * lda + k : (size_t)k * lda + m0);
      x = LH_SEG(X, lseg) + (size_t)n0 * ldx + k;
    }
    const int kn = Ks - k0 - wk * CK;
    if (kn < CK) {
      LH_KEEP_BRANCH();
      if (kn <= 0) {
        if constexpr (CELL)
          a = LH_SEG(A, lseg) + (size_t)(cell0 / kPackCells) * Ks * kPackRows + cell0 % kPackCells * 4;
        else a = LH_SEG(A, lseg) + (TA ? (size_t)m0 * lda : (size_t)m0);
        x = LH_SEG(X, lseg) + (size_t)n0 * ldx;
      }
      if constexpr (TA) {
        pa.load_tail(a, put, lda, lane, kn);
      } else {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
          const int k = a_k(lane + i * 64);
          const unsigned back = (unsigned)(k * lda) * 4u;
          PX::load_unit(a, k < kn ? aoff[i] : (aoff[i] >= back ? aoff[i] - back : 0u), put + 1024u * i);
        }
      }
#pragma unroll
      for (int c = 0; c < FC; ++c) px[c].load_tail(x, put + (kA + c * PX::kFloats) * 4u, ldx, lane, kn);
    } else {
      if constexpr (TA) {
        pa.load(a, put);
      } else {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) PX::load_unit(a, aoff[i], put + 1024u * i);
      }
#pragma unroll
      for (int c = 0; c < FC; ++c) px[c].load(x, put + (kA + c * PX::kFloats) * 4u);
    }
    put = put + kStage * 4u == ring_lds + NB * kStage * 4u ? ring_lds : put + kStage * 4u;
    a += step_a;
    x += SLAB;
    k0 += SLAB;
    new_seg = k0 >= Ks;
    if (new_seg) {
      ++lseg;
      k0 = 0;
    }
  };

  int issued = min(total, NB - 1);
  for (int i = 0; i < issued; ++i) request();

  // what the cell reads from memory
  const int rl = tid % kNarrowCells, nl = tid / kNarrowCells;
  const int r = cell0 + rl, n = n0 + nl;
  const bool ep_ok = CELL && tid < kNarrowCells * BN && r < H && n < N;
  float ep_add[4] = {0.f, 0.f, 0.f, 0.f}, ep_bias[4] = {0.f, 0.f, 0.f, 0.f}, ep_c = 0.f;
  int ep_mask = 0;
  if (ep_ok) {
    int col = n;
    if (g.addend_col) col = min(max(g.addend_col[n], 0), g.addend_ncols - 1);
    const float *ad = g.C + (size_t)col * g.ldc + r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (g.beta != 0.f) ep_add[q] = ad[(size_t)q * H];
      ep_bias[q] = g.bias[q * H + r];
    }
    ep_c = g.c_prev[(size_t)n * H + r];
    ep_mask = g.colmask[n];
  }

  floatx4 acc[FC];
#pragma unroll
  for (int c = 0; c < FC; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
  const float *get = ring;
  int cK = LH_SEG(K, cseg);
  for (int s = 0; s < total; ++s) {
    const int behind = issued - 1 - s;
    if (NB > 3 && behind >= 2) wait_loads<kLoads * 2>();
    else if (behind >= 1) wait_loads<kLoads>();
    else wait_loads<0>();
    float fa[CK / 16][4], fx[FC][CK / 16][4];
#pragma unroll
    for (int grp = 0; grp < CK / 16; ++grp) {
#pragma unroll
      for (int q = 0; q < 4 && !TA; ++q) fa[grp][q] = get[(16 * grp + 4 * q + lq) * 16 + l16];
      if constexpr (TA) {
        const float4 t = *reinterpret_cast<const float4 *>(get + (l16 * PX::U + ((4 * grp + lq) ^ PX::swizzle(l16))) * 4);
        fa[grp][0] = t.x, fa[grp][1] = t.y, fa[grp][2] = t.z, fa[grp][3] = t.w;
      }
#pragma unroll
      for (int c = 0; c < FC; ++c) {
        const float4 t = *reinterpret_cast<const float4 *>(
            get + kA + c * PX::kFloats + (l16 * PX::U + ((4 * grp + lq) ^ PX::swizzle(l16))) * 4);
        fx[c][grp][0] = t.x, fx[c][grp][1] = t.y, fx[c][grp][2] = t.z, fx[c][grp][3] = t.w;
      }
    }
    if (issued < total) {
      request();
      ++issued;
    }
    const int kn = cK - ck - wk * CK;
    if (kn < CK) {
      LH_KEEP_BRANCH();
#pragma unroll
      for (int grp = 0; grp < CK / 16; ++grp)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool in = 16 * grp + 4 * lq + q < kn;
          fa[grp][q] = in ? fa[grp][q] : 0.f;
#pragma unroll
          for (int c = 0; c < FC; ++c) fx[c][grp][q] = in ? fx[c][grp][q] : 0.f;
        }
    }
#pragma unroll
    for (int grp = 0; grp < CK / 16; ++grp)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < FC; ++c)
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(fx[c][grp][q], fa[grp][q], acc[c], 0, 0, 0);
    get = get + kStage == ring + NB * kStage ? ring : get + kStage;
    ck += SLAB;
    if (ck >= cK) {
      LH_KEEP_BRANCH();
      ck = 0;
      ++cseg;
      if (s + 1 < total) cK = LH_SEG(K, cseg);
    }
  }
#undef LH_SEG

  __syncthreads();  // all wavefronts have left their rings
#pragma unroll
  for (int c = 0; c < FC; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) smem[(wk * BN + 16 * c + 4 * lq + j) * kNarrowLd + l16] = acc[c][j];
  __syncthreads();
  if constexpr (!CELL) {
    const bool partial = splits > 1;
    const float alpha = partial ? 1.f : g.alpha, beta = partial ? 0.f : g.beta;
    const int *const colmask = partial ? nullptr : g.colmask;
    const float *const bias = partial ? nullptr : g.bias;
    const int act_rows = partial || g.act != LH_ACT_TANH ? 0 : g.act_rows;
    float *const Cb = partial ? g.ws_part + (size_t)split * g.ws_ld * N : g.C;
    const int ldc = partial ? g.ws_ld : g.ldc;
    const int m = m0 + tid % 16, nn = n0 + tid / 16;
    if (tid >= 16 * BN || m >= M || nn >= N) return;
    const float *src = smem + (tid / 16) * kNarrowLd + tid % 16;
    float sum = src[0];
#pragma unroll
    for (int p = 1; p < 8; ++p) sum += src[p * BN * kNarrowLd];
    float *cp = Cb + (size_t)nn * ldc + m;
    float v = alpha * sum;
    if (beta != 0.f) v += beta * *cp;
    if (bias) v += bias[m];
    if (m < act_rows) v = tanhf(v);
    if (colmask) v *= (float)colmask[nn];
    *cp = v;
    return;
  }
  if (!ep_ok) return;
  const float *src = smem + nl * kNarrowLd + rl * 4;
  float4 sum = *reinterpret_cast<const float4 *>(src);
#pragma unroll
  for (int p = 1; p < 8; ++p) {
    const float4 t = *reinterpret_cast<const float4 *>(src + p * BN * kNarrowLd);
    sum.x += t.x, sum.y += t.y, sum.z += t.z, sum.w += t.w;
  }
  float pre[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) pre[q] = (g.beta != 0.f ? pre[q] + ep_add[q] : pre[q]) + ep_bias[q];
  store_cell(g, pre, ep_c, ep_mask, r, n);
}

template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_kernel(const GemmArgs g) {
  if constexpr (BM == 16) {
    static_assert(WM * WN == 1 && WK == 8 && BK == kNarrowSlab && !TX, "the narrow form");
    narrow_body<BN / 16, TA, false>(g, xcd_logical_id());
  } else gemm_body<BM, BN, WM, WN, WK, BK, TA, TX, false, false>(g, xcd_logical_id());
}

// A kernel of its own for ragged operands, told apart by name.
template <int BM, int BN, int WM, int WN, int WK, int BK, bool TA, bool TX, bool RAGGED>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_kernel(const GemmArgs g) {
  static_assert(RAGGED, "aligned operands: the kernel above");
  gemm_body<BM, BN, WM, WN, WK, BK, TA, TX, false, true>(g, xcd_logical_id());
}
using GemmKernel = void (*)(GemmArgs);  // picks one of the two by the template arguments given

// Stacked gate product W*[x; h; h~] (both operands as stored, no transposes) + LSTM cell.
template <int BM, int BN, int WM, int WN, int WK, int BK>
__global__ __launch_bounds__(64 * WM * WN * WK) void gate_gemm_cell_kernel(const GemmArgs g) {
  gemm_body<BM, BN, WM, WN, WK, BK, false, false, true, false>(g, xcd_logical_id());
}

// The same on packed gate matrices (lda = 32).  A tile of 32 rows takes 8 rows of each gate: 32-byte runs of the
// stored matrix, of which a CU fetches whole 64-byte halves of lines: 1.5 times the bytes of the whole product,
// and 50 GB/s per CU (13 TB/s in all) is what the L2s deliver.  Packed, they are one 128-byte line.
// 1000 hidden units, K = 1000 / 2000: 64 columns 12.7 / 20.6 us streamed from the stored matrix, 10.3 / 16.1 packed
// (staged, the way before: 12.7 / 20.3); 12 columns 11.5 / 17.6 and 9.5 / 14.7; 128 columns 16.5 / 27.3 (64-byte runs)
// and 15.6 / 25.4.
template <int BM, int BN, int WM, int WN, int WK, int BK>
__global__ __launch_bounds__(64 * WM * WN * WK) void gate_gemm_packed_kernel(const GemmArgs g) {
  const int logical = xcd_logical_id();
  stream_body<BM, BN, WM, WN, WK, BK, false, false, true, true>(g, (logical / g.tiles_n) * (BM / 4),
                                                                (logical % g.tiles_n) * BN, 0, 1);
}

// 4H x K stacked gate matrix (gates H rows apart) -> ceil(H / 8) blocks of K x 32 (see stream_body).
// Through LDS, so that both sides are whole lines: 32 rows of a gate in, 32 floats of a block out.  Two
// matrices of 4000 x 1000 take 20.5 us (3.1 TB/s), once per change of the weights.
struct PackArgs {
  const float *src[LH_GATE_PACK_MAX];
  float *dst[LH_GATE_PACK_MAX];
  int ld[LH_GATE_PACK_MAX], K[LH_GATE_PACK_MAX];
  int H;
};
constexpr int kPackK = 8;  // k per workgroup
__global__ __launch_bounds__(256) void gate_pack_kernel(const PackArgs p) {
  // a workgroup: 32 cells (four blocks) of kPackK k
  __shared__ float t[kPackK][4][33];
  const int mat = blockIdx.z, H = p.H, K = p.K[mat];
  const int c0 = blockIdx.x * 32, k0 = blockIdx.y * kPackK;
  if (k0 >= K) return;  // the grid covers the deepest matrix
  for (int i = threadIdx.x; i < kPackK * 4 * 32; i += 256) {
    const int c = i % 32, q = i / 32 % 4, k = i / 128;
    t[k][q][c] = c0 + c < H && k0 + k < K ? p.src[mat][(size_t)(k0 + k) * p.ld[mat] + (size_t)q * H + c0 + c] : 0.f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kPackK * 4 * 32; i += 256) {
    const int r = i % kPackRows, k = i / kPackRows % kPackK, b = i / (kPackRows * kPackK);
    if (c0 + b * kPackCells < H && k0 + k < K)
      p.dst[mat][((size_t)(c0 / kPackCells + b) * K + k0 + k) * kPackRows + r] = t[k][r % 4][b * kPackCells + r / 4];
  }
}

// The packed gate product in its narrow form.
template <int FC>
__global__ __launch_bounds__(512) void gate_gemm_narrow_kernel(const GemmArgs g) {
  narrow_body<FC, false, true>(g, xcd_logical_id());
}

// Several stacked gate products of one decoding step in ONE launch: everything that is known when
// the step starts -- each layer's recurrent product W_h h_{t-1}, and the first layer's whole
// pre-activation with its cell -- so that the GPU sees a few thousand tiles at once instead of a
// few hundred per layer one after the other.  Workgroup ids run through the problems' tiles in
// order; a problem either ends in the LSTM cell (CELL body) or stores its 4H x B product.
constexpr int kMaxGroup = LH_GATE_GROUP_MAX;
struct GroupArgs {
  GemmArgs g[kMaxGroup];
  int tiles[kMaxGroup];  // workgroups of each problem
  int cell[kMaxGroup];   // host only
  int n;
};
// Workgroup ids are dealt to the 8 XCDs round-robin.  The problems of a group differ in depth, so
// every XCD takes its eighth of EVERY problem (a contiguous range of that problem's tiles, n
// fastest, so that the tiles sharing a slice of the weights still meet in one L2): the XCDs finish
// together whatever the mix.  The grid is 8 x the largest per-XCD count; the few workgroups
// beyond an XCD's own count leave at once.
template <int BM, int BN, int WM, int WN, int WK, int BK>
__global__ __launch_bounds__(64 * WM * WN * WK) void gate_gemm_group_kernel(const GroupArgs a) {
  const int xcd = blockIdx.x % 8;
  int w = blockIdx.x / 8;
  int p = 0, tile = -1;
  for (; p < a.n; ++p) {
    const int per = a.tiles[p] / 8, rem = a.tiles[p] % 8;
    const int mine = per + (xcd < rem ? 1 : 0);
    if (w < mine) {
      tile = xcd * per + (xcd < rem ? xcd : rem) + w;
      break;
    }
    w -= mine;
  }
  if (tile < 0) return;
  const GemmArgs g = a.g[p];  // one copy into scalar registers: the K loop must not go back to memory
  gemm_body<BM, BN, WM, WN, WK, BK, false, false, true, false>(g, tile);
}

// Whether a configuration's LDS holds a whole tile, which the cell epilogue needs.
template <int BM, int BN, int WM, int WN, int WK, int BK>
constexpr bool cell_capable() {
  return smem2_floats<BM, BN, WM, WN, WK, BK, false, false>() >= BM * BN;
}

// Second half of a split product: C = epilogue(sum of the partial planes, in split order).
// What bounds it at the sizes that split (a few thousand to a few hundred thousand elements) is
// memory latency, not bytes: a thread owns four consecutive rows of one column and has up to eight
// planes' 16-byte loads in flight at once, so the whole launch is one or two round trips.
// One element and one plane at a time it took 12.0 us for 2000 x 12, 11.1 us for 1000 x 64 and 9.4 us for
// 1000 x 128 elements; it takes 4.9, 4.4 and 4.8 us.
constexpr int kReduceBatch = 8;
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const GemmArgs g) {
  const size_t plane = (size_t)g.ws_ld * g.N;
  const int quads = g.ws_ld / 4;  // a plane's columns are padded to whole quads
  const size_t total = (size_t)quads * g.N;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    const int n = (int)(i / quads), m = (int)(i % quads) * 4;
    const float *p = g.ws_part + (size_t)n * g.ws_ld + m;
    const int rows = min(4, g.M - m);
    float *cp = g.C + (size_t)n * g.ldc + m;
    float old[4] = {0.f, 0.f, 0.f, 0.f}, bv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (g.beta != 0.f && r < rows) old[r] = cp[r];
      if (g.bias && r < rows) bv[r] = g.bias[m + r];
    }
    const float cm = g.colmask ? (float)g.colmask[n] : 1.f;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < g.splits; s0 += kReduceBatch) {
      float4 v[kReduceBatch];
#pragma unroll
      for (int s = 0; s < kReduceBatch; ++s)  // past the last plane: that plane again, not added
        v[s] = *reinterpret_cast<const float4 *>(p + (size_t)min(s0 + s, g.splits - 1) * plane);
#pragma unroll
      for (int s = 0; s < kReduceBatch; ++s) {
        if (s0 + s >= g.splits) break;
        acc[0] += v[s].x, acc[1] += v[s].y, acc[2] += v[s].z, acc[3] += v[s].w;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r >= rows) break;
      float o = g.alpha * acc[r];
      if (g.beta != 0.f) o += g.beta * old[r];
      if (g.bias) o += bv[r];
      if (g.act == LH_ACT_TANH && m + r < g.act_rows) o = tanhf(o);
      if (g.colmask) o *= cm;
      cp[r] = o;
    }
  }
}

// ---- configurations -----------------------------------------------------------------------
struct Config {
  int bm, bn, wm, wn, wk, bk;
  bool streamed;
};
// X(index, BM, BN, WM, WN, WK, BK)
#define LH_GEMM_CONFIGS(X)                                                     \
  X(0, 128, 128, 2, 2, 1, 16)  /* large products: output projection         */ \
  X(1, 128, 128, 2, 2, 1, 32)                                                  \
  X(2, 128, 96, 4, 1, 1, 16)                                                   \
  X(3, 128, 64, 2, 2, 1, 16)                                                   \
  X(4, 128, 64, 2, 2, 1, 32)                                                   \
  X(5, 64, 96, 2, 1, 2, 32)    /* stacked gate products at a few hundred columns */ \
  X(6, 64, 96, 2, 1, 2, 64)                                                    \
  X(7, 64, 64, 2, 2, 1, 16)    /* also the only shape of the generic kernel */ \
  X(8, 64, 64, 2, 2, 1, 64)                                                    \
  X(9, 64, 64, 2, 2, 1, 128)                                                   \
  X(10, 32, 96, 1, 3, 2, 32)   /* M around 1000 */                             \
  X(11, 32, 96, 1, 3, 2, 128)                                                  \
  X(12, 32, 64, 1, 2, 4, 32)   /* skinny */                                    \
  X(13, 32, 64, 1, 2, 4, 64)                                                   \
  X(14, 32, 32, 1, 1, 8, 64)   /* very skinny */                               \
  X(15, 32, 32, 1, 1, 8, 128)                                                  \
  X(16, 128, 32, 4, 1, 1, 16)                                                  \
  X(17, 128, 32, 4, 1, 1, 64)                                                  \
  X(18, 64, 32, 2, 1, 4, 32)                                                   \
  X(19, 64, 32, 2, 1, 4, 64)                                                   \
  X(20, 128, 128, 2, 2, 1, 64) /* deep slabs: one workgroup per CU hides its own latency */ \
  X(21, 128, 64, 2, 2, 1, 64)                                                  \
  X(22, 128, 128, 2, 2, 2, 64) /* ... or two wavefronts per SIMD inside the workgroup */ \
  X(23, 128, 64, 2, 2, 2, 64)                                                  \
  X(24, 128, 96, 4, 1, 2, 64)                                                  \
  X(25, 64, 64, 2, 2, 2, 128)                                                  \
  X(26, 256, 128, 4, 2, 1, 16) /* the batched products of training */          \
  X(27, 256, 128, 4, 2, 1, 32)                                                 \
  X(28, 128, 96, 4, 1, 1, 32)  /* more shapes for the output projection */     \
  X(29, 256, 96, 4, 1, 1, 16)                                                  \
  X(30, 256, 96, 4, 1, 1, 32)                                                  \
  X(31, 128, 96, 4, 1, 2, 32)  /* between the shallow and the deep slabs */    \
  X(32, 128, 64, 2, 2, 2, 32)                                                  \
  X(33, 64, 96, 2, 1, 4, 64)                                                   \
  X(34, 128, 128, 2, 2, 2, 32)                                                 \
  X(35, 64, 64, 2, 2, 2, 64)                                                   \
  X(36, 64, 64, 2, 2, 4, 128)  /* small tiles with 8-16 wavefronts */          \
  X(37, 32, 96, 1, 3, 4, 64)                                                   \
  X(38, 64, 96, 2, 1, 4, 32)                                                   \
  X(39, 128, 64, 2, 2, 4, 64)                                                  \
  X(40, 128, 96, 4, 1, 4, 64)                                                  \
  X(41, 96, 96, 3, 1, 4, 64)   /* three wavefronts along m, twelve in all (three per SIMD): 42 row tiles of the stacked gates at H = 1000 */ \
  X(42, 96, 64, 3, 1, 4, 64)                                                   \
  X(43, 64, 160, 2, 1, 4, 64)  /* 252 tiles of the stacked gates at 580-640 columns */ \
  X(44, 64, 32, 2, 1, 4, 128)  /* few columns against an A that comes from HBM */

#define LH_CFG_ENTRY(I, BM, BN, WM, WN, WK, BK) {BM, BN, WM, WN, WK, BK, streamed<BM, BN, WM, WN, WK, BK>()},
const Config kConfigs[] = {LH_GEMM_CONFIGS(LH_CFG_ENTRY)};
#undef LH_CFG_ENTRY
constexpr int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);
constexpr int kUnalignedConfig = 7;
// The narrow forms, numbered behind them.
const Config kNarrow[] = {{16, 16, 1, 1, 8, kNarrowSlab, false}, {16, 32, 1, 1, 8, kNarrowSlab, false}};
constexpr int kNumNarrow = sizeof(kNarrow) / sizeof(kNarrow[0]);
const Config &config_at(int c) { return c < kNumConfigs ? kConfigs[c] : kNarrow[c - kNumConfigs]; }
// Configurations built for ragged operands as well: those that the cost model gives an aligned output
// projection and its backward products at 5 to 2560 columns of 5000 to 30000 words, or one within
// a few per cent of them.  All of them run the staged form, 15 too, whose aligned
// form is streamed.  In the cost model 12, 15 and 18 have rows of their own: loads that start at any float cost these most
// (32x64: 0.0197 us per k where aligned operands take 0.0115).  With the rows of the aligned kernels 340 products of 30 to
// 30003 rows or words, 1 to 768 columns took 1.021 times the time of the best of a sweep over configurations and splits,
// 1.49 at worst; with these 1.008 and 1.17.  Rows for all ten are no better there, and put 64x64 behind 128x64 where a
// large result has a short K (8830 x 1538, K = 24: 21.4 us and 26.2).
constexpr bool ragged_config(int c) {
  return c == 0 || c == 3 || c == 7 || c == 12 || c == 15 || c == 18 || c == 24 || c == 32 || c == 35 || c == 36;
}

template <typename KernelT>
int launch_kernel(KernelT kernel, int smem_bytes, dim3 grid, dim3 block, hipStream_t st,
                  const GemmArgs &g) {
  if (smem_bytes > 64 * 1024) {
    // more dynamic LDS than the default limit: raised once per kernel instance
    static thread_local const void *raised[64];
    static thread_local int n_raised = 0;
    bool done = false;
    for (int i = 0; i < n_raised; ++i) done = done || raised[i] == (const void *)kernel;
    if (!done) {
      hipError_t e = hipFuncSetAttribute((const void *)kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, smem_bytes);
      if (e != hipSuccess) {
        (void)hipGetLastError();
        return lh::fail_arg("lh_gemm_f32: cannot reserve %d bytes of LDS: %s", smem_bytes,
                            hipGetErrorString(e));
      }
      if (n_raised < 64) raised[n_raised++] = (const void *)kernel;
    }
  }
  hipLaunchKernelGGL(kernel, grid, block, smem_bytes, st, g);
  return lh::check_launch("lh_gemm_f32");
}

// The sum of the partial planes of a split product.
int launch_reduce(const GemmArgs &g, hipStream_t st) {
  // four rows per thread; small products in single-wavefront workgroups, to reach more CUs
  const size_t total = (size_t)(g.ws_ld / 4) * g.N;
  const unsigned nt = total < 65536 ? 64 : 256;
  const size_t blocks = (total + nt - 1) / nt;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(nt), 0, st, g);
  return lh::check_launch("lh_gemm_ws_f32 split reduction");
}

// Shares of the K slabs of a product (bk deep, none across two segments) that is to be split `want` ways: slabs of a
// share, and how many shares hold any.
struct Shares {
  int slabs, n;
};
Shares shares_of(const int *K, int nseg, int bk, int want) {
  int slabs = 0;
  for (int s = 0; s < nseg; ++s) slabs += (K[s] + bk - 1) / bk;
  const int share = (slabs + want - 1) / want;
  return {share, (slabs + share - 1) / share};
}

// What takes a product: the scalar kernel, the main kernel for aligned operands, or its form for
// ragged ones.
enum Form { kGeneric, kRagged, kAligned };

template <int BM, int BN, int WM, int WN, int WK, int BK, bool ALLOW_UNALIGNED, bool ALLOW_RAGGED>
int launch_cfg(const GemmArgs &g0, bool ta, bool tx, Form form, hipStream_t st) {
  GemmArgs g = g0;
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  if (form == kGeneric) g.splits = 1;
  const Shares shares = shares_of(g.K, g.nseg, BK, g.splits);
  g.slabs_per_split = shares.slabs, g.splits = shares.n;
  const dim3 grid(g.tiles_m * g.tiles_n * g.splits), block(64 * WM * WN * WK);
  if (form != kGeneric) {
    int rc = LH_OK;
    if (form == kRagged) {
      if constexpr (!ALLOW_RAGGED) {
        return lh::fail_arg("lh_gemm_f32: internal error, ragged operands reached an aligned-only tile");
      } else {
#define LH_GEMM_LAUNCH(TA, TX)                                                              \
  rc = launch_kernel((GemmKernel)gemm_kernel<BM, BN, WM, WN, WK, BK, TA, TX, true>,         \
                     smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX, true>() * 4, grid, block, st, g)
        if (!ta && !tx) LH_GEMM_LAUNCH(false, false);
        else if (ta) LH_GEMM_LAUNCH(true, false);
        else LH_GEMM_LAUNCH(false, true);
#undef LH_GEMM_LAUNCH
      }
    } else {
#define LH_GEMM_LAUNCH(TA, TX)                                                              \
  rc = launch_kernel((GemmKernel)gemm_kernel<BM, BN, WM, WN, WK, BK, TA, TX>,               \
                     smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX>() * 4, grid, block, st, g)
      if (!ta && !tx) LH_GEMM_LAUNCH(false, false);
      else if (ta) LH_GEMM_LAUNCH(true, false);
      else LH_GEMM_LAUNCH(false, true);
#undef LH_GEMM_LAUNCH
    }
    if (rc != LH_OK || g.splits == 1 || g.leave_partial) return rc;
    return launch_reduce(g, st);
  }
  if constexpr (ALLOW_UNALIGNED) {
    constexpr int bytes = smem_floats<BM, BN, WK, BK>() * 4;
#define LH_GEMM_LAUNCH(TA, TX) \
  return launch_kernel(gemm_generic_kernel<BM, BN, WM, WN, WK, BK, TA, TX, false>, bytes, grid, block, st, g)
    if (!ta && !tx) LH_GEMM_LAUNCH(false, false);
    else if (ta) LH_GEMM_LAUNCH(true, false);
    else LH_GEMM_LAUNCH(false, true);
#undef LH_GEMM_LAUNCH
  }
  return lh::fail_arg("lh_gemm_f32: internal error, unaligned operands reached an aligned-only tile");
}

template <int FC>
int launch_narrow_gemm(const GemmArgs &g0, bool ta, hipStream_t st) {
  GemmArgs g = g0;
  g.tiles_m = (g.M + 15) / 16;
  g.tiles_n = (g.N + 16 * FC - 1) / (16 * FC);
  const Shares shares = shares_of(g.K, g.nseg, kNarrowSlab, g.splits);
  g.slabs_per_split = shares.slabs, g.splits = shares.n;
  const dim3 grid(g.tiles_m * g.tiles_n * g.splits);
  const int rc = ta ? launch_kernel((GemmKernel)gemm_kernel<16, 16 * FC, 1, 1, 8, kNarrowSlab, true, false>,
                                    narrow_smem_floats<FC>() * 4, grid, dim3(512), st, g)
                    : launch_kernel((GemmKernel)gemm_kernel<16, 16 * FC, 1, 1, 8, kNarrowSlab, false, false>,
                                    narrow_smem_floats<FC>() * 4, grid, dim3(512), st, g);
  return rc != LH_OK || g.splits == 1 || g.leave_partial ? rc : launch_reduce(g, st);
}

int launch_index(int c, const GemmArgs &g, bool ta, bool tx, Form form, hipStream_t st) {
  if (c == kNumConfigs) return launch_narrow_gemm<1>(g, ta, st);
  if (c == kNumConfigs + 1) return launch_narrow_gemm<2>(g, ta, st);
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I:                                      \
    return launch_cfg<BM, BN, WM, WN, WK, BK, I == kUnalignedConfig, ragged_config(I)>(g, ta, tx, form, st);
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return lh::fail_arg("lh_gemm_f32: configuration %d does not exist", c);
  }
}

template <int BM, int BN, int WM, int WN, int WK, int BK>
int launch_cell_cfg(const GemmArgs &g0, hipStream_t st) {
  if constexpr (cell_capable<BM, BN, WM, WN, WK, BK>()) {
    GemmArgs g = g0;
    g.tiles_m = (g.cell_H + BM / 4 - 1) / (BM / 4);
    g.tiles_n = (g.N + BN - 1) / BN;
    g.splits = 1;
    g.slabs_per_split = 0;
    for (int s = 0; s < g.nseg; ++s) g.slabs_per_split += (g.K[s] + BK - 1) / BK;
    const dim3 grid(g.tiles_m * g.tiles_n), block(64 * WM * WN * WK);
    return launch_kernel(gate_gemm_cell_kernel<BM, BN, WM, WN, WK, BK>,
                         smem2_floats<BM, BN, WM, WN, WK, BK, false, false>() * 4, grid, block, st, g);
  } else {
    return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: internal error, tile %dx%d cannot hold the cell", BM, BN);
  }
}

template <int BM, int BN, int WM, int WN, int WK, int BK>
int launch_packed_cfg(const GemmArgs &g0, hipStream_t st) {
  if constexpr (streamed<BM, BN, WM, WN, WK, BK>()) {
    GemmArgs g = g0;
    g.tiles_m = (g.cell_H + BM / 4 - 1) / (BM / 4);
    g.tiles_n = (g.N + BN - 1) / BN;
    g.splits = 1;
    g.slabs_per_split = 0;
    for (int s = 0; s < g.nseg; ++s) g.slabs_per_split += (g.K[s] + BK - 1) / BK;
    return launch_kernel(gate_gemm_packed_kernel<BM, BN, WM, WN, WK, BK>,
                         smem2_floats<BM, BN, WM, WN, WK, BK, false, false>() * 4, dim3(g.tiles_m * g.tiles_n),
                         dim3(64 * WM * WN * WK), st, g);
  } else {
    return lh::fail_arg("lh_gate_gemm_lstm_cell_packed_f32: internal error, configuration %dx%d", BM, BN);
  }
}

template <int FC>
int launch_narrow(const GemmArgs &g0, hipStream_t st) {
  GemmArgs g = g0;
  g.tiles_m = (g.cell_H + kNarrowCells - 1) / kNarrowCells;
  g.tiles_n = (g.N + 16 * FC - 1) / (16 * FC);
  g.slabs_per_split = 0;
  for (int s = 0; s < g.nseg; ++s) g.slabs_per_split += (g.K[s] + kNarrowSlab - 1) / kNarrowSlab;
  return launch_kernel(gate_gemm_narrow_kernel<FC>, narrow_smem_floats<FC>() * 4, dim3(g.tiles_m * g.tiles_n),
                       dim3(512), st, g);
}

int launch_packed_index(int c, const GemmArgs &g, hipStream_t st) {
  if (c == kNumConfigs) return launch_narrow<1>(g, st);
  if (c == kNumConfigs + 1) return launch_narrow<2>(g, st);
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I: return launch_packed_cfg<BM, BN, WM, WN, WK, BK>(g, st);
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return lh::fail_arg("lh_gate_gemm_lstm_cell_packed_f32: configuration %d does not exist", c);
  }
}

int launch_cell_index(int c, const GemmArgs &g, hipStream_t st) {
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I: return launch_cell_cfg<BM, BN, WM, WN, WK, BK>(g, st);
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: configuration %d does not exist", c);
  }
}

bool cell_capable_index(int c) {
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I: return cell_capable<BM, BN, WM, WN, WK, BK>();
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return false;
  }
}

int occupancy(GemmKernel kernel, int block, int bytes, int *blocks_per_cu, int *lds_bytes) {
  *lds_bytes = bytes;
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, kernel, block, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return lh::fail_arg("lh_gemm_config_info: occupancy query failed: %s", hipGetErrorString(e));
  }
  return LH_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int BK>
int occupancy_cfg(bool ta, bool tx, int *blocks_per_cu, int *lds_bytes) {
#define LH_GEMM_OCC(TA, TX)                                                                            \
  return occupancy(gemm_kernel<BM, BN, WM, WN, WK, BK, TA, TX>, 64 * WM * WN * WK,                     \
                   smem2_floats<BM, BN, WM, WN, WK, BK, TA, TX>() * 4, blocks_per_cu, lds_bytes)
  if (!ta && !tx) LH_GEMM_OCC(false, false);
  if (ta) LH_GEMM_OCC(true, false);
  LH_GEMM_OCC(false, true);
#undef LH_GEMM_OCC
}

template <int FC>
int occupancy_narrow(bool ta, bool tx, int *blocks_per_cu, int *lds_bytes) {
  if (tx) return lh::fail_arg("lh_gemm_config_info: the narrow forms take no transposed X");
  return occupancy(ta ? (GemmKernel)gemm_kernel<16, 16 * FC, 1, 1, 8, kNarrowSlab, true, false>
                      : (GemmKernel)gemm_kernel<16, 16 * FC, 1, 1, 8, kNarrowSlab, false, false>,
                   512, narrow_smem_floats<FC>() * 4, blocks_per_cu, lds_bytes);
}

int occupancy_index(int c, bool ta, bool tx, int *blocks_per_cu, int *lds_bytes) {
  if (c == kNumConfigs) return occupancy_narrow<1>(ta, tx, blocks_per_cu, lds_bytes);
  if (c == kNumConfigs + 1) return occupancy_narrow<2>(ta, tx, blocks_per_cu, lds_bytes);
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I: return occupancy_cfg<BM, BN, WM, WN, WK, BK>(ta, tx, blocks_per_cu, lds_bytes);
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return lh::fail_arg("lh_gemm_config_info: configuration %d does not exist", c);
  }
}

// Tuning / test aids, see lh_gemm_set_config_override.  Per thread: a tuner or a test on one host
// thread must not change the tiles another thread's model is running with.
thread_local int g_config_override = -1;
thread_local int g_splits_override = 0;

constexpr int kMaxSplits = 16;

// Leading dimension of a partial plane, and the largest split count <= want whose planes fit.
int plane_ld(int M) { return (M + 3) & ~3; }
int fit_splits(int M, int N, int want, size_t workspace_bytes) {
  if (want <= 1) return 1;
  const size_t plane = (size_t)plane_ld(M) * N * sizeof(float);
  const size_t fit = workspace_bytes / plane;
  const size_t s = fit < (size_t)want ? fit : (size_t)want;
  return s < 1 ? 1 : (int)(s > kMaxSplits ? kMaxSplits : s);
}

// ---- choice of tile configuration and K split ------------------------------------------------
// Cost model over a measured table.  For one configuration, T1(K) is the time of a launch that
// gives every CU a single workgroup and Tocc(K) of one that gives every CU as many as fit at once
// (both linear in the K depth of a workgroup's share).  A product whose fullest CU receives n
// workgroups then takes about (n / occ) * Tocc + T(n % occ), T interpolated between T1 and Tocc;
// a split adds the pass that sums the partial planes.  The cheapest (configuration, split) wins.
struct Tuning {
  int occ;           // workgroups resident per CU
  float f1, s1;      // one workgroup per CU: fixed us, us per k
  float focc, socc;  // CU full
};
struct TuningRow {
  int config;
  Tuning t;
};
#include "gemm_tuning.inc"
// The row of a configuration in one of the tables that hold few of them, null where it has none.
template <size_t N>
const Tuning *row_of(const TuningRow (&rows)[N], int config) {
  for (const TuningRow &r : rows)
    if (r.config == config) return &r.t;
  return nullptr;
}
constexpr int kCUs = 256;
// The pass over S partial planes: 4.3 to 4.8 us of 4 planes between other kernels of a stream (1000 x 64 to 2048 x 256),
// 2.1, 2.6 and 3.8 us of 2, 4 and 8 planes of 1000 x 5 and 1.4 us less a launch when replayed from a graph.
constexpr float kReduceFixedUs = 3.5f, kReducePlaneUs = 0.22f, kReduceBytesPerUs = 3.0e6f;
// The LSTM cell as a launch of its own behind its product (us): 4.1 to 4.7 us between other kernels at 12 columns, and 7.2
// and a lookup of 4.6 where the addend is a column of the embedding table.  Behind a short product the dearer price holds
// (the host, which issues two launches for one, is no faster than they are); behind a longer one it made 15 of 240 gate
// products of 64 to 2048 hidden units, 1 to 256 columns 5 % slower or more than the split product they had been, 16 % at
// worst, all of 26 us or longer; now 1 of them, 6 %.
float cell_launch_us(float product_us, int H, int B) {
  return (product_us < 16.f ? 6.f : 4.f) + 28.f * (float)H * (float)B / kReduceBytesPerUs;
}

// What the K loop costs more where its operands come from beyond the L2s, which the table does not show.  A streamed
// wavefront takes a transposed A in 64-byte runs, one per row, and its ring covers the latency of an L2 but not that of
// HBM: from 48 MB of operands on (35 products of 400 to 2000 rows, K = 6000 to 30000) its loop takes 1.28 times the time
// of the table at the median, 1.6 in the worst tenth; with A as stored, in runs of 128 bytes, 1.1 times what staged tiles
// take.  Staged tiles stay within 0.06 of the table, and below 8 MB so do all.
// Transposed, 1536 x 21, K = 8460: 26.1 us on 32x32, 23.3 on staged 64x32; 996 x 109, K = 11516 47.6 and 37.9 (64x64);
// 2048 x 64, K = 8192 33.6 and 30.5.
// The narrow tiles lose the most: a workgroup per CU reads 16 rows and nothing hides it.  Transposed, 1000 x 64, K = 4000
// takes 10.2 us on 16x16 where one matrix is read again and again and 12.3 where twenty take turns (32x32 split in four:
// 12.0 and 14.7), 2000 x 64, K = 8000 29.6 and 39.1 (64x64: 24.2 and 30.0).
// The stored gate matrix of a product with its cell is runs of 32 bytes (8 rows of a gate) and costs what a transposed A
// does: 1.36 at the median of 78 products of at most a workgroup per CU, where staged tiles take 1.06 and packed matrices
// 1.12 (no price for those).  1956 hidden units, 58 columns, K = 3912: 69 us on streamed 64x32, 60 on the staged one, 51
// split with a cell kernel behind.
float cold_share(const Config &k, bool short_runs, int M, int N, const int *K, int nseg) {
  const bool narrow = k.bm == 16;
  if (!k.streamed && !narrow) return 0.f;
  float mb = 0.f;
  for (int s = 0; s < nseg; ++s) mb += 4.0e-6f * (float)K[s] * ((float)M + (float)N);
  return fminf(fmaxf((mb - 8.f) / 24.f, 0.f), 1.f) * (narrow ? 0.5f : (short_runs ? 0.3f : 0.1f));
}

float predict_us(const Tuning &t, const Config &k, int M, int N, const int *K, int nseg, int want,
                 bool reduce_free, int *splits, float cold = 0.f) {
  const long long tiles = (long long)((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn);
  const Shares shares = shares_of(K, nseg, k.bk, want);
  const int S = shares.n;
  *splits = S;
  const float depth = (float)shares.slabs * k.bk;
  // Workgroups per CU: dispatch is dynamic, so a fractional load costs less than a whole extra
  // round but leaves a tail of about half a workgroup.
  const float per_cu = (float)(tiles * S) / kCUs;
  // Not so on streamed tiles: two of their workgroups on a CU do not finish one after the other (and where only one fits,
  // a last round takes as long as any).  1400 x 192, K = 2800 (264 workgroups of 32x32, two to a CU) 30.5 us, 26.1 on the
  // 64x64 tiles that a fractional load would have passed over.
  const float load = k.streamed ? ceilf(per_cu) : fminf(per_cu + 0.5f, ceilf(per_cu));
  // (both are fitted at depths of 512 and 4096: below, several workgroups could come out cheaper than one)
  const float t1 = t.f1 + t.s1 * depth, full = t.focc + t.socc * depth;
  const float tocc = t.occ > 1 ? fmaxf(t1, full) : full;
  const float rounds = floorf(load / (float)t.occ);
  const float rest = load - rounds * (float)t.occ;
  float us = rounds * tocc;
  if (rest > 1e-6f)
    us += rest <= 1.f || t.occ == 1 ? t1 : t1 + (tocc - t1) * (rest - 1.f) / (float)(t.occ - 1);
  us += cold * (us - t.f1);
  if (S > 1 && !reduce_free)
    us += kReduceFixedUs + kReducePlaneUs * (float)S + (float)(S + 1) * (float)M * (float)N * 4.f / kReduceBytesPerUs;
  if (S > 1 && reduce_free)  // the consumer reads S planes instead of one matrix
    us += (float)(S - 1) * (float)M * (float)N * 4.f / kReduceBytesPerUs;
  return us;
}

// max_planes > 0: the caller consumes up to that many partial planes itself (no reduction pass).
// only_cell: restrict the choice to unsplit launches of configurations whose LDS holds a whole
// tile (what the gate product with the cell in its epilogue can use).  *us (optional) receives
// the predicted time of the choice.
// Ragged operands: max_bm / max_bn are the largest tile extents allowed (a ragged extent must hold a
// whole tile), INT_MAX where the extent is a multiple of 4.
void pick_config(int M, int N, const int *K, int nseg, bool ta, bool tx, Form form,
                 size_t workspace_bytes, int max_planes, int *config, int *splits,
                 bool only_cell = false, float *us_out = nullptr, int max_bm = INT_MAX,
                 int max_bn = INT_MAX, bool allow_narrow = true) {
  *splits = 1;
  if (us_out) *us_out = 0.f;
  if (form == kGeneric) {
    *config = kUnalignedConfig;
    return;
  }
  // The decoder repeats a handful of problems thousands of times: remember the answers.
  struct Memo {
    int M, N, K[LH_GEMM_MAX_SEGS], flags, config, splits;
    size_t workspace_bytes;
    float us;
  };
  static thread_local Memo memo[64];
  const int flags = 1 + (ta ? 2 : 0) + (tx ? 4 : 0) + 8 * nseg + 64 * (g_config_override + 1) +
                    4096 * g_splits_override + 131072 * max_planes + (only_cell ? 1048576 : 0) +
                    (max_bm <= M ? 2097152 : 0) + (max_bn <= N ? 4194304 : 0) +
                    (form == kRagged ? 8388608 : 0) + (allow_narrow ? 16777216 : 0);
  int Kk[LH_GEMM_MAX_SEGS] = {0, 0, 0};
  for (int s = 0; s < nseg; ++s) Kk[s] = K[s];
  // Every field into every bit of the slot: the two questions a gate product asks (any launch; an unsplit
  // one that can carry the cell) once shared a slot, each overwrote the other's answer, and a plan took 5.7 us of
  // host time; it takes 0.2.  The workspace is among them: an encoder lane and the main stream ask for the same
  // products with unlike ones.
  unsigned h = 2166136261u;
  for (const int v : {M, N, Kk[0], Kk[1], Kk[2], flags, (int)(workspace_bytes >> 8)})
    h = (h ^ (unsigned)v) * 2654435761u, h ^= h >> 15;
  Memo &e = memo[h % 64];
  if (e.flags == flags && e.M == M && e.N == N && e.K[0] == Kk[0] && e.K[1] == Kk[1] &&
      e.K[2] == Kk[2] && e.workspace_bytes == workspace_bytes) {
    *config = e.config;
    *splits = e.splits;
    if (us_out) *us_out = e.us;
    return;
  }
  static const int kSplitChoices[] = {1, 2, 3, 4, 6, 8, 12, 16};
  // the fourth table is measured on the kernel that carries the LSTM cell in its epilogue
  const Tuning *table = kTuning[only_cell ? 3 : (ta ? 1 : (tx ? 2 : 0))];
  float best = 3.0e38f;
  *config = kUnalignedConfig;
  for (int c = 0; c < kNumConfigs + kNumNarrow; ++c) {
    if (g_config_override >= 0 && c != g_config_override) continue;
    const bool narrow = c >= kNumConfigs;
    if (narrow && (!allow_narrow || only_cell || tx || form != kAligned)) break;
    if (only_cell && !cell_capable_index(c)) continue;
    if (form == kRagged && (!ragged_config(c) || kConfigs[c].bm > max_bm || kConfigs[c].bn > max_bn)) continue;
    const Tuning *t = form == kRagged ? row_of(kRaggedTuning[ta ? 1 : (tx ? 2 : 0)], c)
                      : narrow        ? row_of(kNarrowTuning[ta ? 1 : 0], c)
                                      : nullptr;
    if (!t && narrow) break;
    if (!t) t = &table[c];
    const float cold = tx || form != kAligned ? 0.f : cold_share(config_at(c), ta || only_cell, M, N, K, nseg);
    for (int want : kSplitChoices) {
      if (only_cell && want > 1) break;
      if (!only_cell && g_splits_override > 0) want = fit_splits(M, N, g_splits_override, workspace_bytes);
      if (max_planes > 0 && want > max_planes) want = max_planes;
      if (want > 1 && fit_splits(M, N, want, workspace_bytes) < want) break;
      int S;
      float us = predict_us(*t, config_at(c), M, N, K, nseg, want, max_planes > 0, &S, cold);
      // an override asks for this many shares: too few slabs for them only where no other choice has enough
      if (g_splits_override > 0 && S < want) us += 1.0e6f;
      if (us < best) {
        best = us;
        *config = c;
        *splits = S;
      }
      if (g_splits_override > 0 || (max_planes > 0 && want >= max_planes)) break;
    }
  }
  if (best > 2.9e38f) *config = -1;  // the override names a configuration that cannot run this
  if (us_out) *us_out = best;
  e = Memo{M, N, {Kk[0], Kk[1], Kk[2]}, flags, *config, *splits, workspace_bytes, best};
}

// The packed gate product's configuration and predicted time.
void pick_packed(int H, int B, const int *K, int nseg, int *config, float *us) {
  *config = -1;
  *us = 3.0e38f;
  for (const TuningRow &r : kPackedTuning) {
    if (g_config_override >= 0 && r.config != g_config_override) continue;
    int S;
    const float t = predict_us(r.t, config_at(r.config), 4 * H, B, K, nseg, 1, false, &S);
    if (t < *us) *us = t, *config = r.config;
  }
}

struct Prepared {
  GemmArgs g;
  bool ta, tx;
  Form form;
  int config;
};

int prepare(int M, int N, const lh_gemm_seg *segs, int nseg, int transA, int transX, float alpha,
            float beta, const float *bias, int act, int act_rows, const int *colmask, float *C,
            int ldc, void *workspace, size_t workspace_bytes, int max_planes, Prepared *out) {
  if (M <= 0 || N <= 0) return lh::fail_arg("lh_gemm_f32: M=%d N=%d must be positive", M, N);
  if (!segs || nseg < 1 || nseg > LH_GEMM_MAX_SEGS)
    return lh::fail_arg("lh_gemm_f32: nseg=%d outside [1,%d]", nseg, LH_GEMM_MAX_SEGS);
  if (transA && transX) return lh::fail_arg("lh_gemm_f32: transA && transX is not supported");
  if (act != LH_ACT_NONE && act != LH_ACT_TANH) return lh::fail_arg("lh_gemm_f32: act=%d", act);
  if (!C || ldc < M) return lh::fail_arg("lh_gemm_f32: C=%p ldc=%d (M=%d)", (void *)C, ldc, M);

  GemmArgs &g = out->g;
  g = GemmArgs{};
  bool vec = true, aligned = true;
  for (int s = 0; s < nseg; ++s) {
    const lh_gemm_seg &e = segs[s];
    if (!e.A || !e.X || e.K <= 0)
      return lh::fail_arg("lh_gemm_f32: segment %d has A=%p X=%p K=%d", s, (const void *)e.A,
                          (const void *)e.X, e.K);
    const int min_lda = transA ? e.K : M, min_ldx = transX ? N : e.K;
    if (e.lda < min_lda || e.ldx < min_ldx)
      return lh::fail_arg("lh_gemm_f32: segment %d lda=%d (min %d) ldx=%d (min %d)", s, e.lda,
                          min_lda, e.ldx, min_ldx);
    g.A[s] = e.A;
    g.X[s] = e.X;
    g.lda[s] = e.lda;
    g.ldx[s] = e.ldx;
    g.K[s] = e.K;
    const int a_extent = transA ? e.K : M, x_extent = transX ? N : e.K;
    // the main kernel keeps per-thread byte offsets inside a slab in 32 bits
    constexpr int kMaxLd = 1 << 22;
    vec = vec && e.lda < kMaxLd && e.ldx < kMaxLd;
    aligned = aligned && lh::aligned16(e.A) && lh::aligned16(e.X) && e.lda % 4 == 0 &&
              e.ldx % 4 == 0 && a_extent % 4 == 0 && x_extent % 4 == 0;
    // a unit along k that is short of four values reaches back inside its row
    if ((transA || !transX) && e.K < 4) vec = false;
  }
  // One 16-deep slab is all the scalar kernel has to do, too: 30003 x 1000, K = 16, 29.6 us there and 37.7
  // here, 130 x 33 5.7 and 6.1, 1002 x 1000 6.4 and 6.2; at K = 18 40 and 43, 6.5 and 6.2, 7.3 and 6.8.
  if (!aligned && nseg == 1 && segs[0].K <= 16) vec = false;
  // A tile along a ragged m (n) moves back inside the operand: it must be at least a tile long.  The
  // narrowest tiles are 32 wide; below that the scalar kernel runs a single row of tiles anyway.
  const bool ragged_m = !transA && M % 4 != 0, ragged_n = transX && N % 4 != 0;
  if ((ragged_m && M < 32) || (ragged_n && N < 32)) vec = false;
  g.ragged_m = ragged_m ? 1 : 0;
  g.ragged_n = ragged_n ? 1 : 0;
  for (int s = nseg; s < LH_GEMM_MAX_SEGS; ++s) {  // unused slots mirror segment 0 (never read)
    g.A[s] = g.A[0];
    g.X[s] = g.X[0];
    g.lda[s] = g.lda[0];
    g.ldx[s] = g.ldx[0];
    g.K[s] = g.K[0];
  }
  g.nseg = nseg;
  g.M = M;
  g.N = N;
  g.alpha = alpha;
  g.beta = beta;
  g.bias = bias;
  g.act = act;
  g.act_rows = act_rows;
  g.colmask = colmask;
  g.C = C;
  g.ldc = ldc;
  out->ta = transA != 0;
  out->tx = transX != 0;
  if (!workspace || !lh::aligned16(workspace)) workspace_bytes = 0;
  out->form = !vec ? kGeneric : (aligned ? kAligned : kRagged);
  pick_config(M, N, g.K, nseg, transA != 0, transX != 0, out->form, workspace_bytes, max_planes,
              &out->config, &g.splits, false, nullptr, ragged_m ? M : INT_MAX, ragged_n ? N : INT_MAX);
  if (out->config < 0) {  // the configuration override does not fit a ragged operand
    out->form = kGeneric;
    out->config = kUnalignedConfig;
    g.splits = 1;
  }
  g.leave_partial = max_planes > 0 ? 1 : 0;
  g.ws_part = static_cast<float *>(workspace);
  g.ws_ld = plane_ld(M);
  return LH_OK;
}

}  // namespace

extern "C" int lh_gemm_ws_f32(int M, int N, const lh_gemm_seg *segs, int nseg, int transA,
                              int transX, float alpha, float beta, const float *bias, int act,
                              int act_rows, const int *colmask, float *C, int ldc, void *workspace,
                              size_t workspace_bytes, lh_stream_t stream) {
  if (act_rows < 0 || act_rows > M)
    return lh::fail_arg("lh_gemm_f32: act_rows=%d outside [0,M=%d]", act_rows, M);
  Prepared p;
  const int rc = prepare(M, N, segs, nseg, transA, transX, alpha, beta, bias, act, act_rows,
                         colmask, C, ldc, workspace, workspace_bytes, 0, &p);
  if (rc != LH_OK) return rc;
  return launch_index(p.config, p.g, p.ta, p.tx, p.form, lh::as_stream(stream));
}

extern "C" int lh_gemm_planes_f32(int M, int N, const lh_gemm_seg *segs, int nseg, int transA,
                                  int transX, float beta, float *C, int ldc, void *workspace,
                                  size_t workspace_bytes, int max_planes, int *planes,
                                  lh_stream_t stream) {
  if (!planes || max_planes < 1)
    return lh::fail_arg("lh_gemm_planes_f32: planes=%p max_planes=%d", (void *)planes, max_planes);
  Prepared p;
  const int rc = prepare(M, N, segs, nseg, transA, transX, 1.f, beta, nullptr, LH_ACT_NONE, M,
                         nullptr, C, ldc, workspace, workspace_bytes, max_planes, &p);
  if (rc != LH_OK) return rc;
  // the split the launch will really use (no empty share)
  *planes = shares_of(p.g.K, p.g.nseg, config_at(p.config).bk, p.form != kGeneric ? p.g.splits : 1).n;
  return launch_index(p.config, p.g, p.ta, p.tx, p.form, lh::as_stream(stream));
}

namespace {
// The choice lh_gemm_planes_f32 makes for the stacked gate product of an LSTM cell, and whether
// that choice can carry the cell in its epilogue: aligned operands, no K split, a tile that fits LDS.
int plan_cell(int H, int B, const lh_gemm_seg *segs, int nseg, bool has_addend, const float *addend,
              int ld_addend, size_t workspace_bytes, Prepared *p, bool *fusable) {
  if (H <= 0 || B <= 0) return lh::fail_arg("lh_gate_gemm_lstm_cell: H=%d B=%d", H, B);
  float dummy;
  const int rc = prepare(4 * H, B, segs, nseg, 0, 0, 1.f, has_addend ? 1.f : 0.f, nullptr, LH_ACT_NONE,
                         4 * H, nullptr, has_addend && addend ? const_cast<float *>(addend) : &dummy,
                         has_addend && addend ? ld_addend : 4 * H,
                         workspace_bytes ? (void *)(uintptr_t)256 : nullptr, workspace_bytes,
                         has_addend ? 2 : 3, p);
  if (rc != LH_OK) return rc;
  *fusable = false;
  if (p->form != kAligned || H % 4 != 0) return LH_OK;
  // Best unsplit launch that can carry the cell against the best launch of any kind followed by
  // the cell kernel (a launch of its own that reads the pre-activations, or S planes of them, back).
  // 64 to 640 hidden units, 1 to 3 segments, 1 to 64 columns: on average as fast as the best of a sweep over
  // the configurations and both ways, 22 % behind it at worst (640 units, 2 segments, 32 columns).
  int cfg_any, splits_any, cfg_cell, splits_cell;
  float us_any, us_cell;
  const size_t ws = workspace_bytes;
  // (a product in the narrow form and its cell would often win here: its place is the packed gate product, which
  // is that form with the cell inside; this plan is for callers without packed matrices, one launch a step)
  pick_config(4 * H, B, p->g.K, nseg, false, false, kAligned, ws, has_addend ? 2 : 3, &cfg_any, &splits_any,
              false, &us_any, INT_MAX, INT_MAX, false);
  pick_config(4 * H, B, p->g.K, nseg, false, false, kAligned, ws, has_addend ? 2 : 3, &cfg_cell,
              &splits_cell, true, &us_cell);
  if (cfg_cell < 0) return LH_OK;
  // a configuration override (tuning, tests) asks for the fused form whenever the tile can hold it
  if (g_config_override >= 0 || us_cell <= us_any + cell_launch_us(us_any, H, B)) {
    *fusable = true;
    p->config = cfg_cell;
    p->g.splits = 1;
  }
  return LH_OK;
}
}  // namespace

extern "C" int lh_gate_gemm_lstm_cell_plan(int H, int B, const lh_gemm_seg *segs, int nseg,
                                           int has_addend, size_t workspace_bytes, int *fusable,
                                           char *name, int name_cap) {
  if (!fusable) return lh::fail_arg("lh_gate_gemm_lstm_cell_plan: fusable is NULL");
  Prepared p;
  bool f = false;
  const int rc = plan_cell(H, B, segs, nseg, has_addend != 0, nullptr, 0, workspace_bytes, &p, &f);
  if (rc != LH_OK) return rc;
  *fusable = f ? 1 : 0;
  if (name && name_cap > 0) {
    const Config &k = config_at(p.config);
    if (f) snprintf(name, name_cap, "gate_gemm_cell_kernel<%d, %d, %d, %d, %d, %d>", k.bm, k.bn, k.wm, k.wn, k.wk, k.bk);
    else name[0] = 0;
  }
  return LH_OK;
}

namespace {
int gate_gemm_lstm_cell(int H, int B, const lh_gemm_seg *segs, int nseg, const float *addend,
                        int ld_addend, const int *addend_col, int addend_ncols, const float *bias4h,
                        const float *c_prev, const int *mask01, int sigmoid_f64, float cell_clip,
                        float *gates, float *c, float *h, const float *next_drop_mask, float keep,
                        float *h_drop, size_t workspace_bytes, lh_stream_t stream);
}

extern "C" int lh_gate_gemm_lstm_cell_f32(int H, int B, const lh_gemm_seg *segs, int nseg,
                                          const float *addend, int ld_addend, const int *addend_col,
                                          int addend_ncols, const float *bias4h, const float *c_prev,
                                          const int *mask01, int sigmoid_f64, float cell_clip,
                                          float *c, float *h, size_t workspace_bytes,
                                          lh_stream_t stream) {
  return gate_gemm_lstm_cell(H, B, segs, nseg, addend, ld_addend, addend_col, addend_ncols, bias4h,
                             c_prev, mask01, sigmoid_f64, cell_clip, nullptr, c, h, nullptr, 1.f,
                             nullptr, workspace_bytes, stream);
}

extern "C" int lh_gate_gemm_lstm_cell_train_f32(int H, int B, const lh_gemm_seg *segs, int nseg,
                                                const float *addend, int ld_addend,
                                                const float *bias4h, const float *c_prev,
                                                const int *mask01, int sigmoid_f64, float cell_clip,
                                                float *gates, float *c, float *h,
                                                const float *next_drop_mask, float keep,
                                                float *h_drop, size_t workspace_bytes,
                                                lh_stream_t stream) {
  if (h_drop && (!next_drop_mask || !(keep > 0.f)))
    return lh::fail_arg("lh_gate_gemm_lstm_cell_train_f32: h_drop needs next_drop_mask and keep > 0");
  return gate_gemm_lstm_cell(H, B, segs, nseg, addend, ld_addend, nullptr, 0, bias4h, c_prev, mask01,
                             sigmoid_f64, cell_clip, gates, c, h, next_drop_mask, keep, h_drop,
                             workspace_bytes, stream);
}

namespace {
int gate_gemm_lstm_cell(int H, int B, const lh_gemm_seg *segs, int nseg, const float *addend,
                        int ld_addend, const int *addend_col, int addend_ncols, const float *bias4h,
                        const float *c_prev, const int *mask01, int sigmoid_f64, float cell_clip,
                        float *gates, float *c, float *h, const float *next_drop_mask, float keep,
                        float *h_drop, size_t workspace_bytes, lh_stream_t stream) {
  if (!bias4h || !c_prev || !mask01 || !c || !h)
    return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: a required pointer is NULL");
  if (addend && ld_addend < 4 * H)
    return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: ld_addend=%d < 4H=%d", ld_addend, 4 * H);
  if (addend_col && (!addend || addend_ncols < 1))
    return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: addend_col needs addend and addend_ncols >= 1");
  Prepared p;
  bool f = false;
  const int rc = plan_cell(H, B, segs, nseg, addend != nullptr, addend, ld_addend, workspace_bytes, &p, &f);
  if (rc != LH_OK) return rc;
  if (!f)
    return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: this product does not run fused "
                        "(ask lh_gate_gemm_lstm_cell_plan first)");
  // Other workgroups still read the operands while one writes its cells: the outputs must not
  // overlap any X operand (c may be c_prev: a cell is read and written by one thread).
  for (int s = 0; s < nseg; ++s) {
    const float *x0 = segs[s].X, *x1 = x0 + (size_t)segs[s].ldx * B;
    const float *outs[3] = {c, h, h_drop};
    for (const float *o : outs)
      if (o && o < x1 && x0 < o + (size_t)H * B)
        return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: an output overlaps operand X of segment %d", s);
    if (gates && gates < x1 && x0 < gates + (size_t)4 * H * B)
      return lh::fail_arg("lh_gate_gemm_lstm_cell_f32: gates overlap operand X of segment %d", s);
  }
  GemmArgs &g = p.g;
  g.bias = bias4h;
  g.colmask = mask01;
  g.cell_H = H;
  g.c_prev = c_prev;
  g.c_out = c;
  g.h_out = h;
  g.cell_clip = cell_clip;
  g.sigmoid_f64 = sigmoid_f64;
  g.addend_col = addend_col;
  g.addend_ncols = addend_ncols;
  g.gates_out = gates;
  g.drop_mask = next_drop_mask;
  g.h_drop = h_drop;
  g.keep = keep;
  return launch_cell_index(p.config, g, lh::as_stream(stream));
}
}  // namespace

// ---- gate products on packed gate matrices -----------------------------------------------------
extern "C" size_t lh_gate_pack_floats(int H, int K) {
  return H > 0 && K > 0 ? (size_t)((H + kPackCells - 1) / kPackCells) * kPackRows * (size_t)K : 0;
}

extern "C" int lh_gate_pack_f32(int H, const lh_gate_pack_source *src, int n, lh_stream_t stream) {
  if (H <= 0 || !src || n < 1 || n > LH_GATE_PACK_MAX)
    return lh::fail_arg("lh_gate_pack_f32: H=%d sources=%d (at most %d)", H, n, LH_GATE_PACK_MAX);
  PackArgs p{};
  p.H = H;
  int deepest = 0;
  for (int i = 0; i < n; ++i) {
    if (!src[i].src || !src[i].dst || src[i].K <= 0 || src[i].ld < 4 * H)
      return lh::fail_arg("lh_gate_pack_f32: source %d: src=%p dst=%p K=%d ld=%d (at least 4H)", i,
                          (const void *)src[i].src, (void *)src[i].dst, src[i].K, src[i].ld);
    p.src[i] = src[i].src, p.dst[i] = src[i].dst, p.ld[i] = src[i].ld, p.K[i] = src[i].K;
    deepest = src[i].K > deepest ? src[i].K : deepest;
  }
  const unsigned gy = (unsigned)((deepest + kPackK - 1) / kPackK);
  if (gy > 65535) return lh::fail_arg("lh_gate_pack_f32: K=%d is too deep", deepest);
  hipLaunchKernelGGL(gate_pack_kernel, dim3((unsigned)((H + 31) / 32), gy, (unsigned)n), dim3(256), 0,
                     lh::as_stream(stream), p);
  return lh::check_launch("lh_gate_pack_f32");
}

extern "C" int lh_gate_gemm_lstm_cell_packed_plan(int H, int B, const lh_gemm_seg *segs, int nseg,
                                                  int has_addend, size_t workspace_bytes, int *faster,
                                                  char *name, int name_cap) {
  if (!faster) return lh::fail_arg("lh_gate_gemm_lstm_cell_packed_plan: faster is NULL");
  *faster = 0;
  if (name && name_cap > 0) name[0] = 0;
  Prepared p;
  bool f = false;
  const int rc = plan_cell(H, B, segs, nseg, has_addend != 0, nullptr, 0, workspace_bytes, &p, &f);
  if (rc != LH_OK || p.form != kAligned || H % 4 != 0) return rc;
  // Against what runs without packing: the fused launch, or the product and the cell kernel behind it.
  int c, S, c0 = p.config;
  float us, us0;
  pick_packed(H, B, p.g.K, nseg, &c, &us);
  if (c < 0) return LH_OK;
  pick_config(4 * H, B, p.g.K, nseg, false, false, kAligned, workspace_bytes, has_addend ? 2 : 3, &c0, &S, f, &us0);
  if (!f) us0 += cell_launch_us(us0, H, B);
  if (us > us0) return LH_OK;
  *faster = 1 + (int)(1000.f * fminf(us0 - us, 1.0e6f));
  if (name && name_cap > 0) {
    const Config &k = kConfigs[c < kNumConfigs ? c : 0];
    if (c < kNumConfigs)
      snprintf(name, name_cap, "gate_gemm_packed_kernel<%d, %d, %d, %d, %d, %d>", k.bm, k.bn, k.wm, k.wn, k.wk, k.bk);
    else snprintf(name, name_cap, "gate_gemm_narrow_kernel<%d>", c - kNumConfigs + 1);
  }
  return LH_OK;
}

extern "C" int lh_gate_gemm_lstm_cell_packed_f32(int H, int B, const lh_gemm_seg *segs, int nseg,
                                                 const float *addend, int ld_addend, const int *addend_col,
                                                 int addend_ncols, const float *bias4h, const float *c_prev,
                                                 const int *mask01, int sigmoid_f64, float cell_clip,
                                                 float *gates, float *c, float *h, const float *next_drop_mask,
                                                 float keep, float *h_drop, lh_stream_t stream) {
  const char *const what = "lh_gate_gemm_lstm_cell_packed_f32";
  if (H <= 0 || B <= 0 || !segs || nseg < 1 || nseg > LH_GEMM_MAX_SEGS)
    return lh::fail_arg("%s: H=%d B=%d segments=%d", what, H, B, nseg);
  if (!bias4h || !c_prev || !mask01 || !c || !h) return lh::fail_arg("%s: a required pointer is NULL", what);
  if (addend && ld_addend < 4 * H) return lh::fail_arg("%s: ld_addend=%d < 4H=%d", what, ld_addend, 4 * H);
  if (addend_col && (!addend || addend_ncols < 1))
    return lh::fail_arg("%s: addend_col needs addend and addend_ncols >= 1", what);
  if (h_drop && (!next_drop_mask || !(keep > 0.f)))
    return lh::fail_arg("%s: h_drop needs next_drop_mask and keep > 0", what);
  GemmArgs g{};
  for (int s = 0; s < LH_GEMM_MAX_SEGS; ++s) {
    const lh_gemm_seg &e = segs[s < nseg ? s : 0];
    if (!e.A || !e.X || e.K <= 0 || e.K % 4 != 0 || e.ldx < e.K || e.ldx % 4 != 0 || e.ldx >= 1 << 22 ||
        !lh::aligned16(e.A) || !lh::aligned16(e.X))
      return lh::fail_arg("%s: segment %d: A=%p X=%p K=%d ldx=%d (16-byte aligned, multiples of 4)", what, s,
                          (const void *)e.A, (const void *)e.X, e.K, e.ldx);
    g.A[s] = e.A, g.X[s] = e.X, g.lda[s] = kPackRows, g.ldx[s] = e.ldx, g.K[s] = e.K;
  }
  // other workgroups still read the operands while one writes its cells
  for (int s = 0; s < nseg; ++s) {
    const float *x0 = segs[s].X, *x1 = x0 + (size_t)segs[s].ldx * B;
    const float *outs[4] = {c, h, h_drop, gates};
    for (int o = 0; o < 4; ++o)
      if (outs[o] && outs[o] < x1 && x0 < outs[o] + (size_t)(o == 3 ? 4 : 1) * H * B)
        return lh::fail_arg("%s: an output overlaps operand X of segment %d", what, s);
  }
  int config;
  float us;
  pick_packed(H, B, g.K, nseg, &config, &us);
  if (config < 0) return lh::fail_arg("%s: the configuration override names none of its configurations", what);
  g.nseg = nseg;
  g.M = 4 * H, g.N = B;
  g.beta = addend ? 1.f : 0.f;
  g.C = const_cast<float *>(addend);
  g.ldc = ld_addend;
  g.bias = bias4h;
  g.colmask = mask01;
  g.cell_H = H;
  g.c_prev = c_prev, g.c_out = c, g.h_out = h;
  g.cell_clip = cell_clip;
  g.sigmoid_f64 = sigmoid_f64;
  g.addend_col = addend_col, g.addend_ncols = addend_ncols;
  g.gates_out = gates;
  g.drop_mask = next_drop_mask, g.h_drop = h_drop, g.keep = keep;
  return launch_packed_index(config, g, lh::as_stream(stream));
}

// ---- grouped gate products ----------------------------------------------------------------------
namespace {
template <typename KernelT, typename ArgsT>
int launch_any(KernelT kernel, int smem_bytes, dim3 grid, dim3 block, hipStream_t st, const ArgsT &a,
               const char *what) {
  if (smem_bytes > 64 * 1024) {
    static thread_local const void *raised[64];
    static thread_local int n_raised = 0;
    bool done = false;
    for (int i = 0; i < n_raised; ++i) done = done || raised[i] == (const void *)kernel;
    if (!done) {
      hipError_t e = hipFuncSetAttribute((const void *)kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, smem_bytes);
      if (e != hipSuccess) {
        (void)hipGetLastError();
        return lh::fail_arg("%s: cannot reserve %d bytes of LDS: %s", what, smem_bytes,
                            hipGetErrorString(e));
      }
      if (n_raised < 64) raised[n_raised++] = (const void *)kernel;
    }
  }
  hipLaunchKernelGGL(kernel, grid, block, smem_bytes, st, a);
  return lh::check_launch(what);
}

template <int BM, int BN, int WM, int WN, int WK, int BK>
int launch_group_cfg(GroupArgs &a, hipStream_t st) {
  if constexpr (cell_capable<BM, BN, WM, WN, WK, BK>()) {
    int per_xcd[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int p = 0; p < a.n; ++p) {
      GemmArgs &g = a.g[p];
      // every tile holds BM/4 rows of each gate
      g.tiles_m = (g.cell_H + BM / 4 - 1) / (BM / 4);
      g.tiles_n = (g.N + BN - 1) / BN;
      g.splits = 1;
      g.slabs_per_split = 0;
      for (int s = 0; s < g.nseg; ++s) g.slabs_per_split += (g.K[s] + BK - 1) / BK;
      a.tiles[p] = g.tiles_m * g.tiles_n;
      for (int x = 0; x < 8; ++x) per_xcd[x] += a.tiles[p] / 8 + (x < a.tiles[p] % 8 ? 1 : 0);
    }
    int tiles = 0;
    for (int x = 0; x < 8; ++x) tiles = per_xcd[x] > tiles ? per_xcd[x] : tiles;
    tiles *= 8;
    return launch_any(gate_gemm_group_kernel<BM, BN, WM, WN, WK, BK>,
                      smem2_floats<BM, BN, WM, WN, WK, BK, false, false>() * 4, dim3(tiles),
                      dim3(64 * WM * WN * WK), st, a, "lh_gate_gemm_group_f32");
  } else {
    return lh::fail_arg("lh_gate_gemm_group_f32: internal error, tile %dx%d cannot hold the cell", BM, BN);
  }
}

int launch_group_index(int c, GroupArgs &a, hipStream_t st) {
  switch (c) {
#define LH_CFG_CASE(I, BM, BN, WM, WN, WK, BK) \
  case I: return launch_group_cfg<BM, BN, WM, WN, WK, BK>(a, st);
    LH_GEMM_CONFIGS(LH_CFG_CASE)
#undef LH_CFG_CASE
    default: return lh::fail_arg("lh_gate_gemm_group_f32: configuration %d does not exist", c);
  }
}

// Checks a group and fills the kernel arguments; *config < 0 when the group cannot run as one
// launch (unaligned operands, H not a multiple of 4, no tile that can hold a cell).
int plan_group(int H, int B, const lh_gate_problem *pr, int n, GroupArgs *a, int *config) {
  if (H <= 0 || B <= 0 || !pr || n < 1 || n > kMaxGroup)
    return lh::fail_arg("lh_gate_gemm_group: H=%d B=%d problems=%d (at most %d)", H, B, n, kMaxGroup);
  *config = -1;
  *a = GroupArgs{};
  a->n = n;
  bool vec = H % 4 == 0;
  for (int p = 0; p < n; ++p) {
    const lh_gate_problem &q = pr[p];
    float dummy;
    float *C = q.cell ? (q.addend ? const_cast<float *>(q.addend) : &dummy) : q.out;
    const int ldc = q.cell ? (q.addend ? q.ld_addend : 4 * H) : q.ld_out;
    if (!q.cell && (!q.out || q.ld_out < 4 * H))
      return lh::fail_arg("lh_gate_gemm_group: problem %d: out=%p ld_out=%d", p, (void *)q.out, q.ld_out);
    if (q.cell) {
      if (!q.bias4h || !q.c_prev || !q.mask01 || !q.c || !q.h)
        return lh::fail_arg("lh_gate_gemm_group: problem %d: a required pointer is NULL", p);
      if (q.addend && q.ld_addend < 4 * H)
        return lh::fail_arg("lh_gate_gemm_group: problem %d: ld_addend=%d < 4H", p, q.ld_addend);
      if (q.addend_col && (!q.addend || q.addend_ncols < 1))
        return lh::fail_arg("lh_gate_gemm_group: problem %d: addend_col needs addend and addend_ncols", p);
    }
    Prepared pp;
    const int rc = prepare(4 * H, B, q.segs, q.nseg, 0, 0, 1.f, q.cell && q.addend ? 1.f : 0.f, nullptr,
                           LH_ACT_NONE, 4 * H, nullptr, C, ldc, nullptr, 0, 0, &pp);
    if (rc != LH_OK) return rc;
    vec = vec && pp.form == kAligned && (q.cell || (lh::aligned16(q.out) && q.ld_out % 4 == 0));
    GemmArgs &g = a->g[p];
    g = pp.g;
    a->cell[p] = q.cell ? 1 : 0;
    g.cell_H = H;
    if (!q.cell) {
      g.pre_out = q.out;
      g.pre_ld = q.ld_out;
    }
    if (q.cell) {
      g.bias = q.bias4h;
      g.colmask = q.mask01;
      g.c_prev = q.c_prev;
      g.c_out = q.c;
      g.h_out = q.h;
      g.cell_clip = q.cell_clip;
      g.sigmoid_f64 = q.sigmoid_f64;
      g.addend_col = q.addend_col;
      g.addend_ncols = q.addend_ncols;
      // outputs must not overlap an X operand of ANY problem of the launch
      for (int o = 0; o < n; ++o)
        for (int sgi = 0; sgi < pr[o].nseg; ++sgi) {
          const float *x0 = pr[o].segs[sgi].X, *x1 = x0 + (size_t)pr[o].segs[sgi].ldx * B;
          const float *outs[2] = {q.c, q.h};
          for (const float *w : outs)
            if (w < x1 && x0 < w + (size_t)H * B)
              return lh::fail_arg("lh_gate_gemm_group: an output of problem %d overlaps an X operand "
                                  "of problem %d", p, o);
        }
    } else {
      for (int o = 0; o < n; ++o)
        for (int sgi = 0; sgi < pr[o].nseg; ++sgi) {
          const float *x0 = pr[o].segs[sgi].X, *x1 = x0 + (size_t)pr[o].segs[sgi].ldx * B;
          if (q.out < x1 && x0 < q.out + (size_t)q.ld_out * B)
            return lh::fail_arg("lh_gate_gemm_group: the output of problem %d overlaps an X operand "
                                "of problem %d", p, o);
        }
    }
  }
  if (!vec) return LH_OK;
  // One tile shape for the whole launch.  Cost model as for a single product (predict_us), with
  // the problems' tiles side by side on every CU: n_p tiles of problem p per CU, each taking
  // tocc(depth_p) / occ of a CU's time when the CU is full; a CU that is not full runs its few
  // tiles at a per-tile time between t1 and tocc of the deepest problem.
  float best = 3.0e38f;
  const Tuning *table = kTuning[0];
  for (int c = 0; c < kNumConfigs; ++c) {
    if (g_config_override >= 0 && c != g_config_override) continue;
    if (!cell_capable_index(c)) continue;
    const Config &k = kConfigs[c];
    const Tuning &t = table[c];
    float per_cu = 0.f, packed = 0.f, t1_max = 0.f, tocc_max = 0.f;
    for (int p = 0; p < n; ++p) {
      const float tiles = (float)(((H + k.bm / 4 - 1) / (k.bm / 4)) * ((B + k.bn - 1) / k.bn));
      int slabs = 0;
      for (int sgi = 0; sgi < pr[p].nseg; ++sgi) slabs += (pr[p].segs[sgi].K + k.bk - 1) / k.bk;
      const float depth = (float)slabs * k.bk;
      const float t1 = t.f1 + t.s1 * depth, tocc = t.focc + t.socc * depth;
      per_cu += tiles / kCUs;
      packed += tiles / kCUs * tocc / (float)t.occ;
      t1_max = fmaxf(t1_max, t1);
      tocc_max = fmaxf(tocc_max, tocc);
    }
    float us;
    if (per_cu >= (float)t.occ) {
      us = packed + 0.5f * tocc_max / (float)t.occ;  // dynamic dispatch leaves about half a tile of tail
    } else {
      const float load = fminf(per_cu + 0.5f, ceilf(per_cu));
      us = load <= 1.f || t.occ == 1 ? t1_max
                                     : t1_max + (tocc_max - t1_max) * (load - 1.f) / (float)(t.occ - 1);
    }
    if (us < best) {
      best = us;
      *config = c;
    }
  }
  return LH_OK;
}
}  // namespace

extern "C" int lh_gate_gemm_group_plan(int H, int B, const lh_gate_problem *problems, int n_problems,
                                       int *runnable, char *name, int name_cap) {
  if (!runnable) return lh::fail_arg("lh_gate_gemm_group_plan: runnable is NULL");
  GroupArgs a;
  int config = -1;
  const int rc = plan_group(H, B, problems, n_problems, &a, &config);
  if (rc != LH_OK) return rc;
  *runnable = config >= 0 ? 1 : 0;
  if (name && name_cap > 0) {
    if (config >= 0) {
      const Config &k = kConfigs[config];
      snprintf(name, name_cap, "gate_gemm_group_kernel<%d, %d, %d, %d, %d, %d>", k.bm, k.bn, k.wm,
               k.wn, k.wk, k.bk);
    } else {
      name[0] = 0;
    }
  }
  return LH_OK;
}

extern "C" int lh_gate_gemm_group_f32(int H, int B, const lh_gate_problem *problems, int n_problems,
                                      lh_stream_t stream) {
  GroupArgs a;
  int config = -1;
  const int rc = plan_group(H, B, problems, n_problems, &a, &config);
  if (rc != LH_OK) return rc;
  if (config < 0)
    return lh::fail_arg("lh_gate_gemm_group_f32: this group does not run as one launch "
                        "(ask lh_gate_gemm_group_plan first)");
  return launch_group_index(config, a, lh::as_stream(stream));
}

// ---- the K-split product for callers that cannot allocate ------------------------------------
// The partial planes live in a device array that is part of the library's code object: every GPU
// the library runs on holds its own copy, at its own address, until the process ends.  The name
// of the array is only a handle on the host; the device address is asked for once per device.
namespace {
static __device__ __align__(256) float scratch[LH_GEMM_NOALLOC_WS_BYTES / sizeof(float)];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch_ptr[kMaxDevices];  // per device, null until the first call on it

int scratch_for_current_device(float **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return lh::fail_arg("lh_gemm_noalloc_f32: hipGetDevice: %s", hipGetErrorString(e));
  }
  if (dev < 0 || dev >= kMaxDevices)
    return lh::fail_arg("lh_gemm_noalloc_f32: device %d outside [0,%d)", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return lh::fail_arg("lh_gemm_noalloc_f32: hipGetSymbolAddress on device %d: %s", dev,
                          hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = static_cast<float *>(p);
  }
  *out = g_scratch_ptr[dev];
  return LH_OK;
}
}  // namespace

extern "C" int lh_gemm_noalloc_init(void) {
  float *ws = nullptr;
  return scratch_for_current_device(&ws);
}

extern "C" int lh_gemm_noalloc_f32(int M, int N, const lh_gemm_seg *segs, int nseg, int transA,
                                   int transX, float alpha, float beta, const float *bias, int act,
                                   int act_rows, const int *colmask, float *C, int ldc,
                                   lh_stream_t stream) {
  if (M <= 0 || N <= 0) return lh::fail_arg("lh_gemm_noalloc_f32: M=%d N=%d must be positive", M, N);
  const size_t plane = (size_t)plane_ld(M) * (size_t)N * sizeof(float);
  if (2 * plane > (size_t)LH_GEMM_NOALLOC_WS_BYTES)
    return lh::fail_arg("lh_gemm_noalloc_f32: two partial planes of this %d x %d product need %zu "
                        "bytes, the library's scratch array holds %zu (LH_GEMM_NOALLOC_WS_BYTES); "
                        "use lh_gemm_ws_f32 with a workspace of the caller's",
                        M, N, 2 * plane, (size_t)LH_GEMM_NOALLOC_WS_BYTES);
  float *ws = nullptr;
  const int rc = scratch_for_current_device(&ws);
  if (rc != LH_OK) return rc;
  return lh_gemm_ws_f32(M, N, segs, nseg, transA, transX, alpha, beta, bias, act, act_rows, colmask,
                        C, ldc, ws, (size_t)LH_GEMM_NOALLOC_WS_BYTES, stream);
}

extern "C" int lh_gemm_f32(int M, int N, const lh_gemm_seg *segs, int nseg, int transA, int transX,
                           float alpha, float beta, const float *bias, int act, const int *colmask,
                           float *C, int ldc, lh_stream_t stream) {
  return lh_gemm_ws_f32(M, N, segs, nseg, transA, transX, alpha, beta, bias, act, M, colmask, C,
                        ldc, nullptr, 0, stream);
}

extern "C" int lh_gemm_act_rows_f32(int M, int N, const lh_gemm_seg *segs, int nseg, int transA,
                                    int transX, float alpha, float beta, const float *bias, int act,
                                    int act_rows, const int *colmask, float *C, int ldc,
                                    lh_stream_t stream) {
  return lh_gemm_ws_f32(M, N, segs, nseg, transA, transX, alpha, beta, bias, act, act_rows, colmask,
                        C, ldc, nullptr, 0, stream);
}

extern "C" int lh_gemm_set_config_override(int config) {
  if (config >= kNumConfigs + kNumNarrow)
    return lh::fail_arg("lh_gemm_set_config_override: %d >= %d", config, kNumConfigs + kNumNarrow);
  g_config_override = config < 0 ? -1 : config;
  return kNumConfigs;
}

extern "C" int lh_gemm_set_splits_override(int splits) {
  if (splits > kMaxSplits)
    return lh::fail_arg("lh_gemm_set_splits_override: %d > %d", splits, kMaxSplits);
  g_splits_override = splits < 0 ? 0 : splits;
  return kMaxSplits;
}

extern "C" int lh_gemm_config_info(int config, int transA, int transX, int info[8]) {
  if (config < 0 || config >= kNumConfigs + kNumNarrow || !info || (transA && transX))
    return lh::fail_arg("lh_gemm_config_info: config=%d of %d, info=%p", config, kNumConfigs + kNumNarrow,
                        (void *)info);
  const Config &k = config_at(config);
  info[0] = k.bm, info[1] = k.bn, info[2] = k.wm, info[3] = k.wn, info[4] = k.wk, info[5] = k.bk;
  return occupancy_index(config, transA != 0, transX != 0, &info[6], &info[7]);
}

extern "C" int lh_gemm_kernel_name(int M, int N, const lh_gemm_seg *segs, int nseg, int transA,
                                   int transX, size_t workspace_bytes, int max_planes, char *name,
                                   int name_cap) {
  if (!name || name_cap < 1) return lh::fail_arg("lh_gemm_kernel_name: no output buffer");
  Prepared p;
  float dummy;
  // any aligned non-null address stands in for the workspace: nothing is launched
  const int rc = prepare(M, N, segs, nseg, transA, transX, 1.f, 0.f, nullptr, LH_ACT_NONE, M,
                         nullptr, &dummy, M, workspace_bytes ? (void *)(uintptr_t)256 : nullptr,
                         workspace_bytes, max_planes, &p);
  if (rc != LH_OK) return rc;
  const Config &k = config_at(p.config);
  if (p.form != kGeneric)
    snprintf(name, name_cap, "gemm_kernel<%d, %d, %d, %d, %d, %d, %s, %s%s>", k.bm, k.bn, k.wm, k.wn,
             k.wk, k.bk, p.ta ? "true" : "false", p.tx ? "true" : "false", p.form == kRagged ? ", true" : "");
  else
    snprintf(name, name_cap, "gemm_generic_kernel<%d, %d, %d, %d, %d, %d, %s, %s, false>", k.bm,
             k.bn, k.wm, k.wn, k.wk, k.bk, p.ta ? "true" : "false", p.tx ? "true" : "false");
  return LH_OK;
}
