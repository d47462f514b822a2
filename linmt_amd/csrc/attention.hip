// Attention core (Luong local-p, and the textbook global "general" variant): alignment position,
// window indices, scores, max-subtracted exp, normalisation, Gaussian weighting and the context
// vector in ONE kernel, one workgroup per column b:
//   phase 1  v_p . tanh1[:,b]  -> sigmoid -> p_b -> window [lo,hi]           (block reduction)
//   phase 2  score_j = hs_j . wa[:,b]
//   phase 3  max / exp / sum / Gaussian over the <= W slots
//   phase 4  ctx[:,b] = sum_j a_j hs_j
// The reference materialises the window (LoadInHSKernel) and launches eight kernels for this.
#include "lh_common.h"

namespace {

constexpr int kMaxSlots = 512;
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / lh::kWave;

struct AttnArgs {
  int H, B, D, W;
  const float *tanh1, *v_p, *wa, *hs;
  long long proj_col_stride;  // distance between columns of tanh1 and of wa (>= H)
  long long step_stride, col_stride;
  int hs_steps;
  const int *hs_col, *batch_info, *mask01;
  float *p_t, *sigma;
  int *indices;
  float *align, *cached_exp, *ctx;
  int *viterbi;
  // Projected memory (register kernel only).  ctx_mem != NULL: the context sum runs over ctx_mem
  // (laid out like hs) instead of hs.  out_add / out_bias != NULL are added to that sum (out_add
  // per column, out_add_col_stride apart) and out_tanh applies tanh and the column mask: the
  // output is then the attention layer's h~ rather than the context vector.
  long long wa_col_stride;  // distance between columns of wa
  const float *ctx_mem, *out_add, *out_bias;
  long long out_add_col_stride;
  int out_tanh;
};

// Any window and alignment.  With at most a few columns per CU a launch lasts as long as one workgroup's
// chain of dependent memory round trips, so a column gets up to 16 wavefronts (NT threads), a wavefront has
// the rows of two slots in flight at once (four were slower at every count of columns), every slot's
// exponential is taken once, by the slot's own thread, and the context sum of a row is split over
// as many groups of threads as the workgroup has left (their partial sums meet in LDS in group
// order); its second read of the window comes from L2.  Position and weights do not depend on NT.
constexpr int kSlotBatch = 2;

template <bool VEC, int NT>
__global__ __launch_bounds__(NT) void attn_core_kernel(const AttnArgs a) {
  constexpr int kNW = NT / lh::kWave;
  __shared__ float s_val[kMaxSlots];   // scores, then alignment weights
  __shared__ int s_tau[kMaxSlots];     // encoder timestep of slot j, -1 = no state to read
  __shared__ float s_red[kNW];
  __shared__ float4 s_ctx[NT];
  __shared__ int s_first;

  const int b = lh::xcd_contiguous(blockIdx.x, gridDim.x);  // a sentence's columns on one XCD
  const int tid = threadIdx.x, wave = tid / lh::kWave, lane = tid % lh::kWave;
  const int H = a.H, B = a.B, W = a.W, D = a.D;
  const int len = a.batch_info[b];
  const int off = a.batch_info[B + b];
  const int m = a.mask01[b];
  const int col = a.hs_col ? a.hs_col[b] : b;
  const float *wa = a.wa + (size_t)b * a.proj_col_stride;
  const float *hs_c = a.hs + (size_t)col * a.col_stride;

  float p = 0.f;
  int lo = 0, hi = len - 1;
  if (D >= 0) {
    float part = 0.f;
    const float *t1 = a.tanh1 + (size_t)b * a.proj_col_stride;
    if (tid < kThreads)  // the order of attn_core_regs_kernel: the position must not depend on the kernel
      for (int r = tid; r < H; r += kThreads) part += a.v_p[r] * t1[r];
    const float dot = lh::block_sum<kNW>(part, s_red);
    const float sig = (float)(1.0 / (1.0 + exp(-1.0 * (double)dot)));
    p = (float)len * sig;
    lo = (0 > (int)p - D) ? 0 : ((int)p - D);
    hi = ((len - 1) < (int)p + D) ? (len - 1) : ((int)p + D);
    if (tid == 0) {
      a.p_t[b] = p;
      a.sigma[b] = sig;
    }
  }

  // window indices (reference layout B x W, element (b,j) at b + B*j); thread j owns slot j (W <= NT)
  int idx = -1;
  if (tid < W) {
    if (m == 1 && lo + tid <= hi) idx = lo + tid;
    a.indices[b + (size_t)B * tid] = idx;
    int tau = -1;
    if (idx >= 0) {
      tau = len - 1 - idx + off;
      if (tau < 0 || tau >= a.hs_steps) tau = -1;  // outside the caller's state buffer: zero vector
    }
    s_tau[tid] = tau;
  }
  __syncthreads();

  // scores: wavefront w takes slots w, w + 16, ..., four at a time
  for (int j0 = wave; j0 < W; j0 += kNW * kSlotBatch) {
    const float *row[kSlotBatch];
    float acc[kSlotBatch];
    bool live[kSlotBatch];
#pragma unroll
    for (int u = 0; u < kSlotBatch; ++u) {
      const int j = j0 + u * kNW;
      const int tau = j < W ? s_tau[j] : -1;
      live[u] = tau >= 0;
      row[u] = hs_c + (size_t)(live[u] ? tau : 0) * a.step_stride;
      acc[u] = 0.f;
    }
    if constexpr (VEC) {
#pragma unroll 2
      for (int r = lane * 4; r < H; r += lh::kWave * 4) {
        const float4 y = *reinterpret_cast<const float4 *>(wa + r);
#pragma unroll
        for (int u = 0; u < kSlotBatch; ++u) {
          if (!live[u]) continue;  // the same for the whole wavefront
          const float4 x = *reinterpret_cast<const float4 *>(row[u] + r);
          acc[u] += x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w;
        }
      }
    } else {
#pragma unroll 2
      for (int r = lane; r < H; r += lh::kWave) {
        const float y = wa[r];
#pragma unroll
        for (int u = 0; u < kSlotBatch; ++u)
          if (live[u]) acc[u] += row[u][r] * y;
      }
    }
#pragma unroll
    for (int u = 0; u < kSlotBatch; ++u) {
      const float sc = lh::wave_sum(acc[u]);
      const int j = j0 + u * kNW;
      if (lane == 0 && j < W) s_val[j] = live[u] ? sc : 0.f;
    }
  }
  __syncthreads();

  // normalisation
  const bool valid = tid < W && idx != -1;
  const float val = valid ? s_val[tid] : 0.f;
  const float floor_mx = D >= 0 ? 0.f : -FLT_MAX;
  const float mx = lh::block_max<kNW>(valid ? fmaxf(val, floor_mx) : floor_mx, s_red);
  const float e = valid ? expf(val - mx) : 0.f;
  const float Z = lh::block_sum<kNW>(e, s_red);
  if (tid < W) {
    float al = 0.f, g = 1.f;
    if (valid) {
      if (D >= 0) {
        const float sigma_sq = (float)((D * D) / 4.0);
        const float dlt = p - (float)idx;
        g = expf((-1.f * (dlt * dlt)) / (2.f * sigma_sq));
      }
      al = (Z != 0.f) ? (e / Z) * g : e;
    }
    a.align[b + (size_t)B * tid] = al;
    a.cached_exp[tid + (size_t)W * b] = g;
    s_val[tid] = al;
  }
  if (tid == 0) s_first = W;
  __syncthreads();

  if (a.viterbi) {
    // the first slot of the largest weight (weights are >= 0, slots without a position weigh 0)
    const float al = tid < W ? s_val[tid] : -1.f;
    const float best = lh::block_max<kNW>(fmaxf(al, -1.f), s_red);
    if (tid < W && al == best) atomicMin(&s_first, tid);
    __syncthreads();
    const int first = best > -1.f ? s_first : W;
    if (tid == (first < W ? first : 0)) a.viterbi[b] = first < W ? idx : -1;
  }

  // context vector: the rows (quads of them when aligned) of a column go to `lanes` threads,
  // group g of the workgroup adds the slots j = g, g + groups, ...
  float *ctx = a.ctx + (size_t)b * H;
  const int units = VEC ? H / 4 : H;
  const int lanes = min(NT, (units + lh::kWave - 1) / lh::kWave * lh::kWave);
  const int groups = NT / lanes;
  const int grp = tid / lanes;
  for (int u0 = 0; u0 < units; u0 += lanes) {
    const int unit = u0 + tid % lanes;
    const bool mine = grp < groups && unit < units;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    if (mine) {
#pragma unroll 4
      for (int j = grp; j < W; j += groups) {
        const int tau = s_tau[j];
        const float w = s_val[j];
        // a slot without a state reads column 0's first one, which exists, and drops it
        const float *x = tau >= 0 ? hs_c + (size_t)tau * a.step_stride : a.hs;
        if constexpr (VEC) {
          const float4 v = *reinterpret_cast<const float4 *>(x + (size_t)unit * 4);
          acc.x = tau >= 0 ? acc.x + w * v.x : acc.x;
          acc.y = tau >= 0 ? acc.y + w * v.y : acc.y;
          acc.z = tau >= 0 ? acc.z + w * v.z : acc.z;
          acc.w = tau >= 0 ? acc.w + w * v.w : acc.w;
        } else {
          const float v = x[unit];
          acc.x = tau >= 0 ? acc.x + w * v : acc.x;
        }
      }
    }
    if (groups > 1) {  // then every unit is covered by the first round
      s_ctx[tid] = acc;
      __syncthreads();
      if (grp == 0 && mine)
        for (int g = 1; g < groups; ++g) {
          const float4 o = s_ctx[g * lanes + tid];
          acc.x += o.x, acc.y += o.y, acc.z += o.z, acc.w += o.w;
        }
    }
    if (grp == 0 && mine) {
      if constexpr (VEC) *reinterpret_cast<float4 *>(ctx + (size_t)unit * 4) = acc;
      else ctx[unit] = acc.x;
    }
  }
}

// Sums v[slot] over the 64 lanes of a wavefront for 32 slots at once: at every level a lane keeps
// one half of its slots and hands the other half to its partner, 32 exchanges in place of 6 per
// slot.  Lane l returns the sum of slot l / 2, added in the order of wave_sum.
template <int HALF>
__device__ __forceinline__ void fold_slots(float (&v)[32], int lane) {
  const bool upper = (lane & (2 * HALF)) != 0;
#pragma unroll
  for (int i = 0; i < HALF; ++i) {
    const float keep = upper ? v[i + HALF] : v[i];
    const float send = upper ? v[i] : v[i + HALF];
    v[i] = keep + __shfl_xor(send, 2 * HALF, lh::kWave);
  }
}
__device__ __forceinline__ float wave_sum_slots(float (&v)[32], int lane) {
  fold_slots<16>(v, lane);
  fold_slots<8>(v, lane);
  fold_slots<4>(v, lane);
  fold_slots<2>(v, lane);
  fold_slots<1>(v, lane);
  return v[0] + __shfl_xor(v[0], 1, lh::kWave);
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The same computation for windows of at most WCAP slots (local-p with D <= 10) and 16-byte
// aligned operands: the whole W x H window of the column is read ONCE, straight into registers
// (thread t holds rows 4t..4t+3 -- and 4(t+256).. when H > 1024 -- of every slot, all loads in
// flight together), the scores are block-reduced from per-thread partial dot products, and the
// context vector is accumulated from the same registers.
// A launch lasts as long as one workgroup's chain of dependent steps (few columns per CU, the
// columns of a sentence share their window in L2), so the chain is kept short: the window's bounds
// live in scalar registers (no trip through LDS before its loads), lane j of every wavefront
// normalises slot j by itself, and what all lanes need of it comes back as a lane read.
// H = 1000, D = 10: 12 columns 16.0 -> 7.8 us, 64 columns 14.3 -> 7.0, 768 columns 21.4 -> 15.1.
template <int NQ, int WCAP>
__global__ __launch_bounds__(kThreads) void attn_core_regs_kernel(const AttnArgs a) {
  static_assert(WCAP <= 31, "wave_sum_slots, the bits of live");
  __shared__ float s_part[kWaves][32];
  __shared__ float s_red[kWaves];

  const int b = lh::xcd_contiguous(blockIdx.x, gridDim.x);  // a sentence's columns on one XCD
  const int tid = threadIdx.x, wave = tid / lh::kWave, lane = tid % lh::kWave;
  const int H = a.H, B = a.B, W = a.W, D = a.D;
  const int len = a.batch_info[b];
  const int off = a.batch_info[B + b];
  const int m = a.mask01[b];
  const int col = a.hs_col ? a.hs_col[b] : b;
  const float *wa = a.wa + (size_t)b * a.wa_col_stride;

  // everything that does not depend on the window position is requested first
  float4 w4[NQ], oadd[NQ], obias[NQ];
  bool row_ok[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int r = (tid + q * kThreads) * 4;
    row_ok[q] = r < H;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    w4[q] = row_ok[q] ? *reinterpret_cast<const float4 *>(wa + r) : zero;
    oadd[q] = (row_ok[q] && a.out_add)
                  ? *reinterpret_cast<const float4 *>(a.out_add + (size_t)b * a.out_add_col_stride + r)
                  : zero;
    obias[q] = (row_ok[q] && a.out_bias) ? *reinterpret_cast<const float4 *>(a.out_bias + r) : zero;
  }

  float p = 0.f;
  int lo = 0, hi = len - 1;
  if (D >= 0) {
    float part = 0.f;
    const float *t1 = a.tanh1 + (size_t)b * a.proj_col_stride;
    // rows tid, tid + 256, ... in that order (H <= NQ * 1024), all loads in flight together
    float vv[4 * NQ], tt[4 * NQ];
#pragma unroll
    for (int k = 0; k < 4 * NQ; ++k) {
      const int r = tid + k * kThreads;
      vv[k] = r < H ? a.v_p[r] : 0.f;
      tt[k] = r < H ? t1[r] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 4 * NQ; ++k)
      if (tid + k * kThreads < H) part += vv[k] * tt[k];
    const float dot = lh::block_sum<kWaves>(part, s_red);
    const float sig = (float)(1.0 / (1.0 + exp(-1.0 * (double)dot)));
    p = (float)len * sig;
    lo = (0 > (int)p - D) ? 0 : ((int)p - D);
    hi = ((len - 1) < (int)p + D) ? (len - 1) : ((int)p + D);
    if (tid == 0) {
      a.p_t[b] = p;
      a.sigma[b] = sig;
    }
  }
  // the window's slots: source position lo + j, encoder timestep tau0 - j
  const int lo_s = __builtin_amdgcn_readfirstlane(lo);
  const int slots = __builtin_amdgcn_readfirstlane(m == 1 ? min(W, hi - lo + 1) : 0);
  const int tau0 = __builtin_amdgcn_readfirstlane(len - 1 + off) - lo_s;
  const int steps = a.hs_steps;
  // slots with a state to read (a timestep inside the caller's buffer): one run of them, as bits
  const int j_lo = max(0, tau0 - steps + 1), j_hi = min(slots, tau0 + 1);
  const unsigned live =
      __builtin_amdgcn_readfirstlane(j_hi > j_lo ? ((2u << (j_hi - 1)) - 1u) & ~((1u << j_lo) - 1u) : 0u);

  // The window, once.  A slot without a state to read loads a row that exists instead; its values
  // are never used (no select per loaded register: they were most of this kernel's instructions).
  int rows_at[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) rows_at[q] = row_ok[q] ? (tid + q * kThreads) * 4 : 0;
  // (A column without any such slot, a padded one say, may carry any entry of hs_col: column 0's rows then.)
  const size_t col_at = live ? (size_t)col * a.col_stride : 0;
  auto slot_row = [&](const float *mem, int j) {
    return mem + col_at + (size_t)min(max(tau0 - j, 0), steps - 1) * a.step_stride;
  };
  float4 h[WCAP][NQ];
#pragma unroll
  for (int j = 0; j < WCAP; ++j) {
    const float *row = slot_row(a.hs, j);
#pragma unroll
    for (int q = 0; q < NQ; ++q) h[j][q] = *reinterpret_cast<const float4 *>(row + rows_at[q]);
  }
  // scores: per-thread partial dot products, wavefront sums, then the four wavefronts in order
  float part[32];
#pragma unroll
  for (int j = 0; j < 32; ++j) part[j] = 0.f;
#pragma unroll
  for (int j = 0; j < WCAP; ++j) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const float s = h[j][q].x * w4[q].x + h[j][q].y * w4[q].y + h[j][q].z * w4[q].z + h[j][q].w * w4[q].w;
      part[j] += row_ok[q] ? s : 0.f;
    }
  }
  const float slot_sum = wave_sum_slots(part, lane);
  if (lane % 2 == 0) s_part[wave][lane / 2] = slot_sum;
  if (a.ctx_mem) {
    // the scores are done with the window: the same registers take the window of ctx_mem, whose
    // loads fly while the scores are normalised
#pragma unroll
    for (int j = 0; j < WCAP; ++j) {
      const float *row = slot_row(a.ctx_mem, j);
#pragma unroll
      for (int q = 0; q < NQ; ++q) h[j][q] = *reinterpret_cast<const float4 *>(row + rows_at[q]);
    }
  }
  __syncthreads();
  // every wavefront normalises the whole window, lane j slot j
  const bool valid = lane < slots;
  float sc = 0.f;
  if (lane < WCAP) {
    sc = s_part[0][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sc += s_part[w][lane];
  }
  const float val = lane < WCAP && ((live >> lane) & 1u) ? sc : 0.f;
  const float floor_mx = D >= 0 ? 0.f : -FLT_MAX;
  const float mx = lh::wave_max(valid ? fmaxf(val, floor_mx) : floor_mx);
  const float e = valid ? expf(val - mx) : 0.f;
  float Z = 0.f;  // in slot order
#pragma unroll
  for (int j = 0; j < WCAP; ++j) Z += lane_value(e, j);
  float al = 0.f, g = 1.f;
  if (valid) {
    if (D >= 0) {
      const float sigma_sq = (float)((D * D) / 4.0);
      const float dlt = p - (float)(lo + lane);
      g = expf((-1.f * (dlt * dlt)) / (2.f * sigma_sq));
    }
    al = (Z != 0.f) ? (e / Z) * g : e;
  }
  if (wave == 0) {
    if (lane < W) {
      a.indices[b + (size_t)B * lane] = valid ? lo + lane : -1;
      a.align[b + (size_t)B * lane] = al;
      a.cached_exp[lane + (size_t)W * b] = g;
    }
    if (a.viterbi) {
      // the first slot of the largest weight (weights are >= 0, slots without a position weigh 0)
      const float mine = lane < W ? al : -1.f;
      const float best = lh::wave_max(fmaxf(mine, -1.f));
      const unsigned long long at = __ballot(lane < W && mine == best);
      const int first = at ? __ffsll(at) - 1 : -1;
      if (lane == 0) a.viterbi[b] = best > -1.f && first >= 0 && first < slots ? lo + first : -1;
    }
  }

  float *ctx = a.ctx + (size_t)b * H;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < WCAP; ++j) {
      if (!((live >> j) & 1u)) continue;  // the general kernel skips these slots too
      asm volatile("" ::: "memory");  // a scalar branch over four multiply-adds, not four selects
      const float w = lane_value(al, j);
      acc.x += w * h[j][q].x; acc.y += w * h[j][q].y; acc.z += w * h[j][q].z; acc.w += w * h[j][q].w;
    }
    if (!row_ok[q]) continue;
    const size_t r = (size_t)(tid + q * kThreads) * 4;
    if (a.out_add) {
      acc.x += oadd[q].x; acc.y += oadd[q].y; acc.z += oadd[q].z; acc.w += oadd[q].w;
    }
    if (a.out_bias) {
      acc.x += obias[q].x; acc.y += obias[q].y; acc.z += obias[q].z; acc.w += obias[q].w;
    }
    if (a.out_tanh) {
      const float mf = (float)m;
      acc.x = tanhf(acc.x) * mf; acc.y = tanhf(acc.y) * mf;
      acc.z = tanhf(acc.z) * mf; acc.w = tanhf(acc.w) * mf;
    }
    *reinterpret_cast<float4 *>(ctx + r) = acc;
  }
}

constexpr int kRegsSlots = 21;  // the reference's default window: D = 10

template <int NT>
void launch_general(const AttnArgs &a, bool vec, hipStream_t st) {
  if (vec) hipLaunchKernelGGL((attn_core_kernel<true, NT>), dim3(a.B), dim3(NT), 0, st, a);
  else hipLaunchKernelGGL((attn_core_kernel<false, NT>), dim3(a.B), dim3(NT), 0, st, a);
}

}  // namespace

extern "C" int lh_attn_core_fwd_f32(int H, int B, int D, int max_len, int hs_steps,
                                    const float *tanh1, const float *v_p, const float *wa,
                                    long long proj_col_stride, const float *hs,
                                    long long hs_step_stride,
                                    long long hs_col_stride, const int *hs_col,
                                    const int *batch_info, const int *mask01, float *p_t,
                                    float *sigma, int *indices, float *align, float *cached_exp,
                                    float *ctx, int *viterbi, lh_stream_t stream) {
  if (H <= 0 || B <= 0 || hs_steps <= 0)
    return lh::fail_arg("lh_attn_core_fwd_f32: H=%d B=%d hs_steps=%d", H, B, hs_steps);
  const int W = D >= 0 ? 2 * D + 1 : max_len;
  if (W <= 0 || W > kMaxSlots)
    return lh::fail_arg("lh_attn_core_fwd_f32: window of %d slots outside [1,%d]", W, kMaxSlots);
  if (!wa || !hs || !batch_info || !mask01 || !indices || !align || !cached_exp || !ctx)
    return lh::fail_arg("lh_attn_core_fwd_f32: a required pointer is NULL");
  if (D >= 0 && (!tanh1 || !v_p || !p_t || !sigma))
    return lh::fail_arg("lh_attn_core_fwd_f32: local-p needs tanh1, v_p, p_t and sigma");
  if (hs_step_stride < 0 || hs_col_stride < 0)
    return lh::fail_arg("lh_attn_core_fwd_f32: negative stride");
  if (proj_col_stride == 0) proj_col_stride = H;
  if (proj_col_stride < H)
    return lh::fail_arg("lh_attn_core_fwd_f32: proj_col_stride %lld < H", proj_col_stride);

  AttnArgs a{H, B, D, W, tanh1, v_p, wa, hs, proj_col_stride, hs_step_stride, hs_col_stride, hs_steps, hs_col,
             batch_info, mask01, p_t, sigma, indices, align, cached_exp, ctx, viterbi,
             proj_col_stride, nullptr, nullptr, nullptr, 0, 0};
  const bool vec = H % 4 == 0 && lh::aligned16(wa) && lh::aligned16(hs) && lh::aligned16(ctx) &&
                   hs_step_stride % 4 == 0 && hs_col_stride % 4 == 0 && proj_col_stride % 4 == 0;
  hipStream_t st = lh::as_stream(stream);
  if (vec && W <= kRegsSlots && H <= 4 * kThreads)
    hipLaunchKernelGGL((attn_core_regs_kernel<1, kRegsSlots>), dim3(B), dim3(kThreads), 0, st, a);
  else if (vec && W <= kRegsSlots && H <= 8 * kThreads)
    hipLaunchKernelGGL((attn_core_regs_kernel<2, kRegsSlots>), dim3(B), dim3(kThreads), 0, st, a);
  // Any other: as many wavefronts per column as leave every column resident (256 CUs of 32 wavefronts).
  // Past 2048 columns none of the three does; eight wavefronts then tail off best.  1000 rows, 60 slots, with
  // sixteen / eight / four wavefronts: 512 columns 22 / 25 / 34 us, 768 columns 36 / 33 / 38, 1536 columns
  // 68 / 77 / 67, 3072 columns 121 / 113 / 127; four wavefronts with a slot at a time 38, 41, 63 and 119.
  else if (B <= 512) launch_general<1024>(a, vec, st);
  else if (B <= 1024 || B > 2048 || W > 256) launch_general<512>(a, vec, st);
  else launch_general<256>(a, vec, st);
  return lh::check_launch("lh_attn_core_fwd_f32");
}

extern "C" int lh_attn_core_projected_fwd_f32(int H, int B, int D, int hs_steps, const float *tanh1,
                                              long long tanh1_col_stride, const float *v_p,
                                              const float *h_t, long long h_t_col_stride,
                                              const float *score_mem, const float *ctx_mem,
                                              long long mem_step_stride, long long mem_col_stride,
                                              const int *mem_col, const int *batch_info,
                                              const int *mask01, const float *out_add,
                                              long long out_add_col_stride, const float *out_bias,
                                              float *p_t, float *sigma, int *indices, float *align,
                                              float *cached_exp, float *h_tild, int *viterbi,
                                              lh_stream_t stream) {
  if (H <= 0 || B <= 0 || hs_steps <= 0)
    return lh::fail_arg("lh_attn_core_projected_fwd_f32: H=%d B=%d hs_steps=%d", H, B, hs_steps);
  const int W = 2 * D + 1;
  if (D < 0 || W > LH_ATTN_PROJECTED_MAX_WINDOW || H > LH_ATTN_PROJECTED_MAX_H || H % 4 != 0)
    return lh::fail_arg("lh_attn_core_projected_fwd_f32: D=%d H=%d outside what the kernel holds in "
                        "registers (window <= %d, H <= %d, H %% 4 == 0)", D, H,
                        LH_ATTN_PROJECTED_MAX_WINDOW, LH_ATTN_PROJECTED_MAX_H);
  if (!tanh1 || !v_p || !h_t || !score_mem || !ctx_mem || !batch_info || !mask01 || !out_add ||
      !out_bias || !p_t || !sigma || !indices || !align || !cached_exp || !h_tild)
    return lh::fail_arg("lh_attn_core_projected_fwd_f32: a required pointer is NULL");
  if (tanh1_col_stride == 0) tanh1_col_stride = H;
  if (h_t_col_stride == 0) h_t_col_stride = H;
  if (out_add_col_stride == 0) out_add_col_stride = H;
  if (tanh1_col_stride < H || h_t_col_stride < H || out_add_col_stride < H || mem_step_stride < 0 ||
      mem_col_stride < 0)
    return lh::fail_arg("lh_attn_core_projected_fwd_f32: a stride is too small");
  if (!lh::aligned16(h_t) || !lh::aligned16(score_mem) || !lh::aligned16(ctx_mem) ||
      !lh::aligned16(out_add) || !lh::aligned16(out_bias) || !lh::aligned16(h_tild) ||
      h_t_col_stride % 4 != 0 || out_add_col_stride % 4 != 0 || mem_step_stride % 4 != 0 ||
      mem_col_stride % 4 != 0)
    return lh::fail_arg("lh_attn_core_projected_fwd_f32: operands must be 16-byte aligned with "
                        "strides that are multiples of 4");
  static_assert(LH_ATTN_PROJECTED_MAX_WINDOW == kRegsSlots && LH_ATTN_PROJECTED_MAX_H == 8 * kThreads,
                "limits published in the header");
  AttnArgs a{H, B, D, W, tanh1, v_p, h_t, score_mem, tanh1_col_stride, mem_step_stride, mem_col_stride,
             hs_steps, mem_col, batch_info, mask01, p_t, sigma, indices, align, cached_exp, h_tild,
             viterbi, h_t_col_stride, ctx_mem, out_add, out_bias, out_add_col_stride, 1};
  hipStream_t st = lh::as_stream(stream);
  if (H <= 4 * kThreads)
    hipLaunchKernelGGL((attn_core_regs_kernel<1, kRegsSlots>), dim3(B), dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((attn_core_regs_kernel<2, kRegsSlots>), dim3(B), dim3(kThreads), 0, st, a);
  return lh::check_launch("lh_attn_core_projected_fwd_f32");
}
