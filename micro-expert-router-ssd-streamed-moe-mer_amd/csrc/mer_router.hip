// mer_router.hip -- LinearGate routing on the GPU for gfx950.
//
// Two launches restate LinearGate::route_with_scratch
// (gating.rs:395-476) with its full routing surface (with_routing,
// gating.rs:207-268):
//   logits    = W x                               (W: [n_experts][d_model] f32)
//               router_logits_kernel: one wave per (expert, group of 4
//               tokens), so the gate matrix streams through every CU
//               with many loads in flight (one token reads all of W);
//               router_logits_mfma_kernel: 32 tokens x 32 experts per
//               workgroup, for large batches;
//   the rest, one wave per token (router_kernel; its top-k in registers and
//   the weights of all slots at once: 11.5 -> 7.6 us for 2048 tokens, top-8 of
//   128):
//   scores    = softmax(logits) (transformer.rs:2807, non-finite rows fall
//               back to uniform) or sigmoid (gating.rs:271-279)
//   selection = scores + correction_bias          (bias optional)
//   optional group filter (gating.rs:321-370): groups scored by the sum of
//               their two best selection scores, the best topk_group survive
//   top-k over surviving experts with finite selection (higher first, lower
//               id on ties; insert_top_expert, gating.rs:296-320)
//   weights   = unbiased scores at the chosen experts, renormalised when
//               their sum is finite and > 0, then scaled.
// The dot products are f32 with a different summation order from the
// reference's matvec, so logits agree to f32 rounding, not bit for bit.
#include "mer_internal.hpp"

namespace mer {

namespace {

constexpr int kRouterThreads = 256;
constexpr int kRouterWaves = kRouterThreads / 64;
constexpr uint32_t kRouterTokGroup = 4;  // tokens per logits wave
constexpr uint32_t kRouterTile = 32;      // tokens and experts per workgroup of the MFMA kernel
constexpr int kRouterMWaves = 8;           // its waves
constexpr uint32_t kRouterStage = 16 * kRouterMWaves;  // its k-indices per stage
constexpr uint32_t kRouterStride = kRouterStage + 4;   // LDS row, padded to spread banks
typedef float v4f __attribute__((ext_vector_type(4)));
// The per-token selection runs as one wave: its reductions are shuffles and
// its barriers cost no waiting on other waves.
constexpr int kSelThreads = 64;
constexpr int kSelWaves = 1;

// Total order of f32 (f32::total_cmp) as a signed integer key.
__device__ __forceinline__ int32_t total_key(float v) {
  const int32_t b = __float_as_int(v);
  return b ^ ((b >> 31) & 0x7fffffff);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Candidate (key, id) comparison: better = larger key, then smaller id.
__device__ __forceinline__ bool better(int32_t ka, int32_t ia, int32_t kb, int32_t ib) {
  return ka > kb || (ka == kb && ia < ib);
}

// (key, id) as one unsigned 64-bit value ordered like `better`: the key with
// its sign bit flipped above the complemented id.  0 is below every
// candidate (a real one has a complemented id >= 2^32 - 1024).
__device__ __forceinline__ uint64_t pack_candidate(int32_t key, uint32_t id) {
  return ((uint64_t)((uint32_t)key ^ 0x80000000u) << 32) | (uint64_t)(0xffffffffu - id);
}

// Largest packed candidate of the wave, in every lane: DPP row rotations
// (8, 4, 2, 1) give each lane its row's maximum, then the four row maxima
// are read out.  No LDS-routed permutes on the path.
__device__ __forceinline__ uint64_t wave_max_candidate(uint64_t v) {
  uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
#define MER_ROW_ROR_MAX(CTRL)                                                                     \
  {                                                                                               \
    const uint32_t l2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, CTRL, 0xf, 0xf, false); \
    const uint32_t h2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, CTRL, 0xf, 0xf, false); \
    if (h2 > hi || (h2 == hi && l2 > lo)) {                                                       \
      hi = h2;                                                                                    \
      lo = l2;                                                                                    \
    }                                                                                             \
  }
  MER_ROW_ROR_MAX(0x128)
  MER_ROW_ROR_MAX(0x124)
  MER_ROW_ROR_MAX(0x122)
  MER_ROW_ROR_MAX(0x121)
#undef MER_ROW_ROR_MAX
  uint64_t best = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint64_t c = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, 16 * r) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)lo, 16 * r);
    best = c > best ? c : best;
  }
  return best;
}

}  // namespace

// logit_buf[t][e] = W[e] . x[t] for a group of up to 4 tokens per wave.
// VEC: 16-byte loads (d_model % 4 == 0 and 16-byte aligned gate and x).
template <bool VEC>
__global__ __launch_bounds__(kRouterThreads) void router_logits_kernel(RouterParams p) {
  const uint32_t n_eg = (p.n_experts + kRouterWaves - 1) / kRouterWaves;
  const uint32_t eg = blockIdx.x % n_eg, tg = blockIdx.x / n_eg;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t e = eg * kRouterWaves + wave;
  if (e >= p.n_experts) return;  // the whole wave; nothing below synchronises the workgroup
  const uint32_t t0 = tg * kRouterTokGroup;
  const uint32_t nt = min(kRouterTokGroup, p.n_tokens - t0);
  const float *w = p.gate + (size_t)e * p.d_model;
  const float *x = p.x + (size_t)t0 * p.d_model;
  float acc[kRouterTokGroup] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
#pragma unroll 8
    for (uint32_t d = 4 * lane; d < p.d_model; d += 256) {
      const float4 wv = *reinterpret_cast<const float4 *>(w + d);
#pragma unroll
      for (uint32_t j = 0; j < kRouterTokGroup; ++j)
        if (j < nt) {
          const float4 xv = *reinterpret_cast<const float4 *>(x + (size_t)j * p.d_model + d);
          acc[j] = __builtin_fmaf(wv.x, xv.x, acc[j]);
          acc[j] = __builtin_fmaf(wv.y, xv.y, acc[j]);
          acc[j] = __builtin_fmaf(wv.z, xv.z, acc[j]);
          acc[j] = __builtin_fmaf(wv.w, xv.w, acc[j]);
        }
    }
  } else {
#pragma unroll 8
    for (uint32_t d = lane; d < p.d_model; d += 64) {
      const float wv = w[d];
#pragma unroll
      for (uint32_t j = 0; j < kRouterTokGroup; ++j)
        if (j < nt) acc[j] = __builtin_fmaf(wv, x[(size_t)j * p.d_model + d], acc[j]);
    }
  }
#pragma unroll
  for (uint32_t j = 0; j < kRouterTokGroup; ++j) {
    const float v = wave_sum(acc[j]);
    if (lane == 0 && j < nt) p.logit_buf[(size_t)(t0 + j) * p.n_experts + e] = v;
  }
}

// The same for many tokens: 32 tokens by 32 experts per workgroup on
// v_mfma_f32_16x16x4_f32, so each element of x and W is loaded once per 32
// logits instead of once per logit or per four.  Stages of 128 k-indices go
// through LDS, read whole rows at a time: rows of a power-of-two length start
// in one L2 channel and one L1 set, so 16 rows per load instruction (straight
// from the operand layout) ran at a third of the rate.  Every workgroup takes
// the stages in the same order, so a logit does not depend on the tile that
// its token and its expert fall in and equal gate rows tie exactly (starting
// each workgroup at another stage gains nothing: 128 experts x 2048, 2048
// tokens 24.3 us, 24.5 in order; 256 x 7168, 2048 tokens 90 and 86).  Another
// order than the kernel above, so a call on either side of the choice between
// them differs in the last bits.  Wave w takes the stage's run w of
// 16 k-indices; lane l holds four consecutive elements of row l % 16
// (k-indices 4 (l / 16) .. + 3 of the run), one for each of four products,
// which is the same permutation of k on both sides.  Sums are kept short, as
// they are in the kernel above (32 terms per lane): 16 products, eight of
// those, the rest, then the waves.  Rows and k past the ends are 0.
// ALIGNED: d_model % 4 == 0, so no 16 bytes hold two rows' elements.
template <bool ALIGNED>
__global__ __launch_bounds__(64 * kRouterMWaves) void router_logits_mfma_kernel(RouterParams p) {
  __shared__ __attribute__((aligned(16))) float lds[2][2 * kRouterTile][kRouterStride];
  // the workgroups of one token tile run on one XCD, whose L2 keeps its x
  const uint32_t n_eg = (p.n_experts + kRouterTile - 1) / kRouterTile;
  const uint32_t q = blockIdx.x / 8;
  const uint32_t t0 = ((q / n_eg) * 8 + blockIdx.x % 8) * kRouterTile, e0 = (q % n_eg) * kRouterTile;
  if (t0 >= p.n_tokens) return;  // the whole workgroup
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t row = lane % 16, kg = lane / 16;
  // staging: thread t copies 16 bytes (column t % 32) of rows t / 32 + 16 j;
  // rows 0..31 are tokens (j < 2), 32..63 experts
  const uint32_t nt = min(kRouterTile, p.n_tokens - t0), ne = min(kRouterTile, p.n_experts - e0);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(p.x + (size_t)t0 * p.d_model), 0, nt * p.d_model * 4u, 0x00020000);
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(p.gate + (size_t)e0 * p.d_model), 0, ne * p.d_model * 4u, 0x00020000);
  const uint32_t srow = threadIdx.x / 32, scol = 4 * (threadIdx.x % 32);
  const uint32_t stages = (p.d_model + kRouterStage - 1) / kRouterStage;
  uint32_t next = 0;
  struct Buf {
    v4f v[4];
    uint32_t k;
  };
  auto load = [&](Buf &b) {
    b.k = kRouterStage * next + scol;
    ++next;  // loads past the last stage read zeros
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t o = b.k < p.d_model ? ((srow + 16 * (j % 2)) * p.d_model + b.k) * 4u : 0x80000000u;
      b.v[j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(j < 2 ? xr : gr, o, 0, 0));
    }
  };
  auto store = [&](const Buf &b, uint32_t slab) {
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      v4f v = b.v[j];
      if constexpr (!ALIGNED) {
#pragma unroll
        for (uint32_t i = 1; i < 4; ++i) v[i] = b.k + i < p.d_model ? v[i] : 0.f;
      }
      *reinterpret_cast<v4f *>(&lds[slab][srow + 16 * j][scol]) = v;
    }
  };
  v4f part[4], sum[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) part[i] = sum[i] = v4f{0.f, 0.f, 0.f, 0.f};
  Buf buf[2];
  load(buf[0]);
  load(buf[1]);
  store(buf[0], 0);
  load(buf[0]);
  __syncthreads();
  // stage s is in slab s % 2, s + 1 and s + 2 in buf
  for (uint32_t s = 0; s < stages; s += 2) {
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u) {
      if (s + u >= stages) break;  // uniform
      v4f in[4], t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        in[i] = *reinterpret_cast<const v4f *>(&lds[u][16 * i + row][16 * wave + 4 * kg]);
        t[i] = v4f{0.f, 0.f, 0.f, 0.f};
      }
      store(buf[u ^ 1], u ^ 1);
      load(buf[u ^ 1]);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i)  // tile i: token half i / 2, expert half i % 2
          t[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(in[i / 2][k], in[2 + i % 2][k], t[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) part[i] += t[i];
      __syncthreads();
    }
    if ((s & 7u) == 6u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sum[i] += part[i];
        part[i] = v4f{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  v4f(*red)[4][64] = reinterpret_cast<v4f(*)[4][64]>(lds);  // [wave][tile][lane]
  static_assert(sizeof(lds) >= kRouterMWaves * 4 * 64 * sizeof(v4f), "the reduction fits in the stages' LDS");
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][i][lane] = sum[i] + part[i];
  __syncthreads();
  if (wave >= 4) return;
  v4f v = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < kRouterMWaves; ++w) v += red[w][wave][lane];
  const uint32_t e = e0 + 16 * (wave % 2) + row;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t t = t0 + 16 * (wave / 2) + 4 * kg + i;
    if (t < p.n_tokens && e < p.n_experts) p.logit_buf[(size_t)t * p.n_experts + e] = v[i];
  }
}

// NPER: experts per lane, at least n_experts / 64.
template <int NPER>
__global__ __launch_bounds__(kSelThreads) void router_kernel(RouterParams p) {
  extern __shared__ float smem[];
  float *scores = smem;                               // [n_experts]
  float *selection = scores + p.n_experts;            // [n_experts]
  __shared__ float red_f[kSelWaves];
  __shared__ uint32_t group_ok[kMaxRouterExperts / 32];
  // the group filter's working arrays (thread 0's), in LDS (as private arrays they would live in
  // scratch memory, whose set-up dominates a launch this small)
  __shared__ int32_t sel_g[kMaxRouterGroups];  // surviving groups, best first
  __shared__ float sel_s[kMaxRouterGroups];
  __shared__ int32_t flag_bad;

  const uint32_t t = blockIdx.x;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  if (tid == 0) flag_bad = 0;
  // the token's logits, from router_logits_kernel
  for (uint32_t e = tid; e < p.n_experts; e += kSelThreads) scores[e] = p.logit_buf[(size_t)t * p.n_experts + e];
  __syncthreads();

  // ---- scores -------------------------------------------------------------
  if (p.scoring == 0) {
    // softmax: max over non-NaN values; a NaN or a non-finite max makes the
    // row uniform (softmax_inplace's fallback)
    float m = -INFINITY;
    for (uint32_t e = tid; e < p.n_experts; e += kSelThreads) {
      const float v = scores[e];
      if (v != v) flag_bad = 1;  // benign race: every writer stores 1
      else m = __builtin_fmaxf(m, v);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, off, 64));
    if (lane == 0) red_f[wave] = m;
    __syncthreads();
    m = red_f[0];
    for (int i = 1; i < kSelWaves; ++i) m = __builtin_fmaxf(m, red_f[i]);
    const bool uniform = flag_bad || !__builtin_isfinite(m);
    __syncthreads();
    float s = 0.f;
    for (uint32_t e = tid; e < p.n_experts; e += kSelThreads) {
      const float v = uniform ? 1.f : expf(scores[e] - m);
      scores[e] = v;
      s += v;
    }
    s = wave_sum(s);
    if (lane == 0) red_f[wave] = s;
    __syncthreads();
    float sum = 0.f;
    for (int i = 0; i < kSelWaves; ++i) sum += red_f[i];
    for (uint32_t e = tid; e < p.n_experts; e += kSelThreads)
      scores[e] = uniform ? 1.0f / (float)p.n_experts : (sum > 0.f ? scores[e] / sum : scores[e]);
  } else {
    for (uint32_t e = tid; e < p.n_experts; e += kSelThreads) scores[e] = 1.0f / (1.0f + expf(-scores[e]));
  }
  __syncthreads();
  for (uint32_t e = tid; e < p.n_experts; e += kSelThreads)
    selection[e] = p.bias ? scores[e] + p.bias[e] : scores[e];
  for (uint32_t i = tid; i < kMaxRouterExperts / 32; i += kSelThreads) group_ok[i] = 0xffffffffu;
  __syncthreads();

  // ---- optional group filter ----------------------------------------------
  const bool grouped = p.n_group > 1 && p.topk_group > 0 && p.topk_group < p.n_group && p.n_experts % p.n_group == 0;
  if (grouped && tid == 0) {
    const uint32_t gs = p.n_experts / p.n_group;
    uint32_t c = 0;
    for (uint32_t g = 0; g < p.n_group; ++g) {
      float top1 = -INFINITY, top2 = -INFINITY;
      for (uint32_t i = 0; i < gs; ++i) {
        const float v = selection[g * gs + i];
        if (v > top1) {
          top2 = top1;
          top1 = v;
        } else if (v > top2) {
          top2 = v;
        }
      }
      const float sum = top1 + (__builtin_isfinite(top2) ? top2 : 0.0f);
      // insert_top_group: total order, lower id on ties, keep topk_group
      uint32_t pos = c;
      for (uint32_t i = 0; i < c; ++i)
        if (better(total_key(sum), (int32_t)g, total_key(sel_s[i]), sel_g[i])) {
          pos = i;
          break;
        }
      if (pos == c && c >= p.topk_group) continue;
      const uint32_t last = c < p.topk_group ? c : p.topk_group - 1;
      for (uint32_t i = last; i > pos; --i) {
        sel_g[i] = sel_g[i - 1];
        sel_s[i] = sel_s[i - 1];
      }
      sel_g[pos] = (int32_t)g;
      sel_s[pos] = sum;
      if (c < p.topk_group) ++c;
    }
    for (uint32_t i = 0; i < kMaxRouterExperts / 32; ++i) group_ok[i] = 0u;
    for (uint32_t i = 0; i < c; ++i)
      for (uint32_t e = (uint32_t)sel_g[i] * gs; e < ((uint32_t)sel_g[i] + 1) * gs; ++e) group_ok[e >> 5] |= 1u << (e & 31u);
  }
  __syncthreads();

  // ---- top-k: k rounds of a wave arg-max -------------------------------
  // Each lane keeps its experts' (lane, lane + 64, ...) packed candidates in
  // registers; the winner of a round (the largest) is known to every lane and
  // its owner drops it.
  uint64_t cand[NPER];
#pragma unroll
  for (uint32_t i = 0; i < NPER; ++i) {
    const uint32_t e = lane + 64 * i;
    cand[i] = 0;
    if (e < p.n_experts) {
      const float v = selection[e];
      if (__builtin_isfinite(v) && ((group_ok[e >> 5] >> (e & 31u)) & 1u)) cand[i] = pack_candidate(total_key(v), e);
    }
  }
  uint32_t count = 0;
  int32_t chosen = 0;  // lane r: the expert of round r
  for (uint32_t r = 0; r < p.top_k; ++r) {
    uint64_t mine = cand[0];
#pragma unroll
    for (uint32_t i = 1; i < NPER; ++i) mine = cand[i] > mine ? cand[i] : mine;
    const uint64_t best = wave_max_candidate(mine);
    if (best == 0) break;  // the same in every lane: no eligible expert left
#pragma unroll
    for (uint32_t i = 0; i < NPER; ++i)
      if (cand[i] == best) cand[i] = 0;
    if (lane == r) chosen = (int32_t)(0xffffffffu - (uint32_t)best);
    count = r + 1;
  }

  // ---- weights: lane i's slot; the sum in slot order ------------------------
  static_assert(kMaxRouterTopK <= 64, "one lane per slot");
  float w = lane < count ? scores[chosen] : 0.f;
  float sum = 0.f;
  for (uint32_t i = 0; i < count; ++i) sum = sum + __shfl(w, (int)i, 64);
  if (p.normalise && __builtin_isfinite(sum) && sum > 0.f) w = w / sum;
  if (p.scaling != 1.0f && __builtin_isfinite(p.scaling)) w = w * p.scaling;
  if (lane < p.top_k) {
    p.ids[(size_t)t * p.top_k + lane] = lane < count ? chosen : -1;
    p.weights[(size_t)t * p.top_k + lane] = lane < count ? w : 0.0f;
  }
}

hipError_t launch_router(const RouterParams &p, hipStream_t st) {
  const uint32_t n_eg = (p.n_experts + kRouterWaves - 1) / kRouterWaves;
  const uint32_t n_tg = (p.n_tokens + kRouterTokGroup - 1) / kRouterTokGroup;
  const bool vec = p.d_model % 4 == 0 && (uintptr_t)p.gate % 16 == 0 && (uintptr_t)p.x % 16 == 0;
  // One workgroup of the MFMA kernel takes ~1 us per 128 k-indices whatever
  // the batch; the other kernel's time grows with tokens * experts.  Call us,
  // that kernel / MFMA: 128 experts x 2048: 256 tokens 20 / 22, 512 tokens
  // 32 / 23, 2048 tokens 101 / 25; 256 x 7168: 64 tokens 29 / 54, 2048 tokens
  // 577 / 93; 160 x 3000, 300 tokens 55 / 46; 8 x 4096, 2048 tokens 26 / 35.
  if ((uint64_t)p.n_tokens * p.n_experts >= 40000) {
    const dim3 grid(8 * ((p.n_tokens + 8 * kRouterTile - 1) / (8 * kRouterTile)) * ((p.n_experts + kRouterTile - 1) / kRouterTile));
    if (vec) hipLaunchKernelGGL(router_logits_mfma_kernel<true>, grid, dim3(64 * kRouterMWaves), 0, st, p);
    else hipLaunchKernelGGL(router_logits_mfma_kernel<false>, grid, dim3(64 * kRouterMWaves), 0, st, p);
  } else if (vec) hipLaunchKernelGGL(router_logits_kernel<true>, dim3(n_eg * n_tg), dim3(kRouterThreads), 0, st, p);
  else hipLaunchKernelGGL(router_logits_kernel<false>, dim3(n_eg * n_tg), dim3(kRouterThreads), 0, st, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const size_t lds = sizeof(float) * 2 * (size_t)p.n_experts;
  const dim3 grid(p.n_tokens), block(kSelThreads);
  if (p.n_experts <= 128) hipLaunchKernelGGL(router_kernel<2>, grid, block, lds, st, p);
  else if (p.n_experts <= 256) hipLaunchKernelGGL(router_kernel<4>, grid, block, lds, st, p);
  else hipLaunchKernelGGL(router_kernel<(int)kMaxRouterExperts / 64>, grid, block, lds, st, p);
  return hipGetLastError();
}

}  // namespace mer
