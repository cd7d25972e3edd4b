// mer_grouped.hip -- grouped per-expert path for multi-token batches (gfx950).
//
// A prefill-sized batch routes many tokens to the same expert, so each
// expert's weights can be read once per tile of its tokens.  That turns
// the per-expert work into a real dense contraction: [rows x K] weights by
// [K x tokens], run on MFMA one GGUF block (K = 32) at a
// time.  Reference semantics are those of the decode path: every
// routed (token, slot) pair computes y = W_down (silu(W_gate x) * (W_up x))
// (inference.rs:3291-3306 / :3636-3746) and the token's output is
// [x +] sum_i w_i y_i in slot order (combine_outputs_into,
// inference.rs:4472-4491; the WeightedInto loop, engine.rs:5548-5639).
//
// Launches, all on the caller's stream:
//   group_kernel   block 0 groups the routed pairs by expert (counting
//                  sort) and emits token tiles of one expert's pairs; the
//                  other blocks write x's records (below)
//   gate/up        one workgroup per (token tile, row tile): gate and up rows
//                  for the tile's tokens, SiLU * up
//   [hquant]       gbig only: h's records from f32 h
//   down           one workgroup per (token tile, row tile[, K part]) ->
//                  w_i * y_i per pair
//   combine_kernel out[t] = [x +] sum over slots in slot order
//
// Two projection kernels, by the sizes of the call (mer_grouped_plan.hpp):
//   gproj  int8 MFMA, tiles of 16 pairs, for few pairs, where streaming the
//          weights is everything;
//   gbig   f16 MFMA, tiles of 64 pairs.
//
// Numerics.  The weights are integers (Q8_0 q, or Q4_0 q-8) with one f16
// scale per 32-weight block; they are exact in int8 and in f16.
//
// gproj: each 32-element block b of an input vector (x, or h for the down
// projection) is held as s_b * v with s_b = max|x_b| / 8355711 and
// v = round(x / s_b), split into three signed base-256 digits
// v = v0 + 256 v1 + 65536 v2 (the bytes of v + 0x808080 with their top bits
// flipped).  Per block, MFMA gives the exact int32 sums Pk = sum q*vk
// (|Pk| < 2^19); P1 + 256 P2 is exact in int32, and the block contributes
// (256 (P1 + 256 P2) + P0) * d_w * s_b, formed in f32, to an f32
// accumulator.  The representation error of v is at most 2^-24 of the
// block's largest |x|; non-finite inputs give a NaN scale, so NaN
// propagates.
//
// gbig: an input vector is held as S * (hi + lo) with S a power of two that
// puts its largest element in [2^14, 2^15), hi the f16 nearest to x / S and
// lo the f16 nearest to the rest: an error of at most 2^-23 |x|, and 2^-39 of
// the vector's largest element where lo underflows (elements below 2^-16 of
// it): beside an outlier of more than 2^15 times its own block's largest
// element, an input keeps fewer bits than in gproj.  Per block two chained products, lo first, give sum q (hi + lo) in
// f32; times d_w it goes to an f32 accumulator.  The matrix unit rounds its
// sums towards minus infinity, a bias that would grow with the number of
// blocks, so every other block carries both its weights and its scale
// negated and the biases cancel (Mixtral prefill, 2048 tokens, against
// float64: 3.6e-7 without, 2.1e-7 with; the int8 kernel 2.6e-7).  Partial
// sums of 16 blocks are added up in a second accumulator (one accumulator:
// 4.0e-7, two: 1.7e-7).
//
// gbig under MER_MOE_QMM: the activation is Candle's Q8_0, integers of at most
// 8 bits, exact in one f16; a block's sum is exact in f32 and contributes
// times d_w * d_x.
//
// Operand layout of v_mfma_i32_16x16x32_i8 (gproj): lane l holds 8 int8 of A
// row (l % 16) and of B column (l % 16), covering the same 8 of the block's
// 32 k-indices (chosen by l / 16) in A and B; output lane l holds rows
// 4 (l / 16) + i, i = 0..3, of column l % 16.  Weights are staged through
// LDS as [row][block][32 int8] (rows padded to spread banks) plus f32
// scales [block][row]; the input digits are stored per (vector, block) as
// 4 groups x {8 bytes v0, 8 bytes v1, 8 bytes v2, f32 scale, pad}, so a
// lane reads the B operands of its k-group and the block scale from one
// 32-byte record.
//
// gbig takes the inputs as A rows and the weights as B columns, so an output
// lane's column is one weight row and its scale d_w one register.  Weights go
// to LDS as they are and become f16 in registers.
#include <type_traits>

#include "../../include/mer_hip.h"
#include "mer_internal.hpp"

namespace mer {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr uint32_t kBigTok = 64;             // pairs per token tile of gbig
constexpr uint32_t kGMaxRun[2] = {8, 32};    // consecutive work items on one XCD (gbig: down, gate/up)
constexpr uint32_t kNoLoad = 0x80000000u;    // an offset past every buffer: reads zeros

// ---- gproj geometry -----------------------------------------------------
constexpr uint32_t kGTok = 16;           // pairs per token tile (MFMA N)
constexpr int kGWavesPerEu = 4;
// Workgroup geometry: four waves, RT row tiles of 16 rows (RT = 4 or 8),
// stages of 32 / RT blocks, so every stage holds the same 256 two-block
// chunks (one per thread) whatever RT is.  Each wave computes every row
// tile for its 32 / (4 RT) blocks of the stage: with RT = 8 a B operand
// (one pair column's digit records of one block) serves twice as many
// weight rows, which halves the B bytes loaded per weight byte.
template <int RT>
struct GGeom {
  static constexpr uint32_t kRows = 16 * RT;                       // weight rows per workgroup
  static constexpr uint32_t kStageBlocks = 32 / RT;                // K blocks per stage
  static constexpr uint32_t kStageChunks = kStageBlocks / 2;       // two-block chunks per row per stage
  static constexpr int kWaveBlocks = (int)(kStageBlocks / 4);      // blocks of a stage per wave
  static constexpr uint32_t kRowStride = kStageBlocks * 32 + 16;   // LDS bytes per staged row (padded)
  // scales [block][row]; RT = 4 pads the row to spread the stores' banks,
  // RT = 8 keeps two slabs within a quarter of the CU's LDS
  static constexpr uint32_t kScaleStride = RT == 4 ? kRows + 4 : kRows;
  static_assert(kRows * kStageChunks == 256, "one chunk per thread and stage");
  static_assert(kWaveBlocks >= 1, "every wave has a block in every stage");
};
constexpr float kGIntMax = 8355711.0f;   // |v| bound (0x7f7f7f): v + 0x808080 stays in 24 bits
constexpr uint32_t kGRec = 8;            // dwords per (vector, block, k-group) record: 3 digit planes, scale, pad
static_assert(4 * kGRec == kGroupRecDwords, "four k-groups a block");

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }

__device__ __forceinline__ void record_status(uint32_t *status, uint32_t code) { atomicCAS(status, 0u, code); }

// How a call's input vectors are held: records of one k-group (8 elements)
// of one block.
enum GMode : int {
  kDigits = kGroupDigits,  // gproj: three int8 digit planes and the block scale
  kQ8Act = kGroupQ8Act,    // gbig, QMatMul: Q8_0 integers in f16; one scale per block
  kF16Pair = kGroupF16Pair // gbig: f16 high and low parts; one scale per vector
};

// Quantise 8 elements (one MFMA k-group) of a block whose 4 groups sit in
// 4 adjacent lanes (lane & 3 = group): block max by shuffles, then one
// 32-byte record {v0[8], v1[8], v2[8], f32 block scale, 0}, so a reader
// gets a k-group's three digit planes and the block's scale with two
// 16-byte loads.  Only lanes with `store` write.
// q8: Candle's Q8_0 activation instead (QMatMul, MER_MOE_QMM): scale
// d = amax / 127 kept as f16, q = round(v / d) half away from zero (NaN ->
// 0), so |q| <= 128 lands in plane 0 and planes 1-2 are zero.
__device__ __forceinline__ void quant_group(const float (&v)[8], uint32_t *dst, bool store, bool q8) {
  float amax = 0.f;
  int finite = 1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
    finite &= __builtin_isfinite(v[i]) ? 1 : 0;
  }
#pragma unroll
  for (int off = 1; off < 4; off <<= 1) {
    amax = __builtin_fmaxf(amax, __shfl_xor(amax, off, 64));
    finite &= __shfl_xor(finite, off, 64);
  }
  float s, inv;
  if (q8) {
    const float d = amax / 127.0f;
    inv = d != 0.0f ? 1.0f / d : 0.0f;
    s = (float)(_Float16)d;
  } else if (!finite) {
    s = __builtin_nanf("");
    inv = 0.f;
  } else if (amax == 0.f) {
    s = 0.f;
    inv = 0.f;
  } else {
    s = amax / kGIntMax;
    inv = kGIntMax / amax;
  }
  uint32_t d[6] = {0u, 0u, 0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float q;
    if (q8) {
      q = __builtin_roundf(v[i] * inv);
      q = __builtin_isnan(q) ? 0.f : __builtin_fminf(__builtin_fmaxf(q, -128.0f), 127.0f);
    } else {
      q = __builtin_rintf(v[i] * inv);
      q = __builtin_fminf(__builtin_fmaxf(q, -kGIntMax), kGIntMax);
    }
    const uint32_t u = ((uint32_t)((int32_t)q + 0x808080)) ^ 0x808080u;  // three balanced digits
#pragma unroll
    for (int k = 0; k < 3; ++k) d[2 * k + (i >> 2)] |= ((u >> (8 * k)) & 0xffu) << (8 * (i & 3));
  }
  if (!store) return;
  uint4 *o = reinterpret_cast<uint4 *>(dst);
  o[0] = make_uint4(d[0], d[1], d[2], d[3]);
  o[1] = make_uint4(d[4], d[5], __float_as_uint(s), 0u);
}

// Element of its block at position i of k-group m of gbig's records.
// Q4_0: the eight weights of qs dword m in the order unpack_q4 yields them.
template <int FMT>
__device__ __forceinline__ constexpr uint32_t kgroup_elem(uint32_t m, int i) {
  if constexpr (FMT == FMT_Q4_0) {
    constexpr int o[8] = {0, 2, 16, 18, 1, 3, 17, 19};
    return 4 * m + o[i];
  } else {
    return 8 * m + i;
  }
}

// One k-group of a vector's Q8_0 activation: 8 elements (in kgroup_elem
// order) of a block whose 4 groups sit in 4 adjacent lanes (lane & 3 = group
// m).  `vec`: the vector's region of kRecBytes a block; its first half takes
// the blocks' records (four groups of 16 bytes), the second their f32 scales,
// so a cache line holds two records.  Only lanes with `store` write.
__device__ __forceinline__ void quant_group_q8(const float (&v)[8], uint32_t *vec, uint32_t blocks, uint32_t b, uint32_t m,
                                               bool store) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
#pragma unroll
  for (int off = 1; off < 4; off <<= 1) amax = __builtin_fmaxf(amax, __shfl_xor(amax, off, 64));
  if (!store) return;
  const BlockScale bs = make_block_scale_q8(amax);
  v8h q;
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = (_Float16)quantize_elem_q8(v[i], bs.inv);
  reinterpret_cast<uint4 *>(vec)[(size_t)b * 4 + m] = __builtin_bit_cast(uint4, q);
  if (m == 0) reinterpret_cast<float *>(vec)[(size_t)blocks * (kGroupRecDwords / 2) + b] = bs.s;
}

// Eight elements of block b, k-group m of the f32 vector x, in kgroup_elem order.
template <int FMT>
__device__ __forceinline__ void load_group(const float *x, uint32_t b, uint32_t m, float (&v)[8]) {
  const float *xb = x + (size_t)b * 32;
  const float4 lo = *reinterpret_cast<const float4 *>(xb + kgroup_elem<FMT>(m, 0));
  const float4 hi = *reinterpret_cast<const float4 *>(xb + kgroup_elem<FMT>(m, 0) + (FMT == FMT_Q4_0 ? 16 : 4));
  const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t e = kgroup_elem<FMT>(0, i);
    v[i] = f[e >= 16 ? e - 12 : e];
  }
}

__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }  // -126..127

// kF16Pair records (per block the four k-groups' high parts, then their low
// parts) and scale of one f32 vector of `blocks` blocks, by the whole
// workgroup; a non-finite vector gets a NaN scale.  Two passes over x: the
// second reads caches.  The records may lie on x: a block is read and written
// by four lanes of one wave, and the stores need all of the block's loads.
template <int FMT>
__device__ __forceinline__ void quant_vector(const float *x, uint32_t blocks, uint4 *rec, float *scale) {
  __shared__ float red[16];
  const uint32_t groups = blocks * 4;
  float amax = 0.f;
  int finite = 1;
  for (uint32_t g = threadIdx.x; g < groups; g += blockDim.x) {
    float v[8];
    load_group<FMT>(x, g / 4, g % 4, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
      finite &= __builtin_isfinite(v[i]) ? 1 : 0;
    }
  }
  if (!finite) amax = INFINITY;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = __builtin_fmaxf(amax, __shfl_xor(amax, off, 64));
  if (lane_id() == 0) red[threadIdx.x / 64] = amax;
  __syncthreads();
  for (uint32_t w = 0; w < blockDim.x / 64; ++w) amax = __builtin_fmaxf(amax, red[w]);
  const bool ok = __builtin_isfinite(amax);
  const int e = max((int)(__float_as_uint(amax) >> 23) - 127, -112);  // amax >= 0
  const float inv = ok ? pow2f(14 - e) : 0.f;
  if (threadIdx.x == 0) *scale = ok ? pow2f(e - 14) : __builtin_nanf("");
  for (uint32_t g = threadIdx.x; g < groups; g += blockDim.x) {
    float v[8];
    load_group<FMT>(x, g / 4, g % 4, v);
    if (!ok) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = 0.f;
    }
    v8h hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float y = v[i] * inv;
      hi[i] = (_Float16)y;
      lo[i] = (_Float16)(y - (float)hi[i]);
    }
    uint4 *r = rec + (size_t)(g / 4) * 8 + g % 4;
    r[0] = __builtin_bit_cast(uint4, hi);
    r[4] = __builtin_bit_cast(uint4, lo);
  }
}

// Block 0: group the routed pairs by expert.  Other blocks: x's records.
template <int FMT, int MODE>
__global__ __launch_bounds__(1024) void group_kernel(GroupedParams p) {
  if (blockIdx.x > 0) {
    if constexpr (MODE == kF16Pair) {  // one token per workgroup
      const uint32_t t = blockIdx.x - 1;
      quant_vector<FMT>(p.x + (size_t)t * p.d_model, p.xblocks, reinterpret_cast<uint4 *>(p.xg) + (size_t)t * p.xblocks * 8,
                        p.xs + t);
    } else {
      const uint32_t g = (blockIdx.x - 1) * blockDim.x + threadIdx.x;  // (token, block, group)
      const uint32_t total = p.n_tok * p.xblocks * 4;
      // whole quads stay together for the shuffles; quads past the end idle
      const bool valid = g < total;
      const uint32_t tb = g / 4, m = g % 4;
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if constexpr (MODE == kQ8Act) {
        if (valid) load_group<FMT>(p.x, tb, m, v);
        quant_group_q8(v, p.xg + (size_t)(tb / p.xblocks) * p.xblocks * kGroupRecDwords, p.xblocks, tb % p.xblocks, m, valid);
      } else {
        if (valid) load_group<FMT_Q8_0>(p.x, tb, m, v);  // eight consecutive elements
        quant_group(v, p.xg + ((size_t)tb * 4 + m) * kGRec, valid, p.q8act != 0);
      }
    }
    return;
  }

  constexpr uint32_t kTile = MODE == kDigits ? kGTok : kBigTok;
  extern __shared__ uint32_t sh[];
  uint32_t *cnt = sh;                   // [table_len] pairs per expert, then offsets
  uint32_t *present = sh + p.table_len; // [table_len] the expert has a blob
  // [n_pairs] the pair's expert << 16 | its rank within the expert (both
  // < 4096), so the final scatter needs no second read of the routing
  uint32_t *pos = present + p.table_len;
  __shared__ uint32_t part[1024 * 2];
  const uint32_t tid = threadIdx.x, nth = blockDim.x;
  // Block 0 is a chain of memory round trips, and the other blocks are done
  // before it: the table and the first pair's id and weight are all loaded
  // before any is used, an expert's presence is then looked up in LDS, and
  // with one expert per thread its blob pointer stays in a register.  Against
  // weight, id, table entry and blob pointer one after another, launch to
  // launch: 512 DeepSeek tokens 17.3 -> 12.3 us, 256 Mixtral tokens 8.9 ->
  // 7.2, 64 Qwen3 tokens 7.6 -> 6.7.
  int32_t id = -1;
  float w = 0.f;
  auto fetch = [&](uint32_t q) {
    if (q < p.n_pairs) {
      id = p.ids[q];
      w = p.weights ? p.weights[q] : 1.f;
    }
  };
  fetch(tid);
  const uint8_t *const blob0 = tid < p.table_len ? reinterpret_cast<const uint8_t *>(p.table[tid]) : nullptr;
  for (uint32_t e = tid; e < p.table_len; e += nth) {
    cnt[e] = 0u;
    present[e] = (e == tid ? blob0 : reinterpret_cast<const uint8_t *>(p.table[e])) != nullptr;
  }
  __syncthreads();
  for (uint32_t q = tid; q < p.n_pairs; q += nth) {
    const uint32_t e = (uint32_t)id;
    const bool used = !(w == 0.0f);  // a zero-weight slot is skipped by the combine (engine.rs:5575-5580)
    fetch(q + nth);
    const bool ok = used && e < p.table_len && present[e] != 0u;  // a negative id is past every table
    p.pair_ok[q] = ok ? 1u : 0u;
    if (ok) {
      pos[q] = (e << 16) | atomicAdd(&cnt[e], 1u);
    } else {
      pos[q] = 0xffffffffu;
      if (used) record_status(p.status, 16u /* MER_ERR_RESIDENCY_MISS */);
    }
  }
  __syncthreads();
  // exclusive scans of pairs and tiles per expert: each thread owns a run
  // of consecutive experts
  const uint32_t per = (p.table_len + nth - 1) / nth;
  const uint32_t e0 = tid * per, e1 = min(p.table_len, e0 + per);
  uint32_t sp = 0, st = 0;
  for (uint32_t e = e0; e < e1; ++e) {
    const uint32_t c = cnt[e];
    sp += c;
    st += (c + kTile - 1) / kTile;
  }
  // Inclusive scan of (sp, st) over the block: within each wave by lane
  // shuffles, then each wave adds up the totals before it (one barrier).
  uint32_t ip = sp, it = st;
  for (uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t a = __shfl_up(ip, off, 64), b = __shfl_up(it, off, 64);
    if (lane_id() >= off) {
      ip += a;
      it += b;
    }
  }
  const uint32_t wave = tid / 64;
  if (lane_id() == 63) {
    part[wave] = ip;
    part[nth + wave] = it;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < 15; ++k)  // the totals of the waves before this one
    if (k < wave) {
      ip += part[k];
      it += part[nth + k];
    }
  uint32_t op = ip - sp, ot = it - st;
  for (uint32_t e = e0; e < e1; ++e) {
    const uint32_t c = cnt[e];
    const uint32_t nt = (c + kTile - 1) / kTile;
    cnt[e] = op;
    // full tiles, then the remainder: tiles of equal size are 4% slower at 512
    // Mixtral tokens (a remainder of up to 32 pairs takes half the products)
    for (uint32_t j = 0; j < nt; ++j) {
      GroupTile t;
      t.blob = e == tid ? blob0 : reinterpret_cast<const uint8_t *>(p.table[e]);
      t.start = op + j * kTile;
      t.count = min(kTile, c - j * kTile);
      p.tiles[ot + j] = t;
    }
    op += c;
    ot += nt;
  }
  if (tid == nth - 1) *p.n_tiles = it;
  __syncthreads();
  for (uint32_t q = tid; q < p.n_pairs; q += nth)
    if (pos[q] != 0xffffffffu) p.plist[cnt[pos[q] >> 16] + (pos[q] & 0xffffu)] = q;
}

// ---- gproj: int8 MFMA, tiles of 16 pairs ----------------------------------

// Stage one (16 RT)-row x (32 / RT)-block slab of weights into LDS: one
// two-block chunk per thread, loaded with raw buffer loads into a register
// buffer (a chunk past the row's end reads zeros) and stored as int8 rows
// plus f32 scales.
template <int FMT, int RT>
struct DigitStager {
  using Geo = GGeom<RT>;
  using T = FmtTraits<FMT>;
  static constexpr int kDw = T::kChunkDwords;
  __amdgpu_buffer_rsrc_t rsrc;           // one descriptor for the whole slab (uniform, so no per-lane waterfall)
  uint32_t voff;      // byte offset of this thread's chunk (stage 0)
  uint32_t schunk;
  uint32_t srow;
  using Buf = uint32_t[kDw];

  // fused: slab rows 0 .. 8 RT - 1 are gate rows starting at base, the
  // next 8 RT the same up rows, up_off bytes further; otherwise 16 RT
  // consecutive rows.
  __device__ __forceinline__ void init(const uint8_t *base, uint32_t up_off, uint32_t row_bytes, bool fused) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, 0x7fffffff, 0x00020000);
    const uint32_t c = threadIdx.x;  // chunk of the slab: row c / kStageChunks
    srow = c / Geo::kStageChunks;
    schunk = c % Geo::kStageChunks;
    const bool up = fused && srow >= Geo::kRows / 2;
    const uint32_t r = up ? srow - Geo::kRows / 2 : srow;
    voff = (up ? up_off : 0u) + r * row_bytes + schunk * (uint32_t)T::kChunkBytes;
  }

  // Issue the loads of stage s (its kStageChunks chunks of each row) into
  // w.  Chunks past the row's end (and every chunk of a stage past the
  // last) read zeros, so the loads are issued unconditionally: w is
  // redefined on every path, which keeps the register buffers in place
  // instead of merging two versions of them after a branch.
  __device__ __forceinline__ void load(uint32_t s, uint32_t row_chunks, Buf &w) const {
    const bool ok = s * Geo::kStageChunks + schunk < row_chunks;
    const uint32_t off = ok ? voff + s * Geo::kStageChunks * (uint32_t)T::kChunkBytes : kNoLoad;
#pragma unroll
    for (int v = 0; v < kDw / 4; ++v) {
      const uint4 q = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 16 * v, 0, 0));
      w[4 * v] = q.x;
      w[4 * v + 1] = q.y;
      w[4 * v + 2] = q.z;
      w[4 * v + 3] = q.w;
    }
    w[kDw - 1] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + 16 * (kDw / 4), 0, 0);
  }

  // Write the loaded chunks to LDS: q as int8 [row][block][32], scales
  // as f32 [block][row].
  __device__ __forceinline__ void store(const Buf &w, uint8_t *lq, float *ld) const {
    {
      uint32_t q0[8], q1[8];
      float d0, d1;
      if constexpr (FMT == FMT_Q4_0) {
        // block 0: d = w0[15:0], qs = bytes 2..17; block 1: d = w4[31:16], qs = w5..w8
        const uint32_t a[4] = {realign16(w[0], w[1]), realign16(w[1], w[2]), realign16(w[2], w[3]),
                               realign16(w[3], w[4])};
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          // element j = low nibble of qs[j], j + 16 = high nibble; int8 q - 8
          q0[m] = ((a[m] & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
          q0[4 + m] = (((a[m] >> 4) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
          const uint32_t b = w[5 + m];
          q1[m] = ((b & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
          q1[4 + m] = (((b >> 4) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
        }
        d0 = f16_bits_to_f32(w[0] & 0xffffu);
        d1 = f16_bits_to_f32(w[4] >> 16);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          q0[k] = realign16(w[k], w[k + 1]);
          q1[k] = w[9 + k];
        }
        d0 = f16_bits_to_f32(w[0] & 0xffffu);
        d1 = f16_bits_to_f32(w[8] >> 16);
      }
      const uint32_t b0 = 2 * schunk;
      uint4 *dst = reinterpret_cast<uint4 *>(lq + srow * Geo::kRowStride + b0 * 32);
      dst[0] = make_uint4(q0[0], q0[1], q0[2], q0[3]);
      dst[1] = make_uint4(q0[4], q0[5], q0[6], q0[7]);
      dst[2] = make_uint4(q1[0], q1[1], q1[2], q1[3]);
      dst[3] = make_uint4(q1[4], q1[5], q1[6], q1[7]);
      ld[b0 * Geo::kScaleStride + srow] = d0;
      ld[(b0 + 1) * Geo::kScaleStride + srow] = d1;
    }
  }
};

// One workgroup (4 waves) per (token tile, 16 RT staged rows).  FUSED:
// rows 0 .. 8 RT - 1 are gate rows, the next 8 RT the same up rows; the
// epilogue writes h = silu(g) * u for 8 RT rows = RT / 4 blocks per pair.
// Otherwise 16 RT down rows; the epilogue writes w_i * y_i per pair.
template <int FMT, bool FUSED, int RT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kGWavesPerEu))) void gproj_kernel(GroupedParams p) {
  using Geo = GGeom<RT>;
  using SG = DigitStager<FMT, RT>;
  constexpr uint32_t kRows = Geo::kRows, kSB = Geo::kStageBlocks, kStride = Geo::kRowStride, kSS = Geo::kScaleStride;
  constexpr int kWB = Geo::kWaveBlocks;
  // Two LDS slabs: stage s + 1 is stored into one while stage s is read
  // from the other, so a stage needs one barrier.
  __shared__ __attribute__((aligned(16))) uint8_t lq_buf[2][kRows * kStride];
  __shared__ __attribute__((aligned(16))) float ld_buf[2][kSB * kSS];
  uint8_t *const lq = lq_buf[0];

  const uint32_t row_tiles = FUSED ? p.d_ff / (kRows / 2) : p.d_model / kRows;
  const uint32_t tile = blockIdx.x / row_tiles;
  const uint32_t rt = blockIdx.x % row_tiles;
  if (tile >= *p.n_tiles) return;  // uniform over the workgroup
  const GroupTile gt = p.tiles[tile];
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / 64u;
  // B operands: the lane's column is the tile's pair lane % 16; its k-group
  // is lane / 16.  Every lane reads its column's pair index (16 words per
  // wave) before the weights are issued: loads complete in issue order, so
  // the B addresses never wait for weights.
  const uint32_t col = lane % 16, kg = lane / 16;
  const uint32_t pair = col < gt.count ? p.plist[gt.start + col] : 0xffffffffu;
  const bool col_ok = pair != 0xffffffffu;

  const uint32_t kblocks = FUSED ? p.xblocks : p.hblocks;  // K / 32
  const uint32_t row_chunks = kblocks / 2;
  const uint32_t row_bytes = kblocks * (uint32_t)FmtTraits<FMT>::kBlockBytes;
  SG sg;
  if constexpr (FUSED) {
    sg.init(gt.blob + (size_t)rt * (kRows / 2) * row_bytes, (uint32_t)p.proj_bytes, row_bytes, true);
  } else {
    sg.init(gt.blob + 2 * p.proj_bytes + (size_t)rt * kRows * row_bytes, 0u, row_bytes, false);
  }
  const uint32_t n_stages = (kblocks + kSB - 1) / kSB;
  // Two register buffers of weight loads: W(s) lives in wbuf[s & 1].
  typename SG::Buf wbuf[2];
  sg.load(0, row_chunks, wbuf[0]);
  sg.load(1, row_chunks, wbuf[1]);
  __builtin_amdgcn_sched_barrier(0);  // the weights go out before anything waits for the pair index

  // the lane's record of block 0 (block b's is 4 records = 8 uint4 further):
  // one 32 x 32 -> 64-bit multiply of the vector index by the record stride
  const uint4 *vrec;
  {
    const uint32_t v = col_ok ? (FUSED ? pair / p.top_k : pair) : 0u;
    const uint32_t stride = (FUSED ? p.xblocks : p.hblocks) * 8u;
    vrec = reinterpret_cast<const uint4 *>(FUSED ? p.xg : p.hg) + ((uint64_t)v * stride + kg * 2u);
  }

  float acc[RT][4];
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[a][i] = 0.f;

  // B operands of this wave's blocks of stage s (wave, wave + 4, ...) live
  // in slot s & 1.  A lane without a valid block (or a stage past the last)
  // reads block 0 of its record and gets a zero scale.
  uint2 bv[2][kWB][3];
  float bs[2][kWB];
  bool bok[2][kWB];
  auto load_b = [&](uint32_t s, int slot) {
    const uint32_t left = s < n_stages ? kblocks - s * kSB : 0u;
#pragma unroll
    for (int j = 0; j < kWB; ++j) {
      const uint32_t b = wave + 4 * j;
      bok[slot][j] = col_ok && b < left;
      const uint32_t gb = bok[slot][j] ? s * kSB + b : 0u;
      const uint4 *rp = vrec + gb * 8u;
      const uint4 r0 = rp[0], r1 = rp[1];
      bv[slot][j][0] = make_uint2(r0.x, r0.y);
      bv[slot][j][1] = make_uint2(r0.z, r0.w);
      bv[slot][j][2] = make_uint2(r1.x, r1.y);
      bs[slot][j] = __uint_as_float(r1.z);
    }
  };
  // Loads and slabs alternate between two buffers: at round s the wave
  // issues B(s + 1) and W(s + 2), stores W(s + 1) into the slab stage s
  // does not read, computes stage s and meets the others at the barrier.
  // Every load and store is issued unconditionally (weights past the last
  // stage read zeros without touching memory; B operands past it re-read
  // block 0), so each register buffer is redefined on every path: no
  // branch merges two versions of a buffer, which the compiler would
  // resolve with copies that wait for the loads just issued.  The prologue
  // leaves the loads outstanding in the loop's order (W(s + 1) older than
  // B(s + 1), W(s + 2)), so the wait counts are the same on the first round
  // as on every later one.  (Measured, config 3 gate/up: one slab with two
  // barriers per stage 69 us, two slabs 61-63 us.)
  load_b(0, 0);
  __builtin_amdgcn_sched_barrier(0);  // B(0) issued before the wait for W(0)
  sg.store(wbuf[0], lq_buf[0], ld_buf[0]);
  __syncthreads();
  auto stage = [&](uint32_t s, int slot) {
    const uint8_t *sl = lq_buf[slot];
    const float *sd = ld_buf[slot];
    const uint32_t nb = min(kSB, kblocks - s * kSB);
#pragma unroll
    for (int j = 0; j < kWB; ++j) {
      const uint32_t b = wave + 4 * j;
      if (b >= nb) break;  // uniform
      const float bsj = bok[slot][j] ? bs[slot][j] : 0.f;
      long bk[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) bk[k] = (long)(((uint64_t)bv[slot][j][k].y << 32) | bv[slot][j][k].x);
#pragma unroll
      for (int a = 0; a < RT; ++a) {
        const long av = *reinterpret_cast<const long *>(sl + (a * 16 + col) * kStride + b * 32 + kg * 8);
        const v4i z = {0, 0, 0, 0};
        const v4i p0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bk[0], z, 0, 0, 0);
        const v4i p1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bk[1], z, 0, 0, 0);
        const v4i p2 = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bk[2], z, 0, 0, 0);
        const float4 d = *reinterpret_cast<const float4 *>(&sd[b * kSS + a * 16 + kg * 4]);
        const float dd[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float hi = (float)(p1[i] + (p2[i] << 8));
          const float v = __builtin_fmaf(hi, 256.0f, (float)p0[i]);
          acc[a][i] = __builtin_fmaf(v, dd[i] * bsj, acc[a][i]);
        }
      }
    }
  };
  for (uint32_t s = 0; s < n_stages; s += 2) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t st = s + b;
      load_b(st + 1, b ^ 1);
      sg.load(st + 2, row_chunks, wbuf[b]);
      sg.store(wbuf[b ^ 1], lq_buf[b ^ 1], ld_buf[b ^ 1]);
      if (st < n_stages) stage(st, b);  // uniform
      __syncthreads();
    }
  }

  // Sum the four waves' partials (in the slabs' LDS, free now): wave w
  // then owns row tiles w, w + 4, ...
  constexpr int kOwn = RT / 4;
  typedef float RedT[RT][64][4];  // [row tile][lane][i]
  RedT *red = reinterpret_cast<RedT *>(lq);
  static_assert(sizeof(RedT) * 4 <= sizeof(lq_buf), "reduction fits in the slabs");
#pragma unroll
  for (int a = 0; a < RT; ++a)
    *reinterpret_cast<float4 *>(&red[wave][a][lane][0]) = make_float4(acc[a][0], acc[a][1], acc[a][2], acc[a][3]);
  __syncthreads();
  float4 sum[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    sum[o] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 4; ++w) {  // fixed order
      const float4 v = *reinterpret_cast<const float4 *>(&red[w][wave + 4 * o][lane][0]);
      sum[o].x += v.x;
      sum[o].y += v.y;
      sum[o].z += v.z;
      sum[o].w += v.w;
    }
  }
  // lane holds rows (wave + 4 o) * 16 + 4 * kg + i of column col

  if constexpr (FUSED) {
    __syncthreads();
    float *fin = reinterpret_cast<float *>(lq);  // [16 RT rows][16 cols]
#pragma unroll
    for (int o = 0; o < kOwn; ++o) {
      const uint32_t r = (wave + 4 * o) * 16 + 4 * kg;
      fin[(r + 0) * kGTok + col] = sum[o].x;
      fin[(r + 1) * kGTok + col] = sum[o].y;
      fin[(r + 2) * kGTok + col] = sum[o].z;
      fin[(r + 3) * kGTok + col] = sum[o].w;
    }
    __syncthreads();
    if (tid < 64 * kOwn) {
      // h block hk of the workgroup, pair column c, k-group m: h rows
      // 32 hk + 8m .. +7 (gate rows there, up rows 8 RT further)
      const uint32_t hk = tid / 64, c = (tid / 4) % 16, m = tid % 4;
      float h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float g = fin[(32 * hk + 8 * m + i) * kGTok + c];
        const float u = fin[(kRows / 2 + 32 * hk + 8 * m + i) * kGTok + c];
        h[i] = silu_mul(g, u, p.swiglu_limit);
      }
      const uint32_t pr = __shfl(pair, (int)c, 64);  // lane c of every wave holds column c's pair
      const bool ok = pr != 0xffffffffu;
      const size_t hb = (size_t)(ok ? pr : 0) * p.hblocks + rt * kOwn + hk;
      quant_group(h, p.hg + (hb * 4 + m) * kGRec, ok, p.q8act != 0);
    }
  } else {
    if (col_ok) {
      const float w = p.weights ? p.weights[pair] : 1.0f;
#pragma unroll
      for (int o = 0; o < kOwn; ++o) {
        const uint32_t r = rt * kRows + (wave + 4 * o) * 16 + 4 * kg;
        *reinterpret_cast<float4 *>(p.partial + (size_t)pair * p.d_model + r) =
            make_float4(w * sum[o].x, w * sum[o].y, w * sum[o].z, w * sum[o].w);
      }
    }
  }
}

// ---- gbig: tiles of up to 64 pairs, shared parts ---------------------------

// f16 weights of one MFMA k-group from its raw bytes (exact integers).
// The widely published bit trick: 0x6400 | n is 1024 + n, since an ulp of
// [1024, 2048) is 1.
// Q4_0: qs dword -> q - 8 of bytes' low and high nibbles, in kgroup_elem
// order: (1024 + n) - 1032, and (1024 + 16 n) / 16 - 72 for high nibbles.
// NEG: the negated weights.
template <bool NEG>
__device__ __forceinline__ v8h unpack_q4(uint32_t w) {
  const v2h c1 = {(_Float16)1032.0f, (_Float16)1032.0f};
  const v2h c2 = {(_Float16)72.0f, (_Float16)72.0f};
  const v2h r = {(_Float16)0.0625f, (_Float16)0.0625f};
  const uint32_t w8 = w >> 8;
  const v2h a = __builtin_bit_cast(v2h, (w & 0x000f000fu) | 0x64006400u);
  const v2h b = __builtin_bit_cast(v2h, (w & 0x00f000f0u) | 0x64006400u);
  const v2h c = __builtin_bit_cast(v2h, (w8 & 0x000f000fu) | 0x64006400u);
  const v2h d = __builtin_bit_cast(v2h, (w8 & 0x00f000f0u) | 0x64006400u);
  const v2h e = NEG ? c1 - a : a - c1, f = NEG ? c2 - b * r : b * r - c2;
  const v2h g = NEG ? c1 - c : c - c1, h = NEG ? c2 - d * r : d * r - c2;
  return v8h{e.x, e.y, f.x, f.y, g.x, g.y, h.x, h.y};
}
// Q8_0: eight consecutive int8: (1024 + (q + 128)) - 1152.
template <bool NEG>
__device__ __forceinline__ v8h unpack_q8(uint32_t lo, uint32_t hi) {
  const v2h c = {(_Float16)1152.0f, (_Float16)1152.0f};
  lo ^= 0x80808080u;
  hi ^= 0x80808080u;
  const v2h a = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u));
  const v2h b = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u));
  const v2h d = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u));
  const v2h e = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u));
  const v2h f = NEG ? c - a : a - c, g = NEG ? c - b : b - c, h = NEG ? c - d : d - c, i = NEG ? c - e : e - c;
  return v8h{f.x, f.y, g.x, g.y, h.x, h.y, i.x, i.y};
}

// Asynchronous copy of 16 bytes per lane from a buffer (an offset past its
// end reads zeros) to LDS at `lds` + 16 * lane.  The compiler does not see
// it: the caller waits (wait_vm) before the barrier that publishes it.  M0
// holds the LDS address and is named as written, so the compiler does not
// take an earlier value of its own to be still there (the warning that it does
// not save M0 across the statement is beside the point); s_nop: wait states
// between a write of M0 or of a resource word and its use.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void async_lds16(v4u rsrc, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds) : "memory", "m0");
}
// The same for 4 bytes per lane, to LDS at `lds` + 4 * lane.
__device__ __forceinline__ void async_lds4(v4u rsrc, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
// Wait until at most N of this wave's vector memory operations are in flight.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The same and this wave's LDS reads, then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A workgroup's item: a token tile and a row tile (with a K part folded in by
// the caller).  Items are ordered expert, token tile, row tile, and runs of
// them go to one XCD: its workgroups then share one tile's inputs in their L2
// (Mixtral prefill, 2048 tokens: 3.45 ms, 3.73 with the token tiles of a row
// tile together).  The down projection's items are fewer and longer (K parts
// and d_model / 256 row tiles), so shorter runs end more evenly: with runs of
// 8 it takes 325 us at 512 Mixtral tokens and 1.08 ms at 2048, with 32 363 us
// and 1.11 ms; gate/up is 2-4% slower with runs of 8, 64 or 112.
struct GItem {
  const uint8_t *blob;
  uint32_t start, count, rt;
};
__device__ __forceinline__ bool group_item(const GroupedParams &p, uint32_t row_tiles, uint32_t max_run, GItem *it) {
  const uint32_t total = *p.n_tiles * row_tiles;
  const uint32_t x = blockIdx.x % 8, q = blockIdx.x / 8;
  const uint32_t run = max(1u, min(total / 64, max_run));
  const uint32_t item = ((q / run) * 8 + x) * run + q % run;
  if (item >= total) return false;
  const GroupTile gt = p.tiles[item / row_tiles];
  it->blob = gt.blob;
  it->rt = item % row_tiles;
  it->start = gt.start;
  it->count = gt.count;
  return true;
}

// kBigRows weight rows by NG groups of 32 pairs on v_mfma_f32_32x32x16_f16.
// The waves split the rows (64 each) and share every block of inputs, so
// inputs and weights both go through LDS, copied asynchronously four blocks
// and a stage ahead: no load returns to registers inside the loop, so none
// waits behind another (a wave's loads return in order).  Lane l of a 32 x 32
// product holds weight row l % 32 and pairs 8 (i / 4) + 4 (l / 32) + i % 4.
//
// Bound: matrix unit and vector issue slots at the clock the power limit
// leaves (Mixtral Q4_0, 4096 pairs: 1.74 GHz, 49% and 63% of cycles busy; the
// two f16 products alone take 1.4 ms of the gate/up launch's 2.04 at the
// rate the unit sustains on such data).  One product of a wave's own has to
// saturate the unit while its other wave works on sums, which 32 x 32 tiles
// do and 16 x 16 tiles do not.  Mixtral Q4_0 top-2, 2048 tokens, against the
// int8 kernel: gate/up 4.49 -> 2.04 ms, down 2.16 -> 1.09 ms; 333 tokens under
// MER_MOE_QMM 0.84 -> 0.46 and 0.42 -> 0.24 ms (its products are half as many,
// its sums carry a scale per pair as well: vector issue).
constexpr uint32_t kBigRows = 256;
constexpr uint32_t kBigGran = 5;                          // 16-byte granules per staged row segment
constexpr uint32_t kBigStride = 16 * kBigGran;
constexpr uint32_t kBigSlab = kBigRows * kBigStride;
constexpr uint32_t kXSlots = 5;
constexpr uint32_t kX0 = 2 * kBigSlab;                    // LDS offset of the input slots
constexpr uint32_t kRecBytes = 4 * kGroupRecDwords;       // a block of a vector's inputs in memory
// LDS bytes of a block of 64 pairs' inputs: records, or records and scales
template <int MODE> constexpr uint32_t kXSlot = MODE == kF16Pair ? 64 * 128 : 64 * 64 + 4 * 256;

template <int FMT, int MODE, bool FUSED, int NG>
struct GBig {
  static constexpr int kParts = MODE == kF16Pair ? 2 : 1;  // f16 parts of an input
  static constexpr uint32_t kRec = 64u * kParts;           // bytes of a block's record
  static constexpr uint32_t kBB = FmtTraits<FMT>::kBlockBytes;
  static constexpr int kSB = FMT == FMT_Q4_0 ? 4 : 2;      // blocks per stage: 72 or 68 of 80 bytes
  static constexpr int kNW = (int)(kBigRows * kBigGran / 256);  // weight copies per wave and stage
  static constexpr uint32_t kFlush = 16 / kSB;             // stages per partial sum
  static constexpr int kXCopies = 2 * NG * kParts / 4 ? 2 * NG * kParts / 4 : 1;
  // input copies per wave and block: records, and under kQ8Act scales
  static constexpr int kNX = kXCopies + (MODE == kQ8Act ? 1 : 0);
  static constexpr int kQW = FMT == FMT_Q4_0 ? 3 : 5;      // LDS words a lane reads per row and block
  static_assert(kXSlots == 5, "inputs are copied four blocks ahead");
  static_assert(kBigRows * kBigGran % 256 == 0, "whole copies");

  static __device__ __forceinline__ void run(const GroupedParams &p, const uint8_t *blob, uint32_t start, uint32_t count,
                                             uint32_t rt, uint32_t part, uint8_t *lds) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(tid / 64u);
    const uint32_t rows = FUSED ? p.d_ff : p.d_model;
    const uint32_t row_blocks = FUSED ? p.xblocks : p.hblocks;
    // the blocks of this K part (whole stages; parts divide gate/up never)
    const uint32_t b0 = FUSED ? 0u : part * p.part_blocks;
    const uint32_t kblocks = FUSED ? row_blocks : min(p.part_blocks, row_blocks - b0);
    const uint32_t n_stages = (kblocks + kSB - 1) / kSB;
    constexpr uint32_t kOwnRows = FUSED ? kBigRows / 2 : kBigRows;
    const uint32_t row0 = rt * kOwnRows;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;

    // Weights: staged rows are 128 gate rows then the same 128 up rows
    // (FUSED), or 256 down rows, kBigGran granules each.  Rows past the
    // matrix read zeros; the buffer ends with the projection, so granules
    // that overhang its last row read zeros too.
    const uint64_t wb = reinterpret_cast<uint64_t>(blob) + (FUSED ? 0 : 2 * p.proj_bytes);
    const v4u wr = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)wb),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(wb >> 32)),
                    (uint32_t)((FUSED ? 2 : 1) * p.proj_bytes), 0x00020000u};
    uint32_t woff[kNW];
#pragma unroll
    for (int j = 0; j < kNW; ++j) {
      const uint32_t g = tid + 256u * j;
      const uint32_t r = g / kBigGran, gi = g % kBigGran;
      const uint32_t own = FUSED ? r % kOwnRows : r;
      const bool ok = row0 + own < rows;
      woff[j] = ok ? (FUSED && r >= kOwnRows ? (uint32_t)p.proj_bytes : 0u) + (row0 + own) * (row_blocks * kBB) + b0 * kBB + 16u * gi : kNoLoad;
    }
    uint32_t w_issued = 0;
    auto issue_w = [&]() {
      const uint32_t none = w_issued < n_stages ? 0u : kNoLoad;
#pragma unroll
      for (int j = 0; j < kNW; ++j) {
        async_lds16(wr, woff[j] | none, lds0 + (w_issued & 1u) * kBigSlab + wave * 1024u + 4096u * j);
        woff[j] += kSB * kBB;
      }
      ++w_issued;
    };
    // Inputs: copy i takes part i % kParts of the 16 vectors i / kParts; lane l
    // copies k-group l / 16 of vector l % 16 (64 contiguous bytes per
    // vector).  Wave w makes copies w, w + 4 (of 2 NG kParts; where there are
    // fewer than four, waves repeat them).
    const uint32_t vec_bytes = row_blocks * kRecBytes;
    const uint32_t n_vec = FUSED ? p.n_tok : p.n_pairs;
    const uint64_t xbase = reinterpret_cast<uint64_t>(FUSED ? p.xg : p.hg);
    const v4u xr = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)xbase),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(xbase >> 32)), n_vec * vec_bytes, 0x00020000u};
    uint32_t xoff[kXCopies], soff = kNoLoad;
#pragma unroll
    for (int j = 0; j < kXCopies; ++j) {
      const uint32_t i = (wave + 4u * j) % (2 * NG * kParts);
      const uint32_t n = 16 * (i / kParts) + lane % 16;
      const uint32_t pair = n < count ? p.plist[start + n] : 0u;
      // a column without a pair reads zeros
      const uint32_t vec = (FUSED ? pair / p.top_k : pair) * vec_bytes;
      xoff[j] = n < count ? vec + b0 * kRec + 64u * (i % kParts) + 16u * (lane / 16) : kNoLoad;
      if (MODE == kQ8Act && n < count) soff = vec + row_blocks * kRec + b0 * 4u;
    }
    uint32_t x_issued = 0, x_slot = 0;
    auto issue_x = [&]() {
      const uint32_t none = x_issued < kblocks ? 0u : kNoLoad;
#pragma unroll
      for (int j = 0; j < kXCopies; ++j) {
        async_lds16(xr, xoff[j] | none, lds0 + kX0 + x_slot * kXSlot<MODE> + (wave + 4u * j) % (2 * NG * kParts) * 1024u);
        xoff[j] += kRec;
      }
      if constexpr (MODE == kQ8Act) {  // the scales of the copy's 16 vectors, four times over
        async_lds4(xr, soff | none, lds0 + kX0 + x_slot * kXSlot<MODE> + 4096u + wave % (2 * NG) * 256u);
        soff += 4u;
      }
      ++x_issued;
      x_slot = x_slot + 1 == kXSlots ? 0u : x_slot + 1;
    };

    // Sums over kFlush stages in acc, of those in tot: an f32 rounding error
    // then grows with 16 + K / 512 terms instead of K / 32.
    v16f acc[2][NG], tot[2][NG];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[a][g][i] = tot[a][g][i] = 0.f;

    v8h wv[2][2];
    float dw[2];
    struct Raw {
      uint32_t q[kQW];
      _Float16 d;
    };
    // the wave's two row tiles: 32 gate rows and the same up rows, or 64 down rows
    const uint32_t trow = (FUSED ? 32 * wave : 64 * wave) + lane % 32;
    constexpr uint32_t kTileStep = (FUSED ? kOwnRows : 32) * kBigStride;
    auto fetch = [&](const uint8_t *sl, uint32_t at, int a) {
      const uint8_t *lr = sl + trow * kBigStride + a * kTileStep;
      const uint32_t *q =
          reinterpret_cast<const uint32_t *>(lr + ((at + 2 + (FMT == FMT_Q4_0 ? 8 : 16) * (lane / 32)) & ~3u));
      Raw r;
#pragma unroll
      for (int i = 0; i < kQW; ++i) r.q[i] = q[i];
      r.d = *reinterpret_cast<const _Float16 *>(lr + at);
      return r;
    };
    auto unpack = [&](auto neg, const Raw &r, uint32_t at, uint32_t live, int a) {
      constexpr bool kNeg = decltype(neg)::value;
      const uint32_t sh = (at & 2u) ? 0u : 16u;  // qs start 2 bytes past a dword in even blocks
      uint32_t q[kQW - 1];
#pragma unroll
      for (int i = 0; i + 1 < kQW; ++i) q[i] = __builtin_amdgcn_alignbit(r.q[i + 1], r.q[i], sh);
      if constexpr (FMT == FMT_Q4_0) {
        wv[a][0] = unpack_q4<kNeg>(q[0]);
        wv[a][1] = unpack_q4<kNeg>(q[1]);
      } else {
        wv[a][0] = unpack_q8<kNeg>(q[0], q[1]);
        wv[a][1] = unpack_q8<kNeg>(q[2], q[3]);
      }
      const float d = (float)r.d;
      dw[a] = __uint_as_float(__float_as_uint(kNeg ? -d : d) & live);
    };
    // input operands of group g: [k step][high, low part]; lane l takes
    // vector l % 32, k-group 2 (l / 32) + k (as the weights' words do)
    v8h x[NG][2][kParts];
    float f[16];  // kQ8Act: the scales of the lane's output pairs of one group
    const uint32_t xlane = ((lane % 32) / 16) * (1024u * kParts) + (lane / 32) * 512u + (lane % 16) * 16u;
    auto read_x = [&](const uint8_t *slot, int g) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int part = 0; part < kParts; ++part)
          x[g][k][part] = *reinterpret_cast<const v8h *>(slot + xlane + g * (2048u * kParts) + part * 1024u + k * 256u);
    };
    auto read_f = [&](const uint8_t *slot, int g) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 v = *reinterpret_cast<const float4 *>(slot + 4096u + (2 * g + q / 2) * 256u + (8 * (q % 2) + 4 * (lane / 32)) * 4u);
        f[4 * q] = v.x;
        f[4 * q + 1] = v.y;
        f[4 * q + 2] = v.z;
        f[4 * q + 3] = v.w;
      }
    };

    // Start: the copies of stages 0 and 1 and of blocks 0..3, in the loop's order.
    issue_w();
    issue_x();
    issue_x();
    issue_x();
    issue_w();
    issue_x();
    wait_vm_barrier<3 * kNX + kNW>();
    {
#pragma unroll
      for (int a = 0; a < 2; ++a) unpack(std::false_type{}, fetch(lds, 0u, a), 0u, 0xffffffffu, a);
#pragma unroll
      for (int g = 0; g < NG; ++g) read_x(lds + kX0, g);
    }
    // Block b: at its barrier the inputs of block b + 1 (and, before the
    // stage's last block, the next stage's weights) are complete, and the
    // inputs of block b are in every wave's registers, so the slot of block
    // b - 1 takes block b + 4.
    uint32_t xs = 0;
    auto stage = [&](uint32_t s) {
      const uint8_t *cur = lds + (s & 1u) * kBigSlab, *nxt = lds + ((s & 1u) ^ 1u) * kBigSlab;
      auto block = [&](auto jc) {
        constexpr int j = decltype(jc)::value;
        // Copies started after those of block b + 1 (at block b - 3): the
        // inputs of two blocks, and weights if one of these was a stage's
        // last block.  A stage's last block needs the next stage's weights
        // too, started kSB blocks before.
        constexpr bool kEnd = j == kSB - 1;
        constexpr int kYoungX = 2 * kNX + ((j + kSB - 1) % kSB == kSB - 1 || (j + 2 * kSB - 2) % kSB == kSB - 1 ? kNW : 0);
        constexpr int kYoungW = kSB * kNX;
        wait_vm_barrier<(kEnd && kYoungW < kYoungX ? kYoungW : kYoungX)>();
        // the slab's last block is in registers: the slab takes stage s + 2
        if constexpr (kEnd) issue_w();
        issue_x();
        const uint8_t *xc = lds + kX0 + xs * kXSlot<MODE>;
        xs = xs + 1 == kXSlots ? 0u : xs + 1;
        const uint8_t *xn = lds + kX0 + xs * kXSlot<MODE>;
        constexpr uint32_t nat = kEnd ? 0u : (uint32_t)(j + 1) * kBB;
        const uint8_t *nsl = kEnd ? nxt : cur;
        constexpr std::bool_constant<!kEnd && (j + 1) % 2 == 1> next_odd{};
        const uint32_t live = s * kSB + j + 1 < kblocks ? 0xffffffffu : 0u;
        v16f t[2];
        Raw raw[2];
        auto finish = [&](int g, int a) {
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[a][g][i] = __builtin_fmaf(t[a][i], MODE == kQ8Act ? dw[a] * f[i] : dw[a], acc[a][g][i]);
          if (g == NG - 1) unpack(next_odd, raw[a], nat, live, a);
        };
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            if (g == NG - 1) raw[a] = fetch(nsl, nat, a);
            v16f z;
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = 0.f;
            v16f r = z;
#pragma unroll
            for (int part = kParts - 1; part >= 0; --part)
#pragma unroll
              for (int k = 0; k < 2; ++k) r = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[g][k][part], wv[a][k], r, 0, 0, 0);
            t[a] = r;
            if (g > 0 || a > 0) {
              finish(a ? g : g - 1, a ^ 1);
              // products and sums in turn: a product occupies the matrix unit
              // long enough for sums of the tile before it to issue
              __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
              for (int i = 0; i < 2 * kParts; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (g == NG - 1 && a == 1) __builtin_amdgcn_sched_group_barrier(0x002, MODE == kQ8Act ? 28 : 10, 0);
                else __builtin_amdgcn_sched_group_barrier(0x002, MODE == kQ8Act ? 16 : 4, 0);
              }
            }
            if (MODE == kQ8Act && a == 0) read_f(xc, g);  // (after the sums that use the last group's)
            __builtin_amdgcn_sched_barrier(0);
            if (a == 1) read_x(xn, g);
          }
        finish(NG - 1, 1);
        __builtin_amdgcn_sched_barrier(0);
      };
      block(std::integral_constant<int, 0>{});
      block(std::integral_constant<int, 1>{});
      if constexpr (kSB == 4) {
        block(std::integral_constant<int, 2>{});
        block(std::integral_constant<int, 3>{});
      }
    };
    for (uint32_t s0 = 0; s0 < n_stages; s0 += kFlush) {
      for (uint32_t s = s0; s < min(n_stages, s0 + kFlush); ++s) stage(s);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            tot[a][g][i] += acc[a][g][i];
            acc[a][g][i] = 0.f;
          }
    }
    wait_vm<0>();
    __syncthreads();  // nothing writes LDS any more

    // each pair's output row and factor, read back by every lane's rows
    uint64_t *prow = reinterpret_cast<uint64_t *>(lds);
    float *pscale = reinterpret_cast<float *>(lds + 64 * 8);
    if (tid < 32 * NG && tid < count) {
      const uint32_t pr = p.plist[start + tid];
      prow[tid] = reinterpret_cast<uint64_t>(FUSED ? reinterpret_cast<float *>(p.hg) + (size_t)pr * p.d_ff : p.partial + ((size_t)part * p.n_pairs + pr) * p.d_model);
      const float sc = MODE == kQ8Act ? 1.0f : FUSED ? p.xs[pr / p.top_k] : p.hs[pr];  // the vector's scale
      pscale[tid] = !FUSED && p.weights ? sc * p.weights[pr] : sc;
    }
    __syncthreads();
    const uint32_t r = row0 + trow;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t n = 32 * g + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
        if (n >= count) continue;
        float *out = reinterpret_cast<float *>(prow[n]);
        const float sc = pscale[n];
        if constexpr (FUSED) {
          if (r < rows) out[r] = silu_mul(tot[0][g][i] * sc, tot[1][g][i] * sc, p.swiglu_limit);
        } else {
#pragma unroll
          for (int a = 0; a < 2; ++a)
            if (r + 32 * a < rows) out[r + 32 * a] = sc * tot[a][g][i];
        }
      }
  }
};

template <int FMT, int MODE, bool FUSED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gbig_kernel(GroupedParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kX0 + kXSlots * kXSlot<MODE>];  // two workgroups per CU
  const uint32_t parts = FUSED ? 1u : p.n_parts;
  GItem it;
  if (!group_item(p, ((FUSED ? 2 * p.d_ff : p.d_model) + kBigRows - 1) / kBigRows * parts, kGMaxRun[FUSED], &it)) return;  // uniform
  const uint32_t rt = it.rt / parts, part = it.rt % parts;
  if (it.count > 32) GBig<FMT, MODE, FUSED, 2>::run(p, it.blob, it.start, it.count, rt, part, lds);
  else GBig<FMT, MODE, FUSED, 1>::run(p, it.blob, it.start, it.count, rt, part, lds);
}

// The records of h for gbig's down projection, in h's place, one workgroup per
// routed pair.
template <int FMT, int MODE>
__global__ __launch_bounds__(256) void hquant_kernel(GroupedParams p) {
  const uint32_t pair = blockIdx.x;
  if (!p.pair_ok[pair]) return;
  uint32_t *hg = p.hg + (size_t)pair * p.hblocks * kGroupRecDwords;
  const float *h = reinterpret_cast<const float *>(hg);
  if constexpr (MODE == kF16Pair) {
    quant_vector<FMT>(h, p.hblocks, reinterpret_cast<uint4 *>(hg), p.hs + pair);
  } else {
    // All of h goes to registers before its place takes the records, which
    // lie closer together.  Whole quads of lanes per block: d_ff / 8 groups
    // are a multiple of 8.
    constexpr int kMax = MER_MAX_EXPERT_DIM / 8 / 256;
    const uint32_t groups = p.hblocks * 4;
    float v[kMax][8];
#pragma unroll
    for (int j = 0; j < kMax; ++j) {
      const uint32_t g = threadIdx.x + 256u * j;
      if (g < groups) load_group<FMT>(h, g / 4, g % 4, v[j]);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kMax; ++j) {
      const uint32_t g = threadIdx.x + 256u * j;
      if (g < groups) quant_group_q8(v[j], hg, p.hblocks, g / 4, g % 4, true);
    }
  }
}

// out[t] = [x +] sum over the token's valid slots, in slot order, of the
// pair partials (w_i y_i).  One thread per 4 output elements; the slots'
// validity comes from the grouping kernel, so all loads are independent.
// PARTS: the pairs' sums come in K parts.
template <bool PARTS>
__global__ __launch_bounds__(256) void gcombine_kernel(GroupedParams p) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t per_tok = p.d_model / 4;
  if (q >= p.n_tok * per_tok) return;
  const uint32_t t = q / per_tok, c = (q % per_tok) * 4;
  // Slots are summed in slot order; the loads of up to eight slots are
  // issued before any is used, so the combine costs one memory round trip
  // per eight slots instead of one per slot.
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t k0 = 0; k0 < p.top_k; k0 += 8) {
    bool ok[8];
    float4 v[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) ok[j] = k0 + j < p.top_k && p.pair_ok[t * p.top_k + k0 + j];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j)
      v[j] = ok[j] ? *reinterpret_cast<const float4 *>(p.partial + (size_t)(t * p.top_k + k0 + j) * p.d_model + c)
                   : make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t part = 1; PARTS && part < p.n_parts; ++part) {  // in order
      float4 u[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j)
        u[j] = ok[j] ? *reinterpret_cast<const float4 *>(
                           p.partial + ((size_t)part * p.n_pairs + t * p.top_k + k0 + j) * p.d_model + c)
                     : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) v[j] = make_float4(v[j].x + u[j].x, v[j].y + u[j].y, v[j].z + u[j].z, v[j].w + u[j].w);
    }
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j)
      if (ok[j]) {
        acc.x += v[j].x;
        acc.y += v[j].y;
        acc.z += v[j].z;
        acc.w += v[j].w;
      }
  }
  float4 *o = reinterpret_cast<float4 *>(p.out + (size_t)t * p.d_model + c);
  if (p.flags & (kFlagResidual | kFlagAccumulate)) {
    const float4 base = (p.flags & kFlagResidual) ? *reinterpret_cast<const float4 *>(p.x + (size_t)t * p.d_model + c)
                                                  : *o;
    acc = make_float4(base.x + acc.x, base.y + acc.y, base.z + acc.z, base.w + acc.w);
  }
  *o = acc;
}

}  // namespace

size_t grouped_group_lds_bytes(uint32_t table_len, uint32_t n_pairs) {
  return (size_t)(2 * table_len + n_pairs) * 4;
}

template <int FMT, int MODE>
static hipError_t launch_gprep(const GroupedParams &p, hipStream_t st) {
  const uint32_t quads = p.n_tok * p.xblocks * 4;
  const uint32_t gblocks = 1 + (MODE == kF16Pair ? p.n_tok : (quads + 1023) / 1024);
  hipLaunchKernelGGL((group_kernel<FMT, MODE>), dim3(gblocks), dim3(1024), grouped_group_lds_bytes(p.table_len, p.n_pairs), st,
                     p);
  return hipGetLastError();
}

hipError_t launch_grouped_prep(int fmt, const GroupedParams &p, hipStream_t st) {
  if (p.mode == kDigits) return launch_gprep<FMT_Q8_0, kDigits>(p, st);  // one layout for both formats
  if (p.mode == kQ8Act) return launch_gprep<FMT_Q4_0, kQ8Act>(p, st);
  return fmt == FMT_Q4_0 ? launch_gprep<FMT_Q4_0, kF16Pair>(p, st) : launch_gprep<FMT_Q8_0, kF16Pair>(p, st);
}

static hipError_t launch_gproj(int fmt, bool fused, const GroupedParams &p, uint32_t max_tiles, hipStream_t st) {
  // Down runs 128-row workgroups (RT = 8) wherever d_model divides by 128.
  // Gate/up does so (64 gate + 64 up rows) only from 2048 routed pairs on:
  // with fewer its launch fills too few rounds of the resident workgroup
  // slots.  Measured on the Qwen3 Q8_0 shape, gate/up us at RT = 4 / 8:
  // 16 tokens 36.7 / 41.1, 64 tokens 62.2 / 69.2, 128 tokens 89.2 / 92.1,
  // 256 tokens 144.6 / 136.4; down at 64 tokens 38.9 -> 36.1, at 256
  // tokens 94 -> 75.
  const bool wide = fused ? (p.d_ff % 64 == 0 && p.n_pairs >= 2048) : p.d_model % 128 == 0;
  const uint32_t rows = wide ? 128 : 64;
  const uint32_t grid = max_tiles * (fused ? p.d_ff / (rows / 2) : p.d_model / rows);
#define MER_GPROJ(F, FU, R) hipLaunchKernelGGL((gproj_kernel<F, FU, R>), dim3(grid), dim3(256), 0, st, p)
  if (fmt == FMT_Q4_0) {
    if (fused && wide) MER_GPROJ(FMT_Q4_0, true, 8);
    else if (fused) MER_GPROJ(FMT_Q4_0, true, 4);
    else if (wide) MER_GPROJ(FMT_Q4_0, false, 8);
    else MER_GPROJ(FMT_Q4_0, false, 4);
  } else {
    if (fused && wide) MER_GPROJ(FMT_Q8_0, true, 8);
    else if (fused) MER_GPROJ(FMT_Q8_0, true, 4);
    else if (wide) MER_GPROJ(FMT_Q8_0, false, 8);
    else MER_GPROJ(FMT_Q8_0, false, 4);
  }
#undef MER_GPROJ
  return hipGetLastError();
}

template <int FMT, int MODE, bool FUSED>
static hipError_t launch_gbig(const GroupedParams &p, uint32_t max_tiles, hipStream_t st) {
  const uint32_t row_tiles = ((FUSED ? 2 * p.d_ff : p.d_model) + kBigRows - 1) / kBigRows * (FUSED ? 1u : p.n_parts);
  // whole runs of items on each XCD: up to one run per XCD past the items
  const dim3 grid((max_tiles * row_tiles + 7) / 8 * 8 + 8 * kGMaxRun[FUSED]);
  hipLaunchKernelGGL((gbig_kernel<FMT, MODE, FUSED>), grid, dim3(256), 0, st, p);
  return hipGetLastError();
}

template <int FMT, int MODE>
static hipError_t launch_gbig_mode(bool fused, const GroupedParams &p, uint32_t max_tiles, hipStream_t st) {
  if (!fused) return launch_gbig<FMT, MODE, false>(p, max_tiles, st);
  const hipError_t e = launch_gbig<FMT, MODE, true>(p, max_tiles, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((hquant_kernel<FMT, MODE>), dim3(p.n_pairs), dim3(256), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_grouped_proj(int fmt, bool fused, const GroupedParams &p, uint32_t max_tiles, hipStream_t st) {
  if (p.mode == kDigits) return launch_gproj(fmt, fused, p, max_tiles, st);
  if (p.mode == kQ8Act) return launch_gbig_mode<FMT_Q4_0, kQ8Act>(fused, p, max_tiles, st);
  return fmt == FMT_Q4_0 ? launch_gbig_mode<FMT_Q4_0, kF16Pair>(fused, p, max_tiles, st)
                         : launch_gbig_mode<FMT_Q8_0, kF16Pair>(fused, p, max_tiles, st);
}

hipError_t launch_grouped_combine(const GroupedParams &p, hipStream_t st) {
  const uint32_t cq = p.n_tok * (p.d_model / 4);
  const dim3 grid((cq + 255) / 256);
  if (p.n_parts > 1) hipLaunchKernelGGL(gcombine_kernel<true>, grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL(gcombine_kernel<false>, grid, dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace mer
