// Causal paged attention of prompt tokens on the fp16 matrix cores (the prefill branch of the
// reference's paged_attention, attention.py:249-257, whose gather + SDPA this replaces), over the
// int8 or the fp32 cache.
//
// The row kernel (paged_decode.hip) gives every token a query row of its own: it reads the whole
// context once per token and runs on the VALU (2 prompts of ~900 tokens after ~1000 cached ones and 24
// decode rows: 962 us). Here a workgroup takes 64 query tokens and two query heads of one kv head and
// walks the context in tiles of 64 tokens (fp32 cache: 32) that its four wavefronts share: 79 us for
// the two prompts, 1000 new tokens over the fp32 cache 776 -> 51.
//
// Precision is fp32's: q, the weights and fp32 K / V rows are each split into two fp16 pieces (22
// bits) after scaling by a power of two (per query row and head, per cache row); int8 codes are exact
// in fp16, their scales stay in fp32 on the score and on the weight. Products are exact and summed in
// fp32. Measured against float64, 1000 new tokens: int8 1.2e-7, fp32 1.6e-7 (the row kernel 1.7e-7, 1.6e-7).
//
// Both products are transposed: S^T = K Q^T leaves lane (fr, fc) the scores of query fr for tokens
// 16 tt + 4 fc + e, which is the B operand layout of O^T = V^T P^T when the k order of that product is
// chosen as those tokens. So the weights go from accumulator to operand in place, a query's running
// reference and sum are per-lane scalars, and only a moving reference needs other lanes. V is
// transposed on its way into LDS (4 tokens x 4 dims per thread with byte permutes).
//
// Each wavefront brings its own quarter of the next context tile straight into LDS while the
// current one is computed, then widens it into MFMA fragments (positions in a fragment are permuted so
// that neither the writes nor the reads conflict). Long contexts are split into chunks where the
// tiles alone would leave CUs idle, and a second launch adds the chunks.
// What bounds it: per context tile a wavefront issues 128 products (2048 matrix-core cycles) and about 500
// VALU instructions (exp, the splits, widening, the sums); the two wavefronts of a SIMD overlap them
// only in part: 8192 tokens, in one chunk, run at 500 TFLOP/s of attention, 1 PFLOP/s of fp16 products.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

using lsh::kWave;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kQT = 64;         // query tokens of a tile: 16 per wavefront
constexpr int kHeads = 2;       // query heads of a workgroup (of one kv head)
constexpr int kWaves = 4;
constexpr int kFrag = 1024;     // bytes of a fragment: 64 lanes x 8 fp16
constexpr int kMaxSplits = 64;  // chunks of a tile: one per lane in the search for a workgroup's chunk
constexpr float kLog2e = 1.4426950408889634f;
// Weights: p = exp2(score - ref), ref the running max of score + log2(v scale) (so that p v_scale
// stays below 2^kLazy: the reference moves only past that), times v_scale 2^up, which brings the fp16
// pieces near the top of their range. 2^up is a factor of the staged v scales rather than of p, and a
// chunk takes it from its first token's v scale (kTop - log2 of it, within kUpMin .. kUpMax), so that
// the scales it stages are near 2^kTop: p's exponent stays small, and with it the rounding of its
// argument (with 2^kTop for all the arguments reach 13 and a chunk's reference 20, rounded as such:
// float64 error over the fp32 cache 2.2e-7 instead of 1.6e-7).
constexpr float kLazy = 4.f;
constexpr int kTop = 11, kUpMin = -5, kUpMax = 23;
// A v scale that is not finite (or too large to stage) is staged as kHuge, so that a weight of 0 (a token
// that the query does not see) times it stays 0. The queries that see one are computed again, row by
// row (plain_chunk), and so are those whose scores were not finite.
constexpr float kHuge = 3.402823466e38f, kMaxLv = 100.f;

struct PrefillArgs {
  const float* q;
  const void* kc;
  const void* vc;
  const float* ks;
  const float* vs;
  const int64_t* bt;
  const int64_t* tiles;  // [n][4]: first query row, query rows, tokens the first row sees, table row
  const float* q_mult;
  float* out;
  float* part_acc;  // [chunk of a split tile (part_index)][kv head, head pair][kHeads][kQT][D]
  float* part_rl;   // ... [kHeads][kQT][2] (reference, sum)
  int64_t num_slots;
  int Hq, Hk, G, pairs;  // pairs: head pairs of a kv head
  int max_blocks, bs, bs_shift;
  int chunk, splits;  // most tokens of a context chunk (a multiple of 64), most chunks of a tile
  int whole;          // tiles, at the end of the list, that are one chunk
  float scale;
  // Workgroups in order: the first chunks of all tiles, the second chunks of the tiles that have one (the
  // first so many), ...: start[z] is where the chunks z begin, start[splits] their count.
  int start[kMaxSplits + 1];
};

// Tokens of the chunks of a context: as few chunks of at most `most` tokens as cover it, evened out.
__host__ __device__ inline int chunk_size(int ctx, int most) {
  const int n = (ctx + most - 1) / most, even = (ctx + n - 1) / n;
  return (even + 63) / 64 * 64;
}

// What workgroup `unit` of a head pair computes.
struct Work {
  int tile, chunk;
  int row0, rows, sees, tab;  // the tile
  int ctx, size;              // tokens its last row sees, tokens of a chunk
  int k0, k1;                 // the chunk's tokens (none: k0 >= ctx)
};

__device__ __forceinline__ Work work_of(const PrefillArgs& a, int unit) {
  Work w;
  w.tile = unit;
  w.chunk = 0;
  if (a.splits > 1) {
    const int lane = threadIdx.x % kWave, from = a.start[lane + 1];
    w.chunk = __builtin_popcountll(__ballot(lane + 1 < a.splits && unit >= from));
    w.tile = unit - a.start[w.chunk];
  }
  const int64_t* t = a.tiles + 4 * w.tile;
  w.row0 = static_cast<int>(t[0]);
  w.rows = static_cast<int>(t[1]);
  w.sees = static_cast<int>(t[2]);
  w.tab = static_cast<int>(t[3]);
  w.ctx = w.sees + w.rows - 1;
  w.size = chunk_size(w.ctx, a.chunk);
  w.k0 = w.chunk * w.size;
  w.k1 = min(w.ctx, w.k0 + w.size);
  return w;
}

// Where a tile's chunk lies among the chunks of split tiles.
__device__ __forceinline__ int part_index(const PrefillArgs& a, int tile, int z) {
  return z == 0 ? tile : a.start[z] + tile - a.whole;
}

__device__ __forceinline__ f16x2 as_h2(uint32_t w) { return __builtin_bit_cast(f16x2, w); }
__device__ __forceinline__ uint32_t as_u(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f32x4 mfma(const f16x8& a, const f16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Max over the lanes with the same lane % 16.
__device__ __forceinline__ float max_over_fc(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(a[0])), __builtin_bit_cast(float, static_cast<uint32_t>(a[1])));
  const uint32_t w = __builtin_bit_cast(uint32_t, v);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(b[0])), __builtin_bit_cast(float, static_cast<uint32_t>(b[1])));
}
__device__ __forceinline__ float sum_over_fc(float v) {
  v += __shfl_xor(v, 16, kWave);
  return v + __shfl_xor(v, 32, kWave);
}

__device__ __forceinline__ int exponent_to_15(float top) {  // 2^result brings top to [2^14, 2^15)
  int ex = 0;
  if (top > 0.f && top < __builtin_inff()) ex = 15 - __builtin_amdgcn_frexp_expf(top);
  return ex < -126 ? -126 : (ex > 126 ? 126 : ex);
}

// Two values -> packed hi and lo pieces. The empty asm makes hi one value: left to itself the
// compiler converts a second time for lo's subtraction (fused with the product that made the
// value, which rounds differently).
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  hi = as_u(__builtin_convertvector(f32x2{a, b}, f16x2));
  asm("" : "+v"(hi));
  const f16x2 h = as_h2(hi);
  const f16x2 l = {static_cast<_Float16>(__builtin_fmaf(a, 1.f, -static_cast<float>(h[0]))),
                   static_cast<_Float16>(__builtin_fmaf(b, 1.f, -static_cast<float>(h[1])))};
  lo = as_u(l);
}

// bytes b0, b1 of `pair` (each value + 128) -> two fp16 values, exact
template <uint32_t SEL>
__device__ __forceinline__ uint32_t bytes_to_h2(uint32_t w) {
  const f16x2 k = {1152, 1152};
  return as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, w, SEL)) - k);
}

template <typename E>
struct Geo;
template <>
struct Geo<int8_t> {
  static constexpr int KT = 64, PL = 1;  // tokens of a context tile, fp16 pieces of K and V
};
template <>
struct Geo<float> {
  static constexpr int KT = 32, PL = 2;
};

// Scheduling of a chain of N steps that read PL fragments from LDS and run M products each: the
// reads go kAhead steps before their products (left to itself the compiler reads a fragment right
// before them and waits out the LDS latency at every step).
template <int N, int PL, int M>
__device__ __forceinline__ void read_ahead() {
  constexpr int kAhead = 2, kRead = 0x100, kMfma = 0x8;
  __builtin_amdgcn_sched_group_barrier(kRead, kAhead * PL, 0);
#pragma unroll
  for (int i = 0; i < N - kAhead; ++i) {
    __builtin_amdgcn_sched_group_barrier(kMfma, M, 0);
    __builtin_amdgcn_sched_group_barrier(kRead, PL, 0);
  }
  __builtin_amdgcn_sched_group_barrier(kMfma, kAhead * M, 0);
}

// A chunk for the queries (bits of `redo`) that see a value row (fp32: also a key row) that is not
// finite, as float32 arithmetic row by row has it: an infinity stays in its channel, a score of
// -infinity is a weight of 0. The pieces of such a row would give NaN in every channel, or miss the
// row where its weight is small. Each wavefront takes its 16 query tokens, 4 at a time, lanes over the
// dims; `put` gets (query token, head of the pair, reference, sum, this lane's dims lane + 64 i).
template <typename E, int D, typename Put>
__device__ __forceinline__ void plain_chunk(const PrefillArgs& a, const Work& u, int kvh, int g0,
                                            const uint32_t (&redo)[kHeads], Put put) {
  const int64_t* bt = a.bt + static_cast<int64_t>(u.tab) * a.max_blocks;
  constexpr int kTok = 4, N = kTok * kHeads, W = D / kWave;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  for (int i0 = 0; i0 < 16; i0 += kTok) {
    float q[N][W], m[N], l[N], acc[N][W];
    uint32_t on = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int i = 16 * wave + i0 + j / kHeads;
      const int64_t head = kvh * a.G + min(g0 + j % kHeads, a.G - 1), tok = u.row0 + min(i, u.rows - 1);
      m[j] = -1e30f;
      l[j] = 0.f;
      bool finite = true;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const int d = lane + kWave * w;
        float v = a.q[(tok * a.Hq + head) * D + d];
        if (a.q_mult) v = __fmul_rn(v, a.q_mult[head * D + d]);
        finite &= fabsf(v) < __builtin_inff();
        q[j][w] = v * (a.scale * kLog2e);
        acc[j][w] = 0.f;
      }
      if ((redo[j % kHeads] >> (i0 + j / kHeads) & 1) && i < u.rows && g0 + j % kHeads < a.G) {
        on |= 1u << j;
        if (__ballot(!finite) != 0) l[j] = __builtin_nanf("");  // NaN whatever the cache holds
      }
    }
    uint32_t todo = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) todo |= (on >> j & 1) && l[j] == 0.f ? 1u << j : 0u;
    for (int t = u.k0; t < u.k1 && todo != 0; ++t) {
      const int block = a.bs_shift >= 0 ? t >> a.bs_shift : t / a.bs;
      const int64_t id = bt[block];
      if (id < 0 || id >= a.num_slots / a.bs) continue;
      const int64_t at = (id * a.bs + (t - block * a.bs)) * a.Hk + kvh;
      float k[W], v[W], ks = 1.f, vs = 1.f;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        k[w] = static_cast<float>(static_cast<const E*>(a.kc)[at * D + lane + kWave * w]);
        v[w] = static_cast<float>(static_cast<const E*>(a.vc)[at * D + lane + kWave * w]);
      }
      if constexpr (std::is_same_v<E, int8_t>) {
        ks = a.ks[at];
        vs = a.vs[at];
      }
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if (!(todo >> j & 1) || t >= u.sees + 16 * wave + i0 + j / kHeads) continue;
        float s = q[j][0] * k[0];
#pragma unroll
        for (int w = 1; w < W; ++w) s = __builtin_fmaf(q[j][w], k[w], s);
        s = lsh::group_sum<kWave>(s) * ks;
        const float top = fmaxf(m[j], s), f = __builtin_amdgcn_exp2f(m[j] - top);
        const float p = __builtin_amdgcn_exp2f(s - top);
        m[j] = top;
        l[j] = l[j] * f + p;
#pragma unroll
        for (int w = 0; w < W; ++w) acc[j][w] = __builtin_fmaf(p * vs, v[w], acc[j][w] * f);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (on >> j & 1) put(16 * wave + i0 + j / kHeads, j % kHeads, m[j], l[j], acc[j]);
  }
}

template <typename E, int D>
__global__ __launch_bounds__(kWaves* kWave, 2) void prefill_kernel(PrefillArgs a) {
  constexpr bool kF32 = std::is_same_v<E, float>;
  constexpr int KT = Geo<E>::KT, PL = Geo<E>::PL;
  constexpr int TT = KT / 16;   // 16-token tiles of a context tile
  constexpr int KS = D / 32;    // MFMA steps of q . k
  constexpr int DT = D / 16;    // 16-dim tiles of the output
  constexpr int VS = KT / 32;   // MFMA steps of p v
  constexpr int kKBytes = PL * TT * KS * kFrag, kVBytes = PL * DT * VS * kFrag;
  constexpr int TW = KT / kWaves;                           // context tokens a wavefront stages
  constexpr int kRow = D * static_cast<int>(sizeof(E));     // bytes of a cache row
  constexpr int kLoads = TW * kRow / kFrag;                 // 1 KB loads of a wavefront, K or V
  __shared__ __attribute__((aligned(16))) char conv[kKBytes + kVBytes];            // fp16 fragments
  __shared__ __attribute__((aligned(16))) char raw[kWaves][2][kLoads * kFrag];     // rows as cached
  __shared__ __attribute__((aligned(16))) float sk[KT], sv[KT];                    // the tokens' scales
  __shared__ uint32_t have[kWaves];                                                // bits: the tokens that exist

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int fr = lane % 16, fc = lane / 16;
  const int hp = blockIdx.x, kvh = hp / a.pairs, g0 = hp % a.pairs * kHeads;
  const Work w = work_of(a, blockIdx.y);
  const int rows = w.rows, sees = w.sees, row0 = w.row0, tab = w.tab, k0 = w.k0, k1 = w.k1;
  if (k0 >= w.ctx) return;  // whole workgroup
  const bool whole = w.size >= w.ctx;
  const int part = part_index(a, w.tile, w.chunk);
  const int n_ct = (k1 - k0 + KT - 1) / KT;

  // ---- q: this wavefront's 16 tokens, both heads, as B operands --------------------------------
  const int tok = min(16 * wave + fr, rows - 1);
  int head[kHeads];
  f16x8 qf[kHeads][KS][2];
  float qs[kHeads];  // score = dot * k_scale * qs (log2 units)
#pragma unroll
  for (int c = 0; c < kHeads; ++c) {
    head[c] = kvh * a.G + min(g0 + c, a.G - 1);
    const float* qp = a.q + (static_cast<int64_t>(row0 + tok) * a.Hq + head[c]) * D + 8 * fc;
    float v[KS][8];
    float top = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(qp + 32 * s);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(qp + 32 * s + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[s][e] = lo[e];
        v[s][4 + e] = hi[e];
      }
      if (a.q_mult) {
        const float* mp = a.q_mult + head[c] * D + 32 * s + 8 * fc;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[s][e] = __fmul_rn(v[s][e], mp[e]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(v[s][e]));
    }
    const int ex = exponent_to_15(max_over_fc(top));
    // the sign of the softmax scale goes with q, so that qs >= 0 and the scores' order is the dots'
    const float up = __builtin_copysignf(__builtin_amdgcn_ldexpf(1.f, ex), a.scale);
    qs[c] = fmaxf(__builtin_amdgcn_ldexpf(fabsf(a.scale) * kLog2e, -ex), 1e-37f);  // 0: -inf * 0 below
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t h, l;
        split2(v[s][2 * e] * up, v[s][2 * e + 1] * up, h, l);
        hi[e] = h;
        lo[e] = l;
      }
      qf[c][s][0] = __builtin_bit_cast(f16x8, hi);
      qf[c][s][1] = __builtin_bit_cast(f16x8, lo);
    }
  }

  // ---- staged v scales: times 2^up, from the first token if the tile's first row (so all) sees it --
  const int64_t* bt = a.bt + static_cast<int64_t>(tab) * a.max_blocks;
  auto block_of = [&](int t) { return a.bs_shift >= 0 ? t >> a.bs_shift : t / a.bs; };
  const int64_t blocks = a.num_slots / a.bs, rstride = static_cast<int64_t>(a.Hk) * kRow;
  int up = kTop;
  {
    const int64_t id0 = k0 < sees ? bt[block_of(k0)] : static_cast<int64_t>(-1);
    if (id0 >= 0 && id0 < blocks) {
      const int64_t slot0 = id0 * a.bs + (k0 - block_of(k0) * a.bs);
      float v0 = 0.f;
      if constexpr (kF32) {
        const float* vp = reinterpret_cast<const float*>(static_cast<const char*>(a.vc) + slot0 * rstride + kvh * kRow);
#pragma unroll
        for (int i = 0; i < D / kWave; ++i) v0 = fmaxf(v0, fabsf(vp[i * kWave + lane]));
        v0 = lsh::wave_max_from<1>(v0) * 0x1p-15f;
      } else {
        v0 = a.vs[slot0 * a.Hk + kvh];
      }
      if (v0 > 0.f && v0 < __builtin_inff())
        up = min(max(kTop - __builtin_amdgcn_frexp_expf(v0), kUpMin), kUpMax);
    }
    up = __builtin_amdgcn_readfirstlane(up);
  }
  const float v_up = __builtin_bit_cast(float, static_cast<uint32_t>(up + 127) << 23);

  // ---- staging: wavefront w brings tokens TW w .. + TW of a context tile ------------------------
  // block id of the token this lane looks after (lane % TW of the wavefront's), read a tile ahead
  auto token_of = [&](int it) { return k0 + it * KT + TW * wave + lane % TW; };
  auto fetch_id = [&](int it) {
    const int t = token_of(it);
    return t < k1 ? bt[block_of(t)] : static_cast<int64_t>(-1);
  };
  auto slot_of = [&](int it, int64_t id) {  // cache slot, -1: no such token
    const int t = token_of(it);
    return id < 0 || id >= blocks ? -1 : static_cast<int>(id) * a.bs + (t - block_of(t) * a.bs);
  };
  // starts the loads of a tile's rows (straight into LDS) and of this lane's scale
  float scale = 0.f;
  auto load = [&](int slot) {
    constexpr int kTok = kFrag / kRow;  // tokens of a load
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int s = __shfl(slot, i * kTok + lane / (kWave / kTok), kWave);
      const int64_t at = (s < 0 ? 0 : s) * rstride + kvh * kRow + lane % (kWave / kTok) * 16;
      __builtin_amdgcn_global_load_lds(static_cast<const char*>(a.kc) + at,
                                       (__attribute__((address_space(3))) void*)(raw[wave][0] + i * kFrag), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(static_cast<const char*>(a.vc) + at,
                                       (__attribute__((address_space(3))) void*)(raw[wave][1] + i * kFrag), 16, 0, 0);
    }
    if constexpr (!kF32) {  // lanes 0 .. TW - 1 K scales, the next TW V scales
      const float* const k_scales = a.ks;  // (a choice between the members would load the pointer per lane)
      const float* const v_scales = a.vs;
      const float* p = lane < TW ? k_scales : v_scales;
      scale = slot >= 0 ? p[static_cast<int64_t>(slot) * a.Hk + kvh] : 0.f;
    }
  };
  // V: 4 tokens x VD dims per thread, transposed into [dim][token] on the way
  constexpr int VD = kF32 ? 4 : D / 16;
  constexpr int kVLanes = D / VD;
  const bool v_on = TW / 4 * kVLanes == kWave || lane < TW / 4 * kVLanes;
  const int vd0 = lane % kVLanes * VD, vl0 = lane / kVLanes % (TW / 4) * 4;  // dims, token of the wavefront's
  const int vg = TW / 4 * wave + vl0 / 4;                                    // group of 4 tokens in the tile
  // chunk c (8 dims) of token t: fragment (t / 16, c / 4), lane position t % 16 moved by `swz` so
  // that the writes of a row's lanes fall into different banks
  auto swz = [](int c) { return kF32 ? c & 7 : (c >> 1) * (128 / D); };
  auto k_at = [&](char* base, int pl, int t, int c) {
    return base + ((pl * TT + t / 16) * KS + c / 4) * kFrag + (((t % 16) ^ swz(c)) + 16 * (c % 4)) * 16;
  };
  // dim d, tokens 4 g .. + 3: fragment (d / 16, token / 32), lane d % 16 + 16 (g % 4), its first or
  // second four elements for the even or odd 16-token tile
  auto v_at = [&](char* base, int pl, int d, int g) {
    return base + kKBytes + ((pl * DT + d / 16) * VS + g / 8) * kFrag +
           (((d % 16) ^ (d / 16 % 8)) + 16 * (g % 4)) * 16 + g / 4 % 2 * 8;
  };
  // this wavefront's landed rows -> fragments; `slot` as for their load
  auto convert = [&](int slot) {
    const uint64_t ok = __ballot(slot >= 0);
    if (lane == 0) have[wave] = static_cast<uint32_t>(ok) & ((1u << TW) - 1);
    if constexpr (!kF32) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int j = i * kWave + lane, t = TW * wave + j * 16 / kRow, c = j * 16 % kRow / 8;
        const u32x4 r = *reinterpret_cast<const u32x4*>(raw[wave][0] + j * 16);
        u32x4 lo, hi;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const uint32_t x = r[w] ^ 0x80808080u, y = r[2 + w] ^ 0x80808080u;
          lo[2 * w] = bytes_to_h2<0x04010400u>(x);
          lo[2 * w + 1] = bytes_to_h2<0x04030402u>(x);
          hi[2 * w] = bytes_to_h2<0x04010400u>(y);
          hi[2 * w + 1] = bytes_to_h2<0x04030402u>(y);
        }
        *reinterpret_cast<u32x4*>(k_at(conv, 0, t, c)) = lo;
        *reinterpret_cast<u32x4*>(k_at(conv, 0, t, c + 1)) = hi;
      }
#pragma unroll
      for (int w = 0; w < VD / 4; ++w) {
        uint32_t x[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
          x[t] = *reinterpret_cast<const uint32_t*>(raw[wave][1] + (vl0 + t) * kRow + vd0 + 4 * w) ^ 0x80808080u;
        // bytes of tokens (0, 1) and (2, 3) side by side: [a0 b0 a1 b1], [a2 b2 a3 b3]
        const uint32_t p01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u), p23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
        const uint32_t q01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u), q23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
        const int d = vd0 + 4 * w;
        *reinterpret_cast<u32x2*>(v_at(conv, 0, d, vg)) = u32x2{bytes_to_h2<0x04010400u>(p01), bytes_to_h2<0x04010400u>(p23)};
        *reinterpret_cast<u32x2*>(v_at(conv, 0, d + 1, vg)) = u32x2{bytes_to_h2<0x04030402u>(p01), bytes_to_h2<0x04030402u>(p23)};
        *reinterpret_cast<u32x2*>(v_at(conv, 0, d + 2, vg)) = u32x2{bytes_to_h2<0x04010400u>(q01), bytes_to_h2<0x04010400u>(q23)};
        *reinterpret_cast<u32x2*>(v_at(conv, 0, d + 3, vg)) = u32x2{bytes_to_h2<0x04030402u>(q01), bytes_to_h2<0x04030402u>(q23)};
      }
      if (lane < TW) sk[TW * wave + lane] = scale;
      if (lane >= TW && lane < 2 * TW) sv[TW * wave + lane - TW] = fminf(scale * v_up, kHuge);
    } else {
      // a row's exponent, from the largest magnitude as an integer (NaN and infinity above all)
      auto row_scale = [&](uint32_t top, int lanes, float& up) {
        for (int m = 1; m < lanes; m <<= 1) {
          const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), m, kWave));
          top = top > o ? top : o;
        }
        const int ex = exponent_to_15(__builtin_bit_cast(float, top));
        const bool bad = top >= 0x7f800000u;  // the row reads as zeros, its scale as not finite
        up = bad ? 0.f : __builtin_amdgcn_ldexpf(1.f, ex);
        return bad ? __builtin_nanf("") : __builtin_amdgcn_ldexpf(1.f, -ex);
      };
      auto mag = [](const u32x4& w) {
        uint32_t t = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t b = w[e] & 0x7fffffffu;
          t = t > b ? t : b;
        }
        return t;
      };
      auto value = [](const u32x4& w, int e, float up) {
        const uint32_t u = w[e];
        return up == 0.f ? 0.f : __builtin_bit_cast(float, u) * up;
      };
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int j = i * kWave + lane, tl = j * 16 / kRow, t = TW * wave + tl, p = j * 16 % kRow / 16;
        const u32x4 r = *reinterpret_cast<const u32x4*>(raw[wave][0] + j * 16);
        float up;
        const float down = row_scale(mag(r), kRow / 16, up);
        uint32_t h0, l0, h1, l1;
        split2(value(r, 0, up), value(r, 1, up), h0, l0);
        split2(value(r, 2, up), value(r, 3, up), h1, l1);
        *reinterpret_cast<u32x2*>(k_at(conv, 0, t, p / 2) + p % 2 * 8) = u32x2{h0, h1};
        *reinterpret_cast<u32x2*>(k_at(conv, 1, t, p / 2) + p % 2 * 8) = u32x2{l0, l1};
        if (p == 0) sk[t] = ok >> tl & 1 ? down : 0.f;
      }
      u32x4 r[4];
      float up[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        r[t] = *reinterpret_cast<const u32x4*>(raw[wave][1] + (vl0 + t) * kRow + vd0 * 4);
        const float down = row_scale(mag(r[t]), kVLanes, up[t]);
        if (v_on && vd0 == 0) sv[4 * vg + t] = ok >> (vl0 + t) & 1 ? fminf(down * v_up, kHuge) : 0.f;
      }
      if (v_on) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t h0, l0, h1, l1;
          split2(value(r[0], e, up[0]), value(r[1], e, up[1]), h0, l0);
          split2(value(r[2], e, up[2]), value(r[3], e, up[3]), h1, l1);
          *reinterpret_cast<u32x2*>(v_at(conv, 0, vd0 + e, vg)) = u32x2{h0, h1};
          *reinterpret_cast<u32x2*>(v_at(conv, 1, vd0 + e, vg)) = u32x2{l0, l1};
        }
      }
    }
  };

  // ---- the context ------------------------------------------------------------------------------
  f32x4 acc[kHeads][DT];
  float ref[kHeads], sum[kHeads];
#pragma unroll
  for (int c = 0; c < kHeads; ++c) {
    ref[c] = -1e30f;
    sum[c] = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[c][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int limit = sees + tok;  // tokens this lane's query sees
  uint64_t huge = 0;             // lanes that see a v scale staged as kHuge

  int slot = slot_of(0, fetch_id(0));
  load(slot);
  int64_t id = fetch_id(1);
  for (int it = 0; it < n_ct; ++it) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's rows have landed
    if (it) __syncthreads();             // everyone has read the last tile's fragments
    convert(slot);
    if (it + 1 < n_ct) {  // the rows are read (their values are in use): the next ones may land
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      slot = slot_of(it + 1, id);
      load(slot);
      id = fetch_id(it + 2);
    }
    __syncthreads();
    const char* base = conv;
    __builtin_amdgcn_s_setprio(1);
    f32x4 s[kHeads][TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      // Two sums per score, added at the end: the first half of the hi products in one, the rest, with
      // the small products of lo pieces, in the other. One chain would round at the score's size three
      // times as often; more than two change nothing. lo lo products are small but not nothing:
      // float64 error over the fp32 cache 1.61e-7 without them, 1.57e-7 with.
      f32x4 part[kHeads][2] = {};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int c = 4 * ks + fc, half = 2 * ks / KS;
        const char* p = base + (tt * KS + ks) * kFrag + ((fr ^ swz(c)) + 16 * fc) * 16;
        f16x8 kf[PL];
#pragma unroll
        for (int pl = 0; pl < PL; ++pl)
          kf[pl] = *reinterpret_cast<const f16x8*>(p + pl * TT * KS * kFrag);
#pragma unroll
        for (int c2 = 0; c2 < kHeads; ++c2) part[c2][1] = mfma(kf[0], qf[c2][ks][1], part[c2][1]);
        if constexpr (PL == 2) {
#pragma unroll
          for (int c2 = 0; c2 < kHeads; ++c2) part[c2][1] = mfma(kf[1], qf[c2][ks][0], part[c2][1]);
#pragma unroll
          for (int c2 = 0; c2 < kHeads; ++c2) part[c2][1] = mfma(kf[1], qf[c2][ks][1], part[c2][1]);
        }
#pragma unroll
        for (int c2 = 0; c2 < kHeads; ++c2) part[c2][half] = mfma(kf[0], qf[c2][ks][0], part[c2][half]);
      }
#pragma unroll
      for (int c2 = 0; c2 < kHeads; ++c2) s[c2][tt] = part[c2][0] + part[c2][1];
    }
    read_ahead<TT * KS, PL, kHeads * (PL == 2 ? 4 : 2)>();
    __builtin_amdgcn_s_setprio(0);
    // scores (times qs: log2 units); lane (fr, fc) holds tokens 16 tt + 4 fc + e of its query
    float vtop = 0.f;  // the largest v scale
    const int t0 = k0 + it * KT;
    uint64_t there = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) there |= static_cast<uint64_t>(have[w]) << (TW * w);
    const bool hole = t0 + KT > sees + min(16 * wave, rows - 1) ||  // some lane's query ends in this tile
                      there != (KT == 64 ? ~0ull : (1ull << KT) - 1);
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const f32x4 kk = *reinterpret_cast<const f32x4*>(&sk[16 * tt + 4 * fc]);
      const f32x4 vv = *reinterpret_cast<const f32x4*>(&sv[16 * tt + 4 * fc]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vtop = fmaxf(vtop, vv[e]);
#pragma unroll
        for (int c = 0; c < kHeads; ++c) s[c][tt][e] *= kk[e];
      }
    }
    if (hole) {  // (the largest v scale, too, of the tokens this lane's query sees)
      vtop = 0.f;
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const f32x4 vv = *reinterpret_cast<const f32x4*>(&sv[16 * tt + 4 * fc]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 4 * fc + e;
          const bool in = t0 + 16 * tt + t < limit && (static_cast<uint32_t>(there >> (16 * tt)) >> t & 1);
          vtop = fmaxf(vtop, in ? vv[e] : 0.f);
#pragma unroll
          for (int c = 0; c < kHeads; ++c) s[c][tt][e] = in ? s[c][tt][e] : -__builtin_inff();
        }
      }
    }
    huge |= __ballot(vtop >= kHuge);
    const float lv = fminf(fmaxf(__builtin_amdgcn_logf(max_over_fc(vtop)) - kTop, -kMaxLv), kMaxLv);
    float top[kHeads];
    bool raise = false;
#pragma unroll
    for (int c = 0; c < kHeads; ++c) {
      top[c] = s[c][0][0];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int e = 0; e < 4; ++e) top[c] = fmaxf(top[c], s[c][tt][e]);
      top[c] *= qs[c];
      raise |= top[c] + lv > ref[c] + kLazy;
    }
    if (__ballot(raise) != 0) {
#pragma unroll
      for (int c = 0; c < kHeads; ++c) {
        const float want = max_over_fc(top[c]) + lv;
        const float now = want > ref[c] + kLazy ? want : ref[c];
        const float f = __builtin_amdgcn_exp2f(ref[c] - now);
        ref[c] = now;
        sum[c] *= f;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[c][d][e] *= f;
      }
    }
    // weights and their product with V
    f16x8 ph[VS][kHeads], pl[VS][kHeads];
#pragma unroll
    for (int vs = 0; vs < VS; ++vs) {
      f32x4 vsc[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        vsc[h] = *reinterpret_cast<const f32x4*>(&sv[16 * (2 * vs + h) + 4 * fc]);
#pragma unroll
      for (int c = 0; c < kHeads; ++c) {
        u32x4 hi, lo;
        float eight = 0.f;  // added up apart: an eighth of the roundings at the sum's size
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float w[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c][2 * vs + h][e], qs[c], -ref[c]));
            eight += p;
            w[e] = p * vsc[h][e];
          }
          uint32_t h0, l0, h1, l1;
          split2(w[0], w[1], h0, l0);
          split2(w[2], w[3], h1, l1);
          hi[2 * h] = h0;
          hi[2 * h + 1] = h1;
          lo[2 * h] = l0;
          lo[2 * h + 1] = l1;
        }
        sum[c] += eight;
        ph[vs][c] = __builtin_bit_cast(f16x8, hi);
        pl[vs][c] = __builtin_bit_cast(f16x8, lo);
      }
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      f16x8 vf[VS][PL];
#pragma unroll
      for (int vs = 0; vs < VS; ++vs)
#pragma unroll
        for (int q = 0; q < PL; ++q)
          vf[vs][q] = *reinterpret_cast<const f16x8*>(base + kKBytes + (d * VS + vs) * kFrag +
                                                      ((fr ^ (d % 8)) + 16 * fc) * 16 + q * DT * VS * kFrag);
      // The tile's sum apart, its small products first: one rounding at acc's size (summed into acc product
      // by product, int8, the error against float64 was 1.2e-6 for 2048 tokens after 30000, now 3.6e-7;
      // for 2048 2.0e-7, now 1.4e-7; row kernel 5.3e-7 and 1.9e-7; at the same speed).
      f32x4 t[kHeads] = {};
#pragma unroll
      for (int vs = 0; vs < VS; ++vs) {
        if constexpr (PL == 2) {
#pragma unroll
          for (int c = 0; c < kHeads; ++c) t[c] = mfma(vf[vs][PL - 1], ph[vs][c], t[c]);
        }
#pragma unroll
        for (int c = 0; c < kHeads; ++c) t[c] = mfma(vf[vs][0], pl[vs][c], t[c]);
      }
#pragma unroll
      for (int vs = 0; vs < VS; ++vs)
#pragma unroll
        for (int c = 0; c < kHeads; ++c) t[c] = mfma(vf[vs][0], ph[vs][c], t[c]);
#pragma unroll
      for (int c = 0; c < kHeads; ++c) acc[c][d] += t[c];
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // ---- output: lane (fr, fc) holds dims 16 d + 4 fc + e of its query -----------------------------
  // The arguments, read again (and the work, where it is needed once more): held since the start, they
  // would be spilled around the loop.
  typedef const __attribute__((address_space(4))) PrefillArgs* ArgsPtr;
  ArgsPtr args = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  int unit = blockIdx.y, pair = blockIdx.x;
  asm("" : "+s"(args), "+s"(unit), "+s"(pair));
  const PrefillArgs& b = *(const PrefillArgs*)args;
  const int kv = pair / b.pairs, g = pair % b.pairs * kHeads;
  auto part_at = [&](int tok, int c) {
    return ((static_cast<int64_t>(part) * b.Hk * b.pairs + pair) * kHeads + c) * kQT + tok;
  };
  huge |= huge >> 32;
  huge |= huge >> 16;
  uint32_t redo[kHeads];  // bits: this wavefront's query tokens
#pragma unroll
  for (int c = 0; c < kHeads; ++c) {
    const float l = sum_over_fc(sum[c]);
    redo[c] = static_cast<uint32_t>(huge | __ballot(l != l)) & 0xffffu;
    if (16 * wave + fr >= rows || (redo[c] >> fr & 1) || g + c >= b.G) continue;
    if (whole) {
      const float inv = 1.f / (l * v_up);
      float* o = b.out + (static_cast<int64_t>(row0 + 16 * wave + fr) * b.Hq + kv * b.G + g + c) * D + 4 * fc;
#pragma unroll
      for (int d = 0; d < DT; ++d)
        *reinterpret_cast<f32x4*>(o + 16 * d) = acc[c][d] * inv;
    } else {
      const int64_t at = part_at(16 * wave + fr, c);
      float* o = b.part_acc + at * D + 4 * fc;
#pragma unroll
      for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(o + 16 * d) = acc[c][d] * (1.f / v_up);
      if (fc == 0) {
        b.part_rl[2 * at] = ref[c];  // as the weights used it: any sum with it would round
        b.part_rl[2 * at + 1] = l;
      }
    }
  }
  if (redo[0] | redo[1]) {
    plain_chunk<E, D>(b, work_of(b, unit), kv, g, redo,
                      [&](int t, int c, float m, float l, const float (&v)[D / kWave]) {
                        const int64_t at = part_at(t, c);
                        float* o = b.out + (static_cast<int64_t>(row0 + t) * b.Hq + kv * b.G + g + c) * D;
#pragma unroll
                        for (int i = 0; i < D / kWave; ++i) {
                          if (whole)
                            o[lane + kWave * i] = v[i] / l;
                          else
                            b.part_acc[at * D + lane + kWave * i] = v[i];
                        }
                        if (!whole && lane == 0) {
                          b.part_rl[2 * at] = m;
                          b.part_rl[2 * at + 1] = l;
                        }
                      });
  }
}

// Adds the chunks of the tiles that have several: D / 4 lanes per (query token, head).
//   R = max_j r_j;  out = sum_j 2^(r_j - R) acc_j / sum_j 2^(r_j - R) l_j   (l_j = 0 skipped)
// Bound by one round trip to memory: four chunks' references, sums and rows are loaded together
// (one chunk after another the kernel took 34 us for 30 tiles of up to 8 chunks, this way 17).
template <int D>
__global__ __launch_bounds__(kWaves* kWave) void prefill_merge_kernel(PrefillArgs a) {
  constexpr int LPR = D / 4, kBatch = 4;
  const int tile = blockIdx.y, part = threadIdx.x % LPR;
  const int rows = static_cast<int>(a.tiles[4 * tile + 1]);
  const int ctx = static_cast<int>(a.tiles[4 * tile + 2]) + rows - 1, size = chunk_size(ctx, a.chunk);
  const int n = (ctx + size - 1) / size;
  const int i = blockIdx.x * (kWaves * kWave / LPR) + threadIdx.x / LPR, tok = i / a.Hq, h = i % a.Hq;
  if (n <= 1 || tok >= rows) return;
  const int kvh = h / a.G, g = h % a.G, hp = kvh * a.pairs + g / kHeads, c = g % kHeads;
  float R = -1e30f, L = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < n; j0 += kBatch) {
    float r[kBatch], l[kBatch];
    f32x4 v[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int64_t at =
          ((static_cast<int64_t>(part_index(a, tile, min(j0 + j, n - 1))) * a.Hk * a.pairs + hp) * kHeads + c) * kQT + tok;
      r[j] = a.part_rl[2 * at];
      l[j] = a.part_rl[2 * at + 1];
      v[j] = *reinterpret_cast<const f32x4*>(a.part_acc + at * D + 4 * part);
    }
    float top = R;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) top = fmaxf(top, r[j]);
    const float f = __builtin_amdgcn_exp2f(R - top);
    R = top;
    L *= f;
    o *= f;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const bool on = j0 + j < n && l[j] != 0.f;
      const float w = on ? __builtin_amdgcn_exp2f(r[j] - R) : 0.f;
      L += w * l[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += w * (on ? v[j][e] : 0.f);
    }
  }
  const float inv = 1.f / L;
  *reinterpret_cast<f32x4*>(a.out + (a.tiles[4 * tile] + tok) * a.Hq * D + static_cast<int64_t>(h) * D + 4 * part) =
      o * inv;
}

struct ChunkPlan {
  int chunk, splits, whole;  // as in PrefillArgs
  int64_t units, parts;      // chunks in all, and of the split tiles
  int start[kMaxSplits + 1];
};

// Context tiles (of 64 tokens) of a query tile.
int context_tiles(const int64_t* t) { return static_cast<int>((t[1] + t[2] - 1 + 63) / 64); }

// Chunks of at most `most` context tiles: where they begin in the launch and in the workspace.
// `sorted`: the longest contexts first, so that the tiles with more than z chunks are the first ones.
ChunkPlan lay_out(const int64_t* tiles, int64_t n, int most, int longest, bool sorted) {
  ChunkPlan p{};
  p.chunk = most * 64;
  p.splits = (longest + most - 1) / most;
  int64_t count[kMaxSplits + 1] = {};  // tiles with exactly so many chunks
  for (int64_t i = 0; i < n; ++i) ++count[(context_tiles(tiles + 4 * i) + most - 1) / most];
  int64_t more = n;  // tiles with more than z chunks (not sorted: all, some of them idle)
  for (int z = 0; z < p.splits; ++z) {
    if (sorted) more -= count[z];
    p.start[z] = static_cast<int>(p.units);
    p.units += more;
    if (z == 1) p.whole = static_cast<int>(n - more);
  }
  if (p.splits == 1) p.whole = static_cast<int>(n);
  for (int z = p.splits; z <= kMaxSplits; ++z) p.start[z] = static_cast<int>(p.units);
  p.parts = p.units - p.whole;
  return p;
}

// The chunk size by an estimate in microseconds: a workgroup takes 7 to start and end, 4.26 per context
// tile beside another workgroup on its CU and 3.2 alone; up to two per CU the launch takes its longest
// chunk, above that its work over all places and, where chunks are even, a third of a chunk until the
// last ones end; the merge takes 6 and the partials' bytes at 8 TB/s. Over 51 batches (64 to 16384 new tokens, up
// to 100k cached, 8 to 32 heads, both caches; these are the int8 cache's rates at 128 dims, the others scale
// about alike) the choice is on average 1.7 % and at most 11 % slower than the best of ~20 sizes. 16 / 8 heads,
// int8, us:
//   2048 new: 68 in chunks of 704 tokens (256: 87, whole: 118); after 2000 cached 159 in 2048 (896: 145, 256: 213,
//   whole: 222); after 30000 1081 (8064: 1051, 256: 2011, whole: 1788); 8192 new 566 whole (4096: 589, 256: 1039).
// Partials take at most kMaxParts bytes, whatever the context.
constexpr int64_t kMaxParts = 128LL << 20;
constexpr double kEnds = 7.0, kTile = 4.26, kTileAlone = 3.2, kMerge = 6.0, kBytes = 8e6, kTail = 0.35;

int64_t part_bytes(int64_t parts, int64_t groups, int64_t D) { return parts * groups * kHeads * kQT * (D + 2) * 4; }

ChunkPlan plan_chunks(const int64_t* tiles, int64_t n, int64_t groups, int64_t D) {
  int64_t total = 0;
  int longest = 1, before = INT32_MAX;
  bool sorted = true;
  for (int64_t i = 0; i < n; ++i) {
    const int t = context_tiles(tiles + 4 * i);
    total += t;
    longest = std::max(longest, t);
    sorted = sorted && t <= before;
    before = t;
  }
  const double places = 2.0 * lsh::device_cus();
  double best = 0;
  int take = longest;
  for (int most = longest; most * kMaxSplits >= longest && most > 0; most -= 1 + most / 12) {
    const bool split = most < longest;
    int64_t chunks = n, parts = 0;
    int len = longest;  // of the longest chunk
    if (split) {
      chunks = 0;
      len = 1;
      for (int64_t i = 0; i < n; ++i) {
        const int t = context_tiles(tiles + 4 * i), k = (t + most - 1) / most;
        chunks += k;
        parts += k > 1 ? k : 0;
        len = std::max(len, (t + k - 1) / k);
      }
      if (!sorted) chunks = parts = n * ((longest + most - 1) / most);
      if (chunks >= 65536 || part_bytes(parts, groups, D) > kMaxParts) continue;
    }
    const double units = static_cast<double>(chunks * groups), longest_one = kEnds + kTile * len;
    double us = 2 * units <= places ? kEnds + kTileAlone * len : longest_one;
    if (units > places)
      us = std::max(longest_one, (units * kEnds + static_cast<double>(total * groups) * kTile) / places +
                                     (split ? kTail * longest_one : 0.0));
    if (split) us += kMerge + static_cast<double>(part_bytes(parts, groups, D)) / kBytes;
    if (!split || us < best) {
      best = us;
      take = most;
    }
    if (us > 1.5 * best) break;  // smaller chunks only add to this
  }
  return lay_out(tiles, n, take, longest, sorted);
}

int64_t head_pairs(int64_t Hq, int64_t Hk) { return Hk * ((Hq / Hk + kHeads - 1) / kHeads); }

}  // namespace

extern "C" int64_t llmserve_paged_attention_prefill_workspace_bytes(const int64_t* tiles_host, int64_t n_tiles,
                                                                    int64_t Hq, int64_t Hk, int64_t D) {
  if (n_tiles <= 0 || Hq <= 0 || Hk <= 0 || Hq % Hk || tiles_host == nullptr) return 0;
  const int64_t groups = head_pairs(Hq, Hk);
  return part_bytes(plan_chunks(tiles_host, n_tiles, groups, D).parts, groups, D);
}

extern "C" int llmserve_paged_attention_prefill(const float* q, const void* k_cache, const void* v_cache,
                                                const float* k_scale, const float* v_scale,
                                                const int64_t* block_tables, int64_t table_rows,
                                                const int64_t* tiles, const int64_t* tiles_host, int64_t n_tiles,
                                                float* out, int64_t T, int64_t Hq, int64_t Hk, int64_t D,
                                                int64_t num_slots, int64_t max_blocks, int64_t block_size,
                                                float scale, const float* q_mult, void* workspace,
                                                int64_t workspace_bytes, void* stream) {
  LSH_CHECK(T >= 0 && Hq >= 1 && Hk >= 1 && Hq % Hk == 0 && n_tiles >= 0, "paged_attention_prefill: bad shape");
  LSH_CHECK(D == 64 || D == 128, "paged_attention_prefill: head_dim %lld not 64 or 128", (long long)D);
  if (n_tiles == 0) return LLMSERVE_OK;
  LSH_CHECK(block_size >= 1 && max_blocks >= 1 && num_slots >= block_size && table_rows >= 1,
            "paged_attention_prefill: empty block table or cache");
  LSH_CHECK(max_blocks * block_size < (1LL << 30) && num_slots * Hk < (1LL << 31) && T < (1LL << 24) && Hk <= 4096 &&
                Hq <= 32768 && n_tiles < 65536,
            "paged_attention_prefill: batch, context or cache too large");
  LSH_CHECK(q && k_cache && v_cache && block_tables && tiles && tiles_host && out && (!k_scale == !v_scale),
            "paged_attention_prefill: null pointer");
  LSH_CHECK(lsh::aligned16(q) && lsh::aligned16(k_cache) && lsh::aligned16(v_cache) && lsh::aligned16(out),
            "paged_attention_prefill: q, caches and out must be 16-byte aligned");
  for (int64_t i = 0; i < n_tiles; ++i) {
    const int64_t* t = tiles_host + 4 * i;
    LSH_CHECK(t[0] >= 0 && t[1] >= 1 && t[1] <= kQT && t[0] + t[1] <= T && t[2] >= 1 &&
                  t[2] + t[1] - 1 <= max_blocks * block_size && t[3] >= 0 && t[3] < table_rows,
              "paged_attention_prefill: tile %lld outside the batch or its block table", (long long)i);
  }
  PrefillArgs a{};
  a.G = static_cast<int>(Hq / Hk);
  a.pairs = (a.G + kHeads - 1) / kHeads;
  const int64_t groups = Hk * a.pairs;
  const ChunkPlan plan = plan_chunks(tiles_host, n_tiles, groups, D);
  const int64_t need = part_bytes(plan.parts, groups, D);
  LSH_CHECK(need == 0 || (workspace != nullptr && workspace_bytes >= need && lsh::aligned16(workspace)),
            "paged_attention_prefill: a 16-byte aligned workspace of %lld bytes is needed (%lld given)",
            (long long)need, (long long)workspace_bytes);
  a.q = q;
  a.kc = k_cache;
  a.vc = v_cache;
  a.ks = k_scale;
  a.vs = v_scale;
  a.bt = block_tables;
  a.tiles = tiles;
  a.q_mult = q_mult;
  a.out = out;
  a.part_acc = static_cast<float*>(workspace);
  a.part_rl = a.part_acc + need / 4 / (D + 2) * D;
  a.num_slots = num_slots;
  a.Hq = static_cast<int>(Hq);
  a.Hk = static_cast<int>(Hk);
  a.max_blocks = static_cast<int>(max_blocks);
  a.bs = static_cast<int>(block_size);
  a.bs_shift = -1;
  for (int sh = 0; sh < 30; ++sh)
    if ((1LL << sh) == block_size) a.bs_shift = sh;
  a.chunk = plan.chunk;
  a.splits = plan.splits;
  a.whole = plan.whole;
  std::copy(plan.start, plan.start + kMaxSplits + 1, a.start);
  a.scale = scale;
  hipStream_t st = lsh::as_stream(stream);
  const dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(plan.units));
  const dim3 block(kWaves * kWave);
  const bool once = plan.splits == 1;
  if (k_scale != nullptr && D == 128)
    lsh::launch(prefill_kernel<int8_t, 128>, grid, block, 0, st, once, a);
  else if (k_scale != nullptr)
    lsh::launch(prefill_kernel<int8_t, 64>, grid, block, 0, st, once, a);
  else if (D == 128)
    lsh::launch(prefill_kernel<float, 128>, grid, block, 0, st, once, a);
  else
    lsh::launch(prefill_kernel<float, 64>, grid, block, 0, st, once, a);
  if (!once) {
    const dim3 mgrid(static_cast<unsigned>((kQT * Hq * (D / 4) + 255) / 256), static_cast<unsigned>(n_tiles));
    if (D == 128)
      lsh::launch(prefill_merge_kernel<128>, mgrid, block, 0, st, true, a);
    else
      lsh::launch(prefill_merge_kernel<64>, mgrid, block, 0, st, true, a);
  }
  return lsh::launch_status("paged_attention_prefill");
}
