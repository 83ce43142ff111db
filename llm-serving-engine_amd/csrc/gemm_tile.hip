// Weight-only linears for batches past the decode sizes, on the fp16 matrix cores:
//   int4:  y[m, n] = sum_g s[n, g] sum_{k in g} x'[m, k] q[n, k] + (z - 8 s)[n, g] sum_{k in g} x'[m, k]
//          with x' = x * inv_act_scale (Int4Linear.forward's large-M branch, reference
//          quant.py:141-142, in the group decomposition of int8_gemv.cpp:48-52).
//   int8:  y[m, n] = scale[n] sum_k bf16(x[m, k]) q[n, k], llmserve_int8_linear_prefill's product
//          (gemm_prefill.hip says for which sizes it comes here).
// Operands: q is exact in fp16. Each row of x' is scaled by the power of two that brings its
// largest value to [2^14, 2^15) and split into two fp16 pieces, hi = fp16(x'), lo = fp16(x' - hi):
// 22 significant bits, down to 2^-38 of the row's largest value (int8: bf16(x) is one piece, exact
// down to 2^-31 of it). Products are exact in fp32 and summed there. Measured against float64: 2.7-3.3e-7
// relative (the two bfloat16 pieces of int4_gemm_mfma 5.3e-6, dequantize + fp32 GEMM 8e-7).
//
// Two launches. The split pass (one wavefront per row) writes the pieces as MFMA fragments, the
// sums of x' over each unit of constant group scale, and the constants z - 8 s; for a weight in
// the reference layout it also packs the nibbles, so that the GEMM's weight loads are whole
// kilobytes: read from [N, K / 2], a load instruction touches 16 rows in 64 pieces, and the L1
// answers such loads at 9.4 TB/s over the GPU against 33 TB/s for contiguous ones. The zero
// term sum_g (z - 8 s) sum x' is a product of its own over the units (K / 128 or K / 64 long,
// again two pieces per operand), so the inner loop only does acc += s d.
//
// The GEMM: a wavefront owns TM x 4 tiles of 16 x 16; a workgroup's four wavefronts take WN
// slabs of 64 channels and split the K blocks 4 / WN ways. A stage is 128 channels of K per
// wavefront: x fragments come straight from global memory into LDS (every wavefront of a row
// reads them), the weights into registers, both one stage (weights up to two) ahead, and a
// stage waits once. Two workgroups per CU run out of step, so that one's MFMAs cover the other's
// widening and waits. Measured with parts left out at 2048 x 8192 x 8192: 360 us for the products
// and widening alone (1.5 PFLOP/s of fp16), 558 with the loads.
#include <algorithm>
#include <type_traits>

#include "gemm_tile.h"

namespace {

using lsh::kWave;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlk = 128;      // channels of a K block: four MFMA steps of 32
constexpr int kFrag = 1024;    // bytes of one A fragment: 64 lanes x 8 fp16
constexpr int kWaves = 4;      // wavefronts of a workgroup
constexpr int kSplitRows = 4;  // rows per workgroup of the split pass (one per wavefront)
constexpr int kPadRows = 128;  // activation rows are padded to the tallest tile

// How a lane's 8 channels of step q (lane = fr + 16 fc: row fr, part fc) map to the block's 128
// channels, and in which order. The k order of a product is free as long as both operands
// share it; each order is the one the weight's bytes fall into.
enum Order {
  kInt4G128,  // channels 32 fc + 8 q .. + 8 as [0,4,1,5,2,6,3,7]: 16 nibble bytes per lane and block
  kInt4G64,   // channels 64 (q / 2) + 16 fc + 8 (q % 2) .. + 8, same order: steps 0-1 and 2-3
              // each stay inside one 64-channel group
  kInt8,      // channels as kInt4G64 in index order: 16 bytes per lane and 64 channels
};

constexpr int pieces(Order o) { return o == kInt8 ? 1 : 2; }
// channels of a unit: the pieces of K whose sums and scales are constant
constexpr int unit(Order o) { return o == kInt4G64 ? 64 : 128; }

__host__ __device__ inline int64_t pad_rows(int64_t M) { return (M + kPadRows - 1) / kPadRows * kPadRows; }
__host__ __device__ inline int64_t k_blocks(int64_t K) { return (K + kBlk - 1) / kBlk; }
// K blocks in whole pairs of stages of wk blocks
inline int64_t pad_blocks(int64_t K, int wk) { return (k_blocks(K) + 2 * wk - 1) / (2 * wk) * (2 * wk); }
__host__ __device__ inline int64_t sum_steps(int64_t units) { return (units + 31) / 32; }

// The workspace of a call.
struct SplitOut {
  float* rscale;   // [mp] 2^-e of each row; negative: the split pass has written the row of y
  _Float16* xf;    // [row tile][block][q][piece][lane][8]
  // int4:
  _Float16* xs;    // [row tile][step of 32 units][hi, lo][lane][8]: unit sums of x' 2^e, scaled by 2^-8
  _Float16* zf;    // [channel tile][step][hi, lo][lane][8]: z - 8 s, scaled by 2^f of its channel
  float* zdown;    // [channel] 2^(8 - f)
  uint8_t* w;      // the packed weight, where the call brings none
  float* s;        // ... and its constants
};

inline int64_t sum_bytes(int64_t rows, int64_t K) { return rows * sum_steps((K + 63) / 64) * 32 * 2 * 2; }
__host__ __device__ inline int64_t slabs_of(int64_t N) { return (N + 63) / 64; }
inline int64_t weight_bytes(int64_t N, int64_t K) { return slabs_of(N) * 64 * K / 2; }
inline int64_t const_bytes(int64_t N, int64_t G) { return G * slabs_of(N) * 16 * 8 * 4; }

__device__ __forceinline__ f16x2 as_h2(uint32_t w) { return __builtin_bit_cast(f16x2, w); }
__device__ __forceinline__ uint32_t as_u(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }

__device__ __forceinline__ int exponent_to_15(float top) {  // 2^result brings top to [2^14, 2^15)
  int ex = 0;
  if (top > 0.f && top < __builtin_inff()) ex = 15 - __builtin_amdgcn_frexp_expf(top);
  if (top == __builtin_inff()) ex = -113;  // the largest finite value then stays finite in fp16
  return ex < -126 ? -126 : (ex > 126 ? 126 : ex);
}

// What the split pass reads of an int4 weight: packed (llmserve_int4_gemm_pack's buffer), or
// the reference layout, which it then packs into the workspace.
struct WeightIn {
  const uint8_t* nib;   // [N, K / 2]
  const float* gs;      // [N, G]
  const float* gz;      // [N, G]
  const float* packed;  // constants of a packed weight, or nullptr
  int N, group;
};

// The zero-term constants z - 8 s of one 16-channel tile as the B operand of a product (and
// the tile's constants in packed form, where the weight comes in the reference layout).
template <Order O>
__device__ __forceinline__ void zero_frags(const SplitOut& o, const WeightIn& in, int tile, int K) {
  const int lane = threadIdx.x % kWave, fr = lane % 16, fc = lane / 16;
  const int units = K / unit(O), steps = static_cast<int>(sum_steps(units));
  const unsigned per = static_cast<unsigned>(in.group / unit(O));  // units of a group
  const int G = K / in.group, n = 16 * tile + fr;
  const int64_t row = static_cast<int64_t>(n < in.N ? n : in.N - 1) * G;
  const int64_t slabs = slabs_of(in.N), at = (n / 64 * 16 + fr) * 8 + n % 64 / 16;  // of s in a group's constants
  if (in.packed == nullptr) {
    for (int g = fc; g < G; g += 4) {
      const float s = n < in.N ? in.gs[row + g] : 0.f;
      o.s[g * slabs * 128 + at] = s;
      o.s[g * slabs * 128 + at + 4] = n < in.N ? in.gz[row + g] - 8.f * s : 0.f;
    }
  }
  auto value = [&](int k) {
    const unsigned g = static_cast<unsigned>(k < units ? k : units - 1) / per;
    const float v = in.packed ? in.packed[g * slabs * 128 + at + 4] : in.gz[row + g] - 8.f * in.gs[row + g];
    return k < units ? v : 0.f;
  };
  // the first two steps (64 units) stay in registers: one round of loads for all of them
  float v0[2][8];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int e = 0; e < 8; ++e) v0[st][e] = st < steps ? value(32 * st + 8 * fc + e) : 0.f;
  float top = 0.f;
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(v0[st][e]));
  for (int st = 2; st < steps; ++st)
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(value(32 * st + 8 * fc + e)));
  top = fmaxf(top, __shfl_xor(top, 16, kWave));
  top = fmaxf(top, __shfl_xor(top, 32, kWave));
  const int ex = exponent_to_15(top);
  const float up = __builtin_amdgcn_ldexpf(1.f, ex);
  if (fc == 0) o.zdown[n] = __builtin_amdgcn_ldexpf(1.f, 8 - ex);
  auto store = [&](int st, const float (&v)[8]) {
    f16x8 zh, zl;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = v[e] * up;
      zh[e] = static_cast<_Float16>(t);
      zl[e] = static_cast<_Float16>(t - static_cast<float>(zh[e]));
    }
    _Float16* p = o.zf + (static_cast<int64_t>(tile) * steps + st) * 2 * (kFrag / 2) + lane * 8;
    *reinterpret_cast<f16x8*>(p) = zh;
    *reinterpret_cast<f16x8*>(p + kFrag / 2) = zl;
  };
#pragma unroll
  for (int st = 0; st < 2; ++st)
    if (st < steps) store(st, v0[st]);
  for (int st = 2; st < steps; ++st) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = value(32 * st + 8 * fc + e);
    store(st, v);
  }
}

// Packs the four 16-channel tiles of slab sb / nblk, block sb % nblk.
template <Order O>
__device__ __forceinline__ void pack_block(const SplitOut& o, const WeightIn& in, int64_t sb, int K) {
  const int lane = threadIdx.x % kWave, nblk = K / kBlk;
  const int b = static_cast<int>(sb % nblk);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t n = sb / nblk * 64 + 16 * u + lane % 16;
    u32x4 v = {0, 0, 0, 0};
    if (n < in.N) {
      const uint8_t* p = in.nib + n * (K / 2) + 64 * b;
      if constexpr (O == kInt4G128) {
        v = *reinterpret_cast<const u32x4*>(p + 16 * (lane / 16));
      } else {
        const u32x2 lo = *reinterpret_cast<const u32x2*>(p + 8 * (lane / 16));
        const u32x2 hi = *reinterpret_cast<const u32x2*>(p + 8 * (lane / 16) + 32);
        v = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    }
    *reinterpret_cast<u32x4*>(o.w + (sb * 4 + u) * kFrag + lane * 16) = v;
  }
}

// A row of x' with an infinity: y as float32 arithmetic on the dequantized weight has it (signed
// infinities; NaN where opposite ones meet or the weight is 0). Two pieces, or the sums' split into
// codes and zero term, would give NaN everywhere. No load of the usual rows passes here.
__device__ __forceinline__ void plain_row(const float* x, const float* inv, const WeightIn& in, float* y, int K) {
  const int G = K / in.group;
  for (int n = threadIdx.x % kWave; n < in.N; n += kWave) {
    const uint8_t* row = in.nib + static_cast<int64_t>(n) * (K / 2);
    float sum = 0.f;
    for (int g = 0; g < G; ++g) {
      const float s = in.gs[static_cast<int64_t>(n) * G + g], z = in.gz[static_cast<int64_t>(n) * G + g];
      for (int k = g * in.group; k < (g + 1) * in.group; ++k) {
        const int q = row[k / 2] >> (k % 2 * 4) & 15;
        const float w = __fadd_rn(__fmul_rn(static_cast<float>(q - 8), s), z);
        sum = __builtin_fmaf(inv ? __fmul_rn(x[k], inv[k]) : x[k], w, sum);
      }
    }
    y[n] = sum;
  }
}

// One wavefront per row of x (and of the padding); then, for int4, one per 16-channel tile of
// the zero term and, for a weight in the reference layout, one per packed (slab, block).
template <Order O>
__global__ __launch_bounds__(kSplitRows* kWave) void split_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ inv, SplitOut o, int M, int K, int mp, int nblk,
    WeightIn in, float* __restrict__ y) {
  constexpr int P = pieces(O);
  const int lane = threadIdx.x % kWave;
  const int m = blockIdx.x * kSplitRows + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  if (m >= mp) {  // whole wavefront
    if constexpr (O != kInt8) {
      const int tiles = static_cast<int>(slabs_of(in.N)) * 4, i = m - mp - tiles;
      if (i < 0)
        zero_frags<O>(o, in, m - mp, K);
      else if (in.packed == nullptr && i < tiles / 4 * (K / kBlk))
        pack_block<O>(o, in, i, K);
    }
    return;
  }
  const int chunks = K / 8;
  const float* xr = x + static_cast<int64_t>(m < M ? m : M - 1) * K;
  auto load = [&](int c, float (&v)[8]) {  // x' of chunk c (8 channels)
    const f32x4 a = *reinterpret_cast<const f32x4*>(xr + 8 * c);
    const f32x4 b = *reinterpret_cast<const f32x4*>(xr + 8 * c + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
    if (inv) {
      const f32x4 ia = *reinterpret_cast<const f32x4*>(inv + 8 * c);
      const f32x4 ib = *reinterpret_cast<const f32x4*>(inv + 8 * c + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = __fmul_rn(v[e], ia[e]);
        v[4 + e] = __fmul_rn(v[4 + e], ib[e]);
      }
    }
  };
  constexpr int kHeld = 6;  // chunks a lane keeps between the passes (K up to 3072; the rest is read again)
  float held[kHeld][8];
  float top = 0.f;
#pragma unroll
  for (int i = 0; i < kHeld; ++i) {
#pragma unroll
    for (int e = 0; e < 8; ++e) held[i][e] = 0.f;
    if (m < M && lane + kWave * i < chunks) load(lane + kWave * i, held[i]);
  }
#pragma unroll
  for (int i = 0; i < kHeld; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(held[i][e]));
  if (m < M) {
    for (int c = lane + kWave * kHeld; c < chunks; c += kWave) {
      float v[8];
      load(c, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(v[e]));
    }
  }
  top = lsh::wave_max_from<1>(top);
  // the power of two that brings the row's largest value to [2^14, 2^15)
  const int ex = exponent_to_15(top);
  const float up = m < M ? __builtin_amdgcn_ldexpf(1.f, ex) : 0.f;
  const bool plain = O != kInt8 && top == __builtin_inff();  // uniform; the GEMM leaves such a row alone
  if (lane == 0) o.rscale[m] = plain ? -1.f : __builtin_amdgcn_ldexpf(1.f, -ex);

  const int mt = m / 16, fr = m % 16;
  const int units = K / unit(O);
  _Float16* xs = o.xs + static_cast<int64_t>(mt) * sum_steps(units) * 2 * (kFrag / 2);
  auto store_sum = [&](int u, float s) {  // unit sums as the A operand of the zero term's product
    const _Float16 hi = static_cast<_Float16>(s), lo = static_cast<_Float16>(s - static_cast<float>(hi));
    _Float16* p = xs + (u / 32) * 2 * (kFrag / 2) + (fr + 16 * (u % 32 / 8)) * 8 + u % 8;
    p[0] = hi;
    p[kFrag / 2] = lo;
  };
  const int total = nblk * (kBlk / 8);  // chunks of the padded row
  auto put = [&](int c, float (&v)[8]) {  // every lane calls it (a unit's sum crosses lanes)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (O == kInt8 ? static_cast<float>(static_cast<__bf16>(v[e])) : v[e]) * up;
    // chunk cc of block b -> (q, fc)
    const int b = c / 16, cc = c % 16;
    const int q = O == kInt4G128 ? cc % 4 : 2 * (cc / 8) + cc % 2;
    const int fc = O == kInt4G128 ? cc / 4 : cc % 8 / 2;
    u32x4 hi, lo;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = O == kInt8 ? v[2 * j] : v[j], d = O == kInt8 ? v[2 * j + 1] : v[4 + j];
      const f16x2 h = {static_cast<_Float16>(a), static_cast<_Float16>(d)};
      hi[j] = as_u(h);
      const f16x2 l = {static_cast<_Float16>(a - static_cast<float>(h[0])),
                       static_cast<_Float16>(d - static_cast<float>(h[1]))};
      lo[j] = as_u(l);
    }
    if (c < total) {
      _Float16* p = o.xf + ((static_cast<int64_t>(mt) * nblk + b) * 4 + q) * P * (kFrag / 2) + (fr + 16 * fc) * 8;
      *reinterpret_cast<u32x4*>(p) = hi;
      if constexpr (P == 2) *reinterpret_cast<u32x4*>(p + kFrag / 2) = lo;
    }
    if constexpr (O != kInt8) {
      constexpr int L = unit(O) / 8;  // lanes of a unit
      float s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      s = lsh::group_sum<L>(s);
      if (lane % L == 0 && c < chunks) store_sum(c / L, s * 0x1p-8f);
    }
  };
#pragma unroll
  for (int i = 0; i < kHeld; ++i)
    if (kWave * i < total) put(lane + kWave * i, held[i]);
  for (int c0 = kWave * kHeld; c0 < total; c0 += kWave) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    if (m < M && c0 + lane < chunks) load(c0 + lane, v);
    put(c0 + lane, v);
  }
  if constexpr (O != kInt8) {
    const int padded = static_cast<int>(sum_steps(units)) * 32;
    for (int u = units + lane; u < padded; u += kWave) store_sum(u, 0.f);
    if (plain) plain_row(xr, inv, in, y + static_cast<int64_t>(m) * in.N, K);
  }
}

struct TileArgs {
  SplitOut a;
  const uint8_t* w;  // int4: packed tiles [slab of 64 channels][block][tile of 16][lane][16 bytes]; int8: [N, K]
  const float* s;    // int4: [group][slab][channel of the tile][s of the 4 tiles, z - 8 s of the 4 tiles];
                     // int8: scale [N]
  float* y;          // [M, N]
  int M, N, K, group;
  int blocks;        // K blocks of the fragments (the last ones zero): whole pairs of stages
  int tiles_m, tiles_n;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int64_t bytes) {
  const int n = bytes > 0x7fffffff ? 0x7fffffff : static_cast<int>(bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, n, 0x00020000);
}

// 8 nibbles -> 8 fp16, exact: a nibble at bit 0 (4) of a half's mantissa under the exponent of
// 1024 reads 1024 + q (1024 + 16 q); one packed subtraction (multiply-add) leaves q.
__device__ __forceinline__ f16x8 widen_nibbles(uint32_t w) {
  const f16x2 k1024 = {1024, 1024}, k16th = {0.0625f, 0.0625f}, k64 = {64, 64};
  const uint32_t lo = 0x000f000fu, hi = 0x00f000f0u, e = 0x64006400u, w8 = w >> 8;
  u32x4 r;
  r[0] = as_u(as_h2((w & lo) | e) - k1024);
  r[1] = as_u(__builtin_elementwise_fma(as_h2((w & hi) | e), k16th, -k64));
  r[2] = as_u(as_h2((w8 & lo) | e) - k1024);
  r[3] = as_u(__builtin_elementwise_fma(as_h2((w8 & hi) | e), k16th, -k64));
  return __builtin_bit_cast(f16x8, r);
}

// 8 int8 -> 8 fp16, exact: b ^ 0x80 = b + 128 as the mantissa of 1024 reads 1152 + b.
__device__ __forceinline__ f16x8 widen_int8(uint32_t w0, uint32_t w1) {
  const f16x2 k = {1152, 1152};
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t u = (i ? w1 : w0) ^ 0x80808080u;
    r[2 * i] = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - k);
    r[2 * i + 1] = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - k);
  }
  return __builtin_bit_cast(f16x8, r);
}

__device__ __forceinline__ f32x4 mfma(const f16x8& a, const f16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// A workgroup computes TM row tiles of 16 x WN slabs of 64 channels; WK = 4 / WN wavefronts
// split the K blocks of a slab.
template <Order O, int TM, int WN>
__global__ __launch_bounds__(kWaves* kWave, 2) void gemm_tile_kernel(TileArgs a) {
  constexpr int P = pieces(O), WK = kWaves / WN;
  constexpr int kStage = TM * 4 * P;  // fragments of one K block
  // two stages, as separate arrays: the compiler then sees that the direct-to-LDS loads of one
  // do not touch the fragments read from the other
  __shared__ __attribute__((aligned(16))) char lds0[WK * kStage * kFrag];
  __shared__ __attribute__((aligned(16))) char lds1[WK * kStage * kFrag];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int wn = wave % WN, wk = wave / WN;
  const int fr = lane % 16, fc = lane / 16;
  const int nblk = static_cast<int>(k_blocks(a.K));

  // XCD-aware order: workgroup b runs on XCD b % 8; an XCD takes consecutive tiles of a walk
  // that goes down 8 row tiles before it moves to the next column.
  const int total = a.tiles_m * a.tiles_n;
  const int per = (total + 7) / 8;
  const int id = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (id >= total) return;  // whole workgroup
  const int band = id / (8 * a.tiles_n), first = band * 8;
  const int high = a.tiles_m - first < 8 ? a.tiles_m - first : 8;
  const int r = id - first * a.tiles_n;
  const int tm = first + r % high, tn = r / high;

  const int n0 = (tn * WN + wn) * 64;  // this wavefront's channels
  const int slabs = static_cast<int>(slabs_of(a.N)), slab = min(n0 / 64, slabs - 1);
  const uint8_t* slab_w = a.w + static_cast<int64_t>(slab) * nblk * 4 * kFrag + lane * 16;  // int4
  const float* slab_s = a.s + (slab * 16 + fr) * 8;
  const auto rw = rsrc(a.w, static_cast<int64_t>(a.N) * a.K);  // int8
  int wofs[4];  // byte offset of the lane's weights
#pragma unroll
  for (int u = 0; u < 4; ++u) wofs[u] = min(n0 + 16 * u + fr, a.N - 1) * a.K + 16 * fc;
  constexpr int kScales = O == kInt4G64 ? 2 : 1;
  // The lane's weights for one step of loads: a K block (int4: 32 nibbles and the group scales
  // per tile) or half of one (int8: 16 weights per tile, to spare registers).
  struct Weights {
    uint32_t w[4][4];
    float s[4][kScales];
  };
  auto load_w = [&](int b, int h, Weights& o) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (O == kInt8) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rw, wofs[u], b * 128 + 64 * h, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.w[u][j] = v[j];
      } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(slab_w + (static_cast<int64_t>(b) * 4 + u) * kFrag);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.w[u][j] = v[j];
      }
    }
    if constexpr (O != kInt8) {
#pragma unroll
      for (int i = 0; i < kScales; ++i) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(
            slab_s + static_cast<int64_t>((b * kBlk + i * 64) / a.group) * slabs * 128);
#pragma unroll
        for (int u = 0; u < 4; ++u) o.s[u][i] = v[u];
      }
    }
  };
  // blocks b .. b + WK - 1 of the row tiles, straight into LDS
  constexpr int kBlkBytes = 4 * P * kFrag;  // of one row tile
  const auto rx = rsrc(reinterpret_cast<const char*>(a.a.xf) + static_cast<int64_t>(tm) * TM * a.blocks * kBlkBytes,
                       static_cast<int64_t>(TM) * a.blocks * kBlkBytes);
  auto load_a = [&](int b, char* lds) {
#pragma unroll
    for (int i = 0; i < WK * kStage / kWaves; ++i) {
      const int f = i * kWaves + wave;  // fragment of the stage
      const int k = f / kStage, t = f % kStage / (4 * P), j = f % (4 * P);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(lds + f * kFrag), 16,
                                               lane * 16, (t * a.blocks + b + k) * kBlkBytes + j * kFrag, 0, 0);
    }
  };

  f32x4 acc[TM][4];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One stage: blocks b .. b + WK - 1 from `cur`, while the next stage's loads go to `nxt`
  // (past the end they repeat the last stage, unused: a load under a branch would be waited
  // for before the products). A row's weights of two int4 blocks (two halves of an int8 block)
  // share a 128-byte line, and are loaded together: apart, the line would be fetched twice.
  //   int4: weights wa; `pair`: those of the next two stages go to wb and wa.
  //   int8: halves wa and wb; the next stage's go to wa and wc.
  auto stage = [&](int b, const char* cur, char* nxt, Weights& wa, Weights& wb, Weights& wc, auto pair) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this stage's loads have landed
    __syncthreads();                     // ... everyone's, and the other stage is read
    const char* my = cur + wk * kStage * kFrag + lane * 16;
    const int bn = min(b + WK + wk, nblk - 1);
    load_a(min(b + WK, a.blocks - WK), nxt);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (O == kInt8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q == 2) {
          load_w(bn, 0, wa);
          load_w(bn, 1, wc);
        }
        __builtin_amdgcn_sched_barrier(0);
        const Weights& w = q < 2 ? wa : wb;
        f16x8 bq[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          bq[u] = widen_int8(w.w[u][2 * (q % 2)], w.w[u][2 * (q % 2) + 1]);
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          const f16x8 fa = *reinterpret_cast<const f16x8*>(my + (t * 4 + q) * kFrag);
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[t][u] = mfma(fa, bq[u], acc[t][u]);
        }
      }
    } else {
      f16x8 bq[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) bq[u][q] = widen_nibbles(wa.w[u][q]);
      float sc[4][kScales];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < kScales; ++i) sc[u][i] = wa.s[u][i];
      if constexpr (decltype(pair)::value) {
        __builtin_amdgcn_sched_barrier(0);
        load_w(bn, 0, wb);
        load_w(min(b + 2 * WK + wk, nblk - 1), 0, wa);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        f32x4 d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f16x8 fa[P];
#pragma unroll
          for (int p = 0; p < P; ++p)
            fa[p] = *reinterpret_cast<const f16x8*>(my + ((t * 4 + q) * P + p) * kFrag);
          const bool fresh = q == 0 || (O == kInt4G64 && q == 2);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            d[u] = mfma(fa[0], bq[u][q], fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : d[u]);
#pragma unroll
          for (int u = 0; u < 4; ++u) d[u] = mfma(fa[P - 1], bq[u][q], d[u]);
          if (q == 3 || (O == kInt4G64 && q == 1)) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                acc[t][u][e] = __builtin_fmaf(sc[u][kScales > 1 ? q / 2 : 0], d[u][e], acc[t][u][e]);
          }
        }
      }
    }
  };
  constexpr std::true_type both;
  constexpr std::false_type none;
  Weights w0, w1, w2;
  load_a(0, lds0);
  load_w(min(wk, nblk - 1), 0, w0);
  load_w(O == kInt8 ? min(wk, nblk - 1) : min(WK + wk, nblk - 1), 1, w1);
  for (int b = 0; b < a.blocks; b += 2 * WK) {
    if constexpr (O == kInt8) {
      stage(b, lds0, lds1, w0, w1, w2, none);
      stage(b + WK, lds1, lds0, w0, w2, w1, none);
    } else {
      stage(b, lds0, lds1, w0, w1, w2, none);
      stage(b + WK, lds1, lds0, w1, w0, w2, both);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // no load into LDS is left in flight

  if constexpr (WK > 1) {  // the K parts meet in LDS, added in order by the first wavefront
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(lds0);
    f32x4* red1 = reinterpret_cast<f32x4*>(lds1);
    constexpr int kHalf = WK * kStage;  // tiles of 1 KB one stage array holds
    static_assert(2 * kHalf >= (WK - 1) * WN * TM * 4, "LDS of the K sum");
    auto at = [&](int k, int t, int u) -> f32x4& {
      const int i = ((k - 1) * WN + wn) * TM * 4 + t * 4 + u;
      return (i < kHalf ? red + i * kWave : red1 + (i - kHalf) * kWave)[lane];
    };
    if (wk > 0) {
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          at(wk, t, u) = acc[t][u];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 1; k < WK; ++k)
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          acc[t][u] += at(k, t, u);
  }

  if constexpr (O != kInt8) {
    // the zero term: sum over units of (unit sum) * (z - 8 s), both as two fp16 pieces
    const int steps = static_cast<int>(sum_steps(a.K / unit(O)));
    const _Float16* xs = a.a.xs + static_cast<int64_t>(tm) * TM * steps * 2 * (kFrag / 2) + lane * 8;
    const int last = slabs * 4 - 1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int nt = min(n0 / 16 + u, last);
      const _Float16* zf = a.a.zf + static_cast<int64_t>(nt) * steps * 2 * (kFrag / 2) + lane * 8;
      f32x4 d[TM];
#pragma unroll
      for (int t = 0; t < TM; ++t) d[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int st = 0; st < steps; ++st) {
        const f16x8 zh = *reinterpret_cast<const f16x8*>(zf + st * 2 * (kFrag / 2));
        const f16x8 zl = *reinterpret_cast<const f16x8*>(zf + (st * 2 + 1) * (kFrag / 2));
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          const _Float16* p = xs + (t * steps + st) * 2 * (kFrag / 2);
          const f16x8 xh = *reinterpret_cast<const f16x8*>(p);
          const f16x8 xl = *reinterpret_cast<const f16x8*>(p + kFrag / 2);
          d[t] = mfma(xh, zh, d[t]);
          d[t] = mfma(xl, zh, d[t]);
          d[t] = mfma(xh, zl, d[t]);
          d[t] = mfma(xl, zl, d[t]);
        }
      }
      const float down = a.a.zdown[16 * nt + fr];
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][u][e] = __builtin_fmaf(d[t][e], down, acc[t][u][e]);
    }
  }

  // lane holds rows 4 fc + e, column fr of each 16 x 16 tile; a store past the last row or channel
  // gets a vector offset outside the buffer and is dropped (the scalar offset takes no part in the
  // bounds check, so the row must not go there)
  const int m0 = tm * TM * 16;
  const auto ry = rsrc(a.y + static_cast<int64_t>(m0) * a.N, static_cast<int64_t>(a.M - m0) * a.N * 4);
  f32x4 rm[TM];  // before the stores: a load behind them would wait for them
#pragma unroll
  for (int t = 0; t < TM; ++t) rm[t] = *reinterpret_cast<const f32x4*>(a.a.rscale + m0 + 16 * t + 4 * fc);
  float cs[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) cs[u] = O == kInt8 ? a.s[min(n0 + 16 * u + fr, a.N - 1)] : 1.f;
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * t + 4 * fc + e;
      const bool on = m0 + row < a.M && (O == kInt8 || rm[t][e] > 0.f);
      const uint32_t row_ofs = static_cast<uint32_t>(row) * static_cast<uint32_t>(a.N) * 4;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 16 * u + fr;
        const uint32_t ofs = n < a.N && on ? row_ofs + static_cast<uint32_t>(n) * 4 : 0x80000000u;
        const float v = O == kInt8 ? acc[t][u][e] * cs[u] : acc[t][u][e];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v * rm[t][e]), ry, ofs, 0, 0);
      }
    }
}

// The workspace laid out at p; returns the bytes it takes.
template <Order O>
int64_t lay_out(char* p, int64_t M, int64_t N, int64_t K, int64_t G, bool pack, SplitOut* o) {
  char* const start = p;
  auto take = [&](int64_t bytes) {
    char* at = p;
    p += (bytes + 255) / 256 * 256;
    return at;
  };
  const int64_t mp = pad_rows(M), np = slabs_of(N) * 64;
  SplitOut r{};
  r.rscale = reinterpret_cast<float*>(take(mp * 4));
  r.xf = reinterpret_cast<_Float16*>(take(mp * pad_blocks(K, kWaves) * kBlk * 2 * pieces(O)));
  if (O != kInt8) {
    r.xs = reinterpret_cast<_Float16*>(take(sum_bytes(mp, K)));
    r.zf = reinterpret_cast<_Float16*>(take(sum_bytes(np, K)));
    r.zdown = reinterpret_cast<float*>(take(np * 4));
    if (pack) {
      r.w = reinterpret_cast<uint8_t*>(take(weight_bytes(N, K)));
      r.s = reinterpret_cast<float*>(take(const_bytes(N, G)));
    }
  }
  if (o) *o = r;
  return p - start;
}

template <Order O, int TM, int WN>
void launch_tile(const float* x, const float* inv, const WeightIn& in, TileArgs a, hipStream_t st) {
  const int mp = (a.M + 16 * TM - 1) / (16 * TM) * (16 * TM);
  a.blocks = static_cast<int>(pad_blocks(a.K, kWaves / WN));
  int64_t waves = mp;
  if (O != kInt8) waves += slabs_of(a.N) * (4 + (in.packed ? 0 : a.K / kBlk));
  lsh::launch(split_rows_kernel<O>, dim3(static_cast<unsigned>((waves + kSplitRows - 1) / kSplitRows)),
              dim3(kSplitRows * kWave), 0, st, false, x, inv, a.a, a.M, a.K, mp, a.blocks, in, a.y);
  a.tiles_m = (a.M + 16 * TM - 1) / (16 * TM);
  a.tiles_n = (a.N + 64 * WN - 1) / (64 * WN);
  const int64_t total = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  lsh::launch(gemm_tile_kernel<O, TM, WN>, dim3(static_cast<unsigned>((total + 7) / 8 * 8)),
              dim3(kWaves * kWave), 0, st, true, a);
}

// Tile by the number of workgroups it leaves (256 CUs; us per call, split pass included):
//   64 x 256, no K split, from 1.25 workgroups per CU: 2048 x 6144 x 1024 63 (32 x 128: 83, 16 x 64:
//     ~160), 1024 x 6144 x 1024 42 (46);
//   32 x 128, two K parts, from 0.75 per CU: 777 x 1024 x 2048 25 (64 x 256: 48, 16 x 64: 29),
//     1857 x 1024 x 3072 46 (69);
//   16 x 64, four K parts, below: 64 x 1024 x 3072 17 (32 x 128: 27), 512 x 1024 x 2048 19 (22).
template <Order O>
void run_tile(const float* x, const float* inv, const WeightIn& in, const TileArgs& a, hipStream_t st) {
  auto tiles = [&](int rows, int cols) {
    return static_cast<int64_t>((a.M + rows - 1) / rows) * ((a.N + cols - 1) / cols);
  };
  const int cus = lsh::device_cus();
  if (tiles(64, 256) * 4 >= 5 * cus)
    launch_tile<O, 4, 4>(x, inv, in, a, st);
  else if (tiles(32, 128) * 4 >= 3 * cus)
    launch_tile<O, 2, 2>(x, inv, in, a, st);
  else
    launch_tile<O, 1, 1>(x, inv, in, a, st);
}

}  // namespace

int64_t lsh::int8_tile_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  return lay_out<kInt8>(nullptr, M, N, K, 0, false, nullptr);
}

void lsh::int8_tile_launch(const float* x, const int8_t* qweight, const float* scale, float* y, int64_t M, int64_t N,
                           int64_t K, void* workspace, hipStream_t st) {
  TileArgs a{};
  lay_out<kInt8>(static_cast<char*>(workspace), M, N, K, 0, false, &a.a);
  a.w = reinterpret_cast<const uint8_t*>(qweight);
  a.s = scale;
  a.y = y;
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(N);
  a.K = static_cast<int>(K);
  run_tile<kInt8>(x, nullptr, WeightIn{}, a, st);
}

extern "C" int64_t llmserve_int4_linear_tile_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t group_size) {
  if (M <= 0 || N <= 0 || K <= 0 || group_size <= 0 || K % kBlk || group_size % 64 || K % group_size) return 0;
  return lay_out<kInt4G64>(nullptr, M, N, K, K / group_size, true, nullptr);
}

extern "C" int llmserve_int4_linear_tile(const float* x, const float* inv_act_scale, const uint8_t* nibbles,
                                         const float* g_scale, const float* g_zero, const void* packed, float* y,
                                         int64_t M, int64_t N, int64_t K, int64_t group_size, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  LSH_CHECK(M >= 0 && N >= 1 && K >= 1 && group_size >= 64, "int4_linear_tile: bad shape");
  LSH_CHECK(K % kBlk == 0 && group_size % 64 == 0 && K % group_size == 0,
            "int4_linear_tile: K must be a multiple of 128 and group_size of 64 (K %% group == 0)");
  LSH_CHECK(packed == nullptr || group_size % kBlk == 0,
            "int4_linear_tile: a packed weight needs a group_size multiple of 128");
  LSH_CHECK(M < (1LL << 24) && N < (1LL << 22) && K < (1LL << 20) && M * K < (1LL << 36),
            "int4_linear_tile: shape too large");
  if (M == 0) return LLMSERVE_OK;
  LSH_CHECK(x && y && nibbles && g_scale && g_zero, "int4_linear_tile: null pointer");
  LSH_CHECK(lsh::aligned16(x) && lsh::aligned16(nibbles) && (packed == nullptr || lsh::aligned16(packed)) &&
                (inv_act_scale == nullptr || lsh::aligned16(inv_act_scale)),
            "int4_linear_tile: x, inv_act_scale and the weight must be 16-byte aligned");
  const int64_t need = llmserve_int4_linear_tile_workspace_bytes(M, N, K, group_size);
  LSH_CHECK(workspace != nullptr && workspace_bytes >= need && lsh::aligned16(workspace),
            "int4_linear_tile: a 16-byte aligned workspace of %lld bytes is needed (%lld given)", (long long)need,
            (long long)workspace_bytes);
  TileArgs a{};
  a.y = y;
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(N);
  a.K = static_cast<int>(K);
  a.group = static_cast<int>(group_size);
  const bool g128 = group_size % kBlk == 0;
  char* ws = static_cast<char*>(workspace);
  if (g128)
    lay_out<kInt4G128>(ws, M, N, K, K / group_size, packed == nullptr, &a.a);
  else
    lay_out<kInt4G64>(ws, M, N, K, K / group_size, true, &a.a);
  const float* constants = nullptr;
  if (packed != nullptr)
    constants = reinterpret_cast<const float*>(static_cast<const char*>(packed) +
                                               (weight_bytes(N, K) + 255) / 256 * 256);
  a.w = packed ? static_cast<const uint8_t*>(packed) : a.a.w;
  a.s = packed ? constants : a.a.s;
  const WeightIn in{nibbles, g_scale, g_zero, constants, a.N, a.group};
  hipStream_t st = lsh::as_stream(stream);
  if (g128)
    run_tile<kInt4G128>(x, inv_act_scale, in, a, st);
  else
    run_tile<kInt4G64>(x, inv_act_scale, in, a, st);
  return lsh::launch_status("int4_linear_tile");
}
