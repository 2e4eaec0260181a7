// Device-side building blocks shared by the gfx950 kernels: 64-lane wavefront reductions
// and scans on DPP, 128-bit vector types, exact integer division by a launch constant.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "kernels.hpp"

namespace et {

constexpr int kWave = 64;

// ---- 128-bit / 64-bit movers -----------------------------------------------------------
struct alignas(16) u32x4 { uint32_t x, y, z, w; };
struct alignas(8) u32x2 { uint32_t x, y; };

template <int BYTES> struct vec_bytes;
template <> struct vec_bytes<16> { using type = u32x4; };
template <> struct vec_bytes<8> { using type = u32x2; };
template <> struct vec_bytes<4> { using type = uint32_t; };

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float2v __attribute__((ext_vector_type(2)));

// ---- DPP cross-lane helpers --------------------------------------------------------------
// update_dpp(old, src, ctrl, row_mask, bank_mask, bound_ctrl): lanes whose source is
// disabled keep `old`.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_f32(float old, float src) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old),
                                                               __builtin_bit_cast(int, src), CTRL, ROW_MASK, 0xf, false));
}
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ int dpp_i32(int old, int src) {
  return __builtin_amdgcn_update_dpp(old, src, CTRL, ROW_MASK, 0xf, false);
}

constexpr int kDppQuadXor1 = 0xB1;      // quad_perm:[1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;      // quad_perm:[2,3,0,1]
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kDppRowMirror = 0x140;
constexpr int kDppRowNewBcast = 0x150;  // + n: lane n of every 16 lanes, to all of them
constexpr int kDppRowBcast15 = 0x142;
constexpr int kDppRowBcast31 = 0x143;

// Sum over the 64 lanes of a wavefront; every lane receives the total.
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_f32<kDppQuadXor1>(0.f, v);
  v += dpp_f32<kDppQuadXor2>(0.f, v);
  v += dpp_f32<kDppRowHalfMirror>(0.f, v);
  v += dpp_f32<kDppRowMirror>(0.f, v);
  v += dpp_f32<kDppRowBcast15, 0xa>(0.f, v);
  v += dpp_f32<kDppRowBcast31, 0xc>(0.f, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_f32<kDppQuadXor1>(v, v));
  v = fmaxf(v, dpp_f32<kDppQuadXor2>(v, v));
  v = fmaxf(v, dpp_f32<kDppRowHalfMirror>(v, v));
  v = fmaxf(v, dpp_f32<kDppRowMirror>(v, v));
  v = fmaxf(v, dpp_f32<kDppRowBcast15, 0xa>(v, v));
  v = fmaxf(v, dpp_f32<kDppRowBcast31, 0xc>(v, v));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

__device__ __forceinline__ int wave_sum_i32(int v) {
  v += dpp_i32<kDppQuadXor1>(0, v);
  v += dpp_i32<kDppQuadXor2>(0, v);
  v += dpp_i32<kDppRowHalfMirror>(0, v);
  v += dpp_i32<kDppRowMirror>(0, v);
  v += dpp_i32<kDppRowBcast15, 0xa>(0, v);
  v += dpp_i32<kDppRowBcast31, 0xc>(0, v);
  return __builtin_amdgcn_readlane(v, 63);
}

// Inclusive prefix sum over the 64 lanes (row_shr steps inside each row of 16, then the
// row totals are carried across rows with two broadcasts).
__device__ __forceinline__ int wave_inclusive_scan_i32(int v) {
  v += dpp_i32<0x111>(0, v);                 // row_shr:1
  v += dpp_i32<0x112>(0, v);                 // row_shr:2
  v += dpp_i32<0x114>(0, v);                 // row_shr:4
  v += dpp_i32<0x118>(0, v);                 // row_shr:8
  v += dpp_i32<kDppRowBcast15, 0xa>(0, v);   // rows 1,3 += last lane of rows 0,2
  v += dpp_i32<kDppRowBcast31, 0xc>(0, v);   // rows 2,3 += lane 31
  return v;
}

__device__ __forceinline__ int lane_id() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// ---- exact division of a 32-bit unsigned by a launch-time constant ------------------------
struct fastdiv {
  uint32_t d, magic, shift;
};
inline fastdiv make_fastdiv(uint32_t d) {
  fastdiv f;
  f.d = d;
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  f.shift = s;
  f.magic = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1);
  return f;
}
__device__ __forceinline__ uint32_t div_by(uint32_t n, const fastdiv& f) {
  uint32_t t = __umulhi(n, f.magic);
  return (t + n) >> f.shift;         // valid while t + n < 2^32, i.e. n < 2^31
}

// ---- half helpers ------------------------------------------------------------------------
__device__ __forceinline__ float h2f(_Float16 h) { return (float)h; }
__device__ __forceinline__ _Float16 f2h(float f) { return (_Float16)f; }   // v_cvt_f16_f32, round-to-nearest-even

// ---- stores ------------------------------------------------------------------------------
// Cache policy of buffer stores: sc1 writes through the L2 to the memory side, where the other XCDs find the value; nt keeps less of
// the line in the caches on its way.  What lies dirty in the L2s when a kernel ends is written back before the next one starts, which
// the fp16 products' C and the weights' turned copies are spared so.  Encoders of 12 layers, C in plain stores and written through, one
// card in turn: 16 x 64 in a graph 508 -> 502 us, 8 x 128 from ids 475 -> 467, 100 x 32 753 -> 730, the ops on 217 x 53 1877 -> 1810, 32 x 512
// 2858 -> 2788, 16 x 1024 2841 -> 2692 (another card: 32 x 512 2707 -> 2676, ops level).  So do the small tiles' pieces of 2 and 4 bytes a lane
// (12 layers, two runs of one library within 0.4 %): 5 x 64 of 8 heads in a graph, 2 bytes plain 362, 4 bytes plain 362, all through 359; 5 x 64
// of 12 heads, 4 bytes plain 415, through 411, 2 bytes level; 12 x 64 531 and 529; 31 x 64, the 4 bytes of six columns plain 734, through 727.
// 16 bytes in two stores of 8 are written twice (ops 1809 -> 1895).  Level or worse, and so plain: LayerNorm's fp16 rows, the short fp16
// attention (1000 x 64 7435 -> 7655), the streaming one (8-byte pieces of a head's rows: 64 x 512 5412 -> 5538, 193 x 100 2995 -> 3055), the fp32
// one's 16-byte pieces of pair rows (100 x 64 2770 -> 2805, 500 x 64 10960 -> 11130, 15 x 379 level), the fp32 products' C in floats (500 x 64
// 11330 -> 11440, 210 x 64 5538 -> 5601).  Matrices beyond the last-level cache keep nt (1000 x 64: sc1 instead or both +0.2 to +0.5 %).
constexpr int kPolicyNt = 2, kPolicyThrough = 16;
// 8 bytes, written through.
template <typename V>
__device__ __forceinline__ void store_through(void* p, const V& v) {
  static_assert(sizeof(V) == 8);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#if defined(__HIP_DEVICE_COMPILE__)
// 16 bytes a lane at byte `off` from `base`, which is the same for the whole wavefront, written through.
template <typename V>
__device__ __forceinline__ void store_through(void* base, uint32_t off, const V& v) {
  static_assert(sizeof(V) == 16);
  typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(base, 0, ~0u, 0x00020000);
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, v), r, off, 0, kPolicyThrough);
}
#endif

// ---- bias + GELU arithmetic (reference: cuda/cuda_kernels.cu:29-51) -------------------------
// 0.5*(1+tanh(u)) is evaluated as 1/(1+exp(-2u)), which is the same function without the cancellation of 1+tanh for
// negative u.
__device__ __forceinline__ float gelu_cdf(float x, float x3) {
  // exp(-2u) = 2^(-2u*log2(e)) with u = 0.7978845608028654 * (x + 0.044715 * x3): both factors in one constant
  const float e = __builtin_amdgcn_exp2f((x + 0.044715f * x3) * (-2.8853900817779268f * 0.7978845608028654f));
  return __builtin_amdgcn_rcpf(1.0f + e);
}
// fp16 rounding points of the reference: __hadd2 for the bias, two __hmul2 for the cube, the CDF in float rounded to
// half, __hmul2.  HV is a vector of halves (half4, half8).
template <typename HV, int N>
__device__ __forceinline__ HV bias_gelu_half(HV v, HV bias) {
  const HV x = v + bias;
  const HV x3 = x * (x * x);
  HV cdf;
#pragma unroll
  for (int i = 0; i < N; ++i) cdf[i] = f2h(gelu_cdf(h2f(x[i]), h2f(x3[i])));
  return x * cdf;
}

// ---- split floats ------------------------------------------------------------------------
// x = h + m + l exactly, three bfloat16 pieces, each the rest of the ones before it rounded to nearest (8 significand
// bits and a sign apiece cover the 24 bits of a float).  Two values at a time, packed.  Infinities, NaNs and magnitudes
// that round to a bfloat16 infinity (above 3.38e38) give NaN pieces.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t round_pair_bf16(float& x0, float& x1) {      // returns the pieces, leaves the rests
  const float2v v = {x0, x1};
  const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  x0 -= __builtin_bit_cast(float, p << 16);
  x1 -= __builtin_bit_cast(float, p & 0xffff0000u);
  return p;
}
// N consecutive values (N = 1, 2, 4 or 8; col a multiple of N) of a split row: [k / 32][h, m, l][32] bfloat16
template <int N, typename V>
__device__ __forceinline__ void store_split(uint16_t* row, int col, const V& v) {
  constexpr int W = (N + 1) / 2;
  uint16_t* p = row + (col >> 5) * 96 + (col & 31);
  float x[2 * W];
#pragma unroll
  for (int j = 0; j < 2 * W; ++j) x[j] = j < N ? v[j < N ? j : 0] : 0.f;
#pragma unroll
  for (int piece = 0; piece < 3; ++piece) {
    uint32_t w[W];
#pragma unroll
    for (int j = 0; j < W; ++j) w[j] = round_pair_bf16(x[2 * j], x[2 * j + 1]);
    uint16_t* d = p + piece * 32;
    if constexpr (N == 1) *d = (uint16_t)w[0];
    else if constexpr (N == 2) *reinterpret_cast<uint32_t*>(d) = w[0];
    else if constexpr (N == 4) *reinterpret_cast<u32x2*>(d) = u32x2{w[0], w[1]};
    else *reinterpret_cast<u32x4*>(d) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// ---- floats as pairs of halves -----------------------------------------------------------
// x = 2^e (h + l) for the values of a row that stay below a bound (gemm_pair.hip).  The exponent that puts values up to `bound`
// below 2^15, kept where 2^e and 2^-e are ordinary floats; NaN counts as the largest.
__device__ __forceinline__ int pair_exponent(float bound) {
  return min(max(__builtin_amdgcn_frexp_expf(fminf(bound, 3.4e38f)) - 15, -112), 113);
}
__device__ __forceinline__ float pair_scale(int e) { return __builtin_ldexpf(1.0f, -e); }
// N consecutive values (N = 1, 2, 4 or 8; col a multiple of N) of a pair row: [k / 32][h, l][32] halves; scale = pair_scale(e)
// The epilogues that store pair rows are bound by their arithmetic: with l made from the stored halves a pair of values takes one
// conversion, where the compiler converted every value a second time for l (FFN-up on 20375 rows 277 -> 263 us together with
// gemm_pair_kernel's one lane per exponent, same bits).
// Pieces of 8 bytes, those of FFN-up's large tiles, of LayerNorm and of the short attention, are written through (kPolicyThrough): fp32
// encoders of 12 layers, plain and so, 40 x 64 positions 1680 -> 1650 us, 100 x 64 2803 -> 2778, 160 x 64 4081 -> 4072, 15 x 379 2904 -> 2887; from
// 210 x 64 on level (500 x 64 10995 and 11028, with 0.3 % between two runs of one library).
template <int N, typename V>
__device__ __forceinline__ void store_pair(_Float16* row, int col, const V& v, float scale) {
  typedef _Float16 hvec __attribute__((ext_vector_type(N)));
  hvec h, l;
#pragma unroll
  for (int j = 0; j < N; ++j) h[j] = f2h(v[j] * scale);
  if constexpr (N >= 2) asm("" : "+v"(h));
#pragma unroll
  for (int j = 0; j < N; ++j) l[j] = f2h(__builtin_fmaf(v[j], scale, -h2f(h[j])));
  _Float16* d = row + (col >> 5) * 64 + (col & 31);
  if constexpr (N == 4) {
    store_through(d, h);
    store_through(d + 32, l);
  } else {
    *reinterpret_cast<hvec*>(d) = h;
    *reinterpret_cast<hvec*>(d + 32) = l;
  }
}
// Row r of `out` from a wavefront that holds it, lane + 64 i the i-th four values (zero beyond vpr): the exponent from the
// largest value, and the row's Euclidean norm.  Whoever writes a row writes the same bits.
template <int ITERS, typename V>
__device__ __forceinline__ void store_pair_row(const V (&x)[ITERS], int vpr, const PairRows& out, int r, int n) {
  const int lane = threadIdx.x & (kWave - 1);
  float top = 0.f;
#pragma unroll
  for (int i = 0; i < ITERS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) top = fmaxf(top, fabsf(x[i][j]));
  const int e = pair_exponent(wave_max(top));
  const float scale = pair_scale(e);
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < ITERS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float y = x[i][j] * scale;
      sq = __builtin_fmaf(y, y, sq);
    }
  sq = wave_sum(sq);
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int c = lane + i * kWave;
    if (c < vpr) store_pair<4>(out.rows + (size_t)r * 2 * n, c * 4, x[i], scale);
  }
  if (lane == 0) {
    out.exp[r] = e;
    out.norm[r] = __builtin_ldexpf(__builtin_sqrtf(sq), e);
  }
}
// a < b as an integer, without a compare of its own (what the scalar unit makes of a difference's sign)
__device__ __forceinline__ int uniform_less(int a, int b) { return (int)((unsigned)(a - b) >> 31); }
// a / b, a >= 0, b > 0, same in all lanes.  The compiler's division takes about twice the instructions.
__device__ __forceinline__ int uniform_div(int a, int b) {
  if (__builtin_expect(a >= 1 << 22, 0)) return a / b;     // the quotient of the two floats may be off by more than one
  int q = __builtin_amdgcn_readfirstlane((int)((float)a * __builtin_amdgcn_rcpf((float)b)));
  const int r = a - q * b;
  return q - uniform_less(r, 0) + 1 - uniform_less(r, b);
}
// What bounds a product's columns, from the `stats` of its weight (PairWeightJob): the largest column norm, |bias| and bias (or 0).
struct PairBounds {
  float norm = 0.f, bias = 0.f, above = 0.f;
};
// By one wavefront: nine requests a lane, and what becomes of them and of the words behind them.
struct PairStats {
  float2v pair[8];
  float above;
};
__device__ __forceinline__ void pair_stats_request(const float* __restrict__ stats, int pairs, int i0, float2v (&v)[8]) {
  const float2v* p = reinterpret_cast<const float2v*>(stats);
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = p[min(i0 + u * kWave + (int)(threadIdx.x & (kWave - 1)), pairs - 1)];
}
__device__ __forceinline__ void pair_stats_request(const float* __restrict__ stats, int pairs, int tiles, PairStats& s) {
  pair_stats_request(stats, pairs, 0, s.pair);
  s.above = stats[2 * pairs + min((int)(threadIdx.x & (kWave - 1)), tiles - 1)];
}
__device__ __forceinline__ PairBounds pair_stats_max(const float* __restrict__ stats, int pairs, int tiles, PairStats& s) {
  float2v top = {0.f, 0.f};
  for (int i0 = 0;;) {
#pragma unroll
    for (int u = 0; u < 8; ++u) top = float2v{fmaxf(top[0], s.pair[u][0]), fmaxf(top[1], s.pair[u][1])};
    i0 += 8 * kWave;
    if (i0 >= pairs) break;
    pair_stats_request(stats, pairs, i0, s.pair);
  }
  for (int i = (int)(threadIdx.x & (kWave - 1)) + kWave; i < tiles; i += kWave) s.above = fmaxf(s.above, stats[2 * pairs + i]);
  return {wave_max(top[0]), wave_max(top[1]), wave_max(s.above)};
}
// A bound of |gelu(v)| for all v = x.w + b of a row x of this Euclidean norm: |v| <= |x| |w| + |b|, and gelu(v) lies between -0.171
// and max(v, 0).  Without the second one bias that switches its neuron off took the bits of all others of the row (one of -2^30:
// rows of the layer's result off by 2.9e-3).  What is above the largest value costs no bits: the product's own rounding of a value
// is 2^-24 |x| |w| of its column, a pair's 2^-40 of this, so columns may differ by 2^14 in norm.
__device__ __forceinline__ float pair_gelu_bound(float norm, const PairBounds& b) {
  const float v = norm * (b.norm * 1.01f);
  return fminf(v + b.bias, fmaxf(v + b.above, 0.171f));
}

// seq_start[b] = first packed row of sequence b (b in [0, batch]; seq_start[batch] = T), written by the thread that
// owns packed row t in [0, T]: it covers the sequences that begin at t (token-less sequences included).
__device__ __forceinline__ void seq_start_for_row(const int32_t* __restrict__ batch_idx, int T, int t, int batch,
                                                  int32_t* __restrict__ seq_start) {
  if (t > T) return;
  const int prev = t == 0 ? -1 : batch_idx[t - 1];
  const int cur = t == T ? batch : min(batch_idx[t], batch - 1);
  const int last = t == T ? batch : cur;         // entries (prev, last] start at t
  for (int b = prev + 1; b <= last; ++b) seq_start[b] = t;
}

// order[0..batch) = the sequences sorted by length, longest first (buckets of 16 tokens; the order inside a bucket is
// whatever the atomics give: it only decides which workgroup of the attention kernel starts first).  All THREADS threads
// of one workgroup.
constexpr int kOrderBuckets = kWave + 1;      // lengths up to 1024
template <int THREADS>
__device__ __forceinline__ void sort_sequences(const int32_t* __restrict__ seq_start, int batch, int32_t* __restrict__ order) {
  __shared__ int hist[kOrderBuckets], base[kOrderBuckets];
  for (int i = threadIdx.x; i < kOrderBuckets; i += THREADS) hist[i] = 0;
  __syncthreads();
  auto bucket_of = [&](int b) {
    const int len = seq_start[b + 1] - seq_start[b];
    return kOrderBuckets - 1 - min(max(len, 0) >> 4, kOrderBuckets - 1);      // longest first
  };
  for (int b = threadIdx.x; b < batch; b += THREADS) atomicAdd(&hist[bucket_of(b)], 1);
  __syncthreads();
  if (threadIdx.x < kWave) {                  // 65 buckets: one per lane, and the last one behind them all
    const int mine = hist[threadIdx.x], upto = wave_inclusive_scan_i32(mine);
    base[threadIdx.x] = upto - mine;
    if (threadIdx.x == kWave - 1) base[kWave] = upto;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < batch; b += THREADS) order[atomicAdd(&base[bucket_of(b)], 1)] = b;
}

// The smallest t in [0, T] from which on batch_idx[t] >= b; batch_idx is ascending.  Whole wavefronts.
__device__ __forceinline__ int wave_lower_bound(const int32_t* __restrict__ batch_idx, int T, int b) {
  int lo = 0, hi = T;
  while (hi > lo) {
    const int len = hi - lo, step = (len + kWave - 1) / kWave, probe = lo + lane_id() * step;
    const int c = __popcll(__ballot(probe < hi && batch_idx[min(probe, hi - 1)] < b));
    hi = c == 0 ? lo : min(lo + c * step, hi);
    lo = c == 0 ? lo : lo + (c - 1) * step + 1;
  }
  return lo;
}

// ---- classes of the mask rows --------------------------------------------------------------
// what is known of a block's mask rows behind the last token
constexpr int kMaskPlain = 1, kMaskZeros = 2, kMaskOnes = 4;

// class of a block of 16 query positions: kMaskPlain = the rows of the mask are 1 for keys up to the last token's and 0
// beyond, kMaskZeros / kMaskOnes = they are all 0 / all 1 beyond it.  All 256 threads of a workgroup; the rows of sequence b are
// t0 .. t1.
template <typename T>
__device__ __forceinline__ void mask_class_block(const T* __restrict__ attr_mask, const int32_t* __restrict__ word_idx, int b, int qb,
                                                 int t0, int t1, int seq_len, int blocks, uint8_t* __restrict__ cls) {
  constexpr int kElems = 16 / (int)sizeof(T);
  typedef uint32_t words __attribute__((ext_vector_type(4)));
  if (t1 <= t0) return;
  const int n = min(max(word_idx[t1 - 1], 0), seq_len - 1) + 1;
  if (qb * 16 >= n) return;                                  // never looked at
  const int rows = min(16, n - qb * 16);
  const T* m = attr_mask + ((size_t)b * seq_len + qb * 16) * seq_len;
  // what differs from 1 up to the last token, from 0 behind it, from 1 behind it (bit patterns)
  uint32_t no_token = 0, no_zero = 0, no_one = 0;
  if (seq_len % kElems == 0) {
    constexpr uint32_t kOne = sizeof(T) == 2 ? 0x3c003c00u : 0x3f800000u;
    const int cpr = seq_len / kElems;
#pragma unroll 4
    for (int i = threadIdx.x; i < rows * cpr; i += 256) {
      const words w = reinterpret_cast<const words*>(m)[i];
      const int bits = (n - (i % cpr) * kElems) * (int)sizeof(T) * 8;       // of the 128 here, those up to the last token
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = min(max(bits - j * 32, 0), 32);
        const uint32_t token = (uint32_t)((1ull << t) - 1), one = w[j] ^ kOne;
        no_token |= one & token;
        no_zero |= w[j] & ~token;
        no_one |= one & ~token;
      }
    }
  } else {
    // The rows follow each other without a gap: 16 bytes at a time from the first boundary on, a row's end inside them or not, and
    // the values in front of it and behind the last whole piece one by one.  (Value by value, with a division and a trip to memory
    // for each, it took 62 us a layer call at 32 x 891 positions in fp16, the weights' copies included, where it takes 20 so; 15 x 379
    // positions in fp32, a launch of its own, 13.1 and 5.8.)
    const int all = rows * seq_len;
    auto look_at = [&](int i) {
      const T v = m[i];
      const uint32_t zero = v == (T)0.0f ? 0u : 1u, one = v == (T)1.0f ? 0u : 1u;
      if (i % seq_len < n) {
        no_token |= one;
      } else {
        no_zero |= zero;
        no_one |= one;
      }
    };
    const int front = min((int)((16 - ((uintptr_t)m & 15)) & 15) / (int)sizeof(T), all), pieces = (all - front) / kElems;
    const int behind = front + pieces * kElems;
    if ((int)threadIdx.x < front) look_at(threadIdx.x);
    if ((int)threadIdx.x < all - behind) look_at(behind + threadIdx.x);
    constexpr uint32_t kOne = sizeof(T) == 2 ? 0x3c003c00u : 0x3f800000u, kNoSign = sizeof(T) == 2 ? 0x7fff7fffu : 0x7fffffffu;
    constexpr int kBits = (int)sizeof(T) * 8, kAtOnce = 4;
    const words* piece = reinterpret_cast<const words*>(m + front);
    int key = (front + (int)threadIdx.x * kElems) % seq_len;               // of the piece's first value
    const int on = 256 * kElems % seq_len;
    auto below = [](int bits) { return (uint32_t)((1ull << min(max(bits, 0), 32)) - 1); };
    for (int i = threadIdx.x; i < pieces; i += kAtOnce * 256) {
      words w[kAtOnce];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) w[u] = piece[min(i + u * 256, pieces - 1)];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) {
        // values up to the last token: the first min(n - key, left) of the piece, and of those of the next row, from `left` on, n
        const int left = seq_len - key, first = min(n - key, left) * kBits, next = left * kBits, last = (left + n) * kBits;
        if (i + u * 256 < pieces) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t token = below(first - j * 32) | (below(last - j * 32) & ~below(next - j * 32)), one = w[u][j] ^ kOne;
            no_token |= one & token;
            no_zero |= w[u][j] & kNoSign & ~token;
            no_one |= one & ~token;
          }
        }
        key += on;
        key -= key >= seq_len ? seq_len : 0;
      }
    }
  }
  __shared__ int found[4];
  const bool plain = !__any(no_token != 0), zeros = !__any(no_zero != 0), ones = !__any(no_one != 0);
  if ((threadIdx.x & (kWave - 1)) == 0)
    found[threadIdx.x / kWave] = (plain && zeros ? kMaskPlain : 0) | (zeros ? kMaskZeros : 0) | (ones ? kMaskOnes : 0);
  __syncthreads();
  if (threadIdx.x == 0) cls[(size_t)b * blocks + qb] = (uint8_t)(found[0] & found[1] & found[2] & found[3]);
}

// ---- what a layer needs to know of its batch, by blocks of the launch that prepares its weights ---------------
// (a launch of its own for each of them costs the layer 2 .. 5 us and the calling thread 3 us: seq_order_kernel and
// mask_class_kernel behind the weights' launch, 8.8 + 1.7 + 5.0 us, against 9.6 us with their blocks in it at 39 x 117 positions;
// six layer calls 675 -> 640 us)
constexpr int kTableBatch = 2303;             // sequences whose starts a block keeps in LDS
// Up to this many rows one block looks at all of batch_idx (12 single-layer calls: 1 x 32 positions 719 -> 680 us, 8 x 128 829 ->
// 810 us, 64 x 32 972 -> 946 us against the starts by many blocks and the sort in a launch of its own); beyond, it searches for
// the starts of up to kTableSearch sequences, three to six dependent loads.
constexpr int kTableRows = 2048;
constexpr int kTableSearch = 1024;

// starts[b] for the sequences threadIdx.x + 256 q: a step leaves one part in PROBES + 1 of the rows that may hold the start.
template <int SEQS, int PROBES>
__device__ __forceinline__ void search_starts(const int32_t* __restrict__ batch_idx, int T, int batch, int32_t* starts) {
  int lo[SEQS];
#pragma unroll
  for (int q = 0; q < SEQS; ++q) lo[q] = 0;
  for (int span = T; span > 0;) {              // the start lies in [lo, lo + span]
    const int step = span / (PROBES + 1) + 1;
    int seen[SEQS][PROBES];
#pragma unroll
    for (int q = 0; q < SEQS; ++q)
#pragma unroll
      for (int i = 0; i < PROBES; ++i) seen[q][i] = batch_idx[min(lo[q] + step * (i + 1) - 1, T - 1)];
#pragma unroll
    for (int q = 0; q < SEQS; ++q) {
      const int b = (int)threadIdx.x + q * 256;
      int c = 0;
#pragma unroll
      for (int i = 0; i < PROBES; ++i) c += lo[q] + step * (i + 1) - 1 < T && seen[q][i] < b ? 1 : 0;
      lo[q] += c * step;
    }
    span = max(step - 1, span - PROBES * step);
  }
#pragma unroll
  for (int q = 0; q < SEQS; ++q) {
    const int b = (int)threadIdx.x + q * 256;
    if (b < batch) starts[b] = lo[q];
  }
}

// The whole sequence table by one block of 256 threads, the starts in LDS for the sort.
__device__ __forceinline__ void sequence_table_block(const BatchJobs& jobs, int T, int32_t* starts) {
  const int32_t* __restrict__ batch_idx = jobs.batch_idx;
  if (T <= kTableRows) {
    constexpr int kFly = 8;                                   // rows per thread requested together
    for (int t0 = 0; t0 <= T; t0 += 256 * kFly) {
      int prev[kFly], cur[kFly];
#pragma unroll
      for (int u = 0; u < kFly; ++u) {
        const int t = t0 + u * 256 + (int)threadIdx.x;
        prev[u] = t > 0 && t <= T ? batch_idx[t - 1] : -1;
        cur[u] = t < T ? batch_idx[t] : jobs.batch;
      }
#pragma unroll
      for (int u = 0; u < kFly; ++u) {
        const int t = t0 + u * 256 + (int)threadIdx.x;
        if (t > T) continue;
        const int last = t == T ? jobs.batch : min(cur[u], jobs.batch - 1);
        for (int b = max(prev[u], -1) + 1; b <= last; ++b) starts[b] = t;     // entries (prev, last] start at t
      }
    }
  } else {
    if (jobs.batch <= 256) search_starts<1, 32>(batch_idx, T, jobs.batch, starts);
    else search_starts<kTableSearch / 256, 8>(batch_idx, T, jobs.batch, starts);
    if (threadIdx.x == 0) starts[jobs.batch] = T;
  }
  __syncthreads();
  for (int b = threadIdx.x; b <= jobs.batch; b += 256) jobs.seq_table[b] = starts[b];
  sort_sequences<256>(starts, jobs.batch, jobs.seq_table + jobs.batch + 1);
}

// Block `block` of the jobs' batch_job_blocks() blocks; `scratch`: room for kTableBatch + 1 words of LDS.
__device__ __forceinline__ void batch_job_block(const BatchJobs& jobs, int block, int32_t* scratch) {
  const int T = jobs.rows_dev ? min(*jobs.rows_dev, jobs.rows_bound) : jobs.rows_bound;
  if (block < jobs.table_blocks) {
    if (jobs.one_block_table) sequence_table_block(jobs, T, scratch);
    else seq_start_for_row(jobs.batch_idx, T, block * 256 + (int)threadIdx.x, jobs.batch, jobs.seq_table);
    return;
  }
  // a class block: its sequence's rows, looked for by two of its wavefronts
  block -= jobs.table_blocks;
  const int blocks = (jobs.seq_len + 15) / 16, b = block / blocks, qb = block - b * blocks;
  const int wave = threadIdx.x / kWave;
  if (wave < 2) {
    const int t = b + wave == jobs.batch ? T : wave_lower_bound(jobs.batch_idx, T, b + wave);
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[wave] = t;
  }
  __syncthreads();
  const int t0 = scratch[0], t1 = scratch[1];
  if (jobs.fp32) mask_class_block((const float*)jobs.attr_mask, jobs.word_idx, b, qb, t0, t1, jobs.seq_len, blocks, jobs.cls);
  else mask_class_block((const _Float16*)jobs.attr_mask, jobs.word_idx, b, qb, t0, t1, jobs.seq_len, blocks, jobs.cls);
}

}  // namespace et
