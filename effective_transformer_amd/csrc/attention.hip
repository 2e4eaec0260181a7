// Attention side of the encoder layer on gfx950.
//   qkv_bias_pad      : [T,H] + bias -> zero-padded [B,heads,S,d]   (reference: cuda/attention.cu:105-242,
//                                                                    zero fill tf_op/bert_transformer_op.cu.cc:146)
//   softmax           : masked, scaled softmax in place             (cuda/attention.cu:249-382)
//   transpose_rm_pad  : [B,heads,S,d] -> packed [T,H]               (cuda/attention.cu:387-492)
//   attention (fused) : QK^T, masked softmax, PV and un-padding in one kernel
//                       (tf_op/bert_transformer_op.cu.cc:159-192); reads Q/K/V either from the padded
//                       buffers or straight from packed token rows, writes packed [T,H].
//
// Softmax semantics (all kernels): t = qk*scale + (1-mask)*(-10000); m = max(max_k t, 0), at 1024 keys
// max_k t; e = exp(t-m); p = e / (sum e + 1e-6).  In fp16 the score is rounded to half before the
// softmax, as the reference stores it, and the probability before P.V: up to 64 positions p itself, as
// the reference, beyond (streaming kernel) e, whose rounded values the sum adds up, in float, before the
// division.
#include <type_traits>

#include "et_device.hpp"
#include "kernels.hpp"

namespace et {

namespace {

constexpr float kLog2e = 1.4426950408889634f;

template <typename T> struct Chunk16;
template <> struct Chunk16<float> {
  typedef float4v vec;
  float4v v;
  static constexpr int kElems = 4;
};
template <> struct Chunk16<_Float16> {
  typedef half8 vec;
  half8 v;
  static constexpr int kElems = 8;
};

// ------------------------------------------------------------------------------------------
// add bias + head split + re-pad, one workgroup per (sequence, matrix).  Every 16-byte chunk of
// the padded destination is written once: bias-added data where a token exists, zero elsewhere.
// ------------------------------------------------------------------------------------------
constexpr int kPadThreads = 256;
constexpr int kPadMaxSeq = 1024;

template <typename T>
__global__ __launch_bounds__(kPadThreads) void qkv_bias_pad_kernel(
    const T* __restrict__ Q, const T* __restrict__ bQ, const T* __restrict__ K, const T* __restrict__ bK,
    const T* __restrict__ V, const T* __restrict__ bV, T* __restrict__ q_buf, T* __restrict__ k_buf,
    T* __restrict__ v_buf, const int32_t* __restrict__ seq_start, const int32_t* __restrict__ word_idx, int seq_len,
    int heads, int d) {
  using C = Chunk16<T>;
  __shared__ int tok_of_pos[kPadMaxSeq];
  const int b = blockIdx.x;
  const int mat = blockIdx.y;
  const T* src = mat == 0 ? Q : (mat == 1 ? K : V);
  const T* bias = mat == 0 ? bQ : (mat == 1 ? bK : bV);
  T* dst = mat == 0 ? q_buf : (mat == 1 ? k_buf : v_buf);
  for (int s = threadIdx.x; s < seq_len; s += kPadThreads) tok_of_pos[s] = -1;
  __syncthreads();
  const int t0 = seq_start[b], t1 = seq_start[b + 1];
  for (int t = t0 + threadIdx.x; t < t1; t += kPadThreads) {
    const int s = word_idx[t];
    if (s >= 0 && s < seq_len) tok_of_pos[s] = t;
  }
  __syncthreads();
  const int cpd = d / C::kElems;           // chunks per head row
  const int cph = heads * cpd;             // chunks per token row
  const int total = heads * seq_len * cpd;
  C* out = reinterpret_cast<C*>(dst) + (size_t)b * total;
  const C* in = reinterpret_cast<const C*>(src);
  const C* bi = reinterpret_cast<const C*>(bias);
  for (int i = threadIdx.x; i < total; i += kPadThreads) {
    const int c = i % cpd;
    const int s = (i / cpd) % seq_len;
    const int head = i / (cpd * seq_len);
    const int t = tok_of_pos[s];
    C val;
    if (t >= 0) {
      val.v = in[(size_t)t * cph + head * cpd + c].v + bi[head * cpd + c].v;
    } else {
#pragma unroll
      for (int j = 0; j < C::kElems; ++j) val.v[j] = (T)0;
    }
    out[i] = val;
  }
}

// ------------------------------------------------------------------------------------------
// stand-alone softmax: one wavefront per (b, head, q) row, up to 1024 keys.
// ------------------------------------------------------------------------------------------
constexpr int kSmThreads = 256;
constexpr int kSmMaxIters = 16;

template <typename T>
__global__ __launch_bounds__(kSmThreads) void softmax_kernel(T* __restrict__ qk, const T* __restrict__ attr_mask,
                                                             int rows_total, int heads, int seq_len, float scaler) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row = blockIdx.x * (kSmThreads / kWave) + threadIdx.x / kWave;
  if (row >= rows_total) return;          // wave-uniform
  const int q = row % seq_len;
  const int b = row / (seq_len * heads);
  T* x = qk + (size_t)row * seq_len;
  const T* mk = attr_mask + ((size_t)b * seq_len + q) * seq_len;
  float t[kSmMaxIters];
  // the maximum is clamped below at 0, except at 1024 keys, where the reference's max reduction has no idle lane
  float mx = seq_len < 1024 ? 0.f : -INFINITY;
#pragma unroll
  for (int i = 0; i < kSmMaxIters; ++i) {
    const int k = lane + i * kWave;
    t[i] = -INFINITY;
    if (k < seq_len) {
      t[i] = (float)x[k] * scaler + (1.0f - (float)mk[k]) * -10000.0f;
      mx = fmaxf(mx, t[i]);
    }
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kSmMaxIters; ++i) {
    t[i] = __builtin_amdgcn_exp2f((t[i] - mx) * kLog2e);   // exp2(-inf) = 0 for absent keys
    sum += t[i];
  }
  sum = wave_sum(sum) + 1e-6f;
#pragma unroll
  for (int i = 0; i < kSmMaxIters; ++i) {
    const int k = lane + i * kWave;
    if (k < seq_len) x[k] = (T)(t[i] / sum);
  }
}

// ------------------------------------------------------------------------------------------
// un-pad + head merge: gather flattened over (packed row, 16-byte chunk).
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void transpose_rm_padding_kernel(
    const T* __restrict__ src, T* __restrict__ dst, const int32_t* __restrict__ rows_dev, int rows_bound, int seq_len,
    int heads, int cpd, const int32_t* __restrict__ batch_idx, const int32_t* __restrict__ word_idx) {
  using C = Chunk16<T>;
  const int rows = rows_dev ? min(*rows_dev, rows_bound) : rows_bound;
  const int cph = heads * cpd;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)rows * cph) return;
  const int t = (int)(i / cph);
  const int c = (int)(i - (long)t * cph);
  const int head = c / cpd;
  const int cc = c - head * cpd;
  const int b = batch_idx[t], s = word_idx[t];
  reinterpret_cast<C*>(dst)[i] =
      reinterpret_cast<const C*>(src)[(((size_t)b * heads + head) * seq_len + s) * cpd + cc];
}

// ------------------------------------------------------------------------------------------
// fused attention, size_per_head = 64, seq_len <= 64 in fp16 and <= 32 in fp32 (longer sequences: the kernels below).
//
// One workgroup (4 wavefronts) per (sequence, group of heads).  What does not depend on the
// head is done once: token positions, the zero fill of key/value slots without a token (so that a
// mask that attends to a padded key sees the zero score / zero value the reference's padded buffers
// hold) and the mask rows of each wavefront's queries, which stay in registers.  Per head the K rows
// and the transpose of the V rows are staged in LDS at their padded positions, Q rows beside them,
// while the next head's rows are already in flight into registers.  Each wavefront takes 16-query tiles:
//   S^T = K Q^T   on v_mfma_f32_16x16x32_f16 / v_mfma_f32_16x16x4_f32 -> a lane owns one query
//                 column and 4 keys of every 16-key tile,
//   softmax       over the lane's values + 2 cross-lane steps (lanes l, l^16, l^32, l^48 share a query),
//   O^T = V^T P^T where the lane's own probability registers already are the B operand,
//   then the lane writes 4 consecutive features of its query's packed output row.
// Key tiles that hold no token skip their MFMAs (score 0, value 0) but still go through the
// masked softmax, so the result equals the padded computation exactly.
// ------------------------------------------------------------------------------------------
constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / kWave;
constexpr int kD = 64;

template <typename T> struct AttnCfg;
template <> struct AttnCfg<_Float16> {
  static constexpr int kQkStride = kD + 8;   // halves; 144-byte rows keep 16-byte reads of 8 consecutive rows on distinct banks
  static constexpr int kVtPad = 4;           // halves
  // fp16 keeps V row-major ([key][feature]) and transposes 8x4 blocks in registers: 160-byte rows put the four
  // key groups of an 8-byte operand read 128 bytes apart modulo the 256-byte bank span
  static constexpr int kVStride = kD + 16;
};
template <> struct AttnCfg<float> {
  static constexpr int kQkStride = kD + 4;   // floats; 272-byte rows
  static constexpr int kVtPad = 4;           // floats
};

template <typename T, int NKT>
struct AttnSmem {
  static constexpr int kSp = NKT * 16;
  static constexpr int kVtStride = kSp + AttnCfg<T>::kVtPad;
  static constexpr size_t kQBytes = (size_t)kSp * AttnCfg<T>::kQkStride * sizeof(T);
  static constexpr size_t kVtBytes =
      sizeof(T) == 2 ? (size_t)kSp * AttnCfg<_Float16>::kVStride * sizeof(T) : (size_t)kD * kVtStride * sizeof(T);
  static constexpr size_t kBytes = 2 * kQBytes + kVtBytes + kSp * sizeof(int);
};

// Reductions over the four 16-lane rows of a wavefront (lanes l, l ^ 16, l ^ 32, l ^ 48), the result in all of them.
// v_permlane16_swap exchanges the odd rows of its first operand with the even rows of its second, v_permlane32_swap
// the upper half of the first with the lower half of the second: with both operands a copy of v, the two results hold
// the two rows (halves) that have to be combined, in every lane, without a trip through the LDS crossbar.  The
// operands of each combination are those of the xor shuffle, in one order or the other: same bits.
// (Written as inline assembly on two float copies: with the compiler's builtin, and with integer copies handed back
// as a vector, the second result was lost when both operands hold the same value.  The wait states in front are
// those the compiler itself puts between a VALU write and this instruction.)
__device__ __forceinline__ float xor_lanes_16_32_max(float v) {
  float a = v, b = v;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  v = fmaxf(a, b);
  a = v;
  b = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}
__device__ __forceinline__ float xor_lanes_16_32_sum(float v) {
  float a = v, b = v;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  v = a + b;
  a = v;
  b = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return a + b;
}

// The lane's 16 values of row `row` (-1: none) and head `head`, o[dt][r] = feature 16 dt + 4 g + r (RUN: 16 g + 4 dt + r), as pairs under
// the exponent of the head's largest value.  Whole wavefronts; the four lanes of a query have the same row.
template <bool RUN>
__device__ __forceinline__ void store_head_pairs(float* dst, int row, int H, int head, const float4v (&o)[4], HeadExps head_exp) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int g = (threadIdx.x & (kWave - 1)) >> 4;
  float top = 0.f;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) top = fmaxf(top, fabsf(o[dt][r]));
  const int e = pair_exponent(xor_lanes_16_32_max(top));
  if (row < 0) return;
  const float scale = pair_scale(e);
  _Float16* out = reinterpret_cast<_Float16*>(dst) + (size_t)row * 2 * H;
  if constexpr (RUN) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
      store_pair<8>(out, head * kD + g * 16 + half * 8, __builtin_shufflevector(o[2 * half], o[2 * half + 1], 0, 1, 2, 3, 4, 5, 6, 7), scale);
  } else {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) store_pair<4>(out, head * kD + dt * 16 + g * 4, o[dt], scale);
  }
  if (g == 0) head_exp.exp[(size_t)head * head_exp.stride + row] = (int8_t)e;
#endif
}

// What a launch leaves in dst, as its last argument.  fp16 has one form only, and its instances take no more than that: the host
// issues an encoder of few rows more slowly than the device runs it, and its time goes by the bytes of the arguments too (1 x 32
// positions, 12 layers: 375 us with the 16 of the exponents, 364 without).
template <typename T>
struct AttnOut {
  AttentionOut form = AttentionOut::kPlain;
  int exp_stride = 0;
  int8_t* exp = nullptr;
};
template <>
struct AttnOut<_Float16> {
  AttentionOut form = AttentionOut::kPlain;
};

// WAVES: wavefronts per workgroup, one 16-query tile each.  CPT = 16-byte chunks of
// one matrix a thread moves per head (ceil(seq rows * chunks per row / threads)).
template <typename T, int NKT, int WAVES, int CPT>
__global__ __launch_bounds__(WAVES * kWave) void attention_kernel(
    // (the first 14 words come in registers: what the chain order -> start table -> positions and rows needs)
    const int32_t* __restrict__ seq_start, const int32_t* __restrict__ word_idx, int batch, int seq_len, int heads, int heads_per_wg,
    int layout, int packed_ld, const T* __restrict__ q_src, const T* __restrict__ k_src, const T* __restrict__ v_src,
    const T* __restrict__ attr_mask, T* __restrict__ dst, float scaler, AttnOut<T> out) {
  using Cfg = AttnCfg<T>;
  using Sm = AttnSmem<T, NKT>;
  using C = Chunk16<T>;
  constexpr int kQS = Cfg::kQkStride;
  constexpr int kVS = Sm::kVtStride;
  constexpr int kVR = AttnCfg<_Float16>::kVStride;   // fp16: stride of the row-major V tile
  constexpr int kSp = Sm::kSp;
  constexpr int kCpr = kD / C::kElems;       // 16-byte chunks per head row
  constexpr int kThreads = WAVES * kWave;
  static_assert(NKT <= WAVES, "a wavefront serves one query tile");
  typedef T mask4 __attribute__((ext_vector_type(4)));

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T* Qs = reinterpret_cast<T*>(smem_raw);
  T* Ks = reinterpret_cast<T*>(smem_raw + Sm::kQBytes);
  T* Vt = reinterpret_cast<T*>(smem_raw + 2 * Sm::kQBytes);
  int* tok_of_pos = reinterpret_cast<int*>(smem_raw + 2 * Sm::kQBytes + Sm::kVtBytes);

  // workgroups are dealt out in the order of the table's second half: sequences of similar length side by side, the
  // longest first
  const int b = min(max(seq_start[batch + 1 + blockIdx.y], 0), batch - 1);
  const int h_begin = blockIdx.x * heads_per_wg;
  const int h_end = min(h_begin + heads_per_wg, heads);
  const int t0 = seq_start[b], t1 = seq_start[b + 1];
  const int len = t1 - t0;
  if (len <= 0) return;
  const int H = heads * kD;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int l16 = lane & 15;
  const int g = lane >> 4;

  // ---- everything that does not depend on the head: issued up front, all loads in flight together ----
  // positions are ascending inside a sequence: the last token bounds the occupied 16-row tiles
  const int last_pos_raw = word_idx[t1 - 1];
  int my_t[CPT], my_pos[CPT], my_c[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = threadIdx.x + k * kThreads;
    const int tt = i / kCpr;
    my_c[k] = i - tt * kCpr;
    my_t[k] = tt < len ? t0 + tt : -1;
    my_pos[k] = tt < len ? word_idx[t0 + tt] : -1;
  }
  // the mask rows of this wavefront's queries stay in registers for all heads
  mask4 mreg[NKT];
  const bool vec_mask = (seq_len & 3) == 0;
  {
    const int q = wave * 16 + l16;
    const T* mrow = attr_mask + ((size_t)b * seq_len + min(q, seq_len - 1)) * seq_len;
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      const int key0 = kt * 16 + g * 4;
      mask4 m4 = {(T)0, (T)0, (T)0, (T)0};
      if (vec_mask) {
        if (key0 < seq_len) m4 = *reinterpret_cast<const mask4*>(mrow + key0);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (key0 + r < seq_len) m4[r] = mrow[key0 + r];
      }
      mreg[kt] = m4;
    }
  }
  using V16 = typename C::vec;
  V16 rq[CPT], rk[CPT], rv[CPT];
  // 16-byte chunk k of this thread for `head`: element offset into the source matrices.  Packed rows are addressed by
  // the token alone, so their loads leave without waiting for the positions (one step less in the chain of dependent
  // loads a workgroup starts with: -1.6 us per launch at 1000 x 64 tokens); a position outside the sequence is only
  // sorted out when the chunk goes to LDS.
#define ET_ATTN_LOAD_HEAD(head_)                                                                            \
  _Pragma("unroll") for (int k = 0; k < CPT; ++k) {                                                         \
    if (my_t[k] >= 0 && (layout == 1 || (my_pos[k] >= 0 && my_pos[k] < seq_len))) {                         \
      const size_t off = layout == 1                                                                        \
                             ? (size_t)my_t[k] * packed_ld + (head_) * kD + my_c[k] * C::kElems             \
                             : (((size_t)b * heads + (head_)) * seq_len + my_pos[k]) * kD + my_c[k] * C::kElems; \
      rq[k] = *reinterpret_cast<const V16*>(q_src + off);                                                   \
      rk[k] = *reinterpret_cast<const V16*>(k_src + off);                                                   \
      rv[k] = *reinterpret_cast<const V16*>(v_src + off);                                                   \
    }                                                                                                       \
  }
  ET_ATTN_LOAD_HEAD(h_begin)

  const int last_pos = min(max(last_pos_raw, 0), seq_len - 1);
  const int n_tiles = last_pos / 16 + 1;    // 16-row tiles that hold at least one token (queries and keys)

  // mask value -> additive bias, once for all heads: (1 - m) * -10000 in float as the reference computes it, kept in
  // the element type (exact for 0/1 masks); keys beyond seq_len do not exist
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      mreg[kt][r] = kt * 16 + g * 4 + r < seq_len ? (T)((1.0f - (float)mreg[kt][r]) * -10000.0f) : (T)-INFINITY;

  // ---- position table, then zero the key / value slots that hold no token (once: heads only overwrite tokens) ----
  for (int i = threadIdx.x; i < kSp; i += kThreads) tok_of_pos[i] = -1;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    if (my_t[k] >= 0 && my_c[k] == 0 && my_pos[k] >= 0 && my_pos[k] < seq_len) tok_of_pos[my_pos[k]] = my_t[k];
  __syncthreads();
  {
    // the fp16 P.V contraction runs over pairs of key tiles, so an odd tile count drags one more tile of Vt in
    const int rows = min(kSp, ((n_tiles + 1) / 2) * 32);
    // K: row `pos` (kQS elements), Vt: column `pos` of every feature row
    for (int i = threadIdx.x; i < rows * (kD / 2); i += kThreads) {
      const int pos = i / (kD / 2), w = i - pos * (kD / 2);
      if (tok_of_pos[pos] < 0) {
        if (sizeof(T) == 2) {
          reinterpret_cast<uint32_t*>(Ks + pos * kQS)[w] = 0u;                // 2 halves
          reinterpret_cast<uint32_t*>(Vt + pos * kVR)[w] = 0u;                // V is row-major for fp16
        } else {
          Ks[pos * kQS + 2 * w] = (T)0; Ks[pos * kQS + 2 * w + 1] = (T)0;
          Vt[(2 * w) * kVS + pos] = (T)0;
          Vt[(2 * w + 1) * kVS + pos] = (T)0;
        }
      }
    }
  }

  // where this lane's query writes its output row (head 0; null without a token): the same for every head
  const int tq = wave < n_tiles && wave < NKT ? tok_of_pos[wave * 16 + l16] : -1;
  T* out_row = tq >= 0 ? dst + (size_t)tq * H + g * (sizeof(T) == 2 ? 16 : 4) : nullptr;
  if (sizeof(T) == 4 && out.form == AttentionOut::kSplit && tq >= 0)
    out_row = reinterpret_cast<T*>(reinterpret_cast<uint16_t*>(dst) + (size_t)tq * 3 * H);

  for (int head = h_begin; head < h_end; ++head) {
    if (head != h_begin) __syncthreads();      // every wavefront is done with the previous head's tiles
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int pos = my_pos[k];
      if (my_t[k] >= 0 && pos >= 0 && pos < seq_len) {
        const int c = my_c[k];
        *reinterpret_cast<V16*>(Qs + pos * kQS + c * C::kElems) = rq[k];
        *reinterpret_cast<V16*>(Ks + pos * kQS + c * C::kElems) = rk[k];
        if constexpr (sizeof(T) == 2) {
          *reinterpret_cast<V16*>(Vt + pos * kVR + c * C::kElems) = rv[k];
        } else {
#pragma unroll
          for (int j = 0; j < C::kElems; ++j) Vt[(c * C::kElems + j) * kVS + pos] = rv[k][j];
        }
      }
    }
    __syncthreads();
    if (head + 1 < h_end) { ET_ATTN_LOAD_HEAD(head + 1) }         // flies while this head is computed

    if (wave < n_tiles) {                     // wave-uniform
      const int q = wave * 16 + l16;          // this lane's query position
      float s[NKT][4];
      // ---- S^T = K Q^T -------------------------------------------------------------------
      if constexpr (sizeof(T) == 2) {
        half8 bq[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) bq[ks] = *reinterpret_cast<const half8*>(Qs + q * kQS + ks * 32 + g * 8);
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          float4v acc = {0.f, 0.f, 0.f, 0.f};
          if (kt < n_tiles) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
              const half8 a = *reinterpret_cast<const half8*>(Ks + (kt * 16 + l16) * kQS + ks * 32 + g * 8);
              acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bq[ks], acc, 0, 0, 0);
            }
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) s[kt][r] = h2f(f2h(acc[r]));   // the score is stored in half
        }
      } else {
        float bq[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4v v4 = *reinterpret_cast<const float4v*>(Qs + q * kQS + g * 16 + i * 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) bq[i * 4 + j] = v4[j];
        }
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          float4v acc = {0.f, 0.f, 0.f, 0.f};
          if (kt < n_tiles) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float4v a4 = *reinterpret_cast<const float4v*>(Ks + (kt * 16 + l16) * kQS + g * 16 + i * 4);
#pragma unroll
              for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[j], bq[i * 4 + j], acc, 0, 0, 0);
            }
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) s[kt][r] = acc[r];
        }
      }
      // ---- masked softmax over the keys of query q ------------------------------------------
      float mx = 0.f;                          // clamp of the maximum at 0
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float tv = s[kt][r] * scaler + (float)mreg[kt][r];   // mreg: (1 - mask) * -10000, -inf beyond seq_len
          s[kt][r] = tv;
          mx = fmaxf(mx, tv);
        }
      mx = xor_lanes_16_32_max(mx) * kLog2e;
      float sum = 0.f;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[kt][r] = __builtin_amdgcn_exp2f(s[kt][r] * kLog2e - mx);
          sum += s[kt][r];
        }
      sum = xor_lanes_16_32_sum(sum) + 1e-6f;
      const float inv = 1.0f / sum;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[kt][r] *= inv;
      // ---- O^T = V^T P^T --------------------------------------------------------------------
      float4v o[4];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] = float4v{0.f, 0.f, 0.f, 0.f};
      if constexpr (sizeof(T) == 2) {
        // A operand j = V^T rows {4*l + j}: the lane reads 4 consecutive features of its 8 keys (the keys its
        // probability registers belong to) and transposes the 8x4 block with v_perm_b32
#pragma unroll
        for (int ks = 0; ks < NKT / 2; ++ks) {
          if (2 * ks < n_tiles) {
            half8 p;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              p[r] = f2h(s[2 * ks][r]);
              p[4 + r] = f2h(s[2 * ks + 1][r]);
            }
            typedef uint32_t u2 __attribute__((ext_vector_type(2)));
            typedef uint32_t u4 __attribute__((ext_vector_type(4)));
            u2 raw[8];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
              const int key = ks * 32 + (kk >> 2) * 16 + g * 4 + (kk & 3);
              raw[kk] = *reinterpret_cast<const u2*>(Vt + key * kVR + l16 * 4);
            }
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
              u4 lo, hi;
#pragma unroll
              for (int q4 = 0; q4 < 4; ++q4) {
                lo[q4] = __builtin_amdgcn_perm(raw[2 * q4 + 1][jj], raw[2 * q4][jj], 0x05040100u);
                hi[q4] = __builtin_amdgcn_perm(raw[2 * q4 + 1][jj], raw[2 * q4][jj], 0x07060302u);
              }
              o[2 * jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, lo), p, o[2 * jj], 0, 0, 0);
              o[2 * jj + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, hi), p, o[2 * jj + 1], 0, 0, 0);
            }
          }
        }
      } else {
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          if (kt < n_tiles) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
              const float4v a4 = *reinterpret_cast<const float4v*>(Vt + (dt * 16 + l16) * kVS + kt * 16 + g * 4);
#pragma unroll
              for (int r = 0; r < 4; ++r)
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[r], s[kt][r], o[dt], 0, 0, 0);
            }
          }
        }
      }
      if constexpr (sizeof(T) == 4) {
        if (out.form == AttentionOut::kPairs) {  // (uniform)
          store_head_pairs<false>(dst, tq, H, head, o, HeadExps{out.exp, out.exp_stride});
          continue;
        }
      }
      // ---- write the lane's 16 features of its query's packed row --------------------------
      if (out_row != nullptr) {
        if constexpr (sizeof(T) == 2) {
          // o[j][r] is feature 16*g + 4*r + j: 16 consecutive features
          half8 v0, v1;
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              v0[4 * r + j] = f2h(o[j][r]);
              v1[4 * r + j] = f2h(o[j][2 + r]);
            }
          T* orow = out_row + head * kD;
          *reinterpret_cast<half8*>(orow) = v0;
          *reinterpret_cast<half8*>(orow + 8) = v1;
        } else {
          T* orow = out_row + head * kD;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            typedef T out4 __attribute__((ext_vector_type(4)));
            out4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (T)o[dt][r];
            if (out.form == AttentionOut::kSplit) store_split<4>(reinterpret_cast<uint16_t*>(out_row), head * kD + dt * 16 + g * 4, v);
            else *reinterpret_cast<out4*>(orow + dt * 16) = v;
          }
        }
      }
    }
  }
}

#undef ET_ATTN_LOAD_HEAD

template <typename T, int NKT>
void attention_launch(const void* q, const void* k, const void* v, int layout, int packed_ld, const void* attr_mask,
                      void* dst, const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len, int heads,
                      float scaler, AttentionOut out, HeadExps head_exp, hipStream_t stream) {
  using Sm = AttnSmem<T, NKT>;
  constexpr int kCpr = kD * (int)sizeof(T) / 16;
  constexpr int WAVES = 4;
  constexpr int kThreads = WAVES * kWave;
  constexpr int CPT = (NKT * 16 * kCpr + kThreads - 1) / kThreads;
  static_assert(CPT <= 4, "the next head's chunks, 3 matrices of them, are kept in registers");
  auto kern = attention_kernel<T, NKT, WAVES, CPT>;
  allow_dynamic_lds(reinterpret_cast<const void*>(kern), (int)Sm::kBytes);
  // A workgroup serves several heads of one sequence: mask rows, positions and zero fill are shared by them, and the
  // chain of dependent loads a workgroup starts with (sequence start, positions, rows) is paid once.  Up to 6 heads
  // (4 in fp32), in equal groups, as long as about two workgroups per CU remain: measured best on batches of 100 x 32 and
  // 1000 x 64 tokens.
  int hpw = 1;
  for (int h = sizeof(T) == 2 ? 6 : 4; h > 1; --h)
    if (heads % h == 0 && (long)batch * (heads / h) >= 512) {
      hpw = h;
      break;
    }
  dim3 grid((heads + hpw - 1) / hpw, batch);
  AttnOut<T> form;
  form.form = out;
  if constexpr (sizeof(T) == 4) form.exp = head_exp.exp, form.exp_stride = head_exp.stride;
  kern<<<grid, kThreads, Sm::kBytes, stream>>>(seq_start, word_idx, batch, seq_len, heads, hpw, layout, packed_ld, (const T*)q,
                                               (const T*)k, (const T*)v, (const T*)attr_mask, (T*)dst, scaler, form);
}


// ------------------------------------------------------------------------------------------
// K / V rows brought into LDS by DMA (the streaming kernel below): rows of 128 bytes without padding, one
// `buffer_load ... lds` instruction fills eight of them (lane -> row lane / 8, 16-byte chunk lane & 7).  A row without
// a token is requested beyond its buffer descriptor's range and arrives as zeros.
// Which key a row of an MFMA tile stands for is free as long as K, the mask and V agree: row m of the first tile of a
// pair (32 keys from `base`) is key base + (m >> 2) * 8 + (m & 3), of the second tile 4 keys further.  A lane's scores
// of a pair are then 8 consecutive keys: one 16-byte load of its mask row, and the P operand of the P.V MFMA is in
// natural key order.  Key row `key` lies in slot key ^ ((key >> 3) & 1) (the two rows of a half-wave of the 8-byte V
// reads, 8 keys apart, land on different halves of the banks), and the 16-byte chunks of a slot are XOR-swizzled with
// slot bits 1, 3 and 4 (the 16 rows x one chunk of a K operand read cover all 64 banks).
// ------------------------------------------------------------------------------------------
#define ET_ATTN_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
__device__ __forceinline__ int wide_slot(int key) { return key ^ ((key >> 3) & 1); }
__device__ __forceinline__ int wide_swizzle(int slot) { return ((slot >> 1) & 1) | ((slot >> 2) & 6); }
// s_waitcnt immediates of gfx9: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] at [15:14]
__device__ __forceinline__ void wide_wait_dma() { __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8) | (0 << 14)); }
// barrier without the fence of __syncthreads(), which would wait for every DMA in flight
__device__ __forceinline__ void wide_barrier() { asm volatile("s_barrier" ::: "memory"); }

inline int attention_cu_count() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    return 256;
  return n;
}

// ------------------------------------------------------------------------------------------
// fp16 fused attention for 64 < seq_len <= 1024: one workgroup of 4 wavefronts per (64 QSUB queries, head, sequence),
// a wavefront serves QSUB tiles of 16 queries.  K and V stream through LDS in stages of 64 keys (two stages of 16 KB, the
// next one arriving by DMA under the work on this one), and the softmax runs along with them (a published method: Milakov and
// Gimelshein, 2018): per query the maximum so far, the sum and the output so far, rescaled where the maximum moves.  Nothing grows with the sequence, so several
// workgroups share a CU and fill each other's waits, and a stage's K and V operands serve all queries of a wavefront.
// Bound: VALU issue while it runs (a wavefront and stage of 64 keys x 32 queries: about 1060 cycles of VALU, exp2 at a quarter
// of the rate, against 576 of MFMA), and the start of a workgroup (order -> start table -> rows, then the first stage) over
// the one and a half rounds its grid takes (16 x 1024: 24 of 48 us without the stages' arithmetic).  Measured per launch,
// 12 heads: 8 x 128 positions / 570 tokens 5.4 us (11.3 us with one workgroup's four wavefronts serving a whole head, two
// query tiles each, and scores, mask and next rows in registers), 16 heads and 256 x 128 skewed 30 us (40 us), 16 x 1024 positions
// / 11200 tokens 46 us (172 us with K or V of a whole sequence in 128 KB of LDS, one workgroup per CU and the scores of a query
// in registers), 32 x 512 positions / 12300 tokens 32 us (60 us).  Deeper rings of stages, 8 wavefronts per workgroup or a bound
// of 3 wavefronts per SIMD: 1 to 5 % slower.
// Rounding points: the score to half, the exponentials to half for P.V and, as that product's row of ones, for their sum; sums
// in float, division last.  (The short kernel sums the exponentials before they are rounded, and rounds after the division.
// Relative error of the output against float64, this way and that way, normal operands: 80 positions 4.50e-4 and 4.69e-4, 512
// 5.25e-4 and 5.30e-4, 1024 5.34e-4 and 5.35e-4, 512 with scores nine times as wide 1.527e-3 and 1.534e-3.)
//
// Behind the stage of the last token K and V are zero, so nothing streams there: a score is the mask's bias alone, and a key
// without a value only enters the maximum and the sum (`Unseen`).  `mask_class` says of every block of 16 queries whether its
// mask rows are plain (1 up to the sequence's last token and 0 from there on: then no mask is read), and whether they are all 0
// or all 1 behind the last token; other rows, and those of a caller without classes, are read 64 keys at a time.  Per launch, 12
// heads, fp16, sequences of 16 .. 128 tokens in 32 x 512 positions: plain 13.6 us, causal 16.2, all ones 16.3, random behind
// the tokens 38 (47 each but the first with the stages run over all positions); 64 .. 384 tokens in 64 x 384, causal: 42 (54).
// ------------------------------------------------------------------------------------------
constexpr int kFlKeys = 64;                                  // keys per stage
constexpr int kFlStage = kFlKeys * 128;                      // bytes of K (and of V) per stage
constexpr int kFlWaves = 4;                                  // wavefronts of a workgroup, and per SIMD
constexpr int kFlMaxKeys = 1024;
// Up to 64 positions attention_kernel is the faster one: a head is a single stage there, so nothing streams, and its
// workgroups serve six heads for one start (12 layers, 1000 x 64: 7.79 ms with it, 7.98 ms with this kernel; 217 x 53 in
// single layer calls 2.24 and 2.32 ms).  Beyond, this kernel (12 layers: 8 x 128 from ids 0.67 -> 0.61 ms, 60 x 101
// 1.54 -> 1.25 ms, 300 x 128 7.08 -> 6.87 ms, 500 x 80 5.50 -> 5.47 ms; 24 layers, 256 x 128 skewed 8.63 -> 8.36 ms).
constexpr int kFlMinKeys = 64;
[[maybe_unused]] constexpr float kFlSlack = 10.f;                             // how far (log2) a score may exceed the exponents' reference
[[maybe_unused]] constexpr float kFlLowest = -3e38f;                          // the reference before the first stage; finite, so that scores of
                                                             // -infinity weigh nothing against it
typedef __fp16 half4_fp16 __attribute__((ext_vector_type(4)));
constexpr int kFlSmem = 2 * 2 * kFlStage + kFlMaxKeys * (int)sizeof(int);

// Keys without a value that have not been visited one by one enter the maximum (`lowest`, log2 units: what it is at least) and
// the sum against the exponent `ref` (`extra`; infinity where they leave nothing to the visited keys).  Masked with 0 their score
// is -10000: below 1024 positions, where the maximum is clamped at 0, they weigh exp(-10000 - maximum) = 0; at 1024 there is no
// clamp.  Masked with 1 their score is 0.
struct Unseen {
  float lowest, extra = 0.f;
  __device__ __forceinline__ explicit Unseen(int seq_len) : lowest(seq_len < kFlMaxKeys ? 0.f : -INFINITY) {}
  __device__ __forceinline__ void add_zeros(int seq_len, int keys, float ref) {
    if (seq_len < kFlMaxKeys || keys <= 0) return;
    lowest = fmaxf(lowest, -10000.0f * kLog2e);
    extra += (float)keys * __builtin_amdgcn_exp2f(__builtin_fmaf(-10000.0f, kLog2e, -ref));
  }
  __device__ __forceinline__ void add_ones(int keys, float ref) {
    if (keys <= 0) return;
    lowest = fmaxf(lowest, 0.f);
    extra += (float)keys * __builtin_amdgcn_exp2f(-ref);
  }
};
typedef uint32_t uint4x __attribute__((ext_vector_type(4)));

// The work of workgroup `slot` of XCD `xcd`: a (sequence, head, block of `queries` queries).  Pairs of sequence (in the table's order, the
// longest first) and head are dealt round-robin to the XCDs, whose L2 then fetches a pair's K and V once for all its blocks:
// pair = 8 * (slot / q_blocks) + xcd.
//
// PLACED launches: an XCD hands its workgroups to its shader engines strictly in turn, and one that ends at once leaves its place empty until
// the turn comes round again: so the blocks behind a sequence's tokens come last (they hold queries only where the mask has
// holes).  16 x 1024 positions, 11200 tokens, 12 heads: 3.3 -> 4 workgroups on a CU while there are any, 16 .. 71 -> 49 .. 62 stages
// of keys a CU (12 layers 2776 -> 2753 us, fp32 15 x 379 2902 -> 2889; 6 layers of 16 heads, 64 x 512 with 32 .. 128 tokens 1144 -> 1061).
// Launches that are not placed find their pair and leave in the kernel itself: through this function they started later
// (12 layers of 1 x 1000 positions, fp16, 624 -> 628 us).
struct QueryBlock {
  int b, head, block, t0, t1;
};
constexpr int kPlacedBatch = kWave;        // sequences, one to a lane (more have not been tried)
// More workgroups than four on every CU (fewer all start at once: 8 x 128 positions +0.7 % with it), and, as the kernel finds, about
// 15 % of them without queries: a workgroup starts up to a microsecond later for it, with vector loads where the other way has
// scalar ones (32 x 512 positions, 12 % without queries, +0.5 %).
inline bool query_blocks_placed(int batch, int heads, int q_blocks) {
  return q_blocks > 1 && batch <= kPlacedBatch && (long)batch * heads * q_blocks > 4L * attention_cu_count();
}
__device__ __forceinline__ QueryBlock query_block(const int32_t* __restrict__ seq_start, int batch, int heads, int pair, int block) {
  const int place = uniform_div(pair, heads), b = min(max(seq_start[batch + 1 + place], 0), batch - 1);
  return {b, pair - place * heads, block, seq_start[b], seq_start[b + 1]};
}
// All of a wavefront's lanes; b < 0: nothing.
__device__ __forceinline__ QueryBlock placed_query_block(const int32_t* __restrict__ seq_start, int batch, int heads, int q_blocks, int queries,
                                                         int xcd, int slot) {
  QueryBlock w{-1, 0, 0, 0, 0};
  if (20 * (seq_start[batch] / queries) + 10 * batch < 17 * batch * q_blocks) {
    const int lane = threadIdx.x & (kWave - 1);
    const int b = min(max(seq_start[batch + 1 + min(lane, batch - 1)], 0), batch - 1);
    const int t0 = seq_start[b], t1 = seq_start[b + 1];
    // this XCD's pairs of the lane's sequence: 8 i + xcd from lane * heads on
    const int first = (lane * heads - xcd + 7) >> 3, pairs = lane < batch ? (((lane + 1) * heads - xcd + 7) >> 3) - first : 0;
    const int full = t1 > t0 ? min((t1 - t0 + queries - 1) / queries, q_blocks) : 0;
    const int upto = wave_inclusive_scan_i32(pairs * full), total = __builtin_amdgcn_readlane(upto, kWave - 1);
    const bool behind = slot >= total;
    const int blocks = behind ? q_blocks - full : full;
    const int end = behind ? total + wave_inclusive_scan_i32(pairs * blocks) : upto;
    const uint64_t at = __ballot(slot < end);
    if (at == 0) return w;
    const int rank = __builtin_ctzll(at);
    const int in_rank = slot - (__builtin_amdgcn_readlane(end, rank) - __builtin_amdgcn_readlane(pairs * blocks, rank));
    const int per_pair = __builtin_amdgcn_readlane(blocks, rank), k = uniform_div(in_rank, per_pair);
    w.b = __builtin_amdgcn_readlane(b, rank);
    w.t0 = __builtin_amdgcn_readlane(t0, rank);
    w.t1 = __builtin_amdgcn_readlane(t1, rank);
    w.head = (__builtin_amdgcn_readlane(first, rank) + k) * 8 + xcd - rank * heads;
    w.block = in_rank - k * per_pair + (behind ? __builtin_amdgcn_readlane(full, rank) : 0);
    return w;
  }
  const int of_xcd = uniform_div(slot, q_blocks), pair = of_xcd * 8 + xcd;
  return pair < batch * heads ? query_block(seq_start, batch, heads, pair, slot - of_xcd * q_blocks) : w;
}

template <typename T>
__global__ __launch_bounds__(256) void mask_class_kernel(const T* __restrict__ attr_mask, const int32_t* __restrict__ seq_start,
                                                         const int32_t* __restrict__ word_idx, int seq_len, int blocks,
                                                         uint8_t* __restrict__ cls) {
  const int b = blockIdx.y, qb = blockIdx.x;
  mask_class_block(attr_mask, word_idx, b, qb, seq_start[b], seq_start[b + 1], seq_len, blocks, cls);
}

__device__ __forceinline__ int v_swizzle(int key) { return (((key >> 1) & 1) | ((key >> 2) & 2)) * 2; }
// 16 lanes read four rows of 16 halves (lane i: 8 bytes at row i / 4, halves 4 (i & 3) ..) and each gets one column
__device__ __forceinline__ half4 read_transposed(const unsigned char* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16(
                                       (__attribute__((address_space(3))) half4_fp16*)(p)));
#else
  return half4{};
#endif
}

template <int QSUB, bool PLACED>
__global__ __launch_bounds__(kFlWaves * kWave, 4) void attention_flash_kernel(
    const int32_t* __restrict__ seq_start, int batch, int heads, int q_blocks, int seq_len, int layout, int packed_ld,
    const _Float16* __restrict__ q_src, const _Float16* __restrict__ k_src, const _Float16* __restrict__ v_src,
    const int32_t* __restrict__ word_idx, const _Float16* __restrict__ attr_mask, const uint8_t* __restrict__ mask_class,
    _Float16* __restrict__ dst, float scaler) {
#if defined(__HIP_DEVICE_COMPILE__)   // device-only types in the body; the host pass only needs the stub
  using T = _Float16;
  typedef _Float16 half2x __attribute__((ext_vector_type(2)));
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  unsigned char* kv = smem_raw;                                        // [stage][K, V]
  int* tok_of_pos = reinterpret_cast<int*>(smem_raw + 2 * 2 * kFlStage);

  const int xcd = blockIdx.x & 7, slot_id = blockIdx.x >> 3;
  const int of_xcd = PLACED ? 0 : uniform_div(slot_id, q_blocks), pair = of_xcd * 8 + xcd;
  if (!PLACED && pair >= batch * heads) return;
  const QueryBlock work = PLACED ? placed_query_block(seq_start, batch, heads, q_blocks, 16 * kFlWaves * QSUB, xcd, slot_id)
                                 : query_block(seq_start, batch, heads, pair, slot_id - of_xcd * q_blocks);
  if (PLACED && work.b < 0) return;
  const int b = work.b, head = work.head, qblock = work.block, t0 = work.t0, t1 = work.t1;
  const int len = t1 - t0;
  if (len <= 0) return;
  const int H = heads * kD;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l16 = lane & 15, g = lane >> 4;

  const int first_q = qblock * 16 * kFlWaves * QSUB;
  const int q0 = first_q + wave * 16 * QSUB;                           // this wavefront's: tile u holds q0 + 16 u + l16

  // K / V rows of a stage by DMA: one instruction fills eight slots (lane -> slot 8 i + lane / 8, 16-byte chunk
  // (lane & 7) ^ swizzle).  A row without a token is requested beyond the descriptor's range and arrives as zeros.
  const T* kb = layout == 1 ? k_src + (size_t)t0 * packed_ld + head * kD : k_src + ((size_t)b * heads + head) * seq_len * kD;
  const T* vb = layout == 1 ? v_src + (size_t)t0 * packed_ld + head * kD : v_src + ((size_t)b * heads + head) * seq_len * kD;
  const T* qb = layout == 1 ? q_src + (size_t)t0 * packed_ld + head * kD : q_src + ((size_t)b * heads + head) * seq_len * kD;
  const uint32_t ld = layout == 1 ? (uint32_t)packed_ld : (uint32_t)kD;
  constexpr int kPer = 8 / kFlWaves;                                   // requests of a wavefront for K (and for V) per stage
  uint32_t voff[kPer], voff_v[kPer];
  int dma_key[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int slot = (wave * kPer + i) * 8 + (lane >> 3);
    dma_key[i] = wide_slot(slot);
    voff[i] = ((uint32_t)dma_key[i] * ld + (uint32_t)((lane & 7) ^ wide_swizzle(slot)) * 8u) * 2u;
    // V is read transposed, four rows x 32 bytes by 16 lanes: rows in key order, pairs of chunks XORed with key bits 1 and 3
    voff_v[i] = ((uint32_t)slot * ld + (uint32_t)((lane & 7) ^ v_swizzle(slot)) * 8u) * 2u;
  }
  // `rows`: of the matrices behind kb, vb that exist
  auto issue = [&](int slot, int st, bool dense, int rows) {
    unsigned char* base = kv + slot * 2 * kFlStage;
    const int bytes = (int)(((uint32_t)(rows - 1) * ld + kD) * 2u);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(kb), 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(vb), 0, bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      uint32_t off = voff[i], off_v = voff_v[i];
      uint32_t stage_off = (uint32_t)st * kFlKeys * ld * 2u;
      if (!dense) {
        auto place = [&](uint32_t o, int in_stage) -> uint32_t {       // the row of key `in_stage` of the stage, or nowhere
          const int key = st * kFlKeys + in_stage;
          const int tk = key < kFlMaxKeys ? tok_of_pos[key] : -1;
          const uint32_t row = layout == 1 ? (uint32_t)tk : (uint32_t)key;
          return tk >= 0 ? o + (row - (uint32_t)in_stage) * ld * 2u : 0x80000000u;
        };
        off = place(off, dma_key[i]);
        off_v = place(off_v, (wave * kPer + i) * 8 + (lane >> 3));
        stage_off = 0;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, ET_ATTN_LDS_PTR(base + (wave * kPer + i) * 1024), 16, off, stage_off, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, ET_ATTN_LDS_PTR(base + kFlStage + (wave * kPer + i) * 1024), 16, off_v, stage_off, 0, 0);
    }
  };
  half8 bq[QSUB][2];
  auto load_q = [&](bool dense, int n) {
#pragma unroll
    for (int u = 0; u < QSUB; ++u) {
      const int q = q0 + u * 16 + l16;
      const int tq = q < n ? (dense ? q : tok_of_pos[q]) : -1;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int j = 0; j < 8; ++j) bq[u][ks][j] = (_Float16)0;
        if (tq >= 0)
          bq[u][ks] = *reinterpret_cast<const half8*>(qb + (size_t)(layout == 1 ? tq : q) * ld + ks * 32 + g * 8);
      }
    }
  };

  // Without a hole in the sequence, position p holds token p: the first stage and the queries are requested on that
  // assumption, in one step of the chain of dependent loads with what decides it.
  if (first_q < len) {
    issue(0, 0, true, len);
    load_q(true, len);
  }
  const int n = min(max(word_idx[t1 - 1], 0), seq_len - 1) + 1;        // positions up to the last token
  // the workgroup's blocks of 16 queries all plain: uniform over the workgroup
  const int cblocks = (seq_len + 15) / 16;
  bool plain = false;
  uint32_t zeros_behind = 0, ones_behind = 0;                          // bit i: its block i
  if (mask_class != nullptr) {
    const int c = first_q / 16 + lane;                                 // one class per lane, all of them in one request
    const int got = mask_class[(size_t)b * cblocks + min(c, cblocks - 1)];     // (which does not wait for n)
    const int cl = lane < kFlWaves * QSUB && c * 16 < n ? got : kMaskPlain | kMaskZeros;
    plain = __all(cl & kMaskPlain);
    zeros_behind = (uint32_t)__ballot(cl & kMaskZeros);
    ones_behind = (uint32_t)__ballot(cl & kMaskOnes);
  }
  const bool dense = n == len;
  const bool active = q0 < n;                                          // wave-uniform
  const int stages = (n + kFlKeys - 1) / kFlKeys;
  if (!dense) {
    wide_wait_dma();
    __syncthreads();
    if (first_q >= n) return;                                          // no token among this workgroup's queries
    for (int i = threadIdx.x; i < kFlMaxKeys; i += kFlWaves * kWave) tok_of_pos[i] = -1;
    __syncthreads();
    for (int tt = threadIdx.x; tt < len; tt += kFlWaves * kWave) {
      const int pos = word_idx[t0 + tt];
      if (pos >= 0 && pos < seq_len) tok_of_pos[pos] = tt;             // relative to the sequence's first packed row
    }
    __syncthreads();
    issue(0, 0, false, layout == 1 ? len : n);
    load_q(false, n);
  } else if (first_q >= n) {
    return;                                                            // (nothing has been requested)
  }

  // the queries are waited for here: left pending, they would have the compiler put a wait for every outstanding request,
  // the DMA included, into the stage loop
#pragma unroll
  for (int u = 0; u < QSUB; ++u)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) asm volatile("" : "+v"(bq[u][ks]));

  // operand addresses (see above): a lane constant plus a compile-time offset per pair of key tiles
  int k_rd[2], v_rd[4];
  {
    const int L = wide_slot((l16 >> 2) * 8 + (l16 & 3));
    const int sw = wide_swizzle(L);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) k_rd[ks] = L * 128 + (((ks * 4 + g) ^ sw) * 16);
    // V, transposed read of feature tile dt: the lane's 8 bytes are key g * 8 + l16 / 4, features dt * 16 + (l16 & 3) * 4
    const int key = g * 8 + (l16 >> 2);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      v_rd[dt] = kFlStage + key * 128 + (((dt * 2 + ((l16 >> 1) & 1)) ^ v_swizzle(key)) * 16) + (l16 & 1) * 8;
  }

  // Per query: `ref`, the exponent (log2) its probabilities are taken against, is the maximum of the first stage, moved up
  // only when a score exceeds it by more than kFlSlack (a probability may then reach 2^kFlSlack, far inside half's range,
  // with the same relative precision); `top` is this lane's share of the true maximum.  The sum of the probabilities is
  // one more row of the P.V product (a V^T row of ones).
  float ref[QSUB], top[QSUB];
  float4v o[QSUB][4], l[QSUB];
#pragma unroll
  for (int u = 0; u < QSUB; ++u) {
    ref[u] = kFlLowest;
    top[u] = -INFINITY;
    l[u] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[u][dt] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  const float c_exp = scaler * kLog2e;
  const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(attr_mask + (size_t)b * seq_len * seq_len), 0, seq_len * seq_len * 2, 0x00020000);
  uint32_t mask_row[QSUB];
#pragma unroll
  for (int u = 0; u < QSUB; ++u) mask_row[u] = (uint32_t)min(q0 + u * 16 + l16, seq_len - 1) * (uint32_t)seq_len * 2u;
  half8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (_Float16)1.0f;

  // eight mask values from byte `off` of the sequence's mask; 0 behind the mask
  auto load_mask = [&](uint32_t off) -> half8 {
    half8 mk;
    if ((seq_len & 7) == 0) {
      mk = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(rm, off, 0, 0));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) mk[j] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(rm, off + 2u * j, 0, 0));
    }
    return mk;
  };
  // moves a query's reference up to its lanes' maximum `mx`, where that is far enough above it; returns the factor of what has
  // been summed against the old one
  auto move_ref = [&](int u, float mx) -> float {
    const float up = xor_lanes_16_32_max(mx);
    const float next = up > ref[u] + kFlSlack ? up : ref[u];           // the same in all lanes of a query
    float alpha = __builtin_amdgcn_exp2f(ref[u] - next);
    ref[u] = next;
    asm volatile("s_nop 7" : "+v"(alpha));          // wait states the compiler does not add for the instructions below
    // (in place by hand: the compiler would give the products registers of their own and copy all of them on the way
    // around this block)
    auto scale = [&](float4v& v) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = v[r];
        asm volatile("v_mul_f32 %0, %1, %0" : "+v"(x) : "v"(alpha));
        v[r] = x;
      }
    };
    scale(l[u]);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) scale(o[u][dt]);
    return alpha;
  };

  auto stage = [&](auto PLAINc, int st, int slot) {
    constexpr bool PLAIN = decltype(PLAINc)::value;
    const unsigned char* base = kv + slot * 2 * kFlStage;
    const int key_base = st * kFlKeys + g * 8;                         // this lane's keys: + 32 pair + 0 .. 7
    // ---- S^T = K Q^T: the lane gets 8 consecutive keys per pair of key tiles, rounded to half ----------------------
    half8 sc[QSUB][2];
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        half8 a[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) a[ks] = *reinterpret_cast<const half8*>(base + k_rd[ks] + (pr * 32 + t * 4) * 128);
#pragma unroll
        for (int u = 0; u < QSUB; ++u) {
          float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks], bq[u][ks], acc, 0, 0, 0);
          const half4 h = __builtin_convertvector(acc, half4);
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[u][pr][t * 4 + r] = h[r];
        }
      }
    half8 p[QSUB][2];
#pragma unroll
    for (int u = 0; u < QSUB; ++u) {
      float mx, e[2][8];                                               // mx: of this lane's keys, in log2 units
      if constexpr (PLAIN) {
        if ((st + 1) * kFlKeys > n) {                                  // workgroup-uniform: the last, partial stage
          int key_base = st * kFlKeys + g * 8;
          asm volatile("" : "+v"(key_base));                           // (keeps the comparisons in this block)
#pragma unroll
          for (int pr = 0; pr < 2; ++pr)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (key_base + pr * 32 + j >= n) sc[u][pr][j] = (_Float16)-INFINITY;
        }
        const half8 m8 = __builtin_elementwise_max(sc[u][0], sc[u][1]);
        const half2x m2 = __builtin_elementwise_max(__builtin_elementwise_max(half2x{m8[0], m8[1]}, half2x{m8[2], m8[3]}),
                                                    __builtin_elementwise_max(half2x{m8[4], m8[5]}, half2x{m8[6], m8[7]}));
        mx = fmaxf((float)m2[0], (float)m2[1]) * c_exp;
      } else {
        // additive bias of the mask row: (1 - m) * -10000 as one fma (1 - m is exact in float for a half m)
        mx = -INFINITY;
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          const int k0 = key_base + pr * 32;
          const half8 mk = load_mask(mask_row[u] + (uint32_t)k0 * 2u);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            e[pr][j] = k0 + j < seq_len ? h2f(sc[u][pr][j]) * scaler + __builtin_fmaf((float)mk[j], 10000.0f, -10000.0f) : -INFINITY;
            mx = fmaxf(mx, e[pr][j]);
          }
        }
        mx *= kLog2e;
      }
      top[u] = fmaxf(top[u], mx);
      if (__any(mx > ref[u] + kFlSlack)) move_ref(u, mx);              // the first stage, and seldom after it
#pragma unroll
      for (int pr = 0; pr < 2; ++pr)
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          float2v w;
#pragma unroll
          for (int i = 0; i < 2; ++i)
            w[i] = __builtin_amdgcn_exp2f(PLAIN ? __builtin_fmaf(h2f(sc[u][pr][j + i]), c_exp, -ref[u])
                                                : __builtin_fmaf(e[pr][j + i], kLog2e, -ref[u]));
          const half2x h = __builtin_convertvector(w, half2x);
          p[u][pr][j] = h[0];
          p[u][pr][j + 1] = h[1];
        }
    }
    // ---- O^T += V^T P^T, a pair of key tiles (one MFMA k range) at a time: the transposed reads give the lane features
    // dt * 16 + l16 of keys g * 8 .. + 3 and + 4 .. + 7 ------------------------------------------------------------
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
#pragma unroll
      for (int u = 0; u < QSUB; ++u) l[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, p[u][pr], l[u], 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const half4 lo = read_transposed(base + v_rd[dt] + pr * 32 * 128), hi = read_transposed(base + v_rd[dt] + (pr * 32 + 4) * 128);
        const half8 vt = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int u = 0; u < QSUB; ++u) o[u][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vt, p[u][pr], o[u][dt], 0, 0, 0);
      }
    }
  };

  auto run = [&](auto PLAINc) {
    for (int st = 0; st < stages; ++st) {
      wide_wait_dma();                                                 // this wavefront's share of the stage has landed,
      wide_barrier();                                                  // everybody's has, and the other slot is free
      // (the last stage is loaded once more behind it: a condition here costs the loop registers, 256 x 128 28.5 -> 30.4 us)
      issue((st + 1) & 1, min(st + 1, stages - 1), dense, layout == 1 ? len : n);
      if (active) stage(PLAINc, st, st & 1);
    }
  };
  // (expected, so that the plain loop's code runs straight into the end: 8 x 128 5.6 -> 5.4 us, and nothing is spilled)
  if (__builtin_expect(plain, 1)) run(std::true_type{});
  else run(std::false_type{});
  wide_wait_dma();                                                     // no DMA may still target this workgroup's LDS when it ends

  // What follows starts from the lane number once more, hidden from the compiler: a register that lives through the stage loop
  // for it would be spilled, and its reload waited for at the end of every workgroup (0.7 us).
  int ln = lane_id();
  asm volatile("" : "+v"(ln));
#pragma unroll
  for (int u = 0; u < QSUB; ++u) {
    const int q = q0 + u * 16 + (ln & 15), g = ln >> 4;
    const int tq = q < n ? (dense ? q : tok_of_pos[q]) : -1;
    // the keys behind the last token's stage: no rows, the mask alone
    Unseen unseen(seq_len);
    const int keys = seq_len - stages * kFlKeys;
    if (__builtin_expect(plain, 1)) {
      unseen.add_zeros(seq_len, seq_len - n, ref[u]);
    } else if (zeros_behind >> (wave * QSUB + u) & 1) {
      unseen.add_zeros(seq_len, keys, ref[u]);
    } else if (ones_behind >> (wave * QSUB + u) & 1) {
      unseen.add_ones(keys, ref[u]);
    } else if (active) {
      const uint32_t mask_row = (uint32_t)min(q, seq_len - 1) * (uint32_t)seq_len * 2u;
      int zeros = 0;
      float sum = 0.f;                                                 // of this lane's keys
#pragma unroll 1
      for (int first = stages * kFlKeys; first < seq_len; first += kFlKeys) {
        half8 mk[2];
        uint32_t not_zero = 0;
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          mk[pr] = load_mask(mask_row + (uint32_t)(first + pr * 32 + g * 8) * 2u);
          const uint4x w = __builtin_bit_cast(uint4x, mk[pr]);
          not_zero |= first + pr * 32 + g * 8 < seq_len ? w[0] | w[1] | w[2] | w[3] : 0;
        }
        if (!__any(not_zero != 0)) {
          zeros += min(kFlKeys, seq_len - first);
          continue;
        }
        float mx = -INFINITY;
        auto bias = [&](int pr, int j) {
          return first + pr * 32 + g * 8 + j < seq_len ? __builtin_fmaf((float)mk[pr][j], 10000.0f, -10000.0f) : -INFINITY;
        };
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, bias(j >> 3, j & 7));
        mx *= kLog2e;
        top[u] = fmaxf(top[u], mx);
        if (__any(mx > ref[u] + kFlSlack)) sum *= move_ref(u, mx);
#pragma unroll
        for (int j = 0; j < 16; ++j) sum += __builtin_amdgcn_exp2f(__builtin_fmaf(bias(j >> 3, j & 7), kLog2e, -ref[u]));
      }
      unseen.extra = xor_lanes_16_32_sum(sum);
      unseen.add_zeros(seq_len, zeros, ref[u]);
    }
    // the reference divides by (sum of exp(score - maximum)) + 1e-6, its maximum clamped at 0 below 1024 keys: in units of
    // 2^ref that is the sum here + 1e-6 * 2^(maximum - ref)
    const float mx = fmaxf(xor_lanes_16_32_max(top[u]), unseen.lowest);
    const float inv = 1.0f / (l[u][0] + unseen.extra + 1e-6f * __builtin_amdgcn_exp2f(mx - ref[u]));
    if (tq < 0) continue;
    T* orow = dst + (size_t)(t0 + tq) * H + head * kD + g * 4;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) *reinterpret_cast<half4*>(orow + dt * 16) = __builtin_convertvector(o[u][dt] * inv, half4);
  }
#endif
}

void attention_flash_launch(const void* q, const void* k, const void* v, int layout, int packed_ld, const void* attr_mask,
                            const uint8_t* mask_class, void* dst, const int32_t* seq_start, const int32_t* word_idx,
                            int batch, int seq_len, int heads, float scaler, hipStream_t stream) {
  const int pairs8 = (batch * heads + 7) / 8 * 8;
  auto go = [&](auto qsub) {
    constexpr int QSUB = decltype(qsub)::value;
    const int queries = 16 * kFlWaves * QSUB, q_blocks = (seq_len + queries - 1) / queries;
    auto kern = query_blocks_placed(batch, heads, q_blocks) ? attention_flash_kernel<QSUB, true> : attention_flash_kernel<QSUB, false>;
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), kFlSmem);
    kern<<<pairs8 * q_blocks, kFlWaves * kWave, kFlSmem, stream>>>(
        seq_start, batch, heads, q_blocks, seq_len, layout, packed_ld, (const _Float16*)q, (const _Float16*)k, (const _Float16*)v, word_idx,
        (const _Float16*)attr_mask, mask_class, (_Float16*)dst, scaler);
  };
  // Two query tiles per wavefront halve the LDS reads per score; with few workgroups the CUs are better filled by twice as
  // many of one tile.
  if ((long)batch * heads * ((seq_len + 127) / 128) >= 2L * attention_cu_count()) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 1>{});
}

// ------------------------------------------------------------------------------------------
// fp32 fused attention for 32 < seq_len <= 1024, built like the kernel above: one workgroup of 4 wavefronts per (64 queries, head,
// sequence), 16 queries per wavefront, K and V in stages of 32 keys, the softmax along with them in floats.  The products run on
// the 16-bit matrix instructions with every float as the sum of three bfloat16 pieces (round_pair_bf16): six of the nine
// products of pieces, the others at most 2^-24 of the largest.  A float MFMA takes 16 times as long per product.
// The pieces of K and V are made once per workgroup: a thread brings eight floats of a key's K and of its V into registers under
// the stage in front, splits them and writes them to LDS in rows of 64 values per piece, laid out as in the fp16 kernel (which
// explains the order of the keys).
// Bound: a wavefront and stage issue 768 cycles of MFMA and about 950 of VALU (370 of them the split of K and V, 210 that of the
// probabilities, exp2 at a quarter of the rate), 24 KB of LDS reads; short sequences the start of a workgroup.  One stage in LDS
// and the next in registers take two barriers a stage, but leave room for four workgroups per CU.  15 x 379 positions / 3820
// tokens, 12 heads: 47.0 -> 32.0 us per launch against floats on v_mfma_f32_16x16x4_f32 (2048 cycles of MFMA a stage), 500 x 64 /
// 20375 tokens 64.8 -> 53.1 (33.1 and 59.8 where the result is left as pair rows).  32 queries per wavefront: 35 and 73 us; three
// wavefronts per SIMD instead of four: 34 and 60.
// Relative error against float64 (this / the float instructions), normal operands: 64 positions 1.59e-7 / 2.44e-7, 379 3.01e-7 /
// 4.00e-7, 1000 5.27e-7 / 6.47e-7; with scores nine times as wide 3.9e-7 / 6.4e-7, 6.2e-7 / 9.9e-7, 7.6e-7 / 1.14e-6.
//
// Three pieces are not every float: below 2^-110 the last one ends at 2^-133, the first one is infinite above 3.39e38, and an
// infinity leaves NaN.  A workgroup that meets such operands does its block once more with the float instructions (FLOATS):
//   V with bits below 2^-133;  Q with such bits, or of 2^60 and more (below that, K's bits below 2^-133 move a score by 2^-67);
//   a result that is not finite, which is what an operand without three pieces leaves, as do sums that overflow.
// Probabilities are split 2^24 times as large, where those down to v_exp_f32's smallest have all their bits.  All of it
// costs nothing that shows (in the layer 31.0 -> 31.2 and 59.1 -> 58.3 us a launch).  Where every block is done twice the launches
// take 76 and 111 us, 48 and 64 with the float instructions alone.
// ------------------------------------------------------------------------------------------
constexpr int kF32Keys = 32;                                 // keys per stage
constexpr int kF32Piece = kF32Keys * kD * 2;                 // bytes of a piece of K (and of V) per stage
// Up to 32 positions attention_kernel, whose workgroups serve several heads for one start.  What decides between the two is the
// number of sequences more than their length (per launch, 12 heads, this kernel second: 1000 x 16 32.2 and 51.3 us, 1000 x 31 52.9
// and 66.3, 100 x 20 9.3 and 9.4, but 200 x 32 19.1 and 17.0, 8 x 32 5.8 and 5.1); the rule goes by the
// length alone, as does what depends on it, the making of the mask's classes (mask_class_bytes).
constexpr int kF32MinKeys = 32;
[[maybe_unused]] constexpr float kF32TopQ = 0x1p60f, kF32Raise = 0x1p24f;
constexpr int kF32Smem = 2 * 3 * kF32Piece + (kFlMaxKeys + 4) * (int)sizeof(int);
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// eight floats as three pieces; `rest` collects what the third ones are made of, whose low 16 bits they do not hold
__device__ __forceinline__ void split_eight(float (&x)[8], uint4x (&piece)[3], uint32_t& rest) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i == 2) {
#pragma unroll
      for (int j = 0; j < 8; ++j) rest |= __builtin_bit_cast(uint32_t, x[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) piece[i][j] = round_pair_bf16(x[2 * j], x[2 * j + 1]);
  }
}
// a . b of three pieces each, smallest products first
template <typename F>
__device__ __forceinline__ void piece_products(F&& mfma) {
  mfma(1, 1); mfma(0, 2); mfma(2, 0); mfma(0, 1); mfma(1, 0); mfma(0, 0);
}

// FLOATS: on the float instructions; tid: threadIdx.x
template <bool PLACED, bool FLOATS>
__device__ __forceinline__ void flash_f32_block(
    int tid, const int32_t* __restrict__ seq_start, int batch, int heads, int q_blocks, int seq_len, int layout, int packed_ld,
    const float* __restrict__ q_src, const float* __restrict__ k_src, const float* __restrict__ v_src,
    const int32_t* __restrict__ word_idx, const float* __restrict__ attr_mask, const uint8_t* __restrict__ mask_class,
    float* __restrict__ dst, float scaler, AttentionOut out, HeadExps head_exp, unsigned char* smem_raw) {
#if defined(__HIP_DEVICE_COMPILE__)   // device-only types in the body; the host pass only needs the stub
  unsigned char* kv = smem_raw;                                        // [K, V][piece][key][64]
  int* tok_of_pos = reinterpret_cast<int*>(smem_raw + 2 * 3 * kF32Piece);
  int* votes = tok_of_pos + kFlMaxKeys;                                // a wavefront: its share is to be done again in floats

  const int xcd = blockIdx.x & 7, slot_id = blockIdx.x >> 3;
  const int of_xcd = PLACED ? 0 : uniform_div(slot_id, q_blocks), pair = of_xcd * 8 + xcd;
  if (!PLACED && pair >= batch * heads) return;
  const QueryBlock work = PLACED ? placed_query_block(seq_start, batch, heads, q_blocks, 64, xcd, slot_id)
                                 : query_block(seq_start, batch, heads, pair, slot_id - of_xcd * q_blocks);
  if (PLACED && work.b < 0) return;
  const int b = work.b, head = work.head, qblock = work.block, t0 = work.t0, t1 = work.t1;
  const int len = t1 - t0;
  if (len <= 0) return;
  const int H = heads * kD;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int l16 = lane & 15, g = lane >> 4;
  const int first_q = qblock * 64, q = first_q + wave * 16 + l16;

  const size_t first = layout == 1 ? (size_t)t0 * packed_ld + head * kD : ((size_t)b * heads + head) * seq_len * kD;
  const float *kb = k_src + first, *vb = v_src + first, *qb = q_src + first;
  const uint32_t ld = layout == 1 ? (uint32_t)packed_ld : (uint32_t)kD;

  // this thread's eight features of K and of V: key `my_key` of the stage; a row without a token is requested beyond the
  // descriptor's range and arrives as zeros
  const int my_key = tid >> 3, my_chunk = tid & 7;
  const uint32_t voff = ((uint32_t)my_key * ld + (uint32_t)my_chunk * 8u) * 4u;
  const uint32_t v_swap = (uint32_t)(my_key >> 1 & 1) * 16u;           // (see v_wr)
  float4v in[4];                                                       // K, V
  auto request = [&](int st, bool dense, int rows) {
    const int bytes = (int)(((uint32_t)(rows - 1) * ld + kD) * 4u);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kb), 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(vb), 0, bytes, 0x00020000);
    uint32_t off = voff, stage_off = (uint32_t)st * kF32Keys * ld * 4u;
    if (!dense) {                                                      // the row of the key, or nowhere
      const int key = st * kF32Keys + my_key;
      const int tk = key < kFlMaxKeys ? tok_of_pos[key] : -1;
      const uint32_t row = layout == 1 ? (uint32_t)tk : (uint32_t)key;
      off = tk >= 0 ? off + (row - (uint32_t)my_key) * ld * 4u : 0x80000000u;
      stage_off = 0;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      in[i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rk, off + 16u * i, stage_off, 0));
      in[2 + i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rv, off + (16u * i ^ v_swap), stage_off, 0));
    }
  };
  unsigned char* const k_wr = kv + wide_slot(my_key) * 128 + ((my_chunk ^ wide_swizzle(wide_slot(my_key))) * 16);
  // V is read transposed, four keys x four times four features 16 apart, so that a lane ends up with 16 consecutive features: chunks
  // are XORed with key bit 3, and key bit 1 swaps a chunk's halves (requested the other way round), which spreads a read over all banks
  unsigned char* const v_wr = kv + 3 * kF32Piece + my_key * 128 + ((my_chunk ^ (my_key >> 3 & 1)) * 16);
  // FLOATS: K's and V's rows of 64 floats, their 16-byte chunks XORed so that an operand read covers all banks
  auto write_floats = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ck = my_chunk * 2 + i, cv = my_chunk * 2 + (i ^ (my_key >> 1 & 1));
      *reinterpret_cast<float4v*>(kv + my_key * 256 + ((ck ^ ((my_key >> 3) * 4 + (my_key & 3))) * 16)) = in[i];
      *reinterpret_cast<float4v*>(kv + kF32Keys * 256 + my_key * 256 + ((cv ^ (my_key >> 3)) * 16)) = in[2 + i];
    }
  };
  uint64_t lossy = 0;                                                  // (of K they do not matter)
  auto write = [&] {
    if constexpr (FLOATS) {
      write_floats();
      return;
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      float x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = in[2 * m + (j >> 2)][j & 3];
      uint4x piece[3];
      uint32_t rest = 0;
      split_eight(x, piece, rest);
      if (m) lossy |= __ballot((rest & 0xffffu) != 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4x*>((m ? v_wr : k_wr) + i * kF32Piece) = piece[i];
    }
  };
  int tq;
  float4v q_in[4];                                                     // features 8 g .. and 32 + 8 g .. of the lane's query, FLOATS: 16 g ..
  auto request_q = [&](bool dense, int n) {
    tq = q < n ? (dense ? q : tok_of_pos[q]) : -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      q_in[i] = float4v{0.f, 0.f, 0.f, 0.f};
      const int at = FLOATS ? g * 16 + i * 4 : (i >> 1) * 32 + g * 8 + (i & 1) * 4;
      if (tq >= 0) q_in[i] = *reinterpret_cast<const float4v*>(qb + (size_t)(layout == 1 ? tq : q) * ld + at);
    }
  };

  // without a hole in the sequence position p holds token p: requested on that assumption beside what decides it
  if (first_q < len) {
    request(0, true, len);
    request_q(true, len);
  }
  const int n = min(max(word_idx[t1 - 1], 0), seq_len - 1) + 1;        // positions up to the last token
  const int cblocks = (seq_len + 15) / 16;
  bool plain = false;
  uint32_t zeros_behind = 0, ones_behind = 0;                          // as above
  if (mask_class != nullptr) {
    const int c = first_q / 16 + (lane & 3);
    const int got = mask_class[(size_t)b * cblocks + min(c, cblocks - 1)];
    const int cl = c * 16 < n ? got : kMaskPlain | kMaskZeros;
    plain = __all(cl & kMaskPlain);
    zeros_behind = (uint32_t)__ballot(cl & kMaskZeros);
    ones_behind = (uint32_t)__ballot(cl & kMaskOnes);
  }
  const bool dense = n == len;
  const bool active = first_q + wave * 16 < n;                                          // wave-uniform
  const int stages = (n + kF32Keys - 1) / kF32Keys;
  const int stage_rows = dense || layout == 1 ? len : n;               // of the matrices behind kb, vb that exist
  if (first_q >= n) return;                                            // no token among this workgroup's queries
  if (!dense) {
    for (int i = tid; i < kFlMaxKeys; i += kAttnThreads) tok_of_pos[i] = -1;
    __syncthreads();
    for (int tt = tid; tt < len; tt += kAttnThreads) {
      const int pos = word_idx[t0 + tt];
      if (pos >= 0 && pos < seq_len) tok_of_pos[pos] = tt;             // relative to the sequence's first packed row
    }
    __syncthreads();
    request(0, false, stage_rows);
    request_q(false, n);
  }
  uint4x bq[6];                                                        // [k-step][piece], or floats
  bool again_q = false;
  if constexpr (FLOATS) {
#pragma unroll
    for (int i = 0; i < 4; ++i) bq[i] = __builtin_bit_cast(uint4x, q_in[i]);
  } else {
    uint32_t rest_q = 0;
    float top_q = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[j] = q_in[2 * ks + (j >> 2)][j & 3];
        top_q = fmaxf(top_q, fabsf(x[j]));
      }
      uint4x piece[3];
      split_eight(x, piece, rest_q);
#pragma unroll
      for (int i = 0; i < 3; ++i) bq[ks * 3 + i] = piece[i];
    }
    again_q = __any((rest_q & 0xffffu) != 0 || top_q >= kF32TopQ);
  }

  // operand addresses, as in the fp16 kernel
  int k_rd[2], v_rd[4];
  {
    const int L = wide_slot((l16 >> 2) * 8 + (l16 & 3));
    const int sw = wide_swizzle(L);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) k_rd[ks] = L * 128 + (((ks * 4 + g) ^ sw) * 16);
    const int key = g * 8 + (l16 >> 2);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      v_rd[dt] = 3 * kF32Piece + key * 128 + ((((l16 & 3) * 2 + (dt >> 1)) ^ (key >> 3 & 1)) * 16) + (((dt & 1) ^ (key >> 1 & 1)) * 8);
  }

  float ref = kFlLowest, top = -INFINITY, l = 0.f;                     // as above; l: of this lane's keys
  float4v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = float4v{0.f, 0.f, 0.f, 0.f};
  const float c_exp = scaler * kLog2e;

  const float* mrow = attr_mask + ((size_t)b * seq_len + min(q, seq_len - 1)) * seq_len;

  auto load_mask = [&](int k0) -> float4v {                            // of keys k0 .. k0 + 3, 0 beyond the row
    float4v m4 = {0.f, 0.f, 0.f, 0.f};
    if ((seq_len & 3) == 0) {
      if (k0 < seq_len) m4 = *reinterpret_cast<const float4v*>(mrow + k0);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (k0 + r < seq_len) m4[r] = mrow[k0 + r];
    }
    return m4;
  };
  auto move_ref = [&](float mx) {                                      // as above
    const float up = xor_lanes_16_32_max(mx);
    const float next = up > ref + kFlSlack ? up : ref;                 // the same in all lanes of a query
    const float alpha = __builtin_amdgcn_exp2f(ref - next);
    ref = next;
    l *= alpha;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
  };

  auto stage = [&](auto PLAINc, int st) {
    constexpr bool PLAIN = decltype(PLAINc)::value;
    float4v acc[2];                                                    // keys 32 st + 8 g + 4 t + r
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
    if constexpr (FLOATS) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const unsigned char* row = kv + ((l16 >> 2) * 8 + t * 4 + (l16 & 3)) * 256;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4v a = *reinterpret_cast<const float4v*>(row + (((g * 4 + i) ^ l16) * 16)), b = __builtin_bit_cast(float4v, bq[i]);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc[t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int ks = 0; ks < (FLOATS ? 0 : 2); ++ks) {
      bf16x8 a[2][3];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 3; ++i) a[t][i] = *reinterpret_cast<const bf16x8*>(kv + k_rd[ks] + i * kF32Piece + t * 4 * 128);
      piece_products([&](int i, int j) {
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][i], __builtin_bit_cast(bf16x8, bq[ks * 3 + j]), acc[t], 0, 0, 0);
      });
      __builtin_amdgcn_sched_barrier(0);         // (six operands at a time, for their registers)
    }
    float s[8];                                                        // keys key0 .. key0 + 7
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = acc[j >> 2][j & 3];
    // the exponents' factor: log2 units of the plain scores, of the masked ones otherwise
    const bool no_mask = FLOATS ? plain : PLAIN;
    const float unit = no_mask ? c_exp : kLog2e;
    const int key0 = st * kF32Keys + g * 8;
    float mx = -INFINITY;
    if (no_mask) {
      if ((st + 1) * kF32Keys > n) {                                   // workgroup-uniform: the last, partial stage
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (key0 + j >= n) s[j] = -INFINITY;
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int k0 = key0 + t * 4;
        const float4v m4 = load_mask(k0);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[t * 4 + r] = k0 + r < seq_len ? s[t * 4 + r] * scaler + (1.0f - m4[r]) * -10000.0f : -INFINITY;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) mx = fmaxf(mx, s[j]);
    mx *= unit;
    top = fmaxf(top, mx);
    if (__any(mx > ref + kFlSlack)) move_ref(mx);                      // the first stage, and seldom after it
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j], unit, -ref));
      l += s[j];
    }
    if constexpr (FLOATS) {
      // tile dt's row m is feature 16 (m >> 2) + 4 dt + (m & 3), the chunk (l16 & ~3) + dt of a row
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              *reinterpret_cast<const float*>(kv + (kF32Keys + g * 8 + j) * 256 + ((((l16 & 12) + dt) ^ g) * 16) + (l16 & 3) * 4), s[j], o[dt], 0, 0, 0);
      return;
    }
    uint4x p[3];
    uint32_t rest_p = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] *= kF32Raise;
    split_eight(s, p, rest_p);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      bf16x8 v[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const half4 lo = read_transposed(kv + v_rd[dt] + i * kF32Piece), hi = read_transposed(kv + v_rd[dt] + i * kF32Piece + 4 * 128);
        v[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
      piece_products([&](int i, int j) {
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], __builtin_bit_cast(bf16x8, p[j]), o[dt], 0, 0, 0);
      });
    }
  };
  // this wavefront's LDS reads and writes are complete, and everybody's; requests may be on their way
  auto lds_barrier = [] {
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
    wide_barrier();
  };
  auto run = [&](auto PLAINc) {
    for (int st = 0; st < stages; ++st) {
      if (st > 0) lds_barrier();                                       // everybody has read the stage in front of this one
      write();
      lds_barrier();
      if (st + 1 < stages) request(st + 1, dense, stage_rows);
      if (active) stage(PLAINc, st);
    }
  };
  if (__builtin_expect(plain, 1)) run(std::true_type{});
  else run(std::false_type{});

  // the keys behind the last token's stage, as above
  Unseen unseen(seq_len);
  {
    const int keys = seq_len - stages * kF32Keys;
    if (__builtin_expect(plain, 1)) {
      unseen.add_zeros(seq_len, seq_len - n, ref);
    } else if (zeros_behind >> wave & 1) {
      unseen.add_zeros(seq_len, keys, ref);
    } else if (ones_behind >> wave & 1) {
      unseen.add_ones(keys, ref);
    } else if (active) {
      int zeros = 0;
#pragma unroll 1
      for (int first = stages * kF32Keys; first < seq_len; first += 64) {
        float4v m4[4];
        uint32_t not_zero = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          m4[i] = load_mask(first + i * 16 + g * 4);
          const uint4x w = __builtin_bit_cast(uint4x, m4[i]);
          not_zero |= w[0] | w[1] | w[2] | w[3];
        }
        if (!__any(not_zero != 0)) {
          zeros += min(64, seq_len - first);
          continue;
        }
        float high = -INFINITY;
        auto bias = [&](int i, int r) { return first + i * 16 + g * 4 + r < seq_len ? (1.0f - m4[i][r]) * -10000.0f : -INFINITY; };
#pragma unroll
        for (int j = 0; j < 16; ++j) high = fmaxf(high, bias(j >> 2, j & 3));
        high *= kLog2e;
        top = fmaxf(top, high);
        if (__any(high > ref + kFlSlack)) move_ref(high);
#pragma unroll
        for (int j = 0; j < 16; ++j) l += __builtin_amdgcn_exp2f(__builtin_fmaf(bias(j >> 2, j & 3), kLog2e, -ref));
      }
      unseen.add_zeros(seq_len, zeros, ref);
    }
  }

  const float mx = fmaxf(xor_lanes_16_32_max(top), unseen.lowest);
  const float sum = xor_lanes_16_32_sum(l) + unseen.extra;
  const float inv = 1.0f / (sum + 1e-6f * __builtin_amdgcn_exp2f(mx - ref)) * (FLOATS ? 1.0f : 1.0f / kF32Raise);
  // o[dt][r] is feature 16 g + 4 dt + r
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] *= inv;
  if (out == AttentionOut::kPairs) {
    store_head_pairs<true>(dst, tq < 0 ? -1 : t0 + tq, H, head, o, head_exp);
  } else if (tq >= 0) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const int col = head * kD + g * 16 + dt * 4;
      if (out == AttentionOut::kSplit) store_split<4>(reinterpret_cast<uint16_t*>(dst) + (size_t)(t0 + tq) * 3 * H, col, o[dt]);
      else *reinterpret_cast<float4v*>(dst + (size_t)(t0 + tq) * H + col) = o[dt];
    }
  }
  if constexpr (!FLOATS) {
    // Behind the stores (the second way's come from the same lanes, to the same places), and with what was seen of V in a scalar
    // register: 12 layers of 4 x 100 positions 1035 us without this look, 1042 with it in front of the stores and in a vector
    // register, 1035 as it is.
    float4v not_finite = {0.f, 0.f, 0.f, 0.f};                         // NaN where a result is not
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) not_finite[r] = __builtin_fmaf(o[dt][r], 0.f, not_finite[r]);
    const bool bad = tq >= 0 && !((not_finite[0] + not_finite[1]) + (not_finite[2] + not_finite[3]) == 0.f);
    const int vote = again_q || lossy != 0 || __any(bad);
    if (lane == 0) votes[wave] = vote;
    lds_barrier();                               // (behind it nobody reads K or V any more)
    const uint4x all = *reinterpret_cast<const uint4x*>(votes);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(all[0] | all[1] | all[2] | all[3]) != 0, 0)) {
      int own = wave * kWave + lane_id();        // (nothing of this way through is kept in registers for the other one)
      asm volatile("" : "+v"(own));
      flash_f32_block<PLACED, true>(own, seq_start, batch, heads, q_blocks, seq_len, layout, packed_ld, q_src, k_src, v_src, word_idx,
                                    attr_mask, mask_class, dst, scaler, out, head_exp, smem_raw);
    }
  }
#endif
}

template <bool PLACED>
__global__ __launch_bounds__(kAttnThreads, 4) void attention_flash_f32_kernel(
    const int32_t* __restrict__ seq_start, int batch, int heads, int q_blocks, int seq_len, int layout, int packed_ld,
    const float* __restrict__ q_src, const float* __restrict__ k_src, const float* __restrict__ v_src,
    const int32_t* __restrict__ word_idx, const float* __restrict__ attr_mask, const uint8_t* __restrict__ mask_class,
    float* __restrict__ dst, float scaler, AttentionOut out, HeadExps head_exp) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  flash_f32_block<PLACED, false>(threadIdx.x, seq_start, batch, heads, q_blocks, seq_len, layout, packed_ld, q_src, k_src, v_src, word_idx,
                                 attr_mask, mask_class, dst, scaler, out, head_exp, smem_raw);
}

void attention_flash_f32_launch(const void* q, const void* k, const void* v, int layout, int packed_ld, const void* attr_mask,
                                const uint8_t* mask_class, void* dst, const int32_t* seq_start, const int32_t* word_idx,
                                int batch, int seq_len, int heads, float scaler, AttentionOut out, HeadExps head_exp,
                                hipStream_t stream) {
  const int q_blocks = (seq_len + 63) / 64;
  const int grid = (batch * heads + 7) / 8 * 8 * q_blocks;
  auto kern = query_blocks_placed(batch, heads, q_blocks) ? attention_flash_f32_kernel<true> : attention_flash_f32_kernel<false>;
  kern<<<grid, kAttnThreads, kF32Smem, stream>>>(
      seq_start, batch, heads, q_blocks, seq_len, layout, packed_ld, (const float*)q, (const float*)k, (const float*)v, word_idx,
      (const float*)attr_mask, mask_class, (float*)dst, scaler, out, head_exp);
}

// ------------------------------------------------------------------------------------------
// fused attention for every shape the MFMA kernels above are not built for: size_per_head other than 64 (1 to 256
// elements), head rows off the 16-byte boundaries, and rows further apart than 31 bits reach.  One wavefront per (query, head): the lanes
// split the keys for the scores (full dot products in float, rounded to the element type as the reference stores
// them), the softmax runs on wave reductions, then the lanes split the features for P.V, skipping keys whose
// probability is 0.  Same arithmetic and rounding points as the other kernels; at seq_len = 1024 the reference's block
// of 1024 threads leaves no idle lane in its max reduction, so the clamp of the maximum at 0 disappears there
// (cuda/attention.cu:77-95, 267-270, 345-356: below 1024 the filler -1e-20 of the out-of-range threads acts as the clamp).
// ------------------------------------------------------------------------------------------
constexpr int kGenMaxSeq = 1024;
constexpr int kGenMaxD = 256;

template <typename T>
__global__ __launch_bounds__(kAttnThreads) void attention_generic_kernel(
    const T* __restrict__ q_src, const T* __restrict__ k_src, const T* __restrict__ v_src, int layout, int packed_ld,
    const T* __restrict__ attr_mask, T* __restrict__ dst, const int32_t* __restrict__ seq_start,
    const int32_t* __restrict__ word_idx, int batch, int seq_len, int heads, int d, int rows_16b, float scaler) {
  using C = Chunk16<T>;
  using V16 = typename C::vec;
  constexpr int kPerLane = kGenMaxSeq / kWave;             // keys per lane
  __shared__ int tok_of_pos[kGenMaxSeq];
  __shared__ float prob[kAttnWaves][kGenMaxSeq];
  __shared__ float qrow[kAttnWaves][kGenMaxD];

  const int b = min(max(seq_start[batch + 1 + blockIdx.z], 0), batch - 1), head = blockIdx.y;
  const int t0 = seq_start[b], t1 = seq_start[b + 1];
  const int len = t1 - t0;
  if (len <= 0) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int H = heads * d;
  for (int i = threadIdx.x; i < seq_len; i += kAttnThreads) tok_of_pos[i] = -1;
  __syncthreads();
  for (int tt = threadIdx.x; tt < len; tt += kAttnThreads) {
    const int pos = word_idx[t0 + tt];
    if (pos >= 0 && pos < seq_len) tok_of_pos[pos] = t0 + tt;
  }
  __syncthreads();
  const int q = blockIdx.x * kAttnWaves + wave;            // this wavefront's query position
  if (q >= seq_len) return;
  const int tq = tok_of_pos[q];
  if (tq < 0) return;                                      // no token: the reference drops this row
  auto src_off = [&](int t, int pos) -> size_t {
    return layout == 1 ? (size_t)t * packed_ld + head * d : (((size_t)b * heads + head) * seq_len + pos) * d;
  };
  for (int j = lane; j < d; j += kWave) qrow[wave][j] = (float)q_src[src_off(tq, q) + j];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // ---- scores of the lane's keys: key = lane + 64 i --------------------------------------------------------
  const T* mrow = attr_mask + ((size_t)b * seq_len + q) * seq_len;
  float t[kPerLane];
  float mx = seq_len < kGenMaxSeq ? 0.f : -INFINITY;       // the clamp at 0 holds below 1024 keys
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const int key = lane + i * kWave;
    t[i] = -INFINITY;
    if (key < seq_len) {
      const int tk = tok_of_pos[key];
      float dot = 0.f;
      if (tk >= 0) {
        const T* krow = k_src + src_off(tk, key);
        if (rows_16b) {                                    // wave-uniform: head rows of whole, aligned 16-byte pieces
          for (int c = 0; c < d; c += C::kElems) {
            const V16 kv = *reinterpret_cast<const V16*>(krow + c);
#pragma unroll
            for (int j = 0; j < C::kElems; ++j) dot += qrow[wave][c + j] * (float)kv[j];
          }
        } else {
          for (int c = 0; c < d; ++c) dot += qrow[wave][c] * (float)krow[c];
        }
      }
      const float sc = (float)(T)dot;                      // the score is stored in the element type
      t[i] = sc * scaler + (1.0f - (float)mrow[key]) * -10000.0f;
      mx = fmaxf(mx, t[i]);
    }
  }
  mx = wave_max(mx) * kLog2e;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    t[i] = __builtin_amdgcn_exp2f(t[i] * kLog2e - mx);     // exp2(-inf) = 0 for absent keys
    sum += t[i];
  }
  sum = wave_sum(sum) + 1e-6f;
  const float inv = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const int key = lane + i * kWave;
    if (key < seq_len) prob[wave][key] = (float)(T)(t[i] * inv);     // the probability is stored in the element type
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // ---- P.V: feature = lane + 64 i ------------------------------------------------------------------------------
  constexpr int kFeat = kGenMaxD / kWave;
  float acc[kFeat];
#pragma unroll
  for (int i = 0; i < kFeat; ++i) acc[i] = 0.f;
  for (int key = 0; key < seq_len; ++key) {
    const int tk = tok_of_pos[key];
    const float pk = prob[wave][key];
    if (tk < 0 || pk == 0.f) continue;                     // wave-uniform: a zero value or a zero weight
    const T* vrow = v_src + src_off(tk, key);
#pragma unroll
    for (int i = 0; i < kFeat; ++i) {
      const int j = lane + i * kWave;
      if (j < d) acc[i] += pk * (float)vrow[j];
    }
  }
#pragma unroll
  for (int i = 0; i < kFeat; ++i) {
    const int j = lane + i * kWave;
    if (j < d) dst[(size_t)tq * H + head * d + j] = (T)acc[i];
  }
}

// true when every head row of Q, K and V starts on a 16-byte boundary and is a whole number of 16-byte pieces (what the
// MFMA kernels and the vector loads of the generic one assume)
template <typename T>
bool head_rows_16b(const void* q, const void* k, const void* v, int layout, int packed_ld, int d) {
  const bool ptrs = ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) == 0;
  return ptrs && ((size_t)d * sizeof(T)) % 16 == 0 && (layout != 1 || ((size_t)packed_ld * sizeof(T)) % 16 == 0);
}

template <typename T>
void attention_generic_launch(const void* q, const void* k, const void* v, int layout, int packed_ld, const void* attr_mask,
                              void* dst, const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len,
                              int heads, int d, float scaler, hipStream_t stream) {
  dim3 grid((seq_len + kAttnWaves - 1) / kAttnWaves, heads, batch);
  attention_generic_kernel<T><<<grid, kAttnThreads, 0, stream>>>((const T*)q, (const T*)k, (const T*)v, layout, packed_ld,
                                                                 (const T*)attr_mask, (T*)dst, seq_start, word_idx, batch,
                                                                 seq_len, heads, d,
                                                                 head_rows_16b<T>(q, k, v, layout, packed_ld, d) ? 1 : 0,
                                                                 scaler);
}

template <typename T>
void attention_dispatch(const void* q, const void* k, const void* v, int layout, int packed_ld, const void* attr_mask,
                        void* dst, const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len, int heads,
                        int d, float scaler, AttentionOut out, const uint8_t* mask_class, HeadExps head_exp, hipStream_t stream) {
  // (the streaming kernels address the rows of a sequence with 31 bits)
  const bool far = (uint64_t)seq_len * (uint64_t)(layout == 1 ? packed_ld : kD) * sizeof(T) >= 0x80000000ull;
  if (d != kD || !head_rows_16b<T>(q, k, v, layout, packed_ld, d) || (far && seq_len > kF32MinKeys))
    attention_generic_launch<T>(q, k, v, layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch, seq_len, heads, d,
                                scaler, stream);
  else if (sizeof(T) == 2 && seq_len > kFlMinKeys)
    attention_flash_launch(q, k, v, layout, packed_ld, attr_mask, mask_class, dst, seq_start, word_idx, batch, seq_len, heads,
                           scaler, stream);
  else if (sizeof(T) == 4 && seq_len > kF32MinKeys)
    attention_flash_f32_launch(q, k, v, layout, packed_ld, attr_mask, mask_class, dst, seq_start, word_idx, batch, seq_len,
                               heads, scaler, out, head_exp, stream);
  else if (seq_len <= 32)
    attention_launch<T, 2>(q, k, v, layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch, seq_len, heads,
                           scaler, out, head_exp, stream);
  else if constexpr (sizeof(T) == 2)
    attention_launch<T, 4>(q, k, v, layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch, seq_len, heads,
                           scaler, out, head_exp, stream);
}

}  // namespace

void launch_qkv_bias_pad(DType t, const void* Q, const void* bQ, const void* K, const void* bK, const void* V,
                         const void* bV, void* q_buf, void* k_buf, void* v_buf, const int32_t* seq_start,
                         const int32_t* word_idx, int batch, int seq_len, int heads, int d, hipStream_t stream) {
  if (((size_t)d * elem_size(t)) % 16 != 0) {      // head rows that are no whole number of 16-byte pieces
    launch_qkv_bias_pad_generic(t, Q, bQ, K, bK, V, bV, q_buf, k_buf, v_buf, seq_start, word_idx, batch, seq_len, heads,
                                d, stream);
    return;
  }
  dim3 grid(batch, 3);
  if (t == DType::F32)
    qkv_bias_pad_kernel<float><<<grid, kPadThreads, 0, stream>>>(
        (const float*)Q, (const float*)bQ, (const float*)K, (const float*)bK, (const float*)V, (const float*)bV,
        (float*)q_buf, (float*)k_buf, (float*)v_buf, seq_start, word_idx, seq_len, heads, d);
  else
    qkv_bias_pad_kernel<_Float16><<<grid, kPadThreads, 0, stream>>>(
        (const _Float16*)Q, (const _Float16*)bQ, (const _Float16*)K, (const _Float16*)bK, (const _Float16*)V,
        (const _Float16*)bV, (_Float16*)q_buf, (_Float16*)k_buf, (_Float16*)v_buf, seq_start, word_idx, seq_len, heads,
        d);
}

void launch_softmax(DType t, void* qk, const void* attr_mask, int batch, int heads, int seq_len, float scaler,
                    hipStream_t stream) {
  const int rows = batch * heads * seq_len;
  const int grid = (rows + kSmThreads / kWave - 1) / (kSmThreads / kWave);
  if (t == DType::F32)
    softmax_kernel<float><<<grid, kSmThreads, 0, stream>>>((float*)qk, (const float*)attr_mask, rows, heads, seq_len,
                                                           scaler);
  else
    softmax_kernel<_Float16><<<grid, kSmThreads, 0, stream>>>((_Float16*)qk, (const _Float16*)attr_mask, rows, heads,
                                                              seq_len, scaler);
}

void launch_transpose_rm_padding(DType t, const void* src, void* dst, const int32_t* rows_dev, int rows_bound,
                                 int batch, int seq_len, int heads, int d, const int32_t* batch_idx,
                                 const int32_t* word_idx, hipStream_t stream) {
  (void)batch;
  if (((size_t)d * elem_size(t)) % 16 != 0) {
    launch_transpose_rm_padding_generic(t, src, dst, rows_dev, rows_bound, seq_len, heads, d, batch_idx, word_idx, stream);
    return;
  }
  const int cpd = (int)((size_t)d * elem_size(t) / 16);
  const long total = (long)rows_bound * heads * cpd;
  const int grid = (int)((total + 255) / 256);
  if (grid == 0) return;
  if (t == DType::F32)
    transpose_rm_padding_kernel<float><<<grid, 256, 0, stream>>>((const float*)src, (float*)dst, rows_dev, rows_bound,
                                                                 seq_len, heads, cpd, batch_idx, word_idx);
  else
    transpose_rm_padding_kernel<_Float16><<<grid, 256, 0, stream>>>((const _Float16*)src, (_Float16*)dst, rows_dev,
                                                                    rows_bound, seq_len, heads, cpd, batch_idx,
                                                                    word_idx);
}

bool attention_supported(DType t, int seq_len, int d) {
  (void)t;
  return d >= 1 && d <= kGenMaxD && seq_len >= 1 && seq_len <= kGenMaxSeq;
}

size_t mask_class_bytes(DType t, int batch, int seq_len, int d) {
  return d == kD && seq_len > (t == DType::F16 ? kFlMinKeys : kF32MinKeys) && seq_len <= kFlMaxKeys ? (size_t)batch * ((seq_len + 15) / 16) : 0;
}

size_t mask_class_bytes_max(int batch) { return (size_t)batch * (kFlMaxKeys / 16); }

void launch_mask_class(DType t, const void* attr_mask, const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len,
                       uint8_t* cls, hipStream_t stream) {
  const int blocks = (seq_len + 15) / 16;
  const dim3 grid(blocks, batch);
  if (t == DType::F32)
    mask_class_kernel<<<grid, 256, 0, stream>>>((const float*)attr_mask, seq_start, word_idx, seq_len, blocks, cls);
  else
    mask_class_kernel<<<grid, 256, 0, stream>>>((const _Float16*)attr_mask, seq_start, word_idx, seq_len, blocks, cls);
}

bool attention_writes_pieces(const void* q, const void* k, const void* v, int layout, int packed_ld, int d) {
  return d == kD && head_rows_16b<float>(q, k, v, layout, packed_ld, d);
}

void launch_attention(DType t, const void* q, const void* k, const void* v, int layout, int packed_ld,
                      const void* attr_mask, void* dst, const int32_t* seq_start, const int32_t* word_idx, int batch,
                      int seq_len, int heads, int d, float scaler, hipStream_t stream,
                      AttentionOut out, const uint8_t* mask_class, HeadExps head_exp) {
  if (t == DType::F32)
    attention_dispatch<float>(q, k, v, layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch, seq_len, heads, d,
                              scaler, out, mask_class, head_exp, stream);
  else
    attention_dispatch<_Float16>(q, k, v, layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch, seq_len,
                                 heads, d, scaler, AttentionOut::kPlain, mask_class, HeadExps(), stream);
}

}  // namespace et
