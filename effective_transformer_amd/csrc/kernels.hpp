// Internal launcher interface between the C ABI (et_api.cpp) and the gfx950 kernels.
// Every launcher enqueues on `stream` and returns; none allocates.  Row counts that live on
// the device are passed as `rows_dev` (may be null) next to a host-side upper bound.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace et {

enum class DType : int { F32 = 0, F16 = 1 };
inline size_t elem_size(DType t) { return t == DType::F32 ? 4 : 2; }

// Kernels that need more than 64 KB of dynamic LDS raise the limit once per (kernel, device): the attribute belongs
// to the device a module is loaded on, and a process may hold handles on several GPUs.  `bytes` is the most that any launch of
// the kernel takes: calls after the first change nothing.  (et_api.cpp)
void allow_dynamic_lds(const void* kernel, int bytes);
// The error of a failed allow_dynamic_lds on this thread since the last call (hipSuccess if none); clears it.
hipError_t take_attribute_error();

// A matrix of pair rows (gemm_pair.hip): n values per row as [n / 32][h, l][32] halves, the exponent of each row, and the
// row's Euclidean norm, from which what is computed of it is bounded.  Row arrays have room for 255 entries
// behind the last row (a tile reads them whole).
struct PairRows {
  _Float16* rows = nullptr;
  int32_t* exp = nullptr;
  float* norm = nullptr;             // (not of matrices that nothing is bounded by)
};
// ---- input_output.hip --------------------------------------------------------------------
// Number of int32 words of scratch the scan needs for `length` elements.
size_t scan_scratch_words(int length);
// What the scan of a mask can leave behind on its way, and what the compress launch behind it can (each nullable).
struct ScanExtras {
  int32_t* seq_start = nullptr;      // first half of the batch's sequence table (see launch_seq_start)
  int32_t* packed_row = nullptr;     // of every position: the row it is packed into, -1 if none
  uint64_t* host_word = nullptr;     // pinned host memory: host_tag << 32 | valid-token count, one 8-byte store
  uint32_t host_tag = 0;
};
struct CompressExtras {
  int32_t* seq_table = nullptr;      // the table whose first half the scan wrote: its second half is filled in
  uint16_t* split = nullptr;         // float rows of a multiple of 32 values: the packed rows once more as split rows
  PairRows pair;                     // ... or as pair rows (pair_rows_supported)
};
// Exclusive prefix sum of `in`; optionally (seq_len > 0) also writes batch_idx / word_idx for
// every element > 0 and the valid-token count.  prefix_out may be null.
void launch_scan_index(const int32_t* in, int length, int32_t* prefix_out, int32_t* batch_idx,
                       int32_t* word_idx, int32_t* valid_word_num, int seq_len, int32_t* scratch,
                       hipStream_t stream, const ScanExtras& extras = ScanExtras());
// batch_idx / word_idx from mask + an existing prefix sum.
void launch_index_from_prefix(const int32_t* mask, const int32_t* prefix, int32_t* batch_idx,
                              int32_t* word_idx, int batch, int seq_len, hipStream_t stream);
// to[t,:] = from[batch_idx[t]*S + word_idx[t], :] for t < T.  T comes from *rows_dev when given,
// otherwise from prefix[last] + (mask[last] == 1).
void launch_compress_rows(const void* from, void* to, const int32_t* batch_idx, const int32_t* word_idx,
                          const int32_t* rows_dev, const int32_t* prefix, const int32_t* mask,
                          int batch, int seq_len, int row_bytes, hipStream_t stream,
                          const CompressExtras& extras = CompressExtras());
// Chunks (16, 4 or 2 bytes: the widest piece row_bytes is a whole number of) the two movers below index for n_pos rows;
// must stay below 2^31.
size_t move_chunks(int n_pos, int row_bytes);
// to[B*S rows] = 0 at padding, from[t] at batch_idx[t]*S + word_idx[t]; indices ascending.
void launch_restore_rows(void* to, const void* from, const int32_t* batch_idx, const int32_t* word_idx,
                         const int32_t* rows_dev, int batch, int seq_len, int row_bytes, hipStream_t stream);
// The same where the packed row of every position is at hand (ScanExtras).
void launch_mapped_restore_rows(void* to, const void* from, const int32_t* packed_row, int n_pos, int row_bytes, hipStream_t stream);
// to[b,:] = packed row at position 0 of sequence b (zeros if there is none); indices ascending.
void launch_first_token(void* to, const void* from, const int32_t* batch_idx, const int32_t* word_idx,
                        const int32_t* rows_dev, int rows_bound, int batch, int row_bytes, hipStream_t stream);
// The sequence table of a batch, 2 B + 1 words: seq_start[b] = first packed row of sequence b, b in [0,B];
// seq_start[B] = T; then the B sequence numbers in the order the attention kernels serve them (longest first).
inline size_t seq_table_words(int batch) { return 2 * (size_t)batch + 1; }
void launch_seq_start(const int32_t* batch_idx, const int32_t* rows_dev, int rows_bound, int batch,
                      int32_t* seq_start, hipStream_t stream);
// second half of the table from its first half (for tables whose first half another kernel wrote)
void launch_seq_order(int32_t* seq_table, int batch, hipStream_t stream);

// What a layer that is called without them needs to know of its batch: the sequence table and the classes of its mask rows
// (either may be null).  Extra blocks of 256 threads in front of the launch that prepares the layer's weights; count_batch_jobs
// counts them; a table that one block cannot make needs launch_seq_order behind the launch.
struct BatchJobs {
  const int32_t* batch_idx = nullptr;
  const int32_t* word_idx = nullptr;
  const int32_t* rows_dev = nullptr;
  int rows_bound = 0, batch = 0, seq_len = 0;
  int32_t* seq_table = nullptr;
  const void* attr_mask = nullptr;
  uint8_t* cls = nullptr;
  int fp32 = 0;
  int table_blocks = 0, one_block_table = 0, blocks = 0;      // filled in
};
void count_batch_jobs(BatchJobs* jobs);

// ---- row_kernels.hip ---------------------------------------------------------------------
bool bias_gelu_supported(DType t, int n);
void launch_bias_gelu(DType t, void* out, const void* bias, int m, int n, const int32_t* rows_dev,
                      hipStream_t stream);
bool bias_residual_layernorm_supported(DType t, int n);
// rows the wave-per-row kernels keep in registers (n a multiple of 2 in fp16, up to 4096 elements)
bool layernorm_row_in_registers(DType t, int n);
// Regions whose 128-byte lines a kernel requests on its way (pulled into the last-level cache) for a later kernel that
// would otherwise read them cold.
struct WarmList {
  static constexpr int kMax = 3;
  const uint32_t* p[kMax] = {nullptr, nullptr, nullptr};
  int lines[kMax] = {0, 0, 0};
  int total = 0;
  void add(const void* region, size_t bytes);
};
void launch_bias_residual_layernorm(DType t, void* out, const void* input, const void* bias,
                                    const void* gamma, const void* beta, int m, int n,
                                    const int32_t* rows_dev, hipStream_t stream, const WarmList& warm = WarmList(),
                                    uint16_t* split = nullptr, const PairRows& pair = PairRows());
// split (fp32, rows in registers, n % 32 == 0): the output rows once more as split rows (see gemm_split.hip); pair: as pair
// rows (pair_rows_supported)

// out[t,:] = LayerNorm(word[ids[p]] + type[type_ids[p]] + pos[word_idx[t]]) * gamma + beta for packed row t at padded
// position p = batch_idx[t]*seq_len + word_idx[t]; eps 1e-12.  type_ids/type_table and pos_table may be null.
// n must satisfy bias_residual_layernorm_supported.
void launch_embed_layernorm(DType t, void* out, const int32_t* ids, const int32_t* type_ids, const int32_t* batch_idx,
                            const int32_t* word_idx, const void* word_table, int vocab, const void* type_table,
                            int type_vocab, const void* pos_table, int max_pos, const void* gamma, const void* beta,
                            int m, int n, int seq_len, const int32_t* rows_dev, hipStream_t stream,
                            const CompressExtras& extras = CompressExtras(), int batch = 0);

// ---- attention.hip -----------------------------------------------------------------------
void launch_qkv_bias_pad(DType t, const void* Q, const void* bQ, const void* K, const void* bK,
                         const void* V, const void* bV, void* q_buf, void* k_buf, void* v_buf,
                         const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len,
                         int heads, int d, hipStream_t stream);
void launch_softmax(DType t, void* qk, const void* attr_mask, int batch, int heads, int seq_len,
                    float scaler, hipStream_t stream);
void launch_transpose_rm_padding(DType t, const void* src, void* dst, const int32_t* rows_dev,
                                 int rows_bound, int batch, int seq_len, int heads, int d,
                                 const int32_t* batch_idx, const int32_t* word_idx, hipStream_t stream);
bool attention_supported(DType t, int seq_len, int d);
// What an fp32 launch leaves in dst; the others than float rows only where attention_writes_pieces says so.  kPairs: pair rows whose
// heads have an exponent each (gemm_pair.hip).
enum class AttentionOut { kPlain, kSplit, kPairs };
// [head][row], a byte each, with the bound of the rows rounded up to 4 as the stride; memory aligned to 4 bytes.
constexpr int kMaxHeadExps = 32;       // heads
inline int head_exp_stride(int rows) { return (rows + 3) / 4 * 4; }
struct HeadExps {
  int8_t* exp = nullptr;
  int stride = 0;
};
// layout 0: padded [B,heads,S,d]; layout 1: packed rows with leading dimension packed_ld.
void launch_attention(DType t, const void* q, const void* k, const void* v, int layout, int packed_ld,
                      const void* attr_mask, void* dst, const int32_t* seq_start, const int32_t* word_idx,
                      int batch, int seq_len, int heads, int d, float scaler, hipStream_t stream,
                      AttentionOut out = AttentionOut::kPlain, const uint8_t* mask_class = nullptr, HeadExps head_exp = HeadExps());
// Classes of the mask rows (one byte per 16 query positions of a sequence) for the kernel that makes use of them; the same
// array serves every layer of a batch.  0 bytes: the kernel of this shape has no use for them.
size_t mask_class_bytes(DType t, int batch, int seq_len, int d);
size_t mask_class_bytes_max(int batch);                // at any length
void launch_mask_class(DType t, const void* attr_mask, const int32_t* seq_start, const int32_t* word_idx, int batch, int seq_len,
                       uint8_t* cls, hipStream_t stream);
bool attention_writes_pieces(const void* q, const void* k, const void* v, int layout, int packed_ld, int d);

// ---- gemm.hip ----------------------------------------------------------------------------
// Up to three column groups share one launch (the Q/K/V projections): group g computes
// C[:, g*n : (g+1)*n] = A[g > 0] . B[g] (+ bias[g]) into a row-major C with leading dimension ldc;
// groups 1 and 2 share their A (K and V are made of the same rows).  groups == 1 is the plain GEMM.
struct GemmGroups {
  const void* A[2];                  // of group 0, of groups 1 and 2
  const void* B[3];
  const void* bias[3];
  int groups;
  // true: B[g] holds the transpose, [n][k] row-major (see launch_transpose_weights); only where
  // gemm_takes_transposed_b() says so
  bool b_transposed = false;
  // C = gelu(A.B + bias): bias + GELU as in launch_bias_gelu, same rounding points, applied to each tile on its way
  // out; bias[g] must be set
  bool gelu = false;
  // Hand-over of a wide intermediate between two launches of the persistent k-contiguous kernel (the FFN's [T, 4H]
  // matrix): the producer writes C, the consumer reads A, with every tile of 256 rows stored as consecutive blocks of
  // [256 rows][64 columns] (32 KB each) instead of row-major, so that the consumer's operand fetches, 128 bytes per row
  // and pair of k-steps, are contiguous in memory instead of one row stride apart.  Only where
  // gemm_blocked_handover() says so; the matrix must be allocated for a whole number of 256-row tiles.
  bool c_blocked = false, a_blocked = false;
  // C is read again by the next kernels while it can still be in the last-level cache (the working set of the layer
  // or of the call fits it a few times over): the persistent kernel then writes C through the L2s.  Its non-temporal
  // stores are the better choice when C would only push the weights and the A rows out of that cache.
  bool c_cached = false;
};
// any n, k >= 1 (the MFMA kernels need k % 32 == 0, n % 8 == 0 in fp16 and k % 16 == 0, n % 4 == 0 in fp32; other
// shapes run the element-wise kernel of generic.hip)
bool gemm_supported(DType t, int n, int k, int groups);
// True when both C = A.B1 ([m, wide] from k = narrow) and the product that consumes it (k = wide, n = narrow) run the
// persistent k-contiguous kernel, given k-contiguous copies of both weights.
bool gemm_blocked_handover(DType t, int m_bound, int wide, int narrow);
// The large-M fp16 kernel is faster when B comes k-contiguous ([n][k]): both operands then reach the
// MFMA with 128-bit LDS reads and no register transpose.  True when launch_gemm would use that kernel.
bool gemm_takes_transposed_b(DType t, int m_bound, int ldc, int n, int k, int groups);
// ... and where the encoder layer finds a per-call copy worth its time (everywhere it can be used).
bool gemm_prefers_transposed_b(DType t, int m_bound, int ldc, int n, int k, int groups);
// dst[j] ([n][k], row-major) = transpose of src[j] ([k][n], row-major), fp16, one launch for all jobs.
struct TransposeJobs {
  static constexpr int kMax = 6;
  const void* src[kMax];
  void* dst[kMax];
  int k[kMax], n[kMax];
  int count = 0;
  void add(const void* s, void* d, int k_, int n_) { src[count] = s; dst[count] = d; k[count] = k_; n[count] = n_; ++count; }
};
// `batch` (optional): the same launch makes what the layer needs to know of its batch.
void launch_transpose_weights(const TransposeJobs& jobs, hipStream_t stream, const BatchJobs* batch = nullptr);
void launch_gemm(DType t, const GemmGroups& g, void* C, int ldc, int m_bound, int n, int k,
                 const int32_t* rows_dev, hipStream_t stream);

// ---- gemm_split.hip: fp32 products on the 16-bit matrix cores -----------------------------------------------------
// Operands as split rows (6 k bytes per row, see gemm_split.hip): A [m], B [n] (k-contiguous weights).
// C is float [m][ldc] (+ bias), or with g.gelu the split rows of gelu(A.B + bias) (3 ldc bfloat16 per row).
bool gemm_split_supported(int n, int k);
// float [m][k] -> split rows; float weights [k][n] -> n split rows (k a multiple of 32, n of 4), one launch for all jobs
void launch_split_rows(const float* src, uint16_t* dst, int m, int k, const int32_t* rows_dev, hipStream_t stream);
void launch_split_weights(const TransposeJobs& jobs, hipStream_t stream);
void launch_gemm_split(const GemmGroups& g, void* C, int ldc, int m_bound, int n, int k, const int32_t* rows_dev,
                       hipStream_t stream);

// ---- gemm_pair.hip: fp32 products on the fp16 matrix cores, half the work of split rows ---------------------------
bool gemm_pair_supported(int n, int k);
bool pair_rows_supported(int n);
// float rows -> pair rows.  With batch_idx / word_idx: gathered from the padded tensor, the float rows go to `packed` too;
// seq_table: its second half is filled in on the way.
struct PairRowsJob {
  const float* src = nullptr;
  float* packed = nullptr;            // the packed rows as they are, with indices only (may be null)
  PairRows out;
  const int32_t *batch_idx = nullptr, *word_idx = nullptr;      // of the packed rows in the padded src; null: src is packed
  int m = 0, n = 0, seq_len = 0;
  const int32_t* rows_dev = nullptr;
  int32_t* seq_table = nullptr;       // starts of `batch` sequences; their order is added (see sort_sequences)
  int batch = 0;
};
void launch_pair_rows(const PairRowsJob& job, hipStream_t stream);
struct PairWeightJob {
  const void* src;                   // float [k][n], or (src_split) its n split rows
  bool src_split;
  int k, n;
  _Float16* dst;                     // n pair rows
  int32_t* exp;                      // n
  float* top;                        // scratch: pair_weight_tops(n, k) words
  const float* bias;                 // with stats: n
  // may be null; per 64 k and 64 n a bound of the columns' norms and the largest |bias|, then per 64 n the largest bias (or 0)
  float* stats;
};
inline size_t pair_weight_tops(int n, int k) { return (size_t)((k + 255) / 256) * n; }
inline size_t pair_weight_stat_pairs(int n, int k) { return (size_t)(k / 64) * ((n + 63) / 64); }
inline size_t pair_weight_stats(int n, int k) { return 2 * pair_weight_stat_pairs(n, k) + (n + 63) / 64; }
struct PairWeightJobs {
  static constexpr int kMax = 6;
  PairWeightJob job[kMax] = {};
  int count = 0;
};
// (`rows`: up to two jobs of launch_pair_rows that go along)
void launch_pair_weights(const PairWeightJobs& jobs, hipStream_t stream, const BatchJobs* batch = nullptr, const PairRowsJob* rows = nullptr,
                         int row_jobs = 0);
// C[:, g n : (g + 1) n] = A[g].B[g] + bias[g] (bias may be null), float with leading dimension ldc; with c_exp
// C = gelu(A.B + bias) as pair rows of ldc values, from A[0].norm and the weights' `stats`.
struct PairProduct {
  int groups = 1;
  PairRows A[3];
  const _Float16* B[3] = {};
  const int32_t* b_exp[3] = {};
  const float* bias[3] = {};
  const float* stats = nullptr;
  int32_t* c_exp = nullptr;
  // one group, C float, k up to 64 kMaxHeadExps: A's rows have an exponent per 64 k, and A[0].exp is not read
  const int8_t* head_exp = nullptr;
};
void launch_gemm_pair(const PairProduct& p, void* C, int ldc, int m_bound, int n, int k, const int32_t* rows_dev,
                      hipStream_t stream);

// ---- generic.hip: element-wise kernels for the shapes the tuned kernels do not take ------------------------------
// (rows or head rows that are no whole number of 16-byte pieces, GEMM k / n the MFMA tiles cannot take); the launchers
// above fall back to them by themselves.
void launch_gemm_generic(DType t, const GemmGroups& g, void* C, int ldc, int m_bound, int n, int k,
                         const int32_t* rows_dev, hipStream_t stream);
void launch_bias_gelu_generic(DType t, void* out, const void* bias, int m, int n, const int32_t* rows_dev,
                              hipStream_t stream);
void launch_layernorm_generic(DType t, void* out, const void* input, const void* bias, const void* gamma,
                              const void* beta, int m, int n, const int32_t* rows_dev, float eps, hipStream_t stream);
void launch_qkv_bias_pad_generic(DType t, const void* Q, const void* bQ, const void* K, const void* bK, const void* V,
                                 const void* bV, void* q_buf, void* k_buf, void* v_buf, const int32_t* seq_start,
                                 const int32_t* word_idx, int batch, int seq_len, int heads, int d, hipStream_t stream);
void launch_transpose_rm_padding_generic(DType t, const void* src, void* dst, const int32_t* rows_dev, int rows_bound,
                                         int seq_len, int heads, int d, const int32_t* batch_idx,
                                         const int32_t* word_idx, hipStream_t stream);

// ---- calibrate.hip: measurement aid ---------------------------------------------------------------------
// One launch of `iters` k-steps of the large fp16 GEMM's inner loop (MFMAs + LDS operand reads, no global memory) on
// `cus` workgroups of 8 wavefronts, with zero or random operands; returns the floating-point operations of the launch.
// `sink` receives one float per thread (mfma_ceiling_sink_bytes).
size_t mfma_ceiling_sink_bytes(int cus);
double launch_mfma_ceiling(bool random_operands, int cus, int iters, float* sink, hipStream_t stream);

}  // namespace et
