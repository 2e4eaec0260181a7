// C ABI of libet_hip.so: argument validation, workspace carve-up and launch order of the three
// ops (reference host side: tf_op/bert_transformer_op.cu.cc:33-373) plus the kernel-level entry
// points.  No call allocates device memory; a handle serialises its calls with a mutex like the
// reference's layer op does (tf_op/bert_transformer_op.cc:213).
#include "../../include/et.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "kernels.hpp"

namespace et {

namespace {
// A launcher cannot return a status; a failed attribute call is kept here until the entry point checks its launches.
thread_local hipError_t tls_attr_error = hipSuccess;
}  // namespace

void allow_dynamic_lds(const void* kernel, int bytes) {
  static std::mutex mu;
  static std::vector<std::pair<const void*, int>> done;      // (kernel, device) pairs already raised
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = -1;
  std::lock_guard<std::mutex> lock(mu);
  for (const auto& e : done)
    if (e.first == kernel && e.second == dev) return;
  const hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (err != hipSuccess) {
    tls_attr_error = err;          // reported as ET_RUNTIME_ERROR by the entry point; tried again on the next call
    return;
  }
  if (dev >= 0) done.emplace_back(kernel, dev);
}

hipError_t take_attribute_error() {
  const hipError_t e = tls_attr_error;
  tls_attr_error = hipSuccess;
  return e;
}

}  // namespace et

namespace {

// The persistent GEMM writes C through the L2s while the matrices of a layer (resp. A and C of a stand-alone call)
// are small enough to be found in the 256 MB last-level cache by the kernels that read them next, and with non-temporal
// stores beyond.  12-layer BERT-base, fp16: without non-temporal stores -6 % at 4000 tokens, -2.4 % at 15900, +-0.5 % at 20000,
// +2 % at 30000 and 40000; 24-layer BERT-large at 13100 tokens: -0.4 %.
constexpr double kCachedLayerBytes = 320.0 * 1048576.0;
constexpr double kCachedCallBytes = 96.0 * 1048576.0;
// While the layer's matrices stay below this, weights requested ahead of FFN-up survive until FFN-down reads them.
constexpr double kWarmLayerBytes = 256.0 * 1048576.0;

// Scratch of et_input_static: the tile totals of the mask scan (one int32 per tile of 1024 positions) for up to
// kStaticMaxPositions positions, in kStaticSlots independent slots.  A handle takes a free slot of its device when it
// is created and gives it back when it is destroyed, so that two handles never share tile totals; the handles beyond
// kStaticSlots per device have none.  Every GPU the library runs on holds its own copy of the array until the
// process ends.  In host code the array's name is only a handle for hipGetSymbolAddress: the address a kernel may use
// is looked up once per device (et_create) and kept in static_scratch_ptr.
constexpr int kStaticSlotWords = 1024;
constexpr int kStaticSlots = 8;
constexpr int kStaticMaxPositions = 1024 * 1024;
static __device__ __align__(256) int32_t scratch[kStaticSlots * kStaticSlotWords];

constexpr int kMaxDevices = 64;
std::mutex static_scratch_mu;
int32_t* static_scratch_ptr[kMaxDevices] = {};
unsigned static_slots_taken[kMaxDevices] = {};       // bit s: slot s of the device belongs to a live handle

// Looks up this device's copy of `scratch` (the device must be current).  Called by et_create.
hipError_t resolve_static_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(static_scratch_mu);
  if (static_scratch_ptr[device]) return hipSuccess;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  static_scratch_ptr[device] = static_cast<int32_t*>(p);
  return hipSuccess;
}

// A free slot of the device for a new handle, -1 when all are taken.
int take_static_slot(int device) {
  std::lock_guard<std::mutex> lock(static_scratch_mu);
  for (int s = 0; s < kStaticSlots; ++s)
    if (!(static_slots_taken[device] & (1u << s))) {
      static_slots_taken[device] |= 1u << s;
      return s;
    }
  return -1;
}

void release_static_slot(int device, int slot) {
  if (slot < 0 || device < 0 || device >= kMaxDevices) return;
  std::lock_guard<std::mutex> lock(static_scratch_mu);
  static_slots_taken[device] &= ~(1u << slot);
}

}  // namespace

struct et_context {
  int device = 0;
  std::mutex mu;                   // serialises the calls on this handle
  std::mutex err_mu;               // guards last_error alone: a failure may be recorded before `mu` is taken
  std::string last_error;          // the last failure on this handle by any thread
  // et_input_static: the handle's slot of the device's static scratch (-1: none), and the stream its calls are bound to
  int static_slot = -1;
  bool static_stream_set = false;
  hipStream_t static_stream = nullptr;
};

namespace {

// The calling thread's last failure and the handle it happened on (null: without a handle).  et_last_error prefers it,
// so a thread reads its own message whatever other threads do on the same handle in the meantime.
thread_local std::string tls_error;
thread_local et_handle tls_error_handle = nullptr;
thread_local std::string tls_error_copy;      // et_last_error's copy of another thread's message

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// The smallest buffer a sequence table is taken in.  et_seq_workspace_bytes asks for more: et_attention has the classes of the
// mask rows made behind the table where there is room for them.
inline size_t seq_table_bytes_min(int batch) { return align_up(et::seq_table_words(batch) * sizeof(int32_t), 256); }

et_status fail(et_handle h, et_status s, const std::string& msg) {
  std::string full = std::string("[ET][ERROR] ") + et_status_string(s) + ": " + msg;
  if (h) {
    std::lock_guard<std::mutex> lock(h->err_mu);
    h->last_error = full;
  }
  tls_error = std::move(full);
  tls_error_handle = h;
  return s;
}

et_status check_hip(et_handle h, hipError_t e, const char* what, const char* file, int line) {
  if (e == hipSuccess) return ET_OK;
  return fail(h, ET_RUNTIME_ERROR,
              std::string(what) + ": " + hipGetErrorString(e) + " " + file + ":" + std::to_string(line));
}

et_status check_launch(et_handle h, const char* what) {
  const hipError_t attr = et::take_attribute_error();
  if (attr != hipSuccess) {
    (void)hipGetLastError();
    return fail(h, ET_RUNTIME_ERROR, std::string(what) + ": raising the kernel's LDS limit failed: " + hipGetErrorString(attr));
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return ET_OK;
  return fail(h, ET_LAUNCH_FAILURE, std::string(what) + ": " + hipGetErrorString(e));
}

#define ET_HIP(h, call)                                                        \
  do {                                                                         \
    et_status _s = check_hip((h), (call), #call, __FILE__, __LINE__);          \
    if (_s != ET_OK) return _s;                                                \
  } while (0)

#define ET_REQUIRE(h, cond, msg)                                               \
  do {                                                                         \
    if (!(cond)) return fail((h), ET_INVALID_ARGUMENT, (msg));                 \
  } while (0)

bool dtype_ok(et_dtype d) { return d == ET_FP32 || d == ET_FP16; }
et::DType to_dt(et_dtype d) { return d == ET_FP32 ? et::DType::F32 : et::DType::F16; }

// How fp32 layers run their products: on pair rows (gemm_pair.hip) from 512 hidden values on, where they are closer to float64
// than split rows (k = 512: 1.22e-7 against 1.27e-7, wider: gemm_pair.hip) at half the work, up to the rows the row kernels hold
// in registers; on split rows (gemm_split.hip) at the other multiples of 32; the rest on the fp32 kernels.
bool layer_pairs(et_dtype dtype, int H) {
  return dtype == ET_FP32 && H >= 512 && et::pair_rows_supported(H) && et::gemm_pair_supported(H, 4 * H);
}
bool layer_splits(et_dtype dtype, int H) {
  return dtype == ET_FP32 && !layer_pairs(dtype, H) && H % 32 == 0 && et::gemm_split_supported(H, 4 * H);
}

struct LayerWs {
  size_t qkv, ctx, attn, attn_split, inter, seq, cls, wt, pair, total;
};

// Row arrays and weight arrays of a layer on pair rows, behind its matrices.
struct PairWs {
  int32_t *from_exp, *to_exp, *ctx_exp, *attn_exp, *inter_exp, *w_exp;      // w_exp: Q, K, V, output, up, down
  float *from_norm, *to_norm, *attn_norm, *up_stats, *tops;
};
size_t pair_array_rows(size_t rows) { return align_up(rows + 255, 256); }      // whole tiles of any height up to 256
size_t pair_ws_words(size_t rows, size_t H) {
  const int h = (int)H;
  return 8 * pair_array_rows(rows) + 9 * H + et::pair_weight_stats(4 * h, h) +
         8 * et::pair_weight_tops(h, h) + et::pair_weight_tops(h, 4 * h);
}
PairWs pair_ws(char* p, size_t rows, size_t H) {
  const size_t r = pair_array_rows(rows);
  int32_t* i = (int32_t*)p;
  PairWs w;
  w.from_exp = i; w.to_exp = i + r; w.ctx_exp = i + 2 * r; w.attn_exp = i + 3 * r; w.inter_exp = i + 4 * r;
  float* f = (float*)(i + 5 * r);
  w.from_norm = f; w.to_norm = f + r; w.attn_norm = f + 2 * r;
  w.w_exp = (int32_t*)(f + 3 * r);
  w.up_stats = (float*)(w.w_exp + 9 * H);
  w.tops = w.up_stats + et::pair_weight_stats(4 * (int)H, (int)H);
  return w;
}

LayerWs layer_ws(et_dtype dtype, int B, int S, int heads, int d) {
  const size_t e = dtype == ET_FP32 ? 4 : 2;
  const size_t rows = (size_t)B * S, H = (size_t)heads * d;
  const bool pairs = layer_pairs(dtype, heads * d), split = pairs || layer_splits(dtype, heads * d);
  const size_t ea = split && !pairs ? 6 : e;     // bytes of a value that only a product reads
  LayerWs w;
  size_t off = 0;
  w.qkv = off;   off += align_up(rows * 3 * H * e, 256);
  w.ctx = off;   off += align_up(rows * H * ea, 256);
  w.attn = off;  off += align_up(rows * H * e, 256);
  w.attn_split = off; off += split ? align_up(rows * H * ea, 256) : 0;
  // whole tiles of 256 rows: the FFN's intermediate may be handed over in blocks of [256 rows][64 columns].  The split (pair)
  // rows of from_tensor and to_tensor lie here while the Q/K/V projections read them, those of the layer's output once
  // the intermediate has been consumed.
  w.inter = off; off += align_up(align_up(rows, 256) * 4 * H * ea, 256);
  w.seq = off;   off += align_up(et::seq_table_words(B) * sizeof(int32_t), 256);
  w.cls = off;   off += align_up(et::mask_class_bytes(dtype == ET_FP32 ? et::DType::F32 : et::DType::F16, B, S, d), 256);
  // k-contiguous copies (fp32: split or pair rows) of the six dense kernels (3 H^2 + H^2 + 4 H^2 + 4 H^2 elements)
  w.wt = off;    off += dtype == ET_FP16 || split ? align_up(12 * H * H * ea, 256) : 0;
  w.pair = off;  off += pairs ? align_up(4 * pair_ws_words(rows, H), 256) : 0;
  w.total = off;
  return w;
}

// First statement of every entry point that takes a handle: rejects a null handle, takes the handle's lock (calls on
// one handle are serialised, and the handle's message slot is only written under it) and makes the handle's device
// current for the calling thread.
struct Entry {
  std::unique_lock<std::mutex> lock;
  et_status status = ET_OK;
  explicit Entry(et_handle h) {
    if (!h) {
      status = fail(nullptr, ET_INVALID_ARGUMENT, "null handle");
      return;
    }
    lock = std::unique_lock<std::mutex>(h->mu);
    status = check_hip(h, hipSetDevice(h->device), "hipSetDevice", __FILE__, __LINE__);
  }
};

et_status dims_ok(et_handle h, int B, int S, int heads, int d) {
  ET_REQUIRE(h, B >= 1 && S >= 1 && heads >= 1 && d >= 1, "batch_size, seq_len, head_num, size_per_head must be >= 1");
  ET_REQUIRE(h, (long)B * S < (1L << 30), "batch_size * seq_len too large");
  // row widths and their multiples (3 H, 4 H, bytes per row) are held in 32-bit integers throughout
  ET_REQUIRE(h, (long)heads * d <= (1L << 20), "head_num * size_per_head above 1048576");
  return ET_OK;
}

// the attention kernels put the sequence on a grid dimension that holds 65535 entries
et_status batch_fits_grid(et_handle h, int B) {
  if (B > 65535) return fail(h, ET_UNSUPPORTED, "batch_size above 65535 is not supported by the attention kernels");
  return ET_OK;
}

float softmax_scaler(et_dtype dtype, int d) {
  float s = 1.0f / sqrtf((float)d);
  if (dtype == ET_FP16) s = (float)(_Float16)s;   // the reference holds the scaler in the element type
  return s;
}

et_status embedding_args_ok(et_handle h, et_dtype dtype, const et_embedding_weights* emb, const int32_t* token_type_ids,
                            int seq_len, int H) {
  ET_REQUIRE(h, emb != nullptr, "null embeddings");
  ET_REQUIRE(h, emb->word_embeddings && emb->layernorm_gamma && emb->layernorm_beta, "null embedding table or LayerNorm weight");
  ET_REQUIRE(h, emb->vocab_size >= 1, "vocab_size must be >= 1");
  ET_REQUIRE(h, (emb->token_type_embeddings == nullptr) == (token_type_ids == nullptr),
             "token_type_ids and token_type_embeddings go together");
  ET_REQUIRE(h, emb->token_type_embeddings == nullptr || emb->type_vocab_size >= 1, "type_vocab_size must be >= 1");
  ET_REQUIRE(h, emb->position_embeddings == nullptr || seq_len <= emb->max_position_embeddings,
             "seq_len exceeds max_position_embeddings");
  if (!et::layernorm_row_in_registers(to_dt(dtype), H))
    return fail(h, ET_UNSUPPORTED, "hidden size not supported by the embedding kernel (even, at most 4096)");
  return ET_OK;
}

// What a layer asks of its arguments whoever calls it; the tensors and the entry are the caller's to check.
et_status layer_args_ok(et_handle h, et_dtype dtype, const et_layer_weights* w, const et_layer_prepared* prep, int B, int S,
                        int heads, int d) {
  ET_REQUIRE(h, w != nullptr, "null weights");
  ET_REQUIRE(h, w->attr_kernel_Q && w->attr_kernel_K && w->attr_kernel_V && w->attr_bias_Q && w->attr_bias_K &&
                    w->attr_bias_V && w->attr_output_kernel && w->attr_output_bias && w->attr_output_layernorm_gamma &&
                    w->attr_output_layernorm_beta && w->inter_kernel && w->inter_bias && w->output_kernel &&
                    w->output_bias && w->output_layernorm_gamma && w->output_layernorm_beta,
             "null weight pointer");
  const int H = heads * d, F = 4 * H;
  const et::DType dt = to_dt(dtype);
  et_status s;
  if ((s = batch_fits_grid(h, B)) != ET_OK) return s;
  if (!et::attention_supported(dt, S, d))
    return fail(h, ET_UNSUPPORTED, "attention needs size_per_head <= 256 and seq_len <= 1024");
  if (!et::gemm_supported(dt, H, H, 3) || !et::gemm_supported(dt, F, H, 1) || !et::gemm_supported(dt, H, F, 1))
    return fail(h, ET_UNSUPPORTED, "hidden size not supported by the GEMM kernels");
  if ((uint64_t)B * S * F * et::elem_size(dt) > 0xffffffffull)
    return fail(h, ET_UNSUPPORTED, "activation matrix larger than 4 GB");
  if (!et::bias_gelu_supported(dt, F) || !et::bias_residual_layernorm_supported(dt, H))
    return fail(h, ET_UNSUPPORTED, "hidden size not supported by the row kernels");
  if (prep) {
    if (prep->seq_start && prep->seq_start_bytes < seq_table_bytes_min(B))
      return fail(h, ET_WORKSPACE_TOO_SMALL, "et_layer_prepared.seq_start needs et_seq_workspace_bytes(batch_size) bytes");
    ET_REQUIRE(h, (prep->attr_kernel_Q_t != nullptr) == (prep->attr_kernel_K_t != nullptr) &&
                      (prep->attr_kernel_Q_t != nullptr) == (prep->attr_kernel_V_t != nullptr),
               "prepared Q, K and V kernels go together");
  }
  return ET_OK;
}

// One layer of a batch whose arguments have been checked: launches only.
struct LayerCall {
  et_dtype dtype;
  const et_layer_weights* w;
  const et_layer_prepared* prep;      // may be null
  const void *from, *to, *attr_mask;
  const int32_t *count, *batch_idx, *word_idx;
  const int32_t* seq_start;           // the batch's sequence table, or null: built here
  const uint8_t* mask_class = nullptr;   // the classes of the batch's mask rows, or null: made here where they are used
  void* out;
  int B, S, heads, d;
  int rows;                           // launches are sized for this many rows
  bool rows_exact = false;            //   ... which is the count itself: no kernel asks the device for it
  char* workspace;
  const et::PairRowsJob* input = nullptr;   // fp32 on pair rows: what makes `from` and its pair rows, with this call's first launch
  bool from_split_ready = false;      // fp32: the split (pair) rows of `from` are in the workspace's intermediate already
  bool write_out_split = false;       //   ... and those of `out` are to be left there
  hipStream_t stream;
};
et_status run_layer(et_handle h, const LayerCall& c);

// What the call does not bring along of its batch: the sequence table, and the mask's classes where the attention kernel makes
// use of them.
et::BatchJobs layer_batch_jobs(const LayerCall& c, const LayerWs& ws) {
  et::BatchJobs j;
  if (c.seq_start) return j;
  j.batch_idx = c.batch_idx;
  j.word_idx = c.word_idx;
  j.rows_dev = c.rows_exact ? nullptr : c.count;
  j.rows_bound = c.rows;
  j.batch = c.B;
  j.seq_len = c.S;
  j.seq_table = (int32_t*)(c.workspace + ws.seq);
  j.attr_mask = c.attr_mask;
  j.fp32 = c.dtype == ET_FP32;
  if (!c.mask_class && et::mask_class_bytes(to_dt(c.dtype), c.B, c.S, c.d)) j.cls = (uint8_t*)(c.workspace + ws.cls);
  et::count_batch_jobs(&j);
  return j;
}

// The pair rows of a layer's first input, where et_encoder leaves them and the Q/K/V projections find them.
et::PairRows first_pair_rows(char* layer_base, const LayerWs& ws, int B, int S, int H) {
  const PairWs p = pair_ws(layer_base + ws.pair, (size_t)B * S, (size_t)H);
  return {(_Float16*)(layer_base + ws.inter), p.from_exp, p.from_norm};
}

// fp32 layer on pair rows: launch order of run_layer.
et_status run_layer_pairs(et_handle h, const LayerCall& c) {
  const et_layer_weights* w = c.w;
  static const et_layer_prepared kNoPrep = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
  const et_layer_prepared& pp = c.prep ? *c.prep : kNoPrep;
  const int B = c.B, S = c.S, H = c.heads * c.d, F = 4 * H, rows = c.rows;
  const LayerWs ws = layer_ws(c.dtype, B, S, c.heads, c.d);
  const et::DType dt = et::DType::F32;
  const int32_t* T = c.rows_exact ? nullptr : c.count;
  hipStream_t st = c.stream;
  et_status s;
  char* base = c.workspace;
  const PairWs pw = pair_ws(base + ws.pair, (size_t)B * S, (size_t)H);
  float *qkv = (float*)(base + ws.qkv), *attn = (float*)(base + ws.attn);
  const int32_t* seq_start = c.seq_start ? c.seq_start : (int32_t*)(base + ws.seq);

  // Weights, made anew by every call.  A caller's split copies (et_layer_prepared) hold the same floats: they are what is
  // read where they are handed over.
  _Float16* wt = (_Float16*)(base + ws.wt);
  const size_t HH = (size_t)2 * H * H;
  et::PairWeightJobs jobs;
  float* tops = pw.tops;
  auto weight = [&](const void* plain, const void* split, int k, int n, size_t at, const void* bias, float* stats) {
    jobs.job[jobs.count++] = {split ? split : plain, split != nullptr, k, n, wt + at * HH, pw.w_exp + at * H, tops, (const float*)bias, stats};
    tops += et::pair_weight_tops(n, k);
  };
  weight(w->attr_kernel_Q, pp.attr_kernel_Q_t, H, H, 0, nullptr, nullptr);
  weight(w->attr_kernel_K, pp.attr_kernel_K_t, H, H, 1, nullptr, nullptr);
  weight(w->attr_kernel_V, pp.attr_kernel_V_t, H, H, 2, nullptr, nullptr);
  weight(w->attr_output_kernel, pp.attr_output_kernel_t, H, H, 3, nullptr, nullptr);
  weight(w->inter_kernel, pp.inter_kernel_t, H, F, 4, w->inter_bias, pw.up_stats);
  weight(w->output_kernel, pp.output_kernel_t, F, H, 8, nullptr, nullptr);
  const et::BatchJobs batch = layer_batch_jobs(c, ws);
  // the inputs, in the room of the intermediate, which nothing needs before they have been read
  et::PairRows from = first_pair_rows(base, ws, B, S, H), to = from;
  et::PairRowsJob inputs[2];
  int count = 0;
  auto input = [&](const void* src, const et::PairRows& out) {
    et::PairRowsJob& job = inputs[count++];
    job.src = (const float*)src, job.out = out, job.m = rows, job.n = H, job.rows_dev = T;
  };
  if (c.input) inputs[count++] = *c.input;
  else if (!c.from_split_ready) input(c.from, from);
  if (c.to != c.from) {
    to = {from.rows + (size_t)rows * 2 * H, pw.to_exp, pw.to_norm};
    input(c.to, to);
  }
  et::launch_pair_weights(jobs, st, &batch, inputs, count);
  et::PairProduct p3;
  p3.groups = 3;
  p3.A[0] = from; p3.A[1] = to; p3.A[2] = to;
  const void* qkv_bias[3] = {w->attr_bias_Q, w->attr_bias_K, w->attr_bias_V};
  for (int i = 0; i < 3; ++i) {
    p3.B[i] = wt + i * HH;
    p3.b_exp[i] = pw.w_exp + i * H;
    p3.bias[i] = (const float*)qkv_bias[i];
  }
  et::launch_gemm_pair(p3, qkv, 3 * H, rows, H, H, T, st);
  if ((s = check_launch(h, "QKV projection")) != ET_OK) return s;

  const uint8_t* cls = c.mask_class ? c.mask_class : batch.cls;
  if (!cls && et::mask_class_bytes(dt, B, S, c.d)) {
    et::launch_mask_class(dt, c.attr_mask, seq_start, c.word_idx, B, S, (uint8_t*)(base + ws.cls), st);
    cls = (const uint8_t*)(base + ws.cls);
  }
  const et::PairRows ctx_rows{(_Float16*)(base + ws.ctx), pw.ctx_exp, pw.attn_norm};      // (the norms are rewritten by LayerNorm)
  // The attention kernels leave the context as pair rows with an exponent for each head, from its own largest value: no workgroup
  // sees a whole row, and a bound over all rows of a sequence took the bits of queries that do not see a token of large values
  // (V of that token 2^30 of the others': rows off by 1.9e-3, now 1.1e-6).  Where they cannot (heads of another size than 64) the
  // context takes the attention output's place until a launch of its own has paired its rows.
  const bool by_heads = et::attention_writes_pieces(qkv, qkv + H, qkv + 2 * H, 1, 3 * H, c.d);
  et::HeadExps head_exp;
  if (by_heads) head_exp = {(int8_t*)(base + ws.attn_split), et::head_exp_stride(rows)};      // (LayerNorm's rows come there behind the product)
  et::launch_attention(dt, qkv, qkv + H, qkv + 2 * H, 1, 3 * H, c.attr_mask, by_heads ? (void*)ctx_rows.rows : attn, seq_start, c.word_idx, B,
                       S, c.heads, c.d, softmax_scaler(c.dtype, c.d), st, by_heads ? et::AttentionOut::kPairs : et::AttentionOut::kPlain, cls,
                       head_exp);
  if (!by_heads) {
    et::PairRowsJob context;
    context.src = attn, context.out = ctx_rows, context.m = rows, context.n = H, context.rows_dev = T;
    et::launch_pair_rows(context, st);
  }
  if ((s = check_launch(h, "attention")) != ET_OK) return s;

  auto product = [&](const et::PairRows& a, const int8_t* a_head_exp, int w_at, void* C, int n, int k_) {
    et::PairProduct p;
    p.A[0] = a;
    p.head_exp = a_head_exp;
    p.B[0] = wt + w_at * HH;
    p.b_exp[0] = pw.w_exp + w_at * H;
    et::launch_gemm_pair(p, C, n, rows, n, k_, T, st);
  };
  product(ctx_rows, head_exp.exp, 3, attn, H, H);
  const et::PairRows attn_rows{(_Float16*)(base + ws.attn_split), pw.attn_exp, pw.attn_norm};
  et::launch_bias_residual_layernorm(dt, attn, c.from, w->attr_output_bias, w->attr_output_layernorm_gamma,
                                     w->attr_output_layernorm_beta, rows, H, T, st, et::WarmList(), nullptr, attn_rows);
  if ((s = check_launch(h, "attention output")) != ET_OK) return s;
  et::PairProduct up;
  up.A[0] = attn_rows;
  up.B[0] = wt + 4 * HH;
  up.b_exp[0] = pw.w_exp + 4 * H;
  up.bias[0] = (const float*)w->inter_bias;
  up.stats = pw.up_stats;
  up.c_exp = pw.inter_exp;
  et::launch_gemm_pair(up, base + ws.inter, F, rows, F, H, T, st);
  if ((s = check_launch(h, "FFN up")) != ET_OK) return s;
  product({(_Float16*)(base + ws.inter), pw.inter_exp, nullptr}, nullptr, 8, c.out, H, F);
  et::launch_bias_residual_layernorm(dt, c.out, attn, w->output_bias, w->output_layernorm_gamma, w->output_layernorm_beta, rows, H,
                                     T, st, et::WarmList(), nullptr, c.write_out_split ? from : et::PairRows());
  return check_launch(h, "FFN down");
}

et_status run_layer(et_handle h, const LayerCall& c) {
  if (layer_pairs(c.dtype, c.heads * c.d)) return run_layer_pairs(h, c);
  const et_layer_weights* w = c.w;
  const int B = c.B, S = c.S, H = c.heads * c.d, F = 4 * H, rows = c.rows;
  const LayerWs ws = layer_ws(c.dtype, B, S, c.heads, c.d);
  const et::DType dt = to_dt(c.dtype);
  const int32_t* T = c.rows_exact ? nullptr : c.count;
  hipStream_t st = c.stream;
  et_status s;
  const size_t e = et::elem_size(dt);
  const bool split = layer_splits(c.dtype, H);
  char* base = c.workspace;
  void* qkv = base + ws.qkv;
  void* ctx = base + ws.ctx;
  void* attn = base + ws.attn;
  void* inter = base + ws.inter;
  const int32_t* seq_start = c.seq_start ? c.seq_start : (int32_t*)(base + ws.seq);

  // The large-M fp16 GEMM reads k-contiguous weights with fewer LDS instructions.  Where the caller prepared such
  // copies they are used wherever that kernel runs; otherwise the wide projections get a transposed copy in the
  // workspace on every call (the caller's weights stay as they are).
  static const et_layer_prepared kNoPrep = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
  const et_layer_prepared& pp = c.prep ? *c.prep : kNoPrep;
  const bool can_qkv = et::gemm_takes_transposed_b(dt, rows, 3 * H, H, H, 3);
  const bool can_o = et::gemm_takes_transposed_b(dt, rows, H, H, H, 1);
  const bool can_up = et::gemm_takes_transposed_b(dt, rows, F, F, H, 1);
  const bool can_down = et::gemm_takes_transposed_b(dt, rows, H, H, F, 1);
  // (the split products take their weights as split copies only)
  const bool t_qkv = split || (can_qkv && (pp.attr_kernel_Q_t || et::gemm_prefers_transposed_b(dt, rows, 3 * H, H, H, 3)));
  const bool t_o = split || (can_o && (pp.attr_output_kernel_t || et::gemm_prefers_transposed_b(dt, rows, H, H, H, 1)));
  const bool t_up = split || (can_up && (pp.inter_kernel_t || et::gemm_prefers_transposed_b(dt, rows, F, F, H, 1)));
  const bool t_down = split || (can_down && (pp.output_kernel_t || et::gemm_prefers_transposed_b(dt, rows, H, H, F, 1)));
  char* wt = base + ws.wt;
  const size_t HH = (size_t)H * H * (split ? 6 : e);
  const void* wt_q = wt; const void* wt_k = wt + HH; const void* wt_v = wt + 2 * HH; const void* wt_o = wt + 3 * HH;
  const void* wt_up = wt + 4 * HH; const void* wt_down = wt + 8 * HH;
  const et::BatchJobs batch = layer_batch_jobs(c, ws);
  {
    et::TransposeJobs jobs;
    if (t_qkv && pp.attr_kernel_Q_t) {
      wt_q = pp.attr_kernel_Q_t; wt_k = pp.attr_kernel_K_t; wt_v = pp.attr_kernel_V_t;
    } else if (t_qkv) {
      jobs.add(w->attr_kernel_Q, wt, H, H);
      jobs.add(w->attr_kernel_K, wt + HH, H, H);
      jobs.add(w->attr_kernel_V, wt + 2 * HH, H, H);
    }
    if (t_o && pp.attr_output_kernel_t) wt_o = pp.attr_output_kernel_t;
    else if (t_o) jobs.add(w->attr_output_kernel, wt + 3 * HH, H, H);
    if (t_up && pp.inter_kernel_t) wt_up = pp.inter_kernel_t;
    else if (t_up) jobs.add(w->inter_kernel, wt + 4 * HH, H, F);
    if (t_down && pp.output_kernel_t) wt_down = pp.output_kernel_t;
    else if (t_down) jobs.add(w->output_kernel, wt + 8 * HH, F, H);
    // one launch makes the sequence table, the mask's classes and the transposed copies; none when the caller prepared all
    if (split) {
      et::launch_split_weights(jobs, st);
      jobs.count = 0;
    }
    et::launch_transpose_weights(jobs, st, &batch);
  }
  // split rows of the two inputs, in the room of the intermediate, which nothing needs before they have been read
  const void *from_a = c.from, *to_a = c.to;
  if (split) {
    uint16_t* fs = (uint16_t*)inter;
    if (!c.from_split_ready) et::launch_split_rows((const float*)c.from, fs, rows, H, T, st);
    from_a = to_a = fs;
    if (c.to != c.from) {
      uint16_t* ts = fs + (size_t)rows * 3 * H;
      et::launch_split_rows((const float*)c.to, ts, rows, H, T, st);
      to_a = ts;
    }
  }
  auto gemm = [&](const et::GemmGroups& g, void* C, int ldc, int n, int k) {
    if (split) et::launch_gemm_split(g, C, ldc, rows, n, k, T, st);
    else et::launch_gemm(dt, g, C, ldc, rows, n, k, T, st);
  };
  // Every matrix of the layer is read again by the kernel after the one that wrote it.  While the layer's matrices
  // (from, Q/K/V, context, attention output, [T,4H], out) about fit the last-level cache, the GEMMs leave their
  // outputs there (written through the L2s); beyond that the outputs would only displace the weights and the A rows.
  const bool cached = (double)rows * (7.0 * H + F) * (double)e <= kCachedLayerBytes;
  // Q = from.Wq + bq, K = to.Wk + bk, V = to.Wv + bv into one [T,3H] buffer (bert_transformer_op.cu.cc:105-156)
  et::GemmGroups g3;
  g3.groups = 3;
  g3.c_cached = cached;
  g3.A[0] = from_a; g3.A[1] = to_a;
  g3.B[0] = t_qkv ? wt_q : w->attr_kernel_Q; g3.B[1] = t_qkv ? wt_k : w->attr_kernel_K; g3.B[2] = t_qkv ? wt_v : w->attr_kernel_V;
  g3.bias[0] = w->attr_bias_Q; g3.bias[1] = w->attr_bias_K; g3.bias[2] = w->attr_bias_V;
  g3.b_transposed = t_qkv;
  gemm(g3, qkv, 3 * H, H, H);
  if ((s = check_launch(h, "QKV projection")) != ET_OK) return s;
  // QK^T, softmax, PV, un-pad (:159-192)
  const char *q = (const char*)qkv, *k = q + (size_t)H * e, *v = k + (size_t)H * e;
  const bool ctx_split = split && et::attention_writes_pieces(q, k, v, 1, 3 * H, c.d);
  const uint8_t* cls = c.mask_class ? c.mask_class : batch.cls;
  if (!cls && et::mask_class_bytes(dt, B, S, c.d)) {
    et::launch_mask_class(dt, c.attr_mask, seq_start, c.word_idx, B, S, (uint8_t*)(base + ws.cls), st);
    cls = (const uint8_t*)(base + ws.cls);
  }
  // (where the attention kernel writes floats only, they take the attention output's place until they are split)
  et::launch_attention(dt, q, k, v, 1, 3 * H, c.attr_mask, split && !ctx_split ? attn : ctx, seq_start, c.word_idx, B, S,
                       c.heads, c.d, softmax_scaler(c.dtype, c.d), st, ctx_split ? et::AttentionOut::kSplit : et::AttentionOut::kPlain, cls);
  if (split && !ctx_split) et::launch_split_rows((const float*)attn, (uint16_t*)ctx, rows, H, T, st);
  if ((s = check_launch(h, "attention")) != ET_OK) return s;
  // attention output projection + bias + residual(from_tensor) + LayerNorm (:195-213)
  et::GemmGroups g1;
  g1.groups = 1;
  g1.c_cached = cached;
  g1.A[0] = ctx; g1.B[0] = t_o ? wt_o : w->attr_output_kernel; g1.bias[0] = nullptr;
  g1.b_transposed = t_o;
  gemm(g1, attn, H, H, H);
  // Every weight matrix was last read a whole batch ago, and a GEMM's first round of tiles waits for each cold slice of
  // it (13000 rows: FFN-down 63 us with cold weights, 53 with the weights in the last-level cache; 2000 rows: 20 and
  // 15.6 us).  The two LayerNorm kernels request the matrices that come next on their way: this one the FFN-up weights
  // and, while the layer's matrices are small enough for them to survive FFN-up, the FFN-down weights; the last one the
  // region the caller names, the next layer's attention weights (12-layer BERT-base on three models' weights in turn:
  // -5 % at 700 tokens, -11 % at 2000, -4 % at 8000, -1 % at 16000).
  const bool warm_fits = (double)rows * (7.0 * H + F) * (double)e <= kWarmLayerBytes;
  et::WarmList warm1, warm2;
  // (whichever copy the GEMM reads, unless this call has just written it)
  const void* b_up = t_up ? wt_up : w->inter_kernel;
  const void* b_down = t_down ? wt_down : w->output_kernel;
  if (!(t_up && !pp.inter_kernel_t)) warm1.add(b_up, (size_t)H * F * (split ? 6 : e));
  if (warm_fits && !(t_down && !pp.output_kernel_t)) warm1.add(b_down, (size_t)H * F * (split ? 6 : e));
  warm2.add(pp.warm, pp.warm_bytes);
  // (split layers: the row kernel leaves its output as split rows too; rows it cannot hold in registers take a pass)
  const bool ln_split = split && et::layernorm_row_in_registers(dt, H);
  uint16_t* attn_split = (uint16_t*)(base + ws.attn_split);
  et::launch_bias_residual_layernorm(dt, attn, c.from, w->attr_output_bias, w->attr_output_layernorm_gamma,
                                     w->attr_output_layernorm_beta, rows, H, T, st, warm1, ln_split ? attn_split : nullptr);
  if (split && !ln_split) et::launch_split_rows((const float*)attn, attn_split, rows, H, T, st);
  if ((s = check_launch(h, "attention output")) != ET_OK) return s;
  // FFN up + bias + GELU (:215-227, cuda/cuda_kernels.cu:88-150)
  g1.A[0] = split ? (const void*)attn_split : attn; g1.B[0] = t_up ? wt_up : w->inter_kernel;
  g1.b_transposed = t_up;
  // bias + GELU are applied to each tile on its way out of the GEMM: no pass of its own over [T,4H]
  g1.bias[0] = w->inter_bias; g1.gelu = true;
  // where both FFN projections run the persistent k-contiguous kernel, [T,4H] goes from one to the other in blocks
  const bool blocked = t_up && t_down && et::gemm_blocked_handover(dt, rows, F, H);
  g1.c_blocked = blocked;
  gemm(g1, inter, F, F, H);
  g1.bias[0] = nullptr; g1.gelu = false; g1.c_blocked = false;
  if ((s = check_launch(h, "FFN up")) != ET_OK) return s;
  // FFN down + bias + residual(LN1 output) + LayerNorm (:229-247)
  g1.A[0] = inter; g1.B[0] = t_down ? wt_down : w->output_kernel;
  g1.b_transposed = t_down;
  g1.a_blocked = blocked;
  gemm(g1, c.out, H, H, F);
  g1.a_blocked = false;
  uint16_t* out_split = split && c.write_out_split ? (uint16_t*)inter : nullptr;
  et::launch_bias_residual_layernorm(dt, c.out, attn, w->output_bias, w->output_layernorm_gamma,
                                     w->output_layernorm_beta, rows, H, T, st, warm2, ln_split ? out_split : nullptr);
  if (out_split && !ln_split) et::launch_split_rows((const float*)c.out, out_split, rows, H, T, st);
  if ((s = check_launch(h, "FFN down")) != ET_OK) return s;
  return ET_OK;
}

}  // namespace

extern "C" {

const char* et_status_string(et_status s) {
  switch (s) {
    case ET_OK: return "ET_OK";
    case ET_INVALID_ARGUMENT: return "ET_INVALID_ARGUMENT";
    case ET_WORKSPACE_TOO_SMALL: return "ET_WORKSPACE_TOO_SMALL";
    case ET_UNSUPPORTED: return "ET_UNSUPPORTED";
    case ET_LAUNCH_FAILURE: return "ET_LAUNCH_FAILURE";
    case ET_RUNTIME_ERROR: return "ET_RUNTIME_ERROR";
  }
  return "<unknown>";
}

int et_device_ok(int device) {
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 0;
  return std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
}

et_status et_create(et_handle* out, int device) {
  if (!out) return fail(nullptr, ET_INVALID_ARGUMENT, "null output handle");
  *out = nullptr;
  int count = 0;
  hipError_t e = hipGetDeviceCount(&count);
  if (e != hipSuccess) return fail(nullptr, ET_RUNTIME_ERROR, std::string("hipGetDeviceCount: ") + hipGetErrorString(e));
  if (device < 0 || device >= count) return fail(nullptr, ET_INVALID_ARGUMENT, "no such device");
  if (!et_device_ok(device)) return fail(nullptr, ET_UNSUPPORTED, "device is not gfx950; the kernels are built for MI355X only");
  {
    // the address of the static scratch array on this device (et_input_static), looked up with the device current
    int prev = 0;
    e = hipGetDevice(&prev);
    if (e == hipSuccess) e = hipSetDevice(device);
    if (e == hipSuccess) {
      e = resolve_static_scratch(device);
      (void)hipSetDevice(prev);
    }
    if (e != hipSuccess)
      return fail(nullptr, ET_RUNTIME_ERROR, std::string("static scratch lookup: ") + hipGetErrorString(e));
  }
  et_context* c = new (std::nothrow) et_context();
  if (!c) return fail(nullptr, ET_RUNTIME_ERROR, "out of host memory");
  c->device = device;
  c->static_slot = device < kMaxDevices ? take_static_slot(device) : -1;
  *out = c;
  return ET_OK;
}

et_status et_destroy(et_handle h) {
  if (!h) return ET_OK;
  release_static_slot(h->device, h->static_slot);
  if (tls_error_handle == h) tls_error_handle = nullptr;
  delete h;
  return ET_OK;
}

const char* et_last_error(et_handle h) {
  if (tls_error_handle == h) return tls_error.c_str();       // this thread's own last failure (on h, or without a handle)
  if (!h) return "";
  std::lock_guard<std::mutex> lock(h->err_mu);
  tls_error_copy = h->last_error;
  return tls_error_copy.c_str();
}

size_t et_input_workspace_bytes(int batch_size, int seq_len) {
  if (batch_size < 1 || seq_len < 1) return 0;
  return align_up((et::scan_scratch_words(batch_size * seq_len) + 1) * sizeof(int32_t), 256);
}

size_t et_layer_workspace_bytes(et_dtype dtype, int batch_size, int seq_len, int head_num, int size_per_head) {
  if (batch_size < 1 || seq_len < 1 || head_num < 1 || size_per_head < 1 || !dtype_ok(dtype)) return 0;
  return layer_ws(dtype, batch_size, seq_len, head_num, size_per_head).total;
}

size_t et_seq_workspace_bytes(int batch_size) {
  if (batch_size < 1) return 0;
  return seq_table_bytes_min(batch_size) + et::mask_class_bytes_max(batch_size);
}

et_status et_input(et_handle h, et_dtype dtype, const void* from_tensor, const int32_t* mask, void* to_tensor,
                   int32_t* valid_word_num_dev, int32_t* batch_idx, int32_t* word_idx, int batch_size, int seq_len,
                   int head_num, int size_per_head, void* workspace, size_t workspace_bytes, void* stream,
                   int32_t* valid_word_num_host) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, from_tensor && mask && to_tensor && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  if (workspace_bytes < et_input_workspace_bytes(batch_size, seq_len))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "et_input needs et_input_workspace_bytes(batch_size, seq_len)");
  const size_t row_bytes = (size_t)head_num * size_per_head * et::elem_size(to_dt(dtype));
  if (et::move_chunks(batch_size * seq_len, (int)row_bytes) >= (1ull << 31))
    return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");
  hipStream_t st = (hipStream_t)stream;
  et::launch_scan_index(mask, batch_size * seq_len, nullptr, batch_idx, word_idx, valid_word_num_dev, seq_len,
                        (int32_t*)workspace, st);
  if ((s = check_launch(h, "mask scan")) != ET_OK) return s;
  et::launch_compress_rows(from_tensor, to_tensor, batch_idx, word_idx, valid_word_num_dev, nullptr, nullptr,
                           batch_size, seq_len, (int)row_bytes, st);
  if ((s = check_launch(h, "compress")) != ET_OK) return s;
  if (valid_word_num_host) {
    ET_HIP(h, hipMemcpyAsync(valid_word_num_host, valid_word_num_dev, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    ET_HIP(h, hipStreamSynchronize(st));
  }
  return ET_OK;
}

et_status et_input_static(et_handle h, et_dtype dtype, const void* from_tensor, const int32_t* mask, void* to_tensor,
                          int32_t* valid_word_num_dev, int32_t* batch_idx, int32_t* word_idx, int batch_size,
                          int seq_len, int head_num, int size_per_head, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, from_tensor && mask && to_tensor && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  if ((long)batch_size * seq_len > kStaticMaxPositions ||
      et::scan_scratch_words(batch_size * seq_len) > (size_t)kStaticSlotWords)
    return fail(h, ET_UNSUPPORTED,
                "et_input_static holds scratch for batch_size * seq_len <= 1048576 positions; larger batches go "
                "through et_input with a caller workspace");
  if (h->static_slot < 0)
    return fail(h, ET_UNSUPPORTED,
                "this handle holds no slot of the static scratch (at most 8 live handles per GPU do); use et_input");
  const size_t row_bytes = (size_t)head_num * size_per_head * et::elem_size(to_dt(dtype));
  if (et::move_chunks(batch_size * seq_len, (int)row_bytes) >= (1ull << 31))
    return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");
  int32_t* scratch_dev = h->device < kMaxDevices ? static_scratch_ptr[h->device] : nullptr;
  if (!scratch_dev) return fail(h, ET_RUNTIME_ERROR, "no static scratch on this device");
  scratch_dev += (size_t)h->static_slot * kStaticSlotWords;
  // Calls that share a slot must not overlap on the GPU.  Calls queued on one stream cannot; a call on another stream
  // is accepted only once everything queued on the previous one has finished.
  hipStream_t st = (hipStream_t)stream;
  if (h->static_stream_set && h->static_stream != st) {
    // (any other answer than "not ready", e.g. for a stream that no longer exists, lets the call through)
    const hipError_t q = hipStreamQuery(h->static_stream);
    if (q != hipSuccess) (void)hipGetLastError();
    if (q == hipErrorNotReady) {
      return fail(h, ET_INVALID_ARGUMENT,
                  "et_input_static: the stream of this handle's previous call still has work in flight, and calls on "
                  "two streams would share the handle's scratch slot; wait for that stream or use a second handle");
    }
  }
  h->static_stream_set = true;
  h->static_stream = st;
  // the scan writes every tile total it later reads, so nothing of the previous call's contents has to be cleared
  et::launch_scan_index(mask, batch_size * seq_len, nullptr, batch_idx, word_idx, valid_word_num_dev, seq_len,
                        scratch_dev, st);
  if ((s = check_launch(h, "mask scan")) != ET_OK) return s;
  et::launch_compress_rows(from_tensor, to_tensor, batch_idx, word_idx, valid_word_num_dev, nullptr, nullptr,
                           batch_size, seq_len, (int)row_bytes, st);
  return check_launch(h, "compress");
}

et_status et_embedding_input(et_handle h, et_dtype dtype, const et_embedding_weights* emb, const int32_t* input_ids,
                             const int32_t* token_type_ids, const int32_t* mask, void* to_tensor,
                             int32_t* valid_word_num_dev, int32_t* batch_idx, int32_t* word_idx, int batch_size,
                             int seq_len, int head_num, int size_per_head, void* workspace, size_t workspace_bytes,
                             void* stream, int32_t* valid_word_num_host) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  if ((s = embedding_args_ok(h, dtype, emb, token_type_ids, seq_len, head_num * size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, input_ids && mask && to_tensor && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  if (workspace_bytes < et_input_workspace_bytes(batch_size, seq_len))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "et_embedding_input needs et_input_workspace_bytes(batch_size, seq_len)");
  const int H = head_num * size_per_head;
  hipStream_t st = (hipStream_t)stream;
  et::launch_scan_index(mask, batch_size * seq_len, nullptr, batch_idx, word_idx, valid_word_num_dev, seq_len,
                        (int32_t*)workspace, st);
  if ((s = check_launch(h, "mask scan")) != ET_OK) return s;
  et::launch_embed_layernorm(to_dt(dtype), to_tensor, input_ids, token_type_ids, batch_idx, word_idx,
                             emb->word_embeddings, emb->vocab_size, emb->token_type_embeddings, emb->type_vocab_size,
                             emb->position_embeddings, emb->max_position_embeddings, emb->layernorm_gamma,
                             emb->layernorm_beta, batch_size * seq_len, H, seq_len, valid_word_num_dev, st);
  if ((s = check_launch(h, "embedding")) != ET_OK) return s;
  if (valid_word_num_host) {
    ET_HIP(h, hipMemcpyAsync(valid_word_num_host, valid_word_num_dev, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    ET_HIP(h, hipStreamSynchronize(st));
  }
  return ET_OK;
}

et_status et_layer(et_handle h, et_dtype dtype, const et_layer_weights* w, const void* from_tensor,
                   const void* to_tensor, const void* attr_mask, const int32_t* valid_word_num_dev,
                   const int32_t* batch_idx, const int32_t* word_idx, void* out, int batch_size, int from_seq_len,
                   int to_seq_len, int head_num, int size_per_head, int valid_word_num_hint, void* workspace,
                   size_t workspace_bytes, void* stream) {
  return et_layer_with_prepared(h, dtype, w, nullptr, from_tensor, to_tensor, attr_mask, valid_word_num_dev, batch_idx,
                                word_idx, out, batch_size, from_seq_len, to_seq_len, head_num, size_per_head,
                                valid_word_num_hint, workspace, workspace_bytes, stream);
}

et_status et_sequence_starts(et_handle h, const int32_t* batch_idx, const int32_t* valid_word_num_dev, int batch_size,
                             int seq_len, int32_t* seq_start, size_t seq_start_bytes, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  if ((s = dims_ok(h, batch_size, seq_len, 1, 1)) != ET_OK) return s;
  ET_REQUIRE(h, batch_idx && valid_word_num_dev && seq_start, "null tensor pointer");
  if (seq_start_bytes < seq_table_bytes_min(batch_size))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "the sequence table needs et_seq_workspace_bytes(batch_size)");
  et::launch_seq_start(batch_idx, valid_word_num_dev, batch_size * seq_len, batch_size, seq_start, (hipStream_t)stream);
  return check_launch(h, "sequence starts");
}

et_status et_layer_with_prepared(et_handle h, et_dtype dtype, const et_layer_weights* w, const et_layer_prepared* prep,
                                 const void* from_tensor, const void* to_tensor, const void* attr_mask,
                                 const int32_t* valid_word_num_dev, const int32_t* batch_idx, const int32_t* word_idx,
                                 void* out, int batch_size, int from_seq_len, int to_seq_len, int head_num,
                                 int size_per_head, int valid_word_num_hint, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, from_seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, from_seq_len == to_seq_len, "only support from_seq_len == to_seq_len");
  ET_REQUIRE(h, from_tensor && to_tensor && attr_mask && valid_word_num_dev && batch_idx && word_idx && out,
             "null tensor pointer");
  ET_REQUIRE(h, out != from_tensor && out != to_tensor, "out must not alias from_tensor / to_tensor");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  const int B = batch_size, S = from_seq_len;
  ET_REQUIRE(h, valid_word_num_hint >= -1 && valid_word_num_hint <= B * S, "valid_word_num_hint out of range");
  if (workspace_bytes < layer_ws(dtype, B, S, head_num, size_per_head).total)
    return fail(h, ET_WORKSPACE_TOO_SMALL, "et_layer needs et_layer_workspace_bytes(...)");
  if ((s = layer_args_ok(h, dtype, w, prep, B, S, head_num, size_per_head)) != ET_OK) return s;
  if (valid_word_num_hint == 0) return ET_OK;
  LayerCall c;
  c.dtype = dtype; c.w = w; c.prep = prep;
  c.from = from_tensor; c.to = to_tensor; c.attr_mask = attr_mask;
  c.count = valid_word_num_dev; c.batch_idx = batch_idx; c.word_idx = word_idx;
  c.seq_start = prep ? prep->seq_start : nullptr;
  c.out = out;
  c.B = B; c.S = S; c.heads = head_num; c.d = size_per_head;
  c.rows = valid_word_num_hint > 0 ? valid_word_num_hint : B * S;
  c.workspace = (char*)workspace;
  c.stream = (hipStream_t)stream;
  return run_layer(h, c);
}

// ---- the encoder in one call ------------------------------------------------------------------------------------

namespace {

struct EncoderWs {
  size_t x[2], batch_idx, word_idx, packed_row, count, seq, scan, layer, total;
};

EncoderWs encoder_ws(et_dtype dtype, int B, int S, int heads, int d) {
  const size_t e = dtype == ET_FP32 ? 4 : 2;
  const size_t rows = (size_t)B * S, H = (size_t)heads * d;
  EncoderWs w;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align_up(bytes, 256);
    return at;
  };
  w.x[0] = take(rows * H * e);
  w.x[1] = take(rows * H * e);
  w.batch_idx = take(rows * sizeof(int32_t));
  w.word_idx = take(rows * sizeof(int32_t));
  w.packed_row = take(rows * sizeof(int32_t));
  w.count = take(sizeof(int32_t));
  w.seq = take(seq_table_bytes_min(B));
  w.scan = take(et_input_workspace_bytes(B, S));
  w.layer = take(et_layer_workspace_bytes(dtype, B, S, heads, d));
  w.total = off;
  return w;
}

// Waits until the scan of this call has stored its count (upper half = tag).  The word is written by the GPU in the
// middle of the stream's work, so the host spins on it; now and then the stream is asked whether it has failed or run dry.
et_status wait_for_count(et_handle h, const uint64_t* word, uint32_t tag, const int32_t* count_dev, hipStream_t st, int* T) {
  for (unsigned spin = 1;; ++spin) {
    const uint64_t v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
    if ((uint32_t)(v >> 32) == tag) {
      *T = (int32_t)(uint32_t)v;
      return ET_OK;
    }
    if (spin % 4096 != 0) {
#if !defined(__HIP_DEVICE_COMPILE__)
      __builtin_ia32_pause();
#endif
      continue;
    }
    const hipError_t q = hipStreamQuery(st);
    if (q == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    ET_HIP(h, q);
    // everything has run and the word is not there (memory the GPU's store does not reach): read the count itself
    int32_t value = 0;
    ET_HIP(h, hipMemcpyAsync(&value, count_dev, sizeof value, hipMemcpyDeviceToHost, st));
    ET_HIP(h, hipStreamSynchronize(st));
    *T = value;
    return ET_OK;
  }
}

bool is_capturing(hipStream_t st) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &status) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}

}  // namespace

size_t et_encoder_workspace_bytes(et_dtype dtype, int batch_size, int seq_len, int head_num, int size_per_head) {
  if (batch_size < 1 || seq_len < 1 || head_num < 1 || size_per_head < 1 || !dtype_ok(dtype)) return 0;
  return encoder_ws(dtype, batch_size, seq_len, head_num, size_per_head).total;
}

et_status et_encoder(et_handle h, et_dtype dtype, int num_layers, const et_layer_weights* weights,
                     const et_layer_prepared* prepared, const et_encoder_batch* b, int head_num, int size_per_head,
                     void* workspace, size_t workspace_bytes, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  ET_REQUIRE(h, b != nullptr, "null batch");
  const int B = b->batch_size, S = b->seq_len, H = head_num * size_per_head;
  if ((s = dims_ok(h, B, S, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, num_layers >= 1 && weights != nullptr, "an encoder has at least one layer");
  ET_REQUIRE(h, (b->from_tensor != nullptr) != (b->embeddings != nullptr), "either from_tensor or embeddings");
  ET_REQUIRE(h, b->mask && b->attr_mask && b->out && (b->from_tensor || b->input_ids), "null tensor pointer");
  ET_REQUIRE(h, b->rows_bound >= 0 && b->rows_bound <= B * S, "rows_bound out of range");
  if (b->embeddings && (s = embedding_args_ok(h, dtype, b->embeddings, b->token_type_ids, S, H)) != ET_OK) return s;
  for (int l = 0; l < num_layers; ++l)
    if ((s = layer_args_ok(h, dtype, weights + l, prepared ? prepared + l : nullptr, B, S, head_num, size_per_head)) != ET_OK)
      return s;
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  const EncoderWs ws = encoder_ws(dtype, B, S, head_num, size_per_head);
  if (workspace_bytes < ws.total) return fail(h, ET_WORKSPACE_TOO_SMALL, "et_encoder needs et_encoder_workspace_bytes(...)");
  const et::DType dt = to_dt(dtype);
  const size_t row_bytes = (size_t)H * et::elem_size(dt);
  if (et::move_chunks(B * S, (int)row_bytes) >= (1ull << 31))
    return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");

  char* base = (char*)workspace;
  void* x[2] = {base + ws.x[0], base + ws.x[1]};
  int32_t *batch_idx = (int32_t*)(base + ws.batch_idx), *word_idx = (int32_t*)(base + ws.word_idx);
  int32_t *count = (int32_t*)(base + ws.count), *seq = (int32_t*)(base + ws.seq);
  char* layer_base = base + ws.layer;
  hipStream_t st = (hipStream_t)stream;

  // The count comes back through the caller's pinned word, stored by the scan itself: no copy on the stream, no event.
  // Every call has a tag of its own, so a word left by an earlier batch is never taken for this one's.
  static std::atomic<uint32_t> next_tag{1};
  // The layers of a stack wait for it at every size.  12 layers, waiting and launched for all positions, us per pass in a stream
  // of passes: fp16 1 x 32 405 and 405, 4 x 32 with 41 tokens 414 and 424, 8 x 32 with 120 434 and 457, 12 x 32 with 172 449 and
  // 492, 32 x 32 with 546 545 and 635; fp32 854 and 872, 899 and 968, 964 and 1054, 1019 and 1283, 1379 and 1743.
  // (Nothing runs while a stream is being captured, so there the launches are sized for all positions.)
  const bool wait_for_layers = b->rows_bound == 0 && num_layers > 1 && b->count_word && !is_capturing(st);
  et::ScanExtras scan;
  scan.seq_start = seq;
  scan.packed_row = (int32_t*)(base + ws.packed_row);
  if (wait_for_layers || (b->count_word && b->valid_word_num)) {
    scan.host_word = b->count_word;
    scan.host_tag = next_tag.fetch_add(1, std::memory_order_relaxed);
    if (scan.host_tag == 0) scan.host_tag = next_tag.fetch_add(1, std::memory_order_relaxed);
  }
  et::launch_scan_index(b->mask, B * S, nullptr, batch_idx, word_idx, count, S, (int32_t*)(base + ws.scan), st, scan);
  if ((s = check_launch(h, "mask scan")) != ET_OK) return s;
  const bool split = layer_splits(dtype, H);
  et::CompressExtras extras;
  extras.seq_table = seq;
  // (such layers read their first input from the room of the layer workspace's intermediate)
  const size_t split_off = layer_ws(dtype, B, S, head_num, size_per_head).inter;
  if (split) extras.split = (uint16_t*)(layer_base + split_off);
  const bool pairs = layer_pairs(dtype, H);
  if (pairs) extras.pair = first_pair_rows(layer_base, layer_ws(dtype, B, S, head_num, size_per_head), B, S, H);
  et::PairRowsJob input;
  if (b->embeddings) {
    const et_embedding_weights& emb = *b->embeddings;
    et::launch_embed_layernorm(dt, x[0], b->input_ids, b->token_type_ids, batch_idx, word_idx, emb.word_embeddings,
                               emb.vocab_size, emb.token_type_embeddings, emb.type_vocab_size, emb.position_embeddings,
                               emb.max_position_embeddings, emb.layernorm_gamma, emb.layernorm_beta, B * S, H, S, count, st,
                               extras, B);
  } else if (pairs) {
    input.src = (const float*)b->from_tensor, input.packed = (float*)x[0], input.out = extras.pair;
    input.batch_idx = batch_idx, input.word_idx = word_idx, input.m = B * S, input.n = H, input.seq_len = S, input.rows_dev = count;
    input.seq_table = seq, input.batch = B;
    // (while the host waits for the count there is nothing else to do; where it does not, the first layer's weights take it along)
    if (wait_for_layers) et::launch_pair_rows(input, st);
  } else {
    et::launch_compress_rows(b->from_tensor, x[0], batch_idx, word_idx, count, nullptr, nullptr, B, S, (int)row_bytes, st,
                             extras);
  }
  if ((s = check_launch(h, "input")) != ET_OK) return s;

  LayerCall c;
  if (et::mask_class_bytes(dt, B, S, size_per_head)) {      // once for all layers, in the first one's place for them
    uint8_t* cls = (uint8_t*)(layer_base + layer_ws(dtype, B, S, head_num, size_per_head).cls);
    et::launch_mask_class(dt, b->attr_mask, seq, word_idx, B, S, cls, st);
    c.mask_class = cls;
  }
  c.dtype = dtype;
  c.attr_mask = b->attr_mask;
  c.count = count; c.batch_idx = batch_idx; c.word_idx = word_idx;
  c.seq_start = seq;
  c.B = B; c.S = S; c.heads = head_num; c.d = size_per_head;
  c.rows = b->rows_bound > 0 ? b->rows_bound : B * S;
  c.workspace = layer_base;
  c.stream = st;
  int T = -1;
  if (wait_for_layers) {
    // The count is there when the scan ends and the host has it while the input rows are still being moved: the layers
    // are launched for exactly that many rows (other threads may use the handle meanwhile).
    entry.lock.unlock();
    s = wait_for_count(h, scan.host_word, scan.host_tag, count, st, &T);
    entry.lock.lock();
    if (s != ET_OK) return s;
    c.rows = std::min(std::max(T, 0), B * S);
    c.rows_exact = true;
  }
  int cur = 0;
  for (int l = 0; l < num_layers && c.rows > 0; ++l) {
    c.w = weights + l;
    c.prep = prepared ? prepared + l : nullptr;
    c.from = c.to = x[cur];
    c.out = x[cur ^ 1];
    c.from_split_ready = split || pairs;
    c.input = l == 0 && input.src && !wait_for_layers ? &input : nullptr;
    c.write_out_split = l + 1 < num_layers;
    if ((s = run_layer(h, c)) != ET_OK) return s;
    cur ^= 1;
  }
  et::launch_mapped_restore_rows(b->out, x[cur], scan.packed_row, B * S, (int)row_bytes, st);
  if ((s = check_launch(h, "restore")) != ET_OK) return s;
  if (b->valid_word_num) {
    if (T < 0 && scan.host_word) {
      entry.lock.unlock();
      s = wait_for_count(h, scan.host_word, scan.host_tag, count, st, &T);
      entry.lock.lock();
      if (s != ET_OK) return s;
    } else if (T < 0) {
      ET_HIP(h, hipMemcpyAsync(&T, count, sizeof T, hipMemcpyDeviceToHost, st));
      ET_HIP(h, hipStreamSynchronize(st));
    }
    *b->valid_word_num = T;
  }
  return ET_OK;
}

et_status et_output(et_handle h, et_dtype dtype, const void* from_tensor, const int32_t* valid_word_num_dev,
                    const int32_t* batch_idx, const int32_t* word_idx, void* to_tensor, int batch_size, int seq_len,
                    int head_num, int size_per_head, void* stream) {
  if (head_num < 1 || size_per_head < 1 || (long)head_num * size_per_head >= (1L << 30))
    return fail(h, ET_INVALID_ARGUMENT, "head_num, size_per_head must be >= 1");
  return et_restore(h, dtype, to_tensor, from_tensor, batch_idx, word_idx, valid_word_num_dev, batch_size, seq_len,
                    head_num * size_per_head, stream);
}

et_status et_first_token(et_handle h, et_dtype dtype, const void* from_tensor, const int32_t* valid_word_num_dev,
                         const int32_t* batch_idx, const int32_t* word_idx, void* to_tensor, int batch_size,
                         int seq_len, int hidden_dim, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, 1, hidden_dim)) != ET_OK) return s;
  ET_REQUIRE(h, from_tensor && to_tensor && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  const size_t row_bytes = (size_t)hidden_dim * et::elem_size(to_dt(dtype));
  et::launch_first_token(to_tensor, from_tensor, batch_idx, word_idx, valid_word_num_dev, batch_size * seq_len,
                         batch_size, (int)row_bytes, (hipStream_t)stream);
  return check_launch(h, "first token gather");
}

et_status et_exclusive_scan(et_handle h, int32_t* d_out, const int32_t* d_in, int length, void* workspace,
                            size_t workspace_bytes, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, d_out && d_in, "null tensor pointer");
  ET_REQUIRE(h, length >= 1 && length < (1 << 30), "length out of range");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  if (workspace_bytes < et_input_workspace_bytes(1, length))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "et_exclusive_scan needs et_input_workspace_bytes(1, length)");
  et::launch_scan_index(d_in, length, d_out, nullptr, nullptr, nullptr, 0, (int32_t*)workspace, (hipStream_t)stream);
  return check_launch(h, "exclusive scan");
}

et_status et_compress(et_handle h, et_dtype dtype, const void* from_tensor, const int32_t* mask,
                      const int32_t* prefix_sum, void* to_tensor, int32_t* batch_idx, int32_t* word_idx,
                      int batch_size, int seq_len, int hidden_dim, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, 1, hidden_dim)) != ET_OK) return s;
  ET_REQUIRE(h, from_tensor && mask && prefix_sum && to_tensor && batch_idx && word_idx, "null tensor pointer");
  const size_t row_bytes = (size_t)hidden_dim * et::elem_size(to_dt(dtype));
  if (et::move_chunks(batch_size * seq_len, (int)row_bytes) >= (1ull << 31))
    return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");
  hipStream_t st = (hipStream_t)stream;
  et::launch_index_from_prefix(mask, prefix_sum, batch_idx, word_idx, batch_size, seq_len, st);
  et::launch_compress_rows(from_tensor, to_tensor, batch_idx, word_idx, nullptr, prefix_sum, mask, batch_size, seq_len,
                           (int)row_bytes, st);
  return check_launch(h, "compress");
}

et_status et_restore(et_handle h, et_dtype dtype, void* to_tensor, const void* from_tensor, const int32_t* batch_idx,
                     const int32_t* word_idx, const int32_t* valid_word_num_dev, int batch_size, int seq_len,
                     int hidden_dim, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, 1, hidden_dim)) != ET_OK) return s;
  ET_REQUIRE(h, from_tensor && to_tensor && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  const size_t row_bytes = (size_t)hidden_dim * et::elem_size(to_dt(dtype));
  if (et::move_chunks(batch_size * seq_len, (int)row_bytes) >= (1ull << 31))
    return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");
  et::launch_restore_rows(to_tensor, from_tensor, batch_idx, word_idx, valid_word_num_dev, batch_size, seq_len,
                          (int)row_bytes, (hipStream_t)stream);
  return check_launch(h, "restore");
}

et_status et_add_bias_act(et_handle h, et_dtype dtype, void* out, const void* bias, int m, int n,
                          const int32_t* m_dev, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  ET_REQUIRE(h, out && bias, "null tensor pointer");
  ET_REQUIRE(h, m >= 0 && n >= 1, "bad dimensions");
  if (!et::bias_gelu_supported(to_dt(dtype), n)) return fail(h, ET_UNSUPPORTED, "row bytes must be a multiple of 16");
  if (m == 0) return ET_OK;
  et::launch_bias_gelu(to_dt(dtype), out, bias, m, n, m_dev, (hipStream_t)stream);
  return check_launch(h, "bias + gelu");
}

et_status et_add_bias_input_layernorm(et_handle h, et_dtype dtype, void* out, const void* input, const void* bias,
                                      const void* gamma, const void* beta, int m, int n, const int32_t* m_dev,
                                      void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  ET_REQUIRE(h, out && input && bias && gamma && beta, "null tensor pointer");
  ET_REQUIRE(h, m >= 0 && n >= 1, "bad dimensions");
  if (!et::bias_residual_layernorm_supported(to_dt(dtype), n))
    return fail(h, ET_UNSUPPORTED, "row length not supported by the LayerNorm kernel");
  if (m == 0) return ET_OK;
  et::launch_bias_residual_layernorm(to_dt(dtype), out, input, bias, gamma, beta, m, n, m_dev, (hipStream_t)stream);
  return check_launch(h, "bias + residual + layernorm");
}

et_status et_add_qkv_bias_padding(et_handle h, et_dtype dtype, const void* Q, const void* bias_Q, const void* K,
                                  const void* bias_K, const void* V, const void* bias_V, void* q_buf, void* k_buf,
                                  void* v_buf, const int32_t* valid_word_num_dev, int batch_size, int seq_len,
                                  int head_num, int size_per_head, const int32_t* batch_idx, const int32_t* word_idx,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, Q && K && V && bias_Q && bias_K && bias_V && q_buf && k_buf && v_buf && valid_word_num_dev &&
                    batch_idx && word_idx,
             "null tensor pointer");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  if (workspace_bytes < seq_table_bytes_min(batch_size))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "needs et_seq_workspace_bytes(batch_size)");
  if (seq_len > 1024) return fail(h, ET_UNSUPPORTED, "seq_len <= 1024");
  hipStream_t st = (hipStream_t)stream;
  et::launch_seq_start(batch_idx, valid_word_num_dev, batch_size * seq_len, batch_size, (int32_t*)workspace, st);
  et::launch_qkv_bias_pad(to_dt(dtype), Q, bias_Q, K, bias_K, V, bias_V, q_buf, k_buf, v_buf, (int32_t*)workspace,
                          word_idx, batch_size, seq_len, head_num, size_per_head, st);
  return check_launch(h, "qkv bias + padding");
}

et_status et_softmax(et_handle h, et_dtype dtype, void* qk_buf, const void* attr_mask, int batch_size, int head_num,
                     int seq_len, float scaler, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, 1)) != ET_OK) return s;
  ET_REQUIRE(h, qk_buf && attr_mask, "null tensor pointer");
  if (seq_len > 1024) return fail(h, ET_UNSUPPORTED, "softmax kernel supports seq_len <= 1024");
  et::launch_softmax(to_dt(dtype), qk_buf, attr_mask, batch_size, head_num, seq_len, scaler, (hipStream_t)stream);
  return check_launch(h, "softmax");
}

et_status et_transpose_rm_padding(et_handle h, et_dtype dtype, const void* src, void* dst,
                                  const int32_t* valid_word_num_dev, int batch_size, int seq_len, int head_num,
                                  int size_per_head, const int32_t* batch_idx, const int32_t* word_idx, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, src && dst && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  et::launch_transpose_rm_padding(to_dt(dtype), src, dst, valid_word_num_dev, batch_size * seq_len, batch_size,
                                  seq_len, head_num, size_per_head, batch_idx, word_idx, (hipStream_t)stream);
  return check_launch(h, "transpose + remove padding");
}

et_status et_attention(et_handle h, et_dtype dtype, const void* q, const void* k, const void* v, int qkv_layout,
                       int packed_ld, const void* attr_mask, void* dst, const int32_t* valid_word_num_dev,
                       int batch_size, int seq_len, int head_num, int size_per_head, const int32_t* batch_idx,
                       const int32_t* word_idx, void* workspace, size_t workspace_bytes, void* stream) {
  if (h) {
    ET_REQUIRE(h, workspace != nullptr, "null workspace");
    if (workspace_bytes < seq_table_bytes_min(batch_size))
      return fail(h, ET_WORKSPACE_TOO_SMALL, "needs et_seq_workspace_bytes(batch_size)");
  }
  return et_attention_with_starts(h, dtype, q, k, v, qkv_layout, packed_ld, attr_mask, dst, valid_word_num_dev,
                                  batch_size, seq_len, head_num, size_per_head, batch_idx, word_idx, nullptr,
                                  (int32_t*)workspace, workspace_bytes, stream);
}

et_status et_attention_with_starts(et_handle h, et_dtype dtype, const void* q, const void* k, const void* v,
                                   int qkv_layout, int packed_ld, const void* attr_mask, void* dst,
                                   const int32_t* valid_word_num_dev, int batch_size, int seq_len, int head_num,
                                   int size_per_head, const int32_t* batch_idx, const int32_t* word_idx,
                                   const int32_t* seq_start, int32_t* seq_start_scratch, size_t seq_table_bytes,
                                   void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  if ((s = dims_ok(h, batch_size, seq_len, head_num, size_per_head)) != ET_OK) return s;
  ET_REQUIRE(h, q && k && v && attr_mask && dst && valid_word_num_dev && batch_idx && word_idx, "null tensor pointer");
  ET_REQUIRE(h, qkv_layout == 0 || qkv_layout == 1, "qkv_layout must be 0 (padded) or 1 (packed)");
  ET_REQUIRE(h, qkv_layout == 0 || packed_ld >= head_num * size_per_head, "packed_ld smaller than the hidden size");
  ET_REQUIRE(h, seq_start != nullptr || seq_start_scratch != nullptr, "null sequence start table");
  if (seq_table_bytes < seq_table_bytes_min(batch_size))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "the sequence table needs et_seq_workspace_bytes(batch_size)");
  if ((s = batch_fits_grid(h, batch_size)) != ET_OK) return s;
  if (!et::attention_supported(to_dt(dtype), seq_len, size_per_head))
    return fail(h, ET_UNSUPPORTED, "attention needs size_per_head <= 256 and seq_len <= 1024");
  hipStream_t st = (hipStream_t)stream;
  uint8_t* cls = nullptr;
  if (!seq_start) {
    et::launch_seq_start(batch_idx, valid_word_num_dev, batch_size * seq_len, batch_size, seq_start_scratch, st);
    seq_start = seq_start_scratch;
    const size_t table = seq_table_bytes_min(batch_size), bytes = et::mask_class_bytes(to_dt(dtype), batch_size, seq_len, size_per_head);
    if (bytes > 0 && seq_table_bytes >= table + bytes) {
      cls = (uint8_t*)seq_start_scratch + table;
      et::launch_mask_class(to_dt(dtype), attr_mask, seq_start, word_idx, batch_size, seq_len, cls, st);
    }
  }
  et::launch_attention(to_dt(dtype), q, k, v, qkv_layout, packed_ld, attr_mask, dst, seq_start, word_idx, batch_size,
                       seq_len, head_num, size_per_head, softmax_scaler(dtype, size_per_head), st, et::AttentionOut::kPlain, cls);
  return check_launch(h, "attention");
}

namespace {

et_status gemm_impl(et_handle h, et_dtype dtype, const void* A, const void* B, void* C, const void* bias, int m, int n,
                    int k, const int32_t* m_dev, void* stream, bool gelu, const char* what) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  ET_REQUIRE(h, A && B && C, "null tensor pointer");
  ET_REQUIRE(h, !gelu || bias, "null bias");
  ET_REQUIRE(h, m >= 0 && n >= 1 && k >= 1, "bad dimensions");
  if (!et::gemm_supported(to_dt(dtype), n, k, 1))
    return fail(h, ET_UNSUPPORTED, "GEMM dimensions out of range");
  if ((uint64_t)m * k * et::elem_size(to_dt(dtype)) > 0xffffffffull)
    return fail(h, ET_UNSUPPORTED, "A larger than 4 GB");
  if (m == 0) return ET_OK;
  et::GemmGroups g;
  g.groups = 1;
  g.A[0] = A; g.B[0] = B; g.bias[0] = bias;
  g.gelu = gelu;
  et::launch_gemm(to_dt(dtype), g, C, n, m, n, k, m_dev, (hipStream_t)stream);
  return check_launch(h, what);
}

}  // namespace

et_status et_gemm(et_handle h, et_dtype dtype, const void* A, const void* B, void* C, const void* bias, int m, int n,
                  int k, const int32_t* m_dev, void* stream) {
  return gemm_impl(h, dtype, A, B, C, bias, m, n, k, m_dev, stream, false, "gemm");
}

et_status et_gemm_bias_gelu(et_handle h, et_dtype dtype, const void* A, const void* B, void* C, const void* bias, int m,
                            int n, int k, const int32_t* m_dev, void* stream) {
  return gemm_impl(h, dtype, A, B, C, bias, m, n, k, m_dev, stream, true, "gemm + bias + gelu");
}

et_status et_transpose_weight(et_handle h, et_dtype dtype, const void* src, void* dst, int k, int n, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype_ok(dtype), "dtype must be ET_FP32 or ET_FP16");
  ET_REQUIRE(h, src && dst && src != dst, "null or aliased tensor pointer");
  et::TransposeJobs jobs;
  if (dtype == ET_FP32) {
    ET_REQUIRE(h, k >= 1 && n >= 1 && et::gemm_split_supported(n, k), "k must be a multiple of 32 and n of 4");
    jobs.add(src, dst, k, n);
    et::launch_split_weights(jobs, (hipStream_t)stream);
    return check_launch(h, "weight split");
  }
  ET_REQUIRE(h, k >= 1 && n >= 1 && k % 8 == 0 && n % 8 == 0, "k and n must be positive multiples of 8");
  jobs.add(src, dst, k, n);
  et::launch_transpose_weights(jobs, (hipStream_t)stream);
  return check_launch(h, "weight transpose");
}

et_status et_split_rows(et_handle h, const void* src, void* dst, int m, int k, const int32_t* m_dev, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, src && dst && src != dst, "null or aliased tensor pointer");
  ET_REQUIRE(h, m >= 0 && k >= 1 && k % 32 == 0, "k must be a positive multiple of 32");
  if ((uint64_t)m * k / 8 >= 0x80000000ull) return fail(h, ET_UNSUPPORTED, "tensor too large for one launch");
  et::launch_split_rows((const float*)src, (uint16_t*)dst, m, k, m_dev, (hipStream_t)stream);
  return check_launch(h, "split rows");
}

et_status et_gemm_split(et_handle h, const void* A, const void* Bt, void* C, const void* bias, int gelu, int m, int n,
                        int k, const int32_t* m_dev, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, A && Bt && C, "null tensor pointer");
  ET_REQUIRE(h, !gelu || bias, "null bias");
  ET_REQUIRE(h, m >= 0 && n >= 1 && k >= 1, "bad dimensions");
  if (!et::gemm_split_supported(n, k) || (gelu && n % 32 != 0))
    return fail(h, ET_UNSUPPORTED, "et_gemm_split needs k % 32 == 0 and n % 4 == 0 (with gelu n % 32 == 0)");
  et::GemmGroups g;
  g.groups = 1;
  g.A[0] = A; g.B[0] = Bt; g.bias[0] = bias;
  g.gelu = gelu != 0;
  et::launch_gemm_split(g, C, n, m, n, k, m_dev, (hipStream_t)stream);
  return check_launch(h, "et_gemm_split");
}

size_t et_pair_weight_stats(int n, int k) { return n < 1 || k < 64 ? 0 : et::pair_weight_stats(n, k); }

size_t et_pair_weight_workspace_bytes(int n, int k) { return n < 1 || k < 1 ? 0 : et::pair_weight_tops(n, k) * sizeof(float); }

et_status et_pair_rows(et_handle h, const void* src, const et_pair_matrix* dst, int m, int k, const int32_t* m_dev, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, src && dst && dst->rows && dst->exp && dst->norm && src != dst->rows, "null or aliased tensor pointer");
  ET_REQUIRE(h, m >= 0, "bad dimensions");
  if (!et::pair_rows_supported(k)) return fail(h, ET_UNSUPPORTED, "k must be a multiple of 64 up to 2048");
  const et::PairRows out{(_Float16*)dst->rows, dst->exp, dst->norm};
  et::PairRowsJob job;
  job.src = (const float*)src, job.out = out, job.m = m, job.n = k, job.rows_dev = m_dev;
  et::launch_pair_rows(job, (hipStream_t)stream);
  return check_launch(h, "pair rows");
}

et_status et_pair_weight(et_handle h, const void* src, void* dst, int32_t* exp, const void* bias, float* stats, int k, int n,
                         void* workspace, size_t workspace_bytes, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, src && dst && exp && src != dst, "null or aliased tensor pointer");
  ET_REQUIRE(h, stats == nullptr || bias != nullptr, "stats need the bias");
  ET_REQUIRE(h, workspace != nullptr, "null workspace");
  if (!et::gemm_pair_supported(n, k)) return fail(h, ET_UNSUPPORTED, "k must be a multiple of 64 and n of 16");
  if (workspace_bytes < et_pair_weight_workspace_bytes(n, k))
    return fail(h, ET_WORKSPACE_TOO_SMALL, "et_pair_weight needs et_pair_weight_workspace_bytes(n, k)");
  et::PairWeightJobs jobs;
  jobs.job[jobs.count++] = {src, false, k, n, (_Float16*)dst, exp, (float*)workspace, (const float*)bias, stats};
  et::launch_pair_weights(jobs, (hipStream_t)stream);
  return check_launch(h, "weight pairs");
}

et_status et_gemm_pair(et_handle h, const et_pair_matrix* A, const void* Bt, const int32_t* b_exp, const float* b_stats,
                       const void* bias, void* C, int32_t* c_exp, int m, int n, int k, const int32_t* m_dev, void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, A && A->rows && A->exp && Bt && b_exp && C, "null tensor pointer");
  ET_REQUIRE(h, !c_exp || (A->norm && b_stats && bias), "pair rows as the result need the norms, the bias and the weight's stats");
  ET_REQUIRE(h, m >= 0 && n >= 1 && k >= 1, "bad dimensions");
  if (!et::gemm_pair_supported(n, k) || (c_exp && n % 32 != 0))
    return fail(h, ET_UNSUPPORTED, "et_gemm_pair needs k % 64 == 0 and n % 16 == 0 (with c_exp n % 32 == 0)");
  et::PairProduct p;
  p.A[0] = {(_Float16*)A->rows, A->exp, A->norm};
  p.B[0] = (const _Float16*)Bt;
  p.b_exp[0] = b_exp;
  p.bias[0] = (const float*)bias;
  p.stats = b_stats;
  p.c_exp = c_exp;
  et::launch_gemm_pair(p, C, n, m, n, k, m_dev, (hipStream_t)stream);
  return check_launch(h, "et_gemm_pair");
}

namespace {

et_status gemm_bt_impl(et_handle h, et_dtype dtype, const void* A, const void* Bt, void* C, const void* bias, int m, int n,
                       int k, const int32_t* m_dev, void* stream, bool gelu, const char* what) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, dtype == ET_FP16, "dtype must be ET_FP16");
  ET_REQUIRE(h, A && Bt && C, "null tensor pointer");
  ET_REQUIRE(h, !gelu || bias, "null bias");
  ET_REQUIRE(h, m >= 0 && n >= 1 && k >= 1, "bad dimensions");
  if ((uint64_t)m * k * 2 > 0xffffffffull) return fail(h, ET_UNSUPPORTED, "A larger than 4 GB");
  if (!et::gemm_takes_transposed_b(et::DType::F16, m, n, n, k, 1))
    return fail(h, ET_UNSUPPORTED,
                std::string(what) + " needs k % 64 == 0 and n % 8 == 0");
  et::GemmGroups g;
  g.groups = 1;
  g.A[0] = A; g.B[0] = Bt; g.bias[0] = bias;
  g.b_transposed = true;
  g.gelu = gelu;
  g.c_cached = (double)m * ((double)k + n) * 2.0 <= kCachedCallBytes;     // A and C together: a small call
  et::launch_gemm(et::DType::F16, g, C, n, m, n, k, m_dev, (hipStream_t)stream);
  return check_launch(h, what);
}

}  // namespace

et_status et_gemm_bt(et_handle h, et_dtype dtype, const void* A, const void* Bt, void* C, const void* bias, int m, int n,
                     int k, const int32_t* m_dev, void* stream) {
  return gemm_bt_impl(h, dtype, A, Bt, C, bias, m, n, k, m_dev, stream, false, "et_gemm_bt");
}

et_status et_gemm_bt_bias_gelu(et_handle h, et_dtype dtype, const void* A, const void* Bt, void* C, const void* bias,
                               int m, int n, int k, const int32_t* m_dev, void* stream) {
  return gemm_bt_impl(h, dtype, A, Bt, C, bias, m, n, k, m_dev, stream, true, "et_gemm_bt_bias_gelu");
}

namespace {
int current_cu_count() {
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess || prop.multiProcessorCount <= 0)
    return 256;
  return prop.multiProcessorCount;
}
}  // namespace

size_t et_calibrate_mfma_sink_bytes(et_handle h) {
  Entry entry(h);
  if (entry.status != ET_OK) return 0;
  return et::mfma_ceiling_sink_bytes(current_cu_count());
}

et_status et_calibrate_mfma(et_handle h, int random_operands, int iters, void* sink, size_t sink_bytes, double* flops,
                            void* stream) {
  Entry entry(h);
  et_status s = entry.status;
  if (s != ET_OK) return s;
  ET_REQUIRE(h, sink && flops, "null pointer");
  ET_REQUIRE(h, iters >= 1 && iters <= (1 << 22), "iters must be in 1 .. 4194304");
  const int cus = current_cu_count();
  if (sink_bytes < et::mfma_ceiling_sink_bytes(cus)) return fail(h, ET_WORKSPACE_TOO_SMALL, "sink buffer too small");
  *flops = et::launch_mfma_ceiling(random_operands != 0, cus, iters, (float*)sink, (hipStream_t)stream);
  return check_launch(h, "MFMA calibration");
}

}  // extern "C"
