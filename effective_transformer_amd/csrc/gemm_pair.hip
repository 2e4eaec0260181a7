// fp32 GEMMs of the encoder layer on the fp16 matrix cores of gfx950 (replace the fp32 cublasGemmEx call sites,
// reference: tf_op/bert_transformer_op.cu.cc:110-141, 200-240), for hidden sizes of 512 and more in multiples of 64.
//
// A float x of a row whose values stay below 2^(e+15) is held as the pair h + l of halves, h = x 2^-e rounded to nearest and
// l the rest rounded to nearest (the two-piece split of Ootomo and Yokota, "Recovering single precision accuracy from Tensor Cores
// while surpassing the FP32 theoretical peak performance", 2022, with an exponent per row): off by at most 2^-23 of x, or, below
// 2^-16 of the row's bound, where l is a subnormal half, 2^-39 of the bound.  A product of two such floats is h.h + h.l + l.h (l.l
// is at most 2^-22 of it, 2^-25 in the mean), three products for v_mfma_f32_16x16x32_f16 where three bfloat16 pieces take six
// (gemm_split.hip).  They are summed in chunks of 64 k, smallest first within each 32, and the chunks in float adds: fewer
// roundings at the size of the whole sum than one chain of matrix instructions has.  Error
// against float64, normal operands, relative (this / three bfloat16 pieces / fp32 matrix instructions): k = 512 1.22e-7 /
// 1.27e-7 / 3.8e-7, 768 1.28e-7 / 1.59e-7, 1024 1.34e-7 / 1.87e-7, 3072 1.73e-7 / 3.41e-7 / 9.9e-7, 4096 1.87e-7 / 3.96e-7; all
// operands positive: 5.0e-8 / 1.21e-7 at k = 512, 1.1e-7 / 3.05e-7 at 3072.  Below k = 512 the three pieces are closer, and
// layers of smaller hidden sizes keep them.  Infinities and NaNs give NaN.
//
// Both operands come as "pair rows": [row][k / 32][h, l][32] halves, one 128-byte line per row and k-step of 32.  Both have
// an exponent per row, which are applied to the result.  Input and LayerNorm take it from the row's
// largest value; the FFN's first product, whose workgroups see parts of a row, takes a bound instead (pair_gelu_bound).  The
// attention kernels see a head of a row, 64 values: context rows have an exponent per 64 k, and the output product (HEADS) weighs
// its chunks where it adds them up (20375 rows, attention and product: 141 us with a launch in between that found the rows' own
// exponents, 130 us; 3820 rows 57 and 53; one tile's worth, 160 rows, level; encoders of 12 layers 1 to 2 %).  Weights
// are taken anew by every layer call: pair_weight_top_kernel looks for the largest value of each column, pair_weight_kernel
// writes the rows (8.4 + 10.2 us per layer of BERT-base, split rows 15).
// Bound: at large m the power limit of the matrix cores (20375 rows, k = 768 / n = 2304, 768, 3072 + GELU and k = 3072 / n = 768:
// 171, 68, 259, 226 us in the layer, 1265, 1060, 1113, 1276 TFLOP/s of 16-bit products, 4 to 6 % less on slower cards; split rows
// 307, 112, 451, 413); below a round of the chip the k loop of one tile, which the LDS bounds (134 rows of at
// most 256: 9.4, 6.8, 13.1, 13.9 us; split rows 15.2, 8.7, 16.1, 21.3).
#include <algorithm>
#include <atomic>
#include <iterator>
#include <type_traits>

#include "et_device.hpp"
#include "kernels.hpp"

namespace et {

namespace {

constexpr int kXcds = 8;
constexpr int kLine = 128;                      // bytes of a row and k-step of 32

struct PairGemmArgs {
  const _Float16* A[3];
  const _Float16* B[3];
  const int32_t* a_exp[3];
  const int32_t* b_exp[3];
  const float* bias[3];
  void* C;
  const int32_t* rows_dev;
  // GELU: what bounds the rows of C (pair_gelu_bound)
  const float* a_norm;
  const float* b_stats;
  int32_t* c_exp;
  int stat_pairs;
  int ldc, m_bound, n, k;
  int tiles_n, groups;                          // column tiles per group of B
  int columns;                                  // the tile order takes the column tiles of all groups this many at a time
};

#define ET_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

template <int VM>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (15 << 8) | ((VM >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14)); }
__device__ __forceinline__ void barrier_only() { asm volatile("s_barrier" ::: "memory"); }

// v[i][r]: what lane 4 i + r of the 16 lanes around this one holds
template <int I, int MI>
__device__ __forceinline__ void from_lanes(float4v (&v)[MI], float x) {
  v[I] = float4v{dpp_f32<kDppRowNewBcast + 4 * I>(0.f, x), dpp_f32<kDppRowNewBcast + 4 * I + 1>(0.f, x),
                 dpp_f32<kDppRowNewBcast + 4 * I + 2>(0.f, x), dpp_f32<kDppRowNewBcast + 4 * I + 3>(0.f, x)};
  if constexpr (I + 1 < MI) from_lanes<I + 1>(v, x);
}

// WM x WN wavefronts of MI x NJ blocks of 16 x 16, a ring of ST stages of KS k-steps in LDS.
template <int WM, int WN, int MI, int NJ, int ST, int KS>
struct PairTile {
  static constexpr int BM = WM * 16 * MI, BN = WN * 16 * NJ, WAVES = WM * WN, THREADS = WAVES * kWave;
  static constexpr int A_BYTES = BM * kLine, STEP = (BM + BN) * kLine, SLOT = KS * STEP, SMEM = ST * SLOT;
  static constexpr int DMA_ALL = STEP / 1024, DMA = (DMA_ALL + WAVES - 1) / WAVES;     // instructions per k-step: all, per wavefront
  static constexpr bool BIG = KS == 1;
  static_assert(KS * DMA * (ST - 1) < 64, "the DMA instructions in flight must fit the 6-bit vmcnt");
  static_assert(SMEM <= 160 * 1024, "LDS");
};

// Persistent: a workgroup per CU walks the tiles of its XCD's band, one DMA stream across tile boundaries.
// Per k-step the products run as h.l, l.h, h.h (A's piece first); the chunk's accumulator starts from zero every second k-step
// and is added to the sum there.  The order does not depend on the tile, so a row has the same bits in every batch.
//   KS = 1 (large tiles, two wavefronts per SIMD): the operands of a group of MI x NJ MFMAs are read from LDS under the group in
//   front of it.  At the bar every piece of the k-step has been read: one barrier there frees the slot for the DMA ST k-steps
//   ahead.
//   KS = 2 (small tiles): a stage is a chunk; one barrier per stage, the next stage's operands are read into a second register
//   set under this one's MFMAs.
// GELU: C = gelu(A.B + bias) as pair rows with their exponents in c_exp; otherwise C is float, + bias if given.  HEADS: A's rows
// have an exponent per chunk.
template <int WM, int WN, int MI, int NJ, int ST, int KS, bool GELU, bool HEADS>
__global__ __launch_bounds__(WM * WN * kWave) void gemm_pair_kernel(
    // what comes before the first request, as arguments of their own (gemm_f16_bt_kernel has the reason)
    const _Float16* a0, const _Float16* b0, const int32_t* rows_dev, int m_bound, int N, int K, int tiles_n, int groups, int columns,
    const uint32_t* head_exp, PairGemmArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)   // device-only types in the body; the host pass only needs the stub
  using Tile = PairTile<WM, WN, MI, NJ, ST, KS>;
  constexpr int BM = Tile::BM, BN = Tile::BN;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int rows = rows_dev ? *rows_dev : m_bound;
  uint64_t to_a1 = 0, to_a2 = 0, to_b1 = 0, to_b2 = 0;              // from the operands of the first group, in bytes
  if (groups > 1) {
    to_a1 = (uint64_t)args.A[1], to_a2 = (uint64_t)args.A[2], to_b1 = (uint64_t)args.B[1], to_b2 = (uint64_t)args.B[2];
    asm volatile("" : "+s"(rows), "+s"(to_a1), "+s"(to_a2), "+s"(to_b1), "+s"(to_b2));       // all in one go
    to_a1 -= (uint64_t)a0, to_a2 -= (uint64_t)a0, to_b1 -= (uint64_t)b0, to_b2 -= (uint64_t)b0;
  }
  rows = max(min(rows, m_bound), 0);
  const int tiles_m = (int)((unsigned)(rows + BM - 1) / BM), total = tiles_m * tiles_n * groups;      // tiles that hold valid rows
  // workgroups are dealt round-robin to the XCDs: a contiguous band of tiles for each
  const int per_xcd = (total + kXcds - 1) / kXcds;
  const int xcd = blockIdx.x % kXcds, wgs = gridDim.x / kXcds;      // the grid is a multiple of 8
  const int n_loc = max(0, min(per_xcd, total - xcd * per_xcd));
  int idx = blockIdx.x / kXcds;
  if (idx >= n_loc) return;
  const int nst = (int)((unsigned)K / (32 * KS));                                    // stages of a tile
  const uint32_t row_bytes = (uint32_t)K * 4u;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane & 15, g = lane >> 4;

  struct Src {
    __amdgpu_buffer_rsrc_t a, b;
    int m0, n0, grp;
  };
  auto locate = [&](int i) {
    Src t;
    const int tile = xcd * per_xcd + i;
    const int cg = columns == tiles_n * groups ? 0 : uniform_div(tile, tiles_m * columns), in_group = tile - cg * tiles_m * columns;
    const int tm = uniform_div(in_group, columns);
    const int tn_all = cg * columns + (in_group - tm * columns);
    t.grp = groups == 1 ? 0 : 2 - uniform_less(tn_all, tiles_n) - uniform_less(tn_all, 2 * tiles_n);
    t.m0 = tm * BM;
    t.n0 = (tn_all - t.grp * tiles_n) * BN;
    const uint64_t second = t.grp == 1 ? ~0ull : 0ull, third = t.grp == 2 ? ~0ull : 0ull;
    const char *ptr_a = (const char*)a0 + ((to_a1 & second) | (to_a2 & third)), *ptr_b = (const char*)b0 + ((to_b1 & second) | (to_b2 & third));
    // rows at or beyond the valid count and columns at or beyond n read as zero
    t.a = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ptr_a + (size_t)t.m0 * row_bytes), 0,
                                            min(rows - t.m0, BM) * (int)row_bytes, 0x00020000);
    t.b = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ptr_b + (size_t)t.n0 * row_bytes), 0,
                                            min(N - t.n0, BN) * (int)row_bytes, 0x00020000);
    return t;
  };

  // DMA: one instruction fills 1 KB of LDS, eight lines of 128 bytes, their 16-byte chunks XOR-swizzled with row bits 1-3, so
  // that an operand read (16 rows x one chunk) covers all banks evenly.  LDS row j*16+l of a wave's column group holds column
  // NJ*l+j of the group: a lane then owns NJ consecutive columns of C.  Where the instructions do not divide evenly, the last
  // wavefront repeats the last one (same bytes to the same place).
  uint32_t voff[Tile::DMA];
#pragma unroll
  for (int q = 0; q < Tile::DMA; ++q) {
    const int c = min(wave * Tile::DMA + q, Tile::DMA_ALL - 1) * kWave + lane;
    int row = c / 8;
    const uint32_t in_row = (uint32_t)(((c & 7) ^ ((row >> 1) & 7)) * 16);
    if (row >= BM) {
      row -= BM;
      const int in_wave = row % (16 * NJ);
      row = row - in_wave + (in_wave & 15) * NJ + (in_wave >> 4);
    }
    voff[q] = (uint32_t)row * row_bytes + in_row;
  }
  // instructions [q0, q1) of this wave's share of k-step `u` of stage `t` of tile `c` (past its end: of the first stages of
  // tile `n`) into slot `slot`
  auto issue = [&](int slot, int t, int u, const Src& c, const Src& n, int q0, int q1) {
    const bool over = t >= nst;
    const __amdgpu_buffer_rsrc_t ra = over ? n.a : c.a;
    const __amdgpu_buffer_rsrc_t rb = over ? n.b : c.b;
    const int koff = ((over ? t - nst : t) * KS + u) * kLine;
#pragma unroll
    for (int q = q0; q < q1; ++q) {
      const int i = min(wave * Tile::DMA + q, Tile::DMA_ALL - 1);
      unsigned char* dst = smem + slot * Tile::SLOT + u * Tile::STEP + i * 1024;
      if (i < Tile::A_BYTES / 1024) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, ET_LDS_PTR(dst), 16, voff[q], koff, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, ET_LDS_PTR(dst), 16, voff[q], koff, 0, 0);
    }
  };
  auto issue_stage = [&](int slot, int t, const Src& c, const Src& n) {
#pragma unroll
    for (int u = 0; u < KS; ++u) issue(slot, t, u, c, n, 0, Tile::DMA);
  };

  // chunk g of a piece, swizzled: the pieces h and l are chunks 0-3 and 4-7 of a line
  const int sw = (g ^ ((l16 >> 1) & 7)) * 16;
  const int a_rd = (wm * 16 * MI + l16) * kLine, b_rd = Tile::A_BYTES + (wn * 16 * NJ + l16) * kLine;
  auto read_a = [&](half8 (&v)[MI], int slot, int u, int piece) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      v[i] = *reinterpret_cast<const half8*>(smem + slot * Tile::SLOT + u * Tile::STEP + a_rd + i * 16 * kLine + (sw ^ (piece * 64)));
  };
  auto read_b = [&](half8 (&v)[NJ], int slot, int u, int piece) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      v[j] = *reinterpret_cast<const half8*>(smem + slot * Tile::SLOT + u * Tile::STEP + b_rd + j * 16 * kLine + (sw ^ (piece * 64)));
  };

  float4v sum[MI][NJ], acc[MI][NJ];
  const float4v zero = {0.f, 0.f, 0.f, 0.f};
  // HEADS: behind the ring the exponent of each row of the tile, the largest of its chunks', and per chunk 2^(the chunk's exponent -
  // the row's) as the upper half of the float.  Eight lanes see to four rows (a word of every chunk), every eighth chunk each;
  // `exps` is requested early.
  constexpr int kExpChunks = kMaxHeadExps / 8;
  static_assert(BM * 2 <= Tile::THREADS, "eight lanes for four rows");
  int* const row_exp = reinterpret_cast<int*>(smem + Tile::SMEM);
  uint16_t* const chunk_scale = reinterpret_cast<uint16_t*>(smem + Tile::SMEM + BM * 4);
  uint32_t exps[kExpChunks] = {};
  const int exp_first = threadIdx.x & 7, exp_rows = (int)(threadIdx.x >> 3) * 4;
  auto request_exps = [&](int m0) {
    const int chunks = (int)((unsigned)K / 64), word = min(m0 + min(exp_rows, BM - 4), rows - 1) >> 2;
#pragma unroll
    for (int u = 0; u < kExpChunks; ++u)
      exps[u] = head_exp[(size_t)min(exp_first + u * 8, chunks - 1) * ((unsigned)(m_bound + 3) / 4) + word];
  };
  // (what is made of them stays behind this: between the first requests it would wait for them)
  auto hold_exps = [&] {
#pragma unroll
    for (int u = 0; u < kExpChunks; ++u) asm volatile("" : "+v"(exps[u]));
  };
  auto write_exps = [&] {
    const int chunks = (int)((unsigned)K / 64);
    int top[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      top[r] = -128;
#pragma unroll
      for (int u = 0; u < kExpChunks; ++u)       // (the last chunk stands for those behind it)
        top[r] = max(top[r], (int)(exps[u] << (24 - 8 * r)) >> 24);
      top[r] = max(top[r], dpp_i32<kDppQuadXor1>(top[r], top[r]));
      top[r] = max(top[r], dpp_i32<kDppQuadXor2>(top[r], top[r]));
      top[r] = max(top[r], dpp_i32<kDppRowHalfMirror>(top[r], top[r]));
    }
    if (exp_rows >= BM) return;
    typedef int int4v __attribute__((ext_vector_type(4)));
    if (exp_first == 0) *reinterpret_cast<int4v*>(row_exp + exp_rows) = int4v{top[0], top[1], top[2], top[3]};
#pragma unroll
    for (int u = 0; u < kExpChunks; ++u) {
      if (exp_first + u * 8 >= chunks) break;
      uint32_t s[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = (uint32_t)max(127 + ((int)(exps[u] << (24 - 8 * r)) >> 24) - top[r], 0) << 7;
      *reinterpret_cast<u32x2*>(chunk_scale + (exp_first + u * 8) * BM + exp_rows) = u32x2{s[0] | s[1] << 16, s[2] | s[3] << 16};
    }
  };
  // Read through a vector of halves, as the operands are: in front of a read through a struct the compiler waits for all DMA in
  // flight, every chunk.  Without that, with all first requests out before the exponents are waited for, and with none after the
  // last tile: one layer of 8 x 32 83.1 -> 81.5 us, 12 layers of 15 x 379 2790 -> 2781, of 500 x 64 11083 -> 11044.
  half4 scales[MI] = {};                         // of the chunk that is added next (in front of a tile's first one, of anything: acc is 0)
  auto read_scales = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < MI; ++i) scales[i] = *reinterpret_cast<const half4*>(smem + Tile::SMEM + BM * 4 + 2 * (chunk * BM + wm * 16 * MI + i * 16 + g * 4));
  };
  // the sum with the chunk whose products are in acc
  auto folded = [&](int i, int j, int r) {
    if constexpr (!HEADS) return sum[i][j][r] + acc[i][j][r];
    const u32x2 s2 = __builtin_bit_cast(u32x2, scales[i]);
    const uint32_t w = r < 2 ? s2.x : s2.y;
    return __builtin_fmaf(acc[i][j][r], __builtin_bit_cast(float, r & 1 ? w & 0xffff0000u : w << 16), sum[i][j][r]);
  };
  // one row of blocks; FIRST: the chunk's first product, behind the fold of the chunk before it
  auto mfma_row = [&](auto FIRSTc, const half8 (&a)[MI], const half8 (&b)[NJ], int i) {
    constexpr bool FIRST = decltype(FIRSTc)::value;
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const int j = (i & 1) ? NJ - 1 - jj : jj;          // only one operand changes from one MFMA to the next
      if constexpr (FIRST) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[i][j][r] = folded(i, j, r);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], zero, 0, 0, 0);
      } else {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
      }
    }
  };
  auto mfma = [&](auto FIRSTc, const half8 (&a)[MI], const half8 (&b)[NJ]) {
#pragma unroll
    for (int i = 0; i < MI; ++i) mfma_row(FIRSTc, a, b, i);
  };
  constexpr std::true_type kFirst{};
  constexpr std::false_type kMore{};

  half8 ah[2][MI], al[MI], bh[NJ], bl[NJ];                       // KS = 1
  half8 pa[2][2][2][MI], pb[2][2][2][NJ];                        // KS = 2: [register set][k-step][piece]

  Src cur = locate(idx), nxt = cur;
  if constexpr (HEADS) request_exps(cur.m0);
#pragma unroll
  for (int s = 0; s < ST; ++s) issue_stage(s, min(s, nst - 1), cur, cur);
  // GELU: what bounds the rows of C, the same for every row.  Small tiles look at it, and at all that the epilogue reads, behind
  // the k loop: their launches take little longer than a round trip or two.
  PairBounds bounds;
  PairStats stats;
  if constexpr (GELU) pair_stats_request(args.b_stats, args.stat_pairs, (int)((unsigned)(N + 63) / 64), stats);
  wait_vmcnt<KS * Tile::DMA*(ST - 1)>();
  if constexpr (HEADS) {
    hold_exps();
    write_exps();
    wait_lgkmcnt0();
  }
  barrier_only();
  auto read_set = [&](half8 (&a)[2][2][MI], half8 (&b)[2][2][NJ], int slot) {
#pragma unroll
    for (int u = 0; u < KS; ++u)
#pragma unroll
      for (int piece = 0; piece < 2; ++piece) {
        read_a(a[u][piece], slot, u, piece);
        read_b(b[u][piece], slot, u, piece);
      }
  };
  if constexpr (Tile::BIG) {
    read_a(ah[0], 0, 0, 0);
    read_b(bl, 0, 0, 1);
  } else {
    read_set(pa[0], pb[0], 0);
  }

  if constexpr (GELU && Tile::BIG) bounds = pair_stats_max(args.b_stats, args.stat_pairs, (int)((unsigned)(N + 63) / 64), stats);

  int s = 0;                                     // slot of the current stage
  bool first_tile = true;
  while (true) {
    const int nidx = idx + wgs;
    const bool has_next = nidx < n_loc;
    if (has_next) nxt = locate(nidx);            // otherwise the stream re-loads this tile; the data is never used
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) sum[i][j] = acc[i][j] = zero;
    const int col = cur.n0 + wn * 16 * NJ + l16 * NJ;
    typedef float fvec __attribute__((ext_vector_type(NJ)));
    typedef int int4v __attribute__((ext_vector_type(4)));
    fvec bias = {};
    int ce[NJ] = {};
    int4v re[MI] = {};
    const int row0 = cur.m0 + wm * 16 * MI + g * 4;
    // Pair rows out: the 16 lanes that store the same 4 MI rows see to one row's exponent each, and hand it round (every lane for
    // all of them was a fifth of an epilogue's instructions: store_pair has the figure).
    const int own_row = row0 + min(l16 >> 2, MI - 1) * 16 + (l16 & 3);
    float own_norm = 0.f;
    auto request = [&](const int32_t* a_exp, const int32_t* b_exp, const float* add, const float* norm) {
      if constexpr (GELU) own_norm = norm[own_row];
      if (col >= N) return;
#pragma unroll
      for (int j = 0; j < NJ; ++j) ce[j] = b_exp[col + j];
      if (add != nullptr) bias = *reinterpret_cast<const fvec*>(add + col);
      // (the row arrays reach beyond the last tile: PairRows)
#pragma unroll
      for (int i = 0; i < MI; ++i)
        if constexpr (!HEADS) re[i] = *reinterpret_cast<const int4v*>(a_exp + row0 + i * 16);
    };
    if constexpr (!Tile::BIG) request(args.a_exp[cur.grp], args.b_exp[cur.grp], args.bias[cur.grp], args.a_norm);
    if constexpr (Tile::BIG) {
      auto step = [&](auto Pc, int t) {
        constexpr int P = decltype(Pc)::value;
        read_a(al, s, 0, 1);
        read_b(bh, s, 0, 0);
        mfma(std::integral_constant<bool, P == 0>{}, ah[P], bl);
        __builtin_amdgcn_sched_barrier(0);
        // this wave's share of k-step t+1 has landed, those behind it may fly; right after a tile boundary all of them
        // were confirmed before the C stores went out
        if (first_tile || t >= ST - 1) wait_vmcnt<Tile::DMA*(ST - 2)>();
        wait_lgkmcnt0();                           // its last reads of slot s are complete
        barrier_only();
        if constexpr (HEADS && P == 1) read_scales(t >> 1);
        const int s1 = s + 1 == ST ? 0 : s + 1;
        // the DMA instructions go out between the rows of MFMAs: in one piece they would keep the wavefront from issuing
        constexpr int kPer = (Tile::DMA + 2 * MI - 1) / (2 * MI);
        read_a(ah[1 - P], s1, 0, 0);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          mfma_row(kMore, al, bh, i);
          issue(s, t + ST, 0, cur, nxt, min(i * kPer, Tile::DMA), min((i + 1) * kPer, Tile::DMA));
          __builtin_amdgcn_sched_barrier(0);
        }
        read_b(bl, s1, 0, 1);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          mfma_row(kMore, ah[P], bh, i);
          issue(s, t + ST, 0, cur, nxt, min((MI + i) * kPer, Tile::DMA), min((MI + i + 1) * kPer, Tile::DMA));
          __builtin_amdgcn_sched_barrier(0);
        }
        s = s1;
      };
      for (int t = 0; t < nst; t += 2) {           // (K is a multiple of 64)
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
      }
    } else {
      // one stage on register set P
      auto stage = [&](auto Pc, int t) {
        constexpr int P = decltype(Pc)::value;
        if (first_tile || t >= ST - 1) wait_vmcnt<KS * Tile::DMA*(ST - 2)>();       // as above
        wait_lgkmcnt0();
        barrier_only();
        const int s1 = s + 1 == ST ? 0 : s + 1;
        read_set(pa[1 - P], pb[1 - P], s1);
        __builtin_amdgcn_sched_barrier(0);
        mfma(kFirst, pa[P][0][0], pb[P][0][1]);
        if constexpr (HEADS) read_scales(t);
        issue_stage(s, t + ST, cur, nxt);
        mfma(kMore, pa[P][0][1], pb[P][0][0]);
        mfma(kMore, pa[P][0][0], pb[P][0][0]);
        mfma(kMore, pa[P][1][0], pb[P][1][1]);
        mfma(kMore, pa[P][1][1], pb[P][1][0]);
        mfma(kMore, pa[P][1][0], pb[P][1][0]);
        __builtin_amdgcn_sched_barrier(0);
        s = s1;
      };
      int t = 0;
      for (; t + 1 < nst; t += 2) {
        stage(std::integral_constant<int, 0>{}, t);
        stage(std::integral_constant<int, 1>{}, t + 1);
      }
      if (t < nst) {                              // an odd number of stages
        stage(std::integral_constant<int, 0>{}, t);
        wait_lgkmcnt0();
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int piece = 0; piece < 2; ++piece) {
#pragma unroll
            for (int i = 0; i < MI; ++i) pa[0][u][piece][i] = pa[1][u][piece][i];
#pragma unroll
            for (int j = 0; j < NJ; ++j) pb[0][u][piece][j] = pb[1][u][piece][j];
          }
      }
    }
    wait_vmcnt<0>();
    if constexpr (HEADS) {
      if (has_next) request_exps(nxt.m0);
#pragma unroll
      for (int i = 0; i < MI; ++i) re[i] = *reinterpret_cast<const int4v*>(row_exp + wm * 16 * MI + i * 16 + g * 4);
    }
    if constexpr (Tile::BIG) request(args.a_exp[cur.grp], args.b_exp[cur.grp], args.bias[cur.grp], args.a_norm);
    // the loads are waited for here: left pending on the paths that store nothing, they would have the compiler put a wait
    // for every outstanding load, the DMA included, in front of the k loop's reuse of their registers
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float b = bias[j];
      asm volatile("" : "+v"(b), "+v"(ce[j]));
      bias[j] = b;
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) asm volatile("" : "+v"(re[i]));
    if constexpr (GELU) asm volatile("" : "+v"(own_norm));
    if (HEADS && has_next) {
      hold_exps();
      wait_lgkmcnt0();                             // everybody has read what this tile needs of the exponents:
      barrier_only();
      write_exps();                                // the next one's, which the bar of its first step shows to all
    }
    if constexpr (GELU && !Tile::BIG)
      if (first_tile) bounds = pair_stats_max(args.b_stats, args.stat_pairs, (int)((unsigned)(N + 63) / 64), stats);
    float4v scale[MI];
    if constexpr (GELU) {                          // (every lane is active here)
      const int e = pair_exponent(pair_gelu_bound(own_norm, bounds));
      from_lanes<0>(scale, pair_scale(e));
      if (cur.n0 == 0 && wn == 0 && l16 < 4 * MI && own_row < rows) args.c_exp[own_row] = e;
    }
    if (col < N) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = row0 + i * 16 + r;
          if (row >= rows) continue;
          fvec o;
#pragma unroll
          for (int j = 0; j < NJ; ++j) o[j] = __builtin_ldexpf(folded(i, j, r), re[i][r] + ce[j]) + bias[j];
          if constexpr (GELU) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) o[j] *= gelu_cdf(o[j], o[j] * o[j] * o[j]);
            store_pair<NJ>((_Float16*)args.C + (size_t)row * 2 * args.ldc, cur.grp * N + col, o, scale[i][r]);
          } else {
            *reinterpret_cast<fvec*>((float*)args.C + (size_t)row * args.ldc + (size_t)cur.grp * N + col) = o;
          }
        }
    }
    if (!has_next) break;
    idx = nidx;
    cur = nxt;
    first_tile = false;
  }
  wait_vmcnt<0>();                               // no DMA may still target this workgroup's LDS when it ends
#else
  (void)args;
#endif
}

int device_cu_count() {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cus[kMaxDevices] = {};      // handles on several GPUs may launch from different threads
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    hipDeviceProp_t prop;
    n = hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Tile of a launch.  Below a round of the chip a launch takes the k loop of one tile, so small problems want small tiles;
// large ones want the tile with the fewest operand bytes per product.  A launch takes rounds of tiles over the CUs, each
// as long as its k-steps and a part for filling the ring and storing C.
// 16 x 32 is for launches of one round: a k loop of small tiles is bound by what the LDS takes in and gives out, 12 KB and 16 KB a
// stage of 64 k where 32 x 32 has 16 and 32 (us a launch, 32 x 32 and it: k = 2048, 16 to 64 rows to 768 columns 9.8 and 8.6, 160 rows 10.3 and
// 9.3; k = 768 5.6 and 5.3; k = 512, 240 rows to 512 columns 4.7 and 4.6; in two rounds 300 rows to 768 5.7 and 9.0).
enum PairPick { p256x128, p192x128, p128x128, p96x128, p64x128, p64x64, p32x64, p32x32, p16x32, kPairPicks };
PairPick pick_pair_tile(int m, int n, int k, int groups, bool heads) {
  static constexpr struct { int bm, bn; float step; } kTiles[] = {
      {256, 128, 0.8f}, {192, 128, 0.66f}, {128, 128, 0.48f}, {96, 128, 0.4f}, {64, 128, 0.3f}, {64, 64, 0.19f}, {32, 64, 0.135f}, {32, 32, 0.085f}, {16, 32, 0.07f}};
  const long cus = device_cu_count();
  int best = 0;
  float best_cost = 0.f;
  // (256 rows' exponents of more than 30 chunks do not fit the LDS beside the ring)
  const int first = heads && k > 30 * 64 ? 1 : 0;
  for (int i = first; i < (int)std::size(kTiles); ++i) {
    const long tiles = (long)((m + kTiles[i].bm - 1) / kTiles[i].bm) * ((n + kTiles[i].bn - 1) / kTiles[i].bn) * groups;
    const float cost = (float)((tiles + cus - 1) / cus) * (kTiles[i].step * (float)(k / 32) + 3.f);
    if (i == first || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return (PairPick)best;
}

// `columns` of a launch of one round: the strips of columns with which an XCD's band of tiles touches the fewest operand rows, which is
// what its L2 has to fetch (a band along all columns fetches all of the weights).  us a launch, one strip and so, k = 768: 160 rows to 768
// columns 6.1 -> 5.6, 240 rows 6.5 -> 5.6, 64 rows to 2304 6.2 -> 5.9, 160 rows to 2304 7.9 -> 7.6.  Only where they save more than a
// quarter and the weights are twice as long as A, whose rows the strips fetch more often (480 rows to 768 columns in strips: 12 layers
// 1048 -> 1055 us).
int one_round_columns(int columns, int tiles_m, int tiles_n, int bm, int bn) {
  const int band = (tiles_m * tiles_n + kXcds - 1) / kXcds;
  auto rows = [&](int wide) {
    const int strip = tiles_m * wide;
    if (band <= strip) return std::min(tiles_m, (band + wide - 1) / wide) * bm + std::min(band, wide) * bn;
    return tiles_m * bm + (band + strip - 1) / strip * wide * bn;
  };
  if (tiles_n * bn < 2 * tiles_m * bm) return columns;
  int best = columns, limit = (3 * rows(columns) - 1) / 4;
  for (int strips = 2; strips <= tiles_n; ++strips) {
    if (tiles_n % strips != 0) continue;
    const int r = rows(tiles_n / strips);
    if (r <= limit) best = tiles_n / strips, limit = r - 1;
  }
  return best;
}

template <int WM, int WN, int MI, int NJ, int ST, int KS>
void launch_tile(PairGemmArgs a, bool gelu, int groups, const uint32_t* head_exp, hipStream_t stream) {
  using Tile = PairTile<WM, WN, MI, NJ, ST, KS>;
  a.tiles_n = (a.n + Tile::BN - 1) / Tile::BN;
  a.groups = groups;
  const int tiles_n_all = a.tiles_n * groups;
  // The workgroups of an XCD advance through k side by side, so what its L2 has to deliver per k-step is the distinct
  // rows of A and columns of B they touch: about square blocks of tiles are the best.  Wide outputs take their column
  // tiles in groups of about 1024 columns.
  a.columns = tiles_n_all;
  for (int c = 2; c <= tiles_n_all; ++c)
    if (tiles_n_all % c == 0 && tiles_n_all / c * Tile::BN >= 768) a.columns = tiles_n_all / c;
  const int tiles_m = (a.m_bound + Tile::BM - 1) / Tile::BM, tiles = tiles_m * tiles_n_all;
  if (tiles <= device_cu_count()) a.columns = one_round_columns(a.columns, tiles_m, tiles_n_all, Tile::BM, Tile::BN);
  // (a stream of fewer stages than the ring holds must not cross into a second tile)
  const int grid = ((a.k / (32 * KS) < ST ? tiles : std::min(tiles, device_cu_count())) + kXcds - 1) / kXcds * kXcds;
  auto go = [&](auto kern) {
    auto exps = [&](int chunks) { return head_exp ? Tile::BM * (4 + 2 * chunks) : 0; };
    const int lds = Tile::SMEM + exps(a.k / 64);
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), std::min(Tile::SMEM + exps(kMaxHeadExps), 160 * 1024));
    kern<<<grid, Tile::THREADS, lds, stream>>>(a.A[0], a.B[0], a.rows_dev, a.m_bound, a.n, a.k, a.tiles_n, groups, a.columns, head_exp, a);
  };
  if (gelu) go(gemm_pair_kernel<WM, WN, MI, NJ, ST, KS, true, false>);
  else if (head_exp) go(gemm_pair_kernel<WM, WN, MI, NJ, ST, KS, false, true>);
  else go(gemm_pair_kernel<WM, WN, MI, NJ, ST, KS, false, false>);
}

void launch_pick(PairPick pick, const PairGemmArgs& a, bool gelu, int groups, const uint32_t* head_exp, hipStream_t stream) {
  switch (pick) {
    case p256x128: return launch_tile<4, 2, 4, 4, 3, 1>(a, gelu, groups, head_exp, stream);
    case p192x128: return launch_tile<4, 2, 3, 4, 3, 1>(a, gelu, groups, head_exp, stream);
    case p128x128: return launch_tile<2, 4, 4, 2, 4, 1>(a, gelu, groups, head_exp, stream);
    case p96x128: return launch_tile<2, 4, 3, 2, 4, 1>(a, gelu, groups, head_exp, stream);
    case p64x128: return launch_tile<2, 4, 2, 2, 3, 2>(a, gelu, groups, head_exp, stream);
    case p64x64: return launch_tile<4, 2, 1, 2, 4, 2>(a, gelu, groups, head_exp, stream);
    case p32x64: return launch_tile<2, 4, 1, 1, 5, 2>(a, gelu, groups, head_exp, stream);
    case p32x32: return launch_tile<2, 2, 1, 1, 6, 2>(a, gelu, groups, head_exp, stream);
    case p16x32: return launch_tile<1, 2, 1, 1, 8, 2>(a, gelu, groups, head_exp, stream);
    default: return;
  }
}

// Rows into pair rows: one wavefront per row, which stays in registers (n <= 256 ITERS, a multiple of 4).  With indices the
// source is the padded tensor, and the packed rows are written as well; then the first workgroup sorts the batch's table.
template <int ITERS>
__device__ __forceinline__ void pair_rows_blocks(const PairRowsJob& job, int block, int blocks) {
  const int first = job.seq_table ? 1 : 0;
  if (first && block == 0) {
    sort_sequences<256>(job.seq_table, job.batch, job.seq_table + job.batch + 1);
    return;
  }
  const int rows = job.rows_dev ? min(*job.rows_dev, job.m) : job.m, n = job.n;
  const int lane = threadIdx.x & (kWave - 1);
  const int vpr = n / 4;
  for (int r = (block - first) * 4 + threadIdx.x / kWave; r < rows; r += (blocks - first) * 4) {
    const size_t from = job.batch_idx ? (size_t)job.batch_idx[r] * job.seq_len + job.word_idx[r] : (size_t)r;
    const float4v* s = reinterpret_cast<const float4v*>(job.src + from * n);
    float4v x[ITERS];
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
      const int c = lane + i * kWave;
      x[i] = float4v{0.f, 0.f, 0.f, 0.f};
      if (c < vpr) {
        x[i] = s[c];
        if (job.packed) reinterpret_cast<float4v*>(job.packed + (size_t)r * n)[c] = x[i];
      }
    }
    store_pair_row<ITERS>(x, vpr, job.out, r, n);
  }
}
template <int ITERS>
__global__ __launch_bounds__(256) void pair_rows_kernel(PairRowsJob job) {
  pair_rows_blocks<ITERS>(job, blockIdx.x, gridDim.x);
}
inline int pair_rows_grid(const PairRowsJob& job) { return std::min((job.m + 3) / 4, 2048) + (job.seq_table ? 1 : 0); }

// Weights into n pair rows in two launches, whose loads are whole lines (one launch of workgroups that hold all k of 16 columns
// took 35 .. 45 us at H = 768, of 32 columns with 4 x 8 values a lane 24: one workgroup a CU, whose reads and writes take turns; exponents that go by chunks of 64 k and are applied where a chunk is added need one launch, and
// cost the products 3 to 20 %).  First the largest value of each column in blocks of 256 k, as [k / 256][n].
struct PairWeightArgs {
  PairWeightJobs jobs;
  int tile_begin[PairWeightJobs::kMax + 1];
};
constexpr int kTopRows = 256;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// Rows go along in the first blocks: a launch of their own (8 x 32 tokens: 4 us) would only stand in front of this one.
struct PairRowsArgs {
  PairRowsJob job[2];
  int blocks[2];
};
__global__ __launch_bounds__(256) void pair_weight_top_kernel(PairWeightArgs args, BatchJobs batch, PairRowsArgs rows) {
  __shared__ union {
    float part[16][64];
    int32_t starts[kTableBatch + 1];
  } lds;
  float (&part)[16][64] = lds.part;
  int wg = blockIdx.x;
  if (wg < batch.blocks) {
    batch_job_block(batch, wg, lds.starts);
    return;
  }
  wg -= batch.blocks;
  if (wg < rows.blocks[0] + rows.blocks[1]) {
    const int which = wg < rows.blocks[0] ? 0 : 1;
    const PairRowsJob& job = rows.job[which];
    const int block = wg - (which ? rows.blocks[0] : 0), blocks = rows.blocks[which];
    switch ((job.n / 4 + kWave - 1) / kWave) {
      case 2: return pair_rows_blocks<2>(job, block, blocks);      // (layers on pair rows have 512 values a row and more)
      case 3: return pair_rows_blocks<3>(job, block, blocks);
      case 4: return pair_rows_blocks<4>(job, block, blocks);
      case 5: case 6: return pair_rows_blocks<6>(job, block, blocks);
      default: return pair_rows_blocks<8>(job, block, blocks);
    }
  }
  wg -= rows.blocks[0] + rows.blocks[1];
  int job = 0;
  while (job + 1 < args.jobs.count && wg >= args.tile_begin[job + 1]) ++job;
  const PairWeightJob& jb = args.jobs.job[job];
  const int K = jb.k, N = jb.n, tiles_n = (N + 63) / 64;
  const int t = wg - args.tile_begin[job];
  const int block = t / tiles_n, k0 = block * kTopRows, n0 = (t - block * tiles_n) * 64;
  if (jb.src_split) {                            // rows of three bfloat16 pieces: four lanes per row, every fourth 8 k each
    // (64 consecutive k a lane, value by value: a layer of 32 positions from split copies 74 us, so 69; from floats 67)
    const int r = threadIdx.x >> 2, c = (threadIdx.x & 3) * 8;
    float top = 0.f;
    if (n0 + r < N) {
      const __bf16* p = (const __bf16*)jb.src + (size_t)(n0 + r) * K * 3 + (size_t)(k0 >> 5) * 96 + c;
      const int lines = min(K - k0, kTopRows) / 32;
#pragma unroll 4
      for (int i = 0; i < lines; ++i) {
        const bf16x8 h = *reinterpret_cast<const bf16x8*>(p + i * 96), m = *reinterpret_cast<const bf16x8*>(p + i * 96 + 32),
                     l = *reinterpret_cast<const bf16x8*>(p + i * 96 + 64);
#pragma unroll
        for (int j = 0; j < 8; ++j) top = fmaxf(top, fabsf(((float)h[j] + (float)m[j]) + (float)l[j]));
      }
    }
    top = fmaxf(top, dpp_f32<kDppQuadXor1>(top, top));
    top = fmaxf(top, dpp_f32<kDppQuadXor2>(top, top));
    if (n0 + r < N && (threadIdx.x & 3) == 0) jb.top[(size_t)block * N + n0 + r] = top;
    return;
  }
  const float* __restrict__ src = (const float*)jb.src;
  const int r = threadIdx.x >> 4, c = (threadIdx.x & 15) * 4;
  float4v v[kTopRows / 16];
#pragma unroll
  for (int u = 0; u < kTopRows / 16; ++u) {
    v[u] = float4v{0.f, 0.f, 0.f, 0.f};
    if (k0 + u * 16 + r < K && n0 + c < N) v[u] = *reinterpret_cast<const float4v*>(src + (size_t)(k0 + u * 16 + r) * N + n0 + c);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float top = 0.f;
#pragma unroll
    for (int u = 0; u < kTopRows / 16; ++u) top = fmaxf(top, fabsf(v[u][j]));
    part[r][c + j] = top;
  }
  __syncthreads();
  if (threadIdx.x < 64 && n0 + (int)threadIdx.x < N) {
    float top = part[0][threadIdx.x];
#pragma unroll
    for (int i = 1; i < 16; ++i) top = fmaxf(top, part[i][threadIdx.x]);
    jb.top[(size_t)block * N + n0 + threadIdx.x] = top;
  }
}

// Then 64 x 64 tiles through LDS.  All workgroups are on the chip at once, so the launch takes as long as what stands in front of
// a workgroup's stores: the tile's loads go out first, the columns' largest values behind them, a quarter of a column's to each
// wavefront (28 MB at H = 768: 11.3 -> 10.2 us, 5.6 TB/s of reads and writes; one wavefront that went through a column's values
// one by one before it asked for the tile; tiles on the XCD that read them in the launch before: 10.3).
__global__ __launch_bounds__(256) void pair_weight_kernel(PairWeightArgs args) {
  __shared__ float tile[64][65];
  __shared__ float part[3][4];
  __shared__ float tops[4][64];
  int job = 0;
  while (job + 1 < args.jobs.count && (int)blockIdx.x >= args.tile_begin[job + 1]) ++job;
  const PairWeightJob& jb = args.jobs.job[job];
  const int K = jb.k, N = jb.n, tiles_n = (N + 63) / 64;
  const int t = blockIdx.x - args.tile_begin[job];
  const int chunk = t / tiles_n, k0 = chunk * 64, n0 = (t - chunk * tiles_n) * 64;
  auto find_tops = [&]() {
    const int wave = threadIdx.x / kWave, c = threadIdx.x & (kWave - 1), blocks = (K + kTopRows - 1) / kTopRows;
    float top = 0.f;
    if (n0 + c < N) {
      for (int b0 = 0; b0 < blocks; b0 += 16) {  // (blocks past the last one: the last one again)
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = jb.top[(size_t)min(b0 + 4 * u + wave, blocks - 1) * N + n0 + c];
#pragma unroll
        for (int u = 0; u < 4; ++u) top = fmaxf(top, v[u]);
      }
    }
    tops[wave][c] = top;
  };
  if (jb.src_split) {                            // rows of three bfloat16 pieces, whose sum is the float
    bf16x8 h[2], m[2], l[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = threadIdx.x + u * 256, r = i >> 3, c = (i & 7) * 8;      // row n0+r, k0+c ..
      if (n0 + r >= N) continue;
      const __bf16* p = (const __bf16*)jb.src + (size_t)(n0 + r) * K * 3 + ((k0 + c) >> 5) * 96 + (c & 31);
      h[u] = *reinterpret_cast<const bf16x8*>(p);
      m[u] = *reinterpret_cast<const bf16x8*>(p + 32);
      l[u] = *reinterpret_cast<const bf16x8*>(p + 64);
    }
    find_tops();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = threadIdx.x + u * 256, r = i >> 3, c = (i & 7) * 8;
      if (n0 + r >= N) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j) tile[r][c + j] = ((float)h[u][j] + (float)m[u][j]) + (float)l[u][j];
    }
  } else {
    const float* __restrict__ src = (const float*)jb.src;
    float4v v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = threadIdx.x + u * 256, r = i >> 4, c = (i & 15) * 4;     // source row k0+r, columns n0+c ..
      v[u] = float4v{0.f, 0.f, 0.f, 0.f};
      if (n0 + c < N) v[u] = *reinterpret_cast<const float4v*>(src + (size_t)(k0 + r) * N + n0 + c);
    }
    find_tops();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = threadIdx.x + u * 256, r = i >> 4, c = (i & 15) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) tile[c + j][r] = v[u][j];
    }
  }
  __syncthreads();
  auto exponent = [&](int r) { return pair_exponent(fmaxf(fmaxf(tops[0][r], tops[1][r]), fmaxf(tops[2][r], tops[3][r]))); };
  if (chunk == 0 && threadIdx.x < 64 && n0 + (int)threadIdx.x < N) jb.exp[n0 + threadIdx.x] = exponent(threadIdx.x);
  float norm = 0.f, bias = 0.f, above = 0.f;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = threadIdx.x + u * 256, r = i >> 3, c = (i & 7) * 8;        // row n0+r of the result, k0+c ..
    if (n0 + r >= N) continue;                   // (whole groups of eight lanes)
    const int e = exponent(r);
    const float by = pair_scale(e);
    float sq = 0.f;
    half8 h, l;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float y = tile[r][c + j] * by;
      h[j] = f2h(y);
      l[j] = f2h(y - h2f(h[j]));
      sq = __builtin_fmaf(y, y, sq);
    }
    _Float16* d = jb.dst + (size_t)(n0 + r) * 2 * K + ((k0 + c) >> 5) * 64 + (c & 31);
    *reinterpret_cast<half8*>(d) = h;
    *reinterpret_cast<half8*>(d + 32) = l;
    if (jb.stats != nullptr) {
      sq += dpp_f32<kDppQuadXor1>(0.f, sq);
      sq += dpp_f32<kDppQuadXor2>(0.f, sq);
      sq += dpp_f32<kDppRowHalfMirror>(0.f, sq);
      norm = fmaxf(norm, __builtin_ldexpf(__builtin_sqrtf(sq), e));
      if (chunk == 0) {
        const float b = jb.bias[n0 + r];
        bias = fmaxf(bias, fabsf(b));
        above = fmaxf(above, b);
      }
    }
  }
  if (jb.stats == nullptr) return;
  // |column| <= sqrt(chunks) times the largest part of a column in one chunk
  norm = wave_max(norm) * __builtin_sqrtf((float)(K / 64));
  bias = wave_max(bias);
  above = wave_max(above);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    part[0][threadIdx.x / kWave] = norm;
    part[1][threadIdx.x / kWave] = bias;
    part[2][threadIdx.x / kWave] = above;
  }
  __syncthreads();
  if (threadIdx.x < (chunk == 0 ? 3 : 2))
    jb.stats[threadIdx.x < 2 ? 2 * t + (int)threadIdx.x : 2 * (K / 64) * tiles_n + t] =
        fmaxf(fmaxf(part[threadIdx.x][0], part[threadIdx.x][1]), fmaxf(part[threadIdx.x][2], part[threadIdx.x][3]));
}

}  // namespace

bool gemm_pair_supported(int n, int k) {
  return k % 64 == 0 && k >= 64 && n % 16 == 0 && (uint64_t)k * 4u * 256u < 0x80000000ull;
}

void launch_pair_rows(const PairRowsJob& job, hipStream_t stream) {
  if (job.m <= 0) return;
  const int grid = pair_rows_grid(job);
  auto go = [&](auto kern) { kern<<<grid, 256, 0, stream>>>(job); };
  switch ((job.n / 4 + kWave - 1) / kWave) {
    case 1: return go(pair_rows_kernel<1>);
    case 2: return go(pair_rows_kernel<2>);
    case 3: return go(pair_rows_kernel<3>);
    case 4: return go(pair_rows_kernel<4>);
    case 5: case 6: return go(pair_rows_kernel<6>);
    case 7: case 8: return go(pair_rows_kernel<8>);
    default: return;                             // (pair_rows_supported)
  }
}

bool pair_rows_supported(int n) { return n % 64 == 0 && n >= 64 && n <= 2048; }

void launch_pair_weights(const PairWeightJobs& jobs, hipStream_t stream, const BatchJobs* batch, const PairRowsJob* rows, int row_jobs) {
  if (jobs.count == 0) return;
  PairWeightArgs a;
  a.jobs = jobs;
  auto grid = [&](int rows) {
    int total = 0;
    for (int j = 0; j < jobs.count; ++j) {
      a.tile_begin[j] = total;
      total += ((jobs.job[j].k + rows - 1) / rows) * ((jobs.job[j].n + 63) / 64);
    }
    for (int j = jobs.count; j <= PairWeightJobs::kMax; ++j) a.tile_begin[j] = total;
    return total;
  };
  const int tops = grid(kTopRows);
  const BatchJobs b = batch ? *batch : BatchJobs();
  PairRowsArgs r = {};
  for (int j = 0; j < row_jobs; ++j) {
    r.job[j] = rows[j];
    r.blocks[j] = rows[j].m > 0 ? pair_rows_grid(rows[j]) : 0;
  }
  pair_weight_top_kernel<<<tops + b.blocks + r.blocks[0] + r.blocks[1], 256, 0, stream>>>(a, b, r);
  if (b.seq_table && !b.one_block_table) launch_seq_order(b.seq_table, b.batch, stream);
  const int tiles = grid(64);
  pair_weight_kernel<<<tiles, 256, 0, stream>>>(a);
}

void launch_gemm_pair(const PairProduct& p, void* C, int ldc, int m_bound, int n, int k, const int32_t* rows_dev,
                      hipStream_t stream) {
  if (m_bound <= 0) return;
  PairGemmArgs a = {};
  for (int i = 0; i < p.groups; ++i) {
    a.A[i] = p.A[i].rows;
    a.a_exp[i] = p.A[i].exp;
    a.B[i] = p.B[i];
    a.b_exp[i] = p.b_exp[i];
    a.bias[i] = p.bias[i];
  }
  a.a_norm = p.A[0].norm;
  a.b_stats = p.stats;
  a.stat_pairs = (int)pair_weight_stat_pairs(n, k);
  a.c_exp = p.c_exp;
  a.C = C;
  a.rows_dev = rows_dev;
  a.ldc = ldc;
  a.m_bound = m_bound;
  a.n = n;
  a.k = k;
  launch_pick(pick_pair_tile(m_bound, n, k, p.groups, p.head_exp != nullptr), a, p.c_exp != nullptr, p.groups,
              (const uint32_t*)p.head_exp, stream);
}

}  // namespace et
