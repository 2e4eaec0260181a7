// fp32 GEMMs of the encoder layer on the 16-bit matrix cores of gfx950 (replace the fp32 cublasGemmEx call sites,
// reference: tf_op/bert_transformer_op.cu.cc:110-141, 200-240), for the hidden sizes gemm_pair.hip does not take: multiples of
// 32 below 512, odd multiples of 32, and rows of more than 2048 values.
//
// A float is the exact sum of three bfloat16 numbers h + m + l, each the rest of the ones before it rounded to nearest
// (8 significand bits and a sign apiece cover the 24 bits, in the float's own exponent range).  A product of two such
// floats is nine products of pieces; the three of weight 2^-26 and less (m.l, l.m, l.l) lie below a quarter unit of the
// float product and are left out, the other six go through v_mfma_f32_16x16x32_bf16, each exact and summed in float (splitting
// floats into bfloat16 pieces for such a product is a published method: Henry, Tang and Heinecke, 2019).  Infinities, NaNs and
// magnitudes above 3.38e38 have NaN pieces.  The leading
// products (h.h) and the five corrections have an accumulator of their own: the matrix core cuts an addend that is
// small beside its accumulator, which would otherwise bias every correction towards zero.  Against float64 the result is
// closer than the fp32 matrix instructions' (k = 3072, normal operands: 3.4e-7 relative against 9.9e-7; all operands
// positive: 3.0e-7 against 8.6e-7), at six times the work of a 16-bit product on units sixteen times as fast.
//
// Both operands come as "split rows": [row][k / 32][h, m, l][32] bfloat16, 192 contiguous bytes per row and k-step of 32.
// The kernels that produce A (input, attention, LayerNorm, GELU) write that form themselves; weights are split by every layer
// call unless the caller hands the copies over (15 us per layer of BERT-base in the trace, 9 us of its time).
// Bound: at large m the power limit of the matrix cores (20000 rows, k = 768 / n = 2304, 768, 3072 + GELU and k = 3072 /
// n = 768: 385, 113, 490, 427 us, i.e. 1090 .. 1330 TFLOP/s of 16-bit products; all-zero operands 288, 100, 441, 383 us;
// the fp32 matrix instructions took 617, 211, 780, 767 us); below a round of the chip the k loop of one tile (160 rows:
// 14, 10, 15, 21 us against 17, 17, 19, 59).
#include <algorithm>
#include <atomic>
#include <iterator>
#include <type_traits>

#include "et_device.hpp"
#include "kernels.hpp"

namespace et {

namespace {

constexpr int kXcds = 8;
constexpr int kStepBytes = 192;                 // of a row and k-step

struct SplitGemmArgs {
  const uint16_t* A[3];
  const uint16_t* B[3];
  const float* bias[3];
  void* C;
  const int32_t* rows_dev;
  int ldc, m_bound, n, k;
  int tiles_n, tiles_n_all;                     // column tiles per group of B, and of all groups
  int col_groups;                               // the tile order takes the column tiles in this many groups
};

#define ET_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

template <int VM>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (15 << 8) | ((VM >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14)); }
__device__ __forceinline__ void barrier_only() { asm volatile("s_barrier" ::: "memory"); }

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

// WM x WN wavefronts of MI x NJ blocks of 16 x 16, a ring of ST k-steps in LDS.
template <int WM, int WN, int MI, int NJ, int ST>
struct SplitTile {
  static constexpr int BM = WM * 16 * MI, BN = WN * 16 * NJ, WAVES = WM * WN, THREADS = WAVES * kWave;
  static constexpr int A_BYTES = BM * kStepBytes, SLOT = (BM + BN) * kStepBytes, SMEM = ST * SLOT;
  static constexpr int DMA_ALL = SLOT / 1024, DMA = (DMA_ALL + WAVES - 1) / WAVES;     // instructions: all, per wavefront
  static_assert(DMA * (ST - 1) < 64, "the DMA instructions in flight must fit the 6-bit vmcnt");
  static_assert(SMEM <= 160 * 1024, "LDS");
};

// Persistent: a workgroup per CU walks the tiles of its XCD's band, one DMA stream across tile boundaries.  Per k-step a
// wavefront runs the six products as six groups of MI x NJ MFMAs, ordered so that the operands of the next group are read
// from LDS under the current one and each register set is refilled as soon as its last product has been issued:
// h.h, h.m, h.l, m.h | l.h, m.m (A's piece first).  At the bar every piece of the k-step has been read: one barrier there
// frees the LDS slot for the DMA of the k-step ST ahead, and the h pieces of the next k-step are read behind it.
// The order of the products does not depend on the tile, so a row has the same bits in every batch.
// GELU: C = gelu(A.B + bias) as split rows (the form the next product wants); otherwise C is float, + bias if given.
template <int WM, int WN, int MI, int NJ, int ST, bool GELU>
__global__ __launch_bounds__(WM * WN * kWave) void gemm_split_kernel(SplitGemmArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)   // device-only types in the body; the host pass only needs the stub
  using Tile = SplitTile<WM, WN, MI, NJ, ST>;
  constexpr int BM = Tile::BM, BN = Tile::BN;
  constexpr bool kTwoPerSimd = Tile::WAVES == 8 && MI * NJ >= 12;
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int rows = args.rows_dev ? min(*args.rows_dev, args.m_bound) : args.m_bound;
  const int total = ((rows + BM - 1) / BM) * args.tiles_n_all;      // tiles that hold valid rows
  // workgroups are dealt round-robin to the XCDs: a contiguous band of tiles for each
  const int per_xcd = (total + kXcds - 1) / kXcds;
  const int xcd = blockIdx.x % kXcds, wgs = gridDim.x / kXcds;      // the grid is a multiple of 8
  const int n_loc = max(0, min(per_xcd, total - xcd * per_xcd));
  int idx = blockIdx.x / kXcds;
  if (idx >= n_loc) return;
  const int N = args.n, K = args.k;
  const int nk = K / 32;
  const uint32_t row_bytes = (uint32_t)K * 6u;

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
    const int cpg = args.tiles_n_all / args.col_groups;
    const int per_group = (total / args.tiles_n_all) * cpg;
    const int cg = tile / per_group;
    const int in_group = tile - cg * per_group;
    const int tm = in_group / cpg;
    const int tn_all = cg * cpg + (in_group - tm * cpg);
    t.grp = tn_all / args.tiles_n;
    t.m0 = tm * BM;
    t.n0 = (tn_all - t.grp * args.tiles_n) * BN;
    // rows at or beyond the valid count and columns at or beyond n read as zero
    t.a = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>((const char*)args.A[t.grp] + (size_t)t.m0 * row_bytes), 0,
                                            min(rows - t.m0, BM) * (int)row_bytes, 0x00020000);
    t.b = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>((const char*)args.B[t.grp] + (size_t)t.n0 * row_bytes), 0,
                                            min(N - t.n0, BN) * (int)row_bytes, 0x00020000);
    return t;
  };

  // DMA: one instruction fills 1 KB of LDS.  LDS rows are the 192 bytes of a k-step, the four 16-byte chunks of each
  // piece XOR-swizzled with row bits 2-3, so that an operand read (16 rows x one chunk) covers all banks once.  LDS row
  // j*16+l of a wave's column group holds column NJ*l+j of the group: a lane then owns NJ consecutive columns of C.
  // Where the instructions do not divide evenly, the last wavefront repeats the last one (same bytes to the same place).
  uint32_t voff[Tile::DMA];
#pragma unroll
  for (int q = 0; q < Tile::DMA; ++q) {
    const int c = min(wave * Tile::DMA + q, Tile::DMA_ALL - 1) * kWave + lane;
    int row = c / 12;
    const int ch = c - row * 12;
    const uint32_t in_row = (uint32_t)(ch >> 2) * 64u + (uint32_t)(((ch & 3) ^ ((row >> 2) & 3)) * 16);
    if (row >= BM) {
      row -= BM;
      const int in_wave = row % (16 * NJ);
      row = row - in_wave + (in_wave & 15) * NJ + (in_wave >> 4);
    }
    voff[q] = (uint32_t)row * row_bytes + in_row;
  }
  // instructions [q0, q1) of this wave's share of k-step `t` of tile `c` (past its end: of the first k-steps of tile `n`)
  // into slot `slot`
  auto issue = [&](int slot, int t, const Src& c, const Src& n, int q0, int q1) {
    const bool over = t >= nk;
    const __amdgpu_buffer_rsrc_t ra = over ? n.a : c.a;
    const __amdgpu_buffer_rsrc_t rb = over ? n.b : c.b;
    const int koff = (over ? t - nk : t) * kStepBytes;
#pragma unroll
    for (int q = q0; q < q1; ++q) {
      const int i = min(wave * Tile::DMA + q, Tile::DMA_ALL - 1);
      unsigned char* dst = smem + slot * Tile::SLOT + i * 1024;
      if (i < Tile::A_BYTES / 1024) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, ET_LDS_PTR(dst), 16, voff[q], koff, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, ET_LDS_PTR(dst), 16, voff[q], koff, 0, 0);
    }
  };

  const int sw = (g ^ (l16 >> 2)) * 16;
  const int a_rd = (wm * 16 * MI + l16) * kStepBytes + sw;
  const int b_rd = Tile::A_BYTES + (wn * 16 * NJ + l16) * kStepBytes + sw;
  auto read_a = [&](bf16x8 (&v)[MI], int slot, int piece) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      v[i] = *reinterpret_cast<const bf16x8*>(smem + slot * Tile::SLOT + a_rd + piece * 64 + i * 16 * kStepBytes);
  };
  auto read_b = [&](bf16x8 (&v)[NJ], int slot, int piece) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      v[j] = *reinterpret_cast<const bf16x8*>(smem + slot * Tile::SLOT + b_rd + piece * 64 + j * 16 * kStepBytes);
  };

  float4v main_[MI][NJ], corr[MI][NJ];
  bf16x8 ah[MI], bh[NJ], am[MI], bm[NJ], al[MI], bl[NJ];         // TWO_PER_SIMD
  bf16x8 pa[2][3][MI], pb[2][3][NJ];                             // otherwise: the pieces of this k-step and of the next

  auto mfma_row = [&](float4v (&acc)[MI][NJ], const bf16x8 (&a)[MI], const bf16x8 (&b)[NJ], int i) {
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const int j = (i & 1) ? NJ - 1 - jj : jj;          // only one operand changes from one MFMA to the next
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  };
  auto mfma = [&](float4v (&acc)[MI][NJ], const bf16x8 (&a)[MI], const bf16x8 (&b)[NJ]) {
#pragma unroll
    for (int i = 0; i < MI; ++i) mfma_row(acc, a, b, i);
  };

  Src cur = locate(idx), nxt = cur;
#pragma unroll
  for (int s = 0; s < ST; ++s) issue(s, min(s, nk - 1), cur, cur, 0, Tile::DMA);
  wait_vmcnt<Tile::DMA * (ST - 1)>();
  barrier_only();
  if constexpr (kTwoPerSimd) {
    read_a(ah, 0, 0);
    read_b(bh, 0, 0);
  } else {
#pragma unroll
    for (int piece = 0; piece < 3; ++piece) {
      read_a(pa[0][piece], 0, piece);
      read_b(pb[0][piece], 0, piece);
    }
  }

  int s = 0;                                     // slot of the current k-step
  bool first_tile = true;
  while (true) {
    const int nidx = idx + wgs;
    const bool has_next = nidx < n_loc;
    if (has_next) nxt = locate(nidx);            // otherwise the stream re-loads this tile; the data is never used
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) main_[i][j] = corr[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    if constexpr (kTwoPerSimd) {
      for (int t = 0; t < nk; ++t) {
        read_b(bm, s, 1);
        mfma(main_, ah, bh);
        __builtin_amdgcn_sched_barrier(0);
        read_b(bl, s, 2);
        mfma(corr, ah, bm);
        __builtin_amdgcn_sched_barrier(0);
        read_a(am, s, 1);
        mfma(corr, ah, bl);
        __builtin_amdgcn_sched_barrier(0);
        read_a(al, s, 2);
        mfma(corr, am, bh);
        __builtin_amdgcn_sched_barrier(0);
        // this wave's share of k-step t+1 has landed, those behind it may fly; right after a tile boundary all of them
        // were confirmed before the C stores went out
        if (first_tile || t >= ST - 1) wait_vmcnt<Tile::DMA * (ST - 2)>();
        wait_lgkmcnt0();                           // its last reads of slot s are complete
        barrier_only();
        const int s1 = s + 1 == ST ? 0 : s + 1;
        // the DMA instructions go out between the rows of MFMAs: in one piece they would keep the wavefront from issuing
        constexpr int kPer = (Tile::DMA + 2 * MI - 1) / (2 * MI);
        read_a(ah, s1, 0);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          mfma_row(corr, al, bh, i);
          issue(s, t + ST, cur, nxt, min(i * kPer, Tile::DMA), min((i + 1) * kPer, Tile::DMA));
          __builtin_amdgcn_sched_barrier(0);
        }
        read_b(bh, s1, 0);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          mfma_row(corr, am, bm, i);
          issue(s, t + ST, cur, nxt, min((MI + i) * kPer, Tile::DMA), min((MI + i + 1) * kPer, Tile::DMA));
          __builtin_amdgcn_sched_barrier(0);
        }
        s = s1;
      }
    } else {
      // one k-step on register set P, the next one's pieces read into the other set under its MFMAs
      auto step = [&](auto Pc, int t) {
        constexpr int P = decltype(Pc)::value;
        if (first_tile || t >= ST - 1) wait_vmcnt<Tile::DMA * (ST - 2)>();       // as above
        wait_lgkmcnt0();
        barrier_only();
        const int s1 = s + 1 == ST ? 0 : s + 1;
#pragma unroll
        for (int piece = 0; piece < 3; ++piece) {
          read_a(pa[1 - P][piece], s1, piece);
          read_b(pb[1 - P][piece], s1, piece);
        }
        __builtin_amdgcn_sched_barrier(0);
        mfma(main_, pa[P][0], pb[P][0]);
        mfma(corr, pa[P][0], pb[P][1]);
        issue(s, t + ST, cur, nxt, 0, Tile::DMA);
        mfma(corr, pa[P][0], pb[P][2]);
        mfma(corr, pa[P][1], pb[P][0]);
        mfma(corr, pa[P][2], pb[P][0]);
        mfma(corr, pa[P][1], pb[P][1]);
        __builtin_amdgcn_sched_barrier(0);
        s = s1;
      };
      int t = 0;
      for (; t + 1 < nk; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
      }
      if (t < nk) {                              // an odd number of k-steps
        step(std::integral_constant<int, 0>{}, t);
        wait_lgkmcnt0();
#pragma unroll
        for (int piece = 0; piece < 3; ++piece) {
#pragma unroll
          for (int i = 0; i < MI; ++i) pa[0][piece][i] = pa[1][piece][i];
#pragma unroll
          for (int j = 0; j < NJ; ++j) pb[0][piece][j] = pb[1][piece][j];
        }
      }
    }
    wait_vmcnt<0>();

    const int col = cur.n0 + wn * 16 * NJ + l16 * NJ;
    if (col < N) {
      typedef float fvec __attribute__((ext_vector_type(NJ)));
      fvec bias = {};
      if (args.bias[cur.grp] != nullptr) bias = *reinterpret_cast<const fvec*>(args.bias[cur.grp] + col);
      // the bias is waited for here: left pending on the paths that store nothing, it would have the compiler put a wait
      // for every outstanding load, the DMA included, in front of the k loop's reuse of its registers
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        float b = bias[j];
        asm volatile("" : "+v"(b));
        bias[j] = b;
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = cur.m0 + wm * 16 * MI + i * 16 + g * 4 + r;
          if (row >= rows) continue;
          fvec o;
#pragma unroll
          for (int j = 0; j < NJ; ++j) o[j] = (main_[i][j][r] + corr[i][j][r]) + bias[j];
          if constexpr (GELU) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) o[j] *= gelu_cdf(o[j], o[j] * o[j] * o[j]);
            store_split<NJ>((uint16_t*)args.C + (size_t)row * 3 * args.ldc, cur.grp * N + col, o);
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
// as long as its k-steps (microseconds per k-step below: measured with few workgroups, K = 768 .. 3072) and about 3 us
// for filling the ring and storing C.  (The heights of 192 and 96 rows are there for the part-filled last round: 3850 rows,
// n = 2304 / 768 at k = 768, 3072 + GELU, and 768 at k = 3072: 84, 32, 90, 102 us without them, 70, 28, 84, 90 with; 5500
// rows: 95, 47, 147, 164 and 95, 40, 120, 133.)
enum SplitPick { k256x128, k192x128, k128x128, k96x128, k64x128, k64x64, k32x64, k32x32 };
SplitPick pick_split_tile(int m, int n, int k, int groups) {
  static constexpr struct { int bm, bn; float step; } kTiles[] = {
      {256, 128, 1.58f}, {192, 128, 1.33f}, {128, 128, 0.97f}, {96, 128, 0.79f}, {64, 128, 0.6f}, {64, 64, 0.38f}, {32, 64, 0.26f}, {32, 32, 0.15f}};
  const long cus = device_cu_count();
  int best = 0;
  float best_cost = 0.f;
  for (int i = 0; i < (int)std::size(kTiles); ++i) {
    const long tiles = (long)((m + kTiles[i].bm - 1) / kTiles[i].bm) * ((n + kTiles[i].bn - 1) / kTiles[i].bn) * groups;
    const float cost = (float)((tiles + cus - 1) / cus) * (kTiles[i].step * (float)(k / 32) + 3.f);
    if (i == 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return (SplitPick)best;
}

template <int WM, int WN, int MI, int NJ, int ST>
void launch_tile(SplitGemmArgs a, bool gelu, int groups, hipStream_t stream) {
  using Tile = SplitTile<WM, WN, MI, NJ, ST>;
  a.tiles_n = (a.n + Tile::BN - 1) / Tile::BN;
  a.tiles_n_all = a.tiles_n * groups;
  // The workgroups of an XCD advance through k side by side, so what its L2 has to deliver per k-step is the distinct
  // rows of A and columns of B they touch: about square blocks of tiles are the best.  Wide outputs take their column
  // tiles in groups of about 1024 columns.
  a.col_groups = 1;
  for (int c = 2; c <= a.tiles_n_all; ++c)
    if (a.tiles_n_all % c == 0 && a.tiles_n_all / c * Tile::BN >= 768) a.col_groups = c;
  const int tiles = ((a.m_bound + Tile::BM - 1) / Tile::BM) * a.tiles_n_all;
  // (a stream of fewer k-steps than the ring holds must not cross into a second tile)
  const int grid = ((a.k / 32 < ST ? tiles : std::min(tiles, device_cu_count())) + kXcds - 1) / kXcds * kXcds;
  auto go = [&](auto kern) {
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), Tile::SMEM);
    kern<<<grid, Tile::THREADS, Tile::SMEM, stream>>>(a);
  };
  if (gelu) go(gemm_split_kernel<WM, WN, MI, NJ, ST, true>);
  else go(gemm_split_kernel<WM, WN, MI, NJ, ST, false>);
}

// float rows -> split rows, 8 values per thread (HBM-bound: 4 bytes in, 6 out per value)
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ src, uint16_t* __restrict__ dst, int m,
                                                         fastdiv chunks, const int32_t* __restrict__ rows_dev) {
  const int rows = rows_dev ? min(*rows_dev, m) : m;
  const uint32_t total = (uint32_t)rows * chunks.d;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < total; i += gridDim.x * 256u) {
    const uint32_t row = div_by(i, chunks), c = i - row * chunks.d;
    const float4v* s = reinterpret_cast<const float4v*>(src) + (size_t)i * 2;
    const float4v v0 = s[0], v1 = s[1];
    const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    store_split<8>(dst + (size_t)row * chunks.d * 24, (int)c * 8, v);
  }
}

// [k][n] float weights -> n split rows: 64 x 64 tiles through LDS
struct SplitWeightArgs {
  TransposeJobs jobs;
  int tile_begin[TransposeJobs::kMax + 1];
};
__global__ __launch_bounds__(256) void split_weight_kernel(SplitWeightArgs args) {
  __shared__ float tile[64][65];
  int job = 0;
  while (job + 1 < args.jobs.count && (int)blockIdx.x >= args.tile_begin[job + 1]) ++job;
  const int K = args.jobs.k[job], N = args.jobs.n[job];
  const int tiles_n = (N + 63) / 64;
  const int t = blockIdx.x - args.tile_begin[job];
  const int k0 = (t / tiles_n) * 64, n0 = (t % tiles_n) * 64;
  const float* __restrict__ src = (const float*)args.jobs.src[job];
  uint16_t* __restrict__ dst = (uint16_t*)args.jobs.dst[job];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = threadIdx.x + u * 256, r = i >> 4, c = (i & 15) * 4;       // source row k0+r, columns n0+c ..
    float4v v = {};
    if (k0 + r < K && n0 + c < N) v = *reinterpret_cast<const float4v*>(src + (size_t)(k0 + r) * N + n0 + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) tile[c + j][r] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = threadIdx.x + u * 256, r = i >> 3, c = (i & 7) * 8;        // row n0+r of the result, k0+c ..
    if (n0 + r < N && k0 + c < K) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = tile[r][c + j];
      store_split<8>(dst + (size_t)(n0 + r) * K * 3, k0 + c, v);
    }
  }
}

}  // namespace

void launch_split_rows(const float* src, uint16_t* dst, int m, int k, const int32_t* rows_dev, hipStream_t stream) {
  if (m <= 0) return;
  const long chunks = (long)m * (k / 8);
  const int grid = (int)std::min((chunks + 255) / 256, 256L * 16);
  split_rows_kernel<<<grid, 256, 0, stream>>>(src, dst, m, make_fastdiv((uint32_t)k / 8), rows_dev);
}

void launch_split_weights(const TransposeJobs& jobs, hipStream_t stream) {
  if (jobs.count == 0) return;
  SplitWeightArgs a;
  a.jobs = jobs;
  int total = 0;
  for (int j = 0; j < jobs.count; ++j) {
    a.tile_begin[j] = total;
    total += ((jobs.k[j] + 63) / 64) * ((jobs.n[j] + 63) / 64);
  }
  for (int j = jobs.count; j <= TransposeJobs::kMax; ++j) a.tile_begin[j] = total;
  split_weight_kernel<<<total, 256, 0, stream>>>(a);
}

bool gemm_split_supported(int n, int k) {
  return k % 32 == 0 && k >= 32 && n % 4 == 0 && (uint64_t)k * 6u * 256u < 0x80000000ull;
}

void launch_gemm_split(const GemmGroups& g, void* C, int ldc, int m_bound, int n, int k, const int32_t* rows_dev,
                       hipStream_t stream) {
  if (m_bound <= 0) return;
  SplitGemmArgs a;
  for (int i = 0; i < 3; ++i) {
    a.A[i] = i < g.groups ? (const uint16_t*)g.A[i > 0] : nullptr;
    a.B[i] = i < g.groups ? (const uint16_t*)g.B[i] : nullptr;
    a.bias[i] = i < g.groups ? (const float*)g.bias[i] : nullptr;
  }
  a.C = C;
  a.rows_dev = rows_dev;
  a.ldc = ldc;
  a.m_bound = m_bound;
  a.n = n;
  a.k = k;
  switch (pick_split_tile(m_bound, n, k, g.groups)) {
    case k256x128: return launch_tile<4, 2, 4, 4, 2>(a, g.gelu, g.groups, stream);
    case k192x128: return launch_tile<4, 2, 3, 4, 2>(a, g.gelu, g.groups, stream);
    case k128x128: return launch_tile<2, 4, 4, 2, 3>(a, g.gelu, g.groups, stream);
    case k96x128: return launch_tile<2, 4, 3, 2, 3>(a, g.gelu, g.groups, stream);
    case k64x128: return launch_tile<2, 4, 2, 2, 4>(a, g.gelu, g.groups, stream);
    case k64x64: return launch_tile<4, 2, 1, 2, 6>(a, g.gelu, g.groups, stream);
    case k32x64: return launch_tile<2, 4, 1, 1, 8>(a, g.gelu, g.groups, stream);
    case k32x32: return launch_tile<2, 2, 1, 1, 12>(a, g.gelu, g.groups, stream);
  }
}

}  // namespace et
