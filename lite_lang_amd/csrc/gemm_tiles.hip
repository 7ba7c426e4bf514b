// Prefill projections (M > 64 rows): Y[M, N] = X[M, K] . W[N, K]^T on MFMA,
// gfx950. Replaces the torch.addmm / torch.mm products of the reference's
// prefill (litelang/models/qwen2/layer/transformer_layer.py:80,82,95-109,193)
// for bf16/fp16, and is the int8 x int8 -> int32 product of the W8A8 runtime
// (the reference's SmoothQuant module has no forward, quantize/smooth_quant/
// layer.py:19-59).
//
// One workgroup per CU works off (k split, output tile) items one after the
// other (a persistent grid); tiles are 256 x 256 or 256 x 128 (8 waves, two per
// SIMD) or 128 x 128 (4 waves) by shape (plan_tiles):
//   * stages of 128 bytes of K per row (64 bf16/fp16 or 128 int8) of the
//     tile's weight and activation rows are copied global -> LDS with
//     global_load_lds_dwordx4 (no VGPR staging) into a ring of two to four
//     stage buffers that runs on from one item into the next. A row's 128
//     bytes are one cache line (with 64-byte rows every line was fetched
//     twice);
//   * the ring is refilled in pieces of 128 rows, each as soon as both wave
//     groups have read it, so the copies lead the reads by more than a stage
//     although the 256 x 256 form holds only two stages;
//   * a finished item's rows are turned through the wave's own LDS and stored
//     as whole 128-byte segments with buffer stores that nothing waits for
//     until the ring's own waits reach them;
//   * the 16-byte chunks of every LDS row are XOR-swizzled (tile_swz) so
//     the MFMA operand reads hit distinct banks;
//   * each wave multiplies 64 or 128 weight rows by 32 or 64 activation rows
//     with v_mfma_f32_16x16x32 (v_mfma_i32_16x16x64_i8 for int8) as
//     C^T = W . X^T: the weight rows are the MFMA's row operand, so every
//     lane ends with runs of 4 consecutive output columns of one token row.
//     At 24,000 rows the matrix pipes are busy 63% of the cycles at about
//     1.96 GHz (gate/up + SiLU; the 32 x 32 form with 64-byte rows: 69% at
//     1.55 GHz): the 16 x 16 form, which moves half the accumulator registers
//     per product, draws less and clocks higher, 6% faster than 32 x 32;
//   * the grid is XCD-aware: the workgroups the dispatcher deals to one XCD
//     take a contiguous range of items, tiles in groups of 1, 2 or 4 row
//     tiles by shape (tile_group_m), round robin, so tiles sharing activation
//     or weight rows run together on one L2.
// Measured against 256 x 256 tiles of 64-byte rows and 32 x 32 products (bf16,
// M = 24,000, 3B, 20 launches, both on one card): gate/up + SiLU 1850 -> 1695 us
// (1277 TFLOP/s), down_proj 931 -> 810 (1336), qkv 271 -> 240, o_proj 197 -> 173;
// W8A8 1519 -> 962, 512 -> 415, 210 -> 138, 160 -> 109. down_proj at M = 333
// 204 -> 33 us.
// Epilogues: the model dtype with an optional bias; SiLU_and_Mul of a
// gate/up weight interleaved in 64-row blocks (ll_gemm_interleave_gate_up),
// with the rounding sequence of ll_silu_and_mul; int8 sums dequantised as
// fp32(acc) * s_tok[m] * fp32(s_ch[n]) (+ bias) as ll_dequant_splitk does;
// raw int32 sums.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "ll_common.h"

namespace {

constexpr int kRB = 128;       // bytes of K per row per stage: one cache line
constexpr int kKUnit = 64;     // K spans a multiple of this many bytes
constexpr int kPlanCus = 256;   // CUs the workspace query plans for
constexpr int kMinSplitStages = 6;  // stages per k split on average, at least (the last has the rest)
constexpr int kPieceB = 128 * kRB;  // a piece: 128 rows of one operand (16 KB)

// Tile geometry: NWP pieces of 128 weight rows by NXP pieces of 128
// activation rows (W0, W1 and X0, X1 below).
//
// 256 x 256 (2 x 2): 8 waves in two groups of four that take turns (kPingPong),
// each wave 128 x 64. The phases of stage t, in order, each reading pieces
// from LDS and then multiplying:
//   W0(t) X1(t) -> W0 X0, W0 X1;   W1(t) X0(t + 1) -> W1 X0, W1 X1
// X0 is read a stage ahead, so that both phases read 12 fragments per lane
// for 32 MFMAs: the time of the reads and of the other group's MFMAs is the
// same. A piece's slot in the stage buffer is its place in that order.
//
// 256 x 128 (2 x 1, 8 waves) and 128 x 128 (1 x 1, 4 waves): 64 x 64 per wave,
// every wave reading the next stage's fragments under its MFMAs, one barrier
// per stage. Few workgroups run these, so what counts is the time of one
// stage, bounded by LDS (reads and copies of 96 KB per 128 x 128 stage): 0.74
// and 0.49 us (few workgroups), against 0.87 and 0.56 with two groups taking
// turns on 64 x 32 per wave (128 KB, and a barrier after each turn).
//
// NT: the weight copies are non-temporal, for one row tile (M <= 128) in one k
// split, where every weight byte is read once and would only push the
// activations out of L2 (96 rows, cold weights): gate/up + SiLU 26.9 -> 25.4
// us (22016 x 2048) and 21.0 -> 20.2 (17920 x 1536), lm_head 157 -> 152 and
// 110 -> 102; int8 gate/up + SiLU 21.7 -> 20.9 and 18.9 -> 18.4 (2 to 5% over 65
// to 128 rows). With two row tiles, which share the weights through L2, it
// costs (160 rows, 151936 x 2048: 174 -> 204), and k splits lose too (2048 x
// 11008: 19.0 -> 21.2; 1536 x 8960: 15.7 -> 18.2).
template <int NWP_, int NXP_, bool NT_ = false> struct TileGeo {
  static constexpr bool kNt = NT_;
  static constexpr int NWP = NWP_, NXP = NXP_;
  static constexpr int TN = 128 * NWP, TM = 128 * NXP;
  static constexpr int kPieces = NWP + NXP;
  static constexpr bool kPingPong = kPieces == 4;
  static constexpr int kWaves = kPingPong ? 8 : 4 * NWP;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kDma = 16 / kWaves;      // 16-byte copies per lane per piece
  static constexpr int NH = kPingPong ? 2 : 1;  // 64-row weight blocks per wave
  static constexpr int kStageB = kPieces * kPieceB;
  static constexpr int kNst = kPieces == 4 ? 2 : kPieces == 3 ? 3 : 4;  // stage buffers
  static constexpr int kEpB = kPieces == 3 ? 2048 : 4096;               // epilogue bytes per wave
  static constexpr size_t kLds = (size_t)kNst * kStageB + (size_t)kWaves * kEpB;
  static_assert(kLds <= 160 * 1024, "LDS");
  static constexpr bool is_w(int q) { return q == 0 || q == 2; }
  static constexpr int w_half(int q) { return q / 2; }
  static constexpr int x_half(int q) { return kPingPong && q == 1 ? 1 : 0; }
  // copies of this lane a wave may leave in flight when it waits for the next
  // pieces to be read: two phases of two pieces, or all stages but two
  static constexpr int kInFlight = kPingPong ? 4 * kDma : (kNst - 2) * kPieces * kDma;
};

enum { EPI_STORE = 0, EPI_SILU = 1, EPI_DEQ = 2, EPI_DEQ_SILU = 3, EPI_I32 = 4, EPI_PART = 5 };

template <typename T> struct TileOp;
template <> struct TileOp<__bf16> { typedef bf16x8 V; typedef f32x4 Acc; };
template <> struct TileOp<_Float16> { typedef f16x8 V; typedef f32x4 Acc; };
template <> struct TileOp<int8_t> { typedef i32x4 V; typedef i32x4 Acc; };

// 16 x 16 output block, 32 bf16/fp16 (64 int8) of K per instruction: lane l
// supplies row (or column) l % 16 and the 16-byte K chunk l / 16.
__device__ __forceinline__ f32x4 tile_mma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 tile_mma(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ i32x4 tile_mma(i32x4 a, i32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// 16 B global -> LDS copy of one lane (lane i lands at lds + 16 i); kept out of
// the templates (a dependent call of this builtin drops the host launch stub).
__device__ __forceinline__ void tile_dma16(const void* g, void* lds) {
  __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 0);
}

// the same, non-temporal
__device__ __forceinline__ void tile_dma16_nt(const void* g, void* lds) {
  __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 2 /* nt */);
}

template <int N_> __device__ __forceinline__ void tile_vm_wait() {
  static_assert(N_ >= 0 && N_ < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

// Barrier that waits for this wave's LDS reads only (its own copies were
// waited for with tile_vm_wait; __syncthreads would also drain the copies of
// the stages in flight).
__device__ __forceinline__ void tile_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct TileArgs {
  const char* X; int64_t ldx_b;   // activation rows (K contiguous), row stride in bytes
  const char* W; int64_t ldw_b;   // weight rows [N][K] (EPI_SILU*: interleaved gate/up)
  int M, N;
  int K_b;                        // K in bytes
  int nk;                         // stages of the whole K
  int kps;                        // stages per k split (the last split may have fewer)
  int half;                       // the last stage of K holds 64 bytes per row, not 128
  int tiles_m, tiles_n, splits;
  int group_m;                    // row tiles per group of the tile order (tile_group_m)
  void* Y; int64_t ldy;           // output, row stride in elements of the output type
  int y_bytes;                    // bytes from Y to the end of its last row (< 2^31)
  int64_t split_b;                // bytes between the outputs of consecutive k splits
  int wide;                       // output rows and column counts allow 16-byte stores
  const void* bias;               // [N] in the model dtype, or null
  const float* s_tok;             // int8: activation scale per row [M]
  const void* s_ch; int s_ch_dtype;  // int8: weight scale per channel [N]
};

// Swizzle of the 16-byte chunks of 128-byte LDS row r (an involution on
// 0..7): chunk c of row r sits at chunk c ^ ((r / 2) % 8), so 16 consecutive
// rows read at one chunk index cover all 64 banks once.
__device__ __forceinline__ int tile_swz(int r) { return (r >> 1) & 7; }

// Output tile (m0, n0) of tile t of the grouped order: groups of group_m row
// tiles, each group's column tiles in order with its row tiles innermost.
template <typename G>
__device__ __forceinline__ void tile_coords(const TileArgs& a, int t, int& m0, int& n0) {
  const int gsz = a.group_m * a.tiles_n;
  const int grp = t / gsz, rin = t - grp * gsz;
  const int gm = min(a.group_m, a.tiles_m - grp * a.group_m);
  m0 = (grp * a.group_m + rin % gm) * G::TM;
  n0 = (rin / gm) * G::TN;
}

// A store lane whose offset is kTileNoStore (beyond the buffer's size) stores
// nothing, so every wave issues the same number of store instructions for
// every tile, edges included: the copy ring's vmcnt waits count them. The
// empty asm keeps the compiler from merging stores, which would change that
// count.
constexpr uint32_t kTileNoStore = 0x80000000u;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Scales of channels i[j] .. i[j] + 3 as fp32. The dtype branch is taken once
// for all the loads and conversions, so one wait serves them all.
template <int n>
__device__ __forceinline__ void tile_scales(const void* s, int dtype, const int (&i)[n],
                                            float (&f)[n][4]) {
  if (dtype == LL_F32) {
#pragma unroll
    for (int j = 0; j < n; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) f[j][k] = *(const float*)((const char*)s + (uint32_t)(4 * (i[j] + k)));
  } else {
    uint32_t b[n][4];
#pragma unroll
    for (int j = 0; j < n; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) b[j][k] = *(const uint16_t*)((const char*)s + (uint32_t)(2 * (i[j] + k)));
    if (dtype == LL_F16) {
#pragma unroll
      for (int j = 0; j < n; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) f[j][k] = ll_scale_bits_to_f32(b[j][k], LL_F16);
    } else {
#pragma unroll
      for (int j = 0; j < n; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) f[j][k] = ll_scale_bits_to_f32(b[j][k], LL_BF16);
    }
  }
}

// Every lambda of the kernel is inlined before the arrays it captures are
// split into registers (left to the inliner, they stay in scratch memory).
#define LL_INLINE __attribute__((always_inline))

template <typename T, typename TO, int EPI, typename G>
__global__ __launch_bounds__(G::kThreads, 2) void gemm_tile_kernel(TileArgs a) {
  typedef typename TileOp<T>::V V;
  typedef typename TileOp<T>::Acc Acc;
  constexpr bool kSilu = EPI == EPI_SILU || EPI == EPI_DEQ_SILU;
  constexpr int kNst = G::kNst, NWP = G::NWP, NH = G::NH, kWaves = G::kWaves, kDma = G::kDma;
  constexpr bool kPP = G::kPingPong;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  // ---- work items of this workgroup: (k split, output tile), splits
  // outermost. XCD x (= blockIdx % 8, up to a launch-wide rotation) owns
  // items x * per .. x * per + per - 1; its gridDim / 8 workgroups (one per
  // CU) take them round robin, so the tiles in flight on one XCD at any time
  // are consecutive in the grouped order and share rows in its L2.
  const int tiles = a.tiles_m * a.tiles_n;
  const int items = tiles * a.splits;
  const int per = (items + 7) / 8;
  const int g8 = (int)(gridDim.x >> 3);
  const int i_first = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  const int i_end = min((int)(blockIdx.x & 7) * per + per, items);
  if (i_first >= i_end) return;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wn = kPP ? wave & 1 : wave >> 1, wm = kPP ? wave >> 1 : wave & 1;

  // ---- copy stream: the pieces of all of this workgroup's stages in the
  // order they are read, running on from one item into the next. Instruction
  // u of this wave copies rows 8 j .. 8 j + 7 (j = kWaves u + wave) of a
  // piece; lane -> row 8 j + l / 8, LDS chunk l % 8, that is global chunk
  // (l % 8) ^ swizzle, the same for every piece. Row i of W piece h is tile row
  //   256 x 256:  (2 (i / 64) + h) * 64 + i % 64 (64-row block 2 wn + h of wave column wn);
  //   the others: 128 h + i, or for the SiLU forms
  //               128 h + ((i / 32) % 2) * 64 + (i / 64) * 32 + i % 32,
  // so that a wave holds a gate channel and its up channel.
  const int gch = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
  const uint32_t tail_adj = gch >= 4 ? 64u : 0u;  // half stage: chunks past K re-read the row's last 64 B
  uint32_t soff[G::kPieces][kDma];
  // 32-bit product and sum (the spans are below 4 GiB), kept apart: their
  // 64-bit multiply-add would hold a register pair per offset
  auto row_off = [&](int row, uint32_t ld) LL_INLINE {
    uint32_t o = (uint32_t)row * ld;
    asm volatile("" : "+v"(o));
    return o + (uint32_t)gch * 16;
  };
  auto set_sources = [&](int t) LL_INLINE {
    int m0, n0;
    tile_coords<G>(a, t, m0, n0);
    int sl = lane;  // as a value of its own (no row number is held through the main loop)
    asm volatile("" : "+v"(sl));
#pragma unroll
    for (int q = 0; q < G::kPieces; ++q)
#pragma unroll
      for (int u = 0; u < kDma; ++u) {
        const int i = 8 * (kWaves * u + wave) + (sl >> 3);
        if (G::is_w(q)) {
          int r;
          if constexpr (kPP) r = (2 * (i >> 6) + G::w_half(q)) * 64 + (i & 63);
          else if constexpr (kSilu) r = G::w_half(q) * 128 + ((i >> 5) & 1) * 64 + (i >> 6) * 32 + (i & 31);
          else r = G::w_half(q) * 128 + i;
          soff[q][u] = row_off(min(n0 + r, a.N - 1), (uint32_t)a.ldw_b);
        } else {
          const int r = G::x_half(q) * 128 + i;
          soff[q][u] = row_off(min(m0 + r, a.M - 1), (uint32_t)a.ldx_b);
        }
      }
  };
  // cursor of the copies: item, its first stage, stage within it, ring buffer
  int iss_i = i_first, iss_k = 0, iss_ke = 0, iss_buf = 0;
  auto iss_item = [&]() LL_INLINE {
    const int sp = iss_i / tiles;
    set_sources(iss_i - sp * tiles);
    iss_k = sp * a.kps;
    iss_ke = min(iss_k + a.kps, a.nk);
  };
  iss_item();
  // Copy u of piece q of the cursor's stage. Past the last item every lane
  // copies the operand's first bytes (in bounds, never read, one line), so
  // each wave issues the same number of copies in every stage.
  auto issue_copy = [&](auto qc, int u) LL_INLINE {
    constexpr int q = decltype(qc)::value;
    const bool past = iss_i >= i_end;
    const uint32_t pmask = past ? 0u : ~0u;
    const uint32_t tadj = (a.half && iss_k == a.nk - 1) ? tail_adj : 0u;
    const int64_t kb = past ? 0 : (int64_t)iss_k * kRB;
    uint32_t o = (soff[q][u] - tadj) & pmask;
    asm volatile("" : "+v"(o));  // no 64-bit form of it is held through the loop
    const char* src = (G::is_w(q) ? a.W : a.X) + kb + o;
    char* dst = smem + iss_buf * G::kStageB + q * kPieceB + (kWaves * u + wave) * 1024;
    if constexpr (G::kNt && G::is_w(q)) tile_dma16_nt(src, dst);
    else tile_dma16(src, dst);
  };
  auto issue_piece = [&](auto qc) LL_INLINE {
#pragma unroll
    for (int u = 0; u < kDma; ++u) issue_copy(qc, u);
  };
  auto issue_next = [&]() LL_INLINE {
    iss_buf = iss_buf == kNst - 1 ? 0 : iss_buf + 1;
    if (iss_i < i_end && ++iss_k == iss_ke) {
      iss_i += g8;
      if (iss_i < i_end) iss_item();
    }
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  constexpr std::integral_constant<int, 3> c3{};

  Acc acc[NH][2][4][2];
  auto zero_acc = [&]() LL_INLINE {
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
          for (int q = 0; q < 2; ++q) acc[h][j][p][q] = Acc{0, 0, 0, 0};
  };
  zero_acc();

  // ---- fragments: 64 weight rows as four 16-row blocks (p), 32 activation
  // rows as two (q), twice (j); k step ks is LDS chunks 4 ks .. 4 ks + 3 (lane
  // l / 16). Byte offset of k step ks in a row block of a piece: one register
  // per k step, everything else of the address is scalar or immediate
  // (opaque, so that no other form of it takes registers through the loop).
  int foff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    foff[ks] = (lane & 15) * kRB + (((4 * ks + (lane >> 4)) ^ tile_swz(lane & 15)) << 4);
    asm volatile("" : "+v"(foff[ks]));
  }
  V fw[2][4], fx[3][2][2];  // [ks][p]; [set][ks][q]
  auto read_w = [&](int ks, int buf, int piece, int row) LL_INLINE {
    const int sb = buf * G::kStageB + piece * kPieceB + row * kRB;
#pragma unroll
    for (int p = 0; p < 4; ++p) fw[ks][p] = *(const V*)(smem + (sb + foff[ks]) + 16 * p * kRB);
  };
  auto read_x = [&](int ks, int buf, int piece, int row, V (&f)[2][2]) LL_INLINE {
    const int sb = buf * G::kStageB + piece * kPieceB + row * kRB;
#pragma unroll
    for (int q = 0; q < 2; ++q) f[ks][q] = *(const V*)(smem + (sb + foff[ks]) + 16 * q * kRB);
  };
  // products i0 .. i1 - 1 of the 16 of k step ks: weight block h against both
  // activation sets
  auto multiply = [&](int h, int ks, int i0, int i1) LL_INLINE {
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const int j = i / 8, p = i / 2 % 4, q = i % 2;
      acc[h][j][p][q] = tile_mma(fw[ks][p], fx[j][ks][q], acc[h][j][p][q]);
    }
  };

  // ---- epilogue. acc[h][j][p][q][i] = C[m][n] with m = m0 + (the 32 rows of
  // j and wm) + 16 q + l % 16 and n = n0 + (the 64 columns of h and wn) +
  // 16 p + 4 (l / 16) + i. A lane's run of 4 columns is 8 or 16 bytes, so the rows
  // are turned through the wave's own piece of LDS: stores of whole 128-byte
  // (64-byte where the piece is smaller) row segments, 16 bytes per lane.
  constexpr int kCB = G::kEpB >= 4096 && !(kSilu && !kPP) ? 128 : 64;  // bytes per row segment
  constexpr int kRowsPI = 1024 / kCB;                 // rows per store instruction
  constexpr int kSegCols = kCB / (int)sizeof(TO);     // columns per segment
  constexpr int kOutB = NH * 2 * 64 * 32 * (int)sizeof(TO) / (kSilu ? 2 : 1);  // bytes per wave
  constexpr int kStores = kOutB / 1024;
  char* const ep = smem + kNst * G::kStageB + wave * G::kEpB;
  auto ep_swz = [](int row) LL_INLINE { return kCB == 128 ? (row & 7) : ((row >> 1) & 3); };
  // 4 outputs of row `row` at column c (multiple of 4) of the segment
  auto ep_put = [&](int row, int c, const TO (&o)[4]) LL_INLINE {
    typedef TO V4 __attribute__((ext_vector_type(4)));
    const V4 v = {o[0], o[1], o[2], o[3]};
    const int b = c * (int)sizeof(TO);
    *(V4*)(ep + row * kCB + ((((b >> 4) ^ ep_swz(row)) << 4) | (b & 15))) = v;
  };
  // store the segment: rows mb .. mb + 31, columns nb .. nb + kSegCols - 1 of
  // the nmax columns of the output
  auto ep_store = [&](int el, const __amdgpu_buffer_rsrc_t& r, int mb, int nb, int nmax) LL_INLINE {
    u32x4 v[32 / kRowsPI];
#pragma unroll
    for (int it = 0; it < 32 / kRowsPI; ++it) {
      const int row = it * kRowsPI + el / (kCB / 16), ch = el % (kCB / 16);
      v[it] = *(const u32x4*)(ep + row * kCB + ((ch ^ ep_swz(row)) << 4));
    }
#pragma unroll
    for (int it = 0; it < 32 / kRowsPI; ++it) {
      const int m = mb + it * kRowsPI + el / (kCB / 16);
      const int n = nb + el % (kCB / 16) * (16 / (int)sizeof(TO));
      const uint32_t off = (uint32_t)(((int64_t)m * a.ldy + n) * (int64_t)sizeof(TO));
      if (a.wide) {
        __builtin_amdgcn_raw_buffer_store_b128(v[it], r, (m < a.M && n < nmax) ? off : kTileNoStore, 0, 0);
      } else {  // 8-byte halves: rows 8-byte aligned, or a last chunk of 4 columns
        const u32x2 lo = {v[it][0], v[it][1]}, hi = {v[it][2], v[it][3]};
        const int n2 = n + 8 / (int)sizeof(TO);
        __builtin_amdgcn_raw_buffer_store_b64(lo, r, (m < a.M && n < nmax) ? off : kTileNoStore, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b64(hi, r, (m < a.M && n2 < nmax) ? off + 8 : kTileNoStore, 0, 0);
      }
      asm volatile("" ::: "memory");
    }
  };
  auto epilogue = [&](int item) LL_INLINE {
    const int sp = item / tiles;
    int m0, n0;
    tile_coords<G>(a, item - sp * tiles, m0, n0);
    const __amdgpu_buffer_rsrc_t yres = __builtin_amdgcn_make_buffer_rsrc(
        (char*)a.Y + (int64_t)sp * a.split_b, (short)0, a.y_bytes, 0x00020000);
    const int mw = m0 + wm * (kPP ? 32 : 64);
    constexpr int kMj = kPP ? 128 : 32;  // rows between the two activation sets
    // the lane as a value of its own: nothing that follows from it is
    // computed ahead of the main loop and held in registers through it
    int el = lane;
    asm volatile("" : "+v"(el));
    const int lr = el & 15, lc = el >> 4;
    // The per-row and per-column factors are loaded before the first store
    // that needs them, so the wave waits for them (and for the copies in
    // flight ahead of them) once, not once per store.
    float st[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        st[j][q] = 1.f;
        if constexpr (EPI == EPI_DEQ || EPI == EPI_DEQ_SILU)
          st[j][q] = a.s_tok[min(mw + kMj * j + 16 * q + lr, a.M - 1)];
      }
    if constexpr (!kSilu) {
      typedef TO V4 __attribute__((ext_vector_type(4)));
      const bool has_bias = EPI != EPI_I32 && EPI != EPI_PART && a.bias != nullptr;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int nh = n0 + (kPP ? 2 * wn + h : wn) * 64;
        int nl[4];  // in-range column groups for the loads
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int n = nh + 16 * p + 4 * lc;
          nl[p] = n < a.N ? n : 0;
        }
        V4 bv[4];
        if (has_bias) {
#pragma unroll
          for (int p = 0; p < 4; ++p) bv[p] = *(const V4*)((const char*)a.bias + (uint32_t)(nl[p] * (int)sizeof(TO)));
        }
        float sc[4][4];
        if constexpr (EPI == EPI_DEQ) tile_scales<4>(a.s_ch, a.s_ch_dtype, nl, sc);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            __builtin_amdgcn_sched_barrier(0);  // one group at a time (registers)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              TO o[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                if constexpr (EPI == EPI_I32 || EPI == EPI_PART) {
                  o[i] = (TO)acc[h][j][p][q][i];
                } else if constexpr (EPI == EPI_DEQ) {
                  // the product is rounded before the bias is added (no fused
                  // multiply-add), as in ll_dequant_splitk followed by the add
                  float v = (float)acc[h][j][p][q][i] * st[j][q] * sc[p][i];
                  asm volatile("" : "+v"(v));
                  if (has_bias) v += ll_to_f32(bv[p][i]);
                  o[i] = ll_from_f32<TO>(v);
                } else {
                  o[i] = ll_from_f32<TO>(acc[h][j][p][q][i] + (has_bias ? ll_to_f32(bv[p][i]) : 0.f));
                }
              }
              ep_put(16 * q + lr, 16 * p % kSegCols + 4 * lc, o);
            }
            if (16 * (p + 1) % kSegCols == 0)
              ep_store(el, yres, mw + kMj * j, nh + 16 * (p + 1) - kSegCols, a.N);
          }
      }
    } else {
      // gate/up interleaved in 64-row blocks; this wave's channels:
      //   256 x 256:  n0 / 2 + 64 wn + 16 p, gate acc[0][j][p], up acc[1][j][p]
      //   the others: n0 / 2 + 32 wn + 16 p, gate acc[0][j][p], up acc[0][j][p + 2]
      constexpr int NB = 2 * NH;  // 16-channel blocks of this wave
      const int I = a.N / 2;
      const int cw = n0 / 2 + wn * 16 * NB;
      float sc[2 * NB][4];  // scales of the gate channels, then the up channels
      if constexpr (EPI == EPI_DEQ_SILU) {
        int cl[2 * NB];
#pragma unroll
        for (int p = 0; p < NB; ++p) {
          const int c = cw + 16 * p + 4 * lc;
          cl[p] = c < I ? c : 0;
          cl[NB + p] = I + cl[p];
        }
        tile_scales<2 * NB>(a.s_ch, a.s_ch_dtype, cl, sc);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int p = 0; p < NB; ++p) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const auto ga = acc[0][j][p][q];
            const auto ua = kPP ? acc[NH - 1][j][p][q] : acc[0][j][(p + 2) % 4][q];
            TO o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float gs, us;
              if constexpr (EPI == EPI_DEQ_SILU) {
                gs = (float)ga[i] * st[j][q] * sc[p][i];
                us = (float)ua[i] * st[j][q] * sc[NB + p][i];
              } else {
                gs = ga[i];
                us = ua[i];
              }
              const float gv = ll_to_f32(ll_from_f32<TO>(gs));
              const float u = ll_to_f32(ll_from_f32<TO>(us));
              const TO sv = ll_from_f32<TO>(ll_silu_f32(gv));
              o[i] = ll_from_f32<TO>(u * ll_to_f32(sv));
            }
            ep_put(16 * q + lr, 16 * p % kSegCols + 4 * lc, o);
          }
          if (16 * (p + 1) % kSegCols == 0)
            ep_store(el, yres, mw + kMj * j, cw + 16 * (p + 1) - kSegCols, I);
        }
    }
  };

  // Waits for the copies of the pieces read next. A finished item's stores are
  // not waited for: while the copies waited for were issued before them
  // (since_ep phases or stages after the epilogue, at most kAllow), the wait
  // allows kStores more operations (a count at or below the exact one is
  // always safe; vmcnt retires in issue order).
  static_assert(G::kInFlight + kStores < 64, "vmcnt is a 6-bit counter");
  constexpr int kAllow = kPP ? 1 : kNst - 2;
  int since_ep = 64;
  auto wait_next = [&]() LL_INLINE {
    if (since_ep <= kAllow) tile_vm_wait<G::kInFlight + kStores>();
    else tile_vm_wait<G::kInFlight>();
    ++since_ep;
  };
  auto finish = [&](int item) LL_INLINE {
    epilogue(item);
    zero_acc();
    since_ep = 0;
  };
  // cursor of the multiplications
  int cur_i = i_first, cur_k, cur_ke;
  auto cur_item = [&]() LL_INLINE {
    const int sp = cur_i / tiles;
    cur_k = sp * a.kps;
    cur_ke = min(cur_k + a.kps, a.nk);
  };
  cur_item();
  int buf = 0;
  bool more = true;
  auto cur_next = [&](bool last) LL_INLINE {
    buf = buf == kNst - 1 ? 0 : buf + 1;
    if (!last) {
      ++cur_k;
    } else {
      cur_i += g8;
      more = cur_i < i_end;
      if (more) cur_item();
    }
  };
  // sched_barrier keeps every instruction inside its slot (MFMAs touch no
  // memory, so nothing else stops the scheduler moving them across barriers)
  if constexpr (kPP) {
    // Ping-pong schedule. Waves 0-3 (group A) and 4-7 (group B) hold one wave
    // of each SIMD (the dispatcher places wave w on SIMD w % 4). Time is cut
    // into slots separated by workgroup barriers; phase P is P / 2's W0 or W1
    // half. In slot 2P group A reads the fragments of phase P and issues
    // copies while group B multiplies phase P - 1; in slot 2P + 1 A multiplies
    // phase P while B reads it. So each SIMD's matrix pipe has one wave with a
    // run of MFMAs while the other wave's LDS reads and copies proceed. Ring
    // invariants (four phases in the ring):
    //   * the pieces of phase P have landed before slot 2P: each wave issues
    //     them in its memory slot of phase P - 3 and waits for them before the
    //     barrier that ends slot 2P - 1, with two later phases outstanding;
    //   * the buffers of phase P - 1's pieces are refilled in the memory slots
    //     of phase P (2P and 2P + 1), after the barrier that ends B's read of
    //     them (slot 2P - 1, closed by lgkmcnt(0)).
    // A wave writes a finished item's outputs in its first memory slot after
    // the item's last stage, before that slot's copies.
    auto issue = [&](auto phc) LL_INLINE {
      if constexpr (decltype(phc)::value == 0) {
        issue_piece(c0);
        issue_piece(c1);
      } else {
        issue_piece(c2);
        issue_next();
        issue_piece(c3);
      }
    };
    auto read_x0 = [&](int b) LL_INLINE {
      read_x(0, b, 3, wm * 32, fx[2]);
      read_x(1, b, 3, wm * 32, fx[2]);
    };
    auto read_phase = [&](auto phc, int b) LL_INLINE {
      constexpr int ph = decltype(phc)::value;
      if constexpr (ph == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fx[0][i / 2][i % 2] = fx[2][i / 2][i % 2];
      }
      read_w(0, b, 2 * ph, wn * 64);
      read_w(1, b, 2 * ph, wn * 64);
      if constexpr (ph == 0) {
        read_x(0, b, 1, wm * 32, fx[1]);
        read_x(1, b, 1, wm * 32, fx[1]);
      } else {
        read_x0(1 - b);
      }
    };
    auto multiply_phase = [&](auto phc, bool full) LL_INLINE {  // a half stage has one k step
      __builtin_amdgcn_s_setprio(1);
      multiply(decltype(phc)::value, 0, 0, 16);
      if (full) multiply(decltype(phc)::value, 1, 0, 16);
      __builtin_amdgcn_s_setprio(0);
    };
    // prologue: every phase of the ring but the last one, after the first X0,
    // which both groups read before the first slot
    issue_piece(c3);
    issue(c0);
    issue(c1);
    issue(c0);
    tile_vm_wait<G::kInFlight>();
    tile_barrier();
    read_x0(0);
    tile_barrier();
    auto phase_a = [&](auto phc, bool full, bool last) LL_INLINE {
      constexpr int ph = decltype(phc)::value;
      constexpr std::integral_constant<int, 1 - ph> nxt{};
      __builtin_amdgcn_sched_barrier(0);
      multiply_phase(phc, full);
      __builtin_amdgcn_sched_barrier(0);
      wait_next();
      tile_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (ph == 1) {
        if (last) finish(cur_i);
      }
      read_phase(nxt, ph == 1 ? 1 - buf : buf);
      issue(phc);
      __builtin_amdgcn_sched_barrier(0);
      tile_barrier();
    };
    int done = -1;  // group B: item whose outputs are still in the accumulators
    auto phase_b = [&](auto phc, bool full) LL_INLINE {
      constexpr int ph = decltype(phc)::value;
      constexpr std::integral_constant<int, 1 - ph> prv{};
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (ph == 0) {
        if (done >= 0) {
          finish(done);
          done = -1;
        }
      }
      read_phase(phc, buf);
      issue(prv);
      __builtin_amdgcn_sched_barrier(0);
      wait_next();
      tile_barrier();
      __builtin_amdgcn_sched_barrier(0);
      multiply_phase(phc, full);
      __builtin_amdgcn_sched_barrier(0);
      tile_barrier();
    };
    if (wave < 4) {
      read_phase(c0, 0);
      issue(c1);
      tile_barrier();
      while (more) {
        const bool full = !(a.half && cur_k == a.nk - 1);
        const bool last = cur_k + 1 == cur_ke;  // the item's last stage
        phase_a(c0, full, last);
        phase_a(c1, full, last);
        cur_next(last);
      }
    } else {
      tile_barrier();
      while (more) {
        const bool full = !(a.half && cur_k == a.nk - 1);
        const bool last = cur_k + 1 == cur_ke;
        phase_b(c0, full);
        phase_b(c1, full);
        if (last) done = cur_i;
        cur_next(last);
      }
      epilogue(done);
    }
  } else {
    // Every wave alike, one barrier per stage. At the top of stage t its
    // fragments are in registers (set t % 2); the barrier says that stage t + 1
    // has landed and that everybody has read stage t, whose buffer takes stage
    // t + kNst. The 16 fragment reads of stage t + 1 into the other set and
    // those copies go out between the 32 MFMAs of stage t, so neither LDS
    // latency nor the copies' issue holds them up. (The reads follow the first
    // MFMA: the compiler waits for every outstanding LDS read where it first
    // uses one.)
    V gw[2][2][4], gx[2][2][2][2];  // [set][ks][p]; [set][ks][j][q]
    const int wrow = (wn & 1) * 64, wpc = NWP == 2 ? (wn >> 1) * 2 : 0;
    auto read_frag = [&](auto setc, int b, int r) LL_INLINE {
      constexpr int set = decltype(setc)::value;
      const int ks = r / 8, i = r % 8;
      if (i < 4) {
        const int sb = b * G::kStageB + wpc * kPieceB + wrow * kRB;
        gw[set][ks][i] = *(const V*)(smem + (sb + foff[ks]) + 16 * i * kRB);
      } else {
        const int sb = b * G::kStageB + kPieceB + wm * 64 * kRB;
        gx[set][ks][(i - 4) / 2][i % 2] = *(const V*)(smem + (sb + foff[ks]) + 16 * (i - 4) * kRB);
      }
    };
    auto mul = [&](auto setc, int i) LL_INLINE {  // MFMA i of the stage's 32
      constexpr int set = decltype(setc)::value;
      const int ks = i / 16, j = i / 8 % 2, p = i / 2 % 4, q = i % 2;
      acc[0][j][p][q] = tile_mma(gw[set][ks][p], gx[set][ks][j][q], acc[0][j][p][q]);
    };
    auto copy = [&](int i) LL_INLINE {  // copy i of the stage's kCopies
      if constexpr (kDma == 4) {
        if (i < 4) issue_copy(c0, i);
        else issue_copy(c1, i - 4);
      } else {
        if (i < 2) issue_copy(c0, i);
        else if (i < 4) issue_copy(c1, i - 2);
        else issue_copy(c2, i - 4);
      }
    };
    constexpr int kCopies = G::kPieces * kDma;
    static_assert(kCopies <= 8, "a copy per four MFMAs");
#pragma unroll
    for (int t = 0; t < kNst; ++t) {
#pragma unroll
      for (int i = 0; i < kCopies; ++i) copy(i);
      issue_next();
    }
    tile_vm_wait<(kNst - 1) * kCopies>();
    tile_barrier();
#pragma unroll
    for (int r = 0; r < 16; ++r) read_frag(c0, 0, r);
    auto stage = [&](auto setc) LL_INLINE {
      constexpr int set = decltype(setc)::value;
      constexpr std::integral_constant<int, 1 - set> other{};
      const bool last = cur_k + 1 == cur_ke;
      const int nbuf = buf == kNst - 1 ? 0 : buf + 1;
      wait_next();
      tile_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          mul(setc, 4 * g + i);
          // int8: keeps the sum in one place (the compiler otherwise gives each
          // product's result new registers and runs out of them)
          if constexpr (sizeof(T) == 1) asm volatile("" : "+v"(acc[0][(4 * g + i) / 8 % 2][(4 * g + i) / 2 % 4][i % 2]));
          __builtin_amdgcn_sched_barrier(0);
          if (i % 2 == 0) read_frag(other, nbuf, 2 * g + i / 2);
          if (i == 3 && g < kCopies) copy(g);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      issue_next();
      if (last) finish(cur_i);
      cur_next(last);
    };
    while (true) {
      stage(c0);
      if (!more) break;
      stage(c1);
      if (!more) break;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  tile_vm_wait<0>();
}

// Interleave a [gate; up] weight ([2I, K], I % 128 == 0) into 64-row blocks:
// out row R of tile R / 256: block (R % 256) / 64 alternates gate and up rows
// of channels (R / 256) * 128 + ((R % 256) / 128) * 64 + R % 64.
__global__ void interleave_gate_up_kernel(const u32x4* __restrict__ W, int64_t ldw16,
                                          u32x4* __restrict__ out, int64_t row16, int I,
                                          int64_t total) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= total) return;
  const int64_t R = u / row16, c = u - R * row16;
  const int64_t t = R / 256, r = R % 256;
  const int64_t blk = r / 64, ch = t * 128 + (blk / 2) * 64 + (r % 64);
  const int64_t src = (blk % 2 == 0) ? ch : I + ch;
  out[u] = W[src * ldw16 + c];
}

// Row tiles per group of the tile order, by shape class, as measured with group
// sizes 1, 2, 4 and 8 (us): wide outputs 4 (gate/up + SiLU, 86 column tiles, M =
// 24,000: 1712, 1655, 1634, 1626; 256 x 128 tiles, M = 600: 70.5, 57.2, 56.4,
// 55.3; lm_head of 1536, M = 600: 503, 327, 318, 300; the 8 of these lead the 4 by
// 0.5 to 6%, but not at M = 8192: 565, 557, 546, 547); long K (down_proj, 172
// stages, M = 24,000) 1 (773, 777, 791, 808); the narrow short-K shapes (qkv,
// o_proj) level within 1.5% at every size (2).
int tile_group_m(int64_t tiles_n, int64_t nk) {
  if (tiles_n >= 32) return 4;
  if (nk >= 64) return 1;
  return 2;
}

struct TilePlan {
  int geo;     // 0: 256 x 256, 1: 256 x 128, 2: 128 x 128
  int splits;  // k splits
  int kps;     // stages per split
};

// Tile geometry and k splits by a cost in us, fitted to a sweep of every
// geometry and split count over M 96 .. 24000 at the 3B and 1.5B projections
// (cold weights): a stage costs 1.15 us with few workgroups and 1.5 with all
// CUs busy (256 x 256), 0.76 .. 0.93 (256 x 128), 0.50 (128 x 128); an item
// 6, 2 and 3.3 us of fill and stores; the reduction of splits one more launch
// and the partials' bytes both ways. So large outputs take 256 x 256 tiles
// (M = 24,000, gate/up: 1736 us against 2244 and 2702), outputs of few tiles
// smaller ones and splits (333 x 2048, K = 11008: 33 us with 128 x 128 tiles
// in 5 splits, 98 unsplit, 197 as 16 tiles of 256 x 256), and what lies
// between follows the rounds its tiles take (600 x 22016: 71 us in two
// rounds of 256 x 128, 97 in two of 256 x 256).
// The cost has no term for the weights' bytes: it says 95 us for the lm_head of
// 96 rows, which streams 622 MB in 145 to 152. What it orders are forms of one
// shape, which move the same bytes: with each form forced, its choice was within
// 3% of the best for lm_head and gate/up at 65 to 600 rows, but for a 1536-wide
// lm_head at 256 rows (152 us, best 145) and at 600 (327, best 302).
// A K that ends in half a stage runs on the 256 x 256 form, the only one that
// can leave out a k step; int8 has no 128 x 128 form (its sums and two
// fragment sets do not fit the registers).
TilePlan plan_tiles(int64_t M, int64_t N, int64_t K_b, int es, int64_t max_splits, int cus) {
  const int64_t nk = ll_cdiv(K_b, kRB);
  const int geos = K_b % kRB != 0 ? 1 : es == 1 ? 2 : 3;
  static const int tn[3] = {256, 256, 128}, tm[3] = {256, 128, 128};
  static const double stage_us[3] = {1.15, 0.76, 0.50}, busy_us[3] = {0.35, 0.17, 0.0};
  static const double item_us[3] = {6.0, 2.0, 3.3};
  TilePlan best = {0, 1, (int)nk};
  double best_us = 1e30;
  for (int g = 0; g < geos; ++g) {
    const int64_t tiles = (int64_t)ll_cdiv(M, tm[g]) * ll_cdiv(N, tn[g]);
    for (int64_t sp = 1; sp <= max_splits; ++sp) {
      if (sp > 1 && (sp * kMinSplitStages > nk || tiles * sp > cus)) break;
      const int64_t kps = ll_cdiv(nk, sp);
      if (ll_cdiv(nk, kps) != sp) continue;  // an empty last split
      const int64_t items = tiles * sp, per = ll_cdiv(items, 8);
      const int64_t g8 = std::min<int64_t>(per, std::max(1, cus / 8));
      const double busy = std::min(1.0, (double)items / cus);
      const double us = (double)ll_cdiv(per, g8) * (kps * (stage_us[g] + busy_us[g] * busy) + item_us[g]) +
                        (sp > 1 ? 4.5 + (double)sp * M * N * 8 / 5.5e6 : 0.0);
      if (us < best_us) {
        best_us = us;
        best = {g, (int)sp, (int)kps};
      }
    }
  }
  return best;
}

// The kernel addresses its copy sources with 32-bit row offsets and its
// stores with 31-bit buffer offsets: the weight must span less than 4 GiB
// (checked by the entry points), and the activation and output rows are
// launched in chunks whose spans fit (and whose stage count per workgroup
// fits an int).
template <typename T, typename TO, int EPI, typename G>
int launch_geo(const TileArgs& a0, const TilePlan& plan, int cus, hipStream_t stream) {
  const int64_t yrow_b = a0.ldy * (int64_t)sizeof(TO);
  const int64_t ny = EPI == EPI_SILU || EPI == EPI_DEQ_SILU ? a0.N / 2 : a0.N;
  const int64_t tiles_n = ll_cdiv(a0.N, G::TN);
  const int64_t rows_x = (((int64_t)1 << 32) - 2 * kRB) / a0.ldx_b;
  const int64_t rows_y = (((int64_t)1 << 31) - 1) / yrow_b;
  const int64_t rows_s = ((int64_t)INT32_MAX / a0.nk) * 8 / (tiles_n * plan.splits) * G::TM;
  const int64_t max_rows = std::min(rows_x, std::min(rows_y, rows_s));
  LL_CHECK_ARG(max_rows >= 1, "gemm tiles: output rows or K too large for one launch");
  const int64_t chunk =
      max_rows >= a0.M ? a0.M : (max_rows >= G::TM ? (max_rows / G::TM) * G::TM : max_rows);
  for (int64_t mo = 0; mo < a0.M; mo += chunk) {
    TileArgs a = a0;
    a.X += mo * a0.ldx_b;
    a.Y = (char*)a0.Y + mo * yrow_b;
    if (a0.s_tok != nullptr) a.s_tok = a0.s_tok + mo;
    a.M = (int)(a0.M - mo < chunk ? a0.M - mo : chunk);
    a.y_bytes = (int)((a.M - 1) * yrow_b + ny * (int64_t)sizeof(TO));
    a.wide = yrow_b % 16 == 0 && (uintptr_t)a0.Y % 16 == 0 && (ny * (int64_t)sizeof(TO)) % 16 == 0;
    a.tiles_m = ll_cdiv(a.M, G::TM);
    a.tiles_n = (int)tiles_n;
    a.splits = plan.splits;
    a.kps = plan.kps;
    a.group_m = tile_group_m(tiles_n, a.nk);
    const int64_t per = ((int64_t)a.tiles_m * a.tiles_n * a.splits + 7) / 8;
    const int64_t grid = 8 * std::min<int64_t>(per, std::max(1, cus / 8));
    hipLaunchKernelGGL((gemm_tile_kernel<T, TO, EPI, G>), dim3((unsigned)grid), dim3(G::kThreads),
                       G::kLds, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      ll_set_error("HIP launch failed: %s", hipGetErrorString(e));
      return LL_ERR_HIP;
    }
  }
  return LL_OK;
}

template <typename T, typename TO, int EPI>
int launch_plan(const TileArgs& a, const TilePlan& plan, int cus, hipStream_t stream) {
  if (plan.geo == 0) return launch_geo<T, TO, EPI, TileGeo<2, 2>>(a, plan, cus, stream);
  const bool nt = a.M <= 128 && plan.splits == 1;  // TileGeo: the weights are read once
  if (plan.geo == 1)
    return nt ? launch_geo<T, TO, EPI, TileGeo<2, 1, true>>(a, plan, cus, stream)
              : launch_geo<T, TO, EPI, TileGeo<2, 1>>(a, plan, cus, stream);
  if constexpr (sizeof(T) == 2)
    return nt ? launch_geo<T, TO, EPI, TileGeo<1, 1, true>>(a, plan, cus, stream)
              : launch_geo<T, TO, EPI, TileGeo<1, 1>>(a, plan, cus, stream);
  ll_set_error("gemm tiles: no 128 x 128 form for int8");
  return LL_ERR_UNSUPPORTED;
}

// one k split, outputs in their final form
template <typename T, typename TO, int EPI>
int launch_tiles(const TileArgs& a, hipStream_t stream) {
  int cus = 0;
  const int rc = ll_device_cus(&cus);
  if (rc != LL_OK) return rc;
  return launch_plan<T, TO, EPI>(a, plan_tiles(a.M, a.N, a.K_b, sizeof(T), 1, cus), cus, stream);
}

// Sum of the k splits' partials [splits][M][N], in split order, finished as
// the tile epilogue finishes its sums: fp32 (+ bias), or int32 dequantised.
// 4 columns per thread.
template <typename TP, typename TO>
__global__ __launch_bounds__(256) void tile_reduce_kernel(const TP* __restrict__ part, int splits,
                                                          const void* __restrict__ bias,
                                                          const float* __restrict__ s_tok,
                                                          const void* __restrict__ s_ch,
                                                          int s_ch_dtype, TO* __restrict__ Y,
                                                          int64_t ldy, int M, int N) {
  typedef TO V4 __attribute__((ext_vector_type(4)));
  const int q = N / 4;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int m = (int)(gid / q);
  if (m >= M) return;
  const int n = (int)(gid - (int64_t)m * q) * 4;
  const int64_t idx = (int64_t)m * N + n, ss = (int64_t)M * N;
  V4 o;
  if constexpr (__is_same(TP, float)) {
    const f32x4 v = ll_sum_splits4(part, splits, ss, idx);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = ll_from_f32<TO>(v[e] + (bias != nullptr ? ll_to_f32(((const TO*)bias)[n + e]) : 0.f));
  } else {
    const i32x4 v = ll_sum_splits4_i32(part, splits, ss, idx);
    const float st = s_tok[m];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = (float)v[e] * st * ll_load_scale(s_ch, s_ch_dtype, n + e);
      asm volatile("" : "+v"(x));
      if (bias != nullptr) x += ll_to_f32(((const TO*)bias)[n + e]);
      o[e] = ll_from_f32<TO>(x);
    }
  }
  *(V4*)(Y + (int64_t)m * ldy + n) = o;
}

// Product with the K of few output tiles split over the CUs: partial sums in
// the workspace and a reduction, where the plan splits and the workspace
// holds them; else one split.
template <typename T, typename TO, int EPI>
int launch_tiles_ws(const TileArgs& a, void* ws, int64_t ws_bytes, hipStream_t stream) {
  typedef typename std::conditional<__is_same(T, int8_t), int32_t, float>::type TP;
  int cus = 0;
  const int rc = ll_device_cus(&cus);
  if (rc != LL_OK) return rc;
  const int64_t split_b = (int64_t)a.M * a.N * 4;
  const int64_t room = ws != nullptr && (uintptr_t)ws % 16 == 0 ? ws_bytes / split_b : 0;
  const TilePlan plan = plan_tiles(a.M, a.N, a.K_b, sizeof(T), std::max<int64_t>(1, room), cus);
  if (plan.splits == 1) return launch_plan<T, TO, EPI>(a, plan, cus, stream);
  TileArgs pa = a;
  pa.Y = ws;
  pa.ldy = a.N;
  pa.split_b = split_b;
  std::lock_guard<std::mutex> lock(ll_workspace_mutex(ws));
  const int prc = launch_plan<T, TP, __is_same(T, int8_t) ? EPI_I32 : EPI_PART>(pa, plan, cus, stream);
  if (prc != LL_OK) return prc;
  hipLaunchKernelGGL((tile_reduce_kernel<TP, TO>), dim3((unsigned)ll_cdiv((int64_t)a.M * (a.N / 4), 256)),
                     dim3(256), 0, stream, (const TP*)ws, plan.splits, a.bias, a.s_tok, a.s_ch,
                     a.s_ch_dtype, (TO*)a.Y, a.ldy, a.M, a.N);
  LL_RETURN_LAUNCH();
}

// ldx, ldw in elements of es bytes; ldy in elements of Y, whose rows hold
// ny outputs (N, or N / 2 for the gate/up epilogues).
int check_tile_args(const char* name, const void* X, int64_t ldx, const void* W, int64_t ldw,
                    const void* Y, int64_t ldy, int64_t ny, int64_t M, int64_t N, int64_t K_b,
                    int64_t es) {
  LL_CHECK_ARG(X && W && Y, "%s: null pointer", name);
  LL_CHECK_ARG(M > 0 && N > 0 && N % 4 == 0 && K_b > 0 && K_b % kKUnit == 0,
               "%s: needs M > 0, N %% 4 == 0 and K a multiple of %lld (M=%lld N=%lld K=%lld)", name,
               (long long)(kKUnit / es), (long long)M, (long long)N, (long long)(K_b / es));
  LL_CHECK_ARG(ldx * es >= K_b && ldw * es >= K_b && ldy >= ny,
               "%s: row strides shorter than the rows (ldx=%lld ldw=%lld K=%lld, ldy=%lld for "
               "%lld outputs per row)",
               name, (long long)ldx, (long long)ldw, (long long)(K_b / es), (long long)ldy,
               (long long)ny);
  LL_CHECK_ARG((ldx * es) % 16 == 0 && (ldw * es) % 16 == 0 &&
                   (((uintptr_t)X | (uintptr_t)W) % 16) == 0,
               "%s: X and W rows must be 16 B aligned", name);
  LL_CHECK_ARG(M <= INT32_MAX && N <= INT32_MAX && K_b <= INT32_MAX, "%s: shape too large", name);
  LL_CHECK_ARG((N - 1) * ldw * es + K_b < ((int64_t)1 << 32) && ldx * es < ((int64_t)1 << 31),
               "%s: the weight must span less than 4 GiB", name);
  return LL_OK;
}

TileArgs make_args(const void* X, int64_t ldx_b, const void* W, int64_t ldw_b, int64_t M,
                   int64_t N, int64_t K_b, void* Y, int64_t ldy) {
  TileArgs a = {};
  a.X = (const char*)X; a.ldx_b = ldx_b;
  a.W = (const char*)W; a.ldw_b = ldw_b;
  a.M = (int)M; a.N = (int)N;
  a.K_b = (int)K_b;
  a.nk = a.kps = ll_cdiv(K_b, kRB);
  a.half = K_b % kRB != 0;
  a.Y = Y; a.ldy = ldy;
  return a;
}

}  // namespace

int ll_device_cus(int* cus_out) {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    ll_set_error("hipGetDevice failed");
    return LL_ERR_HIP;
  }
  int n = dev >= 0 && dev < 64 ? cache[dev].load(std::memory_order_relaxed) : 0;
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0) {
      ll_set_error("hipDeviceGetAttribute(MultiprocessorCount) failed");
      return LL_ERR_HIP;
    }
    if (dev >= 0 && dev < 64) cache[dev].store(n, std::memory_order_relaxed);
  }
  *cus_out = n;
  return LL_OK;
}

extern "C" int ll_gemm_tiled_supported(int64_t M, int64_t N, int64_t K, int dtype) {
  if (dtype != LL_BF16 && dtype != LL_F16) return 0;
  return M > 0 && N > 0 && N % 4 == 0 && K > 0 && (K * 2) % kKUnit == 0;
}

int ll_gemm_tiled_ws(const void* X, int64_t ldx, const void* W, int64_t ldw, const void* bias,
                     void* Y, int64_t ldy, int64_t M, int64_t N, int64_t K, int dtype, void* ws,
                     int64_t ws_bytes, hipStream_t stream) {
  LL_CHECK_ARG(dtype == LL_BF16 || dtype == LL_F16, "ll_gemm_tiled: bf16 or fp16 only");
  const int rc = check_tile_args("ll_gemm_tiled", X, ldx, W, ldw, Y, ldy, N, M, N, K * 2, 2);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG(ldy % 4 == 0 && ((uintptr_t)Y) % 8 == 0, "ll_gemm_tiled: Y rows must be 8 B aligned");
  LL_CHECK_ARG(((uintptr_t)bias) % 8 == 0, "ll_gemm_tiled: bias must be 8 B aligned");
  TileArgs a = make_args(X, ldx * 2, W, ldw * 2, M, N, K * 2, Y, ldy);
  a.bias = bias;
  if (dtype == LL_BF16) return launch_tiles_ws<__bf16, __bf16, EPI_STORE>(a, ws, ws_bytes, stream);
  return launch_tiles_ws<_Float16, _Float16, EPI_STORE>(a, ws, ws_bytes, stream);
}

extern "C" int ll_gemm_tiled(const void* X, int64_t ldx, const void* W, int64_t ldw,
                             const void* bias, void* Y, int64_t ldy, int64_t M, int64_t N,
                             int64_t K, int dtype, hipStream_t stream) {
  return ll_gemm_tiled_ws(X, ldx, W, ldw, bias, Y, ldy, M, N, K, dtype, nullptr, 0, stream);
}

extern "C" int64_t ll_gemm_tiles_workspace_size(int64_t M, int64_t N, int64_t K,
                                                int64_t elem_bytes) {
  if (M <= 64 || N <= 0 || N % 4 != 0 || K <= 0 || (elem_bytes != 1 && elem_bytes != 2) ||
      (K * elem_bytes) % kKUnit != 0)
    return 0;
  const TilePlan p = plan_tiles(M, N, K * elem_bytes, (int)elem_bytes, kPlanCus, kPlanCus);
  return p.splits > 1 ? (int64_t)p.splits * M * N * 4 : 0;
}

extern "C" int ll_gemm_tiles_plan(int64_t M, int64_t N, int64_t K, int64_t elem_bytes, int split,
                                  int32_t* tile_n, int32_t* tile_m, int32_t* splits,
                                  int32_t* split_stages) {
  LL_CHECK_ARG(tile_n && tile_m && splits && split_stages, "ll_gemm_tiles_plan: null pointer");
  LL_CHECK_ARG(M > 0 && N > 0 && N % 4 == 0 && K > 0 && (elem_bytes == 1 || elem_bytes == 2) &&
                   (K * elem_bytes) % kKUnit == 0,
               "ll_gemm_tiles_plan: no tile GEMM of this shape (M=%lld N=%lld K=%lld)",
               (long long)M, (long long)N, (long long)K);
  const TilePlan p =
      plan_tiles(M, N, K * elem_bytes, (int)elem_bytes, split ? kPlanCus : 1, kPlanCus);
  *tile_n = p.geo == 2 ? 128 : 256;
  *tile_m = p.geo == 0 ? 256 : 128;
  *splits = p.splits;
  *split_stages = p.kps;
  return LL_OK;
}

// fp32 partial sums for a consumer that finishes them itself: a reduction
// launch (4.5 us and the partials' bytes once more) less per product. Decode
// step of 96 requests (4 layers, 3B): 570 -> 528 us; first token of one prompt
// of 333 (4 layers): 749 -> 737.
extern "C" int ll_gemm_tiles_splitk_count(int64_t M, int64_t N, int64_t K, int dtype) {
  if (!ll_gemm_tiled_supported(M, N, K, dtype)) return 0;
  return plan_tiles(M, N, K * 2, 2, kPlanCus, kPlanCus).splits;
}

extern "C" int ll_gemm_tiles_splitk(const void* X, int64_t ldx, const void* W, int64_t ldw,
                                    int64_t M, int64_t N, int64_t K, int dtype, float* part,
                                    int64_t part_bytes, hipStream_t stream) {
  LL_CHECK_ARG(dtype == LL_BF16 || dtype == LL_F16, "ll_gemm_tiles_splitk: bf16 or fp16 only");
  const int rc = check_tile_args("ll_gemm_tiles_splitk", X, ldx, W, ldw, part, N, N, M, N, K * 2, 2);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG((uintptr_t)part % 16 == 0, "ll_gemm_tiles_splitk: partials must be 16 B aligned");
  const TilePlan plan = plan_tiles(M, N, K * 2, 2, kPlanCus, kPlanCus);
  const int64_t split_b = M * N * 4;
  LL_CHECK_ARG(part_bytes >= plan.splits * split_b,
               "ll_gemm_tiles_splitk: the partials need %lld bytes, got %lld",
               (long long)(plan.splits * split_b), (long long)part_bytes);
  int cus = 0;
  const int crc = ll_device_cus(&cus);
  if (crc != LL_OK) return crc;
  TileArgs a = make_args(X, ldx * 2, W, ldw * 2, M, N, K * 2, part, N);
  a.split_b = split_b;
  if (dtype == LL_BF16) return launch_plan<__bf16, float, EPI_PART>(a, plan, cus, stream);
  return launch_plan<_Float16, float, EPI_PART>(a, plan, cus, stream);
}

extern "C" int ll_gemm_interleave_gate_up(const void* W, int64_t ldw, int64_t I, int64_t K,
                                          int64_t elem_bytes, void* out, hipStream_t stream) {
  LL_CHECK_ARG(W && out, "ll_gemm_interleave_gate_up: null pointer");
  LL_CHECK_ARG(I > 0 && I % 128 == 0 && K > 0 && (K * elem_bytes) % 16 == 0 &&
                   (ldw * elem_bytes) % 16 == 0 && (elem_bytes == 1 || elem_bytes == 2),
               "ll_gemm_interleave_gate_up: needs I %% 128 == 0 and 16 B rows");
  const int64_t row16 = K * elem_bytes / 16, total = 2 * I * row16;
  hipLaunchKernelGGL(interleave_gate_up_kernel, dim3((unsigned)ll_cdiv(total, 256)), dim3(256), 0,
                     stream, (const u32x4*)W, ldw * elem_bytes / 16, (u32x4*)out, row16, (int)I,
                     total);
  LL_RETURN_LAUNCH();
}

extern "C" int ll_gemm_gate_up_silu_tiled(const void* X, int64_t ldx, const void* W_il,
                                          int64_t M, int64_t I, int64_t K, int dtype, void* Y,
                                          int64_t ldy, hipStream_t stream) {
  LL_CHECK_ARG(dtype == LL_BF16 || dtype == LL_F16, "ll_gemm_gate_up_silu_tiled: bf16 or fp16 only");
  LL_CHECK_ARG(I % 128 == 0, "ll_gemm_gate_up_silu_tiled: I must be a multiple of 128");
  const int rc = check_tile_args("ll_gemm_gate_up_silu_tiled", X, ldx, W_il, K, Y, ldy, I, M,
                                 2 * I, K * 2, 2);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG(ldy % 4 == 0 && ((uintptr_t)Y) % 8 == 0,
               "ll_gemm_gate_up_silu_tiled: Y rows must be 8 B aligned");
  TileArgs a = make_args(X, ldx * 2, W_il, K * 2, M, 2 * I, K * 2, Y, ldy);
  if (dtype == LL_BF16) return launch_tiles<__bf16, __bf16, EPI_SILU>(a, stream);
  return launch_tiles<_Float16, _Float16, EPI_SILU>(a, stream);
}

extern "C" int ll_gemm_i8_tiled_ws(const int8_t* Xq, int64_t ldx, const float* s_tok,
                                const int8_t* Wq, int64_t ldw, const void* s_ch, int s_ch_dtype,
                                const void* bias, void* Y, int64_t ldy, int64_t M, int64_t N,
                                int64_t K, int out_dtype, void* workspace,
                                int64_t workspace_bytes, hipStream_t stream) {
  const int rc = check_tile_args("ll_gemm_i8_tiled", Xq, ldx, Wq, ldw, Y, ldy, N, M, N, K, 1);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG(out_dtype == LL_BF16 || out_dtype == LL_F16 || out_dtype == LL_F32,
               "ll_gemm_i8_tiled: bad output dtype %d", out_dtype);
  LL_CHECK_ARG(s_tok && s_ch && (s_ch_dtype == LL_F32 || s_ch_dtype == LL_F16 ||
                                 s_ch_dtype == LL_BF16),
               "ll_gemm_i8_tiled: needs s_tok and s_ch (fp32/fp16/bf16)");
  LL_CHECK_ARG(bias == nullptr || out_dtype != LL_F32,
               "ll_gemm_i8_tiled: a bias needs a 16-bit output dtype");
  LL_CHECK_ARG(ldy % 4 == 0 && ((uintptr_t)Y) % 16 == 0, "ll_gemm_i8_tiled: Y rows must be 16 B aligned");
  LL_CHECK_ARG(((uintptr_t)bias) % 8 == 0, "ll_gemm_i8_tiled: bias must be 8 B aligned");
  TileArgs a = make_args(Xq, ldx, Wq, ldw, M, N, K, Y, ldy);
  a.bias = bias; a.s_tok = s_tok; a.s_ch = s_ch; a.s_ch_dtype = s_ch_dtype;
  if (out_dtype == LL_BF16) return launch_tiles_ws<int8_t, __bf16, EPI_DEQ>(a, workspace, workspace_bytes, stream);
  if (out_dtype == LL_F16) return launch_tiles_ws<int8_t, _Float16, EPI_DEQ>(a, workspace, workspace_bytes, stream);
  return launch_tiles_ws<int8_t, float, EPI_DEQ>(a, workspace, workspace_bytes, stream);
}

extern "C" int ll_gemm_i8_tiled(const int8_t* Xq, int64_t ldx, const float* s_tok,
                                const int8_t* Wq, int64_t ldw, const void* s_ch, int s_ch_dtype,
                                const void* bias, void* Y, int64_t ldy, int64_t M, int64_t N,
                                int64_t K, int out_dtype, hipStream_t stream) {
  return ll_gemm_i8_tiled_ws(Xq, ldx, s_tok, Wq, ldw, s_ch, s_ch_dtype, bias, Y, ldy, M, N, K,
                             out_dtype, nullptr, 0, stream);
}

extern "C" int ll_gemm_i8_i32_tiled(const int8_t* Xq, int64_t ldx, const int8_t* Wq, int64_t ldw,
                                    int32_t* Y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                                    hipStream_t stream) {
  const int rc = check_tile_args("ll_gemm_i8_i32_tiled", Xq, ldx, Wq, ldw, Y, ldy, N, M, N, K, 1);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG(ldy % 4 == 0 && ((uintptr_t)Y) % 16 == 0,
               "ll_gemm_i8_i32_tiled: Y rows must be 16 B aligned");
  TileArgs a = make_args(Xq, ldx, Wq, ldw, M, N, K, Y, ldy);
  return launch_tiles<int8_t, int32_t, EPI_I32>(a, stream);
}

// Shapes outside the tile kernel's layout (K not a multiple of 64, unaligned
// rows; small test models): one thread per output, the int8 dot product over
// K in 4-byte steps where the rows allow (v_dot4_i32_i8), exact int32 sums.
__global__ __launch_bounds__(256) void gemm_i8_plain_kernel(const int8_t* __restrict__ X,
                                                            int64_t ldx,
                                                            const int8_t* __restrict__ W,
                                                            int64_t ldw, int32_t* __restrict__ Y,
                                                            int64_t ldy, int M, int N, int K,
                                                            int vec4) {
  const int n = blockIdx.x * 64 + (threadIdx.x & 63);
  const int m = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (m >= M || n >= N) return;
  const int8_t* xr = X + (int64_t)m * ldx;
  const int8_t* wr = W + (int64_t)n * ldw;
  int32_t acc = 0;
  int k = 0;
  if (vec4) {
    for (; k + 4 <= K; k += 4)
      acc = __builtin_amdgcn_sdot4(*(const int32_t*)(xr + k), *(const int32_t*)(wr + k), acc, false);
  }
  for (; k < K; ++k) acc += (int32_t)xr[k] * (int32_t)wr[k];
  Y[(int64_t)m * ldy + n] = acc;
}

extern "C" int ll_gemm_i8_gate_up_silu_tiled(const int8_t* Xq, int64_t ldx, const float* s_tok,
                                             const int8_t* Wq_il, const void* s_ch,
                                             int s_ch_dtype, int64_t M, int64_t I, int64_t K,
                                             int out_dtype, void* Y, int64_t ldy,
                                             hipStream_t stream) {
  LL_CHECK_ARG(I % 128 == 0, "ll_gemm_i8_gate_up_silu_tiled: I must be a multiple of 128");
  const int rc = check_tile_args("ll_gemm_i8_gate_up_silu_tiled", Xq, ldx, Wq_il, K, Y, ldy, I, M,
                                 2 * I, K, 1);
  if (rc != LL_OK) return rc;
  LL_CHECK_ARG(out_dtype == LL_BF16 || out_dtype == LL_F16,
               "ll_gemm_i8_gate_up_silu_tiled: bf16 or fp16 output");
  LL_CHECK_ARG(s_tok && s_ch && (s_ch_dtype == LL_F32 || s_ch_dtype == LL_F16 ||
                                 s_ch_dtype == LL_BF16),
               "ll_gemm_i8_gate_up_silu_tiled: needs s_tok and s_ch (fp32/fp16/bf16)");
  LL_CHECK_ARG(ldy % 4 == 0 && ((uintptr_t)Y) % 8 == 0,
               "ll_gemm_i8_gate_up_silu_tiled: Y rows must be 8 B aligned");
  TileArgs a = make_args(Xq, ldx, Wq_il, K, M, 2 * I, K, Y, ldy);
  a.s_tok = s_tok; a.s_ch = s_ch; a.s_ch_dtype = s_ch_dtype;
  if (out_dtype == LL_BF16) return launch_tiles<int8_t, __bf16, EPI_DEQ_SILU>(a, stream);
  return launch_tiles<int8_t, _Float16, EPI_DEQ_SILU>(a, stream);
}

extern "C" int ll_gemm_i8_i32(const int8_t* Xq, int64_t ldx, const int8_t* Wq, int64_t ldw,
                              int32_t* Y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                              hipStream_t stream) {
  LL_CHECK_ARG(Xq && Wq && Y, "ll_gemm_i8_i32: null pointer");
  LL_CHECK_ARG(M >= 0 && N > 0 && K > 0 && ldx >= K && ldw >= K && ldy >= N,
               "ll_gemm_i8_i32: bad shape (M=%lld N=%lld K=%lld)", (long long)M, (long long)N,
               (long long)K);
  LL_CHECK_ARG(M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX, "ll_gemm_i8_i32: shape too large");
  if (M == 0) return LL_OK;
  const bool tile = N % 4 == 0 && K % kKUnit == 0 && ldx % 16 == 0 && ldw % 16 == 0 &&
                    (((uintptr_t)Xq | (uintptr_t)Wq) % 16) == 0 && ldy % 4 == 0 &&
                    ((uintptr_t)Y) % 16 == 0;
  if (tile) return ll_gemm_i8_i32_tiled(Xq, ldx, Wq, ldw, Y, ldy, M, N, K, stream);
  const int vec4 = ldx % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)Xq | (uintptr_t)Wq) % 4) == 0;
  // rows in launches of at most 65535 blocks of 4 (the grid's y limit)
  constexpr int64_t kRowsPerLaunch = 65535 * 4;
  for (int64_t m0 = 0; m0 < M; m0 += kRowsPerLaunch) {
    const int64_t mr = M - m0 < kRowsPerLaunch ? M - m0 : kRowsPerLaunch;
    hipLaunchKernelGGL(gemm_i8_plain_kernel, dim3((unsigned)ll_cdiv(N, 64), (unsigned)ll_cdiv(mr, 4)),
                       dim3(256), 0, stream, Xq + m0 * ldx, ldx, Wq, ldw, Y + m0 * ldy, ldy, (int)mr,
                       (int)N, (int)K, vec4);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      ll_set_error("HIP launch failed: %s", hipGetErrorString(e));
      return LL_ERR_HIP;
    }
  }
  return LL_OK;
}
