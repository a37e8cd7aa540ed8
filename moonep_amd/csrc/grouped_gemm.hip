// Expert-side consumer of the dispatched rows: grouped bf16 GEMM on the matrix
// cores of gfx950.  Rows [M,K] are split into G consecutive groups by the
// padded end offsets in cu_seqlens (device memory, as the planner wrote them);
// group g multiplies by its own weight matrix B[g] stored [N,K] (K
// contiguous), so C = A * B[g]^T needs no transposition on either operand.
// With token_padding a multiple of 128 a block of 128 rows never straddles two
// groups.
//
// Four kinds of product:
//   scale  : C[m,n] = bf16(row_scale[m] * acc)               (down projection)
//   swiglu : C[m,n] = bf16(silu(A*Bg^T) * (A*Bu^T))           (gate/up fused)
//   dual   : C = bf16(A*B[g]^T + A2*B2[g]^T): the K loop runs over both pairs
//            (input gradient of the gate/up pair)
//   wgrad  : C[g] = At[:, rows of g] * Bt[:, rows of g]^T in fp32: the K range
//            of a tile is the row range of its group (weight gradients)
// Four kernels:
//   gemm_wide_kernel       (gemm_wide.hip) 256 x 256 tiles, long groups: the products that
//                          tile the rows
//   gemm_pp_kernel         256 x 256 tiles: weight gradients, and the other products where
//                          few of the CUs get a tile
//   gemm_stream_kernel     128 rows x up to 288 weight rows or 256 weight columns:
//                          forward products and input gradients of groups of about
//                          one block, and of few tiles: bound by the weights' bytes
//   grouped_gemm_nt_kernel 128 x 256 tiles: the sum of two products with weights
//                          along K of such groups, and weight gradients that are no
//                          multiples of 256
//
// grouped_gemm_nt_kernel: workgroups of 640 threads on a 128 x 256 tile of (rows
// x weight rows), K in steps of 64: two producer waves stream the tile slices
// from global memory straight into a ring of three LDS stages, eight consumer
// waves own 64 x 64 of the tile each as 2 x 2 MFMA 32x32x16 accumulators.  It is
// bound by the L2 (its channels are ~75 % busy at 0.8 PFLOP/s), i.e. by tile
// bytes per flop.  Tiles are handed out so that the workgroups running at one
// time on an XCD (one L2) work on the same 8 row tiles and neighbouring weight
// tiles.
#include "grouped_gemm.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

using namespace mep_gemm;

constexpr int kStage = kATile + kBTile;        // 48 KB
constexpr int kStages = 3;
constexpr int kConsumers = 8, kProducers = 2;  // waves
constexpr int kGemmThreads = (kConsumers + kProducers) * 64;
constexpr int kPanel = 8;  // row tiles of a long group that share a sweep over the weight tiles
// 1 KB pieces (8 rows x 128 bytes) of a stage that one producer wave moves per step
constexpr int kPiecesPerProducer = (kBM + kBN) / 8 / kProducers;  // 24
static_assert(2 * kPiecesPerProducer < 64, "two steps of loads must fit the 6-bit load counter");

// Producer / consumer waves.  Two producer waves stream the tiles from global
// memory straight into a ring of three LDS stages (global_load_lds, 16 bytes
// per lane: no registers, no LDS store instructions), always two K steps
// ahead; eight consumer waves only read LDS and feed the matrix cores.  One
// s_barrier per K step hands a filled stage to the consumers and a drained one
// back to the producers.  A stage row is the bare 128-byte slice; the 16-byte
// vector q of row r sits at position q ^ (r & 7) ^ ((r >> 3) & 1), so the
// sixteen rows that sixteen consecutive lanes read cover all 64 banks once (a
// 16-byte read runs at 256 bytes per clock then; with q ^ (r & 7) alone, which
// separates only eight rows, at half of that).
template <int MODE>
__global__ __launch_bounds__(kGemmThreads, 1) void grouped_gemm_nt_kernel(GemmArgs a) {
  static_assert(MODE == kModeDual || MODE == kModeWgrad, "the products that need it");
  static_assert(kProducers == 2, "the lane offsets of the pieces assume that a producer wave's pieces share a parity");
  extern __shared__ __attribute__((aligned(1024))) char gsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // ---- which tile.  XCD x (workgroups x, x+8, ...) walks a contiguous eighth of
  // the tile list, in launch order, so the tiles that run on an XCD at one time
  // are neighbours in the list.  Only the row tiles below the last group's end
  // are listed (the row buffer is sized for the worst case; what lies beyond
  // would leave the last XCDs idle).
  //
  // Row-tiled products: the list goes group by group, inside a group weight tile
  // by weight tile, the group's row tiles running fastest.  The h row tiles of
  // a group then read a weight tile at the same time (it leaves HBM once), and
  // the 32 tiles an XCD runs cover 32 / h weight tiles of that group, so its
  // rows are fetched ntiles h / 32 times.  (Panels of eight row tiles whatever
  // the groups were, as before, split most groups over two panels: their
  // weights came from HBM twice.)
  const int mtiles = MODE == kModeWgrad ? a.mtiles : min(a.mtiles, (a.cu[a.G - 1] + kBM - 1) / kBM);
  const int per_group = mtiles * a.ntiles;
  const int total = MODE == kModeWgrad ? per_group * a.G : per_group;
  const int per_xcd = (total + 7) >> 3;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  if (idx >= per_xcd) {
    // no tile: these workgroups are at least as many as the tiles that the unused rows would have
    if (MODE != kModeWgrad && a.zero_tail)
      zero_tail_rows(a, (idx - per_xcd) * 8 + xcd, ((int)(gridDim.x >> 3) - per_xcd) * 8, kGemmThreads);
    return;
  }
  int tg = 0, mt, nt;
  if (MODE == kModeWgrad) {
    if ((mtiles & 7) == 0) {
      // Weight gradient: every XCD takes an eighth of the row tiles of EVERY group,
      // group after group.  Groups differ in length (slots are often empty), so
      // whole groups per XCD would leave the arithmetic to a few of them; this
      // way all finish together and a group's output is written by all XCDs at once.
      const int mpx = mtiles >> 3;
      tg = idx / (mpx * a.ntiles);
      const int r = idx - tg * (mpx * a.ntiles);
      nt = r / mpx;
      mt = xcd * mpx + (r - nt * mpx);
    } else {
      const int L0 = xcd * per_xcd + idx;
      if (L0 >= total) return;
      tg = L0 / per_group;
      const int L = L0 - tg * per_group;
      nt = L / mtiles;
      mt = L - nt * mtiles;
    }
  } else {
    const int L0 = xcd * per_xcd + idx;
    if (L0 >= total) return;
    // the group whose tiles contain list entry L0: the first whose padded end, counted
    // in tiles, lies beyond it (every wave finds it for itself: 64 groups are one ballot)
    tg = -1;
    int beg_tiles = 0, end_tiles = 0;
    for (int c = 0; c < a.G && tg < 0; c += 64) {
      const int e = c + lane < a.G ? a.cu[c + lane] / kBM : 0;
      const uint64_t m = __ballot(c + lane < a.G && e * a.ntiles > L0);
      if (m) {
        const int src = __ffsll((unsigned long long)m) - 1;
        tg = c + src;
        end_tiles = __shfl(e, src);
        const int prev = __shfl(e, src > 0 ? src - 1 : 0);
        beg_tiles = src > 0 ? prev : (c > 0 ? a.cu[c - 1] / kBM : 0);
      }
    }
    if (tg < 0) return;  // cannot happen: L0 < total
    // a long group goes in panels of kPanel row tiles (its weights are then read once per
    // panel, its rows once per 32 / kPanel weight tiles)
    const int h = end_tiles - beg_tiles;
    const int local = L0 - beg_tiles * a.ntiles;
    const int panel = local / (kPanel * a.ntiles);
    const int within = local - panel * (kPanel * a.ntiles);
    const int ph = min(kPanel, h - panel * kPanel);
    nt = within / ph;
    mt = beg_tiles + panel * kPanel + (within - nt * ph);
  }
  const int m0 = mt * kBM;
  const int n0 = nt * kBN;
  const int g = tg;

  // K steps of this tile and where its K range starts in a row
  int kbeg = 0, KT = a.K / kBK;
  if (MODE == kModeDual) KT *= 2;
  if (MODE == kModeWgrad) {
    kbeg = g > 0 ? a.cu[g - 1] : 0;
    KT = (a.cu[g] - kbeg) / kBK;
  }
  const size_t K = (size_t)a.ld;
  const bool any = KT > 0;  // a group without rows: its weight gradient is zero
  if (MODE == kModeWgrad && !any && g >= a.skip_from) return;  // ... and nobody reads it: an unused slot

  if (wave >= kConsumers) {
    // =============================== producer ===============================
    const int p = wave - kConsumers;
    const int r = lane >> 3, kv = lane & 7;
    // piece j of a stage: rows 8j .. 8j+7 of the row tile (j < 16), then of the
    // weight tile; this wave moves the pieces j = p, p + kProducers, ...
    // lane (r, kv) fetches vector kv ^ r ^ (piece & 1) of its row into slot (r, kv); this
    // wave's pieces all have the parity of p
    if (!any) return;
    const size_t goff = MODE == kModeWgrad ? (size_t)kbeg : (size_t)g * a.N * K;
    const size_t lane_off = (size_t)r * K + ((kv ^ r ^ (p & 1)) * 8);
    const uint16_t* Ap = a.A + (size_t)m0 * K + lane_off + (MODE == kModeWgrad ? (size_t)kbeg : 0);
    const uint16_t* Bp0 = a.B + goff + (size_t)n0 * K + lane_off;
    const uint16_t* Bp1 = Bp0 + (size_t)(kBN / 2) * K;
    // dual: the second half of the K loop reads the second pair
    const uint16_t* Aq = MODE == kModeDual ? a.A2 + (size_t)m0 * K + lane_off : Ap;
    const uint16_t* Bq0 = MODE == kModeDual ? a.B2 + goff + (size_t)n0 * K + lane_off : Bp0;
    const uint16_t* Bq1 = Bq0 + (size_t)(kBN / 2) * K;
    auto issue = [&](int k0, int stage) {
      char* base = gsm + stage * kStage;
      const bool second = MODE == kModeDual && k0 >= a.K;
      if (second) k0 -= a.K;
      const uint16_t* pa = second ? Aq : Ap;
      const uint16_t* pb0 = second ? Bq0 : Bp0;
      const uint16_t* pb1 = second ? Bq1 : Bp1;
#pragma unroll
      for (int q = 0; q < kPiecesPerProducer; ++q) {
        const int j = p + q * kProducers;  // 0 .. 47
        const uint16_t* src;
        if (j < kBM / 8) src = pa + (size_t)(8 * j) * K + k0;
        else if (j < kBM / 8 + kBN / 16) src = pb0 + (size_t)(8 * (j - kBM / 8)) * K + k0;
        else src = pb1 + (size_t)(8 * (j - kBM / 8 - kBN / 16)) * K + k0;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(base + j * 1024),
                                         16, 0, 0);
      }
    };
    const int klast = (KT - 1) * kBK;
    issue(0, 0);
    issue(min(kBK, klast), 1);
    mep_wait_vmcnt<kPiecesPerProducer>();  // step 0 has landed
    __builtin_amdgcn_s_barrier();
    int st = 2;  // stage of step kt + 2
    for (int kt = 0; kt < KT; ++kt) {
      issue(min((kt + 2) * kBK, klast), st);
      st = st == kStages - 1 ? 0 : st + 1;
      mep_wait_vmcnt<kPiecesPerProducer>();  // everything up to step kt + 1 has landed
      __builtin_amdgcn_s_barrier();
    }
    mep_wait_vmcnt<0>();
    return;
  }

  // ================================ consumer =================================
  const int wm = wave & 1, wn = wave >> 1;  // 2 x 4 waves, 64 x 64 each
  mep_f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // operand rows of this lane inside a stage (weight rows follow the kBM rows)
  const int arow = 64 * wm + (lane & 31);
  const int brow0 = kBM + 64 * wn + (lane & 31);
  const int brow1 = brow0 + 32;
  const int sw = (lane & 7) ^ ((lane >> 3) & 1);  // (row & 7) ^ ((row >> 3) & 1) of every operand row of this lane
  const int half = lane >> 5;   // which 8 of the 16 K values of an MFMA step
  const int oa0 = arow * kRowBytes, oa1 = (arow + 32) * kRowBytes;
  const int ob0 = brow0 * kRowBytes, ob1 = brow1 * kRowBytes;
  if (any) {
    __builtin_amdgcn_s_barrier();  // stage 0 is filled
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  int st = 0;
  for (int kt = 0; kt < KT; ++kt) {
    const char* sb = gsm + st * kStage;
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      const int col = ((2 * ks + half) ^ sw) * 16;
      const mep_bf16x8 a0 = *(const mep_bf16x8*)(sb + oa0 + col);
      const mep_bf16x8 a1 = *(const mep_bf16x8*)(sb + oa1 + col);
      const mep_bf16x8 b0 = *(const mep_bf16x8*)(sb + ob0 + col);
      const mep_bf16x8 b1 = *(const mep_bf16x8*)(sb + ob1 + col);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, acc[1][1], 0, 0, 0);
    }
    st = st == kStages - 1 ? 0 : st + 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // the reads of this stage are done
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }

  // ---- epilogue.  acc[i][j][v]: row 64*wm + 32*i + 8*(v/4) + 4*(lane/32) + v%4,
  // column (lane % 32) of the j-th 32-wide block
  const int ldc = a.N;
  float* cf = MODE == kModeWgrad ? a.Cf + (size_t)g * a.M * a.N : nullptr;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = m0 + 64 * wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (MODE == kModeWgrad) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          // streaming stores: 58 MB of output per group passing through L2 as ordinary
          // writes evicts the operand lines the other tiles of the group still need (9 % slower)
          __builtin_nontemporal_store(acc[i][j][v], &cf[(size_t)m * ldc + n0 + 64 * wn + 32 * j + (lane & 31)]);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = n0 + 64 * wn + 32 * j + (lane & 31);
          a.C[(size_t)m * ldc + n] = (uint16_t)mep_f32_to_bf16_bits(acc[i][j][v]);
        }
      }
    }
}

// ---------------------------------------------------------------------------
// The weight gradient, and products of long groups of which few CUs get a tile (the others are
// gemm_wide_kernel's): 256 x 256 output tiles, K in steps of 64, 8 waves of 128 x 64 (two on every
// SIMD), one workgroup per CU.
//
// What bounds it: latency of the loads first (a step's 64 KB arrive 1.8 us after they were asked
// for when the chip is busy, and its matrix instructions take 0.9), then the matrix cores at the
// clock their power leaves.  Hence
//  * loads go straight into LDS, half an operand's tile (16 KB) at a time, into five slots per
//    operand that are taken in turn: a half tile is asked for as soon as the one that had the slot
//    five turns before has been read, four of a step's eight half-phases -- two K steps -- before
//    it is wanted, and 64 to 96 KB per CU are in flight at every moment (the whole LDS of a CU is
//    these slots);
//  * s_waitcnt vmcnt(n) waits for the half tiles the next phase reads and leaves the rest in
//    flight.  Neither a workgroup fence nor the compiler's transposing LDS read may stand in the
//    loop: both wait for every load straight into LDS (that alone made the [K, N] forms 20 %
//    slower);
//  * a K step has two phases, rows 0 .. 127 and 128 .. 255 of the tile: read fragments and issue
//    loads | barrier | 16 matrix instructions | barrier.  The waves 4 .. 7 run one barrier behind
//    the waves 0 .. 3, so on every SIMD one wave multiplies while the other reads (without the
//    shift 14 % slower; four phases of 8 instructions 2 % slower);
//  * a workgroup walks its tiles as one stream of K steps: the next tile's loads are on their way
//    while this one is finished and stored (10 % for K = 2048).  It takes kPSteps steps, then
//    leaves its CU to the next one (see there).  The forward products also fetch less from HBM that
//    way, 7.4 GB instead of 9.2 (operands 6.3): an XCD's workgroups drift apart over a long walk,
//    and lines that several tiles share leave L2 in between.
// Groups end on multiples of 128 rows: a group of h 128-row blocks is h / 2 tiles and, if h is
// odd, one of 128 rows whose second phase has no matrix instructions.
//
// Weight gradient at 34 688 rows in 33 groups, H = 7168, H' = 2048 (us, before -> now; before: one
// 256-row kernel with two LDS stages that drained its loads every step): 1555 -> 1314 (1.1 GB of fp32
// zeroes for unused groups included; on another card 1358 -> 1303 with the list by groups, which spreads the zeroes
// over the workgroups, 1052 -> 1027 without zeroes).  A step of it takes 1.2 to 1.6 us: 192 KB of transposing LDS reads (200
// bytes a clock in this layout, half of the 2048 clocks of the matrix instructions) and 64 KB of loads.  What
// it waits for is its own stores: 64 experts of 2048 x 1024, 512 rows each, take 624 us, without stores 395, with
// stores but without loads 453 (loads that follow 256 KB of stores wait behind them, and loads that miss L2 longest).
// gemm_wide_kernel reads 128 KB, but has nothing beside its stores of fp32: from equal (32 steps a tile) to
// 15 % slower (8).  Not faster: stores of 16 bytes in pieces of 32 (6 % slower) or 64 (17 %), in whole 256 bytes
// (0), plain ones (4 % slower) or written through (3 %), waits that leave them in flight for the next tile's first
// steps (1 to 6 % slower), workgroups started a quarter of a tile apart (0), 16 x 16 x 32 instructions (0 to 5 % slower).
//
// LDS layouts.  Operand rows along K: 128 bytes per row and step, 16-byte vector q of row r at
// position q ^ (r & 7) ^ ((r >> 3) & 1): sixteen consecutive lanes cover all banks.  Operands
// given as [K, columns] (weights of the input gradients, activations of the weight gradient): 64
// rows of 256 bytes, vector v of row k at v ^ 4 (k & 3), read with transposing LDS reads (four
// rows of 32 bytes per sixteen lanes): two such blocks side by side cover all banks.
// ---------------------------------------------------------------------------
constexpr int kPThreads = 512;
constexpr int kPHalf = 128 * kRowBytes;   // 16 KB: half of one operand's tile of a K step
constexpr int kPSlots = 5;                // of each operand
constexpr int kPOperand = kPSlots * kPHalf;
constexpr int kPLds = 2 * kPOperand;      // 160 KB
// K steps of a workgroup, about 200 us.  With one share of the whole list per CU a kernel that holds
// 32 CUs beside the product (Buffer(num_sms=32) while the FFN runs on a stream of its own) left 32
// shares waiting until others had ended, and a communication kernel asked for meanwhile waited for
// the whole product.  Beside dispatch and combine on 32 CUs, us, one share -> 128 steps: forward of
// S = 4096, 7168 x 2048, E = 256 3364 -> 2930, forward and backward of S = 4096, 4096 x 2048, E = 128
// 7177 -> 5900 (64 steps 2940 / 5600, 224 steps 3130 / 6130).  With the whole chip 2661 -> 2636 and
// 4816 -> 4824, a layer of small experts 2481 -> 2502 (64 steps: 2 % slower): a change of workgroups
// costs some 4 us, and their shares end more evenly.
constexpr int kPSteps = 128;

// AT, BT: the operand is given as [K, columns].  SCALED: scale mode with row scales.
template <int MODE, bool AT, bool BT, bool SCALED = false>
__global__ __launch_bounds__(kPThreads, 2) void gemm_pp_kernel(GemmArgs a, WgradMap map) {
  constexpr bool DUAL = MODE == kModeDual, WGRAD = MODE == kModeWgrad, FORWARD = MODE == kModeScale && !BT;
  static_assert(!AT || WGRAD, "rows of the other products lie along K");
  static_assert(MODE != kModeSwiglu, "gemm_wide_kernel has it");
  extern __shared__ __attribute__((aligned(1024))) char gsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, half = lane >> 5;

  // ---- loads: a cursor over (tile, K step)
  // pitches; of a weight gradient's operands, [rows, M] and [rows, N], those of the product at hand
  size_t ldA = AT ? (size_t)a.M : (size_t)a.ld, ldB = BT ? (size_t)a.N : (size_t)a.ld;
  const int KT1 = WGRAD ? 0 : a.K / kBK;
  [[maybe_unused]] const bool fold = FORWARD && mep_folds(a.K);
  using Tiles = std::conditional_t<WGRAD, WgradTiles<AT>, PTiles<MODE>>;
  Tiles ld(a, &map, gsm);
  Tiles cp = ld;  // the tiles as they are multiplied; what describes them is read once for both
  // Groups without rows: whole 1 KB rows of zeroes per wave instruction, between the K steps of the workgroup's tiles, as
  // many tiles of zeros to each and not at the same time on all CUs: a CU alone writes 50 bytes a clock, all together 15
  // each.  (16 groups of 4096 x 2048 with 2048 rows and as many without, us: half of the workgroups in front of
  // their tiles, half behind them 1587, this 1549; a row per wave and K step, among the loads, whose waits then are for stores, too, 1617;
  // without zeros 1440 to 1500.)
  auto write_zeros = [&](int tiles) {
    if constexpr (WGRAD) {
      mep_global_f32* out;
      int N;
      for (; tiles > 0 && cp.blank(&out, &N); --tiles) {
        typedef __attribute__((address_space(1))) mep_f32x4 global_f32x4;
        const mep_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int row = wave; row < kPT; row += 8) __builtin_nontemporal_store(zero, (global_f32x4*)(out + (size_t)row * N) + lane);
      }
    }
  };
  const char *pA, *pB;
  uint32_t halfA, halfB;
  int kl = 0;
  uint32_t vA[2], vB[2];
  auto lanes = [&]() {
    const int r = lane >> 3, kv = lane & 7, lk = lane >> 4, lv = lane & 15;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int j = 2 * wave + q;
      vA[q] = AT ? (uint32_t)((4 * j + lk) * ldA * 2 + ((lv ^ (lk << 2)) * 16)) : (uint32_t)((8 * j + r) * ldA * 2 + ((kv ^ r ^ q) * 16));
      vB[q] = BT ? (uint32_t)((4 * j + lk) * ldB * 2 + ((lv ^ (lk << 2)) * 16)) : (uint32_t)((8 * j + r) * ldB * 2 + ((kv ^ r ^ q) * 16));
      vA[q] -= q * 1024;  // what the instruction adds to both addresses (never more than is there: K is at least 64, M and N 256)
      vB[q] -= q * 1024;
    }
  };
  if (!WGRAD) lanes();
  int of = -1;  // weight gradient: the product that the pitches are of
  auto stand = [&](int pair) {  // the pointers at the first K step of the cursor's tile (of its second pair)
    if constexpr (WGRAD) {
      if (of != ld.p) {
        of = ld.p;
        if (AT) ldA = (size_t)map.M(of);
        if (BT) ldB = (size_t)map.N(of);
        lanes();
      }
      pA = ld.A();
      pB = ld.B();
    } else {
      const size_t offB = (size_t)ld.g * a.N * a.K + (BT ? (size_t)ld.n0 : (size_t)ld.n0 * ldB);
      pA = mep_uniform((const char*)((pair ? a.A2 : a.A) + (size_t)ld.m0 * ldA));
      pB = mep_uniform((const char*)((pair ? a.B2 : a.B) + offB));
    }
    halfA = __builtin_amdgcn_readfirstlane(ld.tall ? (AT ? 256u : (uint32_t)(128 * ldA * 2)) : 0u);
    halfB = BT ? 256u : (uint32_t)(128 * ldB * 2);
  };
  bool more = ld.next();
  if (more) stand(0);
  auto advance = [&]() {
    if (!more) return;
    if (kl + 1 < ld.KT) {
      ++kl;
      if (DUAL && kl == KT1) { stand(1); return; }
      const int step = FORWARD && fold ? mep_fold_step(kl - 1) : kRowBytes;
      if (AT) pA += kBK * ldA * 2;
      else pA += step;
      if (BT) pB += kBK * ldB * 2;
      else pB += step;
      return;
    }
    more = ld.next();
    if (more) { kl = 0; stand(0); }  // otherwise the last step is loaded again, for nobody
  };
  // slots are taken in turn: where the next half tile of each operand is written and read
  int wA = 0, wB = kPOperand, rA = 0, rB = kPOperand;
  auto turn = [](int& slot, int first) { slot = slot == first + (kPSlots - 1) * kPHalf ? first : slot + kPHalf; };
  char* lds_w = gsm + wave * 2048;
  auto issueA = [&](int h) {
    mep_load_lds16(pA, vA[0], h ? halfA : 0u, lds_w + wA);
    mep_load_lds16<0, 1024>(pA, vA[1], h ? halfA : 0u, lds_w + wA);
    turn(wA, 0);
  };
  auto issueB = [&](int h) {
    mep_load_lds16(pB, vB[0], h ? halfB : 0u, lds_w + wB);
    mep_load_lds16<0, 1024>(pB, vB[1], h ? halfB : 0u, lds_w + wB);
    turn(wB, kPOperand);
  };

  // ---- fragments
  const int wm = wave >> 2, wn = wave & 3;
  const int sw = (lane & 7) ^ ((lane >> 3) & 1);
  const int ts = lane & 15, tb = (lane >> 4) & 1;
  int adA[4], adB[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int col = ((2 * ks + half) ^ sw) * 16;
    adA[ks] = (64 * wm + l31) * kRowBytes + col;
    adB[ks] = (32 * wn + l31) * kRowBytes + col;
  }
  const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) char*)gsm;
  const int trow = lds0 + (8 * half + (ts >> 2)) * 256 + (ts & 1) * 8;
  const int tvec = 2 * tb + ((ts & 3) >> 1);
  if (AT) {
    adA[0] = trow + (((8 * wm + tvec) ^ ((ts >> 2) << 2)) * 16);
    adA[1] = adA[0] ^ 64;
  }
  if (BT) adB[0] = trow + (((4 * wn + tvec) ^ ((ts >> 2) << 2)) * 16);
  mep_bf16x8 fa[2][4], fb0[4], fb1[4];
  mep_s16x4 ta[2][4][2], tb0[4][2], tb1[4][2];  // transposed reads until they have arrived
  auto readA = [&]() {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (AT) {
#pragma unroll
          for (int u = 0; u < 2; ++u) mep_tr_issue(ta[i][ks][u], adA[i] + rA, ks * 4096 + u * 1024);
        } else {
          fa[i][ks] = *(const mep_bf16x8*)(gsm + (adA[ks] + rA) + i * 32 * kRowBytes);
        }
      }
    turn(rA, 0);
  };
  auto readB = [&](mep_bf16x8* fb, mep_s16x4 (*tbw)[2]) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (BT) {
#pragma unroll
        for (int u = 0; u < 2; ++u) mep_tr_issue(tbw[ks][u], adB[0] + rB, ks * 4096 + u * 1024);
      } else {
        fb[ks] = *(const mep_bf16x8*)(gsm + (adB[ks] + rB));
      }
    }
    turn(rB, kPOperand);
  };
  auto join = [](const mep_s16x4* t) {
    return __builtin_bit_cast(mep_bf16x8, __builtin_shufflevector(t[0], t[1], 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto gotA = [&]() {  // after the wait
    if (!AT) return;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        asm volatile("; arrived %0 %1" : "+v"(ta[i][ks][0]), "+v"(ta[i][ks][1]));
        fa[i][ks] = join(ta[i][ks]);
      }
  };
  auto gotB = [&](mep_bf16x8* fb, mep_s16x4 (*tbw)[2]) {
    if (!BT) return;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      asm volatile("; arrived %0 %1" : "+v"(tbw[ks][0]), "+v"(tbw[ks][1]));
      fb[ks] = join(tbw[ks]);
    }
  };
  mep_f32x16 acc[2][2][2];
  auto mm = [&](int hA) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[hA][0][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][ks], fb0[ks], acc[hA][0][i], 0, 0, 0);
        acc[hA][1][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][ks], fb1[ks], acc[hA][1][i], 0, 0, 0);
      }
    __builtin_amdgcn_s_setprio(0);
  };

  // ---- prologue: the first two K steps
  if (more) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      issueA(0); issueB(0); issueB(1); issueA(1);
      advance();
    }
    mep_wait_vmcnt<10>();
    mep_bar();
    if (wave >= 4) mep_bar();
  }
  bool any = false;
  while (cp.next()) {
    const int KT = cp.KT;
    const bool tall = cp.tall;
    int m0 = 0, n0 = 0, N = a.N;
    mep_global_f32* cf = nullptr;
    if constexpr (WGRAD) {
      cf = cp.C();
      N = map.N(cp.p);
    } else {
      m0 = cp.m0; n0 = cp.n0;
    }
    if (SCALED) __builtin_assume(KT > 0);
    any = true;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[x][y][i][v] = 0.0f;
    // The scales of this wave's rows, one per lane: asked for here, in order before the tile's
    // loads, and there by the epilogue (a load the compiler knows would be waited for there, and
    // with it every load of the next tile).
    float scl0 = 1.0f, scl1 = 1.0f;
    if (SCALED) {
      const float* sp = a.scale + m0 + 64 * wm + lane;
      asm volatile("global_load_dword %0, %1, off" : "=v"(scl0) : "v"(sp));
      asm volatile("global_load_dword %0, %1, off" : "=v"(scl1) : "v"(sp + (tall ? 128 : 0)));
    }
    int zeros_at = -1, zeros = 0;
    if constexpr (WGRAD) {
      const int tiles = 1 + __popcll(cp.left);
      zeros = mep_quotient(__popcll(cp.empties) + tiles - 1, tiles);
      zeros_at = (int)(blockIdx.x >> 3 & 7) * KT >> 3;
    }
    for (int kt = 0; kt < KT; ++kt) {
      if (WGRAD && kt == zeros_at) write_zeros(zeros);
      readA();
      readB(fb0, tb0);
      readB(fb1, tb1);
      issueA(0);
      issueB(0);
      mep_wait_vm_lgkm0<12>();
      gotA();
      gotB(fb0, tb0);
      gotB(fb1, tb1);
      mep_bar();
      mm(0);
      mep_bar();

      readA();
      issueB(1);
      issueA(1);
      advance();
      mep_wait_vm_lgkm0<10>();
      gotA();
      mep_bar();
      if (tall) mm(1);
      mep_bar();
    }

    if (SCALED) {
      mep_wait_vmcnt<8>();  // a K step's loads came after them; the next phase would wait for as many
      asm volatile("; arrived %0 %1" : "+v"(scl0), "+v"(scl1));
    }
    // ---- epilogue: acc[x][y][i][v] is row 128 x + 64 wm + 32 i + 8 (v / 4) + 4 half + v % 4,
    // column 128 y + 32 wn + l31
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      if (x == 1 && !tall) break;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = m0 + 128 * x + 64 * wm + 32 * i + 4 * half;
        if (WGRAD) {
          mep_global_f32* out = cf + (size_t)m * N + n0 + 32 * wn + l31;
#pragma unroll
          for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int y = 0; y < 2; ++y)
              __builtin_nontemporal_store(acc[x][y][i][v], out + (size_t)(8 * (v >> 2) + (v & 3)) * N + 128 * y);
        } else {
          // bf16: two rows of a column pair at a time -- the even lane of a pair stores both
          // columns of the first row, the odd lane both of the second
          int at0 = 16 * half;
          asm volatile("" : "+v"(at0));  // addresses made here, not kept in registers across the main loop
          const bool odd = lane & 1;
          const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
          const size_t first = (size_t)(m + odd) * N + n0 + 32 * wn + (l31 & ~1);
          auto put = [&](uint16_t* c, int v, int col, float v0, float v1) {
            const uint32_t w = mep_cvt_bf16x2(v0, v1);
            const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0xB1, 0xf, 0xf, true);  // the pair's other lane
            *(mep_u1_any*)(c + first + (size_t)(8 * (v >> 2) + (v & 3)) * N + col) = __builtin_amdgcn_perm(o, w, sel);
          };
#pragma unroll
          for (int v = 0; v < 16; v += 2) {
            const float g0 = acc[x][0][i][v], g1 = acc[x][0][i][v + 1], u0 = acc[x][1][i][v], u1 = acc[x][1][i][v + 1];
            if (SCALED) {
              const int at = at0 + 4 * (32 * i + 8 * (v >> 2) + (v & 3));
              const float s0 = __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(x ? scl1 : scl0)));
              const float s1 = __int_as_float(__builtin_amdgcn_ds_bpermute(at + 4, __float_as_int(x ? scl1 : scl0)));
              put(a.C, v, 0, s0 * g0, s1 * g1);
              put(a.C, v, 128, s0 * u0, s1 * u1);
            } else {
              put(a.C, v, 0, g0, g1);
              put(a.C, v, 128, u0, u1);
            }
          }
        }
      }
    }
  }
  if (any && wave < 4) mep_bar();
  mep_wait_vmcnt<0>();  // the loads of steps nobody wanted write LDS, too
  write_zeros(1 << 30);
  if (!WGRAD && a.zero_tail) zero_tail_rows(a, blockIdx.x, gridDim.x, kPThreads);
}
// ---------------------------------------------------------------------------
// Forward products of groups of about one 128-row block (decode batches): every weight is read
// once and its bytes are the time, 805 MB for 16 experts of 4096 x 2048.
//
// A unit is 32 weight rows (SwiGLU: 16 gate rows and the same 16 up rows) times one 128-row block.
// Tiles are 128 rows x one to nine units, so that the tiles of all blocks fill the CUs evenly
// however many groups have rows (whole 128 x 256 tiles leave 17 blocks of 4096 weight rows with
// 272 tiles for 256 CUs: a second round for sixteen of them) and the rows come from L2 once for up
// to 288 weight rows.  A K step of 64 is 16 KB of rows and 4 KB a unit; the whole LDS holds D of
// them, D - 1 on their way (72 KB of weights per CU at nine units) while one is multiplied.
// 8 waves: 32 rows each, every other unit.  In tiles of seven units and more (fewer have little to read in
// a step: 2816 x 256 12.0 us that way, 11.6 in step) the waves 4 .. 7 run one barrier behind the waves 0 .. 3,
// so that one wave of a SIMD multiplies while the other reads: a step's 160 to 192 KB of LDS reads
// take about as long as its matrix instructions, and one after the other, with one barrier a step, the
// two were 1.17 us a step of eight units and 1.33 of nine, however few of the CUs were still at work
// (us, before -> now, 17 blocks: down 4096 x 4096 102 -> 96, 4096 x 7168 176 -> 169, 2048 x 4096
// 61 -> 57, SwiGLU 2048 x 4096 100 -> 98, down 4096 x 2048 the same; the [K, N] form below is 0 to 5 %
// slower that way).  All of a step's fragments are
// asked for before the next loads are issued (behind them they waited: 78 against 54 us where a
// tile has one or two units); weights are loaded nontemporal, so that the rows stay in L2 (183
// against 202 us at 17 blocks).  The order of the K steps is that of the shape (mep_fold_step), as in the
// other kernels: the order of a sum does not depend on where its tile lies.
//
// The tiles of a block divide its units evenly and are as many as fill whole rounds of the grid:
// cut where a CU's even share of the list ends, a tile in two blocks ran its K loop twice with
// half the weights in flight (17 blocks: 209 us).
//
// Measured, FFN forward of 64 tokens, K = 8, experts of 4096 x 2048, E = 128 on 8 ranks, before
// (128 x 256 tiles) -> now: 16 blocks 200 -> 168 us, 17 blocks 290 -> 183 us (4.7 TB/s of
// weights), 18 blocks (two rounds) 323 -> 216 us; 7168 x 2048, 33 blocks 720 -> 582 us.
// The forward of 17 blocks on another card 211 -> 202 us with the epilogue's selects of two values and the row scales read
// before the loads, of 18 232 -> 219, of 24 314 -> 298, 7168 x 2048 with 33 583 -> 558.  What a tile takes beside its
// K steps now: 1.2 us to its group, 0.8 to the last of the first loads, 2 to 3 to their arrival, 1.4 (down) to 4 (SwiGLU) to store.
// With the order of the K steps and the waves' two shifts, 64 tokens at 17 blocks: 190 -> 161 and 170 -> 158 on two cards.
// ---------------------------------------------------------------------------
typedef float mep_f32x4_any __attribute__((ext_vector_type(4), aligned(4)));  // at any element
constexpr int kSThreads = 512;
constexpr int kSUnits = 9;                 // most units of a tile
constexpr int kSA = kBM * kRowBytes;       // 16 KB
constexpr int kSUnit = 32 * kRowBytes;     // 4 KB
constexpr int kSLds = 160 * 1024;
constexpr int kSParts = 2;                 // workgroups that share what a CU does

// Two rows of a pair of neighbouring columns, one column a lane: the even lane stores both columns of the
// first row, the odd lane both of the second.  c: the row and the first column of what this lane stores
// (one value at a time: FFN forward of 64 tokens, 16 experts of 4096 x 2048 198 -> 195.6 us, of 18 tokens,
// 4 experts of 3072 x 512 49 -> 47.6, of 106 tokens, 8 experts of 2816 x 256 36.7 -> 35).
__device__ __forceinline__ void store_two_rows(uint16_t* c, float row0, float row1) {
  const uint32_t w = mep_cvt_bf16x2(row0, row1);
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0xB1, 0xf, 0xf, true);  // the pair's other lane
  *(mep_u1_any*)c = __builtin_amdgcn_perm(o, w, threadIdx.x & 1 ? 0x03020706u : 0x05040100u);
}

template <int MODE, int NU, bool FOLD>
__device__ __forceinline__ void stream_tile(const GemmArgs& a, char* gsm, int m0, int g, int unit0) {
  constexpr bool SWIGLU = MODE == kModeSwiglu;
  constexpr int kStageBytes = kSA + NU * kSUnit;
  constexpr int D = kSLds / kStageBytes < 8 ? kSLds / kStageBytes : 8;
  constexpr bool kShift = NU >= 7;                // the waves 4 .. 7 run one barrier behind the others
  constexpr int kHi = (NU + 1) / 2, kLo = NU / 2;  // units of the waves 0 .. 3 and 4 .. 7; as many pieces to load
  static_assert(D >= 3 && (D - 1) * (2 + kHi) < 64, "the loads on their way must fit the 6-bit counter");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, half = lane >> 5;
  const int rb = wave & 3, uh = wave >> 2;
  const bool lower = wave < 4;
  const size_t ld = (size_t)a.K * 2;
  const int KT = a.K / kBK;

  // ---- loads.  A wave brings the row pieces 2 wave, 2 wave + 1 and the weight pieces wave + 8 i
  // (1 KB: 8 rows of 128 bytes); vector q of LDS row r lies at q ^ (r & 7) ^ ((r >> 3) & 1)
  const int r = lane >> 3, kv = lane & 7;
  const char* pA = mep_uniform((const char*)a.A + (size_t)(m0 + 16 * wave) * ld);
  const uint16_t* mat = SWIGLU && (wave >> 1 & 1) ? a.B2 : a.B;
  const int row0 = SWIGLU ? 16 * (unit0 + (wave >> 2)) + 8 * (wave & 1) : 32 * unit0 + 8 * wave;
  const char* pB = mep_uniform((const char*)mat + ((size_t)g * a.N + row0) * ld);
  const uint32_t strideB = (uint32_t)((SWIGLU ? 32 : 64) * ld);
  uint32_t vA[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) vA[q] = (uint32_t)((8 * q + r) * ld + ((kv ^ r ^ q) * 16));
  const uint32_t vB = (uint32_t)(r * ld + ((kv ^ r ^ (wave & 1)) * 16));
  int kl = 0, ws = 0, rs = 0;
  auto issue = [&]() {
    const int bytes = __builtin_amdgcn_readfirstlane(kl < KT ? -1 : 0);  // past the last step: counted, but nothing is read
    char* slot = gsm + ws;
#pragma unroll
    for (int q = 0; q < 2; ++q) mep_load_lds16(pA, vA[q], 0, slot + (2 * wave + q) * 1024, bytes);
#pragma unroll
    for (int i = 0; i < kLo; ++i) mep_load_lds16<kNontemporal>(pB, vB, i * strideB, slot + kSA + (wave + 8 * i) * 1024, bytes);
    if (kHi > kLo && lower) mep_load_lds16<kNontemporal>(pB, vB, kLo * strideB, slot + kSA + (wave + 8 * kLo) * 1024, bytes);
    const int step = FOLD ? mep_fold_step(kl) : kRowBytes;
    pA += step; pB += step;
    ++kl;
    ws = ws == (D - 1) * kStageBytes ? 0 : ws + kStageBytes;
  };
  // Row scales before all other loads: one that is asked for behind stores is waited for with them, again for every unit
  // (the stores of nine units of 4096 x 2048 took 8.2 us of a down product's 74, now 1.4).
  const int m = m0 + 32 * rb + 4 * half;
  mep_f32x4 scale[4];
  if (!SWIGLU)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      scale[q] = mep_f32x4{1.0f, 1.0f, 1.0f, 1.0f};
      if (a.scale) scale[q] = *(const mep_f32x4_any*)(a.scale + m + 8 * q);
    }
#pragma unroll
  for (int k = 0; k < D - 1; ++k) issue();

  mep_f32x16 acc[kHi];
#pragma unroll
  for (int i = 0; i < kHi; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
  const int sw = (lane & 7) ^ ((lane >> 3) & 1);
  int ad[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) ad[ks] = l31 * kRowBytes + ((2 * ks + half) ^ sw) * 16;

  // this wave's part of the next step is there
  auto next_in = [&]() {
    if (kHi == kLo || lower) mep_wait_vm_lgkm0<(D - 2) * (2 + kHi)>();
    else mep_wait_vm_lgkm0<(D - 2) * (2 + kLo)>();
  };
  if (kShift) {
    next_in();
    mep_bar();
    if (!lower) mep_bar();
  }
  for (int kt = 0; kt < KT; ++kt) {
    if (!kShift) {
      next_in();
      mep_bar();
    }
    // everybody's part of step kt is there, and the slot of the step before has been read by all
    const char* sa = gsm + rs + rb * 32 * kRowBytes;
    const char* sb = gsm + rs + kSA + uh * kSUnit;
    mep_bf16x8 fa[4], fb[4][kHi];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      fa[ks] = *(const mep_bf16x8*)(sa + ad[ks]);
#pragma unroll
      for (int i = 0; i < kHi; ++i)  // one more than the upper waves multiply, where NU is odd
        fb[ks][i] = *(const mep_bf16x8*)(sb + ad[ks] + (i < kLo || lower ? 2 * i * kSUnit : 0));
    }
    __builtin_amdgcn_sched_barrier(0);
    issue();
    __builtin_amdgcn_sched_barrier(0);
    if (kShift) {
      mep_wait_lgkm0();
      if (!lower) next_in();
      mep_bar();
      __builtin_amdgcn_s_setprio(1);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int i = 0; i < kLo; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks], fb[ks][i], acc[i], 0, 0, 0);
      if (kHi > kLo && lower)
        acc[kHi - 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks], fb[ks][kHi - 1], acc[kHi - 1], 0, 0, 0);
    }
    rs = rs == (D - 1) * kStageBytes ? 0 : rs + kStageBytes;
    if (kShift) {
      __builtin_amdgcn_s_setprio(0);
      if (lower) next_in();
      mep_bar();
    }
  }
  if (kShift && lower) mep_bar();
  mep_wait_vm_lgkm0<0>();  // the loads past the last step write LDS, too
  mep_bar();               // the next tile may be loaded

  // ---- epilogue: acc[i][v] is row 32 rb + 8 (v / 4) + 4 half + v % 4, weight row l31 of unit 2 i + uh
#pragma unroll
  for (int i = 0; i < kHi; ++i) {
    if (i >= kLo && !lower) break;
    const int unit = unit0 + 2 * i + uh;
    if (SWIGLU) {
      // gate in the lanes 0 .. 15 of a half wave, up in 16 .. 31: the first take the rows of
      // v = 0 .. 7, the others of v = 8 .. 15, and hand each other what they lack
      const bool up = l31 >= 16;
      const size_t first = (size_t)(m + (up ? 16 : 0) + (lane & 1)) * a.N + 16 * unit + (l31 & 14);
#pragma unroll
      for (int v = 0; v < 8; v += 2) {
        float gv[2], uv[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          // two values: of one element at either of two places the compiler makes fifteen compares and selects
          // (24 854 -> 10 332 instructions; 2.3 us a unit -> 0.7; 2816 x 1408 at 18 blocks SwiGLU 61 -> 56 us)
          float early = acc[i][v + e], late = acc[i][v + 8 + e];
          asm volatile("" : "+v"(early), "+v"(late));
          const float mine = up ? late : early;
          const float other = __shfl_xor(up ? early : late, 16);
          gv[e] = up ? other : mine;
          uv[e] = up ? mine : other;
        }
        const size_t o = first + (size_t)(8 * (v >> 2) + (v & 3)) * a.N;
        store_two_rows(a.C + o, mep_silu(gv[0]) * uv[0], mep_silu(gv[1]) * uv[1]);
        if (a.Cg) store_two_rows(a.Cg + o, gv[0], gv[1]);
        if (a.Cu) store_two_rows(a.Cu + o, uv[0], uv[1]);
      }
    } else {
      uint16_t* c = a.C + (size_t)(m + (lane & 1)) * a.N + 32 * unit + (l31 & ~1);
#pragma unroll
      for (int v = 0; v < 16; v += 2)
        store_two_rows(c + (size_t)(8 * (v >> 2) + (v & 3)) * a.N, scale[v >> 2][v & 3] * acc[i][v], scale[v >> 2][(v & 3) + 1] * acc[i][v + 1]);
    }
  }
}

// The same for weights given as [K, N] (input gradients, alone or as a sum of two pairs).  A unit is 64
// weight columns: a K step of it is 64 rows of 128 bytes in LDS, 16-byte vector v of row k at v ^ 2 (k & 3),
// so that the two blocks of 4 x 16 which 32 lanes read with a transposing read cover all banks.  A wave
// brings eight of the 64 rows and multiplies 32 rows by 32 columns of every unit.  us, dy * down and both
// pairs, 128 x 256 tiles -> this: 4 blocks of K = 5632, 768 columns 97 / 181 -> 44 / 82; 12 of 1024 x 1024
// 26 / 41 -> 13 / 21; 24 of 2048 x 4096 90 / 160 -> 88 / 155 (weights at 4.8 and 5.4 TB/s).
constexpr int kSUnitsKn = 4;
constexpr int kSUnitKn = 64 * kRowBytes;   // 8 KB

template <int MODE, int NU>
__device__ __forceinline__ void stream_tile_kn(const GemmArgs& a, char* gsm, int m0, int g, int unit0) {
  constexpr bool DUAL = MODE == kModeDual;
  constexpr int kStageBytes = kSA + NU * kSUnitKn;
  constexpr int D = kSLds / kStageBytes < 8 ? kSLds / kStageBytes : 8;
  static_assert(D >= 3 && (D - 1) * (2 + NU) < 64, "the loads on their way must fit the 6-bit counter");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, half = lane >> 5;
  const int rb = wave & 3, uh = wave >> 2;
  const size_t ldA = (size_t)a.K * 2, ldB = (size_t)a.N * 2;
  const int KT1 = a.K / kBK, KT = DUAL ? 2 * KT1 : KT1;

  const int r = lane >> 3, kv = lane & 7;
  const size_t offA = (size_t)(m0 + 16 * wave) * ldA;
  const size_t offB = ((size_t)g * a.K + 8 * wave) * ldB + (size_t)unit0 * kRowBytes;
  const char* pA = mep_uniform((const char*)a.A + offA);
  const char* pB = mep_uniform((const char*)a.B + offB);
  uint32_t vA[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) vA[q] = (uint32_t)((8 * q + r) * ldA + ((kv ^ r ^ q) * 16));
  const uint32_t vB = (uint32_t)(r * ldB + ((kv ^ (r & 3) << 1) * 16));
  int kl = 0, ws = 0, rs = 0;
  auto issue = [&]() {
    if (DUAL && kl == KT1) {
      pA = mep_uniform((const char*)a.A2 + offA);
      pB = mep_uniform((const char*)a.B2 + offB);
    }
    const int bytes = __builtin_amdgcn_readfirstlane(kl < KT ? -1 : 0);  // past the last step: counted, but nothing is read
    char* slot = gsm + ws;
#pragma unroll
    for (int q = 0; q < 2; ++q) mep_load_lds16(pA, vA[q], 0, slot + (2 * wave + q) * 1024, bytes);
#pragma unroll
    for (int i = 0; i < NU; ++i)
      mep_load_lds16<kNontemporal>(pB, vB, i * kRowBytes, slot + kSA + i * kSUnitKn + wave * 1024, bytes);
    pA += kRowBytes;
    pB += kBK * ldB;
    ++kl;
    ws = ws == (D - 1) * kStageBytes ? 0 : ws + kStageBytes;
  };
  // row scales before all other loads, as in stream_tile (dy * down with them, 12 blocks of 1024 x 1024 13.9 -> 13.2 us, 4 of K =
  // 5632, 768 columns 43.5 -> 42.6, 18 of K = 4096, 2048 columns 66.6 -> 65.3)
  const int m = m0 + 32 * rb + 4 * half;
  mep_f32x4 scale[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    scale[q] = mep_f32x4{1.0f, 1.0f, 1.0f, 1.0f};
    if (!DUAL && a.scale) scale[q] = *(const mep_f32x4_any*)(a.scale + m + 8 * q);
  }
#pragma unroll
  for (int k = 0; k < D - 1; ++k) issue();

  mep_f32x16 acc[NU];
#pragma unroll
  for (int i = 0; i < NU; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
  const int sw = (lane & 7) ^ ((lane >> 3) & 1);
  int ad[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) ad[ks] = (32 * rb + l31) * kRowBytes + ((2 * ks + half) ^ sw) * 16;
  // a block of sixteen lanes reads four rows of K by sixteen columns
  const int ts = lane & 15, tb = (lane >> 4) & 1;
  const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) char*)gsm;
  const int adB = lds0 + kSA + (8 * half + (ts >> 2)) * kRowBytes +
                  (((4 * uh + 2 * tb + ((ts & 3) >> 1)) ^ (ts >> 2 << 1)) * 16) + (ts & 1) * 8;

  for (int kt = 0; kt < KT; ++kt) {
    // this wave's part of step kt is there; after the barrier everybody's, and the slot of the
    // step before has been read by all
    mep_wait_vm_lgkm0<(D - 2) * (2 + NU)>();
    mep_bar();
    mep_bf16x8 fa[4];
    mep_s16x4 tw[4][NU][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      fa[ks] = *(const mep_bf16x8*)(gsm + rs + ad[ks]);
#pragma unroll
      for (int i = 0; i < NU; ++i)
#pragma unroll
        for (int u = 0; u < 2; ++u) mep_tr_issue(tw[ks][i][u], adB + rs, i * kSUnitKn + ks * 2048 + u * 512);
    }
    __builtin_amdgcn_sched_barrier(0);
    issue();
    __builtin_amdgcn_sched_barrier(0);
    mep_wait_lgkm0();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        asm volatile("; arrived %0 %1" : "+v"(tw[ks][i][0]), "+v"(tw[ks][i][1]));
        const mep_bf16x8 fb =
            __builtin_bit_cast(mep_bf16x8, __builtin_shufflevector(tw[ks][i][0], tw[ks][i][1], 0, 1, 2, 3, 4, 5, 6, 7));
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks], fb, acc[i], 0, 0, 0);
      }
    rs = rs == (D - 1) * kStageBytes ? 0 : rs + kStageBytes;
  }
  mep_wait_vm_lgkm0<0>();  // the loads past the last step write LDS, too
  mep_bar();               // the next tile may be loaded

  // acc[i][v] is row 32 rb + 8 (v / 4) + 4 half + v % 4, column 32 uh + l31 of unit i
  uint16_t* c = a.C + (size_t)(m + (lane & 1)) * a.N + 64 * unit0 + 32 * uh + (l31 & ~1);
#pragma unroll
  for (int v = 0; v < 16; v += 2)
#pragma unroll
    for (int i = 0; i < NU; ++i)
      store_two_rows(c + (size_t)(8 * (v >> 2) + (v & 3)) * a.N + 64 * i, scale[v >> 2][v & 3] * acc[i][v],
                     scale[v >> 2][(v & 3) + 1] * acc[i][v + 1]);
}

// FOLD: a forward product with mep_folds(K).  (As a choice in the kernel it cost the products of few tiles and steps 0.3 to 0.4 us each.)
template <int MODE, bool KN, bool FOLD = false>
__global__ __launch_bounds__(kSThreads, 2) void gemm_stream_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char gsm[];
  constexpr int kUnits = KN ? kSUnitsKn : kSUnits;
  const int per_block = a.N / (KN ? 64 : MODE == kModeSwiglu ? 16 : 32);
  // several ranks (at most 64, one a lane; input gradients only): their blocks are counted through
  const bool ranks = KN && a.G != a.Gr;
  auto rank_blocks = [&]() {
    const int r = (int)(threadIdx.x & 63);
    return r * a.Gr < a.G ? a.cu[r * a.Gr + a.Gr - 1] / kBM : 0;
  };
  int all = a.cu[a.G - 1] / kBM;
  if (ranks) all = __builtin_amdgcn_readlane(mep_wave_incl_scan(rank_blocks()), 63);
  const int blocks = min(a.mtiles, all);
  // `per` tiles of a block: as many as make the tiles of all blocks whole rounds of the CUs
  const int least = (per_block + kUnits - 1) / kUnits;
  const int width = 8 * a.width;
  const int rounds = (blocks * least + width - 1) / width;
  const int per = min(per_block, rounds * width / max(blocks, 1));
  // neighbours in the list on one XCD: a block's rows, and the weights of a group of two blocks.
  // The tiles of a share alternate between kSParts workgroups: where a kernel beside holds some
  // of the CUs, the second half of what could not start there goes to whoever is done first (FFN
  // forward of 64 tokens at 18 blocks beside 32 held CUs: 463 -> 367 us; alone 233 either way).
  const int q = blockIdx.x >> 3;
  const int p = (int)(blockIdx.x & 7) * a.width + q % a.width;
  const int total = blocks * per;
  const int end = (int)((int64_t)total * (p + 1) / width);
  for (int t = (int)((int64_t)total * p / width) + q / a.width; t < end; t += kSParts) {
    const int mt = t / per, tl = t - mt * per;
    const int unit0 = tl * per_block / per;
    const int n = (tl + 1) * per_block / per - unit0;
    // its rank, and the block among that rank's
    int rank = 0, mb = mt;
    if (ranks) {
      const int n_r = rank_blocks(), incl = mep_wave_incl_scan(n_r);
      rank = __ffsll((unsigned long long)__ballot(incl > mt)) - 1;
      if (rank < 0) break;  // cannot happen: the block lies below the sum
      mb -= __builtin_amdgcn_readlane(incl - n_r, rank);
    }
    // the group of this block: the first of the rank whose padded end lies beyond it
    const int* cu = a.cu + rank * a.Gr;
    int g = -1;
    for (int c = 0; c < a.Gr && g < 0; c += 64) {
      const int gi = c + (int)(threadIdx.x & 63);
      const uint64_t mask = __ballot(gi < a.Gr && cu[gi] > mb * kBM);
      if (mask) g = c + __ffsll((unsigned long long)mask) - 1;
    }
    g = __builtin_amdgcn_readfirstlane(g);
    if (g < 0) break;  // cannot happen: the block lies below the last end
    g += rank * a.Gr;
    const int m0 = rank * a.rank_rows + mb * kBM;
    if constexpr (KN) {
      switch (n) {
        case 1: stream_tile_kn<MODE, 1>(a, gsm, m0, g, unit0); break;
        case 2: stream_tile_kn<MODE, 2>(a, gsm, m0, g, unit0); break;
        case 3: stream_tile_kn<MODE, 3>(a, gsm, m0, g, unit0); break;
        default: stream_tile_kn<MODE, 4>(a, gsm, m0, g, unit0); break;
      }
    } else {
      switch (n) {
        case 1: stream_tile<MODE, 1, FOLD>(a, gsm, m0, g, unit0); break;
        case 2: stream_tile<MODE, 2, FOLD>(a, gsm, m0, g, unit0); break;
        case 3: stream_tile<MODE, 3, FOLD>(a, gsm, m0, g, unit0); break;
        case 4: stream_tile<MODE, 4, FOLD>(a, gsm, m0, g, unit0); break;
        case 5: stream_tile<MODE, 5, FOLD>(a, gsm, m0, g, unit0); break;
        case 6: stream_tile<MODE, 6, FOLD>(a, gsm, m0, g, unit0); break;
        case 7: stream_tile<MODE, 7, FOLD>(a, gsm, m0, g, unit0); break;
        case 8: stream_tile<MODE, 8, FOLD>(a, gsm, m0, g, unit0); break;
        default: stream_tile<MODE, 9, FOLD>(a, gsm, m0, g, unit0); break;
      }
    }
  }
  if (a.zero_tail) zero_tail_rows(a, blockIdx.x, gridDim.x, kSThreads);
}

// ---------------------------------------------------------------------------
// [batch, rows, cols] -> [batch, cols, rows] of 2-byte elements through a
// 64 x 64 LDS tile (rows and cols multiples of 64): 128-byte reads and writes.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void transpose16_kernel(const uint16_t* __restrict__ src,
                                                          uint16_t* __restrict__ dst, int rows, int cols) {
  __shared__ uint16_t tile[64][66];
  const size_t plane = (size_t)rows * cols;
  const uint16_t* s = src + (size_t)blockIdx.z * plane;
  uint16_t* d = dst + (size_t)blockIdx.z * plane;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads, two columns each
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = ty + 8 * i;
    const uint32_t v = *(const uint32_t*)(s + (size_t)(r0 + r) * cols + c0 + 2 * tx);
    tile[r][2 * tx] = (uint16_t)v;
    tile[r][2 * tx + 1] = (uint16_t)(v >> 16);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = ty + 8 * i;  // column of the source = row of the destination
    const uint32_t v = (uint32_t)tile[2 * tx][c] | ((uint32_t)tile[2 * tx + 1][c] << 16);
    *(uint32_t*)(d + (size_t)(c0 + c) * rows + r0 + 2 * tx) = v;
  }
}

// ---------------------------------------------------------------------------
// Backward of h = s * silu(g) * u per element, from the gradient dh' of the
// unscaled activation (dh' = dy * Wdown):
//   dgate = s*dh' * u * silu'(g),  dup = s*dh' * silu(g),  hs = s * silu(g) * u,
//   dscale[m] = sum_n dh'[m,n] * silu(g)*u
// One wave per row; rows at or beyond cu_seqlens[G-1] come out as zeros.
// ---------------------------------------------------------------------------
struct SwigluBwdArgs {
  const uint16_t* dh; const uint16_t* gate; const uint16_t* up; const float* scale; const int* cu;
  uint16_t* dgate; uint16_t* dup; uint16_t* hs; float* dscale;
  int M, N, G, rank_rows;  // G groups and rank_rows rows per rank
};

__global__ __launch_bounds__(256) void swiglu_bwd_kernel(SwigluBwdArgs a) {
  const int lane = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= a.M) return;
  const int rank = m / a.rank_rows;
  const bool live = m - rank * a.rank_rows < a.cu[(rank + 1) * a.G - 1];
  const float s = a.scale ? a.scale[m] : 1.0f;
  const size_t row = (size_t)m * a.N;
  float dot = 0.0f;
  for (int n = lane * 8; n < a.N; n += 512) {
    uint4 od = make_uint4(0, 0, 0, 0), og = od, oh = od;
    if (live) {
      const uint4 vd = *(const uint4*)(a.dh + row + n);
      const uint4 vg = *(const uint4*)(a.gate + row + n);
      const uint4 vu = *(const uint4*)(a.up + row + n);
      const uint32_t wd[4] = {vd.x, vd.y, vd.z, vd.w}, wg[4] = {vg.x, vg.y, vg.z, vg.w},
                     wu[4] = {vu.x, vu.y, vu.z, vu.w};
      uint32_t rg[4], ru[4], rh[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float fg[2], fu[2], fh[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float d = e ? mep_bf16_hi(wd[q]) : mep_bf16_lo(wd[q]);
          const float g = e ? mep_bf16_hi(wg[q]) : mep_bf16_lo(wg[q]);
          const float u = e ? mep_bf16_hi(wu[q]) : mep_bf16_lo(wu[q]);
          const float sig = 1.0f / (1.0f + __expf(-g));
          const float act = g * sig;               // silu(g)
          dot += d * act * u;
          const float dhs = s * d;                 // gradient of the scaled activation
          fg[e] = dhs * u * (sig + act * (1.0f - sig));
          fu[e] = dhs * act;
          fh[e] = s * act * u;
        }
        rg[q] = mep_pack_bf16(fg[0], fg[1]);
        ru[q] = mep_pack_bf16(fu[0], fu[1]);
        rh[q] = mep_pack_bf16(fh[0], fh[1]);
      }
      od = make_uint4(rg[0], rg[1], rg[2], rg[3]);
      og = make_uint4(ru[0], ru[1], ru[2], ru[3]);
      oh = make_uint4(rh[0], rh[1], rh[2], rh[3]);
    }
    *(uint4*)(a.dgate + row + n) = od;
    *(uint4*)(a.dup + row + n) = og;
    *(uint4*)(a.hs + row + n) = oh;
  }
  if (a.dscale) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) dot += __shfl_xor(dot, d);
    if (lane == 0) a.dscale[m] = dot;
  }
}

// The grid of a kernel whose workgroups take a CU each, for at most `tiles` tiles per XCD of about
// `steps` K steps: one workgroup per CU at one time (fewer where there are fewer tiles), each for
// kPSteps steps.
unsigned pp_split(GemmArgs& a, int64_t tiles, int64_t steps) {
  const int cus = mep_device_cu_count();
  const int64_t width = std::min<int64_t>(tiles, std::max(cus > 0 ? cus / 8 : 32, 1));
  const int64_t rounds = (tiles + width - 1) / width;
  steps = std::max<int64_t>(steps, 1);
  a.width = (int)width;
  a.rounds = (int)std::min(rounds, std::max<int64_t>((kPSteps + steps / 2) / steps, 1));
  return 8 * (unsigned)(width * ((rounds + a.rounds - 1) / a.rounds));
}

// about how many 256-row tiles the groups have: rows / 128 blocks are filled, about half of the
// groups (the local experts) and a slot or two have rows
int64_t row_tiles_256(const GemmArgs& a) {
  const int64_t rows = std::max((int64_t)a.M - (int64_t)(kBM - 1) * a.G, (int64_t)0);
  const int64_t blocks = std::max<int64_t>(a.G / 2 + 1, rows / kBM + a.G / 4);
  return std::max<int64_t>(a.G / 2 + 1, blocks / 2 + a.G / 8);
}

template <int MODE, bool BKN>
int gemm_256_launch(GemmArgs a, hipStream_t st) {
  // the most row tiles the groups can need: every group has an odd number of 128-row blocks
  const int64_t total = ((int64_t)a.M / kBM + a.G + 1) / 2 * a.ntiles;
  MEP_REQUIRE(total > 0 && total < (1 << 30), MEP_ERR_UNSUPPORTED);
  // lane offsets inside a tile are 32 bits
  MEP_REQUIRE((int64_t)kPT * 2 * (a.K > a.N ? a.K : a.N) < ((int64_t)1 << 31), MEP_ERR_UNSUPPORTED);
  const int irc = mep_ensure_init();  // the LDS opt-in of this kernel, once per device
  if (irc != MEP_OK) return irc;
  const unsigned grid = pp_split(a, (total + 7) / 8, (int64_t)a.K / kBK * (MODE == kModeDual ? 2 : 1));
  // Where at most a quarter of the CUs get a tile, the time is that of one tile, whose steps wait for
  // loads that come from HBM: two waves on a SIMD hide more of that than one.  us, gemm_pp_kernel /
  // gemm_wide_kernel, 64 tiles of 1024 columns: dy * down K = 2048 40.7 / 43.0, K = 7168 117 / 125;
  // down 40.2 / 40.3, 119 / 120; both pairs 74.2 / 74.1, 247 / 241; at 128 tiles 131 / 132, 131 / 125 and
  // 271 / 248, at 256 184 / 179, 185 / 174 and 369 / 343.  SwiGLU is faster on the wide kernel down to 32
  // tiles (48.9 / 41.7, 119 / 116).
  if constexpr (MODE != kModeSwiglu) {
    if (4 * row_tiles_256(a) * a.ntiles <= std::max(mep_device_cu_count(), 8)) {
      if (MODE == kModeScale && a.scale)
        hipLaunchKernelGGL((gemm_pp_kernel<MODE, false, BKN, MODE == kModeScale>), dim3(grid), dim3(kPThreads), kPLds, st, a,
                           WgradMap{});
      else
        hipLaunchKernelGGL((gemm_pp_kernel<MODE, false, BKN>), dim3(grid), dim3(kPThreads), kPLds, st, a, WgradMap{});
      return mep_launch_status();
    }
  }
  return mep_launch_gemm_wide(MODE, BKN, a, grid, st);
}

// 144 KB of dynamic LDS: opted in by mep_init_gemm_kernels
template <int MODE>
int gemm_launch(const GemmArgs& a, int64_t total, hipStream_t st) {
  MEP_REQUIRE(total > 0 && total < (1 << 30), MEP_ERR_UNSUPPORTED);
  const int per_xcd = (int)((total + 7) / 8) + (a.zero_tail ? 1 : 0);
  const size_t lds = (size_t)kStages * kStage;
  const int irc = mep_ensure_init();
  if (irc != MEP_OK) return irc;
  hipLaunchKernelGGL((grouped_gemm_nt_kernel<MODE>), dim3(per_xcd * 8), dim3(kGemmThreads), lds, st, a);
  return mep_launch_status();
}

template <int MODE, bool KN>
int gemm_stream_launch(GemmArgs a, hipStream_t st) {
  const int64_t units = (int64_t)a.mtiles * (a.N / (KN ? 64 : MODE == kModeSwiglu ? 16 : 32));
  MEP_REQUIRE(units > 0 && units < ((int64_t)1 << 30), MEP_ERR_UNSUPPORTED);
  // offsets inside a tile are 32 bits
  MEP_REQUIRE((int64_t)(KN ? 8 : 32 * kSUnits) * 2 * std::max(2 * a.K, KN ? a.N : 0) < ((int64_t)1 << 32), MEP_ERR_UNSUPPORTED);
  const int irc = mep_ensure_init();
  if (irc != MEP_OK) return irc;
  const int cus = mep_device_cu_count();
  a.width = (int)std::min<int64_t>((units + 7) / 8, std::max(cus > 0 ? cus / 8 : 32, 1));
  const dim3 grid(8 * a.width * kSParts), threads(kSThreads);
  if constexpr (!KN) {
    if (mep_folds(a.K)) {
      hipLaunchKernelGGL((gemm_stream_kernel<MODE, KN, true>), grid, threads, kSLds, st, a);
      return mep_launch_status();
    }
  }
  hipLaunchKernelGGL((gemm_stream_kernel<MODE, KN>), grid, threads, kSLds, st, a);
  return mep_launch_status();
}

// weight gradients on 256 x 256 tiles (M, N multiples of 256, a.G even)
template <bool TN>
int wgrad_pp_launch(GemmArgs a, WgradMap map, hipStream_t st) {
  const int longer = map.rows * kPT;
  MEP_REQUIRE((int64_t)map.rows * map.other < (1 << 24), MEP_ERR_UNSUPPORTED);
  map.tiles = map.rows * map.other;
  map.bands = std::max((map.other + 2) / 4, 1);
  const int64_t per_xcd = ((int64_t)map.n * map.tiles * a.G + 7) / 8;
  MEP_REQUIRE(per_xcd < (1 << 27), MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE((int64_t)kPT * 2 * (TN ? longer : a.ld) < ((int64_t)1 << 31), MEP_ERR_UNSUPPORTED);
  const int irc = mep_ensure_init();
  if (irc != MEP_OK) return irc;
  // About half of the groups have rows, the local experts and a slot or two; the tiles of the others are skipped or
  // are the time of a few K steps.  Sets of workgroups for some kPSteps steps each, and enough to list all tiles.
  const int cus = mep_device_cu_count();
  a.width = (int)std::min<int64_t>(per_xcd, std::max(cus > 0 ? cus / 8 : 32, 1));
  const int64_t rounds = (per_xcd + a.width - 1) / a.width, per_group = (a.rank_rows ? a.rank_rows : a.ld) / kBK / a.Gr;
  const int64_t steps = rounds * std::max<int64_t>(per_group + (a.skip_from < a.Gr ? 0 : 3), 1);
  const int64_t sets = std::min(rounds, std::max((steps + kPSteps / 2) / kPSteps, rounds / (kListed * 3 / 4 - 4) + 1));
  a.rounds = rounds == 1 || a.G > kTabled ? (int)((rounds + sets - 1) / sets) : 0;  // WgradTiles
  hipLaunchKernelGGL((gemm_pp_kernel<kModeWgrad, TN, TN>), dim3(8 * (unsigned)(a.width * sets)), dim3(kPThreads), kPLds, st, a, map);
  return mep_launch_status();
}

int check_nt_shapes(const void* A, const void* B, const int32_t* cu, const void* C, int M, int N, int K,
                    int G, int cols_per_tile) {
  MEP_REQUIRE(A && B && cu && C, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(M > 0 && N > 0 && K > 0 && G > 0, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(M % kBM == 0 && K % kBK == 0 && N % cols_per_tile == 0, MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE((int64_t)M * (N > K ? N : K) < ((int64_t)1 << 40), MEP_ERR_UNSUPPORTED);
  return MEP_OK;
}

GemmArgs nt_args(const void* A, const void* B, const void* B2, const int32_t* cu, void* C, const float* scale,
                 int M, int N, int K, int G, int cols_per_tile) {
  GemmArgs a{};
  a.A = (const uint16_t*)A; a.B = (const uint16_t*)B; a.B2 = (const uint16_t*)B2;
  a.cu = cu; a.C = (uint16_t*)C; a.scale = scale;
  a.M = M; a.N = N; a.K = K; a.G = G;
  a.mtiles = M / kBM;
  a.ntiles = N / cols_per_tile;
  a.ld = K;
  a.Gr = G;
  a.rank_rows = M;
  return a;
}

// the arguments of one rank's product made those of `nranks` ranks' whose operands lie behind each other
bool for_ranks(GemmArgs& a, int nranks) {
  if (nranks < 1 || (int64_t)a.M * nranks > INT32_MAX || (int64_t)a.G * nranks > INT32_MAX) return false;
  a.M *= nranks;
  a.G *= nranks;
  a.mtiles *= nranks;
  return true;
}

// Which kernel.  The rows of the groups are only known on the device; M less the padding that G
// groups can have at token_padding = 128 is about what the rows fill.
// mep_set_gemm_row_tile(128 or 256) forces one side (tests run both on small shapes).
std::atomic<int> g_forced_row_tile{0};

bool use_256_tiles(const GemmArgs& a, bool forward, bool kn) {
  const bool ranks = a.G != a.Gr;
  if (ranks && (!kn || a.G / a.Gr > 64)) return true;  // the streaming kernel has a lane for each
  const int forced = g_forced_row_tile.load(std::memory_order_relaxed);
  if (forced) return forced == 256;
  const int64_t rows = std::max((int64_t)a.M - (int64_t)(kBM - 1) * a.G, (int64_t)0);
  // both pairs with weights along K: 256-row tiles unless half of their matrix work would be padding
  if (!forward && !kn) return 2 * rows >= (int64_t)kBM * a.G;
  const int64_t cus = std::max(mep_device_cu_count(), 8);
  const int64_t blocks = std::max<int64_t>(a.G / 2 + 1, rows / kBM + a.G / 4);
  const int64_t tiles = row_tiles_256(a) * a.ntiles, rounds = (tiles + cus - 1) / cus;
  // Several ranks' input gradients: with less than a block a group most 256-row tiles are half empty.  us,
  // backward pass (weight gradients included), streaming / 256 x 256: 8 ranks, 128 groups of 2048 x 1024
  // with 71 blocks 586 / 646, 99 697 / 723, 165 1003 / 916; 16 ranks, 384 of 768 x 768 with 205 617 / 641, 512
  // of 1024 x 512 with 275 724 / 749; 4 ranks, 32 of 512 x 256 with 20 41 / 51; even at 8 ranks, 64 of
  // 1024 x 512 with 41 and 43 126 / 123, 129 / 131.  By the kernels' times, 373 sizes with less than a block
  // a group are 0.7 % off the faster kernel for each product, on 256 x 256 tiles 12 %.  Forward passes,
  // which stay: 246 / 252, 298 / 278, 535 / 358, 257 / 230, 311 / 274, 21 / 24, 52 / 38.
  // Neither bound is where the kernels cross: larger experts and more blocks stay with the 256 x 256 tiles,
  // which are the faster ones for many blocks (4096 x 1024, 128 groups with 164, products 200 and 392 against
  // 254 and 625) and lose where tiles are few (8 groups of 512 x 256 with 12, 17 and 18 against 9 and 8).
  if (ranks) return blocks >= a.G || (int64_t)a.N * a.K > 2048 * 1024;
  if (kn) {
    // Input gradients: the time of either kernel in 10 ns, fitted to 172 products of 4 to 96 blocks of 8 to
    // 96 groups, 256 .. 5632 by 256 .. 5632 (off by 9 and 12 %).  A round of streaming tiles of n units costs
    // 6 + n us and 0.24 + 0.22 n a K step, one of 256 x 256 tiles 6 us and 0.9 to 1.5 a step.  us,
    // streaming / 256 x 256 tiles, dy * down and both pairs: 4 blocks of K = 5632, 768 columns 44 / 76,
    // 82 / 162; 12 of 1024 x 1024 13 / 20, 21 / 36; 17 of 2048 x 4096 68 / 85, 117 / 159; 24 of 2048 x 4096
    // in 13 groups 88 / 56, 155 / 104; 96 of 1024 x 1024 52 / 34, 80 / 61.
    const int64_t steps = (int64_t)a.K / kBK * (a.A2 ? 2 : 1);
    const int64_t units = a.N / 64, least = (units + kSUnitsKn - 1) / kSUnitsKn;
    const int64_t turns = (blocks * least + cus - 1) / cus, per = std::min(units, turns * cus / blocks);
    const int64_t n = (units + per - 1) / per;
    return 200 + 600 * rounds + steps * (90 * rounds + 64 * std::min(tiles, cus) / cus) <
           turns * (600 + 100 * n + steps * (24 + 22 * n));
  }
  // Forward products: what a K step costs either kernel.  The local experts (half of the groups)
  // and a slot or two have rows, the last block of each about half filled.  A round of 256 x 256
  // tiles takes 1.57 us a step whether it is full or not; the streaming kernel 0.21 us for each
  // unit of 128 x 32 that a CU has.  Measured (FFN forward, us, streaming / 256 x 256): experts of
  // 4096 x 2048, E = 128, K = 8: 64 tokens 183 / 289, 256 245 .. 277 / 301; 512 404 / 302;
  // 7168 x 2048, E = 256: 256 tokens 597 / 738, 512 800 / 765; 1024 x 512, E = 64: 512 tokens
  // 44 / 51, 1024 76 / 53; 512 x 256, E = 16, K = 4, 2048 tokens: 34 / 40.
  return 1570 * rounds * cus < 210 * blocks * 8 * a.ntiles;  // a tile is eight units wide
}

// C = rows x weights for the modes that tile the rows; BKN: weights as [K, N]
template <int MODE, bool BKN>
int row_tiled(const GemmArgs& a, hipStream_t st) {
  constexpr bool forward = !BKN && (MODE == kModeScale || MODE == kModeSwiglu);
  if (use_256_tiles(a, forward, BKN)) return gemm_256_launch<MODE, BKN>(a, st);
  if constexpr (forward || BKN) return gemm_stream_launch<MODE, BKN>(a, st);
  else return gemm_launch<MODE>(a, (int64_t)a.mtiles * a.ntiles, st);
}

int gemm_nt_forward(const void* A, const void* B, const void* B_up, const int32_t* cu, int G, void* C,
                    void* C_gate, void* C_up, const float* row_scale, int M, int N, int K, int swiglu,
                    bool zero_tail, void* stream, int nranks = 1) {
  const int cols = swiglu ? kBN / 2 : kBN;
  const int rc = check_nt_shapes(A, B, cu, C, M, N, K, G, cols);
  if (rc != MEP_OK) return rc;
  MEP_REQUIRE(!swiglu || (B_up && !row_scale), MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(swiglu || (!C_gate && !C_up), MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(((uintptr_t)A % 16 == 0) && ((uintptr_t)B % 16 == 0) && ((uintptr_t)B_up % 16 == 0) &&
                  ((uintptr_t)C % 2 == 0) && ((uintptr_t)C_gate % 2 == 0) && ((uintptr_t)C_up % 2 == 0),
              MEP_ERR_ALIGNMENT);
  GemmArgs a = nt_args(A, B, B_up, cu, C, row_scale, M, N, K, G, cols);
  a.Cg = (uint16_t*)C_gate;
  a.Cu = (uint16_t*)C_up;
  a.zero_tail = zero_tail;
  if (!for_ranks(a, nranks)) return MEP_ERR_UNSUPPORTED;
  return swiglu ? row_tiled<kModeSwiglu, false>(a, (hipStream_t)stream)
                : row_tiled<kModeScale, false>(a, (hipStream_t)stream);
}

// input gradients: weights as [K, N], one or two pairs
int gemm_nn(const void* A1, const void* B1, const void* A2, const void* B2, const int32_t* cu, int G, void* C,
            const float* row_scale, int M, int N, int K, bool zero_tail, void* stream, int nranks = 1) {
  const int rc = check_nt_shapes(A1, B1, cu, C, M, N, K, G, kBN);
  if (rc != MEP_OK) return rc;
  MEP_REQUIRE(2 * (int64_t)K < ((int64_t)1 << 30), MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE(((uintptr_t)A1 % 16 == 0) && ((uintptr_t)B1 % 16 == 0) && ((uintptr_t)A2 % 16 == 0) &&
                  ((uintptr_t)B2 % 16 == 0) && ((uintptr_t)C % 2 == 0), MEP_ERR_ALIGNMENT);
  GemmArgs a = nt_args(A1, B1, B2, cu, C, row_scale, M, N, K, G, kBN);
  a.A2 = (const uint16_t*)A2;
  a.zero_tail = zero_tail;
  if (!for_ranks(a, nranks)) return MEP_ERR_UNSUPPORTED;
  return A2 ? row_tiled<kModeDual, true>(a, (hipStream_t)stream) : row_tiled<kModeScale, true>(a, (hipStream_t)stream);
}

// Weight gradients from the activations as they are, in one launch: n products of X1 [rows, M] and
// X2 [rows, N], whose outputs are M x N or N x M; a rank's groups from `split` on go to C2.  As three
// launches each of them has a start and a last round of its own: us, 48 experts of 512 x 512 with 465
// rows each 142 -> 114, 8 of 4864 x 1536 with 1685 rows 771 -> 746, 64 of 2048 x 1024 with 512 rows 761 -> 724.
int wgrad_tn(int n, const void* const* X1, const void* const* X2, const int32_t* cu, int G, float* const* C,
             float* const* C2, int split, const int* M, const int* N, int64_t rows, int skip_empty_from, void* stream,
             int nranks = 1) {
  MEP_REQUIRE(cu && G > 0 && rows > 0 && skip_empty_from >= 0, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(G % 2 == 0 && rows % kBM == 0 && rows * nranks <= INT32_MAX, MEP_ERR_UNSUPPORTED);
  WgradMap map{};
  map.n = n;
  map.rows = std::max(M[0], N[0]) / kPT;
  map.other = std::min(M[0], N[0]) / kPT;
  for (int i = 0; i < n; ++i) {
    MEP_REQUIRE(X1[i] && X2[i] && C[i] && C2[i] && M[i] > 0 && N[i] > 0, MEP_ERR_INVALID_ARG);
    MEP_REQUIRE(M[i] % kPT == 0 && N[i] % kPT == 0, MEP_ERR_UNSUPPORTED);
    MEP_REQUIRE((int64_t)(M[i] > N[i] ? M[i] : N[i]) * rows < ((int64_t)1 << 40), MEP_ERR_UNSUPPORTED);
    MEP_REQUIRE(((uintptr_t)X1[i] % 16 == 0) && ((uintptr_t)X2[i] % 16 == 0) && ((uintptr_t)C[i] % 16 == 0) &&
                    ((uintptr_t)C2[i] % 16 == 0), MEP_ERR_ALIGNMENT);
    MEP_REQUIRE(std::max(M[i], N[i]) == std::max(M[0], N[0]) && std::min(M[i], N[i]) == std::min(M[0], N[0]),
                MEP_ERR_INVALID_ARG);
    map.A[i] = (const uint16_t*)X1[i];
    map.B[i] = (const uint16_t*)X2[i];
    map.C[i] = C[i];
    map.C2[i] = C2[i];
    map.tall |= (M[i] >= N[i]) << i;
  }
  GemmArgs a{};
  a.cu = cu; a.split = split;
  a.G = G * nranks;
  a.ld = rows;
  a.Gr = G;
  a.rank_rows = (int)rows;
  a.skip_from = skip_empty_from;
  return wgrad_pp_launch<true>(a, map, (hipStream_t)stream);
}

template <class Kern>
int opt_in_lds(Kern kern, size_t bytes) {
  MEP_RETURN_IF_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)bytes));
  return MEP_OK;
}

}  // namespace

// Every GEMM kernel uses more dynamic LDS than a kernel gets without asking: the opt-ins
// for the current device, made once from mep_init (never from a launch, which may be
// under stream capture).
int mep_init_gemm_kernels() {
  const size_t ring = (size_t)kStages * kStage;
  int rc = MEP_OK;
#define MEP_OPT(k, b) if (rc == MEP_OK) rc = opt_in_lds(k, b)
  MEP_OPT((gemm_stream_kernel<kModeScale, false>), kSLds);
  MEP_OPT((gemm_stream_kernel<kModeSwiglu, false>), kSLds);
  MEP_OPT((gemm_stream_kernel<kModeScale, false, true>), kSLds);
  MEP_OPT((gemm_stream_kernel<kModeSwiglu, false, true>), kSLds);
  MEP_OPT((gemm_stream_kernel<kModeScale, true>), kSLds);
  MEP_OPT((gemm_stream_kernel<kModeDual, true>), kSLds);
  MEP_OPT((grouped_gemm_nt_kernel<kModeDual>), ring);
  MEP_OPT((grouped_gemm_nt_kernel<kModeWgrad>), ring);
  MEP_OPT((gemm_pp_kernel<kModeScale, false, false>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeScale, false, false, true>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeDual, false, false>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeScale, false, true>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeScale, false, true, true>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeDual, false, true>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeWgrad, false, false>), kPLds);
  MEP_OPT((gemm_pp_kernel<kModeWgrad, true, true>), kPLds);
#undef MEP_OPT
  return rc == MEP_OK ? mep_init_gemm_wide_kernels() : rc;
}

extern "C" int mep_set_gemm_row_tile(int rows) {
  MEP_REQUIRE(rows == 0 || rows == 128 || rows == 256, MEP_ERR_INVALID_ARG);
  g_forced_row_tile.store(rows, std::memory_order_relaxed);
  return MEP_OK;
}

extern "C" int mep_grouped_gemm_nt(const void* A, const void* B, const void* B_up,
                                   const int32_t* cu_seqlens, int G, void* C,
                                   const float* row_scale, int M, int N, int K, int swiglu,
                                   void* stream) {
  return gemm_nt_forward(A, B, B_up, cu_seqlens, G, C, nullptr, nullptr, row_scale, M, N, K, swiglu, false, stream);
}

extern "C" int mep_grouped_swiglu_nt(const void* A, const void* B_gate, const void* B_up,
                                     const int32_t* cu_seqlens, int G, void* C_act, void* C_gate,
                                     void* C_up, int M, int N, int K, void* stream) {
  return gemm_nt_forward(A, B_gate, B_up, cu_seqlens, G, C_act, C_gate, C_up, nullptr, M, N, K, 1, false, stream);
}

extern "C" int mep_grouped_gemm_dual_nt(const void* A1, const void* B1, const void* A2, const void* B2,
                                        const int32_t* cu_seqlens, int G, void* C, int M, int N, int K,
                                        void* stream) {
  const int rc = check_nt_shapes(A1, B1, cu_seqlens, C, M, N, K, G, kBN);
  if (rc != MEP_OK) return rc;
  MEP_REQUIRE(A2 && B2, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(2 * (int64_t)K < ((int64_t)1 << 30), MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE(((uintptr_t)A1 % 16 == 0) && ((uintptr_t)B1 % 16 == 0) && ((uintptr_t)A2 % 16 == 0) &&
                  ((uintptr_t)B2 % 16 == 0) && ((uintptr_t)C % 2 == 0), MEP_ERR_ALIGNMENT);
  GemmArgs a = nt_args(A1, B1, B2, cu_seqlens, C, nullptr, M, N, K, G, kBN);
  a.A2 = (const uint16_t*)A2;
  return row_tiled<kModeDual, false>(a, (hipStream_t)stream);
}

extern "C" int mep_grouped_gemm_nn(const void* A, const void* B, const int32_t* cu_seqlens, int G, void* C,
                                   const float* row_scale, int M, int N, int K, void* stream) {
  return gemm_nn(A, B, nullptr, nullptr, cu_seqlens, G, C, row_scale, M, N, K, false, stream);
}

extern "C" int mep_grouped_gemm_dual_nn(const void* A1, const void* B1, const void* A2, const void* B2,
                                        const int32_t* cu_seqlens, int G, void* C, int M, int N, int K,
                                        void* stream) {
  const int rc = check_nt_shapes(A1, B1, cu_seqlens, C, M, N, K, G, kBN);
  if (rc != MEP_OK) return rc;
  MEP_REQUIRE(A2 && B2, MEP_ERR_INVALID_ARG);
  return gemm_nn(A1, B1, A2, B2, cu_seqlens, G, C, nullptr, M, N, K, false, stream);
}

extern "C" int mep_grouped_gemm_wgrad(const void* At, const void* Bt, const int32_t* cu_seqlens, int G,
                                      float* C, int Ma, int Nb, int64_t ld, int skip_empty_from, void* stream) {
  MEP_REQUIRE(At && Bt && cu_seqlens && C, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(Ma > 0 && Nb > 0 && G > 0 && ld > 0, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(Ma % kBM == 0 && Nb % kBN == 0 && ld % kBM == 0, MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE((int64_t)(Ma > Nb ? Ma : Nb) * ld < ((int64_t)1 << 40), MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE(((uintptr_t)At % 16 == 0) && ((uintptr_t)Bt % 16 == 0) && ((uintptr_t)C % 4 == 0),
              MEP_ERR_ALIGNMENT);
  GemmArgs a{};
  a.A = (const uint16_t*)At; a.B = (const uint16_t*)Bt; a.cu = cu_seqlens; a.Cf = C;
  a.M = Ma; a.N = Nb; a.K = 0; a.G = G;
  a.ld = ld;
  MEP_REQUIRE(skip_empty_from >= 0, MEP_ERR_INVALID_ARG);
  a.skip_from = skip_empty_from;
  a.split = G;
  a.Gr = G;
  // an expert's shapes: 256 x 256 tiles (whose lane offsets are 32 bits).  Groups are experts and as many
  // slots everywhere here, so G is even; the list of tiles would take an odd number, which was not compared.
  if (Ma % kPT == 0 && Nb % kPT == 0 && G % 2 == 0 && (uintptr_t)C % 16 == 0 && ld < ((int64_t)1 << 22)) {
    WgradMap map{};
    map.n = 1;
    map.A[0] = a.A; map.B[0] = a.B; map.C[0] = map.C2[0] = C;
    map.rows = std::max(Ma, Nb) / kPT; map.other = std::min(Ma, Nb) / kPT; map.tall = Ma >= Nb;
    return wgrad_pp_launch<false>(a, map, (hipStream_t)stream);
  }
  a.mtiles = Ma / kBM;
  a.ntiles = Nb / kBN;
  return gemm_launch<kModeWgrad>(a, (int64_t)a.mtiles * a.ntiles * G, (hipStream_t)stream);
}

extern "C" int mep_grouped_gemm_wgrad_tn(const void* X1, const void* X2, const int32_t* cu_seqlens, int G,
                                         float* C, int Ma, int Nb, int64_t rows, int skip_empty_from,
                                         void* stream) {
  return wgrad_tn(1, &X1, &X2, cu_seqlens, G, &C, &C, G, &Ma, &Nb, rows, skip_empty_from, stream);
}

namespace {
int swiglu_bwd_launch(const void* dh, const void* gate_pre, const void* up_pre, const float* row_scale,
                      const int32_t* cu_seqlens, int G, void* dgate, void* dup, void* hs, float* dscale, int M, int N,
                      int rank_rows, void* stream) {
  MEP_REQUIRE(dh && gate_pre && up_pre && cu_seqlens && dgate && dup && hs, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(M > 0 && N > 0 && G > 0, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(N % 8 == 0, MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE(((uintptr_t)dh % 16 == 0) && ((uintptr_t)gate_pre % 16 == 0) && ((uintptr_t)up_pre % 16 == 0) &&
                  ((uintptr_t)dgate % 16 == 0) && ((uintptr_t)dup % 16 == 0) && ((uintptr_t)hs % 16 == 0),
              MEP_ERR_ALIGNMENT);
  SwigluBwdArgs a;
  a.dh = (const uint16_t*)dh; a.gate = (const uint16_t*)gate_pre; a.up = (const uint16_t*)up_pre;
  a.scale = row_scale; a.cu = cu_seqlens;
  a.dgate = (uint16_t*)dgate; a.dup = (uint16_t*)dup; a.hs = (uint16_t*)hs; a.dscale = dscale;
  a.M = M; a.N = N; a.G = G; a.rank_rows = rank_rows;
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3((M + 3) / 4), dim3(256), 0, (hipStream_t)stream, a);
  return mep_launch_status();
}
}  // namespace

extern "C" int mep_swiglu_bwd(const void* dh, const void* gate_pre, const void* up_pre,
                              const float* row_scale, const int32_t* cu_seqlens, int G, void* dgate,
                              void* dup, void* hs, float* dscale, int M, int N, void* stream) {
  return swiglu_bwd_launch(dh, gate_pre, up_pre, row_scale, cu_seqlens, G, dgate, dup, hs, dscale, M, N, M, stream);
}

extern "C" int mep_ffn_forward(const void* rows, const float* slots, const int32_t* cu_seqlens, int G, const void* gate,
                               const void* up, const void* down, void* act, void* gate_pre, void* up_pre, void* y,
                               int nranks, int M, int H, int Hp, void* stream) {
  const int rc = gemm_nt_forward(rows, gate, up, cu_seqlens, G, act, gate_pre, up_pre, nullptr, M, Hp, H, 1, false, stream, nranks);
  if (rc != MEP_OK) return rc;
  return gemm_nt_forward(act, down, nullptr, cu_seqlens, G, y, nullptr, nullptr, slots, M, H, Hp, 0, true, stream, nranks);
}

extern "C" int mep_ffn_backward(const void* dy, const void* rows, const float* slots, const int32_t* cu_seqlens, int G,
                                const void* gate, const void* up, const void* down, const void* gate_pre,
                                const void* up_pre, void* dh, void* dgate, void* dup, void* hs, float* dslots,
                                void* drows, float* const* wgrads, float* const* wgrads_from_split, int split,
                                int nranks, int M, int H, int Hp, int skip_empty_from, void* stream) {
  MEP_REQUIRE(gate && up && wgrads && wgrads_from_split && drows, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE((slots == nullptr) == (dslots == nullptr), MEP_ERR_INVALID_ARG);
  // gradient of the unscaled activation: dy * down[g], down[g] is [H, H'] = [K, N]
  MEP_REQUIRE(nranks > 0 && (int64_t)M * nranks <= INT32_MAX && (int64_t)G * nranks <= INT32_MAX, MEP_ERR_UNSUPPORTED);
  int rc = gemm_nn(dy, down, nullptr, nullptr, cu_seqlens, G, dh, nullptr, M, Hp, H, false, stream, nranks);
  if (rc == MEP_OK)
    rc = swiglu_bwd_launch(dh, gate_pre, up_pre, slots, cu_seqlens, G, dgate, dup, hs, dslots, M * nranks, Hp, M, stream);
  if (rc == MEP_OK) rc = gemm_nn(dgate, gate, dup, up, cu_seqlens, G, drows, nullptr, M, H, Hp, true, stream, nranks);
  const void* x1[3] = {dgate, dup, dy};
  const void* x2[3] = {rows, rows, hs};
  const int m[3] = {Hp, Hp, H}, n[3] = {H, H, Hp};
  return rc == MEP_OK ? wgrad_tn(3, x1, x2, cu_seqlens, G, wgrads, wgrads_from_split, split, m, n, M, skip_empty_from,
                                 stream, nranks)
                      : rc;
}

extern "C" int mep_transpose_bf16(const void* src, void* dst, int batch, int rows, int cols, void* stream) {
  MEP_REQUIRE(src && dst && src != dst, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(batch > 0 && rows > 0 && cols > 0, MEP_ERR_INVALID_ARG);
  MEP_REQUIRE(rows % 64 == 0 && cols % 64 == 0 && batch <= 65535 && rows / 64 <= 65535, MEP_ERR_UNSUPPORTED);
  MEP_REQUIRE(((uintptr_t)src % 4 == 0) && ((uintptr_t)dst % 4 == 0), MEP_ERR_ALIGNMENT);
  hipLaunchKernelGGL(transpose16_kernel, dim3(cols / 64, rows / 64, batch), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)src, (uint16_t*)dst, rows, cols);
  return mep_launch_status();
}

