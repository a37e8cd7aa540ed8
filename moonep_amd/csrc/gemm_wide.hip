// The products that tile the rows (SwiGLU, down, the input gradients) in whole rounds of the chip:
// 256 x 256 output tiles, K in steps of 64, FOUR waves of 128 x 128, one on every SIMD, one workgroup
// per CU.  The walk over the tiles, and what a workgroup takes of it, are those of gemm_pp_kernel
// (grouped_gemm.hip: eight waves of 128 x 64 in two shifts), which this one replaces there.
//
// What bounds it: the power that the chip has for a flop, then the slots of the one instruction
// stream of a SIMD.  Hence
//  * v_mfma_f32_16x16x32_bf16: in a loop of nothing else, on normal data, the chip does 2.06 PFLOP/s
//    with it and 1.79 with 32x32x16 (2.43 with either on zeroes: the difference is power);
//  * 128 x 128 a wave instead of 128 x 64: 128 KB of LDS reads a K step instead of 192.  In the same
//    loop reads of 1/2 KB per 16 x 16 x 32 take it to 1.77 PFLOP/s, of 1/4 KB to 1.94;
//  * the sums fill the accumulation registers (256 a lane).  They are named in the asm statements
//    alone (mep_acc_*): as values of the program the compiler copies or spills them wherever two
//    paths meet.  The build checks that no other instruction touches them;
//  * a wave has nobody to hide behind: what is issued between two matrix instructions (16 cycles
//    each) is at most an LDS read or a load, one every four or eight of them, and every address and
//    slot of the next step is made in there, too.  In front of the matrix instructions of 16 rows
//    instead, two reads and a load cost 10 %; a branch for every four of them (to skip the rows that
//    a short tile does not have) 9 %, so there are two copies of a step, 256 rows and 128.
// Loads go straight into LDS: the weights' tile (32 KB a step) has three slots, the rows' two.  Four
// loads in a row take their place from one M0 and the offset in the instruction, which counts for both
// addresses (an M0 each: 0.2 % slower).  A K
// step goes in two halves (K 0 .. 31, 32 .. 63); while one half's fragments are multiplied, the other
// half's are read.  When the second half's have arrived, one barrier says that the step's slots are
// free and that the next step's are full.  Waiting for older or for younger loads there made no
// difference; the loads cost what they take to issue (with none 9 % faster, with all of them hits in
// L2 5 %).
//
// The first operand of the matrix instruction is the weights: a lane then holds four neighbouring
// columns of one row, and the fragments 2 c and 2 c + 1 take the weight rows 8 a + b and 8 a + 4 + b
// (a, b = 0 .. 3) of a block of 32, so that they make eight neighbouring columns, one 16-byte store.
// Before they are stored, lanes four rows apart trade these 16 bytes for two blocks of columns, so that an
// instruction stores 128 neighbouring bytes of eight rows instead of 64 of sixteen; and the stores are
// nontemporal.  When all CUs store at one time, as they do after tiles of equal length, 128 KB a CU take
// 9000 cycles as plain stores, 9500 to 11 000 nontemporal in pieces of 64 bytes and 6800 in pieces of
// 128 or 256 (one CU alone: 2500), with the matrix cores idle.  us, before -> now: 36 864 rows in 96
// groups, 2048 x 1024: SwiGLU 297 -> 291, down 161 -> 157, dy * down 154 -> 150, both pairs 287 -> 284;
// 32 768 rows in 32 groups, 2048 x 1024 columns 118 -> 108; 7168 x 2048, which power bounds, 1333 ->
// 1324, 716 -> 714, 670 -> 666, 1347 -> 1342 (with the loads below).  Workgroups that begin a quarter of
// the stores' time apart are no faster.
//
// LDS layouts.  The hardware serves 16-byte reads in groups of the lanes 0-3, 12-15, 20-27 (and
// 4-11, 16-19, 28-31), not of sixteen neighbours.  Rows: 128 bytes each, vector q of row r at
// q ^ (r & 6); weights along K: at q ^ (r & 2) ^ 4 (r / 16 % 2); both free of conflicts in those
// groups.  Weights as [K, columns]: 64 rows of 256 bytes per 128 columns, vector v of row k at
// v ^ 4 (k % 4) ^ 2 (k / 8 % 2), read with transposing reads (half of the banks at a time).
//
// Measured, us, gemm_pp_kernel -> this: 34 816 rows in 32 groups, 7168 x 2048: SwiGLU 1774 -> 1610,
// down 888 -> 822, dy * down 866 -> 839, both pairs 1768 -> 1613; 33 792 rows in 16 groups, 4096 x
// 2048: 955 -> 859, 519 -> 469, 501 -> 477, 987 -> 895; 36 864 rows in 64 groups, 2048 x 1024: 303 ->
// 271, 162 -> 146, 162 -> 154, 300 -> 276.  Counters of the first: matrix cores 73 % of all cycles at
// 1.70 GHz (before 72 % at 1.57).
#include "grouped_gemm.h"

#include <type_traits>
#include <utility>

namespace {

using namespace mep_gemm;

constexpr int kWThreads = 256;
constexpr int kWHalf = 128 * kRowBytes;    // 16 KB: half of one operand's tile of a K step
constexpr int kWStep = 2 * kWHalf;
constexpr int kWSlotsA = 2, kWSlotsB = 3;  // K steps of the rows and of the weights in LDS
constexpr int kWFirstB = kWSlotsA * kWStep;
constexpr int kWLds = (kWSlotsA + kWSlotsB) * kWStep;  // 160 KB

#define MEP_INLINE __attribute__((always_inline))

// ---- the sums: block c of 16 x 16 is a[4 c .. 4 c + 3], and only these statements know
template <int C, bool FIRST>
__device__ __forceinline__ void mep_acc_mul(const mep_bf16x8& w, const mep_bf16x8& r) {  // (+)= weights x rows, 16 x 16 x 32
  if (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, 0" ::"n"(4 * C), "n"(4 * C + 3), "v"(w), "v"(r));
  else asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, a[%0:%1]" ::"n"(4 * C), "n"(4 * C + 3), "v"(w), "v"(r));
}
template <int C>
__device__ __forceinline__ mep_f32x4 mep_acc_get() {
  mep_f32x4 v;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v[0]) : "n"(4 * C));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v[1]) : "n"(4 * C + 1));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v[2]) : "n"(4 * C + 2));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v[3]) : "n"(4 * C + 3));
  return v;
}
// the compiler keeps nothing in them across this
#define MEP_A10(p) "a" #p "0", "a" #p "1", "a" #p "2", "a" #p "3", "a" #p "4", "a" #p "5", "a" #p "6", "a" #p "7", "a" #p "8", "a" #p "9"
__device__ __forceinline__ void mep_acc_taken() {
  asm volatile("" ::: "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", MEP_A10(1), MEP_A10(2), MEP_A10(3), MEP_A10(4),
               MEP_A10(5), MEP_A10(6), MEP_A10(7), MEP_A10(8), MEP_A10(9), MEP_A10(10), MEP_A10(11), MEP_A10(12), MEP_A10(13),
               MEP_A10(14), MEP_A10(15), MEP_A10(16), MEP_A10(17), MEP_A10(18), MEP_A10(19), MEP_A10(20), MEP_A10(21), MEP_A10(22),
               MEP_A10(23), MEP_A10(24), "a250", "a251", "a252", "a253", "a254", "a255");
}
#undef MEP_A10

// The order of a half's 16 x 16 x 32 products: two blocks of rows at a time, the blocks of weights back and
// forth, so that one of the two operands stays from each instruction to the next, the other one in turn.  That is
// power: a loop of nothing else does 2.07 PFLOP/s with it, 2.03 where the weights change every time and the rows
// every eighth (back and forth, too) and 2.01 where both change at each eighth, as the rows' order was here.
constexpr int mep_row_block(int n) { return n >> 4 << 1 | ((n ^ n >> 1) & 1); }
constexpr int mep_weight_block(int n) { return (n >> 4 & 1 ? ~n : n) >> 1 & 7; }

// x and y are two blocks of columns of a lane's row.  Of eight lanes the first four take the last four's x for their y: they then
// have one block of their row and of the row four lanes on, the others the other block of the same two.
typedef uint32_t mep_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void mep_trade(mep_u4& x, mep_u4& y) {
  constexpr int kFromBelow = 0x124, kFromAbove = 0x12c;  // row_ror by four lanes and by twelve
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int was = (int)x[d];
    x[d] = (uint32_t)__builtin_amdgcn_update_dpp(was, (int)y[d], kFromBelow, 0xf, 0xa, false);
    y[d] = (uint32_t)__builtin_amdgcn_update_dpp((int)y[d], was, kFromAbove, 0xf, 0x5, false);
  }
}

// f(0), f(1) .. f(N - 1), the numbers as constants
template <class F, int... I>
__device__ __forceinline__ void mep_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void mep_each(F&& f) {
  mep_each(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

// KN: the weights are given as [K, columns].  SCALED: scale mode with row scales.
template <int MODE, bool KN, bool SCALED>
__global__ __launch_bounds__(kWThreads, 1) void gemm_wide_kernel(GemmArgs a) {
  constexpr bool SWIGLU = MODE == kModeSwiglu, DUAL = MODE == kModeDual, FORWARD = !DUAL && !KN;
  static_assert(!(SWIGLU && KN) && (!SCALED || MODE == kModeScale) && MODE != kModeWgrad, "no such product");
  extern __shared__ __attribute__((aligned(1024))) char gsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lq = lane >> 4;

  // ---- loads: a cursor over (tile, K step).  It moves on once a step; the rows of a step (qA) are
  // asked for half a step after its weights
  const size_t ldA = (size_t)a.K, ldB = KN ? (size_t)a.N : (size_t)a.K;
  PTiles<MODE, true> ld(a);
  PTiles<MODE, true> cp = ld;  // the tiles as they are multiplied
  // A tile's operands as the loads take them; a step moves them along K by an offset.  (As addresses, which move on by 64
  // bits and are made into the loads' four words again between the matrix instructions: 32 768 rows, 7168 x 2048,
  // SwiGLU 1334 -> 1329 us, down 719 -> 716; on zeroes, where power bounds less, 1145 -> 1141, 582 -> 580.)
  __amdgpu_buffer_rsrc_t dA = mep_rsrc((const char*)a.A), dB = dA, dB1 = dA;
  uint32_t kA = 0, qkA = 0, halfA = 0, qhalfA = 0;
  uint32_t step = kRowBytes, both = 2 * kRowBytes;  // to the next step; to the one behind it
  const bool fold = FORWARD && mep_folds(a.K);
  int pieces = 0;       // of a folded tile, behind the one that `left` counts
  const uint32_t stepB = KN ? (uint32_t)(kBK * ldB * 2) : 0;
  const uint32_t halfB = SWIGLU ? 0u : KN ? 256u : (uint32_t)(128 * ldB * 2);
  const char* pB = nullptr;
  int left = 0;         // K steps to the end of the tile, or of its first pair
  bool second = false;  // dual: at the second pair
  auto stand = [&]() MEP_INLINE {  // at the first K step of the tile (of its second pair)
    const size_t offA = (size_t)ld.m0 * ldA;
    const size_t offB = (size_t)ld.g * a.N * a.K + (KN ? (size_t)ld.n0 : (size_t)ld.n0 * ldB);
    dA = mep_rsrc(mep_uniform((const char*)((DUAL && second ? a.A2 : a.A) + offA)));
    pB = mep_uniform((const char*)((DUAL && second ? a.B2 : a.B) + offB));
    if (!KN) dB = mep_rsrc(pB);
    if (SWIGLU) dB1 = mep_rsrc(mep_uniform((const char*)(a.B2 + offB)));
    kA = 0;
    halfA = __builtin_amdgcn_readfirstlane(ld.tall ? (uint32_t)(128 * ldA * 2) : 0u);
    left = __builtin_amdgcn_readfirstlane(fold ? kFold : a.K / kBK);
    if (FORWARD) {
      pieces = __builtin_amdgcn_readfirstlane(fold ? a.K / kBK / kFold - 1 : 0);
      step = fold ? (uint32_t)mep_fold_step(0) : kRowBytes;
      both = fold ? kRowBytes : 2 * kRowBytes;
    }
  };
  // more than one tile a workgroup: the next tile's loads wait behind the stores (one: 20 groups of 1792 x 768, down 18.8 us
  // as plain stores, 20 nontemporal)
  const int rounds = __builtin_amdgcn_readfirstlane((int)(ld.count > ld.nw));
  const int some = __builtin_amdgcn_readfirstlane((int)ld.next());
  if (some) stand();
  auto on = [&]() MEP_INLINE {
    kA += step;
    if (FORWARD) step = both - step;
    if (KN && step) pB += stepB;
  };
  auto turned = [&]() MEP_INLINE {  // the cursor has left its tile, or a piece of it
    if (FORWARD && pieces > 0) {
      --pieces;
      left = kFold;
      kA += kRowBytes - (both - step);
      return;
    }
    if (DUAL && !second) {
      second = true;
      stand();
      return;
    }
    second = false;
    if (__builtin_amdgcn_readfirstlane((int)ld.next())) {
      stand();
    } else {  // the last step is loaded again, for nobody
      kA -= FORWARD ? both - step : step;
      pB -= stepB;
      step = both = 0;
      left = 1 << 30;
    }
  };
  uint32_t vA[4], vB[4];  // a wave brings four pieces of 1 KB of either half of a tile: 8 rows, or 4 rows of K
  {
    const int r = lane >> 3, kv = lane & 7;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = 4 * wave + q;
      // less what the instruction adds (no less than that: K and N are at least 64 and 128)
      vA[q] = (uint32_t)((8 * j + r) * ldA * 2 + (kv ^ (r & 6)) * 16) - q * 1024;
      vB[q] = (KN ? (uint32_t)((4 * j + lq) * ldB * 2 + (l15 ^ (lq << 2) ^ (q >> 1 << 1)) * 16)
                  : (uint32_t)((8 * j + r) * ldB * 2 + (kv ^ (r & 2) ^ (q >> 1 << 2)) * 16)) - q * 1024;
    }
  }
  __amdgpu_buffer_rsrc_t dqA = dA;  // the rows' step, behind the weights'
  auto hold = [&]() MEP_INLINE { dqA = dA; qkA = kA; qhalfA = kA + halfA; };
  // where the next step of each operand is written and read
  char* lds_w = gsm + wave * 4096;
  int wA = 0, wB = kWFirstB, rA = 0, rB = kWFirstB;
  auto turnA = [](int& s) MEP_INLINE { s ^= kWStep; };
  auto turnB = [](int& s) MEP_INLINE { s = s == kWLds - kWStep ? kWFirstB : s + kWStep; };
  auto issueA = [&](auto c) MEP_INLINE {  // 0 .. 7
    constexpr int n = c;
    mep_load_lds16<0, (n & 3) * 1024>(dqA, vA[n & 3], n >> 2 ? qhalfA : qkA, lds_w + wA + (n >> 2) * kWHalf);
  };
  auto issueB = [&](auto c) MEP_INLINE {
    constexpr int n = c;
    if (KN) mep_load_lds16<0, (n & 3) * 1024>(pB, vB[n & 3], n >> 2 ? halfB : 0u, lds_w + wB + (n >> 2) * kWHalf);
    else mep_load_lds16<0, (n & 3) * 1024>(SWIGLU && n >> 2 ? dB1 : dB, vB[n & 3], SWIGLU || !(n >> 2) ? kA : kA + halfB, lds_w + wB + (n >> 2) * kWHalf);
  };

  // ---- fragments: set s holds half s of a K step
  const int wm = wave >> 1, wn = wave & 1;
  int adA[2], adB[4];
#pragma unroll
  for (int s = 0; s < 2; ++s) adA[s] = l15 * kRowBytes + ((4 * s + lq) ^ (l15 & 6)) * 16;
  if (KN) {
    const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) char*)gsm;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      adB[c] = lds0 + wn * kWHalf + (8 * lq + (l15 >> 2)) * 256 +
               ((4 * c + (l15 & 3)) ^ (l15 >> 2 << 2) ^ ((lq & 1) << 1)) * 16;
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      adB[s] = ((SWIGLU ? 64 : 128) * wn + 8 * (l15 >> 2) + (l15 & 3)) * kRowBytes +
               ((4 * s + lq) ^ (l15 & 2) ^ (l15 >> 3 << 2)) * 16;
  }
  mep_bf16x8 fr[2][8], fw[2][8];  // rows, weights
  mep_s16x4 tw[2][8][2];          // transposed reads until they have arrived
  auto readA = [&](int s, int i, int at) MEP_INLINE { fr[s][i] = *(const mep_bf16x8*)(gsm + (adA[s] + at) + i * 16 * kRowBytes); };
  auto readB = [&](int s, int j, int at) MEP_INLINE {
    if (KN) {
#pragma unroll
      for (int u = 0; u < 2; ++u) mep_tr_issue(tw[s][j][u], adB[j >> 1] + at, s * 8192 + u * 1024 + (j & 1) * 8);
    } else {
      // SwiGLU: two blocks of 32 gate rows, then the same up rows
      const int row = SWIGLU ? (j >> 2) * 128 + (j >> 1 & 1) * 32 + (j & 1) * 4 : (j >> 1) * 32 + (j & 1) * 4;
      fw[s][j] = *(const mep_bf16x8*)(gsm + (adB[s] + at) + row * kRowBytes);
    }
  };
  auto got = [&](int s) MEP_INLINE {  // after the wait
    if (!KN) return;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      asm volatile("; arrived %0 %1" : "+v"(tw[s][j][0]), "+v"(tw[s][j][1]));
      fw[s][j] = __builtin_bit_cast(mep_bf16x8, __builtin_shufflevector(tw[s][j][0], tw[s][j][1], 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  // x of a half's 16 reads, weights first
  auto read = [&](int s, int x, int at_rows) MEP_INLINE {
    if (x < 8) readB(s, x, rB);
    else readA(s, x - 8, at_rows);
  };

  // ---- prologue: two K steps, the first half's fragments
  if (some) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      hold();
      mep_each<8>(issueA);
      mep_each<8>(issueB);
      turnA(wA); turnB(wB);
      on();
      if (--left == 0) turned();
    }
    mep_wait_vmcnt<16>();
    mep_bar();
  }
  int have = __builtin_amdgcn_readfirstlane((int)cp.next());
  // the wave's rows in a slot: 128 of 256, or 64 of 128
  auto rows_at = [&]() MEP_INLINE { return __builtin_amdgcn_readfirstlane(wm * (cp.tall ? 128 : 64) * kRowBytes); };
  if (have) {
    const int at = rows_at();
#pragma unroll
    for (int x = 0; x < 16; ++x) read(0, x, at + rA);
  }
  mep_wait_lgkm0();
  got(0);
  while (have) {
    const int m0 = cp.m0, n0 = cp.n0, KT = __builtin_amdgcn_readfirstlane(cp.KT);
    const int tall = __builtin_amdgcn_readfirstlane((int)cp.tall);
    const int at_cur = rows_at();
    have = __builtin_amdgcn_readfirstlane((int)cp.next());
    const int at_next = rows_at();
    // The scales of the wave's rows, one per lane: asked for in front of the tile's loads and there by
    // the epilogue (a load the compiler knows would be waited for there, and with it every load of
    // the next tile).
    float scl0 = 1.0f, scl1 = 1.0f;
    auto scales_ask = [&]() MEP_INLINE {
      if (!SCALED) return;
      const float* sp = a.scale + m0 + (tall ? 128 : 64) * wm + lane;
      asm volatile("global_load_dword %0, %1, off" : "=v"(scl0) : "v"(sp));
      asm volatile("global_load_dword %0, %1, off" : "=v"(scl1) : "v"(sp + (tall ? 64 : 0)));
    };
    auto scales_in = [&]() MEP_INLINE {
      if (!SCALED) return;
      mep_wait_vmcnt<16>();  // a K step's loads came after them
      asm volatile("; arrived %0 %1" : "+v"(scl0), "+v"(scl1));
    };
    int kt = 0;
    auto step = [&](auto frags, auto first) MEP_INLINE {
      constexpr int NM = 8 * decltype(frags)::value;  // matrix instructions of a half
      constexpr int R = NM / 16, L = NM / 8;          // one LDS read, one load every so many
      mep_acc_taken();
      int at_rows = at_cur + rA;
      __builtin_amdgcn_sched_barrier(0);
      mep_each<NM>([&](auto c) MEP_INLINE {
        constexpr int n = c;
        if constexpr (n % R == 0) { read(1, n / R, at_rows); __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n % L == L / 2 + 1) { issueB(std::integral_constant<int, n / L>{}); __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n == NM - 2) {
          turnA(rA); turnB(rB);
          at_rows = (kt + 1 < KT ? at_cur : at_next) + rA;
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (n == NM - 1) { turnB(wB); __builtin_amdgcn_sched_barrier(0); }
        constexpr int i = mep_row_block(n), j = mep_weight_block(n);
        mep_acc_mul<8 * i + j, decltype(first)::value>(fw[0][j], fr[0][i]);
        __builtin_amdgcn_sched_barrier(0);
      });
      // the next step is there but for the weights of the one behind it, which were asked for last;
      // this step's slots have been read
      mep_wait_vm_lgkm0<8>();
      got(1);
      mep_bar();
      mep_each<NM>([&](auto c) MEP_INLINE {
        constexpr int n = c;
        if constexpr (n == 1) { hold(); __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n == 2) { on(); --left; __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n % R == 0) { read(0, n / R, at_rows); __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n % L == L / 2 + 1) { issueA(std::integral_constant<int, n / L>{}); __builtin_amdgcn_sched_barrier(0); }
        if constexpr (n == NM - 1) { turnA(wA); __builtin_amdgcn_sched_barrier(0); }
        constexpr int i = mep_row_block(n), j = mep_weight_block(n);
        mep_acc_mul<8 * i + j, false>(fw[1][j], fr[1][i]);
        __builtin_amdgcn_sched_barrier(0);
      });
      if (__builtin_expect(left == 0, 0)) turned();
      mep_wait_lgkm0();
      got(0);
    };
    auto steps = [&](auto frags) MEP_INLINE {
      scales_ask();
      step(frags, std::true_type{});
      for (kt = 1; kt < KT; ++kt) step(frags, std::false_type{});
      scales_in();
    };
    if (tall) steps(std::integral_constant<int, 8>{});
    else steps(std::integral_constant<int, 4>{});
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 15");  // the last sums are there
    __builtin_amdgcn_sched_barrier(0);

    // ---- epilogue: block 8 i + j is row 16 i + l15 of the wave's, its columns 32 (j / 2) + 8 lq +
    // 4 (j % 2) + 0 .. 3 (SwiGLU: gate in j = 0 .. 3, up in 4 .. 7)
    auto store_rows = [&](auto ii) MEP_INLINE {
      constexpr int i = ii;
      __builtin_amdgcn_sched_barrier(0);
      // row and column of what this lane stores first
      const size_t first = (size_t)(m0 + (tall ? 128 : 64) * wm + 16 * i + (l15 & 11)) * a.N + n0 + (SWIGLU ? 64 : 128) * wn +
                           8 * (l15 & 4) + 8 * lq;
      auto pack = [](const mep_f32x4& x, const mep_f32x4& y) MEP_INLINE {
        return mep_u4{mep_cvt_bf16x2(x[0], x[1]), mep_cvt_bf16x2(x[2], x[3]), mep_cvt_bf16x2(y[0], y[1]), mep_cvt_bf16x2(y[2], y[3])};
      };
      auto put = [&](uint16_t* out, mep_u4 x, mep_u4 y) MEP_INLINE {
        mep_trade(x, y);
        mep_u4_any* const at = (mep_u4_any*)(out + first);
        mep_u4_any* const below = (mep_u4_any*)(out + first + 4 * (size_t)a.N);
        if (rounds) {
          __builtin_nontemporal_store((mep_u4_any)x, at);
          __builtin_nontemporal_store((mep_u4_any)y, below);
        } else {
          *at = x;
          *below = y;
        }
      };
      if constexpr (SWIGLU) {
        mep_u4 h[2], g[2], u[2];
        mep_each<2>([&](auto c) MEP_INLINE {
          const mep_f32x4 g0 = mep_acc_get<8 * i + 2 * c>(), g1 = mep_acc_get<8 * i + 2 * c + 1>();
          const mep_f32x4 u0 = mep_acc_get<8 * i + 2 * c + 4>(), u1 = mep_acc_get<8 * i + 2 * c + 5>();
          auto act = [](const mep_f32x4& g, const mep_f32x4& u) MEP_INLINE {
            return mep_f32x4{mep_silu(g[0]) * u[0], mep_silu(g[1]) * u[1], mep_silu(g[2]) * u[2], mep_silu(g[3]) * u[3]};
          };
          h[c] = pack(act(g0, u0), act(g1, u1));
          g[c] = pack(g0, g1);
          u[c] = pack(u0, u1);
        });
        put(a.C, h[0], h[1]);
        if (a.Cg) put(a.Cg, g[0], g[1]);
        if (a.Cu) put(a.Cu, u[0], u[1]);
      } else {
        float sc = 1.0f;
        if (SCALED) sc = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (16 * (i & 3) + l15), __float_as_int(i < 4 ? scl0 : scl1)));
        mep_u4 x[4];
        mep_each<4>([&](auto c) MEP_INLINE {
          mep_f32x4 lo = mep_acc_get<8 * i + 2 * c>(), hi = mep_acc_get<8 * i + 2 * c + 1>();
          if (SCALED) { lo *= sc; hi *= sc; }
          x[c] = pack(lo, hi);
        });
        put(a.C, x[0], x[1]);
        put(a.C + 64, x[2], x[3]);
      }
    };
    mep_each<4>(store_rows);
    if (tall) mep_each<4>([&](auto i) MEP_INLINE { store_rows(std::integral_constant<int, i + 4>{}); });
  }
  mep_wait_vmcnt<0>();  // the loads of steps nobody wanted write LDS, too
  if (a.zero_tail) zero_tail_rows(a, blockIdx.x, gridDim.x, kWThreads);
}

using Kernel = void (*)(GemmArgs);

Kernel kernel_for(int mode, bool kn, bool scaled) {
  switch (mode) {
    case kModeSwiglu: return gemm_wide_kernel<kModeSwiglu, false, false>;
    case kModeDual: return kn ? gemm_wide_kernel<kModeDual, true, false> : gemm_wide_kernel<kModeDual, false, false>;
    default:
      if (kn) return scaled ? gemm_wide_kernel<kModeScale, true, true> : gemm_wide_kernel<kModeScale, true, false>;
      return scaled ? gemm_wide_kernel<kModeScale, false, true> : gemm_wide_kernel<kModeScale, false, false>;
  }
}

}  // namespace

int mep_launch_gemm_wide(int mode, bool kn, const GemmArgs& a, unsigned grid, hipStream_t st) {
  const Kernel kernel = kernel_for(mode, kn, mode == kModeScale && a.scale);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kWThreads), kWLds, st, a);
  return mep_launch_status();
}

int mep_init_gemm_wide_kernels() {
  for (int mode : {kModeScale, kModeSwiglu, kModeDual})
    for (int form = 0; form < 4; ++form)
      MEP_RETURN_IF_HIP(hipFuncSetAttribute((const void*)kernel_for(mode, form & 1, form & 2),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, kWLds));
  return MEP_OK;
}
