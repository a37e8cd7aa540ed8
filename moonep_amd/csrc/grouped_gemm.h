// What the grouped GEMM kernels (grouped_gemm.hip, gemm_wide.hip) share: their arguments, the walk
// over the tiles, loads straight into LDS and the waits for them.
#pragma once

#include "mep_common.h"

namespace mep_gemm {

typedef __bf16 mep_bf16x8 __attribute__((ext_vector_type(8)));
typedef float mep_f32x4 __attribute__((ext_vector_type(4)));
typedef float mep_f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBM = 128, kBN = 256, kBK = 64;  // rows, weight rows, K per step of a tile
constexpr int kRowBytes = kBK * 2;             // an LDS row is one 128-byte slice, no padding
constexpr int kATile = kBM * kRowBytes, kBTile = kBN * kRowBytes;

struct GemmArgs {
  const uint16_t* A;   // [M,K]
  const uint16_t* B;   // [G,N,K]
  const uint16_t* B2;  // [G,N,K] up weights (swiglu) or null
  const int* cu;       // [G] padded end row of each group
  uint16_t* C;         // [M,N]
  const float* scale;  // [M] or null
  int M, N, K, G, mtiles, ntiles;
  const uint16_t* A2;  // dual: rows of the second K segment [M,K]
  uint16_t* Cg;        // swiglu: gate pre-activation [M,N] or null
  uint16_t* Cu;        // swiglu: up pre-activation [M,N] or null
  float* Cf;           // wgrad on 128 x 256 tiles: [G,M,N] fp32
  int64_t ld;          // row stride of A and B in elements (K, or the row count for wgrad)
  int skip_from;       // wgrad: groups g >= skip_from without rows are left unwritten
  int split;           // wgrad: the groups of a rank from here on have an output of their own
  bool zero_tail;      // row-tiled: the rows of C beyond the last group come out as zeros
  // the 256 x 256 kernel takes the groups of several ranks at once: Gr groups per rank, whose rows
  // start at rank_rows * rank (cu counts from there)
  int Gr, rank_rows;
  int width, rounds;  // 256 x 256 and streaming kernel: workgroups of an XCD that work at one time, tiles of one
};

enum { kModeScale = 0, kModeSwiglu = 1, kModeDual = 2, kModeWgrad = 3 };

__device__ __forceinline__ float mep_silu(float x) { return x / (1.0f + __expf(-x)); }

// s_waitcnt vmcnt(n) alone (expcnt and lgkmcnt left at "do not wait")
template <int N>
__device__ __forceinline__ void mep_wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

typedef short mep_s16x4 __attribute__((ext_vector_type(4)));
typedef short mep_s16x8 __attribute__((ext_vector_type(8)));

// bf16 outputs start at any element: stores of two and of eight of them at two-byte addresses (one
// instruction each at any address; the reads keep their 16 bytes)
typedef uint32_t mep_u1_any __attribute__((aligned(2)));
typedef uint32_t mep_u4_any __attribute__((ext_vector_type(4), aligned(2)));

// rows of C beyond a rank's last group, zeroed by `parts` workgroups of `threads` threads
__device__ __forceinline__ void zero_tail_rows(const GemmArgs& a, int part, int parts, int threads) {
  const mep_u4_any zero = {0u, 0u, 0u, 0u};
  for (int r = 0; (r + 1) * a.Gr <= a.G; ++r) {
    const int first = a.cu[(r + 1) * a.Gr - 1];
    const size_t bytes = (size_t)(a.rank_rows - first) * a.N * 2;  // N is a multiple of 128
    char* base = (char*)(a.C + ((size_t)r * a.rank_rows + first) * a.N);
    for (size_t o = ((size_t)part * threads + threadIdx.x) * 16; o < bytes; o += (size_t)parts * threads * 16)
      __builtin_nontemporal_store(zero, (mep_u4_any*)(base + o));
  }
}

// first row / end row of group gi
__device__ __forceinline__ int group_end(const GemmArgs& a, int gi) { return gi / a.Gr * a.rank_rows + a.cu[gi]; }
__device__ __forceinline__ int group_beg(const GemmArgs& a, int gi) {
  const int r = gi / a.Gr;
  return r * a.rank_rows + (gi > r * a.Gr ? a.cu[gi - 1] : 0);
}

constexpr int kPT = 256;                  // tile edge
constexpr int kPPanel = 8;                // row tiles of a long group that share a sweep over the weight tiles

__device__ __forceinline__ const char* mep_uniform(const char* p) {
  const uint64_t v = (uint64_t)p;
  return (const char*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v));
}

constexpr int kNontemporal = 2;  // cache policy of a buffer load

// 16 bytes per lane straight into LDS: lane offsets voff from a uniform base.  bytes = 0: nothing
// is read (every offset is past the end) and the lanes' LDS vectors come out undefined.
template <int AUX = 0>
__device__ __forceinline__ void mep_load_lds16(const char* base, uint32_t voff, uint32_t soff, char* lds, int bytes = -1) {
  __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, AUX);
}
template <int VM>
__device__ __forceinline__ void mep_wait_vm_lgkm0() {
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
}

__device__ __forceinline__ void mep_wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14)); }

__device__ __forceinline__ void mep_bar() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// two floats as bf16, rounded to nearest even by the hardware conversion
__device__ __forceinline__ uint32_t mep_cvt_bf16x2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Four K rows of a column block, transposed: sixteen lanes read a 4 x 16 block, 8 bytes of a row each,
// and each receives one of its columns.  As an instruction of its own: in front of the builtin the
// compiler waits for every load straight into LDS that is in flight.  The result is there after the next
// wait for lgkmcnt(0); nothing may touch it before.  The compiler does not know that: the build reads its
// assembly and fails where a register of a load in an asm statement is touched before its wait, or where
// anything is spilled (moonep_amd/asm_waits.py).
template <class T>
__device__ __forceinline__ void mep_tr_issue(T& x, uint32_t lds, int offset) {
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(x) : "v"(lds), "n"(offset));
}

// Tile list of the weight gradients.  A group's T tiles, those of a row of the longer dimension behind
// each other, are cut into eight runs of T / 8, and XCD x takes the run (x + group) mod 8: all XCDs
// finish together whatever the groups' lengths (slots are often empty) and however few tiles an expert
// has, and the tiles an XCD runs at one time lie in few rows and columns of one group.  (With whole rows
// to an XCD the 3 x 3 tiles of 768 x 768 went to four of the eight: 192 such experts on 16 ranks of 692
// tokens, K = 8, all three products 1140 -> 654 us.)  In eight consecutive groups every XCD has T tiles,
// and its place among them is found without a table: it walks the runs x, x + 1, ... x + 7; run v begins
// at v T / 8, from 8 on run v - 8 counted T further.
// Up to three products whose outputs are M x N or N x M (the projections of an expert) are one list,
// one product behind the other.
constexpr int kProducts = 3;
struct WgradMap {
  int tiles, other;   // T; tiles of the shorter dimension
  int n;              // products
  const uint16_t* A[kProducts];
  const uint16_t* B[kProducts];
  float* C[kProducts];   // [G, M, N]; the groups of a rank from a.split on go to C2
  float* C2[kProducts];
  int M[kProducts], N[kProducts];
  // one of the three without an address, which would put the arguments into memory
  template <class T>
  __host__ __device__ static T pick(const T (&v)[kProducts], int p) { return p == 0 ? v[0] : p == 1 ? v[1] : v[2]; }
  __host__ __device__ int begin(int v) const { return (int)((int64_t)v * tiles / 8); }
  // an XCD's tiles of one product
  __host__ __device__ int64_t count(int xcd, int groups) const {
    return (int64_t)tiles * (groups >> 3) + begin(xcd + (groups & 7)) - begin(xcd);
  }
  // the XCD's tile `item` of a product: its group, row of the longer dimension and place in it
  __host__ __device__ void find(int xcd, int item, int* group, int* row, int* place) const {
    const int octet = item / tiles;
    const int pos = item - octet * tiles + begin(xcd);
    const int v = (8 * pos + 7) / tiles;  // the last run that begins at or before this place
    *group = 8 * octet + v - xcd;
    const int first = begin(v), size = begin(v + 1) - first, rows = size / other;
    int at = pos - first;
    if (rows * other == size) at = at % rows * other + at / rows;  // whole rows: in columns (1 % at 16 x 8 tiles)
    at += first - (v >= 8 ? tiles : 0);
    *row = at / other;
    *place = at - *row * other;
  }
};

// The tiles of one workgroup of the weight gradients, one per lane: all that their divisions and table
// lookups need is done once, side by side, and a change of tiles reads the lane (made anew by both
// cursors at every change they were some hundred dependent instructions: three products of 64 experts of
// 2048 x 1024, 512 rows each, 708 -> 652 us, of 16 of 4096 x 2048, 2048 rows each, 1890 -> 1778).  As in
// PTiles, an XCD's workgroups take `rounds` tiles each in turn, moving on by one place from round to round.
constexpr int kListed = 64;  // most rounds
template <bool TN>
struct WgradTiles {
  int a0, a1, b0, b1, c0, c1;  // addresses: first K step of the operands, first element of the output
  int kp;                      // K steps, product
  uint64_t left;               // the tiles to come
  int KT, p, at;               // the present one
  static constexpr bool tall = true;
  __device__ __forceinline__ WgradTiles(const GemmArgs& a, const WgradMap* of) {
    const WgradMap& map = *of;
    const int lane = threadIdx.x & 63, xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int w = q % a.width, r = q / a.width * a.rounds + lane;
    const int per = (int)map.count(xcd, a.G);
    int item = r * a.width + (w + r) % a.width;
    bool live = lane < a.rounds && item < per * map.n;
    if (!live) item = 0;
    const int pr = (item >= per) + (item >= 2 * per);
    item -= pr * per;
    int g, sl, u;
    map.find(xcd, item, &g, &sl, &u);
    if (!live) g = 0;
    const int rank = g / a.Gr, l = g - rank * a.Gr;
    const int first = l > 0 ? a.cu[g - 1] : 0;
    const int steps = (a.cu[g] - first) / kBK;
    const int64_t kbeg = (int64_t)rank * a.rank_rows + first;
    live = live && (steps > 0 || l < a.skip_from);
    int64_t M = 0, N = 0;
    uint64_t A = 0, B = 0, C = 0;
#pragma unroll
    for (int k = 0; k < kProducts; ++k) {
      const uint64_t own = (uint64_t)map.C[k], other = (uint64_t)map.C2[k];
      const uint64_t to = l < a.split ? own : other;
      M = pr == k ? map.M[k] : M;
      N = pr == k ? map.N[k] : N;
      A = pr == k ? (uint64_t)map.A[k] : A;
      B = pr == k ? (uint64_t)map.B[k] : B;
      C = pr == k ? to : C;
    }
    const int64_t m0 = (M >= N ? sl : u) * kPT, n0 = (M >= N ? u : sl) * kPT;
    A += 2 * (TN ? kbeg * M + m0 : m0 * a.ld + kbeg);
    B += 2 * (TN ? kbeg * N + n0 : n0 * a.ld + kbeg);
    const int64_t row = (l < a.split ? (int64_t)rank * a.split + l : (int64_t)rank * (a.Gr - a.split) + l - a.split) * M + m0;
    C += 4 * (row * N + n0);
    a0 = (int)(uint32_t)A; a1 = (int)(A >> 32);
    b0 = (int)(uint32_t)B; b1 = (int)(B >> 32);
    c0 = (int)(uint32_t)C; c1 = (int)(C >> 32);
    kp = steps * 4 + pr;
    left = __ballot(live);
    KT = 0; p = 0; at = 0;
  }
  __device__ __forceinline__ char* lane_pointer(int lo, int hi) const {
    return (char*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, at) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, at));
  }
  __device__ __forceinline__ const char* A() const { return lane_pointer(a0, a1); }
  __device__ __forceinline__ const char* B() const { return lane_pointer(b0, b1); }
  __device__ __forceinline__ float* C() const { return (float*)lane_pointer(c0, c1); }
  // the next tile to write; false: no more
  __device__ __forceinline__ bool next() {
    if (!left) return false;
    at = __ffsll((unsigned long long)left) - 1;
    left &= left - 1;
    const int v = __builtin_amdgcn_readlane(kp, at);
    KT = v >> 2; p = v & 3;
    return true;
  }
};

// The tiles of one workgroup, in order.  XCD x (workgroups x, x + 8, ...) walks a contiguous
// eighth of the list, `width` workgroups in turn for `rounds` tiles each, then the next ones, so the
// tiles that run on an XCD at one time are neighbours in the list.  Row-tiled products: the list goes group by group, inside a group weight
// tile by weight tile, the group's row tiles fastest; a long group in panels of kPPanel row tiles
// (its weights are read once per panel, its rows once per 32 / kPPanel weight tiles).  From round
// to round a workgroup moves on by one place, so that the short last tiles of the groups do not
// all go to the same ones.
template <int MODE>
struct PTiles {
  const GemmArgs& a;
  int xcd, w, nw, count, first_item, r, last;  // this workgroup among the XCD's, tiles of the XCD, rounds
  int c0, carry;             // row-tiled: 64 groups, one per lane; tiles before them
  int incl, end, blocks;     // tiles up to and including the group, its end, its 128-row blocks
  int g, m0, n0, KT;
  bool tall;
  __device__ __forceinline__ explicit PTiles(const GemmArgs& a_, const WgradMap* = nullptr) : a(a_) {
    xcd = blockIdx.x & 7; nw = a.width; w = (int)(blockIdx.x >> 3) % nw;
    r = (int)(blockIdx.x >> 3) / nw * a.rounds; last = r + a.rounds;
    tall = true; KT = 0; g = 0; m0 = 0; n0 = 0;
    int total_rt = 0;
    for (int c = 0; c < a.G; c += 64) {
      chunk(c);
      total_rt += __shfl(incl, 63);
    }
    const int total = total_rt * a.ntiles;
    const int per_xcd = (total + 7) >> 3;
    first_item = xcd * per_xcd;
    count = min(per_xcd, total - first_item);
    count = __builtin_amdgcn_readfirstlane(count);
    if (a.G > 64) chunk(0);
    carry = 0;
  }
  __device__ __forceinline__ void chunk(int c) {
    c0 = c;
    const int gi = c + (int)(threadIdx.x & 63);
    end = gi < a.G ? group_end(a, gi) : 0;
    int beg = gi < a.G ? group_beg(a, gi) : 0;
    asm volatile("" : "+v"(end), "+v"(beg));  // the loads end here, not inside the main loop
    blocks = (end - beg) / kBM;
    incl = mep_wave_incl_scan((blocks + 1) >> 1);
  }
  // the next tile with work; false: no more
  __device__ __forceinline__ bool next() {
    for (;;) {
      int rot = w + r;
      rot -= rot / nw * nw;
      const int item = r * nw + rot;
      if (r >= last || r * nw >= count) return false;
      ++r;
      if (item >= count) continue;
      return find(item);
    }
  }
  __device__ __forceinline__ bool find(int item) {
    const int L0 = first_item + item;
    for (;;) {
      const uint64_t m = __ballot((carry + incl) * a.ntiles > L0);
      if (m) {
        const int src = __ffsll((unsigned long long)m) - 1;
        g = c0 + src;
        const int before = src > 0 ? __builtin_amdgcn_readlane(incl, src - 1) : 0;
        const int hs = __builtin_amdgcn_readlane(incl, src) - before, first = carry + before;
        const int gend = __builtin_amdgcn_readlane(end, src);
        const int gbeg = gend - __builtin_amdgcn_readlane(blocks, src) * kBM;
        const int local = L0 - first * a.ntiles;
        const int panel = local / (kPPanel * a.ntiles);
        const int within = local - panel * (kPPanel * a.ntiles);
        const int ph = min(kPPanel, hs - panel * kPPanel);
        const int nt = within / ph;
        m0 = gbeg + (panel * kPPanel + (within - nt * ph)) * kPT;
        n0 = nt * (MODE == kModeSwiglu ? kBN / 2 : kBN);
        tall = m0 + kPT <= gend;
        KT = MODE == kModeDual ? 2 * (a.K / kBK) : a.K / kBK;
        return true;
      }
      carry += __builtin_amdgcn_readlane(incl, 63);
      if (c0 + 64 >= a.G) return false;
      chunk(c0 + 64);
    }
  }
};

}  // namespace mep_gemm

// gemm_wide.hip: C = rows x weights on 256 x 256 tiles, four waves of 128 x 128.  kn: weights as [K, N]
// (plain and dual products).  `grid`, a.width and a.rounds as pp_split makes them.
int mep_launch_gemm_wide(int mode, bool kn, const mep_gemm::GemmArgs& a, unsigned grid, hipStream_t st);
int mep_init_gemm_wide_kernels();  // the LDS opt-ins of the current device
