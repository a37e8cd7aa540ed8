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
// AT: added to both addresses, in the instruction.
template <int AUX = 0, int AT = 0>
__device__ __forceinline__ void mep_load_lds16(const char* base, uint32_t voff, uint32_t soff, char* lds, int bytes = -1) {
  __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, AT, AUX);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mep_rsrc(const char* base) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, -1, 0x00020000);
}
template <int AUX = 0, int AT = 0>
__device__ __forceinline__ void mep_load_lds16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, AT, AUX);
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

// n / d for n >= 0, d > 0, in half the instructions of the general division (what a kernel runs once waits for its
// instructions to be fetched): the quotient in fp32, that of what it leaves, and at most one more
__device__ __forceinline__ int mep_quotient(int n, int d) {
  const float inv = __builtin_amdgcn_rcpf((float)d);
  int q = (int)((float)n * inv);
  q += (int)((float)(n - q * d) * inv);
  const int rest = n - q * d;
  return q + (rest >= d) - (rest < 0);
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

// Tile list of the weight gradients: group by group (those with rows), a group's products (up to three, whose
// outputs are M x N or N x M: the projections of an expert) behind each other, a product in bands of about four
// tiles of the shorter dimension, a band row by row.  A group's T tiles are cut into eight runs of T / 8, and of
// the k-th group XCD x takes the run (x + k) mod 8: all XCDs finish together whatever the groups' lengths and
// however few tiles an expert has, the longest groups (local experts come first) early, and the tiles that an XCD
// runs at one time are neighbours in one group, which all XCDs work on at that time.  In eight consecutive groups
// every XCD has T tiles, and its place among them is found without a table: it walks the runs x, x + 1, ...
// x + 7; run v begins at v T / 8, from 8 on run v - 8 counted T further.
// (All groups of one product, then of the next, with the empty ones in their places, put long tiles last and wrote
// the zeros at times when nobody multiplied.  us, that order -> this: 64 experts of 2048 x 1024 on 8 ranks, 512 rows
// each 645 -> 545 (2.6 -> 1.4 GB fetched), 16 of 4096 x 2048 with 2048 rows each and as many empty slots 1730 -> 1640,
// 4 of 2560 x 512 with 5443 250 -> 172.  An eighth of the whole list by work to each XCD fetches less, 0.8 instead of
// 1.4 GB, and takes longer: 617, 1680, 172.)
constexpr int kProducts = 3;
struct WgradMap {
  int tiles, rows, other;   // tiles of an output; of its longer dimension, of the shorter one
  int bands;
  int n;                    // products
  const uint16_t* A[kProducts];
  const uint16_t* B[kProducts];
  float* C[kProducts];   // [G, M, N]; the groups of a rank from a.split on go to C2
  float* C2[kProducts];
  int tall;              // bit p: product p has the longer dimension as its rows
  __host__ __device__ int M(int p) const { return (tall >> p & 1 ? rows : other) * kPT; }
  __host__ __device__ int N(int p) const { return (tall >> p & 1 ? other : rows) * kPT; }
  // one of the three without an address, which would put the arguments into memory
  template <class T>
  __host__ __device__ static T pick(const T (&v)[kProducts], int p) { return p == 0 ? v[0] : p == 1 ? v[1] : v[2]; }
  // tile `item` of a product: its row of the longer dimension and its place in the shorter one
  __device__ __forceinline__ void find(int item, int* row, int* place) const {
    // the band that holds it: the last that begins at or before
    const int band = mep_quotient(bands * (mep_quotient(item, rows) + 1) - 1, other);
    const int first = mep_quotient(band * other, bands), width = mep_quotient((band + 1) * other, bands) - first;
    const int at = item - first * rows;
    *row = mep_quotient(at, width);
    *place = first + at - *row * width;
  }
  __device__ __forceinline__ int begin(int v) const { return (int)((int64_t)v * tiles * n >> 3); }  // of a run
  // an XCD's tiles of the first k groups
  __device__ __forceinline__ int count(int xcd, int k) const { return tiles * n * (k >> 3) + begin(xcd + (k & 7)) - begin(xcd); }
  // where row `row` and place `place` of product p begin, in elements of M and of N
  __device__ __forceinline__ void corner(int p, int row, int place, int* m0, int* n0) const {
    *m0 = (tall >> p & 1 ? row : place) * kPT;
    *n0 = (tall >> p & 1 ? place : row) * kPT;
  }
};

// The tiles of one workgroup of the weight gradients, one per lane: all that their divisions and table
// lookups need is done once, side by side, and a change of tiles reads the lane (made anew by both
// cursors at every change they were some hundred dependent instructions: three products of 64 experts of
// 2048 x 1024, 512 rows each, 708 -> 652 us, of 16 of 4096 x 2048, 2048 rows each, 1890 -> 1778).  An XCD's
// workgroups are sets of a.width that walk its tiles together, moving on by one place from round to round;
// the sets share the rounds, whose number is only known here, evenly.
// a.rounds: the tiles of all groups, with rows or without, stay in their places, as many for a set, and nobody
// looks for the groups with rows first: what that takes, 1 to 3 us, is not made up for where a workgroup has one tile, of
// whatever kind.  216 sizes of one round, 4 to 128 groups of 256 x 256 to 2048 x 1024, 128 to 1024 rows in an
// eighth, half or all of them, against the order by products: the list 0.96 to 1.27 times its time, 1.03 on
// average, this 0.72 to 1.09, 0.96 (4 of 256 x 256 with 128 rows 10.1, 13.0 and 9.6 us).  162 sizes of 2 to 16 rounds: the list
// 0.94, 1.02 where all groups have rows, this 0.98.
constexpr int kListed = 64;           // most tiles of a workgroup
constexpr int kTabled = 64 * 4096;    // most groups in the tables (100 KB); more stay in their places
typedef __attribute__((address_space(1))) float mep_global_f32;
template <bool TN>
struct WgradTiles {
  const GemmArgs& a;
  const WgradMap& map;
  int a0, a1, b0, b1, c0, c1;  // addresses: first K step of the operands, first element of the output
  int kp;                      // K steps, product
  uint64_t left, empties;      // the tiles to come; tiles of zeros
  int KT, p, at;               // the present one
  static constexpr bool tall = true;
  // a group's first row among its rank's, and its K steps; -1: none, and it comes out as zeros
  __device__ __forceinline__ int steps_of(int gi, int* beg) const {
    *beg = 0;
    if (gi >= a.G) return 0;
    const int l = a.G == a.Gr ? gi : gi % a.Gr;
    *beg = l > 0 ? a.cu[gi - 1] : 0;
    const int steps = (a.cu[gi] - *beg) / kBK;
    return steps > 0 ? steps : l < a.skip_from ? -1 : 0;
  }
  // the place of the k-th set bit
  static __device__ __forceinline__ int nth(uint64_t mask, int k) {
    int at = 0;
#pragma unroll
    for (int b = 32; b; b >>= 1) {
      const int c = __popcll(mask >> at & ((1ull << b) - 1));
      if (k >= c) { k -= c; at += b; }
    }
    return at;
  }
  // lds: the kernel's; free again when this returns in all waves
  __device__ __forceinline__ WgradTiles(const GemmArgs& a_, const WgradMap* of, char* lds) : a(a_), map(*of) {
    const int lane = threadIdx.x & 63, xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int set = mep_quotient(q, a.width), w = q - set * a.width;
    auto turn = [&](int r) { return r * a.width + w + r - mep_quotient(w + r, a.width) * a.width; };
    const int per = map.tiles * map.n;
    int k, g, item, first, length;
    bool live;
    // the XCD's tile `at` of a list: which of the groups, and its place among that group's
    auto group = [&](int at) {
      const int octet = mep_quotient(at, per), pos = at - octet * per + map.begin(xcd);
      const int run = mep_quotient(8 * pos + 7, per);  // the last that begins at or before this place
      k = 8 * octet + run - xcd;
      item = pos - map.begin(run) + map.begin(run & 7);
    };
    if (a.rounds) {  // all groups in their places
      const int r = set * a.rounds + lane, at = turn(r);
      live = lane < a.rounds && at < map.count(xcd, a.G);
      group(live ? at : 0);
      g = live ? k : 0;
      length = steps_of(g, &first);
      live = live && length;
    } else {
      // groups with rows and groups that come out as zeros: how many, and of every 64 groups which and how many in
      // front of them.  More than 64 groups: each wave looks at its part of them (one after the other, 1536 groups
      // would be 24 latencies of the memory).
      const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), chunks = (a.G + 63) / 64;
      int beg = 0, steps = steps_of(lane, &beg);
      uint64_t some = __ballot(steps > 0), none = __ballot(steps < 0);
      int full = __popcll(some), empty = __popcll(none), sum = 0;
      uint64_t* const masks = (uint64_t*)lds;                     // [2 chunks]
      int2* const before = (int2*)(lds + 16 * (size_t)chunks);    // [chunks + 8], the waves' sums behind
      if (chunks > 1) {
        full = empty = 0;
        const int mine = wave * chunks / 8, end = (wave + 1) * chunks / 8;
        for (int c = mine; c < end; ++c) {
          steps = steps_of(64 * c + lane, &beg);
          some = __ballot(steps > 0); none = __ballot(steps < 0);
          if (lane == 0) { masks[2 * c] = some; masks[2 * c + 1] = none; before[c] = make_int2(full, empty); }
          full += __popcll(some); empty += __popcll(none);
        }
        if (lane == 0) before[chunks + wave] = make_int2(full, empty);
        __syncthreads();
        full = empty = 0;
#pragma unroll
        for (int v = 0; v < 8; ++v) { const int2 n = before[chunks + v]; full += n.x; empty += n.y; }
        full = __builtin_amdgcn_readfirstlane(full); empty = __builtin_amdgcn_readfirstlane(empty);
      } else {
        sum = __builtin_amdgcn_readlane(mep_wave_incl_scan(max(steps, 0)), 63);
      }
      // This workgroup's tiles, a lane each.  The sets share the rounds of the groups with rows evenly, and all
      // workgroups the tiles of zeros (as a tail of the list, when nothing is left to multiply, those of 15 of 32 groups
      // of 4096 x 2048 are 100 us of 1750), but in a launch of one set the workgroups that have a tile less than the
      // others first take as many of them as make up for it, a tile of zeros being the time of some six K steps.
      const int all_of = (int)(gridDim.x >> 3), sets = mep_quotient(all_of, a.width);
      const int tiles = map.count(xcd, full), blank = map.count(xcd, empty), total = mep_quotient(tiles + a.width - 1, a.width);
      const int base = mep_quotient(total, sets), over = total - base * sets;
      const int first_round = set * base + min(set, over), rounds = base + (set < over);
      int extra = 0, place = q, from = 0, own = 0;
      if (sets == 1 && blank) {
        const int turned = max(total - 1, 0), more = tiles - turned * a.width, less = a.width - more;
        place = w + turned - mep_quotient(w + turned, a.width) * a.width;
        if (less) {
          extra = min(blank, less * min(1 + mep_quotient(sum, 6 * max(full, 1)), kListed / 4));
          const int each = mep_quotient(extra, less), more_of = extra - each * less, light = place - more;
          if (light >= 0) {
            from = light * each + min(light, more_of);
            own = each + (light < more_of);
          }
        }
      }
      const int base2 = mep_quotient(blank - extra, all_of), over2 = blank - extra - base2 * all_of;
      const int back = all_of - 1 - place;
      const int from2 = extra + back * base2 + min(back, over2), own2 = base2 + (back < over2);
      const int z = lane - rounds;
      const bool zero = z >= 0;
      const int at = zero ? (z < own ? from + z : from2 + z - own) : turn(first_round + lane);
      live = zero ? z < own + own2 : at < tiles;
      group(live ? at : 0);
      // that group: among those with rows (zeros: without) the k-th
      if (chunks > 1) {
        // the wave whose part holds it, the chunk in there
        int c = 0, end = 0;
#pragma unroll
        for (int v = 0; v < 8; ++v) {
          const int2 part = before[chunks + v];
          const int n = zero ? part.y : part.x;
          const bool here = c == end && k < n;
          if (here) { c = v * chunks / 8; end = (v + 1) * chunks / 8; }
          else if (c == end) k -= n;
        }
        while (end - c > 1) {  // the last chunk with no more than k in front of it
          const int m = (c + end) / 2;
          const int2 b = before[m];
          if ((zero ? b.y : b.x) <= k) c = m;
          else end = m;
        }
        const int2 b = before[c];
        g = 64 * c + nth(masks[2 * c + zero], k - (zero ? b.y : b.x));
        if (!live) g = 0;
        length = steps_of(g, &first);
        __syncthreads();  // the tables have been read
      } else {
        g = live ? nth(zero ? none : some, k) : 0;
        first = __shfl(beg, g);
        length = __shfl(steps, g);
      }
    }
    const int pr = mep_quotient(item, map.tiles);
    int sl, u, m0, n0;
    map.find(item - pr * map.tiles, &sl, &u);
    map.corner(pr, sl, u, &m0, &n0);
    const int rank = a.G == a.Gr ? 0 : g / a.Gr;
    const int64_t kbeg = (int64_t)rank * a.rank_rows + first;
    const uint64_t A = (uint64_t)WgradMap::pick(map.A, pr) + 2 * (TN ? kbeg * map.M(pr) + m0 : m0 * a.ld + kbeg);
    const uint64_t B = (uint64_t)WgradMap::pick(map.B, pr) + 2 * (TN ? kbeg * map.N(pr) + n0 : n0 * a.ld + kbeg);
    const uint64_t C = (uint64_t)output(pr, g, m0, n0);
    a0 = (int)(uint32_t)A; a1 = (int)(A >> 32);
    b0 = (int)(uint32_t)B; b1 = (int)(B >> 32);
    c0 = (int)(uint32_t)C; c1 = (int)(C >> 32);
    kp = max(length, 0) * 4 + pr;
    left = __ballot(live && length > 0);
    empties = __ballot(live && length < 0);
    KT = 0; p = 0; at = 0;
  }
  __device__ __forceinline__ float* output(int pr, int g, int m0, int n0) const {
    const int rank = a.G == a.Gr ? 0 : g / a.Gr, l = g - rank * a.Gr;
    const int64_t N = map.N(pr);
    const int64_t row = (l < a.split ? (int64_t)rank * a.split + l : (int64_t)rank * (a.Gr - a.split) + l - a.split) * map.M(pr) + m0;
    return (l < a.split ? WgradMap::pick(map.C, pr) : WgradMap::pick(map.C2, pr)) + row * N + n0;
  }
  __device__ __forceinline__ char* lane_pointer(int lo, int hi) const {
    return (char*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, at) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, at));
  }
  __device__ __forceinline__ const char* A() const { return lane_pointer(a0, a1); }
  __device__ __forceinline__ const char* B() const { return lane_pointer(b0, b1); }
  // In global memory by its type: a store through a pointer of unknown kind counts among the LDS operations, too, and a wait
  // for LDS reads then is one for the stores (C1).
  __device__ __forceinline__ mep_global_f32* C() const { return (mep_global_f32*)lane_pointer(c0, c1); }
  // the next of the workgroup's tiles of zeros: its first element, its row length; false: no more
  __device__ __forceinline__ bool blank(mep_global_f32** out, int* N) {
    if (!empties) return false;
    const int now = at;
    at = __ffsll((unsigned long long)empties) - 1;
    empties &= empties - 1;
    *out = C();
    *N = map.N(__builtin_amdgcn_readlane(kp, at) & 3);
    at = now;
    return true;
  }
  // the next tile; false: no more
  __device__ __forceinline__ bool next() {
    if (!left) return false;
    at = __ffsll((unsigned long long)left) - 1;
    left &= left - 1;
    const int v = __builtin_amdgcn_readlane(kp, at);
    KT = v >> 2; p = v & 3;
    return true;
  }
};

// The order of the K steps of forward products (rows and weights along K), the same in every kernel that makes them: the
// forms agree to the bit.  At a pitch that is a multiple of 4 KB the 128 bytes that all CUs ask for in one step lie, of
// every row, on the same few channels of the L2 and the memory; the steps of a 4 KB piece of the rows then alternate between its
// halves, so that the two or three that are on their way at one time use twice as many.  Otherwise they go up.  The order
// is that of the shape alone.  us, up -> this, streaming kernel, 17 blocks of 128 rows (in brackets the time of 128 more columns,
// which go up): down 4096 x 2048 67.7 (54.6) -> 53.8, 4096 x 4096 122.5 -> 97.9, 2048 x 4096 64.3 -> 57.6, SwiGLU 2048 x 2048
// 68.4 -> 53.7, 2048 x 4096 97.1 -> 96.7.  Tiles that begin at 2, 4 or 16 different places take as long as this (55.8, 56.1, 57.0
// for the first), with sums whose order depends on the tile.  At a pitch of 2 KB (K = 1024) beginning at different places gains
// nothing.  The 256 x 256 kernels, whose operands come from the L2 several times, take the same time with either order.
constexpr int kFold = 32;   // K steps of 4 KB
__host__ __device__ __forceinline__ bool mep_folds(int K) { return K % (kFold * kBK) == 0; }
// bytes from step k of a folded product to the next one
__device__ __forceinline__ int mep_fold_step(int k) {
  k &= kFold - 1;
  return k & 1 ? (k == kFold - 1 ? 1 : 1 - kFold / 2) * kRowBytes : kFold / 2 * kRowBytes;
}

// The tiles of one workgroup, in order.  XCD x (workgroups x, x + 8, ...) walks a contiguous
// eighth of the list, `width` workgroups in turn for `rounds` tiles each, then the next ones, so the
// tiles that run on an XCD at one time are neighbours in the list.  Row-tiled products: the list goes group by group, inside a group weight
// tile by weight tile, the group's row tiles fastest; a long group in panels of kPPanel row tiles
// (its weights are read once per panel, its rows once per 32 / kPPanel weight tiles).  From round
// to round a workgroup moves on by one place, so that the short last tiles of the groups do not
// all go to the same ones.
// HALVES: where the last round has a tile for at most half of the workgroups, each goes out as two of
// 128 rows, which take 0.55 to 0.6 of a tile's time.  us, before -> now: 16 groups of 4096 x 2048 with 2048 rows,
// dy * down (4.25 rounds) 505 -> 488; 13 of 1280 x 768 with 8 K steps' rows, SwiGLU and down 130 -> 110; 2 of 1024 x
// 768 with 300 rows 29.6 -> 23.5; 120 drawn sizes 2.7 % on average, 2 % slower at worst (one division more).
template <int MODE, bool HALVES = false>
struct PTiles {
  const GemmArgs& a;
  int xcd, w, nw, count, first_item, r, last;  // this workgroup among the XCD's, tiles of the XCD, rounds
  int whole, items;          // tiles that stay whole, places in the rounds
  int c0, carry;             // row-tiled: 64 groups, one per lane; tiles before them
  int incl, end, blocks;     // tiles up to and including the group, its end, its 128-row blocks
  int g, m0, n0, KT;
  bool tall;
  __device__ __forceinline__ explicit PTiles(const GemmArgs& a_, const WgradMap* = nullptr, char* = nullptr) : a(a_) {
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
    const int rest = count > 0 ? count - mep_quotient(count, nw) * nw : 0;
    whole = HALVES && 2 * rest <= nw ? count - rest : count;
    items = HALVES ? 2 * count - whole : count;
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
      rot -= mep_quotient(rot, nw) * nw;
      const int item = r * nw + rot;
      if (r >= last || r * nw >= items) return false;
      ++r;
      if (item < items && find(item)) return true;
    }
  }
  __device__ __forceinline__ bool find(int item) {
    const int parted = HALVES ? max(item - whole, 0) : 0;
    const int L0 = first_item + item - (parted + 1) / 2;
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
        const int panel = mep_quotient(local, kPPanel * a.ntiles);
        const int within = local - panel * (kPPanel * a.ntiles);
        const int ph = min(kPPanel, hs - panel * kPPanel);
        const int nt = mep_quotient(within, ph);
        m0 = gbeg + (panel * kPPanel + (within - nt * ph)) * kPT;
        n0 = nt * (MODE == kModeSwiglu ? kBN / 2 : kBN);
        tall = m0 + kPT <= gend;
        if (HALVES && item >= whole) {
          if (!tall && (parted & 1)) return false;  // there is no second half
          m0 += (parted & 1) * kBM;
          tall = false;
        }
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
