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
  float* Cf;           // wgrad: [G,M,N] fp32
  int64_t ld;          // row stride of A and B in elements (K, or the row count for wgrad)
  int skip_from;       // wgrad: groups g >= skip_from without rows are left unwritten
  float* Cf2;          // wgrad: the groups from `split` on go here
  int split;
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

// Four K rows of a column block, transposed (see mep_tr_pair).  As an instruction of its own: in
// front of the builtin the compiler waits for every load straight into LDS that is in flight.  The
// result is there after the next wait for lgkmcnt(0); nothing may touch it before.  The compiler does
// not know that: the build reads its assembly and fails where a register of a load in an asm
// statement is touched before its wait, or where anything is spilled (moonep_amd/asm_waits.py).
template <class T>
__device__ __forceinline__ void mep_tr_issue(T& x, uint32_t lds, int offset) {
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(x) : "v"(lds), "n"(offset));
}

// Tile list of the weight gradient: the dimension with more tiles is cut into eight slices, one
// per XCD (mirrored for odd groups, so that 28 tiles give every XCD 3 + 4), and every XCD takes
// its slice of every group, two neighbouring groups at a time: all XCDs finish together whatever
// the groups' lengths, and the tiles an XCD runs at one time are one group's slice times the whole
// other dimension -- each line they load is wanted by 3 to 8 of them.
struct Wgrad2Map {
  int sliced, other;  // tiles of the sliced and of the other dimension
  bool slice_m;       // the sliced dimension is the output row
  __host__ __device__ int lo(int x) const { return x * sliced / 8; }
  __host__ __device__ int size(int x) const { return (x + 1) * sliced / 8 - x * sliced / 8; }
  __host__ __device__ int pair_count(int x) const { return (size(x) + size(7 - x)) * other; }
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
  const Wgrad2Map& map;
  int xcd, w, nw, count, first_item, r, last;  // this workgroup among the XCD's, tiles of the XCD, rounds
  int c0, carry;             // row-tiled: 64 groups, one per lane; tiles before them
  int incl, end, blocks;     // tiles up to and including the group, its end, its 128-row blocks
  int g, m0, n0, kbeg, KT;
  bool tall;
  __device__ __forceinline__ PTiles(const GemmArgs& a_, const Wgrad2Map& map_) : a(a_), map(map_) {
    xcd = blockIdx.x & 7; nw = a.width; w = (int)(blockIdx.x >> 3) % nw;
    r = (int)(blockIdx.x >> 3) / nw * a.rounds; last = r + a.rounds;
    tall = true; kbeg = 0; KT = 0; g = 0; m0 = 0; n0 = 0;
    if (MODE == kModeWgrad) {
      count = map.pair_count(xcd) * (a.G >> 1);
    } else {
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
      if (MODE == kModeWgrad) {
        const int per_pair = map.pair_count(xcd);
        const int pair = item / per_pair;
        int local = item - pair * per_pair;
        const int n_even = map.size(xcd) * map.other;
        g = 2 * pair;
        int xe = xcd;
        if (local >= n_even) { local -= n_even; g += 1; xe = 7 - xcd; }
        const int sz = map.size(xe);
        const int u = local / sz, sl = map.lo(xe) + (local - u * sz);
        m0 = (map.slice_m ? sl : u) * kPT; n0 = (map.slice_m ? u : sl) * kPT;
        typedef const __attribute__((address_space(4))) int* cptr;  // scalar loads
        const int rank = g / a.Gr, l = g - rank * a.Gr;
        const int first = l > 0 ? ((cptr)a.cu)[g - 1] : 0;
        KT = (((cptr)a.cu)[g] - first) / kBK;
        kbeg = rank * a.rank_rows + first;
        if (KT == 0 && l >= a.skip_from) continue;
        return true;
      }
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
