// Pieces shared by the attention kernels: matrix-core fragment types, the
// 32x32x16 MFMA for each 16-bit element type, and 16-byte buffer loads.
#pragma once

#include "api.h"
#include "common.h"

namespace pk {
namespace attn {

constexpr int max_of(int a, int b) { return a > b ? a : b; }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s4;

// D[32x32] += A[32x16] B[16x32]: lane l holds row l%32 of A (K elements
// 8*(l/32) .. +8) and column l%32 of B (the same K elements); the result
// lane l holds column l%32, rows 8*(r/4) + 4*(l/32) + r%4 for r = 0..15.
template <typename T> struct Mma;
template <> struct Mma<bf16> {
  typedef bf16x8 frag;
  static __device__ __forceinline__ f32x16 run(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<f16> {
  typedef f16x8 frag;
  static __device__ __forceinline__ f32x16 run(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// 16 bytes at voffset + soffset of a buffer resource (zeros past its range)
__device__ __forceinline__ uint4 ld_buf(__amdgpu_buffer_rsrc_t r, int voffset, int soffset) {
  typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
  const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, voffset, soffset, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// 16 bytes at voffset + soffset of a buffer resource written straight to LDS:
// lane i's bytes land at lds + 16 * i (lds must be the same for the whole
// wave); zeros past the resource's range. Completion is counted by vmcnt.
__device__ __forceinline__ void ld_buf_lds(__amdgpu_buffer_rsrc_t r, void* lds, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voffset, soffset, 0, 0);
}

// 4 bytes per lane, as ld_buf_lds (lane i's word at lds + 4 * i).
__device__ __forceinline__ void ld_buf_lds4(__amdgpu_buffer_rsrc_t r, void* lds, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, voffset, soffset, 0, 0);
}

// ---- which tile of rows (or keys) block w works on
//
// A "group" is what shares K/V: a (sequence, kv head, quad of q heads), say; a
// sequence's `per_seq` groups are consecutive. Dispatch is round-robin over the
// 8 XCDs, block w running on XCD w % 8.
struct WorkItem {
  int seq, group, tile;  // seq < 0: no work
};

// Dense batches, `groups` = sequences * per_seq of `tiles` tiles each, the last
// of them partial if `partial`. With a multiple of 8 groups, XCD x runs groups
// x, x + 8, ... one after another, so the blocks resident on an XCD share one
// group's K/V in its L2; otherwise the tiles run one after another over all
// groups. DESC (causal rows): the last tiles are the longest and go first.
// Otherwise all tiles are alike but the partial ones, which go last, where a
// short block fills what the whole ones leave (1025 rows of 12 heads of 64, a
// batch of 8: the 96 blocks of one row each took slots of a first round that
// the 768 whole blocks fill).
//
// snake > 0 (DESC, grids that all fit on the device at once; the CUs of an
// XCD): longest first over all groups, every second round of blocks the other
// way, so that a CU's blocks add up to much the same on every CU. In one
// direction the CU with the longest block of one round had that of the next too.
// Causal forward, us: fp32, 32/8 heads of 128, 2 x 1024 tokens 313 -> 187; bf16, 12
// heads of 64, 4 x 2048 52.2 -> 43.1, 32/8 heads of 128, 2048 55.2 -> 50.4; nowhere
// slower.
template <bool DESC>
__device__ __forceinline__ WorkItem dense_item(int w, int groups, int per_seq, int tiles, bool partial, int snake) {
  int tile, rest;
  if (DESC && snake > 0) {
    const int x = w & 7, k = w >> 3, round = k / snake, first = round * snake;
    const int size = min(snake, ((groups * tiles - x + 7) >> 3) - first);  // blocks of this round on the XCD
    const int at = 8 * ((round & 1) ? 2 * first + size - 1 - k : k) + x;
    return {at % groups / per_seq, at % groups % per_seq, tiles - 1 - at / groups};
  }
  if (!DESC && partial && tiles > 1 && w >= (tiles - 1) * groups) {
    tile = tiles - 1;
    rest = w - tile * groups;
  } else {
    if (!DESC && partial && tiles > 1) --tiles;
    if (groups % 8 == 0) {
      const int k = w >> 3;
      tile = k % tiles;
      rest = (w & 7) + 8 * (k / tiles);
    } else {
      tile = w / groups;
      rest = w % groups;
    }
    if (DESC) tile = tiles - 1 - tile;
  }
  return {rest / per_seq, rest % per_seq, tile};
}

// dense_item's snake: for causal grids of more than one block per CU, all resident at once.
inline int snake_cus(bool causal, int64_t blocks, int resident) {
  const int64_t cus = cu_count();
  return causal && blocks > cus && blocks <= resident * cus ? (int)(cus / 8) : 0;
}

// Packed sequences, at most 64 of them: only the tiles that exist, the longest
// sequence first (the blocks that run last are then short), all of a sequence's
// tiles of one group on one XCD where per_seq is a multiple of 8. A grid of the
// longest sequence's tiles for every sequence was three quarters empty blocks at
// 23 documents of 44 to 3048 tokens, and ended with whatever came last. Each wave
// finds its item alone: lane i holds sequence i's tiles and counts those of the
// sequences in front of it.
template <bool DESC>
__device__ __forceinline__ WorkItem packed_item(int w, const int* cu, int seqs, int total, int longest, int rows, int per_seq) {
  int u, group;
  if (per_seq % 8 == 0) {
    const int k = w >> 3, each = per_seq >> 3;
    u = k / each;
    group = (w & 7) + 8 * (k % each);
  } else {
    u = w / per_seq;
    group = w % per_seq;
  }
  const int lane = threadIdx.x & 63;
  int mine = 0;
  if (lane < seqs) {
    const int start = min(max(cu[lane], 0), total);
    const int len = min(min(max(cu[lane + 1], start), total) - start, longest);
    mine = (len + rows - 1) / rows;
  }
  int before = 0;
  for (int j = 0; j < seqs; ++j) {
    const int t = __builtin_amdgcn_readlane(mine, j);
    before += t > mine || (t == mine && j < lane) ? t : 0;
  }
  const uint64_t found = __ballot(u >= before && u < before + mine);
  if (found == 0) return {-1, 0, 0};
  const int seq = __builtin_ctzll(found);
  const int tile = u - __builtin_amdgcn_readlane(before, seq);
  return {seq, group, DESC ? __builtin_amdgcn_readlane(mine, seq) - 1 - tile : tile};
}

// Tiles of `rows` that the packed sequences can have at most, when blocks are
// to be found by packed_item; 0 when every sequence gets the longest one's.
inline int packed_tiles(bool packed, int64_t seqs, int64_t total, int64_t longest, int64_t rows) {
  return packed && seqs > 1 && seqs <= 64 && longest > rows ? (int)(total / rows + seqs) : 0;
}

// A buffer resource as its four words (base, 32-bit range, raw-buffer flags),
// made wave-uniform, for the inline-assembly loads below.
typedef unsigned rsrc_words __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc_words make_rsrc_words(const void* base, int nrec) {
  const uint64_t p = (uint64_t)base;
  rsrc_words r;
  r.x = __builtin_amdgcn_readfirstlane((uint32_t)p);
  r.y = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32) & 0xffffu);
  r.z = __builtin_amdgcn_readfirstlane((uint32_t)nrec);
  r.w = 0x00020000u;
  return r;
}

// ld_buf_lds and ld_buf_lds4 as inline assembly (M0 = the wave's LDS base).
// The compiler does not see these LDS writes, so it waits for none of them
// before later LDS reads, which it must do for the builtin whenever it cannot
// tell the written buffer from the one read (one array indexed by stage). The
// caller waits (lds_loads_landed) before any barrier after which a wave may
// read what it wrote. It must also let the compiler finish its own vector
// loads before issuing these: its waits count loads by number, and loads it
// does not know of would make them wait for more than they mean to.
// (A generic pointer into LDS holds the LDS address in its low 32 bits.)
__device__ __forceinline__ uint32_t lds_base(const void* lds) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
}
__device__ __forceinline__ void ld_lds16_asm(rsrc_words r, const void* lds, int voffset, int soffset) {
  asm volatile("buffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds_base(lds)), "v"(voffset), "s"(r),
               "s"(__builtin_amdgcn_readfirstlane(soffset))
               : "memory");
}
__device__ __forceinline__ void ld_lds4_asm(rsrc_words r, const void* lds, int voffset, int soffset) {
  asm volatile("buffer_load_dword %1, %2, %3 offen lds" ::"{m0}"(lds_base(lds)), "v"(voffset), "s"(r),
               "s"(__builtin_amdgcn_readfirstlane(soffset))
               : "memory");
}

// Wait until this wave's LDS-bound buffer loads have landed.
__device__ __forceinline__ void lds_loads_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Wait until at most N of this wave's vector memory loads are still in flight
// (they complete in issue order).
template <int N> __device__ __forceinline__ void loads_landed_but() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Four 16-bit values as two packed 32-bit words
template <typename T> __device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  return make_uint2((uint32_t)__builtin_bit_cast(uint16_t, from_f32<T>(a)) |
                        ((uint32_t)__builtin_bit_cast(uint16_t, from_f32<T>(b)) << 16),
                    (uint32_t)__builtin_bit_cast(uint16_t, from_f32<T>(c)) |
                        ((uint32_t)__builtin_bit_cast(uint16_t, from_f32<T>(d)) << 16));
}

}  // namespace attn
}  // namespace pk
