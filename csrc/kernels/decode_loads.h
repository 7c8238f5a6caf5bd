// LDS-DMA of paged K / V tiles: the single instructions, the swizzles of the images, and the loads of a decode wave
// (attention.hip, sink_decode.hip).
#pragma once
#include "common.h"

namespace grag {

// Chunk (16 B) swizzle for the K image read as row fragments by ds_read_b128.
template <int D>
__device__ __forceinline__ int kswz(int row) {
  if constexpr (D == 128) return row & 15;
  else if constexpr (D == 64) return (row >> 1) & 7;
  else return (row >> 2) & 3;
}
// Chunk (16 B) swizzle for the V image read with ds_read_b64_tr_b16: a 32-lane
// half reads 8 consecutive rows x 4 8-byte units; these XORs spread them over
// all 64 banks (derivation in docs/kernels.md).
template <int D>
__device__ __forceinline__ int vswz(int row) {
  if constexpr (D == 128) return (row & 7) << 1;
  else if constexpr (D == 64) return ((row >> 1) & 3) << 1;
  else return ((row >> 2) & 1) << 1;
}

// One LDS-DMA wave instruction (global_load_lds_dwordx4): 16 B per lane from
// each lane's `src` into the 1 KiB LDS block at wave-uniform `lds_dst`
// (lane-linear).  Issued from inline asm so hipcc's waitcnt pass does not see
// an LDS write it cannot disambiguate between ring stages (it would put a
// vmcnt(0) in front of every ds_read); completion is tracked only by the
// caller's explicit counted `s_waitcnt vmcnt(N)` (cdna guide §5.7 recipe:
// M0 saved, set, used and restored inside one statement).
template <bool NT = false>
__device__ __forceinline__ void glds16(const void* src, void* lds_dst) {
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds_dst;
  const uint32_t lu = __builtin_amdgcn_readfirstlane(lds);
  uint32_t keep;
  if constexpr (NT) {  // non-temporal: once-read streams (decode K/V, MI355X_MICROARCH 'nt-weights')
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off nt\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(src), "s"(lu)
        : "memory");
  } else {
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(src), "s"(lu)
        : "memory");
  }
}

// The same LDS-DMA with the address as a wave-uniform 64-bit base in SGPRs plus a 32-bit per-lane byte
// offset (global_load_lds saddr form): no 64-bit VALU address arithmetic per load.
template <bool NT = false>
__device__ __forceinline__ void glds16_s(const void* sbase, uint32_t voff, void* lds_dst) {
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds_dst;
  const uint32_t lu = __builtin_amdgcn_readfirstlane(lds);
  uint32_t keep;
  if constexpr (NT) {
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2 nt\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(voff), "s"(sbase), "s"(lu)
        : "memory");
  } else {
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(voff), "s"(sbase), "s"(lu)
        : "memory");
  }
}

// The loads of one wave that walks TK-key tiles of a decode sequence: a ring of NS K and NS V buffers in LDS, filled by LDS-DMA.  A K
// buffer is filled again as soon as its tile's keys are in registers, a V buffer as soon as the values are, so 2 NS - 1 of the
// 2 NS buffers are in flight while the wave computes (tile by tile, 2 NS - 2).  Addresses are formed once per 16 keys, which lie
// in one cache block: a wave-uniform base and an offset a lane that only the context's end changes (with a division a piece and
// lane the addresses took longer than the products).  The block ids of a window of 64 blocks live one per lane; readlane hands
// them to the scalar unit.  Tiles start at multiples of 16 keys and blocks hold multiples of 16.
template <int D, int TK, int NS, bool NT>
struct DecodeLoads {
  static constexpr int DRB = 2 * D, CPR = D / 8, DTILE = TK * DRB, NI = DTILE / 1024;
  static constexpr int RPI = 1024 / DRB, PG = 16 / RPI, NG = TK / 16;
  static_assert((2 * NS - 1) * NI <= 63, "vmcnt range");
  const bf16 *k, *v;
  const int32_t* bt;
  char* ring;
  int BS, G, nblocks, kvh, last, nblk, lane, win, bvec, shift;
  size_t at[NG];  // of the tile whose keys were issued last: its groups' first element, its last valid row
  int lim[NG];

  // `last`: the last key that may be read; `first`: one of the first tile's
  __device__ __forceinline__ DecodeLoads(const bf16* k_, const bf16* v_, const int32_t* bt_, int BS_, int G_, int nblocks_, int kvh_,
                                         int ctx, int last_, int first, char* ring_)
      : k(k_), v(v_), bt(bt_), ring(ring_), BS(BS_), G(G_), nblocks(nblocks_), kvh(kvh_), last(last_), lane(threadIdx.x & 63) {
    nblk = (ctx + BS - 1) / BS;
    shift = (BS & (BS - 1)) == 0 ? __builtin_ctz(BS) : -1;
    win = block_of(first) >> 6;
    load_window();
  }
  __device__ __forceinline__ int block_of(int key) const {
    if (shift >= 0) return key >> shift;
    asm volatile("");
    return key / BS;
  }
  __device__ __forceinline__ void load_window() {
    bvec = bt[min((win << 6) + lane, nblk - 1)];
    if (!index_ok(bvec, nblocks, ERR_BLOCK_DECODE)) bvec = 0;  // reported; block 0 read instead of faulting
  }
  __device__ __forceinline__ void issue_k(int kt0, int stage) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int key = min(kt0 + 16 * g, last & ~15), b = block_of(key);  // (groups past the end re-read the last one)
      if ((b >> 6) != win) {
        win = b >> 6;
        load_window();
      }
      at[g] = (((size_t)__builtin_amdgcn_readlane(bvec, b & 63) * G + kvh) * BS + (key - b * BS)) * D;
      lim[g] = last - key;
#pragma unroll
      for (int i = 0; i < PG; ++i) {
        const int r = i * RPI + lane / CPR;
        glds16_s<NT>(k + at[g], (uint32_t)(min(r, lim[g]) * DRB + (((lane % CPR) ^ kswz<D>(r)) << 4)),
                     ring + stage * 2 * DTILE + (g * PG + i) * 1024);
      }
    }
  }
  __device__ __forceinline__ void issue_v(int stage) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int i = 0; i < PG; ++i) {
        const int r = i * RPI + lane / CPR;
        glds16_s<NT>(v + at[g], (uint32_t)(min(r, lim[g]) * DRB + (((lane % CPR) ^ vswz<D>(r)) << 4)),
                     ring + stage * 2 * DTILE + DTILE + (g * PG + i) * 1024);
      }
  }
  template <int H>
  __device__ __forceinline__ void wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(H * NI) : "memory");
  }
  // all but the `left` buffers issued last have landed
  __device__ __forceinline__ void wait_left(int left) {
    if (left >= 2 * NS - 1) return wait<2 * NS - 1>();
    if constexpr (NS > 3)
      if (left == 6) return wait<6>();
    if constexpr (NS > 3)
      if (left == 5) return wait<5>();
    if constexpr (NS > 2)
      if (left == 4) return wait<4>();
    if constexpr (NS > 2)
      if (left == 3) return wait<3>();
    if (left == 2) return wait<2>();
    if (left == 1) return wait<1>();
    wait<0>();
  }
  // the first tiles' loads: tile t starts at key first + t * step
  __device__ __forceinline__ void start(int first, int step, int n) {
#pragma unroll
    for (int t = 0; t < NS; ++t)
      if (t < n) issue_k(first + t * step, t), issue_v(t);
  }
};

}  // namespace grag
