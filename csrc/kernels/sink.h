// What the sink attention kernels of prompts and of decode share (sink_prefill.hip, sink_decode.hip).
#pragma once
#include "common.h"

namespace grag {

constexpr int SP_BS = 16;          // keys per cache block
constexpr float SP_RESCALE = 8.f;  // the running maximum moves when a score passes it by 2^8

struct SinkArgs {
  const bf16 *q, *k, *v;
  bf16* out;
  const int *bt, *q_start, *ctx_len;
  const float *sinks, *hscale;
  const bf16* hgate;
  int out_ld, bt_stride, H, G, R, nblocks, nseq, tiles, gate_ld, chunk, window, keep;
  float scale, out_scale, softcap;
};

typedef __attribute__((address_space(3))) void sp_lds_t;
typedef __attribute__((address_space(3))) bf16x4_t sp_lds4_t;

// swizzles of the 16-byte chunks of a tile's rows: K is read as row fragments, V by the transposed read (8 rows x 4 units of 8
// bytes at a time); both spread a read over all banks
template <int D> __device__ __forceinline__ int sp_kswz(int row) { return D == 128 ? row & 15 : (row >> 1) & 7; }
template <int D> __device__ __forceinline__ int sp_vswz(int row) { return D == 128 ? (row & 7) << 1 : ((row >> 1) & 3) << 1; }

// 16 bytes a lane from `off` bytes behind a wave-uniform base, with no bound, into 1 KB of LDS, lane after lane, in a form whose
// wait the compiler leaves to the caller: behind the builtin it puts one for everything in flight before each transposed read.
__device__ __forceinline__ void sp_dma_s(const bf16* base, unsigned off, char* dst) {
  const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(sp_lds_t*)dst);
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(off), "s"(base), "s"(lds) : "memory");
}

// first key of the block / window of the query at `pos` (never falls as pos grows)
__device__ __forceinline__ int sp_first(const SinkArgs& p, int pos) {
  const int lo = p.chunk > 0 ? pos - pos % p.chunk : 0;
  return p.window > 0 ? max(lo, pos - p.window + 1) : lo;
}

}  // namespace grag
