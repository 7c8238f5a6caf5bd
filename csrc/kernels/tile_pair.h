// A bf16 tile product of 4 waves for workgroups that share a CU with another (gemm_pair.hip): 2 (rows) x 2 (columns) waves of
// 16 MT x 16 NT outputs, K steps of 64, 16x16x32 matrix-core products, ST LDS buffers refilled by LDS-DMA.
// A wave reads the fragments of half a K step while it multiplies those of the other half, so that a buffer is free for the refill
// of step t + ST in the middle of step t; the other workgroup of the CU multiplies while this one waits or writes its tile out.
// Rows in LDS are 128 bytes, their 16-byte chunks XOR-swizzled by (row >> 1) & 7 on the source address.
#pragma once
#include "common.h"

namespace grag {

constexpr int kPairThreads = 256;
template <int MT, int NT> constexpr int kPairStage = (MT + NT) * 4096;  // bytes of a K step: 32 MT rows of A, 32 NT of B

// The LDS row and 16-byte source chunk of the thread's DMA piece i of an operand (32 rows a piece)
__device__ __forceinline__ int pair_piece_row(int i) { return 32 * i + (threadIdx.x >> 3); }
__device__ __forceinline__ int pair_piece_chunk() { return (threadIdx.x & 7) ^ ((threadIdx.x >> 4) & 7); }

template <int N> __device__ __forceinline__ void pair_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }
// raw barrier: never drains the LDS-DMA in flight (a __syncthreads() would emit vmcnt(0))
__device__ __forceinline__ void pair_bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc += A B^T over nk >= 1 K steps.  offA / offB: byte offsets of the thread's DMA pieces at the first step (pair_piece_row /
// _chunk say which); smem: ST * kPairStage<MT, NT> bytes.  An accumulator's lane holds 4 consecutive columns of one row (the W
// fragment is operand A): row 16 mt + lane % 16, columns 16 nt + 4 (lane / 16) + 0..3 of the wave's block.
template <int MT, int NT, int ST>
__device__ __forceinline__ void pair_loop(char* smem, const void* A, int a_bytes, const void* W, int w_bytes,
                                          const unsigned (&offA)[MT], const unsigned (&offB)[NT], int nk,
                                          f32x4_t (&acc)[MT][NT]) {
  static_assert(ST == 2 || ST == 3, "the waits below");
  constexpr int STAGE = kPairStage<MT, NT>, P = MT + NT;
  const __amdgpu_buffer_rsrc_t rsA = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(A), 0, a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsB = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(W), 0, w_bytes, 0x00020000);
  const int L = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w >> 1, wc = w & 1;
  const int cb = (L >> 4) ^ ((L >> 1) & 7);
  const int off[2] = {(L & 15) * 128 + cb * 16, (L & 15) * 128 + (cb ^ 4) * 16};
  auto issue = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
      lds_dma16(rsA, smem + buf * STAGE + (4 * i + w) * 1024, offA[i], kt * 128);
#pragma unroll
    for (int i = 0; i < NT; ++i)
      lds_dma16(rsB, smem + buf * STAGE + (4 * (MT + i) + w) * 1024, offB[i], kt * 128);
  };
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < nk) issue(s, s);
  bf16x8_t a[2][MT], b[2][NT];
  auto read = [&](int s, int buf) __attribute__((always_inline)) {
    const char* pa = smem + buf * STAGE + wr * MT * 2048 + off[s];
    const char* pb = smem + buf * STAGE + MT * 4096 + wc * NT * 2048 + off[s];
#pragma unroll
    for (int m = 0; m < MT; ++m) a[s][m] = *reinterpret_cast<const bf16x8_t*>(pa + m * 2048);
#pragma unroll
    for (int n = 0; n < NT; ++n) b[s][n] = *reinterpret_cast<const bf16x8_t*>(pb + n * 2048);
  };
  auto mma = [&](int s) __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][n], a[s][m], acc[m][n], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };
  // step t has landed when only the ST - 1 (at the end: fewer) steps behind it are in flight
  auto landed = [&](int behind) __attribute__((always_inline)) {
    if (behind >= ST - 1) pair_wait_vm<(ST - 1) * P>();
    else if (ST > 2 && behind == 1) pair_wait_vm<P>();
    else pair_wait_vm<0>();
  };
  landed(nk - 1);
  pair_bar();
  read(0, 0);
  for (int t = 0, buf = 0; t < nk; ++t) {
    const int next = buf + 1 == ST ? 0 : buf + 1;
    read(1, buf);
    __builtin_amdgcn_sched_barrier(0);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < nk) {
      // the own reads of this buffer and the own pieces of step t + 1 are there; behind the barrier everyone's
      if (t + ST <= nk) pair_wait_vm<(ST - 2) * P>();
      else pair_wait_vm<0>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      pair_bar();
      if (t + ST < nk) issue(t + ST, buf);
      read(0, next);
      __builtin_amdgcn_sched_barrier(0);
    }
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
    buf = next;
  }
}

}  // namespace grag
