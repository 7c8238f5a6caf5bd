// The 256 x 256 bf16 tile product that the dense and the grouped GEMM share (gemm_tile.hip, moe.hip): 8 waves (512
// threads) as 2 (rows) x 4 (columns), K steps of 64, 16x16x32 matrix-core products, two LDS buffers refilled by LDS-DMA.
// Wave (wr, wc) owns rows [128 wr, +128) x columns [64 wc, +64) as 2 x 2 quadrants of 64 x 32.  A buffer holds 4 slots of 16 KB
// (A q0, A q1, B q0, B q1), each the 128 rows (both wave rows / all 4 wave columns) that one quadrant needs; rows are 128
// bytes, their 16-byte chunks XOR-swizzled by (row >> 1) & 7 on the source address.
#pragma once
#include "common.h"

namespace grag {

constexpr int kTileSlot = 128 * 128;        // bytes: 128 rows x 64 bf16
constexpr int kTileBuf = 4 * kTileSlot;     // one K step: A q0, A q1, B q0, B q1
constexpr int kTileThreads = 512;

template <int MT> using TileAccN = f32x4_t[MT][2];  // a quadrant: [16 rows][16 columns]
template <int MT> using TileAN = bf16x8_t[MT][2];   // [16 rows][k step of 32]
typedef TileAccN<4> TileAcc;
typedef TileAN<4> TileA;
typedef bf16x8_t TileB[2][2];    // [16 columns][k step]

template <int MT>
__device__ __forceinline__ void tile_zero(TileAccN<MT>& c) {
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n) c[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}
// (the W fragment is operand A, so that a lane ends with 4 consecutive output columns of one row)
template <int MT>
__device__ __forceinline__ void tile_mma(TileAccN<MT>& acc, const TileAN<MT>& a, const TileB& b) {
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[nt][s], a[mt][s], acc[mt][nt], 0, 0, 0);
  __builtin_amdgcn_s_setprio(0);
}
// raw barrier: never drains the LDS-DMA in flight (a __syncthreads() would emit vmcnt(0))
__device__ __forceinline__ void tile_bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int N> __device__ __forceinline__ void tile_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }
__device__ __forceinline__ void tile_wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The LDS row (0..127) and 16-byte source chunk (0..7) of the thread's DMA piece i (0, 1) of a slot
__device__ __forceinline__ int tile_piece_row(int i) {
  return (2 * (threadIdx.x >> 6) + i) * 8 + ((threadIdx.x & 63) >> 3);
}
__device__ __forceinline__ int tile_piece_chunk(int i) { return (threadIdx.x & 7) ^ ((tile_piece_row(i) >> 1) & 7); }

// Two-phase schedule: 32 MFMAs per barrier interval.  Per K step t (buffer b = t & 1):
//   L1 reads A q0, B q0, B q1 (16 b128)  refill A q1 of step t+1 (buffer b^1; read there in L2(t-1))
//   M1 acc00 = A0 B0, acc01 = A0 B1       (32 MFMAs)
//   L2 reads A q1 (8 b128)                refill A q0, B q0, B q1 of step t+2 (buffer b; read in L1(t))
//   M2 acc10 = A1 B0, acc11 = A1 B1       (32 MFMAs; B q0 / q1 held from L1)
// Waves 4-7 (wr = 1) run one barrier interval behind waves 0-3: on every SIMD one wave loads while its partner multiplies.
// Every load segment ends with a counted vmcnt(8) (its own 2 or 6 refills plus the other segment's are the 8 youngest), which
// retires the batch the NEXT load segment reads -- for the lagging half too, whose load segments coincide with the leading
// half's MFMA segments.  A refill is issued one segment after the barrier that closes the last read of its slot by either
// half.  Refills past the last K step re-load it (clamped index) into slots nobody reads again, so the counts never change.
// offA / offB [quadrant][piece]: byte offsets of the thread's DMA pieces at the first K step (tile_piece_row / _chunk say
// which).  live: rows of this wave's 128 that exist; quadrants without any are not multiplied (PARTIAL only).
template <bool PARTIAL>
__device__ __forceinline__ void tile256_loop(char* smem, const __amdgpu_buffer_rsrc_t& rsA, const __amdgpu_buffer_rsrc_t& rsB,
                                             const unsigned (&offA)[2][2], const unsigned (&offB)[2][2], int nk, int live,
                                             TileAcc& acc00, TileAcc& acc01, TileAcc& acc11, TileAcc& acc10) {
  const int L = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w >> 2, wc = w & 3;
  const bool lag = w >= 4;
  const int cb = (L >> 4) ^ ((L >> 1) & 7);
  const int off0 = (L & 15) * 128 + cb * 16, off1 = (L & 15) * 128 + (cb ^ 4) * 16;
  auto readA = [&](TileA& a, int q, int buf) {
    const char* base = smem + buf * kTileBuf + q * kTileSlot + wr * 64 * 128;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      a[mt][0] = *reinterpret_cast<const bf16x8_t*>(base + mt * 2048 + off0);
      a[mt][1] = *reinterpret_cast<const bf16x8_t*>(base + mt * 2048 + off1);
    }
  };
  auto readB = [&](TileB& b, int q, int buf) {
    const char* base = smem + buf * kTileBuf + (2 + q) * kTileSlot + wc * 32 * 128;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      b[nt][0] = *reinterpret_cast<const bf16x8_t*>(base + nt * 2048 + off0);
      b[nt][1] = *reinterpret_cast<const bf16x8_t*>(base + nt * 2048 + off1);
    }
  };
  auto issueA = [&](int q, int kt, int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, (lds_t*)(smem + buf * kTileBuf + q * kTileSlot + (2 * w + i) * 1024),
                                               16, offA[q][i], kt * 128, 0, 0);
  };
  auto issueB = [&](int q, int kt, int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_t*)(smem + buf * kTileBuf + (2 + q) * kTileSlot + (2 * w + i) * 1024),
                                               16, offB[q][i], kt * 128, 0, 0);
  };
  TileA a;
  TileB b0, b1;
  tile_zero<4>(acc00);
  tile_zero<4>(acc01);
  tile_zero<4>(acc11);
  tile_zero<4>(acc10);
  const int klast = nk - 1;
  issueA(0, 0, 0);
  issueB(0, 0, 0);
  issueB(1, 0, 0);
  issueA(1, 0, 0);
  issueA(0, min(1, klast), 1);
  issueB(0, min(1, klast), 1);
  issueB(1, min(1, klast), 1);
  tile_wait_vm<6>();  // step 0 landed (step 1's A0 / B0 / B1 are the 6 youngest)
  tile_bar();
  if (lag) tile_bar();
  auto step = [&](int kt, auto odd_c) {
    constexpr int buf = decltype(odd_c)::value ? 1 : 0;
    // L1
    readA(a, 0, buf);
    readB(b0, 0, buf);
    readB(b1, 1, buf);
    issueA(1, min(kt + 1, klast), buf ^ 1);
    tile_wait_vm<8>();
    tile_wait_lds();
    tile_bar();
    // M1
    if (!PARTIAL || live > 0) {
      tile_mma<4>(acc00, a, b0);
      tile_mma<4>(acc01, a, b1);
    }
    tile_bar();
    // L2
    readA(a, 1, buf);
    issueA(0, min(kt + 2, klast), buf);
    issueB(0, min(kt + 2, klast), buf);
    issueB(1, min(kt + 2, klast), buf);
    tile_wait_vm<8>();
    tile_wait_lds();
    tile_bar();
    // M2
    if (!PARTIAL || live > 64) {
      tile_mma<4>(acc10, a, b0);
      tile_mma<4>(acc11, a, b1);
    }
    tile_bar();
  };
  int kt = 0;
  for (; kt < klast; kt += 2) {
    step(kt, std::integral_constant<bool, false>{});
    step(kt + 1, std::integral_constant<bool, true>{});
  }
  if (kt == klast) step(kt, std::integral_constant<bool, false>{});
  tile_wait_vm<0>();  // the clamped re-loads land before the LDS is reused
  if (!lag) tile_bar();
}

// The same schedule over a chain of tiles that one workgroup works off: the refills of a tile's last two steps are the next
// tile's first ones, so the loop never drains, and a tile's results are stored while the other half of the waves multiplies and
// the next tile's steps are in flight: its first row quadrants behind the loads of its last step's L2, the others behind those
// of the next tile's first L1.  Loads wait for older stores in the memory counter (it counts in order); the waits of the first step
// behind a tile leave out the 2 * ST2 stores in between, so the stores have a K step's time.
//   next(i, off): byte offsets of the workgroup's i-th tile at its first K step (kTileNone in all: there is none); whether it is
//   emit(q, l, r): stores row quadrant q (columns of acc(q)0, acc(q)1) of the tile in exactly ST2 vector-memory instructions
//   ahead(i): (nk >= 5) called in the second step of tile i - 1; what its vector-memory instructions bring to LDS is there for
//   next(i)
// MT: 16-row tiles of a quadrant: 4, or 3 and 2 for tiles of 192 and 128 rows (a wave's quadrants of 48 and 32).  An A slot then has 96
// and 64 rows; the pieces of the others (tile_piece_row) are kTileNone.
//   live(): rows of this wave's 32 MT that the tile of the last next has; quadrants without any are not multiplied (PARTIAL only)
typedef unsigned TileOff __attribute__((ext_vector_type(8)));  // A [quadrant][piece], B the same (a vector: kept in registers)
constexpr unsigned kTileNone = 0x80000000u;      // past the end of any operand (< 2 GB): loads zeros without a trip to memory

template <int ST2, bool PARTIAL, int MT = 4, typename Next, typename Emit, typename Ahead, typename Live>
__device__ __forceinline__ void tile256_chain(char* smem, const __amdgpu_buffer_rsrc_t& rsA, const __amdgpu_buffer_rsrc_t& rsB,
                                              int nk, Next&& next, Emit&& emit, Ahead&& ahead, Live&& live) {
  const int L = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w >> 2, wc = w & 3;
  const bool lag = w >= 4;
  const int cb = (L >> 4) ^ ((L >> 1) & 7);
  const int off0 = (L & 15) * 128 + cb * 16, off1 = (L & 15) * 128 + (cb ^ 4) * 16;
  auto readA = [&](TileAN<MT>& a, int q, int buf) __attribute__((always_inline)) {
    const char* base = smem + buf * kTileBuf + q * kTileSlot + wr * 16 * MT * 128;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      a[mt][0] = *reinterpret_cast<const bf16x8_t*>(base + mt * 2048 + off0);
      a[mt][1] = *reinterpret_cast<const bf16x8_t*>(base + mt * 2048 + off1);
    }
  };
  auto readB = [&](TileB& b, int q, int buf) __attribute__((always_inline)) {
    const char* base = smem + buf * kTileBuf + (2 + q) * kTileSlot + wc * 32 * 128;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      b[nt][0] = *reinterpret_cast<const bf16x8_t*>(base + nt * 2048 + off0);
      b[nt][1] = *reinterpret_cast<const bf16x8_t*>(base + nt * 2048 + off1);
    }
  };
  auto issueA = [&](const TileOff& o, int q, int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_dma16(rsA, smem + buf * kTileBuf + q * kTileSlot + (2 * w + i) * 1024, o[2 * q + i], kt * 128);
  };
  auto issueB = [&](const TileOff& o, int q, int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      lds_dma16(rsB, smem + buf * kTileBuf + (2 + q) * kTileSlot + (2 * w + i) * 1024, o[4 + 2 * q + i], kt * 128);
  };
  TileAN<MT> a;
  TileB b0, b1;
  TileAccN<MT> acc00, acc01, acc11, acc10;
  TileOff cur;
  next(0, cur);
  issueA(cur, 0, 0, 0);
  issueB(cur, 0, 0, 0);
  issueB(cur, 1, 0, 0);
  issueA(cur, 1, 0, 0);
  issueA(cur, 0, 1, 1);
  issueB(cur, 0, 1, 1);
  issueB(cur, 1, 1, 1);
  tile_wait_vm<6>();  // step 0 landed
  tile_bar();
  if (lag) tile_bar();
  tile_zero<MT>(acc00);
  tile_zero<MT>(acc01);
  int buf = 0, rows = 32 * MT;
  bool more = true, behind = false;  // behind: a tile's stores lie between the loads
  auto step = [&](int i, int kt, auto first_c, auto last_c) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value, LAST = decltype(last_c)::value;
    // L1
    if (FIRST && behind) {  // (its results before the fragments: both would not fit the registers)
      issueA(cur, 1, 1, buf ^ 1);
      emit(1, acc10, acc11);
    }
    if (FIRST) {
      tile_zero<MT>(acc10);
      tile_zero<MT>(acc11);
    }
    readA(a, 0, buf);
    readB(b0, 0, buf);
    readB(b1, 1, buf);
    if (FIRST && behind) {
      tile_wait_vm<8 + 2 * ST2>();
    } else {
      issueA(cur, 1, LAST ? 0 : kt + 1, buf ^ 1);
      tile_wait_vm<8>();
    }
    tile_wait_lds();
    tile_bar();
    // M1
    if (!PARTIAL || rows > 0) {
      tile_mma<MT>(acc00, a, b0);
      tile_mma<MT>(acc01, a, b1);
    }
    tile_bar();
    // L2
    if (!LAST && kt + 2 == nk) more = next(i + 1, cur);
    const int k2 = LAST ? 1 : kt + 2 < nk ? kt + 2 : 0;
    auto refill = [&]() __attribute__((always_inline)) {
      issueA(cur, 0, k2, buf);
      issueB(cur, 0, k2, buf);
      issueB(cur, 1, k2, buf);
    };
    if (LAST) {
      refill();
      tile_wait_vm<8>();  // (behind the stores it took as long: 34 products and 30 of experts, 0.999 - 1.002 in the geometric mean)
      emit(0, acc00, acc01);
      tile_zero<MT>(acc00);
      tile_zero<MT>(acc01);
      readA(a, 1, buf);
    } else {
      readA(a, 1, buf);
      refill();
      if (FIRST && behind) tile_wait_vm<8 + 2 * ST2>();
      else tile_wait_vm<8>();
    }
    tile_wait_lds();
    tile_bar();
    // M2
    if (!PARTIAL || rows > 16 * MT) {
      tile_mma<MT>(acc10, a, b0);
      tile_mma<MT>(acc11, a, b1);
    }
    tile_bar();
    buf ^= 1;
  };
  const std::integral_constant<bool, true> yes{};
  const std::integral_constant<bool, false> no{};
  for (int i = 0;; ++i) {
    if (PARTIAL) rows = live();
    step(i, 0, yes, no);
    ahead(i + 1);
    for (int kt = 1; kt + 1 < nk; ++kt) step(i, kt, no, no);
    step(i, nk - 1, no, yes);
    if (!more) break;
    behind = true;
  }
  emit(1, acc10, acc11);
  tile_wait_vm<0>();  // the loads of the tile that is not there
  if (!lag) tile_bar();
}

// A chain's time, us, for `tiles` tiles of 64 MT rows and 256 columns on ncu CUs, `full` of them if they were all full: begun rounds and
// useful ones, each by K steps and once (the chip's power makes a round that is nearly empty a shorter one).  Least squares over 105
// points of nine products (widths 768 - 37888, K 768 - 18944, 300 - 24000 rows), 5 % off on average there and 6 % at 83 others.
template <int MT> __host__ __device__ inline float tile_chain_us(float tiles, float full, int steps, int ncu) {
  const float begun = ceilf(tiles / (float)ncu), used = full / (float)ncu;
  if (MT == 4) return (.72f * begun + .64f * used) * steps + 9.2f * begun - 2.3f * used + 3.8f;
  if (MT == 3) return (.66f * begun + .43f * used) * steps + 4.0f * begun + 1.8f * used + 5.2f;
  return (.58f * begun + .32f * used) * steps + 2.5f * begun + 1.3f * used + 5.6f;
}

}  // namespace grag
