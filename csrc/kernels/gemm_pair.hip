// Owned bf16 MFMA GEMM in tiles small enough for two and more workgroups a CU (tile_pair.h), for products that would give the 256 x
// 256 tile of gemm_tile.hip too few tiles or a last round that is nearly empty:
//   D[M, N] = A[M, K] W[N, K]^T       bf16 in, fp32 accumulate
// with that kernel's epilogues: store (bias, activation), the SwiGLU product of an interleaved gate / up weight, the gated unit of
// a weight of gate rows and up rows.  The sums run over K in the same order, so the results are that kernel's bit for bit.
//
// What bounds it: one round of tiles is a chain of K / 64 steps, each a trip to memory, LDS and the matrix cores (64 x 64 tiles:
// three steps in flight; 300 rows of 3072 x 768 with GELU 24 us as K parts and their sum -> 6.9).  Over many rounds 128 x 192
// tiles reach 1.15 PF/s where 256 x 256 ones reach 1.45: per product they fetch 1.7 times the bytes, and the LDS-DMA of a CU is
// busy (without it the same loop runs at 1.6, without the fragment reads at 1.3).  Measured: ops/gemm.py pair_plan.
#include "act.h"
#include "tile_pair.h"

using namespace grag;

namespace {

enum { EPI_STORE = 0, EPI_SILU = 1, EPI_GLU = 3 };

struct PairArgs {
  const bf16* A;
  const bf16* W;
  const bf16* bias;
  void* C;
  int lda, ldw, ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  int a_bytes, w_bytes;
  float limit, alpha, shift;  // EPI_GLU
};

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

template <int MT, int NT, int ST, int EPI, int ACT>
__global__ __launch_bounds__(kPairThreads, MT * NT >= 16 ? 2 : 3) void gemm_pair_kernel(PairArgs p) {
  constexpr int BM = 32 * MT, BN = 32 * NT, HN = NT / 2;
  constexpr bool GATED = EPI == EPI_SILU || EPI == EPI_GLU;
  __shared__ __attribute__((aligned(16))) char smem[ST * kPairStage<MT, NT>];
  const int L = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w >> 1, wc = w & 1;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  // bands of 16 row tiles x every column tile, rows first
  constexpr int GM = 16;
  const int band = GM * p.tiles_n, first_m = tile / band * GM, gsz = min(p.tiles_m - first_m, GM);
  const int m0 = (first_m + tile % band % gsz) * BM, n0 = tile % band / gsz * BN;
  unsigned offA[MT], offB[NT];
  const int koff = pair_piece_chunk() * 8;
#pragma unroll
  for (int i = 0; i < MT; ++i) offA[i] = (unsigned)(min(m0 + pair_piece_row(i), p.M - 1) * p.lda + koff) * 2u;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int r = pair_piece_row(i);  // LDS row: wave column r / (16 NT), its column tile, column
    int gn;
    if constexpr (GATED) {  // the wave's first HN column tiles are gate columns, the others the up columns that belong to them
      const int x = r / (16 * NT), nt = r % (16 * NT) / 16, up = nt >= HN;
      const int o = min((n0 / 2) + (x * HN + nt - up * HN) * 16 + (r & 15), p.N / 2 - 1);
      gn = EPI == EPI_GLU ? up * (p.N / 2) + o : (o >> 5) * 64 + up * 32 + (o & 31);
    } else {
      gn = min(n0 + r, p.N - 1);
    }
    offB[i] = (unsigned)(gn * p.ldw + koff) * 2u;
  }
  f32x4_t acc[MT][NT];
  pair_loop<MT, NT, ST>(smem, p.A, p.a_bytes, p.W, p.w_bytes, offA, offB, p.K / 64, acc);

  const int mrow = m0 + wr * 16 * MT + (L & 15), g = L >> 4;
  constexpr int ON = GATED ? HN : NT;  // 16-column tiles of a wave's output
  const int width = GATED ? p.N / 2 : p.N, c0 = (GATED ? n0 / 2 : n0) + wc * 16 * ON;
  bf16* C = (bf16*)p.C;
  // 4 columns of one row as two dwords
  auto value = [&](int m, int n, uint32_t (&d)[2]) __attribute__((always_inline)) {
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (EPI == EPI_GLU) v[r] = glu_f(acc[m][n][r], acc[m][n + HN][r], p.limit, p.alpha, p.shift);
      else if constexpr (EPI == EPI_SILU) v[r] = silu_f(acc[m][n][r]) * acc[m][n + HN][r];
      else v[r] = act_f<ACT>(acc[m][n][r]);
    }
    d[0] = pack_bf16x2(v[0], v[1]);
    d[1] = pack_bf16x2(v[2], v[3]);
  };
  // lanes of 16-lane rows 0 / 2 trade their second pair for the first of rows 1 / 3: 8 consecutive columns a lane
  auto trade = [&](uint32_t (&d0)[2], uint32_t (&d1)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const auto r = __builtin_amdgcn_permlane16_swap(d0[h], d1[h], false, false);
      d0[h] = r[0];
      d1[h] = r[1];
    }
  };
  if (p.bias != nullptr) {  // (per lane: 4 columns of every column tile)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      int col;
      if constexpr (GATED) {
        const int o = c0 + 16 * (n % HN) + 4 * g;
        col = (o >> 5) * 64 + (n >= HN) * 32 + (o & 31);
      } else {
        col = c0 + 16 * n + 4 * g;
      }
      if (col >= p.N) continue;
      const bf16x4_t bv = *reinterpret_cast<const bf16x4_t*>(p.bias + col);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][n][r] += bits2f(bv[r]);
    }
  }
#pragma unroll
  for (int n = 0; n + 1 < ON; n += 2)  // two column tiles of a row: 64 bytes of it in a store
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      uint32_t d0[2], d1[2];
      value(m, n, d0);
      value(m, n + 1, d1);
      trade(d0, d1);
      const int row = mrow + 16 * m, col = c0 + 16 * n + (g & 1) * 16 + (g >> 1) * 8;
      if (row < p.M && col < width) *reinterpret_cast<u32x4_t*>(C + (size_t)row * p.ldc + col) = u32x4_t{d0[0], d0[1], d1[0], d1[1]};
    }
  if constexpr (ON % 2)  // the last one: two row tiles of it
#pragma unroll
    for (int m = 0; m < MT; m += 2) {
      uint32_t d0[2], d1[2];
      value(m, ON - 1, d0);
      value(m + 1, ON - 1, d1);
      trade(d0, d1);
      const int row = mrow + 16 * m + (g & 1) * 16, col = c0 + 16 * (ON - 1) + (g >> 1) * 8;
      if (row < p.M && col < width) *reinterpret_cast<u32x4_t*>(C + (size_t)row * p.ldc + col) = u32x4_t{d0[0], d0[1], d1[0], d1[1]};
    }
}

template <int MT, int NT, int ST>
int launch_pair(const PairArgs& a, int epi, int act, hipStream_t st) {
  const int nwg = a.tiles_m * a.tiles_n;
  if (epi == EPI_SILU) gemm_pair_kernel<MT, NT, ST, EPI_SILU, ACT_NONE><<<nwg, kPairThreads, 0, st>>>(a);
  else if (epi == EPI_GLU) gemm_pair_kernel<MT, NT, ST, EPI_GLU, ACT_NONE><<<nwg, kPairThreads, 0, st>>>(a);
  else if (act == ACT_GELU) gemm_pair_kernel<MT, NT, ST, EPI_STORE, ACT_GELU><<<nwg, kPairThreads, 0, st>>>(a);
  else if (act == ACT_GELU_TANH) gemm_pair_kernel<MT, NT, ST, EPI_STORE, ACT_GELU_TANH><<<nwg, kPairThreads, 0, st>>>(a);
  else gemm_pair_kernel<MT, NT, ST, EPI_STORE, ACT_NONE><<<nwg, kPairThreads, 0, st>>>(a);
  return (int)hipGetLastError();
}

}  // namespace

// shape: 0 = 128 x 192 tiles, 1 = 128 x 128, 2 = 64 x 128, 3 = 64 x 64.  epi 0 store (act 0 none, 1 gelu-erf, 3 gelu-tanh), 1
// SwiGLU (W rows interleaved in 32-row gate / up blocks, C [M, N / 2]), 3 gated unit (W gate rows | up rows, C [M, N / 2], no bias).
// K a multiple of 64, operands that span less than 2 GB, strides multiples of 8, N of 8 (SwiGLU 64, unit 16), A, W and C
// aligned to 16 bytes, the bias to 8.
GRAG_API int grag_gemm_pair(const void* A, const void* W, const void* bias, void* C, int lda, int ldw, int ldc, int M, int N,
                            int K, int epi, int act, int shape, float limit, float alpha, float shift, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 64 != 0 || K < 64 || lda % 8 != 0 || ldw % 8 != 0 || ldc % 8 != 0 || N % 8 != 0 || lda < 0 || ldw < 0 || shape < 0 || shape > 3)
    return (int)hipErrorInvalidValue;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15 || ((uintptr_t)bias & 7)) return (int)hipErrorInvalidValue;
  if ((epi != EPI_STORE && epi != EPI_SILU && epi != EPI_GLU) || (epi == EPI_SILU && N % 64) || (epi == EPI_GLU && (N % 16 || bias)))
    return (int)hipErrorInvalidValue;
  if (act != ACT_NONE && (epi != EPI_STORE || (act != ACT_GELU && act != ACT_GELU_TANH))) return (int)hipErrorInvalidValue;
  const long ab = ((long)(M - 1) * lda + K) * 2, wb = ((long)(N - 1) * ldw + K) * 2;
  if (ab >= (1L << 31) || wb >= (1L << 31)) return (int)hipErrorInvalidValue;
  static const int bm[4] = {128, 128, 64, 64}, bn[4] = {192, 128, 128, 64};
  PairArgs a;
  a.A = (const bf16*)A, a.W = (const bf16*)W, a.bias = (const bf16*)bias, a.C = C;
  a.lda = lda, a.ldw = ldw, a.ldc = ldc, a.M = M, a.N = N, a.K = K;
  a.tiles_m = (M + bm[shape] - 1) / bm[shape], a.tiles_n = (N + bn[shape] - 1) / bn[shape];
  a.a_bytes = (int)ab, a.w_bytes = (int)wb, a.limit = limit, a.alpha = alpha, a.shift = shift;
  if ((long)a.tiles_m * a.tiles_n >= (1L << 30)) return (int)hipErrorInvalidValue;
  if (shape == 0) return launch_pair<4, 6, 2>(a, epi, act, st);
  if (shape == 1) return launch_pair<4, 4, 2>(a, epi, act, st);
  if (shape == 2) return launch_pair<2, 4, 2>(a, epi, act, st);
  return launch_pair<2, 2, 3>(a, epi, act, st);
}
