// Normalisation kernels: fused residual-add + RMSNorm (Qwen2, N1b),
// fused bias + residual + LayerNorm (BERT-family encoders, N2d),
// fused word/pos/type embedding gather + LayerNorm (N2a) and the plain
// token-embedding gather used by the decoder (N1a).
//
// Design: one 256-thread block per row, the row held in registers as 16-B
// bf16x8 vectors (Guideline 13), fp32 statistics, one LDS round trip per
// reduction.  These ops are HBM-bound; at H=3584 a row is 7 KB read + 7 KB
// written (+7 KB residual each way when fused), which is why the residual add
// is folded in instead of being a separate pass.
#include "common.h"
#include <string.h>

using namespace grag;

namespace {

constexpr int kThreads = 256;

template <int VPT>
__global__ __launch_bounds__(kThreads) void rmsnorm_kernel(
    const bf16* __restrict__ x, bf16* __restrict__ residual, const bf16* __restrict__ w,
    bf16* __restrict__ out, int H, float eps) {
  __shared__ float red[kThreads / 64];
  const int row = blockIdx.x;
  const int nvec = H >> 3;
  const bf16x8_t* xr = reinterpret_cast<const bf16x8_t*>(x + (size_t)row * H);
  bf16x8_t* rr = residual ? reinterpret_cast<bf16x8_t*>(residual + (size_t)row * H) : nullptr;
  float v[VPT][8];
  float ss = 0.f;
  // gamma is loaded before the reduction, so its latency overlaps the row loads instead of following the
  // block sum (at decode batches of 1-16 rows these kernels are latency chains, not bandwidth)
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(w);
  bf16x8_t gv[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) gv[i] = wr[idx];
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float a[8];
      unpack8(xr[idx], a);
      if (rr) {
        float b[8];
        unpack8(rr[idx], b);
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += b[j];
        // the residual stream is kept in bf16, so normalise the rounded sum
        bf16x8_t s = pack8(a);
        rr[idx] = s;
        unpack8(s, a);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = a[j];
        ss += a[j] * a[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    }
  }
  ss = block_sum(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)row * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float g[8], o[8];
      unpack8(gv[i], g);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * inv * g[j];
      orow[idx] = pack8(o);
    }
  }
}

// Split-K reduce fused into the decoder's block boundary: h = sum_s ws[s] (fp32
// planes a split-K projection left behind, ops/linear.py linear_deferred),
// residual += h (rounded to bf16, the residual stream's precision), out =
// RMSNorm(residual) * w.  Replaces splitk_reduce (fp32 planes -> bf16 h) +
// rmsnorm (h + residual): one launch and one bf16 round trip of h fewer per
// o_proj / down_proj at decode batches, and h is never rounded before the add.
constexpr int kFewRows = 16;
constexpr int kWideRows = 256;

// Few rows: the launch is as long as its chain of round trips to memory (the planes lie in other dies' caches or beyond), so a
// thread takes four columns -- up to 1024 threads a row, every plane's load, the residual's and the weight's in one trip.
// Width 3584, us with 8 columns a thread -> here: 7 planes 1 row 6.6 -> 3.7, 64 rows 5.2 -> 4.1, 256 rows 7.4 -> 4.9; 9 planes
// 7.8 -> 4.3, 5.6 -> 4.6, 9.2 -> 7.4; 8192, 7 planes 10.1 -> 5.4, 8.3 -> 5.9, 15.0 -> 12.7.  400 rows of 8192 are
// bandwidth's: 19.0 / 19.3 (and 9 planes, walked as 12, 22.5 / 26.3).
template <int V>
__global__ __launch_bounds__(1024) void splitk_rmsnorm_wide_kernel(
    const float* __restrict__ ws, int S, size_t plane, bf16* __restrict__ residual, const bf16* __restrict__ w,
    bf16* __restrict__ out, int H, float eps) {
  __shared__ float red[1024 / 64];
  const size_t r0 = (size_t)blockIdx.x * H;
  f32x4_t x[V];
  bf16x4_t g[V];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int i = (threadIdx.x + k * blockDim.x) * 4;
    x[k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (i < H) {
      g[k] = *reinterpret_cast<const bf16x4_t*>(w + i);
      const bf16x4_t r = *reinterpret_cast<const bf16x4_t*>(residual + r0 + i);
      x[k] = f32x4_t{bits2f(r[0]), bits2f(r[1]), bits2f(r[2]), bits2f(r[3])};
      plane_acc4(x[k], ws + r0 + i, plane, S);  // residual first, then plane order
      const bf16x4_t h = bf16x4_t{f2bits(x[k][0]), f2bits(x[k][1]), f2bits(x[k][2]), f2bits(x[k][3])};
      *reinterpret_cast<bf16x4_t*>(residual + r0 + i) = h;
      x[k] = f32x4_t{bits2f(h[0]), bits2f(h[1]), bits2f(h[2]), bits2f(h[3])};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(x[k][e], x[k][e], ss);
  }
  ss = block_sum(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int i = (threadIdx.x + k * blockDim.x) * 4;
    if (i < H) {
      bf16x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = f2bits(x[k][e] * inv * bits2f(g[k][e]));
      *reinterpret_cast<bf16x4_t*>(out + r0 + i) = o;
    }
  }
}

template <int VPT>
__global__ __launch_bounds__(kThreads) void splitk_rmsnorm_kernel(
    const float* __restrict__ ws, int S, size_t plane, bf16* __restrict__ residual,
    const bf16* __restrict__ w, bf16* __restrict__ out, int H, float eps) {
  __shared__ float red[kThreads / 64];
  const int row = blockIdx.x;
  const int nvec = H >> 3;
  const float* hr = ws + (size_t)row * H;
  bf16x8_t* rr = reinterpret_cast<bf16x8_t*>(residual + (size_t)row * H);
  float v[VPT][8];
  float ss = 0.f;
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(w);
  bf16x8_t gv[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) gv[i] = wr[idx];
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float a[8];
      unpack8(rr[idx], a);
      if (gridDim.x <= kFewRows) {
        // a few rows (small-batch decode): latency-bound, every plane's loads in flight together (common.h
        // plane_acc4; residual first, then plane order, as the loop below)
        f32x4_t a0 = f32x4_t{a[0], a[1], a[2], a[3]}, a1 = f32x4_t{a[4], a[5], a[6], a[7]};
        plane_acc4(a0, hr + idx * 8, plane, S);
        plane_acc4(a1, hr + idx * 8 + 4, plane, S);
#pragma unroll
        for (int j = 0; j < 4; ++j) { a[j] = a0[j]; a[j + 4] = a1[j]; }
      } else {  // many rows: bandwidth-bound, no wasted plane reads (the branch-free pass: 9.3 -> 12.8 us at B176)
#pragma unroll 4
        for (int sp = 0; sp < S; ++sp) {
          const float* q = hr + sp * plane + idx * 8;
          const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(q), x1 = *reinterpret_cast<const f32x4_t*>(q + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) { a[j] += x0[j]; a[j + 4] += x1[j]; }
        }
      }
      bf16x8_t sum = pack8(a);
      rr[idx] = sum;
      unpack8(sum, a);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = a[j];
        ss += a[j] * a[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    }
  }
  ss = block_sum(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)row * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float g[8], o[8];
      unpack8(gv[i], g);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * inv * g[j];
      orow[idx] = pack8(o);
    }
  }
}

// y = LN(x [+ bias] [+ residual]) * gamma + beta.
// WRITEBACK (pre-LN decoders, GPT-2): the bf16-rounded sum x + bias + residual
// is stored back into `residual` (the residual stream) before it is
// normalised, so a pre-LN block boundary is one pass over the row:
// residual += h + b ; y = LN(residual).
//
// Rows of up to 1024 values: one wave a row and four rows a workgroup, so the two reductions are lane exchanges and
// a wave's row is in flight without a barrier (a 768-wide row left 160 of a 256-thread workgroup's lanes idle, and
// its two block sums cost four barriers).  Bound by bandwidth at 24000 rows with bias and residual: 768 wide 33.7 ->
// 18.5 us (6.0 TB/s of reads and writes, partly from the last-level cache), 384 30.2 -> 12.4, 1024 35.4 -> 22.3; at
// 1000 rows and fewer both forms are one launch's time.
template <int VPT, bool WRITEBACK>
__global__ __launch_bounds__(kThreads) void layernorm_wave_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ bias, bf16* __restrict__ residual,
    const bf16* __restrict__ gamma, const bf16* __restrict__ beta, bf16* __restrict__ out, int T, int H,
    float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (row >= T) return;
  const int nvec = H >> 3;
  const bf16x8_t* xr = reinterpret_cast<const bf16x8_t*>(x + (size_t)row * H);
  bf16x8_t* rr = residual ? reinterpret_cast<bf16x8_t*>(residual + (size_t)row * H) : nullptr;
  const bf16x8_t* br = reinterpret_cast<const bf16x8_t*>(bias);
  const bf16x8_t zero = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_t xv[VPT], rv[VPT], bv[VPT], gv[VPT], ev[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = lane + i * 64;
    xv[i] = rv[i] = bv[i] = gv[i] = ev[i] = zero;
    if (idx < nvec) {
      xv[i] = xr[idx];
      if (rr) rv[i] = rr[idx];
      if (br) bv[i] = br[idx];
      gv[i] = reinterpret_cast<const bf16x8_t*>(gamma)[idx];
      ev[i] = reinterpret_cast<const bf16x8_t*>(beta)[idx];
    }
  }
  float v[VPT][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    unpack8(xv[i], v[i]);
    float b[8], r[8];
    unpack8(bv[i], b);
    unpack8(rv[i], r);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = (v[i][j] + b[j]) + r[j];
    if (WRITEBACK) {  // the stream is bf16: normalise the rounded sum
      const bf16x8_t sum = pack8(v[i]);
      if (lane + i * 64 < nvec) rr[lane + i * 64] = sum;
      unpack8(sum, v[i]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[i][j];
  }
  const float mean = wave_sum(s) / (float)H;
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (lane + i * 64 < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = v[i][j] - mean;
        s2 += d * d;
      }
    }
  const float inv = rsqrtf(wave_sum(s2) / (float)H + eps);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)row * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (lane + i * 64 < nvec) {
      float g[8], b[8], o[8];
      unpack8(gv[i], g);
      unpack8(ev[i], b);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * inv * g[j] + b[j];
      orow[lane + i * 64] = pack8(o);
    }
}

// Wider rows: a workgroup each.
template <int VPT, bool WRITEBACK>
__global__ __launch_bounds__(kThreads) void layernorm_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ bias, bf16* __restrict__ residual,
    const bf16* __restrict__ gamma, const bf16* __restrict__ beta, bf16* __restrict__ out, int H,
    float eps) {
  __shared__ float red[kThreads / 64];
  const int row = blockIdx.x;
  const int nvec = H >> 3;
  const bf16x8_t* xr = reinterpret_cast<const bf16x8_t*>(x + (size_t)row * H);
  bf16x8_t* rr = residual ? reinterpret_cast<bf16x8_t*>(residual + (size_t)row * H) : nullptr;
  const bf16x8_t* br = bias ? reinterpret_cast<const bf16x8_t*>(bias) : nullptr;
  float v[VPT][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    if (idx < nvec) {
      unpack8(xr[idx], v[i]);
      if (br) {
        float b[8];
        unpack8(br[idx], b);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += b[j];
      }
      if (rr) {
        float b[8];
        unpack8(rr[idx], b);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += b[j];
        if (WRITEBACK) {  // the stream is bf16: normalise the rounded sum
          const bf16x8_t sum = pack8(v[i]);
          rr[idx] = sum;
          unpack8(sum, v[i]);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[i][j];
    }
  }
  const float mean = block_sum(s, red) / (float)H;
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = v[i][j] - mean;
        s2 += d * d;
      }
    }
  }
  const float inv = rsqrtf(block_sum(s2, red) / (float)H + eps);
  const bf16x8_t* gr = reinterpret_cast<const bf16x8_t*>(gamma);
  const bf16x8_t* er = reinterpret_cast<const bf16x8_t*>(beta);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)row * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float g[8], b[8], o[8];
      unpack8(gr[idx], g);
      unpack8(er[idx], b);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * inv * g[j] + b[j];
      orow[idx] = pack8(o);
    }
  }
}

// BERT embeddings: LN(word[id] + pos[p] + type[tt]).  Up to 1024 columns a wave a token, as layernorm_wave_kernel: 24000 tokens of 768
// 34.3 us in workgroups of 256 threads a token, here 18.0; from 513 columns on at 800 tokens and more, as with fewer a token's chain of two
// loads a lane is longer than the workgroup's (us, workgroups / here: 768 columns 50 / 500 / 800 / 2000 tokens 2.84 / 3.07 / 3.27 /
// 4.24 and 3.00 / 3.12 / 3.24 / 3.75, 1024 2.75 / 3.05 / 3.50 / 4.38 and 3.00 / 3.14 / 3.24 / 3.86; 384 2.82 / 2.95 / 3.16 / 3.93
// and 2.60 / 2.67 / 2.73 / 2.91).
template <int VPT>
__global__ __launch_bounds__(kThreads) void bert_embed_ln_wave_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ pos_ids,
    const int32_t* __restrict__ type_ids, const bf16* __restrict__ word,
    const bf16* __restrict__ pos, const bf16* __restrict__ type, const bf16* __restrict__ gamma,
    const bf16* __restrict__ beta, bf16* __restrict__ out, int T, int H, int V, int P, float eps) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), nvec = H >> 3;
  if (t >= T) return;
  int tid = ids[t], pid = pos_ids[t];
  if (!index_ok(tid, V, ERR_BERT_TOKEN)) tid = 0;  // reported; row 0 read instead
  if (!index_ok(pid, P, ERR_BERT_TOKEN)) pid = 0;
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(word + (size_t)tid * H);
  const bf16x8_t* pr = reinterpret_cast<const bf16x8_t*>(pos + (size_t)pid * H);
  const bf16x8_t* tr = reinterpret_cast<const bf16x8_t*>(type + (size_t)(type_ids ? type_ids[t] : 0) * H);
  const bf16x8_t zero = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_t wv[VPT], pv[VPT], tv[VPT], gv[VPT], ev[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = lane + i * 64;
    wv[i] = pv[i] = tv[i] = gv[i] = ev[i] = zero;
    if (idx < nvec) {
      wv[i] = wr[idx];
      pv[i] = pr[idx];
      tv[i] = tr[idx];
      gv[i] = reinterpret_cast<const bf16x8_t*>(gamma)[idx];
      ev[i] = reinterpret_cast<const bf16x8_t*>(beta)[idx];
    }
  }
  float v[VPT][8], s = 0.f, s2 = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    float a[8], b[8], c[8];
    unpack8(wv[i], a);
    unpack8(pv[i], b);
    unpack8(tv[i], c);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] = a[j] + b[j] + c[j];
      s += v[i][j];
    }
  }
  const float mean = wave_sum(s) / (float)H;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (lane + i * 64 < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = v[i][j] - mean;
        s2 += d * d;
      }
    }
  const float inv = rsqrtf(wave_sum(s2) / (float)H + eps);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)t * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (lane + i * 64 < nvec) {
      float g[8], b[8], o[8];
      unpack8(gv[i], g);
      unpack8(ev[i], b);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * inv * g[j] + b[j];
      orow[lane + i * 64] = pack8(o);
    }
}

// Wider rows, and few tokens of more than 512 columns: a workgroup a token.
template <int VPT>
__global__ __launch_bounds__(kThreads) void bert_embed_ln_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ pos_ids,
    const int32_t* __restrict__ type_ids, const bf16* __restrict__ word,
    const bf16* __restrict__ pos, const bf16* __restrict__ type, const bf16* __restrict__ gamma,
    const bf16* __restrict__ beta, bf16* __restrict__ out, int H, int V, int P, float eps) {
  __shared__ float red[kThreads / 64];
  const int t = blockIdx.x;
  const int nvec = H >> 3;
  int tid = ids[t], pid = pos_ids[t];
  if (!index_ok(tid, V, ERR_BERT_TOKEN)) tid = 0;  // (workgroup-uniform) reported; row 0 read instead
  if (!index_ok(pid, P, ERR_BERT_TOKEN)) pid = 0;
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(word + (size_t)tid * H);
  const bf16x8_t* pr = reinterpret_cast<const bf16x8_t*>(pos + (size_t)pid * H);
  const bf16x8_t* tr =
      reinterpret_cast<const bf16x8_t*>(type + (size_t)(type_ids ? type_ids[t] : 0) * H);
  float v[VPT][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    if (idx < nvec) {
      float a[8], b[8], c[8];
      unpack8(wr[idx], a);
      unpack8(pr[idx], b);
      unpack8(tr[idx], c);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = a[j] + b[j] + c[j];
        s += v[i][j];
      }
    }
  }
  const float mean = block_sum(s, red) / (float)H;
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = v[i][j] - mean;
        s2 += d * d;
      }
    }
  }
  const float inv = rsqrtf(block_sum(s2, red) / (float)H + eps);
  const bf16x8_t* gr = reinterpret_cast<const bf16x8_t*>(gamma);
  const bf16x8_t* er = reinterpret_cast<const bf16x8_t*>(beta);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)t * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * kThreads;
    if (idx < nvec) {
      float g[8], b[8], o[8];
      unpack8(gr[idx], g);
      unpack8(er[idx], b);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * inv * g[j] + b[j];
      orow[idx] = pack8(o);
    }
  }
}

// out[t] = table[ids[t]] — 16 B per lane, grid-stride over (token, vec).
__global__ __launch_bounds__(kThreads) void embed_gather_kernel(const int32_t* __restrict__ ids,
                                                                const bf16* __restrict__ table,
                                                                bf16* __restrict__ out, int T,
                                                                int H, int V) {
  const int nvec = H >> 3;
  const size_t total = (size_t)T * nvec;
  for (size_t i = blockIdx.x * (size_t)kThreads + threadIdx.x; i < total;
       i += (size_t)gridDim.x * kThreads) {
    const int t = (int)(i / nvec), v = (int)(i % nvec);
    int id = ids[t];
    if (!index_ok(id, V, ERR_EMBED_TOKEN)) id = 0;  // reported (ops/_lib.py raises at the next sync)
    reinterpret_cast<bf16x8_t*>(out + (size_t)t * H)[v] =
        reinterpret_cast<const bf16x8_t*>(table + (size_t)id * H)[v];
  }
}

int vpt_for(int H) {
  const int nvec = H / 8;
  if (nvec <= kThreads) return 1;
  if (nvec <= 2 * kThreads) return 2;
  if (nvec <= 4 * kThreads) return 4;
  return 8;
}

}  // namespace

GRAG_API int grag_rmsnorm(const void* x, void* residual, const void* w, void* out, int T, int H,
                          float eps, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0 || H > 8 * 8 * kThreads) return (int)hipErrorInvalidValue;
  const bf16* xp = (const bf16*)x;
  bf16* rp = (bf16*)residual;
  switch (vpt_for(H)) {
    case 1: rmsnorm_kernel<1><<<T, kThreads, 0, stream>>>(xp, rp, (const bf16*)w, (bf16*)out, H, eps); break;
    case 2: rmsnorm_kernel<2><<<T, kThreads, 0, stream>>>(xp, rp, (const bf16*)w, (bf16*)out, H, eps); break;
    case 4: rmsnorm_kernel<4><<<T, kThreads, 0, stream>>>(xp, rp, (const bf16*)w, (bf16*)out, H, eps); break;
    default: rmsnorm_kernel<8><<<T, kThreads, 0, stream>>>(xp, rp, (const bf16*)w, (bf16*)out, H, eps); break;
  }
  return (int)hipGetLastError();
}

// residual += sum_s ws[s] ; out = RMSNorm(residual) * w   (ws: S fp32 planes [T][H], 16-B aligned)
// Small batches (1-16 rows, the reference's 1-4 live sequences): splitk_rmsnorm_kernel gives a row ONE
// workgroup, which then reads all S planes of the row alone (7-9 x 14 KB at Qwen2-7B: 5.6 us at B = 1).
// Here a row is cut into 64-unit chunks (8 columns per unit), one 64-thread workgroup each: every chunk sums
// its planes into the residual (bf16, as the one-block kernel) and its share of sum(h^2); the chunk sums go
// to part_ss and an agent-scope ticket per row names the last arriving chunk (release / acquire fences as
// gemm_stream.hip), which adds the chunk sums in chunk order and normalises the whole row.  The ticket resets
// itself, so the launch replays inside hipGraphs.
__global__ __launch_bounds__(64) void splitk_rmsnorm_small_kernel(
    const float* __restrict__ ws, int S, size_t plane, bf16* __restrict__ residual, const bf16* __restrict__ w,
    bf16* __restrict__ out, int H, float eps, float* __restrict__ part_ss, unsigned* __restrict__ counters) {
  const int row = blockIdx.x, c = blockIdx.y, nch = gridDim.y;
  const int nvec = H >> 3;
  const int u = c * 64 + threadIdx.x;
  const float* hr = ws + (size_t)row * H;
  bf16x8_t* rr = reinterpret_cast<bf16x8_t*>(residual + (size_t)row * H);
  float ss = 0.f;
  if (u < nvec) {
    float a[8];
    unpack8(rr[u], a);
#pragma unroll 8
    for (int sp = 0; sp < S; ++sp) {
      const float* q = hr + sp * plane + u * 8;
      const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(q), x1 = *reinterpret_cast<const f32x4_t*>(q + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) { a[j] += x0[j]; a[j + 4] += x1[j]; }
    }
    const bf16x8_t sum = pack8(a);
    rr[u] = sum;
    unpack8(sum, a);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += a[j] * a[j];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
  __shared__ unsigned last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every lane's residual store landed before the release
  __syncthreads();
  if (threadIdx.x == 0) {
    part_ss[(size_t)row * nch + c] = ss;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned tk = __hip_atomic_fetch_add(&counters[row], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tk >= (unsigned)nch) report_index_error(ERR_TICKET, tk);  // stale / shared ticket word
    last = tk == (unsigned)(nch - 1) ? 1u : 0u;
    if (last) {
      __hip_atomic_store(&counters[row], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  __syncthreads();
  if (!last) return;
  float tot = 0.f;
  for (int k = 0; k < nch; ++k) tot += part_ss[(size_t)row * nch + k];  // chunk order: deterministic
  const float inv = rsqrtf(tot / (float)H + eps);
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(w);
  bf16x8_t* orow = reinterpret_cast<bf16x8_t*>(out + (size_t)row * H);
  for (int v = threadIdx.x; v < nvec; v += 64) {
    float a[8], g[8];
    unpack8(rr[v], a);
    unpack8(wr[v], g);
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = a[j] * inv * g[j];
    orow[v] = pack8(a);
  }
}

// Small-batch form of grag_splitk_add_rmsnorm (T <= 64 rows): part_ss >= T * ceil(H / 512) floats of scratch,
// counters >= T zero-initialised uint32 words (each reset by its last arriver).
GRAG_API int grag_splitk_add_rmsnorm_small(const void* ws, int S, void* residual, const void* w, void* out, int T,
                                           int H, float eps, float* part_ss, unsigned* counters,
                                           hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0 || S < 1 || ws == nullptr || residual == nullptr || !part_ss || !counters || T > 64)
    return (int)hipErrorInvalidValue;
  const int nch = (H / 8 + 63) / 64;
  splitk_rmsnorm_small_kernel<<<dim3(T, nch), 64, 0, stream>>>((const float*)ws, S, (size_t)T * H, (bf16*)residual,
                                                              (const bf16*)w, (bf16*)out, H, eps, part_ss, counters);
  return (int)hipGetLastError();
}

GRAG_API int grag_splitk_add_rmsnorm(const void* ws, int S, void* residual, const void* w, void* out, int T,
                                     int H, float eps, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0 || H > 8 * 8 * kThreads || S < 1 || ws == nullptr || residual == nullptr)
    return (int)hipErrorInvalidValue;
  const size_t plane = (size_t)T * H;
  const float* wp = (const float*)ws;
  bf16* rp = (bf16*)residual;
  // The general form has a row of up to 2048 in flight as well, and past 8 planes (walked as 12 and 16) with fewer registers: us
  // there / here at 512-2048 wide, 1-256 rows: 2-8 planes 2.4-5.1 / 1.9-5.0, 9-16 planes 2.6-7.4 / 2.9-7.7 (up to 16 rows of 16
  // planes 4.6 / 3.7); wider it is never ahead (2304: 2 planes 3.1-3.8 / 2.2-2.8, 16 planes 8.7-13.2 / 3.7-8.2)
  if (T <= kWideRows && H <= 8192 && (H > 2048 || S <= 8)) {
    const int units = H / 4, V = units > 1024 ? 2 : 1, threads = ((units + V - 1) / V + 63) / 64 * 64;
    if (V == 1) splitk_rmsnorm_wide_kernel<1><<<T, threads, 0, stream>>>(wp, S, plane, rp, (const bf16*)w, (bf16*)out, H, eps);
    else splitk_rmsnorm_wide_kernel<2><<<T, threads, 0, stream>>>(wp, S, plane, rp, (const bf16*)w, (bf16*)out, H, eps);
    return (int)hipGetLastError();
  }
#define SRN(V) splitk_rmsnorm_kernel<V><<<T, kThreads, 0, stream>>>(wp, S, plane, rp, (const bf16*)w, (bf16*)out, H, eps)
  switch (vpt_for(H)) {
    case 1: SRN(1); break;
    case 2: SRN(2); break;
    case 4: SRN(4); break;
    default: SRN(8); break;
  }
#undef SRN
  return (int)hipGetLastError();
}

template <bool WB>
static int launch_layernorm(const void* x, const void* bias, void* residual, const void* gamma,
                            const void* beta, void* out, int T, int H, float eps,
                            hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0 || H > 8 * 8 * kThreads) return (int)hipErrorInvalidValue;
  constexpr int rows = kThreads / 64;
  auto wave = [&](auto kern) {
    kern<<<(T + rows - 1) / rows, kThreads, 0, stream>>>((const bf16*)x, (const bf16*)bias, (bf16*)residual,
                                                         (const bf16*)gamma, (const bf16*)beta, (bf16*)out, T, H, eps);
    return (int)hipGetLastError();
  };
  if (H <= 512) return wave(layernorm_wave_kernel<1, WB>);
  if (H <= 1024) return wave(layernorm_wave_kernel<2, WB>);
  auto args = [&](auto kern) {
    kern<<<T, kThreads, 0, stream>>>((const bf16*)x, (const bf16*)bias, (bf16*)residual,
                                     (const bf16*)gamma, (const bf16*)beta, (bf16*)out, H, eps);
  };
  switch (vpt_for(H)) {
    case 1: args(layernorm_kernel<1, WB>); break;
    case 2: args(layernorm_kernel<2, WB>); break;
    case 4: args(layernorm_kernel<4, WB>); break;
    default: args(layernorm_kernel<8, WB>); break;
  }
  return (int)hipGetLastError();
}

GRAG_API int grag_layernorm(const void* x, const void* bias, const void* residual,
                            const void* gamma, const void* beta, void* out, int T, int H,
                            float eps, hipStream_t stream) {
  return launch_layernorm<false>(x, bias, const_cast<void*>(residual), gamma, beta, out, T, H, eps,
                                 stream);
}

// Pre-LN block boundary: residual += x (+ bias), out = LN(residual).
GRAG_API int grag_add_layernorm(const void* x, const void* bias, void* residual,
                                const void* gamma, const void* beta, void* out, int T, int H,
                                float eps, hipStream_t stream) {
  if (residual == nullptr) return (int)hipErrorInvalidValue;
  return launch_layernorm<true>(x, bias, residual, gamma, beta, out, T, H, eps, stream);
}

GRAG_API int grag_bert_embed_ln(const int32_t* ids, const int32_t* pos_ids,
                                const int32_t* type_ids, const void* word, const void* pos,
                                const void* type, const void* gamma, const void* beta, void* out,
                                int T, int H, int V, int P, float eps, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0 || H > 8 * 8 * kThreads) return (int)hipErrorInvalidValue;
  constexpr int rows = kThreads / 64;
  auto wave = [&](auto kern) {
    kern<<<(T + rows - 1) / rows, kThreads, 0, stream>>>(ids, pos_ids, type_ids, (const bf16*)word, (const bf16*)pos, (const bf16*)type,
                                                         (const bf16*)gamma, (const bf16*)beta, (bf16*)out, T, H, V, P, eps);
    return (int)hipGetLastError();
  };
  if (H <= 512) return wave(bert_embed_ln_wave_kernel<1>);
  if (H <= 1024 && T >= 800) return wave(bert_embed_ln_wave_kernel<2>);
  auto args = [&](auto kern) {
    kern<<<T, kThreads, 0, stream>>>(ids, pos_ids, type_ids, (const bf16*)word, (const bf16*)pos,
                                     (const bf16*)type, (const bf16*)gamma, (const bf16*)beta,
                                     (bf16*)out, H, V, P, eps);
  };
  switch (vpt_for(H)) {
    case 1: args(bert_embed_ln_kernel<1>); break;
    case 2: args(bert_embed_ln_kernel<2>); break;
    case 4: args(bert_embed_ln_kernel<4>); break;
    default: args(bert_embed_ln_kernel<8>); break;
  }
  return (int)hipGetLastError();
}

GRAG_API int grag_embed_gather(const int32_t* ids, const void* table, void* out, int T, int H, int V,
                               hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 != 0) return (int)hipErrorInvalidValue;
  const size_t total = (size_t)T * (H / 8);
  int grid = (int)((total + kThreads - 1) / kThreads);
  if (grid > 4096) grid = 4096;
  embed_gather_kernel<<<grid, kThreads, 0, stream>>>(ids, (const bf16*)table, (bf16*)out, T, H, V);
  return (int)hipGetLastError();
}

GRAG_ERR_UNIT(norm)

// The index guard's error block (common.h): pinned, device-mapped, coherent host memory, so a kernel's
// report is visible to the host without a copy.  Returns the host address (nullptr when no device);
// *dev_out receives the device address every unit's grag_err_bind_* takes.
GRAG_API void* grag_err_alloc(void** dev_out) {
  void* h = nullptr;
  if (hipHostMalloc(&h, 256, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) return nullptr;
  memset(h, 0, 256);
  void* d = nullptr;
  if (hipHostGetDevicePointer(&d, h, 0) != hipSuccess) d = h;
  *dev_out = d;
  return h;
}
