// Decode attention of the hybrid decoders on the matrix cores (gfx950): one new token per sequence over the paged cache, with
// what grag_sink_attn_decode describes (sink logit, block or window, cap, temperature, output gate; no kept keys).  Head size
// D = 64 or 128 for keys and values alike, 16-key cache blocks; other calls take the kernel of seqmix.hip.
//
// A workgroup is a part of a sequence's keys for one kv head (and up to 16 of its query heads); wave w walks its tiles of 32 keys
// w, w + NW, ... by itself, without a barrier.  K goes from memory to the registers as the operand of S^T = K Q^T, one tile
// ahead; V by LDS-DMA into the wave's own two buffers and out of them by transposed reads.  Weights are fp32, bf16 hi + lo in
// the second product.  The waves' sums meet in LDS once, at the end.
// Bound by the bytes in flight: 64 sequences of 70000 keys in all, 28 / 4 heads of 128, parts of 512 keys, 42 us with the
// combination (143 MB; 5 us of it the second launch), 82 in the staged 64-key tiles of four waves in step; 12 / 2 heads 45 ->
// 25; 16 / 4 heads of 64 33 -> 21; 128 sequences of 130000 128 -> 67; one of 4000 28 -> 13.  With the compiler's LDS-DMA builtin
// it drained every load before the transposed reads: 54.
#include "sink.h"

GRAG_ERR_UNIT(sink_decode)

namespace grag {

constexpr int SD_KT = 32;  // keys per tile

struct SinkDecodeArgs {
  SinkArgs a;
  int nsplit, split_len;
  float *part_o, *part_ml;
};

// One LDS-DMA instruction: 16 bytes a lane from `src` into the 1 KB of LDS at the wave-uniform `dst`, lane after lane.  As asm
// the compiler does not count it, so that it neither drains the vector memory counter before the transposed reads of the other
// buffer nor reckons with it in its waits for the K registers; the waits below do.
__device__ __forceinline__ void sd_dma(const void* src, char* dst) {
  const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)dst);
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(src), "s"(lds)
      : "memory");
}

template <int D, int NW, bool CAP>
__global__ void __launch_bounds__(64 * NW, D == 64 ? 4 : 2) sink_decode_kernel(const SinkDecodeArgs pa) {
  const SinkArgs& p = pa.a;
  constexpr int RB = 2 * D, CPR = D / 8, NC = D / 32, ND = D / 16, VT = SD_KT * RB;  // VT: bytes of a V tile
  constexpr int NI = VT / 1024, RPI = 1024 / RB;                                     // DMA pieces of a tile, rows of a piece
  __shared__ __attribute__((aligned(16))) char smem[NW * 2 * VT];
  __shared__ float wm[NW][16], wl[NW][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h4 = lane >> 4, li = lane & 15;
  const int R = p.R, ngrp = (R + 15) >> 4;
  const int sp = blockIdx.x, g = blockIdx.y / ngrp, hg = (blockIdx.y - g * ngrp) * 16, seq = blockIdx.z, nseq = gridDim.z;
  const int ctx = p.ctx_len[seq];
  const bool valid = hg + li < R;
  const int head = g * R + (valid ? hg + li : 0);
  const int low = sp_first(p, ctx - 1);  // the first key in sight
  const int hi = pa.nsplit > 1 ? min(ctx, (sp + 1) * pa.split_len) : ctx;
  const int lo = max(pa.nsplit > 1 ? sp * pa.split_len : 0, low & ~(SP_BS - 1));
  const int ntiles = hi > lo ? (hi - lo + SD_KT - 1) / SD_KT : 0;

  const float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;
  const float sc = p.scale * (p.hscale ? p.hscale[head] : 1.f);
  const bool sink = sp == 0 && wave == 0;
  float m = sink ? p.sinks[head] * LOG2E : -INFINITY, lsum = sink && h4 == 0 ? 1.f : 0.f;
  f32x4_t o[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  if (wave < ntiles) {
    bf16x8_t qf[NC];
    const bf16* qp = p.q + ((size_t)seq * p.H + head) * D + 8 * h4;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      qf[c] = valid ? *reinterpret_cast<const bf16x8_t*>(qp + 32 * c) : bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
    const int* bt = p.bt + (size_t)seq * p.bt_stride;
    const int last = (hi - 1) / SP_BS, last_slot = (hi - 1) % SP_BS;
    int base = 0, bvec = 0;  // 64 entries of the block table, one a lane: 1024 keys
    auto block = [&](int i) __attribute__((always_inline)) { return __builtin_amdgcn_readlane(bvec, min(i, last) - base); };
    const int vrow = lane / CPR, vch = lane % CPR;
    char* vbuf = smem + wave * 2 * VT;
    bf16x8_t kf[2][2][NC];
    auto at = [&](int kt0, int tt) __attribute__((always_inline)) {
      return ((size_t)block((kt0 + 16 * tt) / SP_BS) * p.G + g) * SP_BS * D;
    };
    // K of tile t into register set `st`, V into buffer `st`.  Keys past the last one re-read it (their weights are 0, and 0
    // times whatever lies there must be 0).
    auto load_k = [&](int t, auto st) __attribute__((always_inline)) {
      constexpr int S = decltype(st)::value;
      const int kt0 = lo + t * SD_KT;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const bf16* kp = p.k + at(kt0, tt) + (kt0 + 16 * tt + li < hi ? li : last_slot) * D + 8 * h4;
#pragma unroll
        for (int c = 0; c < NC; ++c) kf[S][tt][c] = *reinterpret_cast<const bf16x8_t*>(kp + 32 * c);
      }
    };
    auto load_v = [&](int t, auto st) __attribute__((always_inline)) {
      constexpr int S = decltype(st)::value;
      const int kt0 = lo + t * SD_KT;
      const size_t a[2] = {at(kt0, 0), at(kt0, 1)};
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = i * RPI + vrow, slot = kt0 + r < hi ? r % SP_BS : last_slot;
        sd_dma(p.v + a[i * RPI / SP_BS] + slot * D + ((vch ^ sp_vswz<D>(r)) << 3), vbuf + S * VT + i * 1024);
      }
    };
    auto tile = [&](int t, auto st, auto more) __attribute__((always_inline)) {
      constexpr int S = decltype(st)::value;
      const int kt0 = lo + t * SD_KT;
      f32x4_t s[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        s[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[S][tt][c], qf[c], s[tt], 0, 0, 0);
      }
      if constexpr (CAP) {  // cap in the natural domain, then to log2
        const float ic = 1.f / p.softcap, c2 = p.softcap * LOG2E;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[tt][r] = c2 * tanhf(s[tt][r] * sc * ic);
      } else {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) s[tt] *= sc * LOG2E;
      }
      if (kt0 + SD_KT > hi || kt0 < low) {
        asm volatile("");
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = kt0 + 16 * tt + 4 * h4 + r;
            s[tt][r] = key < hi && key >= low ? s[tt][r] : -INFINITY;
          }
      }
      float cand = m;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) cand = fmaxf(cand, s[tt][r]);
      cand = fmaxf(cand, __shfl_xor(cand, 16, 64));
      cand = fmaxf(cand, __shfl_xor(cand, 32, 64));
      if (__any(cand > m + SP_RESCALE)) {  // (a first key in sight: from -inf)
        const float alpha = cand == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - cand);
        m = cand;
        lsum *= alpha;
#pragma unroll
        for (int n = 0; n < ND; ++n) o[n] *= alpha;
      }
      const float mm = m == -INFINITY ? 0.f : m;
      bf16x8_t ph, pl;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = __builtin_amdgcn_exp2f(s[tt][r] - mm);
          const short b = f2bits(x);
          ph[4 * tt + r] = b;
          pl[4 * tt + r] = f2bits(x - bits2f(b));
          lsum += x;
        }
      // K and V of this tile have landed (loads do in issue order): behind them at least the 2 NC loads of the next tile's K are
      // under way, which no load passes (the asm clobbers memory); more of them, a spill's say, would only wait for longer.  And
      // the reads of the tile before have returned from the buffer that is filled now.
      if constexpr (decltype(more)::value) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * NC) : "memory");
        load_v(t + NW, std::integral_constant<int, 1 - S>{});
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      const char* v_lds = vbuf + S * VT;
      const int r0 = 4 * h4 + (li >> 2), r1 = r0 + 16, tp = li & 3;
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const int unit = 4 * n + tp;
        const bf16x4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (sp_lds4_t*)(v_lds + r0 * RB + ((unit ^ (sp_vswz<D>(r0) << 1)) << 3)));
        const bf16x4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (sp_lds4_t*)(v_lds + r1 * RB + ((unit ^ (sp_vswz<D>(r1) << 1)) << 3)));
        const bf16x8_t a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pl, o[n], 0, 0, 0);
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ph, o[n], 0, 0, 0);
      }
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    const std::true_type more{};
    const std::false_type end{};
    for (int w0 = 0; w0 < ntiles; w0 += 32) {  // the tiles of 64 entries
      const int stop = min(ntiles, w0 + 32);
      int t = w0 + wave;
      if (t >= stop) break;
      base = (lo + w0 * SD_KT) / SP_BS;
      bvec = bt[min(base + lane, last)];
      if (!index_ok(bvec, p.nblocks, ERR_BLOCK_DECODE)) bvec = 0;  // reported; block 0 read instead of faulting
      __builtin_amdgcn_s_waitcnt(0x0F70);                          // vmcnt(0): q and the table
      load_k(t, S0{});
      load_v(t, S0{});
      while (true) {  // one tile ahead: K before this tile's scores, V after them
        if (t + NW >= stop) {
          tile(t, S0{}, end);
          break;
        }
        load_k(t + NW, S1{});
        tile(t, S0{}, more);
        t += NW;
        if (t + NW >= stop) {
          tile(t, S1{}, end);
          break;
        }
        load_k(t + NW, S0{});
        tile(t, S1{}, more);
        t += NW;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (h4 == 0) {
    wm[wave][li] = m;
    wl[wave][li] = lsum;
  }
  // the wave's sums in its own V buffers, [head][D]; a row's 16-byte chunks turned by the row
  float* ow = reinterpret_cast<float*>(smem + wave * 2 * VT);
#pragma unroll
  for (int n = 0; n < ND; ++n) *reinterpret_cast<f32x4_t*>(ow + li * D + (((4 * n + h4) ^ (li & 7)) << 2)) = o[n];
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * D / 4; i += 64 * NW) {  // four values of a head a thread
    const int h = i / (D / 4), c = i % (D / 4);
    if (hg + h >= R) continue;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, wm[w][h]);
    f32x4_t v = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = wm[w][h] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(wm[w][h] - M);
      L = fmaf(wl[w][h], f, L);
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(smem + w * 2 * VT) + h * D +
                                                          ((c ^ (h & 7)) << 2));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(x[e], f, v[e]);
    }
    const int hd = g * R + hg + h;
    if (pa.nsplit > 1) {
      const size_t row = ((size_t)sp * nseq + seq) * p.H + hd;
      *reinterpret_cast<f32x4_t*>(pa.part_o + row * D + 4 * c) = v;
      if (c == 0) {
        pa.part_ml[row * 2] = M * LN2;
        pa.part_ml[row * 2 + 1] = L;
      }
    } else {
      float r = p.out_scale / L;
      if (p.hgate) r /= 1.f + expf(-(float)p.hgate[(size_t)seq * p.gate_ld + hd]);
      *reinterpret_cast<bf16x4_t*>(p.out + (size_t)seq * p.out_ld + (size_t)hd * D + 4 * c) =
          bf16x4_t{f2bits(v[0] * r), f2bits(v[1] * r), f2bits(v[2] * r), f2bits(v[3] * r)};
    }
  }
}

// Whether the kernel takes a call; grag_sink_attn_decode (seqmix.hip) asks before it launches.
bool sink_decode_takes(int d, int vd, int v_ld, int BS, int keep, const void* q, const void* k, const void* v, const void* out,
                       int out_ld) {
  if ((d != 64 && d != 128) || vd != d || v_ld != d || BS != SP_BS || keep > 0 || out_ld % 4) return false;
  return (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0 && ((uintptr_t)out & 7) == 0;
}

hipError_t sink_decode_launch(const void* q, const void* k, const void* v, void* out, int out_ld, const int* bt, int bt_stride,
                              const int* ctx_len, const float* sinks, int nseq, int H, int G, int d, float scale, float out_scale,
                              int nblocks, int nsplit, int split_len, float* part_o, float* part_ml, const float* hscale,
                              const void* hgate, int gate_ld, int chunk, int window, float softcap, hipStream_t st) {
  SinkDecodeArgs pa{};
  SinkArgs& a = pa.a;
  a.q = (const bf16*)q, a.k = (const bf16*)k, a.v = (const bf16*)v, a.out = (bf16*)out;
  a.bt = bt, a.ctx_len = ctx_len, a.sinks = sinks, a.hscale = hscale, a.hgate = (const bf16*)hgate;
  a.out_ld = out_ld, a.bt_stride = bt_stride, a.H = H, a.G = G, a.R = H / G, a.nblocks = nblocks;
  a.gate_ld = gate_ld, a.chunk = chunk, a.window = window;
  a.scale = scale, a.out_scale = out_scale, a.softcap = softcap;
  pa.nsplit = nsplit, pa.split_len = split_len, pa.part_o = part_o, pa.part_ml = part_ml;
  const dim3 grid(nsplit, G * ((a.R + 15) / 16), nseq);
  // four waves where the parts are few, two where they fill the chip anyway (and a smaller unit fills it more evenly): 448 parts
  // of 256 keys 15.5 us with four, 15.8 with two; 1024 of 512 44.5 / 42.2; 16 of 256 13.2 / 14.1
  const bool few = (long)nsplit * G * ((a.R + 15) / 16) * nseq < 512;
#define SINK_DECODE_W(DD, CAP, NW) hipLaunchKernelGGL((sink_decode_kernel<DD, NW, CAP>), grid, dim3(64 * NW), 0, st, pa)
#define SINK_DECODE(DD, CAP)              \
  {                                       \
    if (few) SINK_DECODE_W(DD, CAP, 4);   \
    else SINK_DECODE_W(DD, CAP, 2);       \
  }
  if (d == 64 && softcap > 0.f) SINK_DECODE(64, true)
  else if (d == 64) SINK_DECODE(64, false)
  else if (softcap > 0.f) SINK_DECODE(128, true)
  else SINK_DECODE(128, false)
#undef SINK_DECODE
#undef SINK_DECODE_W
  return hipGetLastError();
}

}  // namespace grag
