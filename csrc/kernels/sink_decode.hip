// Decode attention of the hybrid decoders on the matrix cores (gfx950): one new token per sequence over the paged cache, with
// what grag_sink_attn_decode describes (sink logit, block or window, cap, temperature, output gate; no kept keys).  Head size
// D = 64 or 128 for keys and values alike, 16-key cache blocks; other calls take the kernel of seqmix.hip.
//
// A workgroup is a part of a sequence's keys for one kv head (and up to 16 of its query heads); wave w walks its tiles of 32 keys
// w, w + NW, ... by itself, without a barrier, its loads ahead in a ring of its own (decode_loads.h).  Weights are fp32, bf16 hi +
// lo in the second product.  The waves' sums meet in LDS once, at the end.
// Bound by the bytes in flight and the chain of a wave's tiles.  us with the combination (5 of them the second launch), before, with
// K from memory to the registers (64 bytes a row and instruction, which non-temporal loads tore: 42.9) -> now: 64 sequences of
// 70000 keys in all, 28 / 4 heads of 128, parts of 512 keys (143 MB) 42.4 -> 36.1, 128 of 130000 70.3 -> 60.9, window 1024 of these
// 25.3 -> 21.8 and 46.4 -> 40.3; 12 / 2 heads 128 of 130000 42.0 -> 36.6.
#include "decode_loads.h"
#include "sink.h"

GRAG_ERR_UNIT(sink_decode)

namespace grag {

constexpr int SD_KT = 32;  // keys per tile

struct SinkDecodeArgs {
  SinkArgs a;
  int nsplit, split_len;
  float *part_o, *part_ml;
};

template <int D, int NW, bool CAP>
__global__ void __launch_bounds__(64 * NW) sink_decode_kernel(const SinkDecodeArgs pa) {
  const SinkArgs& p = pa.a;
  constexpr int RB = 2 * D, NC = D / 32, ND = D / 16, NS = 2, TILE = SD_KT * RB, RING = NS * 2 * TILE;
  __shared__ __attribute__((aligned(16))) char smem[NW * RING];
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
    const int first = lo + wave * SD_KT, step = NW * SD_KT, n = (ntiles - wave + NW - 1) / NW;
    DecodeLoads<D, SD_KT, NS, true> ld(p.k, p.v, p.bt + (size_t)seq * p.bt_stride, SP_BS, p.G, p.nblocks, g, hi, hi - 1, first,
                                       smem + wave * RING);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): q and the table, so that the compiler waits for none of them in the loop
#pragma unroll
    for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(qf[c]));
    asm volatile("" : "+v"(ld.bvec));
    ld.start(first, step, n);
    for (int t = 0; t < n; ++t) {
      const int kt0 = first + t * step, stage = t & 1;
      const char *k_lds = ld.ring + stage * 2 * TILE, *v_lds = k_lds + TILE;
      ld.wait_left(2 * (n - t) - 1);
      bf16x8_t kf[2][NC];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          kf[tt][c] = *reinterpret_cast<const bf16x8_t*>(k_lds + (16 * tt + li) * RB + (((4 * c + h4) ^ kswz<D>(16 * tt + li)) << 4));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the keys are in registers
      if (t + NS < n) ld.issue_k(kt0 + NS * step, stage);
      f32x4_t s[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        s[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[tt][c], qf[c], s[tt], 0, 0, 0);
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
        for (int n2 = 0; n2 < ND; ++n2) o[n2] *= alpha;
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
      ld.wait_left(2 * (n - t) - 2);
      const int r0 = 4 * h4 + (li >> 2), r1 = r0 + 16, tp = li & 3;
      bf16x8_t vf[ND];
#pragma unroll
      for (int n2 = 0; n2 < ND; ++n2) {
        const int unit = 4 * n2 + tp;
        const bf16x4_t a0 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((sp_lds4_t*)(v_lds + r0 * RB + ((unit ^ (vswz<D>(r0) << 1)) << 3)));
        const bf16x4_t a1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((sp_lds4_t*)(v_lds + r1 * RB + ((unit ^ (vswz<D>(r1) << 1)) << 3)));
        vf[n2] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the values are in registers
      if (t + NS < n) ld.issue_v(stage);
#pragma unroll
      for (int n2 = 0; n2 < ND; ++n2) {
        o[n2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[n2], pl, o[n2], 0, 0, 0);
        o[n2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[n2], ph, o[n2], 0, 0, 0);
      }
    }
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (h4 == 0) {
    wm[wave][li] = m;
    wl[wave][li] = lsum;
  }
  // the wave's sums in its own buffers, [head][D]; a row's 16-byte chunks turned by the row
  float* ow = reinterpret_cast<float*>(smem + wave * RING);
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
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(smem + w * RING) + h * D +
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

// Waves a part: few parts are each a chain of tiles to be shared, many fill the chip by themselves; a wave's ring is 32 KB of LDS for
// heads of 128 and 16 for heads of 64, so the lines lie where the parts of 4 waves, of 2 no longer have a place at once (heads of 64:
// at twice as many parts).  us of 1 / 2 / 4 waves, cold keys, parts of keys: heads of
// 128 1024 of 512 36.5 / 40.1 / 45.4, 640 of 256 20.5 / 23.6 / 24.9, 384 of 256 20.0 / 16.9 / 19.3, 332 of 20 7.0 / 5.8 / 8.8, 32 of 128 13.8 /
// 11.5 / 10.8; heads of 64 1328 of 512 29.4 / 30.6 / 29.9, 1024 of 900 34.6 / 33.7 / 36.5, 768 of 256 15.0 / 13.3 / 13.4.
static int sink_decode_waves(int D, long parts) {
  const double places = (double)device_cus() * 128 / D;
  return parts > 2.35 * places ? 1 : parts > 1.1 * places ? 2 : 4;
}
GRAG_API int grag_sink_decode_waves(int D, long parts) { return D < 1 ? -1 : sink_decode_waves(D, parts); }  // (for tests)

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
  const long parts = (long)nsplit * G * ((a.R + 15) / 16) * nseq;
  const int waves = sink_decode_waves(d, parts);
#define SINK_DECODE_W(DD, CAP, NW) hipLaunchKernelGGL((sink_decode_kernel<DD, NW, CAP>), grid, dim3(64 * NW), 0, st, pa)
#define SINK_DECODE(DD, CAP)                        \
  {                                                 \
    if (waves == 1) SINK_DECODE_W(DD, CAP, 1);      \
    else if (waves == 2) SINK_DECODE_W(DD, CAP, 2); \
    else SINK_DECODE_W(DD, CAP, 4);                 \
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
