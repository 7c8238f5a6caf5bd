// Prefill attention of the hybrid decoders on the matrix cores (gfx950): causal softmax over the paged cache with a sink logit
// per head, aligned blocks or a sliding window with kept first keys, a score cap, a temperature and an output gate per head
// (grag_sink_attn_prefill says what each does).  Head size D = 64 or 128 for keys and values alike, 16-key cache blocks; other
// sizes take the kernel of seqmix.hip.
//
// Rows are (position, query head) pairs of one kv head, R heads to a position: a workgroup is 8 waves of 16 rows, 128 rows on one
// stream of K / V tiles (the other kernel reads every tile for 64 rows of one head).  Tiles of 64 keys arrive by LDS-DMA, the
// next one in flight while one is computed.  Per tile
//   S^T = K Q^T          bf16 products, exact in fp32,
//   P = 2^(s - m)        fp32; m moves only when a row's scores pass it by 2^8 (its factor is exact then),
//   O^T += V^T P^T       P as bf16 hi + lo, two products: 16 bits of the weights reach the accumulator.
// What bounds it: matrix cores 36 % and vector instructions 46 % of all cycles at window 1024, 2 portions of 8192 tokens, 28 / 4
// heads of 128 (the split is 1.5 times the products of a kernel with 16-bit weights).  Two workgroups share a CU, so that one's
// softmax can meet the other's products.  Tried at that size, us: 128 rows x 2 208; one workgroup of 256 rows, 8 waves of 32
// rows in step 221, half a tile apart 225, 16 waves 223; 128 rows by 4 waves of 32 rows 200, but 49 against 43 on a
// prompt of 1187 tokens, 12 / 2 heads.  Measured, old -> new: window 345 -> 208 us, all keys 811 -> 479, blocks of 1024
// 214 -> 141, 1 x 8192 tokens of all keys 1466 -> 714; 12 / 2 heads, 1 x 1187 tokens 75 -> 43.
#include "sink.h"

GRAG_ERR_UNIT(sink_prefill)

namespace grag {

constexpr int SP_KT = 64;         // keys per tile
constexpr int SP_MAXB = 2048;     // cache blocks a workgroup can walk (32 K keys): its part of the block table, in LDS

template <int D, bool CAP, int NW>
__global__ void __launch_bounds__(64 * NW, 4) sink_prefill_kernel(const SinkArgs p) {
  constexpr int RB = 2 * D, CPR = D / 8, NC = D / 32, ND = D / 16, TILE = SP_KT * RB;
  constexpr int ROWS = 16 * NW, PPW = TILE / 1024 / NW, RPP = 1024 / RB;
  static_assert(PPW >= 1 && SP_BS % (PPW * RPP) == 0, "a wave's DMA rows sit in one cache block");
  __shared__ __attribute__((aligned(16))) char smem[2 * 2 * TILE];
  __shared__ int bt_lds[SP_MAXB];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h4 = lane >> 4, li = lane & 15;
  const int seq = blockIdx.x / p.tiles, kvh = blockIdx.y;
  const int row_base = (p.tiles - 1 - (int)(blockIdx.x % p.tiles)) * ROWS;  // (the longest walks first)
  const int q0 = p.q_start[seq], qlen = p.q_start[seq + 1] - q0, ctx = p.ctx_len[seq], pos0 = ctx - qlen;
  const int R = p.R, nrows = qlen * R;
  if (row_base >= nrows) return;
  const int last_row = min(row_base + ROWS, nrows) - 1;
  const int kv_hi = min(ctx, pos0 + last_row / R + 1);
  // tiles: nkeep of kept keys, then those from the first key that any row sees.  Table entry i of the walk is cache block i, or
  // i + skip behind the kept ones.
  const int kfirst = sp_first(p, pos0 + row_base / R) & ~(SP_KT - 1);
  const int nkeep = min((p.keep + SP_KT - 1) / SP_KT, kfirst / SP_KT);
  const int ntiles = nkeep + (kv_hi - kfirst + SP_KT - 1) / SP_KT;
  const int kb = nkeep * (SP_KT / SP_BS), skip = kfirst / SP_BS - kb;
  const int nb = min((kv_hi + SP_BS - 1) / SP_BS - skip, SP_MAXB);
  const int* bt = p.bt + (size_t)seq * p.bt_stride;
  for (int i = threadIdx.x; i < nb; i += 64 * NW) {
    int b = bt[i < kb ? i : i + skip];
    if (!index_ok(b, p.nblocks, ERR_BLOCK_PREFILL)) b = 0;  // reported; block 0 read instead of faulting
    bt_lds[i] = b;
  }
  auto start = [&](int t) { return t < nkeep ? t * SP_KT : kfirst + (t - nkeep) * SP_KT; };

  // this lane's row
  const float LOG2E = 1.4426950408889634f;
  const int row = row_base + wave * 16 + li;
  const bool valid = row < nrows;
  const int pq = valid ? row / R : 0;
  const int head = kvh * R + (valid ? row - pq * R : 0), tok = q0 + pq;
  const int lim = valid ? min(kv_hi, pos0 + pq + 1) : 0, low = sp_first(p, pos0 + pq);
  const float sc = p.scale * (p.hscale ? p.hscale[head] : 1.f);
  const bool pre = p.hscale || !(p.scale > 0.f);  // scores scaled before the mask and the maximum, else in the exponent's fma
  float m = p.sinks[head] * LOG2E, lsum = h4 == 0 ? 1.f : 0.f;  // the maximum starts at the sink, whose weight is 1 of the sum
  bf16x8_t qf[NC];
  const bf16* qp = p.q + ((size_t)tok * p.H + head) * D + 8 * h4;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    qf[c] = valid ? *reinterpret_cast<const bf16x8_t*>(qp + 32 * c) : bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  // (a compiler-visible wait: the q loads retired, so that the loop needs no vmcnt of its own that would drain the DMA)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();  // the table is there
  // of the wave's rows, the smallest and largest limit and first key
  const int w0 = row_base + wave * 16, w1 = min(w0 + 16, nrows) - 1;
  const int p0 = pos0 + min(w0, nrows - 1) / R, p1 = pos0 + max(w1, 0) / R;
  const int lim_min = w0 + 16 <= nrows ? min(kv_hi, p0 + 1) : 0, lim_max = w0 < nrows ? min(kv_hi, p1 + 1) : 0;
  const int low_min = sp_first(p, p0), low_max = sp_first(p, p1);

  const int lrow = lane / CPR, lch = lane % CPR;
  const int wrow = wave * PPW * RPP, last_slot = (kv_hi - 1) % SP_BS;
  auto issue = [&](int t, int stage) {
    char* kdst = smem + stage * 2 * TILE;
    const int blk = __builtin_amdgcn_readfirstlane(bt_lds[min(t * (SP_KT / SP_BS) + wrow / SP_BS, nb - 1)]);
    const size_t base = ((size_t)blk * p.G + kvh) * SP_BS * D;
    const int kt0 = start(t);
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      const int piece = wave * PPW + i, kr = piece * RPP + lrow;
      // keys past the last one re-read it (their weights are 0, and 0 times whatever lies there must be 0)
      const int slot = kt0 + kr < kv_hi ? kr % SP_BS : last_slot;
      sp_dma(p.k + base, SP_BS * RB, slot * RB + ((lch ^ sp_kswz<D>(kr)) << 4), kdst + piece * 1024);
      sp_dma(p.v + base, SP_BS * RB, slot * RB + ((lch ^ sp_vswz<D>(kr)) << 4), kdst + TILE + piece * 1024);
    }
  };
  f32x4_t o[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bf16x8_t ph[2], pl[2];  // the weights of 32 keys: a lane's row, keys 4 h4 + 0..3 and 16 + 4 h4 + 0..3

  auto scores = [&](int kt0, const char* k_lds) {
    f32x4_t s[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      const int kr = 16 * tt + li;
      s[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c)
        s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8_t*>(k_lds + kr * RB + (((4 * c + h4) ^ sp_kswz<D>(kr)) << 4)), qf[c], s[tt], 0, 0, 0);
    }
    if constexpr (CAP) {  // cap in the natural domain, then to log2
      const float ic = 1.f / p.softcap, c2 = p.softcap * LOG2E;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[tt][r] = c2 * tanhf(s[tt][r] * sc * ic);
    } else if (pre) {  // (a factor of 0 or less: it turns the order, and makes no 0 of a masked score)
      asm volatile("");
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) s[tt] *= sc * LOG2E;
    }
    // a real branch (the empty asm): as selects, the masks would cost every tile what only the edges need
    if (kt0 + SP_KT > lim_min || (kt0 < low_max && kt0 + SP_KT > p.keep)) {
      asm volatile("");
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = kt0 + 16 * tt + 4 * h4 + r;
          s[tt][r] = key < lim && (key >= low || key < p.keep) ? s[tt][r] : -INFINITY;
        }
    }
    const float f = CAP || pre ? 1.f : p.scale * LOG2E;
    float tmax = -INFINITY;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[tt][r]);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float cand = fmaxf(m, tmax * f);
    if (__any(cand > m + SP_RESCALE)) {  // every row takes its exact maximum, so o and lsum see one factor
      const float alpha = __builtin_amdgcn_exp2f(m - cand);
      m = cand;
      lsum *= alpha;
#pragma unroll
      for (int n = 0; n < ND; ++n) o[n] *= alpha;
    }
    float sum = 0.f;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = __builtin_amdgcn_exp2f(fmaf(s[tt][r], f, -m));
        const short hi = f2bits(x);
        ph[tt >> 1][4 * (tt & 1) + r] = hi;
        pl[tt >> 1][4 * (tt & 1) + r] = f2bits(x - bits2f(hi));
        sum += x;
      }
    lsum += sum;
  };
  auto values = [&](const char* v_lds) {
    const int tq = li >> 2, tp = li & 3;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
      const int r0 = 32 * cc + 4 * h4 + tq, r1 = r0 + 16;
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const int unit = 4 * n + tp;
        const bf16x4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (sp_lds4_t*)(v_lds + r0 * RB + ((unit ^ (sp_vswz<D>(r0) << 1)) << 3)));
        const bf16x4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (sp_lds4_t*)(v_lds + r1 * RB + ((unit ^ (sp_vswz<D>(r1) << 1)) << 3)));
        const bf16x8_t a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pl[cc], o[n], 0, 0, 0);
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ph[cc], o[n], 0, 0, 0);
      }
    }
  };
  issue(0, 0);
  for (int t = 0; t < ntiles; ++t) {
    // the wave's own pieces of tile t landed, its reads of tile t - 1 returned; the barrier: everyone's, and the buffer of tile
    // t - 1 is free for the next issue
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < ntiles) issue(t + 1, (t + 1) & 1);
    const int kt0 = start(t);
    if (kt0 >= lim_max || (kt0 + SP_KT <= low_min && kt0 >= p.keep)) continue;  // none of the wave's rows sees a key of it
    const char* k_lds = smem + (t & 1) * 2 * TILE;
    scores(kt0, k_lds);
    values(k_lds + TILE);
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (!valid) return;
  float r = p.out_scale / lsum;
  if (p.hgate) r /= 1.f + expf(-(float)p.hgate[(size_t)tok * p.gate_ld + head]);
  bf16* op = p.out + (size_t)tok * p.out_ld + head * D + 4 * h4;
#pragma unroll
  for (int n = 0; n < ND; ++n)
    *reinterpret_cast<bf16x4_t*>(op + 16 * n) =
        bf16x4_t{f2bits(o[n][0] * r), f2bits(o[n][1] * r), f2bits(o[n][2] * r), f2bits(o[n][3] * r)};
}

// Whether the kernel takes a call; grag_sink_attn_prefill (seqmix.hip) asks before it launches.
bool sink_prefill_takes(int d, int vd, int v_ld, int BS, int max_q_len, int R, int bt_stride, int chunk, int window, int keep,
                        const void* q, const void* k, const void* v, const void* out, int out_ld) {
  if ((d != 64 && d != 128) || vd != d || v_ld != d || BS != SP_BS || max_q_len < 16 || out_ld % 4) return false;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15 || (uintptr_t)out & 7) return false;
  // the most keys a workgroup walks: the kept ones and its rows' windows (or their blocks, two where the rows straddle), or all
  const long rows = 128 / R + 2;
  long keys = (long)bt_stride * BS;
  if (window > 0) keys = keys < window + rows + keep + 3 * SP_KT ? keys : window + rows + keep + 3 * SP_KT;
  if (chunk > 0) keys = keys < chunk + rows + keep + 3 * SP_KT ? keys : chunk + rows + keep + 3 * SP_KT;
  return keys <= (long)SP_MAXB * SP_BS;
}

hipError_t sink_prefill_launch(const void* q, const void* k, const void* v, void* out, int out_ld, const int* bt, int bt_stride,
                               const int* q_start, const int* ctx_len, const float* sinks, int nseq, int max_q_len, int H, int G,
                               int d, float scale, float out_scale, int nblocks, const float* hscale, const void* hgate,
                               int gate_ld, int chunk, int window, float softcap, int keep, hipStream_t st) {
  SinkArgs a{};
  a.q = (const bf16*)q, a.k = (const bf16*)k, a.v = (const bf16*)v, a.out = (bf16*)out;
  a.bt = bt, a.q_start = q_start, a.ctx_len = ctx_len, a.sinks = sinks, a.hscale = hscale, a.hgate = (const bf16*)hgate;
  a.out_ld = out_ld, a.bt_stride = bt_stride, a.H = H, a.G = G, a.R = H / G, a.nblocks = nblocks;
  a.gate_ld = gate_ld, a.chunk = chunk, a.window = window, a.keep = keep;
  a.scale = scale, a.out_scale = out_scale, a.softcap = softcap;
  // 128 rows a workgroup, or 64 where those are few for the chip: a walk's time is the chain of its tiles, shorter with one wave a
  // SIMD than with two.  us of 128 / 64 rows, all keys: 12 / 2 heads, 300 tokens 15 / 13, 1187 (112 workgroups) 43 / 37, 2048
  // (192) 67 / 55; 28 / 4 heads, 1500 (332) 63 / 53; past the line 12 x 300 (360) 22 / 24, 28 / 4 heads, 2048 (448) 76 / 90.
  long tiles = ((long)max_q_len * a.R + 127) / 128;
  const bool few = tiles * nseq * G <= 340;
  if (few) tiles = ((long)max_q_len * a.R + 63) / 64;
  if (tiles * nseq > 0x7fffffffL || G > 65535) return hipErrorInvalidValue;
  a.tiles = (int)tiles;
  const dim3 grid((unsigned)(tiles * nseq), G);
#define SINK_PREFILL(DD, CAP)                                                                                        \
  {                                                                                                                  \
    if (few) hipLaunchKernelGGL((sink_prefill_kernel<DD, CAP, 4>), grid, dim3(256), 0, st, a);                       \
    else hipLaunchKernelGGL((sink_prefill_kernel<DD, CAP, 8>), grid, dim3(512), 0, st, a);                           \
  }
  if (d == 64 && softcap > 0.f) SINK_PREFILL(64, true)
  else if (d == 64) SINK_PREFILL(64, false)
  else if (softcap > 0.f) SINK_PREFILL(128, true)
  else SINK_PREFILL(128, false)
#undef SINK_PREFILL
  return hipGetLastError();
}

}  // namespace grag
