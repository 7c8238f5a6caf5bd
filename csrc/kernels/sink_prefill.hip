// Prefill attention of the hybrid decoders on the matrix cores (gfx950): causal softmax over the paged cache with a sink logit
// per head, aligned blocks or a sliding window with kept first keys, a score cap, a temperature and an output gate per head
// (grag_sink_attn_prefill says what each does).  Head size D = 64 or 128 for keys and values alike, 16-key cache blocks; other
// sizes take the kernel of seqmix.hip.
//
// Rows are (position, query head) pairs of one kv head, R heads to a position: a workgroup is 4 waves of 32 rows, 128 rows on one
// stream of K / V tiles (the other kernel reads every tile for 64 rows of one head), or of 16 rows where those are too few for the
// chip.  Tiles of 64 keys arrive by LDS-DMA, K a tile further ahead than V, a piece at a time between the products.  Per tile
//   S^T = K Q^T          bf16 products, exact in fp32,
//   P = 2^(s - m)        fp32; m moves only when a row's scores pass it by 2^8 (its factor is exact then),
//   O^T += V^T P^T       P as bf16 hi + lo, two products: 16 bits of the weights reach the accumulator; the weights of the next
//                        keys are formed between the products of these.
// What bounds it: the split is 1.5 times the products of a kernel with 16-bit weights, and the chip's power, not its cycles.  At
// window 1024, 2 portions of 8192 tokens, 28 / 4 heads of 128, waves of 16 rows, whose every tile waited for the DMA of the next
// (the compiler's wait before the transposed reads), took 445 k cycles at 2.09 GHz; this takes 356 k at 1.95: matrix cores 45 %,
// vector instructions 46 %, LDS 15 % of them.  The order of the walks, longest first over all portions and heads, is worth 5 to 9 %
// (busy CUs 83 -> 93 % of the time).  Measured, us, before -> after: window 219 -> 200, capped 265 -> 239, blocks of 1024
// 131 -> 121, all keys 7 x 8192 tokens 163 -> 148, 1 x 8192 710 -> 641, 3 x 2405 56 -> 50; 12 / 2 heads 1 x 1187 38 -> 25.
#include "sink.h"

GRAG_ERR_UNIT(sink_prefill)

namespace grag {

constexpr int SP_KT = 64;         // keys per tile
constexpr int SP_MAXB = 2048;     // cache blocks a workgroup can walk (32 K keys): its part of the block table, in LDS

// the larger of a lane's value and that of the lane 32 on, without LDS
__device__ __forceinline__ float sp_max32(float v) {
  const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
}

// the swizzle of V's chunks: a transposed read takes 4 rows x 2 neighbouring units of 32 bytes at a time with 32-row waves
template <int D, int MR> __device__ __forceinline__ int sp_pswz(int row) {
  if constexpr (MR == 16) return sp_vswz<D>(row);
  else return D == 128 ? (row & 3) << 2 : (row & 2) << 1;
}

// MR: rows a wave, the matrix instruction's width (16 x 16 x 32 or 32 x 32 x 16)
// TEAMS: 4 waves each, that walk the tiles of the same rows in turn
template <int D, bool CAP, int MR, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS, MR == 32 || TEAMS > 1 ? 2 : 4) sink_prefill_kernel(const SinkArgs p) {
  constexpr int NW = 4, KD = 512 / MR, AR = MR * MR / 64;  // waves; a product's depth, its results a lane
  constexpr int RB = 2 * D, CPR = D / 8, NC = D / KD, ND = D / MR, NT = SP_KT / MR, TILE = SP_KT * RB;
  constexpr int ROWS = MR * NW, PPW = TILE / 1024 / NW, RPP = 1024 / RB;
  typedef float acc_t __attribute__((ext_vector_type(AR)));
  // With two teams the scores and the first weights go before the SIMD's other waves, whose values' products have instructions between: of
  // 101 launches 2 % less time, of 54 capped ones 6 % (12 / 2 heads of 64, 512 rows on 7000 keys 109 -> 91 us), one longer (45.9 -> 47.9).
  // One team lost as often as it gained, 433 launches 0.94 - 1.10 of the time (8192 rows, 12 / 2 heads of 64 207 -> 222; of 128, 4 x 2048
  // 96 -> 90).
  auto before_others = [](bool on) __attribute__((always_inline)) {
    if constexpr (TEAMS > 1) {
      if (on) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
    }
  };
  auto mma = [](bf16x8_t a, bf16x8_t b, acc_t c) {
    if constexpr (MR == 16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  };
  static_assert(PPW * RPP == SP_BS, "a wave's DMA rows sit in one cache block");
  // (one array: beside a second one the compiler waits for the DMA in flight before every tile's reads)
  __shared__ __attribute__((aligned(16))) char all_lds[TEAMS * 2 * 2 * TILE + 4 * SP_MAXB];
  int* bt_lds = reinterpret_cast<int*>(all_lds + TEAMS * 2 * 2 * TILE);
  const int lane = threadIdx.x & 63, team = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & (NW - 1));
  char* smem = all_lds + team * 2 * 2 * TILE;
  const int hh = lane / MR, li = lane % MR;  // this lane's row is li; its keys (and head numbers) are 8 i + 4 hh + 0..3
  const WalkOrder at = walk_order(blockIdx.x, p.nseq, p.G, p.tiles);
  const int seq = at.seq, kvh = at.kvh;
  const int row_base = at.tile * ROWS;
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
  for (int i = threadIdx.x; i < nb; i += 64 * NW * TEAMS) {
    int b = bt[i < kb ? i : i + skip];
    if (!index_ok(b, p.nblocks, ERR_BLOCK_PREFILL)) b = 0;  // reported; block 0 read instead of faulting
    bt_lds[i] = b;
  }
  auto start = [&](int t) { return t < nkeep ? t * SP_KT : kfirst + (t - nkeep) * SP_KT; };

  // this lane's row
  const float LOG2E = 1.4426950408889634f;
  const int row = row_base + wave * MR + li;
  const bool valid = row < nrows;
  const int pq = valid ? row / R : 0;
  const int head = kvh * R + (valid ? row - pq * R : 0), tok = q0 + pq;
  const int lim = valid ? min(kv_hi, pos0 + pq + 1) : 0, low = sp_first(p, pos0 + pq);
  const float sc = p.scale * (p.hscale ? p.hscale[head] : 1.f);
  const bool pre = p.hscale || !(p.scale > 0.f);  // scores scaled before the mask and the maximum, else in the exponent's fma
  // the maximum starts at the sink, whose weight is 1 of the sum (of the first team's; the others only need a number)
  float m = p.sinks[head] * LOG2E, lsum = hh == 0 && team == 0 ? 1.f : 0.f;
  if (team > 0) m = fmaxf(m, -1e30f);
  bf16x8_t qf[NC];
  const bf16* qp = p.q + ((size_t)tok * p.H + head) * D + 8 * hh;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    qf[c] = valid ? *reinterpret_cast<const bf16x8_t*>(qp + KD * c) : bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  // (a compiler-visible wait: the q loads retired, so that the loop needs no vmcnt of its own that would drain the DMA)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();  // the table is there
  // of the wave's rows, the smallest and largest limit and first key
  const int w0 = row_base + wave * MR, w1 = min(w0 + MR, nrows) - 1;
  const int p0 = pos0 + min(w0, nrows - 1) / R, p1 = pos0 + max(w1, 0) / R;
  const int lim_min = w0 + MR <= nrows ? min(kv_hi, p0 + 1) : 0, lim_max = w0 < nrows ? min(kv_hi, p1 + 1) : 0;
  const int low_min = sp_first(p, p0), low_max = sp_first(p, p1);

  // This wave's keys of a tile are one cache block: a wave-uniform base, a lane's offset behind it.  Keys past the last one re-read
  // it (their weights are 0, and 0 times whatever lies there must be 0); tiles past the last one re-read that one, unused.
  const int lrow = lane / CPR, lch = lane % CPR, last_slot = (kv_hi - 1) % SP_BS;
  auto table = [&](int t) { return bt_lds[min(min(t, ntiles - 1) * (SP_KT / SP_BS) + wave, nb - 1)]; };
  auto slots = [&](int t) {
    const int left = kv_hi - 1 - start(min(t, ntiles - 1)) - wave * SP_BS;
    return left < 0 ? last_slot : left;
  };
  auto base = [&](int blk) { return ((size_t)blk * p.G + kvh) * SP_BS * D; };
  auto dma_k = [&](int i, size_t at, int most, int buf) {
    const int r = i * RPP + lrow;
    sp_dma_s(p.k + at, min(r, most) * RB + ((lch ^ sp_kswz<D>(r)) << 4), smem + (buf & 1) * 2 * TILE + (wave * PPW + i) * 1024);
  };
  auto dma_v = [&](int i, size_t at, int most, int buf) {
    const int r = i * RPP + lrow;
    sp_dma_s(p.v + at, min(r, most) * RB + ((lch ^ sp_pswz<D, MR>(r)) << 4), smem + (buf & 1) * 2 * TILE + TILE + (wave * PPW + i) * 1024);
  };
  acc_t o[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) o[n] = acc_t{};
  constexpr int NP = SP_KT / KD;
  acc_t s[NT];
  bf16x8_t ph[2], pl[2], vf[2][ND];  // of KD keys: the weights of a lane's row, keys 4 hh + 0..3 and KD / 2 + 4 hh + 0..3; the values

  const float f = CAP || pre ? 1.f : p.scale * LOG2E;
  auto scores = [&](int kt0, const char* k_lds) {
    bf16x8_t kf[NT][NC];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        kf[tt][c] = *reinterpret_cast<const bf16x8_t*>(k_lds + (MR * tt + li) * RB + ((((KD / 8) * c + hh) ^ sp_kswz<D>(MR * tt + li)) << 4));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      s[tt] = acc_t{};
      if (tt == 0) before_others(true);
#pragma unroll
      for (int c = 0; c < NC; ++c) s[tt] = mma(kf[tt][c], qf[c], s[tt]);
      if (tt == NT - 1) before_others(false);
    }
    if constexpr (CAP) {  // cap in the natural domain, then to log2
      // Below 1/4 by tanh's power series to x^9, whose next term is 1/10 of fp32's rounding there; a tile with a larger score by
      // tanhf.
      const float ic = 1.f / p.softcap, c2 = p.softcap * LOG2E, k = sc * ic;
      float most = 0.f;
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int r = 0; r < AR; ++r) most = fmaxf(most, fabsf(s[tt][r]));
      if (__any(most * fabsf(k) >= 0.25f)) {
        asm volatile("");
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
          for (int r = 0; r < AR; ++r) s[tt][r] = c2 * tanhf(s[tt][r] * k);
      } else {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
          for (int r = 0; r < AR; ++r) {
            const float x = s[tt][r] * k, z = x * x, cx = c2 * x;
            s[tt][r] = fmaf(cx, z * fmaf(fmaf(fmaf(62.f / 2835.f, z, -17.f / 315.f), z, 2.f / 15.f), z, -1.f / 3.f), cx);
          }
      }
    } else if (pre) {  // (a factor of 0 or less: it turns the order, and makes no 0 of a masked score)
      asm volatile("");
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) s[tt] *= sc * LOG2E;
    }
    // a real branch (the empty asm): as selects, the masks would cost every tile what only the edges need
    if (kt0 + SP_KT > lim_min || (kt0 < low_max && kt0 + SP_KT > p.keep)) {
      asm volatile("");
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int r = 0; r < AR; ++r) {
          const int key = kt0 + MR * tt + 8 * (r >> 2) + 4 * hh + (r & 3);
          s[tt][r] = key < lim && (key >= low || key < p.keep) ? s[tt][r] : -INFINITY;
        }
    }
  };
  auto maximum = [&]() {
    float tmax = -INFINITY;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int r = 0; r < AR; ++r) tmax = fmaxf(tmax, s[tt][r]);
    if constexpr (MR == 16) tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = sp_max32(tmax);
    const float cand = fmaxf(m, tmax * f);
    if (__any(cand > m + SP_RESCALE)) {  // every row takes its exact maximum, so o and lsum see one factor
      const float alpha = __builtin_amdgcn_exp2f(m - cand);
      m = cand;
      lsum *= alpha;
#pragma unroll
      for (int n = 0; n < ND; ++n) o[n] *= alpha;
    }
  };
  auto weights = [&](int u) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = 8 * u + i;
      const float x = __builtin_amdgcn_exp2f(fmaf(s[e / AR][e % AR], f, -m));
      const short hi = f2bits(x);
      ph[u & 1][i] = hi;
      pl[u & 1][i] = f2bits(x - bits2f(hi));
      sum += x;
    }
    lsum += sum;
  };
  auto load_v = [&](const char* v_lds, int u) {
    const int tq = (lane & 15) >> 2, tp = lane & 3;
    const int r0 = KD * u + 4 * hh + tq, r1 = r0 + KD / 2;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const int unit = (MR / 4) * n + (li >> 4) * 4 + tp;
      const bf16x4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (sp_lds4_t*)(v_lds + r0 * RB + ((unit ^ (sp_pswz<D, MR>(r0) << 1)) << 3)));
      const bf16x4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (sp_lds4_t*)(v_lds + r1 * RB + ((unit ^ (sp_pswz<D, MR>(r1) << 1)) << 3)));
      vf[u & 1][n] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  // K of tile t + 1 and V of tile t are there after tile t's barrier, by which everyone has read K of tile t and V of tile t - 1:
  // their buffers take K of tile t + 2 and V of tile t + 1, a piece at a time between the products (all at once, the waves of a
  // CU wait for each other's)
  size_t vat;
  {
    const int t0 = team, t1 = team + TEAMS;
    const int b0 = __builtin_amdgcn_readfirstlane(table(t0)), b1 = __builtin_amdgcn_readfirstlane(table(t1));
#pragma unroll
    for (int i = 0; i < PPW; ++i) dma_k(i, base(b0), slots(t0), 0);
#pragma unroll
    for (int i = 0; i < PPW; ++i) dma_v(i, base(b0), slots(t0), 0);
    vat = base(b1);
#pragma unroll
    for (int i = 0; i < PPW; ++i) dma_k(i, vat, slots(t1), 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PPW) : "memory");  // K of tile 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  for (int j = 0; j * TEAMS < ntiles; ++j) {
    const int t = j * TEAMS + team, kt0 = start(t);
    const char* k_lds = smem + (j & 1) * 2 * TILE;
    const bool sees = t < ntiles && kt0 < lim_max && (kt0 + SP_KT > low_min || kt0 < p.keep);  // a row of the wave, a key of the tile
    const int nblk = table(t + 2 * TEAMS);
    if (sees) scores(kt0, k_lds);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const size_t kat = base(__builtin_amdgcn_readfirstlane(nblk));
    const int kmost = slots(t + 2 * TEAMS), vmost = slots(t + TEAMS);
    if (!sees) {
#pragma unroll
      for (int i = 0; i < PPW; ++i) dma_v(i, vat, vmost, j + 1), dma_k(i, kat, kmost, j);
      vat = kat;
      continue;
    }
    const char* v_lds = k_lds + TILE;
    before_others(true);
    load_v(v_lds, 0);
    maximum();
    weights(0);
    before_others(false);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      if (u + 1 < NP) load_v(v_lds, u + 1);
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        o[n] = mma(vf[u & 1][n], pl[u & 1], o[n]);
        o[n] = mma(vf[u & 1][n], ph[u & 1], o[n]);
      }
#pragma unroll
      for (int i = u * PPW / NP; i < (u + 1) * PPW / NP; ++i) dma_v(i, vat, vmost, j + 1), dma_k(i, kat, kmost, j);
      if (u + 1 < NP) {
        weights(u + 1);
#pragma unroll
        for (int i = 0; i < 2 * ND; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, MR == 32 ? 5 : 2, 0);
          if (MR == 32 || i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    vat = kat;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (TEAMS > 1) {  // the second team's sums through the buffers, lane by lane, to the first
    static_assert(TEAMS == 2 && AR == 4 && NW * (ND + 1) * 1024 <= 2 * 2 * 2 * TILE, "exchange");
    f32x4_t* x = reinterpret_cast<f32x4_t*>(all_lds) + wave * (ND + 1) * 64 + lane;
    __syncthreads();
    if (team == 1) {
#pragma unroll
      for (int n = 0; n < ND; ++n) x[n * 64] = o[n];
      x[ND * 64] = f32x4_t{m, lsum, 0.f, 0.f};
    }
    __syncthreads();
    if (team == 1) return;
    const f32x4_t y = x[ND * 64];
    const float top = fmaxf(m, y[0]), a = __builtin_amdgcn_exp2f(m - top), b = __builtin_amdgcn_exp2f(y[0] - top);
    lsum = lsum * a + y[1] * b;
#pragma unroll
    for (int n = 0; n < ND; ++n) o[n] = o[n] * a + x[n * 64] * b;
  }
  if constexpr (MR == 16) lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (!valid) return;
  float r = p.out_scale / lsum;
  if (p.hgate) r /= 1.f + expf(-(float)p.hgate[(size_t)tok * p.gate_ld + head]);
  bf16* op = p.out + (size_t)tok * p.out_ld + head * D + 4 * hh;
#pragma unroll
  for (int n = 0; n < ND; ++n)
#pragma unroll
    for (int i = 0; i < AR / 4; ++i)
      *reinterpret_cast<bf16x4_t*>(op + MR * n + 8 * i) = bf16x4_t{f2bits(o[n][4 * i] * r), f2bits(o[n][4 * i + 1] * r),
                                                                   f2bits(o[n][4 * i + 2] * r), f2bits(o[n][4 * i + 3] * r)};
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

// The shape of a launch's workgroups: 0 two teams of 4 waves on 64 rows, 1 64 rows by 4 waves of 16, 2 128 rows by 4 waves of 32.  A
// walk's time is its start and the chain of its tiles (kTau each, kStart tiles' worth), shorter with 16 rows a wave than with 32,
// and two teams take the tiles in turn; many walks are paid by the reads a row, in rounds of their workgroups where they are more
// than the chip holds (kSlots a CU).  Of uneven prompts a portion's last tile is half full.  Rounds count by a walk's mean length
// over the longest's, with kPast cached keys before each portion (the host does not know how many there are), at most the
// window; a table of two tiles' blocks has no second team's work.
// 1774 batches of 1 - 128 portions, 30 - 8192 tokens, no, 300 and 1000 cached keys, all keys and window 256, heads of 128 (28 / 4, 12 /
// 2) and 64 (16 / 4, 12 / 12), all three shapes timed: 1.018 of the best in the geometric mean; by the rows' 128-row workgroups alone
// (lines at 200 and 340) 1.05.  us in 128 rows before / by those lines / now, unequal portions: 28 / 4 heads 40 of 800 tokens in all 9.6 /
// 18.8 / 8.7, 12 of 480 7.1 / 11.9 / 8.1; 12 / 2 heads 24 of 1536 8.7 / 13.7 / 9.3.  us of the three, 28 / 4 heads, all keys: 600 x 1 16.0 /
// 21.4 / 27.6, 1187 x 1 - / 38 / 46, 2048 x 4 - / 36.5 / 42.3, 3000 x 8 - / 45.6 / 35.1; 12 / 2 heads 1187 x 1 24.6 / 35.1 / 45.7, 3600 x 12 - /
// 25.0 / 31.4, 8192 x 4 - / 136 / 110.
static int sink_prefill_shape(int D, int nseq, long rows, int max_q_len, int R, int G, long reach, long table) {
  struct Shape {
    float tau, start, slots;
    int rows;
  };
  static const Shape k128[3] = {{0.35f, 2.5f, 0.38f, 64}, {1.36f, 3.6f, 1.75f, 64}, {1.37f, 4.1f, 3.5f, 128}};
  static const Shape k64[3] = {{0.34f, 2.f, 0.42f, 64}, {1.44f, 1.5f, 2.6f, 64}, {2.18f, 1.55f, 2.2f, 128}};
  constexpr double kPast = 1100;
  const Shape* shapes = D == 128 ? k128 : k64;
  const double mean = (double)rows / nseq, far = fmin(max_q_len + kPast, (double)reach + 32);
  const double part = fmin(mean / 2 + kPast, (double)reach) / far, tiles = fmin(max_q_len, (double)reach + 32) / SP_KT;
  const double cus = device_cus();
  int best = -1;
  double least = 0;
  for (int s = table <= 2 * SP_KT ? 1 : 0; s < 3; ++s) {
    const int r = shapes[s].rows;
    const double wgs = G * fmin((double)nseq * (((long)max_q_len * R + r - 1) / r), (double)rows * R / r + 0.5 * nseq);
    const double t = (shapes[s].tau * tiles + shapes[s].start) * fmax(1.0, part * wgs / (shapes[s].slots * cus));
    if (best < 0 || t < least) best = s, least = t;
  }
  return best;
}
static long sink_reach(int chunk, int window) {  // keys that a query sees at most
  long reach = 1L << 40;
  if (chunk > 0) reach = chunk;
  if (window > 0 && window < reach) reach = window;
  return reach;
}
// (for tests)
GRAG_API int grag_sink_prefill_shape(int D, int nseq, int rows, int max_q_len, int R, int G, int chunk, int window, int bt_stride) {
  return nseq < 1 || (D != 64 && D != 128) ? -1 : sink_prefill_shape(D, nseq, rows, max_q_len, R, G, sink_reach(chunk, window),
                                                                     (long)bt_stride * SP_BS);
}

hipError_t sink_prefill_launch(const void* q, const void* k, const void* v, void* out, int out_ld, const int* bt, int bt_stride,
                               const int* q_start, const int* ctx_len, const float* sinks, int nseq, int max_q_len, int rows, int H,
                               int G, int d, float scale, float out_scale, int nblocks, const float* hscale, const void* hgate,
                               int gate_ld, int chunk, int window, float softcap, int keep, hipStream_t st) {
  SinkArgs a{};
  a.q = (const bf16*)q, a.k = (const bf16*)k, a.v = (const bf16*)v, a.out = (bf16*)out;
  a.bt = bt, a.q_start = q_start, a.ctx_len = ctx_len, a.sinks = sinks, a.hscale = hscale, a.hgate = (const bf16*)hgate;
  a.out_ld = out_ld, a.bt_stride = bt_stride, a.H = H, a.G = G, a.R = H / G, a.nblocks = nblocks;
  a.gate_ld = gate_ld, a.chunk = chunk, a.window = window, a.keep = keep;
  a.scale = scale, a.out_scale = out_scale, a.softcap = softcap;
  const int shape = sink_prefill_shape(d, nseq, rows, max_q_len, a.R, G, sink_reach(chunk, window), (long)bt_stride * SP_BS);
  const long per = shape == 2 ? 128 : 64, tiles = ((long)max_q_len * a.R + per - 1) / per;
  if (tiles * nseq * G > 0x7fffffffL - (tiles > 0 ? tiles : 0)) return hipErrorInvalidValue;
  a.tiles = (int)tiles, a.nseq = nseq;
  const dim3 grid((unsigned)(tiles * nseq * G));
#define SINK_PREFILL(DD, CAP)                                                                                           \
  {                                                                                                                     \
    if (shape == 0) hipLaunchKernelGGL((sink_prefill_kernel<DD, CAP, 16, 2>), grid, dim3(512), 0, st, a);               \
    else if (shape == 1) hipLaunchKernelGGL((sink_prefill_kernel<DD, CAP, 16, 1>), grid, dim3(256), 0, st, a);          \
    else hipLaunchKernelGGL((sink_prefill_kernel<DD, CAP, 32, 1>), grid, dim3(256), 0, st, a);                          \
  }
  if (d == 64 && softcap > 0.f) SINK_PREFILL(64, true)
  else if (d == 64) SINK_PREFILL(64, false)
  else if (softcap > 0.f) SINK_PREFILL(128, true)
  else SINK_PREFILL(128, false)
#undef SINK_PREFILL
  return hipGetLastError();
}

}  // namespace grag
