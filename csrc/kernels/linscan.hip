// Chunked linear-attention scan on the matrix cores (gfx950): prompt portions of the decay linear attention and of the
// state-space scan, which are one recurrence with a scalar decay a_t per head and token,
//   S_t = a_t S_(t-1) + c_t k_t v_t^T,   o_t = S_t^T q_t    (S [d, vd] fp32; decay: a_t = lam, c_t = kscale; state space:
//   a_t = exp(-exp(A_log) dt_t), c_t = dt_t, k = B, q = C, v = x, and o_t gains D x_t).
// A chunk is LC = 64 tokens.  With L_t the sum of log2 a up to token t of the chunk and S_0 the state at its start,
//   o_t = 2^(L_t) S_0^T q_t + sum_(s <= t) 2^(L_t - L_s) c_s (k_s . q_t) v_s
//   S_end = 2^(L_63) S_0 + sum_s 2^(L_63 - L_s) c_s k_s v_s^T
// which is four matrix products per chunk.  Only differences L_t - L_s <= 0 of tokens in order appear (for a decay of at most
// 1), so small decays are safe; L is kept as two floats, since it grows with the chunk and its differences need not.
//
// What bounds it: one thread per state column, three vector instructions per state element and token (the kernels of
// seqmix.hip and ssm.hip, which still take decode rows and heads of more than 128 rows), waited on LDS broadcasts at 3 % of
// the fp32 vector rate.  Here a chunk is bound by vector instructions (the splits, SiLU) and the latency of its dependent
// steps.  Measured, those kernels -> this one with workgroups in order of sequence -> longest first (scan_item) -> with pairs split
// together, the halves of q and the table below: decay with SiLU, 28 heads of 128 x 128, 7 portions of 8192 tokens in all 2150 -> 748
// -> 386 -> 311 us, 1 x 1187 635 -> 108 -> 92; without SiLU 2060 -> 214 -> 153 -> 152 and 602 -> 47 -> 45; state space, 56 heads of
// 128 x 64, 3 portions of 4096 tokens 1450 -> 165 -> 100 -> 94.
//
// Precision: nothing is rounded to 16 bits that was not before.  An operand is the sum of bf16 parts of 8 bits of mantissa
// each, and a product of operands is the matrix-core products of their parts (exact, fp32 sums).  What is fp32 (S, the
// weighted triangle, the weighted v) has three parts; q, k and v have one (AP = 1) where they are bf16 numbers as they come,
// and three (AP = 3) after SiLU or rotary, or where the activations are fp32.  Of three by three parts the three products
// below 2^-24 of the result are left out: they lie under the rounding of an fp32 product.
// An infinity has no such parts, and a product of matrices sums 0 times it into tokens that do not see it.  So a part is walked
// token by token, with the recurrence as it stands above, from the first chunk on whose numbers are not all finite and small
// (SCAN_BIG, SCAN_BIG_S: nothing in the products can overflow below them).
//
// A workgroup of 8 waves walks the chunks of one (sequence, head, 64 columns of v).  Wave w has 16 queries (block w % 4)
// against 32 of the columns (half w / 4) for the outputs, and 16 columns (block w % 4) times half of the rows (w / 4) of S,
// in registers.  Products are laid out so that a result is the next product's operand without a shuffle: lane (ql = lane %
// 16, quad = lane / 16) of a 16 x 16 result holds rows 4 quad + i of column ql, and as the order of a sum is free those are
// its share of an operand whose row (or column) is ql and whose summed index runs over the result's rows.  So the triangle is
// formed as [s, t] and the outputs as [column, t]; S leaves through LDS (every wave needs all of it), the triangle does not.
//
// A step with few (sequence, head) pairs is cut into parts of `part` tokens that run side by side:
//   MODE 1  every part's own contribution -> ws, the log2 of its decay -> wa (the first part starts from the carried state;
//           the last part only copies that state into its place in ws, for the first part of MODE 2 to read);
//   MODE 2  the outputs: a part's start state is folded out of the parts before it; the last part leaves the state.
// A portion of one part needs MODE 2 alone.
#include "common.h"

GRAG_ERR_UNIT(linscan)

namespace grag {

constexpr int LC = 64;     // tokens per chunk
constexpr int LVT = 64;    // columns of v per workgroup
constexpr int LTHREADS = 512;
constexpr int LD_MAX = 128;  // rows of S at most
// bounds of what the matrix products take: sums of squares of a thread's elements of q, k, v as they are stored (|x| < 2^20) and
// of S (|S| < 2^60); |c_s| < 2^20 and a decay of at most 1.25 are asked too
constexpr float SCAN_BIG = 0x1p40f, SCAN_BIG_S = 0x1p120f;

struct ScanArgs {
  const void* x;  // q, k, v columns of rows of ld elements
  int ld, qoff, koff, voff, R;  // head h reads q / k head h / R
  float* state;
  const int *slots, *q_start, *ctx_len;
  float* out;
  int nseq, H, d, vd, nslots;
  float *ws, *wa;
  int part, maxparts, full, plain;
  // decay
  const float* decay;
  float kscale;
  int act;
  const int* positions;
  const float* rope;
  int rd, tab_rows;
  // state space
  const void* proj;
  int pld, dtoff;
  const float *dt_bias, *a_log, *skip;
};

// ------------------------------------------------------------------------------------------------ operands
typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;

// An operand with 32 summed indices is 512 bf16 in LDS: lane (ql, quad) has 8 in a row in "slot" 16 quad + ql, summed indices
// 4 quad + 0..3 and 16 + 4 quad + 0..3 (the two halves).
__device__ __forceinline__ bf16x8_t ld8(const bf16* p, int slot) { return *reinterpret_cast<const bf16x8_t*>(p + slot * 8); }
__device__ __forceinline__ bf16x8_t join(bf16x4_t a, bf16x4_t b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
// Rows of k (and v) lie there as row operands (summed over 32 dims).  The same numbers as operands summed over 32 rows: the
// hardware's transposed read, lane (ql, quad) addressing row 4 quad + ql / 4, dims 4 (ql % 4) .. + 3 of 16 and getting dim ql of
// the rows 4 quad + 0..3.  Slots are permuted (place) so that neither the stores nor these reads meet in a bank.
__device__ __forceinline__ int place(int quad, int row, int kg) { return 16 * quad + (row ^ (quad + 4 * kg)); }
__device__ __forceinline__ bf16x4_t ld4t(const bf16* p, int ql, int quad, int kg, int half) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_bf16x4_t*)(p + place(ql & 3, 4 * quad + (ql >> 2), kg) * 8 + 4 * half));
}

template <int N> struct Parts { bf16x8_t p[N]; };
template <int N> __device__ __forceinline__ Parts<N> split8(f32x4_t a, f32x4_t b) {
  bf16x4_t pa[N], pb[N];
  split4<N>(a, pa);
  split4<N>(b, pb);
  Parts<N> s;
#pragma unroll
  for (int j = 0; j < N; ++j) s.p[j] = join(pa[j], pb[j]);
  return s;
}
// The parts of the products a * b, whose rounding the second part takes along: without it the states' error against 64 bits is 1 - 2 %
// larger (8 heads of 128 x 128, 500 + 333 tokens 1.16e-7 -> 1.19e-7), with it state space of 3 portions of 4096 tokens takes 144 us
// for 142.
__device__ __forceinline__ Parts<3> split8(f32x4_t a0, f32x4_t b0, f32x4_t a1, f32x4_t b1) {
  Parts<3> s;
  bf16x4_t lo[2][2], hi[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const f32x4_t a = h ? a1 : a0, b = h ? b1 : b0;
    f32x4_t r;
    hi[h] = pack4(a * b);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = fmaf(a[i], b[i], -bits2f(hi[h][i]));
    split4<2>(r, lo[h]);
  }
  s.p[0] = join(hi[0], hi[1]);
#pragma unroll
  for (int j = 0; j < 2; ++j) s.p[j + 1] = join(lo[0][j], lo[1][j]);
  return s;
}
template <int NA, int NB>
__device__ __forceinline__ f32x4_t mul(const Parts<NA>& a, const Parts<NB>& b, f32x4_t c) {
#pragma unroll
  for (int o = 2; o >= 0; --o)  // the smallest first
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int j = o - i;
      if (j >= 0 && j < NB) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[i], b.p[j], c, 0, 0, 0);
    }
  return c;
}
__device__ __forceinline__ f32x4_t widen(bf16x4_t v) { return f32x4_t{bits2f(v[0]), bits2f(v[1]), bits2f(v[2]), bits2f(v[3])}; }
__device__ __forceinline__ f32x4_t widen(f32x4_t v) { return v; }

// ------------------------------------------------------------------------------------------------ elements
__device__ __forceinline__ float elt(const bf16* p) { return (float)*p; }
__device__ __forceinline__ float elt(const float* p) { return *p; }
__device__ __forceinline__ float softplus_x(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float silu_acc(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float pow2(float x) { return __builtin_amdgcn_exp2f(x); }
// x / (1 + e^-x) to the last bits: e^-x as 2^(hi + lo), with the part of -x log2 e that its fp32 product lost put back; the
// reciprocal with one Newton step.  Below -87 the factor stays at e^-87 (times |x| < 2^20: under 2e-32).
__device__ __forceinline__ float silu_x(float x) {
  constexpr float L2E = 1.4426950408889634f, L2E_LO = 1.9259629911266175e-8f;
  const float m = __builtin_amdgcn_fmed3f(x, -87.f, 0x1p100f), hi = -m * L2E, lo = fmaf(-m, L2E_LO, fmaf(-m, L2E, -hi));
  const float e = pow2(hi), d = 1.f + fmaf(e, lo * 0.6931471805599453f, e);
  const float r = __builtin_amdgcn_rcpf(d);
  return x * fmaf(fmaf(-d, r, 1.f), r, r);
}
// a wave's running sum of fp32 numbers as two floats (sum + rest), by moves between neighbouring lanes
template <int CTRL, int ROWS> __device__ __forceinline__ void scan_step(float& s, float& r) {
  const float us = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), CTRL, ROWS, 0xf, false));
  const float ur = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(r), CTRL, ROWS, 0xf, false));
  const float t = s + us, bb = t - s, e = (s - (t - bb)) + (us - bb) + (r + ur);  // (two-sum: t + e is exact)
  s = t + e;
  r = e - (s - t);
}
__device__ __forceinline__ void wave_scan2(float& s, float& r) {
  scan_step<0x111, 0xf>(s, r);  // 1, 2, 4, 8 lanes down within 16, then lane 15 of rows 0, 2 and lane 31 into those behind
  scan_step<0x112, 0xf>(s, r);
  scan_step<0x114, 0xf>(s, r);
  scan_step<0x118, 0xf>(s, r);
  scan_step<0x142, 0xa>(s, r);
  scan_step<0x143, 0xc>(s, r);
}

// s + the squares of four stored elements
__device__ __forceinline__ float squares(bf16x4_t v, float s) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef short s2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const bf16x2_t p = __builtin_bit_cast(bf16x2_t, s2_t{v[i], v[i + 1]});
    s = __builtin_amdgcn_fdot2_f32_bf16(p, p, s, false);
  }
  return s;
}
__device__ __forceinline__ float squares(f32x4_t v, float s) {
#pragma unroll
  for (int i = 0; i < 4; ++i) s = fmaf(v[i], v[i], s);
  return s;
}

template <typename T> struct V4;
template <> struct V4<bf16> { typedef bf16x4_t t; };
template <> struct V4<float> { typedef f32x4_t t; };
// elements c0 .. c0 + 3 of a row of n (zeros from n on), as they are stored; FULL: all four are there, and aligned
template <bool FULL> __device__ __forceinline__ bf16x4_t raw4(const bf16* row, int c0, int n) {
  if (FULL) return *reinterpret_cast<const bf16x4_t*>(row + c0);
  bf16x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = c0 + e < n ? __builtin_bit_cast(short, row[c0 + e]) : (short)0;
  return v;
}
template <bool FULL> __device__ __forceinline__ f32x4_t raw4(const float* row, int c0, int n) {
  if (FULL) return *reinterpret_cast<const f32x4_t*>(row + c0);
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = c0 + e < n ? row[c0 + e] : 0.f;
  return v;
}
// SiLU of numbers that are multiplied next to each other (one branch: a branch for every four left a wave waiting for its exponentials
// and reciprocals)
template <int N> __device__ __forceinline__ void silu_all(const ScanArgs& a, f32x4_t (&v)[N]) {
  if (!a.act) return;
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[n][e] = silu_x(v[n][e]);
}
// rotary of elements c0 .. c0 + 3 (SiLU behind them) of q or k, where c0 < rd; their partners are read again
template <bool FULL, typename TI>
__device__ __forceinline__ void rotary4(const ScanArgs& a, f32x4_t& v, const TI* row, int c0, int pos) {
  const int half = a.rd >> 1;
  if (FULL) {  // (half is a multiple of 4: the four turn with four in a row)
    if (c0 < a.rd) {
      const bool lo = c0 < half;
      const int fi = lo ? c0 : c0 - half;
      f32x4_t u = widen(raw4<true>(row, lo ? c0 + half : fi, 0));
      if (a.act) {
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = silu_x(u[e]);
      }
      const float* tab = a.rope + (size_t)pos * a.rd + fi;
      const f32x4_t c = *reinterpret_cast<const f32x4_t*>(tab), s = *reinterpret_cast<const f32x4_t*>(tab + half);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = lo ? v[e] * c[e] - u[e] * s[e] : v[e] * c[e] + u[e] * s[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = c0 + e;
      if (i >= a.rd) continue;
      const int fi = i < half ? i : i - half;
      float other = elt(row + (i < half ? i + half : i - half));
      if (a.act) other = silu_x(other);
      const float c = a.rope[(size_t)pos * a.rd + fi], s = a.rope[(size_t)pos * a.rd + half + fi];
      v[e] = i < half ? v[e] * c - other * s : v[e] * c + other * s;
    }
  }
}

// ------------------------------------------------------------------------------------------------ the scan
// The sequence and part of work item `item` (false: there is none).  Longest first: the full parts, then the rests by chunks, so
// that the last workgroups to start are short ones.  Up to 64 sequences, a lane each: what the workgroup reads of all of them comes
// in one trip to memory, and of the rests the item's is found bit by bit of the chunk counts (comparing a rest with all others took
// as long as a short portion).  More sequences, and portions of a chunk, are taken as they come (`plain`): 256 tokens in 64 portions,
// 28 heads of 128 x 128 without SiLU, 60.6 us without any order, 93.5 with each rest compared, 64.4 now; 2950 in 64 90.8 / 107.7 / 85.9.
struct ScanItem { int seq, part, q0, qall, ctx, slot; };
__device__ __forceinline__ bool scan_item(const ScanArgs& a, int item, ScanItem& it) {
  if (a.plain) {
    it.seq = item / a.maxparts, it.part = item % a.maxparts;
    if (it.seq >= a.nseq) return false;
    it.q0 = a.q_start[it.seq], it.qall = a.q_start[it.seq + 1] - it.q0;
    it.ctx = a.ctx_len[it.seq], it.slot = a.slots[it.seq];
    return it.part * a.part < it.qall;
  }
  const int lane = threadIdx.x & 63, own = min(lane, a.nseq - 1);
  const int from = a.q_start[own], to = a.q_start[own + 1], ctx = a.ctx_len[own], slot = a.slots[own];
  const int len = lane < a.nseq ? to - from : 0;
  int full = 0, rest = len, left = item;  // left: the item's place among the rests
  bool found = false;
  if (a.maxparts > 1) {
    full = len / a.part, rest = len - full * a.part;
    int upto = full;  // full parts of the lanes up to this one
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
      const int v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    left -= __builtin_amdgcn_readlane(upto, 63);
    if (left < 0) {
      found = true;
      it.seq = __ffsll((unsigned long long)__ballot(upto > item)) - 1;
      it.part = __builtin_amdgcn_readlane(upto, it.seq) - 1 - item;  // (a sequence's last parts first: they fold the most states)
    }
  }
  if (!found) {
    const int chunks = (rest + LC - 1) / LC;
    unsigned long long at = __ballot(chunks > 0);  // those whose rest may be the item's
    if (left >= __popcll(at)) return false;
    for (int bit = 31 - __clz((a.part + LC - 1) / LC); bit >= 0; --bit) {
      const unsigned long long more = at & __ballot((chunks >> bit) & 1);
      const int n = __popcll(more);
      if (left < n) at = more;
      else at &= ~more, left -= n;
    }
    const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(at >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)at, 0));
    it.seq = __ffsll((unsigned long long)(at & __ballot(before == left))) - 1;  // equal ones by number
    it.part = __builtin_amdgcn_readlane(full, it.seq);
  }
  it.q0 = __builtin_amdgcn_readlane(from, it.seq), it.qall = __builtin_amdgcn_readlane(len, it.seq);
  it.ctx = __builtin_amdgcn_readlane(ctx, it.seq), it.slot = __builtin_amdgcn_readlane(slot, it.seq);
  return true;
}

// grid 8 * ceil(items * H / 8) * ceil(vd / 64): the column tiles of a head beside each other on one XCD (they read the same rows of q
// and k), the next head on the next XCD, the items' heads in the order of scan_item.  With a contiguous range of sequences an XCD the
// XCDs that had the long ones walked on while others were done: 7 portions of 8192 tokens, a CU was busy 48 % of the time.
// ND = ceil(d / 32).  AP = 1 takes 76 KB of LDS and 128 registers: two workgroups share a CU, one's products over the other's
// staging.  FULL: d = 32 ND, vd is a multiple of 64 and rows are aligned for 4-element accesses (rd / 2 a multiple of 4), so that
// nothing is tested per element: of the ~4000 instructions a chunk took with the tests, half were theirs.  Rows behind a portion's
// end are copies of its last row: their weight into the state is 0 (row 5 of sc), and of the queries only they themselves see them.
template <typename TI, int AP, bool SSM, bool FULL, int ND, int MODE>
__global__ void __launch_bounds__(LTHREADS, AP == 1 ? 4 : 2)
linear_scan_kernel(const ScanArgs a) {
  typedef typename V4<TI>::t TI4;
  constexpr bool OUT = MODE == 2;
  constexpr int KN = 4 * ND * 512, VN = 4 * 2 * 512;  // elements of one part of k, v
  __shared__ __attribute__((aligned(16))) bf16 Ks[AP * KN];                      // [part][16 tokens][32 dims]
  __shared__ __attribute__((aligned(16))) bf16 Vs[AP * VN];                      // [part][16 tokens][32 columns]
  __shared__ __attribute__((aligned(16))) bf16 So[OUT ? 4 * ND * 3 * 512 : 8];  // [16 columns][32 dims][part]
  // The two waves of a token block need the same q.  With three parts each makes half of its dims (SiLU is 12 instructions and two slow
  // ones an element, of about 60 elements a thread) and both read all of it as fp32 from LDS, whose splits are the short part: 28
  // heads of 128 x 128 with SiLU, 7 portions of 8192 tokens, 60 us of 450.  The parts themselves would not fit the LDS (158 of 160 KB).
  constexpr bool HALVES = OUT && AP == 3 && ND > 1;
  constexpr int QN = HALVES ? ND / 2 : ND;  // 32-dim groups of q that a wave makes
  __shared__ __attribute__((aligned(16))) float Qs[HALVES ? 4 * ND * 512 : 4];  // [16 tokens][32 dims]
  __shared__ __attribute__((aligned(16))) float sc[2][6][LC];  // L (two floats) | c_s | sign_t | 2^(L_t) | 2^(L_end - L_s) c_s
  __shared__ float pw[OUT && !SSM ? 80 : 1];
  __shared__ float ends[2][3];                                 // 2^(L_end) | L_end | not 0: too large for the products
  __shared__ __attribute__((aligned(16))) int odd[LTHREADS / 64];  // a wave's numbers are too large for the products
  const int ntile = (a.vd + LVT - 1) / LVT;
  const int tile = (blockIdx.x >> 3) % ntile, unit = (blockIdx.x >> 3) / ntile * 8 + (blockIdx.x & 7), h = unit % a.H;
  ScanItem it;
  if (!scan_item(a, unit / a.H, it)) return;
  const int seq = it.seq, part = it.part, q0 = it.q0, qall = it.qall, slot = it.slot;
  const int nparts = (qall + a.part - 1) / a.part;
  const bool last = part == nparts - 1;
  if (MODE == 1 && nparts == 1) return;
  const int qa = q0 + part * a.part, qlen = min(a.part, qall - part * a.part);
  const bool fresh = it.ctx - qall == 0;
  const bool slot_ok = index_ok(slot, a.nslots, ERR_SAMPLER_SLOT);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, ql = lane & 15, quad = lane >> 4;
  const int tb = w & 3, vh = w >> 2;  // outputs: token block, half of the columns; state: column block, half of the rows
  const int col = tile * LVT + 16 * tb + ql;
  const bool col_ok = col < a.vd;
  const size_t dv = (size_t)a.d * a.vd;
  float* Sg = a.state + ((size_t)(slot_ok ? slot : 0) * a.H + h) * dv + col;
  float* wsg = a.ws + ((size_t)seq * a.maxparts * a.H + h) * dv + col;  // part p's is p * H * dv further
  const size_t pstep = (size_t)a.H * dv;
  f32x4_t S[ND];
  auto each = [&](auto&& f) __attribute__((always_inline)) {  // f(register block, element, row of S) of the rows that exist
#pragma unroll
    for (int b = 0; b < ND; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * (vh * ND + b) + 4 * quad + i;
        if (FULL || (col_ok && r < a.d)) f(b, i, r);
      }
  };
#pragma unroll
  for (int b = 0; b < ND; ++b) S[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bool carried = !fresh && slot_ok;
  if (MODE == 1) {
    if (carried && (part == 0 || last)) each([&](int b, int i, int r) { S[b][i] = Sg[(size_t)r * a.vd]; });
    if (last) {
      each([&](int b, int i, int r) { wsg[part * pstep + (size_t)r * a.vd] = S[b][i]; });
      return;
    }
  } else if (part == 0) {
    if (nparts > 1) each([&](int b, int i, int r) { S[b][i] = wsg[(nparts - 1) * pstep + (size_t)r * a.vd]; });
    else if (carried) each([&](int b, int i, int r) { S[b][i] = Sg[(size_t)r * a.vd]; });
  } else {  // two parts' loads in flight at a time
    const float* wa = a.wa + (size_t)seq * a.maxparts * a.H + h;
    for (int p = 0; p < part; p += 2) {
      f32x4_t u[2][ND];
      float f[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const bool on = p + x < part;
        f[x] = on ? pow2(wa[(size_t)(p + x) * a.H]) : 1.f;
#pragma unroll
        for (int b = 0; b < ND; ++b) u[x][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (on) each([&](int b, int i, int r) { u[x][b][i] = wsg[(p + x) * pstep + (size_t)r * a.vd]; });
      }
      if (p == 0) f[0] = 0.f;  // (the first part's holds the carried state)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int b = 0; b < ND; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[b][i] = fmaf(f[x], S[b][i], u[x][b][i]);
    }
  }
  const TI* xq = reinterpret_cast<const TI*>(a.x) + a.qoff + (h / a.R) * a.d;
  const TI* xk = reinterpret_cast<const TI*>(a.x) + a.koff + (h / a.R) * a.d;
  const TI* xv = reinterpret_cast<const TI*>(a.x) + a.voff + h * a.vd + tile * LVT;
  const int vn = min(LVT, a.vd - tile * LVT);
  const int nch = (qlen + LC - 1) / LC;

  // the chunk's rows, fetched while the chunk before is computed (q's behind its outputs): per thread 8 dims of rows krow,
  // krow + 512 / (4 ND), ... of k and 8 columns of a row of v; per wave its 16 rows of q as operands
  constexpr int KT = 4 * ND, KR = LTHREADS / KT, KL = LC / KR > 0 ? LC / KR : 1;  // threads a row, rows a pass, passes
  const int krow = tid / KT, kc = 8 * (tid % KT), vrow = tid >> 3, vc = 8 * (tid & 7);
  TI4 kr[KL][2], vr[2], qr[OUT ? QN : 1][2];
  const int qk = HALVES ? vh * QN : 0;
  Stored<TI> dtr;
  auto fetch = [&](int c) __attribute__((always_inline)) {
    const int end = min(qlen - c * LC, LC) - 1;
    const size_t t0 = (size_t)(qa + c * LC) * a.ld;
#pragma unroll
    for (int x = 0; x < KL; ++x)
#pragma unroll
      for (int e = 0; e < 2; ++e) kr[x][e] = raw4<FULL>(xk + t0 + min(krow + x * KR, end) * a.ld, kc + 4 * e, a.d);
#pragma unroll
    for (int e = 0; e < 2; ++e) vr[e] = raw4<FULL>(xv + t0 + min(vrow, end) * a.ld, vc + 4 * e, vn);
  };
  auto fetch_q = [&](int c) __attribute__((always_inline)) {
    const int end = min(qlen - c * LC, LC) - 1;
    const size_t t0 = (size_t)(qa + c * LC) * a.ld;
    if (OUT) {
#pragma unroll
      for (int k = 0; k < QN; ++k)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          qr[k][b] = raw4<FULL>(xq + t0 + min(16 * tb + ql, end) * a.ld, 32 * (qk + k) + 16 * b + 4 * quad, a.d);
    }
  };
  auto fetch_dt = [&](int c) __attribute__((always_inline)) {
    if (SSM) dtr.load(reinterpret_cast<const TI*>(a.proj) + (size_t)(qa + min(c * LC + lane, qlen - 1)) * a.pld + a.dtoff + h);
  };
  auto position = [&](int t) __attribute__((always_inline)) {
    if (AP == 1 || !a.rd) return 0;
    const int p = a.positions[t];
    return index_ok(p, a.tab_rows, ERR_ROPE_POS) ? p : 0;
  };
  float lsum = 0.f;  // the part's log2 decay
  // the head's constants: log2 of the decay and its sign, or the state-space rate and bias
  const float lam = SSM ? 1.f : a.decay[h], bias = SSM ? a.dt_bias[h] : 0.f, skip = SSM ? a.skip[h] : 0.f;
  const float rate = SSM ? -expf(a.a_log[h]) * 1.4426950408889634f : fmaxf(log2f(fabsf(lam)), -4000.f);  // (lam^n = 0 for 0)
  const bool neg = lam < 0.f;
  auto scalars = [&](int c) __attribute__((always_inline)) {  // by one wave: lane = token of chunk c
    const int buf = c & 1, n = min(qlen - c * LC, LC);
    const float sign = neg && (lane & 1) ? -1.f : 1.f, esign = neg && (n & 1) ? -1.f : 1.f;  // of lam^lane, lam^n
    float cs = 0.f, hi, lo = 0.f, ehi, elo;
    if (SSM) {
      if (lane < n) cs = softplus_x(dtr.value() + bias);
      hi = rate * cs;
      wave_scan2(hi, lo);
      ehi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hi), 63));
      elo = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lo), 63));
    } else {
      if (lane < n) cs = a.kscale;
      const float m = (float)min(lane + 1, n);
      hi = rate * m, lo = fmaf(rate, m, -hi);
      ehi = rate * n, elo = fmaf(rate, (float)n, -ehi);
    }
    // (The first four are read for a state space's outputs alone.  Stored for those alone, decays took 0.4 % less time on average of 84
    // sizes, but 6 portions of 700 tokens, 32 heads of 32 x 64 with SiLU, 54.0 us for 52.5.)
    sc[buf][0][lane] = hi;
    sc[buf][1][lane] = lo;
    sc[buf][2][lane] = cs * sign;
    sc[buf][3][lane] = sign;
    sc[buf][4][lane] = pow2(hi) * (neg ? -sign : 1.f);
    sc[buf][5][lane] = pow2((ehi - hi) + (elo - lo)) * cs * (neg ? -sign * esign : 1.f);
    const bool big = SSM ? __any(!(cs < 0x1p20f)) || !(rate > -0x1p60f) : !(fabsf(lam) <= 1.25f) || !(fabsf(a.kscale) < 0x1p20f);
    if (lane == 0) {
      ends[buf][0] = pow2(ehi) * esign;
      ends[buf][1] = ehi;
      ends[buf][2] = big ? 1.f : 0.f;
    }
  };
  const f32x4_t zero = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // A decay's weights of a triangle are the walk's: lam^n c for n = 63 .. 0 tokens between, then zeros for the keys behind a query: a
  // product and an LDS read a pair where 2^(L_t - L_s) and its mask were nine instructions and a branch.  (The state space's are the
  // tokens'.  Without the branch, the mask on the exponent, they took more registers than there are: 142 us for 3 portions of 4096
  // tokens, 2.5 more.)  With SiLU in one block for all of a thread's elements, 28 heads of 128 x 128, 7 portions of 8192 tokens, 30 us
  // of 390.
  if (OUT && !SSM && tid < 80) {
    const int n = 63 - tid;
    pw[tid] = n < 0 ? 0.f : a.kscale * pow2(rate * (float)n) * (neg && (n & 1) ? -1.f : 1.f);
  }
  if (w == 4) {
    fetch_dt(0);
    scalars(0);
    if (nch > 1) fetch_dt(1);
  }
  fetch(0);
  fetch_q(0);
  int c = 0;
  for (; c < nch; ++c) {
    const int buf = c & 1, t0 = qa + c * LC, n = qlen - c * LC;
    // ---- k, v and S into LDS
    float big = 0.f, big_s = 0.f;
#pragma unroll
    for (int b = 0; b < ND; ++b) big_s = squares(S[b], big_s);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
#pragma unroll
      for (int x = 0; x < KL; ++x) big = squares(kr[x][e], big);
      big = squares(vr[e], big);
#pragma unroll
      for (int k = 0; k < (OUT ? QN : 0); ++k) big = squares(qr[k][e], big);
    }
    const bool fits = __all(fmaf(big_s, SCAN_BIG / SCAN_BIG_S, big) < SCAN_BIG);  // (false for NaN)
    if (lane == 0) odd[w] = !fits;
    auto put_k = [&](int r, int dim, const bf16x4_t (&p)[AP]) __attribute__((always_inline)) {
      const int kg = dim >> 5;
#pragma unroll
      for (int y = 0; y < AP; ++y)
        *reinterpret_cast<bf16x4_t*>(Ks + y * KN + ((r >> 4) * ND + kg) * 512 + place((dim >> 2) & 3, r & 15, kg) * 8 +
                                     4 * ((dim >> 4) & 1)) = p[y];
    };
    auto put_v = [&](int dim, const bf16x4_t (&p)[AP]) __attribute__((always_inline)) {
      const int kg = dim >> 5;
#pragma unroll
      for (int y = 0; y < AP; ++y)
        *reinterpret_cast<bf16x4_t*>(Vs + y * VN + ((vrow >> 4) * 2 + kg) * 512 + place((dim >> 2) & 3, vrow & 15, kg) * 8 +
                                     4 * ((dim >> 4) & 1)) = p[y];
    };
    const bool krows = KR <= LC || krow < LC;  // (more threads than k has rows: one pass)
    if constexpr (AP == 1) {
#pragma unroll
      for (int x = 0; x < KL; ++x)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (krows) put_k(krow + x * KR, kc + 4 * e, {kr[x][e]});
#pragma unroll
      for (int e = 0; e < 2; ++e) put_v(vc + 4 * e, {vr[e]});
    } else {
      if (krows) {
        f32x4_t val[2 * KL];
#pragma unroll
        for (int x = 0; x < 2 * KL; ++x) val[x] = widen(kr[x >> 1][x & 1]);
        silu_all(a, val);
#pragma unroll
        for (int x = 0; x < 2 * KL; ++x) {
          const int r = krow + (x >> 1) * KR, dim = kc + 4 * (x & 1);
          if (a.rd) {
            const int rr = t0 + min(r, min(n, LC) - 1);
            rotary4<FULL>(a, val[x], xk + (size_t)rr * a.ld, dim, position(rr));
          }
          bf16x4_t p[AP];
          split4<AP>(val[x], p);
          put_k(r, dim, p);
        }
      }
      f32x4_t val[2] = {widen(vr[0]), widen(vr[1])};  // (SiLU of the zeros behind the last column is 0)
      silu_all(a, val);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf16x4_t p[AP];
        split4<AP>(val[e], p);
        put_v(vc + 4 * e, p);
      }
    }
    Parts<AP> qf[OUT ? ND : 1];
    if (OUT) {
#pragma unroll
      for (int b = 0; b < ND; ++b) {
        const int j = vh * ND + b;
        bf16x4_t p[3];
        split4<3>(S[b], p);
#pragma unroll
        for (int x = 0; x < 3; ++x)
          *reinterpret_cast<bf16x4_t*>(So + ((tb * ND + (j >> 1)) * 3 + x) * 512 + lane * 8 + 4 * (j & 1)) = p[x];
      }
      if constexpr (AP == 1) {
#pragma unroll
        for (int k = 0; k < ND; ++k) qf[k].p[0] = join(qr[k][0], qr[k][1]);
      } else {
        f32x4_t val[2 * QN];
#pragma unroll
        for (int x = 0; x < 2 * QN; ++x) val[x] = widen(qr[x >> 1][x & 1]);
        silu_all(a, val);
        if (a.rd) {
          const int rr = t0 + min(16 * tb + ql, min(n, LC) - 1), pos = position(rr);
#pragma unroll
          for (int x = 0; x < 2 * QN; ++x)
            rotary4<FULL>(a, val[x], xq + (size_t)rr * a.ld, 32 * (qk + (x >> 1)) + 16 * (x & 1) + 4 * quad, pos);
        }
        if constexpr (HALVES) {
#pragma unroll
          for (int x = 0; x < 2 * QN; ++x)
            *reinterpret_cast<f32x4_t*>(Qs + ((tb * ND + qk) * 2 + x) * 256 + lane * 4) = val[x];
        } else {
#pragma unroll
          for (int k = 0; k < ND; ++k) qf[k] = split8<AP>(val[2 * k], val[2 * k + 1]);
        }
      }
    }
    __syncthreads();
    typedef int i32x4_t __attribute__((ext_vector_type(4)));
    const i32x4_t any = *reinterpret_cast<const i32x4_t*>(odd) | *reinterpret_cast<const i32x4_t*>(odd + 4);
    const bool by_token = __builtin_amdgcn_readfirstlane(any[0] | any[1] | any[2] | any[3]) ||
                          __builtin_amdgcn_readfirstlane(__float_as_int(ends[buf][2]));
    if (by_token) break;
    if (c + 1 < nch) {
      if (w == 4) {  // (before the rows: what it waits for, spills among it, does not wait for them)
        scalars(c + 1);
        if (c + 2 < nch) fetch_dt(c + 2);
      }
      fetch(c + 1);
    }
    if constexpr (HALVES) {
#pragma unroll
      for (int k = 0; k < ND; ++k) {
        const float* q = Qs + (tb * ND + k) * 512 + lane * 4;
        qf[k] = split8<3>(*reinterpret_cast<const f32x4_t*>(q), *reinterpret_cast<const f32x4_t*>(q + 256));
      }
    }
    if (OUT) {
      const int t = 16 * tb + ql;
      const float lt = sc[buf][0][t], lt2 = sc[buf][1][t], ft = sc[buf][3][t], et = sc[buf][4][t];
      // ---- the start state seen by the queries
      f32x4_t o[2] = {zero, zero};
#pragma unroll
      for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          Parts<3> sp;
#pragma unroll
          for (int x = 0; x < 3; ++x) sp.p[x] = ld8(So + (((2 * vh + b) * ND + k) * 3 + x) * 512, lane);
          o[b] = mul(sp, qf[k], o[b]);
          if (b) __builtin_amdgcn_sched_barrier(0);  // (all reads at once would not fit the registers)
        }
      o[0] *= et;
      o[1] *= et;
      // ---- the triangle, two blocks of 16 keys at a time, and its product with v
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (2 * p > tb) continue;
        f32x4_t m[2] = {zero, zero};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int j = 2 * p + e;
          if (j > tb) continue;
#pragma unroll
          for (int k = 0; k < ND; ++k) {
            Parts<AP> kf;
#pragma unroll
            for (int y = 0; y < AP; ++y) kf.p[y] = ld8(Ks + y * KN + (j * ND + k) * 512, place(quad, ql, k));
            m[e] = mul(kf, qf[k], m[e]);
          }
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (SSM) {
            const f32x4_t ls = *reinterpret_cast<const f32x4_t*>(&sc[buf][0][16 * j + 4 * quad]);
            const f32x4_t ls2 = *reinterpret_cast<const f32x4_t*>(&sc[buf][1][16 * j + 4 * quad]);
            const f32x4_t cs = *reinterpret_cast<const f32x4_t*>(&sc[buf][2][16 * j + 4 * quad]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
              m[e][i] = 16 * j + 4 * quad + i <= t ? m[e][i] * (pow2((lt - ls[i]) + (lt2 - ls2[i])) * (cs[i] * ft)) : 0.f;
          } else {
            const float* at = pw + 63 - t + 16 * j + 4 * quad;
#pragma unroll
            for (int i = 0; i < 4; ++i) m[e][i] *= at[i];
          }
        }
        const Parts<3> ms = split8<3>(m[0], m[1]);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          Parts<AP> vf;
#pragma unroll
          for (int y = 0; y < AP; ++y)
            vf.p[y] = join(ld4t(Vs + y * VN + (4 * p + vh) * 512, ql, quad, vh, b),
                           ld4t(Vs + y * VN + (4 * p + 2 + vh) * 512, ql, quad, vh, b));
          o[b] = mul(vf, ms, o[b]);
        }
      }
      if (t < n) {
        // (The address of a decay of 128 registers is made here: carried through the loop it was spilled, and its way back waits as below.
        // 28 heads of 128 x 128 without SiLU, 7 portions of 8192 tokens 165 -> 152 us.  Others spill no less so or lose a little:
        // state space, 3 x 4096 247 -> 261; 32 heads of 32 x 64 with SiLU, 7 x 1000 73.5 -> 76.1.)
        int own = t;
        if constexpr (!SSM && AP == 1) asm volatile("" : "+v"(own));
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int c0 = 16 * (2 * vh + b) + 4 * quad;
          float* op = a.out + (size_t)(t0 + own) * ((size_t)a.H * a.vd) + h * a.vd + tile * LVT + c0;
          if (SSM) {  // (x as it lies in LDS where its one part is all of it: from memory it came behind the next chunk's rows, and
                      // every wave waited for it and for them: state space, 56 heads, 3 portions of 4096 tokens 105 us -> 95)
            if constexpr (AP == 1)
              o[b] += skip * widen(*reinterpret_cast<const bf16x4_t*>(Vs + (2 * tb + vh) * 512 + place(quad, ql, vh) * 8 + 4 * b));
            else o[b] += skip * widen(raw4<FULL>(xv + (size_t)(t0 + t) * a.ld, c0, vn));
          }
          if (FULL) *reinterpret_cast<f32x4_t*>(op) = o[b];
          else
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (c0 + i < vn) op[i] = o[b][i];
        }
      }
    }
    // the next q not before the operands made of this one are done with: registers that spilled otherwise, and a spill's way back
    // waits for the fetches before it (state space, 3 x 1365 tokens: 128 -> 117 us; 7 portions of 8192 without SiLU 281 -> 216)
    __builtin_amdgcn_sched_barrier(0);
    if (c + 1 < nch) fetch_q(c + 1);
    // ---- S at the chunk's end: 16 columns (block tb), rows of half vh
    const float end = ends[buf][0];
#pragma unroll
    for (int b = 0; b < ND; ++b) S[b] *= end;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      f32x4_t v[2], by[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf16x4_t vp[AP];
#pragma unroll
        for (int y = 0; y < AP; ++y) vp[y] = ld4t(Vs + y * VN + (2 * (2 * p + e) + (tb >> 1)) * 512, ql, quad, tb >> 1, tb & 1);
        v[e] = join4<AP>(vp), by[e] = *reinterpret_cast<const f32x4_t*>(&sc[buf][5][32 * p + 16 * e + 4 * quad]);
      }
      const Parts<3> wv = split8(v[0], by[0], v[1], by[1]);
#pragma unroll
      for (int b = 0; b < ND; ++b) {
        const int j = vh * ND + b;
        Parts<AP> kt;
#pragma unroll
        for (int y = 0; y < AP; ++y)
          kt.p[y] = join(ld4t(Ks + y * KN + (2 * p * ND + (j >> 1)) * 512, ql, quad, j >> 1, j & 1),
                         ld4t(Ks + y * KN + ((2 * p + 1) * ND + (j >> 1)) * 512, ql, quad, j >> 1, j & 1));
        S[b] = mul(kt, wv, S[b]);
        if (b & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (MODE == 1) lsum += ends[buf][1];
    if (c + 1 < nch) __syncthreads();
  }
  if (c < nch) {
    // Token by token from chunk c on: q, k and v in LDS as they enter the recurrence, the sums of o over a wave's rows behind
    // them.  (Empty asm around the thread's number and the arguments: what is made of them is not carried through the loop above.)
    int me = threadIdx.x;
    const ScanArgs* ap = (const ScanArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+v"(me), "+s"(ap));
    const int mq = me & 15, mquad = (me & 63) >> 4, mcol = 16 * ((me >> 6) & 3) + mq;
    float* qs = reinterpret_cast<float*>(Ks);
    float *ks = qs + LD_MAX, *vs = ks + LD_MAX, *os = vs + LVT;
    double l2 = 0.;
    for (int t = qa + c * LC, stop = qa + qlen; t < stop; ++t) {
      const TI* row = reinterpret_cast<const TI*>(ap->x) + (size_t)t * ap->ld;
      float step = lam, cs = ap->kscale;
      if (SSM) {
        cs = softplus_x(elt(reinterpret_cast<const TI*>(ap->proj) + (size_t)t * ap->pld + ap->dtoff + h) + bias);
        step = expf(-expf(ap->a_log[h]) * cs);
      }
      if (MODE == 1) l2 += SSM ? rate * cs : rate;
      __syncthreads();
      for (int i2 = me; i2 < 2 * ap->d + vn; i2 += LTHREADS) {
        const bool isv = i2 >= 2 * ap->d, isk = !isv && i2 >= ap->d;
        const int i = isv ? i2 - 2 * ap->d : isk ? i2 - ap->d : i2;
        const TI* x = row + (isv ? ap->voff + h * ap->vd + tile * LVT : (isk ? ap->koff : ap->qoff) + (h / ap->R) * ap->d);
        float val = elt(x + i);
        if (ap->act) val = silu_acc(val);
        if (!isv && i < ap->rd) {
          const int half = ap->rd >> 1, fi = i < half ? i : i - half;
          float other = elt(x + (i < half ? i + half : i - half));
          if (ap->act) other = silu_acc(other);
          const float* tab = ap->rope + (size_t)position(t) * ap->rd + fi;
          val = i < half ? val * tab[0] - other * tab[half] : val * tab[0] + other * tab[half];
        }
        if (isk) val *= cs;
        qs[isv ? 2 * LD_MAX + i : isk ? LD_MAX + i : i] = val;
      }
      __syncthreads();
      const float v = vs[mcol];
      float o = 0.f;
#pragma unroll
      for (int b = 0; b < ND; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * ((me >> 8) * ND + b) + 4 * mquad + i;
          if (!FULL && !(mcol < vn && r < ap->d)) continue;
          S[b][i] = fmaf(step, S[b][i], ks[r] * v);
          o = fmaf(S[b][i], qs[r], o);
        }
      if (OUT) {
        o += __shfl_xor(o, 16, 64);
        o += __shfl_xor(o, 32, 64);
        if (mquad == 0) os[(me >> 6) * 16 + mq] = o;
        __syncthreads();
        if (me < vn) {
          float sum = os[me] + os[64 + me];
          if (SSM) sum += ap->skip[h] * elt(row + ap->voff + h * ap->vd + tile * LVT + me);
          ap->out[(size_t)t * ((size_t)ap->H * ap->vd) + h * ap->vd + tile * LVT + me] = sum;
        }
      }
    }
    lsum += (float)l2;
  }
  if (MODE == 1) {
    each([&](int b, int i, int r) { wsg[part * pstep + (size_t)r * a.vd] = S[b][i]; });
    if (tid == 0 && tile == 0) a.wa[((size_t)seq * a.maxparts + part) * a.H + h] = lsum;
  } else if (last && slot_ok) {
    each([&](int b, int i, int r) { Sg[(size_t)r * a.vd] = S[b][i]; });
  }
}

template <typename TI, int AP, bool SSM, bool FULL, int ND>
static hipError_t launch_scan(const ScanArgs& a_in, int nseq, hipStream_t st) {
  ScanArgs a = a_in;
  a.plain = nseq > 64 || (a.maxparts == 1 && a.part <= LC);
  const long blocks = ((long)nseq * a.maxparts * a.H + 7) / 8 * 8 * ((a.vd + LVT - 1) / LVT);
  if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
  if (a.maxparts > 1)
    hipLaunchKernelGGL((linear_scan_kernel<TI, AP, SSM, FULL, ND, 1>), dim3((unsigned)blocks), dim3(LTHREADS), 0, st, a);
  hipLaunchKernelGGL((linear_scan_kernel<TI, AP, SSM, FULL, ND, 2>), dim3((unsigned)blocks), dim3(LTHREADS), 0, st, a);
  return hipGetLastError();
}
template <int AP, bool SSM>
static hipError_t launch_scan_bf16(const ScanArgs& a, int nseq, hipStream_t st) {
  if (a.full && a.d == 32) return launch_scan<bf16, AP, SSM, true, 1>(a, nseq, st);
  if (a.full && a.d == 64) return launch_scan<bf16, AP, SSM, true, 2>(a, nseq, st);
  if (a.full && a.d == 128) return launch_scan<bf16, AP, SSM, true, 4>(a, nseq, st);
  return launch_scan<bf16, AP, SSM, false, 4>(a, nseq, st);
}

}  // namespace grag

using namespace grag;

GRAG_API int grag_linear_scan_max_dim() { return LD_MAX; }

static bool scan_sizes_ok(int nseq, int H, int d, int vd, int part, int max_q_len, const void* ws, const void* wa) {
  if (nseq < 1 || H < 1 || d < 1 || d > LD_MAX || vd < 1 || vd > 256 || part < LC || part % LC || max_q_len < 1) return false;
  return max_q_len <= part || (ws != nullptr && wa != nullptr);
}

// part: tokens per part (a multiple of 64); ws [nseq * ceil(max_q_len / part)][H][d][vd] and wa [..][H] fp32, unused where
// max_q_len <= part.  dt: 0 = bf16, 1 = fp32 rows.  act / rd as grag_decay_attn_scan.
GRAG_API hipError_t grag_linear_scan_decay(const void* proj, int ld, int qoff, int koff, int voff, const float* decay,
                                           float* state, const int* slots, const int* q_start, const int* ctx_len, float* out,
                                           int nseq, int H, int d, int vd, int nslots, int dt, float* ws, float* wa, int part,
                                           int max_q_len, int act, const int* positions, const float* rope_tab, int rd,
                                           int tab_rows, float kscale, hipStream_t st) {
  if (nseq == 0) return hipSuccess;
  if (!scan_sizes_ok(nseq, H, d, vd, part, max_q_len, ws, wa)) return hipErrorInvalidValue;
  if (rd < 0 || rd > d || (rd & 1) || (rd > 0 && (positions == nullptr || rope_tab == nullptr))) return hipErrorInvalidValue;
  ScanArgs a{};
  a.x = proj, a.ld = ld, a.qoff = qoff, a.koff = koff, a.voff = voff, a.R = 1;
  a.state = state, a.slots = slots, a.q_start = q_start, a.ctx_len = ctx_len, a.out = out;
  a.nseq = nseq, a.H = H, a.d = d, a.vd = vd, a.nslots = nslots, a.ws = ws, a.wa = wa;
  a.part = part, a.maxparts = (max_q_len + part - 1) / part;
  a.decay = decay, a.kscale = kscale, a.act = act, a.positions = positions, a.rope = rope_tab, a.rd = rd, a.tab_rows = tab_rows;
  a.full = !((ld | qoff | koff | voff) & 3) && !(vd & 63) && !(rd & 7) && !((uintptr_t)proj & 7) &&
           !(((uintptr_t)out | (uintptr_t)rope_tab) & 15);
  if (dt != 0) return launch_scan<float, 3, false, false, 4>(a, nseq, st);
  if (act || rd) return launch_scan_bf16<3, false>(a, nseq, st);
  return launch_scan_bf16<1, false>(a, nseq, st);
}

GRAG_API hipError_t grag_linear_scan_ssm(const void* xbc, int C, int boff, int coff, const void* proj, int ld, int dtoff,
                                         const float* dt_bias, const float* A_log, const float* Dv, float* state,
                                         const int* slots, const int* q_start, const int* ctx_len, float* out, int nseq, int H,
                                         int G, int N, int P, int nslots, int dt, float* ws, float* wa, int part,
                                         int max_q_len, hipStream_t st) {
  if (nseq == 0) return hipSuccess;
  if (!scan_sizes_ok(nseq, H, N, P, part, max_q_len, ws, wa) || G < 1 || H % G) return hipErrorInvalidValue;
  ScanArgs a{};
  a.x = xbc, a.ld = C, a.qoff = coff, a.koff = boff, a.voff = 0, a.R = H / G;
  a.state = state, a.slots = slots, a.q_start = q_start, a.ctx_len = ctx_len, a.out = out;
  a.nseq = nseq, a.H = H, a.d = N, a.vd = P, a.nslots = nslots, a.ws = ws, a.wa = wa;
  a.part = part, a.maxparts = (max_q_len + part - 1) / part;
  a.proj = proj, a.pld = ld, a.dtoff = dtoff, a.dt_bias = dt_bias, a.a_log = A_log, a.skip = Dv;
  a.full = !((C | boff | coff) & 3) && !(P & 63) && !((uintptr_t)xbc & 7) && !((uintptr_t)out & 15);
  if (dt != 0) return launch_scan<float, 3, true, false, 4>(a, nseq, st);
  return launch_scan_bf16<1, true>(a, nseq, st);
}
