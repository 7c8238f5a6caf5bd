// Common device helpers for the gfx950 (CDNA4 / MI355X) kernel library.
//
// Conventions used by every kernel in csrc/kernels:
//   * bf16 storage is clang's __bf16; conversions go through plain casts so
//     hipcc emits v_cvt_pk_bf16_f32 (NaN-preserving, RNE) — see
//     MI355X_MICROARCH.md "Correctness boundaries".
//   * wave = 64 lanes; block sizes are multiples of 64.
//   * every global load of bf16 data is vectorised to 16 B/lane (bf16x8).
//   * exported entry points are extern "C", take raw device pointers plus the
//     caller's hipStream_t (PyTorch's current stream), and return hipError_t
//     so the Python side can raise loudly.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define GRAG_API extern "C" __attribute__((visibility("default")))

typedef short bf16x8_t __attribute__((ext_vector_type(8)));
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

typedef __bf16 bf16;

namespace grag {

// compute units of the current device (cached per device; a host query, legal during graph capture)
inline int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): register arrays that its number indexes stay in registers,
// also in loops that the unroller would give up on (they would lie in scratch memory)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(static_cast<F&&>(f));
  }
}

__device__ __forceinline__ float bf2f(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 f2bf(float v) { return (bf16)v; }

__device__ __forceinline__ float bits2f(short s) {
  return __uint_as_float(((uint32_t)(uint16_t)s) << 16);
}
__device__ __forceinline__ short f2bits(float f) {
  bf16 b = (bf16)f;
  return __builtin_bit_cast(short, b);
}
// Two floats as a dword of bf16, four as two: one v_cvt_pk_bf16_f32 a pair, where halves that are rounded by themselves and put
// together with a shift take four instructions.  A tile of gemm_chain_kernel stores 64 pairs a lane, behind which a half of the waves
// waits: 272 -> 176 vector instructions for half a tile, 1168 -> 1072 with GELU; 24000 x 3072 x 768 with GELU 139.8 -> 136.8 us, 12000 x
// 1536 x 384 34.4 -> 33.6, with SwiGLU 24.9 -> 24.3; 34 products 0.98 (GELU), 0.988 (SwiGLU) and 0.994 (none) of the time.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16v2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16v4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo, hi}), bf16v2_t));
}
__device__ __forceinline__ bf16x4_t pack4(f32x4_t v) { return __builtin_bit_cast(bf16x4_t, __builtin_convertvector(v, bf16v4_t)); }

// What the bf16 numbers of a pair (pack_bf16x2) leave of the two floats: x -= its half, one v_dot2_f32_bf16 each (p . (-1, 0) + x) where
// the number's way back to fp32 and the difference are two.  Exact for finite pairs whose remainders are normal numbers (one below 2^-126
// is worth nothing in the products, as before); a pair with an infinity or a NaN leaves NaN in both.  The factors are registers: as a
// literal -1 is encoded as the inline constant of an fp32 operand and multiplies the other half.  In the splits of linscan.hip, with the
// pairs' conversions: state space, 3 portions of 4096 tokens, 149 -> 144 us; a decay scan of a hybrid prompt step of 8192 tokens, 20 us of
// 470.
template <bool ADD>
__device__ __forceinline__ void dot_bf16x2(uint32_t p, float& lo, float& hi) {
  uint32_t kl = ADD ? 0x00003f80u : 0x0000bf80u, kh = kl << 16;
  asm("" : "+s"(kl), "+s"(kh));
  const bf16v2_t v = __builtin_bit_cast(bf16v2_t, p);
  lo = __builtin_amdgcn_fdot2_f32_bf16(v, __builtin_bit_cast(bf16v2_t, kl), lo, false);
  hi = __builtin_amdgcn_fdot2_f32_bf16(v, __builtin_bit_cast(bf16v2_t, kh), hi, false);
}
__device__ __forceinline__ void take_bf16x2(uint32_t p, float& lo, float& hi) { dot_bf16x2<false>(p, lo, hi); }
// ... and x += its half, which is exact where the sum is an fp32 number.
__device__ __forceinline__ void add_bf16x2(uint32_t p, float& lo, float& hi) { dot_bf16x2<true>(p, lo, hi); }
// fp32 numbers as the sum of N bf16 parts, and the sum again (one part: as it is)
template <int N> __device__ __forceinline__ void split4(f32x4_t x, bf16x4_t (&p)[N]) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int j = 0; j < N; ++j) {
    u32x2_t d;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float lo = x[2 * i], hi = x[2 * i + 1];
      d[i] = pack_bf16x2(lo, hi);
      if (j + 1 < N) take_bf16x2(d[i], lo, hi);
      x[2 * i] = lo, x[2 * i + 1] = hi;
    }
    p[j] = __builtin_bit_cast(bf16x4_t, d);
  }
}
template <int N> __device__ __forceinline__ f32x4_t join4(const bf16x4_t (&p)[N]) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  f32x4_t x = {bits2f(p[N - 1][0]), bits2f(p[N - 1][1]), bits2f(p[N - 1][2]), bits2f(p[N - 1][3])};
#pragma unroll
  for (int j = N - 2; j >= 0; --j) {  // (the smallest first)
    const u32x2_t d = __builtin_bit_cast(u32x2_t, p[j]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float lo = x[2 * i], hi = x[2 * i + 1];
      add_bf16x2(d[i], lo, hi);
      x[2 * i] = lo, x[2 * i + 1] = hi;
    }
  }
  return x;
}

// LDS-DMA: 16 bytes a lane from rs + off + soff to dst + 16 * lane (no template: the host's pass knows the builtin in none)
typedef __attribute__((address_space(3))) void lds_t;
__device__ __forceinline__ void lds_dma16(const __amdgpu_buffer_rsrc_t& rs, char* dst, unsigned off, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_t*)dst, 16, off, soff, 0, 0);
}

// The (sequence, kv head) stream and the tile of a sequence that workgroup `id` of a causal prompt attention walks: longest walks first,
// the last tile of every sequence, the last but one, and so on.  Workgroups are dealt to the shader engines in turn, 8 XCDs of 4, and
// run where they were dealt; each tile number's streams are turned against those before it, so that every engine meets every
// sequence, also where the streams are a divisor or a multiple of 32 in number (turned by one a tile, an engine saw two of 4
// sequences and the longest one's engines worked on alone).  A list of 32 engines of 8 CUs each tells the measured times within a few
// percent; over 600 random batches this order takes 1.10 of what the chip's share or the longest walk alone allow in the
// geometric mean, turned by one 1.11, sequence by sequence 1.24.
struct WalkOrder { int seq, kvh, tile; };
__device__ __forceinline__ WalkOrder walk_order(unsigned id, unsigned nseq, unsigned kv_heads, unsigned tiles) {
  const unsigned streams = nseq * kv_heads, rank = id / streams;
  const unsigned stream = (id + (rank + rank / 4 + rank / 8) % nseq * kv_heads) % streams;
  return {(int)(stream / kv_heads), (int)(stream % kv_heads), (int)(tiles - 1 - rank)};
}

// a += four consecutive floats of each of S fp32 split-K planes (plane stride `plane` elements), in plane order.
// Up to 16 planes are walked in one fully unrolled, branch-free pass of 2, 4, 8, 12 or 16 (indices past S re-read
// plane 0 and add zero: fma(1, y, x) rounds as x + y), more in passes of 16 before it, so a pass's loads are all in flight
// together -- a runtime-count loop under "#pragma unroll" runs its remainder iterations one plane per memory round trip.
// The boundary norm of 5 rows of 1536 over 18 planes, a round trip a plane past 16 -> two: 6.8 -> 3.9 us, of 16 rows 10.1 -> 4.7.
template <int MAXS>
__device__ __forceinline__ void plane_acc4_fixed(f32x4_t& a, const float* p, size_t plane, int S) {
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
    const bool on = s < S;
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(p + (on ? s : 0) * plane);
    const float m = on ? 1.f : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = __builtin_fmaf(m, v[r], a[r]);
  }
}
__device__ __forceinline__ void plane_acc4(f32x4_t& a, const float* p, size_t plane, int S) {
  for (; S > 16; S -= 16, p += 16 * plane) plane_acc4_fixed<16>(a, p, plane, 16);
  if (S <= 2) {  // (the pass length: the first of 2, 4, 8, 12, 16 >= S)
    plane_acc4_fixed<2>(a, p, plane, S);
  } else if (S <= 4) {
    plane_acc4_fixed<4>(a, p, plane, S);
  } else if (S <= 8) {
    plane_acc4_fixed<8>(a, p, plane, S);
  } else if (S <= 12) {
    plane_acc4_fixed<12>(a, p, plane, S);
  } else {
    plane_acc4_fixed<16>(a, p, plane, S);
  }
}
// the plane sum alone (from -0, the additive identity of every float, so the bits are the plain sum's)
__device__ __forceinline__ f32x4_t plane_sum4(const float* p, size_t plane, int S) {
  f32x4_t a = f32x4_t{-0.f, -0.f, -0.f, -0.f};
  plane_acc4(a, p, plane, S);
  return a;
}

// Unpack a 16-byte bf16x8 vector into 8 floats.
__device__ __forceinline__ void unpack8(const bf16x8_t& v, float* f) {
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = bits2f(v[i]);
}
__device__ __forceinline__ bf16x8_t pack8(const float* f) {
  bf16x8_t v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = f2bits(f[i]);
  return v;
}

// GELU with the normal distribution, x * Phi(x): Phi(-a) = exp2(P(a)) for a >= 0, P the degree-10 minimax fit (Lawson
// iteration, relative weight 1 up to a = 2 and falling to 1e-4 at 6) of log2 of that tail on [0, 5.5]; its leading
// coefficient is negative and P falls on, so larger a end in 0.  The upper half is 1 - Phi(-a).  Against 64 bits over
// [-8, 8]: at most 3.8e-7 in absolute value, where 0.5 x (1 + erff(x / sqrt 2)) has 4.5e-7, and in [-5, -3] 1.1e-5 of
// the value, where that form's 1 + erf cancels to 4.8e-2.  One hardware exponential and ten fmas without a branch:
// erff takes both of its branches in nearly every wave.  Encoder's 24000 x 3072 x 768 product with bias and GELU in the
// epilogue (73.7 M values): 212 us with erff, 182 with this, 142 without an activation; 4000 rows 38.8 -> 30.7 (26.7).
// inf -> inf, -inf -> NaN (-inf * 0), NaN -> NaN as in that form.
__device__ __forceinline__ float gelu_erf(float x) {
  const float a = fabsf(x);
  float p = fmaf(-3.7635938809899017e-08f, a, 1.035111267810862e-06f);
  p = fmaf(p, a, -1.237917513208231e-05f);
  p = fmaf(p, a, 8.218956645578146e-05f);
  p = fmaf(p, a, -0.00029183205333538353f);
  p = fmaf(p, a, 1.169378992926795e-05f);
  p = fmaf(p, a, 0.006946496199816465f);
  p = fmaf(p, a, -0.05244869366288185f);
  p = fmaf(p, a, -0.4592163562774658f);
  p = fmaf(p, a, -1.1511049270629883f);
  p = fmaf(p, a, -1.f);
  const float q = __builtin_amdgcn_exp2f(p);
  return x * (x < 0.f ? q : 1.f - q);
}

// g sigmoid(alpha g) (u + shift) with g = min(g, limit), u = clamp(u, +-limit).  The exponential is the bare instruction, with what
// its argument's products lost put back (largest error of the sigmoid for gates of -80 to 20, alpha 1 / 1.702: 2.4e-7 / 2.4e-7; with
// expf 1.8e-7 / 3.9e-6; without that part 3.8e-6 / 7.6e-6).  The sigmoid is a reciprocal with one correction step (of the
// reciprocal, not of the product with g: an infinite g stays infinite); where the exponential passes 2^126 it is 0.  The clamp of u
// is one instruction, which pays for that part: 4096 tokens x 4 of 16 experts, width 3584, 1242 us without and with.
__device__ __forceinline__ float glu_f(float g, float u, float limit, float alpha, float shift) {
  constexpr float L2E = 1.4426950408889634f, L2E_LO = 1.9259629911266175e-8f;  // log2 e in two parts
  g = fminf(g, limit);
  u = __builtin_amdgcn_fmed3f(u, -limit, limit);
  const float c = -L2E * alpha, cl = fmaf(-L2E_LO, alpha, fmaf(-L2E, alpha, -c)), e = g * c;
  const float lo = fminf(fmaf(g, cl, fmaf(g, c, -e)), 1.f);  // (no number for an infinite g: 1 then, beside t = 0)
  const float t = __builtin_amdgcn_exp2f(e);
  const float d = 1.f + fmaf(0.6931471805599453f * t, lo, t);
  const float rc = __builtin_amdgcn_rcpf(d);
  const float q = fmaf(fmaf(-d, rc, 1.f), rc, rc);
  return g * (e > 126.f ? 0.f : q) * (u + shift);
}

// ---- wave / block reductions (wave64) ----
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Block-wide sum; `red` must hold >= blockDim.x/64 floats of LDS.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}
__device__ __forceinline__ float block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = -INFINITY;
  for (int i = 0; i < nw; ++i) t = fmaxf(t, red[i]);
  return t;
}

// XCD-aware bijective block remap (cdna_hip_programming.md §5 "XCD swizzle
// must be bijective"): blocks that the dispatcher deals to one XCD
// (orig % 8 equal) get a contiguous range of logical tile ids so neighbouring
// tiles share that XCD's L2.  Speed-only; correctness never depends on it.
__device__ __forceinline__ int xcd_remap(int orig, int nwg) {
  const int q = nwg / 8, r = nwg % 8;
  const int xcd = orig % 8;
  const int base = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
  return base + orig / 8;
}

// an element as it is stored, widened where it is used: nothing waits for it before
template <typename T> struct Stored;
template <> struct Stored<bf16> {
  short v;
  __device__ __forceinline__ void load(const bf16* p) { v = *reinterpret_cast<const short*>(p); }
  __device__ __forceinline__ float value() const { return bits2f(v); }
};
template <> struct Stored<float> {
  float v;
  __device__ __forceinline__ void load(const float* p) { v = *p; }
  __device__ __forceinline__ float value() const { return v; }
};

// The sequence with the item-th longest portion (equal ones, and more than 64 sequences, as they come): for workgroups that walk whole
// portions, so that the last ones to start are short.
__device__ __forceinline__ int by_length(const int* q_start, int nseq, int item) {
  if (nseq > 64) return item;
  const int lane = threadIdx.x & 63, own = min(lane, nseq - 1), len = q_start[own + 1] - q_start[own];
  int rank = 0;
  for (int j = 0; j < nseq; ++j) {
    const int o = __builtin_amdgcn_readlane(len, j);
    rank += o > len || (o == len && j < lane);
  }
  return __ffsll((unsigned long long)__ballot(lane < nseq && rank == item)) - 1;
}

// ---- device-side index guard --------------------------------------------------------------------
// Kernels whose addresses come from index INPUTS (token ids, KV slot ids, block-table entries, row ids,
// cross-workgroup tickets) check them.  An out-of-range index skips its access and records (code, value)
// in a small host-mapped error block instead of faulting the device: an illegal address poisons every
// stream of the process and names no kernel, a recorded code names the kernel and the bad value, and the
// host raises on it at its next sync point (ops/_lib.py check_device_errors).  The block pointer is one
// per translation unit (no relocatable device code here), bound once at library load by
// grag_err_bind_<unit>; it is read with plain (scalar) loads and written only with vector atomics.
enum : unsigned {
  ERR_EMBED_TOKEN = 1u << 0,   // decoder embedding gather: token id >= vocab
  ERR_KV_SLOT = 1u << 1,       // RoPE + KV store: slot id >= KV slots
  ERR_ROPE_POS = 1u << 2,      // RoPE: position >= cos/sin table rows
  ERR_BLOCK_PREFILL = 1u << 3, // prefill attention: block-table entry >= KV blocks
  ERR_BLOCK_DECODE = 1u << 4,  // decode attention: block-table entry >= KV blocks
  ERR_TICKET = 1u << 5,        // a split-merge / stream-K ticket past its part count (shared or stale word)
  ERR_SAMPLER_SLOT = 1u << 6,  // sampler / seen-bit row >= sampler slots
  ERR_TOPK_ROW = 1u << 7,      // top-k merge / IVF scan: candidate row or list range out of range
  ERR_BERT_TOKEN = 1u << 8,    // encoder embedding: token / position id out of range
  ERR_PREFIX_GROUP = 1u << 9,  // shared-prefix decode: group row range or prefix length out of range
};

static __device__ unsigned* g_err_block = nullptr;  // [0] codes (OR), [1] last bad value, [2] count, [3] code of [1]

// The block is pinned host memory mapped into the device address space: plain (non-RMW) system-scope
// stores only -- they travel as posted writes on any host link, where read-modify-write atomics to host
// memory would need link atomics.  Two reporters racing may lose one code bit or count: this is a
// diagnostic that something went wrong and where, not a tally.
__device__ __noinline__ void report_index_error(unsigned code, unsigned value) {
  unsigned* e = g_err_block;
  if (e == nullptr) return;
  const unsigned prev = __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(e, prev | code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(e + 1, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const unsigned cnt = __hip_atomic_load(e + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(e + 2, cnt + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(e + 3, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// true when 0 <= v < n; otherwise reports (code, v) and returns false
__device__ __forceinline__ bool index_ok(long v, long n, unsigned code) {
  if (__builtin_expect(v >= 0 && v < n, 1)) return true;
  report_index_error(code, (unsigned)v);
  return false;
}

}  // namespace grag

// exported per translation unit: bind this unit's error-block pointer (host-mapped memory)
#define GRAG_ERR_UNIT(unit)                                                                 \
  GRAG_API int grag_err_bind_##unit(void* p) {                                              \
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(grag::g_err_block), &p, sizeof(p), 0,          \
                                  hipMemcpyHostToDevice);                                   \
  }
