// Fused cosine-score + metadata-filter + top-k for the GPU vector index.
//
// Vectors are stored L2-normalised in bf16, so cosine == dot product.
// S^T[row][q] = X · Q^T on v_mfma_f32_16x16x32_bf16: A = 16 database rows read
// straight from HBM (16 B per lane; each row is read exactly once per launch),
// B = Q^T from an XOR-swizzled LDS image shared by the workgroup's 8 waves.
// A 16-row tile of 1024-d vectors is 32 KB of HBM traffic against 32*NQT MFMAs,
// so the kernel stays HBM-bound and the per-lane top-k upkeep hides under the
// loads.
//
// Top-k: every lane keeps a sorted register list (KMAX) for each of its query
// columns — a lane sees rows 4*(lane>>4)+r of each tile for query lane&15.
// At the end the four lanes of a query merge with two bitonic xor-shuffle
// rounds (top-K of two sorted lists = elementwise max against the reversed
// partner list, then a half-cleaner network), so each wave emits one list per
// query.  In a flat scan the workgroup's waves merge theirs through LDS (three
// rounds), and topk_lists_merge_kernel picks the best of the workgroups' lists.
// (The lists of all waves through a library sort took 15 launches and 100 us.)
// Work items leave a list per wave for grag_topk_merge.
//
// Filters (N3c): up to 4 predicates over dictionary-encoded int32 columns
// (op 1: col == val, op 2: (col & val) != 0 for multi-valued bitset columns)
// plus an optional allow-bitmap, evaluated per row inside the scan.
//
// Two modes:
//   flat : blockIdx.x = row chunk, blockIdx.y = query tile (NQT*16 queries)
//   work : blockIdx.x = work item {row range, NQT*16 query ids} (IVF probes:
//          rows of one inverted list scanned for the queries that probe it)
#include <algorithm>

#include "common.h"

using namespace grag;

namespace {

constexpr int NWAVES = 8;

struct TopkParams {
  const bf16* X;
  int64_t n_rows;
  int d;
  const bf16* Q;
  int nq;
  int k;
  const int32_t* fcol[4];
  int32_t fval[4];
  int32_t fop[4];
  int nfilt;
  const uint32_t* bitmap;
  const int64_t* row_ids;
  int64_t row_begin, row_end, rows_per_wg;
  int nchunks;
  const int64_t* work_rows;  // [nwork][2]
  const int32_t* work_q;     // [nwork][NQT*16]
  // per-query equality predicate (graph traversal: one query per (edge,
  // value) pair): row passes for query q iff qcols[q_colsel[q]][row] == q_val[q]
  // (q_colsel[q] < 0 disables it for that query)
  const int32_t* qcols[8];
  const int32_t* q_colsel;
  const int32_t* q_val;
  float* out_s;
  int64_t* out_i;
};

// A row of a list is one 64-bit float: the score's bits above, the row's offset below, for scores from 0 on inverted, so that of equal
// scores the lower row is the larger number.  The order of the floats is that of the scores (a float's inf is no double's), and to
// exchange two rows takes one maximum and one minimum, where scores and offsets apart take a compare and four selects.  16
// queries of 20K rows, k = 10 / 30: 27.5 us -> 22.8 / 41 -> 31; 24 of 250K 103 -> 94 / 141 -> 116.
__device__ __forceinline__ double list_row(float x, uint32_t off) {
  const int hi = __float_as_int(x);
  return __hiloint2double(hi, (int)(off ^ ~(uint32_t)(hi >> 31)));
}
constexpr float kNone = -INFINITY;
__device__ __forceinline__ double no_row() { return __hiloint2double(__float_as_int(kNone), -1); }
__device__ __forceinline__ float row_score(double r) { return __int_as_float(__double2hiint(r)); }
__device__ __forceinline__ uint32_t row_off(double r) { return (uint32_t)__double2loint(r) ^ ~(uint32_t)(__double2hiint(r) >> 31); }

template <int K>
__device__ __forceinline__ void list_insert(double (&v)[K], double x) {
  if (x > v[K - 1]) {
#pragma unroll
    for (int i = K - 1; i > 0; --i) v[i] = fmax(v[i], fmin(v[i - 1], x));
    v[0] = fmax(v[0], x);
  }
}

// the best K of a sorted list and of another in rising order (w)
template <int K>
__device__ __forceinline__ void list_merge(double (&v)[K], const double (&w)[K]) {
#pragma unroll
  for (int i = 0; i < K; ++i) v[i] = fmax(v[i], w[i]);
  // bitonic half-cleaners -> descending order
#pragma unroll
  for (int j = K / 2; j > 0; j >>= 1) {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      if ((i & j) == 0) {
        const double a = v[i], b = v[i + j];
        v[i] = fmax(a, b);
        v[i + j] = fmin(a, b);
      }
    }
  }
}

template <int K>
__device__ __forceinline__ void list_merge_xor(double (&v)[K], int mask) {
  double w[K];
#pragma unroll
  for (int i = 0; i < K; ++i) w[i] = __shfl_xor(v[K - 1 - i], mask, 64);
  list_merge<K>(v, w);
}

// What the filters ask of rows row .. row + 3 (rows from r1 on: the last one's): a bit per row of the bitmap, a column's value per
// filter and row
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
struct RowKeys {
  uint32_t alive;
  i32x4_t col[4];
};
__device__ __forceinline__ RowKeys row_keys(const TopkParams& p, int64_t row, int64_t r1) {
  RowKeys k;
  k.alive = 15;
  if (p.bitmap) {
    k.alive = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t at = min(row + r, r1 - 1);
      k.alive |= ((p.bitmap[at >> 5] >> (at & 31)) & 1u) << r;
    }
  }
#pragma unroll
  for (int f = 0; f < 4; ++f)
    if (f < p.nfilt)
#pragma unroll
      for (int r = 0; r < 4; ++r) k.col[f][r] = p.fcol[f][min(row + r, r1 - 1)];
  return k;
}
__device__ __forceinline__ bool row_passes(const TopkParams& p, const RowKeys& k, int r) {
  bool ok = (k.alive >> r) & 1u;
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    if (f < p.nfilt) {
      const int32_t c = r < 2 ? (r == 0 ? k.col[f][0] : k.col[f][1]) : (r == 2 ? k.col[f][2] : k.col[f][3]);
      if (p.fop[f] == 1 && c != p.fval[f]) ok = false;
      if (p.fop[f] == 2 && (c & p.fval[f]) == 0) ok = false;
    }
  }
  return ok;
}

template <int NQT, int KMAX>
__global__ __launch_bounds__(64 * NWAVES) void score_topk_kernel(TopkParams p) {
  constexpr int NQ = NQT * 16;
  extern __shared__ __attribute__((aligned(16))) char qlds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h4 = lane >> 4, li = lane & 15;
  const int d = p.d;
  const int RB = 2 * d;   // bytes per query row in LDS
  const int CPR = d / 8;  // 16-B chunks per row
  // XOR swizzle within aligned blocks of SWZ + 1 chunks: SWZ + 1 = the largest power of two (<= 16) dividing
  // CPR, so (ch ^ m) stays inside the row for every d % 32 == 0 (d = 32 / 64 / 96 rows have 4 / 8 / 12
  // chunks: a plain 15-mask would write past the row and past the tile)
  const int SWZ = min(16, CPR & -CPR) - 1;

  int64_t r0, r1;
  int64_t slot_base;
  if (p.work_rows) {
    r0 = p.work_rows[2 * blockIdx.x];
    r1 = p.work_rows[2 * blockIdx.x + 1];
    slot_base = (int64_t)blockIdx.x * NQ;
  } else {
    r0 = p.row_begin + (int64_t)blockIdx.x * p.rows_per_wg;
    r1 = r0 + p.rows_per_wg;
    if (r1 > p.row_end) r1 = p.row_end;
    slot_base = ((int64_t)blockIdx.y * p.nchunks + blockIdx.x) * NQ;
  }

  // A tile's 32-dim steps in batches of U, two batches of registers: one in flight while the other is multiplied, the next tile's
  // first one too, so that 8 waves a CU keep the stream up.  The filters' columns of a tile's rows are loaded ahead of its batches.
  // The loads leave the rows in the caches: those that pass them by (nontemporal) came to 5.25 TB/s where these come to 5.8 (1M x 768,
  // 16 queries 293 -> 267 us, 500K 153 -> 143, other tables read in between), and where a second workgroup reads the rows for more
  // queries it finds some of them there (1M, 60 queries, k = 30: 625 -> 577).
  constexpr int U = NQT == 1 ? 6 : NQT == 2 ? 4 : 3, STEP = 16 * NWAVES;
  const int nc = d / 32;
  bf16x8_t a0[U], a1[U];
  auto load = [&](bf16x8_t (&a)[U], int64_t t0, int c) __attribute__((always_inline)) {
    const bf16* xp = p.X + min(t0 + li, r1 - 1) * d + 8 * h4 + 32 * c;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + u < nc) a[u] = *reinterpret_cast<const bf16x8_t*>(xp + 32 * u);
  };
  const int64_t first = r0 + wave * 16;
  if (first < r1) load(a0, first, 0);  // (ahead of the queries: a small table's first rows take as long to come)

  // stage the query tile: row qq, chunk ch -> qq*RB + ((ch ^ (qq & SWZ)) << 4)
  for (int c = threadIdx.x; c < NQ * CPR; c += 64 * NWAVES) {
    const int qq = c / CPR, ch = c % CPR;
    int qidx;
    if (p.work_rows) qidx = p.work_q[(int64_t)blockIdx.x * NQ + qq];
    else qidx = blockIdx.y * NQ + qq;
    bf16x8_t val = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
    if (qidx >= 0 && qidx < p.nq) val = *reinterpret_cast<const bf16x8_t*>(p.Q + (int64_t)qidx * d + ch * 8);
    *reinterpret_cast<bf16x8_t*>(qlds + qq * RB + ((ch ^ (qq & SWZ)) << 4)) = val;
  }
  __syncthreads();

  // per-lane per-query predicate (column selector, value)
  int qsel[NQT], qv[NQT];
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) {
    qsel[qt] = -1;
    qv[qt] = 0;
    if (p.q_colsel) {
      const int qq = qt * 16 + li;
      const int qidx = p.work_rows ? p.work_q[(int64_t)blockIdx.x * NQ + qq] : (int)blockIdx.y * NQ + qq;
      if (qidx >= 0 && qidx < p.nq) {
        qsel[qt] = p.q_colsel[qidx];
        qv[qt] = p.q_val[qidx];
      }
    }
  }

  double ls[NQT][KMAX];
  static_for<NQT>([&](auto qt) {
#pragma unroll
    for (int i = 0; i < KMAX; ++i) ls[qt][i] = no_row();
  });

#pragma unroll 1
  for (int64_t t0 = first; t0 < r1; t0 += STEP) {
    const RowKeys keys = row_keys(p, t0 + 4 * h4, r1);
    f32x4_t acc[NQT];
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) acc[qt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](const bf16x8_t (&a)[U], int c) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c + u < nc) {
#pragma unroll
          for (int qt = 0; qt < NQT; ++qt) {
            const int qq = qt * 16 + li;
            const int ch = 4 * (c + u) + h4;
            const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(qlds + qq * RB + ((ch ^ (qq & SWZ)) << 4));
            acc[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b, acc[qt], 0, 0, 0);
          }
        }
      }
    };
#pragma unroll 1
    for (int c = 0; c < nc; c += 2 * U) {
      if (c + U < nc) load(a1, t0, c + U);
      mul(a0, c);
      if (c + 2 * U < nc) load(a0, t0, c + 2 * U);
      else if (t0 + STEP < r1) load(a0, t0 + STEP, 0);
      mul(a1, c + U);
    }
#pragma unroll(NQT * KMAX > 32 ? 1 : 4)
    for (int r = 0; r < 4; ++r) {
      const int64_t row = t0 + 4 * h4 + r;
      const bool ok = row < r1 && row_passes(p, keys, r);
      const uint32_t off = (uint32_t)(row - r0);
      static_for<NQT>([&](auto qt) {
        bool okq = ok;
        if (qsel[qt] >= 0 && okq) okq = p.qcols[qsel[qt]][row] == qv[qt];
        const float x = r < 2 ? (r == 0 ? acc[qt][0] : acc[qt][1]) : (r == 2 ? acc[qt][2] : acc[qt][3]);
        list_insert<KMAX>(ls[qt], okq && x > kNone ? list_row(x, off) : no_row());  // (a NaN is no score)
      });
    }
  }

  static_for<NQT>([&](auto qt) {
    list_merge_xor<KMAX>(ls[qt], 16);
    list_merge_xor<KMAX>(ls[qt], 32);
  });
  int lists = NWAVES, mine = wave;  // lists per query of this workgroup, this wave's
  if (!p.work_rows) {  // the waves' lists into wave 0's, over the query tile's LDS
    double* lv = reinterpret_cast<double*>(qlds);
#pragma unroll 1
    for (int half = NWAVES / 2; half > 0; half >>= 1) {
      __syncthreads();
      if (wave >= half && wave < 2 * half && h4 == 0) {
        static_for<NQT>([&](auto qt) {
#pragma unroll
          for (int i = 0; i < KMAX; ++i) {  // (element-major: 16 lanes in a row)
            lv[(((wave - half) * NQT + qt) * KMAX + KMAX - 1 - i) * 16 + li] = ls[qt][i];
          }
        });
      }
      __syncthreads();
      if (wave < half) {
        static_for<NQT>([&](auto qt) {
          double w[KMAX];
#pragma unroll
          for (int i = 0; i < KMAX; ++i) w[i] = lv[((wave * NQT + qt) * KMAX + i) * 16 + li];
          list_merge<KMAX>(ls[qt], w);
        });
      }
    }
    if (wave != 0) return;
    lists = 1;
  }
  if (h4 != 0) return;
  static_for<NQT>([&](auto qt) {
    const int64_t slot = ((slot_base + qt * 16 + li) * lists + mine) * p.k;
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
      if (i >= p.k) continue;
      const float score = row_score(ls[qt][i]);
      const bool valid = score != kNone;
      const int64_t row = r0 + (int64_t)row_off(ls[qt][i]);
      p.out_s[slot + i] = score;
      p.out_i[slot + i] = valid ? (p.row_ids ? p.row_ids[row] : row) : -1;
    }
  });
}

// (value, number) in falling order of value, ties by rising number
__device__ __forceinline__ bool ahead(float v, uint32_t i, float w, uint32_t j) { return v > w || (v == w && i < j); }
constexpr int kMergeLists = 1024;  // lists of a query at most

// A number as one of the same order among the whole numbers, 0 for what no list holds (-inf; NaN); -0 is 0
__device__ __forceinline__ uint32_t order_key(float v) {
  if (!(v > -INFINITY)) return 0;
  const uint32_t b = __float_as_uint(v + 0.f);
  return b ^ ((b >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}

// The final lists of a flat scan: query q's sorted lists of k are rows (q / G * n + j) * G + q % G, j < n <= kMergeLists, of ps /
// pi.  grid (nq), a multiple of 64 threads, no fewer than n.  Only the k lists with the best heads can hold one of the best k, and of
// those only what is not behind the last of these heads: each wave ranks its 64 heads by counting, the best k of each are ranked
// once more, and the elements of the k lists, loaded at once with their ids, as well.  Bound by three ways to memory (lists folded
// one into the next took one for each of a thread's lists and 64 merges in registers).  The whole search with
// 20K rows, 16 queries: k = 10 32.3 us -> 27.5 and k = 30 61 -> 41, against taking the best head k times, a wave's maximum each.
__global__ __launch_bounds__(1024) void topk_lists_merge_kernel(const float* __restrict__ ps, const int64_t* __restrict__ pi, int n,
                                                                int G, int k, float* __restrict__ out_s, int64_t* __restrict__ out_i) {
  __shared__ __attribute__((aligned(16))) uint32_t heads[kMergeLists];
  __shared__ float cv[32 * 32];
  __shared__ uint32_t hk[kMergeLists / 64 * 32], hj[kMergeLists / 64 * 32], best[32], cnum[32 * 32];
  __shared__ int64_t cid[32 * 32];
  __shared__ uint32_t last_key, last_list;
  __shared__ int count, wave_got[kMergeLists / 64];
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, threads = blockDim.x;
  const int64_t base = (int64_t)(q / G) * n * G + q % G;
  if (tid == 0) count = 0, last_key = last_list = 0;  // (key 0: nothing is behind it)
  int picked = n;
  if (n <= k) {  // every list may hold some: nothing is picked (1000 rows, k = 30, the whole search 72 -> 54 us)
    if (tid < n) best[tid] = tid;
  } else {
    const int waves = (n + 63) / 64;
    if (wave < waves) {
      const uint32_t key = tid < n ? order_key(ps[(base + (int64_t)tid * G) * k]) : 0;
      heads[tid] = key;
      __builtin_amdgcn_wave_barrier();  // (a wave's own 64: LDS takes its accesses in order)
      int rank = 0;
      const u32x4_t* of = reinterpret_cast<const u32x4_t*>(heads + wave * 64);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const u32x4_t w = of[i];
#pragma unroll
        for (int u = 0; u < 4; ++u) rank += w[u] > key;
      }
      unsigned long long in = __ballot(key != 0 && rank < k);
      if (__popcll(in) > k) {  // equal heads at the end of the k: the lower lists
        for (int i = 0; i < 64; ++i) rank += heads[wave * 64 + i] == key && i < lane;
        in = __ballot(key != 0 && rank < k);
      }
      const int got = __popcll(in), place = __popcll(in & ((1ull << lane) - 1));
      if (in >> lane & 1) hk[wave * k + place] = key, hj[wave * k + place] = tid;
      if (lane >= got && lane < k) hk[wave * k + lane] = 0, hj[wave * k + lane] = 0;
      if (lane == 0) wave_got[wave] = got;
    }
    __syncthreads();
    int all = 0;
    for (int w = 0; w < waves; ++w) all += wave_got[w];
    picked = min(all, k);
    for (int x = tid >> 2; x < waves * k; x += threads / 4) {
      const uint32_t key = hk[x], j = hj[x];
      int rank = 0;
      for (int i = tid & 3; i < waves * k; i += 4) rank += hk[i] > key || (hk[i] == key && hj[i] < j);
      rank += __shfl_xor(rank, 1, 64);
      rank += __shfl_xor(rank, 2, 64);
      if ((tid & 3) == 0 && key != 0 && rank < k) {
        best[rank] = j;
        if (rank == k - 1) last_key = key, last_list = j;
      }
    }
  }
  __syncthreads();
  for (int e = tid; e < picked * k; e += threads) {
    const uint32_t j = best[e / k];
    const int t = e % k;
    const int64_t at = (base + (int64_t)j * G) * k + t;
    const float v = ps[at];
    const int64_t id = pi[at];
    const uint32_t key = order_key(v);
    // (of lists with equal values the heads decide: behind the last head's list nothing that equals it is among the best)
    if (key != 0 && (key > last_key || (key == last_key && j <= last_list))) {
      const int c = atomicAdd(&count, 1);
      cv[c] = v, cnum[c] = j * (uint32_t)k + t, cid[c] = id;
    }
  }
  __syncthreads();
  const int c = count;
  for (int x = tid >> 2; x < c; x += threads / 4) {
    const float v = cv[x];
    const uint32_t m = cnum[x];
    int rank = 0;
    for (int i = tid & 3; i < c; i += 4) rank += ahead(cv[i], cnum[i], v, m);
    rank += __shfl_xor(rank, 1, 64);
    rank += __shfl_xor(rank, 2, 64);
    if ((tid & 3) == 0 && rank < k) {
      out_s[(int64_t)q * k + rank] = v;
      out_i[(int64_t)q * k + rank] = cid[x];
    }
  }
  for (int r = c + tid; r < k; r += threads) {
    out_s[(int64_t)q * k + r] = -INFINITY;
    out_i[(int64_t)q * k + r] = -1;
  }
}

template <int NQT, int KMAX>
int launch_topk(const TopkParams& prm, dim3 grid, hipStream_t stream) {
  const size_t merge = (size_t)NWAVES / 2 * NQT * 16 * KMAX * 8;  // the waves' lists, where the query tile was
  const size_t lds = std::max((size_t)NQT * 16 * prm.d * 2, prm.work_rows ? (size_t)0 : merge);
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute((const void*)score_topk_kernel<NQT, KMAX>,
                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_set = true;
  }
  score_topk_kernel<NQT, KMAX><<<grid, 64 * NWAVES, lds, stream>>>(prm);
  return (int)hipGetLastError();
}

int dispatch(const TopkParams& prm, int nqt, int kmax, dim3 grid, hipStream_t stream) {
  if (kmax == 16) {
    if (nqt == 1) return launch_topk<1, 16>(prm, grid, stream);
    if (nqt == 2) return launch_topk<2, 16>(prm, grid, stream);
    if (nqt == 4) return launch_topk<4, 16>(prm, grid, stream);
  } else if (kmax == 32) {
    if (nqt == 1) return launch_topk<1, 32>(prm, grid, stream);
    if (nqt == 2) return launch_topk<2, 32>(prm, grid, stream);
  }
  return (int)hipErrorInvalidValue;
}

void fill_qfilters(TopkParams& prm, const int32_t* const* qcols, int nqcols, const int32_t* q_colsel,
                   const int32_t* q_val) {
  for (int i = 0; i < 8; ++i) prm.qcols[i] = (qcols && i < nqcols) ? qcols[i] : nullptr;
  prm.q_colsel = q_colsel;
  prm.q_val = q_val;
}

void fill_filters(TopkParams& prm, const int32_t* const* fcols, const int32_t* fvals,
                  const int32_t* fops, int nfilt) {
  prm.nfilt = nfilt;
  for (int i = 0; i < 4; ++i) {
    prm.fcol[i] = i < nfilt ? fcols[i] : nullptr;
    prm.fval[i] = i < nfilt ? fvals[i] : 0;
    prm.fop[i] = i < nfilt ? fops[i] : 0;
  }
}

}  // namespace

GRAG_API int grag_topk_num_waves() { return NWAVES; }

// The final top-k of a flat scan's lists (out_s / out_i of grag_score_topk_flat): [nq][k], -1 where fewer rows passed.
GRAG_API int grag_topk_lists_merge(const float* ps, const int64_t* pi, int n, int G, int nq, int k, float* out_s,
                                   int64_t* out_i, hipStream_t stream) {
  if (nq <= 0) return 0;
  if (n < 1 || n > kMergeLists || G < 1 || k < 1 || k > 32) return (int)hipErrorInvalidValue;
  topk_lists_merge_kernel<<<nq, std::max(k > 16 ? 1024 : 256, (n + 63) / 64 * 64), 0, stream>>>(ps, pi, n, G, k, out_s, out_i);
  return (int)hipGetLastError();
}

// Flat scan.  Output slots: [nqtiles][nchunks][nqt*16][k].
GRAG_API int grag_score_topk_flat(const void* X, int64_t row_begin, int64_t row_end,
                                  int64_t rows_per_wg, int d, const void* Q, int nq, int k,
                                  int nqt, int kmax, const int32_t* const* fcols,
                                  const int32_t* fvals, const int32_t* fops, int nfilt,
                                  const uint32_t* bitmap, const int64_t* row_ids,
                                  const int32_t* const* qcols, int nqcols, const int32_t* q_colsel,
                                  const int32_t* q_val, float* out_s, int64_t* out_i,
                                  hipStream_t stream) {
  if (nq <= 0 || row_end <= row_begin) return 0;
  if (nqcols > 8) return (int)hipErrorInvalidValue;
  if (d % 32 != 0 || k > kmax || nfilt > 4 || rows_per_wg <= 0) return (int)hipErrorInvalidValue;
  TopkParams prm{};
  prm.X = (const bf16*)X;
  prm.n_rows = row_end;
  prm.d = d;
  prm.Q = (const bf16*)Q;
  prm.nq = nq;
  prm.k = k;
  fill_filters(prm, fcols, fvals, fops, nfilt);
  prm.bitmap = bitmap;
  prm.row_ids = row_ids;
  prm.row_begin = row_begin;
  prm.row_end = row_end;
  prm.rows_per_wg = rows_per_wg;
  prm.nchunks = (int)((row_end - row_begin + rows_per_wg - 1) / rows_per_wg);
  fill_qfilters(prm, qcols, nqcols, q_colsel, q_val);
  prm.out_s = out_s;
  prm.out_i = out_i;
  const int nqtiles = (nq + nqt * 16 - 1) / (nqt * 16);
  return dispatch(prm, nqt, kmax, dim3(prm.nchunks, nqtiles), stream);
}

// Work-item scan (IVF).  Output slots: [nwork][nqt*16][NWAVES][k].
GRAG_API int grag_score_topk_work(const void* X, int d, const void* Q, int nq, int k, int nqt,
                                  int kmax, const int64_t* work_rows, const int32_t* work_q,
                                  int nwork, const int32_t* const* fcols, const int32_t* fvals,
                                  const int32_t* fops, int nfilt, const uint32_t* bitmap,
                                  const int64_t* row_ids, const int32_t* const* qcols, int nqcols,
                                  const int32_t* q_colsel, const int32_t* q_val, float* out_s,
                                  int64_t* out_i, hipStream_t stream) {
  if (nwork <= 0) return 0;
  if (nqcols > 8) return (int)hipErrorInvalidValue;
  if (d % 32 != 0 || k > kmax || nfilt > 4) return (int)hipErrorInvalidValue;
  TopkParams prm{};
  prm.X = (const bf16*)X;
  prm.d = d;
  prm.Q = (const bf16*)Q;
  prm.nq = nq;
  prm.k = k;
  fill_filters(prm, fcols, fvals, fops, nfilt);
  prm.bitmap = bitmap;
  prm.row_ids = row_ids;
  prm.work_rows = work_rows;
  prm.work_q = work_q;
  fill_qfilters(prm, qcols, nqcols, q_colsel, q_val);
  prm.out_s = out_s;
  prm.out_i = out_i;
  return dispatch(prm, nqt, kmax, dim3(nwork), stream);
}
