// Standalone operators at the reference's kernel boundary
// (suffix_gpu/triton_kernels.py): scatter_append, match_back,
// first_occurrences, sa_search and expand_chain.  The fused decode step
// uses the same device building blocks; these entry points expose them one
// at a time for the index-level API and for parity checks.

#include <algorithm>

#include "launch.h"
#include "pick.h"
#include "sa_search.h"
#include "sfx_common.h"

namespace sfx {

// ---------------------------------------------------------- scatter_append
__global__ __launch_bounds__(64) void k_scatter(sfx_batch bt,
                                                int32_t* new_counts) {
  const int b = blockIdx.x;
  const RowState st = row_state(bt, b);
  const int64_t S = bt.seq;
  const int32_t* sp = bt.sampled + (int64_t)b * bt.num_sampled;
  for (int64_t j = threadIdx.x; j < bt.num_sampled; j += blockDim.x) {
    const int64_t pos = st.base + j;
    const int32_t v = sp[j];
    if (j < st.cnt && v != -1 && pos < S && pos >= 0)
      bt.tokens[(int64_t)b * S + pos] = v;
  }
  if (new_counts && threadIdx.x == 0) new_counts[b] = (int32_t)st.q;
}

// ---------------------------------------------------------- index swap
// Up to three buffer copies in one grid-stride launch: 16-byte words where
// both sides are 16-byte aligned, single words for the rest.
struct CopySpan {
  int32_t* dst;
  const int32_t* src;
  int64_t n;
};

__device__ __forceinline__ void copy_span(const CopySpan& c, int64_t tid,
                                          int64_t nthreads) {
  if (c.n <= 0) return;
  const bool vec = ((reinterpret_cast<uintptr_t>(c.dst) |
                     reinterpret_cast<uintptr_t>(c.src)) & 15u) == 0;
  const int64_t n4 = vec ? c.n / 4 : 0;
  const int4* s4 = reinterpret_cast<const int4*>(c.src);
  int4* d4 = reinterpret_cast<int4*>(c.dst);
  for (int64_t i = tid; i < n4; i += nthreads) d4[i] = s4[i];
  for (int64_t i = 4 * n4 + tid; i < c.n; i += nthreads) c.dst[i] = c.src[i];
}

// The swap's in-place copies of corpus and SA; block 0 also stores the
// key-row selector word (a vector store from one lane).
__global__ __launch_bounds__(256) void k_swap(CopySpan a, CopySpan b,
                                              int32_t* key_select,
                                              int32_t key_select_value) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nth = (int64_t)gridDim.x * blockDim.x;
  copy_span(a, tid, nth);
  copy_span(b, tid, nth);
  if (key_select && tid == 0) *key_select = key_select_value;
}

// ------------------------------------------------------------ delta writes
// Appends up to SFX_APPEND_MAX_DOCS documents: block (x, d) copies a
// grid-stride share of document d, block (0, d) also writes its SEP and
// block (0, 0) the new delta length.
struct AppendDocs {
  sfx_append_doc doc[SFX_APPEND_MAX_DOCS];
};

__global__ __launch_bounds__(256) void k_delta_append(AppendDocs docs,
                                                      int32_t* delta,
                                                      int64_t* delta_len,
                                                      int64_t new_len) {
  const sfx_append_doc& d = docs.doc[blockIdx.y];
  int32_t* out = delta + d.dst;
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nth = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = tid; i < d.n; i += nth) out[i] = d.src[i];
  if (tid == 0) out[d.n] = kSep;
  if (tid == 0 && blockIdx.y == 0 && delta_len) *delta_len = new_len;
}

// delta[0 .. n) = delta[from .. from + n) in place (from > 0), by one
// block in ascending windows: a window's sources are all read before the
// barrier, and its writes only land on sources of outputs at or below the
// window, which are read already.
constexpr int kShiftThreads = 1024;
constexpr int kShiftPer = 8;

__global__ __launch_bounds__(kShiftThreads) void k_delta_shift(
    int32_t* delta, int64_t from, int64_t n, int64_t* delta_len,
    int64_t new_len) {
  constexpr int64_t W = (int64_t)kShiftThreads * kShiftPer;
  for (int64_t k = 0; k < n; k += W) {
    int32_t v[kShiftPer];
#pragma unroll
    for (int u = 0; u < kShiftPer; ++u) {
      const int64_t o = k + u * kShiftThreads + threadIdx.x;
      v[u] = o < n ? delta[from + o] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kShiftPer; ++u) {
      const int64_t o = k + u * kShiftThreads + threadIdx.x;
      if (o < n) delta[o] = v[u];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0 && delta_len) *delta_len = new_len;
}

// -------------------------------------------------------------- match_back
__global__ __launch_bounds__(256) void k_match_back(
    const int32_t* __restrict__ src, int64_t row_stride,
    const int32_t* __restrict__ pat, int P, int64_t n_out, int32_t* out) {
  const int b = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_out) return;
  const int32_t* base = src + (int64_t)b * row_stride;
  const int32_t* pb = pat + (int64_t)b * P;
  int m = 0;
  for (int t = 0; t < P; ++t) {
    const int64_t j = i - 1 - t;
    const int32_t x = j >= 0 ? base[j] : -1;
    if (x != pb[t]) break;
    ++m;
  }
  out[(int64_t)b * n_out + i] = m;
}

// ------------------------------------------------------- first_occurrences
// One workgroup per threshold row, four columns per thread and pass: a pass
// is a chain of a load, a count over the waves and a barrier, so wide passes
// with the next one's columns on their way beat narrow ones as long as the
// workgroups leave room for them (occ_threads).  Rows of at most kOccMin
// columns take one column per thread.  The launch alone, us, a column per
// thread with three barriers a pass / four columns and 1024 threads for every
// row / now: 64 rows of 8,192 columns with 8 thresholds each 13.1 / 5.6 / 4.8
// where few columns reach them (9.8 / 4.8 / 4.0 where many do), 256 such rows
// 21.9 / 18.3 / 13.0, 16 rows of 65,536 85.4 / 16.7 / 15.5, 256 rows of 512
// 4.0 / 11.8 / 4.0, 64 rows of 128 2.6 / 4.5 / 2.6.
typedef int32_t Int4Any __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kOccMin = 256;
constexpr int64_t kOccLongRow = 4096;

// 1024 threads while one such workgroup per CU holds every threshold row, 512
// while two or four do, if a row is long enough for several narrow passes:
// rows of 4,096 columns (64 x 8 thresholds) 4.2 us with 256 threads, 3.7 with
// 512; of 2,048 columns 3.3 and 3.2, of 1,024 2.8 and 3.2.
inline int occ_threads(int64_t n_cols, int64_t rows) {
  if (n_cols < kOccLongRow || rows > 1024) return 256;
  return rows <= 256 ? 1024 : 512;
}

template <int NT, int kCols>
__global__ __launch_bounds__(NT) void k_first_occ(
    const int32_t* __restrict__ mb, int64_t n_cols,
    const int64_t* __restrict__ thr, int64_t per_row, int R, int64_t* pos,
    int64_t* count) {
  static_assert(kCols == 1 || kCols == 4, "one load per thread and pass");
  constexpr int NW = NT / kWave;
  constexpr int64_t kPass = (int64_t)NT * kCols;
  __shared__ int wcnt[2][NW];  // by pass parity: one barrier per pass
  const int64_t row = blockIdx.x;
  const int64_t b = row / per_row;
  const int tid = threadIdx.x;
  const int wv = tid / kWave;
  const int64_t t = thr[row];
  const int32_t* src = mb + b * n_cols;
  int64_t* out = pos + row * R;
  int found = 0;  // the same in every thread
  if (t > 0) {
    auto load = [&](int64_t i, int32_t (&v)[kCols]) {
      if (kCols == 4 && i + kCols <= n_cols) {
        const Int4Any w = *reinterpret_cast<const Int4Any*>(src + i);
#pragma unroll
        for (int u = 0; u < kCols; ++u) v[u] = w[u];
      } else {  // (t > 0: a column past the end never hits)
#pragma unroll
        for (int u = 0; u < kCols; ++u) v[u] = i + u < n_cols ? src[i + u] : 0;
      }
    };
    int32_t cur[kCols], nxt[kCols];
    load((int64_t)tid * kCols, cur);
    int par = 0;
    for (int64_t base = 0; base < n_cols; base += kPass, par ^= 1) {
      const int64_t i = base + (int64_t)tid * kCols;
      if (base + kPass < n_cols) load(i + kPass, nxt);
      bool hit[kCols];
      int below = 0, tot = 0;  // hits of lower lanes, of the wave
#pragma unroll
      for (int u = 0; u < kCols; ++u) {
        hit[u] = (int64_t)cur[u] >= t;
        const uint64_t bm = ballot(hit[u]);
        below += rank_lt(bm);
        tot += popc(bm);
      }
      if (lane_id() == 0) wcnt[par][wv] = tot;
      __syncthreads();
      int slot = found + below;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int c = wcnt[par][w];
        slot += w < wv ? c : 0;
        found += c;
      }
#pragma unroll
      for (int u = 0; u < kCols; ++u) {
        if (hit[u] && slot < R) out[slot] = i + u;
        slot += hit[u];
      }
      if (found >= R) break;
#pragma unroll
      for (int u = 0; u < kCols; ++u) cur[u] = nxt[u];
    }
  }
  const int f = found < R ? found : R;
  for (int r = tid; r < R; r += NT)
    if (r >= f) out[r] = 0;
  if (tid == 0) count[row] = f;
}

// --------------------------------------------------------------- sa_search
// A search is a chain of dependent rounds (a suffix position, then its
// tokens), so what bounds a call is rounds times two memory round trips
// until the lanes fill the chip, and the probes' reads from then on.
// G = 32 lanes per pattern, compared by octets (short patterns by a lane per
// probe), cut 2^22 ranks in 5 rounds; G = 8 with a lane per probe takes 7,
// each with a dependent load per 4 matched tokens, but reads 2.5 times fewer
// probes.  Calls over 4,193,504 suffixes with G = 8 / G = 32, us: patterns of
// 1 .. 32 tokens, 2,048 of them 35.3 / 12.5, 8,192 44.0 / 26.4, 16,384 53.2 /
// 45.2, 32,768 63.0 / 78.0 (over 20,000 suffixes 22.1 / 9.7, 24.6 / 13.8, 26.2
// / 22.3, 28.9 / 37.4); of 1 token, 2,048 9.3 / 7.0, 4,096 10.5 / 8.8, 8,192
// 12.5 / 13.1, 16,384 16.4 / 25.3; of 4 tokens, 4,096 13.3 / 11.5, 8,192 15.8
// / 17.3.  So G = 32 up to 4,096 patterns of at most 4 tokens, and up to 8,192
// longer ones (past that, those that turn out short would lose more than the
// long ones gain).
constexpr int kSearchThreads = 256;

template <int G, bool kOct>
__global__ __launch_bounds__(kSearchThreads) void k_sa_search(
    const int32_t* __restrict__ sa, const int32_t* __restrict__ corpus,
    int64_t n, const int32_t* __restrict__ pattern, int64_t batch,
    int64_t width, const int64_t* __restrict__ plen, int64_t* lower,
    int64_t* upper) {
  const int64_t row = (int64_t)blockIdx.x * (kSearchThreads / G) +
                      threadIdx.x / G;
  if (row >= batch) return;  // whole groups exit together
  const int32_t* pr = pattern + row * width;
  int64_t pl = plen[row];
  pl = pl < 0 ? 0 : (pl > width ? width : pl);
  auto pat_at = [&](int j) -> int32_t { return pr[j]; };
  int64_t lo, hi;
  kary_bounds<G, kOct>(sa, corpus, n, nullptr, 0, pat_at, (int)pl, lo, hi,
                       0u, (uint32_t)n);
  if (threadIdx.x % G == 0) {
    lower[row] = lo;
    upper[row] = hi;
  }
}

// ------------------------------------------------------------ expand_chain
struct ExpandArgs {
  const int32_t* cont;
  int64_t rows;
  int R;
  int K;
  const int64_t* num_occ;
  const int64_t* cap;
  const float* weights;
  float min_prob;
  float alpha;
  int32_t* chain;
  int64_t* num_valid;
  int64_t* num_emit;
  float* score;
  int waves_per_block;
};

__host__ __device__ inline int round16(int x) { return (x + 15) & ~15; }

// Per-wave LDS: continuation cache [R, K + 1], vote buffer A [R],
// weights W [R],
// chain [K]; every region 16-byte aligned.
__host__ __device__ inline int expand_wave_bytes(int R, int K) {
  return round16(R * (K + 1) * 4) + 2 * round16(R * 4) + round16(K * 4) +
         2 * kHashSlots * 4;
}

template <bool kWeighted>
__global__ __launch_bounds__(256) void k_expand(ExpandArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int wv = threadIdx.x / kWave;
  const int ln = threadIdx.x % kWave;
  const int64_t row = (int64_t)blockIdx.x * a.waves_per_block + wv;
  if (wv >= a.waves_per_block || row >= a.rows) return;
  const int R = a.R;
  const int K = a.K;
  unsigned char* base = smem + (size_t)wv * expand_wave_bytes(R, K);
  const int cb = round16(R * (K + 1) * 4);
  int32_t* cache = (int32_t*)base;
  int32_t* A = (int32_t*)(base + cb);
  float* W = (float*)(base + cb + round16(R * 4));
  int32_t* chain = (int32_t*)(base + cb + 2 * round16(R * 4));
  int32_t* H = (int32_t*)(base + cb + 2 * round16(R * 4) + round16(K * 4));
  const int32_t* src = a.cont + row * R * K;
  // rows K + 1 words apart (an odd stride): one depth's rows fall in
  // distinct LDS banks for the expansion's per-lane reads
  for (int e = ln; e < R * K; e += kWave)
    cache[(e / K) * (K + 1) + e % K] = src[e];
  wave_lds_sync();
  const int64_t occ = a.num_occ[row];
  const int64_t cap = a.cap ? a.cap[row] : K;
  auto cont_at = [&](int r, int d) -> int32_t { return cache[r * (K + 1) + d]; };
  const float* wrow = a.weights ? a.weights + row * R : nullptr;
  auto w_at = [&](int r) -> float { return wrow[r]; };
  ExpandResult er;
  if (kWeighted)
    er = expand_wave<true>(cont_at, w_at, R, occ, K, cap, a.min_prob,
                           a.alpha, A, W, H, chain);
  else
    er = expand_wave<false>(cont_at, NoWeight(), R, occ, K, cap, a.min_prob,
                            a.alpha, A, W, H, chain);
  wave_lds_sync();
  for (int d = ln; d < K; d += kWave) a.chain[row * K + d] = chain[d];
  if (ln == 0) {
    const int64_t cap0 = cap > 0 ? cap : 0;
    a.num_valid[row] = er.nv;
    a.num_emit[row] = er.nv < cap0 ? er.nv : cap0;
    a.score[row] = er.score;
  }
}

}  // namespace sfx

using namespace sfx;

#ifdef SFX_TRACE
__constant__ uint64_t* sfx_trace_buf = nullptr;
__constant__ uint64_t* sfx_trace_stats = nullptr;

// Profiling builds only: per-wave expansion counters (8 u64 per wave).
extern "C" int sfx_trace_stats_set(uint64_t* buf) {
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(sfx_trace_stats), &buf,
                                sizeof(buf));
}

// Profiling builds only: point the phase-timestamp buffer (device memory,
// 16 u64 per block) at `buf`, or disable with NULL.
extern "C" int sfx_trace_set(uint64_t* buf) {
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(sfx_trace_buf), &buf,
                                sizeof(buf));
}
#endif

extern "C" int sfx_abi_version(void) { return SFX_ABI_VERSION; }

extern "C" int sfx_index_swap(int32_t* corpus, int32_t* sa,
                              const int32_t* new_corpus,
                              const int32_t* new_sa, int64_t capacity,
                              int32_t* key_select, int32_t key_select_value,
                              hipStream_t stream) {
  if (capacity < 0) return SFX_EINVAL;
  if (capacity == 0 && !key_select) return 0;
  if (capacity > 0 && (!corpus || !sa || !new_corpus || !new_sa))
    return SFX_EINVAL;
  const CopySpan a{corpus, new_corpus, capacity};
  const CopySpan b{sa, new_sa, capacity};
  // Up to eight 256-thread blocks per CU keep every CU streaming (32 MiB
  // of copies at N = 2^22).
  const int64_t want = (capacity / 4 + 255) / 256;
  const unsigned blocks =
      (unsigned)(want < 1 ? 1 : (want > 2048 ? 2048 : want));
  hipLaunchKernelGGL(k_swap, dim3(blocks), dim3(256), 0, stream, a, b,
                     key_select, key_select_value);
  return (int)hipGetLastError();
}

extern "C" int sfx_delta_append(const sfx_append_doc* docs, int32_t ndocs,
                                int32_t* delta, int64_t delta_capacity,
                                int64_t* delta_len, int64_t new_len,
                                hipStream_t stream) {
  if (ndocs < 0 || delta_capacity < 0 || new_len < 0 ||
      new_len > delta_capacity || (ndocs > 0 && (!docs || !delta)))
    return SFX_EINVAL;
  int64_t longest = 0;
  for (int32_t i = 0; i < ndocs; ++i) {
    const sfx_append_doc& d = docs[i];
    if (d.n < 0 || d.dst < 0 || d.dst + d.n + 1 > delta_capacity ||
        (d.n > 0 && !d.src))
      return SFX_EINVAL;
    longest = d.n > longest ? d.n : longest;
  }
  if (ndocs == 0) {
    if (!delta_len) return 0;
    hipLaunchKernelGGL(k_delta_shift, dim3(1), dim3(kShiftThreads), 0,
                       stream, delta, (int64_t)0, (int64_t)0, delta_len,
                       new_len);
    return (int)hipGetLastError();
  }
  const unsigned bx = (unsigned)std::min<int64_t>(
      std::max<int64_t>((longest + 1023) / 1024, 1), 64);
  for (int32_t g = 0; g < ndocs; g += SFX_APPEND_MAX_DOCS) {
    const int32_t cnt = std::min<int32_t>(ndocs - g, SFX_APPEND_MAX_DOCS);
    AppendDocs a = {};
    for (int32_t i = 0; i < cnt; ++i) a.doc[i] = docs[g + i];
    hipLaunchKernelGGL(k_delta_append, dim3(bx, (unsigned)cnt), dim3(256), 0,
                       stream, a, delta, delta_len, new_len);
    const int rc = (int)hipGetLastError();
    if (rc) return rc;
  }
  return 0;
}

extern "C" int sfx_delta_shift(int32_t* delta, int64_t delta_capacity,
                               int64_t from, int64_t n, int64_t* delta_len,
                               hipStream_t stream) {
  if (!delta || from < 0 || n < 0 || from + n > delta_capacity)
    return SFX_EINVAL;
  if (from == 0 && !delta_len) return 0;
  hipLaunchKernelGGL(k_delta_shift, dim3(1), dim3(kShiftThreads), 0, stream,
                     delta, from, from > 0 ? n : 0, delta_len, n);
  return (int)hipGetLastError();
}

extern "C" int sfx_scatter_append(const sfx_batch* bt, int32_t* new_counts,
                                  hipStream_t stream) {
  if (!bt || bt->batch < 0 || bt->seq < 1 || !bt->tokens ||
      !bt->num_tokens || !bt->sampled || bt->num_sampled < 0)
    return SFX_EINVAL;
  if (bt->batch == 0) return 0;
  hipLaunchKernelGGL(k_scatter, dim3((unsigned)bt->batch), dim3(64), 0,
                     stream, *bt, new_counts);
  return (int)hipGetLastError();
}

extern "C" int sfx_match_back(const int32_t* src, int64_t row_stride,
                              const int32_t* pat, int64_t batch,
                              int64_t pattern_len, int64_t n_out,
                              int32_t* out, hipStream_t stream) {
  if (batch < 0 || pattern_len < 0 || n_out < 0 || row_stride < 0)
    return SFX_EINVAL;
  if (batch == 0 || n_out == 0) return 0;
  if (!src || !out || (pattern_len > 0 && !pat)) return SFX_EINVAL;
  if (batch > 65535) return SFX_EINVAL;
  dim3 grid((unsigned)((n_out + 255) / 256), (unsigned)batch);
  hipLaunchKernelGGL(k_match_back, grid, dim3(256), 0, stream, src,
                     row_stride, pat, (int)pattern_len, n_out, out);
  return (int)hipGetLastError();
}

extern "C" int sfx_first_occurrences(const int32_t* mb, int64_t n_cols,
                                     const int64_t* thr, int64_t rows,
                                     int64_t per_row, int64_t max_occ,
                                     int64_t* pos, int64_t* count,
                                     hipStream_t stream) {
  if (rows < 0 || n_cols < 0 || per_row < 1 || max_occ < 1) return SFX_EINVAL;
  if (rows == 0) return 0;
  if (!mb || !thr || !pos || !count) return SFX_EINVAL;
  if (max_occ > 0x7fffffff) return SFX_EINVAL;
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(threads), 0, stream,
                       mb, n_cols, thr, per_row, (int)max_occ, pos, count);
  };
  const int nt = occ_threads(n_cols, rows);
  if (n_cols <= kOccMin)
    launch(k_first_occ<kOccMin, 1>, kOccMin);
  else if (nt == 256)
    launch(k_first_occ<256, 4>, 256);
  else if (nt == 512)
    launch(k_first_occ<512, 4>, 512);
  else
    launch(k_first_occ<1024, 4>, 1024);
  return (int)hipGetLastError();
}

constexpr int64_t kWideSearchMax = 1 << 13;
constexpr int64_t kWideShortMax = 1 << 12;  // patterns of at most 4 tokens

extern "C" int sfx_sa_search(const int32_t* sa, const int32_t* corpus,
                             int64_t n, const int32_t* pattern,
                             int64_t batch, int64_t width,
                             const int64_t* plen, int64_t* lower,
                             int64_t* upper, hipStream_t stream) {
  if (batch < 0 || n < 1 || n > 0x7fffffffLL || width < 0) return SFX_EINVAL;
  if (batch == 0) return 0;
  if (!sa || !corpus || !plen || !lower || !upper ||
      (width > 0 && !pattern))
    return SFX_EINVAL;
  const bool wide = batch <= (width <= 4 ? kWideShortMax : kWideSearchMax);
  const int64_t per_block = kSearchThreads / (wide ? 32 : 8);
  const int64_t blocks = (batch + per_block - 1) / per_block;
  if (wide)
    hipLaunchKernelGGL((k_sa_search<32, true>), dim3((unsigned)blocks),
                       dim3(kSearchThreads), 0, stream, sa, corpus, n,
                       pattern, batch, width, plen, lower, upper);
  else
    hipLaunchKernelGGL((k_sa_search<8, false>), dim3((unsigned)blocks),
                       dim3(kSearchThreads), 0, stream, sa, corpus, n,
                       pattern, batch, width, plen, lower, upper);
  return (int)hipGetLastError();
}

extern "C" int sfx_expand_chain(const int32_t* cont, int64_t rows,
                                int64_t max_occ, int64_t k,
                                const int64_t* num_occ, const int64_t* cap,
                                const float* weights, float min_token_prob,
                                float alpha, int32_t* chain,
                                int64_t* num_valid, int64_t* num_emit,
                                float* score, hipStream_t stream) {
  if (rows < 0 || max_occ < 1 || max_occ > 2048 || k < 1 || k > 4096)
    return SFX_EINVAL;
  if (rows == 0) return 0;
  if (!cont || !num_occ || !chain || !num_valid || !num_emit || !score)
    return SFX_EINVAL;
  ExpandArgs a;
  a.cont = cont;
  a.rows = rows;
  a.R = (int)max_occ;
  a.K = (int)k;
  a.num_occ = num_occ;
  a.cap = cap;
  a.weights = weights;
  a.min_prob = min_token_prob;
  a.alpha = alpha;
  a.chain = chain;
  a.num_valid = num_valid;
  a.num_emit = num_emit;
  a.score = score;
  const size_t per_wave = (size_t)expand_wave_bytes(a.R, a.K);
  if (per_wave > kMaxLds) return SFX_EINVAL;
  int wpb = (int)(kMaxLds / per_wave);
  wpb = wpb > 4 ? 4 : wpb;
  a.waves_per_block = wpb;
  const int64_t blocks = (rows + wpb - 1) / wpb;
  const size_t lds = per_wave * (size_t)wpb;
  static std::atomic<uint64_t> lds_opt_w{0};
  allow_max_lds((const void*)k_expand<true>, lds_opt_w);
  static std::atomic<uint64_t> lds_opt_u{0};
  allow_max_lds((const void*)k_expand<false>, lds_opt_u);
  if (weights)
    hipLaunchKernelGGL(k_expand<true>, dim3((unsigned)blocks), dim3(256),
                       lds, stream, a);
  else
    hipLaunchKernelGGL(k_expand<false>, dim3((unsigned)blocks), dim3(256),
                       lds, stream, a);
  return (int)hipGetLastError();
}
