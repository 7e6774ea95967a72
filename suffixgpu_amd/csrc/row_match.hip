// The match launch of rows that do not fit a CU's LDS (split rows): the parts
// of kRowPart positions of every row are shared out over the chip's
// workgroups, which leave each part's u8 match lengths and, per length, how
// many of its ends match at least that long.  The step launch behind it on
// the stream starts from these (local_split_body), so the row is read by the
// whole chip instead of streamed through one CU.

#include <algorithm>

#include "launch.h"
#include "local_impl.h"

namespace sfx {

constexpr int kMatchThreads = 256;
constexpr int kMatchWaves = kMatchThreads / kWave;
constexpr int kMatchGroups = kRowPart / 4 / kMatchThreads;  // of 4 ends
constexpr int kMaxPat = 255;
// Workgroups of the launch, at most (at least one per row): as many as the
// chip holds at once, five per CU by their LDS.  One per part kept short rows
// of a wide buffer waiting for thousands of workgroups without a part.  Steps
// of 256 rows in a buffer of 131,072 tokens with global memory, us, a
// workgroup per part / these / these without the rows that the step holds in
// LDS: rows of 2% of the buffer 76 / 41 / 37, of 10% 83 / 47 / 46, of 50-100%
// 88 / 86 / 88; 64 rows 40 / 35 / 30, 40 / 36 / 36, 48 / 49 / 49.
constexpr int64_t kMatchGrid = 1280;
// Tokens staged before a part's first position: the longest walk reads
// x(i - 1 - t) for t up to P + 2 (four tokens a step).
__host__ __device__ inline int match_halo(int P) { return stream_halo(P) + 4; }

// nwg workgroups take a row's parts in turn.  Rows of at most a.solo tokens
// are left to the step.
__global__ __launch_bounds__(kMatchThreads) void k_row_match(LocalArgs a,
                                                             int nwg) {
  // ends of one wave that matched four tokens, walked after the scan
  constexpr int kWalkQ = 512;
  __shared__ __align__(16) int32_t row[kRowPart + kMaxPat + 9];
  __shared__ __align__(16) uint8_t mbuf[kRowPart];
  __shared__ int32_t pat[kMaxPat];
  __shared__ int32_t hist[kMaxPat + 1];
  __shared__ int32_t walkq[kMatchWaves][kWalkQ];
  __shared__ int32_t walkn[kMatchWaves];
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int wv = tid / kWave;
  const int ln = tid % kWave;
  const int S = (int)a.bt.seq;
  const int P = a.p.max_pattern_len;
  const RowState st = row_state(a.bt, b);
  int32_t* grow = a.bt.tokens + (int64_t)b * S;
  const int32_t* sp =
      a.bt.sampled ? a.bt.sampled + (int64_t)b * a.bt.num_sampled : nullptr;
  if (st.q <= a.solo) return;
  if (blockIdx.x == 0 && sp) {  // the step's scatter (proposer.py:162-184)
    for (int64_t j = tid; j < a.bt.num_sampled; j += kMatchThreads) {
      const int64_t pos = st.base + j;
      const int32_t v = sp[j];
      if (j < st.cnt && v != -1 && pos < S && pos >= 0) grow[pos] = v;
    }
  }
  const int qe = (int)(st.q < 0 ? 0 : (st.q < S ? st.q : S));
  if (!st.mask) return;

  // Newest-first pattern, -2 fill (local_matcher.py:103-112): the resident
  // token and the sampled id that replaces it are loaded together, and
  // waited for with the first part's tokens.
  static_assert(kMaxPat <= kMatchThreads, "a pattern token per thread");
  int32_t resident = -2, smp = -1;
  if (tid < P) {
    const int64_t idx = st.q - 1 - tid;
    if (idx >= 0) {
      const int64_t at = idx < S - 1 ? idx : S - 1;
      const int64_t j = at - st.base;
      if (sp && j >= 0 && j < st.cnt && j < a.bt.num_sampled) smp = sp[j];
      resident = grow[at];
    }
  }
  for (int k = blockIdx.x; k * kRowPart < qe; k += nwg) {
    const int lo = k * kRowPart;
    const int hi = min(lo + kRowPart, qe);

    // x(lo - halo) .. x(hi - 2), -1 before the row; every word of a thread in
    // flight at once.
    const int halo = match_halo(P);
    const int j0 = lo - halo;
    const int nw = (hi - 1 - j0 + 3) / 4;
    const bool vec4 = (S & 3) == 0 && (((uintptr_t)grow) & 15) == 0;
    constexpr int kLoads =
        (kRowPart + kMaxPat + 9 + 4 * kMatchThreads - 1) / (4 * kMatchThreads);
    int4 v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int w = u * kMatchThreads + tid;
      const int j = j0 + 4 * w;
      if (w >= nw) {
        v[u] = make_int4(0, 0, 0, 0);
      } else if (vec4 && j >= 0 && j + 3 < S) {
        v[u] = reinterpret_cast<const int4*>(grow)[j >> 2];
      } else {
        v[u].x = j < 0 ? -1 : (j < S ? grow[j] : 0);
        v[u].y = j + 1 < 0 ? -1 : (j + 1 < S ? grow[j + 1] : 0);
        v[u].z = j + 2 < 0 ? -1 : (j + 2 < S ? grow[j + 2] : 0);
        v[u].w = j + 3 < 0 ? -1 : (j + 3 < S ? grow[j + 3] : 0);
      }
    }
    if (tid < P) pat[tid] = smp != -1 ? smp : resident;
    for (int i = tid; i <= P; i += kMatchThreads) hist[i] = 0;
    if (tid < kMatchWaves) walkn[tid] = 0;
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int w = u * kMatchThreads + tid;
      if (w < nw) reinterpret_cast<int4*>(row)[w] = v[u];
    }
    __syncthreads();
    if (sp) {  // the scatter again: part 0's stores may not be visible yet
      for (int64_t j = tid; j < a.bt.num_sampled; j += kMatchThreads) {
        const int64_t pos = st.base + j;
        const int32_t x = sp[j];
        if (j < st.cnt && x != -1 && pos < S && pos >= 0 && pos >= j0 &&
            pos < j0 + 4 * nw)
          row[pos - j0] = x;
      }
      __syncthreads();
    }

    // match_back of ends lo .. hi - 1 (zero from hi on): four ends per word,
    // the first four pattern tokens tested without a branch, longer matches
    // queued per wave (a full queue walks in place).
    const int32_t p0 = pat[0];
    const int32_t p1 = P > 1 ? pat[1] : 0;
    const int32_t p2 = P > 2 ? pat[2] : 0;
    const int32_t p3 = P > 3 ? pat[3] : 0;
    const int4* row4 = reinterpret_cast<const int4*>(row) + halo / 4;
    auto walk = [&](int i) -> int {  // i: end - lo
      const int base = halo + i - 1;
      int m = 4;
      while (m < P) {
        int n = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          n += (n == e && m + e < P && row[base - m - e] == pat[m + e]) ? 1 : 0;
        m += n;
        if (n < 4) break;
      }
      return m;
    };
#pragma unroll
    for (int it = 0; it < kMatchGroups; ++it) {
      const int i0 = 4 * (it * kMatchThreads + tid);
      const int4 l4 = row4[i0 / 4 - 1];
      const int4 h4 = row4[i0 / 4];
      const int32_t x[8] = {l4.x, l4.y, l4.z, l4.w, h4.x, h4.y, h4.z, h4.w};
      uint32_t word = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool e0 = lo + i0 + u < hi && x[3 + u] == p0;
        const bool e1 = e0 && P > 1 && x[2 + u] == p1;
        const bool e2 = e1 && P > 2 && x[1 + u] == p2;
        const bool e3 = e2 && P > 3 && x[u] == p3;
        int m = (int)e0 + (int)e1 + (int)e2 + (int)e3;
        bool queued = false;
        if (e3 && P > 4) {
          const int slot = atomicAdd(&walkn[wv], 1);
          queued = slot < kWalkQ;
          if (queued)
            walkq[wv][slot] = i0 + u;
          else
            m = walk(i0 + u);
        }
        word |= (uint32_t)m << (8 * u);
        if (m > 0 && !queued) atomicAdd(&hist[m], 1);
      }
      *reinterpret_cast<uint32_t*>(mbuf + i0) = word;
    }
    wave_lds_sync();
    const int nq = min(walkn[wv], kWalkQ);
    for (int e = ln; e < nq; e += kWave) {
      const int i = walkq[wv][e];
      const int m = walk(i);
      mbuf[i] = (uint8_t)m;
      atomicAdd(&hist[m], 1);
    }
    __syncthreads();

    static_assert(kRowPart == 16 * kMatchThreads, "a 16-byte word per thread");
    reinterpret_cast<uint4*>(a.rs.mb + ((int64_t)b * a.rs.parts + k) *
                                           kRowPart)[tid] =
        reinterpret_cast<const uint4*>(mbuf)[tid];
    // #{mb >= len}: suffix sums of the histogram, longest first
    if (wv == 0) {
      int32_t* out = a.rs.count + (int64_t)b * (P + 1) * a.rs.parts + k;
      uint32_t carry = 0;
      for (int top = P; top >= 1; top -= kWave) {
        const int len = top - ln;
        const uint32_t s =
            carry + wave_incl_scan(len >= 1 ? (uint32_t)hist[len] : 0u);
        if (len >= 1) out[(int64_t)len * a.rs.parts] = (int32_t)s;
        carry = (uint32_t)__builtin_amdgcn_readlane((int)s, kWave - 1);
      }
    }
    __syncthreads();  // the next part rewrites the shared arrays
  }
}

int launch_row_match(const LocalArgs& a, hipStream_t stream) {
  const int64_t share =
      (kMatchGrid + a.bt.batch - 1) / a.bt.batch;  // of the grid, a row's
  const int nwg = (int)std::min<int64_t>(a.rs.parts, share);
  hipLaunchKernelGGL(k_row_match, dim3((unsigned)nwg, (unsigned)a.bt.batch),
                     dim3(kMatchThreads), 0, stream, a, nwg);
  return (int)hipGetLastError();
}

}  // namespace sfx
