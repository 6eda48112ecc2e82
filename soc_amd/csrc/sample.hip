// sample.hip - top-k candidate selection on the device for the sampler (Mac/gpu/src/runtime/sampler.cpp:14-71).
//
// The reference copies the whole logits row to the host and runs
//   std::partial_sort(cand, cand + k, cand + V, [](l, r) { return row[l] / t > row[r] / t; })
// over cand = 0..V-1, then reports cand[0..k). That sort is a heap selection: the first k candidates form a heap,
// and candidate i >= k enters it (replacing the root) exactly when row[i] / t is larger than the current root, i.e.
// than the k-th largest value among candidates 0..i-1; every other candidate is never touched. Running the same
// std::partial_sort over only S = {0..k-1} followed by the candidates that enter, in index order, therefore repeats
// the same comparisons on the same heap and yields the same k candidates in the same order, ties included.
//
// The kernels find S without a sequential scan. With q_i = row[i] / t, candidate i enters iff fewer than k earlier
// candidates j < i have q_j >= q_i, i.e. iff q_i is larger than T_i, the k-th largest of q_0..q_{i-1} (no threshold
// while fewer than k values precede). Two facts make this parallel:
//  - the multiset of the k largest values of any prefix is the top k of the per-chunk top-k lists of the chunks it
//    covers, and also the top k of the candidates of S it holds (the heap holds exactly these values);
//  - a value that is not above the k-th largest of a prefix cannot enter later, and cannot count against a later
//    candidate that is above it.
// k_topk_chunks writes each 2048-value chunk's top-k list. k_topk_accept (one block per chunk) merges the lists of
// the chunks before its own into the prefix top-k list L, then walks its chunk in rounds of 256 values: a value
// survives if it is above L[k-1]; a survivor enters iff L holds fewer than k values >= it minus the earlier
// survivors of its round that are >= it; L then absorbs the round's entrants. k_topk_gather concatenates the chunks'
// entrants. The host sorts the few candidates of S. For k = 1 the heap keeps the lowest index among the largest q,
// which k_topk_one finds in one launch.
//
// Where the k largest q differ from each other and from the rest, the heap's history does not matter: any sort returns
// those k in descending order. k_topk_head finds them in one launch, and where they do not differ a superset of S in
// index order (candidates that do not enter are not touched, so any superset serves). Only where that grows past what
// one block ranks (rising rows) do the three kernels above run.
#include "kernels.h"

#include <type_traits>

namespace soc {
namespace {

constexpr int NT = 256;                // threads per block
constexpr int NW = NT / kWave;         // waves per block
constexpr int EPT = kSampleChunk / NT;  // values per thread in a chunk
constexpr int KM = kSampleMaxK;         // list length (k <= KM)

// Order of a value in the lists; NaN marks an empty list entry (it compares false with everything).
__device__ __forceinline__ float q_of(const float* row, int i, int V, float t) {
  return i < V ? __fdiv_rn(row[i], t) : __builtin_nanf("");
}

// Order-preserving block compaction: this thread's slot among the threads whose flag is set (in thread order), with
// the block's count in *total (the same in every thread). `ws` holds NW ints; two barriers.
__device__ __forceinline__ int block_compact(bool flag, int* ws, int* total) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const uint64_t b = __ballot(flag);
  if (lane == 0) ws[w] = __popcll(b);
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int u = 0; u < NW; ++u) {
    const int n = ws[u];
    off += u < w ? n : 0;
    tot += n;
  }
  __syncthreads();
  *total = tot;
  return off + __popcll(b & ((1ull << lane) - 1));
}

// Block: the top-k values (multiset, descending; entries past the chunk's size are NaN) of chunk c of q, and
// whether the chunk holds a NaN. Each wave extracts the k largest of its 512 values by repeated maxima; the four
// sorted wave lists are then merged by rank (a value's final position is its position in its own list plus the
// count of larger values in the other lists, ties going to the lower-numbered list).
__global__ __launch_bounds__(NT) void k_topk_chunks(const float* __restrict__ row, int V, float t, int k,
                                                     float* __restrict__ chunk_top, int* __restrict__ chunk_nan) {
  __shared__ float wl[NW][KM];
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  float v[EPT];
  uint32_t present = 0;
  bool nan_seen = false;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    // wave w takes elements [512 w, 512 w + 512) of the chunk, lane-interleaved
    const int i = c * kSampleChunk + w * (kWave * EPT) + e * kWave + lane;
    v[e] = q_of(row, i, V, t);
    if (i < V) {
      if (v[e] != v[e]) nan_seen = true;
      else present |= 1u << e;
    }
  }
  const int any_nan = __syncthreads_or(nan_seen);
  if (tid == 0) chunk_nan[c] = any_nan != 0;
  for (int r = 0; r < k; ++r) {
    float best = -INFINITY;
    int be = -1;
#pragma unroll
    for (int e = 0; e < EPT; ++e)
      if (((present >> e) & 1u) && (be < 0 || v[e] > best)) {
        best = v[e];
        be = e;
      }
    const uint64_t any = __ballot(be >= 0);
    if (any == 0) {
      if (lane == 0) wl[w][r] = __builtin_nanf("");
      continue;
    }
    // maximum over lanes that hold a value (-inf is a value here)
    float m = be >= 0 ? best : -INFINITY;
    m = wave_max(m);
    const uint64_t hit = __ballot(be >= 0 && best == m);
    const int src = __builtin_ctzll(hit);
    if (lane == src) present &= ~(1u << be);
    if (lane == 0) wl[w][r] = m;
  }
  for (int r = k; r < KM; ++r)
    if (lane == 0) wl[w][r] = __builtin_nanf("");
  __syncthreads();
  // merge: wave w places its own entry `lane`
  float* out = chunk_top + static_cast<size_t>(c) * KM;
  if (w == 0) out[lane] = __builtin_nanf("");  // KM == 64 entries, one per lane
  __syncthreads();
  const float x = wl[w][lane];
  if (lane < k && x == x) {
    int pos = lane;
    for (int u = 0; u < NW; ++u) {
      if (u == w) continue;
      for (int j = 0; j < k; ++j) {
        const float y = wl[u][j];
        pos += (u < w) ? (y >= x) : (y > x);
      }
    }
    if (pos < k) out[pos] = x;
  }
}

// Block c: writes the indices of the candidates of chunk c that enter the heap, in index order, to
// acc_idx[c * kSampleChunk ..] and their count to acc_cnt[c]. Dynamic LDS: c * k floats (the lists of chunks 0..c-1).
__global__ __launch_bounds__(NT) void k_topk_accept(const float* __restrict__ row, int V, float t, int k,
                                                     const float* __restrict__ chunk_top, int* __restrict__ acc_cnt,
                                                     int* __restrict__ acc_idx) {
  extern __shared__ float lists[];  // list j at lists[j * k], j < c
  __shared__ float q[kSampleChunk];
  __shared__ float rv[NT + 8];  // this round's survivors (values, in index order); 8 pad entries for the unrolled scan
  __shared__ int ri[NT];        // their positions in the chunk
  __shared__ float ev[NT];      // this round's entrants (values, in index order)
  __shared__ float lbuf[2][KM];
  __shared__ int ws[NW];
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  const int c0 = c * kSampleChunk;
  const float qnan = __builtin_nanf("");
  for (int e = 0; e < EPT; ++e) q[e * NT + tid] = q_of(row, c0 + e * NT + tid, V, t);
  for (int j = tid; j < c * k; j += NT) lists[j] = chunk_top[static_cast<size_t>(j / k) * KM + j % k];
  if (tid < 8) rv[NT + tid] = qnan;
  __syncthreads();

  // prefix list: pairwise rank merges, list a = 2 span p absorbing list a + span; a group of g lanes (the power of
  // two >= k) merges one pair, entry gl of each list placed by lane gl
  int g = 1;
  while (g < k) g <<= 1;
  const int gpw = kWave / g, grp = lane / g, gl = lane % g;
  for (int span = 1; span < c; span <<= 1) {
    const int np = (c - span + 2 * span - 1) / (2 * span);  // pairs whose second list exists
    for (int base = 0; base < np; base += NW * gpw) {          // the same trip count in every thread
      const int p = base + w * gpw + grp;
      const bool act = p < np && gl < k;
      float* A = lists + static_cast<size_t>(2 * span * (act ? p : 0)) * k;
      const float* B = A + static_cast<size_t>(span) * k;
      float a = qnan, b = qnan;
      int pa = k, pb = k;
      if (act) {
        a = A[gl];
        b = B[gl];
        int ca = 0, cb = 0;
        for (int j = 0; j < k; ++j) {
          ca += B[j] > a;   // B's larger values go first
          cb += A[j] >= b;  // and A's equal ones too
        }
        if (a == a) pa = gl + ca;
        if (b == b) pb = gl + cb;
      }
      __syncthreads();
      if (act) A[gl] = qnan;
      __syncthreads();
      if (pa < k) A[pa] = a;
      if (pb < k) A[pb] = b;
      __syncthreads();
    }
  }

  float* L = lbuf[0];
  float* Ln = lbuf[1];
  if (tid < KM) L[tid] = (c > 0 && tid < k) ? lists[tid] : qnan;
  __syncthreads();
  int nacc = 0;
  for (int e = 0; e < EPT; ++e) {
    const float th = L[k - 1];
    const int li = e * NT + tid;
    const float x = q[li];
    const bool surv = x == x && !(x <= th);  // q is NaN past the row's end; no threshold while th is NaN
    int nr;
    const int r = block_compact(surv, ws, &nr);
    if (surv) {
      rv[r] = x;
      ri[r] = li;
    }
    __syncthreads();
    if (nr == 0) continue;
    // survivor tid: L's values >= it, then the earlier survivors' (values not above th are below it)
    bool enter = false;
    float v = qnan;
    int cl = 0;
    if (tid < nr) {
      v = rv[tid];
      for (int j = 0; j < k; ++j) cl += L[j] >= v;
      int cnt = cl;
      for (int j = 0; j < tid && cnt < k; j += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) cnt += (j + u < tid) & (rv[j + u] >= v);
      }
      enter = cnt < k;
    }
    int ne;
    const int m = block_compact(enter, ws, &ne);
    if (enter) {
      ev[m] = v;
      acc_idx[c0 + nacc + m] = c0 + ri[tid];
    }
    nacc += ne;
    __syncthreads();
    if (ne == 0) continue;
    // L <- top k of L and the entrants (order: value descending; L before entrants, entrants by index on ties)
    int pl = KM, pe = KM;
    float a = qnan;
    if (tid < k) {
      a = L[tid];
      if (a == a) {
        int cnt = tid;
        for (int j = 0; j < ne; ++j) cnt += ev[j] > a;
        pl = cnt;
      }
    }
    if (enter) {
      int cnt = cl;
      for (int j = 0; j < ne; ++j) {
        const float y = ev[j];
        cnt += (y > v) | ((y == v) & (j < m));
      }
      pe = cnt;
    }
    if (tid < KM) Ln[tid] = qnan;
    __syncthreads();
    if (pl < k) Ln[pl] = a;
    if (pe < k) Ln[pe] = v;
    __syncthreads();
    float* tmp = L;
    L = Ln;
    Ln = tmp;
  }
  if (tid == 0) acc_cnt[c] = nacc;
}

// Block c: copies chunk c's entrants after those of chunks 0..c-1: out[2 + 2 j] = index, out[3 + 2 j] = its raw
// logit's bits, for j < max_out. Block 0 writes out[0] = count of all entrants, out[1] = NaN seen.
__global__ __launch_bounds__(NT) void k_topk_gather(const float* __restrict__ row, int nch,
                                                     const int* __restrict__ chunk_nan,
                                                     const int* __restrict__ acc_cnt, const int* __restrict__ acc_idx,
                                                     int max_out, int* __restrict__ out) {
  __shared__ int red[2][NW];
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  int before = 0, total = 0;
  bool nan_seen = false;
  for (int j = tid; j < nch; j += NT) {
    const int n = acc_cnt[j];
    before += j < c ? n : 0;
    total += n;
    nan_seen |= chunk_nan[j] != 0;
  }
  for (int o = 32; o > 0; o >>= 1) {
    before += __shfl_xor(before, o);
    total += __shfl_xor(total, o);
  }
  if (lane == 0) {
    red[0][w] = before;
    red[1][w] = total;
  }
  const int any_nan = __syncthreads_or(nan_seen);
  before = total = 0;
#pragma unroll
  for (int u = 0; u < NW; ++u) {
    before += red[0][u];
    total += red[1][u];
  }
  const int n = acc_cnt[c];
  for (int r = tid; r < n; r += NT) {
    const int o = before + r;
    if (o < max_out) {
      const int i = acc_idx[static_cast<size_t>(c) * kSampleChunk + r];
      out[2 + 2 * o] = i;
      out[3 + 2 * o] = __float_as_int(row[i]);
    }
  }
  if (c == 0 && tid == 0) {
    out[0] = total;
    out[1] = any_nan != 0;
  }
}

// (value, index) order of the k = 1 search: a larger value, or an equal value at a lower index; index 0x7fffffff
// marks an empty candidate.
__device__ __forceinline__ bool first_max_better(float v, int i, float bv, int bi) {
  return i != 0x7fffffff && (bi == 0x7fffffff || v > bv || (v == bv && i < bi));
}

// Block-wide first maximum of (bv, bi); every thread gets it. sv / si hold NW entries.
__device__ __forceinline__ void block_first_max(float& bv, int& bi, float* sv, int* si) {
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int oi = __shfl_xor(bi, o);
    if (first_max_better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if ((threadIdx.x & (kWave - 1)) == 0) {
    sv[threadIdx.x / kWave] = bv;
    si[threadIdx.x / kWave] = bi;
  }
  __syncthreads();
  bv = sv[0];
  bi = si[0];
#pragma unroll
  for (int u = 1; u < NW; ++u)
    if (first_max_better(sv[u], si[u], bv, bi)) {
      bv = sv[u];
      bi = si[u];
    }
  __syncthreads();
}

// k = 1 in one launch. The one candidate partial_sort keeps is the lowest index among the largest q, so block c
// reduces chunk c to its (largest q, lowest index), publishes it, and the last block to arrive (counter zero before
// the launch, reset by that block) writes out[0] = 1, out[1] = NaN seen, out[2] = the index, out[3] = its raw logit's
// bits. Within a thread indices rise, so the strict `>` keeps the lowest index of equal values.
__global__ __launch_bounds__(NT) void k_topk_one(const float* __restrict__ row, int V, float t,
                                                  float* __restrict__ part_val, int* __restrict__ part_idx,
                                                  int* __restrict__ part_nan, int* __restrict__ counter,
                                                  int* __restrict__ out) {
  __shared__ float sv[NW];
  __shared__ int si[NW];
  __shared__ int last;
  const int c = blockIdx.x, nch = gridDim.x, tid = threadIdx.x;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  bool nan_seen = false;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int i = c * kSampleChunk + e * NT + tid;
    if (i < V) {
      const float x = __fdiv_rn(row[i], t);
      if (x != x) {
        nan_seen = true;
      } else if (bi == 0x7fffffff || x > bv) {
        bv = x;
        bi = i;
      }
    }
  }
  const int any_nan = __syncthreads_or(nan_seen);
  block_first_max(bv, bi, sv, si);
  if (tid == 0) {
    st_dev(part_val + c, bv);
    st_dev(part_idx + c, bi);
    st_dev(part_nan + c, any_nan != 0);
    wait_mem();  // the candidate is visible device-wide before it is counted
    last = atomicAdd(counter, 1) == nch - 1;
  }
  __syncthreads();
  if (!last) return;
  bv = -INFINITY;
  bi = 0x7fffffff;
  nan_seen = false;
  for (int b = tid; b < nch; b += NT) {
    const float pv = ld_dev(part_val + b);
    const int pi = ld_dev(part_idx + b);
    nan_seen |= ld_dev(part_nan + b) != 0;
    if (first_max_better(pv, pi, bv, bi)) {
      bv = pv;
      bi = pi;
    }
  }
  const int nan_all = __syncthreads_or(nan_seen);
  block_first_max(bv, bi, sv, si);
  if (tid == 0) {
    const int idx = bi == 0x7fffffff ? 0 : bi;  // no value at all: every entry NaN, reported by the flag
    out[0] = 1;
    out[1] = nan_all != 0;
    out[2] = idx;
    out[3] = __float_as_int(row[idx]);
    st_dev(counter, 0);
  }
}

// ---- the candidates of a row in one launch ----------------------------------------------------------------------
// Bound by latency, not by the 4 V bytes: a load round trip, the arrival counter, and a chain of short steps in the
// last block to arrive. The row is cut into groups of FE << gshift values (the lanes of a wave that share the tid's
// upper bits); every block publishes its groups' maxima. With T any value that at least k group maxima reach, the k
// largest values are all >= T and lie in the groups whose maximum is, so the last block halves towards T until few
// more than k groups are left (4 V bytes are never sorted; no repeated extraction of maxima), reads those groups
// again, and ranks the values >= T among themselves. Top 50 of 151936 at temperature 0.7, MI355X: 107 us of kernels
// for the general search (74 of them the prefix walk of the last chunk) against 17.5 us, 121 -> 29 us for the call.
//
// Equal values among the k largest (the rule for logits that were rounded to 16 bits) make the heap's history matter.
// The same block then bounds the heap's root from below at doubling prefixes of the row: 128 .. 2048 values of the
// first chunk, 2 .. 64 chunks of group maxima, one wave's search each. A value that enters is above the bound of
// the last such prefix before it, so the first 128 values and the values above their bound, about k per doubling,
// hold S. us a call at 50 of 151936 / 50 of 4096 / 20 of 32000, this kernel followed by the general search, that search
// alone, this: rounded to bf16 149 / 113 / 88, 121 / 90 / 63, 78 / 49 / 46; all but 20 masked 149 / 105 / 78, 118 / 75 /
// 47, 34 / 34 / 35. Two of 32000 that are equal 60, 36, 43. Rows that rise end to end overflow and take both: 258 at 50
// of 4096, 220 for the general search alone.
constexpr int FT = 512;                 // threads per block
constexpr int FW = FT / kWave;
constexpr int FE = kSampleChunk / FT;   // values per thread
constexpr int FR = 16;                  // group maxima per thread of the last block
constexpr int kMaxGroups = FR * FT;
constexpr int kMaxSel = 1024;           // groups read again
constexpr int kMaxRank = 1088;          // values ranked by value
constexpr int kMaxCand = kSampleHeadMax;  // values ranked by index
constexpr int kSlack = 32;              // groups beyond k that end the search for T
constexpr int kPrefixes = 11;           // bounds: prefixes of 128 << b values (b < 5), of 2 << (b - 5) chunks
constexpr int kPrefixRegs = 32;         // keys per lane of a prefix search

// Values in ascending order of q as unsigned words, equal q (+0 and -0 too) as equal words, all above 0; 0 stands for
// no value.
__device__ __forceinline__ uint32_t key_of(float q) {
  const uint32_t b = __float_as_uint(q + 0.0f);
  return (b & 0x80000000u) ? ~b : b | 0x80000000u;
}

// Minimum and maximum over the wave (DPP within rows of 16 lanes, then the four rows).
template <bool MIN>
__device__ __forceinline__ uint32_t wave_pick(uint32_t v) {
  auto pick = [](uint32_t a, uint32_t b) { return MIN ? min(a, b) : max(a, b); };
  auto mov = [](uint32_t a, auto ctrl) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(a), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  v = pick(v, mov(v, std::integral_constant<int, 0xB1>()));
  v = pick(v, mov(v, std::integral_constant<int, 0x4E>()));
  v = pick(v, mov(v, std::integral_constant<int, 0x141>()));
  v = pick(v, mov(v, std::integral_constant<int, 0x140>()));
  const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16),
                 c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
  return pick(pick(a, b), pick(c, d));
}

// The wave's keys (N per lane, those from `regs` on absent) against a pivot: how many reach it, the smallest that does
// (all ones: none) and the largest that does not.
struct Split {
  int n;
  uint32_t least, below;
};
template <int N>
__device__ __forceinline__ Split wave_split(const uint32_t (&key)[N], int regs, uint32_t pivot) {
  Split r{0, 0xFFFFFFFFu, 0u};
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (u < regs) {
      const bool in = key[u] >= pivot;
      r.n += __popcll(__ballot(in));
      r.least = min(r.least, in ? key[u] : 0xFFFFFFFFu);
      r.below = max(r.below, in ? 0u : key[u]);
    }
  r.least = wave_pick<true>(r.least);
  r.below = wave_pick<false>(r.below);
  return r;
}

// Where a search starts: how many keys there are (0: none), the smallest and the largest.
template <int N>
__device__ __forceinline__ Split wave_range(const uint32_t (&key)[N], int regs) {
  Split r{0, 0xFFFFFFFFu, 0u};
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (u < regs) {
      r.n += __popcll(__ballot(key[u] != 0));
      r.least = min(r.least, key[u] - 1);  // (0 becomes all ones)
      r.below = max(r.below, key[u]);
    }
  r.least = wave_pick<true>(r.least) + 1;
  r.below = wave_pick<false>(r.below);
  return r;
}

// A search for a key that at least k keys reach and few more than k do, by halving [lo, hi): n keys reach lo, fewer
// than k reach hi. Both ends move on to a key that is there, so equal keys end it in a step or two (bit by bit they
// took all 32).
struct Search {
  uint32_t lo, hi;
  int n;
  __device__ __forceinline__ bool done(int enough) const { return n <= enough || hi - lo <= 1; }
  __device__ __forceinline__ uint32_t pivot() const { return lo + (hi - lo) / 2; }
  __device__ __forceinline__ void step(const Split& s, int k) {
    if (s.n >= k) {
      lo = s.least;
      n = s.n;
    } else {
      hi = s.below + 1;
    }
  }
};

// out[1]: 0 = out[0] entries follow: either the k largest in descending order or candidates in index order (index, bits
// of the raw logit); 1 = the row holds a NaN; 2 = too many candidates.
__global__ __launch_bounds__(FT) void k_topk_head(const float* __restrict__ row, int V, float t, int k, int gshift,
                                                   int32_t* __restrict__ gmax, int32_t* __restrict__ gnan,
                                                   int* __restrict__ counter, int* __restrict__ out) {
  __shared__ int sel[kMaxSel];
  __shared__ uint32_t ckey[kMaxRank];
  __shared__ int cidx[kMaxCand];
  __shared__ float craw[kMaxCand];
  __shared__ uint32_t bound[kPrefixes];
  __shared__ Split part[2][FW];
  __shared__ int nsel, ncand, last;
  const int c = blockIdx.x, nch = gridDim.x, tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  const int gpb = FT >> gshift;  // groups per block
  float x[FE];
#pragma unroll
  for (int e = 0; e < FE; ++e) x[e] = row[min(c * kSampleChunk + e * FT + tid, V - 1)];
  uint32_t m = 0;
  bool nan_seen = false;
#pragma unroll
  for (int e = 0; e < FE; ++e) {
    const float q = __fdiv_rn(x[e], t);
    if (c * kSampleChunk + e * FT + tid < V) {
      nan_seen |= q != q;
      m = max(m, key_of(q));
    }
  }
  for (int o = 1; o < (1 << gshift); o <<= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o)));
  if ((tid & ((1 << gshift) - 1)) == 0) st_dev(gmax + c * gpb + (tid >> gshift), static_cast<int32_t>(m));
  wait_mem();  // the block's maxima are visible device-wide before the block is counted
  const int any_nan = __syncthreads_or(nan_seen);
  if (tid == 0) {
    st_dev(gnan + c, any_nan != 0);
    wait_mem();
    last = atomicAdd(counter, 1) == nch - 1;
    nsel = ncand = 0;
  }
  __syncthreads();
  if (!last) return;

  const int G = nch * gpb;
  uint32_t g[FR];
#pragma unroll
  for (int u = 0; u < FR; ++u) g[u] = u * FT + tid < G ? static_cast<uint32_t>(ld_dev(gmax + u * FT + tid)) : 0u;
  nan_seen = false;
  for (int b = tid; b < nch; b += FT) nan_seen |= ld_dev(gnan + b) != 0;
  if (tid == 0) st_dev(counter, 0);
  if (__syncthreads_or(nan_seen)) {
    if (tid == 0) {
      out[0] = 0;
      out[1] = 1;
    }
    return;
  }
  // T among all group maxima, one barrier a step
  const int regs = (G + FT - 1) / FT;
  auto block_merge = [&](const Split& p, int buf) {
    if (lane == 0) part[buf][w] = p;
    __syncthreads();
    Split r = part[buf][0];
#pragma unroll
    for (int u = 1; u < FW; ++u) {
      const Split o = part[buf][u];
      r.n += o.n;
      r.least = min(r.least, o.least);
      r.below = max(r.below, o.below);
    }
    return r;
  };
  uint32_t T = 1;  // fewer than k groups: every value
  Split p = wave_range(g, regs);
  if (p.n == 0) p.least = 0xFFFFFFFFu;
  const Split all = block_merge(p, 1);
  if (all.n >= k) {
    Search f{all.least, all.below + 1, all.n};
    for (int buf = 0; !f.done(k + kSlack); buf ^= 1) f.step(block_merge(wave_split(g, regs, f.pivot()), buf), k);
    T = f.lo;
  }
#pragma unroll
  for (int u = 0; u < FR; ++u)
    if (g[u] >= T) {
      const int p = atomicAdd(&nsel, 1);
      if (p < kMaxSel) sel[p] = u * FT + tid;
    }
  __syncthreads();
  const int gs = gshift + 2;  // log2 of the values per group
  static_assert(FE == 4, "values per group");
  // hands every value of the ns selected groups to take(group, index, raw)
  auto read_groups = [&](int ns, auto take) {
    for (int p0 = 0; p0 < (ns << gs); p0 += 8 * FT) {
      int gr[8], ix[8];
      float y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int p = p0 + u * FT + tid;
        gr[u] = 0;
        ix[u] = V;
        if (p < (ns << gs)) {
          const int gi = gr[u] = sel[p >> gs], j = p & ((1 << gs) - 1);
          ix[u] = (gi / gpb) * kSampleChunk + (j >> gshift) * FT + ((gi % gpb) << gshift) + (j & ((1 << gshift) - 1));
        }
        y[u] = row[min(ix[u], V - 1)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (ix[u] < V) take(gr[u], ix[u], y[u]);
    }
  };
  bool give_up = nsel > kMaxSel / 2;
  if (!give_up)
    read_groups(nsel, [&](int, int i, float y) {
      const uint32_t key = key_of(__fdiv_rn(y, t));
      if (key < T) return;
      const int r = atomicAdd(&ncand, 1);
      if (r < kMaxRank) {
        ckey[r] = key;
        cidx[r] = i;
        craw[r] = y;
      }
    });
  __syncthreads();
  int n = ncand;
  give_up |= n > kMaxRank;
  constexpr int RK = (kMaxRank + FT - 1) / FT;
  int rank[RK];
  if (!give_up) {
#pragma unroll
    for (int u = 0; u < RK; ++u) {
      rank[u] = k;
      const int i = tid + u * FT;
      if (i >= n) continue;
      const uint32_t key = ckey[i];
      int above = 0, same = 0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) {
        above += ckey[j] > key;
        same += ckey[j] == key;
      }
      rank[u] = above;
      give_up |= above < k && same > 1;
    }
  }
  if (!__syncthreads_or(give_up)) {
#pragma unroll
    for (int u = 0; u < RK; ++u)
      if (rank[u] < k) {
        out[2 + 2 * rank[u]] = cidx[tid + u * FT];
        out[3 + 2 * rank[u]] = __float_as_int(craw[tid + u * FT]);
      }
    if (tid == 0) {
      out[0] = k;
      out[1] = 0;
    }
    return;
  }

  // Equal values (or many near the k-th): bounds of the heap's root by prefix, a wave each, the long ones in waves of
  // one task. A prefix that does not end before the row's last value bounds nothing.
  if (tid == 0) nsel = ncand = 0;
  for (int task = w; task < kPrefixes; task += FW) {
    // a digit per task, from the right: 128, 256 values, 2 chunks | 2048 values, 64 chunks, 1024 values, 32, 16 chunks |
    // 512 values, 4, 8 chunks
    const int b = static_cast<int>(0x762893A4510ull >> 4 * task) & 15;
    const bool vals = b < 5;
    const int len = vals ? 128 << b : 2 << (b - 5);  // values, or chunks
    uint32_t B = 0;
    if (vals ? len < V : len < nch) {
      const int cnt = vals ? len : min(len * gpb, kPrefixRegs * kWave);  // (of a part of the prefix: a lower bound too)
      uint32_t key[kPrefixRegs];
#pragma unroll
      for (int u = 0; u < kPrefixRegs; ++u) {
        key[u] = 0;
        const int i = u * kWave + lane;
        if (u * kWave < cnt && i < cnt)
          key[u] = vals ? key_of(__fdiv_rn(row[i], t)) : static_cast<uint32_t>(ld_dev(gmax + i));
      }
      const int held = (cnt + kWave - 1) / kWave;
      const Split all = wave_range(key, held);
      Search f{all.least, all.below + 1, all.n};
      while (!f.done(max(k + k / 8, kSlack))) f.step(wave_split(key, held, f.pivot()), k);
      B = f.lo;
    }
    if (lane == 0) bound[b] = B;
  }
  __syncthreads();
  auto chunk_bound = [&](int ch) {  // chunks from 1
    return ch == 1 ? bound[4] : bound[5 + min(31 - __clz(ch), 6) - 1];
  };
  auto put = [&](int i, float y, uint32_t key, uint32_t b) {
    if (key <= b) return;
    const int r = atomicAdd(&ncand, 1);
    if (r < kMaxCand) {
      cidx[r] = i;
      craw[r] = y;
    }
  };
#pragma unroll
  for (int e = 0; e < FE; ++e) {  // the first chunk
    const int i = e * FT + tid;
    if (i < min(V, kSampleChunk)) {
      const float y = row[i];
      put(i, y, key_of(__fdiv_rn(y, t)), i < 128 ? 0u : bound[31 - __clz(i) - 7]);
    }
  }
#pragma unroll
  for (int u = 0; u < FR; ++u) {
    const int gi = u * FT + tid;
    if (gi < G && gi >= gpb && g[u] > chunk_bound(gi / gpb)) {
      const int p = atomicAdd(&nsel, 1);
      if (p < kMaxSel) sel[p] = gi;
    }
  }
  __syncthreads();
  const int ns = nsel;
  if (ns <= kMaxSel)
    read_groups(ns, [&](int gi, int i, float y) { put(i, y, key_of(__fdiv_rn(y, t)), chunk_bound(gi / gpb)); });
  __syncthreads();
  n = ncand;
  if (ns > kMaxSel || n > kMaxCand) {
    if (tid == 0) {
      out[0] = 0;
      out[1] = 2;
    }
    return;
  }
  for (int i = tid; i < n; i += FT) {
    const int at = cidx[i];
    int r = 0;
#pragma unroll 8
    for (int j = 0; j < n; ++j) r += cidx[j] < at;
    out[2 + 2 * r] = at;
    out[3 + 2 * r] = __float_as_int(craw[i]);
  }
  if (tid == 0) {
    out[0] = n;
    out[1] = 0;
  }
}

// Lanes per group (log2) of k_topk_head: groups of 64 values, or 16 where a row of 64-value groups would have few
// more of them than k.
int distinct_gshift(int V) { return V >= 32768 ? 4 : 2; }

}  // namespace

bool sample_head_fits(int V, int k) {
  if (!sample_device_fits(V, k)) return false;
  const size_t nch = (static_cast<size_t>(V) + kSampleChunk - 1) / kSampleChunk;
  return k == 1 || nch * (FT >> distinct_gshift(V)) <= kMaxGroups;
}

hipError_t launch_sample_head(const float* row, int V, float t, int k, void* ws, int* out, hipStream_t s) {
  if (!sample_head_fits(V, k)) return hipErrorInvalidValue;
  const int nch = (V + kSampleChunk - 1) / kSampleChunk;
  int* counter = static_cast<int*>(ws);
  int* chunk_nan = counter + 64;
  int* acc_cnt = chunk_nan + nch;
  float* chunk_top = reinterpret_cast<float*>(acc_cnt + nch);
  int* acc_idx = reinterpret_cast<int*>(chunk_top + static_cast<size_t>(nch) * KM);
  if (k == 1)  // partials in the first entries of the lists' regions
    hipLaunchKernelGGL(k_topk_one, dim3(nch), dim3(NT), 0, s, row, V, t, chunk_top, acc_cnt, chunk_nan, counter, out);
  else  // the group maxima (at most 128 of a chunk's 2048 values) in the entrants' region
    hipLaunchKernelGGL(k_topk_head, dim3(nch), dim3(FT), 0, s, row, V, t, k, distinct_gshift(V), acc_idx, chunk_nan,
                       counter, out);
  return hipGetLastError();
}

bool sample_device_fits(int V, int k) {
  if (V <= 0 || k <= 0 || k > KM) return false;
  const size_t nch = (static_cast<size_t>(V) + kSampleChunk - 1) / kSampleChunk;
  return nch * static_cast<size_t>(k) * 4 <= kSampleTreeBytes;
}

size_t sample_ws_bytes(int V) {
  const size_t nch = (static_cast<size_t>(V) + kSampleChunk - 1) / kSampleChunk;
  return 256 + nch * 4 * 2 + nch * KM * 4 + nch * kSampleChunk * 4;
}

hipError_t launch_sample_topk(const float* row, int V, float t, int k, void* ws, int* out, int max_out,
                              hipStream_t s) {
  if (!sample_device_fits(V, k) || max_out <= 0) return hipErrorInvalidValue;
  const int nch = (V + kSampleChunk - 1) / kSampleChunk;
  int* chunk_nan = static_cast<int*>(ws) + 64;  // (the arrival counter's line comes first)
  int* acc_cnt = chunk_nan + nch;
  float* chunk_top = reinterpret_cast<float*>(acc_cnt + nch);
  int* acc_idx = reinterpret_cast<int*>(chunk_top + static_cast<size_t>(nch) * KM);
  const size_t tree = static_cast<size_t>(nch) * k * 4;
  hipLaunchKernelGGL(k_topk_chunks, dim3(nch), dim3(NT), 0, s, row, V, t, k, chunk_top, chunk_nan);
  hipLaunchKernelGGL(k_topk_accept, dim3(nch), dim3(NT), tree, s, row, V, t, k, chunk_top, acc_cnt, acc_idx);
  hipLaunchKernelGGL(k_topk_gather, dim3(nch), dim3(NT), 0, s, row, nch, chunk_nan, acc_cnt, acc_idx, max_out, out);
  return hipGetLastError();
}

}  // namespace soc
