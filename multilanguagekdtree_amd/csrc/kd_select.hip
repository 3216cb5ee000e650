// kd_select.hip -- standalone selection on gfx950: quickstat_index
// (Parallel/RustVersion/src/quickstat.rs:9-34) for an index slice keyed by
// an FP64 value array.  The element of rank `goal` under the total order
// (value, index) is found over the 64-bit ordered value keys
// (then over the indices, when values tie), and the slice is stably
// partitioned around it: [0, goal) before, the pivot at goal, the rest after
// -- the reference's postcondition (quickstat.rs:199-215).  The common path is
// the selection by narrowing further down; these radix passes take the calls
// that it leaves.
//
// Passes per 8-bit digit: a histogram of the digit over the elements whose
// higher digits match the prefix chosen so far (LDS histograms, one global
// add per bin and block), then a one-block kernel that picks the digit
// holding the wanted rank.  All of it stays on the device.
#include <algorithm>

#include "kd_internal.hpp"

namespace kd {

__device__ __forceinline__ uint64_t ordkey_sel(double v) {
  uint64_t b = (uint64_t)__double_as_longlong(v);
  if ((b << 1) == 0) b = 0;  // -0.0 and +0.0 compare equal
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

// Selection state on the device: prefix and mask of the pivot key (and of
// its index once keys tie), and the rank still wanted inside the prefix.
struct SelState {
  uint64_t key_prefix, key_mask;
  uint64_t idx_prefix, idx_mask;
  uint64_t rank;
  uint64_t hist[256];
};

constexpr int SEL_THREADS = 256;
constexpr int SEL_ITEMS = 16;

__global__ __launch_bounds__(SEL_THREADS) void k_sel_keys(const int64_t *__restrict__ idx,
                                                          const double *__restrict__ vals,
                                                          uint64_t *__restrict__ keys,
                                                          int64_t n, SelState *st,
                                                          uint64_t goal) {
  const int64_t i = (int64_t)blockIdx.x * SEL_THREADS + threadIdx.x;
  if (i == 0) {
    st->key_prefix = st->key_mask = st->idx_prefix = st->idx_mask = 0;
    st->rank = goal;
  }
  if (i < 256) st->hist[i] = 0;
  if (i >= n) return;
  keys[i] = ordkey_sel(vals[idx[i]]);
}

// Histogram of digit `shift` of the key (on_index: of the index) over the
// elements matching the current prefix.
template <bool ON_INDEX>
__global__ __launch_bounds__(SEL_THREADS) void k_sel_hist(const uint64_t *__restrict__ keys,
                                                          const int64_t *__restrict__ idx,
                                                          int64_t n, SelState *st, int shift) {
  __shared__ unsigned int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t kp = st->key_prefix, km = st->key_mask;
  const uint64_t ip = st->idx_prefix, im = st->idx_mask;
  const int64_t base = (int64_t)blockIdx.x * SEL_THREADS * SEL_ITEMS + threadIdx.x;
#pragma unroll 4
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + (int64_t)it * SEL_THREADS;
    if (i >= n) break;
    const uint64_t k = keys[i];
    if ((k & km) != kp) continue;
    if (ON_INDEX) {
      const uint64_t x = (uint64_t)idx[i];
      if (k != kp || (x & im) != ip) continue;
      atomicAdd(&h[(x >> shift) & 255u], 1u);
    } else {
      atomicAdd(&h[(k >> shift) & 255u], 1u);
    }
  }
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd((unsigned long long *)&st->hist[threadIdx.x],
                                (unsigned long long)h[threadIdx.x]);
}

// Pick the digit that holds the wanted rank; clear the histogram.
template <bool ON_INDEX>
__global__ void k_sel_pick(SelState *st, int shift) {
  if (threadIdx.x == 0) {
    uint64_t rank = st->rank, cum = 0;
    int b = 0;
    for (; b < 255; ++b) {
      if (cum + st->hist[b] > rank) break;
      cum += st->hist[b];
    }
    st->rank = rank - cum;
    if (ON_INDEX) {
      st->idx_prefix |= (uint64_t)b << shift;
      st->idx_mask |= (uint64_t)255 << shift;
    } else {
      st->key_prefix |= (uint64_t)b << shift;
      st->key_mask |= (uint64_t)255 << shift;
    }
  }
  __syncthreads();
  st->hist[threadIdx.x] = 0;
}

// Counts of elements equal to the pivot key (decides whether index passes
// are needed) -- reuses hist[0].
__global__ __launch_bounds__(SEL_THREADS) void k_sel_count_eq(const uint64_t *__restrict__ keys,
                                                              int64_t n, SelState *st) {
  __shared__ unsigned int c;
  if (threadIdx.x == 0) c = 0;
  __syncthreads();
  const uint64_t kp = st->key_prefix;
  const int64_t base = (int64_t)blockIdx.x * SEL_THREADS * SEL_ITEMS + threadIdx.x;
  unsigned int local = 0;
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + (int64_t)it * SEL_THREADS;
    if (i < n && keys[i] == kp) ++local;
  }
  if (local) atomicAdd(&c, local);
  __syncthreads();
  if (threadIdx.x == 0 && c) atomicAdd((unsigned long long *)&st->hist[0], (unsigned long long)c);
}

// 0: before the pivot, 1: the pivot, 2: after, under (key, index).
__device__ __forceinline__ int sel_class(uint64_t k, int64_t x, uint64_t pk, int64_t px) {
  if (k != pk) return k < pk ? 0 : 2;
  return x < px ? 0 : (x == px ? 1 : 2);
}

// Per-block counts of the "before" and "after" classes.
__global__ __launch_bounds__(SEL_THREADS) void k_sel_count(const uint64_t *__restrict__ keys,
                                                           const int64_t *__restrict__ idx,
                                                           int64_t n, const SelState *st,
                                                           unsigned long long *cnt_b,
                                                           unsigned long long *cnt_a) {
  __shared__ unsigned int cb, ca;
  if (threadIdx.x == 0) cb = ca = 0;
  __syncthreads();
  const uint64_t pk = st->key_prefix;
  const int64_t px = (int64_t)st->idx_prefix;
  const bool exact = st->idx_mask != 0;
  const int64_t base = (int64_t)blockIdx.x * SEL_THREADS * SEL_ITEMS;
  unsigned int lb = 0, la = 0;
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + (int64_t)it * SEL_THREADS + threadIdx.x;
    if (i >= n) break;
    const uint64_t k = keys[i];
    const int cl = exact ? sel_class(k, idx[i], pk, px) : (k < pk ? 0 : (k == pk ? 1 : 2));
    lb += cl == 0 ? 1u : 0u;
    la += cl == 2 ? 1u : 0u;
  }
  if (lb) atomicAdd(&cb, lb);
  if (la) atomicAdd(&ca, la);
  __syncthreads();
  if (threadIdx.x == 0) {
    cnt_b[blockIdx.x] = cb;
    cnt_a[blockIdx.x] = ca;
  }
}

// Exclusive scan of nb per-block counts (one block).
__global__ __launch_bounds__(1024) void k_sel_scan(unsigned long long *cnt, int64_t nb) {
  __shared__ unsigned long long sh[1024];
  unsigned long long carry = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 1024) {
    const int64_t i = b0 + threadIdx.x;
    const unsigned long long v = i < nb ? cnt[i] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
      const unsigned long long t = threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
      __syncthreads();
      sh[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nb) cnt[i] = carry + sh[threadIdx.x] - v;
    carry += sh[1023];
    __syncthreads();
  }
}

// Stable partition: "before" elements to [0, goal) in order, the pivot to
// goal, "after" elements to (goal, n) in order.
__global__ __launch_bounds__(SEL_THREADS) void k_sel_scatter(const uint64_t *__restrict__ keys,
                                                             const int64_t *__restrict__ idx,
                                                             int64_t n, const SelState *st,
                                                             const unsigned long long *cnt_b,
                                                             const unsigned long long *cnt_a,
                                                             uint64_t goal,
                                                             int64_t *__restrict__ out) {
  __shared__ unsigned int wsum[SEL_THREADS / 64][2];
  const uint64_t pk = st->key_prefix;
  const int64_t px = (int64_t)st->idx_prefix;
  const bool exact = st->idx_mask != 0;
  const int64_t base = (int64_t)blockIdx.x * SEL_THREADS * SEL_ITEMS;
  unsigned long long off_b = cnt_b[blockIdx.x], off_a = goal + 1 + cnt_a[blockIdx.x];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + (int64_t)it * SEL_THREADS + threadIdx.x;
    int cl = 3;
    int64_t x = 0;
    if (i < n) {
      x = idx[i];
      const uint64_t k = keys[i];
      cl = exact ? sel_class(k, x, pk, px) : (k < pk ? 0 : (k == pk ? 1 : 2));
    }
    const uint64_t mb = __builtin_amdgcn_ballot_w64(cl == 0);
    const uint64_t ma = __builtin_amdgcn_ballot_w64(cl == 2);
    if (lane == 0) {
      wsum[w][0] = (unsigned)__builtin_popcountll(mb);
      wsum[w][1] = (unsigned)__builtin_popcountll(ma);
    }
    __syncthreads();
    unsigned int pb = 0, pa = 0, tb = 0, ta = 0;
    for (int q = 0; q < SEL_THREADS / 64; ++q) {
      if (q < w) {
        pb += wsum[q][0];
        pa += wsum[q][1];
      }
      tb += wsum[q][0];
      ta += wsum[q][1];
    }
    if (cl == 0)
      out[off_b + pb + __builtin_popcountll(mb & below)] = x;
    else if (cl == 1)
      out[goal] = x;
    else if (cl == 2)
      out[off_a + pa + __builtin_popcountll(ma & below)] = x;
    off_b += tb;
    off_a += ta;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// selection by narrowing
// ---------------------------------------------------------------------------
//
// The radix passes above read every key eight times and the partition twice
// more.  Here a sample of SAMPLE keys brackets the wanted rank, one pass over
// the elements sorts out which lie below, inside and above the bracket (and
// copies the indices, since the partition is written in place), and only the
// few inside (about 4 %) are looked at again: narrowed by a sample of their
// own until one workgroup holds them all, which picks the pivot under (value,
// index).  The partition then needs two bits an element and the keys of the
// bracket's elements.  Memory traffic is 16 + 8 bytes an element in the first
// pass and 8 + 8 in the partition: 100 M uniform values take 1.13 ms against
// 4.27 ms by radix passes (the first pass and the partition 0.82 ms of it, at
// the rate of a copy), 4 M (in random order) 244 us against 375, 1,000 60 us
// against 178; 100 M equal values 1.13 ms against 8.18.
// The order is that of (value, index) throughout, so equal values are no
// special case.  A bracket that misses the rank (rare, see sample_at) sends the
// call to the radix passes.

// A sample is 8 keys a thread of one workgroup (16 took 30 us longer a sample
// and saved half the candidates); the last candidates may be 16 a thread.
constexpr int SMP_THREADS = 1024, SMP_ITEMS = 8, PIVOT_ITEMS = 16;
constexpr uint32_t SAMPLE = SMP_THREADS * SMP_ITEMS, PIVOT_MAX = SMP_THREADS * PIVOT_ITEMS;

struct NarrowState {
  uint64_t rank;        // wanted, among the elements at hand
  uint64_t count;       // elements at hand
  uint64_t lo, hi;      // the bracket, ends included: ordered keys and, where
  uint64_t lo_idx, hi_idx;  // keys tie, indices
  __device__ bool is_below(uint64_t k, uint64_t x) const {
    return k < lo || (k == lo && x < lo_idx);
  }
  __device__ bool is_inside(uint64_t k, uint64_t x) const {
    return !is_below(k, x) && (k < hi || (k == hi && x <= hi_idx));
  }
  // counted by the last pass over the elements: those below the bracket (high
  // half) and inside it, in one word so that a tile takes one atomic
  unsigned long long tally;
  __device__ uint64_t below() const { return tally >> 32; }
  __device__ uint64_t inside() const { return tally & 0xffffffffu; }
  uint64_t pivot_key;
  int64_t pivot_idx;
  uint32_t bad, fail;   // an index out of range; the radix passes are needed
};

// candidates: (key, index) pairs
struct Cands {
  uint64_t *key;
  int64_t *idx;
  uint64_t cap;
};

// Inclusive sum over the wavefront.
template <typename T>
__device__ __forceinline__ T wave_incl(T v, uint32_t lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T u = __shfl_up(v, o, 64);
    if ((int)lane >= o) v += u;
  }
  return v;
}

// The key of rank `rank` among the workgroup's keys (ITEMS a thread, those
// whose bit in `use` is set): one digit of 8 bits a pass from the first that
// differs, until one key is left.  hist: 256 words; pick: 3 words; found: one.
template <int ITEMS>
__device__ uint64_t block_select(const uint64_t (&k)[ITEMS], uint32_t use, uint32_t rank,
                                 uint32_t *hist, uint32_t *pick, uint64_t *found) {
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if ((use >> i) & 1u) *found = k[i];  // any of them
  if (threadIdx.x < 2) hist[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t ref = *found;
  uint64_t diff = 0;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) diff |= (use >> i) & 1u ? k[i] ^ ref : 0ull;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) diff |= __shfl_xor(diff, o, 64);
  if ((threadIdx.x & 63u) == 0 && diff) {
    atomicOr(&hist[0], (uint32_t)diff);
    atomicOr(&hist[1], (uint32_t)(diff >> 32));
  }
  __syncthreads();
  diff = ((uint64_t)hist[1] << 32) | hist[0];
  if (diff == 0) {
    __syncthreads();  // hist and found are written again
    return ref;
  }
  const int top = (63 - __builtin_clzll(diff)) / 8 * 8;
  uint64_t mask = top == 56 ? 0ull : ~0ull << (top + 8), prefix = ref & mask;
  for (int shift = top; shift >= 0; shift -= 8) {
    __syncthreads();
    if (threadIdx.x < 256) hist[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const bool in = (use >> i) & 1u && (k[i] & mask) == prefix;
      const uint32_t d = (uint32_t)(k[i] >> shift) & 255u;
      // equal digits throughout the wavefront (the leading bytes) count once
      const uint64_t m = __builtin_amdgcn_ballot_w64(in);
      if (m == 0) continue;
      const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, __builtin_ctzll(m));
      if (__builtin_amdgcn_ballot_w64(in && d != d0) == 0) {
        if ((threadIdx.x & 63u) == 0) atomicAdd(&hist[d0], (uint32_t)__builtin_popcountll(m));
      } else if (in) {
        atomicAdd(&hist[d], 1u);
      }
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      // the digit whose range of ranks holds `rank`
      uint32_t c[4], sum = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += c[i] = hist[4 * threadIdx.x + i];
      uint32_t at = wave_incl(sum, threadIdx.x) - sum;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (rank >= at && rank < at + c[i]) {
          pick[0] = 4 * threadIdx.x + i;
          pick[1] = rank - at;
          pick[2] = c[i];
        }
        at += c[i];
      }
    }
    __syncthreads();
    prefix |= (uint64_t)pick[0] << shift;
    mask |= (uint64_t)255 << shift;
    rank = pick[1];
    if (pick[2] == 1 && shift > 0) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i)
        if ((use >> i) & 1u && (k[i] & mask) == prefix) *found = k[i];
      __syncthreads();
      prefix = *found;
      break;
    }
  }
  __syncthreads();
  return prefix;
}

// The element of rank `rank` under (key, index): key and index.  num: two words.
template <int ITEMS>
__device__ void block_select_pair(const uint64_t (&k)[ITEMS], const uint64_t (&x)[ITEMS],
                                  uint32_t use, uint32_t rank, uint32_t *hist, uint32_t *pick,
                                  uint64_t *found, uint32_t *num, uint64_t &key,
                                  uint64_t &index) {
  key = block_select(k, use, rank, hist, pick, found);
  if (threadIdx.x < 2) num[threadIdx.x] = 0;
  __syncthreads();
  uint32_t l = 0, e = 0;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    l += (use >> i) & 1u && k[i] < key ? 1u : 0u;
    e += (use >> i) & 1u && k[i] == key ? 1u : 0u;
    if ((use >> i) & 1u && k[i] == key) *found = x[i];  // of several, any
  }
  if (l) atomicAdd(&num[0], l);
  if (e) atomicAdd(&num[1], e);
  __syncthreads();
  index = *found;
  if (num[1] > 1) {  // equal keys: by index
    uint32_t tied = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) tied |= (use >> i) & 1u && k[i] == key ? 1u << i : 0u;
    index = block_select(x, tied, rank - num[0], hist, pick, found);
  }
  __syncthreads();
}

// Position of sample i of SAMPLE among `count` elements (i itself if there are
// no more): one from every SAMPLE-th part of them, at a place in it that a hash
// of i picks.  At the parts' starts the sample would alias with data of a period: of a 128^3 lattice by its fastest
// coordinate it saw one value, and 99 % of the ranks missed the bracket.  With
// places that have nothing to do with the data, a rank in the sample varies no
// more than in independent draws, so a bracket of 4 standard deviations and 8
// misses about once in 10^4 calls.
__device__ __forceinline__ uint64_t sample_at(uint32_t i, uint64_t count) {
  if (count <= SAMPLE) return i;
  constexpr uint32_t C = 0x9E3779B1u;  // 2^32 / golden ratio, odd
  uint32_t x = (i + 1u) * C;
  x = (x ^ (x >> 15)) * C;
  x = (x ^ (x >> 13)) * C;
  x ^= x >> 16;
  const uint64_t first = i * count / SAMPLE, len = (i + 1u) * count / SAMPLE - first;
  return first + ((x * len) >> 32);  // len is at most 2^32 / SAMPLE
}

// Brackets the wanted rank from a sample (sample_at).  FIRST:
// of the elements themselves; otherwise of the candidates that the last pass
// wrote, whose rank and count are settled first.
template <bool FIRST>
__global__ __launch_bounds__(SMP_THREADS) void k_sel_sample(const int64_t *__restrict__ idx,
                                                            const double *__restrict__ vals,
                                                            int64_t nvals, Cands c, uint64_t n,
                                                            uint64_t goal, NarrowState *st) {
  __shared__ uint32_t hist[256], pick[3], num[2];
  __shared__ uint64_t found;
  uint64_t rank = goal, count = n;
  bool fail = false;
  if (!FIRST) {
    rank = st->rank - st->below();  // below > rank wraps to more than any count
    count = st->inside();
    fail = st->fail || rank >= count || count > c.cap;
  }
  __syncthreads();  // the state has been read
  if (fail) {       // uniform
    if (threadIdx.x == 0) {
      st->fail = 1;
      st->count = 0;
      st->tally = 0;
    }
    return;
  }
  const uint32_t S = (uint32_t)min(count, (uint64_t)SAMPLE);
  const uint32_t have = threadIdx.x < S ? (S - 1 - threadIdx.x) / SMP_THREADS + 1 : 0;
  uint64_t k[SMP_ITEMS], x[SMP_ITEMS];
#pragma unroll
  for (int i = 0; i < SMP_ITEMS; ++i) {
    k[i] = x[i] = 0;
    if ((uint32_t)i >= have) continue;
    const uint64_t j = sample_at(i * SMP_THREADS + threadIdx.x, count);
    if (FIRST) {
      const int64_t v = idx[j];
      x[i] = (uint64_t)v;
      k[i] = v >= 0 && v < nvals ? ordkey_sel(vals[v]) : 0;
    } else {
      k[i] = c.key[j];
      x[i] = (uint64_t)c.idx[j];
    }
  }
  // exact when the sample is everything
  const double p = (double)rank / (double)count;
  const int64_t t = S == count ? (int64_t)rank : (int64_t)(p * S);
  const int64_t w = S == count ? 0 : (int64_t)(4.0 * sqrt((double)S * p * (1.0 - p))) + 8;
  uint64_t lo = 0, hi = ~0ull, lox = 0, hix = ~0ull;
  if (t - w >= 0)
    block_select_pair(k, x, (1u << have) - 1u, (uint32_t)(t - w), hist, pick, &found, num, lo, lox);
  if (w == 0) {
    hi = lo;
    hix = lox;
  } else if (t + w < (int64_t)S) {
    block_select_pair(k, x, (1u << have) - 1u, (uint32_t)(t + w), hist, pick, &found, num, hi, hix);
  }
  if (threadIdx.x == 0) {
    st->rank = rank;
    st->count = count;
    st->lo = lo;
    st->hi = hi;
    st->lo_idx = lox;
    st->hi_idx = hix;
    st->tally = 0;
  }
}

constexpr int NARROW_TILE = SEL_THREADS * SEL_ITEMS;  // 4096 elements, 64 words of 64
static_assert(NARROW_TILE == 64 * 64, "a tile's words are scanned by one wavefront");

// What a tile of the first pass leaves for the partition.
struct Tiles {
  ulonglong2 *masks;    // per 64 elements: below the bracket, inside it
  uint32_t *below, *inside;  // per tile
  uint32_t *first;      // the tile's first candidate
  unsigned long long *before, *after;  // per tile: elements before / after the pivot, then scanned
};

// The first pass: every element against the bracket.  Copies the indices,
// and collects the candidates tile by tile in element order.
__global__ __launch_bounds__(SEL_THREADS) void k_sel_split(const int64_t *__restrict__ idx,
                                                           const double *__restrict__ vals,
                                                           int64_t n, int64_t nvals,
                                                           NarrowState *st,
                                                           int64_t *__restrict__ copy, Tiles t,
                                                           Cands c) {
  __shared__ uint32_t cnt[64];  // candidates per word, then before each word
  __shared__ uint32_t sum_b[SEL_THREADS / 64], base_s;
  const NarrowState br = *st;
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t base = (int64_t)blockIdx.x * NARROW_TILE;
  int64_t x[SEL_ITEMS];
  uint64_t k[SEL_ITEMS];
  bool bad = false;
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + it * SEL_THREADS + threadIdx.x;
    x[it] = i < n ? __builtin_nontemporal_load(idx + i) : 0;
    const bool ok = x[it] >= 0 && x[it] < nvals;
    bad |= i < n && !ok;
    if (!ok) x[it] = 0;  // nvals >= 1; the call is refused
  }
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) k[it] = ordkey_sel(vals[x[it]]);
  uint32_t nb = 0;
  uint64_t ins[SEL_ITEMS];
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + it * SEL_THREADS + threadIdx.x;
    if (i < n) __builtin_nontemporal_store(x[it], copy + i);
    const uint64_t mb = __builtin_amdgcn_ballot_w64(i < n && br.is_below(k[it], (uint64_t)x[it]));
    ins[it] = __builtin_amdgcn_ballot_w64(i < n && br.is_inside(k[it], (uint64_t)x[it]));
    nb += (uint32_t)__builtin_popcountll(mb);
    if (lane == 0) {
      const uint32_t word = it * (SEL_THREADS / 64) + w;
      t.masks[(size_t)blockIdx.x * 64 + word] = make_ulonglong2(mb, ins[it]);
      cnt[word] = (uint32_t)__builtin_popcountll(ins[it]);
    }
  }
  if (lane == 0) sum_b[w] = nb;
  if (bad) st->bad = 1;
  __syncthreads();
  if (w == 0) {
    const uint32_t v = cnt[lane], inc = wave_incl(v, lane);
    cnt[lane] = inc - v;
    if (lane == 63) {
      uint32_t b = 0;
      for (int q = 0; q < SEL_THREADS / 64; ++q) b += sum_b[q];
      t.below[blockIdx.x] = b;
      t.inside[blockIdx.x] = inc;
      base_s = (uint32_t)atomicAdd(&st->tally, ((unsigned long long)b << 32) | inc);
      t.first[blockIdx.x] = base_s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    if (!((ins[it] >> lane) & 1u)) continue;
    const uint64_t at = (uint64_t)base_s + cnt[it * (SEL_THREADS / 64) + w] +
                        __builtin_popcountll(ins[it] & ((1ull << lane) - 1u));
    if (at < c.cap) {
      c.key[at] = k[it];
      c.idx[at] = x[it];
    }
  }
}

// A further pass: the candidates inside the new bracket, in any order.  A
// workgroup takes tiles of 4096 and one atomic a tile (one a wavefront, for
// 64 candidates, took 285 us at 3.2 M candidates).
__global__ __launch_bounds__(SEL_THREADS) void k_sel_narrow(Cands from, Cands to,
                                                            NarrowState *st) {
  __shared__ uint32_t cnt[64];
  __shared__ uint32_t sum_b[SEL_THREADS / 64], base_s;
  const NarrowState br = *st;
  const uint64_t n = br.count;
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (uint64_t base = (uint64_t)blockIdx.x * NARROW_TILE; base < n;
       base += (uint64_t)gridDim.x * NARROW_TILE) {
    uint64_t k[SEL_ITEMS], x[SEL_ITEMS], ins[SEL_ITEMS];
    uint32_t nb = 0;
#pragma unroll
    for (int it = 0; it < SEL_ITEMS; ++it) {
      const uint64_t i = base + it * SEL_THREADS + threadIdx.x;
      k[it] = i < n ? from.key[i] : 0;
      x[it] = i < n ? (uint64_t)from.idx[i] : 0;
    }
#pragma unroll
    for (int it = 0; it < SEL_ITEMS; ++it) {
      const uint64_t i = base + it * SEL_THREADS + threadIdx.x;
      nb += (uint32_t)__builtin_popcountll(
          __builtin_amdgcn_ballot_w64(i < n && br.is_below(k[it], x[it])));
      ins[it] = __builtin_amdgcn_ballot_w64(i < n && br.is_inside(k[it], x[it]));
      if (lane == 0) cnt[it * (SEL_THREADS / 64) + w] = (uint32_t)__builtin_popcountll(ins[it]);
    }
    if (lane == 0) sum_b[w] = nb;
    __syncthreads();
    if (w == 0) {
      const uint32_t v = cnt[lane];
      const uint32_t inc = wave_incl(v, lane);
      cnt[lane] = inc - v;
      if (lane == 63) {
        uint32_t b = 0;
        for (int q = 0; q < SEL_THREADS / 64; ++q) b += sum_b[q];
        base_s = (uint32_t)atomicAdd(&st->tally, ((unsigned long long)b << 32) | inc);
      }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < SEL_ITEMS; ++it) {
      if (!((ins[it] >> lane) & 1u)) continue;
      const uint64_t at = (uint64_t)base_s + cnt[it * (SEL_THREADS / 64) + w] +
                          __builtin_popcountll(ins[it] & ((1ull << lane) - 1u));
      if (at < to.cap) {
        to.key[at] = k[it];
        to.idx[at] = (int64_t)x[it];
      }
    }
    __syncthreads();  // cnt and base_s are written again
  }
}

// The pivot among at most PIVOT_MAX candidates: by key, then by index.
__global__ __launch_bounds__(SMP_THREADS) void k_sel_pivot(Cands c, NarrowState *st) {
  __shared__ uint32_t hist[256], pick[3];
  __shared__ uint64_t found;
  __shared__ uint32_t num[2];
  const uint64_t rank = st->rank - st->below(), count = st->inside();
  if (st->fail || rank >= count || count > c.cap || count > PIVOT_MAX) {
    if (threadIdx.x == 0) st->fail = 1;
    return;
  }
  const uint32_t S = (uint32_t)count;
  const uint32_t have = threadIdx.x < S ? (S - 1 - threadIdx.x) / SMP_THREADS + 1 : 0;
  uint64_t k[PIVOT_ITEMS], x[PIVOT_ITEMS];
#pragma unroll
  for (int i = 0; i < PIVOT_ITEMS; ++i) {
    const bool use = (uint32_t)i < have;
    k[i] = use ? c.key[i * SMP_THREADS + threadIdx.x] : 0;
    x[i] = use ? (uint64_t)c.idx[i * SMP_THREADS + threadIdx.x] : 0;
  }
  uint64_t pk, px;
  block_select_pair(k, x, (1u << have) - 1u, (uint32_t)rank, hist, pick, &found, num, pk, px);
  if (threadIdx.x == 0) {
    st->pivot_key = pk;
    st->pivot_idx = (int64_t)px;
  }
}

// Per tile: elements before and after the pivot (a wavefront a tile).
__global__ __launch_bounds__(SEL_THREADS) void k_sel_tally(const NarrowState *st, Tiles t,
                                                           Cands c, uint32_t ntiles, int64_t n) {
  const uint32_t tile = (blockIdx.x * SEL_THREADS + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (tile >= ntiles) return;
  const uint64_t pk = st->pivot_key;
  const int64_t px = st->pivot_idx;
  const uint32_t m = t.inside[tile], f = t.first[tile];
  uint32_t b = 0, a = 0;
  for (uint32_t i = lane; i < m; i += 64) {
    const int cl = sel_class(c.key[f + i], c.idx[f + i], pk, px);
    b += cl == 0 ? 1u : 0u;
    a += cl == 2 ? 1u : 0u;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    b += __shfl_xor(b, o, 64);
    a += __shfl_xor(a, o, 64);
  }
  if (lane == 0) {
    const int64_t size = min((int64_t)NARROW_TILE, n - (int64_t)tile * NARROW_TILE);
    t.before[tile] = t.below[tile] + b;
    t.after[tile] = (uint64_t)size - t.below[tile] - m + a;
  }
}

// Exclusive scans of the per-tile counts: block 0 `before`, block 1 `after`.
// Each thread takes a run of consecutive tiles.
__global__ __launch_bounds__(1024) void k_sel_scan_tiles(unsigned long long *before,
                                                         unsigned long long *after, uint32_t nb) {
  __shared__ unsigned long long sh[16];
  unsigned long long *v = blockIdx.x ? after : before;
  const uint32_t per = (nb + 1023) / 1024, b = min(threadIdx.x * per, nb), e = min(b + per, nb);
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned long long sum = 0;
#pragma unroll 8
  for (uint32_t i = b; i < e; ++i) sum += v[i];
  const unsigned long long inc = wave_incl(sum, lane);
  if (lane == 63) sh[w] = inc;
  __syncthreads();
  unsigned long long run = inc - sum;
  for (uint32_t q = 0; q < 16; ++q) run += q < w ? sh[q] : 0;
  // eight loads at a time, before any store
  for (uint32_t i0 = b; i0 < e; i0 += 8) {
    unsigned long long c[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) c[q] = i0 + q < e ? v[i0 + q] : 0;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
      if (i0 + q < e) v[i0 + q] = run;
      run += c[q];
    }
  }
}

// Stable partition from the copied indices: "before" elements to [0, goal) in
// order, the pivot to goal, "after" elements to (goal, n) in order.
__global__ __launch_bounds__(SEL_THREADS) void k_sel_place(const int64_t *__restrict__ copy,
                                                           int64_t n, const NarrowState *st,
                                                           Tiles t, Cands c, uint64_t goal,
                                                           int64_t *__restrict__ out) {
  __shared__ uint32_t cnt[2][64];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t pk = st->pivot_key, below = (1ull << lane) - 1u;
  const int64_t px = st->pivot_idx;
  const int64_t base = (int64_t)blockIdx.x * NARROW_TILE;
  // candidates before every word of the tile
  const ulonglong2 mine = t.masks[(size_t)blockIdx.x * 64 + lane];
  const uint32_t c0 = (uint32_t)__builtin_popcountll(mine.y);
  const uint32_t cand0 = t.first[blockIdx.x] + wave_incl(c0, lane) - c0;
  int64_t x[SEL_ITEMS];
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const int64_t i = base + it * SEL_THREADS + threadIdx.x;
    x[it] = i < n ? __builtin_nontemporal_load(copy + i) : 0;
  }
  uint64_t mb[SEL_ITEMS], ma[SEL_ITEMS];
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const uint32_t word = it * (SEL_THREADS / 64) + w;
    const int64_t i = base + it * SEL_THREADS + threadIdx.x;
    const uint64_t b = __shfl(mine.x, word, 64), in = __shfl(mine.y, word, 64);
    int cl = (b >> lane) & 1u ? 0 : 2;
    const uint32_t f = __shfl(cand0, word, 64);
    if ((in >> lane) & 1u)
      cl = sel_class(c.key[f + (uint32_t)__builtin_popcountll(in & below)], x[it], pk, px);
    if (i >= n) cl = 3;
    mb[it] = __builtin_amdgcn_ballot_w64(cl == 0);
    ma[it] = __builtin_amdgcn_ballot_w64(cl == 2);
    if (lane == 0) {
      cnt[0][word] = (uint32_t)__builtin_popcountll(mb[it]);
      cnt[1][word] = (uint32_t)__builtin_popcountll(ma[it]);
    }
  }
  __syncthreads();
  const uint32_t b0 = cnt[0][lane], a0 = cnt[1][lane];
  const uint32_t bi = wave_incl(b0, lane) - b0, ai = wave_incl(a0, lane) - a0;
  int64_t *ob = out + t.before[blockIdx.x], *oa = out + goal + 1 + t.after[blockIdx.x];
#pragma unroll
  for (int it = 0; it < SEL_ITEMS; ++it) {
    const uint32_t word = it * (SEL_THREADS / 64) + w;
    const int64_t i = base + it * SEL_THREADS + threadIdx.x;
    const uint32_t pb = __shfl(bi, word, 64), pa = __shfl(ai, word, 64);
    if (i >= n) continue;
    if ((mb[it] >> lane) & 1u)
      ob[pb + (uint32_t)__builtin_popcountll(mb[it] & below)] = x[it];
    else if ((ma[it] >> lane) & 1u)
      oa[pa + (uint32_t)__builtin_popcountll(ma[it] & below)] = x[it];
    else
      out[goal] = x[it];
  }
}

size_t select_blocks(int64_t n) {
  return (size_t)((n + SEL_THREADS * SEL_ITEMS - 1) / (SEL_THREADS * SEL_ITEMS));
}

// Workspace: keys (n), partitioned copy (n), two count arrays, state, flag.
// Narrowing uses the same bytes: the copied indices (8 n), the words' masks
// (n / 4), the tiles' counts, and (n + n / 4 + n / 16) / 8 candidates of 16.
size_t select_workspace_bytes(int64_t n) {
  const size_t nb = select_blocks(n);
  return 8 * (size_t)n + 8 * (size_t)n + 16 * nb + sizeof(SelState) + 256;
}

// By narrowing: *done is set when it succeeded; otherwise idx is as it was.
// Returns hipErrorInvalidValue if an index is outside [0, nvals).
static hipError_t select_narrow(int64_t *idx, const double *vals, int64_t n, int64_t nvals,
                                int64_t goal, void *ws, hipStream_t s, bool *done) {
  *done = false;
  const uint32_t nb = (uint32_t)select_blocks(n);
  char *w = static_cast<char *>(ws);
  size_t used = 0;
  auto take = [&](size_t bytes) {
    char *p = w + used;
    used += (bytes + 15) / 16 * 16;
    return p;
  };
  NarrowState *st = reinterpret_cast<NarrowState *>(take(sizeof(NarrowState)));
  Tiles t;
  t.masks = reinterpret_cast<ulonglong2 *>(take(1024 * (size_t)nb));
  t.before = reinterpret_cast<unsigned long long *>(take(8 * (size_t)nb));
  t.after = reinterpret_cast<unsigned long long *>(take(8 * (size_t)nb));
  t.below = reinterpret_cast<uint32_t *>(take(4 * (size_t)nb));
  t.inside = reinterpret_cast<uint32_t *>(take(4 * (size_t)nb));
  t.first = reinterpret_cast<uint32_t *>(take(4 * (size_t)nb));
  int64_t *copy = reinterpret_cast<int64_t *>(take(8 * (size_t)n));
  // rounds after the first pass, each leaving a twentieth or so of the
  // candidates, until one workgroup's registers hold them
  const int rounds = n <= (1 << 17) ? 0 : n <= (1 << 22) ? 1 : n <= (1 << 27) ? 2 : 3;
  Cands c[4];
  uint64_t cap = std::max<uint64_t>((uint64_t)n / 8, 16);
  for (int r = 0; r <= rounds; ++r, cap /= 4) {
    c[r].cap = cap;
    c[r].key = reinterpret_cast<uint64_t *>(take(8 * cap));
    c[r].idx = reinterpret_cast<int64_t *>(take(8 * cap));
  }
  // (counts and candidate positions are held in 32 bits)
  if (used > select_workspace_bytes(n) || n > 0xffffffffll) return hipSuccess;  // radix passes
  hipError_t e;
  if ((e = hipMemsetAsync(st, 0, sizeof(NarrowState), s)) != hipSuccess) return e;
  k_sel_sample<true><<<1, SMP_THREADS, 0, s>>>(idx, vals, nvals, Cands{}, (uint64_t)n,
                                               (uint64_t)goal, st);
  k_sel_split<<<nb, SEL_THREADS, 0, s>>>(idx, vals, n, nvals, st, copy, t, c[0]);
  for (int r = 0; r < rounds; ++r) {
    k_sel_sample<false><<<1, SMP_THREADS, 0, s>>>(nullptr, nullptr, 0, c[r], 0, 0, st);
    const unsigned blocks =
        (unsigned)std::min<uint64_t>((c[r].cap + SEL_THREADS - 1) / SEL_THREADS, 1024);
    k_sel_narrow<<<blocks, SEL_THREADS, 0, s>>>(c[r], c[r + 1], st);
  }
  k_sel_pivot<<<1, SMP_THREADS, 0, s>>>(c[rounds], st);
  NarrowState h;
  if ((e = hipMemcpyAsync(&h, st, sizeof(h), hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  if (h.bad) return hipErrorInvalidValue;
  if (h.fail) return hipSuccess;
  k_sel_tally<<<(nb + 3) / 4, SEL_THREADS, 0, s>>>(st, t, c[0], nb, n);
  k_sel_scan_tiles<<<2, 1024, 0, s>>>(t.before, t.after, nb);
  k_sel_place<<<nb, SEL_THREADS, 0, s>>>(copy, n, st, t, c[0], (uint64_t)goal, idx);
  *done = true;
  return hipGetLastError();
}

// Select rank `goal` of idx[0..n) keyed by vals[idx[i]] and partition idx in
// place.  Returns hipErrorInvalidValue if an index is outside [0, nvals).
hipError_t launch_select(int64_t *idx, const double *vals, int64_t n, int64_t nvals,
                         int64_t goal, void *ws, hipStream_t s) {
  bool done = false;
  hipError_t e = select_narrow(idx, vals, n, nvals, goal, ws, s, &done);
  if (e != hipSuccess || done) return e;
  // every index has been checked
  const unsigned nbk = (unsigned)((n + SEL_THREADS - 1) / SEL_THREADS);
  const unsigned nb = (unsigned)select_blocks(n);
  char *w = static_cast<char *>(ws);
  uint64_t *keys = reinterpret_cast<uint64_t *>(w);
  int64_t *out = reinterpret_cast<int64_t *>(w + 8 * (size_t)n);
  unsigned long long *cnt = reinterpret_cast<unsigned long long *>(w + 16 * (size_t)n);
  SelState *st = reinterpret_cast<SelState *>(w + 16 * (size_t)n + 16 * (size_t)nb);
  k_sel_keys<<<std::max(nbk, 1u), SEL_THREADS, 0, s>>>(idx, vals, keys, n, st, (uint64_t)goal);
  for (int shift = 56; shift >= 0; shift -= 8) {
    k_sel_hist<false><<<nb, SEL_THREADS, 0, s>>>(keys, idx, n, st, shift);
    k_sel_pick<false><<<1, 256, 0, s>>>(st, shift);
  }
  k_sel_count_eq<<<nb, SEL_THREADS, 0, s>>>(keys, n, st);
  unsigned long long eq = 0;
  if ((e = hipMemcpyAsync(&eq, &st->hist[0], 8, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  if ((e = hipMemsetAsync(&st->hist[0], 0, 8, s)) != hipSuccess) return e;
  if (eq > 1) {
    // equal values: the pivot is the rank-th of them by index
    for (int shift = 56; shift >= 0; shift -= 8) {
      k_sel_hist<true><<<nb, SEL_THREADS, 0, s>>>(keys, idx, n, st, shift);
      k_sel_pick<true><<<1, 256, 0, s>>>(st, shift);
    }
  }
  k_sel_count<<<nb, SEL_THREADS, 0, s>>>(keys, idx, n, st, cnt, cnt + nb);
  k_sel_scan<<<1, 1024, 0, s>>>(cnt, nb);
  k_sel_scan<<<1, 1024, 0, s>>>(cnt + nb, nb);
  k_sel_scatter<<<nb, SEL_THREADS, 0, s>>>(keys, idx, n, st, cnt, cnt + nb, (uint64_t)goal, out);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  return hipMemcpyAsync(idx, out, sizeof(int64_t) * (size_t)n, hipMemcpyDeviceToDevice, s);
}

}  // namespace kd
