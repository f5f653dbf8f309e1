// Token sampling: greedy argmax and temperature / top-k / top-p / min-p
// inverse-CDF sampling, one 1024-thread workgroup per logits row.
//
// Semantics match ops/torch_ref.py::sample (descending order, ties by index);
// the thresholds and the draw are found without sorting the row, see sampling_row.inc and sample_by_counts.
#include "common.h"

namespace {

constexpr int ST = 1024;     // threads per row

template <typename T> __device__ __forceinline__ float to_f(T v) { return (float)v; }

struct ArgMax { float v; int i; };

__device__ __forceinline__ ArgMax better(ArgMax a, ArgMax b) {
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

// f(value, index) for every element of a row, 16 bytes at a time between the row's first and last 16-byte borders (a
// vocabulary size that is no multiple of eight leaves every row with another offset), four loads in flight per thread.
template <typename T, typename F> __device__ __forceinline__ void for_row(const T* row, int V, F&& f) {
  constexpr int N = 16 / (int)sizeof(T);
  typedef T Vec __attribute__((ext_vector_type(N)));
  const int head = min(V, (int)(((16u - ((unsigned)(uintptr_t)row & 15u)) & 15u) / sizeof(T)));
  const int nvec = (V - head) / N;
  const Vec* body = reinterpret_cast<const Vec*>(row + head);
  if ((int)threadIdx.x < head) f(to_f(row[threadIdx.x]), (int)threadIdx.x);
  int i = threadIdx.x;
  for (; i + 3 * ST < nvec; i += 4 * ST) {
    Vec v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = body[i + e * ST];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < N; ++j) f(to_f((T)v[e][j]), head + (i + e * ST) * N + j);
  }
  for (; i < nvec; i += ST) {
    const Vec v = body[i];
#pragma unroll
    for (int j = 0; j < N; ++j) f(to_f((T)v[j]), head + i * N + j);
  }
  const int rest = head + nvec * N + (int)threadIdx.x;
  if (rest < V) f(to_f(row[rest]), rest);
}

template <typename T>
__global__ __launch_bounds__(ST) void argmax_kernel(int* __restrict__ out, const T* __restrict__ logits, int V,
                                                    long stride) {
  __shared__ float sv[16];
  __shared__ int si[16];
  const T* row = logits + blockIdx.x * stride;
  ArgMax best{-INFINITY, 0x7fffffff};
  for_row(row, V, [&](float v, int i) {
    if (v > best.v || (v == best.v && i < best.i)) best = ArgMax{v, i};     // NaN never wins
  });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax other{__shfl_xor(best.v, o, 64), __shfl_xor(best.i, o, 64)};
    best = better(best, other);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { sv[wid] = best.v; si[wid] = best.i; }
  __syncthreads();
  if (wid == 0) {
    ArgMax b2 = lane < 16 ? ArgMax{sv[lane], si[lane]} : ArgMax{-INFINITY, 0x7fffffff};
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      ArgMax other{__shfl_xor(b2.v, o, 64), __shfl_xor(b2.i, o, 64)};
      b2 = better(b2, other);
    }
    if (lane == 0) out[blockIdx.x] = b2.i == 0x7fffffff ? 0 : b2.i;
  }
}

// block-wide maximum, broadcast to all threads
__device__ __forceinline__ float block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_max(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = lane < 16 ? red[lane] : -INFINITY;
  t = wave_max(t);
  __syncthreads();
  return t;
}

constexpr int BINS = 2048, CAP = 4096;
constexpr unsigned NORMAL_END = 0x40000000u;     // bits of 2.0: weights are at most 1; NaN and infinity lie above

// Weights (positive floats) by the leading bits of their representation: how many, and the sum of the bits below -
// whole numbers, so any order of additions gives the same.  Up to 2^22 elements both share one 64-bit word (19 low bits
// times 2^22 stays under 2^41), a single LDS atomic per element; WIDE keeps them apart.
template <bool WIDE> struct Hist {
  unsigned long long sum[BINS];
  unsigned cnt[WIDE ? BINS : 1];
  __device__ void clear() {
    for (int i = threadIdx.x; i < BINS; i += ST) { sum[i] = 0; if (WIDE) cnt[i] = 0; }
  }
  __device__ void add(int bin, unsigned low) {
    if (WIDE) { atomicAdd(&sum[bin], (unsigned long long)low); atomicAdd(&cnt[bin], 1u); }
    else atomicAdd(&sum[bin], (1ull << 41) | low);
  }
  __device__ unsigned count(int bin) const { return WIDE ? cnt[bin] : (unsigned)(sum[bin] >> 41); }
  __device__ unsigned long long lows(int bin) const { return WIDE ? sum[bin] : sum[bin] & ((1ull << 41) - 1); }
};

__device__ __forceinline__ double pow2(int e) { return __longlong_as_double((long long)(1023 + e) << 52); }
// integer significand and exponent of a weight: value = sig * 2^(lsb)
__device__ __forceinline__ unsigned sig_of(unsigned bits) {
  return (bits & 0x7fffffu) | (bits >> 23 ? 0x800000u : 0u);
}
__device__ __forceinline__ int lsb_of(unsigned bits) { return (int)max(bits >> 23, 1u) - 150; }

// what sample_by_counts keeps beside the counts
struct CountShared { unsigned low, inf, lo, hi, counted, of_stretch[128]; };
struct SampleShared {
  double wmass[16];
  unsigned wcnt[16];
  double mass, above_mass;
  unsigned above_cnt, cnt, n_list;
  int best, n, token, bad;
};

// exclusive scan of (count, mass) over the block in thread order; totals to every thread (by shuffles, which go through LDS, a row's
// two scans of sample_by_counts took 2.5 us more)
__device__ __forceinline__ void block_scan(unsigned c, double m, unsigned& ec, double& em, double& total, SampleShared& s) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned ic = (unsigned)wave_scan((int)c);
  const double im = wave_scan(m);
  if (lane == 63) { s.wcnt[wid] = ic; s.wmass[wid] = im; }
  __syncthreads();
  unsigned bc = 0;
  double bm = 0, all = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wid) { bc += s.wcnt[w]; bm += s.wmass[w]; }
    all += s.wmass[w];
  }
  ec = bc + ic - c;
  em = bm + im - m;
  total = all;
  __syncthreads();
}

// A histogram's two bins of each thread, the heaviest of all first: counts, masses, and what lies in front of them.  Bins hold the
// bits `prefix | bin << shift ..`.
struct Bins {
  unsigned c[2], ec;
  double m[2], em, total;
};
template <bool WIDE> __device__ __forceinline__ Bins sum_bins(const Hist<WIDE>& h, unsigned prefix, int shift, SampleShared& s) {
  Bins t;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int bin = BINS - 1 - (2 * (int)threadIdx.x + e);
    const unsigned bits = prefix | ((unsigned)bin << shift);
    t.c[e] = h.count(bin);
    t.m[e] = t.c[e] ? ((double)t.c[e] * sig_of(bits) + (double)h.lows(bin)) * pow2(lsb_of(bits)) : 0.0;
  }
  block_scan(t.c[0] + t.c[1], t.m[0] + t.m[1], t.ec, t.em, t.total, s);
  return t;
}
// The lowest non-empty bin (at or above `first`) in front of which, `above` included, fewer than K elements and less than M of mass
// lie: its index, count and what lies above it go to `s` (best = -1: none).
__device__ __forceinline__ void find_bin(const Bins& t, int first, unsigned above_cnt, double above_mass, unsigned K, double M,
                                         SampleShared& s) {
  if (threadIdx.x == 0) s.best = -1;
  __syncthreads();
  const unsigned ec = t.ec + above_cnt;
  const double em = t.em + above_mass;
  int mine = -1;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int order = 2 * (int)threadIdx.x + e;
    if (t.c[e] && BINS - 1 - order >= first && ec + (e ? t.c[0] : 0) < K && em + (e ? t.m[0] : 0.0) < M) mine = order;
  }
  // (orders rise with the lanes: a wave's last one speaks for it)
  const unsigned long long those = __ballot(mine >= 0);
  if (mine >= 0 && (those >> (threadIdx.x & 63)) == 1ull) atomicMax(&s.best, mine);
  __syncthreads();
  const int best = s.best;
  __syncthreads();
  if (best >= 0 && best >> 1 == (int)threadIdx.x) {
    const bool second = best & 1;
    s.above_cnt = ec + (second ? t.c[0] : 0);
    s.above_mass = em + (second ? t.m[0] : 0.0);
    s.cnt = second ? t.c[1] : t.c[0];
    s.best = BINS - 1 - best;
  }
  __syncthreads();
}

// sort `n` keys (padded with zeros to a power of two here) in LDS, largest first
__device__ void sort_list(unsigned long long* list, int n) {
  int p = 2;
  while (p < n) p <<= 1;
  for (int i = n + threadIdx.x; i < p; i += ST) list[i] = 0;
  __syncthreads();
  for (int k = 2; k <= p; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < p / 2; t += ST) {
        const int a = 2 * t - (t & (j - 1)), b = a + j;      // the pair `t` of this stage
        const unsigned long long x = list[a], y = list[b];
        if ((x < y) == ((a & k) == 0)) { list[a] = y; list[b] = x; }
      }
      __syncthreads();
    }
}

template <bool WIDE> struct ListShared {
  Hist<WIDE> h1, h2;
  unsigned long long list[CAP];
};

constexpr int PATTERNS = 65536;

// The 16-bit patterns of T in the order of their weights: place d = 0 .. 65535 falls with the value (`flip`: rises)
template <typename T> struct Order16 {
  static constexpr unsigned INF = std::is_same<T, bf16_t>::value ? 0x7f80u : 0x7c00u;
  static constexpr unsigned FIRST = 0x7fffu - INF;               // of the infinity in front of everything; NaNs lie below it
  static constexpr unsigned LOWEST = 0xffffu - FIRST - 1u;       // of the last finite one; the other infinity and NaNs above it
  static __device__ __forceinline__ unsigned place(unsigned bits, unsigned flip) {
    return ((bits & 0x8000u ? bits : bits ^ 0x7fffu) ^ flip) & 0xffffu;
  }
  static __device__ __forceinline__ unsigned bits(unsigned d, unsigned flip) {
    const unsigned e = (d ^ flip) & 0xffffu;
    return e & 0x8000u ? e : e ^ 0x7fffu;
  }
  static __device__ __forceinline__ float value(unsigned d, unsigned flip) {
    return to_f(__builtin_bit_cast(T, (unsigned short)bits(d, flip)));
  }
};
typedef unsigned short Pair16 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Pair16 pair16(unsigned x) { return __builtin_bit_cast(Pair16, x); }
__device__ __forceinline__ unsigned both16(unsigned x) { return x | x << 16; }

// f(the 16 bytes of eight elements, their place among the row's) for the row's part between its first and last 16-byte borders,
// g(element, its index) for the others; every thread of the block takes part in every round (`live`: it has a piece)
template <typename T, typename F, typename G> __device__ __forceinline__ void for_row16(const T* row, int V, F&& f, G&& g) {
  typedef unsigned Vec __attribute__((ext_vector_type(4)));
  const int head = min(V, (int)(((16u - ((unsigned)(uintptr_t)row & 15u)) & 15u) / sizeof(T)));
  const int nvec = (V - head) / 8;
  const Vec* body = reinterpret_cast<const Vec*>(row + head);
  const unsigned short* raw = reinterpret_cast<const unsigned short*>(row);
  if ((int)threadIdx.x < head) g((unsigned)raw[threadIdx.x], (int)threadIdx.x);
  int i = threadIdx.x;
  if (nvec >= 4 * ST) {
    Vec v[4], next[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = body[i + e * ST];
    for (;;) {
      const bool more = i - (int)threadIdx.x + 8 * ST <= nvec;   // (the next four are on their way while these are looked at)
      if (more)
#pragma unroll
        for (int e = 0; e < 4; ++e) next[e] = body[i + (4 + e) * ST];
#pragma unroll
      for (int e = 0; e < 4; ++e) f(v[e], i + e * ST, true);
      i += 4 * ST;
      if (!more) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = next[e];
    }
  }
  for (; i - (int)threadIdx.x < nvec; i += ST) {
    const bool live = i < nvec;
    f(live ? body[i] : Vec{0u, 0u, 0u, 0u}, i, live);
  }
  const int rest = head + nvec * 8 + (int)threadIdx.x;
  if (rest < V) g((unsigned)raw[rest], rest);
}

// Rows of 16-bit logits: the same two questions (see sampling_row.inc), answered from how often each of the 65536 patterns
// occurs.  One pass over the row counts them (16 bits each, 128 KB of LDS); the ones that occur - a few thousand - are packed
// into a list in order, weighed once each, and summed up; what is kept and the pattern that the draw falls on follow from the
// list, with no further look at the row and no sort.  A second pass finds the element: the drawn pattern's elements come in
// the order of their indices, so each wave counts them in its 512 elements at a time, and the one stretch that the wanted one
// lies in is looked at again.  Masses are counts times weights, in doubles: no result depends on the order of additions.
// Bound by the LDS atomics and the vector instructions of the counting pass (10 us of a row of 128256 alone, 16 of 256 rows at
// once, whose logits take 14 from memory), by the second pass (6 and 9) and by a dozen steps of a microsecond or two between
// them.  256 rows of 128256 bf16 logits, every kind of filter among them: 38 us, by bins 118 when this was chosen (93 now); one row
// 29 (62, 53), one of 32000 18 (37, 25).  The patterns are packed by stretches of 512 places a wave: with 64 places a thread the few
// threads that have any were 7 us on their own (3.2 so).
// -1: a pattern occurs 65536 times or more (a count ran over: the counts' sum is then too small), more than 32768 patterns
// occur, or the row is longer than the second pass has counters for.  The type's lowest value and the infinity next to it, which
// masks fill rows with, are counted apart, in registers.
template <typename T>
__device__ int sample_by_counts(const T* row, int V, float inv_t, unsigned k, float tp, float mp, float u, unsigned* tab,
                                SampleShared& s, CountShared& cs) {
  using O = Order16<T>;
  typedef unsigned Vec __attribute__((ext_vector_type(4)));
  if (V > 1 << 23) return -1;
  const unsigned flip = inv_t < 0.f ? 0xffffffffu : 0u;
  const float to_exp2 = inv_t * 1.4426950408889634f;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
#pragma unroll
  for (int j = 0; j < PATTERNS / 2 / (4 * ST); ++j) *reinterpret_cast<Vec*>(tab + 4 * (j * ST + tid)) = Vec{0u, 0u, 0u, 0u};
  if (tid == 0) { s.bad = 0; cs.low = 0; cs.inf = 0; cs.counted = 0; }
  __syncthreads();
  // ---- how often each pattern occurs
  unsigned low = 0, inf = 0, nan = 0;
  const unsigned lowest = O::bits(O::LOWEST, flip), magnitude = lowest & 0x7fffu;
  auto count = [&](unsigned x) { atomicAdd(tab + (x >> 1), x & 1u ? 0x10000u : 1u); };
  auto one = [&](unsigned x) {
    if (x == lowest) ++low;
    else if (x == lowest + 1) ++inf;
    else if ((x & 0x7fffu) > magnitude + 1) nan = 1;
    else count(x);
  };
  for_row16(
      row, V,
      [&](Vec v, int, bool live) {
        if (!live) return;
        const Pair16 most = __builtin_elementwise_max(
            __builtin_elementwise_max(pair16(v[0] & 0x7fff7fffu), pair16(v[1] & 0x7fff7fffu)),
            __builtin_elementwise_max(pair16(v[2] & 0x7fff7fffu), pair16(v[3] & 0x7fff7fffu)));
        if (__builtin_expect(max((unsigned)most[0], (unsigned)most[1]) < magnitude, 1)) {
#pragma unroll
          for (int w = 0; w < 4; ++w) { count(v[w] & 0xffffu); count(v[w] >> 16); }
        } else {
#pragma unroll
          for (int w = 0; w < 4; ++w) { one(v[w] & 0xffffu); one(v[w] >> 16); }
        }
      },
      [&](unsigned x, int) { one(x); });
  if (low) atomicAdd(&cs.low, low);
  if (inf) atomicAdd(&cs.inf, inf);
  if (nan) s.bad = 1;
  __syncthreads();
  // ---- those that occur, in order, as (place, count) words in the counts' stead: 128 stretches of 512 places, eight a lane,
  // dealt to the waves in turn (values lie in a few octaves: most stretches are empty, and neighbours go to different waves)
  unsigned n;
  {
    constexpr int ROUNDS = PATTERNS / 8 / ST;
    Vec v[ROUNDS];
    unsigned pos[ROUNDS], used = 0;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      const unsigned piece = j * ST + tid, there = flip ? PATTERNS / 8 - 1 - piece : piece;     // (positive patterns lie backwards)
      const bool back = (there < PATTERNS / 16) != (flip != 0u);
      v[j] = *reinterpret_cast<const Vec*>(tab + 4 * (there < PATTERNS / 16 ? PATTERNS / 16 - 1 - there : there));
      if (back) v[j] = Vec{v[j][3], v[j][2], v[j][1], v[j][0]};
    }
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      unsigned total = 0;
      if (__any((v[j][0] | v[j][1] | v[j][2] | v[j][3]) != 0)) {
        used |= 1u << j;
        const unsigned there = flip ? PATTERNS / 8 - 1 - (j * ST + tid) : j * ST + tid;
        const bool back = (there < PATTERNS / 16) != (flip != 0u);
        unsigned c = 0, sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (back) v[j][w] = v[j][w] >> 16 | v[j][w] << 16;
          const unsigned lo = v[j][w] & 0xffffu, hi = v[j][w] >> 16;
          c += (lo != 0) + (hi != 0);
          sum += lo + hi;
        }
        if (sum) atomicAdd(&cs.counted, sum);
        unsigned before = 0;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) {
          const unsigned long long have = __ballot(c >> bit & 1u);
          before += (unsigned)__popcll(have & ((1ull << lane) - 1ull)) << bit;
          total += (unsigned)__popcll(have) << bit;
        }
        pos[j] = before;
      }
      if (lane == 0) cs.of_stretch[j * (ST / 64) + wid] = total;
    }
    __syncthreads();
    const unsigned even = cs.of_stretch[2 * lane], odd = cs.of_stretch[2 * lane + 1];
    const unsigned upto = (unsigned)wave_scan((int)(even + odd));
    n = __shfl(upto, 63, 64);
    if (cs.counted != (unsigned)V - cs.low - cs.inf && !s.bad) return -1;
    if (n > PATTERNS / 2) return -1;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      if (!(used >> j & 1u)) continue;
      const int stretch = j * (ST / 64) + wid;
      unsigned at = pos[j] + __shfl(upto - even - odd, stretch >> 1, 64) + (stretch & 1 ? __shfl(even, stretch >> 1, 64) : 0u);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const unsigned d = 8u * (j * ST + tid) + 2u * w;
        if (v[j][w] & 0xffffu) tab[at++] = d << 16 | (v[j][w] & 0xffffu);
        if (v[j][w] >> 16) tab[at++] = (d + 1u) << 16 | v[j][w] >> 16;
      }
    }
    __syncthreads();
  }
  const unsigned lows = cs.low;
  // the row's largest entry (its place: the one in front of all); NaN, and an infinity there, are no distribution
  const unsigned first = n ? tab[0] >> 16 : (lows ? O::LOWEST : O::LOWEST + 1);
  const float top = O::value(first, flip);
  auto weight = [&](unsigned d) { return __float_as_uint(fast_exp2((O::value(d, flip) - top) * to_exp2)); };
  if (s.bad || first <= O::FIRST || (cs.inf && weight(O::LOWEST + 1) >= NORMAL_END)) return 0;
  // ---- entry n is the type's lowest value; a thread has `per` of them in a row
  const unsigned per = (n + 1 + ST - 1) / ST, e0 = min(per * tid, n + 1), e1 = min(e0 + per, n + 1);
  auto entry = [&](unsigned e, unsigned& d, unsigned& c) {
    const unsigned x = e < n ? tab[e] : 0u;
    d = e < n ? x >> 16 : O::LOWEST;
    c = e < n ? x & 0xffffu : lows;
  };
  auto mass_of = [](unsigned w) { return sig_of(w) * pow2(lsb_of(w)); };
  unsigned cnt = 0, ec;
  double m = 0, em, z;
  bool odd = false;
  for (unsigned e = e0; e < e1; ++e) {
    unsigned d, c;
    entry(e, d, c);
    const unsigned w = weight(d);
    if (!c || !w) continue;                        // (a weight of zero is never sampled and adds nothing)
    odd = odd || w >= NORMAL_END;
    cnt += c;
    m += c * mass_of(w);
  }
  if (odd) s.bad = 1;
  block_scan(cnt, m, ec, em, z, s);
  if (s.bad) return 0;
  unsigned kept = (unsigned)V, rank = 0;
  double mass = z;
  for (int step = 0; step < 2; ++step) {
    const unsigned minb = step == 0 && mp > 0.f ? __float_as_uint(fminf(mp, 1.f)) : 0u;
    if (step == 0 && k >= (unsigned)V && tp >= 1.f && minb == 0u) continue;      // everything is kept
    const double M = step == 0 ? (tp >= 1.f ? 1e300 : fmax((double)tp * z, 1e-300)) : fmax((double)u * mass, 1e-300);
    const unsigned K = step == 0 ? k : kept;
    if (tid == 0) s.best = -1;
    __syncthreads();
    int best = -1;
    unsigned in_front = ec, best_c = 0, best_front = 0, best_w = 0;
    double above = em, best_above = 0;
    if (ec < K && em < M)
      for (unsigned e = e0; e < e1; ++e) {
        unsigned d, c;
        entry(e, d, c);
        const unsigned w = weight(d);
        if (!c || !w) continue;
        if (in_front < K && above < M && w >= minb) {
          best = (int)e; best_c = c; best_front = in_front; best_w = w; best_above = above;
        }
        in_front += c;
        above += c * mass_of(w);
      }
    // (entries rise with the lanes: a wave's last one speaks for it)
    if (best >= 0 && (__ballot(best >= 0) >> lane) == 1ull) atomicMax(&s.best, best);
    __syncthreads();
    if (best >= 0 && s.best == best) {
      const double v = mass_of(best_w);
      const double fit = fmin(fmax(ceil((M - best_above) / v), 1.0), (double)best_c);
      const unsigned take = min((unsigned)fit, K - best_front);
      s.above_cnt = best_front + take;
      s.mass = best_above + take * v;
      s.cnt = best_w;
      s.n = (int)take;
    }
    __syncthreads();
    if (s.best < 0) return 0;                      // (no weights at all)
    kept = s.above_cnt;
    mass = s.mass;
    rank = (unsigned)s.n;
    __syncthreads();
  }
  // ---- the rank-th element (from 1) of the patterns that weigh as much: those beside the found one count in front of it
  const int found = s.best;
  const unsigned wanted = s.cnt;
  if (tid == 0) { s.n_list = rank; cs.lo = 0xffffu; cs.hi = 0u; }
  __syncthreads();
  for (unsigned e = e0; e < e1; ++e) {
    unsigned d, c;
    entry(e, d, c);
    if (!c || weight(d) != wanted) continue;
    atomicMin(&cs.lo, d);
    atomicMax(&cs.hi, d);
    if ((int)e < found) atomicAdd(&s.n_list, c);
  }
  __syncthreads();
  rank = s.n_list;
  const unsigned lo = cs.lo, span = cs.hi - lo;
  // ---- how many of them each 512 elements hold: counter 0 for what lies in front of the first 16-byte border
  const int head = min(V, (int)(((16u - ((unsigned)(uintptr_t)row & 15u)) & 15u) / sizeof(T)));
  const int nvec = (V - head) / 8, parts = (nvec + 63) / 64;
  const unsigned short* raw = reinterpret_cast<const unsigned short*>(row);
  auto hit = [&](unsigned x) { return ((O::place(x, flip) - lo) & 0xffffu) <= span; };
  const unsigned drawn = both16(O::bits(lo, flip));
  if (tid == 0) { tab[0] = 0; s.best = -1; s.token = 0; }
  if (tid == 1) tab[parts + 1] = 0;
  __syncthreads();
  auto hits_of = [&](unsigned c, int i, bool live) {             // c: among a thread's eight elements
    unsigned sum = 0;
    if (__any(c != 0))
#pragma unroll
      for (int bit = 0; bit < 4; ++bit) sum += (unsigned)__popcll(__ballot(c >> bit & 1u)) << bit;
    if (lane == 0 && live) tab[1 + (i >> 6)] = sum;
  };
  auto single = [&](unsigned x, int i) { if (hit(x)) atomicAdd(tab + (i < head ? 0 : parts + 1), 1u); };
  if (span == 0)                                   // (one pattern, as good as always)
    for_row16(
        row, V,
        [&](Vec v, int i, bool live) {
          const Pair16 l = {1, 1};
          Pair16 others = {0, 0};
#pragma unroll
          for (int w = 0; w < 4; ++w) others += __builtin_elementwise_min(pair16(v[w] ^ drawn), l);
          hits_of(live ? 8u - others[0] - others[1] : 0u, i, live);
        },
        single);
  else
    for_row16(
        row, V,
        [&](Vec v, int i, bool live) {
          unsigned c = 0;
#pragma unroll
          for (int w = 0; w < 4; ++w) c += hit(v[w] & 0xffffu) + hit(v[w] >> 16);
          hits_of(live ? c : 0u, i, live);
        },
        single);
  __syncthreads();
  // ---- the stretch that the wanted one lies in
  const unsigned each = (parts + 2 + ST - 1) / ST;
  unsigned mine = 0, before;
  for (unsigned e = 0; e < each; ++e) {
    const int i = (int)(each * tid + e);
    if (i < parts + 2) mine += tab[i];
  }
  double none, all;
  block_scan(mine, 0.0, before, none, all, s);
  if (before < rank && rank <= before + mine)
    for (unsigned e = 0; e < each; ++e) {
      const int i = (int)(each * tid + e);
      if (i >= parts + 2) break;
      if (rank <= before + tab[i]) { s.best = i; s.cnt = rank - before; break; }
      before += tab[i];
    }
  __syncthreads();
  const int part = s.best;
  unsigned want = s.cnt;
  if (wid == 0 && part >= 0) {
    if (part == 0 || part == parts + 1) {
      const int from = part == 0 ? 0 : head + 8 * nvec, count = part == 0 ? head : V - from;
      const bool h = lane < count && hit((unsigned)raw[from + (lane < count ? lane : 0)]);
      const unsigned long long hits = __ballot(h);
      if (h && (unsigned)__popcll(hits & ((1ull << lane) - 1ull)) == want - 1u) s.token = from + lane;
    } else {
      const int i = (part - 1) * 64 + lane;
      const bool live = i < nvec;
      const Vec v = live ? reinterpret_cast<const Vec*>(row + head)[i] : Vec{0u, 0u, 0u, 0u};
      unsigned hits = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        hits |= (unsigned)hit(v[w] & 0xffffu) << (2 * w) | (unsigned)hit(v[w] >> 16) << (2 * w + 1);
      if (!live) hits = 0;
      const unsigned c = __popc(hits);
      const unsigned upto = (unsigned)wave_scan((int)c);
      if (upto - c < want && want <= upto) {
        want -= upto - c;
        for (int e = 0; e < 8; ++e)
          if (hits >> e & 1u && --want == 0) s.token = head + 8 * i + e;
      }
    }
  }
  __syncthreads();
  return s.token;
}

// 32-bit logits
template <typename T, bool WIDE>
__global__ __launch_bounds__(ST) void sample_kernel(int* __restrict__ out, const T* __restrict__ logits, int V,
                                                    long stride, const float* __restrict__ temperature,
                                                    const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                    const float* __restrict__ min_p,
                                                    const float* __restrict__ uniform) {
  __shared__ Hist<WIDE> h1, h2;
  __shared__ unsigned long long list[CAP];
  __shared__ SampleShared s;
  __shared__ float red[16];
  __shared__ int s_idx;
  static_assert(sizeof(T) == 4, "");
  unsigned* const tab = nullptr;
  CountShared cs;
#include "sampling_row.inc"
}

// 16-bit logits: the counts take the place of the histograms
template <typename T, bool WIDE>
__global__ __launch_bounds__(ST) void sample16_kernel(int* __restrict__ out, const T* __restrict__ logits, int V,
                                                    long stride, const float* __restrict__ temperature,
                                                    const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                    const float* __restrict__ min_p,
                                                    const float* __restrict__ uniform) {
  __shared__ union {
    ListShared<WIDE> bins;
    unsigned counts[PATTERNS / 2];
  } sh;
  __shared__ SampleShared s;
  __shared__ CountShared cs;
  __shared__ float red[16];
  __shared__ int s_idx;
  static_assert(sizeof(T) == 2, "");
  Hist<WIDE>&h1 = sh.bins.h1, &h2 = sh.bins.h2;
  unsigned long long* const list = sh.bins.list;
  unsigned* const tab = sh.counts;
#include "sampling_row.inc"
}

}  // namespace

VDAMD_API int vdamd_argmax(int* out, const void* logits, int B, int V, long stride, int dtype, hipStream_t s) {
  if (B == 0) return 0;
  if (dtype == DT_BF16)
    hipLaunchKernelGGL(argmax_kernel<bf16_t>, dim3(B), dim3(ST), 0, s, out, (const bf16_t*)logits, V, stride);
  else if (dtype == DT_F16)
    hipLaunchKernelGGL(argmax_kernel<f16_t>, dim3(B), dim3(ST), 0, s, out, (const f16_t*)logits, V, stride);
  else if (dtype == DT_F32)
    hipLaunchKernelGGL(argmax_kernel<float>, dim3(B), dim3(ST), 0, s, out, (const float*)logits, V, stride);
  else return -2;
  HIP_LAUNCH_CHECK();
  return 0;
}

VDAMD_API int vdamd_sample(int* out, const void* logits, int B, int V, long stride, const float* temperature,
                           const int* top_k, const float* top_p, const float* min_p, const float* uniform,
                           int dtype, hipStream_t s) {
  if (B == 0) return 0;
#define L(KERNEL, TY)                                                                                                       \
  do {                                                                                                              \
    if (V <= (1 << 22))                                                                                             \
      hipLaunchKernelGGL((KERNEL<TY, false>), dim3(B), dim3(ST), 0, s, out, (const TY*)logits, V, stride,    \
                         temperature, top_k, top_p, min_p, uniform);                                                \
    else                                                                                                            \
      hipLaunchKernelGGL((KERNEL<TY, true>), dim3(B), dim3(ST), 0, s, out, (const TY*)logits, V, stride,     \
                         temperature, top_k, top_p, min_p, uniform);                                                \
  } while (0)
  if (dtype == DT_BF16) L(sample16_kernel, bf16_t);
  else if (dtype == DT_F16) L(sample16_kernel, f16_t);
  else if (dtype == DT_F32) L(sample_kernel, float);
  else return -2;
#undef L
  HIP_LAUNCH_CHECK();
  return 0;
}
