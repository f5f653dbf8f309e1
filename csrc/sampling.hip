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

// A row's histogram goes by a weight's exponent and its SHIFT1 = 17 lowest bits' neighbours above (six): a bin of a Gaussian row of 128k
// has some 250 entries.  What is cut further goes by the next eleven bits, and by the last six
constexpr int BINS1 = 8192, SHIFT1 = 17, BINS = 2048, SHIFT2 = 6, CAP = 4096;
constexpr unsigned NORMAL_END = 0x40000000u;     // bits of 2.0: weights are at most 1; NaN and infinity lie above

// Weights (positive floats) by the leading bits of their representation: how many, and the sum of the bits below -
// whole numbers, so any order of additions gives the same.  Up to 2^22 elements both share one 64-bit word (17 low bits
// times 2^22 stay under 2^39, the count begins at 2^41), a single LDS atomic per element; WIDE keeps them apart.
template <bool WIDE, int N> struct Hist {
  unsigned long long sum[N];
  unsigned cnt[WIDE ? N : 1];
  __device__ void clear() {
    for (int i = threadIdx.x; i < N; i += ST) { sum[i] = 0; if (WIDE) cnt[i] = 0; }
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
  double wmass[2][16];
  unsigned wcnt[2][16];
  int wbest[2][16];
  double mass, above_mass;
  unsigned above_cnt, cnt, n_list;
  int best, n, token, bad;
};

// The waves' words take turns in two places, so that a step needs no barrier to have its words read before the next one's are written:
// between two uses of a place lies the barrier of the step between.
typedef unsigned Turn;

// exclusive scan of (count, mass) over the block in thread order; totals to every thread (by shuffles, which go through LDS, a row's
// two scans of sample_by_counts took 2.5 us more).  The waves' totals, one a lane, are scanned by every wave: sixteen conditional
// additions of doubles in each of sixteen waves took 0.8 us
__device__ __forceinline__ void block_scan(unsigned c, double m, unsigned& ec, double& em, double& total, SampleShared& s, Turn& turn) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned ic = (unsigned)wave_scan((int)c);
  const double im = wave_scan(m);
  unsigned* const wcnt = s.wcnt[turn & 1];
  double* const wmass = s.wmass[turn & 1];
  ++turn;
  if (lane == 63) { wcnt[wid] = ic; wmass[wid] = im; }
  __syncthreads();
  const bool one = lane < 16;
  const unsigned tc = (unsigned)wave_scan(one ? (int)wcnt[lane & 15] : 0);
  const double tm = wave_scan(one ? wmass[lane & 15] : 0.0);
  auto of = [&](double v, int l) {
    const unsigned long long w = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)w, l), hi = __builtin_amdgcn_readlane((unsigned)(w >> 32), l);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
  };
  const unsigned bc = wid ? (unsigned)__builtin_amdgcn_readlane((int)tc, wid - 1) : 0u;
  const double bm = wid ? of(tm, wid - 1) : 0.0;
  ec = bc + ic - c;
  em = bm + im - m;
  total = of(tm, 15);
}
// the largest of the threads' numbers, which rise with the threads of a wave (-1: none)
__device__ __forceinline__ int block_last(int mine, SampleShared& s, Turn& turn) {
  const int lane = threadIdx.x & 63;
  const unsigned long long those = __ballot(mine >= 0);
  int* const wbest = s.wbest[turn & 1];
  ++turn;
  if (those ? (those >> lane) == 1ull : lane == 0) wbest[threadIdx.x >> 6] = mine;
  __syncthreads();
  int best = wbest[lane & 15];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    const int other = o == 8 ? __builtin_amdgcn_update_dpp(0, best, 0x128, 0xf, 0xf, true)
                    : o == 4 ? __builtin_amdgcn_update_dpp(0, best, 0x124, 0xf, 0xf, true)
                    : o == 2 ? __builtin_amdgcn_update_dpp(0, best, 0x4E, 0xf, 0xf, true)
                             : __builtin_amdgcn_update_dpp(0, best, 0xB1, 0xf, 0xf, true);
    best = max(best, other);
  }
  return __builtin_amdgcn_readfirstlane(best);
}

// A histogram's bins of each thread, the heaviest of all first: counts, masses, and what lies in front of them.  Bins hold the
// bits `prefix | bin << shift ..`.
template <int PER> struct Bins {
  unsigned c[PER], ec;
  double m[PER], em, total;
};
template <bool WIDE, int N>
__device__ __forceinline__ Bins<N / ST> sum_bins(const Hist<WIDE, N>& h, unsigned prefix, int shift, SampleShared& s, Turn& turn) {
  Bins<N / ST> t;
  unsigned c = 0;
  double m = 0;
#pragma unroll
  for (int e = 0; e < N / ST; ++e) {
    const int bin = N - 1 - (N / ST * (int)threadIdx.x + e);
    const unsigned bits = prefix | ((unsigned)bin << shift);
    t.c[e] = h.count(bin);
    t.m[e] = t.c[e] ? ((double)t.c[e] * sig_of(bits) + (double)h.lows(bin)) * pow2(lsb_of(bits)) : 0.0;
    c += t.c[e];
    m += t.m[e];
  }
  block_scan(c, m, t.ec, t.em, t.total, s, turn);
  return t;
}
// The lowest non-empty bin (at or above `first`) in front of which, `above` included, fewer than K elements and less than M of mass
// lie: its index, count and what lies above it go to `s` (best = -1: none).
template <int PER>
__device__ __forceinline__ void find_bin(const Bins<PER>& t, int first, unsigned above_cnt, double above_mass, unsigned K, double M,
                                         SampleShared& s, Turn& turn) {
  unsigned ec = t.ec + above_cnt, best_c = 0, best_ec = 0;
  double em = t.em + above_mass, best_em = 0;
  int mine = -1;
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int order = PER * (int)threadIdx.x + e;
    if (t.c[e] && PER * ST - 1 - order >= first && ec < K && em < M) {
      mine = order;
      best_c = t.c[e];
      best_ec = ec;
      best_em = em;
    }
    ec += t.c[e];
    em += t.m[e];
  }
  const int best = block_last(mine, s, turn);
  if (best < 0) {
    if (threadIdx.x == 0) s.best = -1;
  } else if (best == mine) {
    s.above_cnt = best_ec;
    s.above_mass = best_em;
    s.cnt = best_c;
    s.best = PER * ST - 1 - best;
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
  Hist<WIDE, BINS1> h1;
  Hist<WIDE, BINS> h2;
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

// A row of 16-bit elements between its first and last 16-byte borders, eight elements at a time: a thread's first HELD pieces stay in
// registers from the first pass to the second (64 of the 128 that a thread of 1024 has: rows of up to 131072 entries as a whole), what
// is longer is read again.
template <typename T> struct HeldRow {
  typedef unsigned Vec __attribute__((ext_vector_type(4)));
  static constexpr int HELD = 16;
  const T* row;
  int V, head, nvec;
  Vec held[HELD];
  __device__ __forceinline__ HeldRow(const T* row_, int V_) : row(row_), V(V_) {
    head = min(V, (int)(((16u - ((unsigned)(uintptr_t)row & 15u)) & 15u) / sizeof(T)));
    nvec = (V - head) / 8;
  }
  __device__ __forceinline__ const Vec* body() const { return reinterpret_cast<const Vec*>(row + head); }
  __device__ __forceinline__ void fetch() {
#pragma unroll
    for (int e = 0; e < HELD; ++e) {
      held[e] = Vec{0u, 0u, 0u, 0u};
      if (e * ST < nvec) {                         // (the same for all threads)
        const int i = e * ST + (int)threadIdx.x;
        if (i < nvec) held[e] = body()[i];
      }
    }
  }
  // f(the 16 bytes, their place, whether the thread has a piece at all) for every round, all threads of the block taking part; f comes
  // once a held round: a few instructions, or the code is larger than the instruction cache
  template <typename F> __device__ __forceinline__ void each(F&& f) const {
#pragma unroll
    for (int e = 0; e < HELD; ++e)
      if (e * ST < nvec) f(held[e], e * ST + (int)threadIdx.x, e * ST + (int)threadIdx.x < nvec);
    again(HELD * ST, f);
  }
  // the thread's piece of a held round, the same round for all lanes (a branch: picked by conditions it is 64 instructions)
  __device__ __forceinline__ Vec piece(int round) const {
    switch (round) {
#define OF(e) case e: return held[e];
      OF(0) OF(1) OF(2) OF(3) OF(4) OF(5) OF(6) OF(7) OF(8) OF(9) OF(10) OF(11) OF(12) OF(13) OF(14)
#undef OF
      default: return held[15];
    }
  }
  // the same as `each`, from memory, from the piece `from` on (a multiple of ST)
  template <typename F> __device__ __forceinline__ void again(int from, F&& f) const {
#pragma unroll 1
    for (int i0 = from; i0 < nvec; i0 += ST) {
      const int i = i0 + (int)threadIdx.x;
      Vec v{0u, 0u, 0u, 0u};
      if (i < nvec) v = body()[i];
      f(v, i, i < nvec);
    }
  }
  // g(element, its index) for those in front of the first border and behind the last
  template <typename G> __device__ __forceinline__ void ends(G&& g) const {
    const unsigned short* raw = reinterpret_cast<const unsigned short*>(row);
    const int rest = head + nvec * 8 + (int)threadIdx.x;
    const bool front = (int)threadIdx.x < head, back = rest < V;
    if (front) g((unsigned)raw[threadIdx.x], (int)threadIdx.x);
    if (back) g((unsigned)raw[rest], rest);
  }
};

// Rows of 16-bit logits: the same two questions (see sampling_row.inc), answered from how often each of the 65536 patterns
// occurs.  One pass over the row counts them (16 bits each, 128 KB of LDS); the ones that occur - a few thousand - are packed
// into a list in order, weighed once each, and summed up; what is kept and the pattern that the draw falls on follow from the
// list, with no further look at the row and no sort.  A second pass finds the element: the drawn pattern's elements come in
// the order of their indices, so each wave counts them in its 512 elements at a time, and the one stretch that the wanted one
// lies in is looked at again.  Masses are counts times weights, in doubles: no result depends on the order of additions.
// Bound by the first pass (15 us of 256 rows of 128256 at once, whose logits take 14 from memory; 10 of one row, LDS atomics) and by a
// dozen steps of a microsecond or two behind it.  256 rows of 128256 bf16 logits, every kind of filter among them: 31 us, one row
// 24, 32000 entries 17; with the row read again for the second pass (10 us for 2.5 from registers), the counts' sum as an atomic a
// lane (2 us) and the waves' totals added up by every wave 39, 29 and 18; by bins, as 32-bit rows are, 79, 36 and 18.  The patterns are
// packed by stretches of 512 places a wave: with 64 places a thread the few threads that have any were 7 us on their own.
// -1: a pattern occurs 65536 times or more (a count ran over: the counts' sum is then too small), more than 32768 patterns
// occur or more than 16384 of the likelier sign, or the row is longer than the second pass has counters for.  The type's lowest value and
// the infinity next to it, which masks fill rows with, are counted apart, in registers.
template <typename T>
__device__ __forceinline__ int sample_by_counts(const T* row, int V, float inv_t, unsigned k, float tp, float mp, float u, unsigned* tab,
                                SampleShared& s, CountShared& cs, Turn& turn) {
  using O = Order16<T>;
  typedef unsigned Vec __attribute__((ext_vector_type(4)));
  if (V > 1 << 23) return -1;
  const unsigned flip = inv_t < 0.f ? 0xffffffffu : 0u;
  const float to_exp2 = inv_t * 1.4426950408889634f;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
#pragma unroll
  for (int j = 0; j < PATTERNS / 2 / (4 * ST); ++j) *reinterpret_cast<Vec*>(tab + 4 * (j * ST + tid)) = Vec{0u, 0u, 0u, 0u};
  if (tid == 0) { s.bad = 0; cs.low = 0; cs.inf = 0; cs.counted = 0; }
  __syncthreads();                                 // (in front of the loads: a barrier waits for what is under way)
  HeldRow<T> data(row, V);
  data.fetch();
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
  auto largest = [&](Vec v) {
    const Pair16 most = __builtin_elementwise_max(
        __builtin_elementwise_max(pair16(v[0] & 0x7fff7fffu), pair16(v[1] & 0x7fff7fffu)),
        __builtin_elementwise_max(pair16(v[2] & 0x7fff7fffu), pair16(v[3] & 0x7fff7fffu)));
    return max((unsigned)most[0], (unsigned)most[1]);
  };
  // A piece with elements that are counted apart, or NaN, waits until the plain ones are through: here its round is noted, so that the code
  // for it is there once.  us, 256 rows of 128256 bf16: half masked at random 49, the last half 37, all but 64 39, nothing 36; read again
  // from memory and walked element by element 57, 46 and 49, with the code for both kinds in every round 54, 44 and 43 (nothing masked 44)
  unsigned apart_in = 0;
  data.each([&](Vec v, int i, bool live) {
    const bool plain = largest(v) < magnitude;
    if (live && plain) {
#pragma unroll
      for (int w = 0; w < 4; ++w) { count(v[w] & 0xffffu); count(v[w] >> 16); }
    }
    apart_in |= (__any(!plain) ? 1u : 0u) << min((unsigned)(i - tid) / ST, (unsigned)data.HELD);
  });
  auto apart = [&](Vec v) {
    const unsigned most = largest(v);
    if (most < magnitude) return;                  // (a lane without a piece has zeros)
    const Pair16 l = {1, 1};
    Pair16 not_low = {0, 0}, not_inf = {0, 0};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      not_low += __builtin_elementwise_min(pair16(v[w] ^ both16(lowest)), l);
      not_inf += __builtin_elementwise_min(pair16(v[w] ^ both16(lowest + 1)), l);
    }
    const unsigned lows = 8u - not_low[0] - not_low[1], infs = 8u - not_inf[0] - not_inf[1];
    low += lows;
    inf += infs;
    if (most > magnitude + 1) nan = 1;             // (whatever else is counted: the row has no distribution)
    if (lows + infs < 8u)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (((v[w] & 0xffffu) - lowest) > 1u) count(v[w] & 0xffffu);
        if (((v[w] >> 16) - lowest) > 1u) count(v[w] >> 16);
      }
  };
#pragma unroll 1
  for (unsigned rounds = apart_in & ((1u << data.HELD) - 1u); rounds; rounds &= rounds - 1u) apart(data.piece(__builtin_ctz(rounds)));
  if (apart_in >> data.HELD) data.again(data.HELD * ST, [&](Vec v, int, bool) { apart(v); });
  data.ends([&](unsigned x, int) { one(x); });
  if (__any((low | inf) != 0)) {                   // (one atomic a wave)
    low = (unsigned)wave_scan((int)low);
    inf = (unsigned)wave_scan((int)inf);
    if (lane == 63) { atomicAdd(&cs.low, low); atomicAdd(&cs.inf, inf); }
  }
  if (nan) s.bad = 1;
  __syncthreads();
  // ---- those that occur, in order, as (place, count) words in the counts' stead: 128 stretches of 512 places, eight a lane,
  // dealt to the waves in turn (values lie in a few octaves: most stretches are empty, and neighbours go to different waves).  In two
  // halves, whose counts lie in halves of the table: the first half's words take the place of its own counts
  unsigned n = 0, all_counts = 0;
  const unsigned list0 = flip ? PATTERNS / 4 : 0u;               // where the list begins
  auto word = [&](unsigned e) -> unsigned& { return tab[(list0 + e) & (PATTERNS / 2 - 1)]; };
#pragma unroll 1
  for (unsigned half = 0; half < 2; ++half) {
    constexpr int ROUNDS = PATTERNS / 16 / ST;
    const unsigned piece0 = half * (PATTERNS / 16) + tid;        // of the lane's first round
    const bool back = half == 0;                                 // (positive patterns lie backwards; flipped, the negative ones do)
    Vec v[ROUNDS];
    unsigned pos[ROUNDS], used = 0;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      const unsigned piece = j * ST + piece0, there = flip ? PATTERNS / 8 - 1 - piece : piece;
      v[j] = *reinterpret_cast<const Vec*>(tab + 4 * (there < PATTERNS / 16 ? PATTERNS / 16 - 1 - there : there));
      if (back) v[j] = Vec{v[j][3], v[j][2], v[j][1], v[j][0]};
    }
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      unsigned total = 0;
      if (__any((v[j][0] | v[j][1] | v[j][2] | v[j][3]) != 0)) {
        used |= 1u << j;
        unsigned c = 0, sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (back) v[j][w] = v[j][w] >> 16 | v[j][w] << 16;
          const unsigned lo = v[j][w] & 0xffffu, hi = v[j][w] >> 16;
          c += (lo != 0) + (hi != 0);
          sum += lo + hi;
        }
        all_counts += sum;
        unsigned before = 0;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) {
          const unsigned long long have = __ballot(c >> bit & 1u);
          before += (unsigned)__popcll(have & ((1ull << lane) - 1ull)) << bit;
          total += (unsigned)__popcll(have) << bit;
        }
        pos[j] = before;
      }
      if (lane == 0) cs.of_stretch[half * 64 + j * (ST / 64) + wid] = total;
    }
    if (half == 1) {                               // (one atomic a wave: 64 lanes' on one word are a loop of their own)
      const unsigned wave_counts = (unsigned)wave_scan((int)all_counts);
      if (lane == 63) atomicAdd(&cs.counted, wave_counts);
    }
    __syncthreads();
    const unsigned mine = cs.of_stretch[half * 64 + lane];
    const unsigned upto = (unsigned)wave_scan((int)mine);
    const unsigned before = n;
    n += __shfl(upto, 63, 64);
    if (half == 0 && n > PATTERNS / 4) return -1;
    if (half == 1 && ((cs.counted != (unsigned)V - cs.low - cs.inf && !s.bad) || n > PATTERNS / 2)) return -1;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      if (!(used >> j & 1u)) continue;
      const int stretch = j * (ST / 64) + wid;
      unsigned at = before + pos[j] + __shfl(upto - mine, stretch, 64);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const unsigned d = 8u * (j * ST + piece0) + 2u * w;
        if (v[j][w] & 0xffffu) word(at++) = d << 16 | (v[j][w] & 0xffffu);
        if (v[j][w] >> 16) word(at++) = (d + 1u) << 16 | v[j][w] >> 16;
      }
    }
    // (the first half's words lie where only its own counts were, which nobody reads any more)
    if (half == 1) __syncthreads();
  }
  const unsigned lows = cs.low;
  // the row's largest entry (its place: the one in front of all); NaN, and an infinity there, are no distribution
  const unsigned first = n ? word(0) >> 16 : (lows ? O::LOWEST : O::LOWEST + 1);
  const float top = O::value(first, flip);
  auto weight = [&](unsigned d) { return __float_as_uint(fast_exp2((O::value(d, flip) - top) * to_exp2)); };
  if (s.bad || first <= O::FIRST || (cs.inf && weight(O::LOWEST + 1) >= NORMAL_END)) return 0;
  // ---- entry n is the type's lowest value; a thread has `per` of them in a row
  const unsigned per = (n + 1 + ST - 1) / ST, e0 = min(per * tid, n + 1), e1 = min(e0 + per, n + 1);
  auto entry = [&](unsigned e, unsigned& d, unsigned& c) {
    const unsigned x = e < n ? word(e) : 0u;
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
  block_scan(cnt, m, ec, em, z, s, turn);
  if (s.bad) return 0;
  unsigned kept = (unsigned)V, rank = 0;
  int found = -1;
  double mass = z;
  for (int step = 0; step < 2; ++step) {
    const unsigned minb = step == 0 && mp > 0.f ? __float_as_uint(fminf(mp, 1.f)) : 0u;
    if (step == 0 && k >= (unsigned)V && tp >= 1.f && minb == 0u) continue;      // everything is kept
    const double M = step == 0 ? (tp >= 1.f ? 1e300 : fmax((double)tp * z, 1e-300)) : fmax((double)u * mass, 1e-300);
    const unsigned K = step == 0 ? k : kept;
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
    found = block_last(best, s, turn);
    if (found < 0) return 0;                       // (no weights at all)
    if (found == best) {
      const double v = mass_of(best_w);
      const double fit = fmin(fmax(ceil((M - best_above) / v), 1.0), (double)best_c);
      const unsigned take = min((unsigned)fit, K - best_front);
      s.above_cnt = best_front + take;
      s.mass = best_above + take * v;
      s.cnt = best_w;
      s.n = (int)take;
    }
    __syncthreads();
    kept = s.above_cnt;
    mass = s.mass;
    rank = (unsigned)s.n;
  }
  // ---- the rank-th element (from 1) of the patterns that weigh as much: those beside the found one count in front of it
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
  const int head = data.head, nvec = data.nvec, parts = (nvec + 63) / 64;
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
    data.each([&](Vec v, int i, bool live) {
      Pair16 x[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) x[w] = pair16(v[w] ^ drawn);
      const Pair16 least = __builtin_elementwise_min(__builtin_elementwise_min(x[0], x[1]), __builtin_elementwise_min(x[2], x[3]));
      unsigned sum = 0;
      if (__any(live && (least[0] == 0 || least[1] == 0))) {     // (512 elements seldom have one)
        const Pair16 l = {1, 1};
        Pair16 others = {0, 0};
#pragma unroll
        for (int w = 0; w < 4; ++w) others += __builtin_elementwise_min(x[w], l);
        const unsigned c = live ? 8u - others[0] - others[1] : 0u;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) sum += (unsigned)__popcll(__ballot(c >> bit & 1u)) << bit;
      }
      if (lane == 0 && live) tab[1 + (i >> 6)] = sum;
    });
  else
    data.again(0, [&](Vec v, int i, bool live) {
      unsigned c = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) c += hit(v[w] & 0xffffu) + hit(v[w] >> 16);
      hits_of(live ? c : 0u, i, live);
    });
  data.ends(single);
  __syncthreads();
  // ---- the stretch that the wanted one lies in
  const unsigned each = (parts + 2 + ST - 1) / ST;
  unsigned mine = 0, before;
  for (unsigned e = 0; e < each; ++e) {
    const int i = (int)(each * tid + e);
    if (i < parts + 2) mine += tab[i];
  }
  double none, all;
  block_scan(mine, 0.0, before, none, all, s, turn);
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
  __shared__ Hist<WIDE, BINS1> h1;
  __shared__ Hist<WIDE, BINS> h2;
  __shared__ unsigned long long list[CAP];
  __shared__ SampleShared s;
  __shared__ float red[16];
  __shared__ int s_idx;
  static_assert(sizeof(T) == 4, "");
  unsigned* const tab = nullptr;
  CountShared cs;
  Turn turn = 0;
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
  auto &h1 = sh.bins.h1;
  auto& h2 = sh.bins.h2;
  unsigned long long* const list = sh.bins.list;
  unsigned* const tab = sh.counts;
  Turn turn = 0;
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
