// Token sampling: greedy argmax and temperature / top-k / top-p / min-p
// inverse-CDF sampling, one 1024-thread workgroup per logits row.
//
// Semantics match ops/torch_ref.py::sample (descending order, ties by index);
// the thresholds and the draw are found without sorting the row, see sample_kernel.
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

struct SampleShared {
  double wmass[16];
  unsigned wcnt[16];
  double mass, above_mass;
  unsigned above_cnt, cnt, n_list;
  int best, n, token, bad;
};

// exclusive scan of (count, mass) over the block in thread order; totals to every thread
__device__ __forceinline__ void block_scan(unsigned c, double m, unsigned& ec, double& em, double& total, SampleShared& s) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  unsigned ic = c;
  double im = m;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned oc = __shfl_up(ic, o, 64);
    const double om = __shfl_up(im, o, 64);
    if (lane >= o) { ic += oc; im += om; }
  }
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

// The lowest non-empty bin (at or above `first`) in front of which fewer than K elements and less than M of mass lie:
// its index, count and what lies above it go to `s` (best = -1: none).  Bins hold the bits `prefix | bin << shift ..`.
template <bool WIDE>
__device__ void scan_bins(const Hist<WIDE>& h, unsigned prefix, int shift, int first, unsigned above_cnt, double above_mass,
                          unsigned K, double M, SampleShared& s) {
  unsigned c[2];
  double m[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int bin = BINS - 1 - (2 * (int)threadIdx.x + e);
    const unsigned bits = prefix | ((unsigned)bin << shift);
    c[e] = h.count(bin);
    m[e] = c[e] ? ((double)c[e] * sig_of(bits) + (double)h.lows(bin)) * pow2(lsb_of(bits)) : 0.0;
  }
  unsigned ec;
  double em, total;
  if (threadIdx.x == 0) s.best = -1;
  block_scan(c[0] + c[1], m[0] + m[1], ec, em, total, s);
  ec += above_cnt;
  em += above_mass;
  int mine = -1;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int order = 2 * (int)threadIdx.x + e;
    if (c[e] && BINS - 1 - order >= first && ec + (e ? c[0] : 0) < K && em + (e ? m[0] : 0.0) < M) mine = order;
  }
  if (mine >= 0) atomicMax(&s.best, mine);
  __syncthreads();
  const int best = s.best;
  __syncthreads();
  if (best >= 0 && best >> 1 == (int)threadIdx.x) {
    const bool second = best & 1;
    s.above_cnt = ec + (second ? c[0] : 0);
    s.above_mass = em + (second ? m[0] : 0.0);
    s.cnt = second ? c[1] : c[0];
    s.best = BINS - 1 - best;
  }
  if (threadIdx.x == 0) s.mass = total;
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

// One workgroup per row.  With weights e = exp((logit - max) / T) in descending order (ties by index) an entry is kept
// while fewer than K lie in front of it, less than M of mass lies in front of it, and it is at least min_p; the sampled
// entry is the last one in front of which less than `u * kept mass` lies: the same question, asked twice.
// It is answered without sorting the row: one pass for the maximum, one that counts the weights into 2048 bins by
// their leading bits (exponent and four bits more), a scan over the bins that finds the bin the answer lies in, and a
// pass that lists that bin's entries (a thousand of a Gaussian row of 128k) in LDS, where they are sorted and summed up.
// A bin of more than 4096 entries is cut by the next bits first, and one of equal weights is walked by index.
// Masses are whole multiples of a bin's last bit, added up in 64-bit integers and doubles: no result depends on the
// order of additions.
// A row is read three or four times; a bisection over the bits of both thresholds reads it up to 70 times (256 rows of
// 128256 bf16 logits, every kind of filter among them: 112 - 117 us here, 5.2 - 6.1 ms so; one pass over them at the rate
// of a large copy: 14 us).  What is left is the LDS atomics of the counting pass (25 us), two sorts of about a thousand entries
// (10 us each) and the scans.  One row takes 46 - 80 us: it is one compute unit's work.
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
  const int b = blockIdx.x;
  const T* row = logits + b * stride;
  const float temp = temperature[b];
  // ---- greedy row: plain argmax (lowest index on ties)
  if (temp == 0.f) {
    ArgMax best{-INFINITY, 0x7fffffff};
    for_row(row, V, [&](float v, int i) {
      if (v > best.v || (v == best.v && i < best.i)) best = ArgMax{v, i};
    });
    const float mx = block_max(best.v, red);
    const int cand = (best.v == mx) ? best.i : 0x7fffffff;
    if (threadIdx.x == 0) s_idx = 0x7fffffff;
    __syncthreads();
    atomicMin(&s_idx, cand);
    __syncthreads();
    if (threadIdx.x == 0) out[b] = s_idx == 0x7fffffff ? 0 : s_idx;
    return;
  }
  const float inv_t = 1.f / temp;
  unsigned k = top_k[b] <= 0 || top_k[b] > V ? (unsigned)V : (unsigned)top_k[b];
  const float tp = top_p[b], mp = min_p[b], u = uniform[b];
  h1.clear();
  if (threadIdx.x == 0) s.bad = 0;
  const float sign = inv_t < 0.f ? -1.f : 1.f, to_exp2 = inv_t * 1.4426950408889634f;
  float mx = -INFINITY;
  for_row(row, V, [&](float v, int) { mx = fmaxf(mx, v * sign); });
  const float top = sign * block_max(mx, red);
  // (the difference first: the largest entry weighs exactly 1, and every pass sees the same bits)
  auto weight = [&](float v) { return __float_as_uint(fast_exp2((v - top) * to_exp2)); };
  int bad = 0;
  for_row(row, V, [&](float v, int) {
    const unsigned w = weight(v);
    if (w >= NORMAL_END) bad = 1;                  // (NaN, or a row of infinities)
    else if (w) h1.add(w >> 19, w & 0x7ffffu);     // (a weight of zero is never sampled and adds nothing)
  });
  if (bad) s.bad = 1;
  __syncthreads();
  if (s.bad) { if (threadIdx.x == 0) out[b] = 0; return; }

  unsigned kept = (unsigned)V;
  double mass = 0;
  int listed = -1;                                 // the bin whose entries the list holds
  int token = 0;
  // step 0: how much is kept; step 1: the entry drawn from it
  for (int step = 0; step < 2; ++step) {
    const unsigned minb = step == 0 && mp > 0.f ? __float_as_uint(fminf(mp, 1.f)) : 0u;
    double M;
    if (step == 0) {
      scan_bins<WIDE>(h1, 0u, 19, 0, 0u, 0.0, 1u, 1.0, s);           // (its total is the mass of the row)
      const double z = s.mass;
      mass = z;
      if (k >= (unsigned)V && tp >= 1.f && minb == 0u) continue;     // everything is kept
      M = tp >= 1.f ? 1e300 : fmax((double)tp * z, 1e-300);          // (the first entry always is)
    } else {
      M = fmax((double)u * mass, 1e-300);
    }
    const unsigned K = step == 0 ? k : kept;
    unsigned prefix = 0u;
    int shift = 19;
    scan_bins<WIDE>(h1, 0u, 19, (int)(minb >> 19), 0u, 0.0, K, M, s);
    if (s.best < 0) break;                         // (no weights at all)
    const int bin1 = s.best;
    prefix = (unsigned)bin1 << 19;
    bool some = true;
    while (some && s.cnt > CAP && shift > 0) {
      const int next = shift == 19 ? 8 : 0;
      const unsigned above_cnt = s.above_cnt;
      const double above_mass = s.above_mass;
      h2.clear();
      __syncthreads();
      for_row(row, V, [&](float v, int) {
        const unsigned w = weight(v);
        if (w < NORMAL_END && w >> shift == prefix >> shift && w && w >= minb)
          h2.add((w >> next) & ((1u << (shift - next)) - 1u), w & ((1u << next) - 1u));
      });
      __syncthreads();
      scan_bins<WIDE>(h2, prefix, next, 0, above_cnt, above_mass, K, M, s);
      some = s.best >= 0;
      if (some) prefix |= (unsigned)s.best << next;
      else if (threadIdx.x == 0) { s.above_cnt = above_cnt; s.above_mass = above_mass; }
      shift = next;
      __syncthreads();
    }
    const unsigned above_cnt = s.above_cnt;
    const double above_mass = s.above_mass;
    const int cnt = some ? (int)s.cnt : 0;
    if (cnt > CAP) {
      // entries of one and the same weight, in index order
      const double v = sig_of(prefix) * pow2(lsb_of(prefix));
      const double fit = ceil((M - above_mass) / v);
      int n = (int)fmin(fmin((double)cnt, (double)(K - above_cnt)), fmax(fit, 1.0));
      if (step == 0) { kept = above_cnt + n; mass = above_mass + n * v; continue; }
      int seen = 0;                                // in front of this stretch of the row
      for (int base = 0; base < V; base += ST) {
        const int i = base + threadIdx.x;
        const bool hit = i < V && weight(to_f(row[i])) == prefix;
        unsigned ec;
        double em, total;
        block_scan(hit ? 1u : 0u, hit ? 1.0 : 0.0, ec, em, total, s);
        if (hit && seen + (int)ec == n - 1) s.token = i;
        seen += (int)total;
        if (seen >= n) break;
      }
      __syncthreads();
      token = s.token;
      break;
    }
    if (listed != bin1) {
      listed = shift == 19 ? bin1 : -1;
      if (threadIdx.x == 0) s.n_list = 0;
      __syncthreads();
      if (cnt > 0)
        for_row(row, V, [&](float v, int i) {
          const unsigned w = weight(v);
          if (w < NORMAL_END && w >> shift == prefix >> shift && w && w >= minb) {
            const unsigned pos = atomicAdd(&s.n_list, 1u);
            if (pos < CAP) list[pos] = ((unsigned long long)w << 32) | (0xffffffffu - (unsigned)i);
          }
        });
      __syncthreads();
      sort_list(list, min((int)s.n_list, CAP));
    }
    const int n_list = min((int)s.n_list, CAP);
    // four entries per thread, summed up in order: how many are in front of the border
    unsigned w4[4];
    double m4 = 0;
    const int at = 4 * (int)threadIdx.x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w4[e] = at + e < n_list ? (unsigned)(list[at + e] >> 32) : 0u;
      m4 += sig_of(w4[e]) * pow2(lsb_of(w4[e]));
    }
    unsigned ec;
    double em, total;
    block_scan(0u, m4, ec, em, total, s);
    if (threadIdx.x == 0) { s.n = 0; s.mass = above_mass; }
    __syncthreads();
    double front = above_mass + em, upto = front;
    int n = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (at + e < n_list && above_cnt + at + e < K && front < M) {
        n = at + e + 1;
        front += sig_of(w4[e]) * pow2(lsb_of(w4[e]));
        upto = front;
      } else {
        front = 1e301;
      }
    }
    if (n) atomicMax(&s.n, n);
    __syncthreads();
    if (n && s.n == n) {
      s.mass = upto;
      s.token = (int)(0xffffffffu - (unsigned)list[n - 1]);
    }
    __syncthreads();
    if (step == 0) { kept = above_cnt + s.n; mass = s.mass; }
    else if (s.n) token = s.token;
    __syncthreads();
  }
  if (threadIdx.x == 0) out[b] = token;
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
#define L(TY)                                                                                                       \
  do {                                                                                                              \
    if (V <= (1 << 22))                                                                                             \
      hipLaunchKernelGGL((sample_kernel<TY, false>), dim3(B), dim3(ST), 0, s, out, (const TY*)logits, V, stride,    \
                         temperature, top_k, top_p, min_p, uniform);                                                \
    else                                                                                                            \
      hipLaunchKernelGGL((sample_kernel<TY, true>), dim3(B), dim3(ST), 0, s, out, (const TY*)logits, V, stride,     \
                         temperature, top_k, top_p, min_p, uniform);                                                \
  } while (0)
  if (dtype == DT_BF16) L(bf16_t);
  else if (dtype == DT_F16) L(f16_t);
  else if (dtype == DT_F32) L(float);
  else return -2;
#undef L
  HIP_LAUNCH_CHECK();
  return 0;
}
