// Merge of the KV splits of one attention row: out = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M).
//
// part_o[split][D] and part_ml[split][2] = (m, l) belong to one (token, head).  The weights are made once, a lane per split;
// then the workgroup's threads form as many groups as there are rows of D / 4 of them, each group adds up every n-th split
// with four 16-byte loads in flight, and the groups' sums meet in LDS.  Bound by memory latency, not by bytes: one thread per
// column that walks the splits in turn, with the weight's load and exponential between two adds, takes ~1 us per split
// (latent attention of one sequence, 16 heads x 512 values, 64 splits, merge included: 80 us with it, 21 like this).
#pragma once
#include "common.h"

constexpr int SPLIT_MERGE_MAX_SPLITS = 64;      // a lane of one wave holds a split's weight
constexpr int SPLIT_MERGE_MAX_THREADS = 512;

// Threads for this many splits: whole rows of D / 4 threads, no more rows than splits.
inline int split_merge_threads(int D, int num_splits) {
  const int row = D / 4;
  int groups = SPLIT_MERGE_MAX_THREADS / row;
  if (groups > num_splits) groups = num_splits;
  return (groups * row + 63) / 64 * 64;
}

// Threads below D / 4 return true with the weighted sum of columns 4 threadIdx.x .. + 3 in `o`, and the sum of the
// denominators in `denom`; exp(*sink) (null: none) joins the denominator.  `neg` is below every m, or that of an empty split.
template <int D>
__device__ __forceinline__ bool split_merge(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                            int num_splits, const float* __restrict__ sink, float neg, f32x4& o, float& denom) {
  typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int ROW = D / 4;
  static_assert(D % 4 == 0 && ROW <= SPLIT_MERGE_MAX_THREADS, "unsupported width");
  __shared__ float s_w[SPLIT_MERGE_MAX_SPLITS];
  __shared__ float s_denom;
  __shared__ f32x4 s_sum[SPLIT_MERGE_MAX_THREADS];
  const int tid = threadIdx.x, grp = tid / ROW, col = tid - grp * ROW;
  const int groups = min((int)blockDim.x / ROW, num_splits);
  if (tid < 64) {
    float m = neg, l = 0.f;
    if (tid < num_splits) { m = part_ml[2 * tid]; l = part_ml[2 * tid + 1]; }
    float mm = m;
#pragma unroll
    for (int off = 32; off; off >>= 1) mm = fmaxf(mm, __shfl_xor(mm, off, 64));
    const float w = tid < num_splits ? fast_exp2(m - mm) : 0.f;
    float sum = l * w;
#pragma unroll
    for (int off = 32; off; off >>= 1) sum += __shfl_xor(sum, off, 64);
    s_w[tid] = w;
    if (tid == 0) s_denom = sum + (sink != nullptr ? fast_exp2(*sink * 1.4426950408889634f - mm) : 0.f);
  }
  f32x4 a = {0.f, 0.f, 0.f, 0.f};
  f32x4 v[4];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = *reinterpret_cast<const f32x4_any*>(part_o + (long)min(s0 + i * groups, num_splits - 1) * D + 4 * col);
  };
  const bool live = grp < groups;
  if (live) fetch(grp);                         // (on its way while the weights are made)
  __syncthreads();
  if (live) {
    for (int s0 = grp; s0 < num_splits; s0 += 4 * groups) {
      if (s0 != grp) fetch(s0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + i * groups < num_splits) a += v[i] * s_w[s0 + i * groups];
    }
    s_sum[tid] = a;
  }
  __syncthreads();
  if (tid >= ROW) return false;
  for (int g = 1; g < groups; ++g) a += s_sum[g * ROW + tid];
  o = a;
  denom = s_denom;
  return true;
}
