// Multi-head latent attention (DeepSeek-V2 / V3) over a LATENT paged cache, gfx950.
//
// With the up-projections absorbed into the query and the output (q_lat = q_nope . W_UK, out = o_lat . W_UV^T),
// every query head of a token attends over ONE shared key per position,
//     key   = [ RMSNorm(c_kv) (RANK values) | rotated k_rope (ROPE values) ]      DK = RANK + ROPE
//     value =   RMSNorm(c_kv)                                                      DV = RANK
// so the cache holds DK + DV values per token and layer instead of heads x (DK' + DV') expanded ones
// (DeepSeek-V3: 1088 against 49152).  The two forms of the latent are stored in the layouts the other
// attention kernels use, which make them direct MFMA operands from global memory:
//     k_cache[num_blocks][block_size][DK]                    key rows
//     v_cache[num_blocks][DV/16][block_size/8][16][8]        V^T in fragment order
//
// One workgroup = one token's tile of 16 query heads (x one KV split).  What makes this shape different from
// grouped-query attention is the width: a wave that held all of Q (DK/32 fragments), all of a 32-key K group
// and the whole O^T accumulator (DV/16 tiles) would need ~500 registers.  The four waves of a workgroup split
// BOTH reductions instead:
//   * wave w multiplies its quarter of the DK dimension (Q and K fragments of its k-steps only) and leaves a
//     partial S^T tile pair in LDS; after one barrier every wave adds the four partials - 8 floats per lane,
//     same lane in every wave, conflict-free - and all four run the identical online softmax on the sum;
//   * wave w owns DV/4 columns of the output: its V^T fragments and accumulators are a quarter as well.
// No byte of the cache is read twice by a workgroup, 2 waves per SIMD fit (<= 256 registers), and the exchange
// (2 KiB per group, double-buffered so one barrier per 32 keys suffices) is small next to the 70 KB of cache a
// group streams.  The next group's fragments are requested before the current group is multiplied.
//
// Rows are tokens, not sequences: a prefill chunk, a decode batch and a speculative verification are the same
// launch with `token_seq[t]` naming the block-table row and `seq_lens[t]` = position + 1 the causal limit of
// token t.  (A long prompt therefore streams its keys once per query token - from L2 for the most part, since
// neighbouring tokens run side by side; the expanded-cache prefill kernel reads them once per 128 tokens.)
//
// FlashMLA / vLLM's MLA backends are the CUDA counterparts; the reference framework reaches them through the
// vLLM image it runs (/root/reference/Dockerfile:1).
#include "common.h"
#include "split_merge.h"

namespace {

constexpr float MLA_NEG_BIG = -1.0e30f;
constexpr int MLA_MAX_SPLITS = 64;

// An e4m3 cache (one byte per value, same layouts, scale 1: the normalised latent and the rotated key part are
// O(1) numbers) halves the bytes a decode step streams; fragments are widened in registers on their way in.
template <typename T>
__device__ __forceinline__ typename Vec8<T>::type mla_fp8x8_to(uint2 w) {
  union { uint32_t u[4]; typename Vec8<T>::type v; } r;
  if constexpr (__is_same(T, bf16_t)) {
    r.u[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.f, false));
    r.u[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.f, true));
    r.u[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.f, false));
    r.u[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.f, true));
  } else {
    r.u[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w.x, 1.f, false));
    r.u[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w.x, 1.f, true));
    r.u[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w.y, 1.f, false));
    r.u[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w.y, 1.f, true));
  }
  // (two wait states behind the packed converts: their results are not safe to read earlier, and the
  // compiler's hazard table does not know it - see fp8x8_to in attention.hip)
  asm volatile("s_nop 1" : "+v"(r.u[0]), "+v"(r.u[1]), "+v"(r.u[2]), "+v"(r.u[3]));
  return r.v;
}

// 8 consecutive cache values from element offset `off`, as they are loaded (e4m3: 8 bytes, widened only where
// they are used - a fragment requested one key group ahead must not be waited for at the request)
template <typename T, bool KV8> struct MlaRaw { using type = typename Vec8<T>::type; };
template <typename T> struct MlaRaw<T, true> { using type = uint2; };

template <typename T, bool KV8>
__device__ __forceinline__ typename MlaRaw<T, KV8>::type mla_ld(const void* cache, long off) {
  if constexpr (KV8) {
    return *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(cache) + off);
  } else {
    return ld8<T>(reinterpret_cast<const T*>(cache) + off);
  }
}

template <typename T, bool KV8>
__device__ __forceinline__ typename Vec8<T>::type mla_widen(typename MlaRaw<T, KV8>::type raw) {
  if constexpr (KV8) {
    return mla_fp8x8_to<T>(raw);
  } else {
    return raw;
  }
}

// one value into the cache at element offset `off`
template <typename T, bool KV8>
__device__ __forceinline__ void mla_st(void* cache, long off, float v) {
  if constexpr (KV8) {
    const float c = fminf(fmaxf(v, -448.f), 448.f);
    reinterpret_cast<uint8_t*>(cache)[off] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(c, 0.f, 0, false) & 0xff);
  } else {
    reinterpret_cast<T*>(cache)[off] = (T)v;
  }
}

// What a layer may add to plain causal attention: a sliding window (a token sees its last `window` keys; 0 = all), a
// learned sink per head whose exponential joins the softmax denominator, a sigmoid gate per (token, head) on the output.
struct MlaExtra {
  int window;
  const float* sinks;                // [Hq] or null
  const void* gate; long gate_stride;  // [T, gate_stride] raw values of the element type, or null
  float past_bytes;                  // mla_rows_kernel: read past the caches what is this much and one row's alone (0: nothing)
};

// l (relative to the running maximum m, log2 scale) and the factor the accumulators take when the sink joins
__device__ __forceinline__ void mla_add_sink(float sink_log2, float m, float& l, float& factor) {
  const float m_f = fmaxf(m, sink_log2);
  factor = fast_exp2(m - m_f);
  l = l * factor + fast_exp2(sink_log2 - m_f);
}

// P2: the fp32 softmax weights enter the PV product as a high and a low 16-bit part (two MFMAs per tile, ~16
// mantissa bits) instead of being rounded to 8 bits: for models that define their attention weights in 32-bit.
template <typename T, int DK, int DV, bool KV8, bool P2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void mla_attention_kernel(
    T* __restrict__ out, long out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    const T* __restrict__ q, long q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_table, int bt_stride, const int* __restrict__ token_seq,
    const int* __restrict__ seq_lens, float scale_log2e, int Hq, int block_size, int num_splits, MlaExtra ex) {
  using V = typename Vec8<T>::type;
  constexpr int KSTEPS = DK / 32;              // 32-wide steps of the QK^T reduction
  constexpr int KS = (KSTEPS + 3) / 4;         // ... per wave (the last waves may run short: zero Q there)
  constexpr int VT = DV / 64;                  // 16-row tiles of O^T per wave
  static_assert(DK % 32 == 0 && DV % 64 == 0, "unsupported latent width");
  __shared__ float s_part[2][4][64][8];

  const int split = blockIdx.x, qt = blockIdx.y, t = blockIdx.z;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int qh0 = qt * 16;
  const int nq = min(16, Hq - qh0);
  const int seq_len = seq_lens[t];
  const int* bt_row = block_table + (long)(token_seq != nullptr ? token_seq[t] : t) * bt_stride;

  // keys [win_lo, seq_len): nothing in front of win_lo is read (its pages may have gone back to the pool)
  const int win_lo = ex.window > 0 ? max(seq_len - ex.window, 0) : 0;
  const int g_lo = win_lo >> 5;
  const int n_groups = ((seq_len + 31) >> 5) - g_lo;
  const int gps = (n_groups + num_splits - 1) / num_splits;
  const int g_begin = g_lo + split * gps;
  const int g_end = min(g_begin + gps, g_lo + n_groups);

  // this wave's k-steps: global step wid * KS + s, clamped for the address and zeroed in Q when past the end
  V qf[KS];
  int kstep_off[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int sg = wid * KS + s;
    kstep_off[s] = 32 * min(sg, KSTEPS - 1) + 8 * g4;
    V z;
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] = (T)0.f;
    qf[s] = (sg < KSTEPS && r16 < nq) ? ld8<T>(q + t * q_stride + (long)(qh0 + r16) * DK + kstep_off[s]) : z;
  }
  f32x4 acc[VT];
#pragma unroll
  for (int i = 0; i < VT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = MLA_NEG_BIG, l = 0.f;

  const int slab = block_size * 16;            // elements of one 16-row slab of a V^T block
  using R = typename MlaRaw<T, KV8>::type;
  struct Frag { R ka[KS], kb[KS], vf[VT]; };
  auto load = [&](Frag& f, int g) {
    const int base = g * 32;
    // K rows of the two interleaved S^T tiles: tile 0 row i <-> key 8 (i >> 2) + (i & 3), tile 1 the same + 4
    const int key0 = base + 8 * (r16 >> 2) + (r16 & 3);
    const int ka = max(min(key0, seq_len - 1), win_lo), kb = max(min(key0 + 4, seq_len - 1), win_lo);
    const long ra = ((long)bt_row[ka / block_size] * block_size + (ka % block_size)) * DK;
    const long rb = ((long)bt_row[kb / block_size] * block_size + (kb % block_size)) * DK;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      f.ka[s] = mla_ld<T, KV8>(k_cache, ra + kstep_off[s]);
      f.kb[s] = mla_ld<T, KV8>(k_cache, rb + kstep_off[s]);
    }
    // V^T: this lane's 8 keys are base + 8 g4 .. + 7 (inside one block: block_size % 8 == 0)
    const int vkey = max(min(base + 8 * g4, seq_len - 1), win_lo) & ~7;
    const long vo = (long)bt_row[vkey / block_size] * (DV / 16) * slab + ((vkey % block_size) >> 3) * 128 + 8 * r16;
#pragma unroll
    for (int i = 0; i < VT; ++i) f.vf[i] = mla_ld<T, KV8>(v_cache, vo + (long)(wid * VT + i) * slab);
  };

  Frag cur, nxt;
  if (g_begin < g_end) load(cur, g_begin);
  for (int g = g_begin; g < g_end; ++g) {
    load(nxt, min(g + 1, g_end - 1));          // (past the end: the last group again, never used)
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      s0 = mfma16(mla_widen<T, KV8>(cur.ka[s]), qf[s], s0);
      s1 = mfma16(mla_widen<T, KV8>(cur.kb[s]), qf[s], s1);
    }
    float* mine = &s_part[g & 1][wid][lane][0];
    *reinterpret_cast<f32x4*>(mine) = s0;
    *reinterpret_cast<f32x4*>(mine + 4) = s1;
    __syncthreads();
    // (every wave adds the four partials in the same order, its own included: the softmax state that follows is
    // then bit-identical in all four, which the split-KV merge relies on - only wave 0 reports m and l)
    s0 = *reinterpret_cast<const f32x4*>(&s_part[g & 1][0][lane][0]);
    s1 = *reinterpret_cast<const f32x4*>(&s_part[g & 1][0][lane][4]);
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      s0 += *reinterpret_cast<const f32x4*>(&s_part[g & 1][w][lane][0]);
      s1 += *reinterpret_cast<const f32x4*>(&s_part[g & 1][w][lane][4]);
    }
    // online softmax; key index of element j is base + 8 g4 + j
    const int kidx0 = g * 32 + 8 * g4;
    float p[8];
    float tmax = MLA_NEG_BIG;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float sv = (j < 4 ? s0[j & 3] : s1[j & 3]) * scale_log2e;
      p[j] = (kidx0 + j < seq_len && kidx0 + j >= win_lo) ? sv : MLA_NEG_BIG;
      tmax = fmaxf(tmax, p[j]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m, tmax);
    const float alpha = fast_exp2(m - m_new);
    float psum = 0.f;
    V pf;
    [[maybe_unused]] V pl;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = p[j] <= 0.5f * MLA_NEG_BIG ? 0.f : fast_exp2(p[j] - m_new);
      psum += e;
      pf[j] = (T)e;
      if constexpr (P2) pl[j] = (T)(e - (float)pf[j]);
    }
    l = l * alpha + psum;
    m = m_new;
#pragma unroll
    for (int i = 0; i < VT; ++i) {
      acc[i] *= alpha;
      const V vfrag = mla_widen<T, KV8>(cur.vf[i]);
      acc[i] = mfma16(vfrag, pf, acc[i]);
      if constexpr (P2) acc[i] = mfma16(vfrag, pl, acc[i]);
    }
    cur = nxt;
  }

  float lsum = l;
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (r16 >= nq) return;
  const int qh = qh0 + r16;
  if (num_splits == 1) {
    float factor = 1.f;
    if (ex.sinks != nullptr) mla_add_sink(ex.sinks[qh] * 1.4426950408889634f, m, lsum, factor);
    float inv = lsum > 0.f ? factor / lsum : 0.f;
    if (ex.gate != nullptr) inv *= 1.f / (1.f + __expf(-(float)((const T*)ex.gate)[t * ex.gate_stride + qh]));
    T* orow = out + t * out_stride + (long)qh * DV + 4 * g4;
#pragma unroll
    for (int i = 0; i < VT; ++i) {
      typename Vec4<T>::type o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (T)(acc[i][r] * inv);
      *reinterpret_cast<typename Vec4<T>::type*>(orow + 16 * (wid * VT + i)) = o;
    }
  } else {
    const long pidx = ((long)t * Hq + qh) * num_splits + split;
#pragma unroll
    for (int i = 0; i < VT; ++i)
      *reinterpret_cast<f32x4*>(part_o + pidx * DV + 16 * (wid * VT + i) + 4 * g4) = acc[i];
    if (wid == 0 && g4 == 0) { part_ml[2 * pidx] = m; part_ml[2 * pidx + 1] = lsum; }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Rows of any kind (decoded, of prompts, verified) by 16 heads a workgroup, reading the key rows alone: a row's first DV values ARE
// its value, so the V^T cache need not be read for them.  32 keys at a time go global -> LDS by DMA (one run of 32 * DK values: a group of
// keys never crosses a block here), the next group's while the current one is multiplied, two workgroups per CU.
//   * QK: as above, a wave per quarter of the reduction; K fragments are read from LDS by rows.
//   * PV: a lane reads 4 neighbouring values of each of its 8 keys (8 bytes each) and turns them by byte permutes into V^T
//     fragments of four tiles whose row i is value 4 i + tile of the wave's 64: a permutation of the output's columns that
//     leaves a lane with 16 neighbouring ones of them.
// The 16-byte pieces of a row are XOR-ed with bits 1, 3 and 4 of the key's number (the 16 rows of a K fragment then lie in
// 16 different places of the LDS's 256 bytes).
// Bound by reading the rows: 128 sequences of about 3100 keys, 16 heads, write of the new rows included: 99 us against 211
// through both caches (441 and 833 MB).  ONCE: what one sequence alone reads comes past the caches (nontemporal) where the
// sequences' rows are more than the memory-side cache holds.  Several caches in turn, us, cached / past them / asking first: 128
// sequences of 3100 keys 112 / 104 / 103, 16 of 12000 68 / 61 / 62; with 90 % of the pages shared 60 of 3000 44.9 / 46.2 / 45.5,
// 16 of 3000 (which the cache holds) 21.9 / 24.0 / 22.3.
// ---------------------------------------------------------------------------------------------------------------
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void mla_lds_void;
typedef __attribute__((address_space(1))) void mla_glb_void;

// 16 bytes per lane from global memory straight into LDS: the wave's 64 pieces land at lds_wave_base + 16 * lane
// (NT: cache policy, 2 = nontemporal)
template <int NT> __device__ __forceinline__ void mla_dma16(const void* g, void* lds_wave_base) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the builtin exists in the device pass only)
  __builtin_amdgcn_global_load_lds((mla_glb_void*)const_cast<void*>(g), (mla_lds_void*)lds_wave_base, 16, 0, NT);
#endif
}

template <typename T, int DK, int DV, bool P2, bool ONCE>
__global__ __launch_bounds__(256, 2) void mla_rows_kernel(
    T* __restrict__ out, long out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    const T* __restrict__ q, long q_stride, const T* __restrict__ k_cache, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ token_seq, const int* __restrict__ seq_lens, float scale_log2e, int Hq, int block_size,
    int num_splits, MlaExtra ex) {
  using V = typename Vec8<T>::type;
  constexpr int KSTEPS = DK / 32, KS = (KSTEPS + 3) / 4;
  constexpr int ROW = DK * 2, PIECES = DK / 8, NP = 32 * PIECES / 256;   // bytes, 16-byte pieces of a row; pieces per thread
  constexpr int VI = DV / 256;                                          // runs of 64 values per wave
  static_assert(DK % 64 == 0 && DV % 256 == 0 && 32 * PIECES % 256 == 0, "unsupported latent width");
  // (one object for both uses: the compiler waits for DMA in flight at reads of an object that it knows to be its target)
  __shared__ __attribute__((aligned(1024))) char smem[2 * 32 * ROW + 4 * 2 * 64 * 16];
  float (*s_part)[2][64][4] = reinterpret_cast<float (*)[2][64][4]>(smem + 2 * 32 * ROW);

  const int split = blockIdx.x, qt = blockIdx.y, t = blockIdx.z;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int qh0 = qt * 16;
  const int nq = min(16, Hq - qh0);
  const int seq_len = seq_lens[t];
  const int* bt_row = block_table + (long)(token_seq != nullptr ? token_seq[t] : t) * bt_stride;
  const int win_lo = ex.window > 0 ? max(seq_len - ex.window, 0) : 0;
  const int g_lo = win_lo >> 5;
  const int n_groups = ((seq_len + 31) >> 5) - g_lo;
  const int gps = (n_groups + num_splits - 1) / num_splits;
  const int g_begin = g_lo + split * gps;
  const int g_end = min(g_begin + gps, g_lo + n_groups);

  V qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int sg = wid * KS + s;
    V z;
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] = (T)0.f;
    qf[s] = (sg < KSTEPS && r16 < nq) ? ld8<T>(q + t * q_stride + (long)(qh0 + r16) * DK + 32 * sg + 8 * g4) : z;
  }
  f32x4 acc[VI][4];
#pragma unroll
  for (int i = 0; i < VI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = MLA_NEG_BIG, l = 0.f;

  auto swz = [](int key) { return ((key >> 1) & 1) | (((key >> 3) & 3) << 1); };
  // this thread's pieces of a group: (row, place in LDS) -> piece of the row in memory
  int prow[NP], pbyte[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int c = i * 256 + (int)threadIdx.x;
    prow[i] = c / PIECES;
    pbyte[i] = ((c - prow[i] * PIECES) ^ swz(prow[i])) * 16;
  }
  auto stage = [&](int g, int buf, auto nt) {
    const int base = g * 32;
    const long first = (long)bt_row[base / block_size] * block_size + (base % block_size);
    const char* src = reinterpret_cast<const char*>(k_cache + first * DK);
    // rows that hold no visible key repeat one that does: what a block holds behind the sequence's end is not looked at
    const int lo = max(win_lo - base, 0), hi = min(seq_len - 1 - base, 31);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      mla_dma16<decltype(nt)::value>(src + max(min(prow[i], hi), lo) * ROW + pbyte[i],
                                     smem + buf * 32 * ROW + (i * 256 + wid * 64) * 16);
  };

  const int key_a = 8 * (r16 >> 2) + (r16 & 3);    // K rows of the two interleaved S^T tiles: this one and 4 behind it
  const int off_a = key_a * ROW, off_b = (key_a + 4) * ROW, swz_a = swz(key_a), swz_b = swz(key_a + 4);
  using Cached = std::integral_constant<int, 0>;
  using Past = std::integral_constant<int, 2>;
  if (g_begin < g_end) stage(g_begin, 0, Cached{});
  auto walk = [&](auto nt) {
    for (int g = g_begin; g < g_end; ++g) {
      const int buf = (g - g_begin) & 1;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();                               // the group is in LDS, and nobody reads the other buffer any more
      if (g + 1 < g_end) stage(g + 1, buf ^ 1, nt);
      const char* tile = smem + buf * 32 * ROW;
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int piece = min(wid * KS + s, KSTEPS - 1) * 4 + g4;
        s0 = mfma16(*reinterpret_cast<const V*>(tile + off_a + ((piece ^ swz_a) << 4)), qf[s], s0);
        s1 = mfma16(*reinterpret_cast<const V*>(tile + off_b + ((piece ^ swz_b) << 4)), qf[s], s1);
      }
      *reinterpret_cast<f32x4*>(s_part[wid][0][lane]) = s0;
      *reinterpret_cast<f32x4*>(s_part[wid][1][lane]) = s1;
      // (not __syncthreads(), which would also wait for the next group's rows)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      s0 = *reinterpret_cast<const f32x4*>(s_part[0][0][lane]);
      s1 = *reinterpret_cast<const f32x4*>(s_part[0][1][lane]);
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        s0 += *reinterpret_cast<const f32x4*>(s_part[w][0][lane]);
        s1 += *reinterpret_cast<const f32x4*>(s_part[w][1][lane]);
      }
      const int kidx0 = g * 32 + 8 * g4;
      float p[8];
      float tmax = MLA_NEG_BIG;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sv = (j < 4 ? s0[j & 3] : s1[j & 3]) * scale_log2e;
        p[j] = (kidx0 + j < seq_len && kidx0 + j >= win_lo) ? sv : MLA_NEG_BIG;
        tmax = fmaxf(tmax, p[j]);
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m, tmax);
      const float alpha = fast_exp2(m - m_new);
      float psum = 0.f;
      V pf;
      [[maybe_unused]] V pl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float e = p[j] <= 0.5f * MLA_NEG_BIG ? 0.f : fast_exp2(p[j] - m_new);
        psum += e;
        pf[j] = (T)e;
        if constexpr (P2) pl[j] = (T)(e - (float)pf[j]);
      }
      l = l * alpha + psum;
      m = m_new;
#pragma unroll
      for (int i = 0; i < VI; ++i) {
        // the piece of a row this lane's four values lie in, and which half of it
        const int piece = (wid * VI + i) * 8 + (r16 >> 1), half = (r16 & 1) * 8;
        u32x2 w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = 8 * g4 + j;
          w[j] = *reinterpret_cast<const u32x2*>(tile + key * ROW + ((piece ^ swz(key)) << 4) + half);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          union { uint32_t u[4]; V f; } fr;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t a = w[2 * j][v >> 1], b = w[2 * j + 1][v >> 1];
            fr.u[j] = __builtin_amdgcn_perm(b, a, (v & 1) ? 0x07060302u : 0x05040100u);
          }
          acc[i][v] *= alpha;
          acc[i][v] = mfma16(fr.f, pf, acc[i][v]);
          if constexpr (P2) acc[i][v] = mfma16(fr.f, pl, acc[i][v]);
        }
      }
    }
  };
  bool past = false;
  if constexpr (ONCE)                              // (while the first group is on its way)
    if (g_end - g_begin >= 4)
      past = reads_alone(&s_part[0][0][0][0], t, gridDim.z, seq_lens, block_table, bt_stride, g_begin * 32 / block_size, block_size,
                         ex.window, ROW, ex.past_bytes);
  if constexpr (ONCE) {
    if (past) walk(Past{});
    else walk(Cached{});
  } else {
    walk(Cached{});
  }

  float lsum = l;
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (r16 >= nq) return;
  const int qh = qh0 + r16;
  // acc[i][v][r]: value 64 (wid * VI + i) + 16 g4 + 4 r + v
  if (num_splits == 1) {
    float factor = 1.f;
    if (ex.sinks != nullptr) mla_add_sink(ex.sinks[qh] * 1.4426950408889634f, m, lsum, factor);
    float inv = lsum > 0.f ? factor / lsum : 0.f;
    if (ex.gate != nullptr) inv *= 1.f / (1.f + __expf(-(float)((const T*)ex.gate)[t * ex.gate_stride + qh]));
    T* orow = out + t * out_stride + (long)qh * DV + 16 * g4;
#pragma unroll
    for (int i = 0; i < VI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        typename Vec4<T>::type o;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = (T)(acc[i][v][r] * inv);
        *reinterpret_cast<typename Vec4<T>::type*>(orow + 64 * (wid * VI + i) + 4 * r) = o;
      }
  } else {
    const long pidx = ((long)t * Hq + qh) * num_splits + split;
#pragma unroll
    for (int i = 0; i < VI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f32x4*>(part_o + pidx * DV + 64 * (wid * VI + i) + 16 * g4 + 4 * r) =
            f32x4{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
    if (wid == 0 && g4 == 0) { part_ml[2 * pidx] = m; part_ml[2 * pidx + 1] = lsum; }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// The same rows for FOUR tiles of 16 heads of a token a workgroup.  Groups of 64 keys in LDS, the next one on its way while one is
// multiplied; eight waves:
//   * QK: a wave one tile's whole reduction (its Q in registers) for half of the group's keys, so that a key's score is in one
//     lane.  A tile's two waves trade their maxima through LDS before they form weights, which are then what mla_rows_kernel has (the
//     largest one exact; each half by a maximum of its own in whole powers of two spares a barrier that turned out to cost nothing, and
//     is up to 1.13 times as far from 64-bit sums).
//   * All trade weights through LDS (16 bytes a lane).
//   * PV: a wave a run of 64 values (half of them and two tiles where there are 256) for all keys and tiles: a value is read and turned
//     into a fragment, as in mla_rows_kernel, once for the four.
// The single kernel is bound by turning keys into V^T fragments and by its barriers, 1.25 us per 16 heads and 32 keys of a workgroup;
// here a group costs 2.15 us for four times the heads and twice the keys (a fragment turned serves four tiles, a key read
// from LDS a QK of its own still), though 156 KB of LDS leave one workgroup a CU and nothing beside it while it begins and ends.
// us, single / this (one launch each, 576 of 512 values, 16 bits): 128 heads, 126 rows of 241 keys 56 / 31, 69 of 780 105 / 55, 128 of
// 600 128 / 53, 30 of 2500 109 / 64, 7 of 9212 109 / 55, a prompt of 174 behind 496 110 / 68, three of 293 169 / 119; 64 heads, two
// prompts of 200 111 / 63; 80 heads, 100 tokens behind 2900 166 / 118; one row of 3000, 128 heads, 20 / 26.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int DK, int DV>
__global__ __launch_bounds__(512, 2) void mla_rows4_kernel(
    T* __restrict__ out, long out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    const T* __restrict__ q, long q_stride, const T* __restrict__ k_cache, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ token_seq, const int* __restrict__ seq_lens, float scale_log2e, int Hq, int block_size, int num_splits,
    MlaExtra ex) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the buffer builtins exist in the device pass only)
  using V = typename Vec8<T>::type;
  constexpr int KSTEPS = DK / 32, ROW = DK * 2, PIECES = DK / 8, GROUP = 64;
  constexpr int NP = 32 * PIECES / 256;            // 16-byte pieces of a half group per thread
  constexpr int RUNS = DV / 64, TPW = RUNS / 2;    // of values, one a wave; tiles that a wave multiplies it by
  static_assert(DK % 64 == 0 && (RUNS == 4 || RUNS == 8) && 32 * PIECES % 256 == 0, "unsupported latent width");
  // (one object for all uses, see mla_rows_kernel): two groups | weights of eight waves | their maxima
  __shared__ __attribute__((aligned(1024))) char smem[2 * GROUP * ROW + 8 * 64 * 16 + 8 * 16 * 4];
  char* const s_p = smem + 2 * GROUP * ROW;
  float* const s_m = reinterpret_cast<float*>(s_p + 8 * 64 * 16);

  const int split = blockIdx.x, t = blockIdx.z;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int tile_n = wid & 3, half = wid >> 2;     // of the scores: the wave's tile and half of the keys
  const int run_v = wid % RUNS, tile0 = wid / RUNS * TPW;        // of the products with values: the run, the first of the tiles
  const int seq_len = seq_lens[t];
  const int* const bt_row = block_table + (long)(token_seq != nullptr ? token_seq[t] : t) * bt_stride;
  const int win_lo = ex.window > 0 ? max(seq_len - ex.window, 0) : 0;
  const int g_lo = win_lo / GROUP;
  const int n_groups = (seq_len + GROUP - 1) / GROUP - g_lo;
  const int gps = (n_groups + num_splits - 1) / num_splits;
  const int g_begin = g_lo + split * gps;
  const int g_end = min(g_begin + gps, g_lo + n_groups);

  auto swz = [](int key) { return ((key >> 1) & 1) | (((key >> 3) & 3) << 1); };
  // this thread's pieces of its half of a group (four waves bring a half): their places in 32 rows in memory
  unsigned place[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int c = i * 256 + ((int)threadIdx.x & 255), r = c / PIECES;
    place[i] = r * ROW + ((c - r * PIECES) ^ swz(r)) * 16;
  }
  const int per_block = block_size >> 5, shift = (per_block & (per_block - 1)) == 0 ? __builtin_ctz(per_block) : -1;
  // the wave's half of a group: which 32 keys (a half that holds no visible key repeats one that does), and their block
  int half_of = 0, block_of = 0;
  auto find = [&](int g) {
    half_of = max(min(2 * g + half, (seq_len - 1) >> 5), win_lo >> 5);
    block_of = bt_row[shift >= 0 ? half_of >> shift : half_of / per_block];
  };
  // what `find` has found: the descriptor, and the places of this thread's pieces (rows that hold no visible key repeat one that does)
  auto rows_of = [&](unsigned (&at)[NP]) {
    const int base = half_of * 32, inside = shift >= 0 ? half_of & (per_block - 1) : half_of % per_block;
    const long first = (long)block_of * block_size + inside * 32;
    const int lo = max(win_lo - base, 0), hi = min(seq_len - 1 - base, 31);
#pragma unroll
    for (int i = 0; i < NP; ++i) at[i] = place[i];
    if (lo > 0 || hi < 31) {
      int tid = threadIdx.x & 255;
      asm volatile("" : "+v"(tid));                // (not worth registers in between)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int c = i * 256 + tid, r = c / PIECES;
        at[i] = max(min(r, hi), lo) * ROW + ((c - r * PIECES) ^ swz(r)) * 16;
      }
    }
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(k_cache + first * DK), 0, 32 * ROW, 0x00020000);
  };
  char* const mine = smem + half * 32 * ROW + tile_n * 1024;
  if (g_begin < g_end) {
    find(g_begin);
    unsigned at[NP];
    const auto rows = rows_of(at);
#pragma unroll
    for (int i = 0; i < NP; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (mla_lds_void*)(mine + i * 4096), 16, at[i], 0, 0, 0);
    if (g_begin + 1 < g_end) find(g_begin + 1);
  }
  V qf[KSTEPS];
  {
    const int head = (4 * (int)blockIdx.y + tile_n) * 16 + r16;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      V z;
#pragma unroll
      for (int j = 0; j < 8; ++j) z[j] = (T)0.f;
      qf[s] = head < Hq ? ld8<T>(q + t * q_stride + (long)head * DK + 32 * s + 8 * g4) : z;
    }
  }
  f32x4 acc[TPW][4];
  float M[TPW];                                    // the tiles' maxima, which the sums go by
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    M[i] = MLA_NEG_BIG;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m = MLA_NEG_BIG, l = 0.f;                  // the maximum of the wave's own tile, the sum of its half
  // K rows of the two interleaved S^T tiles: key_a and 4 behind it (whose pieces are turned alike); of 64 values the two pieces.
  // V: keys 8 g4 + j of a half, the pieces of those with bit 1 of j clear and set.  All else is in the instructions' offsets.
  const int key_a = 8 * (r16 >> 2) + (r16 & 3);
  int k_at[2], v_at[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    k_at[e] = key_a * ROW + (((4 * e + g4) ^ swz(key_a)) << 4);
    v_at[e] = 8 * g4 * ROW + (((r16 >> 1) ^ (e | g4 << 1)) << 4) + (r16 & 1) * 8 + run_v * 128;
  }

  for (int g = g_begin; g < g_end; ++g) {
    const int buf = (g - g_begin) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                               // the group is in LDS, and nobody reads the other buffer any more
    const char* const group = smem + buf * GROUP * ROW;
    const char* const keys = group + half * 32 * ROW;
    f32x4 s0[2] = {}, s1[2] = {};
    auto score = [&](int s) {
      const char* const at = keys + k_at[s & 1] + (s >> 1) * 128;
      s0[s & 1] = mfma16(*reinterpret_cast<const V*>(at), qf[s], s0[s & 1]);
      s1[s & 1] = mfma16(*reinterpret_cast<const V*>(at + 4 * ROW), qf[s], s1[s & 1]);
    };
    static_assert(KSTEPS == 2 * NP, "a piece every other step");
    if (g + 1 < g_end) {
      unsigned at[NP];
      const auto rows = rows_of(at);
      // (72 pieces of 1 KB asked for at a time are 0.6 us before the last waves' first product)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (mla_lds_void*)(mine + (buf ^ 1) * GROUP * ROW + i * 4096), 16, at[i], 0, 0, 0);
        score(2 * i);
        score(2 * i + 1);
        __builtin_amdgcn_sched_barrier(0x18e);     // (what reads LDS and multiplies may move across, the pieces stay apart)
      }
      if (g + 2 < g_end) find(g + 2);              // (the table's entry is there when it is wanted)
    } else {
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) score(s);
    }
    const f32x4 sa = s0[0] + s0[1], sb = s1[0] + s1[1];
    const int key0 = g * GROUP + half * 32, kidx0 = key0 + 8 * g4;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = (j < 4 ? sa[j & 3] : sb[j & 3]) * scale_log2e;
    const bool masked = key0 + 32 > seq_len || key0 < win_lo;
    if (masked)
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = (kidx0 + j < seq_len && kidx0 + j >= win_lo) ? p[j] : MLA_NEG_BIG;
    float tmax = fmaxf(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])), fmaxf(fmaxf(p[4], p[5]), fmaxf(p[6], p[7])));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    if (g4 == 0) s_m[wid * 16 + r16] = tmax;
    // (not __syncthreads(), which would also wait for the next group's rows)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const float m_new = fmaxf(m, fmaxf(tmax, s_m[(wid ^ 4) * 16 + r16]));
    float top[TPW];
#pragma unroll
    for (int n = 0; n < TPW; ++n) top[n] = fmaxf(M[n], fmaxf(s_m[(tile0 + n) * 16 + r16], s_m[(tile0 + n + 4) * 16 + r16]));
    V pf;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = fast_exp2(p[j] - m_new);
      p[j] = masked && p[j] <= 0.5f * MLA_NEG_BIG ? 0.f : e;
      pf[j] = (T)p[j];
    }
    const float psum = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    l = l * fast_exp2(m - m_new) + psum;
    m = m_new;
    *reinterpret_cast<V*>(s_p + (wid * 64 + lane) * 16) = pf;
#pragma unroll
    for (int n = 0; n < TPW; ++n) {
      if (__any(top[n] != M[n])) {
        const float alpha = fast_exp2(M[n] - top[n]);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[n][v] *= alpha;
        M[n] = top[n];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    V weights[TPW][2];
#pragma unroll
    for (int n = 0; n < TPW; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h) weights[n][h] = *reinterpret_cast<const V*>(s_p + ((tile0 + n + 4 * h) * 64 + lane) * 16);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      // a lane's four neighbouring values of each of eight keys, turned into V^T fragments of four tiles of columns
      u32x2 w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = *reinterpret_cast<const u32x2*>(group + v_at[j >> 1 & 1] + (kk * 32 + j) * ROW);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        union { uint32_t u[4]; V f; } fr;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t a = w[2 * j][v >> 1], b = w[2 * j + 1][v >> 1];
          fr.u[j] = __builtin_amdgcn_perm(b, a, (v & 1) ? 0x07060302u : 0x05040100u);
        }
#pragma unroll
        for (int n = 0; n < TPW; ++n) acc[n][v] = mfma16(fr.f, weights[n][kk], acc[n][v]);
      }
    }
  }

  // ---- the halves' sums meet
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  __syncthreads();
  float* const s_l = reinterpret_cast<float*>(s_p);
  if (g4 == 0) s_l[wid * 16 + r16] = l;
  __syncthreads();
#pragma unroll
  for (int n = 0; n < TPW; ++n) {
    const int tile = tile0 + n, qh = (4 * (int)blockIdx.y + tile) * 16 + r16;
    if (qh >= Hq) continue;
    float lsum = s_l[tile * 16 + r16] + s_l[(tile + 4) * 16 + r16];
    // acc[n][v][r]: value 64 run_v + 16 g4 + 4 r + v
    if (num_splits == 1) {
      float factor = 1.f;
      if (ex.sinks != nullptr) mla_add_sink(ex.sinks[qh] * 1.4426950408889634f, M[n], lsum, factor);
      float inv = lsum > 0.f ? factor / lsum : 0.f;
      if (ex.gate != nullptr) inv *= 1.f / (1.f + __expf(-(float)((const T*)ex.gate)[t * ex.gate_stride + qh]));
      T* orow = out + t * out_stride + (long)qh * DV + 64 * run_v + 16 * g4;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        typename Vec4<T>::type o;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = (T)(acc[n][v][r] * inv);
        *reinterpret_cast<typename Vec4<T>::type*>(orow + 4 * r) = o;
      }
    } else {
      const long pidx = ((long)t * Hq + qh) * num_splits + split;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f32x4*>(part_o + pidx * DV + 64 * run_v + 16 * g4 + 4 * r) =
            f32x4{acc[n][0][r], acc[n][1][r], acc[n][2][r], acc[n][3][r]};
      if (run_v == 0 && g4 == 0) { part_ml[2 * pidx] = M[n]; part_ml[2 * pidx + 1] = lsum; }
    }
  }
#endif
}

// ---------------------------------------------------------------------------------------------------------------
// Several query tiles per workgroup over ONE stream of cache fragments, for caches that the kernel over key rows does not read (8
// bits, blocks that cut a group of 32 keys, narrow values; where it does, it is 1.2 to 4.6 times as fast: 880 prompt tokens of 128
// heads 902 us here and 584 there).  The kernel over both caches requests every cached
// row once per 16 query rows; wherever more rows share a sequence, that is the L2's bandwidth, not HBM's:
//   * BY_TOKEN (prefill chunks, verification): the NQ tiles are NQ consecutive tokens of one sequence - the token
//     whose position is a multiple of NQ (or the first of its sequence in the step) leads a workgroup, the
//     workgroups of its followers exit at once; every tile masks with its own causal limit;
//   * otherwise (decode, many heads per rank): the NQ tiles are NQ head tiles of one token.
// Same split of the two reductions over the four waves; one wave per SIMD (the NQ accumulator sets and query
// fragments take the registers the second wave had), all NQ partial score tiles exchanged behind one barrier.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int DK, int DV, int NQ, bool BY_TOKEN, bool KV8, bool P2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mla_attention_multi_kernel(
    T* __restrict__ out, long out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    const T* __restrict__ q, long q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_table, int bt_stride, const int* __restrict__ token_seq,
    const int* __restrict__ seq_lens, float scale_log2e, int T_, int Hq, int block_size, int num_splits,
    MlaExtra ex) {
  using V = typename Vec8<T>::type;
  constexpr int KSTEPS = DK / 32;
  constexpr int KS = (KSTEPS + 3) / 4;
  constexpr int VT = DV / 64;
  // [buffer][wave][tile][half][lane][4]: a lane's f32x4 sits next to its neighbours' (conflict-free b128 accesses)
  __shared__ float s_part[2][4][NQ][2][64][4];

  const int split = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  // ---- this workgroup's tiles: (token, first head, visible keys); a tile with 0 keys is absent
  int tok[NQ], qh0[NQ], slen[NQ];
  // BY_TOKEN: leaders are (mostly) every NQ-th token, and consecutive workgroup ids go round the 8 XCDs: with
  // t0 = id they would all land on two of them.  Walk the tokens residue class by residue class instead
  // (ids 0 .. G-1 -> tokens 0, NQ, 2 NQ, ...; the next G ids -> 1, NQ + 1, ...).
  int t0 = blockIdx.z;
  if constexpr (BY_TOKEN) {
    const int G = (T_ + NQ - 1) / NQ;
    t0 = (int)(blockIdx.z % G) * NQ + (int)(blockIdx.z / G);
    if (t0 >= T_) return;
  }
  const int seq_row = token_seq != nullptr ? token_seq[t0] : t0;
  if constexpr (BY_TOKEN) {
    const int pos0 = seq_lens[t0] - 1;
    if (t0 > 0 && token_seq[t0 - 1] == seq_row && pos0 % NQ != 0) return;        // a follower: its leader covers it
    bool live = true;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int t = t0 + n;
      live = live && t < T_ && (n == 0 || (token_seq[t] == seq_row && (seq_lens[t] - 1) % NQ != 0));
      tok[n] = live ? t : t0;
      qh0[n] = blockIdx.y * 16;
      slen[n] = live ? seq_lens[t] : 0;
    }
  } else {
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      tok[n] = t0;
      qh0[n] = (blockIdx.y * NQ + n) * 16;
      slen[n] = qh0[n] < Hq ? seq_lens[t0] : 0;
    }
  }
  int seq_len = 0;
#pragma unroll
  for (int n = 0; n < NQ; ++n) seq_len = max(seq_len, slen[n]);
  const int* bt_row = block_table + (long)seq_row * bt_stride;

  // every tile's own window start; nothing in front of the earliest one is read
  int wlo[NQ];
  int win_lo = seq_len;
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    wlo[n] = ex.window > 0 ? max(slen[n] - ex.window, 0) : 0;
    if (slen[n] > 0) win_lo = min(win_lo, wlo[n]);
  }
  const int g_lo = win_lo >> 5;
  const int n_groups = ((seq_len + 31) >> 5) - g_lo;
  const int gps = (n_groups + num_splits - 1) / num_splits;
  const int g_begin = g_lo + split * gps;
  const int g_end = min(g_begin + gps, g_lo + n_groups);

  V qf[NQ][KS];
  int kstep_off[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kstep_off[s] = 32 * min(wid * KS + s, KSTEPS - 1) + 8 * g4;
#pragma unroll
  for (int n = 0; n < NQ; ++n)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      V z;
#pragma unroll
      for (int j = 0; j < 8; ++j) z[j] = (T)0.f;
      const bool have = wid * KS + s < KSTEPS && slen[n] > 0 && qh0[n] + r16 < Hq;
      qf[n][s] = have ? ld8<T>(q + tok[n] * q_stride + (long)(qh0[n] + r16) * DK + kstep_off[s]) : z;
    }
  f32x4 acc[NQ][VT];
  float m[NQ], l[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m[n] = MLA_NEG_BIG;
    l[n] = 0.f;
#pragma unroll
    for (int i = 0; i < VT; ++i) acc[n][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int slab = block_size * 16;
  using R = typename MlaRaw<T, KV8>::type;
  struct Frag { R ka[KS], kb[KS], vf[VT]; };
  auto load = [&](Frag& f, int g) {
    const int base = g * 32;
    const int key0 = base + 8 * (r16 >> 2) + (r16 & 3);
    const int ka = max(min(key0, seq_len - 1), win_lo), kb = max(min(key0 + 4, seq_len - 1), win_lo);
    const long ra = ((long)bt_row[ka / block_size] * block_size + (ka % block_size)) * DK;
    const long rb = ((long)bt_row[kb / block_size] * block_size + (kb % block_size)) * DK;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      f.ka[s] = mla_ld<T, KV8>(k_cache, ra + kstep_off[s]);
      f.kb[s] = mla_ld<T, KV8>(k_cache, rb + kstep_off[s]);
    }
    const int vkey = max(min(base + 8 * g4, seq_len - 1), win_lo) & ~7;
    const long vo = (long)bt_row[vkey / block_size] * (DV / 16) * slab + ((vkey % block_size) >> 3) * 128 + 8 * r16;
#pragma unroll
    for (int i = 0; i < VT; ++i) f.vf[i] = mla_ld<T, KV8>(v_cache, vo + (long)(wid * VT + i) * slab);
  };

  Frag cur, nxt;
  if (g_begin < g_end) load(cur, g_begin);
  for (int g = g_begin; g < g_end; ++g) {
    load(nxt, min(g + 1, g_end - 1));
    V ka[KS], kb[KS], vf[VT];                    // (an e4m3 cache: widened once, shared by the NQ tiles)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      ka[s] = mla_widen<T, KV8>(cur.ka[s]);
      kb[s] = mla_widen<T, KV8>(cur.kb[s]);
    }
#pragma unroll
    for (int i = 0; i < VT; ++i) vf[i] = mla_widen<T, KV8>(cur.vf[i]);
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma16(ka[s], qf[n][s], s0);
        s1 = mfma16(kb[s], qf[n][s], s1);
      }
      *reinterpret_cast<f32x4*>(&s_part[g & 1][wid][n][0][lane][0]) = s0;
      *reinterpret_cast<f32x4*>(&s_part[g & 1][wid][n][1][lane][0]) = s1;
    }
    __syncthreads();
    const int kidx0 = g * 32 + 8 * g4;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      f32x4 s0 = *reinterpret_cast<const f32x4*>(&s_part[g & 1][0][n][0][lane][0]);
      f32x4 s1 = *reinterpret_cast<const f32x4*>(&s_part[g & 1][0][n][1][lane][0]);
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        s0 += *reinterpret_cast<const f32x4*>(&s_part[g & 1][w][n][0][lane][0]);
        s1 += *reinterpret_cast<const f32x4*>(&s_part[g & 1][w][n][1][lane][0]);
      }
      float p[8];
      float tmax = MLA_NEG_BIG;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sv = (j < 4 ? s0[j & 3] : s1[j & 3]) * scale_log2e;
        p[j] = (kidx0 + j < slen[n] && kidx0 + j >= wlo[n]) ? sv : MLA_NEG_BIG;
        tmax = fmaxf(tmax, p[j]);
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m[n], tmax);
      const float alpha = fast_exp2(m[n] - m_new);
      float psum = 0.f;
      V pf;
      [[maybe_unused]] V pl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float e = p[j] <= 0.5f * MLA_NEG_BIG ? 0.f : fast_exp2(p[j] - m_new);
        psum += e;
        pf[j] = (T)e;
        if constexpr (P2) pl[j] = (T)(e - (float)pf[j]);
      }
      l[n] = l[n] * alpha + psum;
      m[n] = m_new;
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        acc[n][i] *= alpha;
        acc[n][i] = mfma16(vf[i], pf, acc[n][i]);
        if constexpr (P2) acc[n][i] = mfma16(vf[i], pl, acc[n][i]);
      }
    }
    cur = nxt;
  }

#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    float lsum = l[n];
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    const int qh = qh0[n] + r16;
    if (slen[n] <= 0 || qh >= Hq) continue;
    if (num_splits == 1) {
      float factor = 1.f;
      if (ex.sinks != nullptr) mla_add_sink(ex.sinks[qh] * 1.4426950408889634f, m[n], lsum, factor);
      float inv = lsum > 0.f ? factor / lsum : 0.f;
      if (ex.gate != nullptr) inv *= 1.f / (1.f + __expf(-(float)((const T*)ex.gate)[tok[n] * ex.gate_stride + qh]));
      T* orow = out + tok[n] * out_stride + (long)qh * DV + 4 * g4;
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        typename Vec4<T>::type o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (T)(acc[n][i][r] * inv);
        *reinterpret_cast<typename Vec4<T>::type*>(orow + 16 * (wid * VT + i)) = o;
      }
    } else {
      const long pidx = ((long)tok[n] * Hq + qh) * num_splits + split;
#pragma unroll
      for (int i = 0; i < VT; ++i)
        *reinterpret_cast<f32x4*>(part_o + pidx * DV + 16 * (wid * VT + i) + 4 * g4) = acc[n][i];
      if (wid == 0 && g4 == 0) { part_ml[2 * pidx] = m[n]; part_ml[2 * pidx + 1] = lsum; }
    }
  }
}

template <typename T, int DV>
__global__ __launch_bounds__(SPLIT_MERGE_MAX_THREADS) void mla_reduce_kernel(
    T* __restrict__ out, long out_stride, const float* __restrict__ part_o, const float* __restrict__ part_ml, int Hq,
    int num_splits, MlaExtra ex) {
  const int t = blockIdx.y, qh = blockIdx.x;
  const long p0 = ((long)t * Hq + qh) * num_splits;
  f32x4 o;
  float lt;
  if (!split_merge<DV>(part_o + p0 * DV, part_ml + 2 * p0, num_splits, ex.sinks != nullptr ? ex.sinks + qh : nullptr,
                       MLA_NEG_BIG, o, lt)) return;
  float inv = lt > 0.f ? 1.f / lt : 0.f;
  if (ex.gate != nullptr) inv *= 1.f / (1.f + __expf(-(float)((const T*)ex.gate)[t * ex.gate_stride + qh]));
  T* dst = out + t * out_stride + (long)qh * DV + 4 * threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) dst[i] = (T)(o[i] * inv);
}

// One token's latent row into both cache forms.  x[T][DK] (row stride in elements); slot < 0: skipped.
template <typename T, bool KV8>
__global__ void mla_cache_write_kernel(const T* __restrict__ x, long x_stride, void* __restrict__ k_cache,
                                       void* __restrict__ v_cache, const int* __restrict__ slot_mapping, int DK, int DV,
                                       int block_size) {
  const int t = blockIdx.x;
  const int slot = slot_mapping[t];
  if (slot < 0) return;
  const long blk = slot / block_size;
  const int off = slot % block_size;
  const T* row = x + t * x_stride;
  const long krow = ((long)blk * block_size + off) * DK;
  const long slab = (long)block_size * 16;
  const long vblk = blk * (DV / 16) * slab + (off >> 3) * 128 + (off & 7);
  for (int d = threadIdx.x; d < DK; d += blockDim.x) {
    const float v = (float)row[d];
    mla_st<T, KV8>(k_cache, krow + d, v);
    if (d < DV) mla_st<T, KV8>(v_cache, vblk + (d >> 4) * slab + (d & 15) * 8, v);
  }
}

// Everything between the projections and the attention of one token, in one launch (one workgroup per token):
//   * RMSNorm of the latent's first RANK values, rotation of its last ROPE values (half-apart pairs, fp32
//     [cos | sin] table row of the token's position), and the resulting row written into both cache forms;
//   * the absorbed query assembled per head: q_full[t][h] = [ q_lat[h][t] (RANK) | rotated q[t][h][nope:] (ROPE) ].
// Replaces a norm, two slice copies, the rotary kernel, two concatenations and the cache write.
template <typename T, bool KV8>
__global__ __launch_bounds__(256) void mla_prep_kernel(
    T* __restrict__ q_full, const T* __restrict__ q, long q_tok_stride, int q_head_stride, int nope,
    const T* __restrict__ q_lat, long q_lat_head_stride, long q_lat_tok_stride, const T* __restrict__ latent,
    long latent_stride, const T* __restrict__ norm_w, float eps, const float* __restrict__ cos_sin,
    const int* __restrict__ positions, void* __restrict__ k_cache, void* __restrict__ v_cache,
    const int* __restrict__ slot_mapping, int H, int RANK, int ROPE, int block_size) {
  __shared__ float red[17];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int DK = RANK + ROPE, half = ROPE / 2;
  const float* cs = cos_sin + (long)positions[t] * ROPE;
  const T* lat = latent + t * latent_stride;
  float ss = 0.f;
  for (int d = tid; d < RANK; d += 256) { const float v = (float)lat[d]; ss += v * v; }
  const float rinv = rsqrtf(block_sum(ss, red) / (float)RANK + eps);
  const int slot = slot_mapping != nullptr ? slot_mapping[t] : -1;
  if (slot >= 0) {
    const long blk = slot / block_size;
    const int off = slot % block_size;
    const long krow = (blk * block_size + off) * DK;
    const long slab = (long)block_size * 16;
    const long vblk = blk * (RANK / 16) * slab + (off >> 3) * 128 + (off & 7);
    for (int d = tid; d < RANK; d += 256) {
      const float v = (float)(T)((float)lat[d] * rinv * (float)norm_w[d]);      // rounded as the norm kernel rounds
      mla_st<T, KV8>(k_cache, krow + d, v);
      mla_st<T, KV8>(v_cache, vblk + (d >> 4) * slab + (d & 15) * 8, v);
    }
    for (int i = tid; i < half; i += 256) {
      const float x1 = (float)lat[RANK + i], x2 = (float)lat[RANK + half + i];
      mla_st<T, KV8>(k_cache, krow + RANK + i, x1 * cs[i] - x2 * cs[half + i]);
      mla_st<T, KV8>(k_cache, krow + RANK + half + i, x2 * cs[i] + x1 * cs[half + i]);
    }
  }
  T* qo = q_full + (long)t * H * DK;
  for (int e = tid; e < H * RANK; e += 256) {
    const int h = e / RANK, d = e - h * RANK;
    qo[(long)h * DK + d] = q_lat[h * q_lat_head_stride + t * q_lat_tok_stride + d];
  }
  for (int e = tid; e < H * half; e += 256) {
    const int h = e / half, i = e - h * half;
    const T* qr = q + t * q_tok_stride + (long)h * q_head_stride + nope;
    const float x1 = (float)qr[i], x2 = (float)qr[half + i];
    qo[(long)h * DK + RANK + i] = (T)(x1 * cs[i] - x2 * cs[half + i]);
    qo[(long)h * DK + RANK + half + i] = (T)(x2 * cs[i] + x1 * cs[half + i]);
  }
}

template <typename T, int DK, int DV, bool KV8, bool P2>
int launch_mla(void* out, long out_stride, void* part_o, void* part_ml, const void* q, long q_stride,
               const void* k_cache, const void* v_cache, const int* block_table, int bt_stride, const int* token_seq,
               const int* seq_lens, float scale, int T_, int Hq, int block_size, int num_splits, int mode,
               MlaExtra ex, hipStream_t st) {
  const int q_tiles = (Hq + 15) / 16;
  const float sl2 = scale * 1.4426950408889634f;
  constexpr int NQ = 4;
  if (mode == 1 && token_seq != nullptr) {          // NQ consecutive tokens of a sequence share the cache stream
    // (ids walk the tokens residue class by residue class: (T_ + NQ - 1) / NQ ids per class)
    mla_attention_multi_kernel<T, DK, DV, NQ, true, KV8, P2><<<dim3(num_splits, q_tiles, (T_ + NQ - 1) / NQ * NQ), 256, 0, st>>>(
        (T*)out, out_stride, (float*)part_o, (float*)part_ml, (const T*)q, q_stride, k_cache, v_cache, block_table,
        bt_stride, token_seq, seq_lens, sl2, T_, Hq, block_size, num_splits, ex);
  } else if (mode == 2) {                           // NQ head tiles of a token share it
    mla_attention_multi_kernel<T, DK, DV, NQ, false, KV8, P2><<<dim3(num_splits, (q_tiles + NQ - 1) / NQ, T_), 256, 0, st>>>(
        (T*)out, out_stride, (float*)part_o, (float*)part_ml, (const T*)q, q_stride, k_cache, v_cache, block_table,
        bt_stride, token_seq, seq_lens, sl2, T_, Hq, block_size, num_splits, ex);
  } else if (mode == 3) {                           // a workgroup per 16 heads over the key rows alone
    if constexpr (!KV8 && DV % 256 == 0 && DK % 64 == 0) {
      if (block_size % 32) return -1;
#define MLA_ROWS(ONCE)                                                                                                     \
  mla_rows_kernel<T, DK, DV, P2, ONCE><<<dim3(num_splits, q_tiles, T_), 256, 0, st>>>(                                      \
      (T*)out, out_stride, (float*)part_o, (float*)part_ml, (const T*)q, q_stride, (const T*)k_cache, block_table, bt_stride, \
      token_seq, seq_lens, sl2, Hq, block_size, num_splits, ex)
      if (ex.past_bytes > 0) MLA_ROWS(true);
      else MLA_ROWS(false);
#undef MLA_ROWS
    } else {
      return -4;
    }
  } else if (mode == 4) {                           // four tiles of a token's heads over the key rows
    if constexpr (!KV8 && !P2 && DV % 256 == 0 && DK % 64 == 0) {
      if (block_size % 32) return -1;
      mla_rows4_kernel<T, DK, DV><<<dim3(num_splits, (q_tiles + 3) / 4, T_), 512, 0, st>>>(
          (T*)out, out_stride, (float*)part_o, (float*)part_ml, (const T*)q, q_stride, (const T*)k_cache, block_table, bt_stride,
          token_seq, seq_lens, sl2, Hq, block_size, num_splits, ex);
    } else {
      return -4;
    }
  } else {
    mla_attention_kernel<T, DK, DV, KV8, P2><<<dim3(num_splits, q_tiles, T_), 256, 0, st>>>(
        (T*)out, out_stride, (float*)part_o, (float*)part_ml, (const T*)q, q_stride, k_cache, v_cache, block_table,
        bt_stride, token_seq, seq_lens, sl2, Hq, block_size, num_splits, ex);
  }
  HIP_LAUNCH_CHECK();
  if (num_splits > 1) {
    mla_reduce_kernel<T, DV><<<dim3(Hq, T_), split_merge_threads(DV, num_splits), 0, st>>>(
        (T*)out, out_stride, (const float*)part_o, (const float*)part_ml, Hq, num_splits, ex);
    HIP_LAUNCH_CHECK();
  }
  return 0;
}

template <typename T>
int dispatch_mla(int DK, int DV, int kv_fp8, void* out, long out_stride, void* part_o, void* part_ml, const void* q,
                 long q_stride, const void* k_cache, const void* v_cache, const int* block_table, int bt_stride,
                 const int* token_seq, const int* seq_lens, float scale, int T_, int Hq, int block_size,
                 int num_splits, int mode, int precise, MlaExtra ex, hipStream_t st) {
  if (precise && kv_fp8) return -6;       // (split weights over an 8-bit cache: not built)
#define MLA_CASE(DK_, DV_)                                                                                        \
  if (DK == DK_ && DV == DV_) {                                                                                   \
    if (kv_fp8)                                                                                                   \
      return launch_mla<T, DK_, DV_, true, false>(out, out_stride, part_o, part_ml, q, q_stride, k_cache, v_cache, \
                                                  block_table, bt_stride, token_seq, seq_lens, scale, T_, Hq,     \
                                                  block_size, num_splits, mode, ex, st);                          \
    if (precise)                                                                                                  \
      return launch_mla<T, DK_, DV_, false, true>(out, out_stride, part_o, part_ml, q, q_stride, k_cache, v_cache, \
                                                  block_table, bt_stride, token_seq, seq_lens, scale, T_, Hq,     \
                                                  block_size, num_splits, mode, ex, st);                          \
    return launch_mla<T, DK_, DV_, false, false>(out, out_stride, part_o, part_ml, q, q_stride, k_cache, v_cache, \
                                                 block_table, bt_stride, token_seq, seq_lens, scale, T_, Hq,      \
                                                 block_size, num_splits, mode, ex, st);                           \
  }
  MLA_CASE(576, 512) MLA_CASE(96, 64) MLA_CASE(320, 256)
#undef MLA_CASE
  return -4;
}

}  // namespace

// out[T][Hq][DV] = softmax(scale * q[T][Hq][DK] . K^T) . V over the latent cache.  token_seq[T] (may be null:
// token t uses block-table row t) and seq_lens[T] (keys 0 .. seq_lens[t] - 1 are visible to token t).
// part_o / part_ml: num_splits * T * Hq * (DV | 2) floats when num_splits > 1.
// mode 0: one workgroup per (token, 16 heads); 1: four consecutive tokens of a sequence per workgroup (needs
// token_seq; positions inside a sequence must be consecutive); 2: four head tiles of a token per workgroup.
// mode 3: as mode 0, the values taken from the key rows (16-bit caches, blocks of a multiple of 32 tokens, DV a multiple of 256);
// mode 4: as mode 3, four head tiles of a token per workgroup (not with precise).
// past_bytes > 0 (mode 3, token_seq null): where the rows seen are that many bytes, those of one token alone are read past the caches.
// Supported (DK, DV): (576, 512) DeepSeek-V2 / V3, (320, 256), (96, 64).
VDAMD_API int vdamd_mla_attention(void* out, long out_stride, void* part_o, void* part_ml, const void* q,
                                  long q_stride, const void* k_cache, const void* v_cache, const int* block_table,
                                  int bt_stride, const int* token_seq, const int* seq_lens, float scale, int T_,
                                  int Hq, int DK, int DV, int block_size, int num_splits, int mode, int dtype,
                                  int kv_fp8, int precise, int window, const float* sinks, const void* gate,
                                  long gate_stride, long past_bytes, void* stream) {
  if (T_ <= 0) return 0;
  if (window < 0 || (past_bytes > 0 && token_seq != nullptr)) return -1;
  const MlaExtra ex{window, sinks, gate, gate_stride, (float)past_bytes};
  if (block_size % 8 || num_splits < 1 || num_splits > MLA_MAX_SPLITS) return -1;
  if (num_splits > 1 && (part_o == nullptr || part_ml == nullptr)) return -2;
  if (q_stride % 8 || out_stride % 4) return -5;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DT_BF16)
    return dispatch_mla<bf16_t>(DK, DV, kv_fp8, out, out_stride, part_o, part_ml, q, q_stride, k_cache, v_cache,
                                block_table, bt_stride, token_seq, seq_lens, scale, T_, Hq, block_size, num_splits,
                                mode, precise, ex, st);
  if (dtype == DT_F16)
    return dispatch_mla<f16_t>(DK, DV, kv_fp8, out, out_stride, part_o, part_ml, q, q_stride, k_cache, v_cache,
                               block_table, bt_stride, token_seq, seq_lens, scale, T_, Hq, block_size, num_splits,
                               mode, precise, ex, st);
  return -3;
}

// kv_fp8: the caches hold OCP e4m3 bytes (values saturated at +-448, scale 1) instead of elements of the model type.
VDAMD_API int vdamd_mla_cache_write(const void* x, long x_stride, void* k_cache, void* v_cache,
                                    const int* slot_mapping, int T_, int DK, int DV, int block_size, int dtype,
                                    int kv_fp8, void* stream) {
  if (T_ <= 0) return 0;
  if (block_size % 8 || DV % 16 || DV > DK) return -1;
  hipStream_t st = (hipStream_t)stream;
#define MLA_CW(T__, KV8__)                                                                                   \
  mla_cache_write_kernel<T__, KV8__><<<T_, 256, 0, st>>>((const T__*)x, x_stride, k_cache, v_cache, slot_mapping, \
                                                         DK, DV, block_size)
  if (dtype == DT_BF16) { if (kv_fp8) MLA_CW(bf16_t, true); else MLA_CW(bf16_t, false); }
  else if (dtype == DT_F16) { if (kv_fp8) MLA_CW(f16_t, true); else MLA_CW(f16_t, false); }
  else return -3;
#undef MLA_CW
  HIP_LAUNCH_CHECK();
  return 0;
}

// q_full[T][H][RANK + ROPE] and the latent cache rows of T tokens (see mla_prep_kernel).  q[T][H][nope + ROPE]
// with the given token / head strides; q_lat[H][T][RANK] with the given strides; latent[T][RANK + ROPE];
// slot_mapping may be null (no cache bound: only q_full is produced).
VDAMD_API int vdamd_mla_prep(void* q_full, const void* q, long q_tok_stride, int q_head_stride, int nope,
                             const void* q_lat, long q_lat_head_stride, long q_lat_tok_stride, const void* latent,
                             long latent_stride, const void* norm_w, float eps, const float* cos_sin,
                             const int* positions, void* k_cache, void* v_cache, const int* slot_mapping, int T_,
                             int H, int RANK, int ROPE, int block_size, int dtype, int kv_fp8, void* stream) {
  if (T_ <= 0) return 0;
  if (RANK % 16 || ROPE % 2 || (slot_mapping != nullptr && block_size % 8)) return -1;
  hipStream_t st = (hipStream_t)stream;
#define MLA_PREP(T__, KV8__)                                                                                     \
  mla_prep_kernel<T__, KV8__><<<T_, 256, 0, st>>>((T__*)q_full, (const T__*)q, q_tok_stride, q_head_stride, nope,  \
                                                  (const T__*)q_lat, q_lat_head_stride, q_lat_tok_stride,         \
                                                  (const T__*)latent, latent_stride, (const T__*)norm_w, eps,     \
                                                  cos_sin, positions, k_cache, v_cache, slot_mapping, H, RANK,    \
                                                  ROPE, block_size)
  if (dtype == DT_BF16) { if (kv_fp8) MLA_PREP(bf16_t, true); else MLA_PREP(bf16_t, false); }
  else if (dtype == DT_F16) { if (kv_fp8) MLA_PREP(f16_t, true); else MLA_PREP(f16_t, false); }
  else return -3;
#undef MLA_PREP
  HIP_LAUNCH_CHECK();
  return 0;
}
