// Prompt portions of the recurrent mixers in chunks of 64 rows on the matrix cores, values, products and sums of 32 bits, gfx950:
//
//   linear      S <- g S + k v^T ; o = S^T q                            (decayed linear attention, the state-space scan)
//   delta rule  S <- g S ; u = b (v - S^T k) ; S <- S + k u^T ; o = S^T q
//
// per (sequence, head), S [dim, vdim], with a decay g per head, or per head and key channel.  With b_i the product of the
// chunk's decays up to row i, S_0 the state in front of the chunk and G_ij the product of the decays behind row j up to
// row i, a chunk is
//   linear      o_i = (b_i q_i)^T S_0 + sum_(j <= i) A_ij v_j,  A_ij = q_i^T G_ij k_j ;  S = b_64 S_0 + sum_j (G_64,j k_j) v_j^T
//   delta rule  the same with u for v, where (I + diag(beta) L) u = diag(beta) (v - (b k)^T S_0), L_ij = k_i^T G_ij k_j (j < i):
//               u = U - W S_0 with U = T v and W = T (b k), T = (I + diag(beta) L)^-1 diag(beta), known without the state
//
//   chunk_prep  a workgroup per (chunk, head), all chunks at once: A, b q, G k, U and W (everything without S)
//   chunk_walk  a workgroup per (sequence, head, 32 value columns): the chunks one after the other, three products each
//
// The linear kinds come here where segment_scan.hip, which cuts sequences into segments that run side by side, is not ahead
// (segment_rows in ops/hip.py has the rule).  The walk row by row (delta_rule.hip, linear_latent.hip, state_space.hip) is bound by a
// chain of dependent steps per row; here the chain has a link per 64 rows and the sums are matrix instructions: A, L and the linear
// kinds' walk 16x16x4 fp32 ones (a fused multiply-add per term like the vector unit's: no input is narrowed), the delta rule's U, W
// and walk 16-bit ones on operands in three pieces (Thirds in chunk_parts.h).  Products of decays are formed directly, never as
// differences of logarithms: a product between two rows of different groups of 16 is (from the start of i's group up to i) * (whole groups
// between) * (behind j to the end of its group), each at most 1 where decays are, so nothing overflows; inside a group it
// is the quotient of two products from the group's start, unless one of those is smaller than 2^-96 or larger than 2^96,
// where the group's 120 pairs are multiplied out (diag_exact).  A head's products are formed so in 64 bits (2^-960, 2^960).
#include "chunk_parts.h"
#include <utility>

namespace {

constexpr int C = 64;                              // rows of a chunk

struct ChunkArgs {
  const void* x;                                   // [T, x_stride]: q, k, v of head 0 (group 0) at the three columns
  long x_stride;
  int q_off, k_off, v_off;
  const void* beta;                                // [T, beta_stride], raw (delta rule)
  long beta_stride;
  const void* dt;                                  // [T, dt_stride], raw (state space, delta rule)
  long dt_stride;
  const float* dt_bias;
  const float* a_log;
  const float* decay;                              // [H] (LINEAR_HEAD) or [T, H * dim] (LINEAR_CHANNEL)
  float* ws;                                       // per (chunk, head of the launch): A | b q | G k, transposed | b_64 | U,
                                                   // transposed | -W
  long ws_stride;
  const int* qsl;
  int B, H, G, dim, vdim, VP;                      // VP: vdim up to a multiple of 32
  int h0, nh;                                      // the launch's heads
  int silu, vec, vvec;                             // rows of q, k and the decays / of v can be read 16 bytes at a time
  float eps;
};

// What crosses from one kernel to the other lies in pieces of 16x16 as the matrix instruction's operands: 64 lanes of four
// floats, (lane % 16, 4 (lane / 16) + e) = (row, reduction index) of a left operand, (column, row) of U: a wave's load is one
// run of 1 KB.  A[4][4] and b q, -W [4][KB] by (rows, reduction); G k, transposed, [KB][4]; U [tiles][4] by (columns, rows).
struct Layout { int q, kt, bc, u, w, total; };
__device__ __forceinline__ int piece(int index, int lane) { return (index * 64 + lane) * 4; }
__host__ __device__ constexpr Layout layout_of(int DP, int VP, bool delta) {
  Layout l{};
  l.q = C * C;
  l.kt = l.q + C * DP;
  l.bc = l.kt + DP * C;
  l.u = l.bc + DP;
  l.w = l.u + VP * C;
  l.total = l.w + (delta ? C * DP : 0);
  return l;
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The product over 16 reduction indices.  Every product here is summed up in such pieces, each from zero, that are then
// added in turns to two sums: one accumulator running through 192 terms loses twice the digits that the row by row kernels
// lose (relative error in norm of the delta rule's output against 64 bits 4.1e-7; so 2.2e-7, row by row 2.2e-7).  What the
// outputs are sums of (A, and o itself) comes in halves of eight: ten prompts of 450 to 4265 rows under the delta rule per head
// are then 1.00 times as far off as row by row on average (1.05 without, 1.07 with the decays in A's factors as well), for
// 1 to 2 % of the time (55.0 -> 56.2 us on average, 8017 rows per channel 403 -> 409); in u and the state it would cost 5 %.
__device__ __forceinline__ f32x4 dot16(f32x4 a, f32x4 b) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  return mfma4(a[1], b[1], mfma4(a[0], b[0], zero)) + mfma4(a[3], b[3], mfma4(a[2], b[2], zero));
}

// N such products side by side: a matrix instruction of these takes 32 cycles and its result another few, which the others fill
template <int N, bool HALVES = false> __device__ __forceinline__ void dots16(const f32x4* const (&a)[N], const f32x4* const (&b)[N], f32x4 (&c)[N]) {
  f32x4 d[N];
#pragma unroll
  for (int i = 0; i < N; ++i) c[i] = d[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      f32x4& to = HALVES && e >= 2 ? d[i] : c[i];
      to = mfma4((*a[i])[e], (*b[i])[e], to);
    }
  if constexpr (HALVES)
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] += d[i];
}

// 0, or NaN where v has an infinity or a NaN
__device__ __forceinline__ float not_finite(f32x4 v, float so_far) {
#pragma unroll
  for (int e = 0; e < 4; ++e) so_far = fmaf(v[e], 0.f, so_far);
  return so_far;
}
// A lower triangular block (left(i, j / 4, j % 4)) times a right operand with an infinity or a NaN in it.  In the matrix
// instruction the zeros right of the diagonal would meet it and hand it to the rows in front of its own; here they are left out.
template <typename F> __device__ __forceinline__ f32x4 lower16(F&& left, f32x4 x) {
  const int lane = threadIdx.x & 63, lr = lane & 15, kh = lane >> 4;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1                                   // (rare: few registers)
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const float xj = __shfl(x[f], g * 16 + lr, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float l = left(4 * kh + e, g, f);
        if (4 * g + f <= 4 * kh + e) o[e] += l * xj;
      }
    }
  return o;
}

// p[0 .. 3], `fill` from `left` on
template <typename T> __device__ __forceinline__ f32x4 ld4(const T* p, int left, float fill) {
  f32x4 o = {fill, fill, fill, fill};
#pragma unroll
  for (int e = 0; e < 4; ++e) if (e < left) o[e] = ldf(p + e);
  return o;
}

// Sixteen rows of a wave, `cols` values each, on their way into LDS: a row is read by neighbouring lanes, 16 bytes each, whole
// lines at a time (read as operands, four lanes to a row, every line is asked for again while it is on its way: the kernel then
// spends 65 % of its time in such stalls of the vector cache).
template <typename T, int DP> struct RowLoad {
  static constexpr int N = 16 / (int)sizeof(T), PER = DP / N, ROWS = 64 / PER, NI = 16 / ROWS;
  typedef T Vec __attribute__((ext_vector_type(N)));
  Vec v[NI];
  // rows first .. first + valid - 1 of p exist; lanes past `cols` and rows past `valid` get `fill`
  __device__ __forceinline__ void fetch(const T* p, long stride, int valid, int cols, float fill) {
    const int lane = threadIdx.x & 63, j = (lane % PER) * N;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int rr = i * ROWS + lane / PER;
      if (rr < valid && j < cols) v[i] = *reinterpret_cast<const Vec*>(p + (long)rr * stride + j);
      else
#pragma unroll
        for (int e = 0; e < N; ++e) v[i][e] = (T)fill;
    }
  }
  __device__ __forceinline__ void stash(float* dst, int ld) const {
    const int lane = threadIdx.x & 63, j = (lane % PER) * N;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float* d = dst + (i * ROWS + lane / PER) * ld + j;
#pragma unroll
      for (int e = 0; e < N; e += 4)
        *reinterpret_cast<f32x4*>(d + e) = f32x4{(float)v[i][e], (float)v[i][e + 1], (float)v[i][e + 2], (float)v[i][e + 3]};
    }
  }
};
// between one wave's LDS writes and its other lanes' reads of them (a wave's LDS accesses are carried out in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int chunks_of(const int* qsl, int B, int s) {
  const int n = s < B ? qsl[s + 1] - qsl[s] : 0;
  return n > 0 ? (n + C - 1) / C : 0;
}

__device__ __forceinline__ int chunks_before(const int* qsl, int B, int seq) {
  const int lane = threadIdx.x & 63;
  int sum = 0;
  for (int s0 = 0; s0 < seq; s0 += 64) sum += s0 + lane < seq ? chunks_of(qsl, B, s0 + lane) : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  return sum;
}

// grid (bound on the batch's chunks, heads of the launch), 4 waves; wave w has rows 16 w .. 16 w + 15 of the chunk: lane (kh =
// lane / 16, lane % 16) holds channels 16 kb + 4 kh + e of row lane % 16 in registers, which is at once the left operand
// (row, reduction index 4 kh + e) and the right one of the matrix instruction and the lane layout of the products
// over rows (DPP).  Only G k and, for U and W, M, its inverse and b k cross waves, through LDS.
// Bound by what it writes (112 KB per chunk and head, the delta rule 144: linear attention's 6007 rows x 16 heads, 170 MB,
// in 67 us) and, under the delta rule, by instructions: of 65 000 cycles of a workgroup, two to a compute unit, 14 000 wait for its
// rows, 16 000 go into A and L of the last 16 rows, 17 000 into U, W and the inverse, 8 000 into norms and running products (16 heads,
// 8017 rows, a decay per channel).  There 150 us; 195 with the library's exponentials and logarithm (a third of its instructions)
// and with U and W by substitution in fp32, W stored as it left the accumulators, four bytes a lane.
// 64 keys: three workgroups to a compute unit, which takes 168 registers; with the 172 that the compiler likes best a decay per head
// has two, 3736 rows of 32 heads 82 us, now 71 (fp32 rows would not fit, and keep two).
template <typename T, int KIND, int DP>
__global__ __launch_bounds__(256, DP > 64 || sizeof(T) == 4 ? 2 : 3) void chunk_prep_kernel(ChunkArgs a) {
  constexpr bool DELTA = KIND >= DELTA_CHANNEL, CHAN = KIND == LINEAR_CHANNEL || KIND == DELTA_CHANNEL;
  constexpr int KB = DP / 16, NP = CHAN ? KB * 4 : 1, LD = DP + 4, LM = C + 4, LT = C + 8;
  constexpr Layout L0 = layout_of(DP, 0, false);
  __shared__ __attribute__((aligned(16))) float ks[C * LD];
  __shared__ __attribute__((aligned(16))) float tl[CHAN ? 4 * DP : 4];
  // -beta L, and in its place the thirds of (I + beta L)^-1 beta
  __shared__ __attribute__((aligned(16))) union { float l[DELTA ? C * LM : 4]; bf16_t t[3][DELTA ? C * LT : 8]; } m;
  float* const mn = m.l;
  __shared__ __attribute__((aligned(16))) float ti[DELTA ? 4 * 16 * 20 : 4]; // inverses of the diagonal blocks
  __shared__ float bl[C];
  __shared__ double td[4], sd[CHAN ? 1 : C];       // per head: products of whole groups, and of the group's decays behind a row
  int seq, c;
  if (!locate(a.B, blockIdx.x, seq, c, [&](int i) { return chunks_of(a.qsl, a.B, i); })) return;           // (the same for every wave)
  const int hh = blockIdx.y, h = a.h0 + hh, g = h / (a.H / a.G);
  const int q0 = a.qsl[seq], n = a.qsl[seq + 1] - q0;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, kh = lane >> 4;
  const int r = 16 * wave + lr;
  const bool ok = c * C + r < n;
  const long row = q0 + (ok ? c * C + r : 0);
  const T* xr = (const T*)a.x + row * a.x_stride;
  float* ws = a.ws + ((long)hh * gridDim.x + blockIdx.x) * a.ws_stride;   // (a head's chunks side by side: the walk stays in a page)

  // ---- the wave's rows: q, k, the decays
  f32x4 q[KB], k[KB], dk[CHAN ? KB : 1];           // dk: the row's decays (raw dt for the delta rule, until below)
  float p[NP], s[NP];
  // (all on their way at once: loaded where they are used, under the condition there, each was waited for by itself)
  [[maybe_unused]] float bias[KIND == DELTA_CHANNEL ? 4 * KB : 1];
  if constexpr (KIND == DELTA_CHANNEL)
#pragma unroll
    for (int i = 0; i < 4 * KB; ++i) bias[i] = a.dt_bias[h * a.dim + min(16 * (i / 4) + 4 * kh + i % 4, a.dim - 1)];
  [[maybe_unused]] const float raw_beta = DELTA ? ldf((const T*)a.beta + row * a.beta_stride + h) : 0.f;
  const int valid = min(16, n - (c * C + 16 * wave));            // rows of the wave that exist (none: <= 0)
  const long row0 = q0 + c * C + 16 * wave;
  float* mine = ks + 16 * wave * LD;               // the wave's rows of ks, free until it writes G k there
  const float* fr = mine + lr * LD + 4 * kh;
  if (a.vec) {
    RowLoad<T, DP> lq, lk;
    lq.fetch((const T*)a.x + row0 * a.x_stride + a.q_off + (long)g * a.dim, a.x_stride, valid, a.dim, 0.f);
    lk.fetch((const T*)a.x + row0 * a.x_stride + a.k_off + (long)g * a.dim, a.x_stride, valid, a.dim, 0.f);
    using D = std::conditional_t<KIND == LINEAR_CHANNEL, float, T>;
    RowLoad<D, DP> ld;
    if constexpr (KIND == LINEAR_CHANNEL)
      ld.fetch(a.decay + (row0 * a.H + h) * (long)a.dim, (long)a.H * a.dim, valid, a.dim, 1.f);
    else if constexpr (KIND == DELTA_CHANNEL)
      ld.fetch((const T*)a.dt + row0 * a.dt_stride + (long)h * a.dim, a.dt_stride, valid, a.dim, 0.f);
    lq.stash(mine, LD);
    wave_sync();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) q[kb] = *reinterpret_cast<const f32x4*>(fr + 16 * kb);
    wave_sync();
    lk.stash(mine, LD);
    wave_sync();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) k[kb] = *reinterpret_cast<const f32x4*>(fr + 16 * kb);
    if constexpr (CHAN) {
      wave_sync();
      ld.stash(mine, LD);
      wave_sync();
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) dk[kb] = *reinterpret_cast<const f32x4*>(fr + 16 * kb);
    }
    wave_sync();
  } else {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int j = 16 * kb + 4 * kh, left = ok ? a.dim - j : 0;
      q[kb] = ld4(xr + a.q_off + (long)g * a.dim + j, left, 0.f);
      k[kb] = ld4(xr + a.k_off + (long)g * a.dim + j, left, 0.f);
      if constexpr (KIND == LINEAR_CHANNEL) dk[kb] = ld4(a.decay + (row * a.H + h) * (long)a.dim + j, left, 1.f);
      if constexpr (KIND == DELTA_CHANNEL) dk[kb] = ld4((const T*)a.dt + row * a.dt_stride + (long)h * a.dim + j, left, 0.f);
    }
  }
  if (a.silu) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) { q[kb][e] *= sigmoid_f(q[kb][e]); k[kb][e] *= sigmoid_f(k[kb][e]); }
  }
  if constexpr (KIND == DELTA_CHANNEL) {
    const float rate = expf(a.a_log[h]);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float decay = decay_f(dk[kb][e] + bias[4 * kb + e], rate);
        dk[kb][e] = ok && 16 * kb + 4 * kh + e < a.dim ? decay : 1.f;
      }
  }
  if constexpr (DELTA) {
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) { sq += q[kb][e] * q[kb][e]; sk += k[kb][e] * k[kb][e]; }
    sq += __shfl_xor(sq, 16, 64); sk += __shfl_xor(sk, 16, 64);
    sq += __shfl_xor(sq, 32, 64); sk += __shfl_xor(sk, 32, 64);
    const float iq = 1.0f / sqrtf(sq + a.eps) * (1.0f / sqrtf((float)a.dim)), ik = 1.0f / sqrtf(sk + a.eps);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) { q[kb][e] *= iq; k[kb][e] *= ik; }
    if (kh == 0) bl[r] = ok ? sigmoid_f(raw_beta) : 0.f;
  }
  float own = 1.f;                                 // per head: the row's decay,
  double pd = 1.0, after = 1.0;                    // the products of the group's up to the row, and behind it
  if constexpr (CHAN) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * kb + e] = dk[kb][e];
      prefix_products(p[4 * kb], p[4 * kb + 1], p[4 * kb + 2], p[4 * kb + 3]);
      suffix_products(dk[kb], s[4 * kb], s[4 * kb + 1], s[4 * kb + 2], s[4 * kb + 3]);
    }
  } else {
    if (ok) {
      if constexpr (KIND == LINEAR_HEAD) own = a.decay[h];
      else {
        const float step = softplus_f(ldf((const T*)a.dt + row * a.dt_stride + h) + a.dt_bias[h]);
        own = expf(-expf(a.a_log[h]) * step);
        if constexpr (KIND == STATE_SPACE) {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) k[kb] *= step;
        }
      }
    }
    // (a head's decay can be the same number in every row: rounded products of it would be off by the same amount in every
    // chunk.  They are formed in 64 bits, and A and L take the one between their rows, rounded once, behind their sums; with
    // decays in the factors, which rounds each term twice, the error against 64 bits was up to 1.25 times the walk's)
    after = __shfl_down((double)own, 1, 16);
    if (lr == 15) after = 1.0;
    pd = own;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const double before = __shfl_up(pd, o, 16), behind = __shfl_down(after, o, 16);
      if (lr >= o) pd *= before;
      if (lr + o < 16) after *= behind;
    }
    if (lane == 15) td[wave] = pd;
    if (kh == 0) sd[r] = after;
  }
  bool far = false;                                // a product too small or too large to divide by
  if constexpr (CHAN) {
    unsigned beyond = 0;
#pragma unroll
    for (int i = 0; i < NP; ++i) beyond = max(beyond, (bits(p[i]) << 1) - 0x1f000000u);
    far = beyond > 0xc0000000u;                    // (an exponent outside -96 .. 96, infinities and NaN among them)
  } else {
    far = !(fabs(pd) >= 0x1p-960 && fabs(pd) <= 0x1p960);
  }
  if (lr == 15) {
    if constexpr (CHAN) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        *reinterpret_cast<f32x4*>(tl + wave * DP + 16 * kb + 4 * kh) = f32x4{p[4 * kb], p[4 * kb + 1], p[4 * kb + 2], p[4 * kb + 3]};
    }
  }
  [[maybe_unused]] auto P = [&](int kb, int e) { return p[CHAN ? 4 * kb + e : 0]; };
  // per head: the products of the group's decays up to the rows of a lane's accumulator
  [[maybe_unused]] double pr[4];
  if constexpr (!CHAN)
#pragma unroll
    for (int e = 0; e < 4; ++e) pr[e] = __shfl(pd, 4 * kh + e, 16);
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    f32x4 v = k[kb];
    if constexpr (CHAN)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= s[4 * kb + e];
    *reinterpret_cast<f32x4*>(ks + r * LD + 16 * kb + 4 * kh) = v;
  }
  __syncthreads();
  // G k up to the chunk's end, transposed: the wave's rows, a piece per 16 channels
  {
    [[maybe_unused]] float end[4];                 // per head: the products of the decays behind those rows
    if constexpr (!CHAN) {
      double behind = 1.0;
      for (int b = wave + 1; b < 4; ++b) behind *= td[b];
#pragma unroll
      for (int e = 0; e < 4; ++e) end[e] = (float)(sd[16 * wave + 4 * kh + e] * behind);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float groups = 1.f;
      if constexpr (CHAN)
        for (int b = wave + 1; b < 4; ++b) groups *= tl[b * DP + 16 * kb + lr];
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ks[(16 * wave + 4 * kh + e) * LD + 16 * kb + lr] * (CHAN ? groups : end[e]);
      *reinterpret_cast<f32x4*>(ws + L0.kt + piece(kb * 4 + wave, lane)) = v;
    }
    if ((int)threadIdx.x < DP) {
      const int j = threadIdx.x;
      ws[L0.bc + j] = CHAN ? tl[j] * tl[DP + j] * tl[2 * DP + j] * tl[3 * DP + j] : (float)(td[0] * td[1] * td[2] * td[3]);
    }
  }
  // ---- A = q G k and (delta) L = k G k, lower triangles: the wave's rows against the column blocks 0 .. wave
  const bool exact_diag = __any(far);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 da = zero, dl = zero;
  if (!exact_diag) {
    f32x4 sa[2] = {zero, zero}, sb[2] = {zero, zero};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      f32x4 kd = k[kb];
      if constexpr (CHAN)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          kd[e] = quotient(kd[e], P(kb, e));
          q[kb][e] *= P(kb, e);
          k[kb][e] *= P(kb, e);
        }
      sa[kb & 1] += dot16(q[kb], kd);
      if constexpr (DELTA) sb[kb & 1] += dot16(k[kb], kd);
    }
    da = sa[0] + sa[1];
    dl = sb[0] + sb[1];
    if constexpr (!CHAN) {
      const double over = 1.0 / pd;
#pragma unroll
      for (int e = 0; e < 4; ++e) { da[e] *= (float)(pr[e] * over); dl[e] *= (float)(pr[e] * over); }
    }
  } else {
    // diag_exact: pairs (i, i - m) of the wave's group; the product of the decays between them grows with m.  The rows i - m and
    // their decays come by turning the 16 lanes on by one each time, in registers: wave shuffles, which go through LDS, made this
    // a third of such a call's time (16 heads, dim 128, decays of 3e-4 a row: 8017 rows of the delta rule 545 us so, 445 turned,
    // 421 where no group comes here; 60 rows of 8 heads 79, 54 and 46).
    float pa[16], pb[16], between = 1.f, oj = own;
#pragma unroll
    for (int m = 0; m < 16; ++m) pa[m] = pb[m] = 0.f;
    [[maybe_unused]] float by_row[CHAN ? 1 : 16];
    if constexpr (!CHAN)
#pragma unroll
      for (int m = 0; m < 16; ++m) { by_row[m] = between; between *= oj; oj = turn(oj); }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float kj = k[kb][e], dj = dk[CHAN ? kb : 0][e];
        between = 1.f;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          const float kd = kj * (CHAN ? between : by_row[CHAN ? 0 : m]);
          pa[m] += q[kb][e] * kd;
          if constexpr (DELTA) pb[m] += k[kb][e] * kd;
          kj = turn(kj);
          if constexpr (CHAN) { between *= dj; dj = turn(dj); }
        }
      }
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      float sa = pa[m], sb = pb[m];
      sa += __shfl_xor(sa, 16, 64); sa += __shfl_xor(sa, 32, 64);
      sb += __shfl_xor(sb, 16, 64); sb += __shfl_xor(sb, 32, 64);
      // lane (.., i) has the sum of row i, column i - m; as an accumulator, lane (kh, j) has rows 4 kh + e of column j
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float va = __shfl(sa, 4 * kh + e, 64), vb = __shfl(sb, 4 * kh + e, 64);
        if (4 * kh + e - m == lr) { da[e] = va; dl[e] = vb; }
      }
    }
    if constexpr (CHAN)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) { q[kb][e] *= P(kb, e); k[kb][e] *= P(kb, e); }
  }
  // (blocks to the left, nearest first: after each of them its whole product joins the left operands, which end as b q and b k)
  double whole = 1.0;                              // per head: of the groups between
  for (int J = wave - 1; J >= 0; --J) {
    f32x4 sa[2] = {zero, zero}, sb[2] = {zero, zero};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(ks + (16 * J + lr) * LD + 16 * kb + 4 * kh);
      sa[kb & 1] += dot16(q[kb], b);
      if constexpr (DELTA) sb[kb & 1] += dot16(k[kb], b);
      if constexpr (CHAN) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(tl + J * DP + 16 * kb + 4 * kh);
        q[kb] *= t;
        k[kb] *= t;
      }
    }
    f32x4 va = sa[0] + sa[1], vl = sb[0] + sb[1];
    if constexpr (!CHAN) {
      const double left = whole * sd[16 * J + lr];
#pragma unroll
      for (int e = 0; e < 4; ++e) { va[e] *= (float)(pr[e] * left); vl[e] *= (float)(pr[e] * left); }
      whole *= td[J];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 16 * wave + 4 * kh + e;
      ws[piece(wave * 4 + J, (lr >> 2) * 16 + 4 * kh + e) + (lr & 3)] = va[e];
      if constexpr (DELTA) mn[i * LM + 16 * J + lr] = -bl[i] * vl[e];
    }
  }
  if constexpr (!CHAN)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) { q[kb] *= (float)(pd * whole); k[kb] *= (float)(pd * whole); }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = 4 * kh + e;
    ws[piece(wave * 5, (lr >> 2) * 16 + i) + (lr & 3)] = lr <= i ? da[e] : 0.f;
    if constexpr (DELTA) mn[(16 * wave + i) * LM + 16 * wave + lr] = lr < i ? -bl[16 * wave + i] * dl[e] : 0.f;
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) *reinterpret_cast<f32x4*>(ws + L0.q + piece(wave * KB + kb, lane)) = q[kb];

  const int vt = a.VP / 16;
  const T* xv = (const T*)a.x + row0 * a.x_stride + a.v_off + (long)h * a.vdim;
  // columns v0 .. v0 + DP - 1 of the wave's rows of v into its rows of ks
  auto values = [&](int v0) {
    if (a.vvec) {
      RowLoad<T, DP> lv;
      lv.fetch(xv + v0, a.x_stride, valid, a.vdim - v0, 0.f);
      lv.stash(mine, LD);
    } else {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int j = 16 * kb + 4 * kh;
        *reinterpret_cast<f32x4*>(mine + lr * LD + j) = ld4(xv + (long)lr * a.x_stride + v0 + j, lr < valid ? a.vdim - v0 - j : 0, 0.f);
      }
    }
  };
  if constexpr (!DELTA) {
    __syncthreads();                               // G k has been read
    for (int t0 = 0; t0 < vt; t0 += KB) {
      values(16 * t0);
      wave_sync();
#pragma unroll
      for (int t = 0; t < KB; ++t)
        if (t0 + t < vt) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = mine[(4 * kh + e) * LD + 16 * t + lr];
            if (a.silu) v[e] *= sigmoid_f(v[e]);
          }
          *reinterpret_cast<f32x4*>(ws + L0.u + piece((t0 + t) * 4 + wave, lane)) = v;
        }
      wave_sync();
    }
  } else {
    __syncthreads();                               // G k has been read, M is there
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) *reinterpret_cast<f32x4*>(ks + r * LD + 16 * kb + 4 * kh) = k[kb];
    // (I - Mn)^-1 of the wave's diagonal block: lane lr a column, row by row
    {
      float t[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float* m = mn + (16 * wave + i) * LM + 16 * wave;
        float v = i == lr ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) v += m[j] * t[j];
        t[i] = v;
      }
      if (kh == 0)
#pragma unroll
        for (int i = 0; i < 16; ++i) ti[(16 * wave + i) * 20 + lr] = t[i];
    }
    RowLoad<T, DP> lv;                             // the first columns of v, on their way
    if (a.vvec) lv.fetch(xv, a.x_stride, valid, a.vdim, 0.f);
    __syncthreads();
    // the rest of the inverse: a wave 16 columns, block by block; an accumulator's layout is the right operand's
    f32x4 X[4], below[4][3], own_block[4];          // (all read at once: one by one, each is waited for in the chain)
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      own_block[I] = *reinterpret_cast<const f32x4*>(ti + (16 * I + lr) * 20 + 4 * kh);
#pragma unroll
      for (int J = 0; J < I; ++J) below[I][J] = *reinterpret_cast<const f32x4*>(mn + (16 * I + lr) * LM + 16 * J + 4 * kh);
    }
    auto rest = [&](auto apart) {
#pragma unroll
      for (int I = 0; I < 4; ++I) {
        X[I] = zero;
        if (I == wave)
#pragma unroll
          for (int e = 0; e < 4; ++e) X[I][e] = ti[(16 * I + 4 * kh + e) * 20 + lr];
        if (I > wave) {
          f32x4 acc = zero;
#pragma unroll
          for (int J = 0; J < I; ++J)
            if (J >= wave) acc += dot16(below[I][J], X[J]);
          if constexpr (apart) X[I] = lower16([&](int i, int g, int f) { return ti[(16 * I + i) * 20 + 4 * g + f]; }, acc);
          else X[I] = dot16(own_block[I], acc);
        }
      }
    };
    rest(std::false_type{});
    if (__builtin_expect(__any(not_finite(X[3], not_finite(X[2], not_finite(X[1], 0.f))) != 0.f), 0)) rest(std::true_type{});
    const float beta = bl[16 * wave + lr];
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int e = 0; e < 4; ++e) X[I][e] = I > wave || (I == wave && 4 * kh + e >= lr) ? X[I][e] * beta : 0.f;
    __syncthreads();                               // M has been read
#pragma unroll
    for (int I = 0; I < 4; I += 2)
      store_columns<LT, false, 8>(m.t, 16 * I + 4 * kh, 16 * wave + lr, thirds<false>(X[I], X[I + 1]), 16 * (I + 1) + 4 * kh);
    __syncthreads();
    // rows 32 s .. of the columns 16 t .. in ks
    auto column = [&](int t, int s) {
      f32x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = ks[(32 * s + 8 * kh + e) * LD + 16 * t + lr];
        hi[e] = ks[(32 * s + 8 * kh + 4 + e) * LD + 16 * t + lr];
      }
      return std::pair<f32x4, f32x4>(lo, hi);
    };
    auto inverse = [&](int I, int s) { return load_third<8, false>(m.t, (16 * I + lr) * LT + 32 * s + 8 * kh); };
    // term by term, where something is not finite: a zero of the inverse would hand it to the rows in front
    auto apart = [&](int i, int col) {
      float o = 0.f;
#pragma unroll 1
      for (int j = 0; j <= i; ++j) {
        const float h = (float)m.t[0][i * LT + j], sum = h + ((float)m.t[1][i * LT + j] + (float)m.t[2][i * LT + j]);
        o += (sum != sum ? h : sum) * ks[j * LD + col];
      }
      return o;
    };
    // W, transposed (keys by rows: the layout of a left operand as it leaves the accumulator), of 16 keys at a time
    float* wp = ws + L0.u + a.VP * C;
    for (int t = wave; t < KB; t += 4) {
      Thirds keys[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const auto k2 = column(t, s);
        keys[s] = thirds<false>(k2.first, k2.second);
      }
      Sum sum[4] = {};
#pragma unroll
      for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int s = 0; s <= I / 2; ++s) {
          const Thirds rows[1] = {inverse(I, s)};
          products<false, false>(keys[s], rows, *reinterpret_cast<Sum(*)[1]>(&sum[I]));
        }
      f32x4 w[4];
      float odd = 0.f;
#pragma unroll
      for (int I = 0; I < 4; ++I) {
        w[I] = sum[I].h + sum[I].s;
        odd = not_finite(w[I], odd);
      }
      if (__builtin_expect(__any(odd != 0.f), 0))
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
          for (int e = 0; e < 4; ++e) w[I][e] = apart(16 * I + lr, 16 * t + 4 * kh + e);
#pragma unroll
      for (int I = 0; I < 4; ++I) *reinterpret_cast<f32x4*>(wp + piece(I * KB + t, lane)) = -w[I];
    }
    // U, of 16 columns at a time
    for (int t0 = 0; t0 < vt; t0 += KB) {
      __syncthreads();                             // the other waves have read what is there
      if (a.vvec && t0 == 0) lv.stash(mine, LD);
      else values(16 * t0);
      __syncthreads();
      for (int t = wave; t < KB && t0 + t < vt; t += 4) {
        constexpr bool V16 = std::is_same_v<T, bf16_t>;
        Thirds v[2][1];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const auto v2 = column(t, s);
          if constexpr (V16) v[s][0].h = upper(v2.first, v2.second);
          else v[s][0] = thirds<false>(v2.first, v2.second);
        }
        Sum sum[4] = {};
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
          for (int s = 0; s <= I / 2; ++s) products<false, V16>(inverse(I, s), v[s], *reinterpret_cast<Sum(*)[1]>(&sum[I]));
        f32x4 u[4];
        float odd = 0.f;
#pragma unroll
        for (int I = 0; I < 4; ++I) {
          u[I] = sum[I].h + sum[I].s;
          odd = not_finite(u[I], odd);
        }
        if (__builtin_expect(__any(odd != 0.f), 0))
#pragma unroll
          for (int I = 0; I < 4; ++I)
#pragma unroll
            for (int e = 0; e < 4; ++e) u[I][e] = apart(16 * I + 4 * kh + e, 16 * t + lr);
#pragma unroll
        for (int I = 0; I < 4; ++I) *reinterpret_cast<f32x4*>(ws + L0.u + piece((t0 + t) * 4 + I, lane)) = u[I];
      }
    }
  }
}

// grid: (sequence, head) pairs x tiles of 32 value columns, the tiles of a pair on one die (workgroups go round the dies by
// their index: they share what chunk_prep left in its L2), long sequences first.  Eight waves: 0 .. 3 keep rows
// w * DP / 4 .. of the state tile as accumulators and carry it from chunk to chunk, 4 .. 7 form the output of 16 rows of the
// chunk each, so that two waves per SIMD fill each other's waits.  Per chunk
//   state waves    (delta rule) u = U - W S, S of the whole tile from LDS ;  S = b_64 S + (G k)^T u
//   output waves   o = (b q) S + A u
// with two barriers (S is there, u is there), linear kinds with one (u = v comes from memory).  Left operands come from
// memory straight into registers, where the next chunk's take the place of those just used.
// Bound by the chain of a chunk: its matrix instructions (1.1 us of linear kinds at 16 columns, the delta rule 0.6 and as much
// again to split its operands) and its 90 - 115 KB of operands (0.6 - 0.95 us at the 119 - 143 KB per us that a compute unit takes
// from the L2 through its vector cache, about 64 bytes a clock; 45 - 61 KB per us of what comes from the memory-side cache) hardly
// overlap, as all waves wait at the same barriers.  Measured per chunk and workgroup 2.5 / 3.0 us at 16 columns, 4.0 / 3.8 at 32 (the delta
// rule in fp32: 3.5 and 5.0; five prompts of 8017 rows, 16 heads: 221 against 177 us).
template <int DP, int NC> struct LinearWalk {
  static constexpr int KB = DP / 16, NT = DP / 64, LD = DP + 4;
  static constexpr Layout L0 = layout_of(DP, 0, false);
  struct Shared {
    __attribute__((aligned(16))) float sl[2][16 * NC * LD];
  };
  static __device__ __forceinline__ f32x4 at(const float* p, int offset) { return *reinterpret_cast<const f32x4*>(p + offset); }

  const float* ws;                                 // the pair's first chunk
  long step;
  int nc, VP, tile, wave, lane, lr, kh;
  Shared& sh;

  // (chunks past the last are read as the last one: loads without a condition keep the waits for them exact)
  __device__ __forceinline__ const float* chunk_at(int c) const { return ws + step * min(c, nc - 1); }
  __device__ __forceinline__ f32x4 left(const float* p, int offset, int index) const { return at(p, offset + piece(index, lane)); }

  struct StateOps { f32x4 k[NT][4], u[4][NC], b[NT]; };
  struct OutOps { f32x4 q[KB], a[4], u[4][NC]; };

  __device__ __forceinline__ void load_first(StateOps&, int) const {}
  template <typename Ops> __device__ __forceinline__ void load_values(Ops& r, const float* p) const {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) r.u[kb][ct] = left(p, L0.u, (NC * tile + ct) * 4 + kb);
  }
  __device__ __forceinline__ void load_second(StateOps& r, int c) const {
    const float* p = chunk_at(c);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) r.k[t][kb] = left(p, L0.kt, (wave * NT + t) * 4 + kb);
      r.b[t] = at(p, L0.bc + (wave * NT + t) * 16 + 4 * kh);
    }
    load_values(r, p);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void load_first(OutOps& r, int c) const {
    const float* p = chunk_at(c);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) r.q[kb] = left(p, L0.q, wave * KB + kb);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void load_second(OutOps& r, int c) const {
    const float* p = chunk_at(c);
    // (the blocks right of the diagonal are never written: they are read, so that the loads carry no condition, and not used)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) r.a[kb] = left(p, 0, wave * 4 + kb);
    load_values(r, p);
    __builtin_amdgcn_sched_barrier(0);
  }
  // o[ct][0 / 1] += the products of left operands l[0 .. 3] with right ones x[0 .. 3][ct], four chains of instructions side by side
  template <bool HALVES> static __device__ __forceinline__ void four(const f32x4* l, const f32x4 (&x)[4][NC], f32x4 (&o)[NC][2]) {
    if constexpr (NC == 1) {
      f32x4 d[4];
      dots16<4, HALVES>({&l[0], &l[1], &l[2], &l[3]}, {&x[0][0], &x[1][0], &x[2][0], &x[3][0]}, d);
      o[0][0] += d[0] + d[1];
      o[0][1] += d[2] + d[3];
    } else {
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        f32x4 d[4];
        dots16<4, HALVES>({&l[i], &l[i], &l[i + 1], &l[i + 1]}, {&x[i][0], &x[i][1], &x[i + 1][0], &x[i + 1][1]}, d);
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) o[ct][i >> 1] += d[ct] + d[2 + ct];
      }
    }
  }
  // reduction blocks kb .. kb + 3 of a right operand in LDS
  template <int LDR> __device__ __forceinline__ void read_four(const float* right, int kb, f32x4 (&x)[4][NC]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) x[i][ct] = at(right, (16 * ct + lr) * LDR + 16 * (kb + i) + 4 * kh);
  }

  __device__ __forceinline__ void chunk(StateOps& r, int c, f32x4 (&S)[NT][NC]) const {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    float* sl = sh.sl[c & 1];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct)
        *reinterpret_cast<f32x4*>(sl + (16 * ct + lr) * LD + (wave * NT + t) * 16 + 4 * kh) = S[t][ct];
    __syncthreads();
    f32x4 x[4][NC];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) x[i][ct] = r.u[i][ct];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 add[NC][2];
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) add[ct][0] = add[ct][1] = zero;
      four<false>(r.k[t], x, add);
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) S[t][ct] = S[t][ct] * r.b[t] + (add[ct][0] + add[ct][1]);
    }
    load_second(r, c + 1);
  }
  // o of the wave's 16 rows; u: those rows of v
  __device__ __forceinline__ void chunk(OutOps& r, int c, f32x4 (&o)[NC], f32x4 (&u)[NC]) const {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const float* sl = sh.sl[c & 1];
    __syncthreads();
    f32x4 os[NC][2], x[4][NC];
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) os[ct][0] = os[ct][1] = zero;
#pragma unroll
    for (int kb = 0; kb < KB; kb += 4) {
      read_four<LD>(sl, kb, x);
      four<true>(&r.q[kb], x, os);
    }
    load_first(r, c + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) {
        x[i][ct] = r.u[i][ct];
        if (i == wave) u[ct] = r.u[i][ct];
      }
    // (the lower triangle's blocks; the wave's number is the same for all its lanes)
    float odd = 0.f;                               // u of the wave's own rows, which the block on the diagonal meets
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) odd = not_finite(u[ct], odd);
    if (__builtin_expect(__any(odd != 0.f), 0)) {
      f32x4 own, u_own[NC];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < wave)
#pragma unroll
          for (int ct = 0; ct < NC; ++ct) os[ct][i & 1] += dot16(r.a[i], x[i][ct]);
        if (i == wave) {
          own = r.a[i];
#pragma unroll
          for (int ct = 0; ct < NC; ++ct) u_own[ct] = x[i][ct];
        }
      }
#pragma unroll
      for (int ct = 0; ct < NC; ++ct)
        os[ct][0] += lower16([&](int i, int g, int f) { return __shfl(own[f], g * 16 + i, 64); }, u_own[ct]);
    } else if (wave == 3) {
      four<true>(r.a, x, os);
    } else {
#pragma unroll
      for (int kb = 0; kb < 3; ++kb)
        if (kb <= wave)
#pragma unroll
          for (int ct = 0; ct < NC; ++ct) os[ct][kb & 1] += dot16(r.a[kb], x[kb][ct]);
    }
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) o[ct] = os[ct][0] + os[ct][1];
    load_second(r, c + 1);
  }
};

// The delta rule's, its fp32 products as thirds on the 16-bit instructions.  S and u cross through LDS as thirds, split once by
// the wave that has them; what comes from memory is split where it is used (in front of the barriers instead: half a percent of
// calls' times; in the shadow of the products' chain, with loads a chunk ahead: 5 % slower).  A chain of few workgroups over 64 keys
// is bound by its operands, 68 KB a chunk at 45 - 61 KB per us from the memory-side cache, and by what splits them: there the fp32
// instructions were up to 10 % faster (5908 rows of 8 heads of 64 x 64 140 us and 154), and less exact.
template <int DP, int NC> struct DeltaWalk {
  static constexpr int KB = DP / 16, KS = DP / 32, NT = DP / 64, LD = DP + 8, LU = C + 8;
  static constexpr Layout L0 = layout_of(DP, 0, false);
  struct Shared {
    __attribute__((aligned(16))) bf16_t sl[3][16 * NC * LD];
    __attribute__((aligned(16))) bf16_t ul[3][16 * NC * LU];
  };
  static __device__ __forceinline__ f32x4 at(const float* p, int offset) { return *reinterpret_cast<const f32x4*>(p + offset); }

  const float* ws;                                 // the pair's first chunk
  long step;
  int nc, VP, tile, wave, lane, lr, kh;
  Shared& sh;

  // (chunks past the last are read as the last one: loads without a condition keep the waits for them exact)
  __device__ __forceinline__ const float* chunk_at(int c) const { return ws + step * min(c, nc - 1); }
  __device__ __forceinline__ f32x4 left(const float* p, int offset, int index) const { return at(p, offset + piece(index, lane)); }

  struct StateOps { f32x4 w[KB], k[NT][4], u[NC], b[NT]; };
  struct OutOps { f32x4 q[KB], a[4]; };

  __device__ __forceinline__ void load_first(StateOps& r, int c) const {
    const float* p = chunk_at(c);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) r.w[kb] = left(p, L0.u + VP * C, wave * KB + kb);
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) r.u[ct] = left(p, L0.u, (NC * tile + ct) * 4 + wave);
    __builtin_amdgcn_sched_barrier(0);             // (the loads stay where they are put)
  }
  __device__ __forceinline__ void load_second(StateOps& r, int c) const {
    const float* p = chunk_at(c);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) r.k[t][kb] = left(p, L0.kt, (wave * NT + t) * 4 + kb);
      r.b[t] = at(p, L0.bc + (wave * NT + t) * 16 + 4 * kh);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void load_first(OutOps& r, int c) const {
    const float* p = chunk_at(c);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) r.q[kb] = left(p, L0.q, wave * KB + kb);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void load_second(OutOps& r, int c) const {
    const float* p = chunk_at(c);
    // (the blocks right of the diagonal are never written: they are read, so that the loads carry no condition, and not used)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) r.a[kb] = left(p, 0, wave * 4 + kb);
    __builtin_amdgcn_sched_barrier(0);
  }
  // S and u in LDS: a column's rows 32 j + 16 half + 4 kh + e at 32 j + 8 kh + 4 half + e, what a lane takes as one right operand
  template <int LDR, int N> __device__ __forceinline__ Thirds read_right(const bf16_t (&planes)[3][N], int j, int ct) const {
    const int o = (16 * ct + lr) * LDR + 32 * j + 8 * kh;
    return {*reinterpret_cast<const bf16x8*>(planes[0] + o), *reinterpret_cast<const bf16x8*>(planes[1] + o),
            *reinterpret_cast<const bf16x8*>(planes[2] + o)};
  }
  template <int LDR, int N> __device__ __forceinline__ void write_half(bf16_t (&planes)[3][N], int block, int ct, f32x4 v) const {
    const Thirds t = thirds<false>(v, f32x4{0.f, 0.f, 0.f, 0.f});
    const int o = (16 * ct + lr) * LDR + 32 * (block >> 1) + 8 * kh + 4 * (block & 1);
    *reinterpret_cast<bf16x4*>(planes[0] + o) = __builtin_shufflevector(t.h, t.h, 0, 1, 2, 3);
    *reinterpret_cast<bf16x4*>(planes[1] + o) = __builtin_shufflevector(t.m, t.m, 0, 1, 2, 3);
    *reinterpret_cast<bf16x4*>(planes[2] + o) = __builtin_shufflevector(t.l, t.l, 0, 1, 2, 3);
  }
  // reduction blocks 2 j, 2 j + 1 of a right operand in LDS
  template <int LDR, int N> __device__ __forceinline__ void read_columns(const bf16_t (&planes)[3][N], int j, Thirds (&x)[NC]) const {
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) x[ct] = read_right<LDR>(planes, j, ct);
  }

  __device__ __forceinline__ void chunk(StateOps& r, int c, f32x4 (&S)[NT][NC]) const {
    auto& sl = sh.sl;
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) {
      if constexpr (NT == 2) {
        const Thirds t = thirds(S[0][ct], S[1][ct]);
        const int o = (16 * ct + lr) * LD + 32 * wave + 8 * kh;
        *reinterpret_cast<bf16x8*>(sl[0] + o) = t.h;
        *reinterpret_cast<bf16x8*>(sl[1] + o) = t.m;
        *reinterpret_cast<bf16x8*>(sl[2] + o) = t.l;
      } else {
        write_half<LD>(sl, wave, ct, S[0][ct]);
      }
    }
    __syncthreads();
    Thirds x[NC];
    Sum us[NC] = {};
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      read_columns<LD>(sl, j, x);
      products<false, false>(thirds(r.w[2 * j], r.w[2 * j + 1]), x, us);
    }
    f32x4 add_u[NC];
    values(us, add_u);
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) write_half<LU>(sh.ul, wave, ct, r.u[ct] + add_u[ct]);
    load_first(r, c + 1);
    __syncthreads();
    Sum add[NT * NC] = {};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      read_columns<LU>(sh.ul, j, x);
      Thirds keys[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) keys[t] = thirds(r.k[t][2 * j], r.k[t][2 * j + 1]);
      products<false, false>(keys, x, add);
    }
    f32x4 by[NT * NC];
    values(add, by);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) S[t][ct] = S[t][ct] * r.b[t] + by[t * NC + ct];
    load_second(r, c + 1);
  }
  // o of the wave's 16 rows
  __device__ __forceinline__ void chunk(OutOps& r, int c, f32x4 (&o)[NC], f32x4 (&)[NC]) const {
    __syncthreads();
    Sum os[NC] = {};
    Thirds x[NC];
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      read_columns<LD>(sh.sl, j, x);
      products<false, false>(thirds(r.q[2 * j], r.q[2 * j + 1]), x, os);
    }
    load_first(r, c + 1);
    __syncthreads();
    // (the lower triangle's blocks; the wave's number is the same for all its lanes)
    float odd = 0.f;                               // u of the wave's own rows, which the block on the diagonal meets
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(sh.ul[0] + (16 * ct + lr) * LU + 32 * (wave >> 1) + 8 * kh + 4 * (wave & 1));
      odd = not_finite(f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}, odd);
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const bool apart = __builtin_expect(__any(odd != 0.f), 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool last = j == wave >> 1;
      if (j > wave >> 1 || (last && apart && !(wave & 1))) continue;
      const bool both = !last || ((wave & 1) && !apart);
      read_columns<LU>(sh.ul, j, x);
      // (a block that is left out is zeros on both sides: a later row's infinity would come through a zero)
      if (!both)
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
#pragma unroll
          for (int e = 4; e < 8; ++e) x[ct].h[e] = x[ct].m[e] = x[ct].l[e] = (bf16_t)0.f;
      products<false, false>(thirds(r.a[2 * j], both ? r.a[2 * j + 1] : zero), x, os);
    }
    if (apart) {
      f32x4 own = zero;
#pragma unroll
      for (int i = 0; i < 4; ++i) if (i == wave) own = r.a[i];
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int at = (16 * ct + lr) * LU + 32 * (wave >> 1) + 8 * kh + 4 * (wave & 1) + e;
          const float h = (float)sh.ul[0][at], sum = h + ((float)sh.ul[1][at] + (float)sh.ul[2][at]);
          v[e] = sum != sum ? h : sum;
        }
        os[ct].h += lower16([&](int i, int g, int f) { return __shfl(own[f], g * 16 + i, 64); }, v);
      }
    }
    values(os, o);
    load_second(r, c + 1);
  }
};

template <int DP, bool DELTA, int NC>
__global__ __launch_bounds__(512, 2) void chunk_walk_kernel(float* __restrict__ out, const float* __restrict__ wsp, long ws_stride,
                                                            float* __restrict__ state, const int* __restrict__ slots,
                                                            const int* __restrict__ qsl, const int* __restrict__ seq_lens,
                                                            const float* __restrict__ d_skip, int B, int H, int dim, int vdim,
                                                            int VP, int h0, int nh, int chunks, float scale) {
  using W = std::conditional_t<DELTA, DeltaWalk<DP, NC>, LinearWalk<DP, NC>>;
  __shared__ typename W::Shared shared;
  const int tiles = VP / (16 * NC);
  const int id = blockIdx.x, die = id & 7, rest = id >> 3;
  const int tile = rest % tiles, pair = (rest / tiles) * 8 + die;
  if (pair >= B * nh) return;
  const int hh = pair % nh, h = h0 + hh, seq = by_length(qsl, B, pair / nh);
  const int q0 = qsl[seq], n = qsl[seq + 1] - q0;
  if (n <= 0) return;
  const int chunk0 = chunks_before(qsl, B, seq), nc = (n + C - 1) / C;
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  const int lane = threadIdx.x & 63, lr = lane & 15, kh = lane >> 4;
  const int col = 16 * NC * tile + lr;             // (and col + 16)
  W w{wsp + ((long)hh * chunks + chunk0) * ws_stride, ws_stride, nc, VP, tile, wave, lane, lr, kh, shared};
  if (role == 0) {
    float* st = state + ((long)slots[seq] * H + h) * (long)dim * vdim;
    const bool fresh = seq_lens[seq] - n <= 0;     // the rows start the sequence: whatever the slot holds is not ours
    typename W::StateOps r;
    w.load_first(r, 0);
    w.load_second(r, 0);
    f32x4 S[W::NT][NC];
    auto place = [&](int t, int ct, int e) {        // of S[t][ct][e] in the state, -1: outside
      const int d = (wave * W::NT + t) * 16 + 4 * kh + e, v = col + 16 * ct;
      return d < dim && v < vdim ? d * vdim + v : -1;
    };
#pragma unroll
    for (int t = 0; t < W::NT; ++t)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t][ct][e] = !fresh && place(t, ct, e) >= 0 ? st[place(t, ct, e)] : 0.f;
    for (int c = 0; c < nc; ++c) w.chunk(r, c, S);
#pragma unroll
    for (int t = 0; t < W::NT; ++t)
#pragma unroll
      for (int ct = 0; ct < NC; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (place(t, ct, e) >= 0) st[place(t, ct, e)] = S[t][ct][e];
  } else {
    const float skip = d_skip != nullptr ? d_skip[h] : 0.f;
    typename W::OutOps r;
    w.load_first(r, 0);
    w.load_second(r, 0);
    for (int c = 0; c < nc; ++c) {
      f32x4 o[NC], u[NC] = {};
      w.chunk(r, c, o, u);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = c * C + 16 * wave + 4 * kh + e;
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
          if (i < n && col + 16 * ct < vdim)
            out[((long)(q0 + i) * H + h) * vdim + col + 16 * ct] = DELTA ? o[ct][e] * scale : o[ct][e] * scale + skip * u[ct][e];
      }
    }
  }
}

template <typename T, int KIND>
int launch(const ChunkArgs& a, int chunks, int cols, float* out, float* state, const int* slots, const int* seq_lens,
           const float* d_skip, float scale, hipStream_t stream) {
  constexpr bool DELTA = KIND >= DELTA_CHANNEL;
  const dim3 prep(chunks, a.nh);
  const long pairs = ((long)a.B * a.nh + 7) / 8 * 8;
  const dim3 walk((unsigned)(pairs * (a.VP / cols)));
#define WALK(DP_, NC_)                                                                                                       \
  hipLaunchKernelGGL((chunk_walk_kernel<DP_, DELTA, NC_>), walk, dim3(512), 0, stream, out, a.ws, a.ws_stride, state, slots, \
                     a.qsl, seq_lens, d_skip, a.B, a.H, a.dim, a.vdim, a.VP, a.h0, a.nh, chunks, scale)
#define GO(DP_)                                                                                                            \
  do {                                                                                                                     \
    hipLaunchKernelGGL((chunk_prep_kernel<T, KIND, DP_>), prep, dim3(256), 0, stream, a);                                  \
    if (cols == 32) WALK(DP_, 2);                                                                                          \
    else WALK(DP_, 1);                                                                                                     \
  } while (0)
  if (a.dim <= 64) GO(64);
  else GO(128);
#undef GO
#undef WALK
  HIP_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// floats of workspace per chunk and head
VDAMD_API long vdamd_chunk_scan_floats(int kind, int dim, int vdim) {
  return layout_of(dim <= 64 ? 64 : 128, (vdim + 31) / 32 * 32, kind >= DELTA_CHANNEL).total;
}

// Heads h0 .. h0 + nh - 1 of one call.  x [T, x_stride] of type dtype with q, k (of group 0) and v (of head 0) at the three
// columns; dt / beta rows of the same type; out [T, H * vdim] fp32, state [slots, H, dim, vdim] fp32; `chunks`: a bound on the
// batch's chunks of 64 rows; ws: chunks * nh * vdamd_chunk_scan_floats floats, 16-byte aligned; dim <= 128; cols: columns of a
// workgroup of the walk, 16 or 32
VDAMD_API int vdamd_chunk_scan(float* out, int kind, const void* x, long x_stride, int q_off, int k_off, int v_off,
                               const void* beta, long beta_stride, const void* dt, long dt_stride, const float* dt_bias,
                               const float* a_log, const float* decay, const float* d_skip, float* ws, int chunks, float* state,
                               const int* slots, const int* qsl, const int* seq_lens, int B, int H, int G, int dim, int vdim,
                               int h0, int nh, int cols, int silu, float eps, float scale, int dtype, hipStream_t stream) {
  if (B <= 0 || chunks <= 0 || nh <= 0) return 0;
  if (H <= 0 || G <= 0 || H % G || dim <= 0 || dim > 128 || vdim <= 0 || h0 < 0 || h0 + nh > H || nh > 65535 ||
      (cols != 16 && cols != 32))
    return 1;
  ChunkArgs a{};
  a.x = x; a.x_stride = x_stride; a.q_off = q_off; a.k_off = k_off; a.v_off = v_off;
  a.beta = beta; a.beta_stride = beta_stride; a.dt = dt; a.dt_stride = dt_stride; a.dt_bias = dt_bias; a.a_log = a_log;
  a.decay = decay; a.ws = ws; a.ws_stride = vdamd_chunk_scan_floats(kind, dim, vdim); a.qsl = qsl;
  a.B = B; a.H = H; a.G = G; a.dim = dim; a.vdim = vdim; a.VP = (vdim + 31) / 32 * 32; a.h0 = h0; a.nh = nh;
  a.silu = silu; a.eps = eps;
  const int per = dtype == DT_F32 ? 4 : 8;         // elements of 16 bytes
  const bool rows16 = x_stride % per == 0 && (uintptr_t)x % 16 == 0;
  a.vec = rows16 && dim % per == 0 && q_off % per == 0 && k_off % per == 0 &&
          (kind != DELTA_CHANNEL || (dt_stride % per == 0 && (uintptr_t)dt % 16 == 0)) &&
          (kind != LINEAR_CHANNEL || (uintptr_t)decay % 16 == 0);
  a.vvec = rows16 && vdim % per == 0 && v_off % per == 0;
#define KINDS(T)                                                                                                               \
  switch (kind) {                                                                                                              \
    case LINEAR_HEAD: return launch<T, LINEAR_HEAD>(a, chunks, cols, out, state, slots, seq_lens, d_skip, scale, stream);       \
    case LINEAR_CHANNEL: return launch<T, LINEAR_CHANNEL>(a, chunks, cols, out, state, slots, seq_lens, d_skip, scale, stream); \
    case STATE_SPACE: return launch<T, STATE_SPACE>(a, chunks, cols, out, state, slots, seq_lens, d_skip, scale, stream);       \
    case DELTA_CHANNEL: return launch<T, DELTA_CHANNEL>(a, chunks, cols, out, state, slots, seq_lens, d_skip, scale, stream);   \
    case DELTA_HEAD: return launch<T, DELTA_HEAD>(a, chunks, cols, out, state, slots, seq_lens, d_skip, scale, stream);         \
  }
  switch (dtype) {
    case DT_BF16: KINDS(bf16_t) break;
    case DT_F16: KINDS(f16_t) break;
    case DT_F32: KINDS(float) break;
  }
#undef KINDS
  return 1;
}
