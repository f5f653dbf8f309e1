// Prompt portions of the recurrent mixers without a delta rule: decayed linear attention, the state-space scan.  gfx950.
//
//   S <- g S + k v^T ; o = S^T q        per (sequence, head), S [dim, vdim], a decay g per head, or per head and key channel
//
// in chunks of 32 rows on the matrix cores, S kept in registers in 32 bits: with b_i the product of the chunk's decays up to
// row i, G_ij that of the decays behind row j up to row i and S_0 the state in front of the chunk,
//   o_i = (b_i q_i)^T S_0 + sum_(j <= i) A_ij v_j,  A_ij = q_i^T G_ij k_j ;  S = b_32 S_0 + sum_j (G_32,j k_j) v_j^T
//
// Every product is formed in 32 bits on the 16-bit matrix instructions: a 32-bit operand is the sum of three of 16 bits (see
// Thirds), so that six instructions of 16 cycles do what eight of 32 do in 32-bit form; what is 16 bits wide from the start (v,
// and q, k under a decay per head) is one.
//
// A chain of chunks is what a long sequence is; it is cut into segments:
//   segment_kernel<OUT = false>  per (segment, head) that is not its sequence's last: the state that it adds to, from zero, and
//                                the product of its decays
//   segment_starts               the state in front of every segment, from those
//   segment_kernel<OUT = true>   per (segment, head): the outputs, from the state in front; the last one leaves the final state
// Sequences of one segment are the last kernel alone.  Nothing but the states (64 KB each at 128 x 128) passes between them.
//
// Products of decays are formed directly, never as differences of logarithms: b_i and G_32,j are products of at most 32 decays,
// G_ij between the chunk's two groups of 16 rows is (from the second's start up to i) * (behind j to the first's end), each at
// most 1 where decays are, so nothing overflows; inside a group it is the quotient of two products from the group's start,
// unless one of those is smaller than 2^-96 or larger than 2^96, where the group's 120 pairs are multiplied out.  A head's
// products are formed so in 64 bits (2^-960, 2^960) and join sums behind them.
#include "chunk_parts.h"

namespace {

constexpr int R = 32, G16 = 16, LR = R + 8;        // rows of a chunk, of a group; a column of rows in LDS

struct SegArgs {
  const void* x;                                   // [T, x_stride]: q, k of group 0 and v of head 0 at the three columns
  long x_stride;
  int q_off, k_off, v_off;
  const void* dt;                                  // [T, dt_stride], raw (state space)
  long dt_stride;
  const float* dt_bias;
  const float* a_log;
  const float* decay;                              // [H] (LINEAR_HEAD) or [T, H * dim] (LINEAR_CHANNEL)
  const float* d_skip;
  float* out;                                      // [T, H * vdim]
  float* ws;                                       // per (segment, head): the state in front of it | the products of the decays
                                                   // of the segment in front
  float* state;
  const int* slots;
  const int* qsl;
  const int* seq_lens;
  int B, H, G, dim, vdim, tiles;                   // tiles of columns
  int rows;                                        // of a segment (a multiple of 32); 0: a sequence is one
  int silu;
  float scale;
};

// A sequence of n rows comes in the fewest segments of at most `rows`, as even as whole chunks make them
__device__ __forceinline__ int segment_rows(int n, int rows) {
  const int ns = (n + rows - 1) / rows;
  return (n + ns * R - 1) / (ns * R) * R;
}
__device__ __forceinline__ int segments_of(const int* qsl, int s, int rows) {
  const int n = qsl[s + 1] - qsl[s];
  if (n <= 0 || rows == 0) return n > 0;
  const int each = segment_rows(n, rows);
  return (n + each - 1) / each;
}

// a state in the workspace: [tile of 16 keys][tile of 16 values][lane][4] as the matrix instruction's accumulator, then the decays
__host__ __device__ constexpr long state_floats(int DP, int VP) { return (long)DP * VP + DP; }

// Eight waves.  In front of a chunk's products a wave prepares a group of 16 rows and a quarter of the channels and of the value
// columns, lane (lr, kh) has NV channels of row lr; in the products it has half of the keys and a quarter of the columns, S of them as
// accumulators, which is at once the right operand of q S.  Three barriers a chunk: the groups' products of decays are there; the
// operands are; A and the other half's sums are.
// Bound by the chunk's instructions: a wave issues 850 vector instructions (128 x 128, a decay per channel, outputs) of four cycles
// and 90 matrix instructions of 16, two waves to a SIMD, and neither fills the other's time: 13 000 - 14 000 cycles a chunk, 5.5 us,
// of which 3 300 are the barriers' waits.  16 waves of half the columns each spilled and were slower (104 -> 164 us, 6007 rows x 16 heads).
// v_cvt_pk_bf16_f32, products of decays through LDS and a branch for each four values that look for what is not finite cost
// 40 % more.  6007 rows of three prompts, 16 heads of 128 x 128, a decay per channel: states 35, starts 8, outputs 97 us, against
// 67 (preparation) and 143 of the chunked kernels; one prompt of 7000 rows, 8 heads, state space: 74 against 234.
// LDS: 117 KB (137 where v has thirds): one workgroup to a compute unit; 64 x 64 two (54 - 79 KB, 128 registers).
template <typename T, int KIND, bool X, int DP, int VW, bool OUT>
__global__ __launch_bounds__(512, DP * VW > 64 * 64 ? 2 : 4) void segment_kernel(SegArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)              // (the buffer builtins exist in the device pass only)
  constexpr bool CHAN = KIND == LINEAR_CHANNEL, LX = X && !CHAN;
  constexpr int NV = DP / 16, NVV = VW / 16;       // a lane's channels of q and k, columns of v, in the preparation
  constexpr int KS = DP / 64, DB = DP / 32, CT = VW / 64;        // a wave's steps of 32 keys, tiles of 16 keys, of 16 columns
  constexpr int LQ = DP + 8, LP = R + 4;
  __shared__ __attribute__((aligned(16))) bf16_t bq[OUT ? (LX ? 1 : 3) : 1][OUT ? R * LQ : 8];
  __shared__ __attribute__((aligned(16))) bf16_t k0[OUT ? (LX ? 1 : 3) : 1][OUT ? G16 * LQ : 8];
  __shared__ __attribute__((aligned(16))) bf16_t kt[3][DP * LR];
  __shared__ __attribute__((aligned(16))) bf16_t vv[X ? 1 : 3][VW * LR];
  __shared__ __attribute__((aligned(16))) float part[OUT ? 4 * R * LP : 4];      // A, a quarter of the channels each
  __shared__ __attribute__((aligned(16))) f32x4 ox[OUT ? 8 * CT * 64 : 1];       // sums over half of the keys for the other wave
  __shared__ __attribute__((aligned(16))) float tl[2][CHAN ? 2 * DP : 4];        // products of the groups' decays
  __shared__ __attribute__((aligned(16))) float rowf[CHAN ? 4 : R];
  __shared__ double td[2][2], sd[CHAN ? 1 : G16];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, kh = lane >> 4;
  // ---- which segment: neighbours in the grid, which go to the eight dies in turn, are a segment's heads.  (With the segments side by
  // side, 8 sequences or a multiple of it put all heads of one on one die: 32 heads of 128 x 64, 589 rows of 32, one of 376, 274 us,
  // now 76; 2048 rows of 8 in segments of 480 115 and 67)
  const int heads = a.H * a.tiles, want = blockIdx.x / heads, h = (blockIdx.x - want * heads) % a.H;
  const int tile = (blockIdx.x - want * heads) / a.H;
  int seq, s, ns;
  if (a.rows) {
    if (!locate(a.B, want, seq, s, [&](int i) { return segments_of(a.qsl, i, a.rows); })) return;
    seq = __builtin_amdgcn_readfirstlane(seq);     // (the same in all lanes, which the compiler does not see)
    s = __builtin_amdgcn_readfirstlane(s);
    ns = segments_of(a.qsl, seq, a.rows);
  } else {
    seq = __builtin_amdgcn_readfirstlane(by_length(a.qsl, a.B, want));
    s = 0;
    ns = 1;
  }
  const int n_all = a.qsl[seq + 1] - a.qsl[seq];
  if (n_all <= 0 || (!OUT && s == ns - 1)) return;
  const int grp = h / (a.H / a.G), v0 = tile * VW;
  const int each = a.rows ? segment_rows(n_all, a.rows) : n_all;
  const long q0 = a.qsl[seq] + (long)s * each;
  const int n = min(each, n_all - s * each), nc = (n + R - 1) / R;
  const long unit = state_floats(DP, a.tiles * VW);
  float* const wst = a.ws + ((long)want * a.H + h) * unit;

  // ---- the preparation: wave (group of 16 rows, quarter of the channels), lane (row lr, channels kh NV ..)
  const int g = wave >> 2, qt = wave & 3;
  const int ch0 = qt * (DP / 4) + NV * kh, col0 = qt * (VW / 4) + NVV * kh;
  typedef T TV __attribute__((ext_vector_type(NV)));
  typedef T TVV __attribute__((ext_vector_type(NVV)));
  typedef float FV __attribute__((ext_vector_type(NV)));
  typedef float FVV __attribute__((ext_vector_type(NVV)));
  TV rq, rk;
  TVV rv;
  FV rd;
  [[maybe_unused]] T rdt = (T)0.f;
  // (chunks of whole rows and channels are the common case: what lies outside is read from a place inside, and cleared below)
  const int cin = min(ch0, a.dim - NV), vin = min(v0 + col0, a.vdim - NVV);
  const T* const xh = (const T*)a.x + q0 * a.x_stride;
  const unsigned stride = (unsigned)a.x_stride, qk = grp * a.dim + cin, vc = a.v_off + h * a.vdim + vin;
  auto fetch = [&](int c) {
    const T* const xc = xh + (long)min(c * R, n - 1) * a.x_stride;              // (the wave's: one address for all lanes)
    const unsigned row = min(G16 * g + lr, max(n - 1 - c * R, 0));
    if constexpr (OUT) rq = *reinterpret_cast<const TV*>(xc + (row * stride + a.q_off + qk));
    rk = *reinterpret_cast<const TV*>(xc + (row * stride + a.k_off + qk));
    rv = *reinterpret_cast<const TVV*>(xc + (row * stride + vc));
    if constexpr (CHAN) {
      const float* const dc = a.decay + ((q0 + min(c * R, n - 1)) * a.H + h) * (long)a.dim;
      rd = *reinterpret_cast<const FV*>(dc + (row * (unsigned)(a.H * a.dim) + cin));
    }
    if constexpr (KIND == STATE_SPACE) rdt = ((const T*)a.dt)[(q0 + min(c * R, n - 1)) * a.dt_stride + h + row * (unsigned)a.dt_stride];
  };

  // ---- the products: wave (half of the keys, columns cg * 16 CT ..); S as accumulators
  const int dh = wave >> 2, cg = wave & 3;
  f32x4 S[DB][CT];
  const bool fresh = a.seq_lens[seq] - n_all <= 0;               // the rows start the sequence: whatever the slot holds is not ours
  const auto slot = __builtin_amdgcn_make_buffer_rsrc(a.state + ((long)a.slots[seq] * a.H + h) * (long)a.dim * a.vdim, 0,
                                                      a.dim * a.vdim * 4, 0x00020000);
  // (keys past the last lie behind the buffer by themselves; reads from outside are zero, writes are dropped)
  auto place = [&](int db, int ct, int e) {        // of S[db][ct][e] in the state, in bytes
    const int d = dh * (DP / 2) + 16 * db + 4 * kh + e, v = v0 + (cg * CT + ct) * 16 + lr;
    return v < a.vdim ? (d * a.vdim + v) * 4 : 0x40000000;
  };
  auto kept = [&](float* p, int db, int ct) {      // the same in the workspace
    const int at = tile * (VW / 16) + cg * CT + ct;
    return reinterpret_cast<f32x4*>(p + (((long)(dh * DB + db) * (a.tiles * VW / 16) + at) * 64 + lane) * 4);
  };
  fetch(0);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      S[db][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (OUT) {
        if (ns > 1) S[db][ct] = *kept(wst, db, ct);
        else if (!fresh)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            S[db][ct][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(slot, place(db, ct, e), 0, 0));
      }
    }
  float all = 1.f;                                 // OUT = false: the product of the segment's decays, of channel threadIdx.x
  double all_d = 1.0;
  if constexpr (OUT)                               // (the block above the diagonal)
    for (int i = threadIdx.x; i < 4 * G16 * G16; i += 512) part[(i >> 8) * R * LP + (i >> 4 & 15) * LP + G16 + (i & 15)] = 0.f;
  const float head_decay = KIND == LINEAR_HEAD ? a.decay[h] : 1.f;
  [[maybe_unused]] const float bias = KIND == STATE_SPACE ? a.dt_bias[h] : 0.f, rate = KIND == STATE_SPACE ? expf(a.a_log[h]) : 0.f;
  const float skip = KIND == STATE_SPACE && OUT && a.d_skip != nullptr ? a.d_skip[h] : 0.f;

#pragma unroll 1
  for (int c = 0; c < nc; ++c) {
    // (what follows from the lane is made anew in every chunk: kept across them it would not fit the registers)
    int again = lane;
    asm volatile("" : "+v"(again));
    const int lr = again & 15, kh = again >> 4;
    const int ch0 = qt * (DP / 4) + NV * kh, col0 = qt * (VW / 4) + NVV * kh;
    const bool ok = c * R + G16 * g + lr < n;
    f32x4 q[NV / 4], k[NV / 4], v[NVV / 4], p[NV / 4], dk[NV / 4];
    [[maybe_unused]] f32x4 kd[NV / 4], ks[NV / 4]; // k over the products up to the row, times those behind it
    [[maybe_unused]] bool apart = false;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      q[i / 4][i % 4] = (float)rq[i];
      k[i / 4][i % 4] = (float)rk[i];
      dk[i / 4][i % 4] = rd[i];
    }
#pragma unroll
    for (int i = 0; i < NVV; ++i) v[i / 4][i % 4] = (float)rv[i];
    const float dtv = (float)rdt;
    if (c * R + R > n || a.dim < DP || v0 + VW > a.vdim) {
      const bool in = ok && ch0 < a.dim, vin_ = ok && v0 + col0 < a.vdim;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        q[i / 4][i % 4] = in ? q[i / 4][i % 4] : 0.f;
        k[i / 4][i % 4] = in ? k[i / 4][i % 4] : 0.f;
        dk[i / 4][i % 4] = in ? dk[i / 4][i % 4] : 1.f;
      }
#pragma unroll
      for (int i = 0; i < NVV; ++i) v[i / 4][i % 4] = vin_ ? v[i / 4][i % 4] : 0.f;
    }
    fetch(c + 1);                                  // (past the last row: the last row's)
    __builtin_amdgcn_sched_barrier(0);
    if (!X && a.silu) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if constexpr (OUT) q[i / 4][i % 4] = silu_f(q[i / 4][i % 4]);
        k[i / 4][i % 4] = silu_f(k[i / 4][i % 4]);
      }
#pragma unroll
      for (int i = 0; i < NVV; ++i) v[i / 4][i % 4] = silu_f(v[i / 4][i % 4]);
    }
    // ---- products of decays inside the group: up to the row, behind it
    float own = 1.f, step = 1.f;
    double pd = 1.0, after = 1.0;
    [[maybe_unused]] double pr[4];
    if constexpr (CHAN) {
#pragma unroll
      for (int i = 0; i < NV / 4; ++i) {
        p[i] = dk[i];
        prefix_products(p[i]);
        if (lr == 15) *reinterpret_cast<f32x4*>(&tl[c & 1][g * DP + ch0 + 4 * i]) = p[i];
      }
    } else {
      if (ok) {
        if constexpr (KIND == LINEAR_HEAD) own = head_decay;
        else {
          step = softplus_f(dtv + bias);
          own = expf(-rate * step);
        }
      }
      head_products(own, pd, after);
#pragma unroll
      for (int e = 0; e < 4; ++e) pr[e] = __shfl(pd, 4 * kh + e, 16);
      if (lane == 15 && qt == 0) td[c & 1][g] = pd;
    }
    bool far = false;
    if constexpr (CHAN) {
      unsigned beyond = 0;                         // (an exponent outside -96 .. 96, infinities and NaN among them)
#pragma unroll
      for (int i = 0; i < NV; ++i) beyond = max(beyond, (bits(p[i / 4][i % 4]) << 1) - 0x1f000000u);
      far = beyond > 0xc0000000u;
    } else {
      far = !(fabs(pd) >= 0x1p-960 && fabs(pd) <= 0x1p960);
    }
    apart = __any(far);
    // ---- A inside the group, over the wave's channels
    f32x4 da = {0.f, 0.f, 0.f, 0.f};
    Thirds tq;
    if constexpr (OUT) {
      if (apart) da = pairs_apart<CHAN, NV / 4>(q, k, dk, own);
      if constexpr (CHAN)
#pragma unroll
        for (int i = 0; i < NV / 4; ++i) q[i] *= p[i];
      tq = thirds_of<NV / 4, LX>(q);
    }
    if constexpr (CHAN) {
#pragma unroll
      for (int i = 0; i < NV / 4; ++i) ks[i] = k[i] * suffix_products(dk[i]);
      if (OUT && !apart) {
#pragma unroll
        for (int i = 0; i < NV / 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) kd[i][e] = quotient(k[i][e], p[i][e]);
      }
    }
    if constexpr (OUT) {
      if (!apart) {
        Thirds tk[1];
        if constexpr (CHAN) tk[0] = thirds_of<NV / 4, false>(kd);
        else tk[0] = thirds_of<NV / 4, LX>(k);
        Sum sum[1] = {};
        products<LX, LX>(tq, tk, sum);
        da = value<!LX>(sum[0]);
        if constexpr (!CHAN) {
          const double over = 1.0 / pd;
#pragma unroll
          for (int e = 0; e < 4; ++e) da[e] *= (float)(pr[e] * over);
        }
      }
      if constexpr (KIND == STATE_SPACE) da *= step;
    }
    __syncthreads();                               // the groups' products are there; the chunk in front has been used up
    // ---- operands into LDS
    f32x4 other[NV / 4];
    double other_d = 1.0;
    if constexpr (CHAN) {
#pragma unroll
      for (int i = 0; i < NV / 4; ++i) other[i] = *reinterpret_cast<const f32x4*>(&tl[c & 1][(1 - g) * DP + ch0 + 4 * i]);
    } else {
      other_d = td[c & 1][1 - g];
    }
    if constexpr (OUT) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[(qt * R + G16 * g + 4 * kh + e) * LP + G16 * g + lr] = lr <= 4 * kh + e ? da[e] : 0.f;
      Thirds tb = tq;
      if constexpr (CHAN) {
        if (g == 1) {
          f32x4 b[NV / 4];
#pragma unroll
          for (int i = 0; i < NV / 4; ++i) b[i] = q[i] * other[i];
          tb = thirds_of<NV / 4, false>(b);
        }
      } else if (qt == 0 && kh == 0) {
        rowf[G16 * g + lr] = (float)(g == 1 ? pd * other_d : pd);
      }
      // (a row's keys in the order in which S has them: 32 j + 16 half + 4 kh + e at 32 j + 8 kh + 4 half + e)
#pragma unroll
      for (int i = 0; i < NV / 4; ++i) {
        const int ch = ch0 + 4 * i, to = (ch & ~31) + 8 * (ch >> 2 & 3) + 4 * (ch >> 4 & 1);
        store4<LX>(bq, (G16 * g + lr) * LQ + to, tb, i);
      }
    }
    f32x4 end[NV / 4];
    {
      if constexpr (CHAN) {
#pragma unroll
        for (int i = 0; i < NV / 4; ++i)
          end[i] = ks[i];
        if constexpr (OUT)
          if (g == 0) {
            const Thirds t = thirds_of<NV / 4, false>(end);
#pragma unroll
            for (int i = 0; i < NV / 4; ++i) store4<false>(k0, lr * LQ + ch0 + 4 * i, t, i);
          }
        if (g == 0)
#pragma unroll
          for (int i = 0; i < NV / 4; ++i) end[i] *= other[i];
      } else {
        if constexpr (OUT)
          if (g == 0) {
            const Thirds t = thirds_of<NV / 4, LX>(k);
#pragma unroll
            for (int i = 0; i < NV / 4; ++i) store4<LX>(k0, lr * LQ + ch0 + 4 * i, t, i);
            if (qt == 0 && kh == 0) sd[lr] = KIND == STATE_SPACE ? after * step : after;
          }
        const float f = (float)((g == 0 ? after * other_d : after) * (KIND == STATE_SPACE ? (double)step : 1.0));
#pragma unroll
        for (int i = 0; i < NV / 4; ++i) end[i] = k[i] * f;
      }
    }
    store_columns<LR, false, NV>(kt, ch0, G16 * g + lr, thirds_of<NV / 4, false, false>(end));
    store_columns<LR, X, NVV>(vv, col0, G16 * g + lr, thirds_of<NVV / 4, X, false>(v));
    __syncthreads();                               // the operands are there
    // ---- A between the groups, over the wave's channels
    if constexpr (OUT)
      if (g == 1) {
        Thirds t[1];
        t[0] = load_third<NV, LX>(k0, lr * LQ + ch0);
        Sum sum[1] = {};
        products<LX, LX>(tq, t, sum);
        f32x4 dx = value<!LX>(sum[0]);
        if constexpr (!CHAN) {
          const double sj = sd[lr];
#pragma unroll
          for (int e = 0; e < 4; ++e) dx[e] *= (float)(pr[e] * sj);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) part[(qt * R + G16 + 4 * kh + e) * LP + lr] = dx[e];
      }
    // ---- q S over the wave's half of the keys
    f32x4 o[2][CT];
    if constexpr (OUT) {
      Sum os[2 * CT] = {};
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        Thirds x[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) x[ct] = thirds(S[2 * j][ct], S[2 * j + 1][ct]);
        Thirds rows[2];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) rows[rb] = load_third<8, LX>(bq, (G16 * rb + lr) * LQ + dh * (DP / 2) + 32 * j + 8 * kh);
        products<LX, false>(rows, x, os);
      }
      f32x4 ov[2 * CT];
      values(os, ov);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          o[rb][ct] = ov[rb * CT + ct];
          if (rb != dh) ox[(wave * CT + ct) * 64 + lane] = o[rb][ct];
        }
    }
    // ---- S (a head's decay is the same number in every chunk, and so would the error of its rounded product be: two pieces)
    [[maybe_unused]] float bh = 1.f, bl = 0.f;
    if constexpr (!CHAN) {
      const double both = td[c & 1][0] * td[c & 1][1];
      bh = (float)both;
      bl = (float)(both - bh);
    }
    Thirds x[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) x[ct] = load_third<8, X>(vv, ((cg * CT + ct) * 16 + lr) * LR + 8 * kh);
    Sum add[DB * CT] = {};
    f32x4 by[DB * CT];
#pragma unroll
    for (int db = 0; db < DB; db += 2) {
      Thirds keys[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) keys[i] = load_third<8, false>(kt, (dh * (DP / 2) + 16 * (db + i) + lr) * LR + 8 * kh);
      products<false, X>(keys, x, &add[db * CT]);
    }
    values(add, by);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int d = dh * (DP / 2) + 16 * db + 4 * kh;
      f32x4 b;
      if constexpr (CHAN) b = *reinterpret_cast<const f32x4*>(&tl[c & 1][d]) * *reinterpret_cast<const f32x4*>(&tl[c & 1][DP + d]);
      else b = f32x4{bh, bh, bh, bh};
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        if constexpr (!CHAN) by[db * CT + ct] += S[db][ct] * bl;
        S[db][ct] = S[db][ct] * b + by[db * CT + ct];
      }
    }
    if constexpr (!OUT) {
      if constexpr (CHAN) {
        if (threadIdx.x < DP) all *= tl[c & 1][threadIdx.x] * tl[c & 1][DP + threadIdx.x];
      } else {
        all_d *= td[c & 1][0] * td[c & 1][1];
      }
    } else {
      __syncthreads();                             // the other waves' sums and A are there
      // ---- the outputs of rows 16 dh .. of the chunk
      f32x4 al[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float* pa = part + (G16 * dh + lr) * LP + 8 * kh + 4 * i;
        al[i] = (*reinterpret_cast<const f32x4*>(pa) + *reinterpret_cast<const f32x4*>(pa + R * LP)) +
                (*reinterpret_cast<const f32x4*>(pa + 2 * R * LP) + *reinterpret_cast<const f32x4*>(pa + 3 * R * LP));
      }
      float odd = 0.f;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < 8; ++e) odd = fmaf((float)x[ct].h[e], 0.f, odd);
      Sum oo[CT] = {};
      // (a zero above the diagonal would hand a later row's infinity to the rows in front of it: such a chunk term by term)
      if (__builtin_expect(__any(odd != 0.f), 0)) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll 1
          for (int j = 0; j < R; ++j) {
            const int at = ((cg * CT + ct) * 16 + lr) * LR + j;
            float vj = (float)vv[0][at];
            if constexpr (!X) {
              const float sum = vj + ((float)vv[1][at] + (float)vv[2][at]);
              vj = sum != sum ? vj : sum;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = G16 * dh + 4 * kh + e;
              const float* pa = part + i * LP + j;
              const float w = (pa[0] + pa[R * LP]) + (pa[2 * R * LP] + pa[3 * R * LP]);
              if (j <= i) oo[ct].h[e] += w * vj;
            }
          }
      } else {
        products<false, X>(thirds(al[0], al[1]), x, oo);
      }
      f32x4 oov[CT];
      values(oo, oov);
      const int line = a.H * a.vdim * 4;           // bytes of a row; rows past the last lie behind the buffer
      const auto oc = __builtin_amdgcn_make_buffer_rsrc(a.out + ((q0 + c * R) * a.H + h) * (long)a.vdim, 0, min(R, n - c * R) * line,
                                                        0x00020000);
      f32x4 rf = {1.f, 1.f, 1.f, 1.f};
      if constexpr (!CHAN) rf = *reinterpret_cast<const f32x4*>(rowf + G16 * dh + 4 * kh);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const f32x4 mine = dh ? o[1][ct] : o[0][ct];
        f32x4 r = (mine + ox[((wave ^ 4) * CT + ct) * 64 + lane]) * rf + oov[ct];
        const int col = v0 + (cg * CT + ct) * 16 + lr;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float val = r[e] * a.scale;
          if constexpr (KIND == STATE_SPACE) {
            const int at = ((cg * CT + ct) * 16 + lr) * LR + G16 * dh + 4 * kh + e;
            float vj = (float)vv[0][at];
            if constexpr (!X) {
              const float sum = vj + ((float)vv[1][at] + (float)vv[2][at]);
              vj = sum != sum ? vj : sum;
            }
            val += skip * vj;
          }
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, val), oc,
                                                col < a.vdim ? (G16 * dh + 4 * kh + e) * line + col * 4 : 0x40000000, 0, 0);
        }
      }
    }
  }
  if constexpr (OUT) {
    if (s < ns - 1) return;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)S[db][ct][e]), slot, place(db, ct, e), 0, 0);
  } else {
    float* const next = wst + a.H * unit;          // what stands in front of the next segment, but for the state in front of this
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) *kept(next, db, ct) = S[db][ct];
    if (tile == 0 && threadIdx.x < DP) next[unit - DP + threadIdx.x] = CHAN ? all : (float)all_d;
  }
#endif
}

// grid (sequence x head, pieces of 256 x 4 of the state): a value's chain over the segments of a sequence of several
__global__ __launch_bounds__(256) void segment_starts(SegArgs a, int DP, int VP) {
  const int seq = blockIdx.x / a.H, h = blockIdx.x % a.H;
  const int n = a.qsl[seq + 1] - a.qsl[seq], ns = segments_of(a.qsl, seq, a.rows);
  if (ns <= 1) return;
  int first = 0;                                   // segments in front of the sequence's
  for (int i = threadIdx.x & 63; i < seq; i += 64) first += segments_of(a.qsl, i, a.rows);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) first += __shfl_xor(first, o, 64);
  const long unit = state_floats(DP, VP), step = a.H * unit;
  const int idx = blockIdx.y * 256 + threadIdx.x;  // of four values
  if (idx * 4 >= DP * VP) return;
  const int lane = idx & 63, tile = idx >> 6, d = tile / (VP / 16) * 16 + 4 * (lane >> 4), v = tile % (VP / 16) * 16 + (lane & 15);
  float* p = a.ws + ((long)first * a.H + h) * unit + idx * 4;
  const float* b = a.ws + ((long)first * a.H + h) * unit + (long)DP * VP + d;
  const float* st = a.state + ((long)a.slots[seq] * a.H + h) * (long)a.dim * a.vdim;
  const bool fresh = a.seq_lens[seq] - n <= 0;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (!fresh && d + e < a.dim && v < a.vdim) s[e] = st[(d + e) * a.vdim + v];
  *reinterpret_cast<f32x4*>(p) = s;
  constexpr int AHEAD = 4;
  for (int g0 = 1; g0 < ns; g0 += AHEAD) {
    f32x4 add[AHEAD], by[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const long at = min(g0 + i, ns - 1) * step;
      add[i] = *reinterpret_cast<const f32x4*>(p + at);
      by[i] = *reinterpret_cast<const f32x4*>(b + at);
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (g0 + i >= ns) break;
      s = s * by[i] + add[i];
      *reinterpret_cast<f32x4*>(p + (g0 + i) * step) = s;
    }
  }
}

template <typename T, int KIND, bool X, int DP, int VW> int launch(SegArgs a, int segments, hipStream_t st) {
  const int tiles = a.tiles = (a.vdim + VW - 1) / VW;
  if ((long)segments * a.H * tiles * 512 > 0xffffffffl) return 1;                  // (of threads, a launch's limit)
  const dim3 grid(segments * a.H * tiles);
  if (a.rows) {
    hipLaunchKernelGGL((segment_kernel<T, KIND, X, DP, VW, false>), grid, dim3(512), 0, st, a);
    hipLaunchKernelGGL(segment_starts, dim3(a.B * a.H, (DP * tiles * VW + 1023) / 1024), dim3(256), 0, st, a, DP, tiles * VW);
  }
  hipLaunchKernelGGL((segment_kernel<T, KIND, X, DP, VW, true>), grid, dim3(512), 0, st, a);
  HIP_LAUNCH_CHECK();
  return 0;
}
template <typename T, int KIND, bool X> int sizes(const SegArgs& a, int segments, hipStream_t st) {
  if (a.dim <= 64) return a.vdim <= 64 ? launch<T, KIND, X, 64, 64>(a, segments, st) : launch<T, KIND, X, 64, 128>(a, segments, st);
  return a.vdim <= 64 ? launch<T, KIND, X, 128, 64>(a, segments, st) : launch<T, KIND, X, 128, 128>(a, segments, st);
}
template <typename T> int kinds(const SegArgs& a, int kind, int segments, hipStream_t st) {
  constexpr bool B16 = std::is_same_v<T, bf16_t>;
  if (kind == LINEAR_HEAD) return sizes<T, LINEAR_HEAD, false>(a, segments, st);
  if (a.silu) return kind == LINEAR_CHANNEL ? sizes<T, LINEAR_CHANNEL, false>(a, segments, st) : 1;
  if (kind == LINEAR_CHANNEL) return sizes<T, LINEAR_CHANNEL, B16>(a, segments, st);
  return kind == STATE_SPACE ? sizes<T, STATE_SPACE, B16>(a, segments, st) : 1;
}

}  // namespace

// floats of workspace per segment (segments of more than none)
VDAMD_API long vdamd_segment_scan_floats(int heads, int dim, int vdim) {
  const int vw = vdim <= 64 ? 64 : 128;
  return heads * state_floats(dim <= 64 ? 64 : 128, (vdim + vw - 1) / vw * vw);
}

// x [T, x_stride] of type dtype with q, k (of group 0) and v (of head 0) at the three columns, all at multiples of 16 bytes, dim and
// vdim multiples of 8; dt rows of the same type; decay [H] or [T, H, dim]; out
// [T, H * vdim] fp32, state [slots, H, dim, vdim] fp32, dim <= 128.  rows: of a segment, a multiple of 32, with `segments` a bound
// on the batch's and ws segments * vdamd_segment_scan_floats floats, 16-byte aligned; 0: every sequence is one, segments == B
VDAMD_API int vdamd_segment_scan(float* out, int kind, const void* x, long x_stride, int q_off, int k_off, int v_off, const void* dt,
                                 long dt_stride, const float* dt_bias, const float* a_log, const float* decay, const float* d_skip,
                                 float* ws, int rows, int segments, float* state, const int* slots, const int* qsl,
                                 const int* seq_lens, int B, int H, int G, int dim, int vdim, int silu, float scale, int dtype,
                                 hipStream_t stream) {
  if (B <= 0 || segments <= 0) return 0;
  if (H <= 0 || H > 65535 || (long)H * vdim > (1 << 20) || G <= 0 || H % G || dim <= 0 || dim > 128 || vdim <= 0 || rows < 0 ||
      rows % R || (rows && !ws) ||
      (!rows && segments != B) || (kind == STATE_SPACE && (!dt || !dt_bias || !a_log)) ||
      (kind != STATE_SPACE && !decay))
    return 1;
  SegArgs a{};
  a.x = x; a.x_stride = x_stride; a.q_off = q_off; a.k_off = k_off; a.v_off = v_off;
  a.dt = dt; a.dt_stride = dt_stride; a.dt_bias = dt_bias; a.a_log = a_log; a.decay = decay; a.d_skip = d_skip;
  a.out = out; a.ws = ws; a.state = state; a.slots = slots; a.qsl = qsl; a.seq_lens = seq_lens;
  a.B = B; a.H = H; a.G = G; a.dim = dim; a.vdim = vdim; a.rows = rows; a.silu = silu; a.scale = scale;
  const int per = dtype == DT_F32 ? 4 : 8;         // elements of 16 bytes
  if (x_stride % per || (uintptr_t)x % 16 || dim % 8 || vdim % 8 || q_off % per || k_off % per || v_off % per ||
      (kind == LINEAR_CHANNEL && (uintptr_t)decay % 16))
    return 2;
  switch (dtype) {
    case DT_BF16: return kinds<bf16_t>(a, kind, segments, stream);
    case DT_F16: return kinds<f16_t>(a, kind, segments, stream);
    case DT_F32: return kinds<float>(a, kind, segments, stream);
  }
  return 1;
}
