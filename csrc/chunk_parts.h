// What the chunked kernels of the recurrent mixers share (segment_scan.hip, chunk_scan.hip): products in thirds of 32 bits, products
// of decays along rows, finding a workgroup's piece of the batch.
#pragma once
#include "common.h"
#include <math.h>
#include <type_traits>

namespace {

enum { LINEAR_HEAD = 0, LINEAR_CHANNEL = 1, STATE_SPACE = 2, DELTA_CHANNEL = 3, DELTA_HEAD = 4 };

template <typename T> __device__ __forceinline__ float ldf(const T* p) { return (float)(*p); }
// (both sides are formed: a branch around the library functions would keep their latencies from filling each other)
__device__ __forceinline__ float softplus_f(float x) {
  const float l = log1pf(expf(x > 20.f ? 20.f : x));
  return x > 20.f ? x : l;
}
__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
// e^x for x from -200 to zero, or of x and a `rest` that it had no place for.  Cody and Waite's reduction (Software Manual for the
// Elementary Functions, 1980): x = n ln 2 + r with ln 2 in two pieces, the first short enough that n times it is exact, and for
// |r| <= ln 2 / 2 a polynomial whose coefficients are a fit by weighted least squares (off by 5e-9).  Error against 64 bits, root
// mean square / largest, x in -10 .. 0: 2.6e-8 / 7.4e-8 (the library's: 2.6e-8 / 8.3e-8)
template <typename... Rest> __device__ __forceinline__ float exp_inside(float x, Rest... rest) {
  const float n = rintf(x * 1.44269504f);
  float r = fmaf(-n, 1.42860677e-6f, fmaf(-n, 0.693145752f, x));
  ((r += rest), ...);
  float p = fmaf(r, 0.0013814529f, 0.008368751f);
  p = fmaf(r, p, 0.041668393f);
  p = fmaf(r, p, 0.1666652f);
  p = fmaf(r, p, 0.49999994f);
  p = fmaf(r, p, 1.f);
  return ldexpf(fmaf(r, p, 1.f), (int)n);
}
// the same for x below -200 too, where it is zero
__device__ __forceinline__ float exp_f(float x, float rest = 0.f) {
  const bool gone = x < -200.f;                    // (a rest that is no number then, too)
  return exp_inside(gone ? -200.f : x, gone ? 0.f : rest);
}
// e^(-rate softplus(x)).  softplus(x) is softplus(-|x|) more than x where x > 0, and ln(1 + t) = 2 atanh(t / (2 + t)), whose series
// converges for t <= 1 (arguments up to 1 / 3; the coefficients are those of a fit by Chebyshev polynomials, off by 1e-9).  What the
// quotient and the last product lose to rounding goes on as a piece of its own.  Error against 64 bits, root mean square, with the
// library's exponentials and logarithm (several times the instructions) and here: rate 4, x in -6 .. -2 2.20e-8 and 2.17e-8, -2 .. 2
// 1.58e-7 and 1.14e-7, 2 .. 8 7.1e-7 and 4.8e-7; rate 16, -6 .. -2 3.9e-8 and 3.5e-8
__device__ __forceinline__ float decay_f(float x, float rate) {
  const float t = exp_f(-fabsf(x)), w = 2.f + t, wl = t - (w - 2.f), r = __builtin_amdgcn_rcpf(w);
  const float s0 = t * r, more = fmaf(-wl, s0, fmaf(-w, s0, t)) * r, s = s0 + more;
  const float z = s * s;
  const float p = fmaf(fmaf(fmaf(fmaf(0.122047015f, z, 0.106971338f), z, 0.143103123f), z, 0.199993476f), z, 0.333333403f);
  const float l = fmaf(2.f, s0, fmaf(2.f * s, z * p, 2.f * more)), plus = (x > 0.f ? x : 0.f) + l;
  const float y = -rate * plus;
  return exp_f(y, fmaf(-rate, plus, -y));
}
// a / d rounded as the division rounds it, d between 2^-96 and 2^96 and the quotient no denormal: the product with the reciprocal, and
// what that leaves over once more (with the maximum, which drops a remainder that is no number: infinities stay what they are)
__device__ __forceinline__ float quotient(float a, float d) {
  const float r = __builtin_amdgcn_rcpf(d), q = a * r;
  return fmaf(fmaxf(fmaf(-d, q, a), -3.40282347e38f), r, q);
}
// x sigmoid(x), where sigmoid(x) = 1 / (1 + t), or t / (1 + t) below zero, with t = e^-|x|.  No exponent is cut off but where t is zero,
// so that far below zero the result goes to zero as the function does.  The quotient is the product with the reciprocal and what that
// leaves over, with what 1 + t lost to rounding.  Error against 64 bits, root mean square, and of the product with the library's
// sigmoid: x in -8 .. 8 3.8e-8 and 4.5e-8, -20 .. -8 4.4e-8 and 4.6e-8, -60 .. -20 3.7e-8 and 4.4e-8, 8 .. 60 1.5e-8 and 1.8e-8
__device__ __forceinline__ float silu_f(float x) {
  const float t = exp_inside(__builtin_amdgcn_fmed3f(-fabsf(x), -200.f, 0.f));
  const float d = 1.f + t, left_out = t - (d - 1.f), a = x < 0.f ? t : 1.f, r = __builtin_amdgcn_rcpf(d), s = a * r;
  return x * fmaf(fmaf(-left_out, s, fmaf(-d, s, a)), r, s);
}

// A 32-bit value as the exact sum of three of 16 bits, 8 digits each.  Of the nine products of two such sums the six largest are
// formed, each exact, with 32-bit sums; the three left out are below 2^-21 of the product (1.9e-8 root mean square, where a rounding
// of the product is 2.5e-8), with either sign (the first third is about rounded, so that the second is as often below zero as above:
// cut off without that, every product would be 2^-24 too small).  From 3.389e38 on, 0.4 % below the largest number, the first third
// rounds to infinity, and so does the value.  Words of two values all the way: v_cvt_pk_bf16_f32 takes 12 cycles of a SIMD, what is
// here 2 to 3 each.
struct Thirds { bf16x8 h, m, l; };
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned bits(float v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ unsigned tops(float a, float b) { return __builtin_amdgcn_perm(bits(b), bits(a), 0x07060302u); }
// BESIDE: a value that is not finite may turn the second and third of its neighbour (2 i, 2 i + 1) to NaN (a third less work;
// where both belong to the same sums)
template <bool BESIDE = true> __device__ __forceinline__ Thirds thirds(f32x4 a, f32x4 b) {
  // the value less its first third, as one product of two pairs (constants in registers: as inline operands they are read as
  // pairs that hold the number twice)
  unsigned minus0 = 0x0000bf80u, minus1 = 0xbf800000u;
  asm("" : "+s"(minus0), "+s"(minus1));
  u32x4 t[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x = i < 2 ? a[2 * i] : b[2 * i - 4], y = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    float hx = fmaf(x, 0.0027f, x), hy = fmaf(y, 0.0027f, y);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const unsigned w = tops(hx, hy);
      t[p][i] = w;
      if (p == 2) break;
      if constexpr (BESIDE) {
        typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
        x = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, minus0), x, false);
        y = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, minus1), y, false);
      } else {
        x -= __builtin_bit_cast(float, bits(hx) & 0xffff0000u);
        y -= __builtin_bit_cast(float, bits(hy) & 0xffff0000u);
      }
      hx = x;
      hy = y;
    }
  }
  return {__builtin_bit_cast(bf16x8, t[0]), __builtin_bit_cast(bf16x8, t[1]), __builtin_bit_cast(bf16x8, t[2])};
}
// (of values that 16 bits hold)
__device__ __forceinline__ bf16x8 upper(f32x4 a, f32x4 b) {
  return __builtin_bit_cast(bf16x8, u32x4{tops(a[0], a[1]), tops(a[2], a[3]), tops(b[0], b[1]), tops(b[2], b[3])});
}
// What belongs to the large and to the small products of a sum.  An infinity has no thirds (its remainders are no numbers): the
// large products alone are then the result, as they are with it in one piece.
struct Sum {
  f32x4 h = {0.f, 0.f, 0.f, 0.f}, s = {0.f, 0.f, 0.f, 0.f};
};
// the values of N sums.  One instruction a value finds what is not finite, and one branch for all of them
template <int N> __device__ __forceinline__ void values(const Sum (&sum)[N], f32x4 (&v)[N]) {
  f32x4 odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = sum[i].h + sum[i].s;
#pragma unroll
    for (int e = 0; e < 4; ++e) odd[e] = fmaf(v[i][e], 0.f, odd[e]);
  }
  if (__builtin_expect(__any((odd[0] + odd[1]) + (odd[2] + odd[3]) != 0.f), 0))
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = v[i][e] != v[i][e] ? sum[i].h[e] : v[i][e];
}
// SMALL: there were small products
template <bool SMALL = true> __device__ __forceinline__ f32x4 value(const Sum& sum) {
  if constexpr (!SMALL) return sum.h;
  const Sum one[1] = {sum};
  f32x4 v[1];
  values(one, v);
  return v[0];
}
// o[m * N + n] += a[m] . x[n]; AUP, XUP: a, x are their first thirds alone.  An instruction that adds to what another has just
// added to waits for it: the M N sums take turns
template <bool AUP, bool XUP, int M, int N>
__device__ __forceinline__ void products(const Thirds (&a)[M], const Thirds (&x)[N], Sum* o) {
#define EACH(TO, A, X)                  \
  _Pragma("unroll") for (int m = 0; m < M; ++m)   \
  _Pragma("unroll") for (int n = 0; n < N; ++n) o[m * N + n].TO = mfma16(a[m].A, x[n].X, o[m * N + n].TO);
  EACH(h, h, h)
  if constexpr (!AUP) {
    EACH(s, l, h)
    EACH(s, m, h)
  }
  if constexpr (!XUP) {
    EACH(s, h, l)
    if constexpr (!AUP) EACH(s, m, m)
    EACH(s, h, m)
  }
#undef EACH
}
template <bool AUP, bool XUP, int N> __device__ __forceinline__ void products(const Thirds& a, const Thirds (&x)[N], Sum (&o)[N]) {
  const Thirds one[1] = {a};
  products<AUP, XUP>(one, x, o);
}

// a lane's four or eight values; UP: they are 16 bits wide
template <int N4, bool UP, bool BESIDE = true> __device__ __forceinline__ Thirds thirds_of(const f32x4 (&v)[N4]) {
  const f32x4 second = N4 > 1 ? v[N4 - 1] : f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (UP) return {upper(v[0], second), {}, {}};
  else return thirds<BESIDE>(v[0], second);
}
// the lane's i-th four values into LDS planes, side by side
template <bool UP, int P, int N> __device__ __forceinline__ void store4(bf16_t (&planes)[P][N], int at, const Thirds& t, int i) {
  auto four = [&](bf16x8 v) {
    return i ? __builtin_shufflevector(v, v, 4, 5, 6, 7) : __builtin_shufflevector(v, v, 0, 1, 2, 3);
  };
  *reinterpret_cast<bf16x4*>(planes[0] + at) = four(t.h);
  if constexpr (!UP) {
    *reinterpret_cast<bf16x4*>(planes[1] + at) = four(t.m);
    *reinterpret_cast<bf16x4*>(planes[2] + at) = four(t.l);
  }
}
// a lane's N values of row r, columns c0 .. (c1 given: four there and four from c1 on), into planes by column, LD to a column: two
// rows' values of a column are one word, the even row's lane writes the even columns and the odd row's, its neighbour, the odd ones
template <int LD, bool UP, int N, int P, int M>
__device__ __forceinline__ void store_columns(bf16_t (&planes)[P][M], int c0, int r, const Thirds& t, int c1 = -1) {
  const bool odd = r & 1;
  const unsigned pick = odd ? 0x03020706u : 0x05040100u;
  if (c1 < 0) c1 = c0 + 4;
  auto plane = [&](bf16_t* p, bf16x8 v) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4 w = __builtin_bit_cast(i32x4, v);
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const int near = __builtin_amdgcn_update_dpp(0, w[i], 0xB1, 0xf, 0xf, false);        // of the row r ^ 1
      const int column = (i < 2 ? c0 + 2 * i : c1 + 2 * i - 4) + odd;
      *reinterpret_cast<unsigned*>(p + column * LD + (r & ~1)) = __builtin_amdgcn_perm(near, w[i], pick);
    }
  };
  plane(planes[0], t.h);
  if constexpr (!UP) {
    plane(planes[1], t.m);
    plane(planes[2], t.l);
  }
}
template <int M, bool UP, int P, int N> __device__ __forceinline__ Thirds load_third(const bf16_t (&planes)[P][N], int at) {
  auto one = [&](const bf16_t* p) {
    if constexpr (M == 8) return *reinterpret_cast<const bf16x8*>(p + at);
    else {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(p + at);
      return __builtin_shufflevector(v, (bf16x4)(bf16_t)0.f, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  if constexpr (UP) return {one(planes[0]), {}, {}};
  else return {one(planes[0]), one(planes[1]), one(planes[2])};
}

__device__ __forceinline__ float turn(float v) {                // of the lane in front, the first of 16 from the last
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));
}
// Products over the 16 lanes of a row, four values side by side: the lanes up to and including this one, and those behind it.  One
// instruction a step (a lane without a source keeps its value); from the builtin the compiler makes three, and waits between
// them.  (A step reads what was written four instructions before; it has to be two at least, and the s_nop sees to the first.)
#define MUL4(STEP)                                               \
  "v_mul_f32_dpp %0, %0, %0 " STEP " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %1, %1, %1 " STEP " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %2, %2, %2 " STEP " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %3, %3, %3 " STEP " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void prefix_products(float& a, float& b, float& c, float& d) {
  asm("s_nop 1\n\t" MUL4("row_shr:1") MUL4("row_shr:2") MUL4("row_shr:4") MUL4("row_shr:8")
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
__device__ __forceinline__ void suffix_products(const f32x4& v, float& a, float& b, float& c, float& d) {
  a = b = c = d = 1.f;
  asm("s_nop 1\n\t"
      "v_mov_b32_dpp %0, %4 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %1, %5 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %2, %6 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %3, %7 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      MUL4("row_shl:1") MUL4("row_shl:2") MUL4("row_shl:4") MUL4("row_shl:8")
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
}
#undef MUL4
__device__ __forceinline__ void prefix_products(f32x4& v) {
  float a = v[0], b = v[1], c = v[2], d = v[3];
  prefix_products(a, b, c, d);
  v = f32x4{a, b, c, d};
}
__device__ __forceinline__ f32x4 suffix_products(const f32x4& v) {
  float a, b, c, d;
  suffix_products(v, a, b, c, d);
  return f32x4{a, b, c, d};
}

// a row's decay -> the products of its group of 16 rows' up to it, and behind it (lanes without a source get a one; through LDS,
// as __shfl goes, these were 3000 of a chunk's 14500 cycles)
template <int CTRL> __device__ __forceinline__ double row_shift(double v) {
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  const i32x2 w = __builtin_bit_cast(i32x2, v), one = __builtin_bit_cast(i32x2, 1.0);
  return __builtin_bit_cast(double, i32x2{__builtin_amdgcn_update_dpp(one[0], w[0], CTRL, 0xf, 0xf, false),
                                          __builtin_amdgcn_update_dpp(one[1], w[1], CTRL, 0xf, 0xf, false)});
}
__device__ __forceinline__ void head_products(float own, double& upto, double& behind) {
  upto = own;
  behind = row_shift<0x101>(upto);                 // (row_shl: of the lane behind)
  upto *= row_shift<0x111>(upto);
  behind *= row_shift<0x101>(behind);
  upto *= row_shift<0x112>(upto);
  behind *= row_shift<0x102>(behind);
  upto *= row_shift<0x114>(upto);
  behind *= row_shift<0x104>(behind);
  upto *= row_shift<0x118>(upto);
  behind *= row_shift<0x108>(behind);
}
// q_i G_ij k_j of a group of 16 rows with G as the product of the decays between, term by term: lane (lr, kh) has some channels of
// row lr; of the sum over them, rows 4 kh + e of column lr come back.  The rows i - m and their decays come by turning the 16
// lanes on by one each time, in registers.  own: the row's decay where it is one for all channels
template <bool CHAN, int N4>
__device__ __forceinline__ f32x4 pairs_apart(const f32x4 (&q)[N4], const f32x4 (&k)[N4], const f32x4 (&dk)[N4], float own) {
  const int lane = threadIdx.x & 63, lr = lane & 15, kh = lane >> 4;
  float pa[16], between = 1.f, oj = own;
  [[maybe_unused]] float by_row[CHAN ? 1 : 16];
#pragma unroll
  for (int m = 0; m < 16; ++m) pa[m] = 0.f;
  if constexpr (!CHAN)
#pragma unroll
    for (int m = 0; m < 16; ++m) { by_row[m] = between; between *= oj; oj = turn(oj); }
#pragma unroll
  for (int i = 0; i < 4 * N4; ++i) {
    float kj = k[i / 4][i % 4], dj = dk[i / 4][i % 4];
    between = 1.f;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      pa[m] += q[i / 4][i % 4] * (kj * (CHAN ? between : by_row[CHAN ? 0 : m]));
      kj = turn(kj);
      if constexpr (CHAN) { between *= dj; dj = turn(dj); }
    }
  }
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    float sa = pa[m];
    sa += __shfl_xor(sa, 16, 64);
    sa += __shfl_xor(sa, 32, 64);
    // lane (.., i) has the sum of row i, column i - m
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float va = __shfl(sa, 4 * kh + e, 64);
      if (4 * kh + e - m == lr) o[e] = va;
    }
  }
  return o;
}

// the sequence and its piece that the batch's piece `want` is (false: there are fewer), of pieces_of(sequence) pieces each; a
// wave's work
template <typename F> __device__ __forceinline__ bool locate(int B, int want, int& seq, int& c, F&& pieces_of) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int s0 = 0; s0 < B; s0 += 64) {
    const int cnt = s0 + lane < B ? pieces_of(s0 + lane) : 0;
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(incl, o, 64); if (lane >= o) incl += v; }
    const unsigned long long past = __ballot(base + incl > want);
    if (past) {
      const int l = __ffsll(past) - 1;
      seq = s0 + l;
      c = want - base - (__shfl(incl, l, 64) - __shfl(cnt, l, 64));
      return true;
    }
    base += __shfl(incl, 63, 64);
  }
  return false;
}

// the sequence that is place `rank` of the batch by length, longest first (up to 64 sequences; beyond, in their order): what is
// started first is what takes longest
__device__ __forceinline__ int by_length(const int* qsl, int B, int rank) {
  if (B > 64) return rank;
  const int lane = threadIdx.x & 63, n = lane < B ? qsl[lane + 1] - qsl[lane] : -1;
  int place = 0;
  for (int o = 0; o < B; ++o) {
    const int other = __shfl(n, o, 64);
    place += other > n || (other == n && o < lane);
  }
  return __ffsll(__ballot(lane < B && place == rank)) - 1;
}

}  // namespace
