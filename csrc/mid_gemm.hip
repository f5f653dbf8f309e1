// GEMM for batches of 1..1280 rows:  y[M][N] = x[M][K] . W[N][K]^T  (bf16 / f16, fp32 accumulate), plain or with
// SiLU(gate) * up over a [gate ; up] weight.
//
// In this range a step is bound by reading W once from HBM while the MFMA work per weight byte is already substantial
// (M flops per byte), and the output has too few large tiles to fill 256 CUs (N = 8192: 64 tiles of 128 columns).  Hence:
//
//  * a workgroup tile spans BM rows - all of M when M <= 256 - so every W byte is fetched from HBM once, and K is split
//    across workgroups (fp32 partial slabs, summed by a small kernel or by the next one) until the grid covers the chip;
//  * both operands go global -> LDS by LDS-DMA (`buffer_load_dwordx4 ... lds`, 8 rows x 128 bytes per wave instruction,
//    never through registers) into rings of XS and WS images of one 64-deep K tile.  What is in flight is what the rate hangs
//    on: at 5.7 TB/s a CU takes 16 KB of W in 0.73 us, an HBM round trip under load takes about 2.  Per tile the pieces of x
//    are issued before those of W, and loads retire in order: the one counted wait of a K tile leaves two (XS - 1) tiles of W
//    and one of x behind it in flight, and the tile issued right after it makes three;
//  * the 16-byte slots of a row are XOR-ed with (row >> 1) & 7 - on the per-lane SOURCE address, the LDS-DMA destination
//    being lane-linear - so the 16-lane groups of a `ds_read_b128` fragment read hit 16 distinct slots of the 256-byte bank
//    row: no bank conflicts;
//  * the fragments of the next 32-deep K step are read between the MFMAs of this one, column by column, and so are the DMA
//    issues: read in one go in front of them, they held the MFMAs up (70B gate_up at 256 rows 217 -> 187 us);
//  * one barrier per K tile, between its two K steps: behind it every wave has read all of the tile (its place in both rings
//    is free) and every wave's pieces of the next one have landed;
//  * W is read past the caches (nontemporal): it is not used again before it would be evicted, and x stays in the L2
//    (8B gate_up at 48 rows 45.7 -> 41.5 us, 70B gate_up at 256 rows 209 -> 187);
//  * ids are dealt to the XCDs in turn, and an XCD takes one run of the (slice, column tile, row tile) list: its L2 holds
//    one or two slices of x, and the row tiles of a column tile share their W.
//
// Measured in captured graphs over copies of W larger than the caches, us, against the kernels before (W in registers,
// x through LDS; a barrier-free stream at up to 8 rows) or the library; the fp32 slabs of a split K left unreduced:
//   rows          1            16           100           256
//   70B qkv       34 -> 29     36 -> 29     55 -> 37      61 -> 49       (10240 x 8192)
//   70B o         27 -> 24     28 -> 24     34 -> 30      49 -> 40       (8192 x 8192)
//   70B gate_up   162 -> 150   165 -> 154   180 -> 158    215 -> 190     (57344 x 8192, with SiLU * up)
//   70B down      87 -> 77     89 -> 77     (no) -> 87    133 -> 105     (8192 x 28672)
//   8B qkv        16 -> 11     16 -> 12     24 -> 16      28 -> 22       (6144 x 4096)
//   8B gate_up    47 -> 41     68 -> 41     58 -> 51      77 -> 62       (28672 x 4096, with SiLU * up)
// Above 256 rows W comes once a row tile and its neighbours on an XCD share it; what this kernel has over the library there are the K
// splits of long reductions, and tiles of 192 rows for what 256 would pad by a third (library -> here):
//   rows          300          557          768           1024          1280
//   8B down       76 -> 54     114 -> 74    107 -> 90     132 -> 113    147 -> 133    (4096 x 14336)
//   7B down       102 -> 65    142 -> 87    183 -> 102    191 -> 129    230 -> 159    (3584 x 18944)
//   70B down      219 -> 161 (185 in tiles of 256)                                    (8192 x 28672)
// Row-grouped form (sparse experts, rows sorted by expert): a table names each entry's weight matrix, first row and rows; rows may
// be read through the sorted list (gate and up with SiLU * up, then down, us, against tiles of 16 to 128 rows with W straight
// from memory, a gather and the activation kernel; from 72 rows an expert on the large-batch kernel's tiles of 256 are ahead):
//   64 experts of 2048 x 1408, 6 of them a row:  1 row 38 -> 33, 100 rows 228 -> 207, 400 269 -> 240, 600 309 -> 263
//   8 of 4096 x 14336, 2 a row:                  1 row 237 -> 183, 60 rows 622 -> 487, 120 724 -> 492, 200 718 -> 530
// In tiles of 256 rows it is within 7 % of the large-batch kernel both ways between 70 and 160 rows an expert, and not built.
//
// 5.7 to 6.2 TB/s of W up to 48 rows.  At 256 rows the power limit sets the pace: back to back for milliseconds, gate_up takes
// 207 - 211 us and not 187, qkv 56, o 45, down 127 (profiles/mid_gemm_tiles_mi355x.txt).  The LDS traffic of a K tile (x and W
// written once, each wave's fragments read) and its MFMAs take 2048 clocks each of about 3000.  Matrix instructions of 32x32x16
// (fewer, the same LDS reads: gate_up 227 us), four waves of twice the columns (77 / 66 us for 8B's at 256 x 128), each
// workgroup's K loop begun elsewhere and an early touch of x for the XCD's L2 (both within 1 %) were tried and left out.
#include "common.h"

namespace {

constexpr int MG_BK = 64;            // K elements per tile = 128 bytes per row
enum { MG_EPI_NONE = 0, MG_EPI_SILU_MUL = 2 };     // as in stream_gemm.hip
typedef __attribute__((address_space(3))) void mg_lds_void;

// WM waves along the rows, WN along the columns; XS <= WS: images of x and W kept
// GROUPED (rows sorted by expert): tiles [n, 3] = (weight matrix, first row, rows <= BM; 0 = nothing), matrices w_group elements
// apart; src != null: row r of the product is row src[r] of x
template <typename T, int BM, int BN, int WM, int WN, int XS, int WS, int EPI, bool GROUPED>
__global__ __launch_bounds__(WM * WN * 64) void mid_gemm_kernel(const T* x, long x_stride, const T* w, long w_stride, T* out,
                                                          long out_stride, float* partial, int M, int N, int K, int ksplit,
                                                          int ntn, int up_row, const int* __restrict__ tiles, long w_group,
                                                              const int* __restrict__ src, int x_rows, const T* bias) {
#if defined(__HIP_DEVICE_COMPILE__)
  using V8 = typename Vec8<T>::type;
  constexpr int WAVES = WM * WN, FM = BM / WM / 16, FN = BN / WN / 16;
  constexpr int PX = BM / 8 / WAVES, PW = BN / 8 / WAVES;      // 1 KiB pieces per wave and K tile
  constexpr int XB = BM * 128, WB = BN * 128;
  constexpr int MG_NT = 2;           // cache policy of W's loads: nontemporal
  static_assert(XS >= 2 && WS >= XS && WS <= XS + 1 && XS * XB + WS * WB <= 160 * 1024, "unsupported tile");
  static_assert(EPI != MG_EPI_SILU_MUL || FN % 2 == 0, "unsupported tile");
  // loads of a wave behind x and W of the tile that a wait is for: with WS > XS that W is older than that x
  constexpr int AHEAD = WS > XS ? (XS - 1) * PW + (XS - 2) * PX : (XS - 2) * (PX + PW);
  __shared__ __attribute__((aligned(1024))) unsigned char smem[XS * XB + WS * WB];
  unsigned char* const smw = smem + XS * XB;

  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid % WM, wn = wid / WM;
  const int r16 = lane & 15, q = lane >> 4;
  int m0, mrows, ks, tn;
  if constexpr (GROUPED) {                 // (column tiles of an entry side by side: the entries used come first, so the XCDs share them)
    const int entry = blockIdx.x / ntn;
    tn = blockIdx.x - entry * ntn;
    ks = 0;
    m0 = tiles[3 * entry + 1];
    mrows = min(tiles[3 * entry + 2], min(BM, M - m0));
    if (mrows <= 0) return;
    w += tiles[3 * entry] * w_group;
  } else {
    const int per = gridDim.x >> 3, work = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int ntm = (M + BM - 1) / BM;
    if (work >= ntn * ksplit * ntm) return;
    const int mt = work % ntm, wide = work / ntm;
    ks = wide / ntn;
    tn = wide - ks * ntn;
    m0 = mt * BM;
    mrows = min(BM, M - m0);
  }
  const int KT = K / MG_BK;
  const int kt_lo = (int)((long)KT * ks / ksplit), kt_hi = (int)((long)KT * (ks + 1) / ksplit);
  const int nt = kt_hi - kt_lo;
  if (nt <= 0) return;                     // block-uniform; cannot happen for ksplit <= K / 64
  const int last = nt - 1;

  // row of W behind row r of the tile, from the tile's first one: plain, tn * BN ..; with SiLU, BN / 2 gate rows and as many up
  // rows in turns of half a wave's columns, so that a lane holds gate and up of the same column.  Columns past N repeat the last.
  const int first = EPI == MG_EPI_SILU_MUL ? tn * (BN / 2) : tn * BN;
  auto w_row = [&](int r) {
    if constexpr (EPI == MG_EPI_SILU_MUL) {
      constexpr int H = BN / WN / 2;
      const int col = min(r / (2 * H) * H + r % H, up_row - 1 - first);
      return r % (2 * H) < H ? col : up_row + col;
    }
    return min(r, N - 1 - first);
  };
  const int wrows = EPI == MG_EPI_SILU_MUL ? N - first : min(BN, N - first);
  // (the spans fit 32 bits: checked on the host)
  const bool gather = GROUPED && src != nullptr;
  const auto xrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(gather ? x : x + (long)m0 * x_stride), 0,
                                                       (int)((((gather ? x_rows : mrows) - 1) * x_stride + K) * 2), 0x00020000);
  const auto wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(w + (long)first * w_stride), 0,
                                                       (int)(((wrows - 1) * w_stride + K) * 2), 0x00020000);
  unsigned offx[PX], offw[PW];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int r = 8 * (wid * PX + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int row = min(r, mrows - 1);
    offx[i] = ((unsigned)(gather ? src[m0 + row] : row) * (unsigned)x_stride + kt_lo * MG_BK + 8 * c) * 2;
  }
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int r = 8 * (wid * PW + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    offw[i] = ((unsigned)w_row(r) * (unsigned)w_stride + kt_lo * MG_BK + 8 * c) * 2;
  }
  const int swz = (r16 >> 1) & 7;
  const int so[2] = {(q ^ swz) << 4, ((4 + q) ^ swz) << 4};
  const int xro = (wm * FM * 16 + r16) * 128, wro = (wn * FN * 16 + r16) * 128;

  f32x4 acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  V8 xf[2][FM], wf[2][FN];
  constexpr int XR = (FM + FN - 1) / FN, LR = (PX + PW + FN - 1) / FN;
  // the j-th of FN parts of a K step's fragment reads, and of a K tile's DMA
  auto read = [&](int s, int sx, int sw, int j) {
    const unsigned char* bx = smem + sx * XB + xro + so[s];
    const unsigned char* bw = smw + sw * WB + wro + so[s];
#pragma unroll
    for (int i = j * XR; i < (j + 1) * XR && i < FM; ++i) xf[s][i] = *reinterpret_cast<const V8*>(bx + i * 2048);
    wf[s][j] = *reinterpret_cast<const V8*>(bw + j * 2048);
  };
  // (past the last tile it is fetched again and never used: the counted waits need the same loads in every iteration)
  auto load_x = [&](int stage, int t, int p) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, (mg_lds_void*)(smem + stage * XB + (wid * PX + p) * 1024), 16, offx[p],
                                             min(t, last) * 128, 0, 0);
  };
  auto load_w = [&](int stage, int t, int p) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wrsrc, (mg_lds_void*)(smw + stage * WB + (wid * PW + p) * 1024), 16, offw[p],
                                             min(t, last) * 128, 0, MG_NT);
  };
  auto load = [&](int sx, int sw, int t, int j) {
#pragma unroll
    for (int i = j * LR; i < (j + 1) * LR && i < PX + PW; ++i) {
      if (i < PX) load_x(sx, t + XS, i);
      else load_w(sw, t + WS, i - PX);
    }
  };
  auto mma = [&](int s, int j) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = mfma16(wf[s][j], xf[s][i], acc[j][i]);
    __builtin_amdgcn_s_setprio(0);
  };

  // as iterations -WS .. -2 of the loop would have issued them
#pragma unroll
  for (int i = -WS; i < -1; ++i) {
    if (i + XS >= 0)
#pragma unroll
      for (int p = 0; p < PX; ++p) load_x(i + XS, i + XS, p);
#pragma unroll
    for (int p = 0; p < PW; ++p) load_w(i + WS, i + WS, p);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < FN; ++j) load(XS - 1, WS - 1, -1, j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < FN; ++j) read(0, 0, 0, j);
  int sx = 0, sw = 0;
  for (int t = 0; t < nt; ++t) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      read(1, sx, sw, j);
      __builtin_amdgcn_sched_barrier(0);
      mma(0, j);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(AHEAD) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int nx = sx + 1 == XS ? 0 : sx + 1, nw = sw + 1 == WS ? 0 : sw + 1;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      load(sx, sw, t, j);
      read(0, nx, nw, j);
      __builtin_amdgcn_sched_barrier(0);
      mma(1, j);
      __builtin_amdgcn_sched_barrier(0);
    }
    sx = nx;
    sw = nw;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // the tail prefetches must not outlive the LDS

  // ---- lane (r16, q) of fragment (j, i) holds y[row 16 i + r16][column 16 j + 4 q .. + 4] of the wave's part
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + (wm * FM + i) * 16 + r16;
    if (m >= m0 + mrows) continue;
    if constexpr (EPI == MG_EPI_SILU_MUL) {
#pragma unroll
      for (int j = 0; j < FN / 2; ++j) {
        const int n = tn * (BN / 2) + (wn * (FN / 2) + j) * 16 + 4 * q;
        if (n >= up_row) continue;
        typename Vec4<T>::type o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (T)(fast_silu(acc[j][i][r]) * acc[FN / 2 + j][i][r]);
        *reinterpret_cast<typename Vec4<T>::type*>(out + (long)m * out_stride + n) = o;
      }
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = tn * BN + (wn * FN + j) * 16 + 4 * q;
        if (n >= N) continue;                // N % 16 == 0: a fragment column group is all in or all out
        if (ksplit == 1) {
          typename Vec4<T>::type o;
          if (!GROUPED && bias != nullptr) {
            const typename Vec4<T>::type add = *reinterpret_cast<const typename Vec4<T>::type*>(bias + n);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[j][i][r] += (float)add[r];
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (T)acc[j][i][r];
          *reinterpret_cast<typename Vec4<T>::type*>(out + (long)m * out_stride + n) = o;
        } else {
          *reinterpret_cast<f32x4*>(partial + ((size_t)ks * M + m) * N + n) = acc[j][i];
        }
      }
    }
  }
#endif
}

template <typename T>
__global__ void mid_reduce_kernel(T* __restrict__ out, long out_stride, const float* __restrict__ partial, int M,
                                  int N, int ksplit, const T* __restrict__ bias) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int n4 = N >> 2;
  if (idx >= (long)M * n4) return;
  const unsigned mu = (unsigned)idx / (unsigned)n4;        // (M * N / 4 < 2^31: no 64-bit division)
  const int m = (int)mu, n = (int)((unsigned)idx - mu * (unsigned)n4) * 4;
  f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < ksplit; ++k) s += *reinterpret_cast<const f32x4*>(partial + ((size_t)k * M + m) * N + n);
  typename Vec4<T>::type o, add = {};
  if (bias != nullptr) add = *reinterpret_cast<const typename Vec4<T>::type*>(bias + n);
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = (T)(s[r] + (float)add[r]);
  *reinterpret_cast<typename Vec4<T>::type*>(out + (long)m * out_stride + n) = o;
}

template <typename T, int BM, int BN, int WM, int WN, int XS, int WS>
int launch(const void* x, long xs, const void* w, long ws, void* out, long os, const void* bias, void* partial, int M, int N, int K,
           int ksplit, int epi, hipStream_t st) {
  const bool silu = epi == MG_EPI_SILU_MUL;
  const int ntn = silu ? (N / 2 + BN / 2 - 1) / (BN / 2) : (N + BN - 1) / BN;
  const int grid = (ntn * ksplit * ((M + BM - 1) / BM) + 7) / 8 * 8;
#define MG_GO(EPI)                                                                                                             \
  mid_gemm_kernel<T, BM, BN, WM, WN, XS, WS, EPI, false><<<grid, WM * WN * 64, 0, st>>>(                                       \
      (const T*)x, xs, (const T*)w, ws, (T*)out, os, (float*)partial, M, N, K, ksplit, ntn, N / 2, nullptr, 0, nullptr, 0, (const T*)bias)
  if (silu) MG_GO(MG_EPI_SILU_MUL);
  else MG_GO(MG_EPI_NONE);
#undef MG_GO
  HIP_LAUNCH_CHECK();
  if (ksplit > 1 && out != nullptr) {            // out == nullptr: the caller consumes the K-split slabs itself
    const long n = (long)M * (N / 4);
    mid_reduce_kernel<T><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((T*)out, os, (const float*)partial, M, N,
                                                                     ksplit, (const T*)bias);
    HIP_LAUNCH_CHECK();
  }
  return 0;
}

template <typename T, int BM, int BN, int WM, int WN, int XS, int WS>
int launch_grouped(const void* x, long xs, const void* w, long ws, long w_group, void* out, long os, const int* tiles, int num_tiles,
                   const int* src, int x_rows, int M, int N, int K, int epi, hipStream_t st) {
  const bool silu = epi == MG_EPI_SILU_MUL;
  const int ntn = silu ? (N / 2 + BN / 2 - 1) / (BN / 2) : (N + BN - 1) / BN;
#define MG_GO(EPI)                                                                                                             \
  mid_gemm_kernel<T, BM, BN, WM, WN, XS, WS, EPI, true><<<ntn * num_tiles, WM * WN * 64, 0, st>>>(                             \
      (const T*)x, xs, (const T*)w, ws, (T*)out, os, nullptr, M, N, K, 1, ntn, N / 2, tiles, w_group, src, x_rows, nullptr)
  if (silu) MG_GO(MG_EPI_SILU_MUL);
  else MG_GO(MG_EPI_NONE);
#undef MG_GO
  HIP_LAUNCH_CHECK();
  return 0;
}

// 64 rows: two workgroups of four waves to a CU (72 KB), which level out what is left of a round (eight waves, each with half
// the columns, read more of LDS: 70B down at 48 rows 81 us, so 77); larger tiles take a CU each
template <typename T>
int dispatch(const void* x, long xs, const void* w, long ws, void* out, long os, const void* bias, void* partial, int M, int N,
             int K, int ksplit, int bm, int bn, int epi, hipStream_t st) {
#define MG_CASE(BM, BN, WM, WN, XS, WS) \
  if (bm == BM && bn == BN) return launch<T, BM, BN, WM, WN, XS, WS>(x, xs, w, ws, out, os, bias, partial, M, N, K, ksplit, epi, st);
  MG_CASE(256, 256, 4, 2, 2, 3)
  MG_CASE(256, 128, 2, 4, 3, 4)
  MG_CASE(192, 256, 2, 4, 2, 3)
  MG_CASE(192, 128, 4, 2, 3, 4)
  MG_CASE(128, 256, 2, 4, 2, 3)
  MG_CASE(128, 128, 4, 2, 4, 5)
  MG_CASE(64, 128, 2, 2, 3, 3)
#undef MG_CASE
  return -4;
}

}  // namespace

// out = epilogue(x[M][K] . w[N][K]^T).  K % 64 == 0, N % 16 == 0; strides in elements, multiples of 8; pointers 16-byte
// aligned.  (bm, bn) is the workgroup tile: (256 | 192 | 128, 128 | 256), (64, 128).
// epi 0: out[M][N], with bias[N] (or null, 8-byte aligned) added before the one rounding; partial holds ksplit * M * N floats
// when ksplit > 1, and out may be null then: the slabs are the result.
// epi 2: w = [gate ; up], N % 32 == 0, ksplit 1, out[M][N/2] = silu(gate) * up.
VDAMD_API int vdamd_mid_gemm(void* out, long out_stride, const void* x, long x_stride, const void* w, long w_stride,
                             const void* bias, void* partial, int M, int N, int K, int ksplit, int bm, int bn, int epi,
                             int dtype, void* stream) {
  if (M <= 0) return 0;
  if (K % MG_BK || N % 16 || ksplit < 1 || ksplit > K / MG_BK) return -1;
  if (epi != MG_EPI_NONE && (epi != MG_EPI_SILU_MUL || N % 32 || ksplit != 1)) return -1;
  if (ksplit > 1 && partial == nullptr) return -2;
  if (out == nullptr && ksplit == 1) return -2;
  if (bias != nullptr && (epi != MG_EPI_NONE || out == nullptr || (uintptr_t)bias % 8)) return -2;
  if ((x_stride | w_stride) % 8 || out_stride % 4) return -5;
  if (((uintptr_t)x | (uintptr_t)w) % 16 || (uintptr_t)out % 8) return -8;
  const long lim = (1L << 32) - 64;                // bytes that a tile's buffer descriptor spans
  if ((long)(M < bm ? M : bm) * x_stride * 2 >= lim || (long)(epi == MG_EPI_SILU_MUL ? N : bn) * w_stride * 2 >= lim) return -7;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DT_BF16)
    return dispatch<bf16_t>(x, x_stride, w, w_stride, out, out_stride, bias, partial, M, N, K, ksplit, bm, bn, epi, st);
  if (dtype == DT_F16)
    return dispatch<f16_t>(x, x_stride, w, w_stride, out, out_stride, bias, partial, M, N, K, ksplit, bm, bn, epi, st);
  return -3;
}

// Row-grouped form: out rows [tiles[i][1], + tiles[i][2]) = epilogue(x rows . w[tiles[i][0]]^T), tiles [num_tiles, 3] on the device,
// at most bm rows each (0: skipped), every row inside the M of out and x (src != null: of src, whose entries are the rows of
// x [x_rows]); w [groups, N, K] with matrices w_group elements apart.  epi 0 or 2 as above; rows of no tile stay as they are.
VDAMD_API int vdamd_mid_gemm_grouped(void* out, long out_stride, const void* x, long x_stride, const void* w, long w_stride,
                                     long w_group, const int* tiles, int num_tiles, const int* src, int x_rows, int M, int N, int K,
                                     int bm, int bn, int epi, int dtype, void* stream) {
  if (M <= 0 || num_tiles <= 0) return 0;
  if (K % MG_BK || N % 16 || (epi != MG_EPI_NONE && (epi != MG_EPI_SILU_MUL || N % 32))) return -1;
  if ((x_stride | w_stride | w_group) % 8 || out_stride % 4) return -5;
  if (src != nullptr && x_rows <= 0) return -4;
  if (((uintptr_t)x | (uintptr_t)w) % 16 || (uintptr_t)out % 8) return -8;
  const long lim = (1L << 32) - 64;
  if ((long)(src != nullptr ? x_rows : bm) * x_stride * 2 >= lim || (long)(epi == MG_EPI_SILU_MUL ? N : bn) * w_stride * 2 >= lim) return -7;
  hipStream_t st = (hipStream_t)stream;
#define MG_CASE(T, BM, BN, WM, WN, XS, WS) \
  if (bm == BM && bn == BN)                \
    return launch_grouped<T, BM, BN, WM, WN, XS, WS>(x, x_stride, w, w_stride, w_group, out, out_stride, tiles, num_tiles, src, x_rows, M, N, K, epi, st);
#define MG_CASES(T)                \
  MG_CASE(T, 128, 128, 4, 2, 4, 5) \
  MG_CASE(T, 64, 128, 2, 2, 3, 3)
  if (dtype == DT_BF16) { MG_CASES(bf16_t) return -4; }
  if (dtype == DT_F16) { MG_CASES(f16_t) return -4; }
#undef MG_CASES
#undef MG_CASE
  return -3;
}
