// Unquantized-activation GEMMs on the matrix cores over unpacked weights:
// out (rows, N) fp32 = A (rows, K) . W (N, K)^T with A in bf16 or fp32 and W
// in bf16, FP8 (e4m3 with fp32 block scales) or MXFP4 (e2m1 with e8m0 / 32),
// plain or as a SwiGLU pair, for one matrix or for a layer's row tiles.
//
// Serves the bf16-weight MoE layer (moe_layer.hip) and the standalone FP8
// and MXFP4 linears (compat_gemm.hip) from the few rows on at which the
// per-wave GEMV (decode.hip), which multiplies on the vector ALU and passes
// over the weights once per four rows, is not bound by the weight stream any
// more (bf16_gemv, fp8_few_rows, fp4_few_rows).
//
// fp32 precision on bf16 MFMAs. An fp32 activation, times a power of two, is
// the exact sum of three bf16 values, its significand cut in 8 + 8 + 8 bits
// (split3), and every
// weight format here is exact in bf16 (FP8 before its block scale), so the
// three products per weight are exact and are added in fp32: the arithmetic
// of an fp32 dot product, in another order. bf16 activations (x) need one
// product. FP8 block scales multiply the fp32 partial sum of each 64-wide K
// step.
//
// Tile. Eight waves; a workgroup owns BM rows (16, 32 or 64) and WN waves'
// columns, each NC 16-column subtiles wide; the other 8 / WN split every K
// step, so that a few rows still keep eight waves' weight loads in flight
// and the K loop short; their sums meet in LDS at the end, added pairwise.
// Activations go through LDS (bf16 planes, double buffered, one barrier a
// step, split once per workgroup); weights go straight to the wave that
// multiplies them, three K steps ahead, in the K order that makes a
// lane's load 16 or 32 contiguous bytes (lane group g takes K [16 g, +16) of
// a 64-wide step for both operands).
//
// What bounds it: latency, with two waves a SIMD and a barrier a step. Of the
// cycles of an FP8 512 x 4096 x 4096 launch the matrix cores are busy in 24%
// and the vector ALU in 22% (the split, 4.5 instructions an element, is
// repeated by every column tile; the FP8 conversion one per two weights), the
// waves wait for 44% of their time, LDS conflicts take 6%; MXFP4 300 x 2048 x 7168
// 15, 18, 28 and 7% with 160 workgroups on 256 CUs; the bf16 layer's gate/up at
// 1000 tokens 9, 12, 43 and 4%, 64% L2 hits. FP8 512 x 4096 x 4096: 738 us on
// the tiled kernel, 54 here (0.95 PFLOP/s of bf16 products, the product itself
// 317 TFLOP/s); 32 rows 67 -> 12 us. MXFP4 300 x 2048 x 7168: 772 -> 67 us. bf16
// layer (H 1024, E 16, I 512, top-4, a shared expert): 64 tokens 212 -> 43 us,
// 1000 tokens 2712 -> 108 us (32 x 128 tiles: 153 us). Against 64 bits the error
// is below that of the tiled kernel (linears 1.3e-7 and 1.6e-7, there 1.1e-6 and
// 1.4e-6) and of the GEMV with fp32 wave sums that it was measured against
// (layer 1.5e-7 to 1.8e-7 up to 64 tokens).
#include "launch.h"

namespace sllm {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int WD_THREADS = 512;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// upper halves of a (low half of the result) and b
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// v0 and v1 minus the low and the high bf16 of p, exactly: one
// v_dot2_f32_bf16 each, (p.lo, p.hi) . (-1, 0) + v and (0, -1). The (-1, 0)
// operand goes through a register: an inline -1.0 is a 32-bit pattern, which
// this instruction reads as (0, -1).
__device__ __forceinline__ void sub_bf16(float& v0, float& v1, uint32_t p,
                                         uint32_t m1lo) {
  const bf16x2 q = __builtin_bit_cast(bf16x2, p);
  v0 = __builtin_amdgcn_fdot2_f32_bf16(q, __builtin_bit_cast(bf16x2, m1lo), v0, false);
  v1 = __builtin_amdgcn_fdot2_f32_bf16(q, __builtin_bit_cast(bf16x2, 0xBF800000u), v1, false);
}

// fp32 activations are multiplied by 2^A_UP before they are cut, and the sums
// by 2^-A_UP at the end: bf16's smallest step is 2^-133, and v_dot2_f32_bf16
// drops results below 2^-126, so that unscaled the mid and lo parts of values
// below 2^-109 lost bits (2^-118: 2e-5 off, 2^-130: 7%). Scaled, every fp32
// value keeps all of them.
constexpr int A_UP = 40;

// Two fp32 values, scaled, as three bf16 pairs each cut off (truncated) in
// turn: hi + mid + lo is the value exactly (8 + 8 + 8 significand bits). An
// infinity or NaN, or a value past 2^88 (or of less, whose products are past
// it), gives its row's sums infinities or NaN, which are taken again.
__device__ __forceinline__ void split3(float a, float b, uint32_t m1lo,
                                       uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  constexpr float UP = (float)(1ull << A_UP);
  float ra = a * UP, rb = b * UP;
  hi = pack_hi(ra, rb);
  sub_bf16(ra, rb, hi, m1lo);
  mid = pack_hi(ra, rb);
  sub_bf16(ra, rb, mid, m1lo);
  lo = pack_hi(ra, rb);
}

// e4m3 is exact in bf16; v_cvt_scalef32_pk_bf16_fp8 at scale 1 converts two
// bytes (every pair of finite codes is tested)
__device__ __forceinline__ bf16x8 e4m3x8(uint32_t d0, uint32_t d1) {
  const u32x4 r = {
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.f, false)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.f, true)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.f, false)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.f, true))};
  return __builtin_bit_cast(bf16x8, r);
}

// 8 e2m1 values times 2^(sb - 127): exact in bf16; scale byte 0 is zero, 255
// a NaN (the conversion reads 0 as 2^-127, so the data is zeroed)
__device__ __forceinline__ bf16x8 e2m1x8(uint32_t d, uint32_t sb) {
  d = sb ? d : 0u;
  const float s = __uint_as_float(sb << 23);
  const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 0);
  const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 1);
  const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 2);
  const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 3);
  const u32x4 r = {__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1),
                   __builtin_bit_cast(uint32_t, p2), __builtin_bit_cast(uint32_t, p3)};
  return __builtin_bit_cast(bf16x8, r);
}

// One lane's 16 K values of a weight row, as stored.
template <int WF>
struct WBytes {
  static constexpr int regs = WF == WD_BF16 ? 8 : (WF == WD_FP8 ? 4 : 2);
};

// MFMA operand of K half m (8 values) of a lane's 16.
template <int WF>
__device__ __forceinline__ bf16x8 w_frag(const uint32_t* r, int m, uint32_t sb) {
  if constexpr (WF == WD_BF16) {
    const u32x4 v = {r[4 * m], r[4 * m + 1], r[4 * m + 2], r[4 * m + 3]};
    return __builtin_bit_cast(bf16x8, v);
  } else if constexpr (WF == WD_FP8) {
    return e4m3x8(r[2 * m], r[2 * m + 1]);
  } else {
    return e2m1x8(r[m], sb);
  }
}

// Row n of weight block e against the fp32 row a by plain fp32 products, the
// weight scaled first, by a whole wave (each lane 16 values of every 1024).
template <int WF>
__device__ float plain_dot(const WideSeg& S, const float* a, int e, int n, int lane) {
  const int K = S.K;
  const size_t row = (size_t)e * S.N + n;
  float sum = 0.f;
  for (int k = 16 * lane; k < K; k += 1024) {
    float w[16], d = 0.f;
    if constexpr (WF == WD_FP8) {
      const uint4 q = *(const uint4*)(S.w0 + row * K + k);
      const uint32_t b[4] = {q.x, q.y, q.z, q.w};
      const float s = ((const float*)S.s0)[(size_t)(n / S.bh) * ((K + (64 << S.bws) - 1) >> (6 + S.bws)) +
                                           (k >> (6 + S.bws))];
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = e4m3_to_f32(b[i / 4], i & 3) * s;
    } else {
      bf16x8 h[2];
      if constexpr (WF == WD_FP4) {
        const uint2 q = *(const uint2*)(S.w0 + row * (K / 2) + k / 2);
        const uint32_t sb = ((const uint8_t*)S.s0)[row * (K / 32) + k / 32];
        h[0] = e2m1x8(q.x, sb);
        h[1] = e2m1x8(q.y, sb);
      } else {
        h[0] = *(const bf16x8*)(S.w0 + (row * K + k) * 2);
        h[1] = *(const bf16x8*)(S.w0 + (row * K + k) * 2 + 16);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = (float)h[i / 8][i % 8];
    }
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const float4 v = *(const float4*)(a + k + i);
      d = fmaf(v.x, w[i], d);
      d = fmaf(v.y, w[i + 1], d);
      d = fmaf(v.z, w[i + 2], d);
      d = fmaf(v.w, w[i + 3], d);
    }
    sum += d;
  }
  return wave_sum(sum);
}

template <int WF, bool A32, bool SWIGLU, int BM, int WN, int NC>
__global__ __launch_bounds__(WD_THREADS) void wide_kernel(WideSeg S0, WideSeg S1,
                                                          int blocks0, int topk) {
  constexpr int WK = 8 / WN, RB = BM / 16;
  constexpr int KT = 64 * WK;        // K of one step over the K waves
  constexpr int LS = KT + 8;         // LDS row stride (elements, 16 B of pad)
  constexpr int PL = A32 ? 3 : 1;    // bf16 planes of the activations
  constexpr int NO = SWIGLU ? NC / 2 : NC;  // output subtiles of a wave
  constexpr int BN = 16 * NO * WN;   // output columns of the workgroup
  constexpr int CE = A32 ? 4 : 8;    // elements of a 16-byte activation chunk
  constexpr int NA = BM * KT / CE / WD_THREADS;  // such chunks per thread
  constexpr int NW = WBytes<WF>::regs;
  static_assert(NA >= 1 && NA * CE * WD_THREADS == BM * KT, "whole chunks");
  // gate/up up to 32-row tiles: the K steps' sum keeps its rounding errors
  // beside it (of each step whose partial is below the sum, most of it else:
  // the two-operand form). Layer against 64 bits at 64 tokens, H 1024 / 2048: 1.64e-7 /
  // 1.98e-7 without (the GEMV with fp32 wave sums 1.60e-7 / 1.82e-7, now 1.20e-7
  // with 64-bit ones), 1.48e-7 / 1.69e-7 with it, for 1
  // to 3% of the layer's time (41.9 -> 42.9 us, 104 -> 106); in the down launch
  // too 1.46e-7 / 1.64e-7 for twice that. 64-row tiles are below the GEMV that
  // they replaced without it (1.82e-7 against 1.84e-7, 2.3e-7 against 3.6e-7).
  constexpr bool COMP = SWIGLU && BM <= 32;
  constexpr int TILE = PL * BM * LS;  // elements of one step's tile
  constexpr int RED = WK > 1 ? (8 - WN) * RB * NC * 64 * 8 : 0;  // (bf16 sized)
  // (two arrays: a step's reads of one cannot alias its writes of the other)
  __shared__ __attribute__((aligned(16))) uint16_t a_lds0[TILE > RED ? TILE : RED];
  __shared__ __attribute__((aligned(16))) uint16_t a_lds1[TILE];
  __shared__ int rsrc[BM];

  const bool second = (int)blockIdx.x >= blocks0;
  const WideSeg& S = second ? S1 : S0;
  const int b = second ? blockIdx.x - blocks0 : blockIdx.x;
  const int NS = (S.N + BN - 1) / BN;
  // column slabs vary fastest: with a multiple of eight of them a slab's row
  // tiles run on one XCD and share its weights in that L2 (with four, as the
  // bf16 layer's gate/up at I 512, on two)
  const int rt = b / NS, ns = b % NS;
  int e = 0, rb0 = rt * BM, rows;
  if (S.tile_info) {
    if (rt >= *S.num_tiles) return;
    const int4 d = *(const int4*)(S.tile_info + 4 * rt);
    e = d.x;
    rb0 = d.y;
    rows = min(BM, d.z);
  } else {
    rows = min(BM, S.total_rows - rb0);
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lg = lane >> 4, lc = lane & 15;
  const int wk = wave / WN, wn = wave % WN;
  if (tid < BM) {  // rows past the tile repeat its last row; never stored
    const int p = rb0 + min(tid, rows - 1);
    rsrc[tid] = S.gather && S.sorted_idx ? S.sorted_idx[p] / topk : p;
  }
  __syncthreads();

  const int K = S.K, N = S.N;
  const int steps = (K + KT - 1) / KT;
  // ---- addresses ------------------------------------------------------------
  const uint8_t* ap[NA];
  int arow[NA], acol[NA], aoff[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    const int id = q * WD_THREADS + tid;
    const int row = id / (KT / CE), c = id % (KT / CE);
    ap[q] = (const uint8_t*)S.a + (size_t)rsrc[row] * K * (A32 ? 4 : 2);
    arow[q] = row;
    acol[q] = c * CE;
    aoff[q] = row * LS + c * CE;
  }
  const int ncol = ns * BN + wn * 16 * NO;  // the wave's first output column
  const uint8_t* wp[NC];
  const uint8_t* sp[NC];  // MXFP4 scale bytes of the lane's row
  const float* fs[NC];    // FP8: block scales of the subtile's rows
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int oc = SWIGLU ? c % NO : c;
    const int n = min(ncol + oc * 16 + lc, N - 1);
    const uint8_t* base = SWIGLU && c >= NO ? S.w1 : S.w0;
    const size_t row = (size_t)e * N + n;
    if constexpr (WF == WD_BF16) wp[c] = base + (row * K + 16 * lg) * 2;
    else if constexpr (WF == WD_FP8) wp[c] = base + row * K + 16 * lg;
    else wp[c] = base + row * (K / 2) + 8 * lg;
    if constexpr (WF == WD_FP4)
      sp[c] = (const uint8_t*)S.s0 + row * (K / 32) + lg / 2;
    if constexpr (WF == WD_FP8)  // the block of the lane's four result rows
      fs[c] = (const float*)S.s0 + (size_t)(min(ncol + oc * 16 + 4 * lg, N - 1) / S.bh) *
                                       ((K + (64 << S.bws) - 1) >> (6 + S.bws));
  }

  struct Set {
    uint4 a[NA];
    uint32_t w[NC][NW];
    uint32_t sb[NC];
    float f[NC];
  };
  // step s's operands; past the last step (and for a K wave past K) the
  // last ones again, loaded and not used
  auto load = [&](Set& t, int s) {
    const int kb = min(s, steps - 1) * KT;
#pragma unroll
    for (int q = 0; q < NA; ++q)
      t.a[q] = *(const uint4*)(ap[q] + (size_t)min(kb + acol[q], K - CE) * (A32 ? 4 : 2));
    const int kk = min(kb + __builtin_amdgcn_readfirstlane(wk) * 64, K - 64);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (WF == WD_BF16) {
        const uint4 lo = *(const uint4*)(wp[c] + (size_t)kk * 2);
        const uint4 hi = *(const uint4*)(wp[c] + (size_t)kk * 2 + 16);
        t.w[c][0] = lo.x; t.w[c][1] = lo.y; t.w[c][2] = lo.z; t.w[c][3] = lo.w;
        t.w[c][4] = hi.x; t.w[c][5] = hi.y; t.w[c][6] = hi.z; t.w[c][7] = hi.w;
      } else if constexpr (WF == WD_FP8) {
        const uint4 v = *(const uint4*)(wp[c] + kk);
        t.w[c][0] = v.x; t.w[c][1] = v.y; t.w[c][2] = v.z; t.w[c][3] = v.w;
        t.f[c] = fs[c][kk >> (6 + S.bws)];
      } else {
        const uint2 v = *(const uint2*)(wp[c] + kk / 2);
        t.w[c][0] = v.x; t.w[c][1] = v.y;
        t.sb[c] = sp[c][kk / 32];
      }
    }
  };

  f32x4 acc[RB][NC];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[r][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
  f32x4 low[COMP ? RB : 1][COMP ? NC : 1] = {};

  uint32_t m1lo = 0x0000BF80u;  // bf16 (-1, 0), kept in a register
  asm("" : "+v"(m1lo));
  // chunk q of a set's activations -> a step's tile
  auto stage = [&](uint16_t* tile, const Set& t, int q) {
    // 16-row tiles serve a few rows: those past the item are left as they
    // are (their products are never stored) and cost no split
    if (BM == 16 && arow[q] >= rows) return;
    uint16_t* d = tile + aoff[q];
    const uint4 v = t.a[q];
    if constexpr (A32) {
      uint32_t h0, m0, l0, h1, m1, l1;
      split3(__uint_as_float(v.x), __uint_as_float(v.y), m1lo, h0, m0, l0);
      split3(__uint_as_float(v.z), __uint_as_float(v.w), m1lo, h1, m1, l1);
      *(uint2*)d = make_uint2(h0, h1);
      *(uint2*)(d + BM * LS) = make_uint2(m0, m1);
      *(uint2*)(d + 2 * BM * LS) = make_uint2(l0, l1);
    } else {
      *(uint4*)d = v;
    }
  };
  auto multiply = [&](const uint16_t* tile, const Set& cur) {
    const uint16_t* a = tile + lc * LS + wk * 64 + 16 * lg;
    f32x4 part[RB][NC];
    // Fragments are read PL RB units ahead. bf16 weights take both K halves'
    // low parts first, so that the sums round while they are small (64-token
    // layer 1.7e-7 -> 1.6e-7 off 64 bits); the converted formats,
    // which would hold both halves' weights for it (512 x 4096 x 4096 58.9 ->
    // 61.8 us), one K half after the other.
    constexpr int U = PL * RB;  // fragments of a K half; 2 U in all
    constexpr bool LOW = WF == WD_BF16;
    bf16x8 x[U], w[2][NC];
    auto half_of = [](int i) { return LOW ? i / RB % 2 : i / U; };
    auto frag = [&](int i) {
      const int p = PL - 1 - (LOW ? i / (2 * RB) : i % U / RB);
      x[i % U] = *(const bf16x8*)(a + p * BM * LS + i % RB * 16 * LS + 8 * half_of(i));
    };
#pragma unroll
    for (int i = 0; i < U; ++i) frag(i);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int c = 0; c < NC; ++c) w[m][c] = w_frag<WF>(cur.w[c], m, cur.sb[c]);
#pragma unroll
    for (int i = 0; i < 2 * U; ++i) {
      const int m = half_of(i), r = i % RB;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        part[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            w[m][c], x[i % U], i < RB ? z : part[r][c], 0, 0, 0);
      }
      if (i < U) frag(i + U);
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if constexpr (COMP) {
            const float a0 = acc[r][c][v], p0 = part[r][c][v], t = a0 + p0;
            low[r][c][v] += p0 - (t - a0);
            acc[r][c][v] = t;
          } else
          acc[r][c][v] = WF == WD_FP8 ? fmaf(part[r][c][v], cur.f[c], acc[r][c][v])
                                      : acc[r][c][v] + part[r][c][v];
  };
  // Step s multiplies the tile staged in the step before and stages the
  // next one's beside its MFMAs; the scheduling groups keep the fragment
  // reads a half step ahead and spread the split's VALU work over the MFMAs.
  auto step = [&](int s, const uint16_t* tile, uint16_t* ntile, Set& cur,
                  Set& next, Set& far) {
    load(far, s + 3);
    multiply(tile, cur);
#pragma unroll
    for (int q = 0; q < NA; ++q) stage(ntile, next, q);
    if constexpr (BM > 16) {
      constexpr int U = PL * RB;
      constexpr int VALU = (A32 ? 20 * NA : 0) + (WF == WD_BF16 ? 0 : 8 * NC) + 4 * RB * NC;
      constexpr int V = VALU / (2 * U) > 0 ? VALU / (2 * U) : 1;
      // the second half's share, where another one measured better: FP8 32 x
      // 256 (fewer registers live: 62 us at 512 x 4096 x 4096 with V, 54 so),
      // 32-row tiles over MXFP4 (300 x 2048 x 7168 70.0 -> 66.6) and bf16
      // weights (the layer's down launch, 64 tokens: -0.3)
      constexpr int V2 = NC == 4 ? V - 4 : A32 && WF != WD_FP8 && BM == 32 ? V + 2 : V;
      __builtin_amdgcn_sched_group_barrier(0x100, U, 0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        __builtin_amdgcn_sched_group_barrier(0x008, NC, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        __builtin_amdgcn_sched_group_barrier(0x008, NC, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, V2, 0);
      }
    }
    __syncthreads();
  };

  Set t0, t1, t2, t3;
  load(t0, 0);
  load(t1, 1);
  load(t2, 2);
#pragma unroll
  for (int q = 0; q < NA; ++q) stage(a_lds0, t0, q);
  __syncthreads();
  const int full = K / KT;  // steps in which every K wave has a slice
  int s = 0;
  for (; s + 4 <= full; s += 4) {
    step(s, a_lds0, a_lds1, t0, t1, t3);
    step(s + 1, a_lds1, a_lds0, t1, t2, t0);
    step(s + 2, a_lds0, a_lds1, t2, t3, t1);
    step(s + 3, a_lds1, a_lds0, t3, t0, t2);
  }
  // the rest (at most four steps, the last perhaps partial); step s's set
  // is t0 and its tile a_lds0 whatever ran before
  auto rest = [&](const uint16_t* tile, uint16_t* ntile, Set& cur, Set& next) {
    if (s >= steps) return;
    if (s * KT + __builtin_amdgcn_readfirstlane(wk) * 64 < K) multiply(tile, cur);
    if (++s < steps) {
#pragma unroll
      for (int q = 0; q < NA; ++q) stage(ntile, next, q);
    }
    __syncthreads();
  };
  if (s + 3 < steps) load(t3, s + 3);
  rest(a_lds0, a_lds1, t0, t1);
  rest(a_lds1, a_lds0, t1, t2);
  rest(a_lds0, a_lds1, t2, t3);
  rest(a_lds1, a_lds0, t3, t0);

  if constexpr (COMP) {  // (past an infinity the lost part is a NaN)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (__builtin_isfinite(acc[r][c][v])) acc[r][c][v] += low[r][c][v];
  }

  // ---- the K waves' sums ----------------------------------------------------
  if constexpr (WK > 1) {
    f32x4* red = (f32x4*)a_lds0;
    if (wk > 0) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          red[((wave - WN) * RB * NC + r * NC + c) * 64 + lane] = acc[r][c];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        f32x4 t[WK];
        t[0] = acc[r][c];
#pragma unroll
        for (int k = 1; k < WK; ++k)
          t[k] = red[(((k - 1) * WN + wn) * RB * NC + r * NC + c) * 64 + lane];
#pragma unroll
        for (int d = 1; d < WK; d *= 2)
#pragma unroll
          for (int k = 0; k < WK; k += 2 * d) t[k] += t[k + d];
        acc[r][c] = t[0];
      }
  }
  // ---- epilogue: lane = token r * 16 + lc, columns 4 lg + v of a subtile ----
  constexpr float DOWN = A32 ? 1.f / (float)(1ull << A_UP) : 1.f;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int t = r * 16 + lc;
    if (t >= rows) continue;
    const int p = rb0 + t;
    float w = 1.f;
    if (S.row_w) w = S.row_w[S.sorted_idx ? S.sorted_idx[p] : p];
#pragma unroll
    for (int c = 0; c < NO; ++c) {
      const int n = ncol + c * 16 + 4 * lg;
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v)
        o[v] = SWIGLU ? silu_f32(acc[r][c][v]) * acc[r][c + (SWIGLU ? NO : 0)][v]
                      : acc[r][c][v] * DOWN * w;
      float* d = S.out + (size_t)p * N + n;
      if (n + 4 <= N && N % 4 == 0) {
        *(float4*)d = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (n + v < N) d[v] = o[v];
      }
    }
  }
  // An infinite or NaN sum of fp32 activations may be this kernel's own: an
  // FP8 partial that overflows before a small block scale, or an infinite
  // weight (a bf16 one, e8m0 254) against a zero mid or lo part. Those
  // outputs are taken again by plain fp32 products, an output at a time by
  // the whole wave (its weights laid out as the loads above read them). A row
  // that holds a NaN is NaN throughout: left as it is after one of them.
  if constexpr (A32) {
    static_assert(RB * NC * 4 <= 32, "a bit for each of a lane's sums");
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < RB * NC * 4; ++i)
      z = fmaf(acc[i / (4 * NC)][i / 4 % NC][i % 4], 0.f, z);
    // (rows that a 16-row tile leaves unstaged hold anything)
    if (!__ballot(z != 0.f && (RB > 1 || lc < rows))) return;
    uint32_t bad = 0;
#pragma unroll
    for (int i = 0; i < RB * NC * 4; ++i) {
      const int r = i / (4 * NC), c = i / 4 % NC, v = i % 4;
      if (r * 16 + lc < rows && ncol + c * 16 + 4 * lg + v < N &&
          !__builtin_isfinite(acc[r][c][v]))
        bad |= 1u << i;
    }
    uint64_t seen = 0;  // rows looked over for a NaN
    while (const uint64_t m = __ballot(bad != 0)) {
      const int l = __builtin_ctzll(m);
      const int i = __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)bad, l));
      const int t = i / (4 * NC) * 16 + (l & 15), p = rb0 + t;
      const int n = ncol + i / 4 % NC * 16 + 4 * (l >> 4) + i % 4;
      const float* a = (const float*)S.a + (size_t)rsrc[t] * K;
      float y = plain_dot<WF>(S, a, e, n, lane);
      if (__builtin_isnan(y) && !(seen >> t & 1)) {
        seen |= 1ull << t;
        bool nan = false;
        for (int k = 4 * lane; k < K; k += 256) {
          const float4 v = *(const float4*)(a + k);
          nan |= __builtin_isunordered(v.x, v.y) || __builtin_isunordered(v.z, v.w);
        }
        if (__any(nan) && lc == (l & 15))
          bad &= ~(((1u << (4 * NC - 1) << 1) - 1) << (i / (4 * NC) * 4 * NC));
      }
      if (S.row_w) y *= S.row_w[S.sorted_idx ? S.sorted_idx[p] : p];
      if (lane == l) {
        S.out[(size_t)p * N + n] = y;
        bad &= ~(1u << i);
      }
    }
  }
}

template <int WF, bool A32, bool SWIGLU, int BM, int WN, int NC>
int go(const WideSeg& s0, const WideSeg& s1, int topk, hipStream_t st) {
  constexpr int NO = SWIGLU ? NC / 2 : NC, BN = 16 * NO * WN;
  auto blocks = [](const WideSeg& s) -> long {
    if (!s.a) return 0;
    const long rt = s.tile_info ? s.max_tiles : (s.total_rows + BM - 1) / BM;
    return rt * ((s.N + BN - 1) / BN);
  };
  const long b0 = blocks(s0), b1 = blocks(s1);
  if (b0 + b1 <= 0) return 0;
  wide_kernel<WF, A32, SWIGLU, BM, WN, NC>
      <<<(unsigned)(b0 + b1), WD_THREADS, 0, st>>>(s0, s1, (int)b0, topk);
  SLLM_LAUNCHED();
  return 0;
}

}  // namespace

// The linears' tiles (rows x output columns) and the time of a round of their
// workgroups in us at K = 4096, FP8 and MXFP4 weights, by which wide_tile
// weighs them (a launch of one to three rounds over N = 4096, divided by them;
// MXFP4's shortest tiles at a few rows, which cost less than sixteen).
struct WideTile {
  int bm, bn;
  float us;
};
static const WideTile WIDE_FP8[] = {
    {16, 16, 11.5f}, {16, 32, 12.4f}, {32, 64, 22.f}, {32, 128, 31.5f}, {32, 256, 52.f}};
static const WideTile WIDE_FP4[] = {
    {16, 16, 9.5f}, {16, 32, 12.5f}, {32, 64, 23.8f}, {32, 128, 39.f}, {64, 128, 64.f}};

// One workgroup fits a CU (its registers and tile), so a launch takes as
// many rounds as its tiles need over the CUs. FP8 4096 x 4096, us by tile:
// 16 rows 11.5 / 12.4 / 21 / 30 / 48, 32 rows 21.4 / 13.0 / 22 / 31 / 49, 128 rows
// 75 / 44 / 22.3 / 30.7 / 50, 256 rows - / 86 / 43 / 32.9 / 51, 512 rows - / - / 84 /
// 63.2 / 54.6, 513 and 768 rows (three rounds, or two) 90.4 / 98.1 and 94.2 /
// 100.9 of the last two, 1024 rows 125 / 106; 64 x 128 as the tallest spilled 62 at
// 512. The tallest FP8 tile is four waves of 64 columns by two K halves: an
// LDS fragment serves four products, not two, and half as many barriers
// follow (eight waves of 32 columns: 300 / 400 / 512 rows 54.7 / 55.9 / 57.4 us, so
// 51.3 / 51.9 / 54.1); it holds all 256 registers and spills five. MXFP4, whose
// conversions that form holds in registers too, keeps 64 x 128 (7168 <- 2048,
// 150 / 222 / 512 rows 37.3 / 38.4 / 76.0 us there, 44.0 / 44.9 / 88.1 as 32 x
// 256).
int wide_tile(int wf, long rows, long n, int num_cus) {
  const WideTile* tile = wf == WD_FP8 ? WIDE_FP8 : WIDE_FP4;
  int best = 0;
  float t = 0.f;
  for (int i = 0; i < 5; ++i) {
    const long tiles = (rows + tile[i].bm - 1) / tile[i].bm * ((n + tile[i].bn - 1) / tile[i].bn);
    const float c = tile[i].us * (float)((tiles + num_cus - 1) / num_cus);
    if (i == 0 || c < t) {
      best = i;
      t = c;
    }
  }
  return best;
}

int launch_wide(int wf, int swiglu, int tile, const WideSeg& s0,
                const WideSeg* s1, int topk, hipStream_t st) {
  const WideSeg z{};
  const WideSeg& t1 = s1 ? *s1 : z;
#define GO(WF_, BM4_, WN4_, NC4_)                                          \
  (tile == 0   ? go<WF_, true, false, 16, 1, 1>(s0, t1, topk, st)          \
   : tile == 1 ? go<WF_, true, false, 16, 1, 2>(s0, t1, topk, st)          \
   : tile == 2 ? go<WF_, true, false, 32, 2, 2>(s0, t1, topk, st)          \
   : tile == 3 ? go<WF_, true, false, 32, 4, 2>(s0, t1, topk, st)          \
               : go<WF_, true, false, BM4_, WN4_, NC4_>(s0, t1, topk, st))
  if (wf == WD_FP8) return GO(WD_FP8, 32, 4, 4);
  if (wf == WD_FP4) return GO(WD_FP4, 64, 4, 2);
#undef GO
#define GO(A_, SW_)                                                        \
  (tile == 1   ? go<WD_BF16, A_, SW_, 16, 1, 2>(s0, t1, topk, st)          \
   : tile == 2 ? go<WD_BF16, A_, SW_, 32, 2, 2>(s0, t1, topk, st)          \
   : tile == 3 ? go<WD_BF16, A_, SW_, 32, 4, 2>(s0, t1, topk, st)          \
               : go<WD_BF16, A_, SW_, 64, 8, 2>(s0, t1, topk, st))
  SLLM_REQUIRE(tile >= 1 && tile <= 4, "wide gemm: tile %d of bf16 weights", tile);
  return swiglu ? GO(false, true) : GO(true, false);
#undef GO
}

}  // namespace sllm
