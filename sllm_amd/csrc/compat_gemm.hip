// Reference-compatible standalone GEMM entry points.
//
//   sllm_fp8_gemm(_dev)   ref kernels/cuda/fp8.cu:72-110
//   sllm_ds_fp4_gemm      ref kernels/cuda/deepseek.cu:57-73
//   sllm_gemm_ex          ref kernels/cuda/kernels.cu:752-767 (cublasGemmEx)
//   sllm_ds_fp4_gemm_packed  new: packed E2M1 + E8M0 weights on the device
//                         (the reference dequantizes FP4 on the host,
//                         kernels/_deepseek_cuda.py:89-94)
//
// All compute C (M, N) fp32 = A (M, K) . B(N, K)^T with fp32 accumulation.
// Scale orientation for the FP8 weight follows loaders/fp8.py:98-135 and the
// reference's own test (tests/test_fp8_gemm.py:49-55: the kernel must equal
// A @ dequant_weight_blocked(B, scale).T): scale_inv has shape
// (ceil(N/bh), ceil(K/bw)) and W[n, k] = e4m3(B[n, k]) * scale_inv[n/bh,
// k/bw]. The reference kernel's K-block-major index (fp8.cu:66) contradicts
// that contract; the contract is what is implemented.
//
// FP8 and MXFP4 weights of the loader's block shapes run on the matrix cores
// (gemm_wide.hip) or, with few rows, on the layer's unpacked-weight GEMV
// (decode.hip), bf16 gemm_ex with k % 128 == 0 on the MFMA router kernels;
// other shapes take the GEMV up to 64 rows where it fits, else a 32x32
// LDS-tiled fp32 kernel with on-the-fly dequantization of B.
#include "launch.h"

namespace sllm {

enum BFmt { B_F32 = 0, B_BF16 = 1, B_FP8_BLOCK = 2, B_FP4_PACKED = 3 };

struct BDesc {
  int fmt;
  const void* b;
  const void* scale;
  int bh, bw;  // fp8 block shape (N, K); fp4 uses bw along K
};

__device__ __forceinline__ float load_b_elem(const BDesc& d, int n, int k,
                                             int N, int K) {
  switch (d.fmt) {
    case B_F32: return ((const float*)d.b)[(size_t)n * K + k];
    case B_BF16: return bf16_to_f32(((const uint16_t*)d.b)[(size_t)n * K + k]);
    case B_FP8_BLOCK: {
      const uint8_t q = ((const uint8_t*)d.b)[(size_t)n * K + k];
      const int KB = (K + d.bw - 1) / d.bw;
      const float s = ((const float*)d.scale)[(size_t)(n / d.bh) * KB + k / d.bw];
      return __builtin_amdgcn_cvt_f32_fp8((int)q, 0) * s;
    }
    default: {
      const uint8_t byte = ((const uint8_t*)d.b)[(size_t)n * (K / 2) + k / 2];
      const uint32_t nib = (k & 1) ? (byte >> 4) : (byte & 15);
      const uint32_t e = (nib >> 1) & 3u, m = nib & 1u;
      uint32_t bits = e ? ((e + 126u) << 23) | (m << 22) : (m ? 0x3F000000u : 0u);
      const float v = __uint_as_float(bits | ((nib & 8u) << 28));
      const int KB = (K + d.bw - 1) / d.bw;
      const uint8_t sb = ((const uint8_t*)d.scale)[(size_t)n * KB + k / d.bw];
      const float s = sb == 0 ? 0.f : (sb == 255 ? __uint_as_float(0x7FC00000u)
                                                 : __uint_as_float((uint32_t)sb << 23));
      return v * s;
    }
  }
}

// sllm_q4_gemv_rows' post-op, in place: 1 silu(x / scale), 2 sigmoid.
__global__ void post_act_kernel(float* __restrict__ v, long n, int post,
                                float scale) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float x = v[i] / scale;
  v[i] = post == 1 ? silu_f32(x) : sigmoid_f32(x);
}

// 32x32 output tile per 256-thread block; each thread 4 outputs (rows).
__global__ __launch_bounds__(256) void tiled_gemm_kernel(
    const void* __restrict__ a, int a_bf16, BDesc bd, float* __restrict__ c,
    int M, int N, int K) {
  __shared__ float as[32][33];
  __shared__ float bs[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // ty 0..7
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 32) {
    for (int i = threadIdx.x; i < 32 * 32; i += 256) {
      const int r = i / 32, kk = i % 32;
      const int m = m0 + r, n = n0 + r, k = k0 + kk;
      float av = 0.f, bv = 0.f;
      if (m < M && k < K)
        av = a_bf16 ? bf16_to_f32(((const uint16_t*)a)[(size_t)m * K + k])
                    : ((const float*)a)[(size_t)m * K + k];
      if (n < N && k < K) bv = load_b_elem(bd, n, k, N, K);
      as[r][kk] = av;
      bs[r][kk] = bv;
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < 32; ++kk) {
      const float bv = bs[tx][kk];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = fmaf(as[ty * 4 + q][kk], bv, acc[q]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int m = m0 + ty * 4 + q, n = n0 + tx;
    if (m < M && n < N) c[(size_t)m * N + n] = acc[q];
  }
}

int launch_tiled_gemm(const void* a, int a_bf16, const BDesc& bd, float* c,
                      int M, int N, int K, hipStream_t st) {
  SLLM_REQUIRE(a && bd.b && c, "gemm: null pointer");
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: bad dims M=%d N=%d K=%d", M, N,
               K);
  dim3 grid(ceil_div(N, 32), ceil_div(M, 32));
  tiled_gemm_kernel<<<grid, 256, 0, st>>>(a, a_bf16, bd, c, M, N, K);
  SLLM_LAUNCHED();
  return 0;
}

}  // namespace sllm

using namespace sllm;

namespace {

// Where a quantized linear runs: a tile of the matrix-core kernel
// (launch_wide's 0-4), the layer's unpacked-weight GEMV, or the tiled kernel.
enum { LIN_GEMV = 5, LIN_TILED = 6 };

// One row always streams through the GEMV (128 x 128 blocks). Two to four rows
// do where it streams B faster than the matrix cores' tiles, which few rows
// leave mostly empty. us, GEMV / matrix cores, repeated (weights from memory):
// - up to 32 columns a CU (one round of the 16-row tiles) short K only: 2
//   rows 2048 x 2048 4.3 / 5.8 (9 / 9), 4096 x 4096 7.0 / 7.9 (15 / 14), 2048
//   x 7168 8.2 / 9.9 (19 / 16), 7168 x 7168 15.1 / 14.1 (30 / 26); 3 rows 7168
//   x 2048 6.0 / 7.7 (13 / 12), 4096 x 4096 7.8 / 8.0 (18 / 14); 4 rows 9.9 / 8.0
// - up to 48 (one round of three GEMV workgroups of 16 a CU, 32-row tiles
//   there): 12288 x 4096, 2 / 4 / 5 rows 11.8 / 20.9 (26 / 29), 17.0 / 20.9 (32 /
//   29), 23.9 / 20.9 (39 / 29)
// - up to 64 (one round of 32 x 64 tiles, two of the GEMV): 14336 x 4096, 2
//   rows 21.2 / 21.6 (34 / 29)
// - above: 2 rows (17408 x 5120 24.3 / 38.9 (44 / 56), 64000 x 4096 62.1 / 60.1
//   (104 / 130)), 3 up to 96 (18432 x 7168 41.8 / 50.8 (69 / 70), 32000 x 4096
//   41.6 / 32.3 (63 / 67)); 4 rows 17408 x 5120 36.6 / 38.9 (56 / 56), 20480 x
//   2048 18.2 / 17.4 (28 / 26).
bool fp8_few_rows(int M, int N, int K, int cus) {
  if (M == 1) return true;
  if (K < 1024 || M > 4) return false;
  if (N <= 32 * cus) return K <= (M == 2 ? 4096 : M == 3 ? 2048 : 0);
  if (N <= 48 * cus) return true;
  return N > 64 * cus && (M == 2 || (M == 3 && N <= 96 * cus));
}

// The same for MXFP4: 2 rows 4096 x 4096 7.9 / 10.3 (14 / 15), 2048 x 7168 12.5 /
// 13.6 (22 / 19), 8192 x 4096 11.4 / 15.6 (19 / 20), 14336 x 4096 21.1 / 25.3
// (32 / 31), 18432 x 7168 52.3 / 59.8 (70 / 68), 20480 x 2048 15.1 / 29.2 (27 /
// 35), 32000 x 4096 43.8 / 40.2 (58 / 52), 256 x 256 6.2 / 4.3; 3 rows 2048 x 2048
// 6.0 / 7.4 (10 / 11), 20480 x 2048 19.1 / 29.1 (32 / 35), 4096 x 4096 9.6 / 10.2
// (16 / 15), 14336 x 4096 27.5 / 25.2 (39 / 31); 4 rows 7168 x 2048 10.4 / 10.7
// (16 / 15), 20480 x 2048 23.2 / 29.2 (37 / 35).
bool fp4_few_rows(int M, int N, int K, int cus) {
  if (M == 1) return true;
  if (K < 1024 || N > 96 * cus) return false;
  if (M == 2) return K <= 4096 || N > 32 * cus;
  return K <= 2048 && (M == 3 ? K > 1024 : M == 4 && N > 64 * cus);
}

// FP8: the matrix cores take scale blocks of 4 n rows by 64 2^m columns, the
// GEMV the loader's 128 x 128. fits: wide_fits.
int fp8_route(int M, int N, int K, int bh, int bw, bool fits) {
  const int cus = device_cus();
  const bool gemv = bh == 128 && bw == 128 && M <= 64 && N % 128 == 0 && K % 128 == 0;
  const bool wide = M > 1 && fits && bh % 4 == 0 && bw % 64 == 0 && bw == 64 << __builtin_ctz(bw / 64);
  if (gemv && (!wide || fp8_few_rows(M, N, K, cus))) return LIN_GEMV;
  return wide ? wide_tile(WD_FP8, M, N, cus) : LIN_TILED;
}

int fp4_route(int M, int N, int K, int bw, bool fits) {
  const int cus = device_cus();
  const bool gemv = bw == 32 && M <= 64 && K % 32 == 0 && N % 16 == 0;
  const bool wide = M > 1 && N > 0 && fits && bw == 32;
  if (gemv && (!wide || fp4_few_rows(M, N, K, cus))) return LIN_GEMV;
  return wide ? wide_tile(WD_FP4, M, N, cus) : LIN_TILED;
}

struct Tmp {
  void* p = nullptr;
  ~Tmp() {
    if (p) (void)hipFree(p);
  }
};
}  // namespace

extern "C" {

// Host query (no device work): which kernel the FP8 and MXFP4 linears take.
int sllm_linear_plan_query(int fp4, int M, int N, int K, int block_h,
                           int block_w, int aligned) {
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0 && block_h > 0 && block_w > 0,
               "sllm_linear_plan_query: bad dims");
  const bool fits = aligned && wide_fits(nullptr, nullptr, nullptr, K);
  return fp4 ? fp4_route(M, N, K, block_w, fits) : fp8_route(M, N, K, block_h, block_w, fits);
}

int sllm_fp8_gemm_dev(const float* A, const unsigned char* B,
                      const float* scale_inv, float* C, int M, int N, int K,
                      int block_h, int block_w) {
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0 && block_h > 0 && block_w > 0,
               "sllm_fp8_gemm: bad dims");
  SLLM_REQUIRE(A && B && scale_inv && C, "sllm_fp8_gemm: null pointer");
  const int route = fp8_route(M, N, K, block_h, block_w, wide_fits(A, B, C, K));
  if (route < LIN_GEMV) {
    WideSeg s{};
    s.a = A; s.total_rows = M; s.w0 = B; s.s0 = scale_inv; s.bh = block_h;
    s.bws = __builtin_ctz(block_w / 64); s.N = N; s.K = K; s.out = C;
    return launch_wide(WD_FP8, 0, route, s, nullptr, 1, nullptr);
  }
  // (one wave per four weight rows, 16-byte weight loads dequantized in
  // registers; B streamed once per four rows of A)
  if (route == LIN_GEMV)
    return launch_gemv(0, 0, A, 0, 0, nullptr, 1, M, nullptr, nullptr, 1,
                       nullptr, B, scale_inv, nullptr, nullptr, N, K, nullptr,
                       0.f, C, nullptr);
  BDesc bd{B_FP8_BLOCK, B, scale_inv, block_h, block_w};
  return launch_tiled_gemm(A, 0, bd, C, M, N, K, 0);
}

int sllm_fp8_gemm(const float* A, const unsigned char* B,
                  const float* scale_inv, float* C, int M, int N, int K,
                  int block_h, int block_w) {
  SLLM_REQUIRE(A && B && scale_inv && C, "sllm_fp8_gemm: null pointer");
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0 && block_h > 0 && block_w > 0,
               "sllm_fp8_gemm: bad dims");
  const size_t sa = (size_t)M * K * 4, sb = (size_t)N * K,
               sc = (size_t)M * N * 4,
               ss = (size_t)ceil_div(N, block_h) * ceil_div(K, block_w) * 4;
  Tmp dA, dB, dS, dC;
  SLLM_HIP(hipMalloc(&dA.p, sa));
  SLLM_HIP(hipMalloc(&dB.p, sb));
  SLLM_HIP(hipMalloc(&dS.p, ss));
  SLLM_HIP(hipMalloc(&dC.p, sc));
  SLLM_HIP(hipMemcpy(dA.p, A, sa, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dB.p, B, sb, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dS.p, scale_inv, ss, hipMemcpyHostToDevice));
  if (sllm_fp8_gemm_dev((const float*)dA.p, (const unsigned char*)dB.p,
                        (const float*)dS.p, (float*)dC.p, M, N, K, block_h,
                        block_w))
    return -1;
  SLLM_HIP(hipMemcpy(C, dC.p, sc, hipMemcpyDeviceToHost));
  return 0;
}

int sllm_ds_fp4_gemm(float* o, const float* a, const float* b, int M, int N,
                     int K, float scale, float* opts) {
  (void)scale;
  (void)opts;
  SLLM_REQUIRE(o && a && b, "sllm_ds_fp4_gemm: null pointer");
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0, "sllm_ds_fp4_gemm: bad dims");
  const size_t sa = (size_t)M * K * 4, sb = (size_t)N * K * 4,
               sc = (size_t)M * N * 4;
  Tmp dA, dB, dC;
  SLLM_HIP(hipMalloc(&dA.p, sa));
  SLLM_HIP(hipMalloc(&dB.p, sb));
  SLLM_HIP(hipMalloc(&dC.p, sc));
  SLLM_HIP(hipMemcpy(dA.p, a, sa, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dB.p, b, sb, hipMemcpyHostToDevice));
  BDesc bd{B_F32, dB.p, nullptr, 0, 0};
  if (launch_tiled_gemm(dA.p, 0, bd, (float*)dC.p, M, N, K, 0)) return -1;
  SLLM_HIP(hipMemcpy(o, dC.p, sc, hipMemcpyDeviceToHost));
  return 0;
}

// Device pointers: a (M, K) fp32, packed (N, K/2) E2M1, scale (N, K/bw) E8M0.
int sllm_ds_fp4_gemm_packed_dev(float* o, const float* a, const void* packed,
                                const void* scale_e8m0, int M, int N, int K,
                                int block_w) {
  SLLM_REQUIRE(K % 2 == 0 && block_w > 0, "fp4 gemm: K even, block_w > 0");
  SLLM_REQUIRE(M <= 0 || (a && packed && scale_e8m0 && o), "fp4 gemm: null pointer");
  const int route = fp4_route(M, N, K, block_w, wide_fits(a, packed, o, K));
  if (route < LIN_GEMV) {
    WideSeg s{};
    s.a = a; s.total_rows = M; s.w0 = (const uint8_t*)packed; s.s0 = scale_e8m0;
    s.N = N; s.K = K; s.out = o;
    return launch_wide(WD_FP4, 0, route, s, nullptr, 1, nullptr);
  }
  // (the layer's MXFP4 form: the same nibble order, E2M1 values and 0x00 /
  // 0xFF scale convention)
  if (route == LIN_GEMV)
    return launch_gemv(1, 0, a, 0, 0, nullptr, 1, M, nullptr, nullptr, 1,
                       nullptr, (const uint8_t*)packed, scale_e8m0, nullptr,
                       nullptr, N, K, nullptr, 0.f, o, nullptr);
  BDesc bd{B_FP4_PACKED, packed, scale_e8m0, 1, block_w};
  return launch_tiled_gemm(a, 0, bd, o, M, N, K, 0);
}

// Host pointers: same arguments as the device variant.
int sllm_ds_fp4_gemm_packed(float* o, const float* a, const void* packed,
                            const void* scale_e8m0, int M, int N, int K,
                            int block_w) {
  SLLM_REQUIRE(o && a && packed && scale_e8m0, "fp4 gemm: null pointer");
  SLLM_REQUIRE(M > 0 && N > 0 && K > 0 && K % 2 == 0 && block_w > 0,
               "fp4 gemm: bad dims");
  const size_t sa = (size_t)M * K * 4, sp = (size_t)N * (K / 2),
               ss = (size_t)N * ceil_div(K, block_w), sc = (size_t)M * N * 4;
  Tmp dA, dP, dS, dC;
  SLLM_HIP(hipMalloc(&dA.p, sa));
  SLLM_HIP(hipMalloc(&dP.p, sp));
  SLLM_HIP(hipMalloc(&dS.p, ss));
  SLLM_HIP(hipMalloc(&dC.p, sc));
  SLLM_HIP(hipMemcpy(dA.p, a, sa, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dP.p, packed, sp, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dS.p, scale_e8m0, ss, hipMemcpyHostToDevice));
  if (sllm_ds_fp4_gemm_packed_dev((float*)dC.p, (const float*)dA.p, dP.p, dS.p,
                                  M, N, K, block_w))
    return -1;
  SLLM_HIP(hipMemcpy(o, dC.p, sc, hipMemcpyDeviceToHost));
  return 0;
}

// c (m, n) fp32 = a (m, k) . w (n, k)^T; atype 0 = fp32, 1 = bf16 for both a
// and w (dtype tags of kernels/_sllm_cuda.py:490-491). Device pointers.
// bf16 with k % 128 == 0 runs on the router GEMM kernels (the same contract:
// bf16 products on the matrix cores, fp32 accumulation; m <= 64, the decode
// loops' GEMVs, and few tiles of 64 x 128 at larger k on the K-split kernel,
// the rest on the tiles); other batches of at most 64 rows (fp32, or bf16 with
// other k) on the unpacked-weight GEMV; the rest on the tiled kernel.
int sllm_gemm_ex(const void* a, int atype, const void* w, void* c, int m,
                 int n, int k) {
  SLLM_REQUIRE(atype == 0 || atype == 1, "sllm_gemm_ex: atype must be 0 or 1");
  SLLM_REQUIRE(a && w && c && m > 0 && n > 0 && k > 0,
               "sllm_gemm_ex: null pointer or empty shape (m=%d n=%d k=%d)",
               m, n, k);
  if (atype == 1 && k % 128 == 0)
    return launch_bf16_gemm((const uint16_t*)a, (const uint16_t*)w, (float*)c,
                            m, n, k, nullptr);
  // other decode-size batches: the unpacked-weight GEMV (bf16 or fp32 rows)
  if (m <= 64 && n % 16 == 0 && k % (atype == 1 ? 8 : 4) == 0)
    return launch_gemv(atype == 1 ? 2 : 3, 0, a, atype, 0, nullptr, 1, m,
                       nullptr, nullptr, 1, nullptr, (const uint8_t*)w,
                       nullptr, nullptr, nullptr, n, k, nullptr, 0.f,
                       (float*)c, nullptr);
  BDesc bd{atype == 1 ? B_BF16 : B_F32, w, nullptr, 0, 0};
  return launch_tiled_gemm(a, atype, bd, (float*)c, m, n, k, 0);
}

// ref: kernels/cuda/qwen4.cu:98-136, :699-708 (sllm_q4_gemv_rows[_dev]):
// out (rows, O) fp32 = A (rows, K) . W (O, K)^T, then post 1: silu(x /
// scale), post 2: sigmoid(x / scale), other values: none. rows, K or O
// not positive: -1, as the reference. Batches of at most 64 rows on the
// unpacked-weight GEMV (fp32 weight rows), larger ones on the tiled kernel.
int sllm_q4_gemv_rows_dev(const float* A, const float* W, float* out, int rows,
                          int K, int O, int post, float scale) {
  SLLM_REQUIRE(rows > 0 && K > 0 && O > 0,
               "sllm_q4_gemv_rows: rows, K, O must be positive");
  SLLM_REQUIRE(A && W && out, "sllm_q4_gemv_rows: null pointer");
  int rc;
  if (rows <= 64 && O % 16 == 0 && K % 4 == 0) {
    rc = launch_gemv(3, 0, A, 0, 0, nullptr, 1, rows, nullptr, nullptr, 1,
                     nullptr, (const uint8_t*)W, nullptr, nullptr, nullptr, O,
                     K, nullptr, 0.f, out, nullptr);
  } else {
    BDesc bd{B_F32, W, nullptr, 0, 0};
    rc = launch_tiled_gemm(A, 0, bd, out, rows, O, K, 0);
  }
  if (rc || (post != 1 && post != 2)) return rc;
  const long n = (long)rows * O;
  post_act_kernel<<<(unsigned)((n + 255) / 256), 256>>>(out, n, post, scale);
  SLLM_LAUNCHED();
  return 0;
}

int sllm_q4_gemv_rows(const float* A, const float* W, float* out, int rows,
                      int K, int O, int post, float scale) {
  SLLM_REQUIRE(rows > 0 && K > 0 && O > 0,
               "sllm_q4_gemv_rows: rows, K, O must be positive");
  SLLM_REQUIRE(A && W && out, "sllm_q4_gemv_rows: null pointer");
  const size_t sa = (size_t)rows * K * 4, sw = (size_t)O * K * 4,
               so = (size_t)rows * O * 4;
  Tmp dA, dW, dO;
  SLLM_HIP(hipMalloc(&dA.p, sa));
  SLLM_HIP(hipMalloc(&dW.p, sw));
  SLLM_HIP(hipMalloc(&dO.p, so));
  SLLM_HIP(hipMemcpy(dA.p, A, sa, hipMemcpyHostToDevice));
  SLLM_HIP(hipMemcpy(dW.p, W, sw, hipMemcpyHostToDevice));
  if (sllm_q4_gemv_rows_dev((const float*)dA.p, (const float*)dW.p,
                            (float*)dO.p, rows, K, O, post, scale))
    return -1;
  SLLM_HIP(hipMemcpy(out, dO.p, so, hipMemcpyDeviceToHost));
  return 0;
}

}  // extern "C"
