// Block-scaled FP8 / MXFP4 GEMV-GEMM for skinny M (decode widths and up).
//
// C[M,N] (bf16) = sum over 128-wide K-blocks of (A_blk . W_blk^T) * scales
// (wanferenz/kernels/reference.py:235-311 fp8_gemm, :506-591 fp4_gemm; the CPU
// restatement torch_ops.py:93-108).
//
// Decode is bound by streaming W from HBM, so the kernel is shaped around the
// weight stream, not the M dimension:
//   * a workgroup owns 16 output columns (= 16 weight rows) and its four
//     waves split K into four contiguous ranges, so every weight byte is read
//     once, by one lane, in 16-byte loads; partial sums meet in LDS;
//   * each wave batches the loads of UNROLL K-blocks before issuing the MFMAs
//     to keep enough bytes in flight per CU;
//   * tokens ride on the MFMA's M side (16 rows per tile, MT tiles per wave),
//     padded with zero rows, so an M=1..16 GEMV is one V_MFMA_SCALE 16x16x128
//     per 16x128 weight block with no per-byte VALU dequantisation.
#include "mfma_ops.h"

namespace wz {

constexpr int kGemmThreads = 256;

// Rows up to which the skinny kernel serves; above, the tile GEMM (linear_gemm.hip; the same
// summation order, so the same bits).  One M-tile of 16 is padding-free MFMA work of a weight
// stream that is read once; from two on the skinny kernel's re-reads of the rows by every 16
// columns cost more than staging both operands, except where both scales ride in the MFMA and a
// workgroup per 16 columns fits the CUs at once: there its wider weight loads and four K quarters
// win up to 32 rows of a K of up to 2048 (skinny / tile us, e4m3 20 x 4096 x 2048 5.6 / 6.2, 32 x
// 4096 x 1024 4.1 / 4.6, MXFP4 31 x 4096 x 1024 3.9 / 4.3) and, for MXFP4 weights, up to 28 rows of
// a longer one (17 x 2048 x 4096 7.4 / 8.8, 28 rows 8.6 / 8.8, 32 rows 9.0 / 8.8; e4m3 at K = 4096
// 17 rows 8.4 / 8.4).  Wider N and float scales go the other way from 17 rows on (17 x 32768 x 1024
// e4m3 14.8 / 9.2, MXFP4 12.1 / 6.0; 17 x 4096 x 4096 with float scales 16.2 / 9.3).
static int64_t skinny_max_rows(bool fp4, bool pow2, int64_t N, int64_t K) {
  if (!pow2 || N / 16 > cu_count()) return 16;
  return K <= 2048 ? 32 : fp4 ? 28 : 16;
}
bool tile_rows_fits(const void* a, const void* w, const void* w_s, bool fp4, int64_t M, int64_t N, int64_t K);
int launch_tile_rows(const char* name, const uint8_t* a, const void* a_s, int a_kind, const uint8_t* w,
                     const void* w_s, int w_kind, bool fp4, uint16_t* c, int64_t M, int64_t N, int64_t K,
                     hipStream_t stream);

// One workgroup's 16 output columns [n0, n0 + 16) for rows m_base .. m_base + 16 MT.
// kUnroll = K-blocks per load batch (a wave owns about nkb / 4 of them).
template <int WF, bool A_BF16, int MT, int kUnroll>
__device__ __forceinline__ void skinny_body(const void* __restrict__ A, const void* __restrict__ As, int act_kind,
                                            const uint8_t* __restrict__ W, const void* __restrict__ Ws, int w_kind,
                                            uint16_t* __restrict__ C, int M, int N, int K, int m_base, int n0) {
  __shared__ float red[4][MT][kWave][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nl = lane & 15, g = lane >> 4;
  const int nkb = K / 128;
  const int kb0 = (wave * nkb) / 4, kb1 = ((wave + 1) * nkb) / 4;
  const int ldw = WF == kFmtFp4 ? K / 2 : K;
  const uint8_t* wrow = W + int64_t(n0 + nl) * ldw;
  const uint8_t* wsrow = WF == kFmtFp4 ? reinterpret_cast<const uint8_t*>(Ws) + int64_t(n0 + nl) * (K / 32)
                                       : nullptr;
  const bool a_pow2 = act_kind != WZ_SCALE_F32;
  const bool b_pow2 = WF == kFmtFp4 || w_kind == WZ_WSCALE_E8M0;

  v4f acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  for (int kb = kb0; kb < kb1; kb += kUnroll) {
    v8i bb[kUnroll];
    int sbe[kUnroll];
    float sbf[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int k = min(kb + u, kb1 - 1);  // past kb1: a valid re-read whose MFMA is skipped
      if (WF == kFmtFp4) {
        bb[u] = b_fp4(wrow, k, g);
        sbe[u] = b_fp4_scale(wsrow, k, g);
        sbf[u] = 1.0f;
      } else {
        bb[u] = b_fp8(wrow, k, g);
        fp8_wscale(Ws, int64_t(n0 >> 7) * nkb + k, w_kind, sbe[u], sbf[u]);
      }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = m_base + t * 16 + nl;
      if (A_BF16) {
        const bool live = m < M;
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const int k = kb + u;
          if (k < kb1) {
            const AOp a = a_from_bf16(live ? reinterpret_cast<const uint16_t*>(A) + int64_t(m) * K : nullptr, k, g,
                                      a_pow2);
            mma_step<kFmtFp8, WF>(acc[t], a, bb[u], sbe[u], sbf[u], a_pow2, b_pow2, lane);
          }
        }
      } else {
        // the tile's A blocks of this batch are all requested before the first
        // MFMA: rows past M read row M - 1 (their outputs are not stored) and
        // K-blocks past kb1 re-read the last one (their MFMAs are skipped)
        const int mr = min(m, M - 1);
        const uint8_t* arow = reinterpret_cast<const uint8_t*>(A) + int64_t(mr) * K;
        const void* asrow = act_kind == WZ_SCALE_UE8M0
                                ? static_cast<const void*>(reinterpret_cast<const uint8_t*>(As) + int64_t(mr) * nkb)
                                : static_cast<const void*>(reinterpret_cast<const float*>(As) + int64_t(mr) * nkb);
        AOp a[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) a[u] = a_from_fp8_row(arow, asrow, min(kb + u, kb1 - 1), g, act_kind);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
          if (kb + u < kb1) mma_step<kFmtFp8, WF>(acc[t], a[u], bb[u], sbe[u], sbf[u], a_pow2, b_pow2, lane);
      }
    }
  }

#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][t][lane][i] = acc[t][i];
  __syncthreads();
  // Wave w finishes M-tiles t = w, w+4, ...; partials are summed in wave order.
  for (int t = wave; t < MT; t += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = red[0][t][lane][i];
      v += red[1][t][lane][i];
      v += red[2][t][lane][i];
      v += red[3][t][lane][i];
      const int m = m_base + t * 16 + g * 4 + i;
      if (m < M) C[int64_t(m) * N + n0 + nl] = f32_to_bf16(v);
    }
  }
}

template <int WF, bool A_BF16, int MT, int U>
__global__ __launch_bounds__(kGemmThreads) void skinny_gemm_kernel(
    const void* __restrict__ A, const void* __restrict__ As, int act_kind,
    const uint8_t* __restrict__ W, const void* __restrict__ Ws, int w_kind,
    uint16_t* __restrict__ C, int M, int N, int K) {
  skinny_body<WF, A_BF16, MT, U>(A, As, act_kind, W, Ws, w_kind, C, M, N, K, blockIdx.y * (16 * MT), blockIdx.x * 16);
}

// K-blocks per load batch for a wave that owns ceil(nkb / 4) of them.
static inline int skinny_unroll(int64_t K) {
  const int64_t per_wave = (K / 128 + 3) / 4;
  return per_wave >= 8 ? 8 : per_wave >= 4 ? 4 : 2;
}

// Row g of A against its own MXFP4 weight W[g] (the per-expert GEMV of the
// banked decode path): blockIdx.y = g, each row one M=1 skinny product.
template <int U>
__global__ __launch_bounds__(kGemmThreads) void grouped_fp4_kernel(const uint8_t* __restrict__ A,
                                                                   const void* __restrict__ As, int act_kind,
                                                                   const uint8_t* __restrict__ W,
                                                                   const uint8_t* __restrict__ Ws,
                                                                   uint16_t* __restrict__ C, int N, int K) {
  const int64_t g = blockIdx.y;
  const int nkb = K / 128;
  const void* as_g = act_kind == WZ_SCALE_UE8M0
                         ? static_cast<const void*>(static_cast<const uint8_t*>(As) + g * nkb)
                         : static_cast<const void*>(static_cast<const float*>(As) + g * nkb);
  skinny_body<kFmtFp4, false, 1, U>(A + g * K, as_g, act_kind, W + g * N * (K / 2), Ws + g * N * (K / 32),
                                 WZ_WSCALE_E8M0, C + g * N, 1, N, K, 0, blockIdx.x * 16);
}

// The same products with K = 512 U (a wave's K quarter is U K-blocks).  The skinny body asks
// memory 5 U times a wave (a tile, a scale byte per K-block and row, two pieces of the row and
// its scale), most of them for a few bytes of many lines, and that issue rate bounds it: here
// the row and its scales come into LDS once a workgroup, and a weight row's scales of the
// quarter in 16-byte loads, U + U / 4 + 2 requests a wave at 59 registers (seven waves a SIMD)
// instead of 150 (three).  Same products in the same order.  Six rows of 4096 x 4096 17.7 ->
// 15.3 us, 3.5 TB/s; the weights through LDS in whole lines took 15.1, not worth their LDS.
template <int U>
__global__ __launch_bounds__(kGemmThreads) void grouped_fp4_row_kernel(const uint8_t* __restrict__ A,
                                                                       const void* __restrict__ As, int act_kind,
                                                                       const uint8_t* __restrict__ W,
                                                                       const uint8_t* __restrict__ Ws,
                                                                       uint16_t* __restrict__ C, int N) {
  constexpr int K = 512 * U, KB = 4 * U;
  __shared__ __align__(16) uint8_t a_l[K];
  __shared__ uint32_t as_l[KB];  // e8m0 byte, or the float's bits
  __shared__ float red[4][kWave][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nl = lane & 15, g = lane >> 4;
  const int64_t grp = blockIdx.y, row = grp * N + blockIdx.x * 16 + nl;
  const uint8_t* const wr = W + row * (K / 2) + wave * (U * 64) + g * 16;
  const uint8_t* const sr = Ws + row * (K / 32) + wave * (U * 4);
  if (tid * 16 < K) *reinterpret_cast<v4i*>(a_l + tid * 16) = load16(A + grp * K + tid * 16);
  if (tid < KB)
    as_l[tid] = act_kind == WZ_SCALE_UE8M0 ? uint32_t(static_cast<const uint8_t*>(As)[grp * KB + tid])
                                           : static_cast<const uint32_t*>(As)[grp * KB + tid];
  v4i b[U], sd[U / 4];
#pragma unroll
  for (int u = 0; u < U; ++u) b[u] = load16(wr + u * 64);
#pragma unroll
  for (int u = 0; u < U / 4; ++u) sd[u] = load16(sr + u * 16);
  __syncthreads();
  const bool a_pow2 = act_kind != WZ_SCALE_F32;
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int kb = wave * U + u;
    AOp a = a_zero();
    const v4i lo = *reinterpret_cast<const v4i*>(a_l + kb * 128 + g * 16);
    const v4i hi = *reinterpret_cast<const v4i*>(a_l + kb * 128 + g * 16 + 64);
    a.v = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    const uint32_t s = as_l[kb];
    if (act_kind == WZ_SCALE_UE8M0)
      a.se8 = int(s);
    else if (act_kind == WZ_SCALE_UE8M0_F32)
      a.se8 = int((s >> 23) & 0xFFu);
    else
      a.sf = __uint_as_float(s);
    const v8i bv = {b[u][0], b[u][1], b[u][2], b[u][3], 0, 0, 0, 0};
    mma_step<kFmtFp8, kFmtFp4>(acc, a, bv, int((uint32_t(sd[u / 4][u & 3]) >> (8 * g)) & 0xFFu), 1.0f, a_pow2, true,
                               lane);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][lane][i] = acc[i];
  __syncthreads();
  if (tid < 16) {  // row 0 of the tile: element 0 of lane group 0; partials in wave order
    float v = red[0][tid][0];
    v += red[1][tid][0];
    v += red[2][tid][0];
    v += red[3][tid][0];
    C[grp * N + blockIdx.x * 16 + tid] = f32_to_bf16(v);
  }
}

template <int WF, bool A_BF16>
static int launch_skinny(const void* A, const void* As, int act_kind, const void* W, const void* Ws,
                         int w_kind, void* C, int64_t M, int64_t N, int64_t K, hipStream_t stream,
                         const char* what) {
  if (M == 0) return WZ_OK;
  int mt = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8;
  const int64_t rows_per_block = 16 * mt;
  dim3 grid(unsigned(N / 16), unsigned((M + rows_per_block - 1) / rows_per_block));
  const uint8_t* w = static_cast<const uint8_t*>(W);
  uint16_t* c = static_cast<uint16_t*>(C);
  const int u = skinny_unroll(K);
#define WZ_SKINNY(MTV, UV)                                                                            \
  WZ_LAUNCH(what, stream, (skinny_gemm_kernel<WF, A_BF16, MTV, UV>), grid, dim3(kGemmThreads), 0, A, As, \
            act_kind, w, Ws, w_kind, c, int(M), int(N), int(K))
#define WZ_SKINNY_U(MTV)            \
  if (u == 8) {                     \
    WZ_SKINNY(MTV, 8);              \
  } else if (u == 4) {              \
    WZ_SKINNY(MTV, 4);              \
  } else {                          \
    WZ_SKINNY(MTV, 2);              \
  }
  switch (mt) {
    case 1: WZ_SKINNY_U(1); break;
    case 2: WZ_SKINNY_U(2); break;
    case 4: WZ_SKINNY_U(4); break;
    default: WZ_SKINNY_U(8); break;
  }
#undef WZ_SKINNY_U
#undef WZ_SKINNY
  return check_launch(what);
}

static int check_dims(const char* what, int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N <= 0 || K <= 0)
    return set_error(WZ_EINVAL, "%s: bad shape M=%lld N=%lld K=%lld", what, (long long)M,
                     (long long)N, (long long)K);
  if (K % 128)
    return set_error(WZ_EINVAL, "%s: K=%lld must be a multiple of 128", what, (long long)K);
  if (N % 16)
    return set_error(WZ_EINVAL, "%s: N=%lld must be a multiple of 16", what, (long long)N);
  if (M > (1 << 30) || N > (1 << 30) || K > (1 << 30))
    return set_error(WZ_EINVAL, "%s: dimension too large", what);
  return WZ_OK;
}

}  // namespace wz

extern "C" int wz_fp8_gemm(const void* a_e4m3, const void* a_s, const void* w_e4m3, const void* w_s,
                           void* c_bf16, int64_t M, int64_t N, int64_t K, int act_scale_kind,
                           int w_scale_kind, hipStream_t stream) {
  using namespace wz;
  if (int rc = check_dims("fp8_gemm", M, N, K)) return rc;
  if (act_scale_kind < 0 || act_scale_kind > 2 || (w_scale_kind != 0 && w_scale_kind != 1))
    return set_error(WZ_EINVAL, "fp8_gemm: bad scale kinds %d/%d", act_scale_kind, w_scale_kind);
  if (M && (!a_e4m3 || !a_s || !w_e4m3 || !w_s || !c_bf16))
    return set_error(WZ_EINVAL, "fp8_gemm: null pointer");
  const bool pow2 = act_scale_kind != WZ_SCALE_F32 && w_scale_kind == WZ_WSCALE_E8M0;
  if (M > skinny_max_rows(false, pow2, N, K) && tile_rows_fits(a_e4m3, w_e4m3, w_s, false, M, N, K))
    return launch_tile_rows("fp8_gemm", static_cast<const uint8_t*>(a_e4m3), a_s, act_scale_kind,
                            static_cast<const uint8_t*>(w_e4m3), w_s, w_scale_kind, false,
                            static_cast<uint16_t*>(c_bf16), M, N, K, stream);
  return launch_skinny<kFmtFp8, false>(a_e4m3, a_s, act_scale_kind, w_e4m3, w_s, w_scale_kind,
                                       c_bf16, M, N, K, stream, "fp8_gemm");
}

extern "C" int wz_fp8_linear(const void* x_bf16, const void* w_e4m3, const void* w_s, void* y_bf16,
                             int64_t M, int64_t N, int64_t K, int act_scale_kind, int w_scale_kind,
                             hipStream_t stream) {
  using namespace wz;
  if (int rc = check_dims("fp8_linear", M, N, K)) return rc;
  if (act_scale_kind < 0 || act_scale_kind > 2 || (w_scale_kind != 0 && w_scale_kind != 1))
    return set_error(WZ_EINVAL, "fp8_linear: bad scale kinds %d/%d", act_scale_kind, w_scale_kind);
  if (M && (!x_bf16 || !w_e4m3 || !w_s || !y_bf16))
    return set_error(WZ_EINVAL, "fp8_linear: null pointer");
  return launch_skinny<kFmtFp8, true>(x_bf16, nullptr, act_scale_kind, w_e4m3, w_s, w_scale_kind,
                                      y_bf16, M, N, K, stream, "fp8_linear");
}

extern "C" int wz_fp4_gemm(const void* a_e4m3, const void* a_s, const void* w_fp4x2,
                           const void* w_s_e8m0, void* c_bf16, int64_t M, int64_t N, int64_t K,
                           int act_scale_kind, hipStream_t stream) {
  using namespace wz;
  if (int rc = check_dims("fp4_gemm", M, N, K)) return rc;
  if (act_scale_kind < 0 || act_scale_kind > 2)
    return set_error(WZ_EINVAL, "fp4_gemm: bad scale kind %d", act_scale_kind);
  if (M && (!a_e4m3 || !a_s || !w_fp4x2 || !w_s_e8m0 || !c_bf16))
    return set_error(WZ_EINVAL, "fp4_gemm: null pointer");
  if (M > skinny_max_rows(true, act_scale_kind != WZ_SCALE_F32, N, K) &&
      tile_rows_fits(a_e4m3, w_fp4x2, w_s_e8m0, true, M, N, K))
    return launch_tile_rows("fp4_gemm", static_cast<const uint8_t*>(a_e4m3), a_s, act_scale_kind,
                            static_cast<const uint8_t*>(w_fp4x2), w_s_e8m0, WZ_WSCALE_E8M0, true,
                            static_cast<uint16_t*>(c_bf16), M, N, K, stream);
  return launch_skinny<kFmtFp4, false>(a_e4m3, a_s, act_scale_kind, w_fp4x2, w_s_e8m0,
                                       WZ_WSCALE_E8M0, c_bf16, M, N, K, stream, "fp4_gemm");
}

extern "C" int wz_grouped_fp4_gemm(const void* a_e4m3, const void* a_s, const void* w_fp4x2,
                                   const void* w_s_e8m0, void* c_bf16, int64_t G, int64_t N, int64_t K,
                                   int act_scale_kind, hipStream_t stream) {
  using namespace wz;
  if (int rc = check_dims("grouped_fp4_gemm", G, N, K)) return rc;
  if (G > 65535) return set_error(WZ_EINVAL, "grouped_fp4_gemm: G=%lld rows exceed 65535", (long long)G);
  if (act_scale_kind < 0 || act_scale_kind > 2)
    return set_error(WZ_EINVAL, "grouped_fp4_gemm: bad scale kind %d", act_scale_kind);
  if (G == 0) return WZ_OK;
  if (!a_e4m3 || !a_s || !w_fp4x2 || !w_s_e8m0 || !c_bf16)
    return set_error(WZ_EINVAL, "grouped_fp4_gemm: null pointer");
  const dim3 grid(unsigned(N / 16), unsigned(G));
  const uint8_t* a = static_cast<const uint8_t*>(a_e4m3);
  const uint8_t* w = static_cast<const uint8_t*>(w_fp4x2);
  const uint8_t* ws = static_cast<const uint8_t*>(w_s_e8m0);
  uint16_t* c = static_cast<uint16_t*>(c_bf16);
  const int u = skinny_unroll(K);
  // the row kernel reads 16 bytes at a time; other K and unaligned operands take the skinny body
  const bool vec = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) |
                     reinterpret_cast<uintptr_t>(ws)) & 15) == 0 &&
                   (act_scale_kind == WZ_SCALE_UE8M0 || (reinterpret_cast<uintptr_t>(a_s) & 3) == 0);
  if (vec && K == 4096) {
    WZ_LAUNCH("grouped_fp4_gemm", stream, grouped_fp4_row_kernel<8>, grid, dim3(kGemmThreads), 0, a, a_s,
              act_scale_kind, w, ws, c, int(N));
  } else if (vec && K == 2048) {
    WZ_LAUNCH("grouped_fp4_gemm", stream, grouped_fp4_row_kernel<4>, grid, dim3(kGemmThreads), 0, a, a_s,
              act_scale_kind, w, ws, c, int(N));
  } else if (u == 8) {
    WZ_LAUNCH("grouped_fp4_gemm", stream, grouped_fp4_kernel<8>, grid, dim3(kGemmThreads), 0, a, a_s, act_scale_kind,
              w, ws, c, int(N), int(K));
  } else if (u == 4) {
    WZ_LAUNCH("grouped_fp4_gemm", stream, grouped_fp4_kernel<4>, grid, dim3(kGemmThreads), 0, a, a_s, act_scale_kind,
              w, ws, c, int(N), int(K));
  } else {
    WZ_LAUNCH("grouped_fp4_gemm", stream, grouped_fp4_kernel<2>, grid, dim3(kGemmThreads), 0, a, a_s, act_scale_kind,
              w, ws, c, int(N), int(K));
  }
  return check_launch("grouped_fp4_gemm");
}
