// Block-scaled tile GEMM: y[M, N] (bf16) = dequant(xq) . dequant(W)^T for more rows than
// the GEMV and skinny kernels serve well (fp8_gemm reference.py:292-311, fp4_gemm
// reference.py:572-591; CPU statement torch_ops.py:93-108), on three weight forms:
//   packed     the tiles wz_fp8_pack writes ([N/16][K/128][2][1 KB] in MFMA lane order)
//   rows       e4m3 [N, K] as the reference's callers hold it
//   rows, fp4  e2m1 [N, K/2] with one e8m0 scale per 32 K
//
// Summation order.  The order of a shape is fixed by the kernel that serves few rows, so
// an output element has the same bits at every M (the reference enables its decode GEMV
// only where it is bit-equal to its GEMM, fp8_vector.py:235-252): K is cut into slices, each
// accumulated from zero through the MFMA chain (or, for float scales, one scaled partial per
// K-block added on the VALU), and the slices are summed in order.  Packed weights take the
// GEMV's slices (the K range of one GEMV wave: K = 1024 -> 1 K-block, 2048 -> 2, 4096 -> 2,
// 8192 -> 4), row-major ones skinny_gemm_kernel's four K quarters.
//
// Tiles.  A workgroup of WM x WN waves owns BM x BN outputs; a wave owns RT x CT tiles of
// 16 x 16.  Each K-block's A rows (BM x 128 e4m3) and weights are brought into LDS by 16-byte
// buffer loads that write LDS directly, in stages of KS K-blocks, S stages ahead through S + 1
// buffers; a stage's loads go out right after the barrier that frees its buffer, ahead of the
// previous stage's MFMAs.  Row-major operands are staged 128 bytes to a row, their 16-byte
// chunks XOR-swizzled by row so an operand read (one chunk of 16 rows) is free of bank
// conflicts.  No load in the loop has a register destination, so the compiler inserts no memory
// waits there.  The block scales of the whole K range sit in LDS from the start, K-block major.
// The weight is the MFMA's first operand: a lane then holds four consecutive columns of one
// row, scaled by one activation scale, and the bf16 tile goes out through LDS in 16-byte
// stores, whole 128-byte lines for CT = 4.
// Workgroups are renumbered with xcd_runs so the M-tiles of one N-block (which read the same
// weights) run on one XCD, one after the other in its L2.
#include "mfma_ops.h"

#include <algorithm>

namespace wz {

constexpr size_t kTileLds = 160 * 1024;

enum : int { kWPacked = 0, kWRows = 1, kWRowsFp4 = 2 };

template <int RT_, int CT_, int WM_, int WN_, int S_, int KS_, int OCC_>
struct TileCfg {
  static constexpr int RT = RT_, CT = CT_;         // 16 x 16 tiles per wave
  static constexpr int WM = WM_, WN = WN_;         // waves along M and N
  static constexpr int S = S_, KS = KS_;           // stages in flight; K-blocks per stage
  static constexpr int OCC = OCC_;                 // workgroups the registers leave room for on a CU
  static constexpr int W = WM * WN, NT = 64 * W;   // waves, threads
  static constexpr int BM = 16 * RT * WM, BN = 16 * CT * WN;
  static constexpr int NBUF = S + 1;
  static constexpr int LA = BM / 8 / W;            // 1-KB loads of A per wave per K-block
  static_assert(BM % (8 * W) == 0 && BN % (8 * W) == 0, "every wave takes a share of both operands");
  static_assert(128 % (CT * 16) == 0, "a wave's columns share one weight-scale block");
};

// LDS bytes of one stage and the loads each wave issues for it.
template <class C, int WF>
struct StageOf {
  static constexpr int BB = WF == kWRowsFp4 ? 64 : 128;  // weight bytes per column and K-block
  static constexpr int A_BYTES = C::KS * C::BM * 128, B_BYTES = C::KS * C::BN * BB;
  static constexpr int BYTES = A_BYTES + B_BYTES;
  static constexpr int UB = WF == kWRowsFp4 ? 2 : 1;      // K-blocks per 128-byte weight row
  static constexpr int LB = C::BN / 8 / C::W;             // 1-KB weight loads per wave per UB K-blocks
  static constexpr int LW = C::KS * C::LA + (C::KS / UB) * LB;
  static_assert(WF != kWRowsFp4 || C::KS % 2 == 0, "a 128-byte row of fp4 weights holds two K-blocks");
  static_assert((C::S - 1) * LW < 64, "the stage wait is a vmcnt immediate");
};

// slot of the 16-byte chunk q of a staged row r: q ^ gemm_swz(r), so the 16 rows of an
// operand read (one chunk each) fall in distinct banks
__device__ __forceinline__ int gemm_swz(int row) { return (row >> 1) & 7; }

// Activation block scales kept in LDS for the whole K range: power-of-two
// scales as their exponent bytes (what the MFMA takes), float scales as floats.
template <bool AP2>
struct AScaleT {
  using T = float;
};
template <>
struct AScaleT<true> {
  using T = uint8_t;
};

// The end of slice s of the summation order: ((s + 1) num) / den K-blocks.
struct SliceOrder {
  int num, den;
  __device__ __forceinline__ int end(int s) const { return ((s + 1) * num) / den; }
};

struct TileArgs {
  const uint8_t* xq;
  const void* xs;  // [M, K/128]: float, or e8m0 bytes (xs_bytes)
  int xs_bytes;
  const uint8_t* w;
  const void* w_s;
  const uint16_t* res;
  uint16_t *y, *y_hi;  // columns from n_split on go to y_hi
  int n_split, M, N, K;
  SliceOrder order;
  int n_mt, n_nb;
  int vec;  // y, y_hi and res allow 16-byte accesses
};

// SL1: every slice is one K-block, and both scales ride in the MFMA.
template <class C, int WF, bool AP2, bool BP2, bool SL1>
__global__ __launch_bounds__(C::NT, C::OCC * C::W / 4) void tile_gemm_kernel(TileArgs p) {
  using AS = typename AScaleT<AP2>::T;
  using St = StageOf<C, WF>;
  constexpr bool F4 = WF == kWRowsFp4;
  constexpr int FMT = F4 ? kFmtFp4 : kFmtFp8;
  constexpr bool CH = AP2 && BP2;  // both scales ride in the MFMA: the slice chains through it
  static_assert(CH || !SL1);
  extern __shared__ __align__(1024) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int M = p.M, N = p.N, K = p.K, KB = K / 128;
  const int t = xcd_runs(int(blockIdx.x), 0, p.n_mt * p.n_nb);
  const int mt = t % p.n_mt, nb = t / p.n_mt;
  const int m0 = mt * C::BM, n0 = nb * C::BN;
  constexpr int NSB = (C::BN + 127) / 128;  // weight-scale blocks along the tile's columns
  uint8_t* const ws_b = lds + C::NBUF * St::BYTES;  // fp4: [KB][BN][4] bytes; else float [NSB][KB]
  float* const ws_l = reinterpret_cast<float*>(ws_b);
  AS* const as_l = reinterpret_cast<AS*>(ws_b + (F4 ? KB * C::BN * 4 : NSB * KB * 4));  // [KB][BM]

  // this wave's direct loads of a K-block: rows 8i .. 8i+7 (lane l: row 8i + l/8, slot
  // l%8 holding chunk slot ^ swz(row)); packed weights: 1-KB half b%2 of tile b/2
  const __amdgpu_buffer_rsrc_t a_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.xq), short(0), M * K, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), short(0), F4 ? N * (K / 2) : N * K, 0x00020000);
  uint32_t avo[C::LA], bvo[St::LB];
#pragma unroll
  for (int j = 0; j < C::LA; ++j) {
    const int row = 8 * (wave * C::LA + j) + (lane >> 3);
    const int src = min(m0 + row, M - 1);  // rows past M repeat the last; their outputs are dropped
    avo[j] = uint32_t(src) * uint32_t(K) + uint32_t(((lane & 7) ^ gemm_swz(row)) << 4);
  }
#pragma unroll
  for (int j = 0; j < St::LB; ++j) {
    const int b = wave * St::LB + j;
    if constexpr (WF == kWPacked) {
      const int nt = min(n0 / 16 + (b >> 1), N / 16 - 1);  // tiles past N repeat the last; dropped
      bvo[j] = uint32_t(nt) * uint32_t(KB) * 2048u + uint32_t(b & 1) * 1024u + uint32_t(lane) * 16u;
    } else {
      const int row = 8 * b + (lane >> 3), src = min(n0 + row, N - 1);
      bvo[j] = uint32_t(src) * uint32_t(F4 ? K / 2 : K) + uint32_t(((lane & 7) ^ gemm_swz(row)) << 4);
    }
  }
  const uint32_t lds0 = lds_addr(lds);
  // stage q holds K-blocks q KS .. q KS + KS - 1 (past the end: the last, unread)
  auto issue = [&](int q, int buf) {
    const uint32_t sa = lds0 + uint32_t(buf) * St::BYTES, sb = sa + St::A_BYTES;
#pragma unroll
    for (int u = 0; u < C::KS; ++u) {
      const int kb = min(q * C::KS + u, KB - 1);
#pragma unroll
      for (int j = 0; j < C::LA; ++j)
        load_lds_16(a_rs, __builtin_amdgcn_readfirstlane(sa + u * C::BM * 128 + (wave * C::LA + j) * 1024), avo[j],
                    uint32_t(kb) * 128u);
    }
#pragma unroll
    for (int u = 0; u < C::KS; u += St::UB) {
      const int kb = min(q * C::KS + u, KB - St::UB);
#pragma unroll
      for (int j = 0; j < St::LB; ++j)
        load_lds_16(b_rs, __builtin_amdgcn_readfirstlane(sb + (u / St::UB) * C::BN * 128 + (wave * St::LB + j) * 1024),
                    bvo[j], uint32_t(kb) * (WF == kWPacked ? 2048u : uint32_t(St::BB)));
    }
  };

  // the first S stages, then the scales with ordinary loads: the compiler's
  // wait for those drains the stages as well, one round trip for both
  const int NQ = (KB + C::KS - 1) / C::KS;
#pragma unroll
  for (int q = 0; q < C::S; ++q)
    if (q < NQ) issue(q, q);
  for (int i = tid; i < C::BM * KB; i += C::NT) {
    const int r = i / KB, kb = i - r * KB;
    const int64_t si = int64_t(min(m0 + r, M - 1)) * KB + kb;
    if constexpr (AP2)
      as_l[kb * C::BM + r] = p.xs_bytes ? static_cast<const uint8_t*>(p.xs)[si]
                                        : uint8_t((static_cast<const uint32_t*>(p.xs)[si] >> 23) & 0xFFu);
    else
      as_l[kb * C::BM + r] = static_cast<const float*>(p.xs)[si];
  }
  if constexpr (F4) {
    for (int i = tid; i < C::BN * KB; i += C::NT) {
      const int c = i / KB, kb = i - c * KB;
      reinterpret_cast<uint32_t*>(ws_b)[kb * C::BN + c] =
          static_cast<const uint32_t*>(p.w_s)[int64_t(min(n0 + c, N - 1)) * KB + kb];
    }
  } else {
    for (int i = tid; i < NSB * KB; i += C::NT) {
      const int sb = i / KB, kb = i - sb * KB;
      const int64_t si = int64_t(min(n0 / 128 + sb, (N + 127) / 128 - 1)) * KB + kb;
      ws_l[i] = BP2 ? e8m0_to_f32(static_cast<const uint8_t*>(p.w_s)[si]) : static_cast<const float*>(p.w_s)[si];
    }
  }
  __syncthreads();

  // sac: the current slice; tot: the slices summed (-0 is the identity, so the
  // first slice enters as it is)
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  v4f sac[C::RT][C::CT], tot[C::RT][C::CT];
#pragma unroll
  for (int r = 0; r < C::RT; ++r)
#pragma unroll
    for (int c = 0; c < C::CT; ++c) {
      sac[r][c] = zero;
      tot[r][c] = v4f{-0.f, -0.f, -0.f, -0.f};
    }
  const int arow0 = wm * 16 * C::RT, bcol0 = wn * 16 * C::CT;  // the wave's first row and column in the tile
  const int wsb = (n0 % 128 + bcol0) / 128 * KB;
  int s = 0, s_end = p.order.end(0);
  while (s_end <= 0) s_end = p.order.end(++s);

  int buf = 0;
  for (int q = 0; q < NQ; ++q) {
    // this stage's loads have landed: those of the min(S - 1, NQ - 1 - q) later stages may not have
    if (C::S >= 3 && NQ - 1 - q >= 2)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((C::S >= 3 ? 2 : 0) * St::LW) : "memory");
    else if (C::S >= 2 && NQ - 1 - q >= 1)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((C::S >= 2 ? 1 : 0) * St::LW) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    // every wave has finished stage q - 1: its buffer takes stage q + S
    if (q + C::S < NQ) issue(q + C::S, buf == 0 ? C::NBUF - 1 : buf - 1);
    const uint8_t* const st = lds + buf * St::BYTES;
    buf = buf + 1 == C::NBUF ? 0 : buf + 1;
#pragma unroll
    for (int u = 0; u < C::KS; ++u) {
      const int kb = q * C::KS + u;
      if (C::KS > 1 && kb >= KB) break;  // a ragged last stage
      const uint8_t* const sa = st + u * C::BM * 128;
      const uint8_t* const sb = st + St::A_BYTES + (u / St::UB) * C::BN * 128;
      v8i bv[C::CT];
      int wse[C::CT];
      float wsf = 1.0f;
      if constexpr (!F4) wsf = ws_l[wsb + kb];
#pragma unroll
      for (int c = 0; c < C::CT; ++c) {
        const int col = bcol0 + c * 16 + nl;
        if constexpr (F4) {
          const v4i lo = *reinterpret_cast<const v4i*>(sb + col * 128 + (((4 * (u & 1) + g) ^ gemm_swz(col)) << 4));
          bv[c] = v8i{lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
          wse[c] = int(ws_b[(kb * C::BN + col) * 4 + g]);
        } else {
          const uint8_t* const b0 =
              WF == kWPacked ? sb + ((wn * C::CT + c) * 2) * 1024 + lane * 16 : sb + col * 128;
          const int sw = gemm_swz(col);
          const v4i lo = *reinterpret_cast<const v4i*>(WF == kWPacked ? b0 : b0 + ((g ^ sw) << 4));
          const v4i hi = *reinterpret_cast<const v4i*>(WF == kWPacked ? b0 + 1024 : b0 + (((g + 4) ^ sw) << 4));
          bv[c] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          wse[c] = BP2 ? int((__float_as_uint(wsf) >> 23) & 0xFFu) : kE8m0One;
        }
      }
      const bool last = !SL1 && (kb + 1 == s_end || kb + 1 == KB);
#pragma unroll
      for (int r = 0; r < C::RT; ++r) {
        const int row = arow0 + r * 16 + nl, sw = gemm_swz(row);
        const uint8_t* const pa = sa + row * 128;
        const v4i lo = *reinterpret_cast<const v4i*>(pa + ((g ^ sw) << 4));
        const v4i hi = *reinterpret_cast<const v4i*>(pa + (((g + 4) ^ sw) << 4));
        const v8i av = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        const AS as = as_l[kb * C::BM + row];
        const int ase = AP2 ? int(as) : kE8m0One;
        // float scales: (activation scale x weight scale) first, then one multiply-add per
        // K-block, the GEMV's and the skinny kernel's form (mma_step)
        const float sf = (AP2 ? 1.0f : float(as)) * (F4 || BP2 ? 1.0f : wsf);
#pragma unroll
        for (int c = 0; c < C::CT; ++c) {
          if constexpr (CH && !SL1) {
            sac[r][c] = mfma_scaled<FMT, kFmtFp8>(bv[c], av, sac[r][c], wse[c], ase);
          } else {
            const v4f d = mfma_scaled<FMT, kFmtFp8>(bv[c], av, zero, wse[c], ase);
            v4f& a = SL1 ? tot[r][c] : sac[r][c];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] += CH ? d[i] : d[i] * sf;
          }
        }
      }
      if (last) {
#pragma unroll
        for (int r = 0; r < C::RT; ++r)
#pragma unroll
          for (int c = 0; c < C::CT; ++c) {
            tot[r][c] = tot[r][c] + sac[r][c];
            sac[r][c] = zero;
          }
        if (kb + 1 < KB) {
          do s_end = p.order.end(++s);
          while (s_end <= kb + 1);
        }
      }
    }
  }

  // the wave's rows x columns as bf16 in its own part of the stage buffers (every wave has
  // read its last stage), 16-byte chunks XOR-swizzled by row, then out in 16-byte stores
  __syncthreads();
  constexpr int RB = 32 * C::CT, NCH = RB / 16;  // bytes and chunks of a wave's row
  static_assert(C::W * 16 * C::RT * RB <= C::NBUF * StageOf<C, WF>::BYTES, "the bf16 tile fits the stage buffers");
  uint8_t* const so = lds + wave * (16 * C::RT * RB);
#pragma unroll
  for (int r = 0; r < C::RT; ++r)
#pragma unroll
    for (int c = 0; c < C::CT; ++c) {
      const int row = r * 16 + nl, ch = 2 * c + (g >> 1);
      *reinterpret_cast<uint2*>(so + row * RB + ((ch ^ (row & (NCH - 1))) << 4) + (g & 1) * 8) =
          make_uint2(f32x2_to_bf16x2(tot[r][c][0], tot[r][c][1]), f32x2_to_bf16x2(tot[r][c][2], tot[r][c][3]));
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int it = 0; it < (16 * C::RT * NCH + 63) / 64; ++it) {
    const int row = it * (64 / NCH) + lane / NCH, ch = lane % NCH;
    if (row >= 16 * C::RT) continue;  // a wave of one tile: half its lanes
    v4i v = *reinterpret_cast<const v4i*>(so + row * RB + ((ch ^ (row & (NCH - 1))) << 4));
    const int gr = m0 + arow0 + row, col = n0 + bcol0 + ch * 8;
    if (gr >= M || col >= N) continue;
    const bool hi = col >= p.n_split;
    const int64_t o = hi ? int64_t(gr) * (N - p.n_split) + (col - p.n_split) : int64_t(gr) * p.n_split + col;
    uint16_t* const dst = (hi ? p.y_hi : p.y) + o;
    if (p.res) {
      // the residual stream: the product rounded to bf16, then one fp32 add
      const uint16_t* const rp = p.res + o;
      v4i rv;
      if (p.vec) {
        rv = load16(rp);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) rv[i] = int(uint32_t(rp[2 * i]) | (uint32_t(rp[2 * i + 1]) << 16));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = int(f32x2_to_bf16x2(bf16lo(uint32_t(v[i])) + bf16lo(uint32_t(rv[i])),
                                   bf16hi(uint32_t(v[i])) + bf16hi(uint32_t(rv[i]))));
    }
    if (p.vec) {
      *reinterpret_cast<v4i*>(dst) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dst[2 * i] = uint16_t(uint32_t(v[i]) & 0xFFFFu);
        dst[2 * i + 1] = uint16_t(uint32_t(v[i]) >> 16);
      }
    }
  }
}

// ------------------------------------------------------------------ host ----

// A tile shape and its cost: t1 is the time of a grid of at most one workgroup per CU, t2 that
// of a full round of PER_CU workgroups on every CU (us at K = 4096, power-of-two activation
// scales, measured).  Over 17 ... 2048 rows, K = 1024 ... 12288 and both scale kinds the shape of
// the lowest cost takes 0.3 to 1.1 % more time than the fastest on average, 28 % at worst.
template <class C_, int PER_CU_, int T1_, int T2_>
struct TileShape {
  using C = C_;
  static constexpr int PER_CU = PER_CU_;
  static constexpr double T1 = 0.1 * T1_, T2 = 0.1 * T2_;
};

template <class C, int WF>
static size_t tile_lds(int64_t K, bool a_pow2) {
  const size_t kb = size_t(K / 128);
  return size_t(C::NBUF) * StageOf<C, WF>::BYTES + kb * 4 * (WF == kWRowsFp4 ? C::BN : (C::BN + 127) / 128) +
         size_t(C::BM) * kb * (a_pow2 ? 1 : 4);
}

template <class C, int WF, bool AP2, bool BP2, bool SL1>
static int launch_tile(const char* name, TileArgs p, hipStream_t stream) {
  const size_t lds = tile_lds<C, WF>(p.K, AP2);
  static LdsGrant grant;
  if (int rc = allow_lds(name, tile_gemm_kernel<C, WF, AP2, BP2, SL1>, lds, grant)) return rc;
  p.n_mt = (p.M + C::BM - 1) / C::BM;
  p.n_nb = (p.N + C::BN - 1) / C::BN;
  WZ_LAUNCH(name, stream, (tile_gemm_kernel<C, WF, AP2, BP2, SL1>), dim3(unsigned(p.n_mt * p.n_nb)), dim3(C::NT), lds,
            p);
  return check_launch(name);
}

template <class C, int WF, bool AP2, bool SL1>
static int launch_tile_kinds(const char* name, const TileArgs& p, bool b_pow2, hipStream_t stream) {
  if constexpr (SL1 || WF == kWRowsFp4)  // fp4 scales are e8m0
    return launch_tile<C, WF, AP2, true, SL1>(name, p, stream);
  else
    return b_pow2 ? launch_tile<C, WF, AP2, true, false>(name, p, stream)
                  : launch_tile<C, WF, AP2, false, false>(name, p, stream);
}

// Time of the whole grid in rounds of the shape (infinite where its LDS does not fit).  A CU holds
// PER_CU workgroups, or one where the K range's scales (four bytes a row and K-block for float
// ones) leave room for no more: a round of those costs T1.
template <class Sh, int WF>
static double shape_cost(const TileArgs& p, bool a_pow2) {
  using C = typename Sh::C;
  const size_t lds = tile_lds<C, WF>(p.K, a_pow2);
  if (lds > kTileLds) return 1e30;
  const int64_t cus = cu_count(), held = std::min<int64_t>(Sh::PER_CU, kTileLds / lds);
  const int64_t blocks = int64_t((p.M + C::BM - 1) / C::BM) * ((p.N + C::BN - 1) / C::BN);
  if (blocks <= cus) return Sh::T1;
  const int64_t round = cus * held;
  return double((blocks + round - 1) / round) * (held == Sh::PER_CU ? Sh::T2 : Sh::T1);
}

template <int WF, bool AP2, bool SL1, class... Shapes>
static int launch_best(const char* name, const TileArgs& p, bool b_pow2, hipStream_t stream) {
  const double cost[] = {shape_cost<Shapes, WF>(p, AP2)...};
  const int best = int(std::min_element(cost, cost + sizeof...(Shapes)) - cost);
  int i = 0, rc = WZ_OK;
  (void)((i++ == best ? (rc = launch_tile_kinds<typename Shapes::C, WF, AP2, SL1>(name, p, b_pow2, stream), true)
                      : false) ||
         ...);
  return rc;
}

// The shapes, each the fastest of its size in a sweep of waves, stages and K-blocks per stage
// over M = 17 ... 2048 and the projection sizes.  More waves on a CU win (they hide the LDS
// reads and the barriers of each other): 128 x 128 as eight waves of 32 x 64, two workgroups a
// CU with one stage in flight each, 48.6 us at 2048 x 4096 x 4096 (1.41 PFLOP/s) against 63
// as four waves of 64 x 64 with three stages at one a CU, and 104 for the four-wave kernel
// with column-major bf16 stores before it.  Where a grid leaves CUs idle the smaller shapes win
// although they read each operand more often.  At K = 1024 with power-of-two scales (a slice is
// one K-block, so no second accumulator) 256 x 256 fits: 1999 x 40960 x 1024 in 140 us
// against 163 as 128 x 128; in a run of passes 115 us (1.46 PFLOP/s), the four-wave kernel 361.
// Row-major weights against skinny_gemm_kernel, which re-reads the rows once per 16 columns:
// fp8 100 x 4096 x 4096 33 -> 11.4 us, fp4 333 x 2048 x 4096 59 -> 12.5 us.
using Sh32 = TileShape<TileCfg<1, 1, 2, 2, 1, 8, 2>, 1, 105, 105>;
using Sh32w = TileShape<TileCfg<1, 2, 2, 2, 2, 2, 2>, 2, 122, 144>;
// 64 x 64 is one of the choices where float scales leave one 32 x 64 workgroup a CU: 200 x 4096 x
// 8192 in 27.5 us against 45.0, 512 x 2048 x 12288 in 37.0 against 63.4.
using Sh64 = TileShape<TileCfg<1, 2, 4, 2, 2, 2, 2>, 1, 147, 153>;
using Sh64w = TileShape<TileCfg<1, 4, 4, 2, 2, 1, 2>, 2, 184, 297>;
using Sh128 = TileShape<TileCfg<2, 4, 4, 2, 1, 1, 2>, 2, 270, 486>;
using Sh256 = TileShape<TileCfg<8, 4, 2, 4, 1, 1, 1>, 1, 800, 800>;
// fp4 weights: two K-blocks to a staged row, half the weight bytes
using Sf32 = TileShape<TileCfg<1, 1, 2, 2, 2, 4, 2>, 2, 97, 115>;
using Sf32w = TileShape<TileCfg<1, 2, 2, 2, 1, 4, 2>, 2, 122, 138>;
using Sf64 = TileShape<TileCfg<1, 2, 4, 2, 1, 4, 2>, 1, 125, 125>;
using Sf64w = TileShape<TileCfg<1, 4, 4, 2, 1, 2, 2>, 2, 173, 353>;
using Sf128 = TileShape<TileCfg<2, 4, 4, 2, 1, 2, 1>, 1, 250, 290>;

// K-blocks per slice of the canonical summation order (the GEMV's per-wave K
// range at the K it serves; one slice elsewhere).
int gemv_slice_blocks(int64_t K);

// Whether the tile GEMM serves these dimensions: operands addressable by 32-bit buffer offsets,
// and K up to where the smallest shapes hold the K range's scales in LDS.
constexpr int64_t kTileMaxK = 124 * 128;
bool tile_gemm_fits(int64_t M, int64_t N, int64_t K) {
  return M * K < (int64_t(1) << 31) && N * K < (int64_t(1) << 31) && K % 128 == 0 && N % 16 == 0 && K <= kTileMaxK;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// xs: the rows' block scales of kind a_kind (WZ_SCALE_*).
int launch_tile_gemm(const uint8_t* xq, const void* xs, int a_kind, const uint8_t* wp, const void* w_s, int w_kind,
                     const uint16_t* res, uint16_t* y, uint16_t* y_hi, int64_t n_split, int64_t M, int64_t N,
                     int64_t K, hipStream_t stream) {
  if (!tile_gemm_fits(M, N, K))
    return set_error(WZ_EINVAL, "fp8 tile gemm: M=%lld N=%lld K=%lld outside its range", (long long)M, (long long)N,
                     (long long)K);
  const int slice = gemv_slice_blocks(K);
  const bool ap = a_kind != WZ_SCALE_F32, bp = w_kind == WZ_WSCALE_E8M0;
  TileArgs p = {};
  p.xq = xq;
  p.xs = xs;
  p.xs_bytes = a_kind == WZ_SCALE_UE8M0;
  p.w = wp;
  p.w_s = w_s;
  p.res = res;
  p.y = y;
  p.y_hi = y_hi;
  p.n_split = int(n_split);
  p.M = int(M);
  p.N = int(N);
  p.K = int(K);
  p.order = SliceOrder{slice, 1};
  p.vec = aligned16(y) && aligned16(y_hi) && aligned16(res) && n_split % 8 == 0;
  if (slice == 1 && ap && bp)
    return launch_best<kWPacked, true, true, Sh32, Sh32w, Sh64w, Sh128, Sh256>("fp8_tile_gemm", p, bp, stream);
  if (ap) return launch_best<kWPacked, true, false, Sh32, Sh32w, Sh64w, Sh128>("fp8_tile_gemm", p, bp, stream);
  return launch_best<kWPacked, false, false, Sh32, Sh32w, Sh64, Sh64w, Sh128>("fp8_tile_gemm", p, bp, stream);
}

// Row-major weights (e4m3, or e2m1 with fp4) in skinny_gemm_kernel's summation order.  Served where the
// tile GEMM's range holds the operands and its 16-byte loads are aligned; fp4 rows are staged two
// K-blocks at a time, so K must be a multiple of 256, and their scales are read as dwords.
bool tile_rows_fits(const void* a, const void* w, const void* w_s, bool fp4, int64_t M, int64_t N, int64_t K) {
  return tile_gemm_fits(M, N, K) && aligned16(a) && aligned16(w) &&
         (!fp4 || (K % 256 == 0 && (reinterpret_cast<uintptr_t>(w_s) & 3) == 0));
}

int launch_tile_rows(const char* name, const uint8_t* a, const void* a_s, int a_kind, const uint8_t* w,
                     const void* w_s, int w_kind, bool fp4, uint16_t* c, int64_t M, int64_t N, int64_t K,
                     hipStream_t stream) {
  const bool ap = a_kind != WZ_SCALE_F32, bp = fp4 || w_kind == WZ_WSCALE_E8M0;
  TileArgs p = {};
  p.xq = a;
  p.xs = a_s;
  p.xs_bytes = a_kind == WZ_SCALE_UE8M0;
  p.w = w;
  p.w_s = w_s;
  p.y = c;
  p.n_split = int(N);
  p.M = int(M);
  p.N = int(N);
  p.K = int(K);
  p.order = SliceOrder{int(K / 128), 4};
  p.vec = aligned16(c);
  if (fp4)
    return ap ? launch_best<kWRowsFp4, true, false, Sf32, Sf32w, Sf64, Sf64w, Sf128>(name, p, bp, stream)
              : launch_best<kWRowsFp4, false, false, Sf32, Sf32w, Sf64, Sf64w, Sf128>(name, p, bp, stream);
  return ap ? launch_best<kWRows, true, false, Sh32, Sh32w, Sh64w, Sh128>(name, p, bp, stream)
            : launch_best<kWRows, false, false, Sh32, Sh32w, Sh64, Sh64w, Sh128>(name, p, bp, stream);
}

}  // namespace wz
