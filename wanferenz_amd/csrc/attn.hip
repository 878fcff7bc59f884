// Sparse attention over gathered KV rows (decode and chunked prefill).
//
// o[b, s, h, :] = sum_j p_j kv[b, idx_j, :] / (sum_j p_j + exp(sink[h] - m)),
// p_j = exp(q[b, s, h, :] . kv[b, idx_j, :] * scale - m) over the valid
// (idx >= 0) entries of topk_idxs[b, s, :], m the running maximum — the
// blockwise online softmax of wanferenz/kernels/torch_ops.py:114-146 (CPU)
// and reference.py:314-418 (GPU), one KV row shared by all heads (K = V).
// With no valid index in the first block of 64 the reference's
// exp(-inf - -inf) turns its sums into NaN for good, and so does this code.
#include "common.h"

namespace wz {

typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef short v8s_t __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

constexpr int kAttnBlock = 64;     // indices per block (the reference's SPARSE_ATTN_BLOCK)
constexpr int kAttnIdxCap = 2048;  // indices one workgroup covers (32 blocks)
constexpr int kAttnMaxSplit = 64;  // workgroups one query's blocks are split over
constexpr float kLazyMax = 8.0f;   // the running max moves when a block exceeds it by more

__device__ __forceinline__ v4f mfma_bf16_32(v8s_t a, v8s_t b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, a), __builtin_bit_cast(v8bf_t, b), c, 0,
                                                 0, 0);
}

// Floats of one (query, 64 heads, split) partial: m[64], l[64], O[64][D].
__host__ __device__ constexpr int64_t attn_part_floats(int d) { return 128 + 64 * int64_t(d); }

// LDS image of one block of 64 KV rows, row-major, no padding.  The 16-byte chunks of
// row r sit XOR-swizzled (chunk c at slot c ^ swz(r)) so that both read patterns spread
// over the banks.  A 16-byte read of one chunk of 16 rows (the K operand of S^T) is
// served in passes of 16 lanes that mix rows 0-3 and 12-15 of one lane group with rows
// 4-11 of the next, whose chunk is the neighbour: the slots of rows 0-3 and 12-15 are
// closed under ^ 1, so the passes' slots are distinct (conflicts took 44 % of the LDS
// cycles without that, 30 % with it; P's 8-byte writes and the transpose reads are the
// rest).  The transpose reads of V take two adjacent chunks of 8 consecutive rows,
// which have distinct slot pairs.
template <int D>
struct KsLayout {
  static constexpr int RB = 2 * D;             // bytes per row
  static constexpr int RPI = 1024 / RB;        // rows per 1 KB load
  static constexpr int NG = kAttnBlock / RPI;  // loads per block
  static constexpr int BYTES = kAttnBlock * RB;
  static __device__ __forceinline__ int swz(int row) {
    const int hi = (row >> 3) & 1;
    return ((row ^ (hi << 2)) & 7) << 1 | hi;
  }
  // byte address of element `col` (a multiple of 4) of `row`
  static __device__ __forceinline__ int at(int row, int col) {
    return row * RB + (((col >> 3) ^ swz(row)) << 4) + ((col & 7) << 1);
  }
};

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  return f32x2_to_bf16x2(a, b);
}

// Two floats -> packed bf16 pair with the hardware converter (round to nearest
// even, as f32_to_bf16; a NaN stays a NaN).
__device__ __forceinline__ uint32_t cvt_bf16x2(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}

// One workgroup per (query, up to 64 heads, range of 64-index blocks), 8 waves, HT tiles of
// 16 heads.  The LDS reads of the KV rows are what bounds a block, so the waves split both
// products such that a row is read as few times as the registers allow: with Q and O of 64
// heads held in registers, K twice, V once and P once a wave, 256 KB a block of 64 rows
// (2048 cycles at 128 B per cycle, as long as its MFMAs); four waves of 16 heads each, which
// read every row of K and V themselves, took 512 KB and 3.5 us a block, where this takes 2.5.
// 2048 queries of a prompt from position 0 (64 heads of 512, 6.5 of 10 blocks with valid
// indices): 346 -> 174 us, of which 57 us are the workgroups' starts and ends (Q in and O out,
// 268 MB) that one workgroup a CU does not overlap with its products; 640 valid indices for each
// of 2048 queries 347 -> 264 us.
//   * the 64 gathered KV rows sit in LDS row-major; they were loaded while the previous block
//     was computed (double buffer).  A block without a valid index (a prompt's early positions
//     have fewer selected rows than slots) adds nothing and is skipped;
//   * S^T = K Q^T with V_MFMA_F32_16X16X32_BF16: wave w has rows 16 (w & 3) .. +16 and SHT
//     head tiles.  Lane (head n, group g) then holds rows 16rt + 4g + i, four consecutive k
//     slots of the P operand below (k slots 0-3: rows 32kc + 4g + i, slots 4-7: rows 32kc +
//     16 + 4g + i), and P goes to LDS in that operand's order, 8 bytes a lane;
//   * P = exp(S - m) in bf16 (the GPU reference also multiplies a bf16 P,
//     reference.py:404-405), with m moved only when a block's maximum exceeds it by more than
//     kLazyMax (P <= e^8; the final division by the sum taken with the same m makes the result
//     independent of m).  Every wave writes its P with the m of the blocks before and flags a
//     head that needs a new one; only then a second barrier follows, after the maxima have
//     met, O is rescaled and P written again;
//   * O^T[D, heads] += V^T P^T: wave w has columns w D/8 .. +D/8 of every head, V read from
//     the row-major rows with the LDS transpose read (ds_read_b64_tr_b16: in each 16-lane
//     group, lane i addressing row base + (i >> 2), column c0 + 4(i & 3) makes lane j receive
//     rows base..base+3 of column c0 + j).  A lane holds four consecutive columns of one head.
// A workgroup that covers every block normalises (sink term included) and stores bf16, whole
// lines through LDS; for few queries the blocks are split over workgroups that store (m, l, O)
// partials and sparse_attn_combine_kernel merges them.
constexpr int kAttnWaves = 8;

// Row index that an unused entry of a block gets: its byte offset lies past any cache.
template <int D>
constexpr int kNoRow = int(0x80000000u / KsLayout<D>::RB);

// The launch's workgroups cover head groups hq0 .. hq0 + nhq of every query.
template <int D, int HT, bool SPLIT>
__global__ __launch_bounds__(64 * kAttnWaves, 2) void sparse_attn_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kv, const float* __restrict__ sink,
    const int32_t* __restrict__ idx, uint16_t* __restrict__ o, float* __restrict__ part, int S, int H, int N, int topk,
    int bps, int nsplit, int hq0, int nhq, float scale) {
  using L = KsLayout<D>;
  constexpr int KC = D / 32;                  // 32-wide d chunks of S
  constexpr int NT = D / 16 / kAttnWaves;     // 16-column tiles of O per wave
  constexpr int SHT = HT == 4 ? 2 : 1;        // head tiles of S per wave
  constexpr int NL = L::NG / kAttnWaves;      // loads of a block per wave
  static_assert(L::NG % kAttnWaves == 0, "a block's loads must split evenly over the waves");
  static_assert(L::RB / 16 >= 16, "the swizzle permutes 16 chunks of a row");
  __shared__ __align__(1024) uint8_t ksb[2][L::BYTES];
  __shared__ __align__(16) uint8_t s_p[2][16 * HT][64];  // [kc][head]: group g's 8 k slots at 16 g
  __shared__ int s_idx[kAttnIdxCap];
  __shared__ float s_max[4][64], s_l[4][64];  // [row tile][head]
  __shared__ int s_bump[kAttnIdxCap / kAttnBlock], s_used[kAttnIdxCap / kAttnBlock];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const int c = blockIdx.x % nsplit, qh = blockIdx.x / nsplit;
  const int hq = hq0 + qh % nhq, bs = qh / nhq, b = bs / S;
  const int nblk = (topk + kAttnBlock - 1) / kAttnBlock;
  const int blk0 = c * bps, blk1 = min(blk0 + bps, nblk);
  const int nb = blk1 - blk0;  // >= 1: the host never launches an empty split
  const int h0 = hq * 64;
  const int rt = wave & 3, ht0 = (wave >> 2) * SHT;  // this wave's row tile and first head tile of S
  const bool has_s = ht0 < HT;

  // Q rows into the second buffer, in the layout of a block: read from memory once in whole
  // lines, where fragments loaded by the four waves that share them took 4 us more a
  // workgroup; heads past H repeat the last one and are dropped
  const uint32_t ks_lds = lds_addr(&ksb[0][0]);
  const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(q + int64_t(bs) * H * D), short(0), H * L::RB, 0x00020000);
  for (int gi = wave; gi < 16 * HT / L::RPI; gi += kAttnWaves) {
    const int row = gi * L::RPI + lane / (L::RB / 16), slot = lane % (L::RB / 16);
    load_lds_16(q_rsrc, __builtin_amdgcn_readfirstlane(ks_lds + L::BYTES + gi * 1024),
                uint32_t(min(h0 + row, H - 1)) * L::RB + ((slot ^ L::swz(row)) << 4));
  }
  const int32_t* ib = idx + int64_t(bs) * topk + int64_t(blk0) * kAttnBlock;
  for (int j = tid; j < nb * kAttnBlock; j += 64 * kAttnWaves) {
    const int v = blk0 * kAttnBlock + j < topk ? ib[j] : -1;
    const bool ok = v >= 0 && v < N;
    s_idx[j] = ok ? v : kNoRow<D>;
    const uint64_t m = __ballot(ok);  // a wave covers one whole block
    if (lane == 0) {
      s_used[j >> 6] = m != 0;
      s_bump[j >> 6] = 0;
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // Q and the indices are in LDS
  uint32_t todo = uint32_t(__ballot(lane < nb && s_used[min(lane, nb - 1)] != 0));  // nb <= 32
  const bool poisoned = blk0 == 0 && !(todo & 1u);

  // rows of block t -> ksb[buf]; an unused index reads past the end of the
  // buffer, which returns zeros (the reference zero-fills those rows)
  const __amdgpu_buffer_rsrc_t kv_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(kv + int64_t(b) * N * D), short(0), int(int64_t(N) * L::RB), 0x00020000);
  // Load gi of a block fills rows gi * RPI .. +RPI; lane i writes slot i & (RB/16 - 1)
  // of row gi * RPI + i / (RB/16), so it fetches that row's chunk slot ^ swz(row).
  auto issue = [&](int t, int buf) {
    int ln = lane;
    asm volatile("" : "+v"(ln));  // recomputed for each block: the registers go to Q and O
    const int rin = ln / (L::RB / 16), slot = ln % (L::RB / 16);
    int ri[NL];  // every row index first: the asm loads below order memory accesses
#pragma unroll
    for (int j = 0; j < NL; ++j) ri[j] = s_idx[t * kAttnBlock + (j * kAttnWaves + wave) * L::RPI + rin];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int gi = j * kAttnWaves + wave, row = gi * L::RPI + rin;
      const uint32_t vo = uint32_t(ri[j]) * L::RB + ((slot ^ L::swz(row)) << 4);
      load_lds_16(kv_rsrc, __builtin_amdgcn_readfirstlane(ks_lds + buf * L::BYTES + gi * 1024), vo);
    }
  };
  if (todo) issue(__builtin_ctz(todo), 0);
  // Q fragments (B operand of S^T): lane (head nl, group g) holds d 32cc + 8g .. +8
  v8s_t qb[SHT][KC];
#pragma unroll
  for (int h = 0; h < SHT; ++h)
#pragma unroll
    for (int cc = 0; cc < KC; ++cc)
      qb[h][cc] = *reinterpret_cast<const v8s_t*>(ksb[1] + L::at(16 * (has_s ? ht0 + h : 0) + nl, 32 * cc + 8 * g));

  v4f acc[HT][NT];  // acc[ht][nt][i] = O[head 16ht + nl][w D/8 + 16nt + 4g + i]
#pragma unroll
  for (int ht = 0; ht < HT; ++ht)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[ht][nt] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY;  // running max of head `lane`, the same in every wave
  float m_s[SHT], l_s[SHT];  // of this lane's heads of S: the max, and its rows' share of the sum
#pragma unroll
  for (int h = 0; h < SHT; ++h) {
    m_s[h] = -INFINITY;
    l_s[h] = 0.0f;
  }

  int buf = 0;
#pragma unroll 1
  for (bool first = true; todo; first = false, buf ^= 1) {
    const int t = __builtin_ctz(todo);
    todo &= todo - 1;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of block t have landed
    __syncthreads();                // ... and every wave's; the other buffer and s_p are free
    if (todo) issue(__builtin_ctz(todo), buf ^ 1);
    const uint8_t* const ks = ksb[buf];
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int nl = ln & 15, g = ln >> 4;

    // ---- S^T[16 rows, heads]: sacc[h][i] = S[row 16rt + 4g + i][head nl of tile h] ----
    v4f sacc[SHT];
    float p_sum[SHT];
    // P = exp(S - m) in bf16 to LDS, this lane's part of the row sum to p_sum
    auto put_p = [&]() {
#pragma unroll
      for (int h = 0; h < SHT; ++h) {
        float pv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) pv[i] = sacc[h][i] == -INFINITY ? 0.0f : __expf(sacc[h][i] - m_s[h]);
        p_sum[h] = (pv[0] + pv[1]) + (pv[2] + pv[3]);
        *reinterpret_cast<uint2*>(&s_p[rt >> 1][16 * (ht0 + h) + nl][16 * g + 8 * (rt & 1)]) =
            make_uint2(cvt_bf16x2(pv[0], pv[1]), cvt_bf16x2(pv[2], pv[3]));
      }
    };
    if (has_s) {
      const uint64_t vmask = __ballot(s_idx[t * kAttnBlock + lane] != kNoRow<D>);
#pragma unroll
      for (int h = 0; h < SHT; ++h) sacc[h] = v4f{0.f, 0.f, 0.f, 0.f};
      // K fragments are read kAhead d chunks ahead of their MFMAs
      constexpr int kAhead = 3;
      // chunk (4cc + g) ^ swz: its low four bits, and 16 chunks (256 bytes) a step of the rest
      const int krow = (16 * rt + nl) * L::RB, kchunk = (g ^ L::swz(nl)) << 4;
      v8s_t kf[kAhead + 1];
      auto kload = [&](int cc) {
        kf[cc % (kAhead + 1)] = *reinterpret_cast<const v8s_t*>(ks + krow + ((4 * (cc & 3)) << 4 ^ kchunk) + (cc >> 2) * 256);
      };
#pragma unroll
      for (int cc = 0; cc < kAhead; ++cc) kload(cc);
#pragma unroll
      for (int cc = 0; cc < KC; ++cc) {
        if (cc + kAhead < KC) kload(cc + kAhead);
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of their use
#pragma unroll
        for (int h = 0; h < SHT; ++h) sacc[h] = mfma_bf16_32(kf[cc % (kAhead + 1)], qb[h][cc], sacc[h]);
        __builtin_amdgcn_sched_barrier(0);
      }
      bool bump = false;
#pragma unroll
      for (int h = 0; h < SHT; ++h) {
        float bmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sacc[h][i] = (vmask >> (16 * rt + 4 * g + i)) & 1 ? sacc[h][i] * scale : -INFINITY;
          bmax = fmaxf(bmax, sacc[h][i]);
        }
        bmax = fmaxf(bmax, __shfl_xor(bmax, 16, kWave));
        bmax = fmaxf(bmax, __shfl_xor(bmax, 32, kWave));
        bump |= bmax > m_s[h] + kLazyMax;
        if (g == 0) s_max[rt][16 * (ht0 + h) + nl] = bmax;
      }
      if (__ballot(bump)) {
        if (lane == 0) s_bump[t] = 1;
      }
      if (!first) put_p();
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the loads of the next block stay in flight
    if (first || s_bump[t]) {
      // the block's maxima have met: head `lane`
      const int hl = lane < 16 * HT ? lane : 0;
      const float bm = fmaxf(fmaxf(s_max[0][hl], s_max[1][hl]), fmaxf(s_max[2][hl], s_max[3][hl]));
      const bool bump = bm > m_run + kLazyMax;
      // nothing accumulated yet for a head without a maximum
      const float resc = !bump ? 1.0f : (m_run == -INFINITY ? 0.0f : __expf(m_run - bm));
      m_run = bump ? bm : m_run;
#pragma unroll
      for (int h = 0; h < SHT; ++h) {
        m_s[h] = __shfl(m_run, (16 * (ht0 + h) + nl) & 63, kWave);
        l_s[h] *= __shfl(resc, (16 * (ht0 + h) + nl) & 63, kWave);
      }
      if (!first) {
#pragma unroll
        for (int ht = 0; ht < HT; ++ht) {
          const float r = __shfl(resc, 16 * ht + nl, kWave);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[ht][nt] = acc[ht][nt] * r;
        }
      }
      if (has_s) put_p();
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (has_s) {
#pragma unroll
      for (int h = 0; h < SHT; ++h) l_s[h] += p_sum[h];
    }

    // ---- O^T[wave's columns, heads] += V^T[columns, 64 rows] P^T[64 rows, heads] ----
    // V fragments are read two column tiles ahead of their MFMAs
    v8s_t vf[3];
    const int vrow = 4 * g + (nl >> 2);  // rows 16 apart share their swizzle
    auto vload = [&](int j) {  // j = kc NT + nt
      const uint8_t* const p = ks + L::at(vrow, wave * 16 * NT + 16 * (j % NT) + 4 * (nl & 3)) + (j / NT) * 32 * L::RB;
      const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t*)p);
      const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t*)(p + 16 * L::RB));
      vf[j % 3] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    v8s_t pb[HT];  // of 32 rows kc; the second half's are read as the first half's are used up
    auto pload = [&](int kc, int ht) {
      pb[ht] = *reinterpret_cast<const v8s_t*>(&s_p[kc][16 * ht + nl][16 * g]);
    };
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) pload(0, ht);
    vload(0);
    vload(1);
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j) {
      if (j + 2 < 2 * NT) vload(j + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) {
        acc[ht][j % NT] = mfma_bf16_32(vf[j % 3], pb[ht], acc[ht][j % NT]);
        if (j == NT - 1) {
          __builtin_amdgcn_sched_barrier(0);
          pload(1, ht);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  if (has_s) {
#pragma unroll
    for (int h = 0; h < SHT; ++h) {
      l_s[h] += __shfl_xor(l_s[h], 16, kWave);
      l_s[h] += __shfl_xor(l_s[h], 32, kWave);
      if (g == 0) s_l[rt][16 * (ht0 + h) + nl] = l_s[h];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int hl = lane < 16 * HT ? lane : 0;
  const float l_run = (s_l[0][hl] + s_l[1][hl]) + (s_l[2][hl] + s_l[3][hl]);  // of head `lane`
  if constexpr (!SPLIT) {
    // normalise by the sum (sink term included): one reciprocal per head, then products
    // (within 1 fp32 ulp of the quotient, before the bf16 rounding); the tile goes out through
    // this wave's part of the buffer that the last block did not use, 16-byte chunks
    // XOR-swizzled by row
    const float inv_l =
        poisoned ? __builtin_nanf("") : 1.0f / (l_run + __expf(sink[min(h0 + hl, H - 1)] - m_run));
    constexpr int RB = 32 * NT, NCH = RB / 16;  // bytes and chunks of the wave's columns of a head
    uint8_t* const so = ksb[buf] + wave * (16 * HT * RB);
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      const float inv = __shfl(inv_l, 16 * ht + nl, kWave);
      const int row = 16 * ht + nl;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int ch = 2 * nt + (g >> 1);
        const v4f v = acc[ht][nt] * inv;
        *reinterpret_cast<uint2*>(so + row * RB + ((ch ^ (row & (NCH - 1))) << 4) + (g & 1) * 8) =
            make_uint2(cvt_bf16x2(v[0], v[1]), cvt_bf16x2(v[2], v[3]));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    uint16_t* const ow = o + (int64_t(bs) * H + h0) * D + wave * 16 * NT;
#pragma unroll
    for (int it = 0; it < (16 * HT * NCH + 63) / 64; ++it) {
      const int row = it * (64 / NCH) + lane / NCH, ch = lane % NCH;
      if (row >= 16 * HT || h0 + row >= H) continue;
      *reinterpret_cast<v4i*>(ow + int64_t(row) * D + ch * 8) =
          *reinterpret_cast<const v4i*>(so + row * RB + ((ch ^ (row & (NCH - 1))) << 4));
    }
  } else {
    float* const pp = part + int64_t(blockIdx.x) * attn_part_floats(D);
    if (wave == 0) {
      pp[lane] = m_run;
      pp[64 + lane] = poisoned ? __builtin_nanf("") : l_run;
    }
#pragma unroll
    for (int ht = 0; ht < HT; ++ht)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        *reinterpret_cast<v4f*>(pp + 128 + int64_t(16 * ht + nl) * D + (wave * NT + nt) * 16 + 4 * g) = acc[ht][nt];
  }
}

// The same products with a wave per 16 heads: 4 waves, wave w has heads 64 hq + 16w .. +16 (a wave
// past H only helps load).  S^T = K Q^T leaves lane (head n, group g) holding rows 16rt + 4g + i,
// the A operand of O = P V once two row tiles are paired (k slots 0-3: rows 32kc + 4g + i, slots
// 4-7: rows 32kc + 16 + 4g + i), so P stays in registers and a block costs one barrier instead of
// two.  Every wave reads all of K and V from LDS for it, which bounds wider heads (D = 512: 512 KB
// a block, 346 us where the eight waves above take 174), but at D = 128 the eight waves have 16
// MFMAs each between their barriers.  64 heads of 128, us here / there: 2 x 1024 queries of 300
// indices 55.6 / 61, 700 of 640 indices 39.8 / 43, decode of one sequence 9.4 / 10.5; 48 heads
// 52 / 60, 37.8 / 42.6, 9.2 / 9.4.  Up to 32 heads the eight waves win (32: 50 / 38, 37 / 27).
template <int D, bool SPLIT>
__global__ __launch_bounds__(256, 1) void sparse_attn_wave_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kv, const float* __restrict__ sink,
    const int32_t* __restrict__ idx, uint16_t* __restrict__ o, float* __restrict__ part, int S, int H, int N, int topk,
    int bps, int nsplit, float scale) {
  using L = KsLayout<D>;
  constexpr int KC = D / 32;     // 32-wide d chunks of S
  constexpr int NT = D / 16;     // 16-column tiles of O
  constexpr int NL = L::NG / 4;  // loads of a block per wave
  static_assert(L::NG % 4 == 0, "a block's loads must split evenly over the 4 waves");
  static_assert(L::RB / 16 >= 16, "the swizzle permutes 16 chunks of a row");
  __shared__ __align__(1024) uint8_t ksb[2][L::BYTES];
  __shared__ int s_idx[kAttnIdxCap];
  __shared__ int s_used[kAttnIdxCap / kAttnBlock];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const int HQ = (H + 63) / 64;
  const int c = blockIdx.x % nsplit, qh = blockIdx.x / nsplit;
  const int hq = qh % HQ, bs = qh / HQ, b = bs / S;
  const int nblk = (topk + kAttnBlock - 1) / kAttnBlock;
  const int blk0 = c * bps, blk1 = min(blk0 + bps, nblk);
  const int nb = blk1 - blk0;  // >= 1: the host never launches an empty split
  const int hg0 = hq * 64 + 16 * wave;
  const bool active = hg0 < H;  // H % 16 == 0: the whole head group exists

  // Q fragments (B operand of S^T): lane (head nl, group g) holds d 32cc + 8g .. +8
  v8s_t qb[KC];
  const uint16_t* const qrow = q + (int64_t(bs) * H + (active ? hg0 : 0) + nl) * D;
#pragma unroll
  for (int cc = 0; cc < KC; ++cc) qb[cc] = *reinterpret_cast<const v8s_t*>(qrow + 32 * cc + 8 * g);

  const int32_t* const ib = idx + int64_t(bs) * topk + int64_t(blk0) * kAttnBlock;
  for (int j = tid; j < nb * kAttnBlock; j += 256) {
    const int v = blk0 * kAttnBlock + j < topk ? ib[j] : -1;
    const bool ok = v >= 0 && v < N;
    s_idx[j] = ok ? v : kNoRow<D>;
    const uint64_t m = __ballot(ok);  // a wave covers one whole block
    if (lane == 0) s_used[j >> 6] = m != 0;
  }
  __syncthreads();
  uint32_t todo = uint32_t(__ballot(lane < nb && s_used[min(lane, nb - 1)] != 0));  // nb <= 32
  const bool poisoned = blk0 == 0 && !(todo & 1u);

  // rows of block t -> ksb[buf], as in sparse_attn_body
  const __amdgpu_buffer_rsrc_t kv_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(kv + int64_t(b) * N * D), short(0), int(int64_t(N) * L::RB), 0x00020000);
  const uint32_t ks_lds = lds_addr(&ksb[0][0]);
  auto issue = [&](int t, int buf) {
    const int rin = lane / (L::RB / 16), slot = lane % (L::RB / 16);
    int ri[NL];  // every row index first: the asm loads below order memory accesses
#pragma unroll
    for (int j = 0; j < NL; ++j) ri[j] = s_idx[t * kAttnBlock + (j * 4 + wave) * L::RPI + rin];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int gi = j * 4 + wave, row = gi * L::RPI + rin;
      const uint32_t vo = uint32_t(ri[j]) * L::RB + ((slot ^ L::swz(row)) << 4);
      load_lds_16(kv_rsrc, __builtin_amdgcn_readfirstlane(ks_lds + buf * L::BYTES + gi * 1024), vo);
    }
  };
  if (todo) issue(__builtin_ctz(todo), 0);

  v4f acc[NT];  // acc[nt][i] = O[head 4g + i][16nt + nl]
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_use = -INFINITY, l_run = 0.0f;  // head nl: running max, this lane's share of the sum

  for (int buf = 0; todo; buf ^= 1) {
    const int t = __builtin_ctz(todo);
    todo &= todo - 1;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of block t have landed
    __syncthreads();                // ... and every wave's; the other buffer is free
    if (todo) issue(__builtin_ctz(todo), buf ^ 1);
    const uint8_t* const ks = ksb[buf];
    const uint64_t vmask = __ballot(s_idx[t * kAttnBlock + lane] != kNoRow<D>);
    if (!active) continue;

    // ---- S^T[rows, 16 heads]: sacc[rt][i] = S[row 16rt + 4g + i][head nl] ----
    // K fragments are read two d chunks ahead of their MFMAs (three buffers)
    v4f sacc[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) sacc[rt] = v4f{0.f, 0.f, 0.f, 0.f};
    v8s_t kf[3][4];
    auto kload = [&](int cc) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
        kf[cc % 3][rt] = *reinterpret_cast<const v8s_t*>(ks + L::at(16 * rt + nl, 32 * cc + 8 * g));
    };
    kload(0);
    kload(1);
#pragma unroll
    for (int cc = 0; cc < KC; ++cc) {
      if (cc + 2 < KC) kload(cc + 2);
      __builtin_amdgcn_sched_barrier(0);  // keep the reads two chunks ahead of their use
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) sacc[rt] = mfma_bf16_32(kf[cc % 3][rt], qb[cc], sacc[rt]);
      __builtin_amdgcn_sched_barrier(0);
    }
    float bmax = -INFINITY;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sacc[rt][i] = (vmask >> (16 * rt + 4 * g + i)) & 1 ? sacc[rt][i] * scale : -INFINITY;
        bmax = fmaxf(bmax, sacc[rt][i]);
      }
    bmax = fmaxf(bmax, __shfl_xor(bmax, 16, kWave));
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32, kWave));
    const bool bump = bmax > m_use + kLazyMax;
    if (__ballot(bump)) {
      // nothing accumulated yet for a head without a maximum
      const float resc = !bump ? 1.0f : (m_use == -INFINITY ? 0.0f : __expf(m_use - bmax));
      m_use = bump ? bmax : m_use;
      l_run *= resc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float r = __shfl(resc, 4 * g + i, kWave);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt][i] *= r;
      }
    }
    v8s_t pa[2];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      float pv[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pv[i] = sacc[2 * kc][i] == -INFINITY ? 0.0f : __expf(sacc[2 * kc][i] - m_use);
        pv[4 + i] = sacc[2 * kc + 1][i] == -INFINITY ? 0.0f : __expf(sacc[2 * kc + 1][i] - m_use);
        l_run += pv[i] + pv[4 + i];
      }
      pa[kc] = __builtin_bit_cast(v8s_t, make_uint4(cvt_bf16x2(pv[0], pv[1]), cvt_bf16x2(pv[2], pv[3]),
                                                    cvt_bf16x2(pv[4], pv[5]), cvt_bf16x2(pv[6], pv[7])));
    }

    // ---- O[16 heads, D] += P[16 heads, 64 rows] V[64 rows, D] ----
    // V fragments are read two column tiles ahead of their MFMAs (three buffers)
    v8s_t vf[3][2];
    auto vload = [&](int nt) {
      const int col = 16 * nt + 4 * (nl & 3);
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const int row = 32 * kc + 4 * g + (nl >> 2);
        const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t*)(ks + L::at(row, col)));
        const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t*)(ks + L::at(row + 16, col)));
        vf[nt % 3][kc] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    };
    vload(0);
    vload(1);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt + 2 < NT) vload(nt + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) acc[nt] = mfma_bf16_32(pa[kc], vf[nt % 3][kc], acc[nt]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (!active) return;

  l_run += __shfl_xor(l_run, 16, kWave);
  l_run += __shfl_xor(l_run, 32, kWave);
  if constexpr (!SPLIT) {
    // normalise by the sum (sink term included): one reciprocal per head, then
    // products (within 1 fp32 ulp of the quotient, before the bf16 rounding)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int hd = hg0 + 4 * g + i;
      const float lh = __shfl(l_run, 4 * g + i, kWave), mh = __shfl(m_use, 4 * g + i, kWave);
      const float inv = poisoned ? __builtin_nanf("") : 1.0f / (lh + __expf(sink[hd] - mh));
      uint16_t* const orow = o + (int64_t(bs) * H + hd) * D;
#pragma unroll
      for (int nt = 0; nt < NT; nt += 2) {
        const uint32_t pr = cvt_bf16x2(acc[nt][i] * inv, acc[nt + 1][i] * inv);
        orow[16 * nt + nl] = uint16_t(pr & 0xFFFFu);
        orow[16 * nt + 16 + nl] = uint16_t(pr >> 16);
      }
    }
  } else {
    float* const pp = part + int64_t(blockIdx.x) * attn_part_floats(D);
    if (g == 0) {
      pp[16 * wave + nl] = m_use;
      pp[64 + 16 * wave + nl] = poisoned ? __builtin_nanf("") : l_run;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* const orow = pp + 128 + int64_t(16 * wave + 4 * g + i) * D;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) orow[16 * nt + nl] = acc[nt][i];
    }
  }
}

// Merge the (m, l, O) partials of 4 heads of one (query, 64 heads):
// o = sum_c e^(m_c - M) O_c / (sum_c e^(m_c - M) l_c + e^(sink - M)), M = max_c m_c.
// Every partial's (m, l) is loaded at once, then the O partials in batches of
// 16 splits, so each phase costs one memory round trip.
template <int D>
__global__ __launch_bounds__(256) void sparse_attn_combine_kernel(const float* __restrict__ part,
                                                                  const float* __restrict__ sink,
                                                                  uint16_t* __restrict__ o, int H, int nsplit) {
  constexpr int64_t PF = attn_part_floats(D);
  constexpr int kBatch = 16;
  __shared__ float s_m[4][kAttnMaxSplit], s_l[4][kAttnMaxSplit];
  __shared__ float wts[4][kAttnMaxSplit];
  __shared__ float inv[4];
  const int tid = threadIdx.x, HQ = (H + 63) / 64;
  const int k = blockIdx.x & 15, qh = blockIdx.x >> 4;
  const int hq = qh % HQ, bs = qh / HQ;
  const int hl0 = 4 * k;
  if (hq * 64 + hl0 >= H) return;  // heads come in groups of 16 (whole workgroup)
  const float* pb = part + int64_t(qh) * nsplit * PF;
  for (int j = tid; j < 4 * nsplit; j += 256) {
    const int h4 = j & 3, cs = j >> 2;
    s_m[h4][cs] = pb[cs * PF + hl0 + h4];
    s_l[h4][cs] = pb[cs * PF + 64 + hl0 + h4];
  }
  __syncthreads();
  if (tid < 4) {
    float M = -INFINITY;
    for (int cs = 0; cs < nsplit; ++cs) M = fmaxf(M, s_m[tid][cs]);
    float den = __expf(sink[hq * 64 + hl0 + tid] - M);
    for (int cs = 0; cs < nsplit; ++cs) {
      const float w = __expf(s_m[tid][cs] - M);
      wts[tid][cs] = w;
      den += w * s_l[tid][cs];
    }
    inv[tid] = 1.0f / den;
  }
  __syncthreads();
  for (int e = tid * 4; e < 4 * D; e += 256 * 4) {
    const int h4 = e / D, d = e % D;
    const float* src = pb + 128 + int64_t(hl0 + h4) * D + d;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c0 = 0; c0 < nsplit; c0 += kBatch) {
      float4 v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        v[u] = c0 + u < nsplit ? *reinterpret_cast<const float4*>(src + (c0 + u) * PF) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const float w = c0 + u < nsplit ? wts[h4][c0 + u] : 0.0f;
        a.x += w * v[u].x;
        a.y += w * v[u].y;
        a.z += w * v[u].z;
        a.w += w * v[u].w;
      }
    }
    const float s = inv[h4];
    uint16_t* orow = o + (int64_t(bs) * H + hq * 64 + hl0 + h4) * D + d;
    *reinterpret_cast<uint2*>(orow) = make_uint2(pack_bf16x2(a.x * s, a.y * s), pack_bf16x2(a.z * s, a.w * s));
  }
}

// Split of one query's blocks over workgroups: enough workgroups for the chip
// (about 512) when there are few queries, at most kAttnIdxCap indices each.
struct AttnSplit {
  int nsplit, bps;
};

static inline AttnSplit attn_split(int64_t units, int64_t topk) {
  const int nblk = int((topk + kAttnBlock - 1) / kAttnBlock);
  const int cap_bps = kAttnIdxCap / kAttnBlock;
  int want = int(units >= 512 ? 1 : (512 + units - 1) / units);
  want = std::min(std::min(want, nblk), kAttnMaxSplit);
  int bps = (nblk + want - 1) / want;
  if (bps > cap_bps) bps = cap_bps;
  const int nsplit = (nblk + bps - 1) / bps;
  return {nsplit, bps};
}

// The kernel of a shape.  Head groups hold 64 heads, up to four tiles of 16.
//  * Groups of more than two tiles of narrow heads take a wave per tile: heads of 128, and of 256
//    where the blocks are split (there 48 heads of one sequence 9.9 / 11.2 us against the eight
//    waves, 80 of eight with 2048 indices 21.9 / 23.0, 64 of 33 queries 21.7 / 22.6).
//  * Elsewhere the eight waves are compiled for one, two and four tiles.  The last group of H =
//    80, 96 or 144 has one or two, and unsplit queries give it a launch of its own with as many
//    (2 x 1024 queries of 300 indices, 80 heads of 512: 300 us with four tiles for it, 246 so).
template <int D>
static int launch_attn(const uint16_t* q, const uint16_t* kv, const float* sink, const int32_t* idx, uint16_t* o,
                       float* part, int64_t units, int S, int H, int N, int topk, AttnSplit sp, float scale,
                       hipStream_t stream) {
  const int HQ = (H + 63) / 64;
  const bool split = sp.nsplit > 1;
  const int64_t queries = units / HQ;
#define WZ_ATTN_EIGHT(HT, SPLIT, HQ0, NHQ)                                                                           \
  WZ_LAUNCH("sparse_attn", stream, (sparse_attn_kernel<D, HT, SPLIT>), dim3{unsigned(queries * (NHQ) * sp.nsplit)},  \
            dim3(64 * kAttnWaves), 0, q, kv, sink, idx, o, part, S, H, N, topk, sp.bps, sp.nsplit, HQ0, NHQ, scale)
#define WZ_ATTN_WAVE(SPLIT)                                                                                          \
  WZ_LAUNCH("sparse_attn", stream, (sparse_attn_wave_kernel<D, SPLIT>), dim3{unsigned(units * sp.nsplit)},           \
            dim3(256), 0, q, kv, sink, idx, o, part, S, H, N, topk, sp.bps, sp.nsplit, scale)
  if (H <= 16) {
    if (split) WZ_ATTN_EIGHT(1, true, 0, 1); else WZ_ATTN_EIGHT(1, false, 0, 1);
  } else if (H <= 32) {
    if (split) WZ_ATTN_EIGHT(2, true, 0, 1); else WZ_ATTN_EIGHT(2, false, 0, 1);
  } else if (split) {
    if constexpr (D <= 256)
      WZ_ATTN_WAVE(true);
    else
      WZ_ATTN_EIGHT(4, true, 0, HQ);
  } else if constexpr (D == 128) {
    WZ_ATTN_WAVE(false);
  } else {
    const int rest = H & 63;
    const int full = rest != 0 && rest <= 32 ? HQ - 1 : HQ;
    WZ_ATTN_EIGHT(4, false, 0, full);
    if (full < HQ) {
      if (int rc = check_launch("sparse_attn")) return rc;
      if (rest <= 16) WZ_ATTN_EIGHT(1, false, full, 1); else WZ_ATTN_EIGHT(2, false, full, 1);
    }
  }
#undef WZ_ATTN_WAVE
#undef WZ_ATTN_EIGHT
  if (int rc = check_launch("sparse_attn")) return rc;
  if (!split) return WZ_OK;
  WZ_LAUNCH("sparse_attn_combine", stream, sparse_attn_combine_kernel<D>, dim3{unsigned(units * 16)}, dim3(256), 0,
            part, sink, o, H, sp.nsplit);
  return check_launch("sparse_attn_combine");
}

}  // namespace wz

extern "C" int64_t wz_sparse_attn_workspace_bytes(int64_t B, int64_t S, int64_t H, int64_t D, int64_t topk) {
  using namespace wz;
  if (B <= 0 || S <= 0 || H <= 0 || topk <= 0 || H % 16) return 0;
  const int64_t units = B * S * ((H + 63) / 64);
  const AttnSplit sp = attn_split(units, topk);
  if (sp.nsplit <= 1) return 0;
  return units * sp.nsplit * attn_part_floats(int(D)) * int64_t(sizeof(float));
}

extern "C" int wz_sparse_attn(const void* q_bf16, const void* kv_bf16, const float* attn_sink,
                              const int32_t* topk_idxs, void* o_bf16, int64_t B, int64_t S, int64_t H, int64_t D,
                              int64_t N, int64_t topk, float softmax_scale, void* workspace, int64_t workspace_bytes,
                              hipStream_t stream) {
  using namespace wz;
  if (B < 0 || S < 0 || H <= 0 || N <= 0 || topk <= 0 || H % 16)
    return set_error(WZ_EINVAL, "sparse_attn: bad shape B=%lld S=%lld H=%lld (multiple of 16) N=%lld topk=%lld",
                     (long long)B, (long long)S, (long long)H, (long long)N, (long long)topk);
  if (D != 128 && D != 256 && D != 512)
    return set_error(WZ_EINVAL, "sparse_attn: head dim %lld (128, 256 or 512 are built)", (long long)D);
  if (B * S == 0) return WZ_OK;
  if (!q_bf16 || !kv_bf16 || !attn_sink || !topk_idxs || !o_bf16)
    return set_error(WZ_EINVAL, "sparse_attn: null pointer");
  if ((reinterpret_cast<uintptr_t>(q_bf16) | reinterpret_cast<uintptr_t>(kv_bf16) |
       reinterpret_cast<uintptr_t>(o_bf16) | reinterpret_cast<uintptr_t>(workspace)) & 15)
    return set_error(WZ_EINVAL, "sparse_attn: q, kv, o and the workspace must be 16-byte aligned");
  if (N * D * 2 > 0x7FFFFFFFLL)
    return set_error(WZ_EINVAL, "sparse_attn: a KV cache of %lld rows x %lld exceeds 2 GiB per sequence",
                     (long long)N, (long long)D);
  const int64_t units = B * S * ((H + 63) / 64);
  AttnSplit sp = attn_split(units, topk);
  if (sp.nsplit > kAttnMaxSplit)
    return set_error(WZ_EINVAL, "sparse_attn: topk %lld exceeds %d blocks of %d", (long long)topk,
                     kAttnMaxSplit * (kAttnIdxCap / kAttnBlock), kAttnBlock);
  const int64_t need = wz_sparse_attn_workspace_bytes(B, S, H, D, topk);
  if (sp.nsplit > 1 && (!workspace || workspace_bytes < need)) {
    if (workspace)
      return set_error(WZ_EINVAL, "sparse_attn: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
                       (long long)need);
    // no workspace: one workgroup per (query, 64 heads) over every block
    if (topk > kAttnIdxCap)
      return set_error(WZ_EINVAL, "sparse_attn: topk %lld > %d needs a workspace (wz_sparse_attn_workspace_bytes)",
                       (long long)topk, kAttnIdxCap);
    sp = AttnSplit{1, int((topk + kAttnBlock - 1) / kAttnBlock)};
  }
  const uint16_t* q = static_cast<const uint16_t*>(q_bf16);
  const uint16_t* kv = static_cast<const uint16_t*>(kv_bf16);
  uint16_t* o = static_cast<uint16_t*>(o_bf16);
  float* part = static_cast<float*>(workspace);
  if (D == 512)
    return launch_attn<512>(q, kv, attn_sink, topk_idxs, o, part, units, int(S), int(H), int(N), int(topk), sp,
                            softmax_scale, stream);
  if (D == 256)
    return launch_attn<256>(q, kv, attn_sink, topk_idxs, o, part, units, int(S), int(H), int(N), int(topk), sp,
                            softmax_scale, stream);
  return launch_attn<128>(q, kv, attn_sink, topk_idxs, o, part, units, int(S), int(H), int(N), int(topk), sp,
                          softmax_scale, stream);
}
