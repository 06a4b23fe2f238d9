// proj_gemm.hip -- the GEMM on a weight widened to f16 (Q6_K, Q8_0, BF16 in
// their device layouts, f32, and Q4_K of narrow outputs), for prefill rows, and
// the f32 / bf16 weight GEMV of a few rows.
//
// The reference runs these weights as BF16 after widening them at load
// (transformer4.rs:1233-1242) and multiplies on the CPU in f32
// (MatBf16::matmul_by_t, autograd2.rs:757-852).  Here each row of W is
// widened to f16 with a power-of-two scale 2^-ew[n] (max |w'| in
// [2^14, 2^15), exact for BF16, Q8_0 and Q6_K codes times their f16 scales up
// to f16 rounding), A gets the same treatment per row (in the same launch, or
// k_gemm_prep for a set), and k_gemm_f16_t128 or k_gemm_f16_t256 multiplies on
// v_mfma_f32_32x32x16_f16 with the scales restored in the epilogue, as the
// Q4_K GEMM does.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/rt_hip.h"
#include "kquant_layout.hpp"
#include "mfma_common.hpp"
#include "rt_device.hpp"
#include "rt_kernels.hpp"

namespace rt {
namespace {

// Elements 8p .. 8p+7 of row n of a weight in format FMT (decode_*_to_f32 values).
template <int FMT>
RT_DEV void proj_load8(const uint8_t *__restrict__ W, int N, int K, int n, int p, float (&v)[8]) {
#pragma clang fp contract(off)
  if constexpr (FMT == RT_LINEAR_BF16) {
    const uint4 q = reinterpret_cast<const uint4 *>(W)[(size_t)n * (K / 8) + p];
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[2 * i] = bf16_lo(u[i]), v[2 * i + 1] = bf16_hi(u[i]);
  } else if constexpr (FMT == RT_LINEAR_F32) {
    const float4 *r = reinterpret_cast<const float4 *>(W) + (size_t)n * (K / 4) + 2 * p;
    const float4 a = r[0], b = r[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else if constexpr (FMT == RT_LINEAR_Q8_0) {
    const uint2 q = reinterpret_cast<const uint2 *>(W)[(size_t)n * (K / 8) + p];
    const float d = half_bits_to_f32(reinterpret_cast<const uint16_t *>(W + (size_t)N * K)[(size_t)n * (K / 32) + (p >> 2)]);
    const uint32_t u[2] = {q.x, q.y};
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = d * (float)(int8_t)(u[i >> 2] >> (8 * (i & 3)));
  } else if constexpr (FMT == RT_LINEAR_Q4K) {
    const uint8_t *blk = W + ((size_t)n * (K / 256) + (p >> 5)) * kQ4KBlockBytes;
    const int c = (p >> 3) & 3, h = (p >> 2) & 1;  // chunk, its low or high nibbles
    const uint4 hd = *reinterpret_cast<const uint4 *>(blk);
    const uint2 q = *reinterpret_cast<const uint2 *>(blk + 16 + 32 * c + 8 * (p & 3));
    uint32_t sv, mv;
    q4k_scale_min(hd.y, hd.z, hd.w, 2 * c + h, sv, mv);
    const float s = half_bits_to_f32(hd.x & 0xFFFFu) * (float)sv, m = half_bits_to_f32(hd.x >> 16) * (float)mv;
    const uint32_t u[2] = {(q.x >> (4 * h)) & 0x0F0F0F0Fu, (q.y >> (4 * h)) & 0x0F0F0F0Fu};
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = s * (float)((u[i >> 2] >> (8 * (i & 3))) & 0xFu) - m;
  } else {  // RT_LINEAR_Q6K, planar: piece p is l = 8 (p & 3) .. of quarter m of half j (see q6k_value)
    const Q6KPlanes P = q6k_planes(W, (size_t)N * (K / 256));
    const size_t blk = (size_t)n * (K / 256) + (p >> 5);
    const int j = (p >> 4) & 1, m = (p >> 2) & 3, l = 8 * (p & 3);
    const uint2 ql = *reinterpret_cast<const uint2 *>(P.ql + blk * 128 + 64 * j + 32 * (m & 1) + l);
    const uint2 qh = *reinterpret_cast<const uint2 *>(P.qh + blk * 64 + 32 * j + l);
    const float s = half_bits_to_f32(P.d[blk]) * (float)(int8_t)P.sc[blk * 16 + 8 * j + (l >> 4) + 2 * m];
    const uint32_t lo[2] = {(ql.x >> (m < 2 ? 0 : 4)) & 0x0F0F0F0Fu, (ql.y >> (m < 2 ? 0 : 4)) & 0x0F0F0F0Fu};
    const uint32_t hi[2] = {(qh.x >> (2 * m)) & 0x03030303u, (qh.y >> (2 * m)) & 0x03030303u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t c = ((lo[i >> 2] | (hi[i >> 2] << 4)) >> (8 * (i & 3))) & 0x3Fu;
      v[i] = s * (float)((int)c - 32);
    }
  }
}

// One row per wave: its bound and exponent, then its f16 pieces; the first
// 64 * 8 * kKeep values stay in registers between the two, the rest is read
// again.
template <int FMT>
RT_DEV void row_to_f16(const uint8_t *__restrict__ W, int N, int K, int n, _Float16 *__restrict__ w16,
                       int *__restrict__ ew) {
  constexpr int kKeep = 6;
  const int lane = (int)(threadIdx.x & 63), np = K / 8;
  float v[kKeep][8], amax = 0.f;
#pragma unroll
  for (int i = 0; i < kKeep; ++i) {
    if (64 * i >= np) break;  // wave-uniform
    proj_load8<FMT>(W, N, K, n, min(lane + 64 * i, np - 1), v[i]);
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(v[i][k]));
  }
  for (int p = lane + 64 * kKeep; p < np; p += 64) {
    float t[8];
    proj_load8<FMT>(W, N, K, n, p, t);
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(t[k]));
  }
  const int ex = f16_exponent_for(wave_max(amax));
  if (lane == 0) ew[n] = ex;
  auto store = [&](int p, const float (&x)[8]) {
    const uint2 lo = f16x4_scaled(make_float4(x[0], x[1], x[2], x[3]), ex);
    const uint2 hi = f16x4_scaled(make_float4(x[4], x[5], x[6], x[7]), ex);
    reinterpret_cast<uint4 *>(w16)[(size_t)n * np + p] = make_uint4(lo.x, lo.y, hi.x, hi.y);
  };
#pragma unroll
  for (int i = 0; i < kKeep; ++i)
    if (lane + 64 * i < np) store(lane + 64 * i, v[i]);
  for (int p = lane + 64 * kKeep; p < np; p += 64) {
    float t[8];
    proj_load8<FMT>(W, N, K, n, p, t);
    store(p, t);
  }
}

// Rows [0, M) are A's (AFMT: f32 or bf16), the rest W's.  Bound by memory: 16-byte pieces,
// four rows per workgroup.  Element by element with one row per workgroup and
// a second read of every value the same widening took (W alone) 14.3 us for
// BF16 3072x3072 and 15.3 us for Q8_0 6912x1152.
template <int FMT, int AFMT>
__global__ __launch_bounds__(256) void k_rows_to_f16(const void *__restrict__ a, int M, _Float16 *__restrict__ a16,
                                                     int *__restrict__ ea, const uint8_t *__restrict__ W, int N, int K,
                                                     _Float16 *__restrict__ w16, int *__restrict__ ew) {
  const int r = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (r < M)
    row_to_f16<AFMT>(static_cast<const uint8_t *>(a), M, K, r, a16, ea);
  else if (r - M < N)
    row_to_f16<FMT>(W, N, K, r - M, w16, ew);
}

// The tile of workgroup `bid`: XCD b % 8 gets a contiguous run of tiles, walked
// in groups of eight tile rows so neighbours share A and W in L2.
RT_DEV void pick_tile(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int ntiles = tiles_m * tiles_n, x = bid & 7, r = ntiles & 7, q = ntiles >> 3;
  const int tile = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + (bid >> 3);
  const int group = tile / (8 * tiles_n), in_group = tile % (8 * tiles_n), gm = min(8, tiles_m - group * 8);
  tm = group * 8 + in_group % gm;
  tn = in_group / gm;
}

// ---------------------------------------------------------------------------
// C[M][N] = 2^(ea[m]+ew[n]) * sum_k a16[m][k] w16[n][k] (+ bias[n]), C tile
// 128 x 128, for outputs of few tiles.  Eight waves, two per SIMD: four own 64
// x 64 of C each and the other four the same, the two groups taking
// half of every K stage (64 wide), so a stage's fragments are read
// once per group (64 KB of LDS reads per stage where 64 x 32 wave tiles read
// 96) and one wave's waits run under the other's MFMAs.  The groups' sums meet
// in LDS at the end.
//   Stages arrive by global_load_lds_dwordx4 two ahead in a ring of three
//   32 KB slots (four and five slots: the same within 2%); one barrier per
//   stage.  A slot row is 128 B (8 segments of 8 halves), logical segment s at
//   s ^ ((row >> 1) & 7), so the 16 lanes served together by a ds_read_b128
//   hit 16 distinct bank groups.
//   1000 x 3072 x 3072 (192 tiles): 33 us (570 TFLOP/s) against 48 us for the
//   256 x 256 tiles split five ways with their sum; 512 x 2560 x 10240 split
//   three ways 41 us.
// ---------------------------------------------------------------------------
constexpr int kT128Slots = 3;

__global__ __launch_bounds__(512) void k_gemm_f16_t128(const _Float16 *__restrict__ a16, const int *__restrict__ ea,
                                                       const _Float16 *__restrict__ w16, const int *__restrict__ ew,
                                                       const float *__restrict__ bias, float *__restrict__ c, int M,
                                                       int N, int K, int tiles_m, int tiles_n, int ksplit) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kT128Slots][2][128 * 128];
  const int tid = (int)threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  int tm, tn;
  pick_tile((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * 128, n0 = tn * 128;
  // Split-K: blockIdx.y = s takes stages [s*nk/ksplit, (s+1)*nk/ksplit) and,
  // with ksplit > 1, writes its scaled partial tile to c + s*M*N.
  const int nk = K / 64, split = (int)blockIdx.y, kb = split * nk / ksplit, n = (split + 1) * nk / ksplit - kb;  // n >= 1
  if (ksplit > 1) c += (size_t)split * M * N;
  const uint8_t *ab = reinterpret_cast<const uint8_t *>(a16 + (size_t)m0 * K) + (size_t)kb * 128;
  const uint8_t *wb = reinterpret_cast<const uint8_t *>(w16 + (size_t)n0 * K) + (size_t)kb * 128;
  uint32_t ao[2], bo[2];  // copy i: rows 8 (2 wave + i) + [0, 8), eight lanes per row
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * (2 * wave + i) + (lane >> 3), seg = 16 * ((lane & 7) ^ ((r >> 1) & 7));
    ao[i] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K * 2u + seg;
    bo[i] = (uint32_t)(min(n0 + r, N - 1) - n0) * (uint32_t)K * 2u + seg;
  }
  auto issue = [&](int j, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((gvoid *)(ab + (size_t)j * 128 + ao[i]),
                                       (lvoid *)(lds[slot][0] + (2 * wave + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((gvoid *)(wb + (size_t)j * 128 + bo[i]),
                                       (lvoid *)(lds[slot][1] + (2 * wave + i) * 1024), 16, 0, 0);
  };
  uint32_t fa[2], fb[2];  // this group's k-steps 2 kg + t: segment 2 (2 kg + t) + g of the lane's row
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t seg = 16 * ((2 * (2 * kg + t) + g) ^ ((l32 >> 1) & 7));
    fa[t] = (64 * wm + l32) * 128 + seg;
    fb[t] = (64 * wn + l32) * 128 + seg;
  }
  floatx16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx16{};
#pragma unroll
  for (int i = 0; i < kT128Slots - 1; ++i) issue(min(i, n - 1), i);
  // Past the last stage the copies repeat it, so every stage issues four.
  auto stage = [&](int j, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<4 * (kT128Slots - 2)>();  // stage j's copies; the next stage's may be in flight
    wg_barrier();                        // everyone's; the slot refilled below is read out
    issue(min(j + kT128Slots - 1, n - 1), slot == 0 ? kT128Slots - 1 : slot - 1);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 af[2][2], bf[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[t][i] = lds_read16(lds[slot][0] + fa[t] + 4096 * i);
        bf[t][i] = lds_read16(lds[slot][1] + fb[t] + 4096 * i);
      }
    auto mfma4 = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[i][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, af[t][i]),
                                                              __builtin_bit_cast(half8, bf[t][q]), acc[i][q], 0, 0, 0);
    };
    asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(af[0][0]), "+v"(af[0][1]), "+v"(bf[0][0]), "+v"(bf[0][1]));
    mfma4(0);
    lds_wait(af[1][0], af[1][1], bf[1][0], bf[1][1]);
    mfma4(1);
  };
  static_assert(kT128Slots == 3, "the loop below is unrolled by the ring");
  int j = 0;
  for (; j + 3 <= n; j += 3) {
    stage(j, 0);
    stage(j + 1, 1);
    stage(j + 2, 2);
  }
  if (j < n) stage(j, 0);
  if (j + 1 < n) stage(j + 1, 1);
  wait_vmcnt<0>();
  wg_barrier();
  // group 1's sums to LDS, group 0 adds its own and scales, both store
  constexpr int P = 72;
  static_assert(4 * 64 * P * 4 <= kT128Slots * 2 * 128 * 128, "the staged tile fits in the ring");
  float *st = reinterpret_cast<float *>(&lds[0][0][0]) + (wave & 3) * 64 * P;
  if (kg) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[(32 * i + 8 * (r >> 2) + 4 * g + (r & 3)) * P + 32 * q + l32] = acc[i][q][r];
  }
  __syncthreads();
  if (!kg) {
    int ec[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) ec[q] = ew[min(n0 + 64 * wn + 32 * q + l32, N - 1)];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int R = 32 * i + 8 * (r >> 2) + 4 * g + (r & 3), er = ea[min(m0 + 64 * wm + R, M - 1)];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float *p = st + R * P + 32 * q + l32;
          *p = __builtin_amdgcn_ldexpf(acc[i][q][r] + *p, er + ec[q]);
        }
      }
  }
  __syncthreads();
  const bool vec = (N & 3) == 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int R = 32 * kg + 4 * q + (lane >> 4), f = lane & 15, row = m0 + 64 * wm + R, col = n0 + 64 * wn + 4 * f;
    float4 v = *reinterpret_cast<const float4 *>(st + R * P + 4 * f);
    if (bias) v = add_bias4(v, bias, col, N);
    if (row >= M) continue;
    float *dst = c + (size_t)row * N + col;
    if (vec) {
      if (col < N) *reinterpret_cast<float4 *>(dst) = v;
    } else {
      const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (col + k < N) dst[k] = x[k];
    }
  }
}

// ---------------------------------------------------------------------------
// The same product on 256 x 256 tiles, one workgroup per CU: eight waves of
// 128 x 64, two per SIMD.  The two groups of four waves run half a stage apart
// between workgroup barriers: while one multiplies (16 MFMAs), the other reads
// its next fragments and issues its copies, so each SIMD's matrix core always
// has one wave's MFMAs.
//   K moves in stages of 32 through four slots of 16 KB per operand, copied
//   three stages ahead.  A slot row is 64 B (4 segments of 8 halves), logical
//   segment s at s ^ ((row >> 2) & 3): the 16 lanes of a ds_read_b128 hit 16
//   distinct bank groups.
//   4608 x 12288 x 3072 333 us (1.04 PFLOP/s; the four-wave form with 64-wide
//   stages and 128 x 128 wave tiles 400), 4096 x 4096 x 2560 82 us, 2000 x 12000
//   x 3072 159 us.  With zero operands 250 us: the clock is 1.77 GHz under real
//   ones; and the matrix cores are busy 53% of the cycles, where a library f16
//   product keeps them 66% busy (265 us).  Storing C takes 45 us of the 333.
// ---------------------------------------------------------------------------
constexpr int kT256Slot = 256 * 64;  // one operand, one stage

__global__ __launch_bounds__(512, 2) void k_gemm_f16_t256(const _Float16 *__restrict__ a16, const int *__restrict__ ea,
                                                          const _Float16 *__restrict__ w16, const int *__restrict__ ew,
                                                          const float *__restrict__ bias, float *__restrict__ c, int M,
                                                          int N, int K, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(1024))) uint8_t sa[4][kT256Slot], sb[4][kT256Slot];
  const int tid = (int)threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, wn = wave & 3;
  int tm, tn;
  pick_tile((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * 256, n0 = tn * 256, n = K / 32;
  const uint8_t *ab = reinterpret_cast<const uint8_t *>(a16 + (size_t)m0 * K);
  const uint8_t *wb = reinterpret_cast<const uint8_t *>(w16 + (size_t)n0 * K);
  uint32_t ao[2], bo[2];  // copy i: rows 16 (2 wave + i) + [0, 16), four lanes per row
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * (2 * wave + i) + (lane >> 2), seg = 16 * ((lane & 3) ^ ((r >> 2) & 3));
    ao[i] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K * 2u + seg;
    bo[i] = (uint32_t)(min(n0 + r, N - 1) - n0) * (uint32_t)K * 2u + seg;
  }
  auto issue = [&](int j, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((gvoid *)(ab + (size_t)j * 64 + ao[i]), (lvoid *)(sa[slot] + (2 * wave + i) * 1024),
                                       16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((gvoid *)(wb + (size_t)j * 64 + bo[i]), (lvoid *)(sb[slot] + (2 * wave + i) * 1024),
                                       16, 0, 0);
  };
  uint32_t fa[2], fb[2];  // k-step t: segment 2t + g; 32 rows further is 2048 bytes (whole swizzle periods)
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t seg = 16 * ((2 * t + g) ^ ((l32 >> 2) & 3));
    fa[t] = (128 * wm + l32) * 64 + seg;
    fb[t] = (64 * wn + l32) * 64 + seg;
  }
  floatx16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx16{};
  // Past the last stage the copies repeat it, so every stage issues four.
  issue(0, 0);
  issue(min(1, n - 1), 1);
  issue(min(2, n - 1), 2);
  wait_vmcnt<8>();
  wg_barrier();
  if (wm) wg_barrier();  // group 1 runs half a stage behind
  auto stage = [&](int j, int slot) __attribute__((always_inline)) {
    u32x4 af[2][4], bf[2][2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 2; ++i) bf[t][i] = lds_read16(sb[slot] + fb[t] + 2048 * i);
#pragma unroll
      for (int i = 0; i < 4; ++i) af[t][i] = lds_read16(sa[slot] + fa[t] + 2048 * i);
    }
    // the slot of stage j-1: both groups have read it (group 1 in the half
    // stage that the last barrier closed)
    issue(min(j + 3, n - 1), (slot + 3) & 3);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<8>();  // this wave's part of stage j+1, published by the barrier
    lds_wait(af[0][0], af[0][1], af[0][2], af[0][3]);
    lds_wait(af[1][0], af[1][1], af[1][2], af[1][3]);
    lds_wait(bf[0][0], bf[0][1], bf[1][0], bf[1][1]);
    wg_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[i][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, af[t][i]),
                                                              __builtin_bit_cast(half8, bf[t][q]), acc[i][q], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    wg_barrier();
  };
  int j = 0;
  for (; j + 4 <= n; j += 4) {
    stage(j, 0);
    stage(j + 1, 1);
    stage(j + 2, 2);
    stage(j + 3, 3);
  }
  if (j < n) stage(j, 0);
  if (j + 1 < n) stage(j + 1, 1);
  if (j + 2 < n) stage(j + 2, 2);
  if (!wm) wg_barrier();  // as many barriers as group 1
  wait_vmcnt<0>();
  wg_barrier();
  int ec[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) ec[q] = ew[min(n0 + 64 * wn + 32 * q + l32, N - 1)];
  static_assert(32 * 72 * 4 <= kT256Slot, "a staging slice fits in a slot");
  store_c_tile<2>(acc, reinterpret_cast<float *>(wave < 4 ? sa[wave] : sb[wave - 4]), c, M, N, m0 + 128 * wm,
                  n0 + 64 * wn, ea, ec, bias);
}

// ---------------------------------------------------------------------------
// f32 and bf16 weights with a few activation rows (QLinear's f32 branch,
// x.matmul_bt(W), qlinear.rs:102-106, and MatBf16::matmul_by_t,
// autograd2.rs:757-852), M <= 8 per launch row group (blockIdx.y): four weight
// rows per group of kw = 2^lkw waves, streamed once for the MR activation rows, 16-byte
// loads along K (bf16 widened exactly); per output a lane-strided f32 sum, the
// wave's DPP sum, then the kw waves' sums through LDS.  With a bias, out = sum +
// bias[n], the one f32 add of add_bias_rows (qlinear.rs:49-60).
// Bound by the latency of a wave's loads where the rows alone give few waves.
// ---------------------------------------------------------------------------
constexpr int kGemvRowsMaxLkw = 4, kGemvRowsMaxKw = 1 << kGemvRowsMaxLkw;
template <bool BF16, int MR>
__global__ __launch_bounds__(64 * kGemvRowsMaxKw) void k_gemv_rows(const void *__restrict__ W,
                                                                   const float *__restrict__ a,
                                                                   const float *__restrict__ bias,
                                                                   float *__restrict__ c, int M, int N, int K, int lkw,
                                                                   int lgroups) {
  constexpr int RW = 4, V = BF16 ? 8 : 4;  // weights per 16-byte load
  __shared__ float part[kGemvRowsMaxKw][RW * MR];
  const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kw = 1 << lkw, kp = wave & (kw - 1), n0 = (((int)blockIdx.x << lgroups) + (wave >> lkw)) * RW;
  const int m0 = (int)blockIdx.y * 8;
  const int KV = K / V;
  const uint4 *w = static_cast<const uint4 *>(W);
  const float4 *a4 = reinterpret_cast<const float4 *>(a) + (size_t)m0 * (K / 4);
  float acc[RW][MR];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int i = 0; i < MR; ++i) acc[r][i] = 0.f;
#pragma unroll (MR <= 2 ? 4 : 2)
  for (int k = lane + 64 * kp; k < KV; k += 64 * kw) {
    float wf[RW][V];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const uint4 q = w[(size_t)min(n0 + r, N - 1) * KV + k];  // rows past N re-read row N-1, unstored
      const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (BF16)
          wf[r][2 * j] = bf16_lo(u[j]), wf[r][2 * j + 1] = bf16_hi(u[j]);
        else
          wf[r][j] = __uint_as_float(u[j]);
      }
    }
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      const float4 *xr = a4 + (size_t)min(i, M - 1 - m0) * (K / 4) + (V / 4) * k;  // rows past M re-read row M-1
#pragma unroll
      for (int h = 0; h < V / 4; ++h) {
        const float4 x = xr[h];
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          acc[r][i] = fmaf(wf[r][4 * h], x.x, acc[r][i]);
          acc[r][i] = fmaf(wf[r][4 * h + 1], x.y, acc[r][i]);
          acc[r][i] = fmaf(wf[r][4 * h + 2], x.z, acc[r][i]);
          acc[r][i] = fmaf(wf[r][4 * h + 3], x.w, acc[r][i]);
        }
      }
    }
  }
  float v = 0.f;  // lane r MR + i keeps output (r, i)
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      const float t = wave_sum(acc[r][i]);
      if (lane == r * MR + i) v = t;
    }
  if (lkw) {
    if (lane < RW * MR) part[wave][lane] = v;
    __syncthreads();
    if (kp == 0 && lane < RW * MR)
      for (int p = 1; p < kw; ++p) v += part[wave + p][lane];
  }
  if (kp != 0 || lane >= RW * MR) return;
  const int n = n0 + lane / MR, m = m0 + lane % MR;
  if (n < N && m < M) c[(size_t)m * N + n] = bias ? v + bias[n] : v;
}

// add_bias_rows (qlinear.rs:49-60): c[r][j] += bias[j].
__global__ __launch_bounds__(256) void k_add_bias_rows(float *__restrict__ c, const float *__restrict__ bias,
                                                       size_t total, int N) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256)
    c[i] += bias[i % (size_t)N];
}

}  // namespace

template <bool BF16>
static hipError_t gemv_rows(const void *w, const float *a, const float *bias, float *c, int M, int N, int K,
                            hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || K % (BF16 ? 8 : 4) != 0) return hipErrorInvalidValue;
  const int mgroups = (M + 7) / 8, rows = (N + 3) / 4, chunks = (K / (BF16 ? 8 : 4) + 63) / 64;
  // Waves per row group: as many as keep the launch within 8192 waves (4096 of
  // the widest form).  bf16 2560 x 10240 of 5 rows: 1024 waves 44 us, 2048 26,
  // 4096 18.6, 8192 16.4, 16384 24; of 8 rows 45, 27, 21.0, 24.3, 31; f32 of 8
  // rows 78, 44, 29, 24.5, 28.
  const int target = BF16 && M > 6 ? 4096 : 8192;
  int lkw = 0;
  while (lkw < kGemvRowsMaxLkw && (2 << lkw) <= chunks && (long)rows * mgroups * (2 << lkw) <= target) ++lkw;
  const int lgroups = std::max(0, 2 - lkw), groups = 1 << lgroups;  // row groups per workgroup
  const dim3 grid((unsigned)((rows + groups - 1) / groups), (unsigned)mgroups), block((unsigned)(64 << lkw << lgroups));
#define RT_ROWS(MR) hipLaunchKernelGGL((k_gemv_rows<BF16, MR>), grid, block, 0, s, w, a, bias, c, M, N, K, lkw, lgroups)
  switch (std::min(M, 8)) {  // rows of the last group are bounded by M inside
    case 1: RT_ROWS(1); break;
    case 2: RT_ROWS(2); break;
    case 3: RT_ROWS(3); break;
    case 4: RT_ROWS(4); break;
    case 5:
    case 6: RT_ROWS(6); break;
    default: RT_ROWS(8); break;
  }
#undef RT_ROWS
  return hipGetLastError();
}

hipError_t launch_f32_gemv_rows(const float *w, const float *a, const float *bias, float *c, int M, int N, int K,
                                hipStream_t s) {
  return gemv_rows<false>(w, a, bias, c, M, N, K, s);
}

hipError_t launch_bf16_gemv_rows(const uint16_t *w, const float *a, const float *bias, float *c, int M, int N, int K,
                                 hipStream_t s) {
  return gemv_rows<true>(w, a, bias, c, M, N, K, s);
}

hipError_t launch_add_bias_rows(float *c, const float *bias, int M, int N, hipStream_t s) {
  const size_t total = (size_t)M * N;
  const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256, 4096);
  hipLaunchKernelGGL(k_add_bias_rows, dim3(grid), dim3(256), 0, s, c, bias, total, N);
  return hipGetLastError();
}

// Kernel and K split of an M x N x K product, by a time model fitted to
// measurements (us): 256 x 256 tiles, one per CU and round, 0.0267 per unit of K;
// 128 x 128 tiles 0.0100 per unit of K and round, plus 4 per launch; a split
// adds the sum kernel and (2 ks + 1) M N words at 5 TB/s.  1000x3072x3072: 192
// small tiles in one round 33 against 65; 2000x12000x3072: 376 large tiles 159
// against 196; 512x2560x10240: 80 small tiles split three ways 41, whole 79.
// The plan is the same for every M of a 128-row step.
struct ProjPlan {
  bool big;
  int ks;
  double est_us;
};
static ProjPlan proj_plan(int M, int N, int K) {
  const long tb = (long)((M + 255) / 256) * ((N + 255) / 256), ts = (long)((M + 127) / 128) * ((N + 127) / 128);
  ProjPlan best{true, 1, (double)((tb + 255) / 256) * K * 0.0267};
  for (int ks = 1; ks <= 4 && (ks == 1 || K / 64 / ks >= 8); ++ks) {
    const double part = ks > 1 ? 4.0 + (2.0 * ks + 1.0) * ((M + 127) / 128 * 128.0) * N * 4.0 / 5e6 : 0.0;
    const double x = 4.0 + (double)((ts * ks + 255) / 256) * K / ks * 0.0100 + part;
    if (x < best.est_us) best = {false, ks, x};
  }
  return best;
}

double proj_gemm_est_us(int M, int N, int K) { return proj_plan(M, N, K).est_us; }

static size_t proj_r256(size_t b) { return (b + 255) & ~size_t(255); }

size_t proj_gemm_prepped_ws_bytes(int M, int N, int K) {
  const int ks = proj_plan(M, N, K).ks;
  return proj_r256((size_t)N * K * 2) + proj_r256((size_t)N * 4) + (ks > 1 ? (size_t)ks * M * N * 4 : 0);
}

size_t proj_gemm_workspace_bytes(int M, int N, int K) {
  return proj_r256((size_t)M * K * 2) + proj_r256((size_t)M * 4) + proj_gemm_prepped_ws_bytes(M, N, K);
}

// Widens W (and the am rows of a, if any) into ws, then multiplies.
static hipError_t proj_gemm(const void *a, bool a_bf16, int am, _Float16 *a16, int *ea, int fmt, const void *w, const float *bias,
                            float *c, int M, int N, int K, void *ws, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0) return hipErrorInvalidValue;  // K moves in stages of 64
  char *p = static_cast<char *>(ws);
  _Float16 *w16 = reinterpret_cast<_Float16 *>(p);
  p += proj_r256((size_t)N * K * 2);
  int *ew = reinterpret_cast<int *>(p);
  p += proj_r256((size_t)N * 4);
  const uint8_t *wb = static_cast<const uint8_t *>(w);
  const dim3 grid((unsigned)((am + N + 3) / 4)), block(256);
#define RT_WIDEN(F, A) hipLaunchKernelGGL((k_rows_to_f16<F, A>), grid, block, 0, s, a, am, a16, ea, wb, N, K, w16, ew)
  switch (fmt) {
    case RT_LINEAR_Q4K:
      if (a_bf16) RT_WIDEN(RT_LINEAR_Q4K, RT_LINEAR_BF16);
      else RT_WIDEN(RT_LINEAR_Q4K, RT_LINEAR_F32);
      break;
    case RT_LINEAR_Q6K: RT_WIDEN(RT_LINEAR_Q6K, RT_LINEAR_F32); break;
    case RT_LINEAR_Q8_0: RT_WIDEN(RT_LINEAR_Q8_0, RT_LINEAR_F32); break;
    case RT_LINEAR_BF16: RT_WIDEN(RT_LINEAR_BF16, RT_LINEAR_F32); break;
    case RT_LINEAR_F32: RT_WIDEN(RT_LINEAR_F32, RT_LINEAR_F32); break;
    default: return hipErrorInvalidValue;
  }
#undef RT_WIDEN
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const ProjPlan plan = proj_plan(M, N, K);
  float *out = plan.ks > 1 ? reinterpret_cast<float *>(p) : c;
  const float *b = plan.ks > 1 ? nullptr : bias;
  if (plan.big) {
    const int tm = (M + 255) / 256, tn = (N + 255) / 256;
    hipLaunchKernelGGL(k_gemm_f16_t256, dim3(tm * tn), dim3(512), 0, s, a16, ea, w16, ew, b, out, M, N, K, tm, tn);
  } else {
    const int tm = (M + 127) / 128, tn = (N + 127) / 128;
    hipLaunchKernelGGL(k_gemm_f16_t128, dim3(tm * tn, plan.ks), dim3(512), 0, s, a16, ea, w16, ew, b, out, M, N, K, tm,
                       tn, plan.ks);
  }
  e = hipGetLastError();
  if (e != hipSuccess || plan.ks == 1) return e;
  e = launch_gemm_splitk_sum(out, c, (size_t)M * N, plan.ks, s);
  return e == hipSuccess && bias ? launch_add_bias_rows(c, bias, M, N, s) : e;
}

hipError_t launch_proj_gemm_prepped(const _Float16 *a16, const int *ea, int fmt, const void *w, float *c, int M,
                                    int N, int K, void *ws, hipStream_t s) {
  return proj_gemm(nullptr, false, 0, const_cast<_Float16 *>(a16), const_cast<int *>(ea), fmt, w, nullptr, c, M, N, K, ws, s);
}

hipError_t launch_proj_gemm(const void *a, bool a_bf16, int fmt, const void *w, const float *bias, float *c, int M, int N, int K,
                            void *ws, hipStream_t s) {
  char *p = static_cast<char *>(ws);
  _Float16 *a16 = reinterpret_cast<_Float16 *>(p);
  int *ea = reinterpret_cast<int *>(p + proj_r256((size_t)M * K * 2));
  return proj_gemm(a, a_bf16, M, a16, ea, fmt, w, bias, c, M, N, K, p + proj_r256((size_t)M * K * 2) + proj_r256((size_t)M * 4), s);
}

}  // namespace rt
