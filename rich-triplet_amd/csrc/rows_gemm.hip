// rows_gemm.hip -- C[m][n] = sum_k A[m][k] W[n][k] (+ bias[n]) of a few rows
// (a chat turn, the tail of a prompt) on packed Q4_K, Q6_K and Q8_0 weights,
// on the f16 matrix cores.
//
// With few rows the weights' bytes bound the product, so a workgroup takes 32
// columns of W and splits K over its waves: every wave streams its own part
// of the packed rows, dequantises each fragment once in registers and
// multiplies it with every 32-row tile of A (v_mfma_f32_32x32x16_f16).  The
// waves' products meet in LDS, in wave order.  Columns that are too few to
// fill the chip split K over workgroups as well (blockIdx.y; the partial
// products are summed in split order).
//
// Arithmetic as in the tiled GEMMs (q4k_gemm.hip): both operands are f16 with
// a power-of-two scale, f32 accumulation, the scales restored at the end.  A's
// scale is per row (k_rows_prep); W's is per column and wave, from the block
// headers of the wave's own K range, so no pass over the weights precedes the
// kernel.
//
// A lies in HBM in the order the lanes read it: [64-wide chunk][32-row tile]
// [k-step t][lane][8 halves], lane (g, r) = row r of the tile, halves
// k = 16g + 8(t&1) + 32(t>>1) + [0, 8) of the chunk (the order in which a lane
// holding 16 Q4_K bytes meets its weights), so each fragment is one
// contiguous 1 KB load and needs no LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/rt_hip.h"
#include "kquant_layout.hpp"
#include "mfma_common.hpp"
#include "rt_device.hpp"
#include "rt_kernels.hpp"

namespace rt {
namespace {

RT_DEV void rows_load8(const float *p, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
RT_DEV void rows_load8(const uint16_t *p, float (&v)[8]) {
  const uint4 u = *reinterpret_cast<const uint4 *>(p);
  v[0] = bf16_lo(u.x), v[1] = bf16_hi(u.x), v[2] = bf16_lo(u.y), v[3] = bf16_hi(u.y);
  v[4] = bf16_lo(u.z), v[5] = bf16_hi(u.z), v[6] = bf16_lo(u.w), v[7] = bf16_hi(u.w);
}

// One row of A per workgroup: its exponent, then its f16 pieces in the
// fragment order above, the row held in registers between the two (rows
// beyond 8 * kRowsPrepT * 4 values are read again).  Rows past M keep what the
// workspace holds: their products are never stored.
constexpr int kRowsPrepT = 512;
template <typename TA>
__global__ __launch_bounds__(kRowsPrepT) void k_rows_prep(const TA *__restrict__ a, uint8_t *__restrict__ frag,
                                                          int *__restrict__ ea, int K, int tiles) {
  constexpr int KEEP = 4;
  __shared__ float red[kRowsPrepT / 64];
  const int m = (int)blockIdx.x, np = K / 8, tid = (int)threadIdx.x;
  const TA *row = a + (size_t)m * K;
  float v[KEEP][8], amax = 0.f;
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    if (i > 0 && i * kRowsPrepT >= np) break;
    rows_load8(row + 8 * min(tid + i * kRowsPrepT, np - 1), v[i]);
  }
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    if (i > 0 && i * kRowsPrepT >= np) break;
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(v[i][k]));
  }
  for (int s = tid + KEEP * kRowsPrepT; s < np; s += kRowsPrepT) {
    float w[8];
    rows_load8(row + 8 * s, w);
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(w[k]));
  }
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = red[0];
#pragma unroll
  for (int i = 1; i < kRowsPrepT / 64; ++i) amax = fmaxf(amax, red[i]);
  const int e = f16_exponent_for(amax);
  if (tid == 0) ea[m] = e;
  auto store = [&](int s, const float (&x)[8]) {
    const uint2 lo = f16x4_scaled(make_float4(x[0], x[1], x[2], x[3]), e);
    const uint2 hi = f16x4_scaled(make_float4(x[4], x[5], x[6], x[7]), e);
    const int c = s >> 3, q = s & 7, g = (q >> 1) & 1, t = (q & 1) + 2 * (q >> 2);  // chunk; 16 B piece q = k / 8
    *reinterpret_cast<uint4 *>(frag + ((size_t)((c * tiles + (m >> 5)) * 4 + t) * 64 + 32 * g + (m & 31)) * 16) =
        make_uint4(lo.x, lo.y, hi.x, hi.y);
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i)
    if (tid + i * kRowsPrepT < np) store(tid + i * kRowsPrepT, v[i]);
  for (int s = tid + KEEP * kRowsPrepT; s < np; s += kRowsPrepT) {
    float w[8];
    rows_load8(row + 8 * s, w);
    store(s, w);
  }
}

// The same order from rows already in f16 (row-major, prepared with their
// exponents by the kernel that produced them).
__global__ __launch_bounds__(256) void k_rows_pack(const uint4 *__restrict__ a16, uint4 *__restrict__ frag, int M, int K,
                                                   int tiles) {
  const int i = (int)blockIdx.x * 256 + (int)threadIdx.x, np = K / 8;  // piece i % np of row i / np
  if (i >= M * np) return;
  const int m = i / np, s = i - m * np, c = s >> 3, q = s & 7, g = (q >> 1) & 1, t = (q & 1) + 2 * (q >> 2);
  frag[(size_t)((c * tiles + (m >> 5)) * 4 + t) * 64 + 32 * g + (m & 31)] = a16[i];
}

// Eight f16 weights s*(1024 + u) + negc of eight code bytes u (two words), as
// dq_step (q4k_gemm_dev.hpp) forms them, one rounding each.
RT_DEV half8 rows_dq(uint32_t a, uint32_t b, float s, float negc) {
  const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, a, 0x04010400u);
  const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, a, 0x04030402u);
  const uint32_t p2 = __builtin_amdgcn_perm(0x64646464u, b, 0x04010400u);
  const uint32_t p3 = __builtin_amdgcn_perm(0x64646464u, b, 0x04030402u);
  uint32_t r0, r1, r2, r3;
  asm("v_fma_mixlo_f16 %0, %8, %4, %9 op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixhi_f16 %0, %8, %4, %9 op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixlo_f16 %1, %8, %5, %9 op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixhi_f16 %1, %8, %5, %9 op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixlo_f16 %2, %8, %6, %9 op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixhi_f16 %2, %8, %6, %9 op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixlo_f16 %3, %8, %7, %9 op_sel_hi:[0,1,0]\n\t"
      "v_fma_mixhi_f16 %3, %8, %7, %9 op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"
      "s_nop 1"  // a VALU result read by an MFMA: two wait states the compiler cannot see here
      : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
      : "v"(p0), "v"(p1), "v"(p2), "v"(p3), "v"(s), "v"(negc));
  return __builtin_bit_cast(half8, (u32x4){r0, r1, r2, r3});
}

// Weights of one column: load(c) reads the lane's bytes of chunk c, bound()
// the largest |w| its headers allow over chunks [c0, c1) (this lane's half of
// them), frag() the MFMA B operand of k-step t (scaled by 2^-ew).
template <int FMT>
struct RowsW;

template <>
struct RowsW<RT_LINEAR_Q8_0> {
  struct Raw {
    u32x4 q0, q1;
    uint32_t d;
  };
  struct Scale {
    float s[2], c[2];
  };
  const uint8_t *row;
  const uint32_t *dp;  // the f16 scales of a chunk's two blocks
  RT_DEV RowsW(const uint8_t *W, int N, int K, int n)
      : row(W + (size_t)n * K), dp(reinterpret_cast<const uint32_t *>(W + (size_t)N * K) + (size_t)n * (K / 64)) {}
  RT_DEV Raw load(int c, int g) const {
    const uint8_t *b = row + 64 * c + 16 * g;
    return {*reinterpret_cast<const u32x4 *>(b), *reinterpret_cast<const u32x4 *>(b + 32), dp[c]};
  }
  RT_DEV float bound(int c0, int c1, int g) const {
    float m = 0.f;
    for (int c = c0 + g; c < c1; c += 2)
      m = fmaxf(m, fmaxf(fabsf(half_bits_to_f32(dp[c] & 0xFFFFu)), fabsf(half_bits_to_f32(dp[c] >> 16))));
    return 128.f * m;
  }
  RT_DEV Scale scale(const Raw &r, int, int, float unit) const {
    Scale o;
    o.s[0] = half_bits_to_f32(r.d & 0xFFFFu) * unit, o.s[1] = half_bits_to_f32(r.d >> 16) * unit;
    o.c[0] = -1152.f * o.s[0], o.c[1] = -1152.f * o.s[1];  // codes are q + 128
    return o;
  }
  RT_DEV half8 frag(const Raw &r, const Scale &k, int t) const {
    const u32x4 q = t < 2 ? r.q0 : r.q1;
    return rows_dq(q[2 * (t & 1)] ^ 0x80808080u, q[2 * (t & 1) + 1] ^ 0x80808080u, k.s[t >> 1], k.c[t >> 1]);
  }
};

template <>
struct RowsW<RT_LINEAR_Q6K> {
  struct Raw {
    u32x4 l0, l1, h;  // ql of the even and odd quarter, qh
    uint32_t sc, d;
  };
  struct Scale {
    float s[2], c[2];
  };
  Q6KPlanes P;
  size_t blk0;
  RT_DEV RowsW(const uint8_t *W, int N, int K, int n)
      : P(q6k_planes(W, (size_t)N * (K / 256))), blk0((size_t)n * (K / 256)) {}
  // Chunk c of a block is quarters m = 2(c&1), 2(c&1)+1 of half j = (c>>1)&1.
  RT_DEV Raw load(int c, int g) const {
    const size_t b = blk0 + (c >> 2);
    const int j = (c >> 1) & 1;
    const uint8_t *ql = P.ql + b * 128 + 64 * j + 16 * g;
    return {*reinterpret_cast<const u32x4 *>(ql), *reinterpret_cast<const u32x4 *>(ql + 32),
            *reinterpret_cast<const u32x4 *>(P.qh + b * 64 + 32 * j + 16 * g),
            *reinterpret_cast<const uint32_t *>(P.sc + b * 16 + 8 * j + 4 * (c & 1)), P.d[b]};
  }
  RT_DEV float bound(int c0, int c1, int g) const {
    float m = 0.f;
    for (int b = (c0 >> 2) + g; b <= (c1 - 1) >> 2; b += 2) m = fmaxf(m, fabsf(half_bits_to_f32(P.d[blk0 + b])));
    return 4096.f * m;
  }
  RT_DEV Scale scale(const Raw &r, int, int g, float unit) const {
    const float d = half_bits_to_f32(r.d) * unit;
    Scale o;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      o.s[h] = d * (float)(int8_t)((r.sc >> (16 * h + 8 * g)) & 0xFFu);
      o.c[h] = -1056.f * o.s[h];  // codes are q + 32
    }
    return o;
  }
  RT_DEV half8 frag(const Raw &r, const Scale &k, int c, int t) const {
    const int m = 2 * (c & 1) + (t >> 1);  // quarter: nibble m / 2 of ql, bit pair m of qh
    const u32x4 l = t < 2 ? r.l0 : r.l1;
    uint32_t u[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      u[i] = ((l[2 * (t & 1) + i] >> (4 * (m >> 1))) & 0x0F0F0F0Fu) | (((r.h[2 * (t & 1) + i] >> (2 * m)) & 0x03030303u) << 4);
    return rows_dq(u[0], u[1], k.s[t >> 1], k.c[t >> 1]);
  }
};
template <int FMT>
RT_DEV half8 rows_frag(const RowsW<FMT> &w, const typename RowsW<FMT>::Raw &r, const typename RowsW<FMT>::Scale &k, int c,
                       int t) {
  if constexpr (FMT == RT_LINEAR_Q6K) return w.frag(r, k, c, t);
  else return w.frag(r, k, t);
}

constexpr int kRowsWaves = 8, kRowsT = 64 * kRowsWaves;

// Q6_K and Q8_0: MT 32-row tiles per workgroup, tile group blockIdx.z; each lane
// loads its own pieces of W, RING chunks ahead (four or six ahead measured
// slower: the pieces of a line then fall out of the L1 before they are used).
template <int FMT, int MT>
__global__ __launch_bounds__(kRowsT) void k_rows_gemm(const uint8_t *__restrict__ frag, const int *__restrict__ ea,
                                                      const uint8_t *__restrict__ W, const float *__restrict__ bias,
                                                      float *__restrict__ c, int M, int N, int K, int tiles,
                                                      int ksplit) {
  using Wt = RowsW<FMT>;
  constexpr int RING = 2;
  constexpr int P = 36;  // LDS row pitch in floats (16-byte rows, spread over the banks)
  __shared__ __attribute__((aligned(16))) float part[kRowsWaves][32 * P];
  const int tid = (int)threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (int)blockIdx.x * 32, n = min(n0 + l32, N - 1), mt0 = (int)blockIdx.z * MT;
  const int unit = (int)blockIdx.y * kRowsWaves + wave, units = ksplit * kRowsWaves, nch = K / 64;
  const int c0 = (int)((long)unit * nch / units), c1 = (int)((long)(unit + 1) * nch / units);
  const Wt w(W, N, K, n);
  const int last = max(c1 - 1, c0 < nch ? c0 : nch - 1);
  typename Wt::Raw raw[RING];
#pragma unroll
  for (int i = 0; i < RING; ++i) raw[i] = w.load(min(c0 + i, last), g);
  // tiles past the last one (of a group) re-read it
  const uint8_t *ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = frag + (size_t)min(mt0 + i, tiles - 1) * 4096 + lane * 16;
  const size_t astep = (size_t)tiles * 4096;
  u32x4 a[2][MT][4];
  auto load_a = [&](int ch, u32x4(&dst)[MT][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) dst[i][t] = *reinterpret_cast<const u32x4 *>(ap[i] + ch * astep + 1024 * t);
  };
  load_a(min(c0, last), a[0]);
  float bd = w.bound(c0, c1, g);
  bd = fmaxf(bd, __shfl_xor(bd, 32));
  const int ew = f16_exponent_for(bd);
  const float wunit = __builtin_amdgcn_ldexpf(1.0f, -ew);

  floatx16 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = floatx16{};
  for (int cb = c0; cb < c1; cb += RING) {
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      const int ch = cb + j;
      if (ch < c1) {  // wave-uniform
        load_a(min(ch + 1, last), a[(j + 1) & 1]);
        const typename Wt::Scale sc = w.scale(raw[j], ch, g, wunit);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const half8 bf = rows_frag<FMT>(w, raw[j], sc, ch, t);
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a[j & 1][i][t]), bf, acc[i], 0, 0, 0);
        }
        raw[j] = w.load(min(ch + RING, last), g);
      }
    }
  }
  static_assert(RING % 2 == 0, "the A buffers alternate by chunk");

  // One 32-row tile at a time through LDS: the waves' products scaled by
  // 2^ew, then added in wave order by threads of whole 16-byte row pieces.
  if (ksplit > 1) c += (size_t)blockIdx.y * M * N;
  const int r = tid >> 3, f = tid & 7;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row0 = 32 * (mt0 + i);
    if (row0 >= M) break;  // workgroup-uniform
    if (i > 0) __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q)
      part[wave][(8 * (q >> 2) + 4 * g + (q & 3)) * P + l32] = __builtin_amdgcn_ldexpf(acc[i][q], ew);
    __syncthreads();
    if (tid < 256 && row0 + r < M) {
      float4 s = *reinterpret_cast<const float4 *>(&part[0][r * P + 4 * f]);
#pragma unroll
      for (int v = 1; v < kRowsWaves; ++v) {
        const float4 x = *reinterpret_cast<const float4 *>(&part[v][r * P + 4 * f]);
        s.x += x.x, s.y += x.y, s.z += x.z, s.w += x.w;
      }
      const int e = ea[row0 + r], col = n0 + 4 * f;
      const float o[4] = {__builtin_amdgcn_ldexpf(s.x, e), __builtin_amdgcn_ldexpf(s.y, e),
                          __builtin_amdgcn_ldexpf(s.z, e), __builtin_amdgcn_ldexpf(s.w, e)};
      float *dst = c + (size_t)(row0 + r) * N + col;
      if ((N & 3) == 0 && col + 4 <= N) {
        float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
        if (bias) b = make_float4(bias[col], bias[col + 1], bias[col + 2], bias[col + 3]);
        *reinterpret_cast<float4 *>(dst) = bias ? make_float4(o[0] + b.x, o[1] + b.y, o[2] + b.z, o[3] + b.w)
                                                : make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (col + k < N) dst[k] = bias ? o[k] + bias[col + k] : o[k];
      }
    }
  }
}

RT_DEV void lds_wait1(u32x4 &a) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a)); }
RT_DEV void lds_wait2(u32x4 &a, u32x4 &b) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a), "+v"(b)); }

constexpr int kRowsQ4kWaves = 4;
constexpr int kRowsNoExp = -60;  // below the exponent of any non-zero block (f16 headers)

// The Q4_K form: NT 32-column tiles per wave, whole super-blocks per wave.  A
// wave copies the 32 NT x 144 bytes of a super-block's columns to its own LDS
// ring (two blocks) with global_load_lds: nine lanes read one column's block,
// so a copy touches each cache line once, where direct loads (16 bytes per
// lane, 32-byte pieces of 32 columns) fetch every line four times over a
// block.  Column pitch 144 bytes: 16 consecutive columns of a 16-byte read are
// on distinct banks.
template <int MT, int NT>
__global__ __launch_bounds__(64 * kRowsQ4kWaves) void k_rows_gemm_q4k(const uint8_t *__restrict__ frag, const int *__restrict__ ea,
                                                       const uint8_t *__restrict__ W, const float *__restrict__ bias,
                                                       float *__restrict__ c, int M, int N, int K, int tiles,
                                                       int ksplit) {
  constexpr int waves = kRowsQ4kWaves;
  constexpr int COLS = 32 * NT, SLOT = COLS * kQ4KBlockBytes, COPIES = (COLS * 9 + 63) / 64, P = 32 * NT + 4;
  // the waves' rings, then (read out) their products: 37 KB per column tile
  __shared__ __attribute__((aligned(16))) uint8_t rows_lds[waves * 2 * SLOT];
  static_assert(waves * 32 * P * 4 <= waves * 2 * SLOT, "the products fit in the rings");
  const int tid = (int)threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (int)blockIdx.x * COLS, mt0 = (int)blockIdx.z * MT;
  const int nb = K / 256, units = ksplit * waves, unit = (int)blockIdx.y * waves + wave;
  const int b0 = (int)((long)unit * nb / units), b1 = (int)((long)(unit + 1) * nb / units);
  uint8_t *ring = rows_lds + wave * (2 * SLOT);

  // copy i of a block: pieces 64 i + lane of [column][9]; the last copy of an
  // odd count is half a wave (NT = 1: 288 pieces)
  uint32_t off[COPIES];
#pragma unroll
  for (int i = 0; i < COPIES; ++i) {
    const int p = min(64 * i + lane, COLS * 9 - 1), col = p / 9, seg = p - 9 * col;
    off[i] = (uint32_t)((min(n0 + col, N - 1) - n0) * nb) * kQ4KBlockBytes + 16 * seg;
  }
  const uint8_t *wbase = W + (size_t)n0 * nb * kQ4KBlockBytes;
  auto copy = [&](int b) __attribute__((always_inline)) {
    uint8_t *dst = ring + (b & 1) * SLOT;
    const uint8_t *src = wbase + (size_t)b * kQ4KBlockBytes;
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
      if (64 * (i + 1) <= COLS * 9 || lane < COLS * 9 - 64 * i)
        __builtin_amdgcn_global_load_lds((gvoid *)(src + off[i]), (lvoid *)(dst + 1024 * i), 16, 0, 0);
    }
  };
  const uint8_t *ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = frag + (size_t)min(mt0 + i, tiles - 1) * 4096 + lane * 16;
  const size_t astep = (size_t)tiles * 4096;
  constexpr int AR = MT * NT <= 2 ? 4 : 2;  // chunks of A in registers
  u32x4 a[AR][MT][4];
  auto load_a = [&](int ch, u32x4(&dst)[MT][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) dst[i][t] = *reinterpret_cast<const u32x4 *>(ap[i] + ch * astep + 1024 * t);
  };
  floatx16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = floatx16{};
  int ew[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) ew[j] = kRowsNoExp;
  if (b0 < b1) {  // wave-uniform
    copy(b0);
#pragma unroll
    for (int i = 0; i < AR; ++i) load_a(4 * b0 + i, a[i]);
    if (b0 + 1 < b1) copy(b0 + 1);
    for (int b = b0; b < b1; ++b) {
      const uint8_t *blk = ring + (b & 1) * SLOT + l32 * kQ4KBlockBytes;
      // block b's copies have landed; the next block's may be in flight (and
      // A's, whose registers the compiler waits for)
      if (b + 1 < b1) wait_vmcnt<COPIES>();
      else wait_vmcnt<0>();
      u32x4 hd[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) hd[j] = lds_read16(blk + j * 32 * kQ4KBlockBytes);
      if constexpr (NT == 2) lds_wait2(hd[0], hd[1]);
      else lds_wait1(hd[0]);
      // the column's exponent so far, two bits of headroom; a block that
      // needs a larger one rescales the sums (exact)
      float wunit[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float bd = fmaxf(945.f * fabsf(half_bits_to_f32(hd[j][0] & 0xFFFFu)),
                               63.f * fabsf(half_bits_to_f32(hd[j][0] >> 16)));
        const int e = bd > 0.f ? f16_exponent_for(bd) : kRowsNoExp;
        if (__builtin_amdgcn_ballot_w64(e > ew[j])) {  // wave-uniform
          const int e1 = e > ew[j] ? e + 2 : ew[j], de = max(ew[j] - e1, -126);
          ew[j] = e1;
          const float f = __builtin_amdgcn_ldexpf(1.0f, de);
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] *= f;
        }
        wunit[j] = __builtin_amdgcn_ldexpf(g ? 0.0625f : 1.0f, -ew[j]);
      }
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        u32x4 q[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) q[j] = lds_read16(blk + j * 32 * kQ4KBlockBytes + 16 + 32 * cc + 16 * g);
        if constexpr (AR == 2) {
          if (cc > 0 || b > b0) load_a(min(4 * b + cc + 1, 4 * b1 - 1), a[(cc + 1) & 1]);
        }
        if constexpr (NT == 2) lds_wait2(q[0], q[1]);
        else lds_wait1(q[0]);
        float s_lo[NT], s_hi[NT], c_lo[NT], c_hi[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {  // each lane half decodes one sub-block
          uint32_t sv, mv;
          q4k_scale_min(hd[j][1], hd[j][2], hd[j][3], 2 * cc + g, sv, mv);
          const float sf = half_bits_to_f32(hd[j][0] & 0xFFFFu) * (float)sv * wunit[j];
          const float mn = half_bits_to_f32(hd[j][0] >> 16) * (float)mv * (wunit[j] * (g ? 16.f : 1.f));
          const float nc = -(mn + 1024.f * sf);
          const auto s2 = __builtin_amdgcn_permlane32_swap(f32_bits(sf), f32_bits(sf), false, false);
          const auto n2 = __builtin_amdgcn_permlane32_swap(f32_bits(nc), f32_bits(nc), false, false);
          s_lo[j] = bits_f32(s2[0]), s_hi[j] = bits_f32(s2[1]);
          c_lo[j] = bits_f32(n2[0]), c_hi[j] = bits_f32(n2[1]);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const uint32_t mask = t < 2 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
            const half8 bf = rows_dq(q[j][2 * (t & 1)] & mask, q[j][2 * (t & 1) + 1] & mask, t < 2 ? s_lo[j] : s_hi[j],
                                     t < 2 ? c_lo[j] : c_hi[j]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a[cc % AR][i][t]), bf,
                                                                 acc[i][j], 0, 0, 0);
          }
        }
        if constexpr (AR == 4) load_a(min(4 * (b + 1) + cc, 4 * b1 - 1), a[cc]);
      }
      if (b + 2 < b1) copy(b + 2);  // the slot's last reads have been waited for
    }
    wait_vmcnt<0>();
  }
  if (ksplit > 1) c += (size_t)blockIdx.y * M * N;
  float *part = reinterpret_cast<float *>(rows_lds);
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row0 = 32 * (mt0 + i);
    if (row0 >= M) break;  // workgroup-uniform
    __syncthreads();       // the rings, or the previous tile's sums, are read out
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        part[(wave * 32 + 8 * (q >> 2) + 4 * g + (q & 3)) * P + 32 * j + l32] =
            b0 < b1 ? __builtin_amdgcn_ldexpf(acc[i][j][q], ew[j]) : 0.f;
    __syncthreads();
    for (int p = tid; p < 32 * 8 * NT; p += 64 * waves) {
      const int r = p / (8 * NT), col = n0 + 4 * (p % (8 * NT));
      if (row0 + r >= M) continue;
      const float *src = part + r * P + 4 * (p % (8 * NT));
      float4 s = *reinterpret_cast<const float4 *>(src);
      for (int v = 1; v < waves; ++v) {
        const float4 x = *reinterpret_cast<const float4 *>(src + v * 32 * P);
        s.x += x.x, s.y += x.y, s.z += x.z, s.w += x.w;
      }
      const int e = ea[row0 + r];
      const float o[4] = {__builtin_amdgcn_ldexpf(s.x, e), __builtin_amdgcn_ldexpf(s.y, e),
                          __builtin_amdgcn_ldexpf(s.z, e), __builtin_amdgcn_ldexpf(s.w, e)};
      float *dst = c + (size_t)(row0 + r) * N + col;
      if ((N & 3) == 0 && !bias) {
        if (col < N) *reinterpret_cast<float4 *>(dst) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (col + k < N) dst[k] = bias ? o[k] + bias[col + k] : o[k];
      }
    }
  }
}

// MT x NT tiles of the Q4_K form: 2 x 2 (each A fragment feeds two column
// tiles, each dequantised fragment two row tiles) once there are two row
// tiles and the columns still give 96 workgroups.  Rows 10240x2560 of 40: 2 x 2
// 18.5 us a call, 2 x 1 18.9, 1 x 1 18.5; of 300: 40.8, 45.4, 50.0; 12288x3072 of
// 300: 47.3, 56.9, -; 1024x2560 of 40: 1 x 1 10.1 (2 x 2 leaves 16 workgroups).
struct RowsPlanG {
  int mt, nt, ks, tiles;
};
RowsPlanG rows_plan(int fmt, int M, int N, int K) {
  RowsPlanG p{1, 1, 1, (M + 31) / 32};
  const bool q4k = fmt == RT_LINEAR_Q4K;
  if (q4k) {
    if (p.tiles >= 2 && (N + 63) / 64 * ((p.tiles + 1) / 2) * (K >= 4096 ? 3 : 1) >= 96) p.mt = p.nt = 2;
  } else {
    // Q6_K unpacks more per fragment: four row tiles share one (2560x10240 of
    // 100 rows: 32.8 us against 40.3 with two); Q8_0 the same within 5%
    p.mt = p.tiles == 1 ? 1 : (fmt == RT_LINEAR_Q6K && p.tiles > 2 ? 4 : 2);
  }
  // K over workgroups: about one workgroup per CU (two of the Q4_K form, once
  // the rows alone give 80), at least two super-blocks (four 64-wide chunks)
  // per wave.  2560x10240 of 40 rows: ks 3 to 6 20.2-21.0 us, 1 29; of 200
  // rows (160 workgroups): ks 3 37.8, 1 44.
  const int wgs = (N + 32 * p.nt - 1) / (32 * p.nt) * ((p.tiles + p.mt - 1) / p.mt);
  const int most = q4k ? K / 256 / (2 * kRowsQ4kWaves) : K / 64 / (4 * kRowsWaves);
  int ks = (q4k && wgs >= 80 ? 480 : 240) / wgs;
  // Little more than one workgroup per CU leaves the second round nearly empty:
  // halve it where K is long (9636x11776 of 75 rows, 302 workgroups: 71 -> 68;
  // 4096x14336 of 300 rows, 320: 86 -> 81; from 400 workgroups on it loses)
  if (q4k && K >= 8192 && wgs > 256 && wgs <= 400) ks = 2;
  p.ks = std::max(1, std::min(ks, most));
  return p;
}

size_t r256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

bool rows_gemm_ok(int fmt, int M, int N, int K) {
  if (fmt != RT_LINEAR_Q4K && fmt != RT_LINEAR_Q6K && fmt != RT_LINEAR_Q8_0) return false;
  // Up to 384 rows at any width (this path against the tiled ones, us: Q4_K
  // 10240x2560 300 rows 41 / 45, 512 rows 53 / 55; 2560x10240 384 rows 47 / 51,
  // 450 rows 66 / 57; Q8_0 10000x6016 384 rows 154 / 186).  Longer, where the
  // output has too few tiles to fill the chip: 2560x2560 1000 rows 38 / 41,
  // 1024x2560 1000 rows 25 / 38, 6000x2560 640 rows 48 / 47.
  // Not on a large Q4_K weight whose rows fill 128-row tiles (an even number of
  // 64-row pairs): 9636x11776 of 75 rows 68 / 62, of 200 rows 112 / 100, of
  // 140 rows 80 / 97; 10240x10240 of 200 rows 97 / 90; 12000x8192 of 200 86 / 90.
  if (fmt == RT_LINEAR_Q4K && K > 8192 && N > 4096 && ((M + 63) / 64) % 2 == 0) return false;
  return M <= 384 || (M <= 1024 && K <= 4096 && (long)M * N <= 2600000);
}

size_t rows_gemm_workspace_bytes(int fmt, int M, int N, int K) {
  const RowsPlanG p = rows_plan(fmt, M, N, K);
  return r256((size_t)(K / 64) * p.tiles * 4096) + r256((size_t)M * 4) + (p.ks > 1 ? (size_t)p.ks * M * N * 4 : 0);
}

// The product of packed rows; partial products (ks > 1) go to part.
static hipError_t rows_core(int fmt, const RowsPlanG &p, const uint8_t *frag, const int *ea, const void *w,
                            const float *bias, float *c, float *part, int M, int N, int K, hipStream_t s) {
  const uint8_t *wb = static_cast<const uint8_t *>(w);
  float *out = p.ks > 1 ? part : c;
  const float *b = p.ks > 1 ? nullptr : bias;
  const dim3 grid((unsigned)((N + 32 * p.nt - 1) / (32 * p.nt)), (unsigned)p.ks, (unsigned)((p.tiles + p.mt - 1) / p.mt));
  if (fmt == RT_LINEAR_Q4K) {
    const dim3 t(64 * kRowsQ4kWaves);
    if (p.mt == 2)
      hipLaunchKernelGGL((k_rows_gemm_q4k<2, 2>), grid, t, 0, s, frag, ea, wb, b, out, M, N, K, p.tiles, p.ks);
    else
      hipLaunchKernelGGL((k_rows_gemm_q4k<1, 1>), grid, t, 0, s, frag, ea, wb, b, out, M, N, K, p.tiles, p.ks);
  } else {
#define RT_ROWS(F, T)                                                                                              \
  if (fmt == F && p.mt == T)                                                                                       \
    hipLaunchKernelGGL((k_rows_gemm<F, T>), grid, dim3(kRowsT), 0, s, frag, ea, wb, b, out, M, N, K, p.tiles, p.ks);
    RT_ROWS(RT_LINEAR_Q8_0, 1)
    RT_ROWS(RT_LINEAR_Q8_0, 2)
    RT_ROWS(RT_LINEAR_Q6K, 1)
    RT_ROWS(RT_LINEAR_Q6K, 2)
    RT_ROWS(RT_LINEAR_Q6K, 4)
#undef RT_ROWS
  }
  return hipGetLastError();
}

hipError_t launch_rows_gemm(int fmt, const void *a, bool a_bf16, const void *w, const float *bias, float *c, int M,
                            int N, int K, void *ws, hipStream_t s) {
  const RowsPlanG p = rows_plan(fmt, M, N, K);
  uint8_t *frag = static_cast<uint8_t *>(ws);
  int *ea = reinterpret_cast<int *>(frag + r256((size_t)(K / 64) * p.tiles * 4096));
  float *part = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(ea) + r256((size_t)M * 4));
  if (a_bf16)
    hipLaunchKernelGGL(k_rows_prep<uint16_t>, dim3(M), dim3(kRowsPrepT), 0, s, static_cast<const uint16_t *>(a), frag,
                       ea, K, p.tiles);
  else
    hipLaunchKernelGGL(k_rows_prep<float>, dim3(M), dim3(kRowsPrepT), 0, s, static_cast<const float *>(a), frag, ea, K,
                       p.tiles);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = rows_core(fmt, p, frag, ea, w, bias, c, part, M, N, K, s);
  if (e != hipSuccess || p.ks == 1) return e;
  e = launch_gemm_splitk_sum(part, c, (size_t)M * N, p.ks, s);
  return e == hipSuccess && bias ? launch_add_bias_rows(c, bias, M, N, s) : e;
}

size_t rows_pack_bytes(int M, int K) { return r256((size_t)(K / 64) * ((M + 31) / 32) * 4096); }

size_t rows_part_bytes(int fmt, int M, int N, int K) {
  const int ks = rows_plan(fmt, M, N, K).ks;
  return ks > 1 ? r256((size_t)ks * M * N * 4) : 0;
}

hipError_t launch_rows_pack(const _Float16 *a16, int M, int K, void *frag, hipStream_t s) {
  hipLaunchKernelGGL(k_rows_pack, dim3((unsigned)(((size_t)M * (K / 8) + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<const uint4 *>(a16), static_cast<uint4 *>(frag), M, K, (M + 31) / 32);
  return hipGetLastError();
}

hipError_t launch_rows_gemm_packed(int fmt, const void *frag, const int *ea, const void *w, float *c, int M, int N,
                                   int K, float *part, hipStream_t s, GemmLeft *left) {
  const RowsPlanG p = rows_plan(fmt, M, N, K);
  *left = GemmLeft{p.ks > 1 ? part : c, p.ks};
  return rows_core(fmt, p, static_cast<const uint8_t *>(frag), ea, w, nullptr, c, part, M, N, K, s);
}

}  // namespace rt
