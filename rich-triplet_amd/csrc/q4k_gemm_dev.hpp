// q4k_gemm_dev.hpp -- device pieces shared by the Q4_K GEMM kernels
// (q4k_gemm.hip, q4k_gemm_pp.hip): the K chunk, the dequantisation step
// into an MFMA B operand, and the matrix set of a one-launch projection set.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemma3_math.hpp"
#include "mfma_common.hpp"
#include "rt_device.hpp"

namespace rt {

constexpr int kBK = 64;  // K per pipeline stage = one Q4_K chunk (32 qs bytes, 2 sub-blocks)

// ---------------------------------------------------------------------------
// Matrix-core kernels.  All use v_mfma_f32_32x32x16_f16 (lane l: A row / B
// column l%32, k group g = l/32, 8 halves each) and the same K order inside a
// 64-wide chunk (A and B agree on it, so the sum is unchanged):
//   lane group g holds qs bytes [16g, 16g+16) of the chunk's 32; k-step t
//   (0..3) covers chunk-local k = 16g + 8(t&1) + 32(t>>1) + [0, 8): t < 2 are
//   the low nibbles (sub-block 2c), t >= 2 the high nibbles of the same
//   bytes (sub-block 2c+1).
// A (and in the eight-wave kernel the packed W bytes) reaches LDS by
// global_load_lds_dwordx4 (no VGPRs, no ds_write); each ring slot is its own
// __shared__ variable.  In the eight-wave and half-block kernels every lane
// dequantises the qs bytes of its own column straight into the MFMA B operand,
// so no dequantised weight is written back to LDS; the ping-pong kernel
// (q4k_gemm_pp.hip) writes it there once for all the waves of a workgroup.
// ---------------------------------------------------------------------------
// Eight f16 weights of one k-step from two qs words (low or high nibbles).
// v_perm builds halves 1024+q (low nibbles) or 1024+16q (high nibbles), and
// each v_fma_mix computes f16(s*h - c) from them in f32 with one rounding.
// The eight v_fma_mix sit in one asm block that ends with two wait states:
// the compiler's hazard recognizer cannot tell that an asm block is VALU
// work, so it would not separate it from an MFMA that reads its result
// (a VALU write followed by an MFMA read of that VGPR needs two wait states).
template <bool HIGH>
RT_DEV half8 dq_step(uint32_t w0, uint32_t w1, float s, float negc) {
  const uint32_t mask = HIGH ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
  const uint32_t a = w0 & mask, b = w1 & mask;
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
      "s_nop 1"
      : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
      : "v"(p0), "v"(p1), "v"(p2), "v"(p3), "v"(s), "v"(negc));
  const u32x4 r = {r0, r1, r2, r3};
  return __builtin_bit_cast(half8, r);
}

// Up to three matrices sharing A (q|k|v, gate|up) in one launch: their
// 256-column tiles are numbered one after another (tn0), and a workgroup
// takes the matrix its column tile falls in.
struct HMats {
  const uint8_t *w[3];
  const int *ew[3];
  float *c[3];
  int n[3];
  int tn0[3];  // first column tile of each matrix
  int count;
};

// GELU mode's output: h16 [M][N] f16 and its row exponents eh [M]; a_nrm2 and
// gu_bound as store_gelu_tile uses them.
struct GeluOut {
  _Float16 *h16;
  int *eh;
  const float *a_nrm2;
  float gu_bound;
};

// QKV mode: the per-head RMSNorm (gamma g_q for matrix 0, g_k for matrix 1)
// and NeoX RoPE of row m with cos | sin at cs + m*cs_stride (+ head_dim),
// applied before the store; matrix 2 (v) is stored as computed.
struct QkRope {
  const float *cs;
  int cs_stride;
  const float *g_q, *g_k;
  float eps;
};

enum HMode { kHPlain = 0, kHGelu = 1, kHQkv = 2 };

// The GELU epilogue: each staged value is gelu_tanh(g) * u of the wave's gate
// (acc[i][0]) and up (acc[i][1]) accumulators, each scaled by
// 2^(ea[row] + ew of its matrix) as store_c_tile scales them, and h goes out
// as the next GEMM's A operand: f16 scaled by 2^-eh[row] with eh[row] =
// f16_exponent_for(2 * a_nrm2[row] * gu_bound).  By Cauchy-Schwarz
// |g| <= |a| |w_gate|, |u| <= |a| |w_up| and |gelu_tanh(g)| <= |g|, so
// |h| <= |a|^2 max_n |w_gate,n| |w_up,n|: a_nrm2 = |a|^2 of the row of A (f32,
// before its f16 rounding) and gu_bound that maximum; the factor 2 covers
// the f16 operands and the f32 sums.  No value overflows, and f16 rounding is
// relative, so h rounds as with the exponent of its exact row maximum except
// for elements below 2^-14 of the scale.
RT_DEV void store_gelu_tile(const floatx16 (&acc)[4][2], float *stage, _Float16 *h16, int *eh, int M, int N,
                            int row0, int col0, const int *ea, const int (&ecol)[2], const float *a_nrm2,
                            float gu_bound) {
  constexpr int P = 40, F4 = 8, RPI = 8;
  const int lane = (int)(threadIdx.x & 63), g = lane >> 5, l32 = lane & 31;
  const bool vec = (N & 3) == 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int er[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) er[r] = ea[min(row0 + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3), M - 1)];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float gv = __builtin_amdgcn_ldexpf(acc[i][0][r], er[r] + ecol[0]);
      const float uv = __builtin_amdgcn_ldexpf(acc[i][1][r], er[r] + ecol[1]);
      stage[(8 * (r >> 2) + 4 * g + (r & 3)) * P + l32] = mul_nc(gelu_tanh(gv), uv);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int q = 0; q < 32 / RPI; ++q) {
      const int rl = q * RPI + lane / F4, f = lane % F4;
      const int row = row0 + 32 * i + rl, col = col0 + 4 * f;
      const float4 v = *reinterpret_cast<const float4 *>(stage + rl * P + 4 * f);
      if (row < M) {
        const int e = f16_exponent_for(2.0f * a_nrm2[row] * gu_bound);
        if (col == 0) eh[row] = e;
        _Float16 *dst = h16 + (size_t)row * N + col;
        if (vec && col + 4 <= N) {
          *reinterpret_cast<uint2 *>(dst) = f16x4_scaled(v, e);
        } else {
          const float x[4] = {v.x, v.y, v.z, v.w};
          for (int k = 0; k < 4; ++k)
            if (col + k < N) dst[k] = (_Float16)__builtin_amdgcn_ldexpf(x[k], -e);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// The QKV epilogue: the tile is one head (256 columns from n0) of 128 rows from
// row0 on four waves; lane (g, l32) of wave w holds columns c = 32w + l32 (j = 0)
// and c + 128 (j = 1), the RoPE pair.  One 32-row MFMA tile (i) at a time, so
// its accumulators are free once it is stored.  `stage` is this wave's, `wsum`
// the four waves'; a barrier per 32 rows, which the whole workgroup runs.
RT_DEV void store_qkv_tile(const floatx16 (&acc)[4][2], float *stage, float (*wsum)[128], int w, float *c, int M, int N,
                           int row0, int n0, int mi, const int *ea, const int (&ecol)[2], const QkRope &qr) {
  const int lane = (int)(threadIdx.x & 63), g = lane >> 5, l32 = lane & 31;
  const int colp[2] = {n0 + 32 * w, n0 + 128 + 32 * w};
  const int cl = 32 * w + l32;  // the pair's column within the head
  const float *gam = mi == 0 ? qr.g_q : qr.g_k;
  const float g0 = mi < 2 ? 1.0f + gam[cl] : 0.f, g1 = mi < 2 ? 1.0f + gam[cl + 128] : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    floatx16 v0, v1;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int er = ea[min(row0 + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3), M - 1)];
      v0[r] = __builtin_amdgcn_ldexpf(acc[i][0][r], er + ecol[0]);
      v1[r] = __builtin_amdgcn_ldexpf(acc[i][1][r], er + ecol[1]);
    }
    if (mi < 2) {  // workgroup-uniform
      // sums of squares of the 32 rows: this wave's 64 columns through its
      // LDS slot ([row][l32], 16-byte groups swizzled by the row), two
      // lanes per row, then the four waves' sums through wsum
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int R = 8 * (r >> 2) + 4 * g + (r & 3);
        stage[R * 32 + ((((l32 >> 2) ^ R) & 7) << 2) + (l32 & 3)] = v0[r] * v0[r] + v1[r] * v1[r];
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      {
        const int R = lane >> 1;
        float t = 0.f;
#pragma unroll
        for (int m4 = 4 * (lane & 1); m4 < 4 * (lane & 1) + 4; ++m4) {
          const float4 x = *reinterpret_cast<const float4 *>(stage + R * 32 + (((m4 ^ R) & 7) << 2));
          t += (x.x + x.y) + (x.z + x.w);
        }
        t += __shfl_xor(t, 1);
        if ((lane & 1) == 0) wsum[w][32 * i + R] = t;
      }
      wg_barrier();
#pragma unroll
      for (int r = 0; r < 16; ++r) {
#pragma clang fp contract(off)
        const int R = 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
        const float ss = (wsum[0][R] + wsum[1][R]) + (wsum[2][R] + wsum[3][R]);
        const float rinv = rms_inv_from_sumsq(ss, 1.0f / 256.0f, qr.eps);
        const int co = min(row0 + R, M - 1) * qr.cs_stride + cl;  // 32-bit offset from the uniform base
        const float cv = qr.cs[co], sv = qr.cs[co + 128];
        const float a0 = (v0[r] * rinv) * g0, a1 = (v1[r] * rinv) * g1;
        v0[r] = a0 * cv - a1 * sv;
        v1[r] = a0 * sv + a1 * cv;
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // stage and store the tile's 32 rows x (32 + 32) columns
    constexpr int P = 72;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      stage[(8 * (r >> 2) + 4 * g + (r & 3)) * P + l32] = v0[r];
      stage[(8 * (r >> 2) + 4 * g + (r & 3)) * P + 32 + l32] = v1[r];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int rl = q * 4 + lane / 16, f = lane % 16;
      const int row = row0 + 32 * i + rl, cc = colp[f >> 3] + 4 * (f & 7);
      const float4 x = *reinterpret_cast<const float4 *>(stage + rl * P + 4 * f);
      if (row < M) *reinterpret_cast<float4 *>(c + (size_t)row * N + cc) = x;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// The 256 x 256-tile ping-pong kernel (q4k_gemm_pp.hip) on prepared operands:
// tiles_n column tiles over the matrices of `mats` (kHGelu: tiles of 128
// columns of both), K split ksplit ways (kHPlain only; then a single matrix,
// whose c receives ksplit partial products of M x N).
hipError_t launch_q4k_gemm_pp(int mode, const _Float16 *a16, const int *ea, const HMats &mats, int M, int K,
                              int tiles_n, int ksplit, const GeluOut &go, const QkRope &qr, hipStream_t s);

}  // namespace rt
