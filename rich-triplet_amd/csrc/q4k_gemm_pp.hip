// q4k_gemm_pp.hip -- the Q4_K GEMM for outputs of many tiles: C tile 256 x 256,
// one workgroup of eight waves per CU, weights dequantised once per workgroup.
//
// The waves are two groups of four, one wave of each on every SIMD, that run
// half a stage apart between workgroup barriers: while one group multiplies
// (16 MFMAs of its 128 x 64 of C per stage), the other reads its next fragments
// and issues its copies of A, so the matrix cores always have one wave's MFMAs.
// The dequantisation runs in the multiplying half, a few VALU operations after
// each MFMA (in the other half it made that half the longer one: 441 us
// against 353 at 4608 x 12288 x 3072).
//   A stage is 32 of K, one Q4_K sub-block.  A (f16) comes by global_load_lds
//   three stages ahead into a ring of four 16 KB slots.  W: thread t owns half
//   (t & 1) of column t >> 1: it loads the 16 bytes that hold 16 codes of
//   two sub-blocks (low and high nibbles) into registers, and per stage turns
//   16 codes into f16 and stores them to the W slot of two stages ahead.  A
//   weight is dequantised once per 256 rows and read from LDS by the two
//   waves of its columns, where one wave per 64 columns and 128 rows
//   (k_q4k_gemm_h) dequantised it in registers for 128 rows at 1.5 VALU
//   operations between its own MFMAs.
//   Measured (us, the product alone; C stores nontemporal, which gives 4-7%):
//   4608 x 12288 x 3072 351 (0.99 PFLOP/s; k_q4k_gemm_h 385), 4096 x 20480 x 2560
//   396 (1.08; 465), 4096 x 2560 x 10240 214 (1.00; 256 split three ways), 1000
//   x 10240 x 2560 61 (0.86; 100).  Bound by the schedule, then by power: at the
//   first shape the matrix cores are busy 53% of 624,000 cycles (a library f16
//   product: 66% of 509,000), and the clock is 1.72 GHz, where zero operands
//   take as many cycles at 2.13 (285 us).  Storing C takes 45 us.
//   A slot row is 64 B (4 segments of 8 halves), logical segment s at
//   s ^ ((row >> 2) & 3): the 16 lanes of a ds_read_b128 hit 16 distinct bank
//   groups.
#include <hip/hip_runtime.h>

#include "gemma3_math.hpp"
#include "mfma_common.hpp"
#include "q4k_gemm_dev.hpp"
#include "rt_device.hpp"

namespace rt {
namespace {

constexpr int kPSlot = 256 * 64;  // one operand, one stage

// LDS access at a byte address plus a constant (one address register per
// stream instead of one per slot and fragment; see lds_read16).
RT_DEV uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p; }
template <int OFF>
RT_DEV u32x4 lds_read16_at(uint32_t a) {
  static_assert(OFF >= 0 && OFF < 65536, "16-bit offset");
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
  return v;
}
template <int OFF>
RT_DEV void lds_write16_at(uint32_t a, half8 v) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(a), "v"(__builtin_bit_cast(u32x4, v)), "n"(OFF));
}
template <int V>
struct IntC {
  static constexpr int value = V;
};
// f(IntC<0>), ..., f(IntC<N-1>)
template <int N, class F, int I = 0>
RT_DEV void steps(IntC<N> n, F f) {
  if constexpr (I < N) {
    f(IntC<I>{});
    steps<N, F, I + 1>(n, f);
  }
}

template <int MODE>
__global__ __launch_bounds__(512, 2) void k_q4k_gemm_pp(const _Float16 *__restrict__ a16, const int *__restrict__ ea,
                                                        HMats mats, int M, int K, int tiles_m, int tiles_n,
                                                        int ksplit, GeluOut go, QkRope qr) {
  constexpr bool GELU = MODE == kHGelu, QKV = MODE == kHQkv;
  __shared__ __attribute__((aligned(1024))) uint8_t sa[4][kPSlot], sb[4][kPSlot];
  const int tid = (int)threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, wn = wave & 3;
  // XCD b % 8 gets a contiguous run of tiles, walked in groups of eight tile rows
  const int ntiles = tiles_m * tiles_n, x8 = (int)blockIdx.x & 7, r8 = ntiles & 7, q8 = ntiles >> 3;
  const int tile = (x8 < r8 ? x8 * (q8 + 1) : r8 * (q8 + 1) + (x8 - r8) * q8) + ((int)blockIdx.x >> 3);
  const int group = tile / (8 * tiles_n), in_group = tile % (8 * tiles_n), gm = min(8, tiles_m - group * 8);
  const int tm = group * 8 + in_group % gm, tn = in_group / gm;
  const bool in1 = !GELU && mats.count > 1 && tn >= mats.tn0[1], in2 = !GELU && mats.count > 2 && tn >= mats.tn0[2];
  const int mi = in2 ? 2 : (in1 ? 1 : 0);
  float *__restrict__ c = in2 ? mats.c[2] : (in1 ? mats.c[1] : mats.c[0]);
  const int N = in2 ? mats.n[2] : (in1 ? mats.n[1] : mats.n[0]);
  const int m0 = tm * 256, n0 = GELU ? tn * 128 : (tn - (in2 ? mats.tn0[2] : (in1 ? mats.tn0[1] : 0))) * 256;
  const int nblocks = K / 256, split = (int)blockIdx.y;
  const int b0 = split * nblocks / ksplit, b1 = (split + 1) * nblocks / ksplit;  // >= 1 block (host: ksplit <= nblocks)
  const int jlast = 8 * b1 - 1;
  if (ksplit > 1) c += (size_t)split * M * N;

  // Column of tile column tc (0..255) of matrix *w: plain tc; GELU: waves'
  // 64 columns are 32 of gate, then the same 32 of up; QKV: 32 columns of a
  // head, then the 32 that lie 128 further (the RoPE pairs).
  auto col_of = [&](int tc, int &mat) __attribute__((always_inline)) {
    const int w = tc >> 6, r = tc & 63;
    mat = GELU ? r >> 5 : mi;
    return GELU ? 32 * w + (r & 31) : (QKV ? 32 * w + 128 * (r >> 5) + (r & 31) : tc);
  };
  // W: this thread's column and half
  const int wc = tid >> 1, wh = tid & 1;
  int wmat;
  const int wcol = min(n0 + col_of(wc, wmat), N - 1);
  const uint8_t *wbase = GELU ? (wmat ? mats.w[1] : mats.w[0]) : (in2 ? mats.w[2] : (in1 ? mats.w[1] : mats.w[0]));
  const int *ewp = GELU ? (wmat ? mats.ew[1] : mats.ew[0]) : (in2 ? mats.ew[2] : (in1 ? mats.ew[1] : mats.ew[0]));
  const uint8_t *wrow = wbase + (size_t)wcol * nblocks * kQ4KBlockBytes;
  const float unit = __builtin_amdgcn_ldexpf(1.0f, -ewp[wcol]);
  const uint32_t wsw = (wc >> 2) & 3;
  const uint32_t w0 = lds_addr(sb[0]) + wc * 64 + 16 * ((2 * wh) ^ wsw);
  const uint32_t w1 = lds_addr(sb[0]) + wc * 64 + 16 * ((2 * wh + 1) ^ wsw);
  auto load_q = [&](int b, int chunk) __attribute__((always_inline)) {  // codes of sub-blocks 2 chunk, 2 chunk + 1
    return *reinterpret_cast<const u32x4 *>(wrow + (size_t)b * kQ4KBlockBytes + 16 + 32 * chunk + 16 * wh);
  };
  auto load_h = [&](int b) __attribute__((always_inline)) {
    return *reinterpret_cast<const u32x4 *>(wrow + (size_t)b * kQ4KBlockBytes);
  };
  // The 16 codes of sub-block `sub` as f16 into W slot `slot`, in 14 steps of at
  // most about eight VALU operations, one after each MFMA of a stage.
  uint32_t sv = 0, mv = 0, cw = 0, r[8] = {};
  float ds = 0.f, nc = 0.f;
  auto dequant = [&](auto subc, auto slotc, auto stepc, const u32x4 &h, const u32x4 &q) __attribute__((always_inline)) {
    constexpr int sub = decltype(subc)::value, off = decltype(slotc)::value * kPSlot, m = decltype(stepc)::value;
    if constexpr (m == 0) {
      q4k_scale_min(h[1], h[2], h[3], sub, sv, mv);
    } else if constexpr (m == 1) {
      ds = half_bits_to_f32(h[0] & 0xFFFFu) * unit * (sub & 1 ? 0.0625f : 1.0f);  // high nibbles stay in place: 16 q
      nc = half_bits_to_f32(h[0] >> 16) * unit;
    } else if constexpr (m == 2) {
      ds *= (float)sv;
    } else if constexpr (m == 3) {
      nc = -(nc * (float)mv + 1024.f * ds);
    } else if constexpr (m < 12) {  // two halves of code word k: 1024 + code, then s * that + nc
      constexpr int k = (m - 4) >> 1;
      if constexpr (((m - 4) & 1) == 0) cw = q[k] & (sub & 1 ? 0xF0F0F0F0u : 0x0F0F0F0Fu);
      const uint32_t p = __builtin_amdgcn_perm(0x64646464u, cw, ((m - 4) & 1) == 0 ? 0x04010400u : 0x04030402u);
      asm("v_fma_mixlo_f16 %0, %2, %1, %3 op_sel_hi:[0,1,0]\n\t"
          "v_fma_mixhi_f16 %0, %2, %1, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]"
          : "=&v"(r[m - 4])
          : "v"(p), "v"(ds), "v"(nc));
    } else if constexpr (m == 12) {
      lds_write16_at<off>(w0, __builtin_bit_cast(half8, (u32x4){r[0], r[1], r[2], r[3]}));
    } else if constexpr (m == 13) {
      lds_write16_at<off>(w1, __builtin_bit_cast(half8, (u32x4){r[4], r[5], r[6], r[7]}));
    }
  };

  // A copy i: rows 16 (2 wave + i) + [0, 16), four lanes per row
  const uint8_t *ab = reinterpret_cast<const uint8_t *>(a16 + (size_t)m0 * K);
  uint32_t ao[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * (2 * wave + i) + (lane >> 2);
    ao[i] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K * 2u + 16 * ((lane & 3) ^ ((r >> 2) & 3));
  }
  auto issue_a = [&](int j, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds((gvoid *)(ab + (size_t)j * 64 + ao[i]), (lvoid *)(sa[slot] + (2 * wave + i) * 1024),
                                       16, 0, 0);
  };
  uint32_t fa[2], fb[2];  // k-step t: segment 2t + g; 32 rows further is 2048 bytes (whole swizzle periods)
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t seg = 16 * ((2 * t + g) ^ ((l32 >> 2) & 3));
    fa[t] = lds_addr(sa[0]) + (128 * wm + l32) * 64 + seg;
    fb[t] = lds_addr(sb[0]) + (64 * wn + l32) * 64 + seg;
  }
  floatx16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx16{};

  // Prologue: A stages 0..2 on their way, W stages 0 and 1 in LDS.
  u32x4 hc = load_h(b0), hn = hc, q0 = load_q(b0, 0), q1 = load_q(b0, 1);
  issue_a(8 * b0, 0);
  issue_a(8 * b0 + 1, 1);
  issue_a(8 * b0 + 2, 2);
  steps(IntC<14>{}, [&](auto m) { dequant(IntC<0>{}, IntC<0>{}, m, hc, q0); });
  steps(IntC<14>{}, [&](auto m) { dequant(IntC<1>{}, IntC<1>{}, m, hc, q0); });
  wait_vmcnt<4>();  // A stage 0
  wait_lgkmcnt0();
  wg_barrier();
  if (wm) wg_barrier();  // group 1 runs half a stage behind
  auto half_stages = [&](auto uc, int b, int bn) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value, slot = u & 3, off = slot * kPSlot;
    u32x4 af[2][4], bf[2][2];
    __builtin_amdgcn_sched_barrier(0);
    bf[0][0] = lds_read16_at<off>(fb[0]);
    bf[0][1] = lds_read16_at<off + 2048>(fb[0]);
    af[0][0] = lds_read16_at<off>(fa[0]);
    af[0][1] = lds_read16_at<off + 2048>(fa[0]);
    af[0][2] = lds_read16_at<off + 4096>(fa[0]);
    af[0][3] = lds_read16_at<off + 6144>(fa[0]);
    bf[1][0] = lds_read16_at<off>(fb[1]);
    bf[1][1] = lds_read16_at<off + 2048>(fb[1]);
    af[1][0] = lds_read16_at<off>(fa[1]);
    af[1][1] = lds_read16_at<off + 2048>(fa[1]);
    af[1][2] = lds_read16_at<off + 4096>(fa[1]);
    af[1][3] = lds_read16_at<off + 6144>(fa[1]);
    // The slots written below (stage j+2 of W, j+3 of A) were last read two and
    // one stages ago, by both groups before the barrier that opened this half
    // stage.  W's codes come one chunk ahead, the next block's header six stages.
    issue_a(min(8 * b + u + 3, jlast), (slot + 3) & 3);
    if constexpr (u == 0) hn = load_h(bn);
    if constexpr ((u & 3) == 0) q0 = load_q(u < 4 ? b : bn, (u / 2 + 2) & 3);
    if constexpr ((u & 3) == 2) q1 = load_q(u < 4 ? b : bn, (u / 2 + 2) & 3);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<4>();  // this wave's part of A stage j+1 (at least its copies of j+2 and j+3 follow)
    lds_wait(af[0][0], af[0][1], af[0][2], af[0][3]);
    lds_wait(af[1][0], af[1][1], af[1][2], af[1][3]);
    lds_wait(bf[0][0], bf[0][1], bf[1][0], bf[1][1]);
    wg_barrier();
    __builtin_amdgcn_sched_barrier(0);
    steps(IntC<16>{}, [&](auto mc) __attribute__((always_inline)) {
      constexpr int m = decltype(mc)::value, t = m >> 3, i = (m >> 1) & 3, p = m & 1;
      acc[i][p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, af[t][i]),
                                                          __builtin_bit_cast(half8, bf[t][p]), acc[i][p], 0, 0, 0);
      dequant(IntC<(u + 2) & 7>{}, IntC<(slot + 2) & 3>{}, mc, u < 6 ? hc : hn, ((u + 2) / 2) & 1 ? q1 : q0);
      __builtin_amdgcn_sched_barrier(0);
    });
    __builtin_amdgcn_sched_barrier(0);
    wg_barrier();
  };
  for (int b = b0; b < b1; ++b) {
    const int bn = min(b + 1, b1 - 1);  // past the last block its loads repeat
    half_stages(IntC<0>{}, b, bn);
    half_stages(IntC<1>{}, b, bn);
    half_stages(IntC<2>{}, b, bn);
    half_stages(IntC<3>{}, b, bn);
    half_stages(IntC<4>{}, b, bn);
    half_stages(IntC<5>{}, b, bn);
    half_stages(IntC<6>{}, b, bn);
    half_stages(IntC<7>{}, b, bn);
    hc = hn;
  }
  if (!wm) wg_barrier();  // as many barriers as group 1
  wait_vmcnt<0>();
  wait_lgkmcnt0();
  wg_barrier();

  int ecol[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int m;
    const int n = min(n0 + col_of(64 * wn + 32 * j + l32, m), N - 1);
    ecol[j] = (GELU ? (j ? mats.ew[1] : mats.ew[0]) : (in2 ? mats.ew[2] : (in1 ? mats.ew[1] : mats.ew[0])))[n];
  }
  uint8_t *sbase = wave < 4 ? sa[wave] : sb[wave - 4];
  static_assert(32 * 72 * 4 + 2048 <= kPSlot, "a staging slice and the row sums fit in a slot");
  float *stage = reinterpret_cast<float *>(sbase);
  if constexpr (GELU) {
    store_gelu_tile(acc, stage, go.h16, go.eh, M, N, m0 + 128 * wm, n0 + 32 * wn, ea, ecol, go.a_nrm2, go.gu_bound);
  } else if constexpr (QKV) {
    // row sums of squares of a group's four waves: the end of its last slot
    float(*wsum)[128] = reinterpret_cast<float(*)[128]>((wm ? sb[3] : sa[3]) + kPSlot - 2048);
    store_qkv_tile(acc, stage, wsum, wn, c, M, N, m0 + 128 * wm, n0, mi, ea, ecol, qr);
  } else {
    store_c_tile<2>(acc, stage, c, M, N, m0 + 128 * wm, n0 + 64 * wn, ea, ecol);
  }
}

}  // namespace

hipError_t launch_q4k_gemm_pp(int mode, const _Float16 *a16, const int *ea, const HMats &mats, int M, int K,
                              int tiles_n, int ksplit, const GeluOut &go, const QkRope &qr, hipStream_t s) {
  const int tiles_m = (M + 255) / 256;
  const dim3 grid(tiles_m * tiles_n, ksplit);
  switch (mode) {
    case kHGelu:
      hipLaunchKernelGGL(k_q4k_gemm_pp<kHGelu>, grid, dim3(512), 0, s, a16, ea, mats, M, K, tiles_m, tiles_n, ksplit, go, qr);
      break;
    case kHQkv:
      hipLaunchKernelGGL(k_q4k_gemm_pp<kHQkv>, grid, dim3(512), 0, s, a16, ea, mats, M, K, tiles_m, tiles_n, ksplit, go, qr);
      break;
    default:
      hipLaunchKernelGGL(k_q4k_gemm_pp<kHPlain>, grid, dim3(512), 0, s, a16, ea, mats, M, K, tiles_m, tiles_n, ksplit, go, qr);
  }
  return hipGetLastError();
}

}  // namespace rt
