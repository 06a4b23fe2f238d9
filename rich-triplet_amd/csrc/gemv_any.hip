// gemv_any.hip -- the Q4_K, Q6_K and Q8_0 GEMV y = W x for any K (the shapes
// that have no kernel of their own in q4k_kernels.hip and kquant.hip).
//
// Work split ("column resident", as in q4k_gemv.hpp, with the row length a
// run-time value): a row has S slots (Q4_K / Q6_K: four per super-block,
// Q8_0: one per 32-element block).  Thread t of a workgroup owns slot t % S of
// rows t / S + it * rpi (it < ITERS, rpi = T / S): consecutive threads read
// consecutive pieces of a row, all ITERS rows' weights are in flight before
// any arithmetic, and the activations are staged once per workgroup.
//
// Arithmetic, Q6_K and Q8_0: each 64-element activation chunk is scaled to
// integers X = rint(x * s), s = 2^22 / 2^e with the chunk's max |x| < 2^e,
// written as three balanced bytes X = 65536*x2 + 256*x1 + x0 and a fourth
// x3 = rint(254 (x*s - X)).  The weight codes multiply the digits in exact
// integer dot products (v_dot4_i32_i8), so the roundings are the last digit and
// the f32 combine per slot.  Against float64 on N(0,1) rows: Q6_K 0.9e-7 to
// 1.1e-7 (f32 1.4e-7 to 2.8e-7), Q8_0 0.7e-7 to 1.0e-7 (f32 1.0e-7 to 2.3e-7).
// The last digit is 2^-31 of the chunk's bound.  Where that is not enough -- a
// group of 16 that lies 2^6 below the chunk's largest value (one channel far
// above the others), values below 2^-103, infinities and NaNs -- the chunk's
// slots are multiplied in f32, weight by weight (direct()): 12288x3072 with one
// such chunk 10 -> 14 us (Q8_0) and 20 us (Q6_K), since every wave holds one of
// its slots; one wave per row took 46 and 57.
//   Q4_K: f32 activations; per sub-block sum q x in f32 (four chains) and sum x to
// 48 bits, combined as the reference's scale * sum q x - min * sum x
// (autograd2.rs:1671-1698).  The two parts cancel, so their roundings make the
// error: 2.0e-7 to 2.4e-7, where one wave per row gives 2.6e-7 to 6.9e-7.  The
// same time as 24-bit digits (15360x3840 9.4 us, 3840x15360 11.8), which kept
// 24 bits of a chunk's largest value only: 2.4e-7 to 3.1e-7, and nothing of a
// value 2^24 below it.  Finite values whose 16 q x overflows (from 1.4e36 on)
// are multiplied weight by weight.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "../../include/rt_hip.h"
#include "decode.hpp"
#include "gemma3_math.hpp"
#include "kquant_layout.hpp"
#include "q4k_gemv.hpp"
#include "rt_device.hpp"
#include "rt_kernels.hpp"

namespace rt {
namespace {

// Stage of one chunk, in dwords.  Q4_K: the 64 activations, the sums of its two
// halves and what those sums' f32 rounding left.  Else the four digit planes of
// 16 (dword i = elements 4i .. 4i+3), then delta (negative or NaN where the
// digits do not serve the chunk), padding, and for Q6_K per 16-element sub-block
// the integer sums of x0 + 256*x1 and, packed in one dword, of x2 (low half) and
// x3.  The pitches put the 16 lanes that a 16-byte LDS read serves together on
// distinct banks.
template <int FMT>
constexpr int kAnyPitch = 64 + (FMT == RT_LINEAR_Q6K ? 12 : 4);
constexpr uint32_t kAnySpread = 6;  // powers of two from a chunk's largest value down to each group's of 16
constexpr float kAnyTop = 4194304.0f;  // 2^22: the scaling is exact
constexpr float kAnyUnit = 65536.0f / 4194304.0f;  // delta is 2^(e - 16): finite up to the largest x

template <int CTRL>
RT_DEV double dpp_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, (uint64_t)dpp_u32<CTRL>((uint32_t)u) | (uint64_t)dpp_u32<CTRL>((uint32_t)(u >> 32)) << 32);
}

// Elements 4f .. 4f+3 of the vector (zeros and not `in` past K); the 16 lanes of
// a chunk are consecutive lanes of a wave and all call this; `store` masks the
// lanes past the last chunk.
template <int FMT>
RT_DEV void any_stage(uint32_t *dl, int f, float4 v, bool in, bool store) {
  const int sub = f & 15;
  uint32_t *base = dl + (f >> 4) * kAnyPitch<FMT>, *st = base + 64;
  if constexpr (FMT == RT_LINEAR_Q4K) {
    double half = ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
    half += dpp_f64<0xB1>(half);
    half += dpp_f64<0x4E>(half);
    half += dpp_f64<0x141>(half);  // 8 lanes = 32 elements
    if (!store) return;
    reinterpret_cast<float4 *>(base)[sub] = v;
    const float hi = (float)half;
    if ((sub & 7) == 0) st[sub >> 3] = f32_bits(hi), st[2 + (sub >> 3)] = f32_bits((float)(half - (double)hi));
  } else {
    uint32_t mb = max(max(f32_bits(v.x) & 0x7FFFFFFFu, f32_bits(v.y) & 0x7FFFFFFFu),
                      max(f32_bits(v.z) & 0x7FFFFFFFu, f32_bits(v.w) & 0x7FFFFFFFu));
    mb = max(mb, dpp_u32<0xB1>(mb));
    mb = max(mb, dpp_u32<0x4E>(mb));
    uint32_t gb = in ? mb : 0x7F7FFFFFu;  // least largest |x| of a group of 16; none past K
    gb = min(gb, dpp_u32<0x141>(gb));
    gb = min(gb, dpp_u32<0x140>(gb));
    mb = max(mb, dpp_u32<0x141>(mb));
    mb = max(mb, dpp_u32<0x140>(mb));
    // max < 2^e; below 2^-103 the scale stays at the largest normal one
    const int e = max((int)(mb >> 23) - 126, -103);
    const float s = bits_f32(f32_bits(kAnyTop) - ((uint32_t)e << 23));
    float delta = bits_f32(f32_bits(1.0f / 65536.0f) + ((uint32_t)e << 23));
    if (mb >= 0x7F800000u) delta = bits_f32(0x7FC00000u);
    // negative: the digits do not serve the chunk
    if ((mb >> 23) - (gb >> 23) > kAnySpread || ((mb >> 23) < 24 && mb != 0)) delta = -delta;
    const float xs[4] = {v.x, v.y, v.z, v.w};
    // 1.5 * 2^23 + v holds rint(v) in its low mantissa bits: 5 operations per
    // element, where rounding and converting took 10 (0.3 us at K = 9024)
    constexpr float magic = 12582912.0f;
    uint32_t b[4], r[4];  // bytes 0..2: X + 0x808080; byte 0: the fourth digit
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float t = fmaf(xs[i], s, magic);
      b[i] = f32_bits(t) + 0x408080u;
      r[i] = f32_bits(fmaf(fmaf(xs[i], s, magic - t), 254.0f, magic));
      asm volatile("" : "+v"(b[i]), "+v"(r[i]));  // one after the other: registers
    }
    const uint32_t p01 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u);  // b0.0 b1.0 b0.1 b1.1
    const uint32_t p23 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u);
    const uint32_t h01 = __builtin_amdgcn_perm(b[1], b[0], 0x0C0C0602u);  // b0.2 b1.2 0 0
    const uint32_t h23 = __builtin_amdgcn_perm(b[3], b[2], 0x0C0C0602u);
    const uint32_t r01 = __builtin_amdgcn_perm(r[1], r[0], 0x0C0C0400u), r23 = __builtin_amdgcn_perm(r[3], r[2], 0x0C0C0400u);
    uint32_t d[4];
    d[0] = __builtin_amdgcn_perm(p23, p01, 0x05040100u) ^ 0x80808080u;
    d[1] = __builtin_amdgcn_perm(p23, p01, 0x07060302u) ^ 0x80808080u;
    d[2] = __builtin_amdgcn_perm(h23, h01, 0x05040100u) ^ 0x80808080u;
    d[3] = __builtin_amdgcn_perm(r23, r01, 0x05040100u);
    int s01 = 0, s23 = 0;
    if constexpr (FMT == RT_LINEAR_Q6K) {
      auto sum4 = [](uint32_t q) { return __builtin_amdgcn_sdot4((int)q, 0x01010101, 0, false); };
      s01 = sum4(d[0]) + 256 * sum4(d[1]);
      s23 = sum4(d[2]) + 65536 * sum4(d[3]);
      s01 += (int)dpp_u32<0xB1>((uint32_t)s01);
      s23 += (int)dpp_u32<0xB1>((uint32_t)s23);
      s01 += (int)dpp_u32<0x4E>((uint32_t)s01);  // 4 lanes = 16 elements
      s23 += (int)dpp_u32<0x4E>((uint32_t)s23);
    }
    if (!store) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) base[16 * i + sub] = d[i];
    if (sub == 0) st[0] = f32_bits(delta);
    if constexpr (FMT == RT_LINEAR_Q6K) {
      if ((sub & 3) == 0) st[4 + 2 * (sub >> 2)] = (uint32_t)s01, st[5 + 2 * (sub >> 2)] = (uint32_t)s23;
    }
  }
}

// sum_k c_k x_k / delta from a group's digit sums: the middle digits combine
// exactly (|s0 + 256 s1| < 2^28), then one rounding per step.  The product of
// delta and a block's f16 scale is exact and finite, and its product with the
// dot is the slot's value.
RT_DEV float any_dot(const int (&s)[4]) {
  return fmaf((float)s[2], 65536.0f * kAnyUnit, fmaf((float)s[3], 1.0f / 254.0f, (float)(s[0] + 256 * s[1])) * kAnyUnit);
}

// Weights of a thread's slot in ITERS rows, and their dot products with the
// staged chunk(s): p[it] is the slot's part of row it.
template <int FMT, int ITERS>
struct AnyTile;

template <int ITERS>
struct AnyTile<RT_LINEAR_Q4K, ITERS> {
  uint4 hd[ITERS], qa[ITERS], qb[ITERS];
  RT_DEV void load(int it, const uint8_t *W, int, int K, int row, int slot) {
    const uint8_t *bp = W + ((size_t)row * (K / 256) + (slot >> 2)) * kQ4KBlockBytes;
    const int c = slot & 3;
    hd[it] = *reinterpret_cast<const uint4 *>(bp);
    qa[it] = *reinterpret_cast<const uint4 *>(bp + 16 + 32 * c);
    qb[it] = *reinterpret_cast<const uint4 *>(bp + 32 + 32 * c);
  }
  RT_DEV void compute(const uint32_t *dl, int slot, float (&p)[ITERS]) const {
    const float *base = reinterpret_cast<const float *>(dl) + slot * kAnyPitch<RT_LINEAR_Q4K>;
    float l[ITERS][4], h[ITERS][4];  // sums of q x of the low half, 16 q x of the high half
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int k = 0; k < 4; ++k) l[it][k] = h[it][k] = 0.f;
    const uint32_t mlo = opaque_u32(0x0F0F0F0Fu), mhi = opaque_u32(0xF0F0F0F0u);
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // word j: elements 4j .. 4j+3 of the low half and of the high half
      const float4 a = *reinterpret_cast<const float4 *>(base + 4 * j), b = *reinterpret_cast<const float4 *>(base + 32 + 4 * j);
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const uint4 q = j < 4 ? qa[it] : qb[it];
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        const uint32_t lo = w[j & 3] & mlo, hi = w[j & 3] & mhi;
        l[it][0] = fmaf(ubyte0(lo), a.x, l[it][0]);
        l[it][1] = fmaf(ubyte1(lo), a.y, l[it][1]);
        l[it][2] = fmaf(ubyte2(lo), a.z, l[it][2]);
        l[it][3] = fmaf(ubyte3(lo), a.w, l[it][3]);
        h[it][0] = fmaf(ubyte0(hi), b.x, h[it][0]);
        h[it][1] = fmaf(ubyte1(hi), b.y, h[it][1]);
        h[it][2] = fmaf(ubyte2(hi), b.z, h[it][2]);
        h[it][3] = fmaf(ubyte3(hi), b.w, h[it][3]);
      }
      if (ITERS == 4 && (j & 1)) {  // sums in step with the reads: all 64 activations at once would spill
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
#pragma unroll
          for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(l[it][k]), "+v"(h[it][k]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const float4 sum = *reinterpret_cast<const float4 *>(base + 64);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const float d = half_bits_to_f32(hd[it].x & 0xFFFFu), dm = half_bits_to_f32(hd[it].x >> 16);
      uint32_t svp, mvp;
      q4k_scale_min_pair(hd[it].y, hd[it].z, hd[it].w, slot & 3, svp, mvp);
      const float s0 = d * (float)(svp & 0xFFu), s1 = 0.0625f * d * (float)(svp >> 8);  // exact
      const float m0 = dm * (float)(mvp & 0xFFu), m1 = dm * (float)(mvp >> 8);
      const float lo = fmaf(s0, (l[it][0] + l[it][1]) + (l[it][2] + l[it][3]), -(m0 * sum.x));
      const float hi = fmaf(s1, (h[it][0] + h[it][1]) + (h[it][2] + h[it][3]), -(m1 * sum.y));
      p[it] = fmaf(-m0, sum.z, lo) + fmaf(-m1, sum.w, hi);
      asm volatile("" : "+v"(p[it]));  // summed here: sunk into the branch that stores it, the activations stay live
    }
  }
  // Non-finite parts: the codes times the activations overflowed, or an
  // activation is an infinity or a NaN, which makes the slot NaN as scale * inf
  // - min * inf is.
  RT_DEV static bool plain(const uint32_t *, int, const float (&p)[ITERS]) {
    bool ok = true;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) ok = ok && __builtin_isfinite(p[it]);
    return ok;
  }
  // The slot's part p of the (first) row weight by weight, unless the block's
  // scales are what is not finite.
  RT_DEV float direct(const float *x, int slot, float p) const {
    const float4 *xp = reinterpret_cast<const float4 *>(x + 64 * slot);
    uint32_t svp, mvp;
    q4k_scale_min_pair(hd[0].y, hd[0].z, hd[0].w, slot & 3, svp, mvp);
    const float d = half_bits_to_f32(hd[0].x & 0xFFFFu), dm = half_bits_to_f32(hd[0].x >> 16);
    const float s[2] = {d * (float)(svp & 0xFFu), d * (float)(svp >> 8)};
    const float m[2] = {dm * (float)(mvp & 0xFFu), dm * (float)(mvp >> 8)};
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, nan = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {  // elements 4j .. 4j+3
      const float4 v = xp[j];
      const uint4 q = (j & 4) ? qb[0] : qa[0];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w}, c = (w[j & 3] >> (4 * (j >> 3))) & 0x0F0F0F0Fu;
      acc[0] = fmaf(fmaf(s[j >> 3], ubyte0(c), -m[j >> 3]), v.x, acc[0]);
      acc[1] = fmaf(fmaf(s[j >> 3], ubyte1(c), -m[j >> 3]), v.y, acc[1]);
      acc[2] = fmaf(fmaf(s[j >> 3], ubyte2(c), -m[j >> 3]), v.z, acc[2]);
      acc[3] = fmaf(fmaf(s[j >> 3], ubyte3(c), -m[j >> 3]), v.w, acc[3]);
      nan = fmaf(0.f, v.x, fmaf(0.f, v.y, fmaf(0.f, v.z, fmaf(0.f, v.w, nan))));
    }
    const bool scales = (hd[0].x & 0x7C00u) != 0x7C00u && (hd[0].x & 0x7C000000u) != 0x7C000000u;
    return scales ? (acc[0] + acc[1]) + (acc[2] + acc[3]) + nan : p;
  }
};

template <int ITERS>
struct AnyTile<RT_LINEAR_Q6K, ITERS> {  // slot: see Q6KTile (kquant_tile.hpp)
  uint4 qa[ITERS], qb[ITERS], qh[ITERS];
  uint2 sc[ITERS];
  uint32_t dd[ITERS];
  RT_DEV void load(int it, const uint8_t *W, int N, int K, int row, int slot) {
    const Q6KPlanes P = q6k_planes(W, (size_t)N * (K / 256));
    const size_t blk = (size_t)row * (K / 256) + (slot >> 2);
    const int j = (slot >> 1) & 1, a = slot & 1;
    qa[it] = *reinterpret_cast<const uint4 *>(P.ql + blk * 128 + 64 * j + 16 * a);
    qb[it] = *reinterpret_cast<const uint4 *>(P.ql + blk * 128 + 64 * j + 32 + 16 * a);
    qh[it] = *reinterpret_cast<const uint4 *>(P.qh + blk * 64 + 32 * j + 16 * a);
    sc[it] = *reinterpret_cast<const uint2 *>(P.sc + blk * 16 + 8 * j);
    dd[it] = P.d[blk];
  }
  RT_DEV void compute(const uint32_t *dl, int slot, float (&p)[ITERS]) const {
    const int a = slot & 1;
    const uint32_t m4 = opaque_u32(0x0F0F0F0Fu), m2 = opaque_u32(0x30303030u);
    const uint32_t *base = dl + 2 * (slot >> 1) * kAnyPitch<RT_LINEAR_Q6K>;  // the half block's first chunk
    float acc[ITERS][2];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) acc[it][0] = acc[it][1] = 0.f;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t *cb = base + (m >> 1) * kAnyPitch<RT_LINEAR_Q6K>;
      const int w0 = 8 * (m & 1) + 4 * a;
      uint4 x[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) x[d] = *reinterpret_cast<const uint4 *>(cb + 16 * d + w0);
      const uint2 xs = *reinterpret_cast<const uint2 *>(cb + 68 + 2 * (w0 >> 2));
      const int xs01 = 32 * (int)xs.x, xs2 = 32 * (int)(int16_t)(xs.y & 0xFFFFu);
      const int xs3 = 32 * (((int)xs.y - (int)(int16_t)(xs.y & 0xFFFFu)) >> 16);
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const uint4 ql = (m & 1) ? qb[it] : qa[it];
        const uint32_t lw[4] = {ql.x, ql.y, ql.z, ql.w}, hb[4] = {qh[it].x, qh[it].y, qh[it].z, qh[it].w};
        int s[4] = {-xs01, 0, -xs2, -xs3};  // sum X (q - 32), digit by digit
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t nib = (m < 2 ? lw[k] : lw[k] >> 4) & m4;
          const int sh = 2 * m;
          const int q = (int)(nib | ((sh <= 4 ? hb[k] << (4 - sh) : hb[k] >> (sh - 4)) & m2));
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const uint32_t X[4] = {x[d].x, x[d].y, x[d].z, x[d].w};
            s[d] = __builtin_amdgcn_sdot4(q, (int)X[k], s[d], false);
          }
        }
        const float t = any_dot(s);
        const uint32_t scw = m < 2 ? sc[it].x : sc[it].y;  // scales 2m + a of the half block: byte 2*(m&1) + a
        acc[it][m >> 1] = fmaf((float)(int)__builtin_amdgcn_sbfe(scw, 16 * (m & 1) + 8 * a, 8), t, acc[it][m >> 1]);
      }
    }
    const float d0 = fabsf(bits_f32(base[64])), d1 = fabsf(bits_f32(base[kAnyPitch<RT_LINEAR_Q6K> + 64]));
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const float d = half_bits_to_f32(dd[it]);
      p[it] = fmaf(acc[it][1], d * d1, acc[it][0] * (d * d0));
    }
  }
  RT_DEV static bool plain(const uint32_t *dl, int slot, const float (&)[ITERS]) {
    const uint32_t *base = dl + 2 * (slot >> 1) * kAnyPitch<RT_LINEAR_Q6K>;
    return bits_f32(base[64]) > 0.f && bits_f32(base[kAnyPitch<RT_LINEAR_Q6K> + 64]) > 0.f;
  }
  // The slot's part of the (first) row in f32, q6k_value by q6k_value: 16
  // elements of each quarter of its half block.
  RT_DEV float direct(const float *x, int slot, float) const {
    const int a = slot & 1;
    const float4 *xp = reinterpret_cast<const float4 *>(x + 128 * (slot >> 1) + 16 * a);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      asm volatile("" : "+v"(xp), "+v"(acc[0]));  // one quarter after the other: registers
      const uint4 ql = (m & 1) ? qb[0] : qa[0];
      const uint32_t lw[4] = {ql.x, ql.y, ql.z, ql.w}, hb[4] = {qh[0].x, qh[0].y, qh[0].z, qh[0].w};
      const float s = half_bits_to_f32(dd[0]) *
                      (float)(int)__builtin_amdgcn_sbfe(m < 2 ? sc[0].x : sc[0].y, 16 * (m & 1) + 8 * a, 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float4 v = xp[8 * m + k];
        const uint32_t q = ((m < 2 ? lw[k] : lw[k] >> 4) & 0x0F0F0F0Fu) | (((hb[k] >> (2 * m)) & 0x03030303u) << 4);
        acc[0] = fmaf(mul_nc(s, (float)((int)(q & 0xFFu) - 32)), v.x, acc[0]);
        acc[1] = fmaf(mul_nc(s, (float)((int)((q >> 8) & 0xFFu) - 32)), v.y, acc[1]);
        acc[2] = fmaf(mul_nc(s, (float)((int)((q >> 16) & 0xFFu) - 32)), v.z, acc[2]);
        acc[3] = fmaf(mul_nc(s, (float)((int)(q >> 24) - 32)), v.w, acc[3]);
      }
    }
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
};

template <int ITERS>
struct AnyTile<RT_LINEAR_Q8_0, ITERS> {
  uint4 qa[ITERS], qb[ITERS];
  uint32_t dd[ITERS];
  RT_DEV void load(int it, const uint8_t *W, int N, int K, int row, int slot) {
    const uint8_t *q = W + (size_t)row * K + 32 * slot;
    const uint16_t *D = reinterpret_cast<const uint16_t *>(W + (size_t)N * K) + (size_t)row * (K / 32);
    qa[it] = *reinterpret_cast<const uint4 *>(q);
    qb[it] = *reinterpret_cast<const uint4 *>(q + 16);
    dd[it] = D[slot];
  }
  RT_DEV void compute(const uint32_t *dl, int slot, float (&p)[ITERS]) const {
    const uint32_t *base = dl + (slot >> 1) * kAnyPitch<RT_LINEAR_Q8_0>;
    int s[ITERS][4];
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int d = 0; d < 4; ++d) s[it][d] = 0;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      if (ITERS == 4 && g) __builtin_amdgcn_sched_barrier(0);
      uint4 x[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) x[d] = *reinterpret_cast<const uint4 *>(base + 16 * d + 8 * (slot & 1) + 4 * g);
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const uint4 q = g ? qb[it] : qa[it];
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const uint32_t X[4] = {x[d].x, x[d].y, x[d].z, x[d].w};
            s[it][d] = __builtin_amdgcn_sdot4((int)w[j], (int)X[j], s[it][d], false);
          }
      }
    }
    const float delta = fabsf(bits_f32(base[64]));
#pragma unroll
    for (int it = 0; it < ITERS; ++it) p[it] = half_bits_to_f32(dd[it]) * delta * any_dot(s[it]);
  }
  RT_DEV static bool plain(const uint32_t *dl, int slot, const float (&)[ITERS]) {
    return bits_f32(dl[(slot >> 1) * kAnyPitch<RT_LINEAR_Q8_0> + 64]) > 0.f;
  }
  RT_DEV float direct(const float *x, int slot, float) const {
    const float4 *xp = reinterpret_cast<const float4 *>(x + 32 * slot);
    const float d = half_bits_to_f32(dd[0]);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g == 4) asm volatile("" : "+v"(xp), "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
      const float4 v = xp[g];
      const uint4 q = g < 4 ? qa[0] : qb[0];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
      acc[0] = fmaf(d * (float)(int8_t)(w[g & 3] & 0xFFu), v.x, acc[0]);
      acc[1] = fmaf(d * (float)(int8_t)((w[g & 3] >> 8) & 0xFFu), v.y, acc[1]);
      acc[2] = fmaf(d * (float)(int8_t)((w[g & 3] >> 16) & 0xFFu), v.z, acc[2]);
      acc[3] = fmaf(d * (float)(int8_t)(w[g & 3] >> 24), v.w, acc[3]);
    }
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
};

// Dynamic LDS: the staged chunks, then ITERS * T slot sums.  T = blockDim.x as
// an argument: reading blockDim makes the runtime fill the launch's hidden
// arguments, 0.6 us of host time.
// Q8_0 in 80 registers: three workgroups of 512 threads per CU, so that the 615 of
// 12288x3072 run at once (89 registers: 10.0 us against 9.8).
template <int FMT, int ITERS>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(FMT == RT_LINEAR_Q8_0 ? 6 : 4))) void
k_gemv_any(const uint8_t *__restrict__ W, const float *__restrict__ x, float *__restrict__ y, int N, int K, int S, int rpi,
           int T) {
  extern __shared__ __attribute__((aligned(16))) uint32_t any_lds[];
  const int tid = (int)threadIdx.x;
  const int nchunk = (K + 63) / 64, nf = K / 4;
  uint32_t *dl = any_lds;
  float *red = reinterpret_cast<float *>(any_lds + nchunk * kAnyPitch<FMT>);
  // activation loads first (the host makes 16 T >= K), so their wait leaves
  // the weight loads in flight
  float4 xv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xv[i] = reinterpret_cast<const float4 *>(x)[min(tid + i * T, nf - 1)];
  const int slot = tid % S, rsub = tid / S;
  const int row0 = (int)blockIdx.x * rpi * ITERS;
  AnyTile<FMT, ITERS> tile;
  // rows past N, and the threads past rpi * S, re-read a valid row
#pragma unroll
  for (int it = 0; it < ITERS; ++it) tile.load(it, W, N, K, min(row0 + it * rpi + rsub, N - 1), slot);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int f = tid + i * T;
    if (i > 0 && i * T >= 16 * nchunk) break;  // uniform
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    any_stage<FMT>(dl, f, f < nf ? xv[i] : z, f < nf, f < 16 * nchunk);
  }
  __syncthreads();
  float p[ITERS];
  tile.compute(dl, slot, p);
  if (__builtin_expect(!tile.plain(dl, slot, p), 0)) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      // the row's weights again, one row at a time: kept across compute() they spill
      int row = min(row0 + it * rpi + rsub, N - 1);
      asm volatile("" : "+v"(row), "+v"(p[it > 0 ? it - 1 : 0]));
      AnyTile<FMT, 1> again;
      again.load(0, W, N, K, row, slot);
      p[it] = again.direct(x, slot, p[it]);
    }
  }
  if (rsub < rpi) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) red[it * rpi * S + tid] = p[it];
  }
  __syncthreads();
  // 16 lanes per row: strided slot sums, then across the lanes
  const int rows = min(rpi * ITERS, N - row0);
  for (int r = tid >> 4; r < ((rows + 3) & ~3); r += T >> 4) {  // whole waves
    float s = 0.f;
    for (int c = tid & 15; c < S; c += 16) s += red[min(r, rows - 1) * S + c];
    s = row16_sum(s);
    if ((tid & 15) == 0 && r < rows) y[row0 + r] = s;
  }
}

// ---------------------------------------------------------------------------
// The decode step's q|k|v and gate|up launches for any hidden width: the
// prologue of k_qkv / k_gateup (decode_kernels.hip) in front of the same tiles.
// ---------------------------------------------------------------------------
// Sum over the T threads (T/64 waves) of a workgroup; `red` holds 16 floats
// that no earlier call reads.
RT_DEV float any_block_sum(float v, float *red, int T) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < T / 64; ++i) s += red[i];
  return s;
}

// x = EMBED: the token's embedding row * embed_scale, else base + rms(add)
// (1 + g_add); xn = rms(x) (1 + g_out).  Two float4 per thread (8 T >= K).
// load() issues every global load, finish() returns xn and lets workgroup 0
// store x and xn.
template <bool EMBED>
struct AnyPrologue {
  float4 add[2], base[2], ga[2], go[2];
  RT_DEV void load(const DecodeArgs &a, const float *b, const float *ad, const float *g_add, const float *g_out, int K,
                   int T) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int f = min((int)threadIdx.x + i * T, K / 4 - 1);
      if constexpr (EMBED) {
        const uint2 w = reinterpret_cast<const uint2 *>(a.embed + (size_t)a.params[0] * K)[f];
        add[i] = make_float4(mul_nc(bf16_lo(w.x), a.embed_scale), mul_nc(bf16_hi(w.x), a.embed_scale),
                             mul_nc(bf16_lo(w.y), a.embed_scale), mul_nc(bf16_hi(w.y), a.embed_scale));
      } else {
        add[i] = reinterpret_cast<const float4 *>(ad)[f];
        base[i] = reinterpret_cast<const float4 *>(b)[f];
        ga[i] = reinterpret_cast<const float4 *>(g_add)[f];
      }
      go[i] = reinterpret_cast<const float4 *>(g_out)[f];
    }
  }
  RT_DEV void finish(const DecodeArgs &a, float *x_out, float *xn_out, float *red, int K, int T, float4 (&xn)[2]) {
    const float inv_k = 1.0f / (float)K;
    const int f0 = (int)threadIdx.x, nf = K / 4;
    if constexpr (!EMBED) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) ss += f0 + i * T < nf ? sumsq4(add[i]) : 0.f;
      const float r = rms_inv_from_sumsq(any_block_sum(ss, red, T), inv_k, a.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) add[i] = add4(base[i], norm4(add[i], r, ga[i]));
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) ss += f0 + i * T < nf ? sumsq4(add[i]) : 0.f;
    const float r = rms_inv_from_sumsq(any_block_sum(ss, red + 16, T), inv_k, a.eps);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int f = f0 + i * T;
      xn[i] = norm4(add[i], r, go[i]);
      if (blockIdx.x == 0 && f < nf) {
        if (x_out) reinterpret_cast<float4 *>(x_out)[f] = add[i];
        if (xn_out) reinterpret_cast<float4 *>(xn_out)[f] = xn[i];
      }
    }
  }
};

// The fused launches keep the digits in every chunk (32 bits of its largest
// normalised value, where the one-row pass before them kept 16).
template <int FMT>
RT_DEV void any_stage_pro(uint32_t *dl, const float4 (&xn)[2], int K, int T) {
  const int nf = K / 4, nst = 16 * ((K + 63) / 64);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int f = (int)threadIdx.x + i * T;
    if (i > 0 && T >= nst) break;  // uniform
    any_stage<FMT>(dl, f, f < nf ? xn[i] : make_float4(0.f, 0.f, 0.f, 0.f), f < nf, f < nst);
  }
}

// Rows of q, then k, then (nv > 0) v, all of format FMT; a thread picks its
// rows' matrix, so a workgroup may hold rows of two.  x goes to a.hid, xn to
// a.xn (for a v of another format).
template <int FMT, bool EMBED>
__global__ __launch_bounds__(1024) void k_any_qkv(DecodeArgs a, LayerArgs L, LayerArgs prev, int K, int S, int rpi,
                                                  int T, int nv) {
  extern __shared__ __attribute__((aligned(16))) uint32_t any_lds[];
  __shared__ float bred[32];
  const int tid = (int)threadIdx.x;
  uint32_t *dl = any_lds;
  float *red = reinterpret_cast<float *>(any_lds + (K + 63) / 64 * kAnyPitch<FMT>);
  AnyPrologue<EMBED> pro;
  pro.load(a, a.x2, a.dn, prev.g_post_ffn, L.g_in, K, T);
  const int qd = a.n_q_heads * a.head_dim, kvd = a.n_kv_heads * a.head_dim, N = qd + kvd + nv;
  const int slot = tid % S, rsub = tid / S, row0 = (int)blockIdx.x * rpi;
  const int row = min(row0 + rsub, N - 1);
  const bool in_q = row < qd, in_k = !in_q && row < qd + kvd;
  __syncthreads();  // the prologue's loads leave before any weight load of the workgroup
  AnyTile<FMT, 1> tile;
  tile.load(0, in_q ? L.wq : (in_k ? L.wk : L.wv), in_q ? qd : kvd, K, row - (in_q ? 0 : (in_k ? qd : qd + kvd)), slot);
  float4 xn[2];
  pro.finish(a, a.hid, a.xn, bred, K, T, xn);
  any_stage_pro<FMT>(dl, xn, K, T);
  __syncthreads();
  float p[1];
  tile.compute(dl, slot, p);
  if (rsub < rpi) red[tid] = p[0];
  __syncthreads();
  const int rows = min(rpi, N - row0);
  for (int r = tid >> 4; r < ((rows + 3) & ~3); r += T >> 4) {  // whole waves
    float s = 0.f;
    for (int c = tid & 15; c < S; c += 16) s += red[min(r, rows - 1) * S + c];
    s = row16_sum(s);
    const int n = row0 + r;
    if ((tid & 15) == 0 && r < rows)
      (n < qd ? a.q + n : (n < qd + kvd ? a.k + (n - qd) : a.v + (n - qd - kvd)))[0] = s;
  }
}

// PAIRS * rpi gate rows and the same up rows; h = gelu_tanh(g) * u.
template <int FMT, int PAIRS>
__global__ __launch_bounds__(1024) void k_any_gateup(DecodeArgs a, LayerArgs L, int ffn, int K, int S, int rpi, int T) {
  extern __shared__ __attribute__((aligned(16))) uint32_t any_lds[];
  __shared__ float bred[32];
  const int tid = (int)threadIdx.x;
  uint32_t *dl = any_lds;
  float *red = reinterpret_cast<float *>(any_lds + (K + 63) / 64 * kAnyPitch<FMT>);
  AnyPrologue<false> pro;
  pro.load(a, a.hid, a.o, L.g_post_attn, L.g_pre_ffn, K, T);
  const int slot = tid % S, rsub = tid / S, row0 = (int)blockIdx.x * rpi * PAIRS;
  __syncthreads();
  AnyTile<FMT, 2 * PAIRS> tile;
#pragma unroll
  for (int it = 0; it < 2 * PAIRS; ++it)
    tile.load(it, it & 1 ? L.wup : L.wgate, ffn, K, min(row0 + (it >> 1) * rpi + rsub, ffn - 1), slot);
  float4 xn[2];
  pro.finish(a, a.x2, a.xn, bred, K, T, xn);
  any_stage_pro<FMT>(dl, xn, K, T);
  __syncthreads();
  float p[2 * PAIRS];
  tile.compute(dl, slot, p);
  if (rsub < rpi) {
#pragma unroll
    for (int it = 0; it < 2 * PAIRS; ++it) red[(PAIRS * (it & 1) + (it >> 1)) * rpi * S + tid] = p[it];
  }
  __syncthreads();
  const int rows = min(rpi * PAIRS, ffn - row0);
  const float *up = red + PAIRS * rpi * S;
  for (int r = tid >> 4; r < ((rows + 3) & ~3); r += T >> 4) {
    const int rr = min(r, rows - 1) * S;
    float g = 0.f, u = 0.f;
    for (int c = tid & 15; c < S; c += 16) g += red[rr + c], u += up[rr + c];
    g = row16_sum(g);
    u = row16_sum(u);
    if ((tid & 15) == 0 && r < rows) a.h[row0 + r] = mul_nc(gelu_tanh(g), u);
  }
}

// The prologue alone, one workgroup: x to x_out (if any), xn to xn_out.
template <bool EMBED>
__global__ __launch_bounds__(512) void k_any_prologue(DecodeArgs a, const float *base, const float *add,
                                                      const float *g_add, const float *g_out, int K, float *x_out,
                                                      float *xn_out) {
  __shared__ float bred[32];
  AnyPrologue<EMBED> pro;
  pro.load(a, base, add, g_add, g_out, K, 512);
  float4 xn[2];
  pro.finish(a, x_out, xn_out, bred, K, 512, xn);
}

}  // namespace

// Workgroup shape, from a sweep of 256..1024 threads and 1, 2 or 4 rows per
// thread over 19 shapes (distinct matrices in a graph, us; Q4_K then on digits
// of the same time):
//   T: the smallest multiple of 64 from 512 (768 for K >= 8192, whose staging
//   is longer; 320 or, below K = 2048, 192 where 512
//   would leave CUs without a workgroup) whose
//   whole rows fill at least 0.9 of the threads.  Q4_K 15360x3840: 512 threads
//   10.0, 960 (no idle thread) 10.9; 3840x15360: 1024 threads 12.0, 960 12.2.
//   ITERS: the most that keeps about two workgroups per CU (one for K >= 8192:
//   3072x12288 in 192 workgroups 9.4, 384 10.0, 768 10.3; 12288x3072 in 512
//   to 768 workgroups 7.4-7.7).  Q6_K stops at two: four spill registers.
// Before, one wave per row in f32 (kept for longer K): Q4_K 15360x3840 30.3 us
// (1.1 TB/s; now 9.4, 3.5 TB/s, of a 6.7 us streaming floor), 3072x12288
// 24.4 -> 8.9; Q6_K 12288x3072 57.5 -> 9.8, 1152x6912 39.2 -> 5.2; Q8_0
// 12288x3072 47.0 -> 9.8, 6912x1152 8.1 -> 3.7.
constexpr int kAnyMaxK = 16384;  // four float4 of x per thread at T = 1024

// Allows k_gemv_any the LDS of its longest rows (86 KB of the CU's 160), once per
// device: the allowance is the kernel's, so one set per call and to that call's
// size could take it from a launch of another host thread.
template <int FMT, int ITERS>
static hipError_t any_allow_lds() {
  static std::atomic<uint64_t> done{0};  // a bit per device
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev < 64 ? uint64_t(1) << dev : 0;
  if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
  e = hipFuncSetAttribute((const void *)k_gemv_any<FMT, ITERS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          kAnyMaxK / 64 * kAnyPitch<FMT> * 4 + ITERS * 1024 * 4);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}

template <int FMT, int ITERS>
static hipError_t launch_any(const void *W, const float *x, float *y, int N, int K, int S, int T, hipStream_t s) {
  const int rpi = T / S, rows = rpi * ITERS;
  const size_t lds = (size_t)((K + 63) / 64) * kAnyPitch<FMT> * 4 + (size_t)rows * S * 4;
  if (lds > 65536) {
    const hipError_t e = any_allow_lds<FMT, ITERS>();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_gemv_any<FMT, ITERS>), dim3((unsigned)((N + rows - 1) / rows)), dim3(T), lds, s,
                     static_cast<const uint8_t *>(W), x, y, N, K, S, rpi, T);
  return hipGetLastError();
}

bool gemv_any_ok(int K) { return K <= kAnyMaxK; }

// The smallest multiple of 64 threads from t0 (and of at least `per` elements
// of x each) whose whole rows of S slots fill 0.9 of them, else the fullest.
static int any_threads(int S, int K, int per, int t0) {
  t0 = std::max((t0 + 63) / 64 * 64, std::max((S + 63) / 64 * 64, (K / per + 63) / 64 * 64));
  int T = t0 = std::min(t0, 1024);
  for (int t = t0; t <= 1024; t += 64) {
    const int used = t / S * S, best = T / S * S;
    if ((long)used * T > (long)best * t) T = t;
    if (10 * (T / S * S) >= 9 * T) break;
  }
  return T;
}

template <int FMT>
static hipError_t launch_fmt(const void *W, const float *x, float *y, int N, int K, hipStream_t s) {
  const int S = FMT == RT_LINEAR_Q8_0 ? K / 32 : K / 64;
  const bool longk = K >= 8192;
  int t0 = longk ? 768 : 512;
  if (!longk && N < 200 * (512 / S)) t0 = K < 2048 ? 192 : 320;
  const int T = any_threads(S, K, 16, t0);
  const int rpi = T / S, want = longk ? 192 : 448;
  auto wgs = [&](int it) { return (N + rpi * it - 1) / (rpi * it); };
  if (FMT != RT_LINEAR_Q6K && wgs(4) >= want) return launch_any<FMT, FMT == RT_LINEAR_Q6K ? 2 : 4>(W, x, y, N, K, S, T, s);
  if (wgs(2) >= want) return launch_any<FMT, 2>(W, x, y, N, K, S, T, s);
  return launch_any<FMT, 1>(W, x, y, N, K, S, T, s);
}

hipError_t launch_gemv_any(int fmt, const void *W, const float *x, float *y, int N, int K, hipStream_t s) {
  switch (fmt) {
    case RT_LINEAR_Q4K: return launch_fmt<RT_LINEAR_Q4K>(W, x, y, N, K, s);
    case RT_LINEAR_Q6K: return launch_fmt<RT_LINEAR_Q6K>(W, x, y, N, K, s);
    case RT_LINEAR_Q8_0: return launch_fmt<RT_LINEAR_Q8_0>(W, x, y, N, K, s);
    default: return hipErrorInvalidValue;
  }
}

// ---------------------------------------------------------------------------
// The single-token step of a shape without fused templates: six launches per
// layer (q|k|v, attention, its merge, o, gate|up, down) where the formats of a
// set agree, each projection of another mix its own GEMV behind k_any_prologue.
// As a one-row pass of the verify's kernels (eleven launches per layer, split-K
// partial sums between them) the step at Gemma-3-1B widths (26 layers, hidden
// 1152, Q8_0, 700 keys, logits to the host) took 1,685 us; so 1,000 us, of which
// per layer q|k|v 5.0, attention 6.7, merge 4.6, o 4.1, gate|up 7.2 and down
// 6.1 us, and the BF16 head 104 us (5.8 TB/s).  Error against float64 2.6e-4
// before (16-bit digits), 1.7e-5 so.
// ---------------------------------------------------------------------------
static bool any_set_fmt(int fmt) { return fmt == RT_LINEAR_Q4K || fmt == RT_LINEAR_Q6K || fmt == RT_LINEAR_Q8_0; }

template <int FMT>
static void any_qkv(const DecodeArgs &a, const LayerArgs &L, const LayerArgs &P, bool first, int K, int rows, int nv,
                    hipStream_t s) {
  // about one workgroup per CU: 1,536 rows of 1152 in 220 workgroups of 256
  const int S = FMT == RT_LINEAR_Q8_0 ? K / 32 : K / 64;
  const int T = any_threads(S, K, 8, std::max(256, S * ((rows + 255) / 256)));
  const int rpi = T / S;
  const dim3 grid((unsigned)((rows + rpi - 1) / rpi));
  const size_t lds = (size_t)((K + 63) / 64) * kAnyPitch<FMT> * 4 + (size_t)rpi * S * 4;
  if (first)
    hipLaunchKernelGGL((k_any_qkv<FMT, true>), grid, dim3(T), lds, s, a, L, P, K, S, rpi, T, nv);
  else
    hipLaunchKernelGGL((k_any_qkv<FMT, false>), grid, dim3(T), lds, s, a, L, P, K, S, rpi, T, nv);
}

template <int FMT, int PAIRS>
static void any_gateup_p(const DecodeArgs &a, const LayerArgs &L, int ffn, int K, int S, int T, hipStream_t s) {
  const int rpi = T / S;
  const size_t lds = (size_t)((K + 63) / 64) * kAnyPitch<FMT> * 4 + (size_t)2 * PAIRS * rpi * S * 4;
  hipLaunchKernelGGL((k_any_gateup<FMT, PAIRS>), dim3((unsigned)((ffn + rpi * PAIRS - 1) / (rpi * PAIRS))), dim3(T),
                     lds, s, a, L, ffn, K, S, rpi, T);
}

template <int FMT>
static void any_gateup(const DecodeArgs &a, const LayerArgs &L, int ffn, int K, hipStream_t s) {
  const int S = FMT == RT_LINEAR_Q8_0 ? K / 32 : K / 64;
  const int T = any_threads(S, K, 8, 512), rpi = T / S;
  // two gate and two up rows per thread (one each for Q6_K, whose four rows
  // spill) while that leaves most CUs a workgroup: 6,912 rows in 247
  if (FMT != RT_LINEAR_Q6K && ffn >= 2 * rpi * 200) any_gateup_p<FMT, FMT == RT_LINEAR_Q6K ? 1 : 2>(a, L, ffn, K, S, T, s);
  else any_gateup_p<FMT, 1>(a, L, ffn, K, S, T, s);
}

#define RT_ANY_FMT(fmt, call)                                     \
  switch (fmt) {                                                  \
    case RT_LINEAR_Q4K: call(RT_LINEAR_Q4K); break;               \
    case RT_LINEAR_Q6K: call(RT_LINEAR_Q6K); break;               \
    default: call(RT_LINEAR_Q8_0); break;                         \
  }

static hipError_t any_proj(int fmt, const uint8_t *W, const float *x, float *y, int n, int k, hipStream_t s) {
  switch (fmt) {
    case RT_LINEAR_Q6K: return launch_q6k_gemv(W, x, y, n, k, s);
    case RT_LINEAR_Q8_0: return launch_q8_0_gemv(W, x, y, n, k, s);
    case RT_LINEAR_BF16: return launch_bf16_gemv(reinterpret_cast<const uint16_t *>(W), x, y, n, k, s);
    default: return launch_q4k_gemv(W, x, y, n, k, s);
  }
}

hipError_t enqueue_decode_step_any(const DecodeShape &sh, const DecodeArgs &a, const LayerArgs *layers, hipStream_t s) {
  const int H = sh.hidden, qd = sh.n_q_heads * sh.head_dim, kvd = sh.n_kv_heads * sh.head_dim;
  hipError_t e = hipSuccess;
  auto ok = [&](hipError_t r) { return (e = e == hipSuccess ? r : e) == hipSuccess; };
  for (int i = 0; i < sh.n_layers; ++i) {
    const LayerArgs &L = layers[i], &P = layers[i > 0 ? i - 1 : 0];
    const int fq = L.fmt[kProjQ], fv = L.fmt[kProjV];
    if (any_set_fmt(fq) && L.fmt[kProjK] == fq) {
      const int nv = fv == fq ? kvd : 0;
#define RT_QKV(F) any_qkv<F>(a, L, P, i == 0, H, qd + kvd + nv, nv, s)
      RT_ANY_FMT(fq, RT_QKV)
#undef RT_QKV
      ok(hipGetLastError());
      if (nv == 0) ok(any_proj(fv, L.wv, a.xn, a.v, kvd, H, s));
    } else {
      if (i == 0)
        hipLaunchKernelGGL(k_any_prologue<true>, dim3(1), dim3(512), 0, s, a, nullptr, nullptr, nullptr, L.g_in, H, a.hid,
                           a.xn);
      else
        hipLaunchKernelGGL(k_any_prologue<false>, dim3(1), dim3(512), 0, s, a, a.x2, a.dn, P.g_post_ffn, L.g_in, H,
                           a.hid, a.xn);
      ok(hipGetLastError());
      ok(any_proj(fq, L.wq, a.xn, a.q, qd, H, s));
      ok(any_proj(L.fmt[kProjK], L.wk, a.xn, a.k, kvd, H, s));
      ok(any_proj(fv, L.wv, a.xn, a.v, kvd, H, s));
    }
    ok(enqueue_decode_attention(sh, a, L, s));
    ok(any_proj(L.fmt[kProjO], L.wo, a.attn, a.o, H, qd, s));
    const int fg = L.fmt[kProjGate];
    if (any_set_fmt(fg) && L.fmt[kProjUp] == fg) {
#define RT_GU(F) any_gateup<F>(a, L, sh.ffn, H, s)
      RT_ANY_FMT(fg, RT_GU)
#undef RT_GU
      ok(hipGetLastError());
    } else {
      hipLaunchKernelGGL(k_any_prologue<false>, dim3(1), dim3(512), 0, s, a, a.hid, a.o, L.g_post_attn, L.g_pre_ffn, H,
                         a.x2, a.xn);
      ok(hipGetLastError());
      ok(any_proj(fg, L.wgate, a.xn, a.h, sh.ffn, H, s));
      ok(any_proj(L.fmt[kProjUp], L.wup, a.xn, a.u, sh.ffn, H, s));
      ok(launch_gelu_mul_vec(a.h, a.u, sh.ffn, s));
    }
    ok(any_proj(L.fmt[kProjDown], L.wdown, a.h, a.dn, H, sh.ffn, s));
    if (e != hipSuccess) return e;
  }
  // final residual and norm (transformer4.rs:2370-2380), then the head
  hipLaunchKernelGGL(k_any_prologue<false>, dim3(1), dim3(512), 0, s, a, a.x2, a.dn, layers[sh.n_layers - 1].g_post_ffn,
                     a.g_final, H, nullptr, a.xn);
  ok(hipGetLastError());
  if (a.lm_q4k) ok(launch_q4k_gemv(a.lm_q4k, a.xn, a.logits, sh.vocab, H, s));
  else ok(launch_bf16_gemv(a.lm_bf16, a.xn, a.logits, sh.vocab, H, s));
  return e;
}
#undef RT_ANY_FMT

}  // namespace rt
