// Super-tile layouts and their dequantisation to f16 MFMA operands, shared by
// the kernels that stream quantized weights (layouts: gemv.hip).
#pragma once
#include <type_traits>

#include "cwen_internal.h"

namespace {

// Per-format layout of one 16-row x 512-K super-tile of one weight stream.
template <int FMT> struct Fmt;
template <> struct Fmt<GEMV_Q4> {
  static constexpr uint32_t ST_BYTES = 4608, SC_OFS = 4096;
  static constexpr int TV = 1;                 // 16-byte loads per tile per lane
};
template <> struct Fmt<GEMV_Q6K> {
  static constexpr uint32_t ST_BYTES = 6720, HI_OFS = 4096, SC_OFS = 6144, D_OFS = 6656;
  static constexpr int TV = 1;
};
template <> struct Fmt<GEMV_Q8> {
  static constexpr uint32_t ST_BYTES = 8704, SC_OFS = 8192;
  static constexpr int TV = 2;
};
// Q4_1: the Q4_0 nibble layout, then per lane the 4 blocks' (d, m) f16 pairs.
template <> struct Fmt<GEMV_Q41> {
  static constexpr uint32_t ST_BYTES = 5120, SC_OFS = 4096;
  static constexpr int TV = 1;
};
// Q5_K: the low 4 bits in the Q4_0 nibble layout, then per lane one dword
// of fifth bits per tile (kQ5HiPos), then per lane the 4 sub-blocks'
// (d*sc, -dmin*m) f16 pairs.
template <> struct Fmt<GEMV_Q5K> {
  static constexpr uint32_t ST_BYTES = 6144, HI_OFS = 4096, SC_OFS = 5120;
  static constexpr int TV = 1;
};
// (q & mask) | magic in one VOP3 op.  gfx9 VOP3 takes no literal and reads at
// most one scalar, so the mask comes from an SGPR and the magic from a VGPR.
__device__ __forceinline__ uint32_t and_or(uint32_t q, uint32_t mask_s, uint32_t magic_v) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(q), "s"(mask_s), "v"(magic_v));
  return r;
}

struct Unpack {
  uint32_t lo, hi;     // SGPR masks 0x000F000F, 0x00F000F0
  uint32_t h0, h1;     // SGPR masks 0x00300030, 0x03000300 (Q6_K high bits)
  uint32_t b4, b8;     // SGPR masks 0x00100010, 0x01000100 (Q5_K fifth bits)
  uint32_t magic;      // VGPR 0x64006400
};
// Materialise the constants once, opaque to the compiler, so the loop does
// not rebuild them per use.
__device__ __forceinline__ Unpack unpack_consts() {
  Unpack u;
  asm volatile("s_mov_b32 %0, 0x000f000f" : "=s"(u.lo));
  asm volatile("s_mov_b32 %0, 0x00f000f0" : "=s"(u.hi));
  asm volatile("s_mov_b32 %0, 0x00300030" : "=s"(u.h0));
  asm volatile("s_mov_b32 %0, 0x03000300" : "=s"(u.h1));
  asm volatile("s_mov_b32 %0, 0x00100010" : "=s"(u.b4));
  asm volatile("s_mov_b32 %0, 0x01000100" : "=s"(u.b8));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(u.magic));
  return u;
}

__device__ __forceinline__ half8_t pack8(half2_t h0, half2_t h1, half2_t h2, half2_t h3) {
  half8_t r;
  r[0] = h0[0]; r[1] = h0[1]; r[2] = h1[0]; r[3] = h1[1];
  r[4] = h2[0]; r[5] = h2[1]; r[6] = h3[0]; r[7] = h3[1];
  return r;
}
__device__ __forceinline__ half2_t h2c(float v) { return (half2_t){(_Float16)v, (_Float16)v}; }

// Q4_0: 8 nibbles -> 8 f16 weights (n - 8) * d.  (n - 8) is exact; the
// product with the block scale is the one rounding.
__device__ __forceinline__ half8_t unpack8_q4(uint32_t q, const Unpack &u, half2_t dd) {
  const uint32_t q2 = q >> 8;
  const uint32_t t0 = and_or(q, u.lo, u.magic);    // 1024 + n0, 1024 + n4
  const uint32_t t1 = and_or(q, u.hi, u.magic);    // 1024 + 16 n1, 1024 + 16 n5
  const uint32_t t2 = and_or(q2, u.lo, u.magic);   // 1024 + n2, 1024 + n6
  const uint32_t t3 = and_or(q2, u.hi, u.magic);   // 1024 + 16 n3, 1024 + 16 n7
  const half2_t h0 = (__builtin_bit_cast(half2_t, t0) - h2c(1032.f)) * dd;
  const half2_t h1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t1), h2c(0.0625f), h2c(-72.f)) * dd;
  const half2_t h2 = (__builtin_bit_cast(half2_t, t2) - h2c(1032.f)) * dd;
  const half2_t h3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t3), h2c(0.0625f), h2c(-72.f)) * dd;
  return pack8(h0, h1, h2, h3);
}

// Q4_1 (w = n*d + m): the nibble extraction of unpack8_q4, n exact, then
// one fma per pair, rounded once to f16.
__device__ __forceinline__ half8_t unpack8_q41(uint32_t q, const Unpack &u, half2_t dd, half2_t mm) {
  const uint32_t q2 = q >> 8;
  const uint32_t t0 = and_or(q, u.lo, u.magic);    // 1024 + n0, 1024 + n4
  const uint32_t t1 = and_or(q, u.hi, u.magic);    // 1024 + 16 n1, 1024 + 16 n5
  const uint32_t t2 = and_or(q2, u.lo, u.magic);
  const uint32_t t3 = and_or(q2, u.hi, u.magic);
  const half2_t n0 = __builtin_bit_cast(half2_t, t0) - h2c(1024.f);
  const half2_t n1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t1), h2c(0.0625f), h2c(-64.f));
  const half2_t n2 = __builtin_bit_cast(half2_t, t2) - h2c(1024.f);
  const half2_t n3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t3), h2c(0.0625f), h2c(-64.f));
  return pack8(__builtin_elementwise_fma(n0, dd, mm), __builtin_elementwise_fma(n1, dd, mm),
               __builtin_elementwise_fma(n2, dd, mm), __builtin_elementwise_fma(n3, dd, mm));
}

// Q5_K (w = q*D + M, D = d*sc, M = -dmin*m, q = 5 bits): the nibble
// extraction of unpack8_q4 with the fifth bit ORed in (ha = h >> m,
// hb = h >> (8 + m), hc = h << (8 - m) for K run m), q exact, then one fma.
__device__ __forceinline__ half8_t unpack8_q5(uint32_t q, uint32_t ha, uint32_t hb, uint32_t hc, const Unpack &u,
                                              half2_t dd, half2_t mm) {
  const uint32_t q2 = q >> 8;
  const uint32_t t0 = and_or(ha, u.b4, and_or(q, u.lo, u.magic));    // 1024 + q0, 1024 + q4
  const uint32_t t1 = and_or(ha, u.b8, and_or(q, u.hi, u.magic));    // 1024 + 16 q1, 1024 + 16 q5
  const uint32_t t2 = and_or(hb, u.b4, and_or(q2, u.lo, u.magic));
  const uint32_t t3 = and_or(hc, u.b8, and_or(q2, u.hi, u.magic));
  const half2_t n0 = __builtin_bit_cast(half2_t, t0) - h2c(1024.f);
  const half2_t n1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t1), h2c(0.0625f), h2c(-64.f));
  const half2_t n2 = __builtin_bit_cast(half2_t, t2) - h2c(1024.f);
  const half2_t n3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t3), h2c(0.0625f), h2c(-64.f));
  return pack8(__builtin_elementwise_fma(n0, dd, mm), __builtin_elementwise_fma(n1, dd, mm),
               __builtin_elementwise_fma(n2, dd, mm), __builtin_elementwise_fma(n3, dd, mm));
}

// Q6_K: low nibbles as Q4_0 plus the 2 high bits of each weight, laid out in
// `h` so that one masked OR drops them above the nibble: weight e's bits sit
// at 4-5 / 20-21 (e = 0, 1), 8-9 / 24-25 (e = 2, 3) and, after h >> 2, the
// same places for e = 4..7.  The 6-bit value is exact in f16; q6 - 32 too.
__device__ __forceinline__ half8_t unpack8_q6(uint32_t q, uint32_t h, const Unpack &u, half2_t dd) {
  const uint32_t q2 = q >> 8, hs = h >> 2;
  const uint32_t t0 = and_or(h, u.h0, and_or(q, u.lo, u.magic));    // 1024 + q6
  const uint32_t t1 = and_or(h, u.h1, and_or(q, u.hi, u.magic));    // 1024 + 16 q6
  const uint32_t t2 = and_or(hs, u.h0, and_or(q2, u.lo, u.magic));
  const uint32_t t3 = and_or(hs, u.h1, and_or(q2, u.hi, u.magic));
  const half2_t h0 = (__builtin_bit_cast(half2_t, t0) - h2c(1056.f)) * dd;
  const half2_t h1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t1), h2c(0.0625f), h2c(-96.f)) * dd;
  const half2_t h2 = (__builtin_bit_cast(half2_t, t2) - h2c(1056.f)) * dd;
  const half2_t h3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t3), h2c(0.0625f), h2c(-96.f)) * dd;
  return pack8(h0, h1, h2, h3);
}
// The high bits of K run 2r+1 are stored rotated right by 8 in the dword of
// run 2r (their bits are exactly the ones run 2r leaves free).
__device__ __forceinline__ uint32_t rotl8(uint32_t h) { return __builtin_amdgcn_alignbit(h, h, 24); }

// Q8_0: 8 bytes (stored q + 128) -> 8 f16 weights q * d.
__device__ __forceinline__ half8_t unpack8_q8(uint32_t a, uint32_t b, uint32_t magic, half2_t dd) {
  // v_perm: bytes 0-3 come from the second operand, 4-7 from the first.
  // magic = 0x64006400: bytes 5 and 7 are 0x64, the f16 exponent of 1024.
  const uint32_t t0 = __builtin_amdgcn_perm(magic, a, 0x07010500u);  // 1024 + u0, 1024 + u1
  const uint32_t t1 = __builtin_amdgcn_perm(magic, a, 0x07030502u);
  const uint32_t t2 = __builtin_amdgcn_perm(magic, b, 0x07010500u);
  const uint32_t t3 = __builtin_amdgcn_perm(magic, b, 0x07030502u);
  const half2_t h0 = (__builtin_bit_cast(half2_t, t0) - h2c(1152.f)) * dd;
  const half2_t h1 = (__builtin_bit_cast(half2_t, t1) - h2c(1152.f)) * dd;
  const half2_t h2 = (__builtin_bit_cast(half2_t, t2) - h2c(1152.f)) * dd;
  const half2_t h3 = (__builtin_bit_cast(half2_t, t3) - h2c(1152.f)) * dd;
  return pack8(h0, h1, h2, h3);
}

// f16 in the low (hi = false) or high half of `w`, broadcast to both halves.
__device__ __forceinline__ half2_t bcast_half(uint32_t w, bool hi) {
  return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(w, w, hi ? 0x03020302u : 0x01000100u));
}
// Two int8 (stored + 128) in bytes b, b+1 of w -> f16 pair, exactly.
__device__ __forceinline__ half2_t i8pair(uint32_t w, uint32_t magic, bool upper) {
  const uint32_t t = __builtin_amdgcn_perm(magic, w, upper ? 0x07030502u : 0x07010500u);
  return __builtin_bit_cast(half2_t, t) - h2c(1152.f);
}


constexpr int TILES = Q4_ST_TILES;  // tiles per round: one super-tile per stream
// A per-lane buffer offset past any activation range: the load returns zeros.
constexpr uint32_t kPastRange = 0xFFFFFFE0u;
struct GemvParams {
  const uint8_t *w;    // super-tiled weights, round-major: super-tile (st, rg, side) at ((st*nrg + rg)*nsw + side)
  uint32_t wbytes;     // bytes of the tiled weights (buffer range)
  int nsw;             // sides stored per super-tile position (1 or 2)
  int side0;           // first side computed (NS == 1)
  int M, nrg, nst;
  // Workgroups [0, nsplit) each take one piece of a split row tile: piece
  // i % S (rounds (i % S) * rps ..) of tile tile0 + i / S.  The others take
  // whole row tiles 0, 1, ...
  int nsplit, S, rps, tile0;
  const _Float16 *xh;  // activations f16 [B][K]
  uint32_t xbytes;     // buffer range of the activations: columns >= B read as zero
  const float *xf;     // XN: f32 rows [c*xfs + k], converted to f16 while staging
  int xfs;
  // Post-scale (f16 operand w * x, x not yet normalised): output column c is
  // multiplied by 1 / sqrt(sum_p pss[p][c] / K + eps).
  const float *pss;
  int pnpart;
  float eps;
  int K, B;
  float *part;         // split-K partials
  int ncu;             // compute units of the device
  int *cnt;            // per split-tile arrival counters (zero between launches)
  GemvOut out;
};

// 8 f32 activations -> 8 f16, rounded to nearest.
__device__ __forceinline__ uint4 cvt8(const uint4 (&x)[2]) {
  const float4 x0 = __builtin_bit_cast(float4, x[0]), x1 = __builtin_bit_cast(float4, x[1]);
  const half2_t h0 = {(_Float16)x0.x, (_Float16)x0.y}, h1 = {(_Float16)x0.z, (_Float16)x0.w};
  const half2_t h2 = {(_Float16)x1.x, (_Float16)x1.y}, h3 = {(_Float16)x1.z, (_Float16)x1.w};
  return make_uint4(__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1),
                    __builtin_bit_cast(uint32_t, h2), __builtin_bit_cast(uint32_t, h3));
}

// 1 / rms of a column from its npart partial sums of squares: lane l adds
// partials l, l + 64, ... in order, then one DPP tree over the wave, so every
// launch and every block size gets the same scale.  Loads past npart return
// zeros.
struct PostParts {
  float v[CWEN_MAX_PARTS / 64];
};
__device__ __forceinline__ void post_load(PostParts &q, const float *pp, int npart, int lane) {
  const __amdgpu_buffer_rsrc_t r = make_rsrc(pp, (uint32_t)npart * 4);
#pragma unroll
  for (int j = 0; j < CWEN_MAX_PARTS / 64; ++j)
    q.v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4 + j * 256, 0, 0));
}
__device__ __forceinline__ float post_scale(const PostParts &q, float K, float eps) {
  float t = q.v[0];
#pragma unroll
  for (int j = 1; j < CWEN_MAX_PARTS / 64; ++j) t += q.v[j];
  return 1.f / sqrtf(sum64(t) / K + eps);
}

// GatedDeltaNet conv rows (CONV epilogue): lane (g, n) holds positions 4g ..
// 4g+3 of channel `row`; positions 4g-3 .. 4g-1 come from lane (g-1, n), or
// for g = 0 from the history slot the block starts from (h).
__device__ __forceinline__ void conv_store(const GemvOut &o, floatx4_t res, const float (&h)[3], float4 w, int cur, int P,
                                           int row, int lane, int g, int B, bool store) {
  const float p1 = __shfl(res[1], lane - 16), p2 = __shfl(res[2], lane - 16), p3 = __shfl(res[3], lane - 16);
  if (!store) return;
  const size_t hf = (size_t)o.cv_C * 3;
  const float a[7] = {g == 0 ? h[0] : p1, g == 0 ? h[1] : p2, g == 0 ? h[2] : p3, res[0], res[1], res[2], res[3]};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int b = g * 4 + e;
    if (b >= B) continue;
    const float x = conv4(a[e], a[e + 1], a[e + 2], a[e + 3], w);
    o.cv_xc[((size_t)P * CWEN_BMAX + b) * o.cv_C + row] = silu_f(x);
    float *hs = o.cv_H + (size_t)((cur + 1 + b) % o.cv_nslot) * hf + (size_t)row * 3;
    hs[0] = a[e + 1];
    hs[1] = a[e + 2];
    hs[2] = a[e + 3];
  }
}

}  // namespace
