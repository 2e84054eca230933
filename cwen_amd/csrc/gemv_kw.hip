// Batched quantized GEMV for few rows: one 16-row group per workgroup, K split
// over its waves.  Semantics, formats and arithmetic as in gemv.hip.
#include <algorithm>

#include "cwen_internal.h"
#include "gemv_tile.h"

namespace {

constexpr int KW_MAX = GEMV_KW_MAX;   // pieces of K at most

// The few-row form: a launch with at most half as many 64-row tiles as CUs
// (out-projections, down, small matrices) leaves most CUs idle with whole tiles
// and pays a hand-off between workgroups when a tile's K is split over several
// (2.5-2.9 us of a 9-15 us launch: partials out, arrival counter, partials in).
// Here a workgroup takes one 16-row group (for SwiGLU both sides of the pair) and its S
// waves (per side) the S pieces of K, rps rounds each; the pieces meet in LDS and
// are added in piece order, so the sums are those of the split described by
// GemvGrid.  A wave shares nothing with the others before that: it stages its
// own activations, half a round (256 K) at a time, in its own LDS, with no
// barrier in the loop, and keeps one round of weights in flight while it
// computes another.  The residual, the norm weight and the conv's history are
// requested before the loop.
// Measured against the split over workgroups (us, f16 / f32 activations of the
// caller; medians):
//   Q4_0 1000 x 2080  B = 1   6.5 -> 4.4        Q4_0 2048 x 6144  B = 4  7.4 -> 5.2
//   Q4_0 5120 x 5120  B = 1   8.0 -> 7.05       Q8_0 3001 x 4128  B = 5  9.3 -> 6.4
//   Q4_0 8000 x 2048  B = 4   7.2 -> 4.8        Q4_0 6144 x 4096  B = 16 9.0 -> 7.2
//   k/v pair 1024 x 5120  B = 16  9.1 -> 7.1    FFN 2048 x 5632  B = 16  17.1 -> 15.7
// What is left at these sizes is the launch, one round trip to memory for the
// first round of weights and one for the sums: 2-3 us before the first MFMA.
template <int FMT, int NS, int EPI, int CB, bool XN, int RGW>
__global__ __launch_bounds__(64 * KW_MAX * NS) void gemv_kw_kernel(GemvParams p) {
  using F = Fmt<FMT>;
  constexpr int TV = F::TV;
  constexpr int HU = 32;                       // 16-byte units of a column's half round
  constexpr bool DM = FMT == GEMV_Q41 || FMT == GEMV_Q5K;
  using ScT = std::conditional_t<DM, uint4, uint2>;
  extern __shared__ __align__(16) uint4 lds[];  // [waves][CB * HU] activations, then [waves][64] sums
  __shared__ float s_psc[CWEN_BMAX];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwave = (int)blockDim.x >> 6, S = p.S;
  const int n = lane & 15, g = lane >> 4;
  const int rg0 = blockIdx.x * RGW;            // first row group
  const int rg = rg0 + (RGW > 1 ? min(wave, RGW - 1) : 0), row = rg * Q4_ROWS + n;   // of the epilogue
  const int sp = NS == 2 ? wave % S : wave;
  const int side = NS == 2 ? wave / S : EPI == GEMV_EPI_PAIR ? (int)blockIdx.y : p.side0;
  const int st0 = sp * p.rps;
  const int nround = min(p.nst - st0, p.rps);
  uint4 *const act = lds + wave * CB * HU;
  floatx4_t *const red = (floatx4_t *)(lds + nwave * CB * HU);

  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, p.wbytes);
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(XN ? (const void *)p.xf : (const void *)p.xh, p.xbytes);
  const uint32_t sstride = (uint32_t)p.nrg * p.nsw * F::ST_BYTES;
  uint32_t wofs[RGW];
#pragma unroll
  for (int k = 0; k < RGW; ++k)   // a row group past the last one reads that one
    wofs[k] = (((uint32_t)st0 * p.nrg + min(rg0 + k, p.nrg - 1)) * p.nsw + side) * F::ST_BYTES;

  struct Round {
    uint4 q[TILES][TV];
    ScT sc;
    uint4 h5, hq[2];
    uint32_t dq;
  };
  auto load_round = [&](Round (&ws)[RGW], int r) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < RGW; ++k) {
      Round &w = ws[k];
      const uint32_t so = wofs[k] + (uint32_t)r * sstride;
      if constexpr (DM) w.sc = bload16_nt(wr, F::SC_OFS + lane * 16, so);
      else w.sc = bload8_nt(wr, F::SC_OFS + lane * 8, so);
      if constexpr (FMT == GEMV_Q6K) w.dq = bload4_nt(wr, F::D_OFS + n * 4, so);
      if constexpr (FMT == GEMV_Q5K) w.h5 = bload16_nt(wr, F::HI_OFS + lane * 16, so);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int v = 0; v < TV; ++v) w.q[t][v] = bload16_nt(wr, lane * 16 + t * (1024 * TV) + v * 1024, so);
        if constexpr (FMT == GEMV_Q6K) {
          if (t & 1) w.hq[t >> 1] = bload16_nt(wr, F::HI_OFS + (t >> 1) * 1024 + lane * 16, so);
        }
      }
    }
  };
  // Activations of half round h: lane (c2, u) of load i takes unit u (8 K) of
  // column 2 i + c2.  LDS unit c * 32 + (u' ^ (c & 15)), u' = u with bits 2-3
  // negated (see wide.hip: 16-byte reads without bank conflicts).  Units past K
  // and columns past B read as zeros.  The LDS is this wave's own and served in
  // order; wave_fence keeps the compiler from moving a lane's reads past the
  // writes that other lanes made for it.
  const int xc = lane >> 5, xu = lane & 31;
  const int xp = (xu & 16) | (((4 - ((xu >> 2) & 3)) & 3) << 2) | (xu & 3);
  constexpr int XL = CB / 2;                   // staging loads per half round (two columns each)
  constexpr uint32_t XE = XN ? 4 : 2;
  const uint32_t xcol = (uint32_t)(XN ? p.xfs : p.K) * XE;
  uint4 xs[XL][XN ? 2 : 1];
  auto stage_load = [&](int h) __attribute__((always_inline)) {
    const int k = st0 * Q4_ST_K + h * 256 + xu * 8;
#pragma unroll
    for (int i = 0; i < XL; ++i) {   // the column stays in the offset that is range-checked
      const uint32_t vo = k < p.K ? (uint32_t)(xc + 2 * i) * xcol + (uint32_t)k * XE : kPastRange;
      xs[i][0] = bload16(xr, vo);
      if constexpr (XN) xs[i][1] = bload16(xr, vo + 16);
    }
  };
  auto stage_store = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int c = 2 * i + xc;
      if constexpr (XN) act[c * HU + (xp ^ (c & 15))] = cvt8(xs[i]);
      else act[c * HU + (xp ^ (c & 15))] = xs[i][0];
    }
  };

  auto wave_fence = []() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
  };

  stage_load(0);
  Round wa[RGW], wb[RGW];
  load_round(wa, 0);
  __builtin_amdgcn_sched_barrier(0);
  // What the epilogue (wave k < RGW: row group k) needs.
  const GemvOut &o = p.out;
  const bool fin = wave < RGW;
  float *const y0 = (EPI == GEMV_EPI_PAIR && side == 1) ? o.y1 : o.y;
  const bool row_ok = rg < p.nrg && row < p.M;
  float old[4] = {0.f, 0.f, 0.f, 0.f}, nwr = 1.f;
  int cv_cur = 0, cv_P = 0;
  float cv_h[3] = {0.f, 0.f, 0.f};
  float4 cv_w4 = {0.f, 0.f, 0.f, 0.f};
  const bool cv_rows = EPI == GEMV_EPI_CONV && rg * Q4_ROWS < o.cv_C;
  if (fin && row_ok) {
    if (o.yh && o.nwh) nwr = o.nwh[row];
    if (y0 && o.accumulate) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (g * 4 + e < p.B) old[e] = y0[(size_t)(g * 4 + e) * o.ys + row];
    }
    if constexpr (EPI == GEMV_EPI_CONV) {
      cv_cur = o.cv_ctl[0];
      cv_P = o.cv_ctl[3];
      if (cv_rows) {
        cv_w4 = *(const float4 *)(o.cv_w + (size_t)row * 4);
        if (g == 0) {
          const float *hin = o.cv_H + (size_t)cv_cur * o.cv_C * 3 + (size_t)row * 3;
          cv_h[0] = hin[0];
          cv_h[1] = hin[1];
          cv_h[2] = hin[2];
        }
      }
    }
  }
  if (p.pss)
    for (int c = wave; c < p.B; c += nwave) {
      PostParts q;
      post_load(q, p.pss + c * CWEN_MAX_PARTS, p.pnpart, lane);
      const float sc = post_scale(q, (float)p.K, p.eps);
      if (lane == 0) s_psc[c] = sc;
    }

  const Unpack uc = unpack_consts();
  floatx4_t acc[RGW][2];
#pragma unroll
  for (int k = 0; k < RGW; ++k) acc[k][0] = acc[k][1] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
  const int nn = n & (CB - 1);                 // columns past CB repeat staged ones: their outputs are discarded
  int aslot[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) aslot[m] = nn * HU + ((4 * ((4 - g) & 3) + m) ^ nn);

  auto round = [&](int rd, Round (&cur)[RGW], Round (&next)[RGW]) __attribute__((always_inline)) {
    if (rd + 1 < nround) load_round(next, rd + 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wave_fence();
      stage_store();
      wave_fence();
      if (2 * rd + h + 1 < 2 * nround) stage_load(2 * rd + h + 1);
#pragma unroll
      for (int t = 2 * h; t < 2 * h + 2; ++t) {
        half8_t a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = __builtin_bit_cast(half8_t, act[(t & 1) * 16 + aslot[m]]);
#pragma unroll
        for (int k = 0; k < RGW; ++k) {
          const Round &w = cur[k];
          half2_t d0, d1;
          if constexpr (FMT == GEMV_Q6K) {
            const half2_t ds = i8pair(t < 2 ? w.sc.x : w.sc.y, uc.magic, t & 1) * bcast_half(w.dq, t >= 2);
            d0 = (half2_t){ds[0], ds[0]};
            d1 = (half2_t){ds[1], ds[1]};
          } else if constexpr (DM) {
            const uint32_t v = t == 0 ? w.sc.x : t == 1 ? w.sc.y : t == 2 ? w.sc.z : w.sc.w;
            d0 = bcast_half(v, false);
            d1 = bcast_half(v, true);
          } else {
            d0 = d1 = bcast_half(t < 2 ? w.sc.x : w.sc.y, (t & 1) != 0);
          }
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const uint32_t qm = m == 0 ? w.q[t][0].x : m == 1 ? w.q[t][0].y : m == 2 ? w.q[t][0].z : w.q[t][0].w;
            half8_t b;
            if constexpr (FMT == GEMV_Q4) {
              b = unpack8_q4(qm, uc, d0);
            } else if constexpr (FMT == GEMV_Q41) {
              b = unpack8_q41(qm, uc, d0, d1);
            } else if constexpr (FMT == GEMV_Q5K) {
              const uint32_t v = t == 0 ? w.h5.x : t == 1 ? w.h5.y : t == 2 ? w.h5.z : w.h5.w;
              b = unpack8_q5(qm, v >> m, v >> (8 + m), v << (8 - m), uc, d0, d1);
            } else if constexpr (FMT == GEMV_Q6K) {
              const uint4 &h4 = w.hq[t >> 1];
              const uint32_t v = (t & 1) ? (m < 2 ? h4.z : h4.w) : (m < 2 ? h4.x : h4.y);
              b = unpack8_q6(qm, (m & 1) ? rotl8(v) : v, uc, m < 2 ? d0 : d1);
            } else {
              const uint4 &q = w.q[t][TV == 2 ? m >> 1 : 0];
              b = (m & 1) ? unpack8_q8(q.z, q.w, uc.magic, d0) : unpack8_q8(q.x, q.y, uc.magic, d0);
            }
            acc[k][m & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b, acc[k][m & 1], 0, 0, 0);
          }
        }
      }
    }
  };
  int rd = 0;
  for (; rd + 1 < nround; rd += 2) {
    round(rd, wa, wb);
    round(rd + 1, wb, wa);
  }
  if (rd < nround) round(rd, wa, wb);

#pragma unroll
  for (int k = 0; k < RGW; ++k) red[(k * nwave + wave) * 64 + lane] = acc[k][0] + acc[k][1];
  __syncthreads();
  if (!fin) return;
  auto pieces = [&](int s) __attribute__((always_inline)) {
    floatx4_t r = (floatx4_t){0.f, 0.f, 0.f, 0.f};
    if (S == 1) return red[s * 64 + lane];
    for (int k = 0; k < S; ++k) r += red[(s * S + k) * 64 + lane];
    return r;
  };
  floatx4_t res = pieces(RGW > 1 ? wave : 0), up = res;   // sums of side or row group s
  if constexpr (EPI == GEMV_EPI_SWIGLU) up = pieces(1);
  if (p.pss) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sc = g * 4 + e < p.B ? s_psc[g * 4 + e] : 1.f;
      res[e] *= sc;
      up[e] *= sc;
    }
  }
  bool store = row_ok;
  if constexpr (EPI == GEMV_EPI_CONV) {
    if (cv_rows) {
      conv_store(o, res, cv_h, cv_w4, cv_cur, cv_P, row, lane, g, p.B, store);
      store = false;
    }
  }
  float sq[4] = {0.f, 0.f, 0.f, 0.f};
  bool bad = false;
  if (store) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = g * 4 + e;
      if (c >= p.B) continue;
      float v = EPI == GEMV_EPI_SWIGLU ? silu_f(res[e]) * up[e] : res[e];
      if (y0 && o.accumulate) v += old[e];
      if (y0) y0[(size_t)c * o.ys + row] = v;
      if (o.yh) {
        const _Float16 h = (_Float16)f32_of(o.nwh ? v * nwr : v);
        o.yh[(size_t)c * p.M + row] = h;
        bad |= f16_bad(h);
      }
      sq[e] = f32_of(v * v);
    }
  }
  if (bad) raise_flag(o.rflag);
  if (o.ssq) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = sum16(sq[e]);
      if (n == 0 && rg < p.nrg && g * 4 + e < p.B) o.ssq[(g * 4 + e) * CWEN_MAX_PARTS + rg] = t;
    }
  }
}

size_t kw_lds(int nwave, int cb, int rgw) { return (size_t)nwave * ((size_t)cb * 512 + 1024 * rgw); }

template <int FMT, int NS, int EPI, int CB, bool XN>
int launch_one(const GemvParams &p, hipStream_t st) {
  const int nwave = p.S * NS;
  const dim3 block(64u * nwave), grid1((unsigned)p.nrg, EPI == GEMV_EPI_PAIR ? 2u : 1u);
  static_assert(CB * NS <= 16 || (FMT == GEMV_Q4 && NS == 2 && CB == 16), "LDS above 64 KB: see gemv_kw_init");
  // Wide blocks over more row groups than CUs: two row groups per wave, which
  // share its staged activations (5120 x 5120, f16, B = 16: 8.4 against 8.2-9.8 us,
  // unsteady); at B <= 4 the halved workgroup count costs more (4224 x 5120, f32, B = 3,
  // weights from HBM: 8.6 against 8.1), except for f32 activations with weights other than
  // Q4_0 (4224 x 3072 at B = 4, Q5_K 7.2 against 8.0, Q6_K 7.3 against 8.4; 4200 x 3072 Q8_0 7.1
  // against 7.9, weights in cache).  A pair's two sides never exceed the CUs here.
  if constexpr (NS == 1 && EPI != GEMV_EPI_PAIR && !(CB == 16 && XN) && (CB >= 8 || (CB == 4 && XN && FMT != GEMV_Q4))) {
    if (p.S > 1 && (int)(grid1.x * grid1.y) > p.ncu) {
      const dim3 grid2((unsigned)((p.nrg + 1) / 2), grid1.y);
      hipLaunchKernelGGL((gemv_kw_kernel<FMT, NS, EPI, CB, XN, 2>), grid2, block, kw_lds(nwave, CB, 2), st, p);
      return CWEN_OK;
    }
  }
  hipLaunchKernelGGL((gemv_kw_kernel<FMT, NS, EPI, CB, XN, 1>), grid1, block, kw_lds(nwave, CB, 1), st, p);
  return CWEN_OK;
}

template <int FMT, int NS, int EPI>
int launch_cb(const GemvParams &p, hipStream_t st) {
  if (p.xf) {
    if constexpr (EPI == GEMV_EPI_CONV) {
      return CWEN_EINVAL;      // the model's operands are f16
    } else {
      if (p.B <= 2) return launch_one<FMT, NS, EPI, 2, true>(p, st);
      if (p.B <= 4) return launch_one<FMT, NS, EPI, 4, true>(p, st);
      if (p.B <= 8) return launch_one<FMT, NS, EPI, 8, true>(p, st);
      if constexpr (NS == 1) return launch_one<FMT, NS, EPI, 16, true>(p, st);
      else return CWEN_EINVAL;   // converted first: see f32_staged
    }
  }
  if (p.B <= 2) return launch_one<FMT, NS, EPI, 2, false>(p, st);
  if (p.B <= 4) return launch_one<FMT, NS, EPI, 4, false>(p, st);
  if (p.B <= 8) return launch_one<FMT, NS, EPI, 8, false>(p, st);
  return launch_one<FMT, NS, EPI, 16, false>(p, st);
}

}  // namespace

// The instance whose workgroups may hold more than 64 KB of LDS.
int gemv_kw_init() {
  CWEN_HIP_TRY(hipFuncSetAttribute((const void *)gemv_kw_kernel<GEMV_Q4, 2, GEMV_EPI_SWIGLU, 16, false, 1>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kw_lds(2 * KW_MAX, 16, 1)));
  return CWEN_OK;
}

int gemv_kw_launch(int fmt, int epi, const void *params, hipStream_t st) {
  const GemvParams &p = *(const GemvParams *)params;
  if (p.S < 1 || p.S > KW_MAX) return CWEN_EINVAL;
  int rc = CWEN_EINVAL;
  if (epi == GEMV_EPI_SWIGLU) {
    if (fmt == GEMV_Q4) rc = launch_cb<GEMV_Q4, 2, GEMV_EPI_SWIGLU>(p, st);
  } else if (epi == GEMV_EPI_PAIR) {
    if (fmt == GEMV_Q4) rc = launch_cb<GEMV_Q4, 1, GEMV_EPI_PAIR>(p, st);
  } else if (epi == GEMV_EPI_CONV) {
    if (fmt == GEMV_Q4) rc = launch_cb<GEMV_Q4, 1, GEMV_EPI_CONV>(p, st);
  } else if (epi == GEMV_EPI_STORE) {
    switch (fmt) {
      case GEMV_Q4: rc = launch_cb<GEMV_Q4, 1, GEMV_EPI_STORE>(p, st); break;
      case GEMV_Q6K: rc = launch_cb<GEMV_Q6K, 1, GEMV_EPI_STORE>(p, st); break;
      case GEMV_Q8: rc = launch_cb<GEMV_Q8, 1, GEMV_EPI_STORE>(p, st); break;
      case GEMV_Q41: rc = launch_cb<GEMV_Q41, 1, GEMV_EPI_STORE>(p, st); break;
      case GEMV_Q5K: rc = launch_cb<GEMV_Q5K, 1, GEMV_EPI_STORE>(p, st); break;
      default: break;
    }
  }
  if (rc) return rc;
  CWEN_HIP_TRY(hipGetLastError());
  return CWEN_OK;
}
