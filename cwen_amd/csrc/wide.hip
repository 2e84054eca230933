// Quantized matrix products for many positions at once (a prompt's prefill):
// Y[b][i] = sum_k w_ik X[b][k] for b < N, N up to WIDE_MAX, from the same
// super-tiled weights as gemv.hip and with its arithmetic, so a position
// computed here is bit for bit the position gemv_kernel computes in a block.
//
// Reference semantics: prefill_forward's matrix products (run.c:4823-4857,
// through gemvb, run.c:1577-1680).
//
// What must match gemv_kernel for that: every product is a
// v_mfma_f32_16x16x32_f16 over the same 32 K (MFMA m of a tile: K run m of
// each lane's block), products 0 and 2 of a tile add to one accumulator, 1
// and 3 to another, over the tiles in order; the two are added at the end of
// a piece, and the pieces of a row tile that gemv_kernel splits over K (the
// weight's GemvGrid) are added in piece order.
//
// Design (gfx950).  A block of 16 positions re-reads every weight, so a
// prompt in such blocks is bound by HBM (4096 positions: 256 sweeps).  Here a
// workgroup of 4 waves takes SPW weight streams of 16 rows per wave and 64
// positions: the quantized bytes go from memory to registers and are unpacked
// there, once per 64 positions; the activations are staged in LDS 128 K at
// a time (double-buffered), shared by the 4 waves.  With SPW = 4 a wave issues
// 64 MFMAs (1024 matrix-core cycles) per 128 K against 224 VALU operations of
// unpacking (896 cycles) and 16 KB of LDS reads; two workgroups per CU overlap
// them.  128 accumulator registers per lane leave no room for a second set of
// operands: with 8 position tiles and one workgroup per CU the compiler spilled
// loads in flight (739 us for gate/up below), and 8 position tiles of 2 streams,
// half the unpacking per product, came to the same time as this (395 us).
// Measured, gate/up 2 x 17408 x 5120 at 1024 positions: 392-408 us, 0.90-0.93 PFLOP/s
// (a library f16 product of 8192^3 on the same card: 1.18).  4096 positions at
// 4 layers of the 27B shape: 97 ms in blocks of 16, 20.6 ms in passes of 1024.
// The registers fit Q4_0 (2 spilled).  With SPW = 4 the other formats spill: Q4_1 42, Q8_0 59,
// Q5_K 99, Q6_K 115 registers a lane.  The same prompt with Q5_K out- and Q4_1
// down-projections takes 24.6 ms (98.5 in blocks), with Q8_0 and Q6_K 29.7 (102).
#include <algorithm>

#include "cwen_internal.h"
#include "gemv_tile.h"

namespace {

constexpr int WW = 4;                // waves per workgroup
constexpr int TG = 4;                // row groups of a single-sided row tile of gemv_kernel

struct WideParams {
  const uint8_t *w;
  uint32_t wbytes;
  int nrg, nst, M;
  const _Float16 *xh;                // activations, wide_at order
  int K, N, npt;                     // npt: position tiles (16 P positions each)
  int items, perA, perB;             // row items x npt; whole items and pieces per XCD
  // Row items: nA row blocks computed whole, covering row groups [0, rgB);
  // then the row blocks of [rgB, nrg), S pieces of rps rounds each, whose
  // sums go to `part` [piece][side][N][rowsB].
  int nA, rgB, S, rps;
  float *part;
  int rowsB;
  const float *psc;                  // per-position output scale, nullable
  float *y; int ys;                  // STORE
  _Float16 *yh;                      // SWIGLU [N][M]
  int *rflag;
};

// The quantized bytes of one 16-row x 128-K tile of a stream, per lane.
template <int FMT> struct TileRegs {
  uint4 q[Fmt<FMT>::TV];
  uint2 hi;                          // Q6_K high bits; Q5_K fifth bits in .x
};

template <int FMT, int NS, int EPI, int SPW, int P>
__global__ __launch_bounds__(64 * WW, P * SPW > 16 ? 1 : 2) void wide_kernel(WideParams p) {
  using F = Fmt<FMT>;
  constexpr int RGW = SPW / NS;      // row groups per wave
  constexpr bool DM = FMT == GEMV_Q41 || FMT == GEMV_Q5K;
  using ScT = std::conditional_t<DM, uint4, uint2>;
  __shared__ uint4 act[2][P * 256];  // [buf][position][unit ^ (position & 15)]

  // XCD x (workgroups x, x + 8, ...) takes a contiguous range of the whole
  // items and one of the pieces, positions fastest.
  const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
  const bool piece = j >= p.perA;
  const int it = piece ? p.nA * p.npt + x * p.perB + j - p.perA : x * p.perA + j;
  if (it >= (piece ? p.items : p.nA * p.npt)) return;
  const int pt = it % p.npt, item = it / p.npt;
  const int sp = piece ? (item - p.nA) % p.S : 0;
  const int rb = piece ? (item - p.nA) / p.S : item;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int rg0 = (piece ? p.rgB : 0) + (rb * WW + wave) * RGW;   // this wave's first row group
  const int rgend = piece ? p.nrg : p.rgB;
  const int r0 = sp * p.rps;
  const int nround = piece ? min(p.nst - r0, p.rps) : p.nst;
  const int ntile = nround * Q4_ST_TILES;

  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, p.wbytes);
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.xh, (uint32_t)((size_t)p.N * p.K * 2));
  const uint32_t sstride = (uint32_t)p.nrg * NS * F::ST_BYTES;
  uint32_t wofs[SPW];
#pragma unroll
  for (int s = 0; s < SPW; ++s) {
    const int rg = min(rg0 + s / NS, p.nrg - 1);   // idle streams read a valid tile
    wofs[s] = (((uint32_t)r0 * p.nrg + rg) * NS + s % NS) * F::ST_BYTES;
  }

  // Activations: thread t stages LDS unit t & 15 of positions
  // (t >> 4) + 16 i of the tile's positions, 256 contiguous bytes each; those
  // past N read the next tile's first positions, or zeros past the buffer:
  // their sums are never stored.
  // LDS unit of K unit u of position c: c * 16 + (u' ^ (c & 15)), u' = u with
  // its upper two bits negated.  A 16-byte LDS read serves 16 lanes at a time,
  // lanes 0-3, 12-15, 20-23 and 24-27 first: with this order they meet 16
  // different units (u ^ c gave a 2-way conflict on every operand read).
  const int xu = (tid & 15) ^ (tid >> 4);
  const uint32_t xofs = (uint32_t)(pt * 16 * P + (tid >> 4)) * 256 + ((((4 - (xu >> 2)) & 3) << 2) | (xu & 3)) * 16;
  const uint32_t xtile = (uint32_t)p.N * 256, xof0 = (uint32_t)r0 * 4 * xtile;
  uint4 xa[P];
  auto act_load = [&](int t) __attribute__((always_inline)) {
    const uint32_t so = xof0 + (uint32_t)min(t, ntile - 1) * xtile;
#pragma unroll
    for (int i = 0; i < P; ++i) xa[i] = bload16(xr, xofs + i * 4096, so);
  };
  auto act_store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < P; ++i) act[buf][tid + 256 * i] = xa[i];
  };
  TileRegs<FMT> wq[2][SPW];
  auto tile_load = [&](int b, int t) __attribute__((always_inline)) {
    t = min(t, ntile - 1);
    const int u = t & 3;
    const uint32_t so = (uint32_t)(t >> 2) * sstride;
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
#pragma unroll
      for (int v = 0; v < F::TV; ++v)
        wq[b][s].q[v] = bload16(wr, lane * 16 + v * 1024, wofs[s] + so + u * (1024 * F::TV));
      if constexpr (FMT == GEMV_Q6K)
        wq[b][s].hi = bload8_nt(wr, lane * 16, wofs[s] + so + F::HI_OFS + (u >> 1) * 1024 + (u & 1) * 8);
      if constexpr (FMT == GEMV_Q5K) wq[b][s].hi.x = bload4_nt(wr, lane * 16, wofs[s] + so + F::HI_OFS + u * 4);
    }
  };
  ScT sc[SPW];
  uint32_t dq[SPW] = {};
  auto sc_load = [&](ScT (&d)[SPW], uint32_t (&dd)[SPW], int r) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)min(r, nround - 1) * sstride;
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      if constexpr (DM) d[s] = bload16_nt(wr, F::SC_OFS + lane * 16, wofs[s] + so);
      else d[s] = bload8_nt(wr, F::SC_OFS + lane * 8, wofs[s] + so);
      if constexpr (FMT == GEMV_Q6K) dd[s] = bload4_nt(wr, F::D_OFS + n * 4, wofs[s] + so);
    }
  };

  floatx4_t acc[P][SPW][2];
#pragma unroll
  for (int i = 0; i < P; ++i)
#pragma unroll
    for (int s = 0; s < SPW; ++s) acc[i][s][0] = acc[i][s][1] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
  const Unpack uc = unpack_consts();
  int aslot[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) aslot[m] = n * 16 + ((4 * ((4 - g) & 3) + m) ^ n);

  // Scales of tile u of the round (Q4_1 / Q5_K: scale, offset; Q6_K: per half
  // block).
  half2_t d0[SPW], d1[SPW];
  auto scales = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      if constexpr (FMT == GEMV_Q6K) {
        const half2_t s2 = i8pair(u < 2 ? sc[s].x : sc[s].y, uc.magic, u & 1);
        const half2_t ds = s2 * bcast_half(dq[s], u >= 2);
        d0[s] = (half2_t){ds[0], ds[0]};
        d1[s] = (half2_t){ds[1], ds[1]};
      } else if constexpr (DM) {
        const uint32_t w = u == 0 ? sc[s].x : u == 1 ? sc[s].y : u == 2 ? sc[s].z : sc[s].w;
        d0[s] = bcast_half(w, false);
        d1[s] = bcast_half(w, true);
      } else {
        d0[s] = d1[s] = bcast_half(u < 2 ? sc[s].x : sc[s].y, (u & 1) != 0);
      }
    }
  };
  // MFMA operand of K run m of stream s, from tile buffer tb.
  auto operand = [&](int tb, int m, int s) __attribute__((always_inline)) -> half8_t {
    const TileRegs<FMT> &w = wq[tb][s];
    const uint32_t qm = m == 0 ? w.q[0].x : m == 1 ? w.q[0].y : m == 2 ? w.q[0].z : w.q[0].w;
    if constexpr (FMT == GEMV_Q4) {
      return unpack8_q4(qm, uc, d0[s]);
    } else if constexpr (FMT == GEMV_Q41) {
      return unpack8_q41(qm, uc, d0[s], d1[s]);
    } else if constexpr (FMT == GEMV_Q5K) {
      const uint32_t h = w.hi.x;
      return unpack8_q5(qm, h >> m, h >> (8 + m), h << (8 - m), uc, d0[s], d1[s]);
    } else if constexpr (FMT == GEMV_Q6K) {
      const uint32_t h = m < 2 ? w.hi.x : w.hi.y;
      return unpack8_q6(qm, (m & 1) ? rotl8(h) : h, uc, m < 2 ? d0[s] : d1[s]);
    } else {
      const uint4 &q = w.q[m >> 1];
      return (m & 1) ? unpack8_q8(q.z, q.w, uc.magic, d0[s]) : unpack8_q8(q.x, q.y, uc.magic, d0[s]);
    }
  };

  act_load(0);
  sc_load(sc, dq, 0);
  tile_load(0, 0);
  act_store(0);
  act_load(1);
  lds_barrier();

  // One 128-K tile per step.  The scheduling barriers keep the request order
  // (activations of tile t + 2, weights of tile t + 1) and one K run's operands
  // live at a time: without them the scheduler hoists reads until Q4_0 spills too.
  for (int r = 0; r < nround; ++r) {
#pragma unroll
    for (int u = 0; u < Q4_ST_TILES; ++u) {
      const int t = r * Q4_ST_TILES + u;
      act_store((u + 1) & 1);          // tile t + 1 (its buffer's readers passed the last barrier)
      __builtin_amdgcn_sched_barrier(0);
      act_load(t + 2);
      tile_load((u + 1) & 1, t + 1);
      scales(u);
      if (u == 3) sc_load(sc, dq, r + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        half8_t a[P];
#pragma unroll
        for (int i = 0; i < P; ++i) a[i] = __builtin_bit_cast(half8_t, act[u & 1][aslot[m] + 256 * i]);
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
          const half8_t b = operand(u & 1, m, s);
#pragma unroll
          for (int i = 0; i < P; ++i)
            acc[i][s][m & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b, acc[i][s][m & 1], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      lds_barrier();
    }
  }

  bool bad = false;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int c0 = (pt * P + i) * 16 + 4 * g;      // this lane's 4 positions
    float4 sc4 = {1.f, 1.f, 1.f, 1.f};
    if (!piece && p.psc) sc4 = *(const float4 *)(p.psc + c0);
    const float scl[4] = {sc4.x, sc4.y, sc4.z, sc4.w};
#pragma unroll
    for (int k = 0; k < RGW; ++k) {
      const int rg = rg0 + k, row = rg * Q4_ROWS + n;
      if (rg >= rgend || row >= p.M) continue;
      floatx4_t v[NS];
#pragma unroll
      for (int d = 0; d < NS; ++d) v[d] = acc[i][k * NS + d][0] + acc[i][k * NS + d][1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = c0 + e;
        if (c >= p.N) continue;
        if (piece) {
#pragma unroll
          for (int d = 0; d < NS; ++d)
            p.part[((size_t)(sp * NS + d) * p.N + c) * p.rowsB + row - p.rgB * Q4_ROWS] = v[d][e];
          continue;
        }
        float o[NS];
#pragma unroll
        for (int d = 0; d < NS; ++d) o[d] = p.psc ? v[d][e] * scl[e] : v[d][e];
        if constexpr (EPI == GEMV_EPI_SWIGLU) {
          const _Float16 h = (_Float16)f32_of(silu_f(o[0]) * o[NS - 1]);
          p.yh[wide_at(c, row, p.N)] = h;
          bad |= f16_bad(h);
        } else {
          p.y[(size_t)c * p.ys + row] = o[0];
        }
      }
    }
  }
  if (bad) raise_flag(p.rflag);
}

// Rows [row0, M) from their pieces: a wave takes 64 consecutive rows (for a
// single-sided weight a row tile of gemv_kernel) of one position.
template <int NS, int EPI>
__global__ __launch_bounds__(256) void wide_finish_kernel(WideParams p, WideOut o, int row0) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.y * 4 + wave;
  if (c >= p.N) return;
  const int rl = blockIdx.x * 64 + lane, row = row0 + rl;
  const bool ok = row < p.M;
  float v[NS];
#pragma unroll
  for (int d = 0; d < NS; ++d) {
    v[d] = 0.f;
    for (int s = 0; s < p.S; ++s) v[d] += ok ? p.part[((size_t)(s * NS + d) * p.N + c) * p.rowsB + rl] : 0.f;
    if (p.psc) v[d] *= p.psc[c];
  }
  if constexpr (EPI == GEMV_EPI_SWIGLU) {
    if (!ok) return;
    const _Float16 h = (_Float16)f32_of(silu_f(v[0]) * v[NS - 1]);
    p.yh[wide_at(c, row, p.N)] = h;
    if (f16_bad(h)) raise_flag(p.rflag);
  } else {
    float r = v[0], sq = 0.f;
    if (ok) {
      if (o.accumulate) r += p.y[(size_t)c * p.ys + row];
      p.y[(size_t)c * p.ys + row] = r;
      if (o.yh) {
        const _Float16 h = (_Float16)f32_of(r * o.nwh[row]);
        o.yh[wide_at(c, row, p.N)] = h;
        if (f16_bad(h)) raise_flag(p.rflag);
      }
      sq = f32_of(r * r);
    }
    if (o.ssq) {
      sq = sum16(sq);
      if ((lane & 15) == 0 && ok) o.ssq[(size_t)c * CWEN_MAX_PARTS + row / 16] = sq;
    }
  }
}

// Per position: 1 / sqrt(sum_p ssq[c][p] / K + eps), the partials summed as
// gemv_kernel's post-scale sums them.  One wave per position.
__global__ __launch_bounds__(256) void wide_scale_kernel(const float *ssq, int npart, int K, float eps, int N, float *psc) {
  const int lane = threadIdx.x & 63, c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= N) return;
  PostParts q;
  post_load(q, ssq + (size_t)c * CWEN_MAX_PARTS, npart, lane);
  const float s = post_scale(q, (float)K, eps);
  if (lane == 0) psc[c] = s;
}

template <int FMT, int NS, int EPI, int SPW>
void launch(WideParams p, hipStream_t st) {
  constexpr int P = 4, RGB = WW * SPW / NS;
  p.npt = (p.N + 16 * P - 1) / (16 * P);
  p.nA = (p.rgB + RGB - 1) / RGB;
  p.items = (p.nA + (p.nrg - p.rgB + RGB - 1) / RGB * p.S) * p.npt;
  p.perA = (p.nA * p.npt + 7) / 8;
  p.perB = (p.items - p.nA * p.npt + 7) / 8;
  hipLaunchKernelGGL((wide_kernel<FMT, NS, EPI, SPW, P>), dim3((unsigned)(8 * (p.perA + p.perB))), dim3(64 * WW), 0, st, p);
}

}  // namespace

// Row groups [0, rgB) are computed whole, the others in pieces and finished.
static int wide_split_at(const cwen_weight *w, int nsides, bool finish) {
  const GemvGrid &g = w->cfg[nsides - 1];
  if (finish) return 0;
  return g.nsplit ? std::min(g.tile0 * (TG / nsides), w->nrg) : w->nrg;
}

bool wide_takes(const cwen_weight *w, int nsides, bool finish) {
  const GemvGrid &g = w->cfg[nsides - 1];
  return w->nside == nsides && w->ne0 % Q4_ST_K == 0 && !(nsides == 2 && w->fmt != GEMV_Q4) &&
         !(finish && g.nsplit && g.nsplit != g.grid);
}

size_t wide_partial_floats(const cwen_weight *w, int nsides, bool finish, int N) {
  const GemvGrid &g = w->cfg[nsides - 1];
  return (size_t)(g.nsplit ? g.S : 1) * nsides * N * (size_t)(w->nrg - wide_split_at(w, nsides, finish)) * Q4_ROWS;
}

int wide_scale(const float *ssq, int npart, int K, float eps, int N, float *psc, hipStream_t st) {
  hipLaunchKernelGGL(wide_scale_kernel, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, st, ssq, npart, K, eps, N, psc);
  CWEN_HIP_TRY(hipGetLastError());
  return CWEN_OK;
}

int wide_gemm(const cwen_ctx *ctx, const cwen_weight *w, int epi, const _Float16 *xh, int N, const float *psc,
              const WideOut &o, float *part, size_t part_floats, hipStream_t st) {
  const int ns = epi == GEMV_EPI_SWIGLU ? 2 : 1;
  const GemvGrid &g = w->cfg[ns - 1];
  const bool finish = epi == GEMV_EPI_STORE && (o.accumulate || o.yh || o.ssq);
  if (N < 1 || !wide_takes(w, ns, finish) || wide_partial_floats(w, ns, finish, N) > part_floats) return CWEN_EINVAL;
  WideParams p;
  p.w = w->dev;
  p.wbytes = (uint32_t)w->bytes;
  p.nrg = w->nrg;
  p.nst = w->nst;
  p.M = w->ne1;
  p.xh = xh;
  p.K = w->ne0;
  p.N = N;
  p.S = g.nsplit ? g.S : 1;
  p.rps = g.nsplit ? g.rps : w->nst;
  p.rgB = wide_split_at(w, ns, finish);
  p.rowsB = (w->nrg - p.rgB) * Q4_ROWS;
  p.part = part;
  p.psc = psc;
  p.y = o.y;
  p.ys = o.ys;
  p.yh = o.yh;
  p.rflag = o.rflag;
  // Row streams per wave: 4, or the fewest (16 rows, both sides of a pair)
  // while 4 would leave CUs without a workgroup.
  const int big = (w->nrg * ns + 15) / 16 * ((N + 63) / 64) * (g.nsplit == g.grid ? g.S : 1);
  const bool wide4 = big >= ctx->ncu;
  int rc = CWEN_OK;
  if (epi == GEMV_EPI_SWIGLU) {
    if (w->fmt != GEMV_Q4) return CWEN_EINVAL;
    if (wide4) launch<GEMV_Q4, 2, GEMV_EPI_SWIGLU, 4>(p, st);
    else launch<GEMV_Q4, 2, GEMV_EPI_SWIGLU, 2>(p, st);
  } else {
    auto go = [&](auto fmt) {
      constexpr int FMT = decltype(fmt)::value;
      if (wide4) launch<FMT, 1, GEMV_EPI_STORE, 4>(p, st);
      else launch<FMT, 1, GEMV_EPI_STORE, 1>(p, st);
    };
    switch (w->fmt) {
      case GEMV_Q4: go(std::integral_constant<int, GEMV_Q4>{}); break;
      case GEMV_Q6K: go(std::integral_constant<int, GEMV_Q6K>{}); break;
      case GEMV_Q8: go(std::integral_constant<int, GEMV_Q8>{}); break;
      case GEMV_Q41: go(std::integral_constant<int, GEMV_Q41>{}); break;
      case GEMV_Q5K: go(std::integral_constant<int, GEMV_Q5K>{}); break;
      default: rc = CWEN_EINVAL;
    }
  }
  if (rc) return rc;
  CWEN_HIP_TRY(hipGetLastError());
  if (p.rowsB > 0) {
    const dim3 grid((unsigned)((p.rowsB + 63) / 64), (unsigned)((N + 3) / 4));
    if (epi == GEMV_EPI_SWIGLU)
      hipLaunchKernelGGL((wide_finish_kernel<2, GEMV_EPI_SWIGLU>), grid, dim3(256), 0, st, p, o, p.rgB * Q4_ROWS);
    else
      hipLaunchKernelGGL((wide_finish_kernel<1, GEMV_EPI_STORE>), grid, dim3(256), 0, st, p, o, p.rgB * Q4_ROWS);
    CWEN_HIP_TRY(hipGetLastError());
  }
  return CWEN_OK;
}
