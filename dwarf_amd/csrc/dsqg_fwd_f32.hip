// DSQG forward, float32 (gfx950): the dense window on the float32 matrix instructions, the
// long-range taps as row dots on the VALU.
//
// A workgroup owns one (b,h) and 64 query rows; wave w owns 16 of them, n0w = n0 + 16w.
//  1. K/V rows [n0-32, n0+64) go to LDS.  The band's scores are three 16x16 tiles K Q^T
//     (v_mfma_f32_16x16x4_f32): lane (i, g) holds query i and keys 4g + r.  With scale_embed
//     SE Q^T gives q.se of every tap, filed in the wave's [query][tap] table.
//  2. Long-range tap: key rows n0w - delta + 0..15 in the row layout (whole rows, PF taps in
//     flight), dotted with the query rows, DPP sums, the result into the table.
//  3. Softmax of a query over its four lanes: 12 band registers each and every fourth long-range
//     tap; the weights (unnormalised) of the latter go back to the table.
//  4. P V: band tiles V^T P^T on the matrix instructions (the weights already sit in the operand
//     layout), turned into row layout once through LDS; long-range rows are added to it by
//     float32 multiply-adds.  The division by the sum and the IF gain come last.
//
// A matrix product multiplies every value row of a tile by some query's zero weight, so an
// infinity or NaN in the window would reach queries that do not attend it.  Each workgroup looks
// for one while staging (one multiply-add per value); if it finds one, it runs every tap as a
// long-range one, where a row enters only the queries whose weight of it is positive.
//
// Bound by latency at the sizes float32 runs at (a 64-row tile is one of two on a CU at B2 H8
// N2047 D64): what counts is that a tile's loads are all in flight at once and nothing waits per
// tap.  At that size with scale_embed 25 us for 34 MB read and written
// (1.3 TB/s); the VALU kernel, whose every tap re-reads its key row from LDS and whose long-range
// loads sit in a branch each, takes 49.
//
// Semantics: _fwd_v3, kernels/dsqg_attention_v3.py:60-163 (plus score gain and IF gain).
#include "dsqg_f32.hpp"
#include "dsqg_launch.hpp"

namespace dsqg {

template <int D, bool HAS_SE>
__global__ __launch_bounds__(kBlock, D <= 64 ? 2 : 1) void fwd_f32_kernel(FwdParams p) {
  using G_ = GeoF<D>;
  constexpr int DB = G_::DB, RV = G_::RV, CHW = G_::CHW, CPL = G_::CPL, RG = G_::RG, CPR = G_::CPR;
  constexpr int WIN = G_::WIN, CWIN = G_::CWIN;
  constexpr int TS = 52;  // table row stride: rows on distinct banks at every column of a lane quad
  constexpr int PF = D <= 64 ? 6 : 4;  // long-range row blocks in flight

  __shared__ __align__(16) float sK[WIN * RV];
  __shared__ __align__(16) float sV[WIN * RV];
  __shared__ __align__(16) float sSE[HAS_SE ? kMaxTaps * RV : 4];
  __shared__ __align__(16) float sTab[4][16 * TS];
  __shared__ float sBias[kMaxTaps], sGain[kMaxTaps];
  __shared__ int sDelta[kMaxTaps];
  __shared__ float sMark[4], sInv[4][16];

  const int tid = threadIdx.x;
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int bh = lb / p.n_tiles, tile = lb - bh * p.n_tiles;
  const int b = bh / p.H, h = bh - b * p.H;
  const int N = p.N, J = p.taps.J, W = p.taps.W;
  const int n0 = tile * 64;
  const float c = p.scale;
  const int qsn = (int)p.qs.n, ksn = (int)p.ks.n, vsn = (int)p.vs.n;
  const __amdgpu_buffer_rsrc_t rQ = slice_rsrc_f32(p.q, b * p.qs.b + h * p.qs.h, p.qs.n, N, D);
  const __amdgpu_buffer_rsrc_t rK = slice_rsrc_f32(p.k, b * p.ks.b + h * p.ks.h, p.ks.n, N, D);
  const __amdgpu_buffer_rsrc_t rV = slice_rsrc_f32(p.v, b * p.vs.b + h * p.vs.h, p.vs.n, N, D);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, g = l >> 4;
  const int n0w = n0 + 16 * w, n = n0w + i;
  const bool row_ok = n < N;
  float* const sT = sTab[w];

  // ---- Loads: per-tap parameters, window, query rows in both layouts, the first long-range key
  // rows. ----
  TapParams<D, HAS_SE> tp;
  tp.load(p.pos_bias, p.score_gain, p.scale_embed, J, p.H, h, tid);
  const float if_a = p.if_gain ? p.if_gain[h] : 1.0f;
  const int dl_lane = p.taps.delta[l < J ? l : 0];  // lane j holds tap j's offset
  float4 wk[CWIN], wv[CWIN];
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    wk[u] = bload4f(rK, (n0 - kMaxWindow + r) * ksn + cc);
    wv[u] = bload4f(rV, (n0 - kMaxWindow + r) * vsn + cc);
  }
  float4 qB[DB], qR[CHW];
#pragma unroll
  for (int s = 0; s < DB; ++s) qB[s] = bload4f(rQ, n * qsn + 16 * s + 4 * g);
#pragma unroll
  for (int u = 0; u < CHW; ++u) qR[u] = bload4f(rQ, (n0w + rf_row<D>(l, u)) * qsn + rf_col<D>(l, u));
  int klane[CHW], vlane[CHW];
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    klane[u] = opaque(rf_row<D>(l, u) * ksn + rf_col<D>(l, u));
    vlane[u] = opaque(rf_row<D>(l, u) * vsn + rf_col<D>(l, u));
  }
  int j0 = W + 1;                                   // first tap taken as a long-range one
  float4 ring[PF][CHW];
  auto load_k = [&](int j, int slot) {
    const int m0 = n0w - __builtin_amdgcn_readlane(dl_lane, j);
#pragma unroll
    for (int u = 0; u < CHW; ++u) ring[slot][u] = bload4f(rK, m0 * ksn + klane[u]);
  };
  auto load_v = [&](int j, int slot) {
    const int m0 = n0w - __builtin_amdgcn_readlane(dl_lane, j);
#pragma unroll
    for (int u = 0; u < CHW; ++u) ring[slot][u] = bload4f(rV, m0 * vsn + vlane[u]);
  };
#pragma unroll
  for (int t = 0; t < PF; ++t)
    if (j0 + t < J) load_k(j0 + t, t);

  __builtin_amdgcn_sched_barrier(0);  // (every load above is issued before the first wait)
  if (tid < kMaxTaps) sDelta[tid] = dl_lane;  // (wave 0)
  tp.store(sBias, sGain, sSE, J, tid, 0.f);
  float mark = 0.f;
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    if (ci < WIN * CPR) {
      *reinterpret_cast<float4*>(sK + r * RV + cc) = wk[u];
      *reinterpret_cast<float4*>(sV + r * RV + cc) = wv[u];
      mark = nonfinite_mark(wv[u], mark);
    }
  }
  const bool wave_bad = __builtin_amdgcn_ballot_w64(mark != 0.f) != 0;
  if (l == 0) sMark[w] = wave_bad ? 1.f : 0.f;
  __syncthreads();
  const bool bad = __builtin_amdgcn_readfirstlane(sMark[0] + sMark[1] + sMark[2] + sMark[3] != 0.f);

  // ---- q.se of every tap, and the band's scores. ----
  if constexpr (HAS_SE) {
#pragma unroll
    for (int jb = 0; jb < 3; ++jb) {
      const f32x4_t acc = mfma_f32_dot(sSE + (16 * jb + i) * RV + 4 * g, qB);
      *reinterpret_cast<float4*>(sT + i * TS + 16 * jb + 4 * g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    }
    lds_wave_sync();
  }
  float sd[12];
  if (bad) {
    j0 = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e) sd[e] = -INFINITY;
#pragma unroll
    for (int t = 0; t < PF; ++t)
      if (t < J) load_k(t, t);
  } else {
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
      const f32x4_t acc = mfma_f32_dot(sK + (16 * w + 16 * kk + i) * RV + 4 * g, qB);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dl = 32 - 4 * g + i - 16 * kk - r;  // n - m for key m of this register
        const bool ok = row_ok && (unsigned)dl <= (unsigned)W && n >= dl;
        const int j = ok ? dl : 0;
        float x = acc[r] * sGain[j];
        if constexpr (HAS_SE) x += sT[i * TS + j];
        sd[4 * kk + r] = ok ? fmaf(x, c, sBias[j]) : -INFINITY;
      }
    }
  }

  // ---- Long-range scores g q.k (+ q.se) into the table. ----
  for (int jb = j0; jb < J; jb += PF) {
#pragma unroll
    for (int t = 0; t < PF; ++t) {
      const int j = jb + t;
      if (j < J) {
        const float gain = sGain[j];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          float x = 0.f;
#pragma unroll
          for (int pc = 0; pc < CPL; ++pc) x = dot4f(qR[rg * CPL + pc], ring[t][rg * CPL + pc], x);
          x = group_sum<G_::LPR>(x) * gain;
          float* const dst = sT + rf_row<D>(l, rg * CPL) * TS + j;
          if (l % G_::LPR == 0) *dst = HAS_SE ? *dst + x : x;
        }
        if (j + PF < J) load_k(j + PF, t);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < PF; ++t)
    if (j0 + t < J) load_v(j0 + t, t);
  lds_wave_sync();

  // ---- Softmax over the four lanes of each query. ----
  float ss[12];
  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    ss[e] = -INFINITY;
    const int j = j0 + g + 4 * e;
    if (j0 + 4 * e < J) {
      const int jc = j < J ? j : 0;
      const float s = fmaf(sT[i * TS + jc], c, sBias[jc]);
      ss[e] = j < J && row_ok && n >= sDelta[jc] ? s : -INFINITY;
    }
    mx = fmaxf(mx, fmaxf(sd[e], ss[e]));
  }
  mx = col_max(mx);
  if (!row_ok) mx = 0.f;
  float lsum = 0.f;
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    sd[e] = __expf(sd[e] - mx);
    lsum += sd[e];
    if (j0 + 4 * e < J) {
      const float pj = __expf(ss[e] - mx);
      lsum += pj;
      const int j = j0 + g + 4 * e;
      if (j < J) sT[i * TS + j] = pj;
    }
  }
  lsum = col_sum(lsum);
  if (row_ok && g == 0 && p.lse) p.lse[(long long)bh * N + n] = mx + __logf(lsum);
  if (g == 0) sInv[w][i] = if_a / lsum;

  // ---- Band P V, O^T = V^T P^T. ----
  f32x4_t O[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) O[db] = zero4();
  if (!bad) {
#pragma unroll
    for (int kk = 0; kk < 3; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x[DB];
        cols_load<D>(sV + (16 * w + 16 * kk + 4 * g + r) * RV, i, x);
#pragma unroll
        for (int db = 0; db < DB; ++db) O[db] = mfma_f32(x[db], sd[4 * kk + r], O[db]);
      }
  }
  __syncthreads();  // every wave's reads of sK are done: its rows turn the layout
  float* const st = sK + 16 * w * RV;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) x[db] = O[db][r];
    cols_store<D>(st + i * RV, 4 * g + r, x);
  }
  lds_wave_sync();
  float4 acc[CHW];
#pragma unroll
  for (int u = 0; u < CHW; ++u) acc[u] = *reinterpret_cast<const float4*>(st + rf_row<D>(l, u) * RV + rf_col<D>(l, u));

  // ---- Long-range P V, whole rows. ----
  for (int jb = j0; jb < J; jb += PF) {
#pragma unroll
    for (int t = 0; t < PF; ++t) {
      const int j = jb + t;
      if (j < J) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          const float pj = sT[rf_row<D>(l, rg * CPL) * TS + j];
          if (pj > 0.f) {
#pragma unroll
            for (int pc = 0; pc < CPL; ++pc) fma4f(pj, ring[t][rg * CPL + pc], acc[rg * CPL + pc]);
          }
        }
        if (j + PF < J) load_v(j + PF, t);
      }
    }
  }
  float* const ob = static_cast<float*>(p.out) + b * p.os.b + h * p.os.h;
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    const int rr = rf_row<D>(l, u);
    const float inv = sInv[w][rr];
    if (n0w + rr < N)
      store4f_stream(ob + (n0w + rr) * p.os.n + rf_col<D>(l, u),
                     make_float4(acc[u].x * inv, acc[u].y * inv, acc[u].z * inv, acc[u].w * inv));
  }
}

template <int D>
static hipError_t launch_fwd_f32_d(const FwdParams& p0, hipStream_t st) {
  FwdParams p = p0;
  p.n_tiles = (p.N + 63) / 64;
  const long long nblocks = (long long)p.B * p.H * p.n_tiles;
  if (nblocks == 0) return hipSuccess;
  if (p.scale_embed) hipLaunchKernelGGL((fwd_f32_kernel<D, true>), dim3((unsigned)nblocks), dim3(kBlock), 0, st, p);
  else hipLaunchKernelGGL((fwd_f32_kernel<D, false>), dim3((unsigned)nblocks), dim3(kBlock), 0, st, p);
  return hipGetLastError();
}

bool fwd_f32_supported(const FwdParams& p, int D) {
  const long long rs[3] = {p.qs.n, p.ks.n, p.vs.n};
  return f32_mfma_strides_ok(p.N, p.taps.maxd, D, rs, 3);
}

hipError_t launch_fwd_f32(const FwdParams& p, int D, hipStream_t st) {
  switch (D) {
    case 32: return launch_fwd_f32_d<32>(p, st);
    case 64: return launch_fwd_f32_d<64>(p, st);
    case 80: return launch_fwd_f32_d<80>(p, st);
    case 96: return launch_fwd_f32_d<96>(p, st);
    case 128: return launch_fwd_f32_d<128>(p, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsqg
