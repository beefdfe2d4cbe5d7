// DSQG backward, launch 2, float32 (gfx950): key-centric dk and dv.  Same tiling and layouts as
// the float32 forward (dsqg_fwd_f32.hip): 64 key rows of one (b,h) per workgroup, 16 per wave.
//
// Key m is read by the queries n = m + delta_j:
//   dv_m = sum_j a alpha_j(n) dOut_n,   dk_m = c sum_j g_j dS_j(n) q_n,
//   alpha_j(n) = exp(s_j(n) - lse_n),   dS_j(n) = a alpha_j(n) (dOut_n . v_m - D'_n).
//  * Dense window: query and dOut rows [m0, m0+96) in LDS, three 16x16 tiles S = Q K^T and
//    U = dOut V^T per wave on the float32 matrix instructions; their result layout (key l%16,
//    queries 4g + r) is the weight operand of dK^T = Q^T (g dS) and dV^T = dOut^T (a alpha).
//    With scale_embed q.se of the window's queries is a table SE Q^T.
//  * Long-range taps: query rows m0w + delta + 0..15 as whole rows (PF taps in flight) against the
//    wave's key and value rows in the same layout: two row dots, the weights, two row updates.
// An infinity or NaN among the window's rows would reach other keys through their zero weights:
// a workgroup that stages one runs every tap as a long-range one (see dsqg_fwd_f32.hip).
// 34 us at B2 H8 N2047 D64 with scale_embed, the parameter reduction included, which rides in the
// launch as extra workgroups (apart: 33 + 6.5; the VALU kernel: 52 + 6.5).
// Follows _bwd_dkdv_v3 (kernels/dsqg_attention_v3.py:282-352), which also needs no atomics.
#include "dsqg_f32.hpp"
#include "dsqg_launch.hpp"
#include "dsqg_reduce.hpp"

namespace dsqg {

template <int D, bool HAS_SE>
__global__ __launch_bounds__(kBlock, D <= 64 ? 2 : 1) void bwd_dkdv_f32_kernel(BwdParams p) {
  using G_ = GeoF<D>;
  constexpr int DB = G_::DB, RV = G_::RV, CHW = G_::CHW, CPL = G_::CPL, RG = G_::RG, CPR = G_::CPR;
  constexpr int WIN = G_::WIN, CWIN = G_::CWIN;
  constexpr int TS = 33;               // q.se table of the dense taps
  constexpr int PF = D == 32 ? 4 : 2;  // long-range taps in flight, a query and a dOut block each

  __shared__ __align__(16) float sQ[WIN * RV];
  __shared__ __align__(16) float sO[WIN * RV];
  __shared__ __align__(16) float sSE[HAS_SE ? kMaxTaps * RV : 4];
  __shared__ float sT[HAS_SE ? WIN * TS : 1];
  __shared__ float sLse[WIN], sDp[WIN];
  __shared__ float sBias[kMaxTaps], sGain[kMaxTaps];
  __shared__ float sMark[4];

  const int tid = threadIdx.x;
  // Workgroups before and past the dk/dv tiles run the parameter reduction (partials from launch 1).
  const int bid = (int)blockIdx.x - p.red_se_blocks;
  if (bid < 0) {
    reduce_se_block(p.red, (int)blockIdx.x, tid, sQ);
    return;
  }
  const int kv_blocks = (int)gridDim.x - p.red_se_blocks - p.red_blocks;
  if (bid >= kv_blocks) {
    reduce_params_wave(p.red, (bid - kv_blocks) * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tid >> 6), tid & 63);
    return;
  }
  const int lb = xcd_logical_block(bid, kv_blocks);
  const int bh = lb / p.n_tiles_kv, tile = lb - bh * p.n_tiles_kv;
  const int b = bh / p.H, h = bh - b * p.H;
  const int N = p.N, J = p.taps.J, W = p.taps.W;
  const int m0 = tile * 64;
  const float c = p.scale;
  const float a = p.if_gain ? p.if_gain[h] : 1.0f;
  const int qsn = (int)p.qs.n, ksn = (int)p.ks.n, vsn = (int)p.vs.n, dosn = (int)p.dos.n;
  const __amdgpu_buffer_rsrc_t rQ = slice_rsrc_f32(p.q, b * p.qs.b + h * p.qs.h, p.qs.n, N, D);
  const __amdgpu_buffer_rsrc_t rK = slice_rsrc_f32(p.k, b * p.ks.b + h * p.ks.h, p.ks.n, N, D);
  const __amdgpu_buffer_rsrc_t rV = slice_rsrc_f32(p.v, b * p.vs.b + h * p.vs.h, p.vs.n, N, D);
  const __amdgpu_buffer_rsrc_t rO = slice_rsrc_f32(p.dout, b * p.dos.b + h * p.dos.h, p.dos.n, N, D);
  const long long rowbase = (long long)bh * N;
  const __amdgpu_buffer_rsrc_t rL = slice_rsrc_f32(p.lse, rowbase, 1, N, 1);
  const __amdgpu_buffer_rsrc_t rP = slice_rsrc_f32(p.dpre, rowbase, 1, N, 1);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, g = l >> 4;
  const int m0w = m0 + 16 * w, m = m0w + i;
  const bool key_ok = m < N;

  // ---- Loads. ----
  TapParams<D, HAS_SE> tp;
  tp.load(p.pos_bias, p.score_gain, p.scale_embed, J, p.H, h, tid);
  const int wrow = tid < WIN ? m0 + tid : N;
  const float lse_ld = bload1f(rL, wrow), dp_ld = bload1f(rP, wrow);
  const int dl_lane = p.taps.delta[l < J ? l : 0];
  float4 wq[CWIN], wo[CWIN];
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    wq[u] = bload4f(rQ, (m0 + r) * qsn + cc);
    wo[u] = bload4f(rO, (m0 + r) * dosn + cc);
  }
  float4 kB[DB], vB[DB], kR[CHW], vR[CHW];
#pragma unroll
  for (int s = 0; s < DB; ++s) {
    kB[s] = bload4f(rK, m * ksn + 16 * s + 4 * g);
    vB[s] = bload4f(rV, m * vsn + 16 * s + 4 * g);
  }
  int qlane[CHW], olane[CHW];
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    const int rr = rf_row<D>(l, u), cc = rf_col<D>(l, u);
    qlane[u] = opaque(rr * qsn + cc);
    olane[u] = opaque(rr * dosn + cc);
  }
  int j0 = W + 1;  // first tap taken as a long-range one
  float4 qr[PF][CHW], orr[PF][CHW];
  float lr[PF][RG], pr[PF][RG];
  auto load_tap = [&](int j, int slot) {
    const int n0 = m0w + __builtin_amdgcn_readlane(dl_lane, j);
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
      lr[slot][rg] = bload1f(rL, n0 + rf_row<D>(l, rg * CPL));
      pr[slot][rg] = bload1f(rP, n0 + rf_row<D>(l, rg * CPL));
    }
#pragma unroll
    for (int u = 0; u < CHW; ++u) {
      qr[slot][u] = bload4f(rQ, n0 * qsn + qlane[u]);
      orr[slot][u] = bload4f(rO, n0 * dosn + olane[u]);
    }
  };
#pragma unroll
  for (int t = 0; t < PF; ++t)
    if (j0 + t < J) load_tap(j0 + t, t);

  __builtin_amdgcn_sched_barrier(0);  // (every load above is issued before the first wait)
  if (tid < WIN) { sLse[tid] = lse_ld; sDp[tid] = dp_ld; }
  tp.store(sBias, sGain, sSE, J, tid, 0.f);
  float mark = 0.f;
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    if (ci < WIN * CPR) {
      *reinterpret_cast<float4*>(sQ + r * RV + cc) = wq[u];
      *reinterpret_cast<float4*>(sO + r * RV + cc) = wo[u];
      mark = nonfinite_mark(wo[u], nonfinite_mark(wq[u], mark));
    }
  }
  const bool wave_bad = __builtin_amdgcn_ballot_w64(mark != 0.f) != 0;
  if (l == 0) sMark[w] = wave_bad ? 1.f : 0.f;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < CHW; ++u) {  // (after the window's registers are free)
    kR[u] = bload4f(rK, (m0w + rf_row<D>(l, u)) * ksn + rf_col<D>(l, u));
    vR[u] = bload4f(rV, (m0w + rf_row<D>(l, u)) * vsn + rf_col<D>(l, u));
  }
  const bool bad = __builtin_amdgcn_readfirstlane(sMark[0] + sMark[1] + sMark[2] + sMark[3] != 0.f);

  f32x4_t dK[DB], dV[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) { dK[db] = zero4(); dV[db] = zero4(); }
  if (bad) {
    j0 = 0;
#pragma unroll
    for (int t = 0; t < PF; ++t)
      if (t < J) load_tap(t, t);
  } else {
    if constexpr (HAS_SE) {
      // q.se of the window's queries and the dense taps: SE Q^T, 16-row blocks w and w + 4.
      for (int blk = w; blk < WIN / 16; blk += 4) {
        float4 qs[DB];
#pragma unroll
        for (int s = 0; s < DB; ++s) qs[s] = *reinterpret_cast<const float4*>(sQ + (16 * blk + i) * RV + 16 * s + 4 * g);
#pragma unroll
        for (int jb = 0; jb < 3; ++jb) {
          const f32x4_t acc = mfma_f32_dot(sSE + (16 * jb + i) * RV + 4 * g, qs);  // tap 4g + r, query i
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = 16 * jb + 4 * g + r;
            if (j <= W) sT[(16 * blk + i) * TS + j] = acc[r];
          }
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int qb = 0; qb < 3; ++qb) {
      const int row = (16 * w + 16 * qb + i) * RV + 4 * g;
      const f32x4_t aS = mfma_f32_dot(sQ + row, kB), aU = mfma_f32_dot(sO + row, vB);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = 16 * w + 16 * qb + 4 * g + r;  // query row in the window
        const int dl = 16 * qb + 4 * g + r - i;       // query - key
        const bool ok = key_ok && (unsigned)dl <= (unsigned)W && m0 + rr < N;
        const int j = ok ? dl : 0;
        float x = aS[r] * sGain[j];
        if constexpr (HAS_SE) x += sT[rr * TS + j];
        const float alpha = __expf(fmaf(x, c, sBias[j]) - sLse[rr]);
        const float wv = ok ? a * alpha : 0.f;
        const float wk = ok ? c * sGain[j] * (a * alpha * (aU[r] - sDp[rr])) : 0.f;
        float xq[DB], xo[DB];
        cols_load<D>(sQ + rr * RV, i, xq);
        cols_load<D>(sO + rr * RV, i, xo);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          dK[db] = mfma_f32(xq[db], wk, dK[db]);
          dV[db] = mfma_f32(xo[db], wv, dV[db]);
        }
      }
    }
  }
  __syncthreads();  // the windows are read: their rows turn the layout

  float4 ka[CHW], va[CHW];
  {
    float* const sk = sQ + 16 * w * RV;
    float* const sv = sO + 16 * w * RV;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float xk[DB], xv[DB];
#pragma unroll
      for (int db = 0; db < DB; ++db) { xk[db] = dK[db][r]; xv[db] = dV[db][r]; }
      cols_store<D>(sk + i * RV, 4 * g + r, xk);
      cols_store<D>(sv + i * RV, 4 * g + r, xv);
    }
    lds_wave_sync();
#pragma unroll
    for (int u = 0; u < CHW; ++u) {
      ka[u] = *reinterpret_cast<const float4*>(sk + rf_row<D>(l, u) * RV + rf_col<D>(l, u));
      va[u] = *reinterpret_cast<const float4*>(sv + rf_row<D>(l, u) * RV + rf_col<D>(l, u));
    }
  }

  // ---- Long-range taps: one query row per key row. ----
  for (int jb = j0; jb < J; jb += PF) {
#pragma unroll
    for (int t = 0; t < PF; ++t) {
      const int j = jb + t;
      if (j < J) {
        const float gain = sGain[j], bias = sBias[j];
        const int dl = __builtin_amdgcn_readlane(dl_lane, j);
        float4 se[CPL];
        if constexpr (HAS_SE) {
#pragma unroll
          for (int pc = 0; pc < CPL; ++pc) se[pc] = *reinterpret_cast<const float4*>(sSE + j * RV + rf_col<D>(l, pc));
        }
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          float x = 0.f, y = 0.f;
#pragma unroll
          for (int pc = 0; pc < CPL; ++pc) {
            x = dot4f(qr[t][rg * CPL + pc], kR[rg * CPL + pc], x);
            y = dot4f(orr[t][rg * CPL + pc], vR[rg * CPL + pc], y);
          }
          x *= gain;
          if constexpr (HAS_SE) {
#pragma unroll
            for (int pc = 0; pc < CPL; ++pc) x = dot4f(qr[t][rg * CPL + pc], se[pc], x);
          }
          x = group_sum<G_::LPR>(x);
          y = group_sum<G_::LPR>(y);
          if (m0w + rf_row<D>(l, rg * CPL) + dl < N) {
            const float alpha = __expf(fmaf(x, c, bias) - lr[t][rg]);
            const float wv = a * alpha, wk = c * gain * (a * alpha * (y - pr[t][rg]));
#pragma unroll
            for (int pc = 0; pc < CPL; ++pc) {
              fma4f(wk, qr[t][rg * CPL + pc], ka[rg * CPL + pc]);
              fma4f(wv, orr[t][rg * CPL + pc], va[rg * CPL + pc]);
            }
          }
        }
        if (j + PF < J) load_tap(j + PF, t);
      }
    }
  }
  float* const dkb = static_cast<float*>(p.dk) + b * p.dks.b + h * p.dks.h;
  float* const dvb = static_cast<float*>(p.dv) + b * p.dvs.b + h * p.dvs.h;
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    const int rr = rf_row<D>(l, u), cc = rf_col<D>(l, u);
    if (m0w + rr < N) {
      store4f_stream(dkb + (m0w + rr) * p.dks.n + cc, ka[u]);
      store4f_stream(dvb + (m0w + rr) * p.dvs.n + cc, va[u]);
    }
  }
}

template <int D>
static hipError_t launch_dkdv_f32_d(const BwdParams& p, unsigned nb, hipStream_t st) {
  if (p.scale_embed) hipLaunchKernelGGL((bwd_dkdv_f32_kernel<D, true>), dim3(nb), dim3(kBlock), 0, st, p);
  else hipLaunchKernelGGL((bwd_dkdv_f32_kernel<D, false>), dim3(nb), dim3(kBlock), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv_f32(const BwdParams& p, int D, unsigned nblocks, hipStream_t st) {
  switch (D) {
    case 32: return launch_dkdv_f32_d<32>(p, nblocks, st);
    case 64: return launch_dkdv_f32_d<64>(p, nblocks, st);
    case 80: return launch_dkdv_f32_d<80>(p, nblocks, st);
    case 96: return launch_dkdv_f32_d<96>(p, nblocks, st);
    case 128: return launch_dkdv_f32_d<128>(p, nblocks, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsqg
