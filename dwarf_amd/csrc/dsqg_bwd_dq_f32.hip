// DSQG backward, launch 1, float32 (gfx950): query-centric dq, D' and the per-workgroup
// parameter-gradient partials.  Same tiling and layouts as the float32 forward
// (dsqg_fwd_f32.hip): 64 query rows of one (b,h) per workgroup, 16 per wave, the dense window on
// the float32 matrix instructions, long-range taps as row dots on the VALU.
//
//  1. Band: S = K Q^T and U = V dOut^T tiles; alpha_j = exp(s_j - lse), u_j.
//  2. Long-range taps: q.k and dOut.v of each pair by row dots (K and V blocks in flight together),
//     filed in the wave's two [query][tap] tables; the query's four lanes turn them into alpha and
//     u, and with the band's into D' = sum_j alpha_j u_j.
//  3. dS_j = a alpha_j (u_j - D') replaces the scores in the first table (for the parameter sums
//     and scale_embed's products), the weights of dq the second.  dq = c sum_j dS_j (g_j k_j +
//     se_j): the band and the SE term on the matrix instructions, turned into row layout once,
//     then the long-range key rows by float32 multiply-adds.
//  4. dbias / dg / da are sums of the tables over the wave's rows, dse = c dS^T Q a matrix product
//     over the tile's 64 queries; one partial per workgroup, reduced in a fixed order later.
// A tap enters dq only where its alpha is positive.  The matrix products would multiply an
// infinity or NaN of a staged K or scale_embed row by other queries' zero weights, so a workgroup
// that meets one runs every tap as a long-range one (see dsqg_fwd_f32.hip).
//
// Bound by latency like the forward: 37 us at B2 H8 N2047 D64 with scale_embed (the VALU kernel:
// 162, with per-tap register arrays it spills, a branch around each long-range load and dse summed
// one element per thread).
//
// Follows _compute_D_v3 + _bwd_dq_v3 (kernels/dsqg_attention_v3.py:170-275), except that D' is
// computed from the weights and the parameter gradients avoid atomics.
#include "dsqg_f32.hpp"
#include "dsqg_launch.hpp"

namespace dsqg {

// DG: the score gain's gradient is requested (one more table, c q.k of every pair).
template <int D, bool HAS_SE, bool DG>
__global__ __launch_bounds__(kBlock, D <= 64 && !(HAS_SE && DG) ? 2 : 1) void bwd_dq_f32_kernel(BwdParams p) {
  using G_ = GeoF<D>;
  constexpr int DB = G_::DB, RV = G_::RV, CHW = G_::CHW, CPL = G_::CPL, RG = G_::RG, CPR = G_::CPR;
  constexpr int WIN = G_::WIN, CWIN = G_::CWIN;
  constexpr int TS = 52;
  constexpr int PF = D <= 64 ? 3 : 2;  // long-range taps in flight, a K and a V block each

  // K window, then V window.  After the band's products the V window's rows hold the second
  // table and then, with scale_embed, the query rows; the K window turns dq's layout.
  __shared__ __align__(16) float sK[WIN * RV];
  __shared__ __align__(16) float sV[WIN * RV];
  __shared__ __align__(16) float sSE[HAS_SE ? kMaxTaps * RV : 4];
  __shared__ __align__(16) float sDS[4 * 16 * TS];          // scores, then dS
  __shared__ __align__(16) float sRaw[DG ? 4 * 16 * TS : 4];  // c q.k
  __shared__ float sBias[kMaxTaps], sGain[kMaxTaps];
  __shared__ int sDelta[kMaxTaps];
  __shared__ float sMark[4], sDp[4][16];
  static_assert(WIN * RV >= 4 * 16 * TS, "the second table fits the V window");

  const int tid = threadIdx.x;
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int bh = lb / p.n_chunks, tile = lb - bh * p.n_chunks;
  const int b = bh / p.H, h = bh - b * p.H;
  const int N = p.N, J = p.taps.J, W = p.taps.W;
  const int n0 = tile * 64;
  const float c = p.scale;
  const float a = p.if_gain ? p.if_gain[h] : 1.0f;
  const int qsn = (int)p.qs.n, ksn = (int)p.ks.n, vsn = (int)p.vs.n, dosn = (int)p.dos.n;
  const __amdgpu_buffer_rsrc_t rQ = slice_rsrc_f32(p.q, b * p.qs.b + h * p.qs.h, p.qs.n, N, D);
  const __amdgpu_buffer_rsrc_t rK = slice_rsrc_f32(p.k, b * p.ks.b + h * p.ks.h, p.ks.n, N, D);
  const __amdgpu_buffer_rsrc_t rV = slice_rsrc_f32(p.v, b * p.vs.b + h * p.vs.h, p.vs.n, N, D);
  const __amdgpu_buffer_rsrc_t rO = slice_rsrc_f32(p.dout, b * p.dos.b + h * p.dos.h, p.dos.n, N, D);
  const long long rowbase = (long long)bh * N;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, g = l >> 4;
  const int n0w = n0 + 16 * w, n = n0w + i;
  const bool row_ok = n < N;
  float* const sT = sDS + w * 16 * TS;
  float* const sU = sV + w * 16 * TS;
  float* const sR = sRaw + (DG ? w * 16 * TS : 0);

  // ---- Loads. ----
  TapParams<D, HAS_SE> tp;
  tp.load(p.pos_bias, p.score_gain, p.scale_embed, J, p.H, h, tid);
  const float lse = p.lse[rowbase + (row_ok ? n : N - 1)];
  const int dl_lane = p.taps.delta[l < J ? l : 0];
  float4 wk[CWIN], wv[CWIN];
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    wk[u] = bload4f(rK, (n0 - kMaxWindow + r) * ksn + cc);
    wv[u] = bload4f(rV, (n0 - kMaxWindow + r) * vsn + cc);
  }
  float4 qB[DB], oB[DB], qR[CHW], oR[CHW];
#pragma unroll
  for (int s = 0; s < DB; ++s) {
    qB[s] = bload4f(rQ, n * qsn + 16 * s + 4 * g);
    oB[s] = bload4f(rO, n * dosn + 16 * s + 4 * g);
  }
  int klane[CHW], vlane[CHW];
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    const int rr = rf_row<D>(l, u), cc = rf_col<D>(l, u);
    qR[u] = bload4f(rQ, (n0w + rr) * qsn + cc);
    oR[u] = bload4f(rO, (n0w + rr) * dosn + cc);
    klane[u] = opaque(rr * ksn + cc);
    vlane[u] = opaque(rr * vsn + cc);
  }
  int j0 = W + 1;  // first tap taken as a long-range one
  float4 kr[PF][CHW], vr[PF][CHW];
  auto load_k = [&](int j, int slot) {
    const int m0 = n0w - __builtin_amdgcn_readlane(dl_lane, j);
#pragma unroll
    for (int u = 0; u < CHW; ++u) kr[slot][u] = bload4f(rK, m0 * ksn + klane[u]);
  };
  auto load_v = [&](int j, int slot) {
    const int m0 = n0w - __builtin_amdgcn_readlane(dl_lane, j);
#pragma unroll
    for (int u = 0; u < CHW; ++u) vr[slot][u] = bload4f(rV, m0 * vsn + vlane[u]);
  };
#pragma unroll
  for (int t = 0; t < PF; ++t)
    if (j0 + t < J) { load_k(j0 + t, t); load_v(j0 + t, t); }

  __builtin_amdgcn_sched_barrier(0);  // (every load above is issued before the first wait)
  if (tid < kMaxTaps) sDelta[tid] = dl_lane;  // (wave 0)
  float mark = tp.store(sBias, sGain, sSE, J, tid, 0.f);
#pragma unroll
  for (int u = 0; u < CWIN; ++u) {
    const int ci = tid + u * kBlock, r = ci / CPR, cc = 4 * (ci - r * CPR);
    if (ci < WIN * CPR) {
      *reinterpret_cast<float4*>(sK + r * RV + cc) = wk[u];
      *reinterpret_cast<float4*>(sV + r * RV + cc) = wv[u];
      mark = nonfinite_mark(wk[u], mark);
    }
  }
  const bool wave_bad = __builtin_amdgcn_ballot_w64(mark != 0.f) != 0;
  if (l == 0) sMark[w] = wave_bad ? 1.f : 0.f;
  // Table columns past the last tap are read as zeros by the scale_embed products.
  for (int e = tid; e < 4 * 16 * TS; e += kBlock) sDS[e] = 0.f;
  __syncthreads();
  const bool bad = __builtin_amdgcn_readfirstlane(sMark[0] + sMark[1] + sMark[2] + sMark[3] != 0.f);

  if constexpr (HAS_SE) {
#pragma unroll
    for (int jb = 0; jb < 3; ++jb) {
      const f32x4_t acc = mfma_f32_dot(sSE + (16 * jb + i) * RV + 4 * g, qB);
      *reinterpret_cast<float4*>(sT + i * TS + 16 * jb + 4 * g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    }
    lds_wave_sync();
  }

  // ---- 1. Band: alpha, u and their share of D'. ----
  float al[12], uu[12];
  float dlane = 0.f;
#pragma unroll
  for (int e = 0; e < 12; ++e) { al[e] = 0.f; uu[e] = 0.f; }
  if (bad) {
    j0 = 0;
#pragma unroll
    for (int t = 0; t < PF; ++t)
      if (t < J) { load_k(t, t); load_v(t, t); }
  } else {
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
      const int row = (16 * w + 16 * kk + i) * RV + 4 * g;
      const f32x4_t aS = mfma_f32_dot(sK + row, qB), aU = mfma_f32_dot(sV + row, oB);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dl = 32 - 4 * g + i - 16 * kk - r;
        const bool in = (unsigned)dl <= (unsigned)W, ok = in && row_ok && n >= dl;
        const int j = ok ? dl : 0;
        float x = aS[r] * sGain[j];
        if constexpr (HAS_SE) x += sT[i * TS + j];
        al[4 * kk + r] = ok ? __expf(fmaf(x, c, sBias[j]) - lse) : 0.f;
        uu[4 * kk + r] = ok ? aU[r] : 0.f;
        dlane = fmaf(al[4 * kk + r], uu[4 * kk + r], dlane);
        if constexpr (DG) {
          if (in) sR[i * TS + dl] = ok ? c * aS[r] : 0.f;
        }
      }
    }
  }
  __syncthreads();  // the V window is free: the second tables move in

  // ---- 2. Long-range pairs: scores and u into the tables. ----
  for (int jb = j0; jb < J; jb += PF) {
#pragma unroll
    for (int t = 0; t < PF; ++t) {
      const int j = jb + t;
      if (j < J) {
        const float gain = sGain[j];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          float x = 0.f, y = 0.f;
#pragma unroll
          for (int pc = 0; pc < CPL; ++pc) {
            x = dot4f(qR[rg * CPL + pc], kr[t][rg * CPL + pc], x);
            y = dot4f(oR[rg * CPL + pc], vr[t][rg * CPL + pc], y);
          }
          x = group_sum<G_::LPR>(x);
          y = group_sum<G_::LPR>(y);
          const int e = rf_row<D>(l, rg * CPL) * TS + j;
          if (l % G_::LPR == 0) {
            sT[e] = HAS_SE ? sT[e] + x * gain : x * gain;
            sU[e] = y;
            if constexpr (DG) sR[e] = c * x;
          }
        }
        if (j + PF < J) { load_k(j + PF, t); load_v(j + PF, t); }
      }
    }
  }
  lds_wave_sync();
  float als[12], uus[12];
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    als[e] = uus[e] = 0.f;
    if (j0 + 4 * e < J) {
      const int j = j0 + g + 4 * e, jc = j < J ? j : 0;
      const bool ok = j < J && row_ok && n >= sDelta[jc];
      const float s = fmaf(sT[i * TS + jc], c, sBias[jc]), u = sU[i * TS + jc];
      als[e] = ok ? __expf(s - lse) : 0.f;
      uus[e] = ok ? u : 0.f;
      dlane = fmaf(als[e], uus[e], dlane);
    }
  }
  const float Dsum = col_sum(dlane), Dp = row_ok ? Dsum : 0.f;
  // The first key blocks of the second pass travel during the band's product.
#pragma unroll
  for (int t = 0; t < PF; ++t)
    if (j0 + t < J) load_k(j0 + t, t);

  // ---- 3. dS and the weights; the band's and the SE term's share of dq. ----
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    if (j0 + 4 * e < J) {
      const int j = j0 + g + 4 * e;
      const float ds = a * als[e] * (uus[e] - Dp);
      if (j < J) {
        sT[i * TS + j] = ds;
        sU[i * TS + j] = als[e] > 0.f ? ds : 0.f;
      }
    }
  }
  f32x4_t X[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) X[db] = zero4();
  if (!bad) {
#pragma unroll
    for (int kk = 0; kk < 3; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dl = 32 - 4 * g + i - 16 * kk - r;
        const bool in = (unsigned)dl <= (unsigned)W;
        const int j = in ? dl : 0;
        const float al_ = al[4 * kk + r], ds = a * al_ * (uu[4 * kk + r] - Dp);
        const float dq_w = al_ > 0.f ? ds : 0.f;
        if (in) {
          sT[i * TS + dl] = ds;
          sU[i * TS + dl] = dq_w;
        }
        float x[DB];
        cols_load<D>(sK + (16 * w + 16 * kk + 4 * g + r) * RV, i, x);
        const float wq = dq_w * sGain[j];
#pragma unroll
        for (int db = 0; db < DB; ++db) X[db] = mfma_f32(x[db], wq, X[db]);
      }
  }
  lds_wave_sync();
  if constexpr (HAS_SE) {
    if (!bad) {
      // Taps past the last have zero scale_embed rows; their weights must be zero too.
#pragma unroll
      for (int jb = 0; jb < 3; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * jb + 4 * g + r;
          float x[DB];
          cols_load<D>(sSE + j * RV, i, x);
          const float wj = j < J ? sU[i * TS + j] : 0.f;
#pragma unroll
          for (int db = 0; db < DB; ++db) X[db] = mfma_f32(x[db], wj, X[db]);
        }
    }
  }
  __syncthreads();  // every wave's reads of the K window are done: its rows turn the layout
  float* const st = sK + 16 * w * RV;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) x[db] = X[db][r];
    cols_store<D>(st + i * RV, 4 * g + r, x);
  }
  if (g == 0) sDp[w][i] = Dp;
  lds_wave_sync();
  float4 acc[CHW];
#pragma unroll
  for (int u = 0; u < CHW; ++u) acc[u] = *reinterpret_cast<const float4*>(st + rf_row<D>(l, u) * RV + rf_col<D>(l, u));

  // ---- Long-range key rows. ----
  for (int jb = j0; jb < J; jb += PF) {
#pragma unroll
    for (int t = 0; t < PF; ++t) {
      const int j = jb + t;
      if (j < J) {
        const float gain = sGain[j];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          const float ds = sU[rf_row<D>(l, rg * CPL) * TS + j];
          if (ds != 0.f) {
#pragma unroll
            for (int pc = 0; pc < CPL; ++pc) {
              fma4f(ds * gain, kr[t][rg * CPL + pc], acc[rg * CPL + pc]);
              if constexpr (HAS_SE) {
                if (bad) fma4f(ds, *reinterpret_cast<const float4*>(sSE + j * RV + rf_col<D>(l, pc)), acc[rg * CPL + pc]);
              }
            }
          }
        }
        if (j + PF < J) load_k(j + PF, t);
      }
    }
  }
  float* const dqb = static_cast<float*>(p.dq) + b * p.dqs.b + h * p.dqs.h;
#pragma unroll
  for (int u = 0; u < CHW; ++u) {
    const int rr = rf_row<D>(l, u);
    if (n0w + rr < N)
      store4f_stream(dqb + (n0w + rr) * p.dqs.n + rf_col<D>(l, u),
                     make_float4(c * acc[u].x, c * acc[u].y, c * acc[u].z, c * acc[u].w));
  }
  if (row_ok && g == 0) p.dpre[rowbase + n] = Dp;

  // ---- 4. Parameter partials: column sums of the wave's rows, then over the waves in order. ----
  float s_bias = 0.f, s_gain = 0.f, s_if = 0.f;
  if (l < J) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float ds = sT[r * TS + l];
      s_bias += ds;
      if constexpr (DG) s_gain = fmaf(ds, sR[r * TS + l], s_gain);
    }
  }
  if (l == 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s_if += sDp[w][r];
  }
  const bool se_grad = HAS_SE && p.part_se != nullptr;
  __syncthreads();  // the second tables and the layout rows are read
  float* const red = sV;  // 4 x 132 floats of sums
  float* const sQrow = sK;
  if (l < J) { red[w * 132 + l] = s_bias; red[w * 132 + 64 + l] = s_gain; }
  if (l == 0) red[w * 132 + 128] = s_if;
  if (se_grad) {
#pragma unroll
    for (int u = 0; u < CHW; ++u)
      *reinterpret_cast<float4*>(sQrow + (16 * w + rf_row<D>(l, u)) * RV + rf_col<D>(l, u)) = qR[u];
  }
  __syncthreads();
  if (tid < J) {
    p.part_bias[(long long)lb * J + tid] = red[tid] + red[132 + tid] + red[264 + tid] + red[396 + tid];
    if constexpr (DG)
      p.part_gain[(long long)lb * J + tid] = red[64 + tid] + red[196 + tid] + red[328 + tid] + red[460 + tid];
  }
  if (tid == 0 && p.part_if) p.part_if[lb] = red[128] + red[260] + red[392] + red[524];
  if constexpr (HAS_SE) {
    if (se_grad) {
      // dSE^T (d x j) = Q^T dS over the tile's 64 queries, the 16-tap blocks split over the first
      // three waves: lane (i, g), register r of tile db: tap 16 w + i, tile row 4 g + r.
      if (w < 3 && 16 * w < J) {
        f32x4_t E[DB];
#pragma unroll
        for (int db = 0; db < DB; ++db) E[db] = zero4();
#pragma unroll
        for (int ww = 0; ww < 4; ++ww)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x[DB];
            cols_load<D>(sQrow + (16 * ww + 4 * g + r) * RV, i, x);
            const float ds = sDS[(16 * ww + 4 * g + r) * TS + 16 * w + i];
#pragma unroll
            for (int db = 0; db < DB; ++db) E[db] = mfma_f32(x[db], ds, E[db]);
          }
        const int j = 16 * w + i;
        if (j < J) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x[DB];
#pragma unroll
            for (int db = 0; db < DB; ++db) x[db] = c * E[db][r];
            cols_store<D>(p.part_se + ((long long)lb * J + j) * D, 4 * g + r, x);
          }
        }
      }
    }
  }
}

template <int D, bool HAS_SE>
static void launch_dq_f32_se(const BwdParams& p, unsigned nb, hipStream_t st) {
  if (p.part_gain) hipLaunchKernelGGL((bwd_dq_f32_kernel<D, HAS_SE, true>), dim3(nb), dim3(kBlock), 0, st, p);
  else hipLaunchKernelGGL((bwd_dq_f32_kernel<D, HAS_SE, false>), dim3(nb), dim3(kBlock), 0, st, p);
}

template <int D>
static hipError_t launch_dq_f32_d(const BwdParams& p, unsigned nb, hipStream_t st) {
  if (p.tiles_per_block != 1 || p.batches_per_block != 1) return hipErrorInvalidValue;
  // The scale_embed form also serves its gradient requested at se = 0.
  if (p.scale_embed || p.part_se) launch_dq_f32_se<D, true>(p, nb, st);
  else launch_dq_f32_se<D, false>(p, nb, st);
  return hipGetLastError();
}

hipError_t launch_bwd_dq_f32(const BwdParams& p, int D, unsigned nblocks, hipStream_t st) {
  switch (D) {
    case 32: return launch_dq_f32_d<32>(p, nblocks, st);
    case 64: return launch_dq_f32_d<64>(p, nblocks, st);
    case 80: return launch_dq_f32_d<80>(p, nblocks, st);
    case 96: return launch_dq_f32_d<96>(p, nblocks, st);
    case 128: return launch_dq_f32_d<128>(p, nblocks, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsqg
