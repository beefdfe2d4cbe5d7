// Geometry and operand helpers of the float32 MFMA kernels (dsqg_*_f32.hip, gfx950).
//
// v_mfma_f32_16x16x4_f32: A lane l holds row l%16, k = l/16; B lane l holds column l%16,
// k = l/16; C/D lane l holds column l%16, rows 4*(l/16) + r, r = 0..3.  Two choices keep every
// LDS access wide and every operand in the layout the previous step left it in (lane (i, g) =
// (l%16, l/16) throughout):
//  * A contraction over the head dim may visit its columns in any order, as long as both operands
//    agree: one 16-byte read of columns 16s + 4g .. +3 serves four MFMAs.
//  * A product whose contraction runs over rows (P V, dS K, ...) takes for its step r the rows
//    4g + r, which is where the score tile's register r already sits, and its 16-row output tiles
//    take interleaved columns (col_of): the DB tiles' operands of one row are then DB consecutive
//    floats per lane, 16 bytes at a time, and so are the results.
#pragma once

#include "dsqg_common.hpp"
#include "dsqg_mfma.hpp"

namespace dsqg {

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// 16x16 tile of A B over the head dim: A row l%16 from LDS (a: this lane's row at column
// 4 (l/16)), B from registers in the same column order.  Four accumulators, one per column of a
// 16-byte piece: independent chains for the matrix unit, and a sum of four short chains rounds
// less than one long one (at D = 96, N = 27 the whole backward's error against 64 bits falls from
// 3.7e-7 to what the VALU dots have).
template <int DB>
__device__ __forceinline__ f32x4_t mfma_f32_dot(const float* a, const float4 (&b)[DB]) {
  f32x4_t x = zero4(), y = zero4(), z = zero4(), w = zero4();
#pragma unroll
  for (int s = 0; s < DB; ++s) {
    const float4 v = *reinterpret_cast<const float4*>(a + 16 * s);
    x = mfma_f32(v.x, b[s].x, x); y = mfma_f32(v.y, b[s].y, y);
    z = mfma_f32(v.z, b[s].z, z); w = mfma_f32(v.w, b[s].w, w);
  }
  return (x + y) + (z + w);
}

// Row layout of a wave's 16-row block of a [rows][D] float matrix: a row is LPR lanes of CPL
// 16-byte chunks (LPR a power of two up to 16, so that DPP sums run over a row's lanes and no
// lane idles); load u = rg CPL + pc gives lane l chunk l % LPR + LPR pc of row l / LPR + RPL rg.
template <int D>
struct GeoF {
  static_assert(D % 16 == 0 && D >= 32 && D <= 128, "head dim");
  static constexpr int DB = D / 16;  // 16-column operand steps; 16-row output tiles
  static constexpr int LPR = D == 80 ? 4 : (D == 32 || D == 96 ? 8 : 16);
  static constexpr int CPR = D / 4;  // 16-byte chunks of a row
  static constexpr int CPL = CPR / LPR;
  static constexpr int RPL = 64 / LPR;
  static constexpr int RG = 16 / RPL;
  static constexpr int CHW = RG * CPL;
  // LDS row stride: 16 rows' 16-byte pieces at one column fall on distinct banks (D + 4 is an
  // odd multiple of 4 floats).
  static constexpr int RV = D + 4;
  static constexpr int WIN = 64 + kMaxWindow;  // window rows of a 64-row tile
  static constexpr int CWIN = (WIN * CPR + kBlock - 1) / kBlock;
  static_assert(CPL * LPR == CPR, "a row is whole chunks per lane");
};

template <int D>
__device__ __forceinline__ int rf_row(int l, int u) {
  return l / GeoF<D>::LPR + GeoF<D>::RPL * (u / GeoF<D>::CPL);
}
template <int D>
__device__ __forceinline__ int rf_col(int l, int u) {
  return 4 * (l % GeoF<D>::LPR + GeoF<D>::LPR * (u % GeoF<D>::CPL));
}

// Head-dim columns of the DB output tiles at tile row m: whole 64-column groups as four
// consecutive columns 4m + db, then two (2m + db) or one (m) per row of what is left.  cols_load
// reads a row's DB values for row m, cols_store writes them.
template <int D>
__device__ __forceinline__ void cols_load(const float* row, int m, float (&v)[D / 16]) {
#pragma unroll
  for (int b = 0; b < D / 64; ++b) {
    const float4 x = *reinterpret_cast<const float4*>(row + 64 * b + 4 * m);
    v[4 * b] = x.x; v[4 * b + 1] = x.y; v[4 * b + 2] = x.z; v[4 * b + 3] = x.w;
  }
  constexpr int B4 = D / 64 * 4;
  if constexpr (D % 64 == 32) {
    const float2 x = *reinterpret_cast<const float2*>(row + 16 * B4 + 2 * m);
    v[B4] = x.x; v[B4 + 1] = x.y;
  }
  if constexpr (D % 64 == 16) v[B4] = row[16 * B4 + m];
  static_assert(D % 64 == 0 || D % 64 == 32 || D % 64 == 16, "column remainder");
}
template <int D>
__device__ __forceinline__ void cols_store(float* row, int m, const float (&v)[D / 16]) {
#pragma unroll
  for (int b = 0; b < D / 64; ++b)
    *reinterpret_cast<float4*>(row + 64 * b + 4 * m) = make_float4(v[4 * b], v[4 * b + 1], v[4 * b + 2], v[4 * b + 3]);
  constexpr int B4 = D / 64 * 4;
  if constexpr (D % 64 == 32) *reinterpret_cast<float2*>(row + 16 * B4 + 2 * m) = make_float2(v[B4], v[B4 + 1]);
  if constexpr (D % 64 == 16) row[16 * B4 + m] = v[B4];
}

// Buffer resource over one (b,h) slice, rows [0, N) of row stride rs floats (rs >= D): a row
// below 0 or at/after N reads as zeros.  The caller checked (N + max offset + 64) rs 4 < 2^31.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rsrc_f32(const void* base, long long off,
                                                                 long long rs, int N, int D) {
  float* const b = const_cast<float*>(static_cast<const float*>(base)) + off;
  return __builtin_amdgcn_make_buffer_rsrc(b, (short)0, (int)(((long long)(N - 1) * rs + D) * 4), 0x00020000);
}
__device__ __forceinline__ float4 bload4f(__amdgpu_buffer_rsrc_t r, int elem) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, (unsigned)elem * 4u, 0, 0));
}
__device__ __forceinline__ float bload1f(__amdgpu_buffer_rsrc_t r, int elem) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (unsigned)elem * 4u, 0, 0));
}

__device__ __forceinline__ void store4f_stream(float* p, float4 x) { st16_stream(p, __builtin_bit_cast(uint4, x)); }

__device__ __forceinline__ float dot4f(float4 a, float4 b, float acc) {
  return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, fmaf(a.x, b.x, acc))));
}
__device__ __forceinline__ void fma4f(float w, float4 x, float4& acc) {
  acc.x = fmaf(w, x.x, acc.x); acc.y = fmaf(w, x.y, acc.y);
  acc.z = fmaf(w, x.z, acc.z); acc.w = fmaf(w, x.w, acc.w);
}
// Stays 0 over finite values and becomes NaN at the first infinity or NaN.
__device__ __forceinline__ float nonfinite_mark(float4 x, float mark) {
  return fmaf(x.w, 0.f, fmaf(x.z, 0.f, fmaf(x.y, 0.f, fmaf(x.x, 0.f, mark))));
}

// lgkmcnt(0) and a wave barrier: this wave's LDS writes are visible to its lanes.
__device__ __forceinline__ void lds_wave_sync() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
}

// scale_embed [J, D] as 48 rows of stride RV in LDS (rows past J zero), and the per-tap bias and
// gain: requested ahead of a kernel's bulk loads (load) and stored once the window rows are
// (store).  Loads return in order, so requested last they would make the first barrier wait for the
// long-range blocks in flight.
template <int D, bool HAS_SE>
struct TapParams {
  static constexpr int U = HAS_SE ? (kMaxTaps * GeoF<D>::CPR + kBlock - 1) / kBlock : 1;
  float4 x[U];
  float bias, gain;
  __device__ __forceinline__ void load(const float* pos_bias, const float* score_gain, const float* se, int J, int H,
                                       int h, int tid) {
    const int jc = tid < J ? tid : J - 1;
    bias = pos_bias[jc * H + h];
    gain = score_gain ? score_gain[h * J + jc] : 1.0f;
    if constexpr (HAS_SE) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = tid + u * kBlock, j = e / GeoF<D>::CPR, d = 4 * (e - j * GeoF<D>::CPR);
        x[u] = se && j < J ? *reinterpret_cast<const float4*>(se + j * D + d) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  }
  // Returns mark, made NaN by an infinity or NaN of scale_embed.
  __device__ __forceinline__ float store(float* sBias, float* sGain, float* sSE, int J, int tid, float mark) const {
    if (tid < kMaxTaps) {
      sBias[tid] = tid < J ? bias : 0.f;
      sGain[tid] = tid < J ? gain : 1.0f;
    }
    if constexpr (HAS_SE) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = tid + u * kBlock, j = e / GeoF<D>::CPR, d = 4 * (e - j * GeoF<D>::CPR);
        if (e < kMaxTaps * GeoF<D>::CPR) {
          mark = nonfinite_mark(x[u], mark);
          *reinterpret_cast<float4*>(sSE + j * GeoF<D>::RV + d) = x[u];
        }
      }
    }
    return mark;
  }
};

// Whether every row a kernel touches stays within 32-bit buffer offsets, and rows do not overlap.
inline bool f32_mfma_strides_ok(int N, int maxd, int D, const long long* rs, int n) {
  for (int k = 0; k < n; ++k)
    if (rs[k] < D || ((long long)N + maxd + 64) * rs[k] * 4 >= (1LL << 31)) return false;
  return true;
}

}  // namespace dsqg
