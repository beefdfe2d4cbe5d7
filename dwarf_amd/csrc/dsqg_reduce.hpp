// Parameter-gradient reduction (dbias, dscore_gain and dif_gain one wave per output element,
// dscale_embed a workgroup per 32 elements): shared by bwd_reduce_kernel (dsqg_bwd.hip) and the extra workgroups
// of the MFMA dk/dv launches (dsqg_bwd_dkdv_mfma.hip, dsqg_bwd_dkdv_f32.hip), which run it next to
// the dk/dv tiles.
#pragma once

#include "dsqg_common.hpp"

namespace dsqg {

// One wave per parameter-gradient element: lane l sums partials l, l+64, ... in order, then a
// fixed xor-tree combines the lanes, so the result is the same on every run.
__device__ __forceinline__ float wave_sum_fixed(float x) {
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) x += __shfl_xor(x, s, 64);
  return x;
}

__device__ __forceinline__ void reduce_params_wave(const ReduceParams& r, int t, int lane) {
  const int JH = r.J * r.H;
  const int per_h = r.B * r.n_chunks;  // partials per head, ordered (batch group, chunk)
  if (t < JH) {  // dpos_bias[j,h]
    const int j = t / r.H, h = t - j * r.H;
    float s = 0.f;
    for (int k = lane; k < per_h; k += 64) {
      const int bb = k / r.n_chunks, c = k - bb * r.n_chunks;
      s += r.part_bias[((long long)(bb * r.H + h) * r.n_chunks + c) * r.J + j];
    }
    s = wave_sum_fixed(s);
    if (lane == 0) r.dpos_bias[t] = s;
    return;
  }
  t -= JH;
  if (r.dscore_gain) {
    if (t < JH) {  // dscore_gain[h,j]
      const int h = t / r.J, j = t - h * r.J;
      float s = 0.f;
      for (int k = lane; k < per_h; k += 64) {
        const int bb = k / r.n_chunks, c = k - bb * r.n_chunks;
        s += r.part_gain[((long long)(bb * r.H + h) * r.n_chunks + c) * r.J + j];
      }
      s = wave_sum_fixed(s);
      if (lane == 0) r.dscore_gain[t] = s;
      return;
    }
    t -= JH;
  }
  if (r.dif_gain) {
    if (t < r.H) {
      float s = 0.f;
      for (int k = lane; k < per_h; k += 64) {
        const int bb = k / r.n_chunks, c = k - bb * r.n_chunks;
        s += r.part_if[(long long)(bb * r.H + t) * r.n_chunks + c];
      }
      s = wave_sum_fixed(s);
      if (lane == 0) r.dif_gain[t] = s;
      return;
    }
    t -= r.H;
  }
}

// dscale_embed: workgroup blk sums the partials of 32 consecutive elements of [J*D].  A thread
// takes four of them (16 bytes; eight lanes read 128 contiguous bytes) of every 32nd partial row,
// eight rows in flight, and the 32 row sums of an element meet in LDS.  Eight rows are added as a
// tree, sixteen such sums in turn, those in turn again, and the row sums as a tree: rounding grows
// with the levels and not with the rows (rms, relative, of unit normals: 3072 partials 1.0e-7, 65536
// 1.4e-7; one chain per thread and one over the rows 2.1e-7 and 9.0e-7).  lds: 32 x 32 floats.  At
// the start of the dk/dv grid these few workgroups finish long before its tiles do; as a launch of
// its own between dq and dk/dv (a first stage of 256 slices) the sum cost 5 us.
constexpr int kSeGroup = 32;

__device__ __forceinline__ float4 add4f(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

__device__ __forceinline__ void reduce_se_block(const ReduceParams& r, int blk, int tid, float* lds) {
  constexpr int kRowLanes = kBlock / 8;
  const int JD = r.J * r.D;  // a multiple of 16
  const int c = 4 * (tid & 7), row = tid >> 3;
  const int e = blk * kSeGroup + c;
  const int rows = r.B * r.H * r.n_chunks;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (e < JD) {
    const float* src = r.part_se + e;
    float4 run = acc;
    int n = 0;
    for (int k = row; k < rows; k += 8 * kRowLanes) {
      float4 x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int ku = k + u * kRowLanes;
        x[u] = *reinterpret_cast<const float4*>(src + (long long)(ku < rows ? ku : k) * JD);
        if (ku >= rows) x[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      run = add4f(run, add4f(add4f(add4f(x[0], x[1]), add4f(x[2], x[3])), add4f(add4f(x[4], x[5]), add4f(x[6], x[7]))));
      if (++n == 16) {
        acc = add4f(acc, run);
        run = make_float4(0.f, 0.f, 0.f, 0.f);
        n = 0;
      }
    }
    acc = add4f(acc, run);
  }
  *reinterpret_cast<float4*>(lds + row * kSeGroup + c) = acc;
  __syncthreads();
  if (tid < kSeGroup && blk * kSeGroup + tid < JD) {
    float s[kRowLanes];
#pragma unroll
    for (int k = 0; k < kRowLanes; ++k) s[k] = lds[k * kSeGroup + tid];
#pragma unroll
    for (int w = kRowLanes / 2; w > 0; w >>= 1)
#pragma unroll
      for (int k = 0; k < w; ++k) s[k] += s[k + w];
    r.dscale_embed[blk * kSeGroup + tid] = s[0];
  }
}

// Workgroups of the two parts: dscale_embed's (a multiple of the XCD count, so that the workgroups
// after them keep their XCDs) and the one-wave-per-element rest (an upper bound; surplus waves
// return at once).
inline int reduce_se_blocks(const ReduceParams& r) {
  if (!r.dscale_embed) return 0;
  return ((r.J * r.D + kSeGroup - 1) / kSeGroup + kNumXcd - 1) / kNumXcd * kNumXcd;
}
inline int reduce_wave_blocks(const ReduceParams& r) {
  return (int)((2LL * r.J * r.H + r.H + kBlock / 64 - 1) / (kBlock / 64));
}

}  // namespace dsqg
