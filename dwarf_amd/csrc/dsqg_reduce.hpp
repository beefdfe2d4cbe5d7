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
// eight rows in flight, and the 32 row sums of an element meet in LDS in order.  lds: 32 x 32
// floats.  At the start of the dk/dv grid these few workgroups finish long before its tiles do; as
// a launch of its own between dq and dk/dv (a first stage of 256 slices) the sum cost 5 us.
constexpr int kSeGroup = 32;

__device__ __forceinline__ void reduce_se_block(const ReduceParams& r, int blk, int tid, float* lds) {
  const int JD = r.J * r.D;  // a multiple of 16
  const int c = 4 * (tid & 7), row = tid >> 3;
  const int e = blk * kSeGroup + c;
  const int rows = r.B * r.H * r.n_chunks;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (e < JD) {
    const float* src = r.part_se + e;
#pragma unroll 8
    for (int k = row; k < rows; k += kBlock / 8) {
      const float4 x = *reinterpret_cast<const float4*>(src + (long long)k * JD);
      acc.x += x.x; acc.y += x.y; acc.z += x.z; acc.w += x.w;
    }
  }
  *reinterpret_cast<float4*>(lds + row * kSeGroup + c) = acc;
  __syncthreads();
  if (tid < kSeGroup && blk * kSeGroup + tid < JD) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kBlock / 8; ++k) s += lds[k * kSeGroup + tid];
    r.dscale_embed[blk * kSeGroup + tid] = s;
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
