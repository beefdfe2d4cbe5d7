// K/V injection (train/train_2048_condU.py:178-181: k + k_delta, v + v_delta before the attention):
// one pass over a projection output qkv [B,N,3*H*D] and the two deltas, written as the operands the
// attention kernels take, K + k_delta and V + v_delta, and q as well where qkv has another type than
// they compute in (float16 under autocast becomes bfloat16).  Each operand is rounded to the output
// type before the sum, as the casts it replaces did, and the sum once.
//
// Bound by memory: at B8 N2048, 8 heads of 32, bfloat16, 50 MB in 9.8 us (5.1 TB/s; the two adds it
// replaces took 15), and under autocast, with q, 67 MB in 13.9 us (the cast of qkv, the casts of the
// deltas' head-permuted views and the adds took 59).
#include "../../include/dsqg.h"
#include "dsqg_common.hpp"

namespace dsqg {
namespace {

struct InjectParams {
  const void* qkv; long long qb, qn;
  const void* kd; long long kb, kh, kn;
  const void* vd; long long vb, vh, vn;
  void* q_out; void* k_out; void* v_out;
  long long ob, on;
  int N, H, D, E8;  // E8: 8-element pieces of a token's H*D
  long long pieces;
};

template <int DT>
__device__ __forceinline__ void load8(const void* base, long long e, float (&x)[8]) {
  if constexpr (DT == DSQG_F32) {
    Vec8<float>::load(static_cast<const float*>(base) + e, x);
  } else if constexpr (DT == DSQG_BF16) {
    Vec8<bf16_t>::load(static_cast<const bf16_t*>(base) + e, x);
  } else {
    typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
    const f16x8_t v = __builtin_bit_cast(f16x8_t, ld16(static_cast<const bf16_t*>(base) + e));
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (float)v[i];
  }
}

// x rounded to the output type (bf16 or f32).
template <int DT, int ODT>
__device__ __forceinline__ void round8(float (&x)[8]) {
  if constexpr (ODT == DSQG_BF16 && DT != DSQG_BF16) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(f32_to_bf16(x[i]) << 16);
  }
}

template <int ODT>
__device__ __forceinline__ void store8(void* base, long long e, const float (&x)[8]) {
  if constexpr (ODT == DSQG_F32) Vec8<float>::store(static_cast<float*>(base) + e, x);
  else Vec8<bf16_t>::store(static_cast<bf16_t*>(base) + e, x);
}

// DT: type of qkv and of both deltas; ODT: of the outputs.
template <int DT, int ODT>
__global__ __launch_bounds__(kBlock) void kv_inject_kernel(InjectParams p) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= p.pieces) return;
  const long long bn = t / p.E8;
  const int e = 8 * (int)(t - bn * p.E8), E = 8 * p.E8;
  const long long b = bn / p.N, n = bn - b * p.N;
  const int h = e / p.D, d = e - h * p.D;
  const long long src = b * p.qb + n * p.qn + e, dst = b * p.ob + n * p.on + e;
  float k[8], v[8], kd[8], vd[8], q[8];
  load8<DT>(p.qkv, src + E, k);
  load8<DT>(p.qkv, src + 2 * E, v);
  load8<DT>(p.kd, b * p.kb + h * p.kh + n * p.kn + d, kd);
  load8<DT>(p.vd, b * p.vb + h * p.vh + n * p.vn + d, vd);
  if (p.q_out) load8<DT>(p.qkv, src, q);
  round8<DT, ODT>(k); round8<DT, ODT>(v);
  round8<DT, ODT>(kd); round8<DT, ODT>(vd);
#pragma unroll
  for (int i = 0; i < 8; ++i) { k[i] += kd[i]; v[i] += vd[i]; }
  store8<ODT>(p.k_out, dst, k);
  store8<ODT>(p.v_out, dst, v);
  if (p.q_out) store8<ODT>(p.q_out, dst, q);
}

template <int DT, int ODT>
void launch(const InjectParams& p, hipStream_t st) {
  hipLaunchKernelGGL((kv_inject_kernel<DT, ODT>), dim3((unsigned)((p.pieces + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, st, p);
}

}  // namespace
}  // namespace dsqg

using namespace dsqg;

extern "C" int dsqg_kv_inject(const dsqg_kv_inject_args* a, dsqg_stream_t stream) {
  if (!a || a->B < 0 || a->H < 0 || a->N < 0 || a->D <= 0 || a->D % 8 != 0) return DSQG_EINVAL;
  auto size = [](int dt) { return dt == DSQG_F32 ? 4 : (dt == DSQG_BF16 || dt == DSQG_F16) ? 2 : 0; };
  if (!size(a->qkv_dtype) || !size(a->delta_dtype)) return DSQG_EINVAL;
  if (a->out_dtype != DSQG_F32 && a->out_dtype != DSQG_BF16) return DSQG_EINVAL;
  if ((long long)a->B * a->H * a->N == 0) return DSQG_OK;
  auto bad = [](const void* ptr) { return !ptr || (reinterpret_cast<uintptr_t>(ptr) & 15u) != 0; };
  if (bad(a->qkv) || bad(a->k_delta) || bad(a->v_delta) || bad(a->k_out) || bad(a->v_out) || (a->q_out && bad(a->q_out)))
    return DSQG_EINVAL;
  for (int i = 0; i < 2; ++i)
    if (a->qkv_stride[i] < 0 || a->qkv_stride[i] * size(a->qkv_dtype) % 16 != 0 || a->out_stride[i] < 0 ||
        a->out_stride[i] * size(a->out_dtype) % 16 != 0)
      return DSQG_EINVAL;
  for (int i = 0; i < 3; ++i)
    if (a->k_delta_stride[i] < 0 || a->k_delta_stride[i] * size(a->delta_dtype) % 16 != 0 || a->v_delta_stride[i] < 0 ||
        a->v_delta_stride[i] * size(a->delta_dtype) % 16 != 0)
      return DSQG_EINVAL;
  InjectParams p = {};
  p.qkv = a->qkv; p.qb = a->qkv_stride[0]; p.qn = a->qkv_stride[1];
  p.kd = a->k_delta; p.kb = a->k_delta_stride[0]; p.kh = a->k_delta_stride[1]; p.kn = a->k_delta_stride[2];
  p.vd = a->v_delta; p.vb = a->v_delta_stride[0]; p.vh = a->v_delta_stride[1]; p.vn = a->v_delta_stride[2];
  p.q_out = a->q_out; p.k_out = a->k_out; p.v_out = a->v_out;
  p.ob = a->out_stride[0]; p.on = a->out_stride[1];
  p.N = a->N; p.H = a->H; p.D = a->D; p.E8 = a->H * a->D / 8;
  p.pieces = (long long)a->B * a->N * p.E8;
  if (p.pieces > (1ll << 31)) return DSQG_EUNSUPPORTED;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // What the host layer asks for: operands of the output type, and float16 to bf16.
  if (a->delta_dtype != a->qkv_dtype) return DSQG_EUNSUPPORTED;
  if (a->qkv_dtype == DSQG_F32 && a->out_dtype == DSQG_F32) launch<DSQG_F32, DSQG_F32>(p, st);
  else if (a->qkv_dtype == DSQG_BF16 && a->out_dtype == DSQG_BF16) launch<DSQG_BF16, DSQG_BF16>(p, st);
  else if (a->qkv_dtype == DSQG_F16 && a->out_dtype == DSQG_BF16) launch<DSQG_F16, DSQG_BF16>(p, st);
  else return DSQG_EUNSUPPORTED;
  return hipGetLastError() == hipSuccess ? DSQG_OK : DSQG_EHIP;
}
