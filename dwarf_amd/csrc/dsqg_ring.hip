// Loading a prompt's last rows into a layer's K/V ring (gfx950): row m of k and v, for
// m = max(0, N - S) .. N - 1, goes to slot m mod S of the rings, and every sequence's position
// becomes N.  One launch of 16-byte copies, each row read and written once; what it replaces
// (an index range, its remainder and two indexed writes, each with its own launch) took 15 us of
// GPU time and 50 of host time at B1 H8 N77 D32, this launch 2.7.
#include "../../include/dsqg.h"
#include "dsqg_common.hpp"

namespace dsqg {
namespace {

struct RingParams {
  const char* k; long long kb, kh, kn;  // strides in bytes
  const char* v; long long vb, vh, vn;
  char* k_ring; char* v_ring;
  long long* pos;
  int B, H, N, S, rows, lo, cpr;  // rows loaded, the first of them, 16-byte pieces of a row
};

__global__ __launch_bounds__(kBlock) void ring_load_kernel(RingParams p) {
  const int bh = blockIdx.y;
  const int b = bh / p.H, h = bh - b * p.H;
  if (h == 0 && blockIdx.x == 0 && threadIdx.x == 0) p.pos[b] = p.N;
  for (int e = blockIdx.x * kBlock + threadIdx.x; e < p.rows * p.cpr; e += gridDim.x * kBlock) {
    const int r = e / p.cpr, c = e - r * p.cpr;
    const int m = p.lo + r;
    const uint4 x = ld16(p.k + b * p.kb + h * p.kh + m * p.kn + 16 * c);
    const uint4 y = ld16(p.v + b * p.vb + h * p.vh + m * p.vn + 16 * c);
    const long long dst = (((long long)bh * p.S + m % p.S) * p.cpr + c) * 16;
    st16(p.k_ring + dst, x);
    st16(p.v_ring + dst, y);
  }
}

}  // namespace
}  // namespace dsqg

using namespace dsqg;

extern "C" int dsqg_ring_load(const dsqg_ring_load_args* a, dsqg_stream_t stream) {
  if (!a || a->B < 0 || a->H < 0 || a->N < 0 || a->S <= 0 || a->D <= 0) return DSQG_EINVAL;
  if (a->dtype != DSQG_F32 && a->dtype != DSQG_BF16 && a->dtype != DSQG_F16) return DSQG_EINVAL;
  const long long es = a->dtype == DSQG_F32 ? 4 : 2;
  if (a->D * es % 16 != 0) return DSQG_EINVAL;
  if ((long long)a->B * a->H > 65535 || (long long)a->S * (a->D * es / 16) >= (1ll << 31) - (1 << 28)) return DSQG_EUNSUPPORTED;
  if ((long long)a->B * a->H == 0) return DSQG_OK;
  auto bad = [](const void* ptr) { return !ptr || (reinterpret_cast<uintptr_t>(ptr) & 15u) != 0; };
  if (bad(a->k_ring) || bad(a->v_ring) || !a->pos) return DSQG_EINVAL;
  if (a->N > 0 && (bad(a->k) || bad(a->v))) return DSQG_EINVAL;
  for (int i = 0; i < 3; ++i)
    if (a->k_stride[i] < 0 || a->v_stride[i] < 0 || a->k_stride[i] * es % 16 != 0 || a->v_stride[i] * es % 16 != 0)
      return DSQG_EINVAL;
  RingParams p = {};
  p.k = static_cast<const char*>(a->k); p.kb = a->k_stride[0] * es; p.kh = a->k_stride[1] * es; p.kn = a->k_stride[2] * es;
  p.v = static_cast<const char*>(a->v); p.vb = a->v_stride[0] * es; p.vh = a->v_stride[1] * es; p.vn = a->v_stride[2] * es;
  p.k_ring = static_cast<char*>(a->k_ring); p.v_ring = static_cast<char*>(a->v_ring);
  p.pos = reinterpret_cast<long long*>(a->pos);
  p.B = a->B; p.H = a->H; p.N = a->N; p.S = a->S;
  p.lo = a->N > a->S ? a->N - a->S : 0;
  p.rows = a->N - p.lo;
  p.cpr = (int)(a->D * es / 16);
  // A thread per 16-byte piece, up to 32 workgroups per (b,h) (a 1537-slot ring of D = 64 takes 48
  // without the cap).
  const long long pieces = (long long)p.rows * p.cpr;
  long long gx = (pieces + kBlock - 1) / kBlock;
  gx = gx < 1 ? 1 : (gx > 32 ? 32 : gx);
  hipLaunchKernelGGL(ring_load_kernel, dim3((unsigned)gx, (unsigned)(a->B * a->H)), dim3(kBlock), 0,
                     reinterpret_cast<hipStream_t>(stream), p);
  return hipGetLastError() == hipSuccess ? DSQG_OK : DSQG_EHIP;
}
