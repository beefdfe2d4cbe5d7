// Weight and bias gradients of a linear layer y = x W^T + b over many rows (gfx950):
//
//     dW[o,i] = sum_t dy[t,o] x[t,i],     db[o] = sum_t dy[t,o],
//
// dy [T,O], x [T,I], both bf16 or both f16, sums in float32, results in that type (rounded once) or
// in float32 (the parameters' type under autocast: no cast afterwards).
//
// A model's weight is small and its row count is not (256 x 256 over 16384 rows): a product tiled
// over the output alone has a handful of tiles, each walking every row (the library's choice for
// 256 x 256 takes 104 us, its column sum for db another 23).  Here the rows are split too:
// workgroup (split, tile) sums 128 x 128 outputs over its rows into a float32 partial, and a second
// launch adds the partials of every element in order.  At 256 x 256 over 16384 rows (f16) the two
// launches take 17 us for dW and db.  Few rows (one split) go straight to the results in one launch: a
// step of a bf16 layer of 3072 x 768 over 77 rows took 35.0 us of GPU time through partials, takes
// 27.6 so, and 31.9 with the library's product and sum.
//
// The contraction runs over rows, so both operands are read transposed from row-major LDS tiles
// with ds_read_tr16_b64; two reads of 16 rows make one 16x16x32 operand (both operands take the
// rows in the same order).  LDS rows are 144 elements apart: the sixteen rows of a transposed read
// then meet each bank twice, the minimum.  Tiles of 64 rows, two buffers, the next tile's loads in
// flight during the products.  db is summed from the loaded registers by the first column of tiles.
#include "../../include/dsqg.h"
#include "dsqg_common.hpp"
#include "dsqg_mfma.hpp"

namespace dsqg {
namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr int kTile = 128;     // outputs per workgroup and direction
constexpr int kRows = 64;      // rows per LDS tile
constexpr int kRv = kTile + 16;  // LDS row stride (elements)

struct LinearParams {
  const void* dy; long long dys;
  const void* x; long long xs;
  void* dw; void* db;
  float* part;     // [splits][O][I]
  float* part_b;   // [splits][O]
  int T, O, I;
  int splits, rows_per;  // rows per split, a multiple of kRows
  int to, ti;            // tiles per direction
  bool out32;            // results in float32, else in the operands' type
};

template <bool F16>
__device__ __forceinline__ f32x4_t mfma_16(uint4 a, uint4 b, f32x4_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return mfma_16x16x32(as_bf16x8(a), as_bf16x8(b), c);
}

template <bool F16>
__device__ __forceinline__ float elem(unsigned w, int hi) {
  if constexpr (F16) return (float)__builtin_bit_cast(_Float16, (unsigned short)(hi ? w >> 16 : w));
  return __uint_as_float(hi ? w & 0xffff0000u : w << 16);
}

template <bool F16>
__device__ __forceinline__ void store_result(void* out, long long e, float v, bool out32) {
  if (out32) static_cast<float*>(out)[e] = v;
  else if constexpr (F16) static_cast<_Float16*>(out)[e] = (_Float16)v;
  else static_cast<bf16_t*>(out)[e] = (bf16_t)cvt_pk_bf16(v, v);
}

// Rows [r0, r0 + 16) and [r0 + 16, r0 + 32) of 16 columns from c0, transposed: this lane's column
// c0 + l%16, eight rows.
__device__ __forceinline__ uint4 tr_operand(const bf16_t* p) {
  const uint2 a = __builtin_bit_cast(uint2, lds_read_tr16(p));
  const uint2 b = __builtin_bit_cast(uint2, lds_read_tr16(p + 16 * kRv));
  return make_uint4(a.x, a.y, b.x, b.y);
}

template <bool F16>
__global__ __launch_bounds__(kBlock, 2) void linear_wgrad_kernel(LinearParams p) {
  __shared__ __align__(16) bf16_t sY[2][kRows * kRv];
  __shared__ __align__(16) bf16_t sX[2][kRows * kRv];
  const int tid = threadIdx.x;
  // Consecutive workgroups are the tiles of one split: they share its rows, and an XCD's L2.
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int tiles = p.to * p.ti;
  const int split = lb / tiles, tile = lb - split * tiles;
  const int o0 = tile / p.ti * kTile, i0 = (tile % p.ti) * kTile;
  const int r_begin = split * p.rows_per;
  const int r_end = min(p.T, r_begin + p.rows_per);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, g = l >> 4;
  const bool with_db = p.part_b != nullptr && i0 == 0;

  const int dys = (int)p.dys, xs = (int)p.xs;
  const __amdgpu_buffer_rsrc_t rY = slice_rsrc(static_cast<const bf16_t*>(p.dy), p.dys, r_end, p.O);
  const __amdgpu_buffer_rsrc_t rX = slice_rsrc(static_cast<const bf16_t*>(p.x), p.xs, r_end, p.I);
  // This thread's 16-byte piece: column 8 (tid % 16) of rows tid / 16 + 16u; a column past the
  // matrix reads zeros, and so does a row past the split.
  const int rr = tid >> 4, cc = 8 * (tid & 15);
  const int ylane = o0 + cc < p.O ? rr * dys + o0 + cc : kNoElem;
  const int xlane = i0 + cc < p.I ? rr * xs + i0 + cc : kNoElem;
  uint4 ly[4], lx[4];
  auto load = [&](int r) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ly[u] = bload16(rY, (r + 16 * u) * dys + ylane);
      lx[u] = bload16(rX, (r + 16 * u) * xs + xlane);
    }
  };
  float sum[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = 0.f;
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      st16(&sY[buf][(rr + 16 * u) * kRv + cc], ly[u]);
      st16(&sX[buf][(rr + 16 * u) * kRv + cc], lx[u]);
    }
    if (with_db) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const unsigned v[4] = {ly[u].x, ly[u].y, ly[u].z, ly[u].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] += elem<F16>(v[e >> 1], e & 1);
      }
    }
  };

  f32x4_t acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = zero4();

  // Wave w: outputs 64 (w / 2) .. +63 by 64 (w % 2) .. +63 of the tile.
  const int lane = (4 * g + (i >> 2)) * kRv + 4 * (i & 3);
  const int ow = 64 * (w >> 1), iw = 64 * (w & 1);
  load(r_begin);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int r = r_begin; r < r_end; r += kRows, buf ^= 1) {
    const bool more = r + kRows < r_end;
    if (more) load(r + kRows);
#pragma unroll
    for (int k = 0; k < kRows; k += 32) {
      uint4 A[4], B[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        A[t] = tr_operand(&sY[buf][k * kRv + ow + 16 * t + lane]);
        B[t] = tr_operand(&sX[buf][k * kRv + iw + 16 * t + lane]);
      }
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = mfma_16<F16>(A[a], B[b], acc[a][b]);
    }
    if (more) store(buf ^ 1);  // its readers passed the last barrier
    __syncthreads();
  }

  const bool direct = p.splits == 1;
  float* const part = p.part + (long long)split * p.O * p.I;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = o0 + ow + 16 * a + 4 * g + r;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int c = i0 + iw + 16 * b + i;
        if (o < p.O && c < p.I) {
          if (direct) store_result<F16>(p.dw, (long long)o * p.I + c, acc[a][b][r], p.out32);
          else part[(long long)o * p.I + c] = acc[a][b][r];
        }
      }
    }
  if (with_db) {
    float* const red = reinterpret_cast<float*>(sY[0]);  // [16][128] sums, the tiles are done
#pragma unroll
    for (int e = 0; e < 8; ++e) red[rr * kTile + cc + e] = sum[e];
    __syncthreads();
    if (tid < kTile && o0 + tid < p.O) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) s += red[k * kTile + tid];
      if (direct) store_result<F16>(p.db, o0 + tid, s, p.out32);
      else p.part_b[(long long)split * p.O + o0 + tid] = s;
    }
  }
}

// Sum of the splits' partials, four elements per lane; a workgroup's four waves take a quarter of
// the splits each and meet in LDS (in wave order).  n is the element count (a multiple of 4).
template <bool F16, bool OUT32>
__device__ __forceinline__ void reduce_four(const float* part, void* out, long long n, long long blk, int splits,
                                            float4 (&sh)[4][64]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const long long e = (blk * 64 + l) * 4;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (e < n) {
#pragma unroll 8
    for (int k = w; k < splits; k += 4) {
      const float4 v = *reinterpret_cast<const float4*>(part + k * n + e);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
  }
  sh[w][l] = s;
  __syncthreads();
  if (w == 0 && e < n) {
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      s.x += sh[k][l].x; s.y += sh[k][l].y; s.z += sh[k][l].z; s.w += sh[k][l].w;
    }
    if constexpr (OUT32) {
      *reinterpret_cast<float4*>(static_cast<float*>(out) + e) = s;
      return;
    }
    uint2 o;
    if constexpr (F16) {
      typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
      o = __builtin_bit_cast(uint2, (f16x4_t){(_Float16)s.x, (_Float16)s.y, (_Float16)s.z, (_Float16)s.w});
    } else {
      o = pack_bf16x4_u2(s.x, s.y, s.z, s.w);
    }
    *reinterpret_cast<uint2*>(static_cast<bf16_t*>(out) + e) = o;
  }
}

template <bool F16, bool OUT32>
__global__ __launch_bounds__(kBlock) void linear_reduce_kernel(LinearParams p, int w_blocks) {
  __shared__ float4 sh[4][64];
  if ((int)blockIdx.x < w_blocks)
    reduce_four<F16, OUT32>(p.part, p.dw, (long long)p.O * p.I, blockIdx.x, p.splits, sh);
  else
    reduce_four<F16, OUT32>(p.part_b, p.db, p.O, blockIdx.x - w_blocks, p.splits, sh);
}

// One 128 x 128 tile per CU and split: as many splits as give a workgroup to every CU, of at least
// four LDS tiles each.
void linear_plan(LinearParams& p) {
  p.to = (p.O + kTile - 1) / kTile;
  p.ti = (p.I + kTile - 1) / kTile;
  const int tiles = p.to * p.ti;
  int splits = (256 + tiles - 1) / tiles;
  const int most = (p.T + 4 * kRows - 1) / (4 * kRows);
  if (splits > most) splits = most;
  p.rows_per = ((p.T + splits - 1) / splits + kRows - 1) / kRows * kRows;
  p.splits = (p.T + p.rows_per - 1) / p.rows_per;
}

size_t linear_align(size_t x) { return (x + 255) & ~size_t(255); }

int linear_check(const dsqg_linear_wgrad_args* a, LinearParams* p) {
  if (!a || a->T < 0 || a->O <= 0 || a->I <= 0 || a->O % 8 != 0 || a->I % 8 != 0) return DSQG_EINVAL;
  if (a->dtype != DSQG_BF16 && a->dtype != DSQG_F16) return DSQG_EINVAL;
  if (a->out_dtype != a->dtype && a->out_dtype != DSQG_F32) return DSQG_EINVAL;
  if (a->T == 0 || (long long)a->O * a->I >= (1ll << 31)) return DSQG_EUNSUPPORTED;
  *p = LinearParams{};
  p->T = a->T; p->O = a->O; p->I = a->I;
  linear_plan(*p);
  return DSQG_OK;
}

}  // namespace
}  // namespace dsqg

using namespace dsqg;

extern "C" int dsqg_linear_wgrad_workspace_size(const dsqg_linear_wgrad_args* a, size_t* bytes) {
  if (!bytes) return DSQG_EINVAL;
  LinearParams p;
  const int rc = linear_check(a, &p);
  if (rc != DSQG_OK) return rc;
  *bytes = linear_align(sizeof(float) * (size_t)p.splits * p.O * p.I) + linear_align(sizeof(float) * (size_t)p.splits * p.O);
  return DSQG_OK;
}

extern "C" int dsqg_linear_wgrad(const dsqg_linear_wgrad_args* a, dsqg_stream_t stream) {
  LinearParams p;
  const int rc = linear_check(a, &p);
  if (rc != DSQG_OK) return rc;
  auto bad = [](const void* ptr) { return !ptr || (reinterpret_cast<uintptr_t>(ptr) & 15u) != 0; };
  if (bad(a->dy) || bad(a->x) || bad(a->dw) || (a->db && bad(a->db))) return DSQG_EINVAL;
  if (a->dy_stride < a->O || a->dy_stride % 8 != 0 || a->x_stride < a->I || a->x_stride % 8 != 0) return DSQG_EINVAL;
  // Rows are addressed with 32-bit byte offsets, up to a tile past the last.
  if (((long long)a->T + 2 * kRows) * a->dy_stride * 2 >= (1ll << 31) ||
      ((long long)a->T + 2 * kRows) * a->x_stride * 2 >= (1ll << 31))
    return DSQG_EUNSUPPORTED;
  const size_t wbytes = linear_align(sizeof(float) * (size_t)p.splits * p.O * p.I);
  if (!a->workspace || (reinterpret_cast<uintptr_t>(a->workspace) & 255u) ||
      a->workspace_bytes < wbytes + linear_align(sizeof(float) * (size_t)p.splits * p.O))
    return DSQG_EWORKSPACE;
  p.dy = a->dy; p.dys = a->dy_stride;
  p.x = a->x; p.xs = a->x_stride;
  p.dw = a->dw; p.db = a->db;
  p.out32 = a->out_dtype == DSQG_F32;
  p.part = static_cast<float*>(a->workspace);
  p.part_b = a->db ? reinterpret_cast<float*>(static_cast<char*>(a->workspace) + wbytes) : nullptr;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)(p.splits * p.to * p.ti));
  const int w_blocks = (int)(((long long)p.O * p.I + 255) / 256);
  const dim3 rgrid((unsigned)(w_blocks + (a->db ? (p.O + 255) / 256 : 0)));
  if (a->dtype == DSQG_F16) hipLaunchKernelGGL((linear_wgrad_kernel<true>), grid, dim3(kBlock), 0, st, p);
  else hipLaunchKernelGGL((linear_wgrad_kernel<false>), grid, dim3(kBlock), 0, st, p);
  if (p.splits == 1) return hipGetLastError() == hipSuccess ? DSQG_OK : DSQG_EHIP;
  if (p.out32) hipLaunchKernelGGL((linear_reduce_kernel<false, true>), rgrid, dim3(kBlock), 0, st, p, w_blocks);
  else if (a->dtype == DSQG_F16) hipLaunchKernelGGL((linear_reduce_kernel<true, false>), rgrid, dim3(kBlock), 0, st, p, w_blocks);
  else hipLaunchKernelGGL((linear_reduce_kernel<false, false>), rgrid, dim3(kBlock), 0, st, p, w_blocks);
  return hipGetLastError() == hipSuccess ? DSQG_OK : DSQG_EHIP;
}
