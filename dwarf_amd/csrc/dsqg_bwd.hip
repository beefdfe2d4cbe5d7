// DSQG backward, launch 3 and the backward driver.
//
// bwd_reduce_kernel sums the per-workgroup parameter-gradient partials written by launch 1
// (dsqg_bwd_dq.hip / dsqg_bwd_dq_mfma.hip) in a fixed order, so dpos_bias / dscale_embed / dscore_gain / dif_gain are
// deterministic.  The reference accumulates dpb and dse with tl.atomic_add
// (kernels/dsqg_attention_v3.py:265-271), whose summation order varies run to run.
#include "dsqg_common.hpp"
#include "dsqg_launch.hpp"
#include "dsqg_f32.hpp"
#include "dsqg_reduce.hpp"

namespace dsqg {

__global__ __launch_bounds__(kBlock) void bwd_reduce_kernel(ReduceParams r, int se_blocks) {
  __shared__ __align__(16) float lds[kSeGroup * kBlock / 8];
  if ((int)blockIdx.x < se_blocks) {
    reduce_se_block(r, blockIdx.x, threadIdx.x, lds);
    return;
  }
  reduce_params_wave(r, (blockIdx.x - se_blocks) * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                     threadIdx.x & 63);
}

bool bwd_mfma_supported(const BwdParams& p, int D, int dtype) {
  if (dtype != 1) return false;
  long long rs = p.qs.n, rmin = p.qs.n;
  const long long all[4] = {p.qs.n, p.ks.n, p.vs.n, p.dos.n};
  for (long long x : all) { rs = x > rs ? x : rs; rmin = x < rmin ? x : rmin; }
  const long long span = ((long long)p.N + p.taps.maxd + 64) * rs * 2;
  return (D == 32 || D == 64 || D == 80 || D == 96 || D == 128) && p.taps.J - p.taps.W - 1 <= kMaxSparse &&
         rmin >= D && span < (1LL << 31);
}

bool bwd_f32_supported(const BwdParams& p, int D, int dtype) {
  const long long rs[4] = {p.qs.n, p.ks.n, p.vs.n, p.dos.n};
  return dtype == 0 && f32_mfma_strides_ok(p.N, p.taps.maxd, D, rs, 4);
}

// Batches a workgroup of the bf16 scale_embed dq takes (bwd_plan): the choice of 1, 2 and 4 whose
// rounds of resident workgroups times batches cost least, counting a partial's store and re-read
// as 0.6 of a tile.  Whole backward, us, at 1 / 2 / 4 batches, 11 long-range taps, without and with
// the score gain's gradient (fewer workgroups per CU, so other rounds):
//   B4 H4 N256 D64     22.5 / 32.1 / 51.5      23.6 / 33.9 / 55.1
//   B8 H8 N512 D32     21.5 / 26.8 / 39.6      23.0 / 28.3 / 42.3
//   B8 H8 N2048 D32    49.3 / 47.3 / 55.6      60.4 / 60.7 / 59.9
//   B16 H8 N2048 D32   86.3 / 82.9 / 81.1     101.5 / 94.7 / 102.5
//   B4 H8 N1024 D64    29.4 / 35.5 / 54.5      30.1 / 37.1 / 57.9
//   B2 H12 N2048 D64   34.2 / 42.0             45.2 / 46.5
//   B4 H8 N2048 D64    50.9 / 48.3 / 62.4      53.5 / 49.1 / 65.2
//   B8 H12 N2048 D64    113 / 108 / 105         139 / 130 / 138
//   B4 H8 N4096 D64    80.3 / 81.4 / 83.6      96.8 / 90.7 / 88.5
//   B4 H8 N2047 D80    63.5 / 61.5 / 76.8      90.2 / 83.5 / 80.8
//   B8 H8 N2048 D96     123 / 114 / 110         174 / 161 / 155
//   B2 H4 N1024 D128   36.7 / 54.0             37.9 / 57.1
//   B4 H8 N2048 D128    108 / 104 / 130         116 / 110 / 137
//   B8 H6 N2048 D128    156 / 161 / 168         164 / 170 / 180
// It takes the fastest, or one within 5 %, of each but the last (four: 8 and 10 % over one).  With
// one count for every form instead it took 2 at B4 H8 N2047 D80 and 4 at B8 H12 N2048 D64 with the
// gain's gradient, and with 14 taps 2 at B2 H12 N2048 D64 without it (45 us; one batch: 36).
static int se_batches(const BwdParams& p, int D, bool dg) {
  const int slots = 256 * bwd_dq_se_resident(D, p.taps.J - p.taps.W - 1, dg);
  int best = 1;
  double best_cost = 0;
  for (int n : {1, 2, 4}) {
    if (n > 1 && n / 2 >= p.B) break;
    const int nb = n < p.B ? n : (p.B > 0 ? p.B : 1);
    const long long wgs = (long long)((p.B + nb - 1) / nb) * p.H * p.n_tiles;
    const double cost = (double)nb * ((wgs + slots - 1) / slots) + 0.6 * wgs / slots;
    if (n == 1 || cost < best_cost) { best = nb; best_cost = cost; }
  }
  return best;
}

void bwd_plan(BwdParams& p, int D, int dtype, bool se, bool dg, bool compact) {
  const bool mfma = bwd_mfma_supported(p, D, dtype);
  const bool tile64 = mfma || bwd_f32_supported(p, D, dtype);
  const int QPB = tile64 ? 64 : kBlock / lanes_per_row(D);  // dq rows per tile
  const int KPB = tile64 ? 64 : kBlock / lanes_per_row(D);  // dk/dv rows per workgroup
  p.n_tiles = (p.N + QPB - 1) / QPB;
  p.n_tiles_kv = (p.N + KPB - 1) / KPB;
  // One tile per workgroup: the partial rows (J floats) are small next to a tile's loads, and the
  // single-tile form keeps no per-lane addresses across tiles.  The bf16 dq with scale_embed
  // takes the same head and tile of up to four batches per workgroup instead: its [J x D] fp32 dse
  // partial is as large as a tile's dS, so one per tile costs as many bytes again as the tile's
  // dq (written, then read back by the reduction); one per four tiles cuts them to a quarter, where
  // the grid still fills the chip (se_batches; compact: four, the smallest workspace).
  // (Four consecutive tiles of one (b,h) instead put every tile of four times as many (b,h)
  // slices in flight at once, which overflowed L2: 143 MB more L2-miss reads per launch.)
  // dse sums over every b and h, dbias / dg / da over b, so a partial may span batches.
  p.tiles_per_block = 1;
  p.n_chunks = p.n_tiles;
  p.batches_per_block = !(mfma && se) ? 1 : compact ? (p.B < 4 ? (p.B > 0 ? p.B : 1) : 4) : se_batches(p, D, dg);
  p.n_bgroups = (p.B + p.batches_per_block - 1) / p.batches_per_block;
}

hipError_t launch_bwd_reduce(const ReduceParams& r, hipStream_t st) {
  const int se = reduce_se_blocks(r), rest = reduce_wave_blocks(r);
  if (se + rest == 0) return hipSuccess;
  hipLaunchKernelGGL(bwd_reduce_kernel, dim3((unsigned)(se + rest)), dim3(kBlock), 0, st, r, se);
  return hipGetLastError();
}

}  // namespace dsqg
