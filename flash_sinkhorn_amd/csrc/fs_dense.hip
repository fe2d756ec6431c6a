// Planning and launches of the kernels in fs_dense.hpp.
#include "fs_dense.hpp"

#include <algorithm>
#include <cmath>

namespace fs {
namespace {

// Tiles of a result in tiles of the kernel.
template <int WR, int WC, int RB, int CB>
int tile_up(DenseGemmArgs& g) {
  // (the transposed copy is read up to the end of its rows, so every column of it is written)
  g.row_tiles = ((g.out_t ? g.ld_t : g.rows) + 32 * WR * RB - 1) / (32 * WR * RB);
  g.col_tiles = g.ld / (32 * WC * CB);
  return g.row_tiles * g.col_tiles;
}

// Tiles of 64 x 64 run with eight stages of LDS, and two steps to a barrier, where a CU gets so few workgroups that it holds that
// many of each; with four where there are more: they cover each other's waits, four to a CU.
constexpr double kDeepTiles = 512.0;

template <int WR, int WC, int RB, int CB>
int launch_gemm(DenseGemmArgs& g, int items, hipStream_t st) {
  const int tiles = tile_up<WR, WC, RB, CB>(g);
  const dim3 grid((tiles + 7) / 8 * 8, items, g.splits), block(64 * WR * WC);
  if constexpr (WR * RB == 2)
    if ((double)tiles * items * g.splits <= kDeepTiles) {
      hipLaunchKernelGGL((dense_gemm_kernel<WR, WC, RB, CB, 8>), grid, block, 0, st, g);
      return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
    }
  hipLaunchKernelGGL((dense_gemm_kernel<WR, WC, RB, CB, 4>), grid, block, 0, st, g);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <int WR, int WC, int RB, int CB>
int launch_jobs(DenseGemmJobs& g, int jobs, int items, hipStream_t st, bool apart) {
  int tiles = 0;
  for (int i = 0; i < jobs; ++i) tiles = std::max(tiles, tile_up<WR, WC, RB, CB>(g.job[i]));
  const dim3 grid((tiles + 7) / 8 * 8, items, jobs), block(64 * WR * WC);
  if constexpr (WR * RB == 2)
    if ((double)tiles * items * jobs <= kDeepTiles) {
      if (apart) hipLaunchKernelGGL((dense_gemm_jobs_kernel<WR, WC, RB, CB, true, 8>), grid, block, 0, st, g);
      else hipLaunchKernelGGL((dense_gemm_jobs_kernel<WR, WC, RB, CB, false, 8>), grid, block, 0, st, g);
      return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
    }
  if (apart) hipLaunchKernelGGL((dense_gemm_jobs_kernel<WR, WC, RB, CB, true, 4>), grid, block, 0, st, g);
  else hipLaunchKernelGGL((dense_gemm_jobs_kernel<WR, WC, RB, CB, false, 4>), grid, block, 0, st, g);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

// Tiles of 256, 128 or 64 rows and columns: the one whose rounds over the chip cost least, a
// workgroup of the smaller ones taking longer per product (operands are read more often).  In units
// of a 256 x 256 tile's step; writing and adding up a part of a split contraction counts what
// 5 TB/s take.
double tile_cost(const DenseGemmArgs& g, int side, int splits, int items) {
  const int at_once = side == 256 ? 1 : (side == 128 ? 2 : 4);
  const double per = side == 256 ? 1.0 : (side == 128 ? 1.25 / 4 : 2.0 / 16);
  const double tiles = (double)items * splits * std::ceil(g.rows / (double)side) * (g.ld / side);
  const double traffic = splits == 1 ? 0.0 : splits * 8.0 * g.rows * g.ld / 5e6 / 1.3;
  return std::ceil(tiles / (256.0 * at_once)) * at_once * per * ((g.steps + splits - 1) / splits + 6) + traffic;
}
int best_side(const DenseGemmArgs& g, int splits, int items) {
  int best = 64;
  for (int side : {128, 256})
    if (g.ld % side == 0 && tile_cost(g, side, splits, items) <= tile_cost(g, best, splits, items)) best = side;
  return best;
}

// Rows of a wavefront where a step is one launch (dense_rows_kernel), else 0.  It reads the products twice (once
// transposed): while the L2s and the last-level cache serve that faster than a second launch and its merge take.
// Step by sweep and merge -> by rows, us: 500 points 8.2 -> 3.2, 1,000 7.5 -> 4.0, 2,000 13.3 -> 7.3, 2,500
// 16.0 -> 13.3, 3,000 20.5 -> 15.6, 1,000 x 4,000 11.5 -> 11.0, 4,000 points 23.0 -> 24.3.
int dense_rows(const SmallArgs& a, const DenseArgs& t) {
  if (std::max(t.ld, t.ld_t) > kDenseRowKeys || (double)a.items * t.n * t.m > 1.0e7) return 0;
  return (double)a.items * (t.n + t.m) <= 2048 ? 1 : 2;
}

}  // namespace

// How many parts the contraction is cut into (results of few tiles leave most of the chip idle).
void dense_gemm_plan(DenseGemmArgs& g, bool may_split) {
  g.splits = 1;
  if (may_split)
    for (int s = 2; s <= 16 && g.steps / s >= 8; ++s)
      if (tile_cost(g, best_side(g, s, 1), s, 1) < 0.95 * tile_cost(g, best_side(g, g.splits, 1), g.splits, 1)) g.splits = s;
  g.run = (g.steps + g.splits - 1) / g.splits;
  g.splits = (g.steps + g.run - 1) / g.run;
}

int dense_gemm(DenseGemmArgs& g, int items, hipStream_t st) {
  const int side = best_side(g, g.splits, items);
  if (side == 256) return launch_gemm<2, 4, 4, 2>(g, items, st);
  if (side == 128) return launch_gemm<2, 2, 2, 2>(g, items, st);
  return launch_gemm<2, 2, 1, 1>(g, items, st);
}

// (rows of every result padded to 256 columns, so that each takes any of the tiles)
int dense_gemm_jobs(DenseGemmJobs& g, int jobs, int items, hipStream_t st, bool apart) {
  int most = 0;
  for (int i = 1; i < jobs; ++i)
    if ((double)g.job[i].rows * g.job[i].ld > (double)g.job[most].rows * g.job[most].ld) most = i;
  const int side = best_side(g.job[most], 1, items * jobs);
  if (side == 256) return launch_jobs<2, 4, 4, 2>(g, jobs, items, st, apart);
  if (side == 128) return launch_jobs<2, 2, 2, 2>(g, jobs, items, st, apart);
  return launch_jobs<2, 2, 1, 1>(g, jobs, items, st, apart);
}

void dense_plan(const SmallArgs& a, DenseArgs& t) {
  t.n = a.rows[0];
  t.m = a.rows[1];
  t.items = a.items;
  for (int i = 0; i < 2; ++i) t.blocks[i] = (a.rows[i] + 255) / 256 * 8;
  t.ld = t.blocks[1] * 32;
  t.steps = (a.d + 15) / 16;
  // Two workgroups of 64 rows run on a CU at a time, each over a run of columns: the length whose rounds
  // over the chip cost least, counting a 256-column piece's time for what a workgroup does around
  // its run.  (With the longest run that still gives 512 workgroups the last round ran nearly empty
  // at most sizes: 6,000 x 6,000, 564 workgroups, 46.7 us a step against 39.5; 9,000 points 109
  // against 88; 12,000 169 against 145; 4,000 x 5,000 29.6 against 28.5.)
  // Where there is no work for 512, smaller ones, over 256 columns.
  const int iters = t.ld / 256, groups = (t.n + 63) / 64;
  t.large = (double)a.items * groups * iters >= 512.0;
  t.groups = t.large ? groups : (t.n + 31) / 32;
  int run = 1;
  double cost = 0.0;
  for (int r = 1; t.large && r <= iters; ++r) {
    const double c = std::ceil((double)a.items * groups * ((iters + r - 1) / r) / 512.0) * (r + 1);
    if (cost == 0.0 || c < cost) cost = c, run = r;
  }
  t.chunk = run * 256;
  t.chunks = (iters + run - 1) / run;
  t.ld_t = t.blocks[0] * 32;
  t.rows = dense_rows(a, t);
  t.turns = (size_t)a.items * t.n * t.ld * 4 > ((size_t)32 << 20);
}

int dense_prepare(const SmallArgs& a, const DenseArgs& t, hipStream_t st) {
  hipLaunchKernelGGL((dense_stats_kernel<0>), dim3(a.stat_blocks, 2, a.items), dim3(1024), 0, st, a);
  hipLaunchKernelGGL((dense_prep_kernel<0>), dim3(std::max(t.blocks[0], t.blocks[1]) + 1, 2, a.items), dim3(512), 0, st,
                     a, t);
  if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  DenseGemmArgs g;
  g.a = t.planes[0];
  g.b = t.planes[1];
  g.a_blocks = t.blocks[0];
  g.b_blocks = t.blocks[1];
  g.steps = t.steps;
  g.rows = t.n;
  g.ld = t.ld;
  g.scale[0] = a.scale;
  g.scale[1] = a.scale + 1;
  g.step_words = kDenseStep;
  g.plane_words = 64;
  g.out = t.dots;
  g.out_t = t.rows ? t.dots_t : nullptr;
  g.cols = t.m;
  g.ld_t = t.ld_t;
  dense_gemm_plan(g, false);
  return dense_gemm(g, a.items, st);
}

int dense_rows_step(const DenseRowArgs& t, int rows, bool raw, int sides, int items, hipStream_t st) {
  int most = 0;
  for (int i = 0; i < sides; ++i) most = std::max(most, t.s.side[i].nq);
  const dim3 grid((most + 8 * rows - 1) / (8 * rows), sides, items);
  auto* kernel = rows == 1 ? (raw ? dense_rows_kernel<1, true> : dense_rows_kernel<1, false>)
                           : (raw ? dense_rows_kernel<2, true> : dense_rows_kernel<2, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(512), 0, st, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int dense_step(const SmallArgs& a, DenseArgs& t, int step, hipStream_t st) {
  t.step = step;
  for (int i = 0; i < 2; ++i) {
    const size_t half = (size_t)a.items * a.rows[i];
    t.pot[i] = a.pot[i] + (step & 1) * half;
    t.out[i] = a.pot[i] + ((step & 1) ^ 1) * half;
  }
  const dim3 grid(t.groups, t.chunks, a.items);
  if (t.large) hipLaunchKernelGGL((dense_sweep_kernel<8, 8>), grid, dim3(512), 0, st, t);
  else hipLaunchKernelGGL((dense_sweep_kernel<8, 4>), grid, dim3(256), 0, st, t);
  hipLaunchKernelGGL((dense_merge_kernel<0>), dim3((std::max(t.n, t.m) + 63) / 64, 2, a.items), dim3(256), 0, st, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

}  // namespace fs
