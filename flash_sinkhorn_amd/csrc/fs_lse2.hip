// Instantiations and dispatch of the software-pipelined log-sum-exp kernel.
#include "fs_lse2.hpp"
#include "fs_lsecoarse.hpp"
#include "fs_lsecoarse128.hpp"
#include "fs_lsesparse.hpp"

#include "fs_dispatch.hpp"

namespace fs {

template <int DP, int RB, int PREC, bool VEC>
static int launch_cfg(const LaunchArgs& a, int blocks, hipStream_t st) {
  hipLaunchKernelGGL((lse2_kernel<DP, RB, PREC, VEC>), dim3(blocks), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <int DP, int PREC, bool VEC>
static int launch_rb(const LaunchArgs& a, int rb, int blocks, hipStream_t st) {
  if constexpr (DP <= 64) {
    if (rb >= 2) return launch_cfg<DP, 2, PREC, VEC>(a, blocks, st);
  }
  return launch_cfg<DP, 1, PREC, VEC>(a, blocks, st);
}

template <int PREC, bool VEC>
static int launch_dp(const LaunchArgs& a, int dp, int rb, int blocks, hipStream_t st) {
  switch (dp) {
    case 16: return launch_rb<16, PREC, VEC>(a, rb, blocks, st);
    case 32: return launch_rb<32, PREC, VEC>(a, rb, blocks, st);
    case 64: return launch_rb<64, PREC, VEC>(a, rb, blocks, st);
    case 128:
      if constexpr (!VEC) return launch_rb<128, PREC, false>(a, rb, blocks, st);
  }
  return FS_ERR_UNSUPPORTED;
}

int launch_absmax(const float* a, long long na, const float* b, long long nb, float* partial,
                  hipStream_t st) {
  hipLaunchKernelGGL(absmax_kernel, dim3(2 * kAbsmaxBlocks), dim3(256), 0, st, a, na, b, nb, partial);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int launch_fill_zero(unsigned* p, long long n, hipStream_t st) {
  if (n <= 0) return FS_OK;
  const long long grid = (n / 4 + 256) / 256;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)grid), dim3(256), 0, st, p, n);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int launch_split_planes_f16(const SplitArgs& a, hipStream_t st) {
  const int rows = a.n > 1 && a.m[1].rows > a.m[0].rows ? a.m[1].rows : a.m[0].rows;
  const long long items = (long long)(rows + kPlanePadRows) * (a.dp / 4);
  const int grid = (int)((items + 255) / 256);
  hipLaunchKernelGGL(split_planes_f16_kernel, dim3(grid, a.n), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

// fp16 planes, log-sum-exp, rows of at most 64 columns: the pipelined kernel with the coarse
// tile test (two blocks of 32 query rows per wavefront: the launch must be planned with rb = 2)
template <int DP>
static int launch_coarse_dp(const LaunchArgs& a, int blocks, hipStream_t st) {
  hipLaunchKernelGGL((lse_coarse_kernel<DP>), dim3(blocks), dim3(256), 0, st, a);
  // with carried margins both forms are enqueued; per side, the one the state words name runs
  if (a.side[0].margins != nullptr)
    hipLaunchKernelGGL((lse_sparse_kernel<DP>), dim3(a.blocks_sparse), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int launch_row_seeds(const LaunchArgs& a, int dp, int nsides, hipStream_t st) {
  const int sb0 = (a.side[0].nq + kSeedRows - 1) / kSeedRows;
  const int sb1 = nsides > 1 ? (a.side[1].nq + kSeedRows - 1) / kSeedRows : 0;
  LaunchArgs b = a;
  b.sel_pred = 0;
  hipLaunchKernelGGL((coarse_bias_kernel<0>), dim3((sb0 + sb1 + kBiasWaves - 1) / kBiasWaves), dim3(64 * kBiasWaves), 0,
                     st, b, 0, 0, sb0, sb0 + sb1, dp);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

static int launch_coarse(const LaunchArgs& a, int dp, int rb, int blocks, hipStream_t st) {
  if (rb != 2) return FS_ERR_BAD_ARGUMENT;
  // the per-tile records of the key bias, for both sides (tiles past the last key included)
  const int tiles0 = (a.side[0].nk + 63) / 64 + kAuxPadTiles;
  const int tiles1 = blocks > a.blocks0 ? (a.side[1].nk + 63) / 64 + kAuxPadTiles : 0;
  // behind them, per kSeedRows query rows one wavefront that computes where the rows' maxima start
  const bool seeds = a.side[0].seed != nullptr;
  const int sb0 = seeds ? (a.side[0].nq + kSeedRows - 1) / kSeedRows : 0;
  const int sb1 = seeds && blocks > a.blocks0 ? (a.side[1].nq + kSeedRows - 1) / kSeedRows : 0;
  const int groups = (tiles0 + tiles1 + kBiasWaves - 1) / kBiasWaves + (sb0 + sb1 + kBiasWaves - 1) / kBiasWaves;
  hipLaunchKernelGGL((coarse_bias_kernel<0>), dim3(groups), dim3(64 * kBiasWaves), 0, st, a, tiles0,
                     tiles0 + tiles1, sb0, sb0 + sb1, dp);
  if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  switch (dp) {
    case 16: return launch_coarse_dp<16>(a, blocks, st);
    case 32: return launch_coarse_dp<32>(a, blocks, st);
    case 64: return launch_coarse_dp<64>(a, blocks, st);
    case 128:  // lists of keys in place of margins
      if (a.side[0].margins != nullptr) return FS_ERR_BAD_ARGUMENT;
    {
      // in place a workgroup per row group and chunk; by lists the workgroups that test are shared out between the
      // sides by their logits
      LaunchArgs c = a;
      const bool both = blocks > a.blocks0;
      const double l0 = (double)a.side[0].nq * a.side[0].nk, l1 = both ? (double)a.side[1].nq * a.side[1].nk : 0.0;
      const int t0 = both ? std::min(kCoarse128Grid - 8, std::max(8, (int)(kCoarse128Grid * (l0 / (l0 + l1)) + 0.5))) : kCoarse128Grid;
      c.blocks_sparse = t0;
      c.blocks0 = std::max(a.blocks0, t0);
      hipLaunchKernelGGL((lse_coarse128_kernel<0>), dim3(c.blocks0 + (both ? std::max(blocks - a.blocks0, kCoarse128Grid - t0) : 0)),
                         dim3(256), 0, st, c);
      if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
      if (a.side[0].slack == nullptr) return FS_OK;  // (lists would not pay in this launch)
      c.blocks0 = (a.side[0].nq + 31) / 32;
      hipLaunchKernelGGL((lse_listed128_kernel<false>), dim3(c.blocks0 + (both ? (a.side[1].nq + 31) / 32 : 0)), dim3(256), 0, st, c);
      c.blocks0 = both ? kCoarse128Grid / 2 : kCoarse128Grid;
      hipLaunchKernelGGL((lse_listed128_kernel<true>), dim3(kCoarse128Grid), dim3(256), 0, st, c);
    }
      return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
  }
  return FS_ERR_UNSUPPORTED;
}

int launch_lse2(const LaunchArgs& a, int dp, int rb, int prec, bool vec, bool coarse, int blocks,
                hipStream_t st) {
  if (coarse && !vec && prec == kH3 && dp <= 128) return launch_coarse(a, dp, rb, blocks, st);
  if (vec) {  // plan-vector product: fp16 planes, rows of at most 64 columns
    return prec == kH3 ? launch_dp<kH3, true>(a, dp, rb, blocks, st) : FS_ERR_UNSUPPORTED;
  }
  switch (prec) {
    case kF32: return launch_dp<kF32, false>(a, dp, rb, blocks, st);
    case kH3: return launch_dp<kH3, false>(a, dp, rb, blocks, st);
  }
  return FS_ERR_BAD_ARGUMENT;
}

}  // namespace fs
