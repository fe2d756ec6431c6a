// Host side shared by the solvers that look at pinned words while the device runs, and the
// conjugate-gradient launches.
#pragma once

#include <hip/hip_runtime.h>

#include <chrono>

#include "flash_sinkhorn_hip.h"

namespace fs {

// Looks at pinned words until `arrived` says that what the device has to write is there (it
// arrives a few microseconds after the kernel wrote it); after two milliseconds waits for the
// stream instead.
template <typename F>
int wait_for_words(hipStream_t st, F&& arrived) {
  const auto t0 = std::chrono::steady_clock::now();
  for (int looks = 1; !arrived(); ++looks)
    if (looks % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2)) {
      if (hipStreamSynchronize(st) != hipSuccess) return FS_ERR_LAUNCH_FAILED;
      return arrived() ? FS_OK : FS_ERR_LAUNCH_FAILED;
    }
  return FS_OK;
}

// The launches behind fs_cg_init / fs_cg_update.  host: 8 pinned words that receive the state, the
// last of them, an int written behind the others, twice the number of iterations done (0: initialised)
// plus one where there is nothing left to do; or null.
int cg_init(const float* b, float* sol, float* res, float* dir, float* state, long long m, float rtol, float atol,
            float* host, hipStream_t st);
int cg_update(const float* a_dir, float* sol, float* res, float* dir, float* state, long long m, float* host, int iter,
              hipStream_t st);

// The arguments of the kernels of a solve of wide rows that left `workspace` behind (fs_small.hip), with one
// item and an extrapolation.
struct SmallArgs;
struct DenseArgs;
int dense_solved(const fs_small_problem* p, void* workspace, size_t workspace_bytes, SmallArgs& a, DenseArgs& t);

}  // namespace fs
