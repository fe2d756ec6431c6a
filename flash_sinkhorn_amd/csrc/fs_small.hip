// Small problems: planning, workspace and launches of the kernels in fs_small.hpp.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "flash_sinkhorn_hip.h"
#include "fs_small.hpp"

namespace fs {
namespace {

struct EpsTable {
  float e[kSmallTable];
};

// Schedule given by the caller: every item and problem takes the same entries.
template <int T>
__global__ __launch_bounds__(256) void small_table_kernel(const SmallArgs a, const EpsTable t) {
  float* out = a.table + (size_t)blockIdx.x * kSmallTable;
  for (int i = threadIdx.x; i < a.entries; i += 256) out[i] = t.e[i];
  if (threadIdx.x == 0) a.lens[blockIdx.x] = a.full[blockIdx.x] = a.entries;
}

int padded(int64_t d) { return d <= 16 ? 16 : (d <= 32 ? 32 : (d <= 64 ? 64 : 128)); }

int checked(const fs_small_problem* p) {
  if (!p || !p->x || !p->y) return FS_ERR_NULL_POINTER;
  if (p->n <= 0 || p->m <= 0 || p->d <= 0 || p->items <= 0 || p->items > 65535) return FS_ERR_BAD_SIZE;
  if (p->d > kSmallMaxD || p->n > FS_SMALL_MAX_ROWS || p->m > FS_SMALL_MAX_ROWS) return FS_ERR_UNSUPPORTED;
  if (p->dtype < 0 || p->dtype > 2 || p->sched < 0 || p->sched > 2) return FS_ERR_BAD_ARGUMENT;
  if (p->sched != 1 && p->entries <= 0) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 0 && !(p->eps > 0.f)) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 1 && !(p->blur > 0.0 && p->scaling > 0.0 && p->scaling < 1.0)) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 2) {
    if (!p->eps_list) return FS_ERR_NULL_POINTER;
    if (p->entries > kSmallTable) return FS_ERR_UNSUPPORTED;
    for (int i = 0; i < p->entries; ++i)
      if (!(p->eps_list[i] > 0.f)) return FS_ERR_BAD_ARGUMENT;
  }
  if (p->threshold > 0.f && p->check_every <= 0) return FS_ERR_BAD_ARGUMENT;
  return p->self_terms < 0 || p->self_terms > 2 ? FS_ERR_BAD_ARGUMENT : FS_OK;
}

// The kernels' arguments with the workspace laid out from `ws` (null: sizes only); returns the
// bytes the workspace takes.
size_t layout(const fs_small_problem* p, void* ws, SmallArgs& a) {
  std::memset(&a, 0, sizeof(a));
  a.pts[0] = p->x;
  a.pts[1] = p->y;
  a.w[0] = p->a;
  a.w[1] = p->b;
  a.dtype = p->dtype;
  a.normalize = p->normalize;
  a.rows[0] = (int)p->n;
  a.rows[1] = (int)p->m;
  a.d = (int)p->d;
  a.items = (int)p->items;
  a.self = p->self_terms;
  a.threshold = p->threshold;
  a.want_values = p->want_values ? 1 : 0;
  a.cost_scale = p->cost_scale;
  a.sched = p->sched;
  a.entries = p->entries;
  a.cut = p->cut;
  a.extrapolate = p->extrapolate ? 1 : 0;
  a.eps0 = p->eps;
  a.blur = p->blur;
  a.scaling = p->scaling;
  a.rho[0] = p->rho_x;
  a.rho[1] = p->rho_y;
  const int dp = padded(p->d), ndb = (dp + 31) / 32;
  size_t at = 0;
  char* base = static_cast<char*>(ws);
  auto take = [&](auto& ptr, size_t bytes) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(base + at);
    at += (bytes + 255) & ~(size_t)255;
  };
  const size_t items = (size_t)p->items;
  take(a.lens, items * 3 * 4);
  take(a.full, items * 3 * 4);
  take(a.scale, items * 2 * 4);
  take(a.stats, items * 2 * kSmallStatBlocks * kSmallStatWords * 4);
  if (p->sched != 0) take(a.table, items * 3 * kSmallTable * 4);
  for (int i = 0; i < 2; ++i) {
    const size_t rows = (size_t)a.rows[i];
    a.blocks[i] = (int)((rows + 31) / 32);
    const size_t blocks = items * (size_t)a.blocks[i];
    take(a.planes[i], blocks * (size_t)(2 * dp / 16) * 1024);
    if (a.want_values) take(a.values[i], blocks * (size_t)(ndb * 4) * 1024);
    take(a.norm[i], items * rows * 4);
    take(a.wt[i], items * rows * 4);
    take(a.l2w[i], items * rows * 4);
    take(a.pot[i], 2 * items * rows * 4);
    if (a.self) take(a.pot[2 + i], 2 * items * rows * 4);
    if (p->threshold > 0.f) {
      take(a.prev[i], items * rows * 4);
      if (a.self) take(a.prev[2 + i], items * rows * 4);
    }
  }
  return at;
}

template <int DP>
int launch_prep(const SmallArgs& a, hipStream_t st) {
  const int xb = a.blocks[0] > a.blocks[1] ? a.blocks[0] : a.blocks[1];
  hipLaunchKernelGGL((small_stats_kernel<0>), dim3(kSmallStatBlocks, 2, a.items), dim3(256), 0, st, a);
  hipLaunchKernelGGL((small_prep_kernel<DP>), dim3(xb + 1, 2, a.items), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <int DP>
int launch_step(const SmallArgs& a, int step, hipStream_t st) {
  const int blocks = (a.blocks[0] + a.blocks[1]) * (a.self == 1 ? 2 : 1);
#ifndef FS_SMALL_W
#define FS_SMALL_W 8
#endif
  constexpr int W = FS_SMALL_W;
  hipLaunchKernelGGL((small_step_kernel<DP, W>), dim3(blocks, a.items), dim3(64 * W), 0, st, a, step);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

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

template <int DP>
int launch_grad(const SmallArgs& a, const SmallGradArgs& g, hipStream_t st) {
  const int blocks = (g.out[0] ? a.blocks[0] : 0) + (g.out[1] ? a.blocks[1] : 0);
  hipLaunchKernelGGL((small_grad_kernel<DP>), dim3(blocks, a.items), dim3(512), 0, st, a, g);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <typename F>
int by_width(int64_t d, F&& f) {
  switch (padded(d)) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    default: return f(std::integral_constant<int, 128>{});
  }
}

}  // namespace
}  // namespace fs

using namespace fs;

extern "C" {

size_t fs_small_workspace_bytes(const fs_small_problem* p) {
  if (checked(p) != FS_OK) return 0;
  SmallArgs a;
  return layout(p, nullptr, a);
}

int fs_small_solve(const fs_small_problem* p, void* workspace, size_t workspace_bytes, int* host_words,
                   float* loss, float* pots, void* stream) {
  int rc = checked(p);
  if (rc != FS_OK) return rc;
  if ((p->sched == 1 || p->threshold > 0.f) && !host_words) return FS_ERR_NULL_POINTER;
  SmallArgs a;
  if (layout(p, workspace, a) > workspace_bytes || !workspace) return FS_ERR_WORKSPACE_TOO_SMALL;
  hipStream_t st = (hipStream_t)stream;
  int entries = a.entries;
  a.host_words = host_words;
  if (a.sched == 1) {
    static std::atomic<int> tokens{1};
    a.host_token = (tokens.fetch_add(1) & 0x3fffffff) + 1;
    for (int i = 0; i < a.items; ++i) __atomic_store_n(host_words + 4 * i + 3, 0, __ATOMIC_RELAXED);
    __atomic_thread_fence(__ATOMIC_SEQ_CST);
  } else if (a.sched == 2) {
    EpsTable t;
    std::memset(&t, 0, sizeof(t));
    std::memcpy(t.e, p->eps_list, (size_t)a.entries * sizeof(float));
    hipLaunchKernelGGL((small_table_kernel<0>), dim3(a.items * 3), dim3(256), 0, st, a, t);
    if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  }
  rc = by_width(p->d, [&](auto dp) { return launch_prep<decltype(dp)::value>(a, st); });
  if (rc != FS_OK) return rc;
  const int p0 = a.self == 2 ? 1 : 0, p1 = a.self == 0 ? 1 : 3;  // the problems that are solved
  if (a.sched == 1) {
    // how many steps there are is known on the device only
    rc = wait_for_words(st, [&]() {
      for (int i = 0; i < a.items; ++i)
        if (__atomic_load_n(host_words + 4 * i + 3, __ATOMIC_ACQUIRE) != a.host_token) return false;
      return true;
    });
    if (rc != FS_OK) return rc;
    entries = 0;
    for (int i = 0; i < a.items; ++i)
      for (int q = p0; q < p1; ++q) {
        const int k = host_words[4 * i + q];
        if (k <= 0) return k == -1 ? FS_SMALL_NO_DIAMETER : (k == -2 ? FS_SMALL_NOT_A_NUMBER : FS_SMALL_LONG_SCHEDULE);
        if (k > entries) entries = k;
      }
  }
  const int n_steps = entries + 1 + a.extrapolate;
  const bool early = a.threshold > 0.f;
  std::vector<int> length;  // early stopping: entries of every problem's schedule
  if (early)
    for (int i = 0; i < a.items; ++i)
      for (int q = 0; q < 4; ++q) {
        if (q < 3) length.push_back(a.sched == 1 ? host_words[4 * i + q] : entries);
        __atomic_store_n(host_words + 4 * i + q, -1, __ATOMIC_RELAXED);
      }
  int checks = 0;
  bool all_done = false;
  // waits for what check number c has to say; all_done: no problem has entries left to run
  auto check_result = [&](int c) {
    return wait_for_words(st, [&]() {
      all_done = true;
      for (int i = 0; i < a.items; ++i)
        for (int q = p0; q < p1; ++q) {
          const int v = __atomic_load_n(host_words + 4 * i + q, __ATOMIC_ACQUIRE);
          if ((v >= 0 && (v & 1)) || length[3 * i + q] < (c + 1) * p->check_every) continue;
          all_done = false;
          if (v < 2 * c) return false;
        }
      return true;
    });
  };
  for (int s = 0; s < n_steps && rc == FS_OK && !all_done; ++s) {
    rc = by_width(p->d, [&](auto dp) { return launch_step<decltype(dp)::value>(a, s, st); });
    if (rc != FS_OK || !early || s == 0 || s > entries || s % p->check_every != 0) continue;
    hipLaunchKernelGGL((small_check_kernel<0>), dim3(p1 - p0, a.items), dim3(1024), 0, st, a, s, checks);
    if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
    // (asked for with one more stretch of steps enqueued, so that the device does not wait)
    if (checks > 0) rc = check_result(checks - 1);
    ++checks;
  }
  if (rc == FS_OK && early && checks > 0 && !all_done) rc = check_result(checks - 1);
  if (rc != FS_OK || (!loss && !pots)) return rc;
  SmallLossArgs l;
  l.loss = loss;
  l.pots = pots;
  l.relaxed = a.rho[0] > 0.f && a.rho[1] > 0.f ? 1 : 0;
  hipLaunchKernelGGL((small_loss_kernel<0>), dim3(1, a.items), dim3(1024), 0, st, a, l);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int fs_small_grad(const fs_small_problem* p, void* workspace, size_t workspace_bytes, const float* grad_out,
                  float* grad_x, float* grad_y, void* stream) {
  const int rc = checked(p);
  if (rc != FS_OK) return rc;
  if (!grad_out) return FS_ERR_NULL_POINTER;
  if (!p->want_values) return FS_ERR_BAD_ARGUMENT;
  SmallArgs a;
  if (layout(p, workspace, a) > workspace_bytes || !workspace) return FS_ERR_WORKSPACE_TOO_SMALL;
  if (!grad_x && !grad_y) return FS_OK;
  SmallGradArgs g;
  g.grad_out = grad_out;
  g.out[0] = grad_x;
  g.out[1] = grad_y;
  return by_width(p->d, [&](auto dp) { return launch_grad<decltype(dp)::value>(a, g, (hipStream_t)stream); });
}

}  // extern "C"
