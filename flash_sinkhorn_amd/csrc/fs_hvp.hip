// Hessian-vector products on kept inner products: workspace, launches, conjugate gradients.
#include "fs_host.hpp"
#include "fs_hvp.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

namespace fs {
namespace {

int checked(const fs_hvp_problem* p) {
  if (!p || !p->x || !p->y || !p->A || !p->f || !p->g) return FS_ERR_NULL_POINTER;
  if (p->n <= 0 || p->m <= 0 || p->d <= 0) return FS_ERR_BAD_SIZE;
  if (p->m > FS_HVP_MAX_COLUMNS || p->n > FS_SMALL_MAX_ROWS || p->d > FS_SMALL_MAX_D || p->n * p->m > FS_HVP_MAX_PLAN)
    return FS_ERR_UNSUPPORTED;
  if (p->dtype < 0 || p->dtype > 2 || !(p->eps > 0.f) || !(p->cost_scale > 0.f) || p->max_iter < 0) return FS_ERR_BAD_ARGUMENT;
  return FS_OK;
}

struct HvpPlan {
  SmallArgs pts, dir;      // preparation of x and y, of A
  DenseArgs td, ta;        // their planes
  DenseGemmArgs dots, prod, last;
  HvpArgs a;
};

// What a solve of the same points has left: nothing of it is formed again.
struct Kept {
  SmallArgs a;
  DenseArgs t;
};

// `shared`: the products come from a solve, `kept` where more than the sizes is asked for.
size_t layout(const fs_hvp_problem* p, void* ws, HvpPlan& q, bool shared, const Kept* kept = nullptr) {
  std::memset(&q, 0, sizeof(q));
  const int n = (int)p->n, m = (int)p->m, d = (int)p->d;
  size_t at = 0;
  char* base = static_cast<char*>(ws);
  auto take = [&](auto& ptr, size_t bytes) {
    ptr = reinterpret_cast<std::remove_cv_t<std::remove_reference_t<decltype(ptr)>>>(base + at);
    at += (bytes + 255) & ~(size_t)255;
  };
  // ---- the three matrices' planes ----
  auto prepare = [&](SmallArgs& s, DenseArgs& t, const void* first, const void* second, int rows0, int rows1, int dtype,
                     bool mine) {
    s.pts[0] = first;
    s.pts[1] = second;
    s.rows[0] = rows0;
    s.rows[1] = rows1;
    s.dtype = dtype;
    s.d = d;
    s.items = 1;
    s.cost_scale = p->cost_scale;
    s.eps0 = p->eps;
    s.stat_blocks = kSmallStatBlocks;
    s.stat_words = 2;
    s.table_len = 1;
    dense_plan(s, t);
    if (!mine) return;
    take(s.lens, 3 * 4);
    take(s.full, 3 * 4);
    take(s.table, 3 * (size_t)s.table_len * sizeof(float4));
    take(s.scale, 2 * sizeof(float2));
    take(s.stats, 2 * (size_t)s.stat_blocks * s.stat_words * 4);
    for (int i = 0; i < (second ? 2 : 1); ++i) {
      take(t.planes[i], (size_t)t.blocks[i] * t.steps * 2048);
      const size_t rows = s.rows[i];
      take(s.norm[i], rows * 4);
      take(s.wt[i], rows * 4);
      take(s.l2w[i], rows * 4);
      take(s.pot[i], rows * 4);
    }
  };
  prepare(q.pts, q.td, p->x, p->y, n, m, p->dtype, !shared);
  prepare(q.dir, q.ta, p->A, nullptr, n, m, 0, true);
  if (kept) {
    for (int i = 0; i < 2; ++i) {
      q.td.planes[i] = kept->t.planes[i];
      q.pts.norm[i] = kept->a.norm[i];
    }
    q.pts.scale = kept->a.scale;
  }
  HvpArgs& a = q.a;
  a.x = p->x;
  a.y = p->y;
  a.A = p->A;
  a.f = p->f;
  a.g = p->g;
  a.log_a = p->log_a;
  a.log_b = p->log_b;
  a.log_n = std::log((float)(1.0 / n));
  a.log_m = std::log((float)(1.0 / m));
  a.weighted = p->weighted;
  a.out_scale = p->out_scale;
  a.n = n;
  a.m = m;
  a.d = d;
  a.dtype = p->dtype;
  a.eps = p->eps;
  a.cs = p->cost_scale;
  a.lambda = p->lambda_indef;
  a.fac_x = p->rho_x > 0.f ? (p->rho_x + p->eps) / p->rho_x : 1.0f;
  a.fac_y = p->rho_y > 0.f ? (p->rho_y + p->eps) / p->rho_y : 1.0f;
  a.floor = std::max(1e-12f, p->eps * 1e-10f);
  a.ridge = p->rho_x > 0.f || p->rho_y > 0.f ? 0.f : p->eps * p->tau2;
  a.qs = 2.0f * p->cost_scale / p->eps * kLog2e;
  a.ld = q.td.ld;
  a.chunk = q.td.chunk;
  a.chunks = q.td.chunks;
  a.groups = q.td.groups;
  a.norm_x = q.pts.norm[0];
  a.norm_y = q.pts.norm[1];
  a.norm_a = q.dir.norm[0];
  a.scale = q.pts.scale;
  const size_t N = n, M = m, L = a.ld;
  if (!shared) take(a.dots, N * L * 4);
  if (kept) a.dots = kept->t.dots;
  take(a.prod, N * L * 4);
  for (float** r : {&a.xa, &a.ra, &a.mass, &a.r1, &a.inv_diag, &a.w, &a.alpha, &a.s, &a.v_scale}) take(*r, N * 4);
  for (float** r : {&a.cb, &a.denom, &a.r2, &a.vec, &a.sol, &a.res, &a.a_dir}) take(*r, L * 4);
  take(a.row_part, (size_t)a.chunks * N * sizeof(float2));
  take(a.col_part, (size_t)a.groups * M * sizeof(float2));
  // one strip per CU, of whole groups of rows
  const int r = a.ld <= 4096 ? 8 : 4;
  a.strip_rows = std::max(1, (n + 256 * r - 1) / (256 * r)) * r;
  a.strips = (n + a.strip_rows - 1) / a.strip_rows;
  take(a.strip_part, (size_t)a.strips * L * 4);
  take(a.limits, 8);
  take(a.cg, 8 * 4);
  // ---- V y ----
  a.ldo = d <= 64 ? 64 : (d <= 128 ? 128 : (d + 255) / 256 * 256);
  a.yt_blocks = a.ldo / 32;
  const int v_blocks = (n + 255) / 256 * 8;
  take(a.vplanes, (size_t)v_blocks * (L / 16) * 2048);
  take(a.yt, (size_t)a.yt_blocks * (L / 16) * 2048);
  auto product = [&](DenseGemmArgs& g, const u32x4* rows, int row_blocks, const u32x4* cols, int col_blocks, int steps, int ld,
                     const float2* scale_a, const float2* scale_b, const float* out, bool split) {
    g.a = rows;
    g.b = cols;
    g.a_blocks = row_blocks;
    g.b_blocks = col_blocks;
    g.steps = steps;
    g.rows = n;
    g.ld = ld;
    g.scale[0] = scale_a;
    g.scale[1] = scale_b;
    g.step_words = kDenseStep;
    g.plane_words = 64;
    g.out = const_cast<float*>(out);
    dense_gemm_plan(g, split);
  };
  product(q.dots, q.td.planes[0], q.td.blocks[0], q.td.planes[1], q.td.blocks[1], q.td.steps, a.ld, q.pts.scale,
          q.pts.scale + 1, a.dots, false);
  product(q.prod, q.ta.planes[0], q.ta.blocks[0], q.td.planes[1], q.td.blocks[1], q.td.steps, a.ld, q.dir.scale,
          q.pts.scale + 1, a.prod, false);
  product(q.last, a.vplanes, v_blocks, a.yt, a.yt_blocks, (int)(L / 16), a.ldo, nullptr, nullptr, nullptr, true);
  a.splits = q.last.splits;
  take(a.prod_out, (size_t)a.splits * N * a.ldo * 4);
  q.last.out = const_cast<float*>(a.prod_out);
  return at;
}

// The planes of x and y, where no solve has left them, and of the direction (one matrix, the second operand of its
// product is y's), what of the operands is taken row by row, and the products.
int prepare(HvpPlan& q, bool kept, hipStream_t st) {
  const HvpArgs& a = q.a;
  const int mats = kept ? 0 : 2, blocks = kept ? q.ta.blocks[0] : std::max(q.td.blocks[0], q.td.blocks[1]);
  hipLaunchKernelGGL((hvp_stats_kernel<0>), dim3(kSmallStatBlocks, mats + 1), dim3(1024), 0, st, q.pts, q.dir, mats);
  hipLaunchKernelGGL((hvp_prep_kernel<0>), dim3(blocks + 1, mats + 1), dim3(512), 0, st, q.pts, q.td, q.dir, q.ta, mats);
  const TransposedArgs yt = {a.y, a.scale, a.yt, a.m, a.d, a.ld, a.dtype};
  hipLaunchKernelGGL((hvp_rows_kernel<0>), dim3((a.n + a.ld + 3) / 4 + (a.ld / 16 + 3) / 4 * a.yt_blocks), dim3(256), 0, st, a, yt);
  if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  if (kept) return dense_gemm(q.prod, 1, st);
  DenseGemmJobs jobs;
  std::memset(&jobs, 0, sizeof(jobs));
  jobs.job[0] = q.dots;
  jobs.job[1] = q.prod;
  return dense_gemm_jobs(jobs, 2, 1, st, false);
}

template <int MODE>
int strips(const HvpArgs& a, hipStream_t st) {
  const int wgs = a.strips + (MODE == 2 ? 1 : 0);
  if (a.ld <= 2048) hipLaunchKernelGGL((hvp_strip_kernel<1, 8, MODE>), dim3(wgs), dim3(512), 0, st, a);
  else if (a.ld <= 4096) hipLaunchKernelGGL((hvp_strip_kernel<2, 8, MODE>), dim3(wgs), dim3(512), 0, st, a);
  else hipLaunchKernelGGL((hvp_strip_kernel<4, 4, MODE>), dim3(wgs), dim3(512), 0, st, a);
  if constexpr (MODE < 2) hipLaunchKernelGGL((hvp_columns_kernel<MODE>), dim3((a.m + 63) / 64), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

// The planes, sums and products behind a gradient on kept products.
struct GradPlan {
  DenseGradArgs g;
  TransposedArgs yt;
  DenseGemmArgs product;
};

size_t grad_layout(const SmallArgs& s, const DenseArgs& t, void* ws, GradPlan& q) {
  std::memset(&q, 0, sizeof(q));
  size_t at = 0;
  auto take = [&](auto& ptr, size_t bytes) {
    ptr = reinterpret_cast<std::remove_cv_t<std::remove_reference_t<decltype(ptr)>>>(static_cast<char*>(ws) + at);
    at += (bytes + 255) & ~(size_t)255;
  };
  DenseGradArgs& g = q.g;
  g.ldo = (s.d + 255) / 256 * 256;
  const size_t steps = t.ld / 16;
  take(g.planes, (size_t)t.blocks[0] * steps * 2048);
  take(q.yt.yt, (size_t)(g.ldo / 32) * steps * 2048);
  take(g.sums, (size_t)(t.ld / 256) * t.n * 4);
  q.yt.y = s.pts[1];
  q.yt.scale = s.scale;
  q.yt.m = t.m;
  q.yt.d = s.d;
  q.yt.ld = t.ld;
  q.yt.dtype = s.dtype;
  DenseGemmArgs& m = q.product;
  m.a = g.planes;
  m.b = q.yt.yt;
  m.a_blocks = t.blocks[0];
  m.b_blocks = g.ldo / 32;
  m.steps = (int)steps;
  m.rows = t.n;
  m.ld = g.ldo;
  m.step_words = kDenseStep;
  m.plane_words = 64;
  dense_gemm_plan(m, true);
  g.splits = m.splits;
  take(m.out, (size_t)m.splits * t.n * g.ldo * 4);
  g.prod = m.out;
  return at;
}

int run_hvp(const fs_hvp_problem* p, const Kept* kept, void* workspace, size_t workspace_bytes, float* out,
            float* host_state, hipStream_t st);

}  // namespace
}  // namespace fs

using namespace fs;

extern "C" {

size_t fs_hvp_workspace_bytes(const fs_hvp_problem* p) {
  if (checked(p) != FS_OK) return 0;
  HvpPlan q;
  return layout(p, nullptr, q, false);
}

size_t fs_hvp_solved_workspace_bytes(const fs_hvp_problem* p) {
  if (checked(p) != FS_OK) return 0;
  HvpPlan q;
  return layout(p, nullptr, q, true);
}

int fs_hvp(const fs_hvp_problem* p, void* workspace, size_t workspace_bytes, float* out, float* host_state, void* stream) {
  return run_hvp(p, nullptr, workspace, workspace_bytes, out, host_state, (hipStream_t)stream);
}

int fs_hvp_solved(const fs_hvp_problem* p, const fs_small_problem* solved, void* solved_workspace, size_t solved_bytes,
                  void* workspace, size_t workspace_bytes, float* out, float* host_state, void* stream) {
  if (!p || !solved || !solved_workspace) return FS_ERR_NULL_POINTER;
  Kept kept;
  const int rc = dense_solved(solved, solved_workspace, solved_bytes, kept.a, kept.t);
  if (rc != FS_OK) return rc;
  if (solved->n != p->n || solved->m != p->m || solved->d != p->d || solved->cost_scale != p->cost_scale) return FS_ERR_BAD_SIZE;
  return run_hvp(p, &kept, workspace, workspace_bytes, out, host_state, (hipStream_t)stream);
}

size_t fs_dense_grad_workspace_bytes(const fs_small_problem* p) {
  SmallArgs a;
  DenseArgs t;
  GradPlan q;
  return dense_solved(p, nullptr, ~(size_t)0, a, t) == FS_OK ? grad_layout(a, t, nullptr, q) : 0;
}

int fs_dense_grad(const fs_small_problem* p, void* solved_workspace, size_t solved_bytes, const float* grad_out,
                  float* grad_x, void* workspace, size_t workspace_bytes, void* stream) {
  if (!p || !solved_workspace || !workspace || !grad_out || !grad_x) return FS_ERR_NULL_POINTER;
  SmallArgs a;
  DenseArgs t;
  GradPlan q;
  int rc = dense_solved(p, solved_workspace, solved_bytes, a, t);
  if (rc != FS_OK) return rc;
  if (grad_layout(a, t, workspace, q) > workspace_bytes) return FS_ERR_WORKSPACE_TOO_SMALL;
  hipStream_t st = (hipStream_t)stream;
  q.g.grad_out = grad_out;
  q.g.out = grad_x;
  hipLaunchKernelGGL((dense_plan_kernel<0>), dim3((t.n + 255) / 256 * 8, t.ld / 256), dim3(256), 0, st, a, t, q.g);
  hipLaunchKernelGGL((hvp_yt_kernel<0>), dim3((t.ld / 16 + 3) / 4, q.g.ldo / 32), dim3(256), 0, st, q.yt);
  if ((rc = dense_gemm(q.product, 1, st)) != FS_OK) return rc;
  hipLaunchKernelGGL((dense_grad_kernel<0>), dim3(t.n), dim3(256), 0, st, a, t, q.g);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

}  // extern "C"

namespace fs {
namespace {

// On a few thousand points no launch but the mass' and V's takes longer than a launch does (3 to 6 us), so there are as few as the
// data's way allows: the operands of both products prepared together, the two products in one launch, y^T with the rows,
// the limits with the last strips, the weights and the outer factor in kernels that read the potentials and
// write the result (26 launches and some 15 small ones around them -> 21 and none: loss, gradient and product of 2,048 x
// 2,048 x 64 717 -> 640 us, 1,500 x 1,400 x 20 668 -> 493, 7,000 x 5,000 x 60 1,458 -> 1,400, 6,000 x 7,500 x 900 3,061 -> 3,014).
int run_hvp(const fs_hvp_problem* p, const Kept* kept, void* workspace, size_t workspace_bytes, float* out,
            float* host_state, hipStream_t st) {
  int rc = checked(p);
  if (rc != FS_OK) return rc;
  if (!out || !host_state) return FS_ERR_NULL_POINTER;
  HvpPlan q;
  if (!workspace || layout(p, workspace, q, kept != nullptr, kept) > workspace_bytes) return FS_ERR_WORKSPACE_TOO_SMALL;
  HvpArgs& a = q.a;
  a.out = out;
  if ((rc = prepare(q, kept != nullptr, st)) != FS_OK) return rc;
  if (q.td.large) hipLaunchKernelGGL((hvp_mass_kernel<8>), dim3(a.groups, a.chunks), dim3(512), 0, st, a);
  else hipLaunchKernelGGL((hvp_mass_kernel<4>), dim3(a.groups, a.chunks), dim3(256), 0, st, a);
  hipLaunchKernelGGL((hvp_merge_kernel<0>), dim3((std::max(a.n, a.m) + 63) / 64, 2), dim3(256), 0, st, a);
  if ((rc = strips<0>(a, st)) != FS_OK) return rc;
  // ---- conjugate gradients: the host looks one iteration behind the one it enqueues, and what it
  // enqueued behind the last one does nothing ----
  int* count = reinterpret_cast<int*>(host_state) + 7;
  bool done = false;  // (from the word that arrives last: the report is then whole)
  auto seen = [&](int k) {
    const int c = __atomic_load_n(count, __ATOMIC_ACQUIRE);
    done = c >= 0 && (c & 1);
    return done || c >= 2 * k;
  };
  __atomic_store_n(count, -1, __ATOMIC_RELEASE);
  if ((rc = cg_init(a.a_dir, a.sol, a.res, a.vec, a.cg, a.m, p->rtol, p->atol, host_state, st)) != FS_OK) return rc;
  for (int k = 0; k < p->max_iter && !done; ++k) {
    if ((rc = strips<1>(a, st)) != FS_OK) return rc;
    if ((rc = cg_update(a.a_dir, a.sol, a.res, a.vec, a.cg, a.m, host_state, k, st)) != FS_OK) return rc;
    if ((rc = wait_for_words(st, [&]() { return seen(k); })) != FS_OK) return rc;
  }
  a.vec = a.sol;
  if ((rc = strips<2>(a, st)) != FS_OK) return rc;
  hipLaunchKernelGGL((hvp_v_kernel<0>), dim3((a.n + 255) / 256 * 8, a.ld / 256), dim3(256), 0, st, a);
  if ((rc = dense_gemm(q.last, 1, st)) != FS_OK) return rc;
  const int blocks = (int)std::min<size_t>(4096, ((size_t)a.n * ((a.d + 3) / 4) + 255) / 256);
  hipLaunchKernelGGL((hvp_result_kernel<0>), dim3(blocks), dim3(256), 0, st, a);
  if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  // (the last iteration's state, for the caller's report)
  return done ? FS_OK : wait_for_words(st, [&]() { return seen(p->max_iter); });
}

}  // namespace
}  // namespace fs
