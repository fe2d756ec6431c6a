// Small problems: planning, workspace and launches of the kernels in fs_small.hpp.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <type_traits>

#include "flash_sinkhorn_hip.h"
#include "fs_dense.hpp"
#include "fs_host.hpp"
#include "fs_pair.hpp"
#include "fs_small.hpp"

namespace fs {
namespace {

struct EpsTable {
  float e[kSmallTable];
};

// Schedule given by the caller: every item and problem takes the same entries.
template <int T>
__global__ __launch_bounds__(256) void small_table_kernel(const SmallArgs a, const EpsTable t) {
  float4* out = a.table + (size_t)blockIdx.x * a.table_len;
  for (int i = threadIdx.x; i <= a.entries; i += 256) out[i] = small_coef(a.cost_scale, t.e[min(i, a.entries - 1)]);
  if (threadIdx.x == 0) a.lens[blockIdx.x] = a.full[blockIdx.x] = a.entries;
}

// Which kernels a problem takes.  d <= 64: both sides of a step from one sweep (fs_pair.hpp) where
// that saves more than its second launch per step costs.  Fixed eps: from 2e7 logits per step on
// (one problem of 4,500 points, d = 64, 40 steps: 1.08 against 1.47 ms, d = 3 0.74 against 0.82; 3,600 points, d = 64:
// 0.88 against 0.78 ms).  A schedule rewrites the planes behind every step and has few steps: 5e7 (d = 3, 6,500 points:
// 0.40 against 0.40 ms; 9,000: 0.56 against 0.71), 2e7 where the planes are wide (d = 64, 4,500: 0.54 against
// 0.58 ms; 3,600: 0.44 against 0.33).  Items of a batch fill the chip without it: 12 x 2,048 x 8, debiased, 0.96
// against 0.74 ms.  Early stopping on a schedule is only built for the small kernels.
bool use_pair(const fs_small_problem* p) {
  if (p->alternating || p->d > 64 || (p->threshold > 0.f && p->sched != 0)) return false;
  const double n = (double)p->n, m = (double)p->m;
  const double logits = (p->self_terms < 2 ? n * m : 0.) + (p->self_terms ? 0.5 * (n * n + m * m) : 0.);
  return logits >= (p->sched == 0 || p->d > 32 ? 2.0e7 : 5.0e7);
}

// Wide rows: the products are formed once and kept (fs_dense.hpp).
bool use_dense(const fs_small_problem* p) { return p->d > kSmallMaxD; }

// Narrower rows whose products are formed once and kept for the steps of a solve (dense_rows_kernel).  A workgroup
// of small_step_kernel reads the planes of all keys for 32 rows, 2, 4, 6, 8, 12 or 16 bytes a logit by the padded width, from the
// caches; a kept product is 4.  `read`: the bytes of a step, which come from the last-level cache, against the narrower
// planes.  Potentials after 50 steps at a fixed eps, and after a schedule of 14, planes -> products, us:
//   d = 64:  256 points 243 -> 196, 91 -> 94; 1,000: 370 -> 238, 131 -> 102; 2,048 (32 MiB): 553 -> 395, 187 -> 152;
//            2,500 (49 MiB): 657 -> 712, 177 -> 201; with self problems 1,000 (16 MiB): 388 -> 306, 110 -> 101;
//            1,500 (35 MiB): 477 -> 507, 137 -> 159
//   d = 48 (planes of 48 columns): 1,000: 334 -> 244, 110 -> 94; 2,048: 504 -> 401, 153 -> 138
//   d = 96 (planes of 96): 256: 282 -> 207, 103 -> 97; 1,000: 448 -> 248, 149 -> 104; 2,000: 725 -> 411, 226 -> 155; 3,000: 1,000 ->
//            860, 310 -> 295; 4,000: 1,370 -> 1,345, 411 -> 411; with self problems 1,000: 461 -> 308, 154 -> 120; 2,000: 840 -> 750,
//            248 -> 260; 2,500: 1,557 -> 1,092, 478 -> 370
//   d = 128: 256: 320 -> 201, 110 -> 96; 1,000: 563 -> 246, 175 -> 104; 3,000 (70 MiB): 1,143 -> 849, 344 -> 290; 4,000
//            (125 MiB): 1,639 -> 1,447, 413 -> 391 (d = 100: 401 -> 417); with self problems 2,500 (98 MiB): 1,957 -> 1,083
//   d = 32, fixed eps: 512: 233 -> 200; 1,000 (8 MiB): 295 -> 236; 1,500 (18 MiB): 359 -> 345; its schedules 85 -> 86 and
//            102 -> 101; d <= 16: 270 -> 230 at 1,000, 0.93 to 1.0 at 256 and 1,500
bool use_products(const fs_small_problem* p) {
  if (p->alternating || p->d <= 16 || use_dense(p) || use_pair(p)) return false;
  const double n = (double)p->n, m = (double)p->m;
  const double ldx = std::ceil(n / 256) * 256, ldy = std::ceil(m / 256) * 256;
  if (std::max(ldx, ldy) > kDenseRowKeys) return false;
  if (p->sched != 1 && p->entries < 8) return false;  // (forming them takes what some six steps gain)
  // (a schedule by diameter is not replayed, and below this the host, with one launch and one tensor more, is what its
  // caller waits for: 64 x 64 points at 40, 64 and 100 columns 88 -> 94, 89 -> 93, 91 -> 95 us; debiased 256 x 64 96 -> 92,
  // 128 x 128 101 -> 95)
  if (p->sched == 1 && (double)p->items * std::max(n, m) * (p->d <= 64 ? 64 : 128) < 16384.0) return false;
  const double read = 4.0 * (double)p->items *
                      ((p->self_terms < 2 ? n * ldy + m * ldx : 0.) + (p->self_terms ? n * ldx + m * ldy : 0.));
  if (p->d <= 32) return p->sched == 0 && read <= 9.0e6;
  return read <= (p->d <= 64 ? 3.4e7 : 1.1e8);
}

// The products of every side [items][rows][ld] and bytes they take.
struct Products {
  float* dots[4];
  int ld[4];
  size_t bytes;
};
Products products_at(const SmallArgs& a, void* at) {
  Products t;
  char* p = static_cast<char*>(at);
  for (int side = 0; side < 4; ++side) {
    const int mat = side & 1, keys = side < 2 ? mat ^ 1 : mat;
    t.dots[side] = nullptr;
    t.ld[side] = (a.rows[keys] + 255) / 256 * 256;
    if (side < 2 ? a.self == 2 : a.self == 0) continue;
    t.dots[side] = reinterpret_cast<float*>(p);
    p += (size_t)a.items * a.rows[mat] * t.ld[side] * 4;  // (a multiple of 1 KiB)
  }
  t.bytes = (size_t)(p - static_cast<char*>(at));
  return t;
}

// Forms them, from the planes of small_prep_kernel.  Both sides of a problem get a product of their own: a
// transposed copy would add a logit's cross products in the other order (those of its key first), and a cloud solved
// against itself would have f and g that differ by a rounding.
int form_products(const SmallArgs& a, const Products& t, int steps, hipStream_t st) {
  DenseGemmJobs jobs;
  std::memset(&jobs, 0, sizeof(jobs));
  int n = 0;
  for (int side = 0; side < 4; ++side) {
    if (t.dots[side] == nullptr) continue;
    const int r = side & 1, c = side < 2 ? r ^ 1 : r;
    DenseGemmArgs& g = jobs.job[n++];
    g.a = a.planes[r];
    g.b = a.planes[c];
    g.a_blocks = a.blocks[r];
    g.b_blocks = a.blocks[c];
    g.steps = steps;
    g.step_words = 64;
    g.plane_words = steps * 64;
    g.rows = a.rows[r];
    g.cols = a.rows[c];
    g.scale[0] = a.scale + r;
    g.scale[1] = a.scale + c;
    g.out = t.dots[side];
    g.ld = t.ld[side];
    dense_gemm_plan(g, false);
  }
  return dense_gemm_jobs(jobs, n, a.items, st);
}

// Workgroups over which the loss of an item is spread: one for what a workgroup does in three rounds.
int loss_parts(const SmallArgs& a) {
  const int rows = std::max(a.rows[0], a.rows[1]);
  return rows <= 3072 ? 1 : std::min(64, (rows + 1023) / 1024);
}

// Columns that planes hold: as few 16-column steps as the rows fill, in steps of 32 from 64 on (80 and 112 columns were not
// built).  A step streams and multiplies all of them, so the last quarter counts: with 64 and 128 columns -> 48 and 96,
// loss and gradient, us: schedules 3,001 x 4,567 x 33 315 -> 283, 5,000 x 5,100 x 40 492 -> 385 and x 80 1,210 -> 953, 30,000 x
// 29,000 x 40 5,730 -> 4,020; 3,112 x 2,124 x 37, debiased, 73 steps 1,592 -> 1,399; 10,000 x 44, 60 steps, mostly along lists
// 2,327 -> 2,170.  Products of narrow rows are formed two steps at a time, so a solve on these takes 64 for 48.
int padded(const fs_small_problem* p) {
  if (p->d <= 32) return p->d <= 16 ? 16 : 32;
  if (p->d <= 64) return p->d <= 48 && !use_products(p) ? 48 : 64;
  return p->d <= 96 ? 96 : 128;
}

// `solved`: the problem has been, and its list of eps is not looked at again (the workspace has the table).
int checked(const fs_small_problem* p, bool solved = false) {
  if (!p || !p->x || !p->y) return FS_ERR_NULL_POINTER;
  if (p->n <= 0 || p->m <= 0 || p->d <= 0 || p->items <= 0 || p->items > 65535) return FS_ERR_BAD_SIZE;
  if (p->n > FS_SMALL_MAX_ROWS || p->m > FS_SMALL_MAX_ROWS || p->d > FS_SMALL_MAX_D) return FS_ERR_UNSUPPORTED;
  if (p->d > kSmallMaxD && p->items * p->n * p->m > FS_SMALL_MAX_PRODUCTS) return FS_ERR_UNSUPPORTED;
  if (p->d > kSmallMaxD && (p->self_terms || p->want_values || p->sched == 1)) return FS_ERR_UNSUPPORTED;
  if (p->dtype < 0 || p->dtype > 2 || p->sched < 0 || p->sched > 2) return FS_ERR_BAD_ARGUMENT;
  if (p->sched != 1 && p->entries <= 0) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 0 && !(p->eps > 0.f)) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 1 && !(p->blur > 0.0 && p->scaling > 0.0 && p->scaling < 1.0)) return FS_ERR_BAD_ARGUMENT;
  if (p->sched == 2 && p->entries >= kSmallTable) return FS_ERR_UNSUPPORTED;
  if (p->sched == 2 && !solved) {
    if (!p->eps_list) return FS_ERR_NULL_POINTER;
    for (int i = 0; i < p->entries; ++i)
      if (!(p->eps_list[i] > 0.f)) return FS_ERR_BAD_ARGUMENT;
  }
  if (p->threshold > 0.f && p->check_every <= 0) return FS_ERR_BAD_ARGUMENT;
  if (p->alternating && (p->sched != 0 || p->self_terms || p->want_values || p->d > kSmallMaxD)) return FS_ERR_UNSUPPORTED;
  return p->self_terms < 0 || p->self_terms > 2 ? FS_ERR_BAD_ARGUMENT : FS_OK;
}

// Entries that a schedule of this problem can have (at a fixed eps one stands for all).  By diameter: of
// clouds whose squared diameter fp32 holds (small_schedule refuses others), one more for what the
// logarithms round.
int table_entries(const fs_small_problem* p) {
  if (p->sched == 0) return 1;
  if (p->sched == 2) return p->entries;
  const double most = 3.0 + std::ceil(std::max(0.0, (std::log(1.845e19) - std::log(p->blur)) / -std::log(p->scaling)));
  int k = (int)std::min<double>(most, kSmallTable - 1);
  if (p->cut > 0) k = std::min(k, p->cut);
  return k;
}

// Clouds of few columns are not peaked at the eps they are solved at: there is nothing to skip, and the kernel
// without that is 3 to 6 % faster (9,000 x 3 at eps 0.01).
bool skips(int d) { return d > 8; }

// Work items of a medium problem's launch: 256-row groups of the stationary rows times chunks of the
// streamed ones, one chunk length for all problems.  Two workgroups per CU run at a time, so
// the length is the one whose last round of 512 is fullest, counting two tiles' worth of time for
// what an item costs around its tiles.
void plan_pair(const SmallArgs& a, PairArgs& t) {
  t.items = a.items;
  t.first_prob = a.self == 2 ? 1 : 0;
  t.nprob = a.self ? 3 : 1;
  t.sched = a.sched;
  t.extrapolate = a.extrapolate;
  for (int q = t.first_prob; q < t.nprob; ++q) {
    PairProblem& pr = t.prob[q];
    const int s = q == 2 ? 1 : 0, k = q == 0 ? 1 : s;
    pr.self = q > 0;
    pr.n_st = a.rows[s];
    pr.n_str = a.rows[k];
    pr.st_blocks = a.pblocks[s];
    pr.str_blocks = a.pblocks[k];
    pr.groups = (pr.n_st + 255) / 256;
    // (a row's few units are a smaller share the more there are: at 4,500 x 64 such a step takes as long as
    // one that computes everything and its merge 5 us longer, at 10,000 x 64 62 against 92 us)
    pr.ends = skips(a.d) && (double)pr.n_st * pr.n_str >= 6.0e7;
    pr.strict = !(a.rho[s] > 0.f) && !(a.rho[k] > 0.f);
    pr.units = 0.f;
    for (int g = 0; g < pr.groups && skips(a.d); ++g) pr.units += 16.f * (float)((pr.n_str - (pr.self ? 256 * g : 0) + 63) / 64);
  }
  auto items_at = [&](int tiles, PairArgs& u) {
    int n = 0;
    for (int q = t.first_prob; q < t.nprob; ++q) {
      PairProblem& pr = u.prob[q];
      pr.chunk = tiles * 64;
      pr.chunks = (pr.n_str + pr.chunk - 1) / pr.chunk;
      pr.n_items = 0;
      for (int c = 0; c < pr.chunks; ++c)
        pr.n_items += pr.self ? self_groups_of_chunk(c, pr.chunk, pr.n_str, pr.groups) : pr.groups;
      pr.two_first = pr.groups * pr.chunks;
      pr.two_items = pr.two_first;
      if (!pr.self)
        pr.two_items += (pr.n_str + 255) / 256 * ((pr.n_st + pr.chunk - 1) / pr.chunk);
      n += pr.n_items;
    }
    return n;
  };
  int best = 4;
  double cost = 0.0;
  for (int tiles = 4; tiles <= kPairMostTiles; ++tiles) {
    const double n = (double)items_at(tiles, t) * a.items;
    const double c = std::ceil(n / 512.0) * (tiles + 2);
    if (cost == 0.0 || c < cost - 1e-9) cost = c, best = tiles;
  }
  items_at(best, t);
  t.per_xcd = 0;
  for (int q = t.first_prob; q < t.nprob; ++q) t.per_xcd += (t.prob[q].n_items + 7) / 8;
  t.merge_groups = (std::max(a.pblocks[0], a.pblocks[1]) + 7) / 8;
  for (int i = 0; i < 4; ++i) {
    PairSide& sd = t.side[i];
    const int mat = i & 1;
    sd.rows = a.rows[mat];
    sd.blocks = a.pblocks[mat];
  }
}

// Pointers of a medium problem's kernels once the workspace is laid out.
void bind_pair(const SmallArgs& a, PairArgs& t) {
  t.table = a.table;
  t.table_len = a.table_len;
  t.lens = a.lens;
  t.limits = a.limits;
  t.reach = a.reach;
  for (int q = t.first_prob; q < t.nprob; ++q) {
    PairProblem& pr = t.prob[q];
    const int s = q == 2 ? 1 : 0, k = q == 0 ? 1 : s;
    const int ss = q == 0 ? 0 : 1 + q, ks = q == 0 ? 1 : ss;  // sides of the stationary and the streamed rows
    auto planes = [&](int m) { return q > 0 && a.self_planes[m] ? a.self_planes[m] : a.planes[m]; };
    pr.st_planes = planes(s);
    pr.str_planes = planes(k);
    pr.st_bias = t.side[ss].bias;
    pr.str_bias = t.side[ks].bias;
    pr.st_bias32 = t.side[ss].bias32;
    pr.str_bias32 = t.side[ks].bias32;
    for (int i : {ss, ks}) {
      PairSide& sd = t.side[i];
      const int mat = i & 1;
      sd.part = i == ss ? pr.st_part : pr.str_part;
      sd.parts = i == ss ? pr.chunks : pr.groups;
      sd.col = pr.str_part;
      sd.ms = i == ss ? pr.st_ms : pr.str_ms;
      sd.best = i == ss ? pr.st_best : pr.str_best;
      sd.other = a.pts[q == 0 ? mat ^ 1 : mat];
      sd.others = a.rows[q == 0 ? mat ^ 1 : mat];
      sd.ms_parts = i == ss ? pr.chunks : (pr.n_st + pr.chunk - 1) / pr.chunk;
      sd.self = pr.self;
      sd.chunk = pr.chunk;
      sd.pot = a.pot[i];
      sd.norm = a.norm[mat];
      sd.l2w = a.l2w[mat];
      sd.pts = a.pts[mat];
      sd.dtype = a.dtype;
      sd.d = a.d;
      sd.rho = a.rho[mat];
      // (where all problems share their eps, the first of them writes the planes they share)
      sd.planes = a.self_planes[mat] ? (i < 2 ? a.planes[mat] : a.self_planes[mat])
                                     : (i < 2 || a.self == 2 ? a.planes[mat] : nullptr);
    }
  }
}

// The kernels' arguments with the workspace laid out from `ws` (null: sizes only); returns the
// bytes the workspace takes.
size_t layout(const fs_small_problem* p, void* ws, SmallArgs& a, PairArgs* pa = nullptr, DenseArgs* da = nullptr,
              PairArgs** pair_at = nullptr) {
  std::memset(&a, 0, sizeof(a));
  a.pair = use_pair(p) ? 1 : 0;
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
  a.alternating = p->alternating ? 1 : 0;
  a.extrapolate = p->extrapolate || p->alternating ? 1 : 0;  // (the parity of the last potentials)
  a.eps0 = p->eps;
  a.blur = p->blur;
  a.scaling = p->scaling;
  a.rho[0] = p->rho_x;
  a.rho[1] = p->rho_y;
  const int dp = use_dense(p) ? 0 : padded(p), ndb = (dp + 31) / 32;
  size_t at = 0;
  char* base = static_cast<char*>(ws);
  auto take = [&](auto& ptr, size_t bytes) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(base + at);
    at += (bytes + 255) & ~(size_t)255;
  };
  const size_t items = (size_t)p->items;
  take(a.lens, items * 3 * 4);
  take(a.full, items * 3 * 4);
  take(a.scale, items * 2 * sizeof(float2));
  // (what the device leaves per item follows the clouds: 4,096 clouds of 32 points take 70 MB with
  // it, 700 MB with the largest of both)
  a.stat_blocks = use_dense(p) ? kSmallStatBlocks : (int)std::min<int64_t>(kSmallStatBlocks, (std::max(p->n, p->m) + 31) / 32);
  a.stat_words = use_dense(p) ? 2 : 4 + 2 * a.d;
  a.table_len = table_entries(p) + 1;
  take(a.stats, items * 2 * (size_t)a.stat_blocks * (size_t)a.stat_words * 4);
  take(a.table, items * 3 * (size_t)a.table_len * sizeof(float4));
  for (int i = 0; i < 2; ++i) {
    const size_t rows = (size_t)a.rows[i];
    a.blocks[i] = (int)((rows + 31) / 32);
    // (whole 256-row groups, and the tiles that are fetched past the end)
    a.pblocks[i] = a.pair ? (int)((rows + 255) / 256) * 8 + 8 : a.blocks[i];
    const size_t blocks = items * (size_t)a.blocks[i], pblocks = items * (size_t)a.pblocks[i];
    if (!use_dense(p)) take(a.planes[i], pblocks * (size_t)(2 * dp / 16) * 1024);
    if (a.pair && a.self && a.sched != 0) take(a.self_planes[i], pblocks * (size_t)(2 * dp / 16) * 1024);
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
  if (use_dense(p)) {
    DenseArgs scratch;
    DenseArgs& t = da ? *da : scratch;
    std::memset(&t, 0, sizeof(t));
    dense_plan(a, t);
    // Where the rows of products start within a 4 KiB page shows in the sweep, which is bound by reading
    // them: 1 KiB behind its start 3.56 ms (8,192 x 8,192 x 256, 60 steps) and 14.60 (16,384), 2 KiB 3.65
    // and 14.53, at it 3.61 and 14.57, 2.75 KiB 3.58 and 15.7; other sizes lie within 1 %.
    at = ((at + 4095) & ~(size_t)4095) + 1024;
    take(t.dots, items * (size_t)t.n * (size_t)t.ld * 4);
    if (t.rows) take(t.dots_t, items * (size_t)t.m * (size_t)t.ld_t * 4);
    for (int i = 0; i < 2; ++i) take(t.planes[i], items * (size_t)t.blocks[i] * (size_t)t.steps * 2048);
    take(t.part[0], items * (size_t)t.chunks * (size_t)t.n * sizeof(float2));
    take(t.part[1], items * (size_t)t.groups * (size_t)t.m * sizeof(float2));
    take(t.top, items * (size_t)t.n * 4);
    t.table = a.table;
    t.table_len = a.table_len;
    t.lens = a.lens;
    t.sched = a.sched;
    t.extrapolate = a.extrapolate;
    for (int i = 0; i < 2; ++i) {
      t.l2w[i] = a.l2w[i];
      t.norm[i] = a.norm[i];
      t.rho[i] = a.rho[i];
    }
  }
  if (a.pair) {
    take(a.limits, items * sizeof(float4));
    take(a.reach, items * sizeof(float4));
    PairArgs scratch;
    PairArgs& t = pa ? *pa : scratch;
    std::memset(&t, 0, sizeof(t));
    plan_pair(a, t);
    take(t.state, items * 3 * kPairStateWords * 4);
    take(t.work, 8 * (size_t)t.per_xcd * sizeof(int4));
    for (int q = t.first_prob; q < t.nprob; ++q) {
      PairProblem& pr = t.prob[q];
      take(pr.st_part, items * (size_t)pr.chunks * (size_t)pr.n_st * 4);
      take(pr.str_part, items * (size_t)pr.groups * (size_t)pr.n_str * 4);
      take(pr.list, items * (size_t)pr.n_items * (4 * kPairListWords * 8));
      take(pr.two_list, items * (size_t)pr.two_items * (4 * kPairListWords * 8));
      take(pr.st_ms, items * (size_t)pr.chunks * (size_t)pr.n_st * sizeof(float2));
      take(pr.st_best, items * (size_t)pr.chunks * (size_t)pr.n_st * 4);
      if (!pr.self) {
        const size_t parts = items * (size_t)((pr.n_st + pr.chunk - 1) / pr.chunk) * (size_t)pr.n_str;
        take(pr.str_ms, parts * sizeof(float2));
        take(pr.str_best, parts * 4);
      }
    }
    for (int i = a.self == 2 ? 2 : 0; i < (a.self ? 4 : 2); ++i) {
      PairSide& sd = t.side[i];
      take(sd.bias, items * (size_t)sd.blocks * 32 * sizeof(u32x4));
      take(sd.bias32, items * (size_t)sd.blocks * 32 * 4);
      take(sd.sum2, items * (size_t)sd.rows * 4);
      take(sd.key, items * (size_t)sd.rows * 4);
      take(sd.dot, items * (size_t)sd.rows * 4);
    }
    PairArgs* args;
    take(args, sizeof(PairArgs));
    if (pair_at) *pair_at = args;
    if (pa) bind_pair(a, t);
  }
  return at;
}

// Values of a matrix from which on 1,024 threads a workgroup take its statistics, in place of 256: 64 workgroups wait for their
// loads.  10,000 x 64 16.6 -> 9.4 us, 30,011 x 64 43.5 -> 18.4, 50,000 x 64 71 -> 27; 256,000 values 6.9 -> 7.2, 99,000 5.4 -> 6.6.
constexpr int64_t kWideStats = 3 << 17;

template <int DP>
int launch_prep(const SmallArgs& a, const PairArgs& pa, PairArgs* pair_at, hipStream_t st) {
  const int xb = a.blocks[0] > a.blocks[1] ? a.blocks[0] : a.blocks[1];
  if ((int64_t)std::max(a.rows[0], a.rows[1]) * a.d >= kWideStats)
    hipLaunchKernelGGL((small_stats_kernel<1024>), dim3(a.stat_blocks, 2, a.items), dim3(1024), 0, st, a);
  else
    hipLaunchKernelGGL((small_stats_kernel<256>), dim3(a.stat_blocks, 2, a.items), dim3(256), 0, st, a);
  const dim3 grid(xb + 1, 2, a.items);
  if constexpr (DP <= 64)
    if (a.pair) hipLaunchKernelGGL((small_prep_kernel<DP, PairArgs>), grid, dim3(256), 0, st, a, pa, pair_at);
  if (!a.pair)
    hipLaunchKernelGGL((small_prep_kernel<DP, SmallNothing>), grid, dim3(256), 0, st, a, SmallNothing(),
                       static_cast<SmallNothing*>(nullptr));
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

SmallStepArgs step_args(const SmallArgs& a, int step) {
  SmallStepArgs t;
  std::memset(&t, 0, sizeof(t));
  t.scale = reinterpret_cast<const float4*>(a.scale);
  t.step = step;
  t.extrapolate = a.extrapolate;
  t.coef_stride = 3 * a.table_len;
  const int first = a.self == 2 ? 2 : 0, sides = a.self == 1 ? 4 : 2;
  for (int i = 0; i < sides; ++i) {
    const int side = first + i, qm = side & 1, km = side < 2 ? qm ^ 1 : qm, prob = side < 2 ? 0 : side - 1;
    SmallStepSide& s = t.side[i];
    const size_t nq = (size_t)a.items * a.rows[qm], nk = (size_t)a.items * a.rows[km];
    s.kplanes = a.planes[km];
    s.qplanes = a.planes[qm];
    s.kpot = a.pot[side < 2 ? side ^ 1 : side] + (step & 1) * nk;
    s.kl2w = a.l2w[km];
    // (the entry past the last repeats it, for the extrapolation)
    s.coef = a.table + prob * a.table_len + (a.sched == 0 ? 0 : std::min(std::max(step - 1, 0), a.table_len - 1));
    s.lens = a.lens + prob;
    s.old = a.pot[side] + (step & 1) * nq;
    s.out = a.pot[side] + ((step & 1) ^ 1) * nq;
    s.norm = a.norm[qm];
    s.nq = a.rows[qm];
    s.nk = a.rows[km];
    s.nqb = a.blocks[qm];
    s.nkb = a.blocks[km];
    s.rho = a.rho[qm];
    s.qm = qm;
    s.km = km;
  }
  return t;
}

int launch_rows(const SmallArgs& a, int step, const float* const* dots, const int* ld, float* top, int rows, hipStream_t st) {
  DenseRowArgs t;
  t.s = step_args(a, step);
  const int first = a.self == 2 ? 2 : 0, sides = a.self == 1 ? 4 : 2;
  for (int i = 0; i < 4; ++i) {
    t.dots[i] = i < sides ? dots[first + i] : nullptr;
    t.ld[i] = i < sides ? ld[first + i] : 0;
  }
  t.top = top;
  return dense_rows_step(t, rows, top == nullptr, sides, a.items, st);  // (wide rows have `top`)
}

// Wavefronts that share the keys of 32 rows: sixteen where eight would leave the chip half empty and
// there are keys for them (3,001 x 4,567 x 33: 326 against 424 us a solve; from 257 workgroups on, and
// at 128 columns, where they cost registers, eight are faster).
template <int DP>
int launch_small(const SmallStepArgs& t, dim3 grid, int64_t working, int key_blocks, hipStream_t st) {
  if constexpr (DP <= 64)
    if (working <= 256 && key_blocks >= 48) {
      hipLaunchKernelGGL((small_step_kernel<DP, 16>), grid, dim3(1024), 0, st, t);
      return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
    }
  hipLaunchKernelGGL((small_step_kernel<DP, 8>), grid, dim3(512), 0, st, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <int DP>
int launch_step(const SmallArgs& a, int step, hipStream_t st) {
  const int xb = std::max(a.blocks[0], a.blocks[1]);
  return launch_small<DP>(step_args(a, step), dim3(xb, a.self == 1 ? 4 : 2, a.items),
                          (int64_t)(a.blocks[0] + a.blocks[1]) * (a.self == 1 ? 2 : 1) * a.items, xb, st);
}

// One alternating iteration: f from the newest g, then g from that f.
template <int DP>
int launch_alternating(const SmallArgs& a, int it, hipStream_t st) {
  for (int side = 0; side < 2; ++side) {
    SmallStepArgs t = step_args(a, it);
    t.side[0] = t.side[side];
    t.full = 1;
    t.extrapolate = -1;  // (iteration `it` is one of the first lens)
    if (side == 1) t.side[0].kpot = a.pot[0] + ((it & 1) ^ 1) * (size_t)a.items * a.rows[0];
    const int rc = launch_small<DP>(t, dim3(a.blocks[side], 1, a.items), (int64_t)a.blocks[side] * a.items,
                                    a.blocks[side ^ 1], st);
    if (rc != FS_OK) return rc;
  }
  return FS_OK;
}

template <int DP>
int launch_pair_merge(const SmallArgs& a, const PairArgs& t, PairArgs* at, int step, hipStream_t st) {
  const int blocks = std::max(a.pblocks[0], a.pblocks[1]);
  // (at one eps the planes are written once, before the first step)
  const int planes = step < 0 || a.sched != 0 ? (blocks + 3) / 4 : 0;
  const int grid = t.merge_groups + planes + (step < 0 ? (8 * t.per_xcd + 1023) / 1024 : 0);
  const auto kernel = DP > 16 || skips(a.d) ? pair_merge_kernel<DP, true> : pair_merge_kernel<DP, DP != 16>;
  hipLaunchKernelGGL(kernel, dim3(grid, a.self == 1 ? 4 : 2, a.items), dim3(1024), 0, st,
                     (PairArgsPtr)at, step, planes);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <int DP>
int launch_pair_step(const SmallArgs& a, const PairArgs& t, PairArgs* at, int step, hipStream_t st) {
  const int blocks = std::min(8 * t.per_xcd, kPairGrid);
  const auto kernel = DP > 16 || skips(a.d) ? pair_sweep_kernel<DP, true> : pair_sweep_kernel<DP, DP != 16>;
  hipLaunchKernelGGL(kernel, dim3(blocks, a.items), dim3(256), 0, st, (PairArgsPtr)at, step);
  return launch_pair_merge<DP>(a, t, at, step, st);
}

template <int DP>
int launch_grad(const SmallArgs& a, const PairArgs& pa, const SmallGradArgs& g, hipStream_t st) {
  const int xb = a.blocks[0] > a.blocks[1] ? a.blocks[0] : a.blocks[1];
  const dim3 grid(!g.out[0] ? a.blocks[1] : (!g.out[1] ? a.blocks[0] : xb), g.out[0] && g.out[1] ? 2 : 1, a.items);
  if constexpr (DP <= 64)
    if (a.pair && skips(a.d)) {
      hipLaunchKernelGGL((small_grad_kernel<DP, PairBlocks>), grid, dim3(512), 0, st, a, g, pair_blocks(pa, a.extrapolate));
      return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
    }
  hipLaunchKernelGGL((small_grad_kernel<DP, SmallAllBlocks>), grid, dim3(512), 0, st, a, g, SmallAllBlocks{});
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

template <typename F>
int by_width(const fs_small_problem* p, F&& f) {
  switch (padded(p)) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    case 48: return f(std::integral_constant<int, 48>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 96: return f(std::integral_constant<int, 96>{});
    default: return f(std::integral_constant<int, 128>{});
  }
}

}  // namespace

int dense_solved(const fs_small_problem* p, void* workspace, size_t workspace_bytes, SmallArgs& a, DenseArgs& t) {
  const int rc = checked(p, true);
  if (rc != FS_OK) return rc;
  if (!use_dense(p) || p->items != 1 || !p->extrapolate) return FS_ERR_UNSUPPORTED;
  return layout(p, workspace, a, nullptr, &t) > workspace_bytes ? FS_ERR_WORKSPACE_TOO_SMALL : FS_OK;
}

}  // namespace fs

using namespace fs;

extern "C" {

size_t fs_small_workspace_bytes(const fs_small_problem* p) {
  if (checked(p) != FS_OK) return 0;
  SmallArgs a;
  return layout(p, nullptr, a);
}

size_t fs_small_products_bytes(const fs_small_problem* p) {
  if (checked(p) != FS_OK || !use_products(p)) return 0;
  SmallArgs a;
  layout(p, nullptr, a);
  return products_at(a, nullptr).bytes;
}

size_t fs_small_last_step_offset(const fs_small_problem* p, int item, int prob) {
  if (checked(p) != FS_OK || !use_pair(p) || item < 0 || item >= p->items || prob < 0 || prob > 2) return 0;
  SmallArgs a;
  PairArgs t;
  layout(p, nullptr, a, &t);
  if (prob < t.first_prob || prob >= t.nprob) return 0;
  return reinterpret_cast<size_t>(t.state) + (((size_t)item * 3 + prob) * kPairStateWords + kPairModes) * 4;
}

int fs_small_solve(const fs_small_problem* p, void* workspace, size_t workspace_bytes, int* host_words,
                   float* loss, float* pots, void* stream) {
  return fs_small_solve_products(p, workspace, workspace_bytes, nullptr, 0, host_words, loss, pots, stream);
}

int fs_small_solve_products(const fs_small_problem* p, void* workspace, size_t workspace_bytes, void* products,
                            size_t products_bytes, int* host_words, float* loss, float* pots, void* stream) {
  int rc = checked(p);
  if (rc != FS_OK) return rc;
  if ((p->sched == 1 || p->threshold > 0.f) && !host_words) return FS_ERR_NULL_POINTER;
  SmallArgs a;
  PairArgs pa, *pair_at = nullptr;
  DenseArgs da;
  if (!workspace || layout(p, workspace, a, &pa, &da, &pair_at) > workspace_bytes) return FS_ERR_WORKSPACE_TOO_SMALL;
  hipStream_t st = (hipStream_t)stream;
  const bool dense = use_dense(p);
  const bool kept = products && use_products(p);
  Products by_rows = products_at(a, products);
  if (kept && by_rows.bytes > products_bytes) return FS_ERR_WORKSPACE_TOO_SMALL;
  if (dense) by_rows = Products{{da.dots, da.dots_t}, {da.ld, da.ld_t}, 0};
  const double rows = (double)a.items * (a.rows[0] + a.rows[1]) * (a.self == 1 ? 2 : 1);
  const int wave_rows = dense ? da.rows : (kept ? (rows <= 2048 ? 1 : 2) : 0);
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
  rc = dense ? dense_prepare(a, da, st) : by_width(p, [&](auto dp) {
    constexpr int DP = decltype(dp)::value;
    const int r = launch_prep<DP>(a, pa, pair_at, st);
    if constexpr (DP <= 64)
      if (r == FS_OK && a.pair) return launch_pair_merge<DP>(a, pa, pair_at, -1, st);
    if (r == FS_OK && kept) return form_products(a, by_rows, DP / 16, st);
    return r;
  });
  if (rc != FS_OK) return rc;
  const int p0 = a.self == 2 ? 1 : 0, p1 = a.self == 0 ? 1 : 3;  // the problems that are solved
  auto run_step = [&](int s) {
    if (wave_rows) return launch_rows(a, s, by_rows.dots, by_rows.ld, dense ? da.top : nullptr, wave_rows, st);
    if (dense) return dense_step(a, da, s, st);
    return by_width(p, [&](auto dp) {
      constexpr int DP = decltype(dp)::value;
      if (a.alternating) return launch_alternating<DP>(a, s, st);
      if constexpr (DP <= 64)
        if (a.pair) return launch_pair_step<DP>(a, pa, pair_at, s, st);
      return launch_step<DP>(a, s, st);
    });
  };
  int ahead = 0;  // steps enqueued already
  if (a.sched == 1) {
    // how many steps there are is known on the device only.  The first ones are enqueued before the
    // host looks, so that the device does not wait for it (a step past the end of a schedule does
    // nothing: 256 x 256 x 16 debiased 12 us less)
    for (; a.threshold <= 0.f && ahead < 6 && rc == FS_OK; ++ahead) rc = run_step(ahead);
    if (rc != FS_OK) return rc;
    rc = wait_for_words(st, [&]() {
      for (int i = 0; i < a.items; ++i)
        if (__atomic_load_n(host_words + 4 * i + 3, __ATOMIC_ACQUIRE) != a.host_token) return false;
      return true;
    });
    if (rc != FS_OK) return rc;
    for (int i = 0; i < a.items; ++i) {  // (see small_schedule)
      const int lens = __atomic_load_n(host_words + 4 * i + 2, __ATOMIC_RELAXED);
      for (int q = 0; q < 3; ++q) __atomic_store_n(host_words + 4 * i + q, (lens >> (10 * q) & 1023) - 3, __ATOMIC_RELAXED);
    }
    entries = 0;
    for (int i = 0; i < a.items; ++i)
      for (int q = p0; q < p1; ++q) {
        const int k = host_words[4 * i + q];
        if (k <= 0) return k == -1 ? FS_SMALL_NO_DIAMETER : (k == -2 ? FS_SMALL_NOT_A_NUMBER : FS_SMALL_LONG_SCHEDULE);
        if (k > entries) entries = k;
      }
  }
  const int n_steps = a.alternating ? entries : entries + 1 + a.extrapolate;
  const bool early = a.threshold > 0.f;
  // early stopping: entries of every problem's schedule (no memory for them: an error, not an exception
  // that would leave a C entry point)
  const std::unique_ptr<int[]> length(early ? new (std::nothrow) int[3 * (size_t)a.items] : nullptr);
  if (early && !length) return FS_ERR_LAUNCH_FAILED;
  if (early)
    for (int i = 0; i < a.items; ++i)
      for (int q = 0; q < 4; ++q) {
        if (q < 3) length[3 * (size_t)i + q] = a.sched == 1 ? host_words[4 * i + q] : entries;
        __atomic_store_n(host_words + 4 * i + q, -1, __ATOMIC_RELAXED);
      }
  int checks = 0;
  bool all_done = false, ahead_of_us = false;
  // waits for what check number c has to say; all_done: no problem has entries left to run;
  // ahead_of_us: one of them stopped at a later check, which the device has run as well by now
  auto check_result = [&](int c) {
    return wait_for_words(st, [&]() {
      all_done = true;
      ahead_of_us = false;
      for (int i = 0; i < a.items; ++i)
        for (int q = p0; q < p1; ++q) {
          const int v = __atomic_load_n(host_words + 4 * i + q, __ATOMIC_ACQUIRE);
          ahead_of_us = ahead_of_us || (v >= 0 && v > 2 * c + 1);
          if ((v >= 0 && (v & 1)) || length[3 * i + q] < (c + 1) * p->check_every) continue;
          all_done = false;
          if (v < 2 * c) return false;
        }
      return true;
    });
  };
  int s = ahead;
  for (; s < n_steps && rc == FS_OK && !all_done; ++s) {
    rc = run_step(s);
    const int done = a.alternating ? s + 1 : s;  // averaged steps or iterations
    if (rc != FS_OK || !early || done == 0 || done > entries || done % p->check_every != 0) continue;
    hipLaunchKernelGGL((small_check_kernel<0>), dim3(p1 - p0, a.items), dim3(1024), 0, st, a, done, checks);
    if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
    // (asked for with one more stretch of steps enqueued, so that the device does not wait)
    if (checks > 0) rc = check_result(checks - 1);
    ++checks;
  }
  // (the extrapolation of a problem that stopped at the newest check is the next step; for the others
  // it does nothing)
  if (rc == FS_OK && all_done && ahead_of_us && s < n_steps && !a.alternating) rc = run_step(s);
  if (rc == FS_OK && early && checks > 0 && !all_done) rc = check_result(checks - 1);
  if (rc != FS_OK || (!loss && !pots)) return rc;
  SmallLossArgs l;
  l.loss = loss;
  l.pots = pots;
  l.relaxed = a.rho[0] > 0.f && a.rho[1] > 0.f ? 1 : 0;
  const int parts = loss_parts(a);
  l.parts = a.stats;  // (done with since the preparation)
  hipLaunchKernelGGL((small_loss_kernel<0>), dim3(parts, a.items), dim3(1024), 0, st, a, l);
  if (loss && parts > 1) hipLaunchKernelGGL((small_loss_sum_kernel<0>), dim3(a.items), dim3(64), 0, st, l, parts);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int fs_small_potentials(const fs_small_problem* p, void* workspace, size_t workspace_bytes, float* const* pots,
                        void* stream) {
  const int rc = checked(p);
  if (rc != FS_OK) return rc;
  if (!pots) return FS_ERR_NULL_POINTER;
  SmallArgs a;
  if (layout(p, workspace, a) > workspace_bytes || !workspace) return FS_ERR_WORKSPACE_TOO_SMALL;
  SmallPotArgs t;
  std::memcpy(t.pots, pots, sizeof(t.pots));
  const dim3 grid((std::max(a.rows[0], a.rows[1]) + 1023) / 1024, a.self == 1 ? 4 : 2, a.items);
  hipLaunchKernelGGL((small_potentials_kernel<0>), grid, dim3(1024), 0, (hipStream_t)stream, a, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int fs_small_grad(const fs_small_problem* p, void* workspace, size_t workspace_bytes, const float* grad_out,
                  float* grad_x, float* grad_y, void* stream) {
  const int rc = checked(p);
  if (rc != FS_OK) return rc;
  if (!grad_out) return FS_ERR_NULL_POINTER;
  if (!p->want_values) return FS_ERR_BAD_ARGUMENT;
  SmallArgs a;
  PairArgs pa;
  if (layout(p, workspace, a, &pa) > workspace_bytes || !workspace) return FS_ERR_WORKSPACE_TOO_SMALL;
  if (!grad_x && !grad_y) return FS_OK;
  SmallGradArgs g;
  g.grad_out = grad_out;
  g.out[0] = grad_x;
  g.out[1] = grad_y;
  return by_width(p, [&](auto dp) { return launch_grad<decltype(dp)::value>(a, pa, g, (hipStream_t)stream); });
}

}  // extern "C"
