// Symmetric steps on the kept matrix of inner products, for wide rows.
//
// A step evaluates n m logits.  Formed anew each costs 3 d matrix-core multiply-adds (two fp16 planes a
// side), kept it costs reading four bytes: from a few hundred columns on reading wins, at
// 8192 x 8192 x 1536 by six (495 us for a one-sweep step that forms them, about 70 for one that reads
// 268 MB).  So the products x_i.y_j are formed once per solve, in the same two-plane arithmetic, and
// kept as fp32 [n][ld]; 288 GB of HBM hold them many times over, and up to 256 MB of them stay
// in the last-level cache between steps.  Kernels:
//   dense_gemm_kernel   C = A B^T on two-plane operands in MFMA order
//   dense_sweep_kernel  both half-updates' soft-max statistics from one reading of the products
//   dense_merge_kernel  the new potentials from them
//   dense_rows_kernel   both in one launch, on the products and their transpose (up to 1e7 of them)
#pragma once

#include "fs_common.hpp"
#include "fs_small.hpp"

namespace fs {

// Planes in operand order, hi and lo next to each other: per 32 rows and 16 columns two blocks of
// 64 16-byte words, word (h, row % 32) holding columns 8 h .. 8 h + 7.
constexpr int kDenseStep = 2 * 64;

struct DenseArgs {
  float* dots;             // [items][n][ld], ld a multiple of 256, zero beyond the m-th column
  u32x4* planes[2];        // [items][blocks][steps][2][64]
  int blocks[2];           // 32-row blocks, a multiple of 8 (zero rows behind the last one)
  int steps;               // 16-column steps
  int n, m, ld, items, chunk, chunks, groups;
  float2* part[2];         // (maximum, sum): [items][chunks][n] of the rows, [items][groups][m] of the columns
  float* top;              // [items][n] the largest logit of a row of x in the extrapolation, for dense_plan_kernel
  const float* pot[2];     // this step's potentials, log weights, norms
  float* out[2];
  const float* l2w[2];
  const float* norm[2];
  const float4* table;      // [items][3][table_len]
  const int* lens;
  float rho[2];
  int table_len;
  int step, sched, extrapolate;
  int large;               // the shape of dense_sweep_kernel
  int turns;               // every other step reads the products backwards
  // (not read by the kernels that take this, and behind what they read)
  float* dots_t;           // [items][m][ld_t]: the products transposed, where a step is one launch (`rows`)
  int ld_t, rows;          // rows: rows of a wavefront in dense_rows_kernel, 0: dense_sweep_kernel
};

// Largest magnitude and sum of the weights of a slice of one matrix (small_stats_kernel's first two
// words; no bounding boxes: a schedule comes as a table here).  Bound by memory.
__device__ __forceinline__ void dense_stats_of(const SmallArgs& a, int mat, int item) {
  const int tid = threadIdx.x;
  const size_t count = (size_t)a.rows[mat] * a.d, base = item * count;
  const bool wide = small_wide(a.pts[mat], a.d, a.dtype);
  float am = 0.f, ws = 0.f;
  const size_t stride = (size_t)gridDim.x * 1024 * 8;
#pragma unroll 2
  for (size_t i = ((size_t)blockIdx.x * 1024 + tid) * 8; i < count; i += stride) {
    float v[8];
    if (i + 8 <= count) {
      small_load8(v, a.pts[mat], base + i, a.dtype, wide);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = i + k < count ? small_load(a.pts[mat], base + i + k, a.dtype) : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) am = fmaxf(am, fabsf(v[k]));
  }
  if (a.w[mat] != nullptr)
    for (int i = blockIdx.x * 1024 + tid; i < a.rows[mat]; i += gridDim.x * 1024)
      ws += a.w[mat][(size_t)item * a.rows[mat] + i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    am = fmaxf(am, __shfl_xor(am, o, 64));
    ws += __shfl_xor(ws, o, 64);
  }
  __shared__ float sh[2][16];
  if ((tid & 63) == 0) sh[0][tid >> 6] = am, sh[1][tid >> 6] = ws;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w) am = fmaxf(am, sh[0][w]), ws += sh[1][w];
    float* out = a.stats + (((size_t)item * 2 + mat) * a.stat_blocks + blockIdx.x) * a.stat_words;
    out[0] = am;
    out[1] = ws;
  }
}
template <int T>
__global__ __launch_bounds__(1024) void dense_stats_kernel(const SmallArgs a) {
  dense_stats_of(a, blockIdx.y, blockIdx.z);
}

// Planes of 32 rows, their norms, log weights and initial potentials.  Grid (blocks of the larger
// matrix and one more, which fills the table of a fixed eps; matrices; items).
__device__ __forceinline__ void dense_prep_of(const SmallArgs& a, const DenseArgs& t, int mat, int item) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x == gridDim.x - 1) {
    if (mat == 0) small_schedule(a, item);
    return;
  }
  const int rb = blockIdx.x, rows = a.rows[mat], d = a.d;
  if (rb >= t.blocks[mat]) return;
  const int wave = tid >> 6, lane = tid & 63, li = lane & 31, h = lane >> 5;
  float am, ws;
  small_merge_stats(a, item, mat, am, ws);
  const float sc = f16_plane_scale(am);
  if (rb == 0 && tid == 0) a.scale[item * 2 + mat] = make_float2(sc, 1.0f / sc);
  const int row = rb * 32 + li;
  const bool live = row < rows, wide = small_wide(a.pts[mat], d, a.dtype);
  const size_t base = ((size_t)item * rows + min(row, rows - 1)) * d;
  u32x4* po = t.planes[mat] + ((size_t)item * t.blocks[mat] + rb) * (size_t)t.steps * kDenseStep + lane;
  float q = 0.f;
  for (int kk = wave; kk < t.steps; kk += 8) {
    float v[8];
    const int c0 = 16 * kk + 8 * h;
    if (c0 + 8 <= d) {
      small_load8(v, a.pts[mat], base + c0, a.dtype, wide);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = c0 + k < d ? small_load(a.pts[mat], base + c0 + k, a.dtype) : 0.f;
    }
    u32x4 hi, lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float v0 = live ? sc * v[2 * k] : 0.f, v1 = live ? sc * v[2 * k + 1] : 0.f;
      const _Float16 h0 = (_Float16)v0, h1 = (_Float16)v1;
      hi[k] = pack_f16((float)h0, (float)h1);
      lo[k] = pack_f16(v0 - (float)h0, v1 - (float)h1);
      q = __builtin_fmaf(v0, v0, __builtin_fmaf(v1, v1, q));
    }
    po[(size_t)kk * kDenseStep] = hi;
    po[(size_t)kk * kDenseStep + 64] = lo;
  }
  __shared__ float sh[8][64];
  sh[wave][lane] = q;
  __syncthreads();
  if (tid >= 32 || !live) return;
  q = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w) q += sh[w][tid] + sh[w][tid + 32];
  const float inv = 1.0f / sc, al = a.cost_scale * (q * inv * inv);
  const size_t at = (size_t)item * rows + row;
  a.norm[mat][at] = al;
  float w = a.w[mat] == nullptr ? 1.0f / (float)rows : a.w[mat][at];
  if (a.w[mat] != nullptr && a.normalize) w = w / fmaxf(ws, 1e-40f);
  a.wt[mat][at] = w;
  a.l2w[mat][at] = w > 0.f ? small_log2(w, 0.f) : -100000.0f * kLog2e;
  a.pot[mat][at] = -al;
}
template <int T>
__global__ __launch_bounds__(512) void dense_prep_kernel(const SmallArgs a, const DenseArgs t) {
  dense_prep_of(a, t, blockIdx.y, blockIdx.z);
}

// One operand's tile stream and C = A B^T: a workgroup of WR x WC wavefronts owns 32 WR RB rows and
// 32 WC CB columns; per 16-column step both operands' blocks come into one of ST LDS stages by
// direct global -> LDS loads of 1 KiB per wavefront: with four stages three steps ahead and a barrier per step, with eight six
// steps ahead and a barrier per two (dense_gemm_tile).
// Bound by the matrix pipe: RB CB 3 MFMAs per wavefront and step against 2 (RB + CB) LDS reads.
// LDS reads are written out by hand (the compiler would have each wait for the loads in flight).
struct DenseGemmArgs {
  const u32x4* a;           // rows, columns: planes
  const u32x4* b;
  int a_blocks, b_blocks;   // blocks per item
  int steps, rows, ld;      // rows: of the result, per item
  int splits, run;          // parts of the contraction (each a result of its own) and their steps
  const float2* scale[2];   // of the rows' and of the columns' planes, with inverses, two words an item; null: none
  float* out;               // [splits or items][rows][ld]
  float* out_t;             // [items][cols][ld_t], the result transposed, or null
  int cols, ld_t;
  int row_tiles, col_tiles;
  // words from one 16-column step to the next and from the hi to the lo plane (of both operands): kDenseStep and 64,
  // or those of planes in the order of small_prep_kernel, whose blocks are not padded to whole tiles
  int step_words, plane_words;
};

// APART: the cross products of all steps before hi * hi of the first, in a second pass (see dense_gemm_jobs_kernel), a
// stage of which is the hi planes of two steps (an even number of them).
//
// With eight stages a barrier lies between two steps and the next two: a tile of 64 x 64 has three products a step and
// wavefront, and where a CU has one or two workgroups nothing covers the barrier and the LDS reads in front of them (with
// eight stages and a barrier a step nothing was gained).  1,000 x 1,000 x 784 13.4 -> 12.3 us, 600 x 700 x 1,400 16.5 -> 13.9,
// 900 x 1,300 x 163 8.4 -> 8.2, of which some 5 are the launch, the first loads and the results.
template <int WR, int WC, int RB, int CB, bool APART, int ST>
__device__ __forceinline__ void dense_gemm_tile(const DenseGemmArgs& g, int split) {
  constexpr int W = WR * WC, TR = WR * RB, TC = WC * CB, PIECES = 2 * (TR + TC), LOADS = PIECES / W;
  constexpr int PER = ST == 8 ? 2 : 1;  // steps between two barriers
  static_assert((ST & (ST - 1)) == 0 && (ST - 2 * PER) * LOADS < 64, "stages in turn, and loads in flight that a wait can count");
  static_assert(PIECES % W == 0, "every wavefront moves the same number of pieces");
  static_assert(2 * RB * 1024 <= 65535 && 2 * CB * 1024 <= 65535, "offsets of the LDS reads");
  __shared__ __attribute__((aligned(16))) u32x4 lds[ST * PIECES * 64];
  // XCD x takes the x-th eighth of the tiles in the order (4 row tiles, column tile, row tile):
  // what shares an L2 shares operands
  const int tiles = g.row_tiles * g.col_tiles, per_xcd = (tiles + 7) / 8;
  int item = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per_xcd || item >= tiles) return;
  const int band = item / (4 * g.col_tiles), within = item % (4 * g.col_tiles);
  const int nb = min(4, g.row_tiles - 4 * band);
  const int rt = 4 * band + within % nb, ct = within / nb, z = blockIdx.y;
  const int k_begin = split * g.run, steps = min(g.steps - k_begin, g.run);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 31, h = lane >> 5, wr = wave / WC, wc = wave % WC;

  // piece p of a stage: block p / 2 (the rows' first), plane p % 2
  const u32x4* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int p = wave * LOADS + i, blk = p / 2;
    const bool of_a = blk < TR;
    // (past the last block: that one again, for results that nobody takes)
    const int gb = of_a ? min(rt * TR + blk, g.a_blocks - 1) : min(ct * TC + blk - TR, g.b_blocks - 1);
    src[i] = (of_a ? g.a + ((size_t)z * g.a_blocks + gb) * (size_t)g.steps * kDenseStep
                   : g.b + ((size_t)z * g.b_blocks + gb) * (size_t)g.steps * kDenseStep) +
             ((size_t)k_begin * g.step_words + (p & 1) * g.plane_words + lane);
  }
  const int total = APART ? steps + steps / 2 : steps;
  static_assert(LOADS % 2 == 0, "load i of a wavefront is of plane i % 2");
  auto stage = [&](int k, int buf) {
    k = min(k, total - 1);
    const bool hi = APART && k >= steps;
    if (hi) k = 2 * (k - steps);
    const long long at[2] = {(long long)k * g.step_words, (long long)(k + (hi ? 1 : 0)) * g.step_words - (hi ? g.plane_words : 0)};
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src[i] + at[i & 1]),
          (__attribute__((address_space(3))) void*)(&lds[(buf * PIECES + wave * LOADS + i) * 64]), 16, 0, 0);
  };
  const unsigned base = (unsigned)(size_t)(const __attribute__((address_space(3))) u32x4*)&lds[0] + lane * 16;
  const unsigned abase = base + wr * RB * 2 * 1024, bbase = base + (TR + wc * CB) * 2 * 1024;

  f32x16 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

#pragma unroll
  for (int k = 0; k < ST - PER; ++k) stage(k, k);
  for (int k = 0; k < total; k += PER) {
    constexpr int newer = (ST - 2 * PER) * LOADS;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (newer & 15) | ((newer >> 4) << 14));  // the steps from k on have landed
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();  // for everyone, and those before have been read by everyone
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < PER; ++q) stage(k + ST - PER + q, (k + ST - PER + q) & (ST - 1));
    u32x4 x[PER][RB][2], y[PER][CB][2];
    static_for<PER>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const unsigned off = ((k + q) & (ST - 1)) * (PIECES * 1024);
      static_for<2 * RB>([&](auto i) { x[q][i / 2][i % 2] = lds_read16<decltype(i)::value * 1024>(abase + off); });
      static_for<2 * CB>([&](auto i) { y[q][i / 2][i % 2] = lds_read16<decltype(i)::value * 1024>(bbase + off); });
    });
    static_for<PER * CB>([&](auto at) {
      constexpr int q = decltype(at)::value / CB, j = decltype(at)::value % CB;
      // this column block has been read; LDS returns in order
      constexpr int later = 2 * (CB - 1 - j) + 2 * (PER - 1 - q) * (RB + CB);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F | (later << 8));
      __builtin_amdgcn_sched_barrier(0);
      if (q > 0 && k + q >= total) return;  // (an odd number of steps)
      if (!APART || k < steps) {
#pragma unroll
        for (int prod = 0; prod < (APART ? 2 : 3); ++prod)
#pragma unroll
          for (int i = 0; i < RB; ++i)
            acc[i][j] = small_mfma(x[q][i][prod == 0 ? 1 : 0], y[q][j][prod == 1 ? 1 : 0], acc[i][j]);
      } else {
#pragma unroll
        for (int step = 0; step < 2; ++step)
#pragma unroll
          for (int i = 0; i < RB; ++i) acc[i][j] = small_mfma(x[q][i][step], y[q][j][step], acc[i][j]);
      }
    });
  }
  __builtin_amdgcn_s_waitcnt(0);
  const float inv = g.scale[0] == nullptr ? 1.0f : g.scale[0][z * 2].y * g.scale[1][z * 2].y;
  float* out = g.out + (size_t)(z + split) * g.rows * g.ld;  // (one item where the contraction is split)
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = (rt * TR + wr * RB + i) * 32 + 8 * (r / 4) + 4 * h + r % 4;
      if (row < g.rows)
#pragma unroll
        for (int j = 0; j < CB; ++j) out[(size_t)row * g.ld + (ct * TC + wc * CB + j) * 32 + li] = acc[i][j][r] * inv;
    }
  if (g.out_t == nullptr) return;
  // (a lane holds four consecutive rows of one column, four times)
  float* out_t = g.out_t + (size_t)z * g.cols * g.ld_t;
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int col = (ct * TC + wc * CB + j) * 32 + li;
    if (col < g.cols)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(out_t + (size_t)col * g.ld_t + (rt * TR + wr * RB + i) * 32 + 8 * q + 4 * h) =
              make_float4(acc[i][j][4 * q] * inv, acc[i][j][4 * q + 1] * inv, acc[i][j][4 * q + 2] * inv,
                          acc[i][j][4 * q + 3] * inv);
  }
}

template <int WR, int WC, int RB, int CB, int ST>
__global__ __launch_bounds__(64 * WR * WC, 2) void dense_gemm_kernel(const DenseGemmArgs g) {
  dense_gemm_tile<WR, WC, RB, CB, false, ST>(g, blockIdx.z);
}

// Up to four products of the same depth in one launch, summed in the order of steps on planes: the cross products before
// hi * hi.  (Added to hi * hi step by step, each is rounded to the last place of a sum 2^11 times as large, and not alike
// for both sides of a pair: potentials of 1,000 to 2,500 points after 40 steps were 1.1 to 1.6 times as far from fp64, with
// the logits of dense_rows_kernel in base 2; now they are as far.  The second pass takes 13 us for 11 at 2,048 x 64, 37 for 28 at
// 3,000 x 2,800 x 100.)
struct DenseGemmJobs {
  DenseGemmArgs job[4];
};
template <int WR, int WC, int RB, int CB, bool APART, int ST>
__global__ __launch_bounds__(64 * WR * WC, 2) void dense_gemm_jobs_kernel(const DenseGemmJobs g) {
  dense_gemm_tile<WR, WC, RB, CB, APART, ST>(g.job[blockIdx.z], 0);
}

__device__ __forceinline__ void dense_join(float& m, float& s, float m2, float s2) {
  const float M = fmaxf(m, m2);
  s = s * fast_exp2(m - M) + s2 * fast_exp2(m2 - M);
  m = M;
}

// Soft-max statistics of all rows (over the columns' biases) and of all columns (over the rows').  A
// wavefront reads RW rows of 256 columns (1 KiB a row) at a time, a lane four columns of them; the
// rows' running statistics stay lane-private over the workgroup's run of columns and cross lanes
// once, the columns' are lane-private over the rows and cross wavefronts through LDS.  Bound by
// memory (HBM or last-level cache); two exponentials per product hide behind it with four
// wavefronts per SIMD.  Both directions carry running maxima: no step needs permission.
//
// Every other step over more products than the L2s hold goes from the last to the first, and finds in the
// 256 MB of the last-level cache what the step before has read last (in one order, what does not fit pushes
// out all of it).  50 steps of 9,000 x 9,000 (324 MB) 5.15 -> 4.18 ms, 12,000 points 7.87 -> 7.13, 16,000 13.0 ->
// 12.2, 4,000 x 5,000 1.59 -> 1.52; 8,192 points (268 MB) 3.07 as before.  Up to 32 MB one order
// is faster: 2,000 points 0.80 ms for 0.86.
template <int RW, int WV>
__global__ __launch_bounds__(64 * WV, 4) void dense_sweep_kernel(const DenseArgs a) {
  constexpr int B = 8;  // rows in registers
  static_assert(RW % B == 0, "");
  __shared__ float2 sh[2][WV][256];
  const bool back = a.turns && (a.step & 1);
  const int group = back ? gridDim.x - 1 - blockIdx.x : blockIdx.x, ch = back ? gridDim.y - 1 - blockIdx.y : blockIdx.y;
  const int item = back ? gridDim.z - 1 - blockIdx.z : blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int entries = a.lens[item * 3];
  if (a.step > entries + a.extrapolate) return;
  const float4 coef = a.table[(size_t)item * 3 * a.table_len + (a.sched == 0 ? 0 : min(max(a.step - 1, 0), a.table_len - 1))];
  const float qs = coef.y, kc = coef.w;
  const int r0 = (group * WV + wave) * RW;
  const float* dots = a.dots + (size_t)item * a.n * a.ld;
  // the rows' biases, one per lane
  float rb;
  {
    const int row = r0 + (lane & (RW - 1));
    const size_t at = (size_t)item * a.n + min(row, a.n - 1);
    rb = row < a.n ? fmaxf(__builtin_fmaf(kc, a.pot[0][at], a.l2w[0][at]), kNegBig) : kNegBig;
  }
  float rm[RW], rs[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) rm[r] = kNegBig, rs[r] = 0.f;
  const int c_first = ch * a.chunk, pieces = (min(a.ld, c_first + a.chunk) - c_first) / 256;
  int buf = 0;
  for (int piece = 0; piece < pieces; ++piece, buf ^= 1) {
    const int c0 = c_first + 256 * (back ? pieces - 1 - piece : piece);
    float kb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int col = c0 + 4 * lane + k;
      const size_t at = (size_t)item * a.m + min(col, a.m - 1);
      kb[k] = col < a.m ? fmaxf(__builtin_fmaf(kc, a.pot[1][at], a.l2w[1][at]), kNegBig) : kNegBig;
    }
    float cm[4], cs[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) cm[k] = kNegBig, cs[k] = 0.f;
#pragma unroll
    for (int b0 = 0; b0 < RW; b0 += B) {
      float4 v[B];
#pragma unroll
      for (int r = 0; r < B; ++r)
        v[r] = *reinterpret_cast<const float4*>(dots + (size_t)min(r0 + b0 + r, a.n - 1) * a.ld + c0 + 4 * lane);
      float mc[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) mc[k] = cm[k];
#pragma unroll
      for (int r = 0; r < B; ++r) {
        // ---- the row ----
        const float l0 = __builtin_fmaf(v[r].x, qs, kb[0]), l1 = __builtin_fmaf(v[r].y, qs, kb[1]);
        const float l2 = __builtin_fmaf(v[r].z, qs, kb[2]), l3 = __builtin_fmaf(v[r].w, qs, kb[3]);
        float& m = rm[b0 + r];
        float& s = rs[b0 + r];
        const float M = fmaxf(fmaxf(fmaxf(l0, l1), fmaxf(l2, l3)), m);
        s = s * fast_exp2(m - M) + ((fast_exp2(l0 - M) + fast_exp2(l1 - M)) + (fast_exp2(l2 - M) + fast_exp2(l3 - M)));
        m = M;
        // ---- the columns' maxima ----
        const float br = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, rb), b0 + r));
        v[r].x = __builtin_fmaf(v[r].x, qs, br);
        v[r].y = __builtin_fmaf(v[r].y, qs, br);
        v[r].z = __builtin_fmaf(v[r].z, qs, br);
        v[r].w = __builtin_fmaf(v[r].w, qs, br);
        mc[0] = fmaxf(mc[0], v[r].x);
        mc[1] = fmaxf(mc[1], v[r].y);
        mc[2] = fmaxf(mc[2], v[r].z);
        mc[3] = fmaxf(mc[3], v[r].w);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float s = cs[k] * fast_exp2(cm[k] - mc[k]);
#pragma unroll
        for (int r = 0; r < B; ++r) s += fast_exp2((k == 0 ? v[r].x : k == 1 ? v[r].y : k == 2 ? v[r].z : v[r].w) - mc[k]);
        cs[k] = s;
        cm[k] = mc[k];
      }
    }
    float4* o = reinterpret_cast<float4*>(&sh[buf][wave][4 * lane]);
    o[0] = make_float4(cm[0], cs[0], cm[1], cs[1]);
    o[1] = make_float4(cm[2], cs[2], cm[3], cs[3]);
    __syncthreads();  // (the other buffer is free once everyone is here)
    for (int c = threadIdx.x; c < 256; c += 64 * WV) {
      float m = sh[buf][0][c].x, s = sh[buf][0][c].y;
#pragma unroll
      for (int w = 1; w < WV; ++w) dense_join(m, s, sh[buf][w][c].x, sh[buf][w][c].y);
      if (c0 + c < a.m) a.part[1][((size_t)item * a.groups + group) * a.m + c0 + c] = make_float2(m, s);
    }
  }
  // ---- the rows' statistics over the lanes: halves of the rows change places ----
#pragma unroll
  for (int o = 32, n = RW / 2; n > 0; o >>= 1, n >>= 1) {
    const bool up = lane & o;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const float gm = up ? rm[r] : rm[r + n], gs = up ? rs[r] : rs[r + n];
      float m = up ? rm[r + n] : rm[r], s = up ? rs[r + n] : rs[r];
      dense_join(m, s, __shfl_xor(gm, o, 64), __shfl_xor(gs, o, 64));
      rm[r] = m;
      rs[r] = s;
    }
  }
  constexpr int LEFT = 64 / RW;  // lanes that share a row
#pragma unroll
  for (int o = LEFT / 2; o > 0; o >>= 1) dense_join(rm[0], rs[0], __shfl_xor(rm[0], o, 64), __shfl_xor(rs[0], o, 64));
  const int row = r0 + lane / LEFT;
  if (lane % LEFT == 0 && row < a.n) a.part[0][((size_t)item * a.chunks + ch) * a.n + row] = make_float2(rm[0], rs[0]);
}

// The new potentials: 64 rows of one side per workgroup, its four wavefronts share the parts.
template <int T>
__global__ __launch_bounds__(256) void dense_merge_kernel(const DenseArgs a) {
  const int side = blockIdx.y, item = blockIdx.z, rows = side ? a.m : a.n;
  if ((int)blockIdx.x * 64 >= rows) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int entries = a.lens[item * 3];
  if (a.step > entries + a.extrapolate) return;
  const float eps = a.table[(size_t)item * 3 * a.table_len + (a.sched == 0 ? 0 : min(max(a.step - 1, 0), a.table_len - 1))].x;
  const int row = blockIdx.x * 64 + lane, rc = min(row, rows - 1), parts = side ? a.groups : a.chunks;
  const size_t at = (size_t)item * rows + rc;
  const float old = a.pot[side][at], norm = a.norm[side][at];
  const float2* p = a.part[side] + (size_t)item * parts * rows + rc;
  float M = kNegBig, S = 0.f;
#pragma unroll 8
  for (int c = wave; c < parts; c += 4) {
    const float2 v = p[(size_t)c * rows];
    dense_join(M, S, v.x, v.y);
  }
  __shared__ float2 sh[4][64];
  sh[wave][lane] = make_float2(M, S);
  __syncthreads();
  if (wave > 0 || row >= rows) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) dense_join(M, S, sh[w][lane].x, sh[w][lane].y);
  const float rho = a.rho[side], damp = rho > 0.f ? 1.0f / (1.0f + eps / rho) : 1.0f;
  const float alpha = (a.step == 0 || a.step > entries) ? 1.0f : 0.5f;
  float f = alpha * (-eps * damp * kLn2 * small_log2(fmaxf(S, 1e-40f), M));
  if (alpha != 1.0f) f += (1.0f - alpha) * old;
  if (damp < 1.0f) f -= alpha * (1.0f - damp) * norm;
  a.out[side][at] = f;
  if (side == 0 && a.step > entries) a.top[at] = M;
}

// A step of every problem in one launch, where the products and their transposes stay in the last-level
// cache: a wavefront owns R rows of one side and reads all of their products, so nothing is left to a merge; the
// columns of the xy products are rows of a transposed copy, which the product's epilogue writes beside the
// other.  Bound by the launch and the chain of loads in front of the first logit (1,000 points: 4.0 us a
// step, 7.5 by sweep and merge), so the products' first piece is on its way before the biases of the keys, which
// the workgroup's eight wavefronts share in LDS; from 2,000 points on by reading 2 x 4 bytes a product (7.3 us,
// 4.4 TB/s).  RAW: logits in units of the products, as the steps on planes of the same problems have them (there a row's
// logit and that of its column, which each hold the other's potential, are rounded alike, and what does not cancel adds
// up in the slow modes of a peaked plan).  Grid (rows of the largest side, sides, items).
constexpr int kDenseRowKeys = 4096;  // most keys (their biases in LDS)
struct DenseRowArgs {
  SmallStepArgs s;        // (the planes are not read)
  const float* dots[4];   // [items][rows][ld] of every side
  int ld[4];
  float* top;             // [items][nq] the largest logit of a row of side 0 in the extrapolation, or null
};
template <int R, bool RAW>
__global__ __launch_bounds__(512) void dense_rows_kernel(const DenseRowArgs a) {
  constexpr int P = 4;  // 16-byte words of a row per lane and piece: 1024 keys
  __shared__ __attribute__((aligned(16))) float bias[kDenseRowKeys];
  const int side = blockIdx.y, item = blockIdx.z, tid = threadIdx.x;
  const SmallStepSide& sd = a.s.side[side];
  const int nq = sd.nq, nk = sd.nk, ld = a.ld[side];
  if ((int)blockIdx.x * 8 * R >= nq) return;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int row0 = ((int)blockIdx.x * 8 + wave) * R;
  const float* dots = a.dots[side] + (size_t)item * nq * ld + 4 * lane;
  const float* row[R];
#pragma unroll
  for (int r = 0; r < R; ++r) row[r] = dots + (size_t)min(row0 + r, nq - 1) * ld;
  // (a piece may end behind a row's last word: that word again, for nobody)
  auto load = [&](float4 (&v)[R][P], int c0) {
#pragma unroll
    for (int k = 0; k < P; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) v[r][k] = *reinterpret_cast<const float4*>(row[r] + min(c0 + 256 * k, ld - 256));
  };
  float4 v[R][P];
  load(v, 0);
  const int entries = sd.lens[item * 3], step = a.s.step;
  const float4 coef = sd.coef[(size_t)item * a.s.coef_stride];
  const size_t at = (size_t)item * nq + min(row0 + min(lane, R - 1), nq - 1);
  const float old = sd.old[at], norm = sd.norm[at];
  const float* kpot = sd.kpot + (size_t)item * nk;
  const float* kl2w = sd.kl2w + (size_t)item * nk;
  const float eps = coef.x, qs = coef.y, kc = coef.w;
  const float raw = RAW ? coef.z : 1.0f, masked = fmaxf(kNegBig * raw, -3.0e38f);
  const float no_max = RAW ? 0.5f * masked * qs : kNegBig;
  for (int j = tid; j < ld; j += 512) {
    const float b = __builtin_fmaf(kc, kpot[min(j, nk - 1)], kl2w[min(j, nk - 1)]) * raw;
    bias[j] = j < nk ? fmaxf(b, masked) : masked;
  }
  __syncthreads();
  if (step > entries + a.s.extrapolate) return;  // (its schedule is shorter)

  float m[R], s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) m[r] = no_max, s[r] = 0.f;
  for (int c0 = 0; c0 < ld; c0 += 256 * P) {
    float4 next[R][P];
    if (c0 + 256 * P < ld) load(next, c0 + 256 * P);
    if constexpr (RAW) {  // one maximum and rescale for the piece
      float M[R];
#pragma unroll
      for (int r = 0; r < R; ++r) M[r] = 0.5f * masked;
#pragma unroll
      for (int k = 0; k < P; ++k) {
        if (c0 + 256 * k >= ld) break;
        const float4 kb = *reinterpret_cast<const float4*>(&bias[c0 + 256 * k + 4 * lane]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float4& l = v[r][k];
          l = make_float4(l.x + kb.x, l.y + kb.y, l.z + kb.z, l.w + kb.w);
          M[r] = fmaxf(M[r], fmaxf(fmaxf(l.x, l.y), fmaxf(l.z, l.w)));
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        M[r] *= qs;
        asm("" : "+v"(M[r]));  // (rounded once, whatever it is used for)
        M[r] = fmaxf(M[r], m[r]);
        s[r] *= fast_exp2(m[r] - M[r]);
        m[r] = M[r];
      }
#pragma unroll
      for (int k = 0; k < P; ++k) {
        if (c0 + 256 * k >= ld) break;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float4 l = v[r][k];
          s[r] += (fast_exp2(__builtin_fmaf(l.x, qs, -m[r])) + fast_exp2(__builtin_fmaf(l.y, qs, -m[r]))) +
                  (fast_exp2(__builtin_fmaf(l.z, qs, -m[r])) + fast_exp2(__builtin_fmaf(l.w, qs, -m[r])));
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < P; ++k) {
        if (c0 + 256 * k >= ld) break;
        const float4 kb = *reinterpret_cast<const float4*>(&bias[c0 + 256 * k + 4 * lane]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float l0 = __builtin_fmaf(v[r][k].x, qs, kb.x), l1 = __builtin_fmaf(v[r][k].y, qs, kb.y);
          const float l2 = __builtin_fmaf(v[r][k].z, qs, kb.z), l3 = __builtin_fmaf(v[r][k].w, qs, kb.w);
          const float M = fmaxf(fmaxf(fmaxf(l0, l1), fmaxf(l2, l3)), m[r]);
          s[r] = s[r] * fast_exp2(m[r] - M) +
                 ((fast_exp2(l0 - M) + fast_exp2(l1 - M)) + (fast_exp2(l2 - M) + fast_exp2(l3 - M)));
          m[r] = M;
        }
      }
    }
    if (c0 + 256 * P < ld)
#pragma unroll
      for (int k = 0; k < P; ++k)
#pragma unroll
        for (int r = 0; r < R; ++r) v[r][k] = next[r][k];
  }
  float M = kNegBig, S = 0.f;  // lane r: row r
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float t = m[r];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t = fmaxf(t, __shfl_xor(t, o, 64));
    float u = s[r] * fast_exp2(m[r] - t);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) u += __shfl_xor(u, o, 64);
    if (lane == r) M = t, S = u;
  }
  if (lane >= R || row0 + lane >= nq) return;
  const float rho = sd.rho, damp = rho > 0.f ? 1.0f / (1.0f + eps / rho) : 1.0f;
  const float alpha = (step == 0 || step > entries) ? 1.0f : 0.5f;
  float f = alpha * (-eps * damp * kLn2 * small_log2(RAW ? small_sum(S, M) : fmaxf(S, 1e-40f), M));
  if (alpha != 1.0f) f += (1.0f - alpha) * old;
  if (damp < 1.0f) f -= alpha * (1.0f - damp) * norm;
  sd.out[at] = f;
  if (side == 0 && a.top != nullptr && step > entries) a.top[at] = M;
}

// Host side (fs_dense.hip).
void dense_plan(const SmallArgs& a, DenseArgs& t);
void dense_gemm_plan(DenseGemmArgs& g, bool may_split);
int dense_gemm(DenseGemmArgs& g, int items, hipStream_t st);
int dense_gemm_jobs(DenseGemmJobs& g, int jobs, int items, hipStream_t st, bool apart = true);
int dense_prepare(const SmallArgs& a, const DenseArgs& t, hipStream_t st);
int dense_step(const SmallArgs& a, DenseArgs& t, int step, hipStream_t st);
int dense_rows_step(const DenseRowArgs& t, int rows, bool raw, int sides, int items, hipStream_t st);

}  // namespace fs
