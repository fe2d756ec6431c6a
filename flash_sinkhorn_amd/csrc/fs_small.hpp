// Whole solves of small problems, one launch per step (d <= 128, fp16 planes).
//
// A small solve is bound by launches, not by arithmetic: at 2000 x 2000 x 3 a step of the xy
// problem and of the two self problems of a debiased loss is a few microseconds of work, and a
// launch costs about 3 us on the host and 2 us on the device whatever it does.  So this family
// spends one launch per step on ALL problems of a loss (the xy pair and the two self problems, for
// every item of a batch): a workgroup owns 32 query rows of one half-update and ALL their keys, its
// wavefronts share the keys, merge their soft-max statistics in LDS and run the epilogue, so
// nothing is left to a merge launch and nothing is written but the new potentials.  What used
// to be dozens of small launches around the steps (norms, log weights, bounding boxes, plane
// conversion, the eps schedule, the loss) is one statistics launch and one preparation launch in
// front and one launch behind.
//
// The planes are kept in MFMA operand order only (per 32 rows, plane and 16-column step one
// 1 KiB block with lane (h, row % 32)'s 16 bytes at 16 * (32 h + row % 32)): the same block
// serves as the stationary and as the streamed operand, a wavefront reads it with one fully
// coalesced load, and at these sizes every read hits the L2.
//
#pragma once

#include "fs_common.hpp"

namespace fs {

constexpr int kSmallStatBlocks = 64;            // most workgroups per matrix and item of small_stats_kernel
constexpr int kSmallMaxD = 128;
constexpr int kSmallTable = 512;                // most entries of an eps schedule kept on the device

// A run of small problems.  Sides: 0 f of the xy problem (rows of x against keys y), 1 g of it
// (rows of y against keys x), 2 the self problem of x, 3 that of y.  Problems: 0 xy, 1 xx, 2 yy.
struct SmallArgs {
  const void* pts[2];     // x [items, n, d], y [items, m, d]
  const float* w[2];      // weights [items, rows], null: uniform
  int dtype;              // 0 fp32, 1 fp16, 2 bf16
  int normalize;          // divide the weights by their sum
  int rows[2], blocks[2];  // rows of x and y, 32-row blocks of them
  int d, items;
  int self;               // 1: the self problems are solved as well, 2: only they are
  int want_values;        // value operands for small_grad_kernel are written
  float cost_scale;
  // eps schedule: 0 eps0 in every entry, 1 from the diameter of the clouds, 2 the table as given
  int sched, entries, cut, extrapolate;
  float eps0;
  double blur, scaling;
  float rho[2];           // <= 0: strict marginal
  // workspace
  // statistics of every matrix by stat_blocks workgroups, stat_words each: absmax; weights: sum, smallest,
  // largest; column minima, maxima (the first four, or the first two, where no more is needed)
  int stat_blocks, stat_words;
  float* stats;           // [items][2][stat_blocks][stat_words]
  float2* scale;          // [items][2] power-of-two scales of the planes, and their inverses
  u32x4* planes[2];       // [items][blocks][2 planes][DP / 16][64]
  u32x4* values[2];       // [items][blocks][DP / 32][2 steps][2 planes][64]
  float* norm[2];         // [items][rows] cost_scale * |row|^2
  float* wt[2];           // [items][rows] weights as the solve takes them
  float* l2w[2];          // [items][rows] their base-2 logarithms
  float* pot[4];          // [2 parities][items][rows of the side]: shifted potentials
  int table_len;          // entries a schedule can have and one more
  float4* table;          // [items][3][table_len] per entry: eps and what the kernels derive from
                          // it (small_coef); one entry past the last repeats it
  int* full;              // [items][3] entries of the schedules
  int* lens;              // [items][3] those the problem runs: fewer once it has converged
  int* host_words;        // pinned host memory, 4 words per item (see small_schedule, small_check_kernel)
  int host_token;
  int alternating;        // full steps, one side after the other, from the newest potentials
  // early stopping (threshold > 0): the potentials of the last check
  float threshold;
  float* prev[4];         // [items][rows of the side]
  // medium problems (fs_pair.hpp): their planes carry the square root of the logits' scale, a set
  // per problem where each has an eps of its own
  int pair;
  int pblocks[2];         // 32-row blocks of the planes of x and y, padding included
  u32x4* self_planes[2];
  float4* limits;
  float4* reach;
};

__device__ __forceinline__ float small_load(const void* p, size_t i, int dtype) {
  if (dtype == 0) return static_cast<const float*>(p)[i];
  if (dtype == 1) return (float)static_cast<const _Float16*>(p)[i];
  return __builtin_bit_cast(float, (unsigned)static_cast<const unsigned short*>(p)[i] << 16);
}

// Eight consecutive elements as floats; `wide`: by whole 16-byte words.
__device__ __forceinline__ void small_load8(float (&v)[8], const void* p, size_t at, int dtype, bool wide) {
  if (wide && dtype == 0) {
    const float4* q = reinterpret_cast<const float4*>(static_cast<const float*>(p) + at);
    const float4 u = q[0], w = q[1];
    v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w, v[4] = w.x, v[5] = w.y, v[6] = w.z, v[7] = w.w;
  } else if (wide) {
    const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const unsigned short*>(p) + at);
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const unsigned short b = (unsigned short)(w[k >> 1] >> (16 * (k & 1)));
      v[k] = dtype == 1 ? (float)__builtin_bit_cast(_Float16, b) : __builtin_bit_cast(float, (unsigned)b << 16);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = small_load(p, at + k, dtype);
  }
}
// Do rows of d elements start at multiples of 16 bytes?
__device__ __forceinline__ bool small_wide(const void* p, int d, int dtype) {
  return ((size_t)p & 15) == 0 && (d & (dtype == 0 ? 3 : 7)) == 0;
}

// What a step derives from its eps: eps, base-2 logit per unit of x.y, its inverse, base-2 units
// per unit of a potential.
__device__ __forceinline__ float4 small_coef(float cost_scale, float eps) {
  const float qs = 2.0f * cost_scale / eps * kLog2e;
  return make_float4(eps, qs, 1.0f / qs, kLog2e / eps);
}
__device__ __forceinline__ const float4* small_table(const SmallArgs& a, int item, int prob) {
  return a.table + ((size_t)item * 3 + prob) * a.table_len;
}
// The coefficients behind the cost and the gradient: those of the schedule's last entry (which a
// problem that stopped early keeps).
__device__ __forceinline__ float4 small_last_coef(const SmallArgs& a, int item, int prob) {
  const float4* t = small_table(a, item, prob);
  return t[a.sched == 0 ? 0 : a.full[item * 3 + prob] - 1];
}

// Partial statistics of a slice of one matrix of one item: largest magnitude (the plane scale),
// sum of the weights, and per column the smallest and largest value (the bounding box behind a
// schedule by diameter).  A thread stays on one column.  Bound by the loads in flight: NT
// threads a workgroup, 256 or 1,024 (kWideStats).
template <int NT>
__global__ __launch_bounds__(NT) void small_stats_kernel(const SmallArgs a) {
  const int mat = blockIdx.y, item = blockIdx.z, tid = threadIdx.x;
  const int rows = a.rows[mat], d = a.d;
  const int per = (rows + a.stat_blocks - 1) / a.stat_blocks;
  const int r0 = min(rows, (int)blockIdx.x * per), r1 = min(rows, r0 + per);
  const int reps = NT / d, act = reps * d;
  __shared__ float mn[NT], mx[NT];
  float lo = 3.0e38f, hi = -3.0e38f, ws = 0.f;
  bool nan = false;
  if (tid < act) {
    const size_t base = (size_t)item * rows * d;
#pragma unroll 8
    for (size_t e = (size_t)r0 * d + tid; e < (size_t)r1 * d; e += act) {
      const float v = small_load(a.pts[mat], base + e, a.dtype);
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
      nan = nan || !(v == v);
    }
  }
  float wl = 3.0e38f, wh = 0.f;
  if (a.w[mat] != nullptr)
    for (int r = r0 + tid; r < r1; r += NT) {
      const float w = a.w[mat][(size_t)item * rows + r];
      ws += w;
      wl = fminf(wl, w);
      wh = fmaxf(wh, w);
    }
  if (nan) lo = hi = __builtin_nanf("");
  mn[tid] = lo;
  mx[tid] = hi;
  for (int k = reps; k > 1;) {  // columns repeat every d threads: halve the number of repeats
    const int half = (k + 1) / 2;
    __syncthreads();
    if (tid < (k - half) * d) {
      const float l = mn[tid + half * d], u = mx[tid + half * d];
      mn[tid] = (l < mn[tid] || !(l == l)) ? l : mn[tid];
      mx[tid] = (u > mx[tid] || !(u == u)) ? u : mx[tid];
    }
    k = half;
  }
  __syncthreads();
  float* out = a.stats + (((size_t)item * 2 + mat) * a.stat_blocks + blockIdx.x) * a.stat_words;
  if (tid < d) {
    out[4 + tid] = mn[tid];
    out[4 + d + tid] = mx[tid];
  }
  __syncthreads();
  // (a NaN does not reach the plane scale: fmaxf drops it, as absmax_kernel does)
  float am = (r1 > r0 && tid < d) ? fmaxf(fabsf(mn[tid]), fabsf(mx[tid])) : 0.f;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    am = fmaxf(am, __shfl_xor(am, o, 64));
    ws += __shfl_xor(ws, o, 64);
    wl = fminf(wl, __shfl_xor(wl, o, 64));
    wh = fmaxf(wh, __shfl_xor(wh, o, 64));
  }
  __syncthreads();
  constexpr int NW = NT / 64;
  if ((tid & 63) == 0) {
    mn[tid >> 6] = am;
    mx[tid >> 6] = ws;
    mn[NW + (tid >> 6)] = wl;
    mx[NW + (tid >> 6)] = wh;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < NW; ++w) {
      am = fmaxf(am, mn[w]);
      ws += mx[w];
      wl = fminf(wl, mn[NW + w]);
      wh = fmaxf(wh, mx[NW + w]);
    }
    out[0] = am;
    out[1] = ws;
    out[2] = wl;
    out[3] = wh;
  }
}

// log2(v) + c for positive v: the exponent joins c before the fraction's logarithm does, so that one
// rounding is left where v is far from one or the two nearly cancel.
__device__ __forceinline__ float small_log2(float v, float c) {
  int e;
  float f = frexpf(v, &e);
  const bool low = f < 0.70710678f;
  f = low ? 2.0f * f : f;
  return ((float)(low ? e - 1 : e) + c) + __log2f(f);
}

// The schedules of one item from its bounding boxes (numpy's arange and exp in double, as the
// host builds it for larger problems): [D^2] + exp(2 ln D + i * 2 ln scaling) while above blur^2
// + [blur^2].  By one workgroup; diameters of the union, of x and of y.
__device__ void small_schedule(const SmallArgs& a, int item) {
  const int tid = threadIdx.x;
  __shared__ float sq[3];
  __shared__ int len[3], full[3];
  if (a.sched == 0 && tid < 3) {  // one entry stands for all
    a.lens[item * 3 + tid] = a.full[item * 3 + tid] = a.entries;
    a.table[((size_t)item * 3 + tid) * a.table_len] = small_coef(a.cost_scale, a.eps0);
  }
  if (a.sched != 1 && !a.pair) return;
  // The partial results, all on their way at once: of the boxes up to sixteen threads a column, whose minima and maxima
  // meet in LDS (a thread a column, sixteen blocks at a time, was eight round trips; with the logarithms below side by side and no
  // fence the kernel went from 9.4 to 8.2 us at 256 points, 16.0 to 10.1 at 4,567 and 20.5 to 14.4 at 30,011; it takes
  // 4.3 where there is no schedule).
  const int wave_lane = tid & 63;
  float4 part[2];
  if (a.pair && tid < 64) {
#pragma unroll
    for (int mat = 0; mat < 2; ++mat) {
      const float* st = a.stats + (((size_t)item * 2 + mat) * a.stat_blocks + (tid < a.stat_blocks ? tid : 0)) * a.stat_words;
      part[mat] = make_float4(st[0], st[1], st[2], st[3]);
    }
  }
  __shared__ float box[2][2][256];
  const int groups = min(16, 256 / a.d), group = tid / a.d, col = tid - group * a.d;
  if (tid < 3) sq[tid] = 0.f;
  if (group < groups) {
#pragma unroll
    for (int mat = 0; mat < 2; ++mat) {
      const float* st = a.stats + ((size_t)item * 2 + mat) * a.stat_blocks * a.stat_words + 4 + col;
      float lo = 3.0e38f, hi = -3.0e38f;
      for (int b0 = group; b0 < a.stat_blocks; b0 += 8 * groups) {  // (eight on their way, the last one again)
        float l[8], u[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float* at = st + (size_t)min(b0 + k * groups, a.stat_blocks - 1) * a.stat_words;
          l[k] = at[0];
          u[k] = at[a.d];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          lo = (l[k] < lo || !(l[k] == l[k])) ? l[k] : lo;
          hi = (u[k] > hi || !(u[k] == u[k])) ? u[k] : hi;
        }
      }
      box[mat][0][tid] = lo;
      box[mat][1][tid] = hi;
    }
  }
  __syncthreads();
  float r[3] = {0.f, 0.f, 0.f};
  if (tid < a.d) {
    float lo[2] = {3.0e38f, 3.0e38f}, hi[2] = {-3.0e38f, -3.0e38f};
#pragma unroll
    for (int mat = 0; mat < 2; ++mat)
#pragma unroll
      for (int g = 0; g < 16; ++g) {
        const int at = tid + min(g, groups - 1) * a.d;
        const float l = box[mat][0][at], u = box[mat][1][at];
        lo[mat] = (l < lo[mat] || !(l == l)) ? l : lo[mat];
        hi[mat] = (u > hi[mat] || !(u == u)) ? u : hi[mat];
      }
    const float e0 = (lo[0] < lo[1] || !(lo[0] == lo[0]) ? lo[0] : lo[1]);
    const float e1 = (hi[0] > hi[1] || !(hi[0] == hi[0]) ? hi[0] : hi[1]);
    r[0] = e1 - e0;
    r[1] = hi[0] - lo[0];
    r[2] = hi[1] - lo[1];
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    float s = r[p] * r[p];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0 && tid < 128) atomicAdd(&sq[p], s);
  }
  __syncthreads();
  if (a.pair && tid < 64) {
    float am = 0.f, mass = 1.f, lim[4];
#pragma unroll
    for (int mat = 0; mat < 2; ++mat) {
      const bool live = tid < a.stat_blocks;
      float m = part[mat].x, ws = live ? part[mat].y : 0.f, wl = part[mat].z, wh = part[mat].w;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        m = fmaxf(m, __shfl_xor(m, o, 64));
        ws += __shfl_xor(ws, o, 64);
        wl = fminf(wl, __shfl_xor(wl, o, 64));
        wh = fmaxf(wh, __shfl_xor(wh, o, 64));
      }
      am = fmaxf(am, m);
      if (a.w[mat] == nullptr) wl = wh = 1.0f / (float)a.rows[mat];
      else if (a.normalize) wl /= fmaxf(ws, 1e-40f), wh /= fmaxf(ws, 1e-40f);
      else mass = (ws > mass || !(ws == ws)) ? ws : mass;  // (NaN too, of either matrix)
      lim[2 * mat] = wl > 0.f ? small_log2(wl, 0.f) : -100000.0f * kLog2e;
      lim[2 * mat + 1] = wh > 0.f ? small_log2(wh, 0.f) : -100000.0f * kLog2e;
    }
    if (tid == 0) {
      a.limits[item] = make_float4(lim[0], lim[1], lim[2], lim[3]);
      // (the diagonal of the joint bounding box bounds every distance)
      const float far = a.cost_scale * sq[0];
      a.reach[item] = make_float4(am, far, 2.0f * (far + a.cost_scale * (float)a.d * am * am), small_log2(mass, 0.01f));
    }
  }
  if (a.sched != 1) return;
  __shared__ double from[3], per_step;
  if (tid < 64) {  // one logarithm a lane: of the diameters, of the end and of a step
    const double D = (double)sqrtf(sq[min(tid, 2)]);
    const double twice = 2.0 * log(wave_lane == 3 ? a.blur : (wave_lane == 4 ? a.scaling : D));
    const double stop = __shfl(twice, 3, 64), step = __shfl(twice, 4, 64);
    if (tid < 3) {
      int k = -2;                      // not a number
      if (D <= 0.0) k = -1;            // one point
      else if (D < 3.0e38) {
        const double cnt = ceil((stop - twice) / step);
        const double total = 2.0 + (cnt > 0.0 ? cnt : 0.0);
        k = total > (double)(kSmallTable - 1) ? -3 : (int)total;  // -3: longer than the table
        full[tid] = k;
        if (k > 0 && a.cut > 0) k = min(k, a.cut);
        if (k >= a.table_len) k = -3;
      }
      len[tid] = k;
      from[tid] = twice;
      if (tid == 0) per_step = step;
      a.lens[item * 3 + tid] = k;
      a.full[item * 3 + tid] = k;
    }
  }
  __syncthreads();
  // One store, so that nothing has to be ordered (a fence in front of the token writes back an L2): three lengths in
  // one word, ten bits each from -3 up, and the token in the next.
  if (tid == 0) {
    const unsigned lens = (unsigned)(len[0] + 3) | (unsigned)(len[1] + 3) << 10 | (unsigned)(len[2] + 3) << 20;
    int* words = a.host_words + item * 4 + 2;
    if ((reinterpret_cast<size_t>(words) & 7) == 0) {
      __hip_atomic_store(reinterpret_cast<unsigned long long*>(words), (unsigned long long)(unsigned)a.host_token << 32 | lens,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else {  // (words of a caller that are only aligned as such)
      __hip_atomic_store(words, (int)lens, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __threadfence_system();
      __hip_atomic_store(words + 1, a.host_token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  const int n0 = max(0, len[0] + (len[0] > 0)), n1 = max(0, len[1] + (len[1] > 0)), n2 = max(0, len[2] + (len[2] > 0));
  for (int k = tid; k < n0 + n1 + n2; k += 256) {  // (the entries of all three)
    const int p = k < n0 ? 0 : (k < n0 + n1 ? 1 : 2), i = k - (p == 0 ? 0 : (p == 1 ? n0 : n0 + n1));
    const double D = (double)sqrtf(sq[p]);
    const int c = min(i, len[p] - 1);
    const double e = c == 0 ? D * D : (c == full[p] - 1 ? a.blur * a.blur : exp(from[p] + (c - 1) * per_step));
    a.table[((size_t)item * 3 + p) * a.table_len + i] = small_coef(a.cost_scale, (float)e);
  }
}

// Largest magnitude of a matrix and the sum of its weights, by every lane of a wavefront.
__device__ __forceinline__ void small_merge_stats(const SmallArgs& a, int item, int mat, float& am, float& ws) {
  static_assert(kSmallStatBlocks == 64, "one partial result per lane");
  const int lane = threadIdx.x & 63;
  const bool live = lane < a.stat_blocks;
  const float* st = a.stats + (((size_t)item * 2 + mat) * a.stat_blocks + (live ? lane : 0)) * a.stat_words;
  am = st[0];
  ws = live ? st[1] : 0.f;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    am = fmaxf(am, __shfl_xor(am, o, 64));
    ws += __shfl_xor(ws, o, 64);
  }
}

// Everything the steps read, from one block of 32 rows: planes and (with want_values) value operands
// in MFMA order, cost_scale * |row|^2, base-2 log weights and the initial potentials.  The last
// workgroup column (x = blocks of the larger matrix) writes the schedules, and where `Kept` is not empty the
// arguments that later launches read from the workspace (a launch of its own for these made 487 us of
// 484.6 at 8,023 x 7,300 x 18).
struct SmallNothing {};
template <int DP, typename Kept>
__global__ __launch_bounds__(256) void small_prep_kernel(const SmallArgs a, const Kept kept, Kept* out) {
  constexpr int KK = DP / 16, NDB = (DP + 31) / 32, LDW = NDB * 32 + 1;
  const int mat = blockIdx.y, item = blockIdx.z, tid = threadIdx.x;
  if ((int)blockIdx.x == gridDim.x - 1) {
    if (mat == 0) {
      small_schedule(a, item);
    } else if constexpr (sizeof(Kept) >= sizeof(int)) {
      static_assert(sizeof(Kept) % sizeof(int) == 0, "whole words");
      if (item == 0)
        for (int i = tid; i < (int)(sizeof(Kept) / sizeof(int)); i += 256)
          reinterpret_cast<int*>(out)[i] = reinterpret_cast<const int*>(&kept)[i];
    }
    return;
  }
  const int rb = blockIdx.x, rows = a.rows[mat], d = a.d;
  if (rb >= a.blocks[mat]) return;
  __shared__ float s[32 * LDW];
  // (the points are on their way beside the statistics)
  const int r0 = rb * 32;
  const size_t base = ((size_t)item * rows + r0) * d;
  float point[DP / 8];
#pragma unroll
  for (int k = 0; k < DP / 8; ++k) {
    const int e = min(tid + 256 * k, (min(32, rows - r0) * d) - 1);
    point[k] = small_load(a.pts[mat], base + e, a.dtype);
  }
  float am, ws;
  small_merge_stats(a, item, mat, am, ws);
  const float sc = f16_plane_scale(am);
  if (rb == 0 && tid == 0) a.scale[item * 2 + mat] = make_float2(sc, 1.0f / sc);
  if (d < NDB * 32)
    for (int e = tid; e < 32 * LDW; e += 256) s[e] = 0.f;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < DP / 8; ++k) {
    const int e = tid + 256 * k, r = e / d;
    if (e < 32 * d) s[r * LDW + (e - r * d)] = r0 + r < rows ? sc * point[k] : 0.f;
  }
  __syncthreads();
  // planes
  u32x4* po = a.planes[mat] + ((size_t)item * a.blocks[mat] + rb) * (2 * KK * 64);
  for (int e = tid; e < KK * 64 && !a.pair; e += 256) {
    const int kk = e >> 6, lane = e & 63;
    const float* v = s + (lane & 31) * LDW + 16 * kk + 8 * (lane >> 5);
    u32x4 hi, lo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v0 = v[2 * q], v1 = v[2 * q + 1];
      const _Float16 h0 = (_Float16)v0, h1 = (_Float16)v1;
      hi[q] = pack_f16((float)h0, (float)h1);
      lo[q] = pack_f16(v0 - (float)h0, v1 - (float)h1);
    }
    po[kk * 64 + lane] = hi;
    po[(KK + kk) * 64 + lane] = lo;
  }
  if (a.want_values) {
    // lane (li, h), slot i of step t: key 16 t + (i < 4 ? 4 h + i : 4 + 4 h + i), the order in which
    // the accumulator of a logits tile holds the keys; column 32 cb + li
    u32x4* vo = a.values[mat] + ((size_t)item * a.blocks[mat] + rb) * (NDB * 2 * 2 * 64);
    for (int e = tid; e < NDB * 2 * 64; e += 256) {
      const int lane = e & 63, t = (e >> 6) & 1, cb = e >> 7;
      const int h = lane >> 5, col = 32 * cb + (lane & 31);
      u32x4 hi, lo;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int key = 16 * t + 4 * h + (q < 2 ? 2 * q : 4 + 2 * q);
        const float v0 = s[key * LDW + col], v1 = s[(key + 1) * LDW + col];
        const _Float16 h0 = (_Float16)v0, h1 = (_Float16)v1;
        hi[q] = pack_f16((float)h0, (float)h1);
        lo[q] = pack_f16(v0 - (float)h0, v1 - (float)h1);
      }
      vo[((cb * 2 + t) * 2 + 0) * 64 + lane] = hi;
      vo[((cb * 2 + t) * 2 + 1) * 64 + lane] = lo;
    }
  }
  // norms: eight threads a row
  {
    const int r = tid >> 3, c = tid & 7;
    float q = 0.f;
    for (int k = c; k < d; k += 8) q = __builtin_fmaf(s[r * LDW + k], s[r * LDW + k], q);
    q += __shfl_xor(q, 1, 64);
    q += __shfl_xor(q, 2, 64);
    q += __shfl_xor(q, 4, 64);
    const int row = r0 + r;
    if (c == 0 && row < rows) {
      const float inv = 1.0f / sc;
      const float al = a.cost_scale * (q * inv * inv);
      const size_t at = (size_t)item * rows + row;
      a.norm[mat][at] = al;
      float w = a.w[mat] == nullptr ? 1.0f / (float)rows : a.w[mat][at];
      if (a.w[mat] != nullptr && a.normalize) w = w / fmaxf(ws, 1e-40f);
      a.wt[mat][at] = w;
      a.l2w[mat][at] = w > 0.f ? small_log2(w, 0.f) : -100000.0f * kLog2e;
      a.pot[mat][at] = -al;
      if (a.self) a.pot[2 + mat][at] = -al;
    }
  }
}

__device__ __forceinline__ f32x16 small_mfma(const u32x4& x, const u32x4& y, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), c, 0,
                                                0, 0);
}

// Keys of one 32-key block: both planes, and potential and log weight of key li.
template <int KK>
struct SmallKeys {
  u32x4 p[2][KK];
  float pot, l2w;
};

// The keys a wavefront streams: everything that does not change from block to block.
template <int KK>
struct SmallStream {
  const u32x4* planes;
  const float* pot;
  const float* l2w;
  int nk, nkb, lane;
  float kc, raw, masked;  // base 2 per unit of a potential; accumulator units per base-2 unit; bias past the end

  // (past the last block: the last one again, for nobody)
  __device__ __forceinline__ void load(SmallKeys<KK>& k, int blk) const {
    const int b = min(blk, nkb - 1);
    const u32x4* at = planes + (size_t)b * (2 * KK * 64) + lane;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) k.p[p][kk] = at[(p * KK + kk) * 64];
    const int j = min(b * 32 + (lane & 31), nk - 1);
    k.pot = pot[j];
    k.l2w = l2w[j];
  }
  // A tile of logits in accumulator units: the three plane products from the lowest weight to
  // hi * hi, then the key bias by one fp32 MFMA.  Keys past the last one get a bias of -1e30 in
  // base 2 (where that can be held); half of it is where a row's maximum starts: above the masked
  // keys, whose exponentials are then zero (a wavefront may see nothing else), and below every
  // real logit.
  __device__ __forceinline__ f32x16 logits(const SmallKeys<KK>& k, const u32x4 (&q)[2][KK], int blk) const {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) acc = small_mfma(k.p[1][kk], q[0][kk], acc);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) acc = small_mfma(k.p[0][kk], q[1][kk], acc);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) acc = small_mfma(k.p[0][kk], q[0][kk], acc);
    float v = __builtin_fmaf(kc, k.pot, k.l2w) * raw;
    asm volatile("" : "+v"(v));  // (the loads stay ahead of the select below, which is not a branch)
    const float bias = (blk * 32 + (lane & 31) < nk) ? fmaxf(v, masked) : masked;
    const bool h = lane >= 32;
    return __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 0.f : bias, h ? 0.f : 1.0f, acc, 0, 0, 0);
  }
};

__device__ __forceinline__ float small_max16(float m, const f32x16& a) {
#pragma unroll
  for (int r = 0; r < 16; r += 2) m = fmaxf(fmaxf(m, a[r]), a[r + 1]);
  return m;
}

// A row's sum of exponentials, with its maximum in base 2.  In units of the products the rounding of that maximum is part of every
// exponential, which the logarithm of the sum takes out again; past 2^31 (clouds some 1e9 eps apart) it is 128 and more, and the sum
// zero, infinite or neither.  The largest key counts as one there: no number of keys weighs up against the rounding.
__device__ __forceinline__ float small_sum(float s, float m) {
  if (__builtin_amdgcn_classf(s, 0x267))  // (NaN, infinite, zero)
    if (fabsf(m) > 0x1p30f && fabsf(m) < 3.0e38f) s = 1.0f;
  return fmaxf(s, 1e-40f);
}

// What one step of one side needs, laid out so that a workgroup has it after one round of
// argument loads (pointers of item 0).
struct SmallStepSide {
  const u32x4* kplanes;
  const u32x4* qplanes;
  const float* kpot;   // potentials of the keys
  const float* kl2w;
  const float4* coef;  // of this step's entry; the items' are coef_stride apart
  const int* lens;     // the items' are 3 apart
  const float* old;    // this side's potentials, before ...
  float* out;          // ... and behind the step
  const float* norm;
  int nq, nk, nqb, nkb;
  float rho;
  int qm, km;          // which of the two matrices: query and key rows
};
struct SmallStepArgs {
  SmallStepSide side[4];
  const float4* scale;  // [items] scale of x, its inverse, scale of y, its inverse
  int step, extrapolate, coef_stride;
  int full;             // alternating: full steps, the whole shifted potential is damped
};

// One step of every problem.  Grid (32-row blocks of the larger cloud, sides, items).
// At these sizes the kernel is bound by the chain of memory round trips in front of its first
// logits and by the vector pipe behind it, so everything the first loads need comes from the
// kernel arguments, what the first logits need (coefficients, scales) arrives beside the keys,
// and the products of the next block run under the exponentials of the one before.
template <int DP, int W>
__global__ __launch_bounds__(64 * W) void small_step_kernel(const SmallStepArgs a) {
  constexpr int KK = DP / 16;
  const SmallStepSide& sd = a.side[blockIdx.y];
  const int rb = blockIdx.x, item = blockIdx.z;
  const int nq = sd.nq, nk = sd.nk, nkb = sd.nkb, qm = sd.qm, km = sd.km;
  if (rb >= sd.nqb) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;

  SmallStream<KK> ks;
  ks.planes = sd.kplanes + (size_t)item * nkb * (2 * KK * 64);
  ks.pot = sd.kpot + (size_t)item * nk;
  ks.l2w = sd.kl2w + (size_t)item * nk;
  ks.nk = nk;
  ks.nkb = nkb;
  ks.lane = lane;
  SmallKeys<KK> kr;
  ks.load(kr, wave);
  u32x4 q[2][KK];
  {
    const u32x4* b = sd.qplanes + ((size_t)item * sd.nqb + rb) * (2 * KK * 64) + lane;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) q[p][kk] = b[(p * KK + kk) * 64];
  }
  const int entries = sd.lens[item * 3];
  const float4 coef = sd.coef[(size_t)item * a.coef_stride];
  const float4 sc = a.scale[item];
  const float lscale = coef.y * (qm ? sc.w : sc.y) * (km ? sc.w : sc.y);
  ks.kc = coef.w;
  ks.raw = coef.z * (qm ? sc.z : sc.x) * (km ? sc.z : sc.x);
  ks.masked = fmaxf(kNegBig * ks.raw, -3.0e38f);

  float mr = 0.5f * ks.masked, m = mr * lscale, s = 0.f;  // the running maximum, raw and base 2
  const float no_max = m;
  auto soft = [&](const f32x16& acc) {
    mr = small_max16(mr, acc);
    float mn = mr * lscale;
    asm("" : "+v"(mn));  // (rounded once: an unchanged maximum has to give a factor of exactly one)
    s *= fast_exp2(m - mn);
    m = mn;
    float p0 = 0.f, p1 = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      p0 += fast_exp2(__builtin_fmaf(acc[r], lscale, -m));
      p1 += fast_exp2(__builtin_fmaf(acc[r + 1], lscale, -m));
    }
    s += p0 + p1;
  };
  if (wave < nkb) {
    f32x16 acc0 = ks.logits(kr, q, wave), acc1;
    ks.load(kr, wave + W);
    for (int blk = wave;; blk += 2 * W) {
      if (blk + W < nkb) {
        acc1 = ks.logits(kr, q, blk + W);
        ks.load(kr, blk + 2 * W);
      }
      soft(acc0);
      if (blk + W >= nkb) break;
      if (blk + 2 * W < nkb) {
        acc0 = ks.logits(kr, q, blk + 2 * W);
        ks.load(kr, blk + 3 * W);
      }
      soft(acc1);
      if (blk + 2 * W >= nkb) break;
    }
  }
  // ---- the row's statistics over the wavefronts and half-waves ----
  __shared__ float2 sh[W][64];
  sh[wave][lane] = make_float2(m, s);
  const int row = rb * 32 + tid, step = a.step;
  const size_t at = (size_t)item * nq + min(row, nq - 1);
  const float old = sd.old[at], shift = sd.norm[at];
  __syncthreads();
  if (tid >= 32 || row >= nq || step > entries + a.extrapolate) return;  // (its schedule is shorter)
  float M = no_max, S = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) M = fmaxf(M, fmaxf(sh[w][tid].x, sh[w][tid + 32].x));
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float2 u = sh[w][tid], v = sh[w][tid + 32];
    S += u.y * fast_exp2(u.x - M) + v.y * fast_exp2(v.x - M);
  }
  const float eps = coef.x, rho = sd.rho;
  const float damp = rho > 0.f ? 1.0f / (1.0f + eps / rho) : 1.0f;
  const float alpha = (a.full || step == 0 || step > entries) ? 1.0f : 0.5f;
  float r = alpha * (-eps * damp * kLn2 * small_log2(small_sum(S, M), M));
  if (alpha != 1.0f) r += (1.0f - alpha) * old;
  if (damp < 1.0f && !a.full) r -= alpha * (1.0f - damp) * shift;
  sd.out[at] = r;
}

// Convergence check behind averaged step `step` (the check_every-th since the last check): a
// problem none of whose potentials has moved by the threshold since then runs no further entries
// (its extrapolation, if any, is the next step); the others' potentials are kept for the next
// check.  The first check only keeps them.  One workgroup per item and problem; it leaves
// 2 * check + converged in the problem's host word.
template <int T>
__global__ __launch_bounds__(1024) void small_check_kernel(const SmallArgs a, int step, int check) {
  const int prob = blockIdx.x + (a.self == 2 ? 1 : 0), item = blockIdx.y, tid = threadIdx.x;
  if (a.lens[item * 3 + prob] < step) return;  // stopped before, or a shorter schedule
  const int newest = a.alternating ? step & 1 : (step & 1) ^ 1;
  const int s0 = prob == 0 ? 0 : 1 + prob, s1 = prob == 0 ? 1 : s0;
  float change = 0.f;
  for (int side = s0; side <= s1; ++side) {
    const int rows = a.rows[side & 1];
    const float* now = a.pot[side] + ((size_t)newest * a.items + item) * rows;
    float* prev = a.prev[side] + (size_t)item * rows;
    for (int i = tid; i < rows; i += 1024) {
      // (alternating: the first check compares with the initial potentials)
      const float before = a.alternating && check == 0 ? -a.norm[side & 1][(size_t)item * rows + i] : prev[i];
      const float d = fabsf(now[i] - before);
      change = d > change || !(d == d) ? d : change;
    }
  }
  __shared__ float sh[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float d = __shfl_xor(change, o, 64);
    change = d > change || !(d == d) ? d : change;
  }
  if ((tid & 63) == 0) sh[tid >> 6] = change;
  __syncthreads();
  bool stop = check > 0 || a.alternating;
  for (int w = 0; w < 16; ++w) stop = stop && sh[w] < a.threshold;
  if (!stop)
    for (int side = s0; side <= s1; ++side) {
      const int rows = a.rows[side & 1];
      const float* now = a.pot[side] + ((size_t)newest * a.items + item) * rows;
      float* prev = a.prev[side] + (size_t)item * rows;
      for (int i = tid; i < rows; i += 1024) prev[i] = now[i];
    }
  if (tid == 0) {
    if (stop) {
      a.lens[item * 3 + prob] = step;
      // (the extrapolation, next, takes the schedule's last eps)
      if (a.sched != 0)
        a.table[((size_t)item * 3 + prob) * a.table_len + step] = small_last_coef(a, item, prob);
    }
    __hip_atomic_store(a.host_words + item * 4 + prob, 2 * check + (stop ? 1 : 0), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// The loss of every item, and the standard potentials (of the last step, and of the one before
// when there was an extrapolation) of every side.  Grid (parts, items): a part takes every
// parts-th run of 1024 rows; several parts leave their sums to small_loss_sum_kernel.
// pots: per side and kind (0: of the cost, 1: of the gradient) [items][rows], in that order.
struct SmallLossArgs {
  float* loss;        // [items] or null
  float* parts;       // [items][parts], where there are several
  float* pots;        // or null
  int relaxed;        // both marginals relaxed: the other cost formula
};

template <int T>
__global__ __launch_bounds__(1024) void small_loss_kernel(const SmallArgs a, const SmallLossArgs l) {
  const int item = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
  float total = 0.f;
  size_t off = a.self == 2 ? 2 * (size_t)a.items * (a.rows[0] + a.rows[1]) : 0;
  const int first = a.self == 2 ? 2 : 0, sides = a.self ? 4 : 2;
  // What a thread's first row of every side needs is loaded before the first sum, both potentials for the one that the
  // schedule's length names (each side a chain of its own: 7.5 us at 2,000 points debiased, now 4.8).
  struct Row {
    float norm, weight, pot[2];
  };
  auto load = [&](int side, int i) {
    const int mat = side & 1, rows = a.rows[mat];
    const size_t half = (size_t)a.items * rows, at = (size_t)item * rows + min(i, rows - 1);
    return Row{a.norm[mat][at], a.wt[mat][at], {a.pot[side][at], a.pot[side][half + at]}};
  };
  Row row[4];
  int lens[4];
  float eps_last[4];
  const int i0 = part * 1024 + tid;
#pragma unroll
  for (int side = 0; side < 4; ++side)
    if (side >= first && side < sides) {
      const int prob = side < 2 ? 0 : side - 1;
      row[side] = load(side, i0);
      lens[side] = a.lens[item * 3 + prob];
      eps_last[side] = l.relaxed ? small_last_coef(a, item, prob).x : 0.f;
    }
#pragma unroll
  for (int side = 0; side < 4; ++side) {
    if (side < first || side >= sides) continue;
    const int mat = side & 1, rows = a.rows[mat];
    const int last = (lens[side] + 1 + a.extrapolate) & 1;
    const size_t half = (size_t)a.items * rows;
    const float rho = a.rho[mat];
    // (a self problem has this potential twice: its cost is 2 <a, f>)
    const float sign = side < 2 ? 1.0f : -1.0f;
    float sum = 0.f;
    Row v = row[side];
    for (int i = i0; i < rows;) {
      const size_t at = (size_t)item * rows + i;
      const float f = (last ? v.pot[1] : v.pot[0]) + v.norm;
      if (l.pots != nullptr) {
        l.pots[off + at] = f;
        l.pots[off + half + at] = a.extrapolate ? (last ? v.pot[0] : v.pot[1]) + v.norm : f;
      }
      sum += v.weight * (l.relaxed ? 1.0f - expf(-f / rho) : f);
      i += 1024 * gridDim.x;
      if (i < rows) v = load(side, i);
    }
    if (l.relaxed) sum *= rho + 0.5f * eps_last[side];
    total += sign * sum;
    off += 2 * half;
  }
  if (l.loss == nullptr) return;
  __shared__ float sh[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o, 64);
  if ((tid & 63) == 0) sh[tid >> 6] = total;
  __syncthreads();
  if (tid == 0) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += sh[w];
    if (gridDim.x == 1) l.loss[item] = t;
    else l.parts[(size_t)item * gridDim.x + part] = t;
  }
}

// The standard potentials alone, every side and kind into memory of its own (a program that keeps or
// changes one of them does not hold or touch the others).  Grid (1024-row pieces, sides, items).
struct SmallPotArgs {
  float* pots[4][2];  // [side][of the cost, of the gradient]: [items][rows] or null
};

template <int T>
__global__ __launch_bounds__(1024) void small_potentials_kernel(const SmallArgs a, const SmallPotArgs p) {
  const int side = blockIdx.y + (a.self == 2 ? 2 : 0), item = blockIdx.z, mat = side & 1, rows = a.rows[mat];
  const int i = blockIdx.x * 1024 + threadIdx.x;
  if (i >= rows) return;
  const int last = a.lens[item * 3 + (side < 2 ? 0 : side - 1)] + 1 + a.extrapolate;
  const size_t half = (size_t)a.items * rows, at = (size_t)item * rows + i;
  const float al = a.norm[mat][at];
  if (p.pots[side][0] != nullptr) p.pots[side][0][at] = a.pot[side][(last & 1) * half + at] + al;
  if (p.pots[side][1] != nullptr)
    p.pots[side][1][at] = a.pot[side][(a.extrapolate ? (last & 1) ^ 1 : last & 1) * half + at] + al;
}

template <int T>
__global__ __launch_bounds__(64) void small_loss_sum_kernel(const SmallLossArgs l, int parts) {
  float t = 0.f;
  for (int i = threadIdx.x; i < parts; i += 64) t += l.parts[(size_t)blockIdx.x * parts + i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if (threadIdx.x == 0) l.loss[blockIdx.x] = t;
}

// Gradients of the loss in x and y at the potentials before the extrapolation.  A workgroup owns
// 32 rows; with self problems it sweeps the keys of the other cloud, then its own cloud's, and
// takes the difference of the two barycentres:
//   xy alone   2 cs gs w_i (q_i - T_i),      with the self terms   2 cs gs w_i (T'_i - T_i).
struct SmallGradArgs {
  const float* grad_out;  // [items]
  float* out[2];          // [items, rows, d] or null
};

// The key blocks that matter to a block of query rows, where the solve has kept that (fs_pair.hpp).
struct SmallAllBlocks {
  static constexpr int kMost = 1;
  __device__ __forceinline__ int find(int, int, int, int, int, unsigned short*) const { return -1; }
};

template <int DP, typename Lists>
__global__ __launch_bounds__(512, 2) void small_grad_kernel(const SmallArgs a, const SmallGradArgs g, const Lists lists) {
  constexpr int KK = DP / 16, NDB = (DP + 31) / 32, W = 8;
  constexpr int LDW = NDB * 32 + 4;                 // padded row of a wavefront's partial output
  constexpr int PER = NDB * 32 * 32 / 512;          // outputs per thread
  __shared__ __attribute__((aligned(16))) float sh_o[W][32 * LDW];
  __shared__ float2 sh_ms[W][32];
  __shared__ unsigned short sh_blocks[Lists::kMost];
  const int rb = blockIdx.x, item = blockIdx.z, tid = threadIdx.x;
  const int qm = g.out[0] == nullptr ? 1 : blockIdx.y;
  if (rb >= a.blocks[qm]) return;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, h = lane >> 5;
  const int nq = a.rows[qm], d = a.d;
  u32x4 q[2][KK];
  float bary[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) bary[i] = 0.f;

  // (what either pass starts from is on its way before the first one)
  const int len0 = a.lens[item * 3], len1 = a.self ? a.lens[item * 3 + 1 + qm] : 0;
  const float4 coef0 = small_last_coef(a, item, 0), coef1 = a.self ? small_last_coef(a, item, 1 + qm) : coef0;
  const float2 sq = a.scale[item * 2 + qm], other = a.scale[item * 2 + (qm ^ 1)];
  for (int pass = 0; pass <= a.self; ++pass) {
    const int km = pass == 0 ? qm ^ 1 : qm;
    const int kside = pass == 0 ? km : 2 + km;
    const int prob = pass == 0 ? 0 : 1 + km;
    const int nk = a.rows[km], nkb = a.blocks[km];
    const int last = (pass == 0 ? len0 : len1) + 1;  // (the step before the extrapolation)
    const float4 coef = pass == 0 ? coef0 : coef1;
    const float2 sk = pass == 0 ? other : sq;
    const u32x4* qp = pass == 0 || a.self_planes[qm] == nullptr ? a.planes[qm] : a.self_planes[qm];
    const u32x4* kp = pass == 0 || a.self_planes[km] == nullptr ? a.planes[km] : a.self_planes[km];
    if (pass == 0 || qp != a.planes[qm]) {
      const u32x4* b = qp + ((size_t)item * a.pblocks[qm] + rb) * (2 * KK * 64) + lane;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) q[p][kk] = b[(p * KK + kk) * 64];
    }
    float lscale = coef.y * sq.y * sk.y, raw = coef.z * sq.x * sk.x;
    if (a.pair) {  // (see pair_scale)
      const float most = a.reach[item].x, ps = f16_plane_scale(most);
      const bool root = most * sqrtf(coef.y) < 30000.f;
      lscale = root ? 1.0f : coef.y / (ps * ps);
      raw = root ? 1.0f : coef.z * (ps * ps);
    }
    SmallStream<KK> ks;
    ks.planes = kp + (size_t)item * a.pblocks[km] * (2 * KK * 64);
    ks.pot = a.pot[kside] + ((size_t)(last & 1) * a.items + item) * nk;
    ks.l2w = a.l2w[km] + (size_t)item * nk;
    ks.nk = nk;
    ks.nkb = nkb;
    ks.lane = lane;
    ks.kc = coef.w;
    ks.raw = raw;
    ks.masked = fmaxf(kNegBig * ks.raw, -3.0e38f);
    const float no_max = 0.5f * ks.masked * lscale;
    const u32x4* vp = a.values[km] + (size_t)item * nkb * (NDB * 4 * 64) + lane;

    float m = no_max, s = 0.f;
    f32x16 o[NDB];
#pragma unroll
    for (int cb = 0; cb < NDB; ++cb)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[cb][r] = 0.f;
    const int found = lists.find(item, prob, qm, rb, nkb, sh_blocks);  // (with barriers, or -1: all of them)
    const int count = found < 0 ? nkb : found;
    auto block_at = [&](int i) { return found < 0 ? i : (int)sh_blocks[min(i, count - 1)]; };
    SmallKeys<KK> kr;
    if (wave < count) ks.load(kr, block_at(wave));
    for (int i = wave; i < count; i += W) {
      const int blk = __builtin_amdgcn_readfirstlane(block_at(i));
      const u32x4* v = vp + (size_t)blk * (NDB * 4 * 64);
      const f32x16 acc = ks.logits(kr, q, blk);
      if (i + W < count) ks.load(kr, block_at(i + W));
      // the two half-waves of a column feed one sum: they share its maximum
      float mx = small_max16(ks.masked, acc) * lscale;
      mx = fmaxf(mx, xor32(mx));
      if (wave_any(mx > m)) {
        const float mn = fmaxf(m, mx);
        const float f = fast_exp2(m - mn);
        m = mn;
        s *= f;
#pragma unroll
        for (int cb = 0; cb < NDB; ++cb)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[cb][r] *= f;
      }
      // probabilities times 2^11, as two fp16 planes in the order of the value operands' keys
      const float one = opaque_one();
      u32x4 ph[2], pl[2];
      float ps = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int r = 8 * t + 2 * c;
          const float e0 = fast_exp2(__builtin_fmaf(acc[r], lscale, 11.0f - m));
          const float e1 = fast_exp2(__builtin_fmaf(acc[r + 1], lscale, 11.0f - m));
          ps += e0 + e1;
          const unsigned both = pack_f16(e0, e1);
          const f16x2 hi = __builtin_bit_cast(f16x2, both);
          ph[t][c] = both;
          pl[t][c] = pack_f16(f16_rest(e0, hi[0], one), f16_rest(e1, hi[1], one));
        }
      s += ps;
#pragma unroll
      for (int cb = 0; cb < NDB; ++cb) {
        u32x4 vh[2], vl[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          vh[t] = v[((cb * 2 + t) * 2 + 0) * 64];
          vl[t] = v[((cb * 2 + t) * 2 + 1) * 64];
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) o[cb] = small_mfma(vl[t], ph[t], o[cb]);
#pragma unroll
        for (int t = 0; t < 2; ++t) o[cb] = small_mfma(vh[t], pl[t], o[cb]);
#pragma unroll
        for (int t = 0; t < 2; ++t) o[cb] = small_mfma(vh[t], ph[t], o[cb]);
      }
    }
    s += xor32(s);
    // ---- the wavefronts' sums under a common maximum ----
    if (h == 0) sh_ms[wave][li] = make_float2(m, s);
    __syncthreads();
    float M = no_max;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, sh_ms[w][li].x);
    const float fac = fast_exp2(m - M);
#pragma unroll
    for (int cb = 0; cb < NDB; ++cb)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<float4*>(&sh_o[wave][li * LDW + 32 * cb + 8 * c + 4 * h]) =
            make_float4(o[cb][4 * c] * fac, o[cb][4 * c + 1] * fac, o[cb][4 * c + 2] * fac, o[cb][4 * c + 3] * fac);
    __syncthreads();
    const float inv_v = sk.y;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 512 * i, row = e / (NDB * 32), col = e % (NDB * 32);
      float mm = no_max, sum = 0.f, O = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) mm = fmaxf(mm, sh_ms[w][row].x);
#pragma unroll
      for (int w = 0; w < W; ++w) {
        sum += sh_ms[w][row].y * fast_exp2(sh_ms[w][row].x - mm);
        O += sh_o[w][row * LDW + col];
      }
      const float t = O * inv_v / fmaxf(sum, 1e-40f);  // (2^11 is in both)
      bary[i] = pass == 0 ? t : t - bary[i];
    }
    __syncthreads();  // the next pass writes the same buffers
  }

  const float coef = 2.0f * a.cost_scale * g.grad_out[item];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = tid + 512 * i, col = e % (NDB * 32), row = rb * 32 + e / (NDB * 32);
    if (row < nq && col < d) {
      const size_t r = (size_t)item * nq + row;
      const float diff = a.self ? bary[i] : small_load(a.pts[qm], r * d + col, a.dtype) - bary[i];
      g.out[qm][r * d + col] = coef * a.wt[qm][r] * diff;
    }
  }
}

}  // namespace fs
