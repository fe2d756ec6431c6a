// Hessian-vector product of the cost in x on kept products.
//
// With P the plan, A the direction, F_ij = A_i.(x_i - y_j), cs the cost's scale:
//   r1 = 2 cs rowsum(P F),  r2 = 2 cs colsum(P F)
//   (denom - P^T diag_x^-1 P) z = r2 - P^T (r1 / diag_x)                   (conjugate gradients)
//   z1 = (r1 - P z) / diag_x
//   H A = s_i x_i + 2 cs rowsum(P)_i A_i + sum_j V_ij y_j,
//   s_i = (2 cs / eps)(rowsum(P)_i z1_i + (P z)_i) - lambda (2 / eps) r1_i,
//   V_ij = P_ij (-(2 cs / eps)(z1_i + z_j) + lambda (4 cs / eps) F_ij).
// So three contractions over the columns or the points carry everything: x.y, A.y and V.y (formed
// plan by plan it was two matrix products and four vector products for the right-hand side, one
// more product and the second-order term, each evaluating the plan anew: nine evaluations at
// about 500 us and five products at 1.1 ms more at 8192 x 8192 x 1536).  Everything else reads the two kept
// matrices once per pass and is bound by memory.
#pragma once

#include "fs_dense.hpp"

namespace fs {

struct HvpArgs {
  const void* x;
  const void* y;
  const float* A;
  const float* f;            // potentials with P_ij = exp((f_i + g_j - C_ij) / eps)
  const float* g;
  const float* log_a;        // weighted: ... of a_i b_j exp(..) instead, with the weights' logarithms (null: uniform ones)
  const float* log_b;
  float log_n, log_m;        // of uniform weights
  int weighted;
  const float* out_scale;    // the result is multiplied by it, or null
  float* out;
  int n, m, d, ld, dtype;
  float eps, cs, lambda, fac_x, fac_y, floor, ridge;
  float qs;                  // base-2 logit per unit of x.y
  const float* dots;         // [n][ld] x.y
  const float* prod;         // [n][ld] A.y
  const float* norm_x;       // cs |x|^2, cs |y|^2, cs |A|^2
  const float* norm_y;
  const float* norm_a;
  float* xa;                 // [n] x.A
  float* ra;                 // [n] base-2 potential minus norm
  float* cb;                 // [ld]
  float2* row_part;          // [chunks][n]: sums of P and of P F
  float2* col_part;          // [groups][m]
  int chunk, chunks, groups;
  float* mass;               // [n]
  float* r1;
  float* inv_diag;
  float* w;                  // [n] r1 / diag_x
  float* denom;              // [m]
  float* r2;
  float* strip_part;         // [strips][ld]
  int strip_rows, strips;
  float* vec;                // [m] the vector the strips multiply by
  float* alpha;              // [n] -(2 cs / eps) z1
  float* s;                  // [n]
  float* limits;             // largest |z|, largest |y|
  float* v_scale;            // [n] power-of-two scale of a row of V
  u32x4* vplanes;            // [n blocks][ld / 16][2][64]
  u32x4* yt;                 // [column blocks][ld / 16][2][64]
  int yt_blocks;
  const float2* scale;       // of x, y
  const float* prod_out;     // [splits][n][ldo]
  int ldo, splits;
  float* cg;                 // state (see fs_cg.hip)
  float* sol;
  float* res;
  float* a_dir;
};

// The preparation of x and y (where no solve has kept it: mats = 2, else 0) and of A, each of its two launches for all
// of them (a launch on a few blocks takes 3.5 to 4.5 us, whatever it does).
template <int T>
__global__ __launch_bounds__(1024) void hvp_stats_kernel(const SmallArgs pts, const SmallArgs dir, int mats) {
  if ((int)blockIdx.y < mats) dense_stats_of(pts, blockIdx.y, 0);
  else dense_stats_of(dir, 0, 0);
}
template <int T>
__global__ __launch_bounds__(512) void hvp_prep_kernel(const SmallArgs pts, const DenseArgs td, const SmallArgs dir,
                                                       const DenseArgs ta, int mats) {
  if ((int)blockIdx.y < mats) dense_prep_of(pts, td, blockIdx.y, 0);
  else dense_prep_of(dir, ta, 0, 0);
}

// Planes of y^T: the rows are y's columns.  A wavefront per 32 columns and 16 points.
struct TransposedArgs {
  const void* y;
  const float2* scale;  // of x, y
  u32x4* yt;            // [column blocks][ld / 16][2][64]
  int m, d, ld, dtype;
};
__device__ __forceinline__ void hvp_yt_of(const TransposedArgs& a, int blk, int kk) {
  const int lane = threadIdx.x & 63;
  if (kk >= a.ld / 16) return;
  const int col = blk * 32 + (lane & 31), j0 = 16 * kk + 8 * (lane >> 5);
  const float sc = a.scale[1].x;
  float v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    v[q] = col < a.d && j0 + q < a.m ? sc * small_load(a.y, (size_t)(j0 + q) * a.d + col, a.dtype) : 0.f;
  u32x4 hi, lo;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const _Float16 h0 = (_Float16)v[2 * q], h1 = (_Float16)v[2 * q + 1];
    hi[q] = pack_f16((float)h0, (float)h1);
    lo[q] = pack_f16(v[2 * q] - (float)h0, v[2 * q + 1] - (float)h1);
  }
  u32x4* out = a.yt + ((size_t)blk * (a.ld / 16) + kk) * kDenseStep + lane;
  out[0] = hi;
  out[64] = lo;
}
template <int T>
__global__ __launch_bounds__(256) void hvp_yt_kernel(const TransposedArgs a) {
  hvp_yt_of(a, blockIdx.y, blockIdx.x * 4 + (threadIdx.x >> 6));
}

// A potential in the convention of the product, from one that leaves the weight to the plan (no weight, or one below
// zero: a logarithm of -100,000).
__device__ __forceinline__ float hvp_potential(const HvpArgs& a, const float* pot, const float* log_w, float uniform, int i) {
#pragma clang fp contract(off)  // (the number that a caller would hand over otherwise)
  if (!a.weighted) return pot[i];
  const float l = log_w == nullptr ? uniform : log_w[i], t = a.eps * (l > -__builtin_inff() ? l : -100000.0f);
  return pot[i] + t;
}

// x_i.A_i and the base-2 biases: a wavefront per row, the rows of y behind those of x.  Behind them the planes of y^T,
// which the last product reads (by itself that launch took 5.4 us at 2,048 x 64).
template <int T>
__global__ __launch_bounds__(256) void hvp_rows_kernel(const HvpArgs a, const TransposedArgs t) {
  const int row_blocks = (a.n + a.ld + 3) / 4;
  if ((int)blockIdx.x >= row_blocks) {
    const int b = blockIdx.x - row_blocks, per = (t.ld / 16 + 3) / 4;
    hvp_yt_of(t, b / per, b % per * 4 + (threadIdx.x >> 6));
    return;
  }
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const float k = kLog2e / a.eps;
  if (row < a.n) {
    float s = 0.f;
    for (int c = lane; c < a.d; c += 64)
      s = __builtin_fmaf(small_load(a.x, (size_t)row * a.d + c, a.dtype), a.A[(size_t)row * a.d + c], s);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) {
      a.xa[row] = s;
      a.ra[row] = k * (hvp_potential(a, a.f, a.log_a, a.log_n, row) - a.norm_x[row]);
    }
  } else if (row - a.n < a.ld && lane == 0) {
    const int j = row - a.n;
    a.cb[j] = j < a.m ? k * (hvp_potential(a, a.g, a.log_b, a.log_m, j) - a.norm_y[j]) : kNegBig;
  }
}

// Sums of P and of P F along rows and columns, from one reading of both matrices: the shape of
// dense_sweep_kernel, without maxima (the plan's entries are what they are).
template <int WV>
__global__ __launch_bounds__(64 * WV, 4) void hvp_mass_kernel(const HvpArgs a) {
  constexpr int RW = 8;
  __shared__ float2 sh[2][WV][256];
  const int group = blockIdx.x, ch = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r0 = (group * WV + wave) * RW;
  const int mine = min(r0 + (lane & (RW - 1)), a.n - 1);
  const float rb = r0 + (lane & (RW - 1)) < a.n ? a.ra[mine] : kNegBig, xa = a.xa[mine];
  float rp[RW], rf[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) rp[r] = rf[r] = 0.f;
  const int c_end = min(a.ld, (ch + 1) * a.chunk);
  int buf = 0;
  for (int c0 = ch * a.chunk; c0 < c_end; c0 += 256, buf ^= 1) {
    float kb[4], cp[4], cf[4];
    *reinterpret_cast<float4*>(kb) = *reinterpret_cast<const float4*>(a.cb + c0 + 4 * lane);
#pragma unroll
    for (int k = 0; k < 4; ++k) cp[k] = cf[k] = 0.f;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const size_t at = (size_t)min(r0 + r, a.n - 1) * a.ld + c0 + 4 * lane;
      float v[4], e[4];
      *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(a.dots + at);
      *reinterpret_cast<float4*>(e) = *reinterpret_cast<const float4*>(a.prod + at);
      const float br = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, rb), r));
      const float xr = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, xa), r));
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float p = fast_exp2(__builtin_fmaf(v[k], a.qs, br + kb[k])), t = p * (xr - e[k]);
        rp[r] += p;
        rf[r] += t;
        cp[k] += p;
        cf[k] += t;
      }
      if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (four rows' loads at a time: registers)
    }
    float4* o = reinterpret_cast<float4*>(&sh[buf][wave][4 * lane]);
    o[0] = make_float4(cp[0], cf[0], cp[1], cf[1]);
    o[1] = make_float4(cp[2], cf[2], cp[3], cf[3]);
    __syncthreads();  // (the other buffer is free once everyone is here)
    for (int c = threadIdx.x; c < 256; c += 64 * WV) {
      float2 s = sh[buf][0][c];
#pragma unroll
      for (int w = 1; w < WV; ++w) s.x += sh[buf][w][c].x, s.y += sh[buf][w][c].y;
      if (c0 + c < a.m) a.col_part[(size_t)group * a.m + c0 + c] = s;
    }
  }
#pragma unroll
  for (int o = 32, n = RW / 2; n > 0; o >>= 1, n >>= 1) {
    const bool up = lane & o;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const float gp = up ? rp[r] : rp[r + n], gf = up ? rf[r] : rf[r + n];
      rp[r] = (up ? rp[r + n] : rp[r]) + __shfl_xor(gp, o, 64);
      rf[r] = (up ? rf[r + n] : rf[r]) + __shfl_xor(gf, o, 64);
    }
  }
#pragma unroll
  for (int o = 32 / RW; o > 0; o >>= 1) {
    rp[0] += __shfl_xor(rp[0], o, 64);
    rf[0] += __shfl_xor(rf[0], o, 64);
  }
  const int row = r0 + lane / (64 / RW);
  if (lane % (64 / RW) == 0 && row < a.n) a.row_part[(size_t)ch * a.n + row] = make_float2(rp[0], rf[0]);
}

// Diagonals and right-hand sides from those sums: 64 rows of one side per workgroup.
template <int T>
__global__ __launch_bounds__(256) void hvp_merge_kernel(const HvpArgs a) {
  const int side = blockIdx.y, rows = side ? a.m : a.n, parts = side ? a.groups : a.chunks;
  if ((int)blockIdx.x * 64 >= rows) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, row = blockIdx.x * 64 + lane;
  const float2* p = (side ? a.col_part : a.row_part) + min(row, rows - 1);
  float mass = 0.f, t = 0.f;
#pragma unroll 8
  for (int c = wave; c < parts; c += 4) {
    const float2 v = p[(size_t)c * rows];
    mass += v.x;
    t += v.y;
  }
  __shared__ float2 sh[4][64];
  sh[wave][lane] = make_float2(mass, t);
  __syncthreads();
  if (wave > 0 || row >= rows) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) mass += sh[w][lane].x, t += sh[w][lane].y;
  const float r = 2.0f * a.cs * t, diag = (side ? a.fac_y : a.fac_x) * fmaxf(mass, a.floor);
  if (side) {
    a.denom[row] = diag + a.ridge;
    a.r2[row] = r;
  } else {
    a.mass[row] = mass;
    a.r1[row] = r;
    a.inv_diag[row] = 1.0f / diag;
    a.w[row] = r / diag;
  }
}

// Largest |z| and |y_j|, for the scales of V's rows, by a workgroup of 512 threads.
__device__ __forceinline__ void hvp_limits(const HvpArgs& a) {
  float z = 0.f, y = 0.f;
  for (int j = threadIdx.x; j < a.m; j += 512) z = fmaxf(z, fabsf(a.sol[j])), y = fmaxf(y, a.norm_y[j]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) z = fmaxf(z, __shfl_xor(z, o, 64)), y = fmaxf(y, __shfl_xor(y, o, 64));
  __shared__ float sh[2][8];
  if ((threadIdx.x & 63) == 0) sh[0][threadIdx.x >> 6] = z, sh[1][threadIdx.x >> 6] = y;
  __syncthreads();
  if (threadIdx.x > 0) return;
  for (int w = 1; w < 8; ++w) z = fmaxf(z, sh[0][w]), y = fmaxf(y, sh[1][w]);
  a.limits[0] = z;
  a.limits[1] = sqrtf(y / a.cs);
}

// Whole rows of the plan in registers: a workgroup owns `strip_rows` rows, R at a time, its 512
// threads 4 CP columns each.  MODE 0: column sums of P_ij w_i; 1: the same with w = P vec / diag_x, so
// that one reading serves both products of a Schur-complement step; 2: P vec alone, and what the
// result needs of it; one workgroup more finds hvp_limits.  Bound by memory; the next R rows are in flight while the
// sums cross the workgroup.
template <int CP, int R, int MODE>
__global__ __launch_bounds__(512, 2) void hvp_strip_kernel(const HvpArgs a) {
  if (MODE == 1 && a.cg[4] != 0.f) return;  // converged: what was enqueued behind it does nothing
  if (MODE == 2 && (int)blockIdx.x == a.strips) return hvp_limits(a);
  __shared__ float sh[2][8][R];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int first = blockIdx.x * a.strip_rows, last = min(a.n, first + a.strip_rows);
  float4 cb[CP], v[CP], acc[CP], p[R][CP], next[R][CP];
  bool in[CP];
#pragma unroll
  for (int c = 0; c < CP; ++c) {
    const int col = 4 * (tid + 512 * c);
    in[c] = col < a.ld;
    cb[c] = in[c] ? *reinterpret_cast<const float4*>(a.cb + col) : make_float4(kNegBig, kNegBig, kNegBig, kNegBig);
    acc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    v[c] = acc[c];
    if (MODE > 0) {
      v[c].x = col < a.m ? a.vec[col] : 0.f;
      v[c].y = col + 1 < a.m ? a.vec[col + 1] : 0.f;
      v[c].z = col + 2 < a.m ? a.vec[col + 2] : 0.f;
      v[c].w = col + 3 < a.m ? a.vec[col + 3] : 0.f;
    }
  }
  auto load = [&](int i0) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CP; ++c)
        next[r][c] = *reinterpret_cast<const float4*>(a.dots + (size_t)min(i0 + r, a.n - 1) * a.ld + (in[c] ? 4 * (tid + 512 * c) : 0));
  };
  load(first);
  int buf = 0;
  for (int i0 = first; i0 < last; i0 += R, buf ^= 1) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CP; ++c) p[r][c] = next[r][c];
    if (i0 + R < last) load(i0 + R);
    float s[R], wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float b = i0 + r < last ? a.ra[i0 + r] : kNegBig;
      wr[r] = MODE == 0 ? (i0 + r < last ? a.w[i0 + r] : 0.f) : (MODE == 1 ? a.inv_diag[min(i0 + r, a.n - 1)] : 0.f);
      s[r] = 0.f;
#pragma unroll
      for (int c = 0; c < CP; ++c) {
        float4& q = p[r][c];
        q.x = fast_exp2(__builtin_fmaf(q.x, a.qs, b + cb[c].x));
        q.y = fast_exp2(__builtin_fmaf(q.y, a.qs, b + cb[c].y));
        q.z = fast_exp2(__builtin_fmaf(q.z, a.qs, b + cb[c].z));
        q.w = fast_exp2(__builtin_fmaf(q.w, a.qs, b + cb[c].w));
        if (MODE > 0) s[r] += (q.x * v[c].x + q.y * v[c].y) + (q.z * v[c].z + q.w * v[c].w);
      }
    }
    if (MODE > 0) {
      // over the wavefront: halves of the rows change places, then over the eight of them
#pragma unroll
      for (int o = 32, n = R / 2; n > 0; o >>= 1, n >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int r = 0; r < n; ++r) {
          const float g = up ? s[r] : s[r + n];
          s[r] = (up ? s[r + n] : s[r]) + __shfl_xor(g, o, 64);
        }
      }
#pragma unroll
      for (int o = 32 / R; o > 0; o >>= 1) s[0] += __shfl_xor(s[0], o, 64);
      if (lane % (64 / R) == 0) sh[buf][wave][lane / (64 / R)] = s[0];
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) t += sh[buf][w][r];
        s[r] = t;
        if (MODE == 1) wr[r] *= t;
      }
      if (MODE == 2 && tid < R && i0 + tid < last) {
        float pz = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) pz = tid == r ? s[r] : pz;
        const int i = i0 + tid;
        const float z1 = a.w[i] - pz * a.inv_diag[i], k = 2.0f * a.cs / a.eps;
        a.alpha[i] = -k * z1;
        a.s[i] = k * (a.mass[i] * z1 + pz) - a.lambda * (2.0f / a.eps) * a.r1[i];
      }
    }
    if (MODE < 2) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < CP; ++c) {
          acc[c].x = __builtin_fmaf(p[r][c].x, wr[r], acc[c].x);
          acc[c].y = __builtin_fmaf(p[r][c].y, wr[r], acc[c].y);
          acc[c].z = __builtin_fmaf(p[r][c].z, wr[r], acc[c].z);
          acc[c].w = __builtin_fmaf(p[r][c].w, wr[r], acc[c].w);
        }
    }
  }
  if (MODE < 2)
#pragma unroll
    for (int c = 0; c < CP; ++c)
      if (in[c]) *reinterpret_cast<float4*>(a.strip_part + (size_t)blockIdx.x * a.ld + 4 * (tid + 512 * c)) = acc[c];
}

// The strips' column sums: MODE 0 leaves r2 - sum in a_dir (the right-hand side), 1 the
// Schur-complement product denom vec - sum.
template <int MODE>
__global__ __launch_bounds__(256) void hvp_columns_kernel(const HvpArgs a) {
  if (MODE == 1 && a.cg[4] != 0.f) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = blockIdx.x * 64 + lane;
  float t = 0.f;
#pragma unroll 8
  for (int g = wave; g < a.strips; g += 4) t += a.strip_part[(size_t)g * a.ld + col];
  __shared__ float sh[4][64];
  sh[wave][lane] = t;
  __syncthreads();
  if (wave > 0 || col >= a.m) return;
  t = (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
  a.a_dir[col] = MODE == 0 ? a.r2[col] - t : __builtin_fmaf(a.denom[col], a.vec[col], -t);
}

// Power of two that takes a row of V below 2^15 (f16_plane_scale without its clamp at 2^40: the
// plan of a cloud with many points is small).
__device__ __forceinline__ float hvp_scale(float most) {
  const int e = (int)((__builtin_bit_cast(unsigned, most) >> 23) & 255u);
  if (e == 0 || e == 255) return 1.0f;
  return __builtin_bit_cast(float, (unsigned)max(1, min(253, 127 + 14 - (e - 127))) << 23);
}

// Planes of V, 32 rows x 256 columns per workgroup: read in rows of 1 KiB, turned into operand order in
// LDS (units of one plane, 16-column step and half-wave, 512 + 16 bytes apart so that the eight
// units that 64 lanes write at a time lie on different banks).  Bound by memory.
template <int T>
__global__ __launch_bounds__(256) void hvp_v_kernel(const HvpArgs a) {
  constexpr int UNIT = 528;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * 32 * UNIT];
  const int blk = blockIdx.x, c0 = blockIdx.y * 256;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const float k2 = 2.0f * a.cs / a.eps, k4 = a.lambda * 4.0f * a.cs / a.eps;
  const float zmax = a.limits[0], ymax = a.limits[1];
  float kb[4], z[4];
  *reinterpret_cast<float4*>(kb) = *reinterpret_cast<const float4*>(a.cb + c0 + 4 * lane);
#pragma unroll
  for (int k = 0; k < 4; ++k) z[k] = c0 + 4 * lane + k < a.m ? k2 * a.sol[c0 + 4 * lane + k] : 0.f;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int i = wave * 8 + r, row = blk * 32 + i, rc = min(row, a.n - 1);
    const size_t at = (size_t)rc * a.ld + c0 + 4 * lane;
    float v[4], e[4];
    *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(a.dots + at);
    *reinterpret_cast<float4*>(e) = *reinterpret_cast<const float4*>(a.prod + at);
    const float b = row < a.n ? a.ra[rc] : kNegBig, al = a.alpha[rc], xa = a.xa[rc];
    // |F_ij| <= |x_i.A_i| + |A_i| |y_j|, P_ij <= the row's sum
    const float most = a.mass[rc] * (fabsf(al) + k2 * zmax + fabsf(k4) * (fabsf(xa) + sqrtf(a.norm_a[rc] / a.cs) * ymax));
    const float sc = hvp_scale(most);
    if (c0 == 0 && lane == 0 && row < a.n) a.v_scale[row] = sc;
    _Float16 hi[4], lo[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float p = fast_exp2(__builtin_fmaf(v[k], a.qs, b + kb[k]));
      const float t = sc * p * (al - z[k] + k4 * (xa - e[k]));
      hi[k] = (_Float16)t;
      lo[k] = (_Float16)(t - (float)hi[k]);
    }
    // columns 4 lane .. 4 lane + 3: step lane / 4, half-wave lane / 2 % 2, half of its 16 bytes
    unsigned char* o = lds + (lane >> 1) * UNIT + i * 16 + (lane & 1) * 8;
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_f16((float)hi[0], (float)hi[1]), pack_f16((float)hi[2], (float)hi[3]));
    *reinterpret_cast<uint2*>(o + 32 * UNIT) =
        make_uint2(pack_f16((float)lo[0], (float)lo[1]), pack_f16((float)lo[2], (float)lo[3]));
  }
  __syncthreads();
  u32x4* out = a.vplanes + ((size_t)blk * (a.ld / 16) + c0 / 16) * kDenseStep;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int w = threadIdx.x + 256 * q;  // 16-byte word: [step][plane][half-wave][row]
    const int kk = w >> 7, plane = (w >> 6) & 1, half = (w >> 5) & 1, i = w & 31;
    out[w] = *reinterpret_cast<const u32x4*>(lds + (plane * 32 + kk * 2 + half) * UNIT + i * 16);
  }
}

// The gradient in x of a solve whose products are kept:
//   2 cs gs w_i (x_i - sum_j P_ij y_j / sum_j P_ij),  P_ij = 2^(qs x_i.y_j + c_j - M_i),
// c_j the biases of y before the extrapolation and M_i the largest logit of the row, which the extrapolation has
// formed of the same numbers by the same instruction: a row's largest P is one, whatever the sizes of its
// logits.  (Not from the potential that it left: with weak relaxations, damp << 1, that is the norm and next
// to nothing of the row's sum, and what is got back by dividing by damp is off by many powers of two.)
struct DenseGradArgs {
  const float* grad_out;
  float* out;
  u32x4* planes;             // of P, [n blocks][ld / 16][2][64]
  float* sums;               // [n][ld / 256] sums of a row's P over 256 columns
  const float* prod;         // [splits][n][ldo] P y
  int ldo, splits;
};
constexpr float kDenseGradScale = 4096.f;

// Planes of P, in the shape of hvp_v_kernel, and the sums of its rows.  Bound by memory: 8,192 x 8,192 in 116 us (4.6
// TB/s); the product behind it 520, the result 48, where forming the plan's products again took 1.65 ms.
template <int T>
__global__ __launch_bounds__(256) void dense_plan_kernel(const SmallArgs a, const DenseArgs t, const DenseGradArgs g) {
  constexpr int UNIT = 528;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * 32 * UNIT];
  const int blk = blockIdx.x, c0 = blockIdx.y * 256;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int last = a.lens[0] + 2;
  const float4 coef = small_last_coef(a, 0, 0);
  const float* y = a.pot[1] + (size_t)((last & 1) ^ 1) * t.m;      // before the extrapolation
  float kb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int col = c0 + 4 * lane + k, cc = min(col, t.m - 1);
    kb[k] = col < t.m ? fmaxf(__builtin_fmaf(coef.w, y[cc], a.l2w[1][cc]), kNegBig) : kNegBig;
  }
  float sum[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int i = wave * 8 + r, row = blk * 32 + i, rc = min(row, t.n - 1);
    float v[4];
    *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(t.dots + (size_t)rc * t.ld + c0 + 4 * lane);
    const float top = t.top[rc];
    _Float16 hi[4], lo[4];
    sum[r] = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float p = row < t.n ? kDenseGradScale * fast_exp2(__builtin_fmaf(v[k], coef.y, kb[k]) - top) : 0.f;
      sum[r] += p;
      hi[k] = (_Float16)p;
      lo[k] = (_Float16)(p - (float)hi[k]);
    }
    unsigned char* o = lds + (lane >> 1) * UNIT + i * 16 + (lane & 1) * 8;  // (as in hvp_v_kernel)
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_f16((float)hi[0], (float)hi[1]), pack_f16((float)hi[2], (float)hi[3]));
    *reinterpret_cast<uint2*>(o + 32 * UNIT) =
        make_uint2(pack_f16((float)lo[0], (float)lo[1]), pack_f16((float)lo[2], (float)lo[3]));
  }
  // the rows' sums over the lanes: halves of the rows change places, then what is left of each
#pragma unroll
  for (int o = 32, n = 4; n > 0; o >>= 1, n >>= 1) {
    const bool up = lane & o;
#pragma unroll
    for (int r = 0; r < n; ++r) sum[r] = (up ? sum[r + n] : sum[r]) + __shfl_xor(up ? sum[r] : sum[r + n], o, 64);
  }
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) sum[0] += __shfl_xor(sum[0], o, 64);
  const int mine = blk * 32 + wave * 8 + (lane >> 3);
  if ((lane & 7) == 0 && mine < t.n) g.sums[(size_t)mine * (t.ld / 256) + blockIdx.y] = sum[0];
  __syncthreads();
  u32x4* out = g.planes + ((size_t)blk * (t.ld / 16) + c0 / 16) * kDenseStep;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int w = threadIdx.x + 256 * q;
    const int kk = w >> 7, plane = (w >> 6) & 1, half = (w >> 5) & 1, i = w & 31;
    out[w] = *reinterpret_cast<const u32x4*>(lds + (plane * 32 + kk * 2 + half) * UNIT + i * 16);
  }
}

// Four columns of a row: by a 16-byte word where every row of floats starts at one, else element by element up to
// the d-th.
__device__ __forceinline__ bool hvp_wide(const void* p, int d, int dtype) { return dtype == 0 && small_wide(p, d, 0); }
__device__ __forceinline__ float4 hvp_load4(const void* p, size_t at, int dtype, bool wide, int left) {
  if (wide) return *reinterpret_cast<const float4*>(static_cast<const float*>(p) + at);
  float4 v = make_float4(small_load(p, at, dtype), 0.f, 0.f, 0.f);
  if (left > 1) v.y = small_load(p, at + 1, dtype);
  if (left > 2) v.z = small_load(p, at + 2, dtype);
  if (left > 3) v.w = small_load(p, at + 3, dtype);
  return v;
}
__device__ __forceinline__ void hvp_store4(float* p, size_t at, float4 v, bool wide, int left) {
  if (wide) {
    *reinterpret_cast<float4*>(p + at) = v;
    return;
  }
  p[at] = v.x;
  if (left > 1) p[at + 1] = v.y;
  if (left > 2) p[at + 2] = v.z;
  if (left > 3) p[at + 3] = v.w;
}
// The parts of a split contraction (their rows are padded to whole words).
__device__ __forceinline__ float4 hvp_parts(const float* p, size_t stride, int splits) {
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int k = 0; k < splits; ++k) {
    const float4 u = *reinterpret_cast<const float4*>(p + k * stride);
    v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
  }
  return v;
}

// A workgroup per row, a thread four columns.  Bound by memory: 8,192 x 1,536 in four parts (302 MB) 48 us, 6.2
// TB/s (by single columns, each thread adding up the row's sums by itself, 113).
template <int T>
__global__ __launch_bounds__(256) void dense_grad_kernel(const SmallArgs a, const DenseArgs t, const DenseGradArgs g) {
  const int row = blockIdx.x, lane = threadIdx.x & 63, parts = t.ld / 256;
  const bool wx = hvp_wide(a.pts[0], a.d, a.dtype), wo = hvp_wide(g.out, a.d, 0);
  float s = 0.f;
  for (int c = lane; c < parts; c += 64) s += g.sums[(size_t)row * parts + c];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  const float inv = a.scale[1].y / fmaxf(s, 1e-40f), coef = 2.0f * a.cost_scale * g.grad_out[0] * a.wt[0][row];
  for (int col = 4 * threadIdx.x; col < a.d; col += 1024) {
    const size_t e = (size_t)row * a.d + col;
    const float4 x = hvp_load4(a.pts[0], e, a.dtype, wx, a.d - col);
    const float4 v = hvp_parts(g.prod + (size_t)row * g.ldo + col, (size_t)t.n * g.ldo, g.splits);
    hvp_store4(g.out, e,
               make_float4(coef * (x.x - v.x * inv), coef * (x.y - v.y * inv), coef * (x.z - v.z * inv), coef * (x.w - v.w * inv)),
               wo, a.d - col);
  }
}

// The result, four columns at a time.  Bound by memory: 8,192 x 1,536 in four parts (352 MB) 62 us, 5.7
// TB/s (by single columns, with a 64-bit division each, 91).
template <int T>
__global__ __launch_bounds__(256) void hvp_result_kernel(const HvpArgs a) {
  const unsigned quads = (unsigned)(a.d + 3) / 4, count = (unsigned)a.n * quads;  // (at most 65,536 x 4,096)
  const bool wx = hvp_wide(a.x, a.d, a.dtype), wa = hvp_wide(a.A, a.d, 0), wo = hvp_wide(a.out, a.d, 0);
  const float gs = a.out_scale == nullptr ? 1.0f : *a.out_scale;
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
    const unsigned row = i / quads;
    const int col = 4 * (int)(i - row * quads), left = a.d - col;
    const size_t e = (size_t)row * a.d + col;
    const float4 x = hvp_load4(a.x, e, a.dtype, wx, left), A = hvp_load4(a.A, e, 0, wa, left);
    const float4 v = hvp_parts(a.prod_out + (size_t)row * a.ldo + col, (size_t)a.n * a.ldo, a.splits);
    const float k = a.scale[1].y / a.v_scale[row], s = a.s[row], w = 2.0f * a.cs * a.mass[row];
    hvp_store4(a.out, e,
               make_float4(gs * (s * x.x + w * A.x + v.x * k), gs * (s * x.y + w * A.y + v.y * k),
                           gs * (s * x.z + w * A.z + v.z * k), gs * (s * x.w + w * A.w + v.w * k)),
               wo, left);
  }
}

}  // namespace fs
