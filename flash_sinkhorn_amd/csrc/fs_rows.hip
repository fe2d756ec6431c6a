// What a solve of the general path starts from and looks at between its steps, a launch each.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "flash_sinkhorn_hip.h"

namespace fs {
namespace {

struct RowStart {
  const float* pts[2];
  const float* w[2];     // weights, null: no logarithms
  const float* less[2];  // taken off the norms, null: nothing
  float *norm[2], *logw[2], *pot[2];
  int rows[2], blocks0, d, wide;
  float cost_scale;
};

// cost_scale |row|^2, its negative (the potential that a solve starts from) and the logarithm of a row's weight, of both
// clouds.  Sixteen lanes a row, sixteen rows a workgroup.  Bound by reading the points.  As operations of their own products, sums,
// logarithms and selections were fourteen launches of 65 us together at 50,000 rows of 128 columns, and the host took longer
// than they did: ten alternating iterations with this and change_kernel 3,998 -> 3,850 us, of 7,000 x 7,500 x 100 1,435 ->
// 1,305, of 15,000 x 14,000 x 8 1,300 -> 1,163.  Norms and biases of a c-transform were seven: 2,716 x 2,506 x 35 77 -> 46 us,
// 20,000 x 15,000 x 8 105 -> 87, 48,000 x 48,000 x 100 1,591 -> 1,548.
constexpr int kRowsOfBlock = 16;
__global__ __launch_bounds__(256) void row_start_kernel(const RowStart a) {
  const int mat = (int)blockIdx.x >= a.blocks0 ? 1 : 0, tid = threadIdx.x, lane = tid & 15;
  const int row = ((int)blockIdx.x - (mat ? a.blocks0 : 0)) * kRowsOfBlock + (tid >> 4), rows = a.rows[mat], d = a.d;
  const float* p = a.pts[mat] + (size_t)min(row, rows - 1) * d;
  const float w = a.w[mat] != nullptr ? a.w[mat][min(row, rows - 1)] : 0.f;
  const float less = a.less[mat] != nullptr ? a.less[mat][min(row, rows - 1)] : 0.f;
  float s = 0.f;
  if (a.wide) {
#pragma unroll 4
    for (int c = 4 * lane; c < d; c += 64) {
      const float4 v = *reinterpret_cast<const float4*>(p + c);
      s = __builtin_fmaf(v.x, v.x, __builtin_fmaf(v.y, v.y, __builtin_fmaf(v.z, v.z, __builtin_fmaf(v.w, v.w, s))));
    }
  } else {
#pragma unroll 4
    for (int c = lane; c < d; c += 16) s = __builtin_fmaf(p[c], p[c], s);
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane > 0 || row >= rows) return;
  s *= a.cost_scale;
  a.norm[mat][row] = s - less;
  if (a.w[mat] == nullptr) return;
  a.pot[mat][row] = -s;
  a.logw[mat][row] = w > 0.f ? logf(w) : -100000.0f;
}

// out[i]: the largest |now[i] - before[i]| (not a number where one of the differences is none).  A workgroup each: mostly its launch.
struct Change {
  const float *now[2], *before[2];
  int rows[2];
  float* out;
};
__global__ __launch_bounds__(1024) void change_kernel(const Change a) {
  const int i = blockIdx.x, tid = threadIdx.x, rows = a.rows[i];
  unsigned most = 0;  // (of numbers without a sign, and of what is none behind them)
#pragma unroll 8
  for (int r = tid; r < rows; r += 1024) {
    const float v = a.now[i][r] - a.before[i][r];
    most = max(most, __builtin_bit_cast(unsigned, v) & 0x7fffffffu);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, o, 64));
  __shared__ unsigned sh[16];
  if ((tid & 63) == 0) sh[tid >> 6] = most;
  __syncthreads();
  if (tid > 0) return;
#pragma unroll
  for (int w = 1; w < 16; ++w) most = max(most, sh[w]);
  a.out[i] = __builtin_bit_cast(float, most);
}

// The diagonal of the joint bounding box of two clouds: per column the smallest and largest value of a run of rows, from 64
// workgroups a cloud, then one workgroup over all of them.  What is not a number stays.  10,500 and 7,532 rows of 90 12 us, where
// reductions down the columns of a row-major matrix, one each, took 80 in eleven launches.
struct Box {
  const float* pts[2];
  int rows[2], d, blocks;
  float* part;  // [clouds * blocks][2][d]
  int parts;
};
constexpr int kBoxBlocks = 64, kBoxThreads = 512;
__device__ __forceinline__ float box_low(float a, float b) { return (b < a || !(b == b)) ? b : a; }
__device__ __forceinline__ float box_high(float a, float b) { return (b > a || !(b == b)) ? b : a; }

__global__ __launch_bounds__(kBoxThreads) void box_kernel(const Box a) {
  const int mat = blockIdx.y, tid = threadIdx.x, rows = a.rows[mat], d = a.d;
  const int per = (rows + a.blocks - 1) / a.blocks, r0 = min(rows, (int)blockIdx.x * per), r1 = min(rows, r0 + per);
  float* out = a.part + ((size_t)mat * a.blocks + blockIdx.x) * 2 * d;
  const float* p = a.pts[mat];
  const int reps = max(1, kBoxThreads / d), step = d <= kBoxThreads ? reps : 1;
  __shared__ float sh[2][kBoxThreads];
  for (int c0 = 0; c0 < d; c0 += kBoxThreads) {  // (once, but for rows of more columns than threads)
    const int col = d <= kBoxThreads ? tid % d : c0 + tid, rep = d <= kBoxThreads ? tid / d : 0;
    const bool live = col < d && rep < reps;
    float lo = __builtin_inff(), hi = -lo;
    if (live)
#pragma unroll 8
      for (int r = r0 + rep; r < r1; r += step) {
        const float v = p[(size_t)r * d + col];
        lo = box_low(lo, v);
        hi = box_high(hi, v);
      }
    if (d > kBoxThreads) {
      if (live) out[col] = lo, out[d + col] = hi;
      continue;
    }
    sh[0][tid] = lo;
    sh[1][tid] = hi;
    for (int k = reps; k > 1;) {  // columns repeat every d threads: halve the number of repeats
      const int half = (k + 1) / 2;
      __syncthreads();
      if (tid < (k - half) * d) {
        sh[0][tid] = box_low(sh[0][tid], sh[0][tid + half * d]);
        sh[1][tid] = box_high(sh[1][tid], sh[1][tid + half * d]);
      }
      k = half;
    }
    __syncthreads();
    if (tid < d) out[tid] = sh[0][tid], out[d + tid] = sh[1][tid];
  }
}

__global__ __launch_bounds__(1024) void diameter_kernel(const Box a, float* out) {
  const int tid = threadIdx.x, d = a.d;
  __shared__ float sh[2][1024];
  __shared__ float sums[16];
  float sum = 0.f;
  const int groups = d <= 1024 ? min(16, 1024 / d) : 1, width = min(d, 1024);
  for (int c0 = 0; c0 < d; c0 += 1024) {
    const int group = tid / width, col = c0 + tid - group * width;
    float lo = __builtin_inff(), hi = -lo;
    if (group < groups && col < d)
#pragma unroll 8
      for (int b = group; b < a.parts; b += groups) {
        lo = box_low(lo, a.part[(size_t)b * 2 * d + col]);
        hi = box_high(hi, a.part[((size_t)b * 2 + 1) * d + col]);
      }
    __syncthreads();
    sh[0][tid] = lo;
    sh[1][tid] = hi;
    __syncthreads();
    if (tid < width && c0 + tid < d) {
      for (int g = 1; g < groups; ++g) {
        lo = box_low(lo, sh[0][tid + g * width]);
        hi = box_high(hi, sh[1][tid + g * width]);
      }
      sum = __builtin_fmaf(hi - lo, hi - lo, sum);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if ((tid & 63) == 0) sums[tid >> 6] = sum;
  __syncthreads();
  if (tid > 0) return;
#pragma unroll
  for (int w = 1; w < 16; ++w) sum += sums[w];
  *out = sqrtf(sum);
}

int launch_rows(RowStart& t, hipStream_t st) {
  t.wide = t.d % 4 == 0 && ((reinterpret_cast<size_t>(t.pts[0]) | reinterpret_cast<size_t>(t.pts[1])) & 15) == 0;
  t.blocks0 = (t.rows[0] + kRowsOfBlock - 1) / kRowsOfBlock;
  const int blocks = t.blocks0 + (t.rows[1] + kRowsOfBlock - 1) / kRowsOfBlock;
  hipLaunchKernelGGL(row_start_kernel, dim3(blocks), dim3(256), 0, st, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

bool bad_rows(int64_t n, int64_t m) { return n <= 0 || m <= 0 || n > (1 << 30) || m > (1 << 30); }

}  // namespace
}  // namespace fs

extern "C" {

int fs_row_start(const float* x, const float* y, const float* a, const float* b, int64_t n, int64_t m, int64_t d,
                 float cost_scale, float* const* out, void* stream) {
  using namespace fs;
  if (!x || !y || !a || !b || !out) return FS_ERR_NULL_POINTER;
  for (int i = 0; i < 6; ++i)
    if (!out[i]) return FS_ERR_NULL_POINTER;
  if (bad_rows(n, m) || d <= 0 || d > (1 << 20)) return FS_ERR_BAD_SIZE;
  RowStart t{{x, y}, {a, b}, {nullptr, nullptr}, {out[0], out[1]}, {out[2], out[3]}, {out[4], out[5]}, {(int)n, (int)m}, 0, (int)d, 0, cost_scale};
  return launch_rows(t, (hipStream_t)stream);
}

int fs_c_bias(const float* x, const float* y, const float* psi, int64_t n, int64_t m, int64_t d, float cost_scale,
              float* x_norm, float* bias, void* stream) {
  using namespace fs;
  if (!x || !y || !psi || !x_norm || !bias) return FS_ERR_NULL_POINTER;
  if (bad_rows(n, m) || d <= 0 || d > (1 << 20)) return FS_ERR_BAD_SIZE;
  RowStart t{{x, y}, {nullptr, nullptr}, {nullptr, psi}, {x_norm, bias}, {nullptr, nullptr}, {nullptr, nullptr}, {(int)n, (int)m}, 0, (int)d, 0, cost_scale};
  return launch_rows(t, (hipStream_t)stream);
}

size_t fs_diameter_workspace_bytes(int64_t d) { return d <= 0 || d > (1 << 20) ? 0 : (size_t)4 * fs::kBoxBlocks * d * sizeof(float); }

int fs_diameter(const float* x, const float* y, int64_t n, int64_t m, int64_t d, float* out, void* workspace,
                size_t workspace_bytes, void* stream) {
  using namespace fs;
  if (!x || !y || !out || !workspace) return FS_ERR_NULL_POINTER;
  if (bad_rows(n, m) || d <= 0 || d > (1 << 20)) return FS_ERR_BAD_SIZE;
  if (workspace_bytes < fs_diameter_workspace_bytes(d)) return FS_ERR_WORKSPACE_TOO_SMALL;
  const int clouds = x == y && n == m ? 1 : 2;
  const int blocks = (int)std::min<int64_t>(kBoxBlocks, (std::max(n, m) + 31) / 32);
  const Box b{{x, y}, {(int)n, (int)m}, (int)d, blocks, static_cast<float*>(workspace), clouds * blocks};
  hipLaunchKernelGGL(box_kernel, dim3(blocks, clouds), dim3(kBoxThreads), 0, (hipStream_t)stream, b);
  if (hipGetLastError() != hipSuccess) return FS_ERR_LAUNCH_FAILED;
  hipLaunchKernelGGL(diameter_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, b, out);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

int fs_change(const float* f, const float* f_before, int64_t n, const float* g, const float* g_before, int64_t m, float* out,
              void* stream) {
  using namespace fs;
  if (!f || !f_before || !g || !g_before || !out) return FS_ERR_NULL_POINTER;
  if (bad_rows(n, m)) return FS_ERR_BAD_SIZE;
  const Change t{{f, g}, {f_before, g_before}, {(int)n, (int)m}, out};
  hipLaunchKernelGGL(change_kernel, dim3(2), dim3(1024), 0, (hipStream_t)stream, t);
  return hipGetLastError() == hipSuccess ? FS_OK : FS_ERR_LAUNCH_FAILED;
}

}  // extern "C"
