// Symmetric steps of medium problems from one sweep over the logits (d <= 64, fp16 planes), two
// launches per step for the xy problem, the two self problems and every item of a batch.
//
// With S_ij = qs x_i.y_j + r_i + c_j (qs = 2 cs log2(e) / eps, r_i and c_j the biases of x_i and y_j
// as keys), the row sums R_i and the column sums C_j of 2^S give both half-updates of a step:
// LSE_j(x_i.y_j + c_j) = log2 R_i - r_i, LSE_i(x_i.y_j + r_i) = log2 C_j - c_j (see
// fs_lsesweep.hpp, which takes the same two sums).  What bounds such a sweep is the issue of vector
// instructions beside the matrix pipe, so here a logit costs two of them and a third of an
// exponential's share of nothing else:
//   * the planes carry sqrt(qs), so the accumulator holds base-2 logits and nothing scales them;
//   * both biases ride in the matrix product: each is three fp16 pieces at 2^12, 1 and 2^-12
//     (33 bits), [c1 c2 c3 s1 s2 s3] against [s1 s2 s3 r1 r2 r3], one more 16-column MFMA
//     (3 * DP / 16 + 1 per tile) where an fp32 FMA and the preloading of the accumulator were;
//   * the rows that stay in registers are the A operand, so a lane holds 16 of THEM and one
//     streamed row: the sums of the stationary rows are 16 lane-private accumulators that cross
//     lanes once per work item, and a streamed row's sum over a wavefront's 64 stationary rows is
//     lane-private too: no cross-lane step per tile at all.
// 32 instructions per 32 x 32 tile and 16 exponentials: 256 cycles of the vector pipe beside
// 416 cycles of the matrix pipe at 64 columns.
//
// No maximum lies under the exponentials.  Whether a step may be taken this way is decided before
// it runs, from what the step before left behind: bounds on all sums (pair_mode) from the extremes
// of the last sums, of the changes of the potentials, and the ratio of the two eps.  Where
// they do not guarantee that every sum is exact in fp32, the launch runs the step two-sided with
// running maxima (pair_item_two_sided): the first steps of a solve at a small fixed eps, empty
// weights, plans that move fast.  So nothing is ever redone, and a step is these two launches.
#pragma once

#include <type_traits>

#include "fs_colsum.hpp"
#include "fs_common.hpp"
#include "fs_small.hpp"

namespace fs {

constexpr int kPairSlots = 8;        // copies of a step's extremes, over which the workgroups spread
constexpr int kPairStateWords = 3 * kPairSlots * 8;  // three steps' worth, eight extremes each
constexpr float kPairFar = -2.4e8f;  // bias of rows past the last one, in base 2 (2^12 times -58594)

// One problem: stationary rows against streamed rows.  Pointers of item 0.
struct PairProblem {
  const u32x4* st_planes;   // [items][blocks][2 KK][64]
  const u32x4* str_planes;
  const u32x4* st_bias;     // [items][blocks * 32] one piece per row: (s1 s2)(s3 b1)(b2 b3)(0 0)
  const u32x4* str_bias;
  const float* st_bias32;   // [items][blocks * 32] the same as fp32 numbers
  const float* str_bias32;
  float* st_part;           // [items][chunks][rows] sums of the stationary rows
  float* str_part;          // [items][groups][rows] sums of the streamed rows
  int n_st, n_str;
  int st_blocks, str_blocks;  // 32-row blocks, padding included
  int groups, chunks, chunk;  // 256-row groups of the stationary rows; chunks (of rows) of the others
  int self;                 // a matrix with itself: a group streams only rows at or behind its first
  int first_item, n_items;  // work items of this problem in the launch
  // two-sided steps: (maximum, sum) per row and chunk of keys, and their work items (those of the
  // streamed rows' own half-update from two_first on; a self problem has none)
  float2* st_ms;            // [items][chunks][n_st]
  float2* str_ms;           // [items][chunks of n_st][n_str]
  int two_first, two_items;
};

// One side of a problem in the merge: the rows whose potentials it updates.
struct PairSide {
  const float* part;        // sums: [parts][rows]
  const float* col;         // self problems: the column sums that the groups before took
  const float2* ms;         // two-sided steps: (maximum, sum) per chunk of keys, and row
  int ms_parts;
  const float* old;
  float* out;
  const float* norm;
  const float* l2w;
  u32x4* bias;              // written for the next step
  float* bias32;
  u32x4* planes;            // written when the next step has another eps (null: another side does)
  const void* pts;
  int rows, blocks, parts, self, chunk, dtype, d;
  float rho;
};

struct PairArgs {
  PairProblem prob[3];
  PairSide side[4];         // 2 problem + (0 stationary, 1 streamed) for xy, then xx, yy
  const float4* table;      // [items][3][table_len]
  const int* lens;          // [items][3]
  float* state;             // [items][3][kPairStateWords]
  const float4* limits;     // [items] smallest and largest base-2 weight of x, of y
  const float4* reach;      // [items] largest |value|, bound of the costs, bound of a potential
  int step, extrapolate, sched, items, nprob, first_prob, total_items, table_len;
  int merge_groups;         // 256-row groups of the larger cloud: workgroups beyond them write planes
};

// Largest bias that its three pieces hold, with room to spare.
constexpr float kPairMostBias = 6.0e7f;

// Scale of an operand's planes: sqrt(qs), said as 0, or where the planes cannot hold that, a power
// of two (the steps are two-sided then).
__device__ __forceinline__ float pair_scale(float most, float qs) {
  return most * sqrtf(qs) < 30000.f ? 0.f : f16_plane_scale(most);
}

// Which entry of its schedule a step takes.
__device__ __forceinline__ float4 pair_coef(const PairArgs& a, int item, int prob, int step) {
  const float4* t = a.table + ((size_t)item * 3 + prob) * a.table_len;
  return t[a.sched == 0 ? 0 : min(max(step - 1, 0), a.table_len - 1)];
}

// Extremes a merge leaves behind, as values whose largest is kept: largest and minus smallest
// log2 of a row's sum over its weight, of a streamed row's, of the changes of both sides' potentials.
__device__ __forceinline__ unsigned pair_key(float v) {  // order-preserving
  const unsigned u = __builtin_bit_cast(unsigned, v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float pair_value(unsigned k) {
  return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// May step `step` of a problem take both sides from one sweep?  x: log2(R_i / a_i) = log2 of
// sum_j b_j 2^(e_ij), e = the exponent without weights.  The next step's sum is
// sum_j b_j 2^(rho e_ij + kappa (df_i + dg_j)), rho = eps / eps', kappa = log2(e) / eps'.  With
// B = sum b: for rho >= 1 the power means give  rho x - (rho - 1) log2 B <= log2 sum_j b_j 2^(rho e)
// <= rho x - (rho - 1) log2 b_min  (and the other way round for rho < 1).  The biases count the
// weights from the largest of their side (so that logits are small where eps is large, and what a
// matrix product rounds off them is too).  Every sum taken so has to lie in [2^-80, 2^100]: then no exponential overflows, and what is lost below 2^-126 is less
// than 2^-26 of a sum with a million terms.  Before the first step the potentials are minus the norms,
// so e_ij = -C_ij / eps >= -bound / eps.
// By every lane of a wavefront with the same result; `set`: which of the three sets to read.
__device__ __forceinline__ bool pair_mode(const PairArgs& a, int item, int prob, int step) {
  // (every load is issued before anything is decided)
  const float4 now = pair_coef(a, item, prob, step), before = pair_coef(a, item, prob, step - 1);
  const float4 w = a.limits[item], reach = a.reach[item];
  const unsigned* st = reinterpret_cast<const unsigned*>(a.state) +
                       ((size_t)item * 3 + prob) * kPairStateWords + ((step + 2) % 3) * kPairSlots * 8;
  const int lane = threadIdx.x & 63;
  unsigned v = st[lane];  // [slot][8]
  const float4 lim = prob == 0 ? w : (prob == 1 ? make_float4(w.x, w.y, w.x, w.y) : make_float4(w.z, w.w, w.z, w.w));
  bool ok = (pair_scale(reach.x, now.y) == 0.f) & (lim.x > -1000.f) & (lim.z > -1000.f) &
            (now.w * reach.z < kPairMostBias);
  if (step == 0) return ok & (fminf(lim.x - lim.y, lim.z - lim.w) - reach.y * now.w > -80.f);
  const float rho = before.x / now.x, kappa = now.w;
#pragma unroll
  for (int o = 8; o < 64; o <<= 1) v = max(v, (unsigned)__shfl_xor((int)v, o, 64));
  const float mine = pair_value(v);  // lane % 8: which extreme
  float e[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) e[k] = __shfl(mine, k, 64);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    // this side's sums: weights of its own rows (w) and of the others' (k)
    const float hi = e[4 * s], lo = -e[4 * s + 1];
    const float dfh = e[4 * s + 2], dfl = -e[4 * s + 3], dgh = e[4 * (s ^ 1) + 2], dgl = -e[4 * (s ^ 1) + 3];
    const float wmin = s ? lim.z : lim.x, wmax = s ? lim.w : lim.y, kmin = s ? lim.x : lim.z;
    const float kmax = s ? lim.y : lim.w, mass = kmax + 20.f;  // log2 B is at most that, with up to a million keys
    const float up = rho >= 1.f ? rho * hi - (rho - 1.f) * kmin : rho * hi + (1.f - rho) * mass;
    const float dn = rho >= 1.f ? rho * lo - (rho - 1.f) * mass : rho * lo + (1.f - rho) * kmin;
    const float U = up + kappa * (dfh + dgh) - kmax, L = dn + kappa * (dfl + dgl) + (wmin - wmax) - kmax;
    ok = ok & (U < 100.f) & (L > -80.f);
  }
  return ok;  // (false where anything is not a number)
}

__device__ __forceinline__ u32x4 pair_bias(float b) {
  const _Float16 s1 = (_Float16)4096.f, s2 = (_Float16)1.f, s3 = (_Float16)0.000244140625f;
  const _Float16 p1 = (_Float16)(b * 0.000244140625f);
  const float r1 = __builtin_fmaf(-4096.f, (float)p1, b);
  const _Float16 p2 = (_Float16)r1;
  const _Float16 p3 = (_Float16)((r1 - (float)p2) * 4096.f);
  u32x4 v;
  v[0] = pack_f16((float)s1, (float)s2);
  v[1] = pack_f16((float)s3, (float)p1);
  v[2] = pack_f16((float)p2, (float)p3);
  v[3] = 0u;
  return v;
}
// The same row as an A operand: (b1 b2)(b3 s1)(s2 s3), nothing in the upper half-wave.
__device__ __forceinline__ u32x4 pair_bias_a(const u32x4& v, int h) {
  u32x4 r;
  r[0] = __builtin_amdgcn_alignbit(v[2], v[1], 16);
  r[1] = __builtin_amdgcn_alignbit(v[0], v[2], 16);
  r[2] = __builtin_amdgcn_alignbit(v[1], v[0], 16);
  r[3] = 0u;
  if (h) r = u32x4{0u, 0u, 0u, 0u};
  return r;
}

// The streamed operand of a work item: tiles of 64 rows (both planes and the biases) in a ring of three
// LDS buffers, filled by direct global -> LDS loads of 1 KiB per wavefront, two tiles ahead.  LDS
// is read by hand: the compiler cannot tell a read of one buffer from the loads filling another.
// TWO: the biases are fp32 numbers (two-sided steps, which take them at any size) instead of pieces.
template <int DP, bool TWO>
struct PairStream {
  static constexpr int KK = DP / 16, NM = 3 * KK + 1;  // MFMAs of a unit
  static constexpr int PIECES = 2 * 2 * KK;            // 1 KiB pieces of a tile, without the bias
  static constexpr int BUF = PIECES * 64 + 64;         // 16-byte words of a buffer
  static constexpr int LOADS = PIECES / 4 + 1;         // per wavefront and tile
  using Bias = std::conditional_t<TWO, float, u32x4>;
  struct Keys {
    u32x4 p[2][KK];
    Bias b;
  };
  u32x4* lds;
  const u32x4* gsrc;
  const Bias* bsrc;
  int wave, lane;

  __device__ __forceinline__ void begin(u32x4* buffers, const u32x4* planes, const Bias* bias, int blocks, int batch,
                                        int j_begin) {
    lds = buffers;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    gsrc = planes + ((size_t)batch * blocks + j_begin / 32) * (2 * KK * 64) + lane;
    bsrc = bias + (size_t)batch * blocks * 32 + j_begin + lane;
  }
  __device__ __forceinline__ void stage(int tile, int buf) const {
#pragma unroll
    for (int c = 0; c < PIECES / 4; ++c)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(gsrc + (size_t)tile * (PIECES * 64) + (c * 4 + wave) * 64),
          (__attribute__((address_space(3))) void*)(&lds[buf * BUF + (c * 4 + wave) * 64]), 16, 0, 0);
    // (every wavefront moves the bias piece, so that all count the same loads)
    const auto* src = (const __attribute__((address_space(1))) void*)(bsrc + (size_t)tile * 64);
    auto* dst = (__attribute__((address_space(3))) void*)(&lds[buf * BUF + PIECES * 64]);
    if constexpr (TWO) __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
    else __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
  }
  static __device__ __forceinline__ u32x4 read(const u32x4* ptr) {
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1"
                 : "=v"(v)
                 : "v"((unsigned)(size_t)(const __attribute__((address_space(3))) u32x4*)ptr)
                 : "memory");
    return v;
  }
  __device__ __forceinline__ void read_piece(Keys& k, int q, int kk, int buf, int js) const {
    k.p[q][kk] = read(&lds[buf * BUF + (js * (2 * KK) + q * KK + kk) * 64 + lane]);
  }
  __device__ __forceinline__ void read_bias(Keys& k, int buf, int js) const {
    const Bias* at = reinterpret_cast<const Bias*>(&lds[buf * BUF + PIECES * 64]) + js * 32 + (lane & 31);
    if constexpr (TWO) {
      asm volatile("ds_read_b32 %0, %1"
                   : "=v"(k.b)
                   : "v"((unsigned)(size_t)(const __attribute__((address_space(3))) float*)at)
                   : "memory");
    } else {
      k.b = read(at);
    }
  }
  // (low plane, high plane, bias: the order in which a unit needs them)
  __device__ __forceinline__ void read_all(Keys& k, int buf, int js) const {
#pragma unroll
    for (int q = 1; q >= 0; --q)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) read_piece(k, q, kk, buf, js);
    read_bias(k, buf, js);
  }
  // One set of registers holds the streamed operands: in the last unit of a sub-tile every piece is
  // followed, behind the last MFMA that reads it, by the read of the next sub-tile's.
  __device__ __forceinline__ void read_next(Keys& y, int k, int buf, int js) const {
    if (k < KK) read_piece(y, 1, k, buf, js);
    if (k >= 2 * KK && k < 3 * KK) read_piece(y, 0, k - 2 * KK, buf, js);
    if (k == 3 * KK) read_bias(y, buf, js);
  }
  static __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
  // all LDS accesses but the newest N are done
  template <int N>
  static __device__ __forceinline__ void wait_lds() {
    __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
  }
  // every tile but the newest has landed, and all LDS accesses are done
  static __device__ __forceinline__ void wait_tile() {
    __builtin_amdgcn_s_waitcnt(0x0070 | (LOADS & 15) | ((LOADS >> 4) << 14));
  }
  static __device__ __forceinline__ void wait_all() {
    fence();
    __builtin_amdgcn_s_waitcnt(0x0070);
    fence();
  }
  static __device__ __forceinline__ void barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  __device__ __forceinline__ void start(Keys& y) const {
    stage(0, 0);
    stage(1, 1);
    fence();
    wait_tile();
    fence();
    barrier();
    read_all(y, 0, 0);
  }
};

// Both planes of two blocks of 32 rows in registers.
template <int KK>
__device__ __forceinline__ void pair_load_rows(u32x4 (&x)[2][2][KK], const u32x4* planes, int lane) {
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) x[rb][q][kk] = planes[((rb * 2 + q) * KK + kk) * 64 + lane];
}

// A work item with running maxima: 256 query rows (B operand: a lane holds one row and 16 keys)
// against a chunk of keys, as lse2_kernel does it on the same tiles.
template <int DP>
__device__ __forceinline__ void pair_item_two_sided(const PairArgs& a, int batch, const PairProblem& pr, int prob, int it,
                                                    u32x4* lds) {
  using S = PairStream<DP, true>;
  constexpr int KK = DP / 16, NM = S::NM;
  const int side = it >= pr.two_first ? 1 : 0;  // the streamed rows' own half-update
  if (side) it -= pr.two_first;
  const int n_k = side ? pr.n_st : pr.n_str, n_q = side ? pr.n_str : pr.n_st;
  const int groups = (n_q + 255) / 256, chunk = it / groups, group = it % groups;
  const int kblocks = side ? pr.st_blocks : pr.str_blocks, qblocks = side ? pr.str_blocks : pr.st_blocks;
  const int lane = threadIdx.x & 63, li = lane & 31, h = lane >> 5;
  const int j_begin = chunk * pr.chunk, j_end = min(n_k, j_begin + pr.chunk);
  const int ntiles = (j_end - j_begin + 63) / 64;
  const float4 coef = pair_coef(a, batch, prob, a.step);
  // (planes that cannot carry sqrt(qs) carry a power of two instead)
  const float ps = pair_scale(a.reach[batch].x, coef.y);
  const float lscale = ps == 0.f ? 1.0f : coef.y / (ps * ps);
  S ks;
  ks.begin(lds, side ? pr.st_planes : pr.str_planes, side ? pr.st_bias32 : pr.str_bias32, kblocks, batch, j_begin);
  const int blk0 = group * 8 + ks.wave * 2;
  u32x4 x[2][2][KK];
  pair_load_rows(x, (side ? pr.str_planes : pr.st_planes) + ((size_t)batch * qblocks + blk0) * (2 * KK * 64), lane);
  float m[2], s[2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    m[rb] = 0.5f * kNegBig;  // above the rows past the last one, below every real logit
    s[rb] = 0.f;
  }
  typename S::Keys y;
  int cur = 0, nxt = 1, nx2 = 2;
  ks.start(y);
  f32x16 R0, R1;
#pragma unroll
  for (int r = 0; r < 16; ++r) R1[r] = kNegBig;
  // the soft-max of the unit before, cut into NM pieces: maximum, rescale, exponentials
  auto soft = [&](int k, const f32x16& v, int rb, float& mx, float (&e)[16], float& p0, float& p1) {
    constexpr int K0 = (NM + 3) / 4;  // pieces of the maximum
    if (k == 0) mx = m[rb];
    if (k < K0) {
      const int v0 = k * 8 / K0, v1 = (k + 1) * 8 / K0;
#pragma unroll
      for (int c = v0; c < v1; ++c) mx = fmaxf(fmaxf(mx, v[2 * c]), v[2 * c + 1]);
      if (k == K0 - 1) {
        s[rb] *= fast_exp2(m[rb] - mx);
        m[rb] = mx;
        p0 = p1 = 0.f;
      }
    } else {
      const int n = NM - K0, v0 = (k - K0) * 16 / n, v1 = (k - K0 + 1) * 16 / n;
#pragma unroll
      for (int r = v0; r < v1; ++r) e[r] = fast_exp2(v[r] - mx);
      if (k > K0) {
        const int u0 = (k - K0 - 1) * 16 / n;
#pragma unroll
        for (int r = u0; r < v0; ++r) {
          if (r & 1) p1 += e[r]; else p0 += e[r];
        }
      }
      if (k == NM - 1) {
#pragma unroll
        for (int r = v0; r < 16; ++r) {
          if (r & 1) p1 += e[r]; else p0 += e[r];
        }
        s[rb] += p0 + p1;
      }
    }
  };
  for (int t = 0; t < ntiles; ++t) {
#pragma unroll
    for (int js = 0; js < 2; ++js)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        f32x16& acc = rb ? R1 : R0;
        f32x16& prev = rb ? R0 : R1;
        if (rb == 0) ks.template wait_lds<KK + 1>();
        S::fence();
        float e[16], mx, p0, p1;
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          if (k == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          }
          if (rb == 0 && k == KK) {
            ks.template wait_lds<0>();
            S::fence();
          }
          if (k < 3 * KK) {
            const int prod = k / KK, kk = k % KK;
            acc = small_mfma(y.p[prod == 0 ? 1 : 0][kk], x[rb][prod == 1 ? 1 : 0][kk], acc);
          } else {
            if (lscale != 1.0f) {
#pragma unroll
              for (int r = 0; r < 16; ++r) acc[r] *= lscale;
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 0.f : y.b, h ? 0.f : 1.0f, acc, 0, 0, 0);
          }
          if (js == 0 && rb == 0 && k == 0) ks.stage(t + 2, nx2);
          if (rb == 1 && js == 1 && k == 0) {
            ks.wait_tile();
            S::barrier();
          }
          if (rb == 1) ks.read_next(y, k, js == 0 ? cur : nxt, js ^ 1);
          soft(k, prev, rb ^ 1, mx, e, p0, p1);
          S::fence();
        }
      }
    const int c = cur;
    cur = nxt;
    nxt = nx2;
    nx2 = c;
  }
  {
    float e[16], mx, p0, p1;
#pragma unroll
    for (int k = 0; k < NM; ++k) soft(k, R1, 1, mx, e, p0, p1);
  }
  S::wait_all();
  __syncthreads();  // (the next item fills the same buffers)
  float2* out = (side ? pr.str_ms : pr.st_ms) + ((size_t)batch * ((n_k + pr.chunk - 1) / pr.chunk) + chunk) * n_q;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float mo = xor32(m[rb]), so = xor32(s[rb]);
    const float M = fmaxf(m[rb], mo);
    const float sum = s[rb] * fast_exp2(m[rb] - M) + so * fast_exp2(mo - M);
    const int row = (blk0 + rb) * 32 + li;
    if (h == 0 && row < n_q) out[row] = make_float2(M, sum);
  }
}

// One step.  Grid (work items of all problems, rounded up to a multiple of 8; items of the batch).
// A workgroup of four wavefronts owns 256 stationary rows (two blocks of 32 per wavefront, operands
// in registers) and streams a chunk of the other matrix.  The exponentials of one 32 x 32 unit sit
// between the MFMAs of the next in program order.
template <int DP>
__global__ __launch_bounds__(256, 2) void pair_sweep_kernel(const PairArgs a) {
  using S = PairStream<DP, false>;
  constexpr int KK = DP / 16, NM = S::NM;
  __shared__ __attribute__((aligned(16))) u32x4 lds[3 * S::BUF];
  __shared__ float lds_col[2][4][2][64];        // [tile parity][wavefront][half-wave][row]

  const int batch = blockIdx.y;
  // XCD-aware: workgroups are dealt round-robin to the 8 XCDs; XCD x takes the x-th eighth of the
  // items, whose order is chunk by chunk: what runs on an XCD at one time shares a chunk in its L2
  const int per = (a.total_items + 7) / 8;
  int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || item >= a.total_items) return;
  int p = a.first_prob;
  while (p + 1 < a.nprob && item >= a.prob[p + 1].first_item) ++p;
  const PairProblem& pr = a.prob[p];
  if (a.step > a.lens[batch * 3 + p] + a.extrapolate) return;  // its schedule is shorter
  item -= pr.first_item;
  if (!pair_mode(a, batch, p, a.step)) {
    for (int it = item; it < pr.two_items; it += pr.n_items) pair_item_two_sided<DP>(a, batch, pr, p, it, lds);
    return;
  }
  int chunk = 0, group = item;
  if (pr.self) {
    for (;;) {
      const int g = self_groups_of_chunk(chunk, pr.chunk, pr.n_str, pr.groups);
      if (group < g) break;
      group -= g;
      ++chunk;
    }
  } else {
    chunk = item / pr.groups;
    group = item % pr.groups;
  }
  const int lane = threadIdx.x & 63, li = lane & 31, h = lane >> 5;
  const int j_begin = pr.self ? max(chunk * pr.chunk, group * 256) : chunk * pr.chunk;
  const int j_end = min(pr.n_str, (chunk + 1) * pr.chunk);
  const int ntiles = (j_end - j_begin + 63) / 64;
  S ks;
  ks.begin(lds, pr.str_planes, pr.str_bias, pr.str_blocks, batch, j_begin);
  const int wave = ks.wave;

  // ---- stationary operands ----
  const int blk0 = group * 8 + wave * 2;
  u32x4 xa[2][2][KK], xb[2];
  pair_load_rows(xa, pr.st_planes + ((size_t)batch * pr.st_blocks + blk0) * (2 * KK * 64), lane);
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) xb[rb] = pair_bias_a(pr.st_bias[((size_t)batch * pr.st_blocks + blk0 + rb) * 32 + li], h);
  // MFMA k of a unit: the cross products, hi * hi, the biases
  auto mfma_k = [&](int k, const f32x16& acc, const typename S::Keys& y, int rb) {
    if (k == 3 * KK) return small_mfma(xb[rb], y.b, acc);
    const int prod = k / KK, kk = k % KK;
    return small_mfma(xa[rb][prod == 1 ? 1 : 0][kk], y.p[prod == 0 ? 1 : 0][kk], acc);
  };

  float st[2][16];  // sums of the stationary rows, over the streamed rows this lane sees
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[rb][r] = 0.f;
  const unsigned col_at = (unsigned)(size_t)(const __attribute__((address_space(3))) float*)&lds_col[0][0][0][0];
  auto put_sum = [&](int tile, int js, float v) {
    asm volatile("ds_write_b32 %0, %1" : : "v"(col_at + 4 * ((((tile & 1) * 4 + wave) * 2 + h) * 64 + js * 32 + li)), "v"(v)
                 : "memory");
  };
  float* colp = pr.str_part + ((size_t)batch * pr.groups + group) * pr.n_str;
  auto flush = [&](int tile) {  // a tile's sums over the four wavefronts, in a fixed order
    float c[8];
#pragma unroll
    for (int w = 0; w < 8; ++w)
      asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(c[w]) : "v"(col_at + 4 * ((tile & 1) * 512 + lane)), "n"(w * 256)
                   : "memory");
    S::fence();
    ks.template wait_lds<0>();
    S::fence();
    float v = c[0] + c[1];
#pragma unroll
    for (int w = 1; w < 4; ++w) v += c[2 * w] + c[2 * w + 1];
    const int j = j_begin + tile * 64 + lane;
    if (j < j_end) colp[j] = v;
  };

  typename S::Keys y;
  int cur = 0, nxt = 1, nx2 = 2;
  ks.start(y);
  f32x16 R0, R1;  // running chain and the unit whose exponentials are taken
#pragma unroll
  for (int r = 0; r < 16; ++r) R1[r] = -1.0e30f;
  float ps0 = 0.f, ps1 = 0.f, pend = 0.f;
  for (int t = 0; t < ntiles; ++t) {
#pragma unroll
    for (int js = 0; js < 2; ++js) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        f32x16& acc = rb ? R1 : R0;
        f32x16& prev = rb ? R0 : R1;
        const int prb = rb ^ 1;
        if (rb == 0) ks.template wait_lds<KK + 1>();  // the low plane is there
        S::fence();
        float e[16];
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          if (k == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          }
          if (rb == 0 && k == KK) {
            ks.template wait_lds<0>();  // everything is
            S::fence();
          }
          acc = mfma_k(k, acc, y, rb);
          if (js == 0 && rb == 0 && k == 0) ks.stage(t + 2, nx2);
          if (rb == 1 && js == 1 && k == 0) {
            // tile t + 1 has landed, and every wavefront is through with reading tile t and with
            // its sums of tile t - 1
            ks.wait_tile();
            S::barrier();
            // (written behind the barrier: the reader of the tile before last is done)
            put_sum(t, 0, pend);
            if (t >= 1 && wave == (t & 3)) flush(t - 1);
          }
          if (rb == 1) ks.read_next(y, k, js == 0 ? cur : nxt, js ^ 1);
          // the exponentials of the unit before
          const int v0 = k * 16 / NM, v1 = (k + 1) * 16 / NM;
#pragma unroll
          for (int r = v0; r < v1; ++r) e[r] = fast_exp2(prev[r]);
          if (k > 0) {
            const int u0 = (k - 1) * 16 / NM, u1 = k * 16 / NM;
#pragma unroll
            for (int r = u0; r < u1; ++r) {
              st[prb][r] += e[r];
              if (r & 1) ps1 += e[r]; else ps0 += e[r];
            }
          }
          S::fence();
        }
        {
#pragma unroll
          for (int r = (NM - 1) * 16 / NM; r < 16; ++r) {
            st[prb][r] += e[r];
            if (r & 1) ps1 += e[r]; else ps0 += e[r];
          }
        }
        if (prb == 1) {  // the streamed rows of the sub-tile before are complete
          const float v = ps0 + ps1;
          ps0 = ps1 = 0.f;
          if (js == 1) {
            pend = v;
          } else {
            if (t >= 1) put_sum(t - 1, 1, v);
          }
        }
        S::fence();
      }
    }
    const int c = cur;
    cur = nxt;
    nxt = nx2;
    nx2 = c;
  }
  // ---- the last unit, the last tile's sums ----
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float e = fast_exp2(R1[r]);
    st[1][r] += e;
    if (r & 1) ps1 += e; else ps0 += e;
  }
  put_sum(ntiles - 1, 1, ps0 + ps1);
  S::wait_all();  // (also what was fetched past the chunk)
  __syncthreads();
  if (wave == 0) flush(ntiles - 1);
  // ---- the stationary rows' sums over the lanes ----
  float* rowp = pr.st_part + ((size_t)batch * pr.chunks + chunk) * pr.n_st;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    float v = colsum_all(st[rb], li);
    v += __shfl_xor(v, 16, 64);
    const int row = (blk0 + rb) * 32 + colsum_key(li & 15, h);
    if (li < 16 && row < pr.n_st) rowp[row] = v;
  }
}

// Operand planes of one block of 32 rows at an eps: sqrt(qs) times the rows (as a sum of two floats,
// so that the product of two of them is qs to 2^-46), two fp16 planes.  By 256 threads.
template <int DP>
__device__ __forceinline__ void pair_write_planes(u32x4* out, const void* pts, size_t row0, int rows_here, int d,
                                                  int dtype, float scale, float qs, int tid, int threads) {
  constexpr int KK = DP / 16;
  float s_hi = scale, s_lo = 0.f;
  if (scale == 0.f) {
    s_hi = sqrtf(qs);
    s_lo = __builtin_fmaf(-s_hi, s_hi, qs) / (2.0f * s_hi);
  }
  for (int e = tid; e < KK * 64; e += threads) {
    const int kk = e >> 6, lane = e & 63, row = lane & 31, c0 = 16 * kk + 8 * (lane >> 5);
    u32x4 hi, lo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float f[2], g[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int c = c0 + 2 * q + i;
        const float v = (row < rows_here && c < d) ? small_load(pts, (row0 + row) * d + c, dtype) : 0.f;
        const _Float16 hh = (_Float16)(v * s_hi);
        f[i] = (float)hh;
        g[i] = __builtin_fmaf(v, s_hi, -f[i]) + v * s_lo;
      }
      hi[q] = pack_f16(f[0], f[1]);
      lo[q] = pack_f16(g[0], g[1]);
    }
    out[kk * 64 + lane] = hi;
    out[(KK + kk) * 64 + lane] = lo;
  }
}

// Behind a step (or, with step = -1, before the first): the new potentials from the sums, and what the
// next step reads: the rows' biases, their planes when its eps is another one, and the extremes
// that say how it may run.  Grid (256-row groups, then 128-row ones that write planes, of the larger
// cloud; sides; items).  Bound by memory latency: four wavefronts share the partial sums of 64 rows.  The
// extremes are combined in the workgroup first: with an atomic maximum per 64 rows a merge took
// 13.6 us at 10,000 points, debiased, half of it for them.
template <int DP>
__global__ __launch_bounds__(1024) void pair_merge_kernel(const PairArgs a) {
  const int side = blockIdx.y + (a.first_prob ? 2 : 0), item = blockIdx.z, tid = threadIdx.x;
  const PairSide& sd = a.side[side];
  const int prob = side < 2 ? 0 : side - 1, step = a.step;
  const int entries = a.lens[item * 3 + prob];
  const float4 next = pair_coef(a, item, prob, min(step + 1, entries + a.extrapolate));
  if (step > entries + a.extrapolate) return;
  if ((int)blockIdx.x >= a.merge_groups) {
    // ---- planes for a step with another eps: a quarter of a workgroup per 32 rows ----
    const int blk = (blockIdx.x - a.merge_groups) * 4 + (tid >> 8);
    if (sd.planes == nullptr || blk >= sd.blocks || step >= entries + a.extrapolate) return;
    if (step >= 0 && pair_coef(a, item, prob, step).x == next.x) return;
    pair_write_planes<DP>(sd.planes + ((size_t)item * sd.blocks + blk) * (2 * (DP / 16) * 64), sd.pts,
                          (size_t)item * sd.rows + blk * 32, sd.rows - blk * 32, sd.d, sd.dtype,
                          pair_scale(a.reach[item].x, next.y), next.y, tid & 255, 256);
    return;
  }
  if ((int)blockIdx.x * 256 >= sd.blocks * 32) return;
  unsigned* state = reinterpret_cast<unsigned*>(a.state) + ((size_t)item * 3 + prob) * kPairStateWords;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int part = wave & 3, quarter = wave >> 2, row = blockIdx.x * 256 + quarter * 64 + lane;
  const bool live = row < sd.rows;
  const size_t at = (size_t)item * sd.rows + min(row, sd.rows - 1);
  const float old = sd.old[at], norm = sd.norm[at];
  // the row's log weight from the largest of its side, and the other side's largest
  const float4 lim = a.limits[item];
  const bool of_x = side == 0 || side == 2;
  const float own = of_x ? lim.y : lim.w, others = side >= 2 ? own : (of_x ? lim.w : lim.y);
  const float l2w = sd.l2w[at] - own;
  float f = old;
  if (step < 0) {
    if (part > 0) return;
    // (nothing is known of the sums yet)
    if (blockIdx.x == 0 && quarter == 0 && (side == 0 || side >= 2))
      for (int i = lane; i < kPairStateWords; i += 64) state[i] = 0u;
  } else {
    __shared__ float2 sh[4][4][64];
    __shared__ float sh_ex[4][4];
    const float4 coef = pair_coef(a, item, prob, step);
    const float r = __builtin_fmaf(coef.w, old, l2w);  // the row's bias in this step
    const bool sweep = pair_mode(a, item, prob, step);
    float2 mine = make_float2(kNegBig, 0.f);
    const int rc = min(row, sd.rows - 1);
    if (sweep) {
      float s = 0.f;
      const float* p = sd.part + (size_t)item * sd.parts * sd.rows + rc;
      if (sd.self) {
        const int own = rc >> 8;
#pragma unroll 4
        for (int c = own * 256 / sd.chunk + part; c < sd.parts; c += 4) s += p[(size_t)c * sd.rows];
        const float* q = sd.col + (size_t)item * ((sd.rows + 255) / 256) * sd.rows + rc;
#pragma unroll 8
        for (int g = part; g < own; g += 4) s += q[(size_t)g * sd.rows];
      } else {
#pragma unroll 8
        for (int c = part; c < sd.parts; c += 4) s += p[(size_t)c * sd.rows];
      }
      mine.y = s;
    } else {
      const float2* p = sd.ms + (size_t)item * sd.ms_parts * sd.rows + rc;
#pragma unroll 8
      for (int c = part; c < sd.ms_parts; c += 4) {
        const float2 v = p[(size_t)c * sd.rows];
        const float M = fmaxf(mine.x, v.x);
        mine.y = mine.y * fast_exp2(mine.x - M) + v.y * fast_exp2(v.x - M);
        mine.x = M;
      }
    }
    sh[quarter][part][lane] = mine;
    __syncthreads();
    const float2(&all)[4][64] = sh[quarter];
    float lse;
    if (sweep) {
      lse = small_log2((all[0][lane].y + all[1][lane].y) + (all[2][lane].y + all[3][lane].y), others) - r;
    } else {
      float M = kNegBig, s = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) M = fmaxf(M, all[w][lane].x);
#pragma unroll
      for (int w = 0; w < 4; ++w) s += all[w][lane].y * fast_exp2(all[w][lane].x - M);
      lse = small_log2(fmaxf(s, 1e-40f), M + others);
    }
    const float rho = sd.rho, eps = coef.x;
    const float damp = rho > 0.f ? 1.0f / (1.0f + eps / rho) : 1.0f;
    const float alpha = (step == 0 || step > entries) ? 1.0f : 0.5f;
    f = alpha * (-eps * damp * kLn2 * lse);
    if (alpha != 1.0f) f += (1.0f - alpha) * old;
    if (damp < 1.0f) f -= alpha * (1.0f - damp) * norm;
    float ex[4] = {-3.0e38f, -3.0e38f, -3.0e38f, -3.0e38f};
    if (live && part == 0) {
      sd.out[at] = f;
      const float x = __builtin_fmaf(coef.w, old, lse), df = f - old;
      ex[0] = x; ex[1] = -x; ex[2] = df; ex[3] = -df;
      if (!(x == x) || !(df == df) || !(fabsf(next.w * f) < kPairMostBias)) ex[0] = ex[1] = ex[2] = ex[3] = 3.0e38f;
    }
    // (the set that the next merge writes into)
    if (blockIdx.x == 0 && (side == 0 || side >= 2) && tid < kPairSlots * 8)
      state[((step + 1) % 3) * kPairSlots * 8 + tid] = 0u;
    if (part == 0) {
      // halves of the four change places, then what is left of each
#pragma unroll
      for (int o = 32, n = 2; n > 0; o >>= 1, n >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int k = 0; k < n; ++k) ex[k] = fmaxf(up ? ex[k + n] : ex[k], __shfl_xor(up ? ex[k] : ex[k + n], o, 64));
      }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) ex[0] = fmaxf(ex[0], __shfl_xor(ex[0], o, 64));
      if ((lane & 15) == 0) sh_ex[lane >> 4][quarter] = ex[0];
    }
    __syncthreads();
    if (tid < 8 && (tid < 4 || side >= 2)) {  // (a self problem's two sides are one)
      const float* e = sh_ex[tid & 3];
      unsigned* slot = state + (step % 3) * kPairSlots * 8 + (blockIdx.x % kPairSlots) * 8;
      atomicMax(&slot[side == 1 ? 4 + tid : tid], pair_key(fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3]))));
    }
  }
  // ---- for the next step ----
  if (part > 0 || step >= entries + a.extrapolate || row >= sd.blocks * 32) return;
  const float b = live ? fmaxf(__builtin_fmaf(next.w, f, l2w), kNegBig) : kNegBig;
  sd.bias[(size_t)item * sd.blocks * 32 + row] = pair_bias(fmaxf(b, kPairFar));
  sd.bias32[(size_t)item * sd.blocks * 32 + row] = b;
}

}  // namespace fs
