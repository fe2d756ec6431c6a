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
//
// At small eps a plan is peaked: of the 32 x 32 units of logits all but a few have none within 44 base-2
// units of any sum (10,000 x 10,000 x 64, N(0, I), eps = 0.01: 84 %, of a self problem 99.4).  Such units
// end at their coarse products (pair_run_coarse), and where the potentials settle at one eps the units
// that do not are kept as lists, which the next steps go along without a look at the others
// (pair_run_list).  Which form a step takes follows from the same words as above (pair_mode).  Launch
// of the 10,000 x 64 debiased step: 85 us every logit, 43 the coarse form, 27 the lists (of which
// some 8 are the chain of loads in front of the first unit).
#pragma once

#include <type_traits>

#include "fs_colsum.hpp"
#include "fs_common.hpp"
#include "fs_small.hpp"

namespace fs {

constexpr int kPairSlots = 8;        // copies of a step's extremes, over which the workgroups spread
// three steps' worth: eight extremes in each slot, then the units that went on, a cache line per slot, then
// what is known of the lists (pair_mode), a cache line per step
constexpr int kPairCounts = 3 * kPairSlots * 8;
constexpr int kPairLists = kPairCounts + 3 * kPairSlots * 32;
constexpr int kPairTaken = kPairLists + 3 * 32;  // per step and XCD, of the first problem: work items taken
constexpr int kPairModes = kPairTaken + 3 * 8 * 32;  // how the newest step was taken (PairMode)
constexpr int kPairStateWords = kPairModes + 32;
constexpr int kPairListWords = 4;    // 64-bit words per wavefront of a work item: [row block][half of the sub-tiles]
constexpr int kPairMostTiles = 64;   // of a chunk
constexpr float kPairGap = 44.f;     // base-2 distance below every sum at which a logit is left out
// Share of units that go on up to which the coarse test pays.  The line is flat: 30 steps at a fixed eps with 0.25 /
// 0.4 / 0.5 / 0.7 here, 12,000 x 9 (share 0.35) 1,512 / 1,250 / 1,260 / 1,351 us, 12 columns 1,240 / 1,380 / 1,385 /
// 1,531 at eps 0.05, 18 columns there 1,600 / 1,656 / 1,655 / 1,540, 32 at 0.1 - / 1,627 / 1,715 / 1,606.
constexpr float kPairOn = 0.4f;
constexpr float kPairTwoOn = 0.7f;   // the same of two-sided steps
constexpr float kPairLeast = -84.f, kPairMost = 120.f;  // log2 of the smallest and largest sum of a one-sweep step
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
  float units;              // 32 x 32 units of all its work items; 0: every logit is computed
  int ends;                 // two-sided steps may end units as well
  int strict;               // neither marginal is relaxed
  unsigned long long* list; // [items][n_items][wavefront][kPairListWords] units to visit
  unsigned long long* two_list;  // [items][two_items][wavefront][kPairListWords] those that a two-sided step ran
  int n_items;              // work items of this problem
  // two-sided steps: (maximum, sum) per row and chunk of keys, and their work items (those of the
  // streamed rows' own half-update from two_first on; a self problem has none)
  float2* st_ms;            // [items][chunks][n_st]
  float2* str_ms;           // [items][chunks of n_st][n_str]
  int* st_best;             // ... and the key of that maximum, where a coarse step has seen one (else -1)
  int* str_best;
  int two_first, two_items;
};

// How a step is taken (pair_mode): both sides from one sweep, and with which units.  Found where the step begins, by the
// sweep's workgroups, and left in the problem's state for the merge, which has to add the very shift that the sweep took off
// (found a second time there, a settled step of 4,500 x 3 took 15.1 us, now 14.7, 4,500 x 8 the same, 4,800 x 4,300 x 16
// 16.9 -> 16.3, 10,850 x 7,531 x 23 30.9 -> 30.4, 10,000 x 64 37.0 -> 36.4).
struct PairMode {  // (the first five are an interface: fs_small_last_step_offset)
  int sweep;     // else two-sided with running maxima
  int list;      // only the units on the lists
  int coarse;    // units are ended by their coarse products where these allow it
  float low;     // log2 of every sum is above that
  float shift;   // taken off every base-2 logit of a one-sweep step, so that its sums fit fp32
  float ratio;   // the next step's logits over this one's, where its eps is smaller
  float drift;   // with a list: what a logit may have risen by since it was made
  float base;    // ... and what no logit off it reached then
  float reserve; // how far below this step's line a list made now begins
  int two;       // a two-sided step whose units are ended by their coarse products
  float rho;     // its logits over those of the step before
  float least[2];  // what the least change of the other rows' potentials adds to a logit of the rows of a side
};
static_assert(sizeof(PairMode) <= 32 * sizeof(float), "a cache line of the state");

// One side of a problem in the merge: the rows whose potentials it updates.
struct PairSide {
  const float* part;        // sums: [parts][rows]
  const float* col;         // self problems: the column sums that the groups before took
  const float2* ms;         // two-sided steps: (maximum, sum) per chunk of keys, and row
  const int* best;
  int ms_parts;
  // of every row: log2 of its last sum in the kernels' units, the key of its largest logit when a two-sided
  // step last saw one (-1: none has), the two points' inner product
  float* sum2;
  int* key;
  float* dot;
  const void* other;        // points and number of the rows that its keys are
  int others;
  float* pot;               // [2 parities][items][rows] potentials
  const float* norm;
  const float* l2w;
  u32x4* bias;              // written for the next step
  float* bias32;
  u32x4* planes;            // written when the next step has another eps (null: another side does)
  const void* pts;
  int rows, blocks, parts, self, chunk, dtype, d;
  float rho;
};

// What the two kernels of a step read besides the step's number.  It lies in the workspace: a kernel's
// arguments are read past the L2 caches, a line at a time where what is needed of them depends on what was
// read (touching all of their lines first made a launch 3 us longer).  So the only argument beside the
// step is this address, which the command processor preloads into registers: a settled step of
// 4,500 x 64 takes 19.9 us in two launches, 21.8 with everything in the arguments.
struct PairArgs {
  PairProblem prob[3];
  PairSide side[4];         // 2 problem + (0 stationary, 1 streamed) for xy, then xx, yy
  const float4* table;      // [items][3][table_len]
  const int* lens;          // [items][3]
  float* state;             // [items][3][kPairStateWords]
  const float4* limits;     // [items] smallest and largest base-2 weight of x, of y
  const float4* reach;      // [items] largest |value|, bound of the costs, bound of a potential, log2 of the larger mass
  int extrapolate, sched, items, nprob, first_prob, table_len;
  int merge_groups;         // 256-row groups of the larger cloud: workgroups beyond them write planes
  int per_xcd;              // work items of an XCD: an eighth of every problem's
  int4* work;               // [8][per_xcd]: problem + 4 * item of it, or -1; chunk + 65536 * group; first and last streamed row
};

typedef const __attribute__((address_space(4))) PairArgs* PairArgsPtr;  // (read by scalar loads)

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
// log2 of a row's sum over its weight with the row's new potential, of a streamed row's, of the changes of both
// sides' potentials.
__device__ __forceinline__ unsigned pair_key(float v) {  // order-preserving
  const unsigned u = __builtin_bit_cast(unsigned, v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float pair_value(unsigned k) {
  return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// May step `step` of a problem take both sides from one sweep?  x: log2(R_i / a_i) = log2 of
// sum_j b_j 2^(e_ij), e = the exponent without weights.  The next step's sum is
// sum_j b_j 2^(rho (e_ij + kappa (df_i + dg_j))), rho = eps / eps', kappa = log2(e) / eps.  The merge leaves the
// extremes of z_i = x_i + kappa df_i, so at the old eps the new logarithms lie between z_i + kappa min dg and
// z_i + kappa max dg (the extremes of x_i and of df_i by themselves would count a change twice where an averaged
// step halves x_i: 30,011 x 29,989 x 64 to blur 0.05 took two steps more two-sided, 0.70 and 0.96 ms for 0.33
// each).  Where neither marginal is relaxed and the step was averaged, kappa df_i = -x_i / 2 and
// kappa dg_j = -y_j / 2, so a new term is the geometric mean of b_j 2^(e_ij - x_i), of which a row's sum is one, and
// of b_j 2^(e_ij - y_j) <= b_j / a_i: the sum is at most sqrt(B / a_i), B = sum b.  From there to the
// new eps, for rho >= 1 the power means give  rho x - (rho - 1) log2 B <= log2 sum_j b_j 2^(rho e)
// <= rho x - (rho - 1) log2 b_min  (and the other way round for rho < 1).  The biases count the
// weights from the largest of their side (so that logits are small where eps is large, and what a
// matrix product rounds off them is too).  Every sum has to lie in [2^-84, 2^120] once all logits are
// shifted by one number: then no exponential overflows (kappa f is up to 6e7 units, where a float's step is 4 and a
// logit's rounding as much: see the merge), and what is lost below 2^-126 is less
// than 2^-26 of a sum with 65,536 terms.  Before the first step the potentials are minus the norms,
// so e_ij = -C_ij / eps >= -bound / eps.
// By every lane of a wavefront with the same result; `set`: which of the three sets to read.
struct PairKnown {  // what pair_mode decides from: all loaded before anything is waited for
  float4 now, before, next, w, reach, list;
  float twos;        // two-sided steps with coarse products so far
  unsigned ext, on;  // lane: [slot][which extreme]; units that went on, of slot lane % 8
};
__device__ __forceinline__ PairKnown pair_known(const PairArgs& a, int item, int prob, int step) {
  PairKnown k;
  k.now = pair_coef(a, item, prob, step);
  k.before = pair_coef(a, item, prob, step - 1);
  k.next = pair_coef(a, item, prob, step + 1);
  k.w = a.limits[item];
  k.reach = a.reach[item];
  const float* st = a.state + ((size_t)item * 3 + prob) * kPairStateWords;
  k.list = *reinterpret_cast<const float4*>(st + kPairLists + (step % 3) * 32);
  k.twos = st[kPairLists + (step % 3) * 32 + 4];
  const unsigned* at = reinterpret_cast<const unsigned*>(st);
  const int set = (step + 2) % 3;
  k.ext = at[set * kPairSlots * 8 + (threadIdx.x & 63)];
  k.on = at[kPairCounts + (set * kPairSlots + (threadIdx.x & 7)) * 32];
  __builtin_amdgcn_sched_barrier(0);
  return k;
}
__device__ __forceinline__ PairMode pair_mode(const PairKnown& k, float units, bool ends, bool strict, int prob, int step) {
  const float4 now = k.now, before = k.before, next = k.next, w = k.w, reach = k.reach;
  const float4 lim = prob == 0 ? w : (prob == 1 ? make_float4(w.x, w.y, w.x, w.y) : make_float4(w.z, w.w, w.z, w.w));
  const bool ok0 = (pair_scale(reach.x, now.y) == 0.f) & (now.w * reach.z < kPairMostBias);
  bool ok = ok0 & (lim.x > -1000.f) & (lim.z > -1000.f);
  PairMode mode;
  mode.ratio = next.x < now.x ? now.x * __builtin_amdgcn_rcpf(next.x) : 1.f;
  mode.coarse = mode.list = mode.two = 0;
  mode.rho = 1.f;
  mode.least[0] = mode.least[1] = 0.f;
  mode.drift = mode.base = mode.reserve = mode.shift = 0.f;
  const float mass = reach.w;  // log2 of the larger sum of weights
  float most = -3.0e38f;       // log2 of every sum is below that
  // (whole numbers, which fp16 holds)
  auto fit = [&]() {
    // (one of the two is zero, or no number fits; by branches 0.15 us of a step at 10,850 x 7,531 x 23)
    mode.shift = fmaxf(ceilf(most - kPairMost), 0.f) + fminf(floorf(mode.low - kPairLeast), 0.f);
    return (most - mode.shift <= kPairMost) & (mode.low - mode.shift >= kPairLeast) & (fabsf(mode.shift) < 2000.f);
  };
  if (step == 0) {
    mode.low = fminf(lim.x - lim.y, lim.z - lim.w) - reach.y * now.w;
    most = mass - fminf(lim.y, lim.w);
    mode.sweep = ok & fit();
    return mode;
  }
  const float rho = before.x == now.x ? 1.f : before.x * __builtin_amdgcn_rcpf(now.x), kappa = now.w;
  static_assert(kPairSlots == 8, "a wavefront holds them");
  unsigned v = k.ext, on = k.on;
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) {
    v = max(v, (unsigned)__shfl_xor((int)v, 8 * o, 64));
    on += (unsigned)__shfl_xor((int)on, o, 64);
  }
  float e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = pair_value((unsigned)__builtin_amdgcn_readlane((int)v, i));
  // (behind a two-sided step nothing is known: tried)
  mode.coarse = (float)on < kPairOn * units;
  // (the first one finds the keys from which the next can tell what is far)
  // (before the second step the potentials jump: nothing of the last one says what is far)
  mode.two = ends && step >= 2 && ok0 && rho >= 1.f && (k.twos == 1.f || (float)on < kPairTwoOn * units);
  mode.rho = rho;
  mode.least[0] = -kappa * e[7];
  mode.least[1] = -kappa * e[3];
  mode.low = 3.0e38f;
  // (no bound by the mean, where the step before was no average; a select: this is in front of every step)
  const float slack = strict & (step >= 2) ? 1.f : 3.0e38f;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    // this side's sums: weights of its own rows (w) and of the others' (k)
    const float dgh = e[4 * (s ^ 1) + 2], dgl = -e[4 * (s ^ 1) + 3];
    const float hi = e[4 * s] + before.w * dgh, lo = -e[4 * s + 1] + before.w * dgl;
    const float wmin = s ? lim.z : lim.x, wmax = s ? lim.w : lim.y, kmin = s ? lim.x : lim.z, kmax = s ? lim.y : lim.w;
    const float up = rho >= 1.f ? -(rho - 1.f) * kmin : (1.f - rho) * mass;
    const float dn = rho >= 1.f ? -(rho - 1.f) * mass : (1.f - rho) * kmin;
    // (linear in the row's own weight, so largest at one end of it)
    const float mean = fmaxf(rho * 0.5f * (mass - wmin) + (wmin - wmax), rho * 0.5f * (mass - wmax)) + slack;
    const float U = fminf(rho * hi, mean) + up - kmax, L = rho * lo + dn + (wmin - wmax) - kmax;
    ok = ok & (U < 3.0e38f) & (L > -3.0e38f);  // (false where anything is not a number)
    most = fmaxf(most, U);
    mode.low = fminf(mode.low, L);
  }
  mode.sweep = ok & fit();
  // Between two steps at one eps a logit rises by no more than the potentials of its two rows do.
  const float rise = kappa * (e[2] + e[6]);
  mode.drift = k.list.x + rise;
  mode.base = k.list.y;
  mode.list = mode.sweep && mode.coarse && k.list.z != 0.f && mode.base + mode.drift <= mode.low - kPairGap;
  // (changes of the potentials shrink from step to step, at first to about a half where a plan is peaked, slowly
  // later: a list that reaches further costs its steps 0.28 us a unit, a new one 320 us, at 50,000 x 64)
  mode.reserve = next.x == now.x ? fminf(16.f + 24.f * __builtin_amdgcn_sqrtf(fmaxf(rise, 0.f)), 256.f) : 0.f;
  return mode;
}

// A row's bias as three pieces, what its part in the cross products of the planes can add to a
// logit (pair_cross), in a column that the matrix product multiplies by zero, and a one for the logits' shift.
__device__ __forceinline__ u32x4 pair_bias(float b, float cross) {
  const _Float16 s1 = (_Float16)4096.f, s2 = (_Float16)1.f, s3 = (_Float16)0.000244140625f;
  const _Float16 p1 = (_Float16)(b * 0.000244140625f);
  const float r1 = __builtin_fmaf(-4096.f, (float)p1, b);
  const _Float16 p2 = (_Float16)r1;
  const _Float16 p3 = (_Float16)((r1 - (float)p2) * 4096.f);
  u32x4 v;
  v[0] = pack_f16((float)s1, (float)s2);
  v[1] = pack_f16((float)s3, (float)p1);
  v[2] = pack_f16((float)p2, (float)p3);
  v[3] = pack_f16(cross, 1.f);
  return v;
}
// The two cross products of a logit come to at most 2^-10 |x~_i| |y~_j| (|lo| <= 2^-11 |hi|, x~ the rows as
// the planes hold them), so to no more than the sum of 2^-11 |x~_i|^2 and 2^-11 |y~_j|^2.  On top of a row's
// share: what fp32 sums of that size round off, values below fp16's normal range, the rounding to fp16 here.
__device__ __forceinline__ float pair_cross(float kappa, float norm, float reach) {
  return 1.004f * (kappa * norm * 0.0009765625f) + kappa * reach * 9.5367431640625e-07f + 0.25f;
}
__device__ __forceinline__ float pair_cross_of(const u32x4& bias) {
  return (float)__builtin_bit_cast(_Float16, (unsigned short)(bias[3] & 0xffffu));
}
// The same row as an A operand: (b1 b2)(b3 s1)(s2 s3)(0 -shift), nothing in the upper half-wave.
__device__ __forceinline__ u32x4 pair_bias_a(const u32x4& v, int h, float shift) {
  u32x4 r;
  r[0] = __builtin_amdgcn_alignbit(v[2], v[1], 16);
  r[1] = __builtin_amdgcn_alignbit(v[0], v[2], 16);
  r[2] = __builtin_amdgcn_alignbit(v[1], v[0], 16);
  r[3] = pack_f16(0.f, -shift);
  if (h) r = u32x4{0u, 0u, 0u, 0u};
  return r;
}

// (Not to be computed with ahead of the path of the kernel that asks: each fills the registers.)
__device__ __forceinline__ int pair_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
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
    lane = pair_lane();
    gsrc = planes + ((size_t)batch * blocks + j_begin / 32) * (2 * KK * 64);
    bsrc = bias + (size_t)batch * blocks * 32 + j_begin;
  }
  __device__ __forceinline__ void stage(int tile, int buf) const {
#pragma unroll
    for (int c = 0; c < PIECES / 4; ++c)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(gsrc + (size_t)tile * (PIECES * 64) + (c * 4 + wave) * 64 + lane),
          (__attribute__((address_space(3))) void*)(&lds[buf * BUF + (c * 4 + wave) * 64]), 16, 0, 0);
    // (every wavefront moves the bias piece, so that all count the same loads)
    const auto* src = (const __attribute__((address_space(1))) void*)(bsrc + (size_t)tile * 64 + lane);
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
__device__ __forceinline__ void pair_item_two_sided(const PairArgs& a, int batch, const PairProblem& pr, int prob, int step, int it,
                                                    u32x4* lds) {
  using S = PairStream<DP, true>;
  constexpr int KK = DP / 16, NM = S::NM;
  const int side = it >= pr.two_first ? 1 : 0;  // the streamed rows' own half-update
  if (side) it -= pr.two_first;
  const int n_k = side ? pr.n_st : pr.n_str, n_q = side ? pr.n_str : pr.n_st;
  const int groups = (n_q + 255) / 256, chunk = it / groups, group = it % groups;
  const int kblocks = side ? pr.st_blocks : pr.str_blocks, qblocks = side ? pr.str_blocks : pr.st_blocks;
  const int lane = pair_lane(), li = lane & 31, h = lane >> 5;
  const int j_begin = chunk * pr.chunk, j_end = min(n_k, j_begin + pr.chunk);
  const int ntiles = (j_end - j_begin + 63) / 64;
  const float4 coef = pair_coef(a, batch, prob, step);
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

// The key that accumulator register r of half-wave h belongs to, in the sub-tile whose first key is `first`; -1
// behind the last one.  There the bias is kPairFar, and so is that of real keys whose potential or weight is not a
// number or off every scale (one weight of infinity makes all of its side's such), so the padding
// may hold a row's largest logit: pair_merge_kernel reads the point of the key that is kept.
constexpr int pair_key_of(int first, int r, int h, int keys) {
  const int key = first + 8 * (r >> 2) + 4 * h + (r & 3);
  return key < keys ? key : -1;
}
constexpr bool pair_keys_end_at_the_last_row() {
  for (int keys = 1; keys <= 130; ++keys)
    for (int first = 0; first < (keys + 63) / 64 * 64; first += 32) {
      int seen = 0;
      for (int e = 0; e < 32; ++e) {
        const int key = pair_key_of(first, e >> 1, e & 1, keys);
        if (key >= keys || key < -1 || (key >= 0 && key < first)) return false;
        seen += key >= 0;
      }
      const int left = keys - first;
      if (seen != (left < 0 ? 0 : left > 32 ? 32 : left)) return false;
    }
  return true;
}
static_assert(pair_keys_end_at_the_last_row(), "no key behind the last row, and every other one");

// A work item with running maxima in a step in which most units are empty: as pair_item_two_sided, but
// a unit ends at its hi * hi products where these, the key bias and the bound on the cross products stay
// kPairGap base-2 units below a lower bound on the logarithm of every row's sum.  That bound is the
// larger of two: the last step's sum, less what the potentials of the keys may have fallen by (with eps' <
// eps and rho = eps / eps', power means give rho times the old logarithm less (rho - 1) log2 of the
// weights' sum, which counts them from the largest), and the row's logit at the key that held its
// largest when a step last saw it (pair_merge_kernel keeps the two points' inner product).  The running
// maximum starts there, so that every larger logit that is found raises the line.  A lane holds
// one query row and 16 keys, the key's bias and its share of the bound ride in the matrix product.
template <int DP>
__device__ __forceinline__ unsigned pair_item_two_coarse(const PairArgs& a, int batch, const PairProblem& pr, int prob,
                                                         int step, const PairMode& mode, int it, u32x4* lds) {
  using S = PairStream<DP, false>;
  constexpr int KK = DP / 16;
  const int side = it >= pr.two_first ? 1 : 0;  // the streamed rows' own half-update
  unsigned long long* put = pr.two_list + ((size_t)batch * pr.two_items + it) * (4 * kPairListWords);
  if (side) it -= pr.two_first;
  const PairSide& sd = a.side[prob == 0 ? side : 1 + prob];
  const int n_k = side ? pr.n_st : pr.n_str, n_q = side ? pr.n_str : pr.n_st;
  const int groups = (n_q + 255) / 256, chunk = it / groups, group = it % groups;
  const int kblocks = side ? pr.st_blocks : pr.str_blocks, qblocks = side ? pr.str_blocks : pr.st_blocks;
  const int lane = pair_lane(), li = lane & 31, h = lane >> 5;
  const int j_begin = chunk * pr.chunk, j_end = min(n_k, j_begin + pr.chunk);
  const int ntiles = (j_end - j_begin + 63) / 64;
  const float4 coef = pair_coef(a, batch, prob, step);
  const float* kbias = (side ? pr.st_bias32 : pr.str_bias32) + (size_t)batch * kblocks * 32;
  S ks;
  ks.begin(lds, side ? pr.st_planes : pr.str_planes, side ? pr.st_bias : pr.str_bias, kblocks, batch, j_begin);
  const int blk0 = group * 8 + ks.wave * 2;
  ks.stage(0, 0);
  ks.stage(1, 1);
  ks.stage(2, 2);
  u32x4 x[2][2][KK];
  pair_load_rows(x, (side ? pr.str_planes : pr.st_planes) + ((size_t)batch * qblocks + blk0) * (2 * KK * 64), lane);
  float m[2], s[2], off[2];  // a unit goes on where a logit exceeds m - off
  int best[2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const int row = (blk0 + rb) * 32 + li;
    const size_t at = (size_t)batch * n_q + min(row, n_q - 1);
    const int key = sd.key[at];
    const float sum2 = sd.sum2[at], dot = sd.dot[at];
    const float cross = pair_cross_of((side ? pr.str_bias : pr.st_bias)[((size_t)batch * qblocks + blk0 + rb) * 32 + li]);
    const float there = __builtin_fmaf(coef.y, dot, kbias[max(key, 0)]) - 0.5f - 9.5367431640625e-07f * coef.w * a.reach[batch].z;
    float low = mode.rho * sum2 - (mode.rho - 1.f) * __log2f((float)n_k) + fminf(mode.least[side], 0.f) - 0.5f;
    low = fmaxf(fmaxf(low, key >= 0 ? there : -3.0e38f), 0.5f * kNegBig);  // (also where it is not a number)
    m[rb] = low;
    s[rb] = 0.f;
    best[rb] = -1;
    off[rb] = row < n_q ? kPairGap + cross : -3.0e38f;
  }
  const unsigned one = 0x3c00u, s1 = 0x6c00u, s2 = 0x3c00u, s3 = 0x0c00u;  // fp16 1, 2^12, 1, 2^-12
  // the key's bias with its share of the bound, and without
  u32x4 qb = {0u, s1 << 16, s2 | s3 << 16, one}, qexact = {0u, s1 << 16, s2 | s3 << 16, 0u};
  if (h) qb = qexact = u32x4{0u, 0u, 0u, 0u};
  u32x4 y[KK], yb;
  f32x16 acc[2][2];  // [parity of the sub-tile][row block]
  unsigned long long list[2][2] = {{0ull, 0ull}, {0ull, 0ull}};  // [row block][half of the sub-tiles]
  auto read_key = [&](int k, int buf, int js) {
    if (k < KK) y[k] = S::read(&lds[buf * S::BUF + (js * (2 * KK) + k) * 64 + lane]);
    else yb = S::read(&lds[buf * S::BUF + S::PIECES * 64 + js * 32 + li]);
  };
  auto wait_reads = [&]() {
    S::fence();
    ks.template wait_lds<0>();
    S::fence();
  };
  auto run = [&](int to, int buf, int js, bool test, float (&mx)[2]) {
#pragma unroll
    for (int k = 0; k <= KK; ++k) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        f32x16& c = acc[to][rb];
        if (k == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) c[r] = 0.f;
        }
        c = k < KK ? small_mfma(y[k < KK ? k : 0], x[rb][0][k < KK ? k : 0], c) : small_mfma(yb, qb, c);
        if (rb == 1) read_key(k, buf, js);
        if (test) {
          constexpr int N = 2 * (KK + 1);
          const int i = 2 * k + rb, v0 = i * 32 / N, v1 = (i + 1) * 32 / N;
#pragma unroll
          for (int v = v0; v < v1; ++v) {
            const float l = acc[to ^ 1][v >> 4][v & 15];
            mx[v >> 4] = (v & 15) == 0 ? l : fmaxf(mx[v >> 4], l);
          }
        }
        S::fence();
      }
    }
  };
  auto finish = [&](int of, int sub, int buf, const float (&mx)[2]) {
    const int js = sub & 1;
    const bool on0 = wave_any(mx[0] > m[0] - off[0]), on1 = wave_any(mx[1] > m[1] - off[1]);
    if (!(on0 || on1)) return;
    const unsigned long long bit = 1ull << (sub & 63);
    list[0][0] |= on0 && sub < 64 ? bit : 0ull;
    list[0][1] |= on0 && sub >= 64 ? bit : 0ull;
    list[1][0] |= on1 && sub < 64 ? bit : 0ull;
    list[1][1] |= on1 && sub >= 64 ? bit : 0ull;
    u32x4 z[2][KK], zb;
#pragma unroll
    for (int q = 1; q >= 0; --q)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) z[q][kk] = S::read(&lds[buf * S::BUF + (js * (2 * KK) + q * KK + kk) * 64 + lane]);
    zb = S::read(&lds[buf * S::BUF + S::PIECES * 64 + js * 32 + li]);
    wait_reads();
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      if (rb ? !on1 : !on0) continue;
      // (anew, from the lowest weight to the bias: fewest roundings at the size of the whole)
      f32x16 c;
#pragma unroll
      for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) c = small_mfma(z[1][kk], x[rb][0][kk], c);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) c = small_mfma(z[0][kk], x[rb][1][kk], c);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) c = small_mfma(z[0][kk], x[rb][0][kk], c);
      c = small_mfma(zb, qexact, c);
      const float top = small_max16(c[0], c);
      if (wave_any(top > m[rb])) {
        if (top > m[rb]) {
          s[rb] *= fast_exp2(m[rb] - top);
          m[rb] = top;
          int at = 0;
#pragma unroll
          for (int r = 1; r < 16; ++r) at = c[r] == top ? r : at;
          best[rb] = pair_key_of(j_begin + sub * 32, at, h, n_k);
        }
      }
      float p0 = 0.f, p1 = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        p0 += fast_exp2(c[r] - m[rb]);
        p1 += fast_exp2(c[r + 1] - m[rb]);
      }
      s[rb] += p0 + p1;
    }
  };
  S::fence();
  S::wait_all();
  S::barrier();
  float mx[2];
#pragma unroll
  for (int k = 0; k <= KK; ++k) read_key(k, 0, 0);
  wait_reads();
  run(0, 0, 1, false, mx);
  wait_reads();
  for (int t = 0; t < ntiles; ++t) {
    const int cur = t & 3, nxt = (t + 1) & 3;
    // tile t + 1 has landed, and every wavefront is through with tile t - 1
    S::fence();
    S::wait_tile();
    S::fence();
    S::barrier();
    ks.stage(t + 3, (t + 3) & 3);
    S::fence();
    run(1, nxt, 0, true, mx);
    wait_reads();
    finish(0, 2 * t, cur, mx);
    S::fence();
    run(0, nxt, 1, true, mx);
    wait_reads();
    finish(1, 2 * t + 1, cur, mx);
  }
  S::wait_all();
  __syncthreads();  // (the next item fills the same buffers)
  const size_t to = ((size_t)batch * ((n_k + pr.chunk - 1) / pr.chunk) + chunk) * n_q;
  float2* out = (side ? pr.str_ms : pr.st_ms) + to;
  int* keys = (side ? pr.str_best : pr.st_best) + to;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float mo = xor32(m[rb]), so = xor32(s[rb]);
    const int bo = __shfl_xor(best[rb], 32, 64);
    const float M = fmaxf(m[rb], mo);
    const float sum = s[rb] * fast_exp2(m[rb] - M) + so * fast_exp2(mo - M);
    const int row = (blk0 + rb) * 32 + li;
    if (h == 0 && row < n_q) {
      out[row] = make_float2(M, sum);
      keys[row] = bo >= 0 && (mo > m[rb] || best[rb] < 0) ? bo : best[rb];
    }
  }
  if (lane < kPairListWords)
    put[ks.wave * kPairListWords + lane] = lane < 2 ? (lane ? list[0][1] : list[0][0]) : (lane == 3 ? list[1][1] : list[1][0]);
  return __popcll(list[0][0]) + __popcll(list[0][1]) + __popcll(list[1][0]) + __popcll(list[1][1]);
}

// What a work item of the one-sweep forms is: 256 stationary rows against a chunk of streamed ones.
struct PairItem {
  int prob, index, chunk, group, j_begin, j_end;
};
typedef int PairWord __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) PairWord* PairWork;  // (read by scalar loads)
__device__ __forceinline__ PairItem pair_item(PairWord w) {
  PairItem t;
  t.prob = w[0] < 0 ? -1 : w[0] & 3;
  t.index = w[0] >> 2;
  t.chunk = w[1] & 65535;
  t.group = w[1] >> 16;
  t.j_begin = w[2];
  t.j_end = w[3];
  return t;
}

// The work items, once per solve.  XCD-aware: workgroups are dealt round-robin to the 8 XCDs; XCD x takes
// the x-th eighth of every problem's items, whose order is chunk by chunk: what runs on an XCD at one
// time shares a chunk in its L2.
__device__ void pair_write_work(const PairArgs& a, int at) {
  if (at >= 8 * a.per_xcd) return;
  const int xcd = at / a.per_xcd;
  int i = at - xcd * a.per_xcd, p = a.first_prob;
  int4 w = make_int4(-1, 0, 0, 0);
  for (; p < a.nprob; ++p) {
    const int per = (a.prob[p].n_items + 7) / 8;
    if (i < per) break;
    i -= per;
  }
  const PairProblem& pr = a.prob[p];
  const int index = xcd * ((pr.n_items + 7) / 8) + i;
  if (index < pr.n_items) {
    int chunk = index / pr.groups, group = index % pr.groups;
    if (pr.self) {
      chunk = 0;
      group = index;
      for (;;) {
        const int g = self_groups_of_chunk(chunk, pr.chunk, pr.n_str, pr.groups);
        if (group < g) break;
        group -= g;
        ++chunk;
      }
    }
    w.x = p + 4 * index;
    w.y = chunk + 65536 * group;
    w.z = pr.self ? max(chunk * pr.chunk, group * 256) : chunk * pr.chunk;
    w.w = min(pr.n_str, (chunk + 1) * pr.chunk);
  }
  a.work[at] = w;
}

// The streamed rows' sums on their way from the four wavefronts to memory.
struct PairCols {
  unsigned at;  // LDS address of [tile parity][wavefront][half-wave][row]
  int wave, lane;
  __device__ __forceinline__ void put(int tile, int js, float v) const {
    asm volatile("ds_write_b32 %0, %1"
                 :
                 : "v"(at + 4 * ((((tile & 1) * 4 + wave) * 2 + (lane >> 5)) * 64 + js * 32 + (lane & 31))), "v"(v)
                 : "memory");
  }
  // a tile's sums over the wavefronts, in a fixed order; `left`: streamed rows from its first to the chunk's end
  __device__ __forceinline__ void flush(int tile, float* out, int left) const {
    float c[8];
#pragma unroll
    for (int w = 0; w < 8; ++w)
      asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(c[w]) : "v"(at + 4 * ((tile & 1) * 512 + lane)), "n"(w * 256)
                   : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
    float v = c[0] + c[1];
#pragma unroll
    for (int w = 1; w < 4; ++w) v += c[2 * w] + c[2 * w + 1];
    if (lane < left) out[lane] = v;
  }
};

// The stationary rows' sums over the lanes of a wavefront.
__device__ __forceinline__ void pair_put_rows(const PairProblem& pr, int batch, int chunk, int blk0, float (&st)[2][16],
                                              int lane) {
  const int li = lane & 31, h = lane >> 5;
  float* rowp = pr.st_part + ((size_t)batch * pr.chunks + chunk) * pr.n_st;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    float v = colsum_all(st[rb], li);
    v += __shfl_xor(v, 16, 64);
    const int row = (blk0 + rb) * 32 + colsum_key(li & 15, h);
    if (li < 16 && row < pr.n_st) rowp[row] = v;
  }
}

// Work items of steps in which most units (32 x 32 logits) are empty, from index `at` of the workgroup's
// on, as long as they are such; returns the index of the first that was not taken.
//
// A unit's hi * hi products and biases alone (KK + 1 of 3 KK + 1 MFMAs, no exponential) say that every
// logit of it lies kPairGap base-2 units below every sum of the step (pair_mode's lower bound on them):
// it ends there unless hi * hi + biases + the bound on the cross products reaches that line.  What
// is left out is below 2^-28 of any sum even with 65,536 terms.  The products of a sub-tile's two
// units go to the matrix pipe while the units of the sub-tile before are tested between them in program order;
// those that go on then take all of their products and their exponentials, with the streamed
// operands read again from LDS.  No accumulator and no LDS read on its way crosses the branch.
//
// The tiles of all items run through one ring of four buffers, three ahead, across the ends of items:
// an item of nine tiles spent 5 us on its way to the first product and 10 in its tiles (10,000 x 64).
template <int DP>
__device__ __forceinline__ int pair_run_coarse(const PairArgs& a, int batch, PairWork work, int at, int stride,
                                               int count, unsigned which, const PairMode* modes, unsigned* went,
                                               u32x4* lds, float* lds_col) {
  using S = PairStream<DP, false>;
  constexpr int KK = DP / 16;
  const int lane = pair_lane(), li = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  PairCols cols{(unsigned)(size_t)(const __attribute__((address_space(3))) float*)lds_col, wave, lane};
  S ks;
  // ---- the tiles to come ----
  int s_at = at - stride, s_tile = 0, s_left = 0;
  PairWord ahead = work[at];
  bool dry = false;
  auto stage = [&](int buf) {
    if (s_left == 0 && !dry) {
      s_at += stride;
      const PairItem n = pair_item(ahead);
      dry = s_at >= count || n.prob < 0 || !((which >> n.prob) & 1);
      s_tile = 0;
      if (!dry) {
        const PairProblem& pr = a.prob[n.prob];
        ks.begin(lds, pr.str_planes, pr.str_bias, pr.str_blocks, batch, n.j_begin);
        s_left = (n.j_end - n.j_begin + 63) / 64;
        ahead = work[min(s_at + stride, count - 1)];
      }
    }
    ks.stage(s_tile, buf);  // (behind the last item: a tile again, for nobody)
    if (!dry) {
      ++s_tile;
      --s_left;
    }
  };
  PairItem t = pair_item(ahead);
  stage(0);
  stage(1);

  u32x4 xa[2][2][KK], xb[2];
  float on_at[2];  // a unit goes on where a logit and the streamed row's share of the bound exceed that
  float far = 0.f;
  auto load_rows = [&]() {
    const PairProblem& pr = a.prob[t.prob];
    const int blk0 = t.group * 8 + wave * 2;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) xb[rb] = pr.st_bias[((size_t)batch * pr.st_blocks + blk0 + rb) * 32 + li];
    pair_load_rows(xa, pr.st_planes + ((size_t)batch * pr.st_blocks + blk0) * (2 * KK * 64), lane);
  };
  auto derive_rows = [&]() {
    const float shift = modes[t.prob].shift;
    far = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
              __builtin_bit_cast(int, modes[t.prob].low - shift - modes[t.prob].reserve))) - kPairGap;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      float c = pair_cross_of(xb[rb]);
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) c = fmaxf(c, __shfl_xor(c, o, 64));
      on_at[rb] = far - c;
      xb[rb] = pair_bias_a(xb[rb], h, shift);
    }
  };
  load_rows();

  u32x4 y[KK], yb;       // high plane and bias of the sub-tile to be multiplied
  f32x16 acc[2][2];      // [parity of the sub-tile][row block]
  float bound[2];        // the streamed rows' share of the bound
  float st[2][16];       // sums of the stationary rows, over the streamed rows this lane sees
  auto read_key = [&](int k, int buf, int js) {
    if (k < KK) y[k] = S::read(&lds[buf * S::BUF + (js * (2 * KK) + k) * 64 + lane]);
    else yb = S::read(&lds[buf * S::BUF + S::PIECES * 64 + js * 32 + li]);
  };
  auto wait_reads = [&]() {
    S::fence();
    ks.template wait_lds<0>();
    S::fence();
  };
  // products of the sub-tile in y, parity `to`; the maxima of the units of the other parity between
  // them; y is read anew from (buf, js) behind the last MFMA that uses a piece of it
  auto step = [&](int to, int buf, int js, bool test, float (&mx)[2]) {
#pragma unroll
    for (int k = 0; k <= KK; ++k) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        f32x16& c = acc[to][rb];
        if (k == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) c[r] = 0.f;
        }
        c = k < KK ? small_mfma(xa[rb][0][k < KK ? k : 0], y[k < KK ? k : 0], c) : small_mfma(xb[rb], yb, c);
        if (k == KK && rb == 1) bound[to] = pair_cross_of(yb);
        if (rb == 1) read_key(k, buf, js);
        if (test) {
          constexpr int N = 2 * (KK + 1);
          const int i = 2 * k + rb, v0 = i * 32 / N, v1 = (i + 1) * 32 / N;
#pragma unroll
          for (int v = v0; v < v1; ++v) {
            const float l = acc[to ^ 1][v >> 4][v & 15];
            mx[v >> 4] = (v & 15) == 0 ? l : fmaxf(mx[v >> 4], l);
          }
        }
        S::fence();
      }
    }
  };
  // the units of parity `of` that go on, of sub-tile js in buffer buf; returns the streamed rows' sums
  unsigned long long list[2][2];  // [row block][half of the sub-tiles]
  auto finish = [&](int of, int sub, int buf, const float (&mx)[2]) {
    float ps0 = 0.f, ps1 = 0.f;
    const int js = sub & 1;
    const bool on0 = wave_any(mx[0] + bound[of] > on_at[0]), on1 = wave_any(mx[1] + bound[of] > on_at[1]);
    if (on0 || on1) {
      u32x4 z[2][KK], zb;
#pragma unroll
      for (int q = 1; q >= 0; --q)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) z[q][kk] = S::read(&lds[buf * S::BUF + (js * (2 * KK) + q * KK + kk) * 64 + lane]);
      zb = S::read(&lds[buf * S::BUF + S::PIECES * 64 + js * 32 + li]);
      wait_reads();
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        if (rb ? !on1 : !on0) continue;
        // (anew, from the lowest weight on, to the same bits as the plain form and the gradient)
        f32x16 c;
#pragma unroll
        for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][0][kk], z[1][kk], c);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][1][kk], z[0][kk], c);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][0][kk], z[0][kk], c);
        c = small_mfma(xb[rb], zb, c);
        // (its logits themselves, which the bound is far above, say whether it is kept)
        if (wave_any(small_max16(c[0], c) > far - 0.5f)) {
          const unsigned long long bit = 1ull << (sub & 63);
          list[rb][0] |= sub < 64 ? bit : 0ull;
          list[rb][1] |= sub >= 64 ? bit : 0ull;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = fast_exp2(c[r]);
          st[rb][r] += e;
          if (r & 1) ps1 += e; else ps0 += e;
        }
      }
    }
    return ps0 + ps1;
  };

  S::fence();
  S::wait_tile();  // (the first tile; the second may be on its way)
  S::fence();
  S::barrier();
  stage(2);
  float* out = nullptr;  // where the sums of the tile before go
  int left = 0;
  for (int g = 0;;) {
    const PairProblem& pr = a.prob[t.prob];
    const int blk0 = t.group * 8 + wave * 2;
    derive_rows();
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[rb][r] = 0.f;
    list[0][0] = list[0][1] = list[1][0] = list[1][1] = 0ull;
    float mx[2];
#pragma unroll
    for (int k = 0; k <= KK; ++k) read_key(k, g & 3, 0);
    wait_reads();
    step(0, g & 3, 1, false, mx);
    wait_reads();
    const PairWord following = work[min(at + stride, count - 1)];
    float* colp = pr.str_part + ((size_t)batch * pr.groups + t.group) * pr.n_str + t.j_begin;
    int sub = 0;
    for (int n = t.j_end - t.j_begin; n > 0; n -= 64, ++g, sub += 2) {
      const int cur = g & 3, nxt = (g + 1) & 3;
      // tile g + 1 has landed, and every wavefront is through with tile g - 1 and its sums
      S::fence();
      S::wait_tile();
      S::fence();
      S::barrier();
      stage((g + 3) & 3);
      if (left > 0 && wave == (g & 3)) cols.flush(g - 1, out, left);
      out = colp;
      left = n;
      colp += 64;
      S::fence();
      step(1, nxt, 0, true, mx);
      wait_reads();
      cols.put(g, 0, finish(0, sub, cur, mx));
      S::fence();
      step(0, nxt, 1, true, mx);
      wait_reads();
      cols.put(g, 1, finish(1, sub + 1, cur, mx));
    }
    {
      const unsigned went_on = __popcll(list[0][0]) + __popcll(list[0][1]) + __popcll(list[1][0]) + __popcll(list[1][1]);
      if (lane == 0 && went_on) atomicAdd(&went[t.prob], went_on);
      unsigned long long* put = pr.list + (((size_t)batch * pr.n_items + t.index) * 4 + wave) * kPairListWords;
      if (lane < kPairListWords) put[lane] = lane < 2 ? (lane ? list[0][1] : list[0][0]) : (lane == 3 ? list[1][1] : list[1][0]);
    }
    // (the next item's rows are on their way while the sums of these cross the lanes)
    const PairItem done = t;
    at += stride;
    t = pair_item(following);
    const bool more = at < count && t.prob >= 0 && ((which >> t.prob) & 1);
    if (more) load_rows();
    S::fence();
    pair_put_rows(pr, batch, done.chunk, blk0, st, lane);
    if (!more) {
      S::wait_all();
      __syncthreads();
      if (wave == 0) cols.flush(g - 1, out, left);
      return at;
    }
  }
}

// Work items of steps whose lists hold, from index `at` of the workgroup's on, as long as they are such:
// only the units on the lists are visited, without a test, with the streamed operands straight from global
// memory, one sub-tile ahead.  The sub-tiles on the lists of an item's four blocks of 64 rows are shared
// out evenly between the wavefronts (some rows have near keys everywhere: with a block to each a settled
// launch at 50,000 x 64 took 103 us, with even shares 80), so a wavefront may finish one block's list and
// begin the next one's.  Both kinds of sums lie in LDS until the item is done: of streamed rows per block, of stationary
// rows per block and wavefront, each added in a fixed order.
template <int DP>
__device__ __forceinline__ int pair_run_list(const PairArgs& a, int batch, PairWork work, int at, int stride,
                                             int count, unsigned which, const PairMode* modes, float* cols, float* rows) {
  constexpr int KK = DP / 16;
  typedef unsigned long long u64;
  struct Keys {
    u32x4 p[2][KK], b;
  };
  const int lane = pair_lane(), li = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // lane (4 block + word) % 16: one of the item's words
  auto words_of = [&](const PairItem& t) {
    const PairProblem& pr = a.prob[t.prob];
    return pr.list[((size_t)batch * pr.n_items + t.index) * (4 * kPairListWords) + (lane & 15)];
  };
  PairItem t = pair_item(work[at]);
  PairWord ahead = work[min(at + stride, count - 1)];
  u64 w = words_of(t);
  // (what lies there may be the other forms' tiles; each item leaves zeros again)
  for (int i = threadIdx.x; i < 4 * a.prob[t.prob].chunk; i += 256) cols[i] = 0.f;
  __syncthreads();
  for (;;) {
    const PairProblem& pr = a.prob[t.prob];
    const PairItem now = t;
    const int chunk = pr.chunk, len = now.j_end - now.j_begin;
    auto word = [&](u64 v, int i) {
      return (u64)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, i) |
             (u64)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), i) << 32;
    };
    const u64 mine = w;
    at += stride;
    t = pair_item(ahead);
    const bool more = at < count && t.prob >= 0 && ((which >> t.prob) & 1);
    if (more) {
      ahead = work[min(at + stride, count - 1)];
      w = words_of(t);
    }
    int total = 0;
#pragma unroll
    for (int o = 0; o < 4; ++o)
      total += __popcll(word(mine, 4 * o) | word(mine, 4 * o + 2)) + __popcll(word(mine, 4 * o + 1) | word(mine, 4 * o + 3));
    const int from = wave * total / 4, to = (wave + 1) * total / 4;
    int before = 0;
#pragma unroll 1
    for (int o = 0; o < 4; ++o) {
      const u64 on00 = word(mine, 4 * o), on01 = word(mine, 4 * o + 1), on10 = word(mine, 4 * o + 2), on11 = word(mine, 4 * o + 3);
      u64 left0 = on00 | on10, left1 = on01 | on11;
      const int here = __popcll(left0) + __popcll(left1);
      int skip = max(from - before, 0), left = min(to - before, here) - skip;
      before += here;
      float* sum = rows + (o * 4 + wave) * 64;
      if (left <= 0) {
        sum[lane] = 0.f;
        continue;
      }
      float st[2][16];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[rb][r] = 0.f;
      const int blk0 = now.group * 8 + o * 2;
      u32x4 xa[2][2][KK], xb[2];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
        xb[rb] = pair_bias_a(pr.st_bias[((size_t)batch * pr.st_blocks + blk0 + rb) * 32 + li], h, modes[now.prob].shift);
      pair_load_rows(xa, pr.st_planes + ((size_t)batch * pr.st_blocks + blk0) * (2 * KK * 64), lane);
      const u32x4* planes = pr.str_planes + ((size_t)batch * pr.str_blocks + now.j_begin / 32) * (2 * KK * 64);
      const u32x4* bias = pr.str_bias + (size_t)batch * pr.str_blocks * 32 + now.j_begin;
      const int low = __popcll(left0);
      for (int k = min(skip, low); k > 0; --k) left0 &= left0 - 1;
      for (int k = skip - low; k > 0; --k) left1 &= left1 - 1;
      auto take = [&]() {  // the next sub-tile, -1 behind the last
        int sub = -1;
        if (left > 0) {
          if (left0) {
            sub = __builtin_ctzll(left0);
            left0 &= left0 - 1;
          } else {
            sub = 64 + __builtin_ctzll(left1);
            left1 &= left1 - 1;
          }
          --left;
        }
        return sub;
      };
      auto load = [&](Keys& k, int sub) {
        const u32x4* src = planes + (size_t)max(sub, 0) * (2 * KK * 64) + lane;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int kk = 0; kk < KK; ++kk) k.p[q][kk] = src[(q * KK + kk) * 64];
        k.b = bias[max(sub, 0) * 32 + li];
        __builtin_amdgcn_sched_barrier(0);
      };
      auto run = [&](const Keys& k, int sub) {
        const u64 bit = 1ull << (sub & 63);
        float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          if (!((sub < 64 ? (rb ? on10 : on00) : (rb ? on11 : on01)) & bit)) continue;
          f32x16 c;
#pragma unroll
          for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll
          for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][0][kk], k.p[1][kk], c);
#pragma unroll
          for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][1][kk], k.p[0][kk], c);
#pragma unroll
          for (int kk = 0; kk < KK; ++kk) c = small_mfma(xa[rb][0][kk], k.p[0][kk], c);
          c = small_mfma(xb[rb], k.b, c);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float e = fast_exp2(c[r]);
            st[rb][r] += e;
            if (r & 1) ps1 += e; else ps0 += e;
          }
        }
        float ps = ps0 + ps1;
        ps += xor32(ps);
        if (h == 0) cols[o * chunk + sub * 32 + li] = ps;
      };
      Keys k0, k1;
      int s0 = take();
      load(k0, s0);
      for (;;) {
        const int s1 = take();
        load(k1, s1);
        run(k0, s0);
        if (s1 < 0) break;
        s0 = take();
        load(k0, s0);
        run(k1, s1);
        if (s0 < 0) break;
      }
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        float v = colsum_all(st[rb], li);
        v += __shfl_xor(v, 16, 64);
        if (li < 16) sum[rb * 32 + colsum_key(li, h)] = v;
      }
    }
    __syncthreads();
    {
      const float* sum = rows + (threadIdx.x >> 6) * 256 + lane;
      const int row = now.group * 256 + threadIdx.x;
      if (row < pr.n_st)
        pr.st_part[((size_t)batch * pr.chunks + now.chunk) * pr.n_st + row] = (sum[0] + sum[64]) + (sum[128] + sum[192]);
    }
    float* out = pr.str_part + ((size_t)batch * pr.groups + now.group) * pr.n_str + now.j_begin;
    for (int j = threadIdx.x; j < len; j += 256) {
      float v = cols[j];
      cols[j] = 0.f;
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        v += cols[k * chunk + j];
        cols[k * chunk + j] = 0.f;
      }
      out[j] = v;
    }
    __syncthreads();
    if (!more) return at;
  }
}

// A work item of a step that takes both sides from one sweep, every logit of it: the exponentials
// of one 32 x 32 unit sit between the MFMAs of the next in program order.
template <int DP>
__device__ __forceinline__ void pair_item_plain(const PairProblem& pr, int batch, const PairItem& it, const PairMode& mode,
                                                unsigned* went, u32x4* lds, float* lds_col) {
  using S = PairStream<DP, false>;
  constexpr int KK = DP / 16, NM = S::NM;
  const int lane = pair_lane(), li = lane & 31, h = lane >> 5;
  const int j_begin = it.j_begin, j_end = it.j_end, ntiles = (j_end - j_begin + 63) / 64;
  S ks;
  ks.begin(lds, pr.str_planes, pr.str_bias, pr.str_blocks, batch, j_begin);
  const int wave = ks.wave;
  const PairCols cols{(unsigned)(size_t)(const __attribute__((address_space(3))) float*)lds_col, wave, lane};

  // ---- stationary operands ----
  const int blk0 = it.group * 8 + wave * 2;
  u32x4 xa[2][2][KK], xb[2];
  pair_load_rows(xa, pr.st_planes + ((size_t)batch * pr.st_blocks + blk0) * (2 * KK * 64), lane);
  float cross = 0.f;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const u32x4 v = pr.st_bias[((size_t)batch * pr.st_blocks + blk0 + rb) * 32 + li];
    xb[rb] = pair_bias_a(v, h, mode.shift);
    cross = pair_cross_of(v);
  }
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
  float* colp = pr.str_part + ((size_t)batch * pr.groups + it.group) * pr.n_str + j_begin;
  auto flush = [&](int tile) { cols.flush(tile, colp + tile * 64, j_end - j_begin - tile * 64); };

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
            cols.put(t, 0, pend);
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
            if (t >= 1) cols.put(t - 1, 1, v);
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
  float mx = R1[0];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    mx = fmaxf(mx, R1[r]);
    const float e = fast_exp2(R1[r]);
    st[1][r] += e;
    if (r & 1) ps1 += e; else ps0 += e;
  }
  cols.put(ntiles - 1, 1, ps0 + ps1);
  {
    // this unit says for all of the wavefront's whether the coarse test of the next step would end them
    // (its logits and cross products are about `ratio` times these, the streamed rows' share of the
    // latter about that of the others)
    if (went != nullptr && wave_any((mx + mode.shift + 2.0f * cross) * mode.ratio > mode.low - mode.reserve - kPairGap) && lane == 0) atomicAdd(went, 4u * (unsigned)ntiles);
  }
  S::wait_all();  // (also what was fetched past the chunk)
  __syncthreads();
  if (wave == 0) flush(ntiles - 1);
  pair_put_rows(pr, batch, it.chunk, blk0, st, lane);
}

// One step.  Grid (workgroups of an item of the batch, items of the batch).  A workgroup of four
// wavefronts owns 256 stationary rows (two blocks of 32 per wavefront, operands in registers) and
// streams a chunk of the other matrix; it takes every (workgroups)-th of its XCD's work items.
constexpr int kPairGrid = 512;  // two workgroups per CU
template <int DP, bool SKIP>
__global__ __launch_bounds__(256, 2) void pair_sweep_kernel(PairArgsPtr args, int step) {
  const PairArgs& a = *(const PairArgs*)args;
  using S = PairStream<DP, false>;
  // (four tiles, or the sums of a chunk's streamed rows per wavefront)
  constexpr int kWords = !SKIP ? 3 * S::BUF : (4 * S::BUF > kPairMostTiles * 64 ? 4 * S::BUF : kPairMostTiles * 64);
  __shared__ __attribute__((aligned(16))) u32x4 lds[kWords];
  __shared__ float lds_col[2][4][2][64];        // [tile parity][wavefront][half-wave][row]
  __shared__ PairMode modes[3];
  __shared__ unsigned went[3];                  // units that went on
  __shared__ int next_item[2];
  __shared__ __attribute__((aligned(16))) unsigned mode_bits[4];

  const int batch = blockIdx.y, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, mine = blockIdx.x >> 3, stride = gridDim.x >> 3, count = a.per_xcd;
  const PairWork work = (PairWork)(a.work + xcd * count);
  PairWord word = work[mine];
  // The modes: of a single problem by every wavefront for itself, without a barrier (what they write to LDS for
  // later is the same), of three by one wavefront each.
  const bool single = a.nprob - a.first_prob == 1;
  const int own = single ? a.first_prob : max(min(wave, a.nprob - 1), a.first_prob);
  unsigned bits;
  {
    const PairKnown known = pair_known(a, batch, own, step);
    const int entries = a.lens[batch * 3 + own];
    const PairMode m = pair_mode(known, SKIP ? a.prob[own].units : 0.f, SKIP && a.prob[own].ends, a.prob[own].strict, own, step);
    // (where its schedule is shorter nothing is done)
    const bool live = step <= entries + a.extrapolate;
    bits = (live ? 1u : 0u) | (live && m.sweep ? 8u : 0u);
    if (SKIP)
      bits |= (live && m.sweep && m.coarse && !m.list ? 64u : 0u) | (live && m.list ? 512u : 0u) | (m.two ? 4096u : 0u);
    bits <<= own;
    if (lane == 0 && (single || own == wave)) {
      modes[own] = m;
      if (blockIdx.x == 0 && live) *reinterpret_cast<PairMode*>(a.state + ((size_t)batch * 3 + own) * kPairStateWords + kPairModes) = m;
    }
    if (threadIdx.x < 3) went[threadIdx.x] = 0u;
  }
  if (!single) {
    if (lane == 0) mode_bits[wave] = own == wave ? bits : 0u;
    __syncthreads();
    const uint4 all = *reinterpret_cast<const uint4*>(mode_bits);
    bits = all.x | all.y | all.z | all.w;
  }
  bits = __builtin_amdgcn_readfirstlane(bits);
  // (bit p: problem p)
  const unsigned live = bits & 7u, sweep = bits >> 3 & 7u, coarse = bits >> 6 & 7u, list = bits >> 9 & 7u, ends = bits >> 12 & 7u;
  // (items of these forms take long and are all alike: whoever is free takes the next)
  int* taken = reinterpret_cast<int*>(a.state) + (size_t)batch * 3 * kPairStateWords + kPairTaken + ((step % 3) * 8 + xcd) * 32;
  int turn = 0;
  for (unsigned two = live & ~sweep; two; two &= two - 1) {
    const int p = __builtin_ctz(two);
    const PairProblem& pr = a.prob[p];
    const int per = (pr.two_items + 7) / 8, end = min(pr.two_items, (xcd + 1) * per);
    for (int k = xcd * per + mine; k < end; ++turn) {
      if (threadIdx.x == 0) next_item[turn & 1] = xcd * per + stride + atomicAdd(taken + p * kPairStateWords, 1);
      // (with a barrier in them)
      if (SKIP && ((ends >> p) & 1)) {
        const unsigned on = pair_item_two_coarse<DP>(a, batch, pr, p, step, modes[p], k, lds);
        // (both sides of the xy problem count)
        if (lane == 0 && on) atomicAdd(&went[p], pr.self ? on : (on + 1) / 2);
      } else {
        pair_item_two_sided<DP>(a, batch, pr, p, step, k, lds);
      }
      k = __builtin_amdgcn_readfirstlane(next_item[turn & 1]);
    }
  }
  const bool fetch = (coarse | list) == 0 && count > stride;
  for (int i = mine; i < count;) {
    const PairItem t = pair_item(word);
    if (t.prob < 0 || !((live & sweep) >> t.prob & 1)) {
      i += stride;
    } else if (SKIP && ((list >> t.prob) & 1)) {
      i = pair_run_list<DP>(a, batch, work, i, stride, count, list, modes, reinterpret_cast<float*>(lds),
                            &lds_col[0][0][0][0]);
    } else if (SKIP && ((coarse >> t.prob) & 1)) {
      i = pair_run_coarse<DP>(a, batch, work, i, stride, count, coarse, modes, went, lds, &lds_col[0][0][0][0]);
    } else {
      if (fetch && threadIdx.x == 0) next_item[turn & 1] = stride + atomicAdd(taken + a.first_prob * kPairStateWords + 1, 1);
      pair_item_plain<DP>(a.prob[t.prob], batch, t, modes[t.prob], SKIP ? &went[t.prob] : nullptr, lds, &lds_col[0][0][0][0]);
      i = fetch ? __builtin_amdgcn_readfirstlane(next_item[turn & 1]) : i + stride;
      ++turn;
    }
    if (i < count) word = work[i];
  }
  if (!SKIP) return;
  __syncthreads();
  if (threadIdx.x >= a.first_prob && threadIdx.x < a.nprob && went[threadIdx.x])
    atomicAdd(reinterpret_cast<unsigned*>(a.state) + ((size_t)batch * 3 + threadIdx.x) * kPairStateWords + kPairCounts +
                  ((step % 3) * kPairSlots + blockIdx.x % kPairSlots) * 32,
              went[threadIdx.x]);
}

// Operand planes of one block of 32 rows at an eps: sqrt(qs) times the rows (as a sum of two floats,
// so that the product of two of them is qs to 2^-46), two fp16 planes.  By 256 threads, a lane eight columns of a row, by whole
// words where rows start at 16 bytes (value by value a merge of 30,011 and 29,989 rows of 64 took 21.2 us, so 15.5; without
// planes 10.4).
template <int DP>
__device__ __forceinline__ void pair_write_planes(u32x4* out, const void* pts, size_t row0, int rows_here, int d,
                                                  int dtype, float scale, float qs, int tid, int threads) {
  constexpr int KK = DP / 16;
  float s_hi = scale, s_lo = 0.f;
  if (scale == 0.f) {
    s_hi = sqrtf(qs);
    s_lo = __builtin_fmaf(-s_hi, s_hi, qs) / (2.0f * s_hi);
  }
  const bool wide = small_wide(pts, d, dtype);
  for (int e = tid; e < KK * 64; e += threads) {
    const int kk = e >> 6, lane = e & 63, row = lane & 31, c0 = 16 * kk + 8 * (lane >> 5);
    const size_t at = (row0 + row) * d + c0;
    float v[8];
    if (row < rows_here && c0 + 8 <= d) {
      small_load8(v, pts, at, dtype, wide);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (row < rows_here && c0 + k < d) ? small_load(pts, at + k, dtype) : 0.f;
    }
    u32x4 hi, lo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float f[2], g[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const _Float16 hh = (_Float16)(v[2 * q + i] * s_hi);
        f[i] = (float)hh;
        g[i] = __builtin_fmaf(v[2 * q + i], s_hi, -f[i]) + v[2 * q + i] * s_lo;
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
template <int DP, bool SKIP>
__global__ __launch_bounds__(1024) void pair_merge_kernel(PairArgsPtr args, int step, int plane_groups) {
  const PairArgs& a = *(const PairArgs*)args;
  const int side = blockIdx.y + (a.first_prob ? 2 : 0), item = blockIdx.z, tid = threadIdx.x;
  const PairSide& sd = a.side[side];
  const int prob = side < 2 ? 0 : side - 1;
  if ((int)blockIdx.x >= a.merge_groups) {
    // ---- planes for a step with another eps: a quarter of a workgroup per 32 rows ----
    if ((int)blockIdx.x >= a.merge_groups + plane_groups) {
      if (step < 0 && item == 0 && blockIdx.y == 0) pair_write_work(a, (blockIdx.x - a.merge_groups - plane_groups) * 1024 + tid);
      return;
    }
    const int entries = a.lens[item * 3 + prob];
    const float4 next = pair_coef(a, item, prob, min(step + 1, entries + a.extrapolate));
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
  // (everything is on its way before anything is waited for)
  const int from = step < 0 ? 0 : step & 1;
  const float old = sd.pot[from * (size_t)a.items * sd.rows + at], norm = sd.norm[at], weight = sd.l2w[at];
  const int entries = a.lens[item * 3 + prob];
  const PairMode mode = *reinterpret_cast<const PairMode*>(state + kPairModes);
  const PairKnown known = pair_known(a, item, prob, max(step, 0));
  if (step > entries + a.extrapolate) return;
  const float4 next = step < 0 ? known.now : known.next;
  // the row's log weight from the largest of its side, and the other side's largest
  const float4 lim = known.w;
  const bool of_x = side == 0 || side == 2;
  const float own = of_x ? lim.y : lim.w, others = side >= 2 ? own : (of_x ? lim.w : lim.y);
  const float l2w = weight - own;
  float f = old;
  if (step < 0) {
    if (part > 0) return;
    // (nothing is known of the sums yet)
    if (SKIP && live) sd.key[at] = -1;
    if (blockIdx.x == 0 && quarter == 0 && (side == 0 || side >= 2))
      for (int i = lane; i < kPairStateWords; i += 64) state[i] = 0u;
  } else {
    __shared__ float2 sh[4][4][64];
    __shared__ int sh_best[4][4][SKIP ? 64 : 1];
    __shared__ float sh_dot[4][4][SKIP ? 64 : 1];
    __shared__ float sh_ex[4][4];
    const float4 coef = known.now;
    const float r = __builtin_fmaf(coef.w, old, l2w);  // the row's bias in this step
    const bool sweep = __builtin_amdgcn_readfirstlane(mode.sweep), ended = __builtin_amdgcn_readfirstlane(mode.two);
    float2 mine = make_float2(kNegBig, 0.f);
    int best = -1;
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
      const int* q = sd.best + (size_t)item * sd.ms_parts * sd.rows + rc;
      float most = kNegBig;
#pragma unroll 8
      for (int c = part; c < sd.ms_parts; c += 4) {
        const float2 v = p[(size_t)c * sd.rows];
        const int k = SKIP && ended ? q[(size_t)c * sd.rows] : -1;
        const float M = fmaxf(mine.x, v.x);
        mine.y = mine.y * fast_exp2(mine.x - M) + v.y * fast_exp2(v.x - M);
        mine.x = M;
        best = k >= 0 && v.x > most ? k : best;
        most = k >= 0 ? fmaxf(most, v.x) : most;
      }
      if (SKIP) sh_best[quarter][part][lane] = best;
    }
    if (SKIP && blockIdx.x == 0 && (side == 0 || side >= 2) && tid == 0) {
      // (what the next step knows of the lists)
      float* out = a.state + ((size_t)item * 3 + prob) * kPairStateWords + kPairLists + ((step + 1) % 3) * 32;
      const bool made = sweep && mode.coarse && !mode.list;
      out[0] = mode.list ? mode.drift : 0.f;
      out[1] = mode.list ? mode.base : mode.low - kPairGap - mode.reserve;
      out[2] = next.x == coef.x && (made || mode.list) ? 1.f : 0.f;
      // (for the gradient: whose lists hold the units of this step, the one-sweep or the two-sided form's)
      out[4] = known.twos + (!sweep && mode.two ? 1.f : 0.f);
      out[3] = made || mode.list ? 1.f : (!sweep && mode.two ? 2.f : 0.f);
    }
    sh[quarter][part][lane] = mine;
    __syncthreads();
    const float2(&all)[4][64] = sh[quarter];
    float lse;
    if (sweep) {
      // (fp32 holds every sum, by eight units from the bounds; where potentials of some 10^7 units cancel, logits and bounds are
      // off by rounding themselves: what that takes past the range ends there, no further off than its logits are, and a
      // potential stays a number.  NaN stays.)
      const float sum = (all[0][lane].y + all[1][lane].y) + (all[2][lane].y + all[3][lane].y);
      lse = small_log2(sum > 3.4e38f ? 3.4e38f : (sum < 1.2e-38f ? 1.2e-38f : sum), others + mode.shift) - r;
    } else {
      float M = kNegBig, s = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) M = fmaxf(M, all[w][lane].x);
#pragma unroll
      for (int w = 0; w < 4; ++w) s += all[w][lane].y * fast_exp2(all[w][lane].x - M);
      lse = small_log2(fmaxf(s, 1e-40f), M + others);
    }
    if (SKIP && !sweep && ended) {
      // the key of the largest logit that any chunk has seen beyond where it began, the pair's inner product
      const float2(&ms)[4][64] = sh[quarter];
      float most = kNegBig;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int k = sh_best[quarter][w][lane];
        best = k >= 0 && ms[w][lane].x > most ? k : (w == 0 ? -1 : best);
        most = k >= 0 ? fmaxf(most, ms[w][lane].x) : most;
      }
      const bool fresh = live && best >= 0 && best != sd.key[at];
      float dot = 0.f;
      if (fresh) {
        const size_t u = at * sd.d, v = ((size_t)item * sd.others + best) * sd.d;
#pragma unroll 4
        for (int k = part; k < sd.d; k += 4)
          dot = __builtin_fmaf(small_load(sd.pts, u + k, sd.dtype), small_load(sd.other, v + k, sd.dtype), dot);
      }
      sh_dot[quarter][part][lane] = dot;
      __syncthreads();
      if (fresh && part == 0) {
        sd.key[at] = best;
        sd.dot[at] = (sh_dot[quarter][0][lane] + sh_dot[quarter][1][lane]) + (sh_dot[quarter][2][lane] + sh_dot[quarter][3][lane]);
      }
    }
    const float rho = sd.rho, eps = coef.x;
    const float damp = rho > 0.f ? 1.0f / (1.0f + eps / rho) : 1.0f;
    const float alpha = (step == 0 || step > entries) ? 1.0f : 0.5f;
    f = alpha * (-eps * damp * kLn2 * lse);
    if (alpha != 1.0f) f += (1.0f - alpha) * old;
    if (damp < 1.0f) f -= alpha * (1.0f - damp) * norm;
    float ex[4] = {-3.0e38f, -3.0e38f, -3.0e38f, -3.0e38f};
    if (live && part == 0) {
      sd.pot[(from ^ 1) * (size_t)a.items * sd.rows + at] = f;
      if (SKIP) sd.sum2[at] = lse - others;
      const float z = __builtin_fmaf(coef.w, f, lse), df = f - old;
      ex[0] = z; ex[1] = -z; ex[2] = df; ex[3] = -df;
      if (!(z == z) || !(df == df) || !(fabsf(next.w * f) < kPairMostBias)) ex[0] = ex[1] = ex[2] = ex[3] = 3.0e38f;
    }
    // (the set that the next merge writes into)
    if (blockIdx.x == 0 && (side == 0 || side >= 2) && tid < kPairSlots * 9 + 16) {
      const int set = (step + 1) % 3, k = tid - kPairSlots * 8, x = k - kPairSlots;
      state[k < 0 ? set * kPairSlots * 8 + tid
                  : x < 0 ? kPairCounts + (set * kPairSlots + k) * 32 : kPairTaken + (set * 8 + x / 2) * 32 + x % 2] = 0u;
    }
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
  const float cross = live ? pair_cross(next.w, norm, known.reach.z) : 0.f;
  sd.bias[(size_t)item * sd.blocks * 32 + row] = pair_bias(fmaxf(b, kPairFar), fminf(cross, 60000.f));
  sd.bias32[(size_t)item * sd.blocks * 32 + row] = b;
}

// The key blocks (32 keys) that matter to a block of 32 query rows of the gradient: those whose unit the
// extrapolation, which read the same potentials, did not end.  By a workgroup of 512 threads; as many blocks
// as it returns are in `ids`, in their order (-1: that step computed every logit).
//
// Everything comes by value from the workspace that the gradient is given (pair_blocks), nothing from PairArgs: an
// autograd node's workspace need not be the memory that the solve ran in (a replayed graph's is the next
// call's, and hooks of saved tensors bring it back elsewhere), so the addresses inside say nothing.
struct PairBlocks {
  static constexpr int kMost = 2048;
  struct Lists {
    const unsigned long long* list;
    const unsigned long long* two_list;
    int n_items, two_items, two_first, n_st, n_str, chunk, groups, self;
  };
  Lists prob[3];
  const int* lens;
  const float* state;
  int extrapolate;
  __device__ __forceinline__ int find(int item, int prob_at, int qm, int qb, int nkb, unsigned short* ids) const {
    const int prob = __builtin_amdgcn_readfirstlane(prob_at);
    const Lists& pr = this->prob[prob];
    const int step = lens[item * 3 + prob] + 1;
    const float kind = state[((size_t)item * 3 + prob) * kPairStateWords + kPairLists + ((step + 1) % 3) * 32 + 3];
    if (!extrapolate || kind == 0.f) return -1;
    const bool two = kind == 2.f;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per = pr.chunk / 32;  // blocks of a chunk
    const int side = prob == 0 && qm == 1 ? 1 : 0;
    __shared__ unsigned long long mask[kMost / 64];
    __syncthreads();
    for (int seg = wave; seg * 64 < nkb; seg += 8) {
      const int kb = seg * 64 + lane;
      bool on = false;
      if (kb < nkb) {
        // stationary and streamed block of the unit
        const bool turned = two ? false : (pr.self ? kb / 8 < qb / 8 : side == 1);
        const int st = turned ? kb : qb, str = turned ? qb : kb, group = st / 8;
        const int chunk = str / per;
        int first = chunk * per, index;
        if (two) {
          index = (side ? pr.two_first : 0) + chunk * (((side ? pr.n_str : pr.n_st) + 255) / 256) + group;
        } else if (pr.self) {
          index = group;
          for (int c = 0; c < chunk; ++c) index += self_groups_of_chunk(c, pr.chunk, pr.n_str, pr.groups);
          first = max(first, group * 8);
        } else {
          index = chunk * pr.groups + group;
        }
        const int sub = str - first;
        const unsigned long long* w = two ? pr.two_list + (size_t)item * pr.two_items * (4 * kPairListWords)
                                          : pr.list + (size_t)item * pr.n_items * (4 * kPairListWords);
        on = (w[((size_t)index * 4 + (st & 7) / 2) * kPairListWords + (st & 1) * 2 + (sub >> 6)] >> (sub & 63)) & 1;
      }
      const unsigned long long m = __builtin_amdgcn_ballot_w64(on);
      if (lane == 0) mask[seg] = m;
    }
    __syncthreads();
    int count = 0;
    for (int seg = 0; seg * 64 < nkb; ++seg) {
      const unsigned long long m = mask[seg];
      if (wave == (seg & 7) && ((m >> lane) & 1)) ids[count + __popcll(m & ((1ull << lane) - 1))] = (unsigned short)(seg * 64 + lane);
      count += __popcll(m);
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(count);
  }
};

// The lists of a solve whose workspace is laid out in `t` (host side).
inline PairBlocks pair_blocks(const PairArgs& t, int extrapolate) {
  PairBlocks b = {};
  b.lens = t.lens;
  b.state = t.state;
  b.extrapolate = extrapolate;
  for (int q = t.first_prob; q < t.nprob; ++q) {
    const PairProblem& pr = t.prob[q];
    b.prob[q] = {pr.list, pr.two_list, pr.n_items, pr.two_items, pr.two_first, pr.n_st, pr.n_str, pr.chunk, pr.groups, pr.self};
  }
  return b;
}

}  // namespace fs
