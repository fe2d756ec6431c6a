// Log-sum-exp with the coarse tile test for rows of 65 .. 128 columns (fp16 planes): in place, or by lists.
//
// The test is the one of lse_coarse_kernel (fs_lsecoarse.hpp): the hi*hi plane product of a
// 32 x 32 logits tile (a unit), plus the exact key bias and a bound on the two cross products,
// shows whether any logit of the unit lies within 2^40 of its row's maximum; a unit
// where none does is left out, after a third of its MFMAs and without a single exponential.
//
// In place (lse_coarse128_kernel): a unit that goes on is finished where it is.  It holds up its
// workgroup's other wavefronts at the next barrier: with a tenth of the units going on the matrix pipe is
// busy 38 % of the time.  This form runs where rows have no start yet, or much goes on.
//
// By lists, in three launches, which are enqueued in every call that may go by them: the test (a launch that comes back at
// once where no unit is tested again), the keys on the lists, and what is left over of them (mostly nothing); in place
// the latter two find nothing to do, 9 us.  On a peaked plan nearly every unit that goes on does so for one logit
// (20,000 x 30,000 x 128, eps 0.0025: 1.04 a unit, 37,000 units of 586,000), and which ones these are
// hardly changes from one half-update to the next.  coarse128_test is nothing but the hi*hi products
// and their test, and leaves per unit which keys any of its 32 rows needs (Side::marks) and by how much all other logits
// stay below (Side::slack).  lse_listed128_kernel gathers the keys of 32 rows, 32 at a time, forms their
// logits from the start and runs the online soft-max.  Where the slack of an earlier launch covers what
// biases and maxima have moved by since, the test is not run at all (slack_renewed); units where it
// does not are taken whole, or but for one key where that one alone has risen.
//
// A half-update of the 20,000 x 30,000 x 128 problem, launches around it included: 290 - 310 us in place; 235 - 255 by lists
// with their test (185 - 195 of it), 60 - 140 without, of which 30 are launches that find nothing
// to do and the merge.  Ten iterations 5.9 -> 3.9 ms; 40 symmetric steps of 30,000 x 28,000 x 128 in eight clusters at
// eps 0.01 32 -> 13 ms; 100 of three problems of 10,000 x 128 23.8 -> 11.4 ms.  Where no lists pay the two launches
// are lost: flat plans of 12,000 - 16,000 rows take 2 - 3 % longer than without (16,000 x 12,000 x 100, eps 0.5: 3.32 -> 3.40 ms).
//
// What a row's logits are tested against is a lower bound of its maximum: its logit at the key that
// held its maximum in the launch before (Side::seed, computed by coarse_bias_kernel's seed blocks from
// Side::best_key), or the largest hi*hi logit so far less the bound on its cross products.
//
// LDS reads are written out by hand, with their wait: the compiler, which cannot tell a read
// of one buffer from the loads still filling another, would make every LDS access wait
// for all of them.
#pragma once

#include "fs_common.hpp"
#include "fs_stream.hpp"

namespace fs {

// The line that a unit's logits have to stay below, from a lower bound of a row's largest logit: 2^40 under it.
__device__ __forceinline__ float slack_line(float bound, float gap) { return bound - fabsf(bound) * 0x1p-20f - gap; }

// The least over each half of the wavefront, in lanes 31 and 63 (DPP row shifts, then a row broadcast).
__device__ __forceinline__ float half_min(float v) {
  int x = __builtin_bit_cast(int, v);
#define FS_MIN_STEP(ctrl, rmask, bmask)                                                          \
  {                                                                                               \
    const int o = __builtin_amdgcn_update_dpp(x, x, ctrl, rmask, bmask, false);                   \
    x = __builtin_bit_cast(int, fminf(__builtin_bit_cast(float, x), __builtin_bit_cast(float, o))); \
  }
  FS_MIN_STEP(0x111, 0xf, 0xf)  // row_shr:1
  FS_MIN_STEP(0x112, 0xf, 0xf)  // row_shr:2
  FS_MIN_STEP(0x114, 0xf, 0xe)  // row_shr:4
  FS_MIN_STEP(0x118, 0xf, 0xc)  // row_shr:8
  FS_MIN_STEP(0x142, 0xa, 0xf)  // row_bcast:15
#undef FS_MIN_STEP
  return __builtin_bit_cast(float, x);
}
// Keys that come this close to the line, in base-2 units, are taken as well, so that what is left out stays so for a while.
// More of it makes fewer tests and longer lists.  64, 256, 512 and 1,024 units, ms: ten alternating iterations of 20,000 x
// 30,000 x 128 at eps 0.0025 4.0, 4.0, 3.6, 3.4, at 0.05 3.4, 3.2, 3.5, 5.9; twenty of 12,000 x 14,000 x 80 at 0.01 2.9, 2.5, 2.5, 2.7; 40
// symmetric steps of 30,000 x 28,000 x 96 at 0.05 11.3, 9.9, 14.4, 29.9, of x 128 in clusters at 0.01 12.4, 13.1, 12.5, 10.9.
constexpr float kTakeReserve = 256.f;
// fp16, rounded towards zero
__device__ __forceinline__ unsigned pack_down(float v) {
  return __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(v, 0.f)) & 0xffffu;
}

// The units of 96 query rows a wavefront, tested.  Tiles of 64 keys have their hi planes in LDS (two buffers, the next
// in flight); the key bias is where the accumulators start; the launch is two workgroups per CU, each with an
// equal run of (row group, 128 keys) pieces, and every barrier finds its wavefronts with the same work
// behind them.  Bound by the matrix pipe (1.1 PFLOP/s; a large fp16 product reaches 1.34 on this card).
__device__ __forceinline__ void coarse128_test(const LaunchArgs& args, const Side& sd, unsigned tag, int bid, int grid,
                                               unsigned* lds) {
  constexpr int DP = 128, RB = 3, JT = 64, NSUB = JT / 32, KK16 = DP / 16;
  constexpr int ROWW = DP;        // 32-bit words per two-plane row in global memory
  constexpr int ROWH = DP / 2;    // words per hi-plane row in LDS
  constexpr int PPRH = ROWH / 4;  // 16-byte pieces per hi-plane row
  constexpr int LOADS = JT * PPRH / 256;  // direct loads per lane of a tile
  static_assert(PPRH == 16 && LOADS == 4, "64 keys x 16 pieces: four direct loads per lane");
  static_assert(kCoarse128Rows == 4 * 32 * RB, "");

  unsigned (*lds_k)[JT * ROWH] = reinterpret_cast<unsigned (*)[JT * ROWH]>(lds);  // [2]
  // the key bias in raw units, and kAuxMax behind it, a copy per wavefront
  float (*lds_b)[4][2 * JT] = reinterpret_cast<float (*)[4][2 * JT]>(lds + 2 * JT * ROWH);  // [2]
  static_assert(2 * (JT * ROWH + 4 * 2 * JT) <= kTest128Lds, "");
  if (!slack_renewed(args.sel, tag, sd.ps_q)) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 31;
  const int h = lane >> 5;
  // this workgroup's pieces: 128 keys (two tiles) of a row group, keys fastest
  const int per_group = (sd.nk + 2 * JT - 1) / (2 * JT), ntiles = (sd.nk + JT - 1) / JT;
  const long long n_pieces = (long long)((sd.nq + kCoarse128Rows - 1) / kCoarse128Rows) * per_group;
  const long long first = bid * n_pieces / grid, last = (bid + 1) * n_pieces / grid;
  if (first >= last) return;

  // MFMAs produce raw products of the scaled planes; lscale turns them into base-2 logits
  const float lscale = sd.qscale / (sd.plane_scale[sd.ps_q] * sd.plane_scale[sd.ps_k]);
  const float inv_lscale = 1.0f / lscale;

  auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto lds_addr = [](const void* p) {
    return (unsigned)(size_t)(const __attribute__((address_space(3))) void*)p;
  };
  auto direct = [](const void* from, void* to) {  // 16 bytes a lane
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                     (__attribute__((address_space(3))) void*)to, 16, 0, 0);
  };
  auto direct4 = [](const void* from, void* to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                     (__attribute__((address_space(3))) void*)to, 4, 0, 0);
  };

  // ---- key tiles: lane idx of instruction c fills LDS slot idx of the tile's buffer and fetches
  // the piece that belongs there (slot = piece ^ (row & 15)); the plane buffers end in zero
  // rows, and keys past the last are masked by their bias ----
  // (the four rounds of a tile are 16 rows apart and share the slot permutation)
  const unsigned koff = (unsigned)(((tid / PPRH) * ROWW + (((tid % PPRH) ^ ((tid / PPRH) & 15)) * 4)) * 4);
  const unsigned* kplanes = sd.kplanes;
  const unsigned* records = sd.key_aux + kAuxB;
  asm volatile("" : "+s"(kplanes), "+s"(records));  // (kept: loaded again in every tile otherwise, behind its barrier)
  auto issue_tile = [&](int tile, int buf) {
    const char* ktile = reinterpret_cast<const char*>(kplanes + (size_t)tile * (JT * ROWW)) + koff;
#pragma unroll
    for (int c = 0; c < LOADS; ++c)
      direct(ktile + c * (256 / PPRH) * ROWW * 4, &lds_k[buf][(c * 256 + wave * 64) * 4]);
    direct4(records + (size_t)tile * kAuxWords + lane, &lds_b[buf][wave][0]);
    direct4(records + (size_t)tile * kAuxWords + (kAuxMax - kAuxB) + lane, &lds_b[buf][wave][JT]);
  };
  // the hi planes of a sub-tile's keys and the bias of the keys behind a lane's 16 logits
  // (register r: key 8 (r / 4) + 4 h + r % 4), with the tile's bounds: read and waited for in one block
  auto read_sub = [&](const unsigned* keys, const float* bias, int js, u32x4 (&k)[KK16], f32x16& start, f32x2& most) {
    unsigned at[KK16];
#pragma unroll
    for (int kk = 0; kk < KK16; ++kk) at[kk] = lds_addr(keys + li * ROWH + (((2 * kk + h) ^ (li & 15)) << 2));
    f32x4 b0, b1, b2, b3;
    asm volatile(
        "ds_read_b128 %0, %13\n\tds_read_b128 %1, %13 offset:32\n\t"
        "ds_read_b128 %2, %13 offset:64\n\tds_read_b128 %3, %13 offset:96\n\tds_read_b64 %12, %22\n\t"
        "ds_read_b128 %4, %14\n\tds_read_b128 %5, %15\n\tds_read_b128 %6, %16\n\tds_read_b128 %7, %17\n\t"
        "ds_read_b128 %8, %18\n\tds_read_b128 %9, %19\n\tds_read_b128 %10, %20\n\tds_read_b128 %11, %21\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(b0), "=&v"(b1), "=&v"(b2), "=&v"(b3), "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3]),
          "=&v"(k[4]), "=&v"(k[5]), "=&v"(k[6]), "=&v"(k[7]), "=&v"(most)
        : "v"(lds_addr(bias + js * 32 + 4 * h)), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "v"(at[4]), "v"(at[5]),
          "v"(at[6]), "v"(at[7]), "v"(lds_addr(bias + JT + 2))
        : "memory");
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      start[e] = b0[e];
      start[4 + e] = b1[e];
      start[8 + e] = b2[e];
      start[12 + e] = b3[e];
    }
  };
  auto mfma16 = [](const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  };
  auto swap_halves = [&](float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  };
  auto max16 = [](const f32x16& a) {
    float m = fmaxf(a[0], a[1]);
#pragma unroll
    for (int r = 2; r < 16; ++r) m = fmaxf(m, a[r]);
    return m;
  };


  u32x4 xh[RB][KK16];  // hi planes of the query rows: [block][16-column step]
  // A unit is left out where each of its hi*hi logits, whatever the cross products add, lies 2^40 below
  // a lower bound of its row's maximum: below `floor`, in raw units, which is the bound less 2^40.  The cross
  // products come to at most |X_lo| |Y_hi| + |X_hi| |Y_lo| in 2-norms: the row's, and the largest of the tile's
  // keys.  (The bound of lse_coarse_kernel, element by element, is some eight times as large: 645 base-2 units in
  // place of 80 on N(0, I) clouds at eps 0.0025.)  The fp32 roundings of the chain, which starts from the bias,
  // are below 2^-20 of the logit and of |X_hi| |Y_hi| (kAuxMax) and one base-2 unit.
  float floor[RB], norm_hi[RB], norm_lo[RB];
  const float gap = -args.skip_log2 * inv_lscale, reserve = kTakeReserve * inv_lscale;
  int buf = 0;
  issue_tile((int)(first % per_group) * 2, 0);

  for (long long piece = first; piece < last;) {
    const int ig = (int)(piece / per_group);
    const int t0 = (int)(piece % per_group) * 2;  // a run of tiles of one row group
    const int t1 = (int)min((long long)ntiles, t0 + 2 * (last - piece));
    piece += (t1 - t0 + 1) / 2;
    const int row0 = (ig * 4 + wave) * (32 * RB);
    bool seeded = sd.seed != nullptr;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int row = min(row0 + rb * 32 + li, sd.nq - 1);
      const unsigned* qrow = sd.qplanes + (size_t)row * (size_t)ROWW;
#pragma unroll
      for (int kk = 0; kk < KK16; ++kk) xh[rb][kk] = *reinterpret_cast<const u32x4*>(qrow + 8 * kk + 4 * h);
      norm_hi[rb] = 1.0001f * sd.qnorms[row];
      norm_lo[rb] = 1.0001f * sd.qnorms[((sd.nq + 3) & ~3) + row];
      floor[rb] = -3.0e38f;
      if (sd.seed != nullptr) {
        const float sv = sd.seed[row];
        seeded = seeded && sv > -3.0e38f;
        floor[rb] = slack_line(sv, gap);
        if (row0 + rb * 32 + li < sd.nq && h == 0) sd.slack_floor[row] = floor[rb];
      }
    }
    seeded = __builtin_amdgcn_ballot_w64(seeded) == ~0ull;
    if (!seeded && args.sel != nullptr && lane == 0) args.sel[kSelBump + sd.ps_q] = 1u;
    float left[2 * NSUB][RB];  // by how much the units of 128 keys lie below the line, the least of a lane's logits
    unsigned marks[2 * NSUB][RB];  // the keys of theirs that do not
#pragma unroll
    for (int k = 0; k < 2 * NSUB; ++k)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) left[k][rb] = 3.0e38f, marks[k][rb] = 0u;

    for (int t = t0; t < t1; ++t, buf ^= 1) {
      // this wavefront's part of the tile has landed; after the barrier all parts have, and every
      // wavefront has left the tile before, whose buffer the next one takes
      fence();
      __builtin_amdgcn_s_waitcnt(0x0F70);
      fence();
      barrier();
      if (t + 1 < t1 || piece < last) issue_tile(t + 1 < t1 ? t + 1 : (int)(piece % per_group) * 2, buf ^ 1);
      fence();
#pragma unroll
      for (int js = 0; js < NSUB; ++js) {
        u32x4 ks[KK16];
        f32x16 start;
        f32x2 most;
        read_sub(lds_k[buf] + js * 32 * ROWH, lds_b[buf][wave], js, ks, start, most);
        f32x16 acc[RB];
#pragma unroll
        for (int kk = 0; kk < KK16; ++kk)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) acc[rb] = mfma16(ks[kk], xh[rb][kk], kk == 0 ? start : acc[rb]);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const float tmax = max16(acc[rb]);
          const float corr = __builtin_fmaf(norm_lo[rb], most[0], __builtin_fmaf(norm_hi[rb], most[1], inv_lscale));
          float below = floor[rb] - (tmax + corr);
          unsigned mark = 0u;
          if (wave_any(!(below > reserve))) {
            // some row's logit is above the line or close to it: its key is taken, for all rows
            float rest = -3.0e38f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const unsigned long long hit = __builtin_amdgcn_ballot_w64(!(floor[rb] - (acc[rb][r] + corr) > reserve));
              const bool lo = (unsigned)hit != 0u, hi = (unsigned)(hit >> 32) != 0u;
              mark |= (lo ? 1u : 0u) << (8 * (r / 4) + r % 4) | (hi ? 16u : 0u) << (8 * (r / 4) + r % 4);
              rest = fmaxf(rest, (h ? hi : lo) ? -3.0e38f : acc[rb][r]);
            }
            below = floor[rb] - (rest + corr);
          }
          if (t & 1) left[NSUB + js][rb] = below, marks[NSUB + js][rb] = mark;
          else left[js][rb] = below, marks[js][rb] = mark;
          // (rows without a start: by what has come so far)
          if (!seeded) floor[rb] = fmaxf(floor[rb], __builtin_fmaf(fabsf(tmax), -0x1p-20f, tmax - corr) - gap);
        }
        fence();
      }
      if ((t & 1) == 0 && t + 1 < t1) continue;
      // the units of 128 keys: the least over the lanes
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        unsigned word[2];
#pragma unroll
        for (int k = 0; k < NSUB; ++k) {
          float a = left[2 * k][rb], b = left[2 * k + 1][rb];
          swap_halves(a, b);  // a: the first unit's, b: the second's, 32 lanes each
          float v = half_min(fminf(a, b)) * lscale;
          v = fminf(v, 60000.f);
          const unsigned half16 = pack_down(v);
          word[k] = (unsigned)__builtin_amdgcn_readlane((int)half16, 31) |
                    ((unsigned)__builtin_amdgcn_readlane((int)half16, 63) << 16);
          left[2 * k][rb] = left[2 * k + 1][rb] = 3.0e38f;
        }
        // (rows without a start take their first unit whatever it holds: they may hold NaN)
        if (!seeded && t < 2) word[0] = (word[0] & 0xffff0000u) | 0xbc00u;
        const int block = (ig * 4 + wave) * RB + rb;
        if (block * 32 < sd.nq && lane == 0) {
          const size_t at = (size_t)block * sd.slack_stride + t / 2 * 4;
          *reinterpret_cast<uint2*>(sd.slack + at) = make_uint2(word[0], word[1]);
          *reinterpret_cast<uint4*>(sd.marks + at) = make_uint4(marks[0][rb], marks[1][rb], marks[2][rb], marks[3][rb]);
        }
#pragma unroll
        for (int k = 0; k < 2 * NSUB; ++k) marks[k][rb] = 0u;
      }
    }
  }
}

// Units that go on are finished where they are, by the online soft-max.  A wavefront keeps both planes of 64
// query rows; tiles of 64 keys have both planes in LDS (two buffers, the next tile in flight), a
// unit that goes on adds the cross products from there, and nothing in it waits for memory.
__device__ __forceinline__ void coarse128_in_place(const LaunchArgs& args, const Side& sd, int bid, unsigned* lds) {
  constexpr int DP = 128, RB = 2, JT = 64, NSUB = JT / 32, KK16 = DP / 16;
  constexpr int ROWW = DP;        // 32-bit words per two-plane row in global memory
  constexpr int ROWH = DP / 2;    // words per hi-plane row in LDS
  constexpr int PPRH = ROWH / 4;  // 16-byte pieces per hi-plane row
  constexpr int PER_PLANE = JT * PPRH / 256;  // direct loads per lane and plane of a tile
  static_assert(PPRH == 16 && PER_PLANE == 4, "64 keys x 16 pieces: four direct loads per lane and plane");

  unsigned (*lds_k)[2][JT * ROWH] = reinterpret_cast<unsigned (*)[2][JT * ROWH]>(lds);  // [buffer][plane]
  float (*lds_b)[2][JT] = reinterpret_cast<float (*)[2][JT]>(lds + 4 * JT * ROWH);      // [buffer], bias and kAuxMax
  static_assert(4 * JT * ROWH + 4 * JT <= kCoarse128Lds, "");
  const int split = bid % sd.splits;
  const int ig = bid / sd.splits;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int li = lane & 31;
  const int h = lane >> 5;
  const int row0 = (ig * 4 + wave) * (32 * RB);
  const int j_begin = split * sd.chunk;
  const int j_end = min(sd.nk, j_begin + sd.chunk);
  const int ntiles = (j_end > j_begin) ? (j_end - j_begin + JT - 1) / JT : 0;

  // MFMAs produce raw products of the scaled planes; lscale turns them into base-2 logits
  const float lscale = sd.qscale / (sd.plane_scale[sd.ps_q] * sd.plane_scale[sd.ps_k]);
  const float inv_lscale = 1.0f / lscale;

  // ---- stationary planes of the query rows: [block][16-column step] ----
  u32x4 xh[RB][KK16], xl[RB][KK16];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = min(row0 + rb * 32 + li, sd.nq - 1);
    const unsigned* qrow = sd.qplanes + (size_t)row * (size_t)ROWW;
#pragma unroll
    for (int kk = 0; kk < KK16; ++kk) {
      xh[rb][kk] = *reinterpret_cast<const u32x4*>(qrow + 8 * kk + 4 * h);
      xl[rb][kk] = *reinterpret_cast<const u32x4*>(qrow + ROWH + 8 * kk + 4 * h);
    }
  }
  float norm_hi[RB], norm_lo[RB];  // (the bound on the cross products: see coarse128_test)
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = min(row0 + rb * 32 + li, sd.nq - 1);
    norm_hi[rb] = 1.0001f * sd.qnorms[row];
    norm_lo[rb] = 1.0001f * sd.qnorms[((sd.nq + 3) & ~3) + row];
  }

  // ---- LDS access by hand ----
  auto lds_addr = [](const void* p) {
    return (unsigned)(size_t)(const __attribute__((address_space(3))) void*)p;
  };
  auto ds_read16 = [&](const unsigned* p) -> u32x4 {
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(lds_addr(p)) : "memory");
    return v;
  };
  auto ds_read4 = [&](const float* p) -> float {
    float v;
    asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(lds_addr(p)) : "memory");
    return v;
  };
  auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
  auto wait_lds = [&]() {  // lgkmcnt(0), and nothing moves across
    fence();
    __builtin_amdgcn_s_waitcnt(0xC07F);
    fence();
  };
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- key tiles: lane idx of instruction c fills LDS slot idx of a plane's buffer and fetches
  // the piece that belongs there (slot = piece ^ (row & 15)); the plane buffers end in zero
  // rows, so tiles past the chunk are fetched like any other and masked by their bias ----
  // (the four rounds of a plane are 16 rows apart and share the slot permutation)
  const unsigned koff = (unsigned)(((tid / PPRH) * ROWW + (((tid % PPRH) ^ ((tid / PPRH) & 15)) * 4)) * 4);
  const char* ktile = reinterpret_cast<const char*>(sd.kplanes + (size_t)j_begin * (size_t)ROWW);
  auto issue_tile = [&](int buf) {  // the next tile in sequence
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int c = 0; c < PER_PLANE; ++c)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(ktile + (p * ROWH + c * (256 / PPRH) * ROWW) * 4 + koff),
            (__attribute__((address_space(3))) void*)(&lds_k[buf][p][(c * 256 + wave * 64) * 4]), 16, 0, 0);
    ktile += JT * ROWW * 4;
  };
  // ---- key bias: wavefront 0 brings those of the tile's 64 keys and the tile's bounds, by direct loads
  // issued ahead of the tile's keys (the same wait covers both) ----
  const unsigned* records = sd.key_aux + (size_t)(j_begin / JT) * kAuxWords + kAuxB + lane;
  auto issue_bias = [&](int t, int buf) {
    if (wave == 0) {
      const unsigned* r = records + (size_t)t * kAuxWords;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)r,
                                       (__attribute__((address_space(3))) void*)(&lds_b[buf][0][0]), 4, 0, 0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(r + (kAuxMax - kAuxB)),
                                       (__attribute__((address_space(3))) void*)(&lds_b[buf][1][0]), 4, 0, 0);
    }
  };
  auto mfma16 = [](const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  };
  auto swap_halves = [&](float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  };
  auto max16 = [](const f32x16& a) {
    float m = fmaxf(a[0], a[1]);
#pragma unroll
    for (int r = 2; r < 16; ++r) m = fmaxf(m, a[r]);
    return m;
  };

  const float clear = args.skip_log2 - kTakeReserve;

  // ---- running statistics.  The logits stay in absolute raw units (of the full logit with
  // its key bias); the running maximum M is kept as run_c = -M * lscale, rounded once: the
  // constant of the exponentials and what the test compares with (subtracted inside the
  // accumulator, M would cost the logits their digits whenever it lies far below them) ----
  float run_c[RB], run_s[RB], best_v[RB];
  int best_j[RB];
  const bool track = sd.best_key != nullptr;
  bool seeded = sd.seed != nullptr;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    run_c[rb] = 0.f;
    run_s[rb] = 0.f;
    best_v[rb] = -3.0e38f;
    best_j[rb] = -1;
    if (sd.seed != nullptr) {
      const float sv = sd.seed[min(row0 + rb * 32 + li, sd.nq - 1)];
      seeded = seeded && sv > -3.0e38f;
      run_c[rb] = -sv * lscale;
    }
  }
  // (wavefront-uniform: without a starting value for every row the first unit sets the maxima)
  seeded = __builtin_amdgcn_ballot_w64(seeded) == ~0ull;
  if (!seeded && args.sel != nullptr && sd.slack != nullptr && lane == 0) args.sel[kSelBump + sd.ps_q] = 1u;
  bool started[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    started[rb] = seeded;
    if (!seeded) run_c[rb] = 0.f;
  }
  unsigned n_ended = 0, n_clear = 0;  // n_clear: units of which lists would take nothing

  // ---- prologue: tile 0 and its bias terms ----
  if (ntiles > 0) {
    issue_bias(0, 0);
    issue_tile(0);
    fence();
    __builtin_amdgcn_s_waitcnt(0x0070);  // everything has landed
    fence();
  }
  barrier();

  int buf = 0;
  for (int t = 0; t < ntiles; ++t) {
    const int j0 = j_begin + t * JT;
    const int nbuf = buf ^ 1;
    // the other buffer was read during tile t - 1, which every wavefront has left
    issue_bias(t + 1, nbuf);
    issue_tile(nbuf);
    fence();

#pragma unroll
    for (int js = 0; js < NSUB; ++js) {
      const unsigned* yrow = lds_k[buf][0] + (js * 32 + li) * ROWH;
      float kbias = ds_read4(&lds_b[buf][0][js * 32 + li]);
      float most_hi = ds_read4(&lds_b[buf][1][2]), most_lo = ds_read4(&lds_b[buf][1][3]);
      // hi*hi of both row blocks, the key operands one step ahead of their MFMAs
      u32x4 ks[2];
      ks[0] = ds_read16(yrow + (((0 + h) ^ (li & 15)) << 2));
      f32x16 acc[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[rb][r] = 0.f;
#pragma unroll
      for (int kk = 0; kk < KK16; ++kk) {
        wait_lds();
        if (kk + 1 < KK16) ks[(kk + 1) & 1] = ds_read16(yrow + (((2 * (kk + 1) + h) ^ (li & 15)) << 2));
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = mfma16(ks[kk & 1], xh[rb][kk], acc[rb]);
      }
      fence();
      asm volatile("" : "+v"(kbias), "+v"(most_hi), "+v"(most_lo));  // (read before the first wait above)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        // + key bias: A = [bias_j, 1], B = [1, 0]
        acc[rb] = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 1.0f : kbias, h ? 0.0f : 1.0f,
                                                       acc[rb], 0, 0, 0);
        const float tmax = max16(acc[rb]);
        const float corr = __builtin_fmaf(norm_lo[rb], most_hi, __builtin_fmaf(norm_hi[rb], most_lo, inv_lscale));
        // every logit of the unit at least 2^40 below its row's running maximum, whatever the
        // cross products add: nothing of it could change the fp32 sums
        const float above = __builtin_fmaf(tmax + corr, lscale, run_c[rb]);
        n_clear += wave_any(above > clear) ? 0u : 1u;
        if (started[rb] && !wave_any(above > args.skip_log2)) {
          ++n_ended;
          continue;
        }
        // ---- the unit goes on: cross products on the lo planes, then the online soft-max ----
        {
          // (both planes of the keys again from LDS, two steps at a time: the registers of the
          // first pass are free by now.  The cross products are summed on their own, where they
          // are small, and join the logits with one addition: added one by one to logits of a
          // few thousand base-2 units they would each be rounded to those logits' last place.)
          const unsigned* ylo = lds_k[buf][1] + (js * 32 + li) * ROWH;
          f32x16 cr;
#pragma unroll
          for (int r = 0; r < 16; ++r) cr[r] = 0.f;
#pragma unroll
          for (int part = 0; part < KK16 / 2; ++part) {
            u32x4 kh[2], kl[2];
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
              const int kk = part * 2 + k2;
              kh[k2] = ds_read16(yrow + (((2 * kk + h) ^ (li & 15)) << 2));
              kl[k2] = ds_read16(ylo + (((2 * kk + h) ^ (li & 15)) << 2));
            }
            wait_lds();
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
              const int kk = part * 2 + k2;
              cr = mfma16(kh[k2], xl[rb][kk], cr);
              cr = mfma16(kl[k2], xh[rb][kk], cr);
            }
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[rb][r] += cr[r];
          const float lane_max = max16(acc[rb]);
          float tm = lane_max;
          {
            float a = tm, b = tm;
            swap_halves(a, b);
            tm = fmaxf(a, b);  // the row's largest logit of the unit
          }
          // the key of the row's largest logit so far (absolute raw units; lane-private, the two
          // half-waves are merged at the end)
          // (searched only when some lane's largest value of the unit beats what it has)
          if (track && wave_any(lane_max > best_v[rb])) {
            const int jb = j0 + js * 32 + 4 * h;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float v = acc[rb][r];
              if (v > best_v[rb]) {
                best_v[rb] = v;
                best_j[rb] = jb + 8 * (r / 4) + (r % 4);
              }
            }
          }
          const bool first = !started[rb];
          float cc = -tm * lscale;
          asm volatile("" : "+v"(cc));  // the exponents, the rescale and the result see one number
          cc = first ? cc : fminf(cc, run_c[rb]);
          float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            ps0 += fast_exp2(__builtin_fmaf(acc[rb][r], lscale, cc));
            ps1 += fast_exp2(__builtin_fmaf(acc[rb][r + 1], lscale, cc));
          }
          const float resc = first ? 0.f : fast_exp2(cc - run_c[rb]);
          run_s[rb] = run_s[rb] * resc + (ps0 + ps1);
          run_c[rb] = cc;
          started[rb] = true;
        }
      }
    }

    // tile t + 1 has landed (and with it the bias terms requested ahead of it); after the barrier
    // both are visible and every wavefront is done reading tile t
    fence();
    __builtin_amdgcn_s_waitcnt(0x0070);
    fence();
    barrier();
    buf = nbuf;
  }
  fence();
  __builtin_amdgcn_s_waitcnt(0x0070);  // what was fetched past the chunk: let it land before the end

  // unit counts of this wavefront for the variant choice on the device
  if (args.sel != nullptr && lane == 0 && ntiles > 0) {
    const int slot = blockIdx.x % kSelSlots;
    atomicAdd(&args.sel[kSelEnded + slot], n_ended);
    atomicAdd(&args.sel[kSelUnits + slot], (unsigned)(ntiles * NSUB * RB));
    if (n_clear > 0 && sd.slack != nullptr) atomicAdd(&args.sel[kSelDmax + sd.ps_q * kDmaxSlots + (blockIdx.x & (kDmaxSlots - 1))], n_clear);
  }

#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = row0 + rb * 32 + li;
    const float s = run_s[rb] + xor32(run_s[rb]);
    const float M2 = -run_c[rb];
    float bv = best_v[rb];
    int bj = best_j[rb];
    const float ov = xor32(bv);
    const int oj = __shfl_xor(bj, 32, 64);
    if (ov > bv || (ov == bv && oj >= 0 && (bj < 0 || oj < bj))) bj = oj;
    if (row < sd.nq && h == 0) {
      if (sd.splits == 1) {
        epilogue_scalar(sd.ep, row, M2, s, 0.f);
        if (track && bj >= 0) sd.best_key[row] = bj;
      } else {
        const size_t pr = (size_t)split * (size_t)sd.nq + (size_t)row;
        *reinterpret_cast<float2*>(&sd.part_ms[2 * pr]) = make_float2(M2, s);
        if (sd.part_best != nullptr) sd.part_best[pr] = bj;
      }
    }
  }
}

// Either form of both sides in one launch (as two, one of them found nothing to do: 4 us of a step).  Side 0 has
// the first blocks0 workgroups, as many as the larger of its forms; the test's are blocks_sparse of them (and what is
// left of kCoarse128Grid on side 1).
template <int T>
__global__ __launch_bounds__(256, 2) void lse_coarse128_kernel(const LaunchArgs args) {
  static_assert(kTest128Lds <= kCoarse128Lds, "");
  __shared__ __attribute__((aligned(16))) unsigned lds[kCoarse128Lds];
  // variant chosen on the device: the launch of the variant that was not chosen ends here
  if (args.sel_pred && args.sel[kSelWord] != args.sel_want) return;
  int bid = blockIdx.x;
  const bool second = bid >= args.blocks0;
  if (second) bid -= args.blocks0;
  const Side& sd = second ? args.side[1] : args.side[0];
  int lists = __builtin_amdgcn_readfirstlane(sd.slack != nullptr && coarse128_lists(args.sel, args.tag[second ? 1 : 0], sd.ps_q) ? 1 : 0);
  if (lists == 0 && bid < sd.igroups * sd.splits) coarse128_in_place(args, sd, bid, lds);
  // (one behind the other for the compiler: as two branches of one condition they shared what the form in place had no
  // registers for, and it spilled: 20,000 x 30,000 x 128 at eps 0.2 256 and 284 us a half-update for 244 and 262)
  asm volatile("" : "+s"(lists));
  if (lists != 0) {
    const int grid = second ? kCoarse128Grid - args.blocks_sparse : args.blocks_sparse;
    if (bid < grid) coarse128_test(args, sd, args.tag[second ? 1 : 0], bid, grid, lds);
  }
}

// A workgroup takes 32 query rows, each of its wavefronts a quarter of the keys.  First the keys on the list; what
// they make of the rows' maxima tells by how much the rows' lines have fallen at most (the key that a
// row's maximum was held by may have lost its lead to another on the list), and which units' slack that uses up:
// their other keys follow.  Bound by the chain of loads in front of the first logits and behind it, so each wavefront has three
// quarters of a unit in flight.
//
// A row block whose lines have fallen by more than most of its units' slack (one row of the 32 will do) is left to a
// second launch, REST, which shares its units out over up to 16 workgroups: alone, it took 250 us.
// (Left to it from more than this many keys on: 256, 1,024, 4,096 and never take 4.65, 4.0, 4.25 and 4.3 ms for the ten iterations
// at 20,000 x 30,000 x 128, 11.8, 13.1, 13.5 and 14.2 for 40 steps in clusters; at larger eps and of fewer columns all are within 3 %.)
constexpr int kRestKeys = 1024;  // (as many are a workgroup's own)
template <bool REST>
__global__ __launch_bounds__(256, 2) void lse_listed128_kernel(const LaunchArgs args) {
  constexpr int DP = 128, KK16 = DP / 16;
  constexpr int ROWW = DP, ROWH = DP / 2;  // words of a two-plane row, and of one plane of it
  // per wavefront: a quarter of the columns of 32 keys, [plane][key], three times; the unit's bias
  __shared__ __attribute__((aligned(16))) unsigned lds_q[4][3][2 * 32 * 16];
  __shared__ __attribute__((aligned(16))) float lds_qb[4][64];
  constexpr int kListKeys = 256;
  __shared__ unsigned short lds_keys[4][kListKeys];  // of the batch's first key
  __shared__ float sh_max[4][32], sh_sum[4][32], sh_top[4][32];
  __shared__ int sh_key[4][32], sh_count[4];

  if (args.sel_pred && args.sel[kSelWord] != args.sel_want) return;
  int bid = blockIdx.x;
  const bool second = bid >= args.blocks0;
  if (second) bid -= args.blocks0;
  const Side& sd = second ? args.side[1] : args.side[0];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 31, h = lane >> 5;
  if (!coarse128_lists(args.sel, args.tag[second ? 1 : 0], sd.ps_q)) return;
  // (left to the second launch: their number, the row blocks, and by how much their lines have fallen)
  int* put_off = sd.slack_rest;
  float* put_off_fall = reinterpret_cast<float*>(sd.slack_rest) + (sd.nq + 31) / 32 + 4;
  const int parts = min(16, sd.splits - 1);  // workgroups of a row block there, and partial results
  const int items = REST ? min(put_off[0], (sd.nq + 31) / 32) * parts : 1, step = second ? gridDim.x - args.blocks0 : args.blocks0;
  for (int item = REST ? bid : 0; item < items; item += REST ? step : 1) {
  const int block = REST ? put_off[4 + item / parts] : bid, row = block * 32 + li;
  const int slice = REST ? item % parts * 4 + wave : wave, slices = REST ? 4 * parts : 4;
  const float lscale = sd.qscale / (sd.plane_scale[sd.ps_q] * sd.plane_scale[sd.ps_k]);
  const int pieces = (sd.nk + 127) / 128;
  const int piece0 = (int)((long long)slice * pieces / slices), piece1 = (int)((long long)(slice + 1) * pieces / slices);

  auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
  auto lds_addr = [](const void* p) {
    return (unsigned)(size_t)(const __attribute__((address_space(3))) void*)p;
  };
  // The logits stay in absolute raw units (of the full logit with its key bias); the running maximum M
  // is kept as run_c = -M * lscale, rounded once: the constant of the exponentials (subtracted
  // inside the accumulator, M would cost the logits their digits whenever it lies far below them).
  float run_c = 0.f, run_s = 0.f, best_v = -3.0e38f;
  int best_j = -1;
  const bool track = sd.best_key != nullptr;
  bool started = sd.seed != nullptr;
  if (sd.seed != nullptr) {
    const float sv = sd.seed[min(row, sd.nq - 1)];
    started = sv > -3.0e38f;
    run_c = -sv * lscale;
  }
  const bool renewed = slack_renewed(args.sel, args.tag[second ? 1 : 0], sd.ps_q);
  const float line = renewed ? 0.f : sd.slack_floor[min(row, sd.nq - 1)];
  float fall = REST ? put_off_fall[item / parts] : 0.f;
  // (wavefront-uniform: without a starting value for every row the first unit sets the maxima)
  started = __builtin_amdgcn_ballot_w64(started) == ~0ull;

  // ---- the keys that are taken, in order, of 64 pieces of 128 at a time (one a lane) ----
  unsigned taken[4] = {0u, 0u, 0u, 0u};
  int n_taken = 0;
  auto load_marks = [&](int from, bool rest) {
    const int piece = min(from + lane, piece1 - 1);
    const size_t at = (size_t)block * sd.slack_stride + piece * 4;
    const uint4 m = *reinterpret_cast<const uint4*>(sd.marks + at);
    const uint2 w = *reinterpret_cast<const uint2*>(sd.slack + at);
    const unsigned mk[4] = {m.x, m.y, m.z, m.w}, sl[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int sub = piece * 4 + k, keys = sd.nk - sub * 32;  // (keys of this unit that exist)
      const float s = (float)__builtin_bit_cast(_Float16, (unsigned short)sl[k]) - fall;
      unsigned t = mk[k];
      if (rest) {
        const unsigned* rec = sd.key_aux + (size_t)(max(sub, 0) / 2) * kAuxWords + kAuxMax + 4 + (sub & 1);
        const float rise = __builtin_bit_cast(float, rec[0]) * lscale, rise2 = __builtin_bit_cast(float, rec[2]) * lscale;
        t = ~mk[k] & (s > rise ? 0u : (s > rise2 ? 1u << rec[4] : ~0u));
      }
      if (from + lane >= piece1 || keys <= 0) t = 0u;
      else if (keys < 32) t &= (1u << keys) - 1u;
      taken[k] = t;
    }
  };
  // (a list of what fits of them from key number `first` of the batch on)
  auto list_keys = [&](int first, int rank) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      unsigned t = taken[k];
      while (t != 0u) {
        if (rank >= first && rank < first + kListKeys) lds_keys[wave][rank - first] = (unsigned short)(lane * 128 + k * 32 + __builtin_ctz(t));
        ++rank;
        t &= t - 1u;
      }
    }
  };

  // ---- a quarter of a unit's keys: half the columns of one plane, 128 bytes a key (hi before lo; a cache line
  // each, where a quarter of the columns of both planes was two requests for as many bytes).  Instruction c
  // brings eight keys; LDS slot = piece ^ (key / 2 % 8) ----
  const unsigned *kplanes = sd.kplanes, *qplanes = sd.qplanes;
  // (row c of eight: where the eight lanes of a key find it, in bytes)
  auto issue_quarter = [&](const unsigned* planes, const unsigned (&at)[4], int q, int slot) {
    const char* k = reinterpret_cast<const char*>(planes + (q & 1) * ROWH + (q >> 1) * 32);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(k + at[c]),
          (__attribute__((address_space(3))) void*)(&lds_q[wave][slot][c * 256]), 16, 0, 0);
  };
  int batch0 = piece0 * 128, n_list = 0;  // the batch's first key, keys on the list
  auto find_keys = [&](int unit, unsigned (&at)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int key = batch0 + lds_keys[wave][min(unit * 32 + c * 8 + (lane >> 3), n_list - 1)];
      at[c] = (unsigned)key * (ROWW * 4) + (unsigned)(((lane & 7) ^ ((c & 1) * 4 + (lane >> 4))) * 16);
    }
  };
  auto issue_bias = [&](int unit) {
    const int key = batch0 + lds_keys[wave][min(unit * 32 + li, n_list - 1)];
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(sd.key_aux + (size_t)(key / 64) * kAuxWords + kAuxB + key % 64),
        (__attribute__((address_space(3))) void*)(&lds_qb[wave][0]), 4, 0, 0);
  };
  unsigned qat[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) qat[k] = lds_addr(&lds_q[wave][0][li * 32 + (((2 * k + h) ^ ((li >> 1) & 7)) << 2)]);
  const unsigned qatb = lds_addr(&lds_qb[wave][li]);
  auto read_quarter = [&](u32x4* k, int slot) {
    const unsigned by = (unsigned)slot * 4096u;
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3])
        : "v"(qat[0] + by), "v"(qat[1] + by), "v"(qat[2] + by), "v"(qat[3] + by) : "memory");
  };

  auto mfma16 = [](const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  };
  auto swap_halves = [&](float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  };
  auto max16 = [](const f32x16& a) {
    float m = fmaxf(a[0], a[1]);
#pragma unroll
    for (int r = 2; r < 16; ++r) m = fmaxf(m, a[r]);
    return m;
  };

  u32x4 xh[KK16], xl[KK16];
#pragma unroll
  for (int kk = 0; kk < KK16; ++kk) xh[kk] = xl[kk] = u32x4{0u, 0u, 0u, 0u};
  bool rows_in = false;
#pragma unroll 1
  for (int rest = REST ? 1 : 0; rest < 2; ++rest) {
  if (!REST && rest != 0) {
    // By how much the units have come closer to the line since they were tested: the rise of their keys' biases
    // (kAuxMax) and the largest fall of a row's line.  One base-2 unit covers the roundings.
    if (h == 0) sh_max[wave][li] = started ? -run_c : kNegBig;
    __syncthreads();
    const float most = fmaxf(fmaxf(sh_max[0][li], sh_max[1][li]), fmaxf(sh_max[2][li], sh_max[3][li]));
    __syncthreads();
    if (!renewed) {
      fall = (line - slack_line(most / lscale, -args.skip_log2 / lscale)) * lscale + 1.0f;
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) fall = fmaxf(fall, __shfl_xor(fall, o, 64));
    }
    int keys = 0;
    for (int from = piece0; from < piece1; from += 64) {
      load_marks(from, true);
#pragma unroll
      for (int k = 0; k < 4; ++k) keys += __builtin_popcount(taken[k]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) keys += __shfl_xor(keys, o, 64);
    if (lane == 0) sh_count[wave] = keys;
    __syncthreads();
    keys = sh_count[0] + sh_count[1] + sh_count[2] + sh_count[3];
    __syncthreads();
    if (keys == 0) break;
    if (keys > kRestKeys && sd.splits > 1) {
      if (threadIdx.x == 0) {
        const int at = atomicAdd(put_off, 1);
        put_off[4 + at] = block;
        put_off_fall[at] = fall;
      }
      break;
    }
  }
  for (int from = piece0; from < piece1; from += 64) {
   batch0 = from * 128;
   load_marks(from, rest != 0);
   int mine = 0;
#pragma unroll
   for (int k = 0; k < 4; ++k) mine += __builtin_popcount(taken[k]);
   int rank = mine;  // keys of the lanes in front
#pragma unroll
   for (int o = 1; o < 64; o <<= 1) {
     const int v = __shfl_up(rank, o, 64);
     if (lane >= o) rank += v;
   }
   const int all = __shfl(rank, 63, 64);
   rank -= mine;
   n_taken += all;
   for (int first = 0; first < all; first += kListKeys) {
    list_keys(first, rank);
    n_list = min(kListKeys, all - first);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // (the list is this wavefront's own)
    const int n_units = (n_list + 31) / 32;
    unsigned at[4];
    int slot = 1;
    if (!rows_in) {
      // the query rows' planes the same way, the first unit's quarters behind them.  The planes end in zero rows.
      rows_in = true;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        at[c] = (unsigned)(block * 32 + c * 8 + (lane >> 3)) * (ROWW * 4) + (unsigned)(((lane & 7) ^ ((c & 1) * 4 + (lane >> 4))) * 16);
      fence();
#pragma unroll
      for (int q = 0; q < 3; ++q) issue_quarter(qplanes, at, q, q);
      fence();
      __builtin_amdgcn_s_waitcnt(0x0F78);
      fence();
      read_quarter(xh, 0);
      issue_quarter(qplanes, at, 3, 0);
      fence();
      __builtin_amdgcn_s_waitcnt(0x0F78);
      fence();
      read_quarter(xl, 1);
      find_keys(0, at);
      fence();
      __builtin_amdgcn_s_waitcnt(0x0F74);
      fence();
      read_quarter(xh + 4, 2);
      fence();
      __builtin_amdgcn_s_waitcnt(0x0F70);
      fence();
      read_quarter(xl + 4, 0);
    } else {
      find_keys(0, at);
    }
    fence();
    issue_bias(0);
    issue_quarter(kplanes, at, 0, 1);
    issue_quarter(kplanes, at, 1, 2);
    issue_quarter(kplanes, at, 2, 0);
    float batch_v = -3.0e38f;  // the largest logit of the list so far and its place on it
    int batch_j = -1;
  for (int unit = 0; unit < n_units; ++unit) {
    const bool more = unit + 1 < n_units;
    // The cross products are summed on their own, where they are small, and join the logits
    // with one addition: added one by one to logits of a few thousand base-2 units they
    // would each be rounded to those logits' last place.
    f32x16 acc, cr;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = cr[r] = 0.f;
    float kbias = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // this quarter has landed; the two behind it may be in flight (four loads each, and a bias with a unit's first)
      fence();
      if (q < 2) __builtin_amdgcn_s_waitcnt(0x0F78);
      else if (more) __builtin_amdgcn_s_waitcnt(0x0F79);
      else if (q == 2) __builtin_amdgcn_s_waitcnt(0x0F74);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      fence();
      u32x4 k[4];
      const unsigned by = (unsigned)slot * 4096u;
      if (q == 0)
        asm volatile(
            "ds_read_b32 %4, %9\n\t"
            "ds_read_b128 %0, %5\n\tds_read_b128 %1, %6\n\tds_read_b128 %2, %7\n\tds_read_b128 %3, %8\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3]), "=&v"(kbias)
            : "v"(qat[0] + by), "v"(qat[1] + by), "v"(qat[2] + by), "v"(qat[3] + by), "v"(qatb) : "memory");
      else
        read_quarter(k, slot);
      // the quarter three ahead takes the place of this one
      if (q == 0) {
        issue_quarter(kplanes, at, 3, slot);
      } else if (more) {
        if (q == 1) find_keys(unit + 1, at), issue_bias(unit + 1);
        issue_quarter(kplanes, at, q - 1, slot);
      }
      slot = slot == 2 ? 0 : slot + 1;
      fence();
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) {
        const int kk = (q >> 1) * 4 + k2;
        if ((q & 1) == 0) {
          acc = mfma16(k[k2], xh[kk], acc);
          cr = mfma16(k[k2], xl[kk], cr);
        } else {
          cr = mfma16(k[k2], xh[kk], cr);
        }
      }
    }
    if (unit * 32 + li >= n_list) kbias = -3.0e38f;  // (behind the list: the last key again, masked)
    // + key bias: A = [bias_j, 1], B = [1, 0]
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 1.0f : kbias, h ? 0.0f : 1.0f, acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += cr[r];
    const float lane_max = max16(acc);
    float tm = lane_max;
    {
      float a = tm, b = tm;
      swap_halves(a, b);
      tm = fmaxf(a, b);  // the row's largest logit of the unit
    }
    // the key of the row's largest logit so far (absolute raw units; lane-private, the two
    // half-waves are merged at the end)
    // (searched only when some lane's largest value of the unit beats what it has)
    if (track && wave_any(lane_max > batch_v)) {
      const int jb = unit * 32 + 4 * h;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float v = acc[r];
        if (v > batch_v) {
          batch_v = v;
          batch_j = jb + 8 * (r / 4) + (r % 4);
        }
      }
    }
    const bool first = !started;
    float cc = -tm * lscale;
    asm volatile("" : "+v"(cc));  // the exponents, the rescale and the result see one number
    cc = first ? cc : fminf(cc, run_c);
    float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      ps0 += fast_exp2(__builtin_fmaf(acc[r], lscale, cc));
      ps1 += fast_exp2(__builtin_fmaf(acc[r + 1], lscale, cc));
    }
    const float resc = first ? 0.f : fast_exp2(cc - run_c);
    run_s = run_s * resc + (ps0 + ps1);
    run_c = cc;
    started = true;
  }
    if (batch_j >= 0 && batch_v > best_v) {
      best_v = batch_v;
      best_j = batch0 + lds_keys[wave][batch_j];
    }
   }
  }
  }

  // ---- the four wavefronts' results become one ----
  {
    const float s = run_s + xor32(run_s), ov = xor32(best_v);
    const int oj = __shfl_xor(best_j, 32, 64);
    if (ov > best_v || (ov == best_v && oj >= 0 && (best_j < 0 || oj < best_j))) best_v = ov, best_j = oj;
    if (h == 0) {
      sh_max[wave][li] = started ? -run_c : kNegBig;
      sh_sum[wave][li] = s;
      sh_top[wave][li] = best_v;
      sh_key[wave][li] = best_j;
    }
    if (lane == 0) sh_count[wave] = n_taken;
  }
  __syncthreads();
  // unit counts for the variant choice on the device (one set of atomics per workgroup: one per wavefront took 17 us
  // of a launch's 51)
  if (args.sel != nullptr && threadIdx.x == 0) {
    unsigned gathered = 0u;
#pragma unroll
    for (int w = 0; w < 4; ++w) gathered += (unsigned)((sh_count[w] + 31) / 32);
    if (!REST) atomicAdd(&args.sel[kSelSkip + blockIdx.x % kSelSlots], (unsigned)(4 * pieces));
    atomicAdd(&args.sel[kSelDmax + sd.ps_q * kDmaxSlots + (blockIdx.x & (kDmaxSlots - 1))], gathered);
  }
  if (row < sd.nq && h == 0) {
  float M2 = kNegBig, s = 0.f, top = -3.0e38f;
  int bj = -1;
#pragma unroll
  for (int w = 0; w < 4; ++w) M2 = fmaxf(M2, sh_max[w][li]);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    s += sh_sum[w][li] * fast_exp2(sh_max[w][li] - M2);
    if (sh_key[w][li] >= 0 && sh_top[w][li] > top) top = sh_top[w][li], bj = sh_key[w][li];  // (of equal ones the smallest key)
  }
  if (sd.splits == 1) {
    if (wave == 0) {
      epilogue_scalar(sd.ep, row, M2, s, 0.f);
      if (track && bj >= 0) sd.best_key[row] = bj;
    }
  } else {
    // (the other partial results are empty, unless the second launch fills them)
    const int mine = REST ? 1 + item % parts : 0;
    for (int part = REST ? (wave == 0 ? mine : sd.splits) : wave; part < (REST ? mine + 1 : sd.splits); part += 4) {
      const size_t pr = (size_t)part * (size_t)sd.nq + (size_t)row;
      *reinterpret_cast<float2*>(&sd.part_ms[2 * pr]) = part == mine ? make_float2(M2, s) : make_float2(kNegBig, 0.f);
      if (sd.part_best != nullptr) sd.part_best[pr] = part == mine ? bj : -1;
    }
  }
  }
  __syncthreads();
  }
}

}  // namespace fs
