// Splitting the last work items of a launch over the loop they run.
//
// The attention passes give one workgroup one work item: a tile of queries (or
// keys) of one head, walked against all keys (or queries). A grid that is not a
// whole number of rounds over the chip leaves most CUs idle in its last round:
// 588 items of one workgroup per CU run 2.3 rounds of work in the time of 3, and
// 156 items keep 100 of the 256 CUs idle throughout. A split launch runs the
// items of the full rounds as before and cuts each of the `rest` items after them
// into `n` pieces along its loop. A piece writes its fp32 accumulators to a
// partial buffer, and a second, small kernel sums an item's pieces in a fixed
// order (no atomics: repeated calls agree bit for bit) and writes the outputs.
// What a launch does is decided on the host, on every call (plan_split, 0.1-0.7 us),
// as a function of the items, the steps of an item's loop and the costs of the kernel
// that runs it alone.
#pragma once
#include <type_traits>
#include "common.h"

namespace dmad {

// Kernel arguments of a split launch (rest == 0: an ordinary launch).
struct SplitParams {
  int whole;    // work items [0, whole) run whole, one workgroup each
  int rest;     // work items [whole, whole + rest) run in pieces
  int n;        // pieces per split item
  int len;      // steps of pieces 0 .. n - 2; the last piece takes what is left
  float* part;  // partials, [rest][n] blocks
};

// What this workgroup of a split launch runs.
struct SplitWork {
  int item;      // work item; -1: none (a padding workgroup of the last ids)
  int piece;     // -1: the whole item
  int slot;      // (item - whole) n + piece: index of the piece's partial block
  int beg, end;  // steps of the item's loop
};

// Workgroups of a split launch: the whole items, then per XCD its share of the
// split items, piece-major, so that the equal, longer pieces start first and a
// shorter last piece fills the gaps they leave, and an item's pieces (which read
// the same rows of one head) share an L2.
__host__ __device__ inline int64_t split_grid(int64_t whole, int64_t rest, int64_t n) {
  return whole + 8 * ((rest + 7) / 8) * n;
}

__device__ __forceinline__ SplitWork split_work(const SplitParams& sp, int xcd_order, int steps) {
  const int bid = (int)blockIdx.x;
  if (bid < sp.whole) return SplitWork{xcd_order ? xcd_remap(bid, sp.whole) : bid, -1, 0, 0, steps};
  const int id = bid - sp.whole, xcd = id & 7, k = id >> 3;
  const int per = sp.rest >> 3, rem = sp.rest & 7;
  const int first = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  const int mine = per + (xcd < rem ? 1 : 0);  // split items of this XCD
  if (mine == 0 || k >= mine * sp.n) return SplitWork{-1, 0, 0, 0, 0};
  const int piece = k / mine, j = first + (k - piece * mine);
  const int beg = piece * sp.len;
  return SplitWork{sp.whole + j, piece, j * sp.n + piece, beg, piece + 1 < sp.n ? beg + sp.len : steps};
}

// Partial block of one piece: per wave and tensor, the wave's 32 x D accumulator
// tile in the 32x32 MFMA layout (lane: row lane % 32, columns 32 d + 8 jj +
// 4 (lane / 32) + 0..3), 16 bytes per lane and (d, jj), so every store and load
// instruction moves 1 KiB in a row.
template <int D>
__host__ __device__ constexpr int split_tile_floats() { return 32 * D; }
template <int D>
__device__ __forceinline__ void split_put(float* tile, int lane, int d, int jj, f32x4_t v) {
  *(f32x4_t*)(tile + ((4 * d + jj) * 64 + lane) * 4) = v;
}
__device__ __forceinline__ f32x4_t split_get(const float* tile, int lane, int g) {
  return *(const f32x4_t*)(tile + (g * 64 + lane) * 4);
}

// ---------------------------------------------------------------- host: the plan
// Costs of one kernel of a split launch, in microseconds on an MI355X whose clock the
// power limit does not lower: those of launches of a few rounds. Long launches take
// longer (the 64-wide query pass of 4 x 32 heads of 2048 tokens 201 us, 149 by its
// costs), so that what a split of theirs saves is overrated by as much.
struct SplitCost {
  int occ;          // workgroups that fit a CU
  float step;       // one step of the loop, one workgroup per CU
  float shared;     // factor on a step's time per further workgroup on the CU
  float fixed;      // a workgroup's time outside its loop
  int part_bytes;   // partial block of one piece
};
struct SplitPlan {
  int64_t whole = 0, rest = 0, grid = 0, bytes = 0;
  int n = 1, len = 0;
};

constexpr int kSplitCus = 256;
constexpr int kSplitMaxPieces = 64;
constexpr int64_t kSplitMaxBytes = (int64_t)128 << 20;  // partials of one launch

// Time of `a` workgroups of la steps followed by `b` of lb <= la on `slots` slots,
// in that order.
inline double split_queue(int64_t slots, int64_t a, double ta, int64_t b, double tb) {
  const double t = (double)(a / slots) * ta;  // full rounds of the long ones
  const int64_t busy = a % slots;             // slots busy for another ta
  if (b == 0) return t + (busy ? ta : 0.);
  double best = 0.;
  for (int64_t r = 1;; ++r) {  // r short ones in a row on a free slot
    const double end = (double)r * tb;
    const int64_t after = end > ta ? (int64_t)((end - ta) / tb) : 0;
    if ((slots - busy) * r + busy * after >= b) {
      best = end;
      break;
    }
  }
  if (busy && best < ta) best = ta;
  return t + best;
}

// The same for a grid of `a` and then `b` workgroups per XCD. Workgroups go to the
// XCDs in turn, and within an XCD to its four engines of eight CUs in turn, whether
// or not another engine is idle: 168 fp32 tiles of 55 steps in pieces of 37 and 18
// took 55 steps' time (680 us, whole 671), because the engine that got six of the 21
// long pieces got five short ones as well, where the chip's 88 free CUs would have
// run all 168 in 37; in three even pieces they take 490 us. Forty shapes whose pieces
// this changed, against counting the chip's CUs as one pool: all 1-58% faster (plain
// and JVP 2-4%, backward 2-29%, fp32 2-58%).
inline double split_makespan(const SplitCost& k, int64_t a, double la, int64_t b, double lb) {
  constexpr int64_t kEngines = 4, kCus = kSplitCus / 8 / kEngines;
  const int64_t total = a + b, most = (total + kEngines - 1) / kEngines, per = (most + kCus - 1) / kCus;
  if (total == 0) return 0.;
  const int occ = (int)(per < k.occ ? per : k.occ);  // workgroups sharing a CU
  const double step = k.step * (1. + k.shared * (occ - 1));
  double t = 0.;
  for (int64_t e = 0; e < kEngines; ++e) {
    const int64_t longs = (a + kEngines - 1 - e) / kEngines, all = (total + kEngines - 1 - e) / kEngines;
    const double te = split_queue(kCus * occ, longs, la * step + k.fixed, all - longs, lb * step + k.fixed);
    if (te > t) t = te;
  }
  return t;
}

// The plan that runs the last `rest` of `items` work items in n pieces, `len` steps each
// but the last.
inline SplitPlan split_cut(int64_t items, int64_t rest, int n, int len, int64_t part_bytes) {
  SplitPlan pl;
  pl.whole = items - rest;
  pl.rest = rest;
  pl.n = n;
  pl.len = len;
  pl.grid = split_grid(pl.whole, rest, n);
  pl.bytes = rest * n * part_bytes;
  return pl;
}

// How to run `items` work items of `steps` steps: in full rounds, then the rest in
// the pieces that finish soonest by the costs above (even_only: in pieces of one
// length), where that saves at least a twentieth of the launch and 8 us (of a backward
// in several launch pairs: of all pairs, of which only the last is cut): the second
// kernel and its scratch cost the host 4-5 us, and calls that short wait for the
// host (a training call of two 64-wide heads of 999 tokens: 45 us of kernels split,
// 67 whole, in 200 us of host time, 12 of them for the three splits). The partials
// are written and read once, at about 3.3 TB/s, by a second kernel that takes 5 us
// at least (all measured). Over 56 random shapes, each also cut by hand into 2 to 8
// pieces, the choice was within 3% of the best in 48.
inline SplitPlan plan_split(int64_t items, int64_t steps, const SplitCost& k, bool even_only = false) {
  SplitPlan pl;
  pl.whole = items;
  pl.grid = items;
  const int64_t slots = (int64_t)kSplitCus * k.occ, rest = items % slots, rounds = items / slots;
  if (rest == 0 || steps < 4) return pl;
  const double round = (1. + k.shared * (k.occ - 1)) * k.step * (double)steps + k.fixed;
  const int64_t mine = (rest + 7) / 8;  // items of the fullest XCD
  const double as_is = split_makespan(k, mine, (double)steps, 0, 0.);
  const double least = 0.05 * (as_is + (double)rounds * round);
  double best = as_is - (least > 8. ? least : 8.);
  for (int64_t n = 2; n <= kSplitMaxPieces && n <= steps && rest * n * k.part_bytes <= kSplitMaxBytes; ++n) {
    const double extra = 5. + 2. * (double)(rest * n) * k.part_bytes / 3.3e6;
    const int64_t even = (steps + n - 1) / n;
    // the shorter last piece runs in the slots the n - 1 long ones leave free
    const int64_t left = slots - (n - 1) * rest;
    int64_t lens[3] = {even, 0, 0};
    if (!even_only && left > 0 && left < rest) {
      const int64_t q = (rest + left - 1) / left;  // short pieces in a row (an engine may get one more)
      lens[1] = (steps * q + (n - 1) * q) / ((n - 1) * q + 1);
      lens[2] = (steps * (q + 1) + (n - 1) * (q + 1)) / ((n - 1) * (q + 1) + 1);
    }
    for (const int64_t a : lens) {
      const int64_t b = steps - (n - 1) * a;
      if (a < 1 || b < 1 || b > a) continue;
      const double t = split_makespan(k, (n - 1) * mine, (double)a, mine, (double)b) + extra;
      if (t < best) {
        best = t;
        pl.n = (int)n;
        pl.len = (int)a;
      }
    }
  }
  return pl.n > 1 ? split_cut(items, rest, pl.n, pl.len, k.part_bytes) : pl;
}

// ---------------------------------------------------------------- forward
// Partial block of the forward, 128 queries: per wave [O (, C)][ROWS x D], then per
// wave [m, l (, mu)][ROWS]: l the sum of exp2(score - m) over the piece's keys,
// O = O~ / l and C = C~ / l. A piece weighs exp2(m) l; m + log2(l) in one float
// would lose l beside scores of a large common value (2^24 and more: all of it).
// ROWS = 32: tiles as above. ROWS = 16 (fp32 operands): the
// 16x16 layout (lane: row lane % 16, columns 16 d + 4 (lane / 16) + 0..3), again
// 16 bytes per lane and d.
template <int D, bool JVP, int ROWS = 32>
struct FwdPart {
  static constexpr int WAVES = 128 / ROWS;
  static constexpr int NT = JVP ? 2 : 1;
  static constexpr int TILE = ROWS * D;
  static constexpr int STATS = WAVES * NT * TILE;
  static constexpr int NS = JVP ? 3 : 2;
  static constexpr int FLOATS = STATS + WAVES * NS * ROWS;
};

// ---------------------------------------------------------------- backward
// Partial block of a backward pass: [waves][tensors][32 x D] accumulator tiles,
// unscaled. The passes' pieces add up without weights.
struct SplitSumParams {
  SplitParams sp;
  void* out[2];  // dK, dV or dQ, dQd; out[1] may be null (its tiles are then not read)
  int64_t sb[2], sh[2], sl[2];
  float scale[2];
  int H, L;      // rows of an output's head
  int tiles;     // work items per head
  int bh0;       // head of work item 0
};

// One workgroup per wave tile (32 rows) of a split item, four pieces' loads in
// flight at a time (as fwd_combine_kernel). WAVES waves per work item, NT tiles
// per wave.
template <typename T, int D, int WAVES, int NT>
__global__ __launch_bounds__(256) void split_sum_kernel(SplitSumParams p) {
  constexpr int TILE = split_tile_floats<D>(), FLOATS = WAVES * NT * TILE;
  const int item = (int)blockIdx.x / WAVES, wave = (int)blockIdx.x - item * WAVES;
  const int lane = lane_id(), col = lane & 31, half = lane >> 5, grp = threadIdx.x >> 6;
  const int work = p.sp.whole + item, slice = work / p.tiles, tile_no = work - slice * p.tiles;
  const int bh = p.bh0 + slice, b = bh / p.H, h = bh - b * p.H;
  const int row = (tile_no * WAVES + wave) * 32 + col;
  const float* part = p.sp.part + (int64_t)item * p.sp.n * FLOATS + wave * NT * TILE;
  constexpr int U = 4, NG = D / 32;
  const int n = p.sp.n;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (p.out[t] == nullptr) continue;
    f32x4_t acc[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) acc[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < n; i += U) {
      f32x4_t v[U][NG];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* tile = part + (int64_t)min(i + u, n - 1) * FLOATS + t * TILE;
#pragma unroll
        for (int g = 0; g < NG; ++g) v[u][g] = split_get(tile, lane, 4 * g + grp);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (i + u >= n) break;
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[g] += v[u][g];
      }
    }
    if (row < p.L) {
      char* out = (char*)p.out[t] + (b * p.sb[t] + h * p.sh[t] + (int64_t)row * p.sl[t]) * 2;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const f32x4_t a = acc[g] * p.scale[t];
        *(u32x2_t*)(out + (32 * g + 8 * grp + 4 * half) * 2) =
            u32x2_t{Elem<T>::pack2(a[0], a[1]), Elem<T>::pack2(a[2], a[3])};
      }
    }
  }
}

}  // namespace dmad
