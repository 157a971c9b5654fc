// Combines the pieces of a split forward (split.h): O, Od, LSE and mu of the split
// query tiles from their pieces' normalised sums.
#pragma once
#include <type_traits>
#include "attn_fwd.h"
#include "split.h"

namespace dmad {

// One workgroup per wave tile (ROWS queries) of a split item; thread = (lane of the
// tile, one of 4 groups of columns). Bound by reading the partials once. MAGI: a
// piece is its share of the task's own key tiles, empty for a task of fewer tiles
// than pieces, and only the group's rows are written.
template <typename T, int D, bool JVP, int ROWS = 32, bool MAGI = false>
__global__ __launch_bounds__(256) void fwd_combine_kernel(FwdParams p) {
  using P = FwdPart<D, JVP, ROWS>;
  constexpr int GROUPS = ROWS * D / 256;          // 16-byte column groups of a tile's lane
  constexpr int NG = (GROUPS + 3) / 4;            // ... per thread: groups grp, grp + 4, ...
  constexpr int U = NG * (JVP ? 2 : 1) > 8 ? 2 : 4;  // pieces in flight
  const int item = (int)blockIdx.x / P::WAVES, wave = (int)blockIdx.x % P::WAVES;
  const int lane = lane_id(), col = lane % ROWS, half = lane / ROWS, grp = threadIdx.x >> 6;
  if (grp >= GROUPS) return;
  const int per_head = MAGI ? p.T : (p.Lq + 127) / 128;
  const int work = p.sp.whole + item, bh = work / per_head;
  int row0 = (work - bh * per_head) * 128, q_lo = 0, q_hi = p.Lq, ntiles = 0;
  if constexpr (MAGI) {
    const MagiTask t = magi_task(p, work - bh * per_head, 128);
    row0 = t.row0;
    q_lo = t.q_lo;
    q_hi = t.q_hi;
    ntiles = magi_ntiles(p, t, 32);
    if (ntiles == 0) return;  // a group without keys: its first piece wrote the rows
  }
  const int query = row0 + wave * ROWS + col;
  auto empty = [&](int i) { return MAGI && magi_piece(ntiles, i, p.sp.n) == magi_piece(ntiles, i + 1, p.sp.n); };
  const float* part = p.sp.part + (int64_t)item * p.sp.n * P::FLOATS;
  const float* st = part + P::STATS + wave * P::NS * ROWS + col;
  // pieces are taken U at a time with all of their loads in flight together (the
  // partials come from other XCDs' workgroups, about a microsecond away); past
  // the last piece the last one is read again and left out
  const int n = p.sp.n;
  float m = -__builtin_inff();
  for (int i = 0; i < n; i += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = st[(int64_t)min(i + u, n - 1) * P::FLOATS];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (!empty(min(i + u, n - 1))) m = fmaxf(m, v[u]);
    }
  }
  float w = 0.f, mu = 0.f;
  f32x4_t o[NG], c[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) o[g] = c[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < n; i += U) {
    f32x4_t ov[U][NG], cv[U][NG];
    float ms[U], ls[U], mus[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float* pi = part + (int64_t)min(i + u, n - 1) * P::FLOATS;
      const float* si = st + (pi - part);
      ms[u] = si[0];
      ls[u] = si[ROWS];
      if constexpr (JVP) mus[u] = si[2 * ROWS];
      const float* tile = pi + wave * P::NT * P::TILE;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int j = 4 * g + grp < GROUPS ? 4 * g + grp : grp;
        ov[u][g] = split_get(tile, lane, j);
        if constexpr (JVP) cv[u][g] = split_get(tile + P::TILE, lane, j);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i + u >= n) break;
      if (empty(i + u)) continue;
      const float wi = fast_exp2(ms[u] - m) * ls[u];
      w += wi;
      if constexpr (JVP) mu += wi * mus[u];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[g][e] = fmaf(wi, ov[u][g][e], o[g][e]);
          if constexpr (JVP) c[g][e] = fmaf(wi, cv[u][g][e], c[g][e]);
        }
      }
    }
  }
  if (query >= p.Lq || query < q_lo || query >= q_hi) return;
  const float inv = 1.0f / w;
  mu *= inv;
  const int b = bh / p.H, h = bh - b * p.H;
  const int64_t off = b * p.o_sb + h * p.o_sh + (int64_t)query * p.o_sl;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (4 * g + grp >= GROUPS) break;
    const int dc = (4 * g + grp) * (256 / ROWS) + 4 * half;  // a group is 256 / ROWS columns wide
    f32x4_t ov, tv;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ov[e] = o[g][e] * inv;
      tv[e] = c[g][e] * inv - mu * ov[e];
    }
    if constexpr (std::is_same<T, float>::value) {
      *(f32x4_t*)((float*)p.o + off + dc) = ov;
      if constexpr (JVP) *(f32x4_t*)((float*)p.to + off + dc) = tv;
    } else {
      *(u32x2_t*)((char*)p.o + (off + dc) * 2) = u32x2_t{Elem<T>::pack2(ov[0], ov[1]), Elem<T>::pack2(ov[2], ov[3])};
      if constexpr (JVP)
        *(u32x2_t*)((char*)p.to + (off + dc) * 2) = u32x2_t{Elem<T>::pack2(tv[0], tv[1]), Elem<T>::pack2(tv[2], tv[3])};
    }
  }
  if (half == 0 && grp == 0) {
    const int64_t si = (int64_t)bh * p.Lq + query;
    p.lse[si] = (m + __builtin_log2f(w)) * 0.6931471805599453f;
    if constexpr (JVP) p.mu[si] = mu;
  }
}

}  // namespace dmad
