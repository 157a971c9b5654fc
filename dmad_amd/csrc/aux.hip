// Layout kernels around the attention passes (HBM-bound, O(L*D) work).
#include "launch.h"
#include "attn_bwd.h"

namespace dmad {

// Transposed, zero-padded copies of up to six [L, D] operands in one launch: one
// TL (l) x TD (d) tile of one tensor per workgroup through LDS. A thread reads 16
// bytes of two consecutive rows and puts their eight columns as (l, l + 1) pairs
// into the LDS tile, from which 16 bytes of an output row (8 l) leave as they lie:
// 16-byte loads and stores on both sides (TD = 64: whole 128-byte lines; the
// 32-wide tile of heads up to 32 takes twice the rows instead). The pitch of an odd
// number of words keeps the pair stores of a wave on different banks.
// Bound by HBM at large sizes and by the launch at small ones, hence one launch:
// element-wise loads and stores, a launch per tensor, took 14.5 us for each of the
// five copies of a training call (B=4, H=32, 1500 tokens, D=32), 7-9 us for each of
// six at 12 heads of 876 tokens.
template <int TD>
struct TransposeCfg {
  static constexpr int TL = 64 * 64 / TD;  // rows of a tile: 256 threads, one row pair and 8 columns each
  static constexpr int CR = TD / 8;        // 16-byte chunks per tile row
  static constexpr int PITCH = TL / 2 + 1;  // words per LDS row (one column, TL / 2 pairs)
};

template <int TD>
__global__ __launch_bounds__(256) void transpose_pad_kernel(TransposeParams p, int BH) {
  using C = TransposeCfg<TD>;
  __shared__ uint32_t tile[TD * C::PITCH];
  const TransposeParams::Tensor t = p.t[blockIdx.z];
  const int nlt = (t.LP + C::TL - 1) / C::TL;
  if (nlt == 0 || blockIdx.x >= (unsigned)(nlt * BH)) return;  // the grid fits the longest tensor
  const int bh = blockIdx.x / nlt;
  const int b = bh / p.H, h = bh - b * p.H;
  const int l0 = (blockIdx.x - bh * nlt) * C::TL, d0 = blockIdx.y * TD;
  const int tid = threadIdx.x;
  {
    const int chunk = tid % C::CR, pair = tid / C::CR;
    const int l = l0 + 2 * pair, d = d0 + 8 * chunk;
    const uint16_t* x = (const uint16_t*)t.x + b * t.sb + h * t.sh + (int64_t)l * t.sl + d;
    i32x4_t r0 = {0, 0, 0, 0}, r1 = {0, 0, 0, 0};
    if (d < p.D) {
      if (l < t.L) r0 = *(const i32x4_t*)x;
      if (l + 1 < t.L) r1 = *(const i32x4_t*)(x + t.sl);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t u = (uint32_t)r0[e], v = (uint32_t)r1[e];
      tile[(8 * chunk + 2 * e) * C::PITCH + pair] = (u & 0xffff) | (v << 16);
      tile[(8 * chunk + 2 * e + 1) * C::PITCH + pair] = (u >> 16) | (v & 0xffff0000u);
    }
  }
  __syncthreads();
  uint16_t* y = (uint16_t*)t.y + (int64_t)bh * p.DP * t.LP;
  constexpr int CO = C::TL / 8;  // 16-byte chunks per output row of the tile
#pragma unroll
  for (int i = tid; i < TD * CO; i += 256) {
    const int dd = i / CO, c = i % CO;
    const int l = l0 + 8 * c, d = d0 + dd;
    const uint32_t* w = tile + dd * C::PITCH + 4 * c;
    if (d < p.DP && l < t.LP)
      *(i32x4_t*)(y + (int64_t)d * t.LP + l) = i32x4_t{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
  }
}

template <int TD>
static hipError_t launch_transpose(const TransposeParams& p, int BH, hipStream_t s) {
  constexpr int TL = TransposeCfg<TD>::TL;
  int most = 0;
  for (int i = 0; i < p.count; ++i) most = p.t[i].LP > most ? p.t[i].LP : most;
  if (most == 0) return hipSuccess;
  hipLaunchKernelGGL((transpose_pad_kernel<TD>), dim3((most + TL - 1) / TL * BH, (p.DP + TD - 1) / TD, p.count),
                     dim3(256), 0, s, p, BH);
  return hipGetLastError();
}

hipError_t launch_transpose_pad(const TransposeParams& p, int BH, hipStream_t s) {
  if (p.count == 0 || BH == 0) return hipSuccess;
  return p.DP <= 32 ? launch_transpose<32>(p, BH, s) : launch_transpose<64>(p, BH, s);
}


// ---------------------------------------------------------------- backward helpers

template <typename T>
__device__ __forceinline__ float dot8(const uint16_t* a, const uint16_t* b) {
  const i32x4_t x = *(const i32x4_t*)a, y = *(const i32x4_t*)b;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t u = (uint32_t)x[i], w = (uint32_t)y[i];
    s = fmaf(Elem<T>::to_f32((uint16_t)(u & 0xffff)), Elem<T>::to_f32((uint16_t)(w & 0xffff)), s);
    s = fmaf(Elem<T>::to_f32((uint16_t)(u >> 16)), Elem<T>::to_f32((uint16_t)(w >> 16)), s);
  }
  return s;
}

// D/8 consecutive lanes share one query row, each lane reading 16 bytes of O,
// dO (and Od, dOd): every load instruction reads whole rows, and the per-row
// dot products finish with a butterfly over those lanes.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_prep_kernel(PrepParams p) {
  constexpr int LPR = D / 8;        // lanes per row
  constexpr int RPB = 256 / LPR;    // rows per workgroup
  const int sub = threadIdx.x % LPR;
  const int64_t gid = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  const bool live = gid < (int64_t)p.BH * p.LQP;
  const int bh = live ? (int)(gid / p.LQP) : 0, q = live ? (int)(gid - (int64_t)bh * p.LQP) : p.Lq;
  const int b = bh / p.H, h = bh - b * p.H;
  const bool full = p.dto != nullptr;
  float d_o = 0.f, d_to = 0.f, rho = 0.f;
  if (q < p.Lq) {
    const int d = 8 * sub;
    const uint16_t* o = (const uint16_t*)p.o + b * p.o_sb + h * p.o_sh + (int64_t)q * p.o_sl + d;
    const uint16_t* dd = (const uint16_t*)p.dout + b * p.do_sb + h * p.do_sh + (int64_t)q * p.do_sl + d;
    d_o = dot8<T>(dd, o);
    if (full) {
      const uint16_t* to = (const uint16_t*)p.to + b * p.o_sb + h * p.o_sh + (int64_t)q * p.o_sl + d;
      const uint16_t* dt = (const uint16_t*)p.dto + b * p.do_sb + h * p.do_sh + (int64_t)q * p.do_sl + d;
      d_to = dot8<T>(dt, to);
      rho = dot8<T>(dt, o);
    }
  }
#pragma unroll
  for (int m = 1; m < LPR; m <<= 1) {
    d_o += __shfl_xor(d_o, m);
    if (full) {
      d_to += __shfl_xor(d_to, m);
      rho += __shfl_xor(rho, m);
    }
  }
  if (!live || sub != 0) return;
  float lse2 = __builtin_inff(), mu = 0.f;
  if (q < p.Lq) {
    lse2 = p.lse[(int64_t)bh * p.Lq + q] * 1.4426950408889634f;
    if (full) mu = p.mu[(int64_t)bh * p.Lq + q];
  }
  if (p.stats_a) {
    float* s = p.stats_a + ((int64_t)bh * (p.LQP / p.BA) + q / p.BA) * 2 * p.BA + q % p.BA;
    s[0] = lse2;
    s[p.BA] = d_o;
  }
  if (p.stats_b) {
    float* s = p.stats_b + ((int64_t)bh * (p.LQP / 32) + q / 32) * 4 * 32 + q % 32;
    s[0] = lse2;
    s[32] = d_o + d_to - mu * rho;
    s[64] = mu;
    s[96] = rho;
  }
  if (p.stats_bt) {
    float* s = p.stats_bt + ((int64_t)bh * (p.LQP / p.BA) + q / p.BA) * 2 * p.BA + q % p.BA;
    s[0] = lse2;
    s[p.BA] = rho;
  }
}

template <typename T>
static hipError_t launch_prep_t(const PrepParams& p, hipStream_t s) {
  const int64_t rows = (int64_t)p.BH * p.LQP;
  auto go = [&](auto kern, int lpr) {
    const int64_t nb = (rows * lpr + 255) / 256;
    hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(256), 0, s, p);
  };
  switch (p.D) {
    case 16: go(bwd_prep_kernel<T, 16>, 2); break;
    case 32: go(bwd_prep_kernel<T, 32>, 4); break;
    case 64: go(bwd_prep_kernel<T, 64>, 8); break;
    case 128: go(bwd_prep_kernel<T, 128>, 16); break;
    case 256: go(bwd_prep_kernel<T, 256>, 32); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_bwd_prep(const PrepParams& p, int dtype, hipStream_t s) {
  if ((int64_t)p.BH * p.LQP == 0) return hipSuccess;
  return dtype == 0 ? launch_prep_t<__bf16>(p, s) : launch_prep_t<_Float16>(p, s);
}

}  // namespace dmad
