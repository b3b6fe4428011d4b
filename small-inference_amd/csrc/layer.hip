// The decoder layer's own operations around the paged attention, for gfx950: projections of a few tokens fused with
// the operations next to them, and the same elementwise operations alone for the large batches whose projections
// are left to the GEMM library. bf16 in and out, fp32 inside.
//
// Reference: engine/model.py:101-175 (RMSNorm, fused QKV with bias, rotary embedding, SwiGLU MLP, residuals), there
// about 30 separate torch operations a layer.
#include "decode_common.h"

namespace sipa {

// ---- skinny_linear: y = epilogue(norm(x) W^T), few tokens -----------------------------------------------------------
//
// Bound: the weights' read from HBM and, for a layer's 2 to 17 MB, as much the latency of one launch: load, reduce,
// store. So a workgroup owns whole rows of W (16 rows times RT tiles, all of K), its WV waves take 64-channel slices
// of K, the loads of two slices ahead are in flight, and nothing is written before the result: one launch, no
// partials, no second pass. Against a GEMM library's tiles (56 workgroups of a 4864-long serial loop for the MLP's
// down projection) every wave's share of K is a few loads.
//
// W enters the MFMA as the A operand straight from memory, lane (r, q4) holding row r's channels 16 q4 .. 16 q4 + 15
// of a slice (four lanes read one 128-byte line of a row), x as the B operand in the same channel order, so D[n][t]
// comes out with lane (t, q4) holding outputs n = 4 q4 .. 4 q4 + 3 of token t. The waves' partial sums meet in LDS.
//
// RMSNorm (NORM): the row scale rstd[t] factors out of the product, so x * w_norm is rounded to bf16 for the MFMA
// (one rounding, where norm-then-multiply in bf16 has two), the squares of x are summed on the way, and the
// accumulators are scaled in the epilogue: no pass over x before the product and no barrier.
//
// Split K (RESIDUAL): 896 outputs are 56 row tiles, and a CU's share of a 4864-long K, 155 KB, is more than one CU has
// in flight; four workgroups share it and the last one adds their sums.
//
// Measured in a graph, weights from memory, 8 tokens, against the GEMM library and the operations around it one by one
// (us): norm + QKV 1152 x 896 + bias + rotary 4.8 (library product 5.5, with 12 launches around it); o 896 x 896 +
// residual 4.0 (5.5 + 2); norm + gate/up 9728 x 896 + SwiGLU 8.8 (8.5 + 10 launches); down 896 x 4864 + residual 7.0
// with four splits, 8.8 with two, 11.6 with one (16.8 + 2). A whole decode step of 8 sequences (24 layers) 3018 -> 972.
//
// Row tiles: for ROPE and SILU a tile's 16 rows are 8 rows and their 8 partners (channels c and c + D/2 of a head;
// gate and up), so one thread holds both halves of a pair.
enum { kEpiResidual = 0, kEpiRope = 1, kEpiSilu = 2 };

struct LinearArgs {
  const uint16_t* x;       // [T, K] rows
  int64_t x_st;
  const uint16_t* w;       // [N, K] contiguous
  const uint16_t* norm_w;  // [K] (NORM)
  float eps;
  const uint16_t* bias;    // [N] or null
  const uint16_t* res;     // [T, N] rows (RESIDUAL) or null
  int64_t res_st;
  uint16_t* out;
  int64_t out_st;
  const uint16_t* cos;     // [T, D] (ROPE)
  const uint16_t* sin;     // [T, D], the sign of rotate-half folded in
  int32_t T, K, D, rot;    // rot: output channels that are rotated (whole heads, the first ones)
  int32_t tiles;           // row tiles in all
  int32_t inter;           // SILU: gate rows (the up rows follow)
  int32_t units;           // 64-channel slices of K a workgroup takes
  int32_t splits;          // workgroups that share a row tile's K (RESIDUAL)
  float* part;             // [row tile][token group][splits][RT][TT][256] partial sums
  int32_t* counters;       // [row tile][token group] workgroups done, zero between calls
};

template <int EPI>
__device__ __forceinline__ int linear_row(const LinearArgs& a, int tile, int r) {
  if (EPI == kEpiSilu) return tile * 8 + (r & 7) + (r < 8 ? 0 : a.inter);
  if (EPI == kEpiRope && tile * 16 < a.rot) {
    const int per = a.D >> 4;  // tiles a head
    const int head = tile / per, c0 = (tile - head * per) * 8;
    return head * a.D + c0 + (r & 7) + (r < 8 ? 0 : a.D >> 1);
  }
  return tile * 16 + r;
}

__device__ __forceinline__ u32x4 weight_load(const uint16_t* p) { return stream_load(p); }

// x * w per channel, rounded to bf16, and the sum of x's squares.
__device__ __forceinline__ u32x4 scale_channels(u32x4 x, u32x4 w, float& ss) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = __uint_as_float(x[i] << 16), b = __uint_as_float(x[i] & 0xffff0000u);
    const float c = __uint_as_float(w[i] << 16), d = __uint_as_float(w[i] & 0xffff0000u);
    ss = fmaf(a, a, ss);
    ss = fmaf(b, b, ss);
    o[i] = pack_bf16x2(a * c, b * d);
  }
  return o;
}

// U: 64-channel slices of a stage; NST: stages in flight (one where the wave's whole share is one stage).
template <int EPI, bool NORM, int TT, int RT, int WV, int U, int NST>
__global__ void __launch_bounds__(64 * WV) skinny_linear(const LinearArgs a) {
  __shared__ __align__(16) float red[WV][RT][TT][256];
  __shared__ float ssq[NORM ? WV : 1][TT * 16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r = lane & 15, q4 = lane >> 4;
  const int tile0 = blockIdx.x * RT;
  const int t_base = blockIdx.y * (16 * TT);
  // slices [unit0, unit1) of K are this workgroup's; wave v takes unit0 + v, unit0 + v + WV, ...
  const int unit0 = blockIdx.z * a.units, unit1 = min(unit0 + a.units, a.K >> 6);
  const int units = unit1 - unit0;
  const int mine = units > wave ? (units - wave + WV - 1) / WV : 0;

  const uint16_t* wrow[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
    wrow[i] = a.w + (int64_t)linear_row<EPI>(a, min(tile0 + i, a.tiles - 1), r) * a.K + 16 * q4;
  const uint16_t* xrow[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) xrow[i] = a.x + (int64_t)min(t_base + 16 * i + r, a.T - 1) * a.x_st + 16 * q4;
  const uint16_t* nrow = NORM ? a.norm_w + 16 * q4 : nullptr;

  struct Stage {
    u32x4 w[U][RT][2], x[U][TT][2], n[U][2];
  };
  Stage st[NST];
  // Slices past the wave's last re-read its last one and are not multiplied.
  auto load = [&](Stage& s, int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = 64 * (unit0 + wave + WV * min(k + u, mine - 1));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < RT; ++i) s.w[u][i][h] = weight_load(wrow[i] + c + 8 * h);
#pragma unroll
        for (int i = 0; i < TT; ++i) s.x[u][i][h] = *(const u32x4*)(xrow[i] + c + 8 * h);
        if (NORM) s.n[u][h] = *(const u32x4*)(nrow + c + 8 * h);
      }
    }
  };
  f32x4 acc[RT][TT];
  float ss[TT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < TT; ++j) ss[j] = 0.f;
  auto multiply = [&](Stage& s, int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // A slice past the wave's share is masked to zeros, not branched around: with a branch here the compiler sinks
      // the slice's loads into it, and their latencies add up instead of overlapping.
      const uint32_t live = k + u < mine ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) s.w[u][i][h] &= live;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          u32x4 xv = s.x[u][j][h] & live;
          if (NORM) xv = scale_channels(xv, s.n[u][h], ss[j]);
#pragma unroll
          for (int i = 0; i < RT; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, s.w[u][i][h]),
                                                                __builtin_bit_cast(bf16x8, xv), acc[i][j], 0, 0, 0);
        }
    }
  };
  if (mine > 0) {
    load(st[0], 0);
    if constexpr (NST == 1) {
      multiply(st[0], 0);
    } else {
      if (mine > U) load(st[1], U);
      for (int k = 0; k < mine; k += 2 * U) {
        multiply(st[0], k);
        if (k + 2 * U < mine) load(st[0], k + 2 * U);
        if (k + U < mine) {
          multiply(st[1], k + U);
          if (k + 3 * U < mine) load(st[1], k + 3 * U);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) *(f32x4*)&red[wave][i][j][lane * 4] = acc[i][j];
  if (NORM) {
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      const float s = sum_over_rows(ss[j]);
      if (q4 == 0) ssq[wave][16 * j + r] = s;
    }
  }
  __syncthreads();

  if (EPI == kEpiResidual && a.splits > 1) {
    // Split K: every workgroup stores its sums through to memory; the last to arrive adds them in split order.
    constexpr int E = RT * TT * 256;
    const int pair = blockIdx.y * gridDim.x + blockIdx.x;
    float* const part = a.part + (int64_t)pair * a.splits * E;
    float* const flat = &red[0][0][0][0];
    __shared__ int last;
    for (int e = threadIdx.x; e < E; e += 64 * WV) {
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < WV; ++v) s += flat[v * E + e];
      store_coherent(part + blockIdx.z * E + e, s);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      last = __hip_atomic_fetch_add(a.counters + pair, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             a.splits - 1;
    __syncthreads();
    if (!last) return;
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(part, (short)0, a.splits * E * 4, 0x00020000);
    for (int e = threadIdx.x; e < E; e += 64 * WV) {
      float s = 0.f;
      for (int v0 = 0; v0 < a.splits; v0 += 4) {
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          x[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                               rows, (min(v0 + u, a.splits - 1) * E + e) * 4, 0, kAuxSc1));
#pragma unroll
        for (int u = 0; u < 4; ++u) s += v0 + u < a.splits ? x[u] : 0.f;
      }
      flat[e] = s;
#pragma unroll
      for (int v = 1; v < WV; ++v) flat[v * E + e] = 0.f;
    }
    if (threadIdx.x == 0)
      __hip_atomic_store(a.counters + pair, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
  }

  // Pairs (n, n + 8) of a tile's outputs for one token; eight neighbouring threads store eight neighbouring channels.
  for (int p = threadIdx.x; p < RT * TT * 128; p += 64 * WV) {
    const int n = p & 7, tl = (p >> 3) & 15, j = (p >> 7) % TT, i = p / (128 * TT);
    const int t = t_base + 16 * j + tl, tile = tile0 + i;
    if (t >= a.T || tile >= a.tiles) continue;
    const int at = ((n >> 2) * 16 + tl) * 4 + (n & 3);  // output n's place; n + 8 is 128 words on
    float lo = 0.f, hi = 0.f;
#pragma unroll
    for (int v = 0; v < WV; ++v) {
      lo += red[v][i][j][at];
      hi += red[v][i][j][at + 128];
    }
    if (NORM) {
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < WV; ++v) s += ssq[v][16 * j + tl];
      const float rstd = rsqrtf(s / (float)a.K + a.eps);
      lo *= rstd;
      hi *= rstd;
    }
    const int nlo = linear_row<EPI>(a, tile, n), nhi = linear_row<EPI>(a, tile, n + 8);
    if (EPI == kEpiSilu) {
      a.out[t * a.out_st + nlo] = f32_to_bf16_bits(lo / (1.f + expf(-lo)) * hi);
      continue;
    }
    if (a.bias != nullptr) {
      lo += bf16_bits_to_f32(a.bias[nlo]);
      hi += bf16_bits_to_f32(a.bias[nhi]);
    }
    if (EPI == kEpiRope && tile * 16 < a.rot) {
      const int c = nlo % a.D, c2 = c + (a.D >> 1);
      const uint16_t *cs = a.cos + (int64_t)t * a.D, *sn = a.sin + (int64_t)t * a.D;
      const float x0 = lo, x1 = hi;
      lo = x0 * bf16_bits_to_f32(cs[c]) + x1 * bf16_bits_to_f32(sn[c]);
      hi = x1 * bf16_bits_to_f32(cs[c2]) + x0 * bf16_bits_to_f32(sn[c2]);
    }
    if (EPI == kEpiResidual && a.res != nullptr) {
      lo += bf16_bits_to_f32(a.res[t * a.res_st + nlo]);
      hi += bf16_bits_to_f32(a.res[t * a.res_st + nhi]);
    }
    a.out[t * a.out_st + nlo] = f32_to_bf16_bits(lo);
    a.out[t * a.out_st + nhi] = f32_to_bf16_bits(hi);
  }
}

template <int EPI, bool NORM, int TT, int RT, int WV, int U, int NST>
static void launch_linear(LinearArgs& a, hipStream_t st) {
  const dim3 grid((a.tiles + RT - 1) / RT, (a.T + 16 * TT - 1) / (16 * TT), a.splits);
  skinny_linear<EPI, NORM, TT, RT, WV, U, NST><<<grid, 64 * WV, 0, st>>>(a);
}

template <int EPI, bool NORM>
static void dispatch_linear(LinearArgs& a, hipStream_t st) {
  const int units = a.K >> 6;
  a.units = (units + a.splits - 1) / a.splits;
  a.splits = (units + a.units - 1) / a.units;
  if (a.T <= 16) {
    if (a.units <= 16) return launch_linear<EPI, NORM, 1, 1, 8, 2, 1>(a, st);
    if (a.units <= 24) return launch_linear<EPI, NORM, 1, 1, 8, 3, 1>(a, st);
    if constexpr (!NORM) {
      if (a.units >= 64) return launch_linear<EPI, NORM, 1, 1, 16, 2, 2>(a, st);
    }
    return launch_linear<EPI, NORM, 1, 1, 8, 2, 2>(a, st);
  }
  const int tt = a.T <= 32 ? 2 : 4;
  if (a.tiles >= 512) {  // two row tiles a workgroup share its x loads and still fill the chip
    if (tt == 2) return launch_linear<EPI, NORM, 2, 2, 8, 1, 2>(a, st);
    return launch_linear<EPI, NORM, 4, 2, 8, 1, 2>(a, st);
  }
  if (a.units <= 16) {
    if (tt == 2) return launch_linear<EPI, NORM, 2, 1, 8, 2, 1>(a, st);
    return launch_linear<EPI, NORM, 4, 1, 8, 2, 1>(a, st);
  }
  if (tt == 2) return launch_linear<EPI, NORM, 2, 1, 8, NORM ? 1 : 2, 2>(a, st);
  return launch_linear<EPI, NORM, 4, 1, 8, NORM ? 1 : 2, 2>(a, st);
}

// ---- the elementwise operations alone (large batches) -----------------------------------------------------------------
//
// Bound: HBM or L2 traffic of one read and one write, 16 bytes a lane; at a few hundred tokens, launch latency. Measured
// at 128 x 896 / 128 x 4864 in a graph: norm with residual 3.0 us (9 torch launches before), rotary 2.1 (4), SwiGLU 2.6
// (2); an empty launch there is about 2.

// out = bf16(bf16(x * rstd) * w), x = a (+ b rounded to bf16, stored to sum): one wave a row, the row in registers.
template <int CH>
__global__ void __launch_bounds__(256) rms_norm_kernel(const uint16_t* __restrict__ x, int64_t x_st,
                                                       const uint16_t* __restrict__ add, int64_t add_st,
                                                       const uint16_t* __restrict__ w, float eps,
                                                       uint16_t* __restrict__ sum, int64_t sum_st,
                                                       uint16_t* __restrict__ out, int64_t out_st, int T, int K) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  u32x4 v[CH];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = 8 * (lane + 64 * i);
    v[i] = u32x4{0, 0, 0, 0};
    if (c < K) v[i] = *(const u32x4*)(x + t * x_st + c);
    if (add != nullptr && c < K) {
      const u32x4 d = *(const u32x4*)(add + t * add_st + c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[i][e] = pack_bf16x2(__uint_as_float(v[i][e] << 16) + __uint_as_float(d[e] << 16),
                              __uint_as_float(v[i][e] & 0xffff0000u) + __uint_as_float(d[e] & 0xffff0000u));
      *(u32x4*)(sum + t * sum_st + c) = v[i];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = __uint_as_float(v[i][e] << 16), hi = __uint_as_float(v[i][e] & 0xffff0000u);
      ss = fmaf(lo, lo, ss);
      ss = fmaf(hi, hi, ss);
    }
  }
  const float rstd = rsqrtf(wave_sum(ss) / (float)K + eps);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = 8 * (lane + 64 * i);
    if (c >= K) continue;
    const u32x4 g = *(const u32x4*)(w + c);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t n = pack_bf16x2(__uint_as_float(v[i][e] << 16) * rstd,
                                     __uint_as_float(v[i][e] & 0xffff0000u) * rstd);
      o[e] = pack_bf16x2(__uint_as_float(n << 16) * __uint_as_float(g[e] << 16),
                         __uint_as_float(n & 0xffff0000u) * __uint_as_float(g[e] & 0xffff0000u));
    }
    *(u32x4*)(out + t * out_st + c) = o;
  }
}

// Rotary embedding in place on the first H heads of rows [T, >= H D]: a thread takes 8 channels and their partners.
__global__ void __launch_bounds__(256) rope_kernel(uint16_t* __restrict__ x, int64_t x_st,
                                                   const uint16_t* __restrict__ cos,
                                                   const uint16_t* __restrict__ sin, int T, int H, int D) {
  const int per_head = D >> 4, per = H * per_head;
  const int id = blockIdx.x * 256 + threadIdx.x;
  const int t = id / per;
  if (t >= T) return;
  const int e = id - t * per, h = e / per_head, c = 8 * (e - h * per_head);
  uint16_t* p = x + t * x_st + h * D + c;
  const uint16_t *cs = cos + (int64_t)t * D + c, *sn = sin + (int64_t)t * D + c;
  const int half = D >> 1;
  const u32x4 a = *(const u32x4*)p, b = *(const u32x4*)(p + half);
  const u32x4 c0 = *(const u32x4*)cs, c1 = *(const u32x4*)(cs + half);
  const u32x4 s0 = *(const u32x4*)sn, s1 = *(const u32x4*)(sn + half);
  u32x4 lo, hi;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    auto f = [](uint32_t u, int k) { return __uint_as_float(k ? u & 0xffff0000u : u << 16); };
    lo[i] = pack_bf16x2(f(a[i], 0) * f(c0[i], 0) + f(b[i], 0) * f(s0[i], 0),
                        f(a[i], 1) * f(c0[i], 1) + f(b[i], 1) * f(s0[i], 1));
    hi[i] = pack_bf16x2(f(b[i], 0) * f(c1[i], 0) + f(a[i], 0) * f(s1[i], 0),
                        f(b[i], 1) * f(c1[i], 1) + f(a[i], 1) * f(s1[i], 1));
  }
  *(u32x4*)p = lo;
  *(u32x4*)(p + half) = hi;
}

// out[t, i] = silu(gu[t, i]) * gu[t, I + i], 8 channels a thread.
__global__ void __launch_bounds__(256) silu_mul_kernel(const uint16_t* __restrict__ gu, int64_t gu_st,
                                                       uint16_t* __restrict__ out, int64_t out_st, int T, int I) {
  const int per = I >> 3;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int t = (int)(id / per);
  if (t >= T) return;
  const int c = 8 * (int)(id - (int64_t)t * per);
  const u32x4 g = *(const u32x4*)(gu + t * gu_st + c), u = *(const u32x4*)(gu + t * gu_st + I + c);
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float g0 = __uint_as_float(g[i] << 16), g1 = __uint_as_float(g[i] & 0xffff0000u);
    const float u0 = __uint_as_float(u[i] << 16), u1 = __uint_as_float(u[i] & 0xffff0000u);
    o[i] = pack_bf16x2(g0 / (1.f + expf(-g0)) * u0, g1 / (1.f + expf(-g1)) * u1);
  }
  *(u32x4*)(out + t * out_st + c) = o;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

static int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SIPA_OK : fail(SIPA_EHIP, "%s: %s", what, hipGetErrorString(e));
}

}  // namespace sipa

using namespace sipa;

extern "C" int32_t sipa_fused_linear(const sipa_linear_params* p, void* stream) {
  SIPA_CHECK(p != nullptr && p->struct_size == (int32_t)sizeof(sipa_linear_params), SIPA_EINVAL,
             "sipa_linear_params: wrong size");
  SIPA_CHECK(p->num_tokens >= 0 && p->in_features > 0 && p->out_features > 0, SIPA_EINVAL, "linear: bad sizes");
  if (p->num_tokens == 0) return SIPA_OK;
  SIPA_CHECK(p->num_tokens <= 1 << 20 && p->out_features <= 1 << 24 && p->in_features <= 1 << 20, SIPA_EUNSUPPORTED,
             "linear: sizes out of range");
  SIPA_CHECK(p->in_features % 64 == 0, SIPA_EUNSUPPORTED, "linear: in_features %d is not a multiple of 64",
             p->in_features);
  SIPA_CHECK(p->x && p->weight && p->out, SIPA_EINVAL, "linear: null pointer");
  SIPA_CHECK(aligned16(p->x) && aligned16(p->weight) && aligned16(p->norm_weight) && p->x_stride % 8 == 0,
             SIPA_EUNSUPPORTED, "linear: x, weight and norm weight need 16-byte rows");
  SIPA_CHECK(p->x_stride >= 0 && p->out_stride >= 0 && p->res_stride >= 0, SIPA_EINVAL, "linear: negative stride");
  SIPA_CHECK(p->norm_weight == nullptr || p->eps >= 0.f, SIPA_EINVAL, "linear: eps");
  LinearArgs a{};
  a.x = (const uint16_t*)p->x, a.x_st = p->x_stride, a.w = (const uint16_t*)p->weight;
  a.norm_w = (const uint16_t*)p->norm_weight, a.eps = p->eps, a.bias = (const uint16_t*)p->bias;
  a.res = (const uint16_t*)p->residual, a.res_st = p->res_stride;
  a.out = (uint16_t*)p->out, a.out_st = p->out_stride;
  a.cos = (const uint16_t*)p->rot_cos, a.sin = (const uint16_t*)p->rot_sin;
  a.T = p->num_tokens, a.K = p->in_features, a.D = p->head_dim;
  a.splits = 1;
  if (p->num_splits > 1) {
    SIPA_CHECK(p->epilogue == SIPA_LINEAR_RESIDUAL && p->norm_weight == nullptr, SIPA_EINVAL,
               "linear: only the residual epilogue without norm splits K");
    SIPA_CHECK(p->num_splits <= 64 && p->part && p->counters, SIPA_EWORKSPACE, "linear: split buffers missing");
    a.splits = p->num_splits, a.part = (float*)p->part, a.counters = (int32_t*)p->counters;
  }
  const hipStream_t st = (hipStream_t)stream;
  const int N = p->out_features;
  switch (p->epilogue) {
    case SIPA_LINEAR_RESIDUAL:
      SIPA_CHECK(N % 16 == 0, SIPA_EUNSUPPORTED, "linear: out_features %d is not a multiple of 16", N);
      a.tiles = N / 16;
      if (a.norm_w) dispatch_linear<kEpiResidual, true>(a, st);
      else dispatch_linear<kEpiResidual, false>(a, st);
      break;
    case SIPA_LINEAR_ROPE:
      SIPA_CHECK(N % 16 == 0 && a.D > 0 && a.D % 16 == 0, SIPA_EUNSUPPORTED, "linear: heads of %d channels", a.D);
      SIPA_CHECK(p->rot_channels >= 0 && p->rot_channels <= N && p->rot_channels % a.D == 0, SIPA_EINVAL,
                 "linear: %d rotated channels", p->rot_channels);
      SIPA_CHECK(p->rot_channels == 0 || (a.cos && a.sin), SIPA_EINVAL, "linear: rotary tables missing");
      SIPA_CHECK(p->residual == nullptr, SIPA_EINVAL, "linear: no residual with the rotary epilogue");
      a.rot = p->rot_channels;
      a.tiles = N / 16;
      if (a.norm_w) dispatch_linear<kEpiRope, true>(a, st);
      else dispatch_linear<kEpiRope, false>(a, st);
      break;
    case SIPA_LINEAR_SILU:
      SIPA_CHECK(N % 16 == 0, SIPA_EUNSUPPORTED, "linear: out_features %d is not a multiple of 16", N);
      SIPA_CHECK(p->residual == nullptr && p->bias == nullptr, SIPA_EINVAL, "linear: no residual or bias with SiLU");
      a.inter = N / 2;
      a.tiles = a.inter / 8;
      if (a.norm_w) dispatch_linear<kEpiSilu, true>(a, st);
      else dispatch_linear<kEpiSilu, false>(a, st);
      break;
    default:
      return fail(SIPA_EINVAL, "linear: epilogue %d", p->epilogue);
  }
  return launched("linear");
}

extern "C" int32_t sipa_rms_norm(const void* x, int64_t x_stride, const void* add, int64_t add_stride,
                                 const void* weight, float eps, void* sum, int64_t sum_stride, void* out,
                                 int64_t out_stride, int32_t T, int32_t K, void* stream) {
  SIPA_CHECK(T >= 0 && K > 0, SIPA_EINVAL, "rms_norm: bad sizes");
  if (T == 0) return SIPA_OK;
  SIPA_CHECK(x && weight && out && (add == nullptr) == (sum == nullptr), SIPA_EINVAL, "rms_norm: null pointer");
  SIPA_CHECK(K % 8 == 0 && K <= 8192, SIPA_EUNSUPPORTED, "rms_norm: rows of %d channels", K);
  SIPA_CHECK(aligned16(x) && aligned16(add) && aligned16(weight) && aligned16(sum) && aligned16(out) &&
                 x_stride % 8 == 0 && add_stride % 8 == 0 && sum_stride % 8 == 0 && out_stride % 8 == 0,
             SIPA_EUNSUPPORTED, "rms_norm: rows must be 16-byte aligned");
  const int grid = (T + 3) / 4;
  const hipStream_t st = (hipStream_t)stream;
#define SIPA_NORM(CH)                                                                                              \
  rms_norm_kernel<CH><<<grid, 256, 0, st>>>((const uint16_t*)x, x_stride, (const uint16_t*)add, add_stride,        \
                                            (const uint16_t*)weight, eps, (uint16_t*)sum, sum_stride,              \
                                            (uint16_t*)out, out_stride, T, K)
  if (K <= 1024) SIPA_NORM(2);
  else if (K <= 2048) SIPA_NORM(4);
  else SIPA_NORM(16);
#undef SIPA_NORM
  return launched("rms_norm");
}

extern "C" int32_t sipa_rope(void* x, int64_t x_stride, const void* cos, const void* sin, int32_t T, int32_t H,
                             int32_t D, void* stream) {
  SIPA_CHECK(T >= 0 && H >= 0 && D > 0, SIPA_EINVAL, "rope: bad sizes");
  if (T == 0 || H == 0) return SIPA_OK;
  SIPA_CHECK(x && cos && sin, SIPA_EINVAL, "rope: null pointer");
  SIPA_CHECK(D % 16 == 0 && (int64_t)T * H * D < 1ll << 34, SIPA_EUNSUPPORTED, "rope: %d heads of %d channels", H, D);
  SIPA_CHECK(aligned16(x) && aligned16(cos) && aligned16(sin) && x_stride % 8 == 0, SIPA_EUNSUPPORTED,
             "rope: rows must be 16-byte aligned");
  const int64_t n = (int64_t)T * H * (D / 16);
  rope_kernel<<<(int)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>((uint16_t*)x, x_stride, (const uint16_t*)cos,
                                                                      (const uint16_t*)sin, T, H, D);
  return launched("rope");
}

extern "C" int32_t sipa_silu_mul(const void* gate_up, int64_t gu_stride, void* out, int64_t out_stride, int32_t T,
                                 int32_t I, void* stream) {
  SIPA_CHECK(T >= 0 && I > 0, SIPA_EINVAL, "silu_mul: bad sizes");
  if (T == 0) return SIPA_OK;
  SIPA_CHECK(gate_up && out, SIPA_EINVAL, "silu_mul: null pointer");
  SIPA_CHECK(I % 8 == 0 && (int64_t)T * I < 1ll << 34 && aligned16(gate_up) && aligned16(out) &&
                 gu_stride % 8 == 0 && out_stride % 8 == 0,
             SIPA_EUNSUPPORTED, "silu_mul: rows must be 16-byte aligned, %d channels", I);
  const int64_t n = (int64_t)T * (I / 8);
  silu_mul_kernel<<<(int)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>((const uint16_t*)gate_up, gu_stride,
                                                                          (uint16_t*)out, out_stride, T, I);
  return launched("silu_mul");
}
