// The decoder layer's own operations around the paged attention, for gfx950: projections of a few tokens fused with
// the operations next to them, and the same elementwise operations alone for the large batches whose projections
// are left to the GEMM library. bf16 in and out, fp32 inside.
//
// Reference: engine/model.py:101-175 (RMSNorm, fused QKV with bias, rotary embedding, SwiGLU MLP, residuals), there
// about 30 separate torch operations a layer.
#include <algorithm>

#include "decode_common.h"

namespace sipa {

// Two kernels compute y = epilogue(norm(x) W^T), a projection fused with what stands before and after it.
//
// W enters the MFMA as the A operand, x as the B operand, so D[n][t] comes out with lane (t, q4) holding outputs
// n = 4 q4 .. 4 q4 + 3 of token t.
//
// RMSNorm (NORM): the row factor rstd[t] factors out of the product, so x * w_norm is rounded to bf16 for the MFMA (one
// rounding, where norm-then-multiply in bf16 has two), the squares of x are summed on the way, and the accumulators
// are scaled at the end: no pass over x before the product.
//
// Row tiles of 16: for ROPE and SILU they are 8 rows and their 8 partners (channels c and c + D/2 of a head; gate and
// up), so that both halves of a pair meet in one tile.
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
  // ROPE: the K and V channels (from kv0 on, kv_heads heads each) go straight to the paged pools [heads, blocks, offsets,
  // D] instead of out, token t at (blocks[t], offsets[t]); kv_heads 0: everything to out
  int32_t kv_heads, kv0;
  uint16_t *k_pool, *v_pool;
  int64_t kv_sh, kv_sn, kv_sb;
  const int64_t *blocks, *offsets;
  int32_t tiles;           // row tiles in all
  int32_t inter;           // SILU: gate rows (the up rows follow)
  int32_t units;           // 64-channel slices of K a workgroup takes
  int32_t splits;          // workgroups that share a tile's K (RESIDUAL)
  float* part;             // [tile][splits][tokens x rows of a tile] partial sums
  int32_t* counters;       // [tile] workgroups done, zero between calls
  int32_t* clear;          // counters of a later launch, zeroed by this one's first workgroup
  int32_t clear_n;
};

// A split launch needs its counters at zero. The projection launched before it on the stream clears them (clear), so that
// they can lie in memory of the call's own: no launch is added, and calls share nothing.
__device__ __forceinline__ void clear_counters(const LinearArgs& a) {
  if (blockIdx.x + blockIdx.y + blockIdx.z != 0) return;
  for (int i = threadIdx.x; i < a.clear_n; i += blockDim.x)
    __hip_atomic_store(a.clear + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void __launch_bounds__(256) clear_kernel(int32_t* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

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

// Where channel c of token t is stored. K and V straight to the pools: a separate store launch took 2.5 to 3.8 us a layer
// (kernel and the gap before it) for a few KB; without it a replayed 24-layer step of 8 sequences went from 950 to 889 us,
// and 24 layers over 544 mixed tokens from 2306 to 2230.
template <int EPI>
__device__ __forceinline__ uint16_t* out_at(const LinearArgs& a, int t, int c) {
  if (EPI == kEpiRope && a.kv_heads > 0 && c >= a.kv0) {
    int h = (c - a.kv0) / a.D;
    const int ch = c - a.kv0 - h * a.D;
    uint16_t* pool = a.k_pool;
    if (h >= a.kv_heads) h -= a.kv_heads, pool = a.v_pool;
    return pool + h * a.kv_sh + a.blocks[t] * a.kv_sn + a.offsets[t] * a.kv_sb + ch;
  }
  return a.out + t * a.out_st + c;
}

// x / (1 + e^-x) in fp32: the hardware's exp2 and reciprocal, each within an ulp or two, 2^-8 of the bf16 step the
// result is rounded to. (Very negative x: e^-x = inf, and x * 0 = -0.)
__device__ __forceinline__ float silu(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + fast_exp2(-1.4426950408889634f * x));
}

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

// ---- skinny_linear: up to 16 tokens, few rows ---------------------------------------------------------------------------
//
// Bound: the latency of one launch (load, reduce, store) more than the 1.6 to 6 MB of weights. A workgroup owns 16 rows
// and all of K, its 8 waves take 64-channel slices straight from memory into registers (lane (r, q4) channels
// 16 q4 .. + 15 of row r: four lanes read one 128-byte line; x in the same channel order), at most U slices each, all in
// flight together, and their sums meet in LDS.
//
// Measured in a graph, weights from memory, 8 tokens, against tile_linear's smallest tile and the GEMM library's product
// alone (us): norm + QKV 1152 x 896 + bias + rotary 5.1, 6.2, 5.7; 2048 x 1536 6.3, 8.3, 7.2; 896 x 896 + residual 4.1,
// 4.2, 5.5. An empty launch there is about 2.
constexpr int kSkinnyWaves = 8;

template <int EPI, bool NORM, int U>
__global__ void __launch_bounds__(64 * kSkinnyWaves) skinny_linear(const LinearArgs a) {
  constexpr int WV = kSkinnyWaves;
  __shared__ __align__(16) float red[WV][256];
  __shared__ float ssq[WV][16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r = lane & 15, q4 = lane >> 4;
  const int tile = blockIdx.x;
  clear_counters(a);
  const int units = a.K >> 6;
  const uint16_t* const wrow = a.w + (int64_t)linear_row<EPI>(a, tile, r) * a.K + 16 * q4;
  const uint16_t* const xrow = a.x + (int64_t)min(r, a.T - 1) * a.x_st + 16 * q4;
  const uint16_t* const nrow = NORM ? a.norm_w + 16 * q4 : nullptr;
  u32x4 w[U][2], x[U][2], nw[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = 64 * min(wave + WV * u, units - 1);  // past the end: the last slice again, masked below
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[u][h] = stream_load(wrow + c + 8 * h);
      x[u][h] = *(const u32x4*)(xrow + c + 8 * h);
      if (NORM) nw[u][h] = *(const u32x4*)(nrow + c + 8 * h);
    }
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    // masked to zeros, not branched around: with a branch the compiler sinks the slice's loads into it, and their
    // latencies add up instead of overlapping
    const uint32_t live = wave + WV * u < units ? 0xffffffffu : 0u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 xv = x[u][h] & live;
      if (NORM) xv = scale_channels(xv, nw[u][h], ss);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[u][h] & live),
                                                    __builtin_bit_cast(bf16x8, xv), acc, 0, 0, 0);
    }
  }
  *(f32x4*)&red[wave][lane * 4] = acc;
  if (NORM) {
    const float s = sum_over_rows(ss);
    if (q4 == 0) ssq[wave][r] = s;
  }
  __syncthreads();

  // Pairs (n, n + 8) of the tile's outputs for one token; eight neighbouring threads store eight neighbouring channels.
  const int n = threadIdx.x & 7, t = threadIdx.x >> 3;
  if (t >= min(a.T, 16)) return;
  const int at = ((n >> 2) * 16 + t) * 4 + (n & 3);  // output n's place; n + 8 is 128 words on
  float lo = 0.f, hi = 0.f;
#pragma unroll
  for (int v = 0; v < WV; ++v) {
    lo += red[v][at];
    hi += red[v][at + 128];
  }
  if (NORM) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < WV; ++v) s += ssq[v][t];
    const float rstd = rsqrtf(s / (float)a.K + a.eps);
    lo *= rstd;
    hi *= rstd;
  }
  const int nlo = linear_row<EPI>(a, tile, n), nhi = linear_row<EPI>(a, tile, n + 8);
  if (EPI == kEpiSilu) {
    a.out[t * a.out_st + nlo] = f32_to_bf16_bits(silu(lo) * hi);
    return;
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
  *out_at<EPI>(a, t, nlo) = f32_to_bf16_bits(lo);
  *out_at<EPI>(a, t, nhi) = f32_to_bf16_bits(hi);
}

// ---- tile_linear: everything else -----------------------------------------------------------------------------------------
//
// Bound: at up to some hundred tokens neither HBM (2 to 17 MB of weights) nor the matrix cores (1 to 10 GFLOP) but the
// latency of a short K loop on few workgroups, and for larger tiles the norm's VALU work. 4 waves (2 x 2) share a tile
// of 32 TT tokens and 32 TN rows of W; both operands go through LDS (one read from L2 per workgroup), 64 channels a
// step, two buffers, one barrier a step, with the loads of NR steps in flight in registers ahead of them. Rows of 128
// bytes are stored with their 16-byte chunks xor-ed by the row, so the fragment reads of 16 rows spread over all
// banks. The norm's products and squares are formed once per workgroup, on the way into LDS. A token's partner channel
// is 32 lanes away, so the rotary and gated epilogues exchange accumulators with a shuffle.
//
// Split K (RESIDUAL): 896 outputs are 28 tiles of 32 rows, and one workgroup would take 76 steps of a 4864-long K; up to
// six share it and the last one to arrive adds their sums in split order.
//
// Measured in a graph, weights from memory, against the GEMM library's product alone (us; the library needs a norm, 2.9,
// a rotary, 2.1, a SwiGLU, 2.2 to 6, or a residual launch, 2, besides): 64 tokens: QKV 1152 x 896 6.4 (8.0), o 896 x 896
// 4.4 (7.9), gate/up 9728 x 896 10.0 (11.9), down 896 x 4864 8.4 (13.6); 544 tokens: 9.6 (8.4), 5.5 (7.9), 26.3 (17.7),
// 15 to 16 (16.5).
template <int EPI, bool NORM, int TT, int TN, int NR>
__global__ void __launch_bounds__(256) tile_linear(const LinearArgs a) {
  static_assert(NR % 2 == 0, "a ring slot always meets the same LDS buffer");
  constexpr int BT = 32 * TT, BN = 32 * TN;  // tokens, rows of W
  __shared__ __align__(16) uint16_t xs[2][BT * 64];
  __shared__ __align__(16) uint16_t wsh[2][BN * 64];
  __shared__ float rstd_s[NORM ? BT : 1];
  __shared__ int last;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wt = wave & 1, wn = wave >> 1;
  const int lane = threadIdx.x & 63, r = lane & 15, q4 = lane >> 4;
  const int tile0 = blockIdx.x * (2 * TN), t_base = blockIdx.y * BT;
  const int unit0 = blockIdx.z * a.units;
  const int n = min(a.units, (a.K >> 6) - unit0);
  clear_counters(a);

  // this thread's chunk of rows (tid / 8) + 32 i
  const int row0 = threadIdx.x >> 3, ch = threadIdx.x & 7;
  const int lds_at = row0 * 64 + ((ch ^ (row0 & 7)) << 3);
  const uint16_t *xp[TT], *wp[TN];
#pragma unroll
  for (int i = 0; i < TT; ++i)
    xp[i] = a.x + (int64_t)min(t_base + row0 + 32 * i, a.T - 1) * a.x_st + 64 * unit0 + 8 * ch;
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int wr = row0 + 32 * i;
    wp[i] = a.w + (int64_t)linear_row<EPI>(a, min(tile0 + (wr >> 4), a.tiles - 1), wr & 15) * a.K + 64 * unit0 + 8 * ch;
  }
  const uint16_t* np = NORM ? a.norm_w + 64 * unit0 + 8 * ch : nullptr;

  struct Stage {
    u32x4 x[TT], w[TN], nw;
  };
  Stage ring[NR];
  auto load = [&](Stage& s, int k) {
#pragma unroll
    for (int i = 0; i < TN; ++i) s.w[i] = *(const u32x4*)(wp[i] + 64 * k);
#pragma unroll
    for (int i = 0; i < TT; ++i) s.x[i] = *(const u32x4*)(xp[i] + 64 * k);
    if (NORM) s.nw = *(const u32x4*)(np + 64 * k);
  };
  float ss[TT];
  f32x4 acc[TN][TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    ss[j] = 0.f;
#pragma unroll
    for (int i = 0; i < TN; ++i) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // One step: the slot's operands into LDS buffer b, then (after the caller's next loads) the barrier and the products.
  // A buffer is written again two steps on, behind a barrier that every wave passes after its reads of it.
  auto stage = [&](Stage& s, int b) {
#pragma unroll
    for (int i = 0; i < TN; ++i) *(u32x4*)(wsh[b] + lds_at + 32 * 64 * i) = s.w[i];
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      u32x4 v = s.x[i];
      if (NORM) v = scale_channels(v, s.nw, ss[i]);
      *(u32x4*)(xs[b] + lds_at + 32 * 64 * i) = v;
    }
  };
  auto multiply = [&](int b) {
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = r * 64 + (((4 * h + q4) ^ (r & 7)) << 3);
      bf16x8 wf[TN], xf[TT];
#pragma unroll
      for (int i = 0; i < TN; ++i) wf[i] = *(const bf16x8*)(wsh[b] + (wn * TN + i) * 16 * 64 + at);
#pragma unroll
      for (int j = 0; j < TT; ++j) xf[j] = *(const bf16x8*)(xs[b] + (wt * TT + j) * 16 * 64 + at);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
  };
  // NR steps in flight; the steady state refills every slot unconditionally, so the compiler's waits are exact there.
#pragma unroll
  for (int j = 0; j < NR; ++j) load(ring[j], min(j, n - 1));
  int k = 0;
  for (; k + 2 * NR <= n; k += NR) {
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      stage(ring[j], j & 1);
      load(ring[j], k + j + NR);
      multiply(j & 1);
    }
  }
#pragma unroll
  for (int j = 0; j < NR; ++j)
    if (k + j < n) {  // uniform over the workgroup
      stage(ring[j], j & 1);
      if (k + j + NR < n) load(ring[j], k + j + NR);
      multiply(j & 1);
    }
#pragma unroll
  for (int j = 0; j < NR; ++j)
    if (k + NR + j < n) {
      stage(ring[j], j & 1);
      multiply(j & 1);
    }

  if (NORM) {
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      float s = ss[i];
      s += __shfl_xor(s, 1);
      s += __shfl_xor(s, 2);
      s += __shfl_xor(s, 4);
      if (ch == 0) rstd_s[row0 + 32 * i] = rsqrtf(s / (float)a.K + a.eps);
    }
    __syncthreads();
  }

  if (EPI == kEpiResidual && a.splits > 1) {
    // Split K: the sums go through to memory, and the last workgroup to arrive adds them in split order (the split
    // merge of the decode kernels: stores complete, then a relaxed counter).
    const int pair = blockIdx.y * gridDim.x + blockIdx.x;
    float* const part = a.part + (int64_t)pair * a.splits * (BT * BN);
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(part, (short)0, a.splits * BT * BN * 4, 0x00020000);
    const auto at = [&](int sp, int i, int j) { return (((sp * TN + i) * TT + j) * 256 + (int)threadIdx.x) * 16; };
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TT; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), rows, at(blockIdx.z, i, j), 0,
                                               kAuxSc1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      last = __hip_atomic_fetch_add(a.counters + pair, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             a.splits - 1;
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0)
      __hip_atomic_store(a.counters + pair, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int sp = 0; sp < a.splits; ++sp)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
          acc[i][j] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, at(sp, i, j), 0, kAuxSc1));
  }

  auto unpack = [](uint2 u) {
    return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                 __uint_as_float(u.y & 0xffff0000u)};
  };
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int tile = tile0 + wn * TN + i;
    const bool in = tile < a.tiles;
    const int c = linear_row<EPI>(a, min(tile, a.tiles - 1), 4 * q4);  // this lane's 4 channels: c .. c + 3
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      const int tl = (wt * TT + j) * 16 + r, t = t_base + tl;
      f32x4 v = acc[i][j];
      if (NORM) v *= rstd_s[tl];
      if (EPI == kEpiSilu) {
        // Lanes q4 < 2 hold four gate channels, their partners the up channels: each side gives the other half of its
        // own and finishes two channels.
        const bool gate = q4 < 2;
        const float s0 = __shfl_xor(gate ? v[2] : v[0], 32), s1 = __shfl_xor(gate ? v[3] : v[1], 32);
        const float g0 = gate ? v[0] : s0, g1 = gate ? v[1] : s1, u0 = gate ? s0 : v[2], u1 = gate ? s1 : v[3];
        if (in && t < a.T)
          *(uint32_t*)(a.out + t * a.out_st + tile * 8 + 4 * (q4 & 1) + (gate ? 0 : 2)) =
              pack_bf16x2(silu(g0) * u0, silu(g1) * u1);
        continue;
      } else {
        if (a.bias != nullptr) v += unpack(*(const uint2*)(a.bias + c));
        if (EPI == kEpiRope && tile * 16 < a.rot) {
          f32x4 u;
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = __shfl_xor(v[e], 32);
          const int64_t at = (int64_t)min(t, a.T - 1) * a.D + c % a.D;
          v = v * unpack(*(const uint2*)(a.cos + at)) + u * unpack(*(const uint2*)(a.sin + at));
        }
        if (EPI == kEpiResidual && a.res != nullptr && t < a.T) v += unpack(*(const uint2*)(a.res + t * a.res_st + c));
      }
      if (!in || t >= a.T) continue;
      *(uint2*)out_at<EPI>(a, t, c) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
}

template <int EPI, bool NORM, int TT, int TN, int NR>
static void launch_tile(const LinearArgs& a, hipStream_t st) {
  const dim3 grid((a.tiles + 2 * TN - 1) / (2 * TN), (a.T + 32 * TT - 1) / (32 * TT), a.splits);
  tile_linear<EPI, NORM, TT, TN, NR><<<grid, 256, 0, st>>>(a);
}

// Tile shapes of tile_linear by number: tokens and rows of W.
struct TileShape {
  int tokens, rows;
};
constexpr TileShape kTiles[] = {{32, 32}, {32, 64}, {64, 64}, {64, 128}, {128, 128}};
constexpr int kNumTiles = 5, kSkinny = kNumTiles;

struct LinearPlan {
  int shape;   // index into kTiles, or kSkinny
  int splits;  // workgroups that share a tile's K
  int64_t part_bytes;
  int64_t counters;
};

// Tiles 64 x 64, 64 x 128 and 128 x 128 of a gated projection by the workgroups each makes: its time at K = 896 is close
// to 6 + 4.1 c, 4 + 8 c and (17.5, 25, 13 c from three on) us, c the most workgroups a CU gets (in proportion at 1536),
// measured at 33 to 1000 tokens on both model shapes. Against 128 x 128 throughout: 0.5B 160 tokens 18.0 -> 13.4 us, 800
// 37.1 -> 33.5, 1.5B 160 36.8 -> 32.5.
static int gated_tile(int64_t g2, int64_t g3, int64_t g4, int cus) {
  const auto per_cu = [&](int64_t g) { return (double)((g + cus - 1) / cus); };
  const double t2 = 6 + 4.1 * per_cu(g2), t3 = 4 + 8 * per_cu(g3);
  const double t4 = g4 <= cus ? 17.5 : g4 <= 2 * cus ? 25 : 13 * per_cu(g4);
  return t4 <= t2 && t4 <= t3 ? 4 : t3 <= t2 ? 3 : 2;
}

// The smallest tile whose grid stays within a number of workgroups that depends on the epilogue (given for 256 CUs): small
// tiles fill the chip, large ones read less. ROPE: 640 (K is short and the tiles' norm is their cost; QKV 0.5B at 544
// tokens 9.4 us with 612 workgroups, 10.8 with 162). SILU: 200 workgroups of 32 x 64, gated_tile above them. RESIDUAL: 256,
// and a K from 4096 on is then split, at most six ways (896 x 4864 at 8 tokens 7.7 us with six, 8.2 with eight, 10.6 with
// one): tiles of 32 x 32 until the grid has about 256 again, larger ones only as far as one workgroup a CU goes (896 x
// 4864, whole and in halves: 300 tokens, 140 tiles, 14.3 and 17.6; 800 tokens, 182 tiles, 21.2 and 25.6). From 96 slices of
// K on, a grid too large to split takes the next larger tile in halves (us without and with: 1536 x 8960 160 tokens 23.4
// and 20.0, 300 28.9 and 25.0; 1536 x 6144, 96 slices, 17.2 and 15.3, 21.4 and 19.1; 896 x 4864, 76 slices, 544 tokens 14.7
// and 17.0: not there). num_splits and shape of the caller come first (0: the rule).
static LinearPlan plan_linear(int epi, bool norm, int T, int tiles, int K, int want_splits, int want_shape, int cus) {
  LinearPlan p{};
  const int units = K >> 6;
  auto grid = [&](int s) {
    return (int64_t)((16 * tiles + kTiles[s].rows - 1) / kTiles[s].rows) * ((T + kTiles[s].tokens - 1) / kTiles[s].tokens);
  };
  if (want_shape > 0) {
    p.shape = want_shape - 1;
  } else if (T <= 16 && units <= 24 && tiles <= cus && want_splits <= 1) {
    p.shape = kSkinny;
  } else {
    const int most = epi == kEpiRope ? 5 * cus / 2 : epi == kEpiSilu ? 25 * cus / 32 : cus;
    p.shape = epi == kEpiSilu ? 1 : 0;
    if (epi != kEpiSilu)
      while (p.shape + 1 < kNumTiles && grid(p.shape) > most) ++p.shape;
    else if (grid(1) > most)
      p.shape = gated_tile(grid(2), grid(3), grid(4), cus);
    // a long K in whole workgroups of one tile against two halves of the next larger one
    if (epi == kEpiResidual && !norm && want_splits <= 0 && units >= 96 && p.shape < 2 &&
        (p.shape == 0 ? grid(0) * 5 > 4 * cus : 2 * grid(1) > cus) && 2 * grid(p.shape + 1) <= cus)
      ++p.shape;
  }
  p.splits = 1;
  if (p.shape != kSkinny && epi == kEpiResidual && !norm) {
    const int64_t g = grid(p.shape);
    if (want_splits > 0)
      p.splits = want_splits;
    else if (K >= 4096 && p.shape == 0 && g * 5 <= 4 * cus)
      p.splits = (int)std::min<int64_t>(6, (cus + g - 1) / g);
    else if (K >= 4096 && p.shape > 0)
      p.splits = (int)std::min<int64_t>(6, std::max<int64_t>(1, cus / g));
    const int per = (units + p.splits - 1) / p.splits;
    p.splits = (units + per - 1) / per;
    if (p.splits > 1) {
      p.part_bytes = g * p.splits * kTiles[p.shape].tokens * kTiles[p.shape].rows * 4;
      p.counters = g;
    }
  }
  return p;
}

template <int EPI, bool NORM>
static void launch_linear(const LinearArgs& a, int shape, hipStream_t st) {
  switch (shape) {
    case 0: return launch_tile<EPI, NORM, 1, 1, 4>(a, st);
    case 1: return launch_tile<EPI, NORM, 1, 2, 4>(a, st);
    case 2: return launch_tile<EPI, NORM, 2, 2, 4>(a, st);
    case 3: return launch_tile<EPI, NORM, 2, 4, 4>(a, st);
    case 4: return launch_tile<EPI, NORM, 4, 4, 2>(a, st);
    default:
      if (a.K <= 16 * 64)
        skinny_linear<EPI, NORM, 2><<<a.tiles, 64 * kSkinnyWaves, 0, st>>>(a);
      else
        skinny_linear<EPI, NORM, 3><<<a.tiles, 64 * kSkinnyWaves, 0, st>>>(a);
  }
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
    o[i] = pack_bf16x2(silu(g0) * u0, silu(g1) * u1);
  }
  *(u32x4*)(out + t * out_st + c) = o;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool aligned8(const void* p) { return ((uintptr_t)p & 7) == 0; }

static int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SIPA_OK : fail(SIPA_EHIP, "%s: %s", what, hipGetErrorString(e));
}

}  // namespace sipa

using namespace sipa;

static int check_linear(const sipa_linear_params* p) {
  SIPA_CHECK(p != nullptr && p->struct_size == (int32_t)sizeof(sipa_linear_params), SIPA_EINVAL,
             "sipa_linear_params: wrong size");
  const int T = p->num_tokens, K = p->in_features, N = p->out_features;
  SIPA_CHECK(T >= 0 && K > 0 && N > 0, SIPA_EINVAL, "linear: bad sizes");
  SIPA_CHECK(T <= 1 << 20 && N <= 1 << 22 && K <= 1 << 20, SIPA_EUNSUPPORTED, "linear: sizes out of range");
  SIPA_CHECK(K % 64 == 0, SIPA_EUNSUPPORTED, "linear: in_features %d is not a multiple of 64", K);
  SIPA_CHECK(N % 16 == 0, SIPA_EUNSUPPORTED, "linear: out_features %d is not a multiple of 16", N);
  SIPA_CHECK(p->epilogue >= SIPA_LINEAR_RESIDUAL && p->epilogue <= SIPA_LINEAR_SILU, SIPA_EINVAL, "linear: epilogue %d",
             p->epilogue);
  SIPA_CHECK(p->tile >= 0 && p->tile <= kNumTiles + 1 && p->num_splits >= 0 && p->num_splits <= 64, SIPA_EINVAL,
             "linear: tile %d, %d splits", p->tile, p->num_splits);
  SIPA_CHECK(p->tile != kSkinny + 1 || (T <= 16 && K <= 24 * 64 && p->num_splits <= 1), SIPA_EUNSUPPORTED,
             "linear: the skinny kernel takes up to 16 tokens and %d in_features, unsplit", 24 * 64);
  if (p->epilogue == SIPA_LINEAR_ROPE) {
    SIPA_CHECK(p->head_dim > 0 && p->head_dim % 16 == 0, SIPA_EUNSUPPORTED, "linear: heads of %d channels", p->head_dim);
    SIPA_CHECK(p->rot_channels >= 0 && p->rot_channels <= N && p->rot_channels % p->head_dim == 0, SIPA_EINVAL,
               "linear: %d rotated channels", p->rot_channels);
  }
  SIPA_CHECK(p->kv_heads >= 0 && (p->kv_heads == 0 || p->epilogue == SIPA_LINEAR_ROPE), SIPA_EINVAL,
             "linear: only the rotary epilogue stores to K and V pools");
  SIPA_CHECK(p->kv_heads == 0 || (p->kv_heads <= (1 << 16) && p->rot_channels >= p->kv_heads * p->head_dim &&
                                  N == p->rot_channels + p->kv_heads * p->head_dim),
             SIPA_EINVAL, "linear: %d K and V heads of %d channels do not end %d rotated of %d channels", p->kv_heads,
             p->head_dim, p->rot_channels, N);
  SIPA_CHECK(p->num_splits <= 1 || (p->epilogue == SIPA_LINEAR_RESIDUAL && p->norm_weight == nullptr), SIPA_EINVAL,
             "linear: only the residual epilogue without norm splits K");
  SIPA_CHECK(p->clear_count >= 0 && p->clear_count <= kMaxCounters && (p->clear_count == 0 || p->clear), SIPA_EINVAL,
             "linear: %d counters to clear", p->clear_count);
  return SIPA_OK;
}

static LinearPlan plan_of(const sipa_linear_params* p) {
  const int tiles = p->out_features / 16;  // SILU: 8 gate and 8 up rows each
  // of the first device asked for (a process's GPUs are alike; a layer's call plans eight times); 256 without one
  static const int cus = [] {
    const int n = sipa_device_cu_count(-1);
    return n > 0 ? n : 256;
  }();
  return plan_linear(p->epilogue, p->norm_weight != nullptr, p->num_tokens, tiles, p->in_features, p->num_splits,
                     p->tile, cus);
}

extern "C" int64_t sipa_linear_scratch_bytes(const sipa_linear_params* p) {
  const int rc = check_linear(p);
  if (rc != SIPA_OK) return rc;
  return p->num_tokens == 0 ? 0 : plan_of(p).part_bytes;
}

extern "C" int32_t sipa_fused_linear(const sipa_linear_params* p, void* stream) {
  const int rc = check_linear(p);
  if (rc != SIPA_OK) return rc;
  if (p->num_tokens == 0) return SIPA_OK;
  SIPA_CHECK(p->x && p->weight && p->out, SIPA_EINVAL, "linear: null pointer");
  SIPA_CHECK(aligned16(p->x) && aligned16(p->weight) && aligned16(p->norm_weight) && p->x_stride % 8 == 0,
             SIPA_EUNSUPPORTED, "linear: x, weight and norm weight need 16-byte rows");
  SIPA_CHECK(aligned8(p->bias) && aligned8(p->residual) && aligned8(p->out) && aligned8(p->rot_cos) &&
                 aligned8(p->rot_sin) && p->res_stride % 4 == 0 && p->out_stride % 4 == 0,
             SIPA_EUNSUPPORTED, "linear: bias, residual, rotary tables and out need 8-byte rows");
  SIPA_CHECK(p->x_stride >= 0 && p->out_stride >= 0 && p->res_stride >= 0, SIPA_EINVAL, "linear: negative stride");
  SIPA_CHECK(p->norm_weight == nullptr || p->eps >= 0.f, SIPA_EINVAL, "linear: eps");
  SIPA_CHECK(p->epilogue == SIPA_LINEAR_RESIDUAL || p->residual == nullptr, SIPA_EINVAL,
             "linear: only the residual epilogue takes a residual");
  SIPA_CHECK(p->epilogue != SIPA_LINEAR_SILU || p->bias == nullptr, SIPA_EINVAL, "linear: no bias with SiLU");
  SIPA_CHECK(p->epilogue != SIPA_LINEAR_ROPE || p->rot_channels == 0 || (p->rot_cos && p->rot_sin), SIPA_EINVAL,
             "linear: rotary tables missing");
  SIPA_CHECK(p->kv_heads == 0 || (p->k_pool && p->v_pool && p->kv_blocks && p->kv_offsets), SIPA_EINVAL,
             "linear: K and V pools or slots missing");
  SIPA_CHECK(p->kv_heads == 0 || (aligned8(p->k_pool) && aligned8(p->v_pool) && p->kv_stride_h % 4 == 0 &&
                                  p->kv_stride_n % 4 == 0 && p->kv_stride_b % 4 == 0),
             SIPA_EUNSUPPORTED, "linear: K and V pools need 8-byte rows");
  const LinearPlan plan = plan_of(p);
  LinearArgs a{};
  a.kv_heads = p->kv_heads;
  if (p->kv_heads > 0) {
    a.kv0 = p->rot_channels - p->kv_heads * p->head_dim;
    a.k_pool = (uint16_t*)p->k_pool, a.v_pool = (uint16_t*)p->v_pool;
    a.kv_sh = p->kv_stride_h, a.kv_sn = p->kv_stride_n, a.kv_sb = p->kv_stride_b;
    a.blocks = p->kv_blocks, a.offsets = p->kv_offsets;
  }
  a.x = (const uint16_t*)p->x, a.x_st = p->x_stride, a.w = (const uint16_t*)p->weight;
  a.norm_w = (const uint16_t*)p->norm_weight, a.eps = p->eps, a.bias = (const uint16_t*)p->bias;
  a.res = (const uint16_t*)p->residual, a.res_st = p->res_stride;
  a.out = (uint16_t*)p->out, a.out_st = p->out_stride;
  a.cos = (const uint16_t*)p->rot_cos, a.sin = (const uint16_t*)p->rot_sin;
  a.T = p->num_tokens, a.K = p->in_features, a.D = p->head_dim;
  a.tiles = p->out_features / 16, a.inter = p->out_features / 2;
  a.rot = p->epilogue == SIPA_LINEAR_ROPE ? p->rot_channels : 0;
  a.clear = (int32_t*)p->clear, a.clear_n = p->clear_count;
  a.splits = plan.splits;
  const int units = a.K >> 6;
  a.units = (units + a.splits - 1) / a.splits;
  if (plan.splits > 1) {
    SIPA_CHECK(p->scratch != nullptr && p->scratch_bytes >= plan.part_bytes && aligned16(p->scratch) && p->counters,
               SIPA_EWORKSPACE, "linear: %lld bytes of scratch needed for %d splits", (long long)plan.part_bytes,
               plan.splits);
    SIPA_CHECK(plan.counters <= kMaxCounters, SIPA_EUNSUPPORTED, "linear: %lld tiles exceed the %d merge counters",
               (long long)plan.counters, kMaxCounters);
    a.part = (float*)p->scratch, a.counters = (int32_t*)p->counters;
  }
  const hipStream_t st = (hipStream_t)stream;
  switch (p->epilogue * 2 + (a.norm_w != nullptr)) {
    case 0: launch_linear<kEpiResidual, false>(a, plan.shape, st); break;
    case 1: launch_linear<kEpiResidual, true>(a, plan.shape, st); break;
    case 2: launch_linear<kEpiRope, false>(a, plan.shape, st); break;
    case 3: launch_linear<kEpiRope, true>(a, plan.shape, st); break;
    case 4: launch_linear<kEpiSilu, false>(a, plan.shape, st); break;
    default: launch_linear<kEpiSilu, true>(a, plan.shape, st); break;
  }
  return launched("linear");
}

// The three projections of sipa_layer_out over its scratch: h, the gated activations, then one split's partial sums at
// a time.
static int layer_out_parts(const sipa_layer_out_params* p, sipa_linear_params (&l)[3], int64_t* bytes) {
  SIPA_CHECK(p != nullptr && p->struct_size == (int32_t)sizeof(sipa_layer_out_params), SIPA_EINVAL,
             "sipa_layer_out_params: wrong size");
  SIPA_CHECK(p->num_tokens >= 0 && p->num_tokens <= 1 << 20 && p->hidden > 0 && p->hidden <= 1 << 20 && p->inter > 0 &&
                 p->inter <= 1 << 20,
             SIPA_EINVAL, "layer: bad sizes");
  auto align = [](int64_t n) { return (n + 255) & ~(int64_t)255; };
  const int64_t h_bytes = align((int64_t)p->num_tokens * p->hidden * 2);
  const int64_t act_bytes = align((int64_t)p->num_tokens * p->inter * 2);
  char* const base = (char*)p->scratch;
  char* const h = base;
  char* const act = base == nullptr ? nullptr : base + h_bytes;
  for (auto& q : l) {
    q = sipa_linear_params{};
    q.struct_size = sizeof(q);
    q.num_tokens = p->num_tokens;
    q.scratch = base == nullptr ? nullptr : act + act_bytes;
    q.scratch_bytes = p->scratch_bytes - h_bytes - act_bytes;
  }
  l[0].epilogue = SIPA_LINEAR_RESIDUAL, l[0].in_features = p->attn_features, l[0].out_features = p->hidden;
  l[0].x = p->attn, l[0].x_stride = p->attn_stride, l[0].weight = p->o_w, l[0].residual = p->x;
  l[0].res_stride = p->x_stride, l[0].out = h, l[0].out_stride = p->hidden;
  l[1].epilogue = SIPA_LINEAR_SILU, l[1].in_features = p->hidden, l[1].out_features = 2 * p->inter, l[1].eps = p->eps;
  l[1].x = h, l[1].x_stride = p->hidden, l[1].weight = p->gate_up_w, l[1].norm_weight = p->post_norm;
  l[1].out = act, l[1].out_stride = p->inter;
  l[2].epilogue = SIPA_LINEAR_RESIDUAL, l[2].in_features = p->inter, l[2].out_features = p->hidden;
  l[2].x = act, l[2].x_stride = p->inter, l[2].weight = p->down_w, l[2].residual = h, l[2].res_stride = p->hidden;
  l[2].out = p->out, l[2].out_stride = p->hidden;
  int64_t part = 0;
  for (const auto& q : l) {
    const int64_t b = sipa_linear_scratch_bytes(&q);
    if (b < 0) return (int)b;
    part = std::max(part, b);
  }
  *bytes = h_bytes + act_bytes + part;
  return SIPA_OK;
}

extern "C" int64_t sipa_layer_out_scratch_bytes(const sipa_layer_out_params* p) {
  sipa_linear_params l[3];
  int64_t bytes = 0;
  const int rc = layer_out_parts(p, l, &bytes);
  return rc != SIPA_OK ? rc : bytes;
}

extern "C" int32_t sipa_layer_out(const sipa_layer_out_params* p, void* stream) {
  sipa_linear_params l[3];
  int64_t bytes = 0;
  const int rc = layer_out_parts(p, l, &bytes);
  if (rc != SIPA_OK) return rc;
  if (p->num_tokens == 0) return SIPA_OK;
  SIPA_CHECK(p->x && p->attn && p->o_w && p->post_norm && p->gate_up_w && p->down_w && p->out && p->counters,
             SIPA_EINVAL, "layer: null pointer");
  SIPA_CHECK(p->scratch != nullptr && p->scratch_bytes >= bytes && ((uintptr_t)p->scratch & 255) == 0, SIPA_EWORKSPACE,
             "layer: %lld bytes of 256-byte aligned scratch needed", (long long)bytes);
  const int n0 = (int)plan_of(&l[0]).counters, n2 = (int)plan_of(&l[2]).counters;
  SIPA_CHECK(n0 <= SIPA_LAYER_COUNTERS / 2 && n2 <= SIPA_LAYER_COUNTERS / 2, SIPA_EUNSUPPORTED,
             "layer: %d and %d split tiles exceed the %d counters", n0, n2, SIPA_LAYER_COUNTERS);
  int32_t* const counters = (int32_t*)p->counters;
  l[0].counters = counters, l[2].counters = counters + SIPA_LAYER_COUNTERS / 2;
  if (n0 > 0) {  // from 4096 attention features on: no projection of this call runs before it
    clear_kernel<<<1, 256, 0, (hipStream_t)stream>>>(counters, n0);
    const int r = launched("layer counters");
    if (r != SIPA_OK) return r;
  }
  l[0].clear = l[2].counters, l[0].clear_count = n2;
  for (const auto& q : l) {
    const int r = sipa_fused_linear(&q, stream);
    if (r != SIPA_OK) return r;
  }
  return SIPA_OK;
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
