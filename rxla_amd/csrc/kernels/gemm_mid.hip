// W8A16 linear for a few dozen to a few hundred rows (chunked prompts, short
// prompts, batched decode beyond 16 rows), same cast points as gemm.hip:
//
//   y[m, n] = bf16( sum_k x[m, k] * bf16((u8[n, k] - 128) * s[n, k / G]) )
//
// Bound: at 17-64 rows the weights' HBM bytes, beyond that the matrix rate
// while the weight tiles stay in L2. The GEMV streams the weights once per 32
// rows and the 128-row GEMM tiles leave most CUs idle at these sizes, so:
//   * weights go global -> registers -> bf16 fragments, each wave its own 16
//     RG weight rows: no LDS traffic and no barrier for them, and every code is
//     converted once per 16 FJ rows of x. A lane holds 16 consecutive codes of
//     row lane % 16 (both weight layouts); its two 8-code halves are the A
//     operands of two MFMAs, and x is read in that k order.
//   * the 16 FJ rows of x go through LDS in chunks of 256 k, double-buffered
//     by LDS DMA, shared by the 4 waves of a wave group (64 RG weight rows).
//   * the weights of chunk c + 1 load into a second register set while chunk c
//     is multiplied.
//   * K splits over KG wave groups of a workgroup (merged through LDS) and over
//     `ksplit` workgroups (f32 partials, rxw8_gemv_splitk_reduce).
// Measured (bf16 rows, per-channel row-major unless noted): 48 x 6144 x 4096
// 28.8 -> 14.1 us (f32 rows, G = 128: 33.4 -> 17.8), 64 x 12288 x 4096 54.7 ->
// 19.7, 60 x 24576 x 4096 (f32, packed) 148 -> 39, 100 x 2048 x 6144 29.4 ->
// 13.6, 655 x 2048 x 2048 31.1 -> 18.6. What is left at 48 rows (25 MB, 5 us
// of HBM time): a launch and a reduce launch, and one memory round trip per
// chunk of which the other wave group hides a part.
#include "common.h"

// (matches gemm.hip and ops.cpp)
struct GemmArgs {
  const void *x;       // [M, K] bf16 (f32: the _xf kernels)
  const uint8_t *w;    // [N, K] u8 or packed [N/16, K/64, 1024]
  const float *scale;  // [N, K / G]
  void *y;             // [M, N]
  int M, N, K, G;
  int y_f32, y_mode, w_packed;
  int group_n;
  int ksplit;
  float *ws;           // [ksplit, M, N] f32 partials when ksplit > 1
};

namespace {

constexpr int CK = 256;  // k per chunk
constexpr int ROWB = CK * 2;

// lane holds y[m, n .. n+3] (see gemm.hip gemm_store)
__device__ __forceinline__ void store4(const GemmArgs &a, int m, int n, f32x4 v) {
  if (a.y_mode == 2) {
    f32x4 up;
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(v[i], 32);
    if ((n & 15) < 8 && m < a.M && n < a.N) {
      const int c = (n >> 4) * 8 + (n & 7);
      *(uint2 *)((uint16_t *)a.y + (int64_t)m * (a.N / 2) + c) =
          uint2{pack_bf16x2(silu_mul_f32(round_bf16(v[0]), round_bf16(up[0])),
                            silu_mul_f32(round_bf16(v[1]), round_bf16(up[1]))),
                pack_bf16x2(silu_mul_f32(round_bf16(v[2]), round_bf16(up[2])),
                            silu_mul_f32(round_bf16(v[3]), round_bf16(up[3])))};
    }
    return;
  }
  if (m >= a.M || n >= a.N) return;  // (N % 16 == 0: a lane's 4 channels are all in or all out)
  if (a.y_mode == 1) {
    float4 *h = (float4 *)((float *)a.y + (int64_t)m * a.N + n);
    float4 o = *h;
    o.x += round_bf16(v[0]);
    o.y += round_bf16(v[1]);
    o.z += round_bf16(v[2]);
    o.w += round_bf16(v[3]);
    *h = o;
  } else if (a.y_f32) {
    *(float4 *)((float *)a.y + (int64_t)m * a.N + n) =
        float4{round_bf16(v[0]), round_bf16(v[1]), round_bf16(v[2]), round_bf16(v[3])};
  } else {
    *(uint2 *)((uint16_t *)a.y + (int64_t)m * a.N + n) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
}

template <int FJ, int RG, bool GRP, bool XF>
__device__ __forceinline__ void gemm_mid(const GemmArgs &a) {
  constexpr int KG = 2;  // wave groups
  constexpr int TM = 16 * FJ, TN = 64 * RG, XBUF = TM * ROWB;
  constexpr int XDMA = XBUF / 1024 / 4;  // LDS-DMA instructions per wave per chunk
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wv & 3, kg = wv >> 2;
  // work items (split, tile), each XCD a contiguous share; tiles in groups of
  // GN n tiles with n fastest, so that the 32 CUs of an XCD cover about GN n x
  // 32 / GN m tiles and share both operands through its L2
  const int tiles_m = (a.M + TM - 1) / TM, tiles_n = (a.N + TN - 1) / TN, ntiles = tiles_m * tiles_n;
  const int per_xcd = (ntiles * a.ksplit + 7) / 8;
  const int t_all = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (t_all >= ntiles * a.ksplit) return;
  const int split = t_all / ntiles, t = t_all - split * ntiles;
  constexpr int GN = 8;
  const int group = t / (GN * tiles_m), in = t - group * GN * tiles_m, gw = min(GN, tiles_n - group * GN);
  const int n0 = (group * GN + in % gw) * TN + wn * 16 * RG, m0 = in / gw * TM;
  const int KT = a.K / 64, chunks = a.K / CK, groups = a.K / a.G;
  const int cb = split * chunks / a.ksplit, ce = (split + 1) * chunks / a.ksplit;
  const int iters = (ce - cb + KG - 1) / KG;  // of every wave group; chunk cb + kg + KG i

  char *xs = smem + kg * 2 * XBUF;
  // f32 rows: a thread's 2 FJ pieces of 8 values, loaded with the chunk's
  // weights and rounded to bf16 (the reference's x.cast(BF16)) into LDS once
  // the chunk before has been multiplied
  constexpr int XP = XF ? 2 * FJ : 1;
  float4 xr[XP][2];
  const int tid = threadIdx.x & 255;
  auto load_x = [&](int c) {
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int p = tid + 256 * i, m = min(m0 + (p >> 5), a.M - 1);
      const float4 *src = (const float4 *)((const float *)a.x + (int64_t)m * a.K + c * CK + (p & 31) * 8);
      xr[i][0] = src[0], xr[i][1] = src[1];
    }
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int p = tid + 256 * i, row = p >> 5;
      *(u32x4 *)(xs + buf * XBUF + row * ROWB + (((p & 31) ^ (row & 15)) << 4)) =
          u32x4{pack_bf16x2(xr[i][0].x, xr[i][0].y), pack_bf16x2(xr[i][0].z, xr[i][0].w),
                pack_bf16x2(xr[i][1].x, xr[i][1].y), pack_bf16x2(xr[i][1].z, xr[i][1].w)};
    }
  };
  uint32_t xoff[XDMA];
#pragma unroll
  for (int i = 0; i < XDMA; ++i) {
    const int row = 2 * (wn * XDMA + i) + (lane >> 5);
    const int m = min(m0 + row, a.M - 1);  // rows past M repeat the last row (not stored)
    xoff[i] = (uint32_t)m * (uint32_t)a.K * 2u + ((uint32_t)((lane & 31) ^ (row & 15)) << 4);
  }
  auto issue_x = [&](int c, int buf) {
#pragma unroll
    for (int i = 0; i < XDMA; ++i)
      dma16(a.x, xoff[i] + (uint32_t)c * ROWB, lds_addr(xs + buf * XBUF + (wn * XDMA + i) * 1024));
  };
  const int kstride = a.w_packed ? 1024 : 64;  // bytes between 64-k steps of a lane's codes
  uint32_t woff[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int n = min(n0 + 16 * g + r16, a.N - 1);
    woff[g] = a.w_packed ? (uint32_t)(n >> 4) * (uint32_t)KT * 1024u + (uint32_t)((n & 15) + 16 * kq) * 16u
                         : (uint32_t)n * (uint32_t)a.K + (uint32_t)kq * 16u;
  }
  // Grouped scales: the split's own groups of the workgroup's rows go to LDS
  // as [group][row] first, behind the first chunk's loads (read from memory
  // step by step, 4 bytes of 16 rows each, they cost 2 to 4 us of 14 at 48 x
  // 6144 x 4096, G = 128). A 64-k step's group is step / (G / 64), by a
  // reciprocal (exact below 2^16 steps).
  float *scl = (float *)(smem + 2 * KG * XBUF);
  const uint32_t gk = (uint32_t)a.G / 64, ginv = gk > 1 ? 0xffffffffu / gk + 1 : 0;
  auto group_of = [&](int step) { return (int)(gk > 1 ? __umulhi((uint32_t)step, ginv) : (uint32_t)step); };
  const int g_lo = GRP ? group_of(4 * cb) : 0, g_n = GRP ? group_of(4 * ce - 1) + 1 - g_lo : 1;
  auto stage_scales = [&]() {
    const int nt = n0 - wn * 16 * RG;  // the workgroup's first weight row
    for (int e = threadIdx.x; e < TN * g_n; e += 256 * KG) {
      const int row = e / g_n, g = e - row * g_n;
      scl[g * TN + row] = a.scale[(int64_t)min(nt + row, a.N - 1) * groups + g_lo + g];
    }
  };
  struct WSet {
    u32x4 w[4][RG];
  };
  float sc[RG];
  auto load_w = [&](int c, WSet &ws) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int g = 0; g < RG; ++g)
        ws.w[s][g] = *(const u32x4 *)(a.w + woff[g] + (uint32_t)(4 * c + s) * (uint32_t)kstride);
  };
  const int last = ce - 1;
  auto chunk_of = [&](int i) { return min(cb + kg + KG * i, last); };  // past the end: re-read, not multiplied
  WSet w0, w1;
  if constexpr (XF) load_x(chunk_of(0));
  else issue_x(chunk_of(0), 0);
  if constexpr (!GRP) {
#pragma unroll
    for (int g = 0; g < RG; ++g) sc[g] = a.scale[(int64_t)min(n0 + 16 * g + r16, a.N - 1)];
  }
  load_w(chunk_of(0), w0);
  if constexpr (GRP) stage_scales();
  if constexpr (XF) store_x(0);
  f32x4 acc[RG][FJ];
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[g][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Chunk i from `cur`, while chunk i + 1 loads: its copies and weights are
  // all requested first and so have the whole step to arrive.
  auto step = [&](int i, const WSet &cur, WSet &nxt) {
    // chunk i is in LDS; buffer i + 1 is free
    if constexpr (XF) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const char *xb = xs + (i & 1) * XBUF;
    const int cn = chunk_of(i + 1);
    if constexpr (XF) load_x(cn);
    else issue_x(cn, (i + 1) & 1);
    load_w(cn, nxt);
    const bool live = cb + kg + KG * i < ce;  // (wave-uniform) this group has a chunk left
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (!live) break;
      float scs[RG];
      if constexpr (GRP) {
        const float *sp = scl + (group_of(4 * (cb + kg + KG * i) + s) - g_lo) * TN + wn * 16 * RG + r16;
#pragma unroll
        for (int g = 0; g < RG; ++g) scs[g] = sp[16 * g];
      }
      bf16x8 xf[2][FJ];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
          xf[h][j] = as_bf16x8(*(const u32x4 *)(xb + (16 * j + r16) * ROWB + (((8 * s + 2 * kq + h) ^ r16) << 4)));
      u32x4 wf[RG][2];
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        const float scale = GRP ? scs[g] : sc[g], ms = -128.0f * scale;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint2 lo = u8x4_to_dq_bf16x4(cur.w[s][g][2 * h], scale, ms);
          const uint2 hi = u8x4_to_dq_bf16x4(cur.w[s][g][2 * h + 1], scale, ms);
          wf[g][h] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
          for (int j = 0; j < FJ; ++j) acc[g][j] = mfma16x16x32(as_bf16x8(wf[g][h]), xf[h][j], acc[g][j]);
    }
    if constexpr (XF) store_x((i + 1) & 1);
  };
  int i = 0;
  for (; i + 2 <= iters; i += 2) {
    step(i, w0, w1);
    step(i + 1, w1, w0);
  }
  if (i < iters) step(i, w0, w1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the last chunk
  __syncthreads();
  f32x4 *red = (f32x4 *)smem;
  if (kg > 0)
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
      for (int j = 0; j < FJ; ++j) red[(wn * RG * FJ + g * FJ + j) * 64 + lane] = acc[g][j];
  __syncthreads();
  if (kg > 0) return;
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[g][j] += red[(wn * RG * FJ + g * FJ + j) * 64 + lane];
  // lane holds D[n = 16 g + 4 kq + e][m = 16 j + r16]
#pragma unroll
  for (int j = 0; j < FJ; ++j)
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      const int m = m0 + 16 * j + r16, n = n0 + 16 * g + 4 * kq;
      if (a.ksplit == 1)
        store4(a, m, n, acc[g][j]);
      else if (m < a.M && n < a.N)
        *(f32x4 *)(a.ws + ((int64_t)split * a.M + m) * a.N + n) = acc[g][j];
    }
}

// ---- F32 compute (gemm.hip rxw8_gemm_f32c's product and contract) -------------
//   y[m, n] = sum_g s[n, g] * sum_{k in g} (xh[m, k] + xl[m, k]) * (u8[n, k] - 128)
// on the same scheme: weights global -> registers -> exact bf16 codes, each
// wave its own 64 weight rows; 64 (16 FJ) rows of xh and xl through LDS in
// chunks of 128 k. 256 x 64 output tiles of 4 waves, two workgroups per CU
// with waits and barriers of their own, where the 256 x 128 tiles of gemm.hip
// hold a CU each with 8 waves in lockstep and, at a few hundred rows, leave
// half the CUs without a tile or split K into a reduce pass. A scale group's
// f32 sum is scaled into the total at the group's end (a split's part of a
// group scales its own part).
struct LinearF32GemmArgs {
  const uint16_t *xh, *xl;  // [M, K] bf16 hi / lo parts of x
  const uint8_t *w;         // [N, K] u8 codes, or packed [N/16, K/64, 1024]
  const float *scale;       // [N, K / G]
  float *y;                 // [M, N]
  int M, N, K, G;
  int y_mode;               // 0: y = result; 1: y += result
  int w_packed;
  int ksplit;               // 1, or the number of K splits
  float *ws;                // [ksplit, M, N] f32 partials when ksplit > 1
};

// Four codes u -> the bf16 pairs of u - 128 (exact): the top bit flipped they
// are signed bytes, one sign-extending conversion each
__device__ __forceinline__ uint2 signed_bf16x4(uint32_t w) {
  w ^= 0x80808080u;
  const float f0 = (float)(int8_t)w, f1 = (float)(int8_t)(w >> 8);
  const float f2 = (float)(int8_t)(w >> 16), f3 = (float)((int32_t)w >> 24);
  return uint2{pack_bf16x2(f0, f1), pack_bf16x2(f2, f3)};
}

template <int FJ>
__device__ __forceinline__ void gemm_f32m(const LinearF32GemmArgs &a) {
  constexpr int RG = 4, TM = 16 * FJ, TN = 256, CKF = 128, RB = CKF * 2, XB = TM * RB;
  constexpr int XDMA = XB / 1024 / 4;  // LDS-DMA instructions per wave, part and chunk
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // [2 buffers][xh | xl], scales
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wn = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_m = (a.M + TM - 1) / TM, tiles_n = (a.N + TN - 1) / TN, ntiles = tiles_m * tiles_n;
  const int per_xcd = (ntiles * a.ksplit + 7) / 8;
  const int t_all = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (t_all >= ntiles * a.ksplit) return;
  const int split = t_all / ntiles, t = t_all - split * ntiles;
  constexpr int GN = 8;  // n tiles per tile-order group (n fastest): an XCD's 64 tiles are about 8 x 8
  const int group = t / (GN * tiles_m), in = t - group * GN * tiles_m, gw = min(GN, tiles_n - group * GN);
  const int nt = (group * GN + in % gw) * TN, n0 = nt + wn * 64, m0 = in / gw * TM;
  const int KT = a.K / 64, chunks = a.K / CKF, ng = a.K / a.G;
  const int cb = split * chunks / a.ksplit, ce = (split + 1) * chunks / a.ksplit, last = ce - 1;
  const uint32_t gk = (uint32_t)a.G / 64, ginv = gk > 1 ? 0xffffffffu / gk + 1 : 0;
  auto group_of = [&](int step) { return (int)(gk > 1 ? __umulhi((uint32_t)step, ginv) : (uint32_t)step); };
  float *scl = (float *)(smem + 4 * XB);  // [group][row], the split's groups
  const int g_lo = group_of(2 * cb), g_n = group_of(2 * ce - 1) + 1 - g_lo;

  uint32_t xoff[XDMA];
#pragma unroll
  for (int i = 0; i < XDMA; ++i) {
    const int row = 4 * (wn * XDMA + i) + (lane >> 4);
    const int m = min(m0 + row, a.M - 1);  // rows past M repeat the last row (not stored)
    xoff[i] = (uint32_t)m * (uint32_t)a.K * 2u + ((uint32_t)((lane & 15) ^ (row & 15)) << 4);
  }
  auto issue_x = [&](int c, int buf) {
#pragma unroll
    for (int i = 0; i < XDMA; ++i) {
      const uint32_t l = lds_addr(smem + buf * 2 * XB + (wn * XDMA + i) * 1024);
      dma16(a.xh, xoff[i] + (uint32_t)c * RB, l);
      dma16(a.xl, xoff[i] + (uint32_t)c * RB, l + XB);
    }
  };
  const int kstride = a.w_packed ? 1024 : 64;
  uint32_t woff[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int n = min(n0 + 16 * g + r16, a.N - 1);
    woff[g] = a.w_packed ? (uint32_t)(n >> 4) * (uint32_t)KT * 1024u + (uint32_t)((n & 15) + 16 * kq) * 16u
                         : (uint32_t)n * (uint32_t)a.K + (uint32_t)kq * 16u;
  }
  u32x4 w[2][RG];
  auto load_w = [&](int c, int s) {
#pragma unroll
    for (int g = 0; g < RG; ++g)
      w[s][g] = *(const u32x4 *)(a.w + woff[g] + (uint32_t)(2 * c + s) * (uint32_t)kstride);
  };
  issue_x(cb, 0);
  load_w(cb, 0);
  load_w(cb, 1);
  for (int e = threadIdx.x; e < TN * g_n; e += 256) {
    const int row = e / g_n, g = e - row * g_n;
    scl[g * TN + row] = a.scale[(int64_t)min(nt + row, a.N - 1) * ng + g_lo + g];
  }
  f32x4 acc[RG][FJ], tot[RG][FJ];
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[g][j] = tot[g][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c = cb; c < ce; ++c) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // chunk c is here; the other buffer is free
    const char *xb = smem + ((c - cb) & 1) * 2 * XB;
    const int cn = min(c + 1, last);
    issue_x(cn, (c + 1 - cb) & 1);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u32x4 wf[RG][2];
#pragma unroll
      for (int g = 0; g < RG; ++g)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint2 lo = signed_bf16x4(w[s][g][2 * h]), hi = signed_bf16x4(w[s][g][2 * h + 1]);
          wf[g][h] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
      load_w(cn, s);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8 xf[2][FJ];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int j = 0; j < FJ; ++j)
            xf[p][j] = as_bf16x8(*(const u32x4 *)(xb + p * XB + (16 * j + r16) * RB + (((8 * s + 2 * kq + h) ^ r16) << 4)));
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int j = 0; j < FJ; ++j) acc[g][j] = mfma16x16x32(as_bf16x8(wf[g][h]), xf[p][j], acc[g][j]);
      }
      const int step = 2 * c + s, gi = group_of(step);
      if (step + 1 == 2 * ce || group_of(step + 1) != gi) {  // (uniform) the group's, or the split's, end
#pragma unroll
        for (int g = 0; g < RG; ++g) {
          const f32x4 sv = *(const f32x4 *)(scl + (gi - g_lo) * TN + wn * 64 + 16 * g + 4 * kq);
#pragma unroll
          for (int j = 0; j < FJ; ++j) {
            tot[g][j] += sv * acc[g][j];
            acc[g][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the last chunk
  // lane holds D[n = 16 g + 4 kq + e][m = 16 j + r16]
#pragma unroll
  for (int j = 0; j < FJ; ++j) {
    const int m = m0 + 16 * j + r16;
    if (m >= a.M) continue;
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      const int n = n0 + 16 * g + 4 * kq;
      if (n >= a.N) continue;
      if (a.ksplit > 1) {
        *(f32x4 *)(a.ws + ((int64_t)split * a.M + m) * a.N + n) = tot[g][j];
      } else {
        f32x4 *yp = (f32x4 *)(a.y + (int64_t)m * a.N + n);
        *yp = a.y_mode == 1 ? *yp + tot[g][j] : tot[g][j];
      }
    }
  }
}

}  // namespace

// Launch contract (checked by the host): x bf16, or f32 for the _xf kernels
// (all 16-byte aligned); N % 16 == 0, K % 256 == 0, G % 64 == 0
// (or G == K: the per-channel kernels), M * K * 2 < 2^31, N * K < 2^32, ksplit
// <= K / 256, LDS 4 * 16 FJ * 512 bytes (+ the
// split's groups x 64 RG floats of grouped scales); 512 threads; grid =
// 8 * ceil(tiles * ksplit / 8).
#define RXW8_GEMM_MID(FJ, RG, GRP, XF, SUFFIX)                                                   \
  extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))      \
      rxw8_gemm_mid_m##FJ##_r##RG##SUFFIX(GemmArgs a) {                                          \
    gemm_mid<FJ, RG, GRP, XF>(a);                                                             \
  }
#define RXW8_GEMM_MID_FJ(FJ)                 \
  RXW8_GEMM_MID(FJ, 1, false, false, )       \
  RXW8_GEMM_MID(FJ, 2, false, false, )       \
  RXW8_GEMM_MID(FJ, 1, true, false, _g)      \
  RXW8_GEMM_MID(FJ, 2, true, false, _g)      \
  RXW8_GEMM_MID(FJ, 1, false, true, _xf)     \
  RXW8_GEMM_MID(FJ, 2, false, true, _xf)     \
  RXW8_GEMM_MID(FJ, 1, true, true, _g_xf)    \
  RXW8_GEMM_MID(FJ, 2, true, true, _g_xf)
RXW8_GEMM_MID_FJ(1)
RXW8_GEMM_MID_FJ(2)
RXW8_GEMM_MID_FJ(3)
RXW8_GEMM_MID_FJ(4)

// Launch contract as rxw8_gemm_f32c (gemm.hip), and: K % 128 == 0, ksplit <= K
// / 128, LDS 4 * 16 FJ * 256 bytes + the split's groups x 256 floats; 256
// threads; grid = 8 * ceil(tiles * ksplit / 8).
#define RXW8_GEMM_F32M(FJ)                                                                      \
  extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))    \
      rxw8_gemm_mid_f32_m##FJ(LinearF32GemmArgs a) {                                           \
    gemm_f32m<FJ>(a);                                                                          \
  }
RXW8_GEMM_F32M(2)
RXW8_GEMM_F32M(4)
