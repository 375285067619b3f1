// Grouped-query attention with f32 scores and f32 probabilities on the matrix
// cores (attention.rs:83-135 with SDPA :150-252), for head widths 64, 128 and
// 256: the masked / any-length form (f32 q, k, v and an additive mask), causal
// prefill over bf16 caches of the widths and group sizes the bf16 flash kernel
// does not take.
//
// v_mfma_f32_16x16x4_f32 multiplies f32 operands exactly as f32 FMAs would, so
// bf16 operands are only widened and nothing is rounded below f32. The G
// query heads of a kv head and the queries fold into one list of rows, row
// r = i * G + g (query i, head g of the group): every row of a tile shares
// the K/V tile, whatever the group size, and causal limits grow with r.
//
// Operand layouts (lane l: col = l % 16, j = l / 16), per tile of 16 keys:
//   S^T = K Q^T: A = K (row = key col, k index j), B = q of row col. A lane's
//     16-byte piece of a K row feeds one MFMA per element, with the k index j
//     standing for element e of piece 4 u + j; q sits in registers in that
//     order. The result gives lane l the scores of row col, keys 4 j + 0..3.
//   O^T += V^T P^T: k index j of MFMA c stands for key 4 j + c, so P's operand
//     is the score register c itself: no exchange between lanes. A lane's
//     4 elements of V row 4 j + c feed 4 MFMAs. A lane owns row col's outputs
//     d = 64 u + 16 j + 4 i + e, so the running maximum's rescale factor is
//     lane-local too.
// Bound: the f32 matrix rate (154 TFLOP/s for a large product). Measured: 16 / 8
// heads x 512 x 512 keys at D = 128 under a causal mask 34.5 us against 1,292 us
// for one wave per row on the VALU; causal prefill of 7 x 425 rows, 32 / 4
// heads, D = 256: 245 us (85 TFLOP/s) against 9.7 ms. What is left between
// that and the rate is the softmax and copy issue, which overlap the other
// waves' MFMAs only in part; under the causal mask (MFMA pipes 21% busy) also
// the round of workgroups, which lasts as long as the row tile that sees every
// key.
// A tile whose mask entries are all -inf for a wave's rows adds exactly nothing
// when its K and V values are ordinary numbers; the wave then skips its
// products (after a look at the tile in LDS: NaN and infinities still reach the
// output as in the reference).
#include <type_traits>
#include <utility>

#include "common.h"

// (matches ops.cpp)
struct GqaTileArgs {
  const void *q, *k, *v;
  const float *mask;         // additive, or null
  void *out;
  int64_t bdim[4];           // batch prefix dims (innermost last), 1 where absent
  int64_t mb[4];             // mask stride of each batch dim (0: broadcast)
  int64_t msh, msi;          // mask strides of head, query (0: broadcast)
  int64_t msj;               // of key: 1, or 0 (broadcast)
  int64_t q_sb, q_sh, q_si;  // element strides of q (batch, head, row)
  int64_t o_sb, o_sh, o_si;  // of out
  int64_t k_sb, k_sh;        // of k (rows of D contiguous), v: v_sb, v_sh
  int64_t v_sb, v_sh;
  const int32_t *starts;     // [NB] causal: query i sees keys 0 .. st + i, st = clamp(starts[b], 0, Sk - Sq); or null
  const int32_t *lens;       // [NB] decode: keys 0 .. clamp(lens[b], 1, Sk) - 1; or null
  const int32_t *slots;      // [NB] K/V batch index of query batch b, or null (b)
  float *part;               // nsplit > 1: [unit][split][row][4 + D] partials (m, l, -, -, o)
  int *counters;             // nsplit > 1: [unit] arrivals, zero between launches
  int NB, Hq, Hkv, Sq, Sk, tiles, nsplit;
  float scale;
  int q_bf16, out_bf16;
};

// Split partials and counters of a runtime's calls, one block for calls that
// run and one for calls that a stream capture records (16 MiB and 64 KiB each,
// as the no-allocation entry's array). This code object is loaded once per
// runtime, so each runtime has its own, and a captured pointer is good until
// the runtime ends: no later call moves the block, and none that runs beside a
// replay uses it. runtime_create takes the address and clears the counters.
extern "C" {
__attribute__((used)) __device__ __align__(256) unsigned char rxw8_f32_attention_blocks[2][(64 << 10) + (16 << 20)];
}

namespace {

constexpr float kNegInf = -__builtin_huge_valf();
// Bits of 2^60: for |q|, |k| below it, products and their sums over 256 dims
// stay finite. (NaN and infinities have larger bits.)
constexpr uint32_t kTameBits = (127u + 60u) << 23, kInfBits = 255u << 23;

__device__ __forceinline__ float max4(float v) {
  uint2 p = pair_xor16(v);
  v = fmaxf(__uint_as_float(p.x), __uint_as_float(p.y));
  p = pair_xor32(v);
  return fmaxf(__uint_as_float(p.x), __uint_as_float(p.y));
}
__device__ __forceinline__ float sum4(float v) { return sum_xor32(sum_xor16(v)); }

// 4 bytes per lane from the lane's own address to LDS at lds + 4 * lane (see dma16)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma4(const float *p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off"
               :: "v"(p), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// K / V elements: ES bytes each, EPC per 16-byte piece
template <bool BF>
struct Kv;
template <>
struct Kv<false> {
  static constexpr int ES = 4, EPC = 4;
  typedef f32x4 Piece;  // one K piece
  typedef f32x4 Four;   // four V elements
  static __device__ __forceinline__ float el(const Piece &v, int e) { return v[e]; }
  static __device__ __forceinline__ float four(const Four &v, int e) { return v[e]; }
};
template <>
struct Kv<true> {
  static constexpr int ES = 2, EPC = 8;
  typedef u32x4 Piece;
  typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned Four;
  static __device__ __forceinline__ float el(const Piece &v, int e) {
    return __uint_as_float(e & 1 ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16);
  }
  static __device__ __forceinline__ float four(const Four &v, int e) {
    return __uint_as_float(e & 1 ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16);
  }
};

// Whether every value of a staged tile of BYTES (read by the whole wave) has
// magnitude bits below `bits`
template <bool BF, int BYTES>
__device__ __forceinline__ bool below(const char *t, int lane, uint32_t bits) {
  uint32_t hi = 0, lo = 0;
#pragma unroll
  for (int o = 0; o < BYTES; o += 1024) {
    const u32x4 v = *(const u32x4 *)(t + o + 16 * lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      hi = max(hi, v[e] & (BF ? 0x7fff0000u : 0x7fffffffu));
      if constexpr (BF) lo = max(lo, v[e] & 0x7fffu);
    }
  }
  return __all(max(hi, lo << 16) < bits);
}

// One row's softmax state and its outputs held by a lane: o[u][e][i] is
// d = 64 u + 16 j + 4 i + e (unnormalised)
template <int D>
struct RowState {
  float m = kNegInf, l = 0.f;
  f32x4 o[D / 64][4];
  __device__ RowState() {
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[u][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // pp: the row's [4 + D] record (16-byte aligned) of another range of keys
  __device__ __forceinline__ void merge(const float *pp, int j) {
    const float m2 = pp[0], l2 = pp[1];
    const float M = fmaxf(m, m2);
    const float f1 = m == kNegInf ? 0.f : expf(m - M), f2 = m2 == kNegInf ? 0.f : expf(m2 - M);
    l = l * f1 + l2 * f2;
    m = M;
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 v = *(const f32x4 *)(pp + 4 + 64 * u + 16 * j + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[u][e][i] = o[u][e][i] * f1 + v[e] * f2;
      }
  }
  __device__ __forceinline__ void save(float *pp, int j) const {
    if (j == 0) pp[0] = m, pp[1] = l;
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(f32x4 *)(pp + 4 + 64 * u + 16 * j + 4 * i) = f32x4{o[u][0][i], o[u][1][i], o[u][2][i], o[u][3][i]};
  }
};

// Device-coherent (sc1: write-through, respectively past this XCD's caches)
// 16-byte stores and loads of split records
__device__ __forceinline__ void store_coherent(float *base, uint32_t byte, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), buf_rsrc(base, 0x7fffffffu), byte, 0, 16);
}
__device__ __forceinline__ f32x4 load_coherent(const float *base, uint32_t byte) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buf_rsrc(base, 0x7fffffffu), byte, 0, 16));
}

// Exchange between the 4 lanes of a row (j = 0..3): on return o[u][e][i] is
// d = 64 u + 16 i + 4 j + e, so that the lanes' 16-byte pieces of one i are 64
// contiguous bytes.
template <int D>
__device__ __forceinline__ void by_pieces(RowState<D> &s) {
#pragma unroll
  for (int u = 0; u < D / 64; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f32x4 &o = s.o[u][e];
      unsigned x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = __float_as_uint(o[i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(x[i], x[i + 2], false, false);
        x[i] = r[0], x[i + 2] = r[1];
      }
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const auto r = __builtin_amdgcn_permlane16_swap(x[i], x[i + 1], false, false);
        x[i] = r[0], x[i + 1] = r[1];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(x[i]);
    }
}

// out element offset oo of a row (state by_pieces); y = o / l. A row that saw
// no key (m = -inf) is NaN, the reference's softmax of an all-masked row.
template <int D>
__device__ __forceinline__ void store_row(const GqaTileArgs &a, const RowState<D> &s, int64_t oo, int j) {
  const float inv = s.m == kNegInf ? __builtin_nanf("") : 1.0f / s.l;
#pragma unroll
  for (int u = 0; u < D / 64; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t at = oo + 64 * u + 16 * i + 4 * j;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = s.m == kNegInf ? inv : s.o[u][e][i] * inv;
      if (a.out_bf16)
        *(uint2 *)((uint16_t *)a.out + at) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      else
        *(f32x4 *)((float *)a.out + at) = f32x4{y[0], y[1], y[2], y[3]};
    }
}

// Row r = i * G + g of (batch b, kv head): where its q, out and mask rows are
// and how many keys it sees
struct RowAt {
  int64_t q, o;
  const float *mask;
  int vis;
};
__device__ __forceinline__ int row_vis(const GqaTileArgs &a, int b, int i) {
  if (a.starts) return min(max(a.starts[b], 0), a.Sk - a.Sq) + i + 1;
  if (a.lens) return min(max(a.lens[b], 1), a.Sk);
  return a.Sk;
}
__device__ __forceinline__ RowAt row_at(const GqaTileArgs &a, int b, int kvh, int r) {
  const int G = a.Hq / a.Hkv;
  const int i = r / G, h = kvh * G + (r - i * G);
  RowAt x;
  x.q = b * a.q_sb + h * a.q_sh + i * a.q_si;
  x.o = b * a.o_sb + h * a.o_sh + i * a.o_si;
  x.vis = row_vis(a, b, i);
  x.mask = nullptr;
  if (a.mask) {
    int64_t off = 0;
    int rest = b;
    for (int t = 3; t >= 0; --t) {
      const int n = (int)a.bdim[t];  // (the batch count fits an int)
      if (n == 1) continue;
      const int digit = rest % n;
      rest /= n;
      off += digit * a.mb[t];
    }
    x.mask = a.mask + off + h * a.msh + i * a.msi;
  }
  return x;
}

// q of one row in MFMA order: qr[u * EPC + e] = q[(4 u + j) * EPC + e]
__device__ __forceinline__ void four_bf16(const uint2 &w, float *x) {
  x[0] = __uint_as_float(w.x << 16), x[1] = __uint_as_float(w.x & 0xffff0000u);
  x[2] = __uint_as_float(w.y << 16), x[3] = __uint_as_float(w.y & 0xffff0000u);
}
template <int D, int EPC>
__device__ __forceinline__ void load_q(const GqaTileArgs &a, int64_t at, int j, float (&qr)[D / 4]) {
  // (one branch around all the loads: a branch per load would wait for each)
  if (a.q_bf16) {
    uint2 w[D / 16];
#pragma unroll
    for (int x = 0; x < D / 16; ++x)
      w[x] = *(const uint2 *)((const uint16_t *)a.q + at + (4 * (4 * x / EPC) + j) * EPC + 4 * x % EPC);
#pragma unroll
    for (int x = 0; x < D / 16; ++x) four_bf16(w[x], qr + 4 * x);
  } else {
#pragma unroll
    for (int x = 0; x < D / 16; ++x) {
      const f32x4 w = *(const f32x4 *)((const float *)a.q + at + (4 * (4 * x / EPC) + j) * EPC + 4 * x % EPC);
#pragma unroll
      for (int e = 0; e < 4; ++e) qr[4 * x + e] = w[e];
    }
  }
}

// e^(s - m); before any visible key (m = -inf) every score is -inf and weighs
// nothing, or is NaN and stays it.
// (__expf rounds (s - m) log2(e), an error that grows with |s - m| but stays
// below that of the score itself. Against 64 bits, at widths 64 / 128 / 256, 1
// and 200 queries, 700 keys, scores of width 1 to 64: 1.8e-7 to 1.9e-6 with it
// where the scalar kernels with expf give 5.1e-7 to 8.1e-6; equal, 1e-6 to
// 4.5e-6 on both, with 200 added to every score.)
__device__ __forceinline__ float prob(float s, float m) {
  return m == kNegInf ? (s != s ? s : 0.f) : __expf(s - m);
}

// The tile's scores (already scaled and masked) -> probabilities in p against
// the row's reference maximum m. The reference moves (and l and the outputs
// are rescaled) only when a score exceeds it by more than 8: p then stays
// below e^8, l and o carry the same factor, and most tiles need neither the
// maximum over the row's lanes nor the rescale. l sums this lane's own keys
// (the lanes of a row share m, so their sums add up at the end).
template <int D>
__device__ __forceinline__ void softmax_step(RowState<D> &s, float (&p)[4]) {
  const float top = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
  if (__any(top > s.m + 8.f)) {  // (m = -inf: any key that is not masked)
    const float mn = fmaxf(s.m, max4(top));
    const float alpha = s.m == kNegInf ? 0.f : expf(s.m - mn);
    s.l *= alpha;
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) s.o[u][e] *= alpha;
    s.m = mn;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) p[c] = prob(p[c], s.m);
  s.l += (p[0] + p[1]) + (p[2] + p[3]);
}

// Publish this workgroup's rows and, in the workgroup that completes the
// unit's nsplit arrivals, return true once its records can be read. The
// records' device-coherent stores have completed (vmcnt 0, then the barrier)
// before the arrival is counted, and the last arriver reads them with
// device-coherent loads: no release fence, which would write back the whole
// L2. Uniform per workgroup.
__device__ __forceinline__ bool last_arrival(int *counter, int nsplit, int *flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
  __syncthreads();
  return *flag;
}

// Merge the nsplit (<= 32) records of each of `rows` rows (record (split, row)
// at base + (split * rows_per + row) * (4 + D)) in split order and write the
// outputs: the rows' factors in LDS (fac: [rows][nsplit + 1], 1 / l last)
// first, then 4 outputs per thread, 8 records in flight.
template <int D, typename OUT>
__device__ __forceinline__ void merge_units(const GqaTileArgs &a, const float *base, int rows, int rows_per,
                                            float *fac, OUT out_at) {
  const int S = a.nsplit, NT = blockDim.x;
  const int sp = S <= 2 ? 2 : S <= 4 ? 4 : S <= 8 ? 8 : S <= 16 ? 16 : 32;  // lanes per row
  for (int t = threadIdx.x; t < (rows * sp + 63) / 64 * 64; t += NT) {      // whole waves
    const int r = t / sp, s = t - r * sp;
    float m = kNegInf, l = 0.f;
    if (r < rows && s < S) {
      const f32x4 v = load_coherent(base, (uint32_t)(s * rows_per + r) * (4 + D) * 4);
      m = v[0], l = v[1];
    }
    float M = m;
    for (int x = 1; x < sp; x <<= 1) M = fmaxf(M, __shfl_xor(M, x));
    const float e = m == kNegInf ? 0.f : expf(m - M);
    float L = e * l;
    for (int x = 1; x < sp; x <<= 1) L += __shfl_xor(L, x);
    if (r < rows && s < S) fac[r * (S + 1) + s] = e;
    if (r < rows && s == 0) fac[r * (S + 1) + S] = M == kNegInf ? __builtin_nanf("") : 1.0f / L;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < rows * (D / 4); t += NT) {
    const int r = t / (D / 4), d = 4 * (t - r * (D / 4));
    const float *f = fac + r * (S + 1);
    f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < S; s0 += 8) {
      f32x4 v[8];
#pragma unroll
      for (int s = 0; s < 8; ++s)
        v[s] = load_coherent(base, ((uint32_t)(min(s0 + s, S - 1) * rows_per + r) * (4 + D) + 4 + d) * 4);
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (s0 + s < S) y += f[s0 + s] * v[s];
    }
    y *= f[S];
    const int64_t at = out_at(r) + d;
    if (a.out_bf16)
      *(uint2 *)((uint16_t *)a.out + at) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    else
      *(f32x4 *)((float *)a.out + at) = y;
  }
}

// ---- many rows per kv head: K/V tiles shared through LDS ---------------------
// A workgroup of RG x KG waves owns 16 RG rows of one (batch, kv head). Its KG
// wave groups take alternate tiles of 16 keys, each through a ring of NB
// buffers filled by LDS DMA (NB - 1 tiles in flight), and merge at the end.
// Every wave issues the same number of copies per step (past the last tile
// they repeat it), so the waits count them exactly.
template <int D, bool BF, int RG, int KG, int NB>
__device__ void gqa_tile(const GqaTileArgs &a) {
  typedef Kv<BF> T;
  constexpr int ROWB = D * T::ES, TILEB = 16 * ROWB, CH = ROWB / 16, NI = TILEB / 1024;
  constexpr int OPS = 2 * NI / RG;      // K/V copies of a wave per tile, 1 KiB each
  constexpr int UK = D / (4 * T::EPC);  // K pieces per lane
  constexpr bool PRE = D < 256 || BF || KG > 1;  // registers to hold fragments ahead
  static_assert((2 * NI) % RG == 0 && (NB - 2) * (OPS + 4) < 64, "");
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  __shared__ int flag;
  const int lane = threadIdx.x & 63, j = lane >> 4, col = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rg = wv % RG, kg = wv / RG;
  const int NBH = a.NB * a.Hkv, G = a.Hq / a.Hkv, R = G * a.Sq;
  int blk = blockIdx.x;
  const int bh = blk % NBH;
  blk /= NBH;
  const int split = blk % a.nsplit;
  const int tile = a.tiles - 1 - blk / a.nsplit;  // the longest causal tiles first
  const int b = bh / a.Hkv, kvh = bh - b * a.Hkv;
  const int slot = a.slots ? a.slots[b] : b;
  const char *kp = (const char *)a.k + (slot * a.k_sb + kvh * a.k_sh) * T::ES;
  const char *vp = (const char *)a.v + (slot * a.v_sb + kvh * a.v_sh) * T::ES;
  const int r0 = tile * 16 * RG + rg * 16;  // this wave's rows r0 .. r0 + 15
  const RowAt row = row_at(a, b, kvh, min(r0 + col, R - 1));
  // keys that some row of the workgroup sees; of this wave's rows, some and all
  const int nkeys = row_vis(a, b, (min((tile + 1) * 16 * RG, R) - 1) / G);
  const int vis_max = row_vis(a, b, min(r0 + 15, R - 1) / G), vis_min = row_vis(a, b, min(r0, R - 1) / G);
  const int ntiles = (nkeys + 15) / 16, per = (ntiles + a.nsplit - 1) / a.nsplit;
  const int t0 = split * per, t1 = min(ntiles, t0 + per);
  char *ring = tile_lds + kg * NB * 2 * TILEB;
  float *mring = (float *)(tile_lds + KG * NB * 2 * TILEB) + wv * NB * 256;  // mask values, per wave
  // step n of this wave group is tile t0 + kg + KG n. The copies' offsets
  // within a tile are fixed; only the last tile clamps its rows to the last key.
  int krow[OPS];
  uint32_t voff[OPS];
#pragma unroll
  for (int x = 0; x < OPS; ++x) {
    const int in = x * RG + rg, kv = in >= NI;  // wave-uniform
    const int o = (kv ? in - NI : in) * 1024 + 16 * lane;
    const int ch = (o % ROWB) / 16;
    krow[x] = o / ROWB;
    const int sw = CH >= 16 ? krow[x] & 15 : (krow[x] >> 1) & 7;  // K pieces swizzled: fragment reads conflict-free
    voff[x] = 16 * (kv ? ch : ch ^ sw);
  }
  auto issue = [&](int n) {
    const int t = min(t0 + kg + KG * n, t1 - 1), bsel = n % NB;
    char *dst = ring + bsel * 2 * TILEB;
    if (a.mask) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dma4(row.mask + (a.msj ? min(16 * t + 4 * j + c, a.Sk - 1) : 0), lds_addr((char *)(mring + bsel * 256 + 64 * c)));
    }
    const bool whole = 16 * t + 16 <= nkeys;
#pragma unroll
    for (int x = 0; x < OPS; ++x) {
      const int in = x * RG + rg, kv = in >= NI;
      const uint32_t kr = whole ? krow[x] : min(16 * t + krow[x], nkeys - 1) - 16 * t;
      dma16((kv ? vp : kp) + (int64_t)t * TILEB, kr * ROWB + voff[x], lds_addr(dst + in * 1024));
    }
  };
  const int steps = t1 > t0 ? (t1 - t0 + KG - 1) / KG : 0;  // uniform per workgroup
  if (steps)
    for (int n = 0; n < NB - 1; ++n) issue(n);
  float qr[D / 4];
  load_q<D, T::EPC>(a, row.q, j, qr);
  uint32_t qmax = 0;
#pragma unroll
  for (int x = 0; x < D / 4; ++x) qmax = max(qmax, __float_as_uint(qr[x]) & 0x7fffffffu);
  const bool q_tame = __all(qmax < kTameBits);
  RowState<D> st;
  for (int n = 0; n < steps; ++n) {
    const int t = t0 + kg + KG * n, bsel = n % NB;
    const char *kt = ring + bsel * 2 * TILEB, *vt = kt + TILEB;
    if (a.mask)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * (OPS + 4)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * OPS) : "memory");
    // V rows past the last key repeat it, with weight 0, which would make NaN of
    // an infinity: each wave puts zeros over those that it has copied
    if (t < t1 && 16 * t + 16 > nkeys) {
      int at = lane;
      unsigned z = 0;
      asm volatile("" : "+v"(at), "+v"(z));  // (formed here: kept through the loop they cost D = 256 registers)
#pragma unroll
      for (int x = 0; x < OPS; ++x) {
        const int in = x * RG + rg;
        if (in >= NI && 16 * t + krow[x] >= nkeys)
          *(u32x4 *)(ring + bsel * 2 * TILEB + in * 1024 + 16 * at) = u32x4{z, z, z, z};
      }
    }
    __syncthreads();
    issue(n + NB - 1);  // into the buffer read before this barrier
    bool work = t < t1 && 16 * t < vis_max;  // wave-uniform
    float mc[4] = {0.f, 0.f, 0.f, 0.f};
    if (work && a.mask) {
      bool none = true;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        mc[c] = mring[bsel * 256 + 64 * c + lane];
        none &= mc[c] == kNegInf || 16 * t + 4 * j + c >= row.vis;
      }
      if (__all(none) && q_tame && below<BF, TILEB>(kt, lane, kTameBits) && below<BF, TILEB>(vt, lane, kInfBits))
        work = false;
    }
    if (__builtin_amdgcn_readfirstlane(work)) {
      // fragments ahead of their MFMAs: left to itself the compiler reads each
      // piece just before the 4 MFMAs it feeds and waits out the LDS latency
      // every time
      const int sw = CH >= 16 ? col : (col >> 1) & 7;
      constexpr int KH = D < 256 ? UK : UK / 2;  // pieces at a time, by registers
      f32x4 s4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) s4[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < UK / KH; ++h) {
        typename T::Piece kf[KH];
#pragma unroll
        for (int u = 0; u < KH; ++u)
          kf[u] = *(const typename T::Piece *)(kt + col * ROWB + 16 * ((4 * (h * KH + u) + j) ^ sw));
        if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < KH; ++u)
#pragma unroll
          for (int e = 0; e < T::EPC; ++e)
            s4[e & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(T::el(kf[u], e), qr[(h * KH + u) * T::EPC + e],
                                                             s4[e & 3], 0, 0, 0);
      }
      typename T::Four vf[4][D / 64];
      auto read_v = [&](int c) {
#pragma unroll
        for (int u = 0; u < D / 64; ++u)
          vf[c][u] = *(const typename T::Four *)(vt + (4 * j + c) * ROWB + (64 * u + 4 * col) * T::ES);
      };
      if constexpr (PRE) {
        read_v(0), read_v(1);
        if constexpr (D < 256) read_v(2), read_v(3);
        __builtin_amdgcn_sched_barrier(0);
      }
      const f32x4 dot = (s4[0] + s4[1]) + (s4[2] + s4[3]);
      float p[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float s = dot[c] * a.scale;
        if (a.mask) s += mc[c];
        p[c] = 16 * t + 4 * j + c < row.vis ? s : kNegInf;
      }
      softmax_step<D>(st, p);
      // a key that some row of the wave must not see (causal starts) may hold
      // anything: a product 0 x NaN or 0 x inf would reach that row, so such a
      // tile's products are formed per row and key
      bool plain = true;
      if (16 * t + 16 > vis_min && vis_min < nkeys) plain = below<BF, TILEB>(vt, lane, kInfBits);
      if (plain) {
        if constexpr (!PRE) read_v(0), read_v(1);
        if constexpr (D == 256) read_v(2), read_v(3);
        if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int u = 0; u < D / 64; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              st.o[u][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(T::four(vf[c][u], e), p[c], st.o[u][e], 0, 0, 0);
      } else {
        for (int kk = 0; kk < 16; ++kk) {
          const float pk = __shfl(kk & 2 ? (kk & 1 ? p[3] : p[2]) : (kk & 1 ? p[1] : p[0]), (kk >> 2) * 16 + col);
          if (16 * t + kk < row.vis) {
#pragma unroll
            for (int u = 0; u < D / 64; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const typename T::Four x =
                    *(const typename T::Four *)(vt + kk * ROWB + (64 * u + 16 * j + 4 * i) * T::ES);
#pragma unroll
                for (int e = 0; e < 4; ++e) st.o[u][e][i] += pk * T::four(x, e);
              }
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the last tile
  st.l = sum4(st.l);
  if constexpr (KG > 1) {
    __syncthreads();  // the ring is free
    float *rec = (float *)tile_lds;
    if (kg > 0) st.save(rec + (((kg - 1) * RG + rg) * 16 + col) * (4 + D), j);
    __syncthreads();
    if (kg == 0)
      for (int x = 0; x < KG - 1; ++x) st.merge(rec + ((x * RG + rg) * 16 + col) * (4 + D), j);
  }
  if (kg == 0) by_pieces<D>(st);
  if (a.nsplit == 1) {
    if (kg == 0 && r0 + col < R) store_row<D>(a, st, row.o, j);
    return;
  }
  const int unit = bh * a.tiles + tile;
  float *base = a.part + (int64_t)unit * a.nsplit * (16 * RG) * (4 + D);
  if (kg == 0) {
    const uint32_t at = (uint32_t)(split * 16 * RG + rg * 16 + col) * (4 + D) * 4;
    if (j == 0) store_coherent(base, at, f32x4{st.m, st.l, 0.f, 0.f});
#pragma unroll
    for (int u = 0; u < D / 64; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        store_coherent(base, at + (4 + 64 * u + 16 * i + 4 * j) * 4,
                       f32x4{st.o[u][0][i], st.o[u][1][i], st.o[u][2][i], st.o[u][3][i]});
  }
  if (!last_arrival(a.counters + unit, a.nsplit, &flag)) return;
  const int first = tile * 16 * RG;
  merge_units<D>(a, base, min(16 * RG, R - first), 16 * RG, (float *)tile_lds,
                 [&](int r) { return row_at(a, b, kvh, first + r).o; });
  if (threadIdx.x == 0) __hip_atomic_store(a.counters + unit, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- up to 8 rows per kv head (decode steps) ----------------------------------
// v_mfma_f32_4x4x1_16b_f32: 16 blocks of 4 lanes, each a 4 x 4 outer product,
// so 4 rows fill it where a 16-row tile would leave 12 of 16 rows empty (at
// D = 256 a 16-key tile is 0.4 us of matrix time instead of 1.7), and the
// q and output registers shrink to a quarter, which leaves room for K and V
// in flight. NS sets of 4 rows share every K/V byte. Lane l: block b = l / 4,
// r = l % 4.
//   scores: A = K row 16 t + 4 kq + r, B = q of row r, both at the block's own
//     dims; 4 blocks of keys kq. Each block ends with a partial sum of its
//     dims, [key][row]; a reduce-scatter over the 16 blocks leaves lane 4 k + r
//     with the score of key k, row r.
//   P V: A = p, taken from block k (cbsz / abid broadcast) for key k, B = a
//     16-byte piece of V row k, the row's pieces over LPR lanes; with more
//     lanes than a row has pieces, lane groups take different keys.
// Each of the 8 waves walks its own tiles straight from memory: the next
// tile's K is in flight through the softmax and P V of this one, its V through
// the next scores. Bound: HBM for long caches (8 x 32 / 8 heads, D = 128, f32,
// lengths 2048-4096: 43.5 us, 4.6 TB/s), else the chain of round trips (lengths,
// first tile, merge): 4 x 8 / 2 heads, D = 256, f32, lengths 300-2048: 15.4 us
// against 517 us for one workgroup per query head with scalar loads.
template <int CB, int AB>
__device__ __forceinline__ f32x4 mfma4x4(float x, float y, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(x, y, c, CB, AB, 0);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kRor8 = 0x128, kRor4 = 0x124, kHalfMirror = 0x141, kQuadReverse = 0x1b;

template <int... I, typename F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// x[16] per lane, summed over the 16 blocks: block b returns sum of x[b]
__device__ __forceinline__ float reduce_scatter16(float (&x)[16], int lane) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[i]), __float_as_uint(x[i + 8]), false, false);
    x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]), __float_as_uint(x[i + 4]), false, false);
    x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  const bool b1 = lane & 8, b0 = lane & 4;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float send = b1 ? x[i] : x[i + 2], keep = b1 ? x[i + 2] : x[i];
    x[i] = keep + dpp<kRor8>(send);
  }
  const float send = b0 ? x[0] : x[1], keep = b0 ? x[1] : x[0];
  return keep + dpp<kQuadReverse>(dpp<kHalfMirror>(send));  // lane ^ 4
}
__device__ __forceinline__ float max_blocks(float v) {
  v = max4(v);
  v = fmaxf(v, dpp<kRor8>(v));
  return fmaxf(v, dpp<kRor4>(v));
}
__device__ __forceinline__ float sum_blocks(float v) {
  v = sum4(v);
  v += dpp<kRor8>(v);
  return v + dpp<kRor4>(v);
}

template <int D, bool BF, int NS>
__device__ void gqa_quad(const GqaTileArgs &a) {
  typedef Kv<BF> T;
  constexpr int NW = 8, ES = T::ES, EPC = T::EPC, ROWB = D * ES;
  constexpr int EPK = EPC < D / 16 ? EPC : D / 16, NK = D / (16 * EPK);  // K elements per load, loads per key block
  constexpr int LPR = ROWB / 16, BPG = LPR / 4;                         // lanes per V row, V loads per tile
  constexpr int CB = BPG == 16 ? 4 : BPG == 8 ? 3 : BPG == 4 ? 2 : 1;
  typedef typename std::conditional<EPK == EPC, typename T::Piece, typename T::Four>::type KPiece;
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  __shared__ int flag;
  const int lane = threadIdx.x & 63, blkn = lane >> 2, r = lane & 3;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NBH = a.NB * a.Hkv, G = a.Hq / a.Hkv, R = G * a.Sq;
  const int bh = blockIdx.x % NBH, split = blockIdx.x / NBH;
  const int b = bh / a.Hkv, kvh = bh - b * a.Hkv;
  const int slot = __builtin_amdgcn_readfirstlane(a.slots ? a.slots[b] : b);
  const char *kp = (const char *)a.k + (slot * a.k_sb + kvh * a.k_sh) * ES;
  const char *vp = (const char *)a.v + (slot * a.v_sb + kvh * a.v_sh) * ES;
  const int nkeys = __builtin_amdgcn_readfirstlane(row_vis(a, b, a.Sq - 1)), vis_min = row_vis(a, b, 0);
  // (V rows past the last key read as zeros: weight 0 times what that key holds
  // would be NaN for an infinity)
  const __amdgpu_buffer_rsrc_t v_rsrc = buf_rsrc(vp, (uint32_t)nkeys * ROWB);
  const int ntiles = (nkeys + 15) / 16, per = (ntiles + a.nsplit - 1) / a.nsplit;
  const int t0 = split * per, t1 = min(ntiles, t0 + per);
  KPiece kf[4][NK];
  typename T::Piece vf[BPG];
  auto load_k = [&](int t) {
#pragma unroll
    for (int kq = 0; kq < 4; ++kq) {
      const char *p = kp + (uint32_t)min(16 * t + 4 * kq + r, nkeys - 1) * ROWB + EPK * ES * blkn;
#pragma unroll
      for (int i = 0; i < NK; ++i) kf[kq][i] = *(const KPiece *)(p + 16 * EPK * ES * i);
    }
  };
  const int grp = lane / LPR, vcol = lane % LPR;
  auto load_v = [&](int t) {
#pragma unroll
    for (int x = 0; x < BPG; ++x)
      vf[x] = __builtin_bit_cast(typename T::Piece, __builtin_amdgcn_raw_buffer_load_b128(
                                                        v_rsrc, (uint32_t)(16 * t + grp * BPG + x) * ROWB + 16 * vcol, 0, 0));
  };
  const int tb = t0 + wv;
  if (tb < t1) {
    load_k(tb);
    load_v(tb);
  }
  RowAt row[NS];
  float qr[NS][D / 16];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    row[s] = row_at(a, b, kvh, min(4 * s + r, R - 1));
    if (a.q_bf16) {
      uint2 w[D / 64];
#pragma unroll
      for (int x = 0; x < D / 64; ++x)
        w[x] = *(const uint2 *)((const uint16_t *)a.q + row[s].q + EPK * (blkn + 16 * (4 * x / EPK)) + 4 * x % EPK);
#pragma unroll
      for (int x = 0; x < D / 64; ++x) four_bf16(w[x], qr[s] + 4 * x);
    } else {
#pragma unroll
      for (int x = 0; x < D / 64; ++x) {
        const f32x4 w = *(const f32x4 *)((const float *)a.q + row[s].q + EPK * (blkn + 16 * (4 * x / EPK)) + 4 * x % EPK);
#pragma unroll
        for (int e = 0; e < 4; ++e) qr[s][4 * x + e] = w[e];
      }
    }
  }
  float m[NS], l[NS];
  f32x4 o[NS][EPC];  // component: row 4 s + i; dim EPC * vcol + e, this lane group's keys
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    m[s] = kNegInf, l[s] = 0.f;
#pragma unroll
    for (int e = 0; e < EPC; ++e) o[s][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int t = tb; t < t1; t += NW) {
    const int key = 16 * t + blkn;
    float mk[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) mk[s] = a.mask ? row[s].mask[(int64_t)min(key, a.Sk - 1) * a.msj] : 0.f;
    f32x4 acc[NS][4];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int kq = 0; kq < 4; ++kq) acc[s][kq] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int e = 0; e < EPK; ++e) {
        if constexpr (BF) __builtin_amdgcn_sched_barrier(0);  // widen K and V as they are used, not all ahead
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int kq = 0; kq < 4; ++kq) {
            float kx;
            if constexpr (EPK == EPC) kx = T::el(kf[kq][i], e); else kx = T::four(kf[kq][i], e);
            acc[s][kq] = mfma4x4<0, 0>(kx, qr[s][i * EPK + e], acc[s][kq]);
          }
      }
    const int tn = min(t + NW, t1 - 1);  // (the last tile is read again rather than branched over)
    load_k(tn);
    float p[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float x[16];
#pragma unroll
      for (int y = 0; y < 16; ++y) x[y] = acc[s][y >> 2][y & 3];
      float sc = reduce_scatter16(x, lane) * a.scale;
      if (a.mask) sc += mk[s];
      if (key >= row[s].vis) sc = kNegInf;
      if (__any(sc > m[s] + 8.f)) {  // (see softmax_step)
        const float mn = fmaxf(m[s], max_blocks(sc));
        const float alpha = m[s] == kNegInf ? 0.f : expf(m[s] - mn);
        l[s] *= alpha;
        const f32x4 f = f32x4{dpp<0x00>(alpha), dpp<0x55>(alpha), dpp<0xaa>(alpha), dpp<0xff>(alpha)};
#pragma unroll
        for (int e = 0; e < EPC; ++e) o[s][e] *= f;
        m[s] = mn;
      }
      p[s] = prob(sc, m[s]);
      l[s] += p[s];
    }
    bool plain = true;
    if (16 * t + 16 > vis_min && vis_min < nkeys) {  // keys that some row must not see (see gqa_tile)
      // (on the raw bits: sharing the widened values with the products would
      // keep them all in registers)
      uint32_t hi = 0, lo = 0;
#pragma unroll
      for (int x = 0; x < BPG; ++x) {
        const u32x4 v = __builtin_bit_cast(u32x4, vf[x]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hi = max(hi, v[e] & 0x7fff0000u);
          if constexpr (BF) lo = max(lo, v[e] & 0x7fffu);
        }
      }
      plain = __all(hi < 0x7f800000u && lo < 0x7f80u);
    }
    if (plain) {
      unrolled(std::make_integer_sequence<int, BPG>{}, [&](auto xc) {
        constexpr int X = decltype(xc)::value;
        if constexpr (BF) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < EPC; ++e)
#pragma unroll
          for (int s = 0; s < NS; ++s) o[s][e] = mfma4x4<CB, X>(p[s], T::el(vf[X], e), o[s][e]);
      });
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int vis = __shfl(row[s].vis, i);
#pragma unroll 1
          for (int x = 0; x < BPG; ++x) {
            const float pk = __shfl(p[s], 4 * (grp * BPG + x) + i);
            const int kx = 16 * t + grp * BPG + x;
            if (kx < vis) {
              const typename T::Piece v = *(const typename T::Piece *)(vp + (uint32_t)kx * ROWB + 16 * vcol);
#pragma unroll
              for (int e = 0; e < EPC; ++e) o[s][e][i] += pk * T::el(v, e);
            }
          }
        }
    }
    load_v(tn);
  }
  // lane groups, then waves (through LDS, all threads on the outputs)
  float *ml = (float *)tile_lds, *rec = ml + NW * 8 * NS;  // [wave][row][2], [wave][row][D]
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    l[s] = sum_blocks(l[s]);
    if (lane < 4) ml[(wv * 4 * NS + 4 * s + r) * 2] = m[s], ml[(wv * 4 * NS + 4 * s + r) * 2 + 1] = l[s];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y[EPC];
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        y[e] = o[s][e][i];
        if constexpr (LPR <= 32) y[e] = sum_xor32(y[e]);
        if constexpr (LPR <= 16) y[e] = sum_xor16(y[e]);
        if constexpr (LPR <= 8) y[e] += dpp<kRor8>(y[e]);
      }
      if (lane < LPR)
#pragma unroll
        for (int e = 0; e < EPC; e += 4)
          *(f32x4 *)(rec + (wv * 4 * NS + 4 * s + i) * D + EPC * vcol + e) = f32x4{y[e], y[e + 1], y[e + 2], y[e + 3]};
    }
  }
  __syncthreads();
  float *base = a.part + (int64_t)bh * a.nsplit * R * (4 + D);
  for (int x = threadIdx.x; x < R * (D / 4); x += 64 * NW) {
    const int rr = x / (D / 4), d = 4 * (x - rr * (D / 4));
    float M = kNegInf, L = 0.f;
    f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[(w * 4 * NS + rr) * 2]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = ml[(w * 4 * NS + rr) * 2], f = mw == kNegInf ? 0.f : expf(mw - M);
      L += f * ml[(w * 4 * NS + rr) * 2 + 1];
      y += f * *(const f32x4 *)(rec + (w * 4 * NS + rr) * D + d);
    }
    if (a.nsplit == 1) {
      y *= M == kNegInf ? __builtin_nanf("") : 1.0f / L;
      const int64_t at = row_at(a, b, kvh, rr).o + d;
      if (a.out_bf16)
        *(uint2 *)((uint16_t *)a.out + at) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      else
        *(f32x4 *)((float *)a.out + at) = y;
    } else {
      const uint32_t at = (uint32_t)(split * R + rr) * (4 + D) * 4;
      if (d == 0) store_coherent(base, at, f32x4{M, L, 0.f, 0.f});
      store_coherent(base, at + (4 + d) * 4, y);
    }
  }
  if (a.nsplit == 1) return;
  if (!last_arrival(a.counters + bh, a.nsplit, &flag)) return;
  merge_units<D>(a, base, R, R, ml, [&](int x) { return row_at(a, b, kvh, x).o; });
  if (threadIdx.x == 0) __hip_atomic_store(a.counters + bh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

// (matches the plans of ops.cpp attention_f32_launch)
#define RXW8_GQA_TILE(D, T, BF, NB4, KG2, NB2)                                                           \
  extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))              \
      rxw8_gqa_tile_##T##_d##D##_r4(GqaTileArgs a) {                                                     \
    gqa_tile<D, BF, 4, 1, NB4>(a);                                                                       \
  }                                                                                                      \
  extern "C" __global__ void __launch_bounds__(128 * KG2) __attribute__((amdgpu_waves_per_eu(KG2 / 2)))  \
      rxw8_gqa_tile_##T##_d##D##_r2(GqaTileArgs a) {                                                     \
    gqa_tile<D, BF, 2, KG2, NB2>(a);                                                                     \
  }
RXW8_GQA_TILE(64, f32, false, 3, 4, 3)
RXW8_GQA_TILE(128, f32, false, 3, 4, 2)
RXW8_GQA_TILE(256, f32, false, 2, 2, 2)
RXW8_GQA_TILE(64, bf16, true, 3, 4, 3)
RXW8_GQA_TILE(128, bf16, true, 3, 4, 3)
RXW8_GQA_TILE(256, bf16, true, 3, 4, 2)

#define RXW8_GQA_QUAD(D, T, BF)                                                                          \
  extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))              \
      rxw8_gqa_quad_##T##_d##D##_s1(GqaTileArgs a) {                                                     \
    gqa_quad<D, BF, 1>(a);                                                                               \
  }                                                                                                      \
  extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))              \
      rxw8_gqa_quad_##T##_d##D##_s2(GqaTileArgs a) {                                                     \
    gqa_quad<D, BF, 2>(a);                                                                               \
  }
RXW8_GQA_QUAD(64, f32, false)
RXW8_GQA_QUAD(128, f32, false)
RXW8_GQA_QUAD(256, f32, false)
RXW8_GQA_QUAD(64, bf16, true)
RXW8_GQA_QUAD(128, bf16, true)
RXW8_GQA_QUAD(256, bf16, true)
