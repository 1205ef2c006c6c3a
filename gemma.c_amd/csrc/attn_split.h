// attn_split.h -- the fp32 modes' attention on the f16 matrix cores, shared
// by the prompt pass (prefill.hip) and the vision tower (vision.hip).
//
// Every fp32 operand x of the two products (q, k, the weights p and v) is
// scaled by a power of two into the upper range of f16 and split into two
// f16 pieces, x = x0 + x1 (each rounded to nearest, x1 from the exact
// remainder: 22 significant bits), and every product a b is summed from a1 b0,
// a0 b1 and a0 b0 on v_mfma_f32_32x32x16_f16 with fp32 accumulation.  f16 x
// f16 products are exact there; what a product leaves out is at most about
// 2^-21 |a b| (2^-23 rms), below the rounding of the fp32 sums it goes into,
// and the sums take half the roundings of three bf16 pieces with six
// products.  Measured against 64-bit sums: see the tests' bars.
//
// Scales are exact powers of two: one per query, one per 32-key tile of K
// and one per tile of V (attn_pack_kernel), so a tile of outliers costs no
// other tile its precision.  K's goes into the softmax's scale, V's into the
// weights (the value sums are kept in units of a running exponent, as the
// weights are relative to a running maximum).
//
// K and V are split once per key and layer by attn_pack_kernel into tiles of
// 32 keys whose pieces lie in the order in which a wave reads its operands:
// fragment f of a tile is 64 lanes x 16 bytes.  A tile so goes from memory to
// LDS by linear DMA and from LDS to the matrix cores by conflict-free
// 16-byte reads, and the attention kernel spends no instruction on splitting
// or transposing.  (Splitting in the attention kernel, once per workgroup
// and tile, took as long as the products: 16 row blocks each split the same
// keys.)
#pragma once

#include <float.h>
#include <limits.h>

#include <type_traits>

#include "gh_arith.h"
#include "gh_kernels.h"

namespace gh {
namespace {

// Fragments of a 32-key tile.  A wave computes S^T = K Q^T (rows: 32 keys,
// columns: 32 queries) and O^T = V^T P^T (rows: 32 dims).  Operand layout of
// the 32x32x16 MFMA: lane l holds row (or column) l % 32 and the eight k
// values 8 (l / 32) .. + 7; result element r of lane l is row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
//   K: fragment 2 s + p: piece p of dims 16 s .. 16 s + 15, lane l: key l % 32
//   V: fragment (2 b + s) 2 + p: piece p of dims 32 b .. + 31 (rows) over the
//      keys of step s, lane l: dim 32 b + l % 32, element e: key
//      8 (2 s + e / 4) + 4 (l / 32) + e % 4 -- the keys whose scores lane l
//      holds in elements 8 s .. 8 s + 7, so its weights are the other operand
//      as they stand
// A head dim 8 above a multiple of 32 (SigLIP's 72) has a tail of 8 dims:
//   K: one fragment, lanes 0-31 piece 0 and lanes 32-63 piece 1 of the 8 dims
//   V: one fragment per step, rows 0-7 piece 0 and rows 8-15 piece 1
template <int HD>
struct AttnTile {
  static constexpr bool kTail = HD % 32 == 8;
  static constexpr int KF = HD / 16;                       // whole 16-dim steps
  static constexpr int NBF = kTail ? HD / 32 : (HD + 31) / 32;  // 32-dim blocks
  static constexpr int NB = NBF + (kTail ? 1 : 0);         // accumulator blocks
  static constexpr int KFR = 2 * KF + (kTail ? 1 : 0);     // K fragments
  static constexpr int VFR = 4 * NBF + (kTail ? 2 : 0);    // V fragments
  static constexpr size_t kBytes = (size_t)(KFR + VFR) * 1024;
  static_assert(HD % 16 == 0 || kTail, "head dim");
};

// The pieces of eight values.
__device__ __forceinline__ void split8(const float (&x)[8], h8 *hi, h8 *lo) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const h2 a = cvt_pk_f16(x[e], x[e + 1]);
    const h2 b = cvt_pk_f16(x[e] - (float)a[0], x[e + 1] - (float)a[1]);
    (*hi)[e] = a[0];
    (*hi)[e + 1] = a[1];
    (*lo)[e] = b[0];
    (*lo)[e + 1] = b[1];
  }
}
// E such that amax 2^-E lies in [2^14, 2^15), f16's upper range; 0 for 0.
__device__ __forceinline__ int scale_exp(float amax) {
  return amax > 0.0f ? ilogbf(amax) - 14 : 0;
}
// ... rounded up to a multiple of 4: the V tiles of ordinary layers then
// share one exponent and the running one rarely moves.
__device__ __forceinline__ int scale_exp4(float amax) {
  return amax > 0.0f ? (scale_exp(amax) + 3 + 1024) / 4 * 4 - 1024 : 0;
}

// Two workgroups per (32-key tile, kv head), K and V: rows 32 t .. 32 t + 31
// (rows from `keys` on are zero) with their biases, scaled and split into the
// tile's fragments.  Memory-bound: reads and writes 4 bytes a value once.
struct AttnPack {
  const float *k, *v;            // row r of head h at r * stride + h * hstride
  size_t stride, hstride;
  const float *bk, *bv;          // biases [heads][HD], or null
  int tile0, ntiles, keys;
  char *planes;                  // [head][ntiles] tiles, tile0 first
  int2 *exps;                    // [head][ntiles] exponents of K and V
};

// Threads of a packing workgroup: one item of eight values each, up to 512.
template <int HD>
constexpr int kPackThreads = HD >= 128 ? 512 : (4 * HD + 63) / 64 * 64;

// z = 0 packs the tile's K, z = 1 its V: twice the workgroups, and each
// thread's loads (rows past the last clamped to it, zeroed afterwards) are all
// in flight at once.
template <int HD>
__global__ __launch_bounds__(kPackThreads<HD>) void attn_pack_kernel(AttnPack a) {
  typedef AttnTile<HD> G;
  constexpr int NT = kPackThreads<HD>;
  constexpr int N = 4 * HD;                // items of the tile: 32 HD / 8
  constexpr int PT = (N + NT - 1) / NT;    // per thread
  __shared__ float red[NT / 64];
  const int tid = threadIdx.x, h = blockIdx.y;
  const bool isv = blockIdx.z != 0;
  const int t0 = (a.tile0 + blockIdx.x) * 32;
  const float *src = (isv ? a.v : a.k) + h * a.hstride;
  const float *bias = isv ? a.bv : a.bk;

  float x[PT][8];
  if (!isv) {  // item: key i % 32, dims 8 (i / 32) .. + 7
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int i = min(tid + j * NT, N - 1), key = t0 + i % 32, d = 8 * (i / 32);
      const float *row = src + (size_t)min(key, a.keys - 1) * a.stride + d;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const v4f t = *reinterpret_cast<const v4f *>(row + e);
        const v4f b = bias != nullptr ? *reinterpret_cast<const v4f *>(bias + h * HD + d + e)
                                      : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u) x[j][e + u] = bias != nullptr ? t[u] + b[u] : t[u];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] = key < a.keys ? x[j][e] : 0.0f;
    }
  } else {  // item: dim i % HD; step s and lane half of i / HD give the keys
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int i = min(tid + j * NT, N - 1), d = i % HD, q = i / HD, s = q >> 1, half = q & 1;
      const float b = bias != nullptr ? bias[h * HD + d] : 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = t0 + 8 * (2 * s + e / 4) + 4 * half + e % 4;
        const float t = src[(size_t)min(key, a.keys - 1) * a.stride + d];
        x[j][e] = key < a.keys ? (bias != nullptr ? t + b : t) : 0.0f;
      }
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, finite_abs(x[j][e]));
  amax = wave_max_dpp(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) amax = fmaxf(amax, red[w]);
  const int ex = isv ? scale_exp4(amax) : scale_exp(amax);
  const size_t at = (size_t)h * a.ntiles + blockIdx.x;
  if (tid == 0) reinterpret_cast<int *>(a.exps + at)[isv ? 1 : 0] = ex;
  char *kf = a.planes + at * G::kBytes, *vf = kf + G::KFR * 1024;
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int i = tid + j * NT;
    if (i >= N) break;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[j][e] = ldexpf(x[j][e], -ex);
    h8 hi, lo;
    split8(x[j], &hi, &lo);
    char *f;
    int next;  // from a fragment's piece 0 to its piece 1
    if (!isv) {
      const int key = i % 32, g = i / 32;  // dims 8 g .. + 7
      const bool tail = G::kTail && g == 2 * G::KF;
      f = kf + (tail ? 2 * G::KF * 1024 + key * 16 : (g >> 1) * 2048 + (32 * (g & 1) + key) * 16);
      next = tail ? 512 : 1024;
    } else {
      const int d = i % HD, q = i / HD, s = q >> 1, half = q & 1, b = d / 32, r = d % 32;
      const bool tail = G::kTail && b == G::NBF;
      f = vf + (tail ? 4 * G::NBF + s : (2 * b + s) * 2) * 1024 + (32 * half + r) * 16;
      next = tail ? 128 : 1024;
    }
    *reinterpret_cast<h8 *>(f) = hi;
    *reinterpret_cast<h8 *>(f + next) = lo;
  }
  // rows of V's fragments that no dim fills
  const h8 zero = {};
  if (isv && G::kTail && tid < 2 * 32) {
    const int s = tid / 32, half = (tid / 16) % 2, r = 16 + tid % 16;
    *reinterpret_cast<h8 *>(vf + (4 * G::NBF + s) * 1024 + (32 * half + r) * 16) = zero;
  }
  if (isv && HD < 32)
    for (int i = tid; i < 4 * 32; i += NT) {
      const int f = i / 32, half = (i / 16) % 2, r = 16 + i % 16;
      *reinterpret_cast<h8 *>(vf + f * 1024 + (32 * half + r) * 16) = zero;
    }
}

// One LDS DMA load: lane l's 16 bytes at base + 16 l land at lds + 16 l (base
// and lds wave-uniform).  From inline asm so that the compiler does not wait
// for the pending load before later LDS reads; the kernel waits itself.  m0
// has no other user in the kernels that call this.
__device__ __forceinline__ void attn_dma(const char *base, uint32_t off, const void *lds) {
  const uint32_t m = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)lds;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m), "v"(off),
               "s"(base)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// What a lane's query sees: keys ws .. p_top; every query of its wave sees keys
// f_lo .. f_hi.
struct AttnSee {
  int ws, p_top, f_lo, f_hi;
};

constexpr float kAttnFloor = -0x1p55f;  // the reference before a query has seen a key
constexpr int kAttnTop = 15;          // weights stay below 2^15
constexpr int kAttnSet = 7;           // a moved reference puts the largest at 2^6 .. 2^7
constexpr int kAttnReach = 64;        // octaves between tiles of V that one query's sums can hold

// The attention of one wave's 32 queries over tiles ta .. tb (packed tiles of
// its kv head; the workgroup's waves share them through LDS).  On return
// o[b][r] holds the value sums in units of 2^e_o, relative to the reference
// 2^m2 (a whole number), and l the weights' sum over the keys that this lane
// holds.
// Tiles are double-buffered, one barrier each; the next tile's scores are
// computed in the same stretch as this tile's weights, so that the vector
// unit works while the matrix cores do.
template <int HD, int NW, bool CAP = false>
struct AttnWave {
  typedef AttnTile<HD> G;
  h8 q[G::KF][2];
  h8 qt1, qt2;
  v16f o[G::NB];
  float m2, l;
  int e_o;

  // x: the query's dims in operand order, scaled; its exponent comes back
  __device__ __forceinline__ int load_q(const float *row, const float *bias, int half) {
    float x[G::KF + 1][8];
    float amax = 0.0f;
#pragma unroll
    for (int s = 0; s < G::KF + (G::kTail ? 1 : 0); ++s) {
      const int d = s < G::KF ? 16 * s + 8 * half : 16 * s;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        v4f t = *reinterpret_cast<const v4f *>(row + d + e);
        if (bias != nullptr) t += *reinterpret_cast<const v4f *>(bias + d + e);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          x[s][e + u] = t[u];
          amax = fmaxf(amax, finite_abs(t[u]));
        }
      }
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    const int eq = scale_exp(amax);
#pragma unroll
    for (int s = 0; s < G::KF + (G::kTail ? 1 : 0); ++s) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[s][e] = ldexpf(x[s][e], -eq);
      h8 hi, lo;
      split8(x[s], &hi, &lo);
      if (s < G::KF) {
        q[s][0] = hi;
        q[s][1] = lo;
      } else {  // against (k0 | k1): k0 q1 + k1 q0, then k0 q0
        const h8 zero = {};
        qt1 = half ? hi : lo;
        qt2 = half ? zero : hi;
      }
    }
    return eq;
  }

  // The products of a tile as chunks of up to three, in order: the score
  // products of K (kQ chunks), then the value products of V's two key steps
  // (kV chunks each).  A chunk reads one or two fragments.
  static constexpr int kQ = G::KF + (G::kTail ? 1 : 0), kV = G::NB, kChunks = kQ + 2 * kV;
  static constexpr int kAhead = 2;  // chunks whose fragments are read ahead

  // The fragments of chunk I: K at kf (tile t + 1), V at vf (tile t), both
  // with the lane's offset.
  template <int I>
  static __device__ __forceinline__ void read(const char *kf, const char *vf, h8 (&f)[2]) {
    if constexpr (I < kQ) {
      f[0] = *reinterpret_cast<const h8 *>(kf + (2 * I) * 1024);
      if constexpr (I < G::KF) f[1] = *reinterpret_cast<const h8 *>(kf + (2 * I + 1) * 1024);
    } else {
      constexpr int s = (I - kQ) / kV, b = (I - kQ) % kV;
      constexpr int at = b < G::NBF ? (2 * b + s) * 2 : 4 * G::NBF + s;
      f[0] = *reinterpret_cast<const h8 *>(vf + at * 1024);
      if constexpr (b < G::NBF) f[1] = *reinterpret_cast<const h8 *>(vf + (at + 1) * 1024);
    }
  }
  template <int I>
  __device__ __forceinline__ void product(const h8 (&f)[2], const h8 (&p)[2][2], v16f &s) {
    auto mma = [](h8 a, h8 b, v16f c) {
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    };
    if constexpr (I < G::KF) {
      s = mma(f[1], q[I][0], s);
      s = mma(f[0], q[I][1], s);
      s = mma(f[0], q[I][0], s);
    } else if constexpr (I < kQ) {
      s = mma(f[0], qt1, s);
      s = mma(f[0], qt2, s);
    } else {
      constexpr int st = (I - kQ) / kV, b = (I - kQ) % kV;
      if constexpr (b < G::NBF) o[b] = mma(f[1], p[st][0], o[b]);
      o[b] = mma(f[0], p[st][1], o[b]);
      o[b] = mma(f[0], p[st][0], o[b]);
    }
  }
  // Softmax weights 2 j and 2 j + 1 of the lane's 16 (2^(x (c1 + c2) - m)),
  // their sum and their pieces.
  static __device__ __forceinline__ void weights(int j, const v16f &x, float c1, float c2, float m,
                                                 float (&sum)[8], h8 (&p)[2][2]) {
    const float a = __builtin_amdgcn_exp2f(fmaf(x[2 * j], c1, fmaf(x[2 * j], c2, -m)));
    const float b = __builtin_amdgcn_exp2f(fmaf(x[2 * j + 1], c1, fmaf(x[2 * j + 1], c2, -m)));
    sum[j] = a + b;
    const h2 hi = cvt_pk_f16(a, b);
    const h2 lo = cvt_pk_f16(a - (float)hi[0], b - (float)hi[1]);
    const int s = j / 4, e = 2 * (j % 4);
    p[s][0][e] = hi[0];
    p[s][0][e + 1] = hi[1];
    p[s][1][e] = lo[0];
    p[s][1][e + 1] = lo[1];
  }
  template <int I = 0, int N, class F>
  static __device__ __forceinline__ void each_chunk(std::integral_constant<int, N> n, F &&f) {
    if constexpr (I < N) {
      f(std::integral_constant<int, I>{});
      each_chunk<I + 1>(n, f);
    }
  }

  __device__ __forceinline__ void scale_o(float f) {
#pragma unroll
    for (int b = 0; b < G::NB; ++b) o[b] *= f;
  }
  // Moves the running maximum and exponent for a tile whose largest score of
  // the lane is top2 (base 2) and whose V has exponent ev.  Rarely does
  // anything: the maximum has kAttnTop - kAttnSet octaves of slack, V's
  // exponent goes up at once and down with slack (settled() says whether it
  // would).  Returns how far the tile's
  // units lie below the sums' (<= 0), for the weights to carry.  A tile more
  // than kAttnReach octaves below the sums is out of their reach: it only adds
  // its weights to l, here (with the returned -1000 they vanish elsewhere).
  __device__ __forceinline__ int refer(const v16f &x, float c1, float c2, float top2, int ev,
                                       bool first) {
    if (__any(top2 > m2 + (float)kAttnTop)) {
      const float rmax = fmaxf(top2, __shfl_xor(top2, 32, 64));
      const float m_new = fmaxf(m2, ceilf(rmax) - (float)kAttnSet);
      const float alpha = __builtin_amdgcn_exp2f(m2 - m_new);  // a power of two, or 0
      m2 = m_new;
      l *= alpha;
      if (!first) scale_o(alpha);
    }
    int df = ev - e_o;
    if (df > 0 || df < -8) {  // wave-uniform
      if (df >= -kAttnReach) {
        if (!first) scale_o(ldexpf(1.0f, max(-df, -300)));
        e_o = ev;
        df = 0;
      } else {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          s += __builtin_amdgcn_exp2f(fmaf(x[r], c1, fmaf(x[r], c2, -m2)));
        l += s;
        df = -1000;
      }
    }
    return df;
  }

  __device__ __forceinline__ bool settled(float top2, int df) const {
    return !__any(top2 > m2 + (float)kAttnTop) && df <= 0 && df >= -8;
  }

  // lds: 2 K tiles, then 2 V tiles.  c_hi + c_lo: the scores' scale (asc)
  // times log2 e, without the tiles' exponents; cap: the soft cap of the
  // scaled scores (0: none).
  __device__ __forceinline__ void run(const char *tiles, const int2 *exps, int ta, int tb,
                                      const AttnSee &see, float asc, float c_hi, float c_lo,
                                      float cap, char *lds, int wave, int lane) {
    const int half = lane >> 5;
    char *kbuf = lds, *vbuf = lds + 2 * G::KFR * 1024;
    const uint32_t loff = lane * 16;
    auto fetch = [&](const char *src, char *dst, auto count) {
      constexpr int N = decltype(count)::value;
#pragma unroll
      for (int i = 0; i < (N + NW - 1) / NW; ++i) {
        const int f = i * NW + wave;  // wave-uniform
        if (N % NW == 0 || f < N) attn_dma(src + f * 1024, loff, dst + f * 1024);
      }
    };
    auto fetch_k = [&](int t) {
      fetch(tiles + (size_t)t * G::kBytes, kbuf + (t & 1) * (G::KFR * 1024),
            std::integral_constant<int, G::KFR>{});
    };
    auto fetch_v = [&](int t) {
      fetch(tiles + (size_t)t * G::kBytes + G::KFR * 1024, vbuf + (t & 1) * (G::VFR * 1024),
            std::integral_constant<int, G::VFR>{});
    };
    // tile exponents are loaded a tile ahead into vector registers, so that
    // the wait for the tile's DMAs covers them
    int zero;
    asm("v_mov_b32 %0, 0" : "=v"(zero));

#pragma unroll
    for (int b = 0; b < G::NB; ++b) o[b] = v16f{};
    m2 = kAttnFloor;
    l = 0.0f;
    e_o = -(1 << 20);  // below every exponent: the first tile sets it

    int2 ex = exps[ta + zero];
    fetch_k(ta);
    fetch_v(ta);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's DMAs landed
    lds_barrier();                       // every wave's did
    if (ta < tb) fetch_k(ta + 1);
    v16f sc = {};
    {
      const char *k0 = kbuf + (ta & 1) * (G::KFR * 1024) + loff;
      const h8 none[2][2] = {};
      h8 f[kQ][2];
      each_chunk(std::integral_constant<int, (kQ < 4 ? kQ : 4)>{}, [&](auto I) { read<I>(k0, nullptr, f[I]); });
      __builtin_amdgcn_sched_barrier(0);
      each_chunk(std::integral_constant<int, kQ>{}, [&](auto I) {
        if constexpr (I + 4 < kQ) read<I + 4>(k0, nullptr, f[I + 4]);
        product<I>(f[I], none, sc);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    // The tile loop is turned so that what rarely happens (refer) lies outside
    // the inner loop: in it the value sums are touched by the matrix cores
    // alone and stay in the accumulation registers.
    h8 pre[kAhead][2];  // the first chunks' fragments
    float c1, c2, top2;
    int ev;
    auto begin = [&](int t) {
      __builtin_amdgcn_s_waitcnt(0x0F70);
      // K of tile t + 1 and V of tile t are in; every wave is done with K of
      // tile t and V of tile t - 1
      lds_barrier();
      const char *kn = kbuf + ((t + 1) & 1) * (G::KFR * 1024) + loff;
      const char *vt = vbuf + (t & 1) * (G::VFR * 1024) + loff;
      each_chunk(std::integral_constant<int, kAhead>{}, [&](auto I) { read<I>(kn, vt, pre[I]); });
      __builtin_amdgcn_sched_barrier(0);
      const int ek = __builtin_amdgcn_readfirstlane(ex.x);
      ev = __builtin_amdgcn_readfirstlane(ex.y);
      if (t < tb) {
        ex = exps[t + 1 + zero];
        fetch_v(t + 1);
        if (t + 1 < tb) fetch_k(t + 2);
      }
      // a scale below 2^-70 changes no score by 2^-32 (the raw ones are below
      // 2^38) and would let the masked ones come up
      c1 = fmaxf(ldexpf(c_hi, ek), 0x1p-70f);
      c2 = ldexpf(c_lo, ek);
      if constexpr (CAP) {  // capped scores, in units of the scaled score
        const float as = ldexpf(asc, ek);
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = tanhf(sc[r] * as / cap) * cap;
        c1 = 1.44269502162933349609375f;  // fl(log2 e)
        c2 = 1.92596298909109e-8f;        // log2 e - fl(log2 e)
      }
      if (32 * t < see.f_lo || 32 * t + 31 > see.f_hi) {  // wave-uniform: some key masked
        // a score whose weight is 0: -2^118 once scaled, or -2^57 and below
        const float off = ldexpf(-1.0f, min(118 - ilogbf(c1), 127));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = 32 * t + 8 * (r >> 2) + 4 * half + (r & 3);
          sc[r] = key <= see.p_top && key >= see.ws ? sc[r] : off;
        }
      }
      float top = sc[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) top = fmaxf(top, sc[r]);
      top2 = top * c1;
    };
    int t = ta;
    begin(t);
    for (;;) {
      int df = refer(sc, c1, c2, top2, ev, t == ta);
      do {
        const float m = m2 - (float)df;
        const char *kn = kbuf + ((t + 1) & 1) * (G::KFR * 1024) + loff;
        const char *vt = vbuf + (t & 1) * (G::VFR * 1024) + loff;
        // the chunks, each with the reads of a later one and a share of the
        // weights: all eight pairs before the second key step, the first four
        // before the first.  (Past the last tile the scores are of no use.)
        h8 f[kChunks][2];
        float sum[8];
        h8 p[2][2];
        v16f sn = {};
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          f[i][0] = pre[i][0];
          f[i][1] = pre[i][1];
        }
        each_chunk(std::integral_constant<int, kChunks>{}, [&](auto I) {
          constexpr int n = kQ + kV;  // chunks that take weights
          if constexpr (I + kAhead < kChunks) read<I + kAhead>(kn, vt, f[I + kAhead]);
          product<I>(f[I], p, sn);
          if constexpr (I < n)
#pragma unroll
            for (int j = 8 * I / n; j < 8 * (I + 1) / n; ++j) weights(j, sc, c1, c2, m, sum, p);
          if constexpr (I == n)
            l += (((sum[0] + sum[1]) + (sum[2] + sum[3])) +
                  ((sum[4] + sum[5]) + (sum[6] + sum[7]))) * ldexpf(1.0f, df < -8 ? 0 : -df);
          __builtin_amdgcn_sched_barrier(0);
        });
        sc = sn;
        if (++t > tb) break;
        begin(t);
        df = ev - e_o;
      } while (settled(top2, df));
      if (t > tb) break;
    }
    l += __shfl_xor(l, 32, 64);
  }

  // The value sums of dims 32 b + 8 j + 4 (lane / 32) .. + 3, in units of 2^e_o
  // (j < dims / 8 of the block).
  __device__ __forceinline__ v4f dims(int b, int j) const {
    v4f t;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      t[i] = G::kTail && b == G::NBF ? o[b][i] + o[b][4 + i] : o[b][4 * j + i];
    return t;
  }
  // calls f(first dim, value sums) for every group of four dims that the lane holds
  template <class F>
  __device__ __forceinline__ void each(int half, F &&f) const {
#pragma unroll
    for (int b = 0; b < G::NB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (32 * b + 8 * j < HD) f(32 * b + 8 * j + 4 * half, dims(b, j));
  }
};

__device__ __forceinline__ v4f ldexp4(v4f x, int e) {
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = ldexpf(x[i], e);
  return x;
}

// c_hi + c_lo = scale * log2 e, times 2^e.
__device__ __forceinline__ void log2_scale(float scale, int e, float *c_hi, float *c_lo) {
  const double c = (double)scale * 1.4426950408889634074;
  const float hi = (float)c;
  *c_hi = ldexpf(hi, e);
  *c_lo = ldexpf((float)(c - (double)hi), e);
}

}  // namespace
}  // namespace gh
