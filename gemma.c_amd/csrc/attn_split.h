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
// and one per tile of V (attn_pack_kernel).  K's goes into the softmax's scale,
// V's into the weights: the value sums are kept in units of the largest V tile
// of the workgroup's keys.
//
// Two f16 pieces hold a value's 22 bits only down to 2^-17 of its tile's
// largest, and a weight's down to 2^-8 of its query's largest.  So a workgroup
// first looks at what its tiles hold (TileRange, kept by attn_pack_kernel) and
// computes its queries by AttnBf3, three bf16 pieces and six products at any
// magnitude, unless all of this holds:
//  - K and V are finite.
//  - Every key's largest V, and every dim's in every tile (of kThin keys or
//    more) but for dims of zeros, is within 2^6 of the largest V of all.  A
//    weight's pieces drop at most 2^-31 of the query's largest weight, in units
//    of the largest V (about 2^-26 rms over 4096 keys): 2^-20 of the least such
//    key or dim, of ordinary ones far less.
//  - HD 2^-9 of a raw score's unit, the most that q's and k's pieces drop from a
//    score by ending at 2^-25, is below 2^-19 octaves.
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
#include <math.h>

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
// The bits of |x|, which order as the magnitudes do, what isn't finite above all.
__device__ __forceinline__ int abs_bits(float x) { return __float_as_int(x) & 0x7fffffff; }
constexpr int kInfBits = 0x7f800000;
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
// Max over the 64 lanes of a wave.
__device__ __forceinline__ int wave_max_i32(int v) {
  v = max(v, dpp_i32<kDppXor1>(v));
  v = max(v, dpp_i32<kDppXor2>(v));
  v = max(v, dpp_i32<kDppHalfMirror>(v));
  v = max(v, dpp_i32<kDppMirror>(v));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
// Lane l's result: the largest t[l % 8] of its eight lanes.  Each step hands
// half of a lane's values to a lane that keeps that half.
__device__ __forceinline__ int max_across_8(const int (&t)[8], int lane) {
  int a[4], b[2];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    a[e] = max(lane & 4 ? t[4 + e] : t[e], dpp_i32<kDppHalfMirror>(lane & 4 ? t[e] : t[4 + e]));
#pragma unroll
  for (int e = 0; e < 2; ++e)
    b[e] = max(lane & 2 ? a[2 + e] : a[e], dpp_i32<kDppXor2>(lane & 2 ? a[e] : a[2 + e]));
  return max(lane & 1 ? b[1] : b[0], dpp_i32<kDppXor1>(lane & 1 ? b[0] : b[1]));
}
// E such that amax 2^-E lies in [2^14, 2^15), f16's upper range; for 0 one that
// is below any other's.
__device__ __forceinline__ int scale_exp(float amax) {
  return amax > 0.0f ? ilogbf(amax) - 14 : -200;
}
// ... rounded up to a multiple of 4, which most V tiles of ordinary layers
// share; 0 for 0.
__device__ __forceinline__ int scale_exp4(float amax) {
  return amax > 0.0f ? (scale_exp(amax) + 3 + 1024) / 4 * 4 - 1024 : 0;
}

// What a packed tile holds, for the choice between the two forms.
struct TileRange {
  int ek, ev;   // exponents of K and V; ek INT_MAX: K is not finite
  float vtop;   // V's largest magnitude; infinite: V is not finite
  float vlow;   // f16 pieces keep this tile's V beside others of up to this magnitude
};
constexpr float kVReach = 0x1p6f;  // how far V's keys and dims may lie apart
// Tiles of fewer keys don't speak for their dims: by chance alone one of a few
// values lies far below the rest (ordinary rows of one key: one dim in 70).
constexpr int kThin = 8;

// Two workgroups per (32-key tile, kv head), K and V: rows 32 t .. 32 t + 31
// (rows from `keys` on are zero) with their biases, scaled and split into the
// tile's fragments.  Memory-bound: reads and writes 4 bytes a value once.
struct AttnPack {
  const float *k, *v;            // row r of head h at r * stride + h * hstride
  size_t stride, hstride;
  const float *bk, *bv;          // biases [heads][HD], or null
  int tile0, ntiles, keys;
  char *planes;                  // [head][ntiles] tiles, tile0 first
  TileRange *range;              // [head][ntiles]
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
  __shared__ int red[NT / 64];             // K's largest magnitude, as bits
  __shared__ int keytop[32], dimtop[HD];  // V's, of each key and dim
  const int tid = threadIdx.x, h = blockIdx.y;
  const bool isv = blockIdx.z != 0;
  if (isv) {
    if (tid < 32) keytop[tid] = 0;
    for (int i = tid; i < HD; i += NT) dimtop[i] = 0;
    __syncthreads();
  }
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
  int top = 0;
  if (!isv) {
#pragma unroll
    for (int j = 0; j < PT; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) top = max(top, abs_bits(x[j][e]));
    top = wave_max_i32(top);
    if ((tid & 63) == 0) red[tid >> 6] = top;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) top = max(top, red[w]);
  } else {
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int i = min(tid + j * NT, N - 1), d = i % HD, q = i / HD, s = q >> 1, half = q & 1;
      int t[8], most = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) most = max(most, t[e] = abs_bits(x[j][e]));
      // eight lanes hold eight dims of the same keys (HD % 8 == 0)
      const int e = tid % 8;
      atomicMax(&keytop[8 * (2 * s + e / 4) + 4 * half + e % 4], max_across_8(t, tid));
      atomicMax(&dimtop[d], most);
    }
    __syncthreads();
    top = wave_max_i32(keytop[tid % 32]);
  }
  const bool finite = top < kInfBits;  // if not, the pieces are of no use
  const float amax = finite ? __int_as_float(top) : 0.0f;
  const int ex = isv ? scale_exp4(amax) : scale_exp(amax);
  const size_t at = (size_t)h * a.ntiles + blockIdx.x;
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
  if (tid >= 64) return;
  TileRange *r = a.range + at;
  if (!isv) {
    if (tid == 0) r->ek = finite ? ex : INT_MAX;
    return;
  }
  const int keys = min(32, a.keys - t0);
  int low = INT_MAX;
  if (tid < keys) low = keytop[tid];
  if (keys >= kThin)
    for (int d = tid; d < HD; d += 64)
      if (dimtop[d] != 0) low = min(low, dimtop[d]);
  low = -wave_max_i32(-low);
  if (tid == 0) {
    r->ev = ex;
    r->vtop = finite ? amax : INFINITY;
    r->vlow = __int_as_float(low) * kVReach;
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

// ... and each lane's 16 bytes from an address of its own.
__device__ __forceinline__ void attn_dma_rows(const float *src, const void *lds) {
  const uint32_t m = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)lds;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m), "v"(src)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// What a lane's query sees: keys ws .. p_top; every query of its wave sees keys
// f_lo .. f_hi.
struct AttnSee {
  int ws, p_top, f_lo, f_hi;
};

constexpr float kLog2e = 1.44269502162933349609375f;  // fl(log2 e)
constexpr float kLog2eLo = 1.92596298909109e-8f;      // log2 e - fl(log2 e)
constexpr float kAttnFloor = -0x1p55f;  // the reference before a query has seen a key
constexpr int kAttnTop = 15;          // weights stay below 2^15
constexpr float kAttnVTop = 0x1p100f;  // the value sums stay finite below
constexpr int kAttnSet = 7;           // a moved reference puts the largest at 2^6 .. 2^7

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
  // Moves the running maximum for a tile whose largest score of the lane is
  // top2 (base 2).  Rarely does anything: the maximum has kAttnTop - kAttnSet
  // octaves of slack (settled() says whether it would).
  __device__ __forceinline__ void refer(float top2, bool first) {
    if (settled(top2)) return;
    const float rmax = fmaxf(top2, __shfl_xor(top2, 32, 64));
    const float m_new = fmaxf(m2, ceilf(rmax) - (float)kAttnSet);
    const float alpha = __builtin_amdgcn_exp2f(m2 - m_new);  // a power of two, or 0
    m2 = m_new;
    l *= alpha;
    if (!first) scale_o(alpha);
  }

  __device__ __forceinline__ bool settled(float top2) const {
    return !__any(top2 > m2 + (float)kAttnTop);
  }

  // lds: 2 K tiles, then 2 V tiles; red: a v4f per wave.  c_hi + c_lo: the
  // scores' scale (asc) times log2 e, without the tiles' exponents; cap: the
  // soft cap of the scaled scores (0: none); keys: how many there are.  False,
  // for the whole workgroup and with nothing computed, where the tiles hold
  // what two f16 pieces don't.
  __device__ __forceinline__ bool run(const char *tiles, const TileRange *range, int ta, int tb,
                                      int keys, const AttnSee &see, float asc, float c_hi,
                                      float c_lo, float cap, char *lds, v4f *red, int wave,
                                      int lane) {
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

    auto exps = [&](int t) { return *reinterpret_cast<const int2 *>(&range[t].ek); };
    int2 ex = exps(ta + zero);
    fetch_k(ta);
    fetch_v(ta);
    float vtop = 0.0f, vlow = FLT_MAX, ek = -1e9f;
    for (int t = ta + 64 * wave + lane; t <= tb; t += 64 * NW) {
      const TileRange r = range[t];
      vtop = fmaxf(vtop, r.vtop);
      vlow = fminf(vlow, r.vlow);
      ek = fmaxf(ek, (float)r.ek);
    }
    red[wave] = v4f{wave_max_dpp(vtop), -wave_max_dpp(-vlow), wave_max_dpp(ek), wave_max_dpp(c_hi)};
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's DMAs landed
    lds_barrier();                       // every wave's did
    v4f all = red[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const v4f r = red[w];
      all = v4f{fmaxf(all[0], r[0]), fminf(all[1], r[1]), fmaxf(all[2], r[2]), fmaxf(all[3], r[3])};
    }
    vtop = all[0];
    const bool fit = vtop <= kAttnVTop && all[1] >= vtop && all[2] < 1e6f &&
                     ldexpf(all[3], (int)all[2]) <= 0x1p-10f / HD &&
                     (tb > ta || keys - 32 * ta >= kThin);
    if (!__builtin_amdgcn_readfirstlane((int)fit)) return false;
    e_o = __builtin_amdgcn_readfirstlane(scale_exp4(vtop));  // the largest tile's exponent
    if (ta < tb) fetch_k(ta + 1);
    v16f sc = {};
    {
      const char *k0 = kbuf + (ta & 1) * (G::KFR * 1024) + loff;
      const h8 none[2][2] = {};
      h8 f[kQ][2];
      each_chunk(std::integral_constant<int, (kQ < 4 ? kQ : 4)>{},
                 [&](auto I) { read<I>(k0, nullptr, f[I]); });
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
        ex = exps(t + 1 + zero);
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
        c1 = kLog2e;
        c2 = kLog2eLo;
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
      refer(top2, t == ta);
      do {
        const int df = ev - e_o;  // the tile's units below the sums', for the weights to carry
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
                  ((sum[4] + sum[5]) + (sum[6] + sum[7]))) * ldexpf(1.0f, -df);
          __builtin_amdgcn_sched_barrier(0);
        });
        sc = sn;
        if (++t > tb) break;
        begin(t);
      } while (settled(top2));
      if (t > tb) break;
    }
    l += __shfl_xor(l, 32, 64);
    return true;
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

// The same attention at any magnitude, on the bf16 matrix cores: every fp32
// operand x of the two products (q, k, the weights p and v) as three bf16
// pieces x = x0 + x1 + x2 (split3x2: 24 significant bits, fp32's exponents),
// each product a b from the six piece products whose orders add up to at most
// 2, the small ones first, on v_mfma_f32_16x16x32_bf16 (lane l: A[l%16][8(l/16)
// .. +7], B[8(l/16) .. +7][l%16], D[4(l/16) + r][l%16]) with fp32 accumulation:
// the dropped ones are below 3 * 2^-24 |a b|, and bf16 x bf16 products are
// exact there.  NW waves x 16 queries of one head, 32-key tiles of
// K and V as they stand in memory: a tile's K rows come by LDS DMA into a
// staging buffer while the tile before is in use, and its V rows likewise (VS)
// or at its start; there they get their biases and are split,
// once per workgroup, into planes: K [key][dim] (head dims padded to whole
// 32-dim chunks) and V^T [dim][k], where k = 8 g + 4 b + r is the value
// product's index of key 16 b + 4 g + r, the key whose score lane (query, g)
// holds in element r of block b, so a lane's eight weights are its operand of
// that product as they stand.  Lane (query col, g) ends with dims 16 nb + 4 g
// .. + 3 in o[nb].  A wave skips the tiles that none of its queries sees.
struct AttnRows {
  const float *k, *v;    // row r at r * stride
  size_t stride;
  const float *bk, *bv;  // biases, or null
};
// What a lane's query sees, what each of its wave's 16 sees and what any does.
struct AttnGroup {
  int ws, p_top, f_lo, f_hi, w_lo, w_hi;
};

// VS: V's rows come through the staging buffer too, during the tile before; not
// where the LDS for it would cost the f16 form of the same kernel a workgroup.
// BIAS: K, V and the queries have biases.
template <int HD, int NW, bool BIAS, bool VS>
struct AttnBf3 {
  static constexpr int TK = 32;              // keys per tile
  static constexpr int NT = NW * 64;
  static constexpr int CH = (HD + 31) / 32;  // 32-dim chunks of the score product
  static constexpr int DP = CH * 32;         // padded head dim of the K planes
  // A last chunk of 8 dims (head dim 72) takes two MFMAs instead of six: its
  // k index carries four piece products over the 8 dims, k = 8 g + e for
  // dim 32 CF + e of piece pair g (first MFMA: k2 q0, k1 q1, k0 q2, k1 q0;
  // second: k0 q1, k0 q0 and two zero pairs)
  static constexpr bool kTail8 = HD % 32 == 8;
  static constexpr int CF = kTail8 ? CH - 1 : CH;  // chunks summed piece by piece
  static constexpr int NB = (HD + 15) / 16;  // 16-dim output blocks
  static constexpr int RK = DP + 8;          // K plane row (bf16): 16 rows in distinct banks
  static constexpr int RV = TK + 8;          // V^T plane row (bf16)
  static constexpr int C4 = HD / 4;          // float4 per key row
  static constexpr int SG = TK * C4;         // float4 of a K tile
  static constexpr int VB = 8 * C4;          // V blocks of a tile
  static constexpr int kUnroll = VS ? 4 : 1;
  // planes 16 bytes apart in the banks: the first tail MFMA reads three of
  // them at one offset
  static constexpr int kKPlane = TK * RK + 8, kVPlane = NB * 16 * RV;
  static constexpr size_t kBytes =
      (size_t)(kKPlane + kVPlane) * 6 + (size_t)((VS ? 2 : 1) * SG + 2 * C4) * 16;
  static_assert(HD % 8 == 0 && SG % 64 == 0 && kKPlane % 8 == 0, "head dim");

  v4f o[NB];
  float m, l;  // base-2 reference maximum (a whole number) and weights' sum

  // qrow, see: the lane's query.  vexp: V enters as v 2^-vexp (for
  // values whose pieces bf16 would not hold), and so do the sums.
  __device__ __forceinline__ void run(const AttnRows &rows, int k_lo, int k_end,
                                      const float *qrow, const float *qbias,
                                      const AttnGroup &see, float asc, float cap, int vexp,
                                      char *lds, int wave, int lane) {
    __bf16 *kt = reinterpret_cast<__bf16 *>(lds);
    __bf16 *vt = kt + 3 * kKPlane;
    v4f *stg = reinterpret_cast<v4f *>(vt + 3 * kVPlane);
    v4f *kvb = stg + (VS ? 2 : 1) * SG;  // K's bias, then V's
    const int tid = 64 * wave + lane, col = lane & 15, grp = lane >> 4;

    // the queries' pieces: lane (col, g) holds dims 32 c + 8 g .. + 7
    bf8 qa[3][CH];
    bf8 qt1 = {}, qt2 = {};
    int tsel = 0;  // the K plane lane (col, g) reads in the first tail MFMA
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      u4 w0, w1, w2;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const int d = 32 * c + 8 * grp + e;  // HD is even: d and d + 1 are both in or out
        float x0 = 0.0f, x1 = 0.0f;
        if (HD % 32 == 0 || d < HD) {
          x0 = BIAS ? qrow[d] + qbias[d] : qrow[d];
          x1 = BIAS ? qrow[d + 1] + qbias[d + 1] : qrow[d + 1];
        }
        const Bf3x2 sp = split3x2(x0, x1);
        w0[e / 2] = sp.q0;
        w1[e / 2] = sp.q1;
        w2[e / 2] = sp.q2;
      }
      qa[0][c] = as_bf8(w0);
      qa[1][c] = as_bf8(w1);
      qa[2][c] = as_bf8(w2);
    }
    // the tail chunk's operands: lane (col, 0) holds dims 32 CF .. + 7 of
    // every piece in qa[p][CF]; lane (col, g) takes the piece of pair g
    if constexpr (kTail8) {
      u4 t[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const u4 v = __builtin_bit_cast(u4, qa[p][CF]);
#pragma unroll
        for (int d = 0; d < 4; ++d) t[p][d] = (uint32_t)__shfl((int)v[d], col, 64);
      }
      qt1 = as_bf8(grp == 1 ? t[1] : grp == 2 ? t[2] : t[0]);          // q0 q1 q2 q0
      qt2 = as_bf8(grp == 0 ? t[1] : grp == 1 ? t[0] : u4{0, 0, 0, 0});  // q1 q0 0 0
      tsel = grp == 0 ? 2 : grp == 2 ? 0 : 1;                               // k2 k1 k0 k1
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) o[nb] = v4f{0.f, 0.f, 0.f, 0.f};
    m = kFloor;
    l = 0.0f;
    const float c1 = kLog2e, c2 = kLog2eLo;

    // zero padding: K dims HD .. DP-1 and V^T rows HD .. 16 NB - 1, never staged
    const __bf16 bz = (__bf16)0.0f;
    constexpr int KP = DP - HD > 0 ? DP - HD : 1, VP = 16 * NB - HD > 0 ? 16 * NB - HD : 1;
    for (int i = tid; i < 3 * TK * (DP - HD); i += NT) {
      const int p = i / (TK * KP), j = i % (TK * KP);
      kt[p * kKPlane + (j / KP) * RK + HD + j % KP] = bz;
    }
    for (int i = tid; i < 3 * (16 * NB - HD) * RV; i += NT) {
      const int p = i / (VP * RV), j = i % (VP * RV);
      vt[p * kVPlane + HD * RV + j] = bz;
    }
    if constexpr (BIAS)
      for (int i = tid; i < 2 * C4; i += NT)
        kvb[i] = reinterpret_cast<const v4f *>(i < C4 ? rows.bk : rows.bv)[i % C4];

    auto fetch = [&](int t0) {  // rows past the last repeat it: their weights are 0
      for (int i = wave; i < (VS ? 2 : 1) * SG / 64; i += NW) {  // wave-uniform
        const int ch = (64 * i + lane) % SG, t = ch / C4;
        attn_dma_rows((i < SG / 64 ? rows.k : rows.v) +
                          (size_t)min(t0 + t, k_end) * rows.stride + 4 * (ch - t * C4),
                      stg + 64 * i);
      }
    };
    fetch(k_lo);
    for (int t0 = k_lo; t0 <= k_end; t0 += TK) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's DMAs landed
      lds_barrier();  // every wave's did, and every wave is done with the planes
#pragma unroll kUnroll
      for (int j = 0; j < (SG + NT - 1) / NT; ++j) {
        const int i = tid + j * NT;
        if (i >= SG) break;
        const int t = i / C4, c4 = i - t * C4;
        v4f kv = stg[i];
        if constexpr (BIAS) kv += kvb[c4];
        const Bf3x2 lo = split3x2(kv[0], kv[1]), hi = split3x2(kv[2], kv[3]);
        __bf16 *at = kt + t * RK + 4 * c4;
        *reinterpret_cast<u2 *>(at) = u2{lo.q0, hi.q0};
        *reinterpret_cast<u2 *>(at + kKPlane) = u2{lo.q1, hi.q1};
        *reinterpret_cast<u2 *>(at + 2 * kKPlane) = u2{lo.q2, hi.q2};
      }
      // 4 keys x 4 dims, first by the threads that have the least of K
      for (int b = NT - 1 - tid; b < VB; b += NT) {
        const int tq = b % 8, c4 = b / 8;
        const int k0i = 8 * (tq % 4) + 4 * (tq / 4);  // the value product's k of key 4 tq
        v4f x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if constexpr (VS)
            x[u] = stg[SG + (4 * tq + u) * C4 + c4];
          else
            x[u] = *reinterpret_cast<const v4f *>(
                rows.v + (size_t)min(t0 + 4 * tq + u, k_end) * rows.stride + 4 * c4);
        }
        if constexpr (BIAS)
#pragma unroll
          for (int u = 0; u < 4; ++u) x[u] += kvb[C4 + c4];
        if (vexp != 0)  // workgroup-uniform
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[u][e] = ldexpf(x[u][e], -vexp);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Bf3x2 lo = split3x2(x[0][e], x[1][e]), hi = split3x2(x[2][e], x[3][e]);
          __bf16 *at = vt + (4 * c4 + e) * RV + k0i;
          *reinterpret_cast<u2 *>(at) = u2{lo.q0, hi.q0};
          *reinterpret_cast<u2 *>(at + kVPlane) = u2{lo.q1, hi.q1};
          *reinterpret_cast<u2 *>(at + 2 * kVPlane) = u2{lo.q2, hi.q2};
        }
      }
      lds_barrier();  // the planes are complete; the staging buffer is free
      if (t0 + TK <= k_end) fetch(t0 + TK);

      if (t0 > see.w_hi || t0 + TK - 1 < see.w_lo) continue;  // wave-uniform
      // sc[b][r] = q(col) . k(t0 + 16 b + 4 grp + r)
      v4f sc[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        sc[b] = v4f{0.f, 0.f, 0.f, 0.f};
        if constexpr (kTail8) {
          const __bf16 *at = kt + (16 * b + col) * RK + 32 * CF;
          const bf8 a1 = *reinterpret_cast<const bf8 *>(at + tsel * kKPlane);
          const bf8 a2 = *reinterpret_cast<const bf8 *>(at);
          sc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, qt1, sc[b], 0, 0, 0);
          sc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, qt2, sc[b], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < CF; ++c)
          sc[b] = six(kt + (16 * b + col) * RK + 32 * c + 8 * grp, kKPlane, qa[0][c],
                      qa[1][c], qa[2][c], sc[b]);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        sc[b] *= asc;
        if (cap != 0.0f)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[b][r] = tanhf(sc[b][r] / cap) * cap;
      }
      if (t0 < see.f_lo || t0 + TK - 1 > see.f_hi) {  // wave-uniform: some key masked
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = t0 + 16 * b + 4 * grp + r;
            sc[b][r] = key <= see.p_top && key >= see.ws ? sc[b][r] : -FLT_MAX;
          }
      }
      float top = -FLT_MAX;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) top = fmaxf(top, sc[b][r]);
      const float top2 = top * c1;
      if (__any(top2 > m + kSlack)) {
        float rmax = fmaxf(top2, __shfl_xor(top2, 16, 64));
        rmax = fmaxf(rmax, __shfl_xor(rmax, 32, 64));
        const float m_new = fmaxf(m, ceilf(rmax));
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) o[nb] *= alpha;
      }
      u4 w0, w1, w2;  // weight k = 4 b + r of the lane's eight is dword 2 b + r / 2
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          float p[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float x = sc[b][r + u];
            p[u] = x > -FLT_MAX ? __builtin_amdgcn_exp2f(fmaf(x, c1, fmaf(x, c2, -m))) : 0.0f;
            l += p[u];
          }
          const Bf3x2 sp = split3x2(p[0], p[1]);
          w0[2 * b + r / 2] = sp.q0;
          w1[2 * b + r / 2] = sp.q1;
          w2[2 * b + r / 2] = sp.q2;
        }
      const bf8 p0 = as_bf8(w0), p1 = as_bf8(w1), p2 = as_bf8(w2);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        o[nb] = six(vt + (16 * nb + col) * RV + 8 * grp, kVPlane, p0, p1, p2, o[nb]);
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
  }

 private:
  static constexpr float kSlack = 16.0f;  // weights stay below 2^16
  static constexpr float kFloor = -0x1p100f;  // below any score
  // acc + a b from the planes of a (at, at + plane, at + 2 plane) and b's pieces
  static __device__ __forceinline__ v4f six(const __bf16 *at, int plane, bf8 b0, bf8 b1, bf8 b2,
                                            v4f acc) {
    const bf8 a0 = *reinterpret_cast<const bf8 *>(at);
    const bf8 a1 = *reinterpret_cast<const bf8 *>(at + plane);
    const bf8 a2 = *reinterpret_cast<const bf8 *>(at + 2 * plane);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b2, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b1, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc, 0, 0, 0);
  }
};

// The power of two that AttnBf3 takes out of V, from what run() left in `red`:
// 0 but for values so small that their third pieces would be subnormal.
__device__ __forceinline__ int any_vexp(const v4f *red, int waves) {
  float vtop = 0.0f;
  for (int w = 0; w < waves; ++w) vtop = fmaxf(vtop, red[w][0]);
  return __builtin_amdgcn_readfirstlane(vtop < 0x1p-60f ? -64 : 0);
}

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
