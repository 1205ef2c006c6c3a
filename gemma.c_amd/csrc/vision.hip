// vision.hip -- the SigLIP vision tower of forward_vision (gemma.c:4394-4725)
// on the GPU: patch embedding, position embedding, the encoder layers
// (layer norm, q/k/v with biases, full attention over the patches, o, layer
// norm, fc1 with bias and GELU, fc2), the post layer norm, average pooling
// down to the image tokens, the soft-embedding RMSNorm and the projection
// into the text model's width.  The int8 projections are the library's
// GEMMs (gemm_i8.hip, bit-exact); these kernels are the fp32 glue between
// them, evaluated as the decode step's glue is (decode.hip): in fp64 from
// the reference's formulas, rounded to fp32 once where the reference stores
// an fp32 tensor, with single fp32 additions (biases, residuals, the
// dequantized position embedding) kept as the single fp32 operations they
// are.
#include <type_traits>

#include <cstdlib>
#include <cstring>

#include "attn_split.h"
#include "dec_common.h"

namespace gh {
namespace {

// One workgroup per row.  With y: x[r] = clamp((y[r] + bias) + x[r]) (the
// output bias and the residual, gemma.c:4575-4590, 4641-4656), stored back
// as the new residual.  Then LayerNorm (layernorm, gemma.c:2526-2549) in
// fp64: mean, variance about it, (x - mean) / sqrt(var + eps) * w + b,
// rounded once; the row is quantized into xq[r] / xs[r] (quantize_acts)
// when xq is given, else stored to h[r].
template <int NPT, int NT>
__global__ __launch_bounds__(NT) void vis_ln_rows_kernel(VisLn a) {
  __shared__ double red[NT / 64];
  __shared__ float redf[NT / 64];
  const int tid = threadIdx.x, n4 = a.dim >> 2;
  const size_t r = blockIdx.x;
  float *xr = a.x + r * a.dim;
  v4f xv[NPT];
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * NT;
    xv[j] = c < n4 ? reinterpret_cast<const v4f *>(xr)[c] : zero;
    if (a.y != nullptr && c < n4) {
      const v4f yv = reinterpret_cast<const v4f *>(a.y + r * a.dim)[c];
      const v4f bv = reinterpret_cast<const v4f *>(a.bias)[c];
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[j][e] = clamp_f32((yv[e] + bv[e]) + xv[j][e]);
      reinterpret_cast<v4f *>(xr)[c] = xv[j];
    }
  }
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < NPT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) s += (double)xv[j][e];
  const double mean = block_sum<NT>(s, red) / (double)a.dim;
  double ss = 0.0;
#pragma unroll
  for (int j = 0; j < NPT; ++j)
    if (tid + j * NT < n4)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double d = (double)xv[j][e] - mean;
        ss += d * d;
      }
  const double inv = 1.0 / sqrt(block_sum<NT>(ss, red) / (double)a.dim + (double)a.eps);
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * NT;
    if (c >= n4) {
      xv[j] = zero;
      continue;
    }
    const v4f wv = reinterpret_cast<const v4f *>(a.w)[c];
    const v4f bv = reinterpret_cast<const v4f *>(a.b)[c];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xv[j][e] = (float)(((double)xv[j][e] - mean) * inv * (double)wv[e] + (double)bv[e]);
      amax = fmaxf(amax, abs_daz(xv[j][e]));
    }
  }
  if (a.xq == nullptr) {
#pragma unroll
    for (int j = 0; j < NPT; ++j)
      if (tid + j * NT < n4) reinterpret_cast<v4f *>(a.h + r * a.dim)[tid + j * NT] = xv[j];
    return;
  }
  amax = block_max<NT>(amax, redf);
  const QuantParams qp = quant_params(amax);
  int8_t *row = a.xq + r * a.dim;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * NT;
    if (c < n4)
      reinterpret_cast<uint32_t *>(row)[c] =
          pack4(quant_one(xv[j].x, qp.inv), quant_one(xv[j].y, qp.inv),
                quant_one(xv[j].z, qp.inv), quant_one(xv[j].w, qp.inv));
  }
  if (tid == 0) a.xs[r] = qp.scale;
}

// Full (non-causal) attention of every patch over every patch, per head
// (gemma.c:4533-4561): q, k and v are the GEMM outputs plus their biases
// (single fp32 additions, 4517-4526), scores q.k * scale with scale =
// 1 / sqrtf(hdim) in fp32, softmax over all patches, value sums -- on the
// fp64 matrix cores.  v_mfma_f64_16x16x4f64 takes A[16][4] as lane l ->
// A[l%16][l/16], B[4][16] as lane l -> B[l/16][l%16], and leaves D[16][16]
// as lane l, element r -> D[4r + l/16][l%16] (checked on this GPU).
//
// The products are taken transposed, S^T = K . Q^T and O^T = V^T . P^T, so
// that a lane (query j = l%16, g = l/16) holds the scores of query j for the
// keys 4r + g of a 16-key block, which are exactly the P^T operand the value
// product wants: the probabilities never leave registers.  A workgroup is
// 4 waves x 16 queries of one head; the queries stay in registers as fp64
// operands (lane g holds dims [g HD/4, (g+1) HD/4) of its query).  Per tile of
// 32 keys: K and V (biases added, fp32) are staged in LDS -- V transposed,
// its keys permuted so that the 4 a lane needs for one MFMA step are
// adjacent -- then two 16-key score blocks, the softmax weights, and P . V
// into the fp64 output block O^T[16 NB][16].  K and V are held in LDS as
// fp64, converted once when staged.
//
// Softmax: p = exp(s - m) with m a running reference maximum per query.
// Shifting by any m gives the same softmax; m is moved up (to the exact row
// maximum seen so far, rescaling O and the sums by exp(m_old - m_new)) only
// when some score of the wave exceeds it by more than kVaSlack, which keeps
// every p <= e^kVaSlack and lets most tiles skip the row reductions.  The
// row sums are per-lane partials, added across the 4 lanes of a query at
// the end.  Every sum is fp64; each output is rounded to fp32 once.
constexpr int kVaKeys = 32;          // keys per tile
constexpr int kVaWaves = 8;          // waves (16 queries each) per workgroup
constexpr int kVbWaves = 16;         // ... of the three-bf16 kernel (head dims <= 72)
constexpr double kVaSlack = 64.0;    // e^64 * 3.4e38 * n keys stays far below DBL_MAX

template <int HD, int NW>
__global__ __launch_bounds__(NW * 64, 8 / NW) void vis_attn_kernel(VisAttn a) {
  constexpr int NT = NW * 64, QB = NW * 16;  // threads, queries per workgroup
  static_assert(HD % 8 == 0 && HD <= 128, "head dim");
  constexpr int KS = HD / 4;            // MFMA steps of a score block (dims per lane)
  constexpr int NB = (HD + 15) / 16;    // 16-dim output blocks
  constexpr int RK = HD + 2;            // K row in LDS (doubles)
  constexpr int VS = kVaKeys + 2;       // V^T row in LDS (doubles)
  constexpr int C4 = HD / 4;            // float4 per key row
  constexpr int PF = (kVaKeys * C4 + NT - 1) / NT;  // float4 of K (and of V) per thread
  __shared__ double kt[kVaKeys * RK];
  __shared__ double vt[16 * NB * VS];
  __shared__ double etab[128];
  __shared__ v4f kvb[2][C4];  // the k and v biases of this head
  typedef double v2d __attribute__((ext_vector_type(2)));
  typedef double v4d __attribute__((ext_vector_type(4)));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // blocks of one head share K and V: give each XCD (blocks b, b+8, ...) a
  // contiguous run of (head, query block) pairs so they meet in its L2
  const int nqb = (a.n + QB - 1) / QB, nblk = nqb * a.n_heads;
  int blk = blockIdx.x;
  if (nblk % 8 == 0) blk = (blk % 8) * (nblk / 8) + blk / 8;
  const int h = blk / nqb;
  const int q0 = (blk - h * nqb) * QB + wave * 16;
  const int col = lane & 15, grp = lane >> 4;

  double qa[KS];
  {
    const int qr = min(q0 + col, a.n - 1);
    const float *qrow = a.qkv + (size_t)qr * a.stride + h * HD + grp * KS;
    const float *bq = a.bias + h * HD + grp * KS;
#pragma unroll
    for (int s = 0; s < KS; ++s) qa[s] = (double)(qrow[s] + bq[s]);
  }
  v4d o[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) o[nb] = v4d{0.0, 0.0, 0.0, 0.0};
  double m_ref = -DBL_MAX, l_part = 0.0;
  const double scale = (double)a.scale;
  const float *bk = a.bias + a.dim + h * HD;
  const float *bv = a.bias + 2 * a.dim + h * HD;
  const float *kbase = a.qkv + a.dim + h * HD;
  const float *vbase = a.qkv + 2 * a.dim + h * HD;

  // padding dims of V^T (never overwritten by the staging below)
  for (int i = HD * VS + tid; i < 16 * NB * VS; i += NT) vt[i] = 0.0;
  exp_tab_load(etab);
  for (int i = tid; i < 2 * C4; i += NT)
    kvb[i / C4][i % C4] = reinterpret_cast<const v4f *>(i < C4 ? bk : bv)[i % C4];
  const ExpConsts ec = exp_consts();

  v4f kx[PF], vx[PF];
  auto fetch = [&](int t0) {  // rows clamped into range: every load is unconditional
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int i = min(tid + j * NT, kVaKeys * C4 - 1);
      const int t = i / C4, c4 = i - t * C4;
      const size_t row = (size_t)min(t0 + t, a.n - 1) * a.stride;
      kx[j] = *reinterpret_cast<const v4f *>(kbase + row + 4 * c4);
      vx[j] = *reinterpret_cast<const v4f *>(vbase + row + 4 * c4);
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < a.n; t0 += kVaKeys) {
    lds_barrier();  // every wave is done with the previous tile
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int i = tid + j * NT;
      if (i >= kVaKeys * C4) break;
      const int t = i / C4, c4 = i - t * C4;
      const bool ok = t0 + t < a.n;
      const v4f zero = {0.f, 0.f, 0.f, 0.f};
      const v4f kv = ok ? kx[j] + kvb[0][c4] : zero;
      const v4f vv = ok ? vx[j] + kvb[1][c4] : zero;
      *reinterpret_cast<v2d *>(&kt[t * RK + 4 * c4]) = v2d{(double)kv[0], (double)kv[1]};
      *reinterpret_cast<v2d *>(&kt[t * RK + 4 * c4 + 2]) = v2d{(double)kv[2], (double)kv[3]};
      const int tp = (t & 16) | ((t & 3) << 2) | ((t >> 2) & 3);  // key 16b+4s+g -> 16b+4g+s
#pragma unroll
      for (int e = 0; e < 4; ++e) vt[(4 * c4 + e) * VS + tp] = (double)vv[e];
    }
    lds_barrier();
    if (t0 + kVaKeys < a.n) fetch(t0 + kVaKeys);

    // scores: sc[b][r] = q(col) . k(t0 + 16 b + 4 r + grp)
    v4d sc[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      sc[b] = v4d{0.0, 0.0, 0.0, 0.0};
      const double *kr = &kt[(16 * b + col) * RK + grp * KS];
#pragma unroll
      for (int s = 0; s < KS; s += 2) {
        const v2d k2 = *reinterpret_cast<const v2d *>(kr + s);
        sc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(k2[0], qa[s], sc[b], 0, 0, 0);
        sc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(k2[1], qa[s + 1], sc[b], 0, 0, 0);
      }
    }
    double tmax = -DBL_MAX;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = t0 + 16 * b + 4 * r + grp < a.n;
        sc[b][r] = ok ? sc[b][r] * scale : -DBL_MAX;
        tmax = fmax(tmax, sc[b][r]);
      }
    if (__any(tmax > m_ref + kVaSlack)) {
      double rmax = fmax(tmax, __shfl_xor(tmax, 16, 64));
      rmax = fmax(rmax, __shfl_xor(rmax, 32, 64));
      const double m_new = fmax(m_ref, rmax);
      const double alpha = exp_tab(m_ref - m_new, etab, ec);
      m_ref = m_new;
      l_part *= alpha;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) o[nb] *= alpha;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // a masked key (-DBL_MAX) lands on exp_tab's clamp and gives 0
        const double pr = exp_tab(sc[b][r] - m_ref, etab, ec);
        l_part += pr;
        sc[b][r] = pr;
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const double *vr = &vt[(16 * nb + col) * VS + 16 * b + 4 * grp];
        const v2d v01 = *reinterpret_cast<const v2d *>(vr);
        const v2d v23 = *reinterpret_cast<const v2d *>(vr + 2);
        o[nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(v01[0], sc[b][0], o[nb], 0, 0, 0);
        o[nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(v01[1], sc[b][1], o[nb], 0, 0, 0);
        o[nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(v23[0], sc[b][2], o[nb], 0, 0, 0);
        o[nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(v23[1], sc[b][3], o[nb], 0, 0, 0);
      }
    }
  }
  double l = l_part + __shfl_xor(l_part, 16, 64);
  l = l + __shfl_xor(l, 32, 64);
  const int qr = q0 + col;
  if (qr < a.n) {
    float *orow = a.out + (size_t)qr * a.dim + h * HD;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * nb + 4 * r + grp;
        if (d < HD) orow[d] = (float)(o[nb][r] / l);
      }
  }
}

// The same attention on the fp32 matrix cores (v_mfma_f32_16x16x4f32, twice
// the fp64 rate): q, k, v, scores, weights and value sums in fp32, as the
// reference computes them (gemm_fpx, softmax, gemm_fpx_nn), in a different
// order, so the result agrees with the fp64 form to fp32 rounding rather
// than bit for bit.  The fp32 MFMA takes A and B as the fp64 one does but
// leaves D as lane l, element r -> D[4 (l/16) + r][l%16] (checked on this
// GPU), so a lane (query col, g = l/16) holds the scores of keys 4g + r of a
// 16-key block, and the value product's MFMA step r takes keys 4g + r from
// lane group g: V^T stays in natural key order and a lane reads its four
// keys as one float4.  The reference maximum moves when a score exceeds it
// by more than 16 (e^16 * n keys * |v| stays far below FLT_MAX).  The
// exponential is __expf (v_exp_f32 on x log2 e: a relative error near
// |x| 2^-24 for the arguments here, |x| <= 16 past the masked keys), and two
// workgroups share a CU (113 registers at head dim 72): 880 -> 785 us per
// SigLIP layer against expf at one workgroup per CU.
constexpr float kVaSlackF = 16.0f;
constexpr int kVaKeysF = 32;  // keys per tile (fp32 kernel; 64 measured 2% slower)

template <int HD, int NW, int TK>
__global__ __launch_bounds__(NW * 64, 16 / NW) void vis_attn_f32_kernel(VisAttn a) {
  constexpr int NS = TK / 16;         // 16-key score blocks per tile
  constexpr int NT = NW * 64, QB = NW * 16;
  static_assert(HD % 8 == 0 && HD <= 128, "head dim");
  constexpr int KS = HD / 4;          // MFMA steps of a score block (dims per lane)
  constexpr int NB = (HD + 15) / 16;  // 16-dim output blocks
  constexpr int RK = HD + 2;          // K row in LDS (floats)
  constexpr int VS = TK + 4;     // V^T row in LDS (floats)
  constexpr int C4 = HD / 4;
  constexpr int PF = (TK * C4 + NT - 1) / NT;
  __shared__ float kt[TK * RK];
  __shared__ float vt[16 * NB * VS];
  __shared__ v4f kvb[2][C4];
  typedef float v2f __attribute__((ext_vector_type(2)));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nqb = (a.n + QB - 1) / QB, nblk = nqb * a.n_heads;
  int blk = blockIdx.x;
  if (nblk % 8 == 0) blk = (blk % 8) * (nblk / 8) + blk / 8;
  const int h = blk / nqb;
  const int q0 = (blk - h * nqb) * QB + wave * 16;
  const int col = lane & 15, grp = lane >> 4;

  float qa[KS];
  {
    const int qr = min(q0 + col, a.n - 1);
    const float *qrow = a.qkv + (size_t)qr * a.stride + h * HD + grp * KS;
    const float *bq = a.bias + h * HD + grp * KS;
#pragma unroll
    for (int s = 0; s < KS; ++s) qa[s] = qrow[s] + bq[s];
  }
  v4f o[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) o[nb] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_ref = -FLT_MAX, l_part = 0.0f;
  const float *bk = a.bias + a.dim + h * HD;
  const float *bv = a.bias + 2 * a.dim + h * HD;
  const float *kbase = a.qkv + a.dim + h * HD;
  const float *vbase = a.qkv + 2 * a.dim + h * HD;

  for (int i = HD * VS + tid; i < 16 * NB * VS; i += NT) vt[i] = 0.0f;  // padding dims
  for (int i = tid; i < 2 * C4; i += NT)
    kvb[i / C4][i % C4] = reinterpret_cast<const v4f *>(i < C4 ? bk : bv)[i % C4];

  // K: float4 i of the tile is key i / C4, dims 4 (i % C4) .. +3.  V goes
  // to LDS transposed in blocks of 4 keys x 4 dims: block b = (tq, c4) =
  // (b % 8, b / 8) holds keys 4 tq .. 4 tq + 3 of dims 4 c4 .. 4 c4 + 3 and
  // is written as 4 float4 of V^T; eight consecutive lanes differ in tq, so
  // with the row pitch VS = TK + 4 their 16-byte writes fall in eight
  // different bank groups (scattering single floats instead put a
  // half-wave's writes on two banks).
  static_assert(TK % 4 == 0 && TK / 4 == 8, "V blocks: 8 key quads per tile");
  constexpr int VB = 8 * C4;               // V blocks per tile
  constexpr int PV = (VB + NT - 1) / NT;   // V blocks per thread
  v4f kx[PF], vx[PV][4];
  auto fetch = [&](int t0) {  // rows clamped into range: every load is unconditional
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int i = min(tid + j * NT, TK * C4 - 1);
      const int t = i / C4, c4 = i - t * C4;
      kx[j] = *reinterpret_cast<const v4f *>(kbase + (size_t)min(t0 + t, a.n - 1) * a.stride +
                                             4 * c4);
    }
#pragma unroll
    for (int j = 0; j < PV; ++j) {
      const int b = min(tid + j * NT, VB - 1);
      const int tq = b % 8, c4 = b / 8;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        vx[j][u] = *reinterpret_cast<const v4f *>(
            vbase + (size_t)min(t0 + 4 * tq + u, a.n - 1) * a.stride + 4 * c4);
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < a.n; t0 += TK) {
    lds_barrier();  // every wave is done with the previous tile
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int i = tid + j * NT;
      if (i >= TK * C4) break;
      const int t = i / C4, c4 = i - t * C4;
      const v4f kv = t0 + t < a.n ? kx[j] + kvb[0][c4] : zero;
      *reinterpret_cast<v2f *>(&kt[t * RK + 4 * c4]) = v2f{kv[0], kv[1]};
      *reinterpret_cast<v2f *>(&kt[t * RK + 4 * c4 + 2]) = v2f{kv[2], kv[3]};
    }
#pragma unroll
    for (int j = 0; j < PV; ++j) {
      const int b = tid + j * NT;
      if (b >= VB) break;
      const int tq = b % 8, c4 = b / 8;
      v4f r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) r[u] = t0 + 4 * tq + u < a.n ? vx[j][u] + kvb[1][c4] : zero;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<v4f *>(&vt[(4 * c4 + e) * VS + 4 * tq]) =
            v4f{r[0][e], r[1][e], r[2][e], r[3][e]};
    }
    lds_barrier();
    if (t0 + TK < a.n) fetch(t0 + TK);

    // scores: sc[b][r] = q(col) . k(t0 + 16 b + 4 grp + r)
    v4f sc[NS];
#pragma unroll
    for (int b = 0; b < NS; ++b) {
      sc[b] = v4f{0.f, 0.f, 0.f, 0.f};
      const float *kr = &kt[(16 * b + col) * RK + grp * KS];
#pragma unroll
      for (int s = 0; s < KS; s += 2) {
        const v2f k2 = *reinterpret_cast<const v2f *>(kr + s);
        sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(k2[0], qa[s], sc[b], 0, 0, 0);
        sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(k2[1], qa[s + 1], sc[b], 0, 0, 0);
      }
    }
    float tmax = -FLT_MAX;
#pragma unroll
    for (int b = 0; b < NS; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = t0 + 16 * b + 4 * grp + r < a.n;
        sc[b][r] = ok ? sc[b][r] * a.scale : -FLT_MAX;
        tmax = fmaxf(tmax, sc[b][r]);
      }
    if (__any(tmax > m_ref + kVaSlackF)) {
      float rmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      rmax = fmaxf(rmax, __shfl_xor(rmax, 32, 64));
      const float m_new = fmaxf(m_ref, rmax);
      const float alpha = __expf(m_ref - m_new);
      m_ref = m_new;
      l_part *= alpha;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) o[nb] *= alpha;
    }
#pragma unroll
    for (int b = 0; b < NS; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pr = sc[b][r] > -FLT_MAX ? __expf(sc[b][r] - m_ref) : 0.0f;
        l_part += pr;
        sc[b][r] = pr;
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const v4f v4 = *reinterpret_cast<const v4f *>(&vt[(16 * nb + col) * VS + 16 * b + 4 * grp]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          o[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v4[r], sc[b][r], o[nb], 0, 0, 0);
      }
    }
  }
  float l = l_part + __shfl_xor(l_part, 16, 64);
  l = l + __shfl_xor(l, 32, 64);
  const int qr = q0 + col;
  if (qr < a.n) {
    float *orow = a.out + (size_t)qr * a.dim + h * HD;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * nb + 4 * grp + r;
        if (d < HD) orow[d] = o[nb][r] / l;
      }
  }
}

// One workgroup per row: (float)gelu_tanh(h + b1) (gemma.c:4600-4604 with
// gelu 4150-4172: the bias added in fp32, the GELU in fp64 rounded once),
// quantized into xq[r] / xs[r].
template <int NPT, int NT>
__global__ __launch_bounds__(NT) void vis_gelu_quant_kernel(const float *hbuf, const float *bias,
                                                            int mlp, int8_t *xq, float *xs,
                                                            WarmRegions warm) {
  __shared__ float redf[NT / 64];
  __shared__ double etab[128];
  exp_tab_load(etab);
  const GeluConsts gc = gelu_consts();
  const int tid = threadIdx.x, n4 = mlp >> 2;
  const float *row = hbuf + (size_t)blockIdx.x * mlp;
  v4f hv[NPT], bv[NPT];
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * NT;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    hv[j] = c < n4 ? reinterpret_cast<const v4f *>(row)[c] : zero;
    bv[j] = c < n4 ? reinterpret_cast<const v4f *>(bias)[c] : zero;
  }
  lds_barrier();  // the exp table
  v4f out[NPT];
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NPT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      out[j][e] = (float)gelu(hv[j][e] + bv[j][e], etab, gc);
      amax = fmaxf(amax, abs_daz(out[j][e]));
    }
  amax = block_max<NT>(amax, redf);
  const QuantParams qp = quant_params(amax);
  int8_t *dst = xq + (size_t)blockIdx.x * mlp;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * NT;
    if (c < n4)
      reinterpret_cast<uint32_t *>(dst)[c] =
          pack4(quant_one(out[j].x, qp.inv), quant_one(out[j].y, qp.inv),
                quant_one(out[j].z, qp.inv), quant_one(out[j].w, qp.inv));
  }
  if (tid == 0) xs[blockIdx.x] = qp.scale;
  warm_share(warm, blockIdx.x, gridDim.x, tid, NT);
}

// One workgroup per image token: the mean of its ksize x ksize patches
// (AvgPool2d, gemma.c:4673-4694) in fp64 rounded once, the soft-embedding
// RMSNorm (4698-4704) and the row quantized for the projection.
template <int NPT>
__global__ __launch_bounds__(kNT) void vis_pool_kernel(VisPool a) {
  __shared__ double red[kWaves];
  __shared__ float redf[kWaves];
  const int tid = threadIdx.x, n4 = a.dim >> 2;
  const int side = a.ppi / a.ksize;
  const int oy = blockIdx.x / side, ox = blockIdx.x % side;
  v4f pv[NPT];
  double ss = 0.0;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * kNT;
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    if (c < n4)
      for (int ky = 0; ky < a.ksize; ++ky)
        for (int kx = 0; kx < a.ksize; ++kx) {
          const int p = (oy * a.ksize + ky) * a.ppi + ox * a.ksize + kx;
          const v4f x = reinterpret_cast<const v4f *>(a.h + (size_t)p * a.dim)[c];
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] += (double)x[e];
        }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pv[j][e] = (float)(sum[e] / (double)(a.ksize * a.ksize));
      ss += (double)pv[j][e] * (double)pv[j][e];
    }
  }
  const double rms = rms_of(block_sum<kNT>(ss, red), a.dim, a.eps);
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * kNT;
    if (c >= n4) continue;
    const v4f wv = reinterpret_cast<const v4f *>(a.w)[c];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pv[j][e] = norm_one(pv[j][e], rms, wv[e]);
      amax = fmaxf(amax, abs_daz(pv[j][e]));
    }
  }
  if (a.xq == nullptr) {  // fp32 rows for an fp32 projection
#pragma unroll
    for (int j = 0; j < NPT; ++j) {
      const int c = tid + j * kNT;
      if (c < n4) reinterpret_cast<v4f *>(a.out + (size_t)blockIdx.x * a.dim)[c] = pv[j];
    }
    return;
  }
  amax = block_max<kNT>(amax, redf);
  const QuantParams qp = quant_params(amax);
  int8_t *row = a.xq + (size_t)blockIdx.x * a.dim;
#pragma unroll
  for (int j = 0; j < NPT; ++j) {
    const int c = tid + j * kNT;
    if (c < n4)
      reinterpret_cast<uint32_t *>(row)[c] =
          pack4(quant_one(pv[j].x, qp.inv), quant_one(pv[j].y, qp.inv),
                quant_one(pv[j].z, qp.inv), quant_one(pv[j].w, qp.inv));
  }
  if (tid == 0) a.xs[blockIdx.x] = qp.scale;
}

// h = gelu(h + bias) in place, grid (ceil(mlp / 4 / kNT), rows): the fp32
// tower's fc1 epilogue (gemma.c:4620-4622), each value as the quantizing
// kernel computes it.
__global__ __launch_bounds__(kNT) void vis_bias_gelu_kernel(float *h, const float *bias, int mlp) {
  __shared__ double etab[128];
  exp_tab_load(etab);
  const GeluConsts gc = gelu_consts();
  const int c = blockIdx.x * kNT + threadIdx.x;
  float *row = h + (size_t)blockIdx.y * mlp;
  const bool ok = c < mlp / 4;
  v4f hv = {0.f, 0.f, 0.f, 0.f}, bv = hv;
  if (ok) {
    hv = reinterpret_cast<const v4f *>(row)[c];
    bv = reinterpret_cast<const v4f *>(bias)[c];
  }
  lds_barrier();  // the exp table
  if (!ok) return;
  v4f out;
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = (float)gelu(hv[e] + bv[e], etab, gc);
  reinterpret_cast<v4f *>(row)[c] = out;
}

template <int C, int CMAX, class F>
hipError_t by_npt(int npt, F &&launch) {
  if (npt == C) return launch(std::integral_constant<int, C>{});
  if constexpr (C < CMAX) return by_npt<C + 1, CMAX>(npt, launch);
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_vis_ln_rows(const VisLn &a, int n, hipStream_t stream) {
  // the fewest threads per row that cover it in kPfMaxNpt chunks: more rows
  // in flight per CU (SigLIP's 1152 columns: one wave, 5 chunks)
  const int n4 = a.dim / 4;
  auto go = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    return by_npt<1, kPfMaxNpt>((n4 + NT - 1) / NT, [&](auto c) {
      vis_ln_rows_kernel<decltype(c)::value, NT><<<n, NT, 0, stream>>>(a);
      return hipGetLastError();
    });
  };
  if ((n4 + 63) / 64 <= kPfMaxNpt) return go(std::integral_constant<int, 64>{});
  if ((n4 + 127) / 128 <= kPfMaxNpt) return go(std::integral_constant<int, 128>{});
  return go(std::integral_constant<int, 256>{});
}

// 16 queries of one head from q0 on by AttnBf3: K, V and the queries with their
// biases, every key for every query.
template <int HD, int NW, bool VS>
__device__ __forceinline__ void vis_attn_any(const VisAttn &a, int h, int q0, int vexp, char *lds,
                                             int wave, int lane) {
  const int qr = q0 + (lane & 15), grp = lane >> 4;
  const float *qrow = a.qkv + (size_t)min(qr, a.n - 1) * a.stride + h * HD;
  const float *k = a.qkv + a.dim + h * HD, *bk = a.bias + a.dim + h * HD;
  const AttnRows rows{k, k + a.dim, (size_t)a.stride, bk, bk + a.dim};
  typedef AttnBf3<HD, NW, true, VS> Any;
  Any w;
  w.run(rows, 0, a.n - 1, qrow, a.bias + h * HD,
        AttnGroup{0, a.n - 1, 0, a.n - 1, 0, a.n - 1}, a.scale, 0.0f, vexp, lds, wave, lane);
  if (qr >= a.n) return;
  float *orow = a.out + (size_t)qr * a.dim + h * HD + 4 * grp;
#pragma unroll
  for (int nb = 0; nb < Any::NB; ++nb)
    if (16 * nb + 4 * grp < HD)
      *reinterpret_cast<v4f *>(orow + 16 * nb) = ldexp4(w.o[nb] / w.l, vexp);
}

// The fp32 mode's attention without a workspace, by AttnBf3 alone: calls under
// stream capture, which can't allocate one.
template <int HD, int NW>
__global__ __launch_bounds__(NW * 64, 16 / NW) void vis_attn_bf3_kernel(VisAttn a) {
  __shared__ __attribute__((aligned(16))) char lds[AttnBf3<HD, NW, true, true>::kBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nqb = (a.n + NW * 16 - 1) / (NW * 16), nblk = nqb * a.n_heads;
  int blk = blockIdx.x;
  if (nblk % 8 == 0) blk = (blk % 8) * (nblk / 8) + blk / 8;
  const int h = blk / nqb;
  vis_attn_any<HD, NW, true>(a, h, (blk - h * nqb) * NW * 16 + wave * 16, 0, lds, wave, lane);
}

// The fp32 mode's attention on the f16 matrix cores in split precision
// (attn_split.h): NW waves x 32 queries of one head over tiles that
// attn_pack_kernel made of K and V with their biases.  Bound by the matrix
// cores at the clock that the chip holds under them: SigLIP at 896 px (4096
// patches, 16 heads of 72) takes 30 products per 32 queries and tile, 258
// GFLOP of f16 in 215-235 us (1.1-1.2 PFLOP/s; v_mfma_f32_32x32x16_f16 on random
// registers alone sustains 1.6), packing 17.8 us.  Three bf16 pieces take 430
// by themselves (vis_attn_bf3_kernel) at the same matrix rate with twice the
// products, and their error against 64-bit sums is larger: 9.6e-7 relative, here
// 7.0e-7 (fewer fp32 roundings per sum).  Where the tiles need them all the
// same, the layer takes 710 us (V's tiles 2^24 apart).  The tower's image (9 of
// 27 layers): 6.73 -> 4.7 ms.
template <int HD, int NW>
__global__ __launch_bounds__(NW * 64, 2) void vis_attn_split_kernel(VisAttn a, const char *planes,
                                                                   const TileRange *range,
                                                                   int ntiles) {
  typedef AttnTile<HD> G;
  constexpr bool kVs = HD <= 72;
  typedef AttnBf3<HD, NW, true, kVs> Any;
  constexpr int QB = NW * 32;
  __shared__ __attribute__((aligned(16))) char
      lds[2 * G::kBytes > Any::kBytes ? 2 * G::kBytes : Any::kBytes];
  __shared__ v4f red[NW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  // each XCD's workgroups share one head's tiles in its L2
  const int nqb = (a.n + QB - 1) / QB, nblk = nqb * a.n_heads;
  int blk = blockIdx.x;
  if (nblk % 8 == 0) blk = (blk % 8) * (nblk / 8) + blk / 8;
  const int h = blk / nqb;
  const int q0 = (blk - h * nqb) * QB + wave * 32, qr = q0 + (lane & 31);
  AttnWave<HD, NW> w;
  const int eq = w.load_q(a.qkv + (size_t)min(qr, a.n - 1) * a.stride + h * HD, a.bias + h * HD,
                          half);
  float c_hi, c_lo;
  log2_scale(a.scale, eq, &c_hi, &c_lo);
  const AttnSee see{0, a.n - 1, 0, a.n - 1};
  if (!w.run(planes + (size_t)h * ntiles * G::kBytes, range + (size_t)h * ntiles, 0, ntiles - 1,
             a.n, see, 0.0f, c_hi, c_lo, 0.0f, lds, red, wave, lane)) {
    const int vexp = any_vexp(red, NW);
#pragma unroll 1
    for (int g = 0; g < 32; g += 16)
      vis_attn_any<HD, NW, kVs>(a, h, q0 + g, vexp, lds, wave, lane);
    return;
  }
  if (qr >= a.n) return;
  float *orow = a.out + (size_t)qr * a.dim + h * HD;
  const float f = 1.0f / w.l;
  w.each(half, [&](int d, v4f x) { *reinterpret_cast<v4f *>(orow + d) = ldexp4(x * f, w.e_o); });
}

template <int HD>
void launch_vis_split(const VisAttn &a, char *planes, const DeviceInfo &dev, hipStream_t stream) {
  const int ntiles = (a.n + 31) / 32;
  TileRange *range =
      reinterpret_cast<TileRange *>(planes + (size_t)a.n_heads * ntiles * AttnTile<HD>::kBytes);
  const AttnPack pk{a.qkv + a.dim, a.qkv + 2 * a.dim, (size_t)a.stride, (size_t)HD,
                    a.bias + a.dim, a.bias + 2 * a.dim, 0, ntiles, a.n, planes, range};
  attn_pack_kernel<HD><<<dim3(ntiles, a.n_heads, 2), kPackThreads<HD>, 0, stream>>>(pk);
  // 128 queries a workgroup while those have a CU each (784 patches, 16 heads:
  // 39 us against 50 with 256; 2401 patches, 12 heads: 77 against 103), else
  // 256, which share each tile's way to LDS (4096 patches: 243 against 250)
  const int few = (a.n + 127) / 128 * a.n_heads;
  if (few <= dev.cus)
    vis_attn_split_kernel<HD, 4><<<few, 256, 0, stream>>>(a, planes, range, ntiles);
  else
    vis_attn_split_kernel<HD, 8><<<(a.n + 255) / 256 * a.n_heads, 512, 0, stream>>>(a, planes,
                                                                                   range, ntiles);
}

// The fp32 mode's kernel: a split one by default (f16 pieces with a workspace,
// bf16 pieces without), the fp32-MFMA one with GEMMA_HIP_VIS_ATTN=f32.  Read at
// every launch (one getenv per layer), so that one process can time or check both.
bool vis_attn_split() {
  const char *e = getenv("GEMMA_HIP_VIS_ATTN");
  return e == nullptr || strcmp(e, "f32") != 0;
}

size_t attn_planes_bytes(int hdim, int heads, int keys) {
  const size_t tiles = (size_t)heads * ((keys + 31) / 32);
  size_t tile = 0;
  switch (hdim) {
    case 16: tile = AttnTile<16>::kBytes; break;
    case 32: tile = AttnTile<32>::kBytes; break;
    case 64: tile = AttnTile<64>::kBytes; break;
    case 72: tile = AttnTile<72>::kBytes; break;
    case 128: tile = AttnTile<128>::kBytes; break;
    case 256: tile = AttnTile<256>::kBytes; break;
  }
  return tiles * (tile + sizeof(TileRange));
}

hipError_t launch_vis_attention(const VisAttn &a, int hdim, bool f32, char *planes,
                                const DeviceInfo &dev, hipStream_t stream) {
  constexpr int NW = kVaWaves;
  const dim3 grid((a.n + NW * 16 - 1) / (NW * 16) * a.n_heads);
  if (f32 && planes != nullptr && vis_attn_split()) {
    switch (hdim) {
      case 16: launch_vis_split<16>(a, planes, dev, stream); break;
      case 32: launch_vis_split<32>(a, planes, dev, stream); break;
      case 64: launch_vis_split<64>(a, planes, dev, stream); break;
      case 72: launch_vis_split<72>(a, planes, dev, stream); break;
      case 128: launch_vis_split<128>(a, planes, dev, stream); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  if (f32 && vis_attn_split()) {
    // 16-wave workgroups (256 queries share each staged and split tile):
    // SigLIP 896 px 19.24-19.39 -> 17.86-17.95 ms per image against 8 waves
    // (4 waves: 25.5); head dim 128 keeps 8, its registers exceed the 128 of
    // four waves per SIMD
    constexpr int W = kVbWaves;
    const dim3 gw((a.n + W * 16 - 1) / (W * 16) * a.n_heads);
    switch (hdim) {
      case 16: vis_attn_bf3_kernel<16, W><<<gw, W * 64, 0, stream>>>(a); break;
      case 32: vis_attn_bf3_kernel<32, W><<<gw, W * 64, 0, stream>>>(a); break;
      case 64: vis_attn_bf3_kernel<64, W><<<gw, W * 64, 0, stream>>>(a); break;
      case 72: vis_attn_bf3_kernel<72, W><<<gw, W * 64, 0, stream>>>(a); break;
      case 128: vis_attn_bf3_kernel<128, NW><<<grid, NW * 64, 0, stream>>>(a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  if (f32) {
    switch (hdim) {
      case 16: vis_attn_f32_kernel<16, NW, kVaKeysF><<<grid, NW * 64, 0, stream>>>(a); break;
      case 32: vis_attn_f32_kernel<32, NW, kVaKeysF><<<grid, NW * 64, 0, stream>>>(a); break;
      case 64: vis_attn_f32_kernel<64, NW, kVaKeysF><<<grid, NW * 64, 0, stream>>>(a); break;
      case 72: vis_attn_f32_kernel<72, NW, kVaKeysF><<<grid, NW * 64, 0, stream>>>(a); break;
      case 128: vis_attn_f32_kernel<128, NW, kVaKeysF><<<grid, NW * 64, 0, stream>>>(a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  switch (hdim) {
    case 16: vis_attn_kernel<16, NW><<<grid, NW * 64, 0, stream>>>(a); break;
    case 32: vis_attn_kernel<32, NW><<<grid, NW * 64, 0, stream>>>(a); break;
    case 64: vis_attn_kernel<64, NW><<<grid, NW * 64, 0, stream>>>(a); break;
    case 72: vis_attn_kernel<72, NW><<<grid, NW * 64, 0, stream>>>(a); break;
    case 128: vis_attn_kernel<128, NW><<<grid, NW * 64, 0, stream>>>(a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_vis_gelu_quant(const float *h, const float *bias, int n, int mlp, int8_t *xq,
                                 float *xs, const WarmRegions &warm, hipStream_t stream) {
  // the fewest threads per row that cover it in kPfMaxNpt chunks: at SigLIP's
  // 4304 columns, 256 threads leave 16% of the slots empty, 1024 threads 47%
  // (54.7 -> 36.7 us per layer measured)
  const int n4 = mlp / 4;
  auto go = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    return by_npt<1, kPfMaxNpt>((n4 + NT - 1) / NT, [&](auto c) {
      vis_gelu_quant_kernel<decltype(c)::value, NT><<<n, NT, 0, stream>>>(h, bias, mlp, xq, xs,
                                                                             warm);
      return hipGetLastError();
    });
  };
  if ((n4 + 255) / 256 <= kPfMaxNpt) return go(std::integral_constant<int, 256>{});
  if ((n4 + 511) / 512 <= kPfMaxNpt) return go(std::integral_constant<int, 512>{});
  return go(std::integral_constant<int, 1024>{});
}

hipError_t launch_vis_bias_gelu(float *h, const float *bias, int n, int mlp, hipStream_t stream) {
  if (n <= 0 || mlp <= 0 || mlp % 4 != 0) return hipErrorInvalidValue;
  vis_bias_gelu_kernel<<<dim3((mlp / 4 + kNT - 1) / kNT, n), kNT, 0, stream>>>(h, bias, mlp);
  return hipGetLastError();
}

hipError_t launch_vis_pool(const VisPool &a, int ntok, hipStream_t stream) {
  return by_npt<1, kPfMaxNpt>((a.dim / 4 + kNT - 1) / kNT, [&](auto c) {
    vis_pool_kernel<decltype(c)::value><<<ntok, kNT, 0, stream>>>(a);
    return hipGetLastError();
  });
}

}  // namespace gh
