// gemm_f32.hip -- fp32 GEMM for unquantized model files (gemma.c:3304-3399
// gemm_fpx): in split precision on the f16 matrix cores (gemm_h2_kernel), or
// on fp32 MFMA (v_mfma_f32_32x32x2_f32, gemm_f32_kernel).
//
//   dst[i][j] = sum_l src[i][l]*mat[j][l]
//
// The fp32-MFMA kernel: 256 threads, 2x2 waves, 128x128 or 64x64 block tiles, a K step of 16
// floats (64 bytes per row) double-buffered in LDS.  A lane
// owns 8 consecutive k of each step (lane / 32 picks the half) for A and B
// alike, so each of the 8 MFMA sub-steps pairs matching k.  The reference's
// fp32 sum has no fixed order (vectorised, KC-chunked, gemma.c:3287-3299), so
// parity for this path is a tolerance on |y - y_exact| / sum|a*b|.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "gh_arith.h"
#include "gh_kernels.h"

namespace gh {
namespace {

constexpr int kThreads = 256;
constexpr int kBK = 16;                   // floats of K per step
constexpr int kRowChunks = kBK / 4 + 1;   // float4 chunks per LDS row (+1 pad)

// WM x WN: each wave's sub-tile in 32x32 MFMA tiles; the 2x2 waves make a
// (64 WM) x (64 WN) block tile.
template <int WM, int WN>
__global__ __launch_bounds__(kThreads) void gemm_f32_kernel(
    float *__restrict__ dst, int dstr, const float *__restrict__ mat, int mstr,
    const float *__restrict__ src, int sstr, int m, int n, int k, F32Epilogue ep) {
  constexpr int kBM = 64 * WM, kBN = 64 * WN;
  __shared__ v4f lds_a[2][kBM][kRowChunks];
  __shared__ v4f lds_b[2][kBN][kRowChunks];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1;
  const int wn = wave & 1;
  const int m0 = blockIdx.y * kBM;
  const int n0 = blockIdx.x * kBN;
  const int ld_row = tid >> 2;
  const int ld_chunk = tid & 3;

  v4f ra[WM], rb[WN];
  auto load_tiles = [&](int kt) {
    const int kb = kt * kBK + ld_chunk * 4;
#pragma unroll
    for (int h = 0; h < WM; ++h) {
      const int gm = m0 + ld_row + 64 * h;
      ra[h] = (gm < m && kb < k)
                  ? *reinterpret_cast<const v4f *>(src + (size_t)gm * sstr + kb)
                  : v4f{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int h = 0; h < WN; ++h) {
      const int gn = n0 + ld_row + 64 * h;
      rb[h] = (gn < n && kb < k)
                  ? *reinterpret_cast<const v4f *>(mat + (size_t)gn * mstr + kb)
                  : v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int h = 0; h < WM; ++h) lds_a[buf][ld_row + 64 * h][ld_chunk] = ra[h];
#pragma unroll
    for (int h = 0; h < WN; ++h) lds_b[buf][ld_row + 64 * h][ld_chunk] = rb[h];
  };

  v16f acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = v16f{};

  const int nk = (k + kBK - 1) / kBK;
  load_tiles(0);
  store_tiles(0);
  __syncthreads();

  const int frag_row = lane & 31;
  const int half = lane >> 5;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load_tiles(kt + 1);
    v4f a[WM][2], b[WN][2];
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      a[i][0] = lds_a[cur][wm * 32 * WM + i * 32 + frag_row][half * 2];
      a[i][1] = lds_a[cur][wm * 32 * WM + i * 32 + frag_row][half * 2 + 1];
    }
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      b[j][0] = lds_b[cur][wn * 32 * WN + j * 32 + frag_row][half * 2];
      b[j][1] = lds_b[cur][wn * 32 * WN + j * 32 + frag_row][half * 2 + 1];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              a[i][s >> 2][s & 3], b[j][s >> 2][s & 3], acc[i][j], 0, 0, 0);
    if (kt + 1 < nk) store_tiles(cur ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int col = n0 + wn * 32 * WN + j * 32 + (lane & 31);
    if (col >= n) continue;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row =
            m0 + wm * 32 * WM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < m) dst[(size_t)row * dstr + col] = ep.apply(acc[i][j][r], row, col, dstr);
      }
  }
}

// The same GEMM on the f16 matrix cores in split precision (gh_arith.h): two
// scaled f16 pieces per operand, three products (v_mfma_f32_16x16x32_f16) with
// fp32 accumulation.  Three bf16 pieces with six products took twice the matrix
// work at about the same rate and rounded each sum twice as often.  Both in us
// and against the 64-bit sums (rms): 512x13824x1152 105 -> 76, 5.3e-7 ->
// 3.8e-7; 2048x20480x2560 1128 -> 758, 7.9e-7 -> 5.6e-7; 4096x4304x1152 276 ->
// 166.  That is 0.85 PFLOP/s of f16 products.  Bound by the vector work of the
// split (six sevenths of the time are left without it), the LDS traffic and the
// matrix cores together, none of them alone.
//
// Scales.  Each row of A and of B has its own power of two, set from its first
// K step so that the step's largest value lies in [2^10, 2^11): four octaves
// below what flags it, and with both pieces whole down to 2^-13 of it.  A later
// step with a scaled value of 2^15 or more flags it; the workgroup then moves
// those rows' scales, splits the step again and rescales its sums (exactly).
// Rows of zeros start at the least scale.
// Range.  The second piece ends at 2^-25, a full one for values from 2^-2 on.
// Each lane keeps the largest of its part of a row (four of every 32 floats)
// over eight to fifteen steps; a workgroup in which one of those is below 2^-2,
// and not zero, does its steps over with three bf16 pieces and six products,
// which hold any magnitudes.  So a value's error is at most 2^-23 of it or of the
// largest of those 32 to 60, whichever is more.  (An outlier 2^24 above its row
// and met by zeros left 2e-4 of the result.)  Over so many, rows in which values
// near zero are common pass: gelu(gate) up with three of five below 2^-12 of
// the largest; and over steps, not lanes, because the kernel is bound by the
// vector work: the first product above takes 76 us so, 73 without any check and
// 86 with the maxima of each step over four lanes.  Where every tile is done
// over, it takes 165.
//
// 256 threads, 2x2 waves of 2 WM x 2 WN 16x16 tiles.  Per 32-float K step the
// workgroup splits its A and B rows into two f16 planes each in LDS, doubly
// buffered: a wave's products of one step run between the vector instructions
// that split the next (one barrier a step; 77 -> 72 us against splitting, a
// barrier, and the products), and each row's registers are loaded again with
// the step after as soon as they are split.  The product is taken transposed
// (D = B A^T: lane l, element r holds row l % 16 of A and columns
// 4 (l / 16) + r), so a lane's four outputs are neighbours in memory.
//
// B comes as segments (F32Segs: q, k, v or gate, up side by side in the
// output); each thread resolves the rows it loads to their segment once.
// Split-K (SK, splits > 1): workgroup (x, y, z) computes K steps
// [z nk / splits, (z + 1) nk / splits) of tile (x, y), stores its fp32
// partial tile to the workspace, and counts itself in on the tile's counter;
// the workgroup that arrives last sums the splits' partials in split order
// (its own from registers), so the result does not depend on the order of
// arrival, runs the epilogue and resets the counter.
struct F32Split {
  int splits;
  int *ws;   // [tiles][splits][kThreads * WM * WN * 16] fp32 bits
  int *cnt;  // [tiles], zero between launches
};

constexpr int kScaleSet = 10, kScaleTop = 15;   // octaves of a row's scaled values
constexpr int kScaleMin = -126, kScaleMax = 117;  // whose scales are normal floats

// The largest of eight consecutive lanes' values.
__device__ __forceinline__ float max_of_8(float v) {
  v = fmaxf(v, dpp_f32<kDppXor1>(v));
  v = fmaxf(v, dpp_f32<kDppXor2>(v));
  return fmaxf(v, dpp_f32<kDppHalfMirror>(v));
}

template <int WM, int WN, bool SK>
__global__ __launch_bounds__(kThreads, WM * WN == 4 ? 2 : WM * WN == 2 ? 3 : 4) void gemm_h2_kernel(
    float *__restrict__ dst, int dstr, F32Segs b, int mstr, const float *__restrict__ src,
    int sstr, int m, int k, F32Epilogue ep, F32Split sk) {
  constexpr int kBM = 64 * WM, kBN = 64 * WN;
  constexpr int MI = 2 * WM, NJ = 2 * WN;  // 16x16 tiles of a wave
  constexpr int BK = 32;                   // floats of K per step
  constexpr int CPR = BK / 4;              // float4 chunks per row and step
  constexpr int RPP = kThreads / CPR;      // rows per load pass
  constexpr int HA = kBM / RPP, HB = kBN / RPP, H = HA + HB;
  static_assert(kBM % RPP == 0 && kBN % RPP == 0 && CPR == 8, "tile");
  // two steps' planes of A's rows then B's; a row's 16-byte chunk c stands at
  // c ^ (row / 4) % 4, which spreads 16 rows' equal chunks over all banks
  __shared__ __attribute__((aligned(16))) _Float16 plane[2][2][(kBM + kBN) * BK];
  __shared__ int exps[kBM + kBN], moved[kBM + kBN];
  __shared__ int flag[2];  // the step that left its range, by its parity
  __shared__ int wide;     // some row holds more than two pieces do

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1;
  const int wn = wave & 1;
  const int n = b.end[b.nseg - 1];
  const int m0 = blockIdx.y * kBM;
  const int n0 = blockIdx.x * kBN;
  const int ld_row = tid / CPR, ld_c = tid % CPR;  // chunk ld_c of rows ld_row + RPP h

  // the rows this thread loads, A's then B's (past the last: the last again,
  // whose outputs are not stored)
  const float *row[H];
#pragma unroll
  for (int h = 0; h < HA; ++h)
    row[h] = src + (size_t)min(m0 + ld_row + RPP * h, m - 1) * sstr;
#pragma unroll
  for (int h = 0; h < HB; ++h) {
    const int gn = min(n0 + ld_row + RPP * h, n - 1);
    const int t = (b.nseg > 1 && gn >= b.end[0]) + (b.nseg > 2 && gn >= b.end[1]);
    const int first = t == 0 ? 0 : t == 1 ? b.end[0] : b.end[1];
    const float *w = t == 0 ? b.w[0] : t == 1 ? b.w[1] : b.w[2];
    row[HA + h] = w + (size_t)(gn - first) * mstr;
  }

  v4f x[H];
  auto load = [&](int kt) {  // past the end of the rows: their last floats again
    const int kb = min(kt * BK + 4 * ld_c, k - 4);
#pragma unroll
    for (int h = 0; h < H; ++h) {
      x[h] = *reinterpret_cast<const v4f *>(row[h] + kb);
      __builtin_amdgcn_sched_barrier(0);  // in order: the steps wait for them one by one
    }
  };
  float f[H];  // 2^-E of those rows; 0 for what load() repeated
  auto step_max = [&](int h) {
    return max_of_8(fmaxf(fmaxf(finite_abs(x[h][0]), finite_abs(x[h][1])),
                          fmaxf(finite_abs(x[h][2]), finite_abs(x[h][3]))));
  };
  auto set = [&](int h, float top) {
    const int e = min(max((__float_as_int(top) >> 23) - 127 - kScaleSet, kScaleMin), kScaleMax);
    f[h] = __int_as_float((127 - e) << 23);
    if (ld_c == 0) exps[ld_row + RPP * h] = e;
  };
  // the largest magnitude of the lane's part of row h since the last check, and
  // the bits (less 1: zeros don't count) of the least of those
  float g[H];
  uint32_t low = ~0u;
  auto check = [&]() {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      low = min(low, (uint32_t)__float_as_int(g[h]) - 1u);
      g[h] = 0.0f;
    }
  };
  constexpr uint32_t kLeast = 0x3e800000u;  // 2^-2
  constexpr int kSteps = 8;                 // between checks, and at least before the last
  // splits row h of the step into the planes at `buf`; the largest magnitude
  const int st_at = ld_row * BK + ((ld_c / 2) ^ (ld_row / 4 % 4)) * 8 + ld_c % 2 * 4;
  static_assert(RPP % 16 == 0, "rows RPP apart swizzle alike");
  auto split_store = [&](int buf, int h) {
    const v4f y = x[h] * f[h];
    const h2 a = cvt_pk_f16(y[0], y[1]), c = cvt_pk_f16(y[2], y[3]);
    auto rest = [&](int e, _Float16 p) { return __builtin_fmaf(x[h][e], f[h], -(float)p); };
    const h2 a1 = cvt_pk_f16(rest(0, a[0]), rest(1, a[1]));
    const h2 c1 = cvt_pk_f16(rest(2, c[0]), rest(3, c[1]));
    const int at = st_at + RPP * h * BK;
    *reinterpret_cast<u2 *>(&plane[buf][0][at]) =
        u2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, c)};
    *reinterpret_cast<u2 *>(&plane[buf][1][at]) =
        u2{__builtin_bit_cast(uint32_t, a1), __builtin_bit_cast(uint32_t, c1)};
    return fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3])));
  };
  // the rows' last step: nothing past their end
  auto trim = [&](int kt) {
    if ((kt + 1) * BK > k && kt * BK + 4 * ld_c >= k) {
#pragma unroll
      for (int h = 0; h < H; ++h) f[h] = 0.0f;
    }
  };

  v4f acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, grp = lane >> 4;
  const int arow = wm * 16 * MI, bcol = wn * 16 * NJ;  // the wave's first row and column
  const int rd_at = fr * BK + (grp ^ (fr / 4)) * 8;
  // acc[i][j][r] is output row m0 + out_row(i), column n0 + out_col(j, r)
  auto out_row = [&](int i) { return arow + 16 * i + fr; };
  auto out_col = [&](int j, int r) { return bcol + 16 * j + 4 * grp + r; };

  const int nk = (k + BK - 1) / BK;
  int kt0 = 0, kt1 = nk;
  if constexpr (SK) {
    kt0 = (int)((long)blockIdx.z * nk / sk.splits);
    kt1 = (int)((long)(blockIdx.z + 1) * nk / sk.splits);
  }
  if (tid < 2) flag[tid] = -1;
  if (tid == 2) wide = 0;
  load(kt0);
  lds_barrier();  // flag and wide are set
#pragma unroll
  for (int h = 0; h < H; ++h) set(h, step_max(h));
  trim(kt0);
#pragma unroll
  for (int h = 0; h < H; ++h) g[h] = split_store(kt0 & 1, h);
  load(min(kt0 + 1, kt1 - 1));
  for (int kt = kt0; kt < kt1; ++kt) {
    const int buf = kt & 1;
    lds_barrier();  // the step's planes and flags are complete, the other planes are free
    if (__builtin_amdgcn_readfirstlane(flag[buf]) == kt) {
      // rows that left their range: new scales, the step split again, the sums
      // of those rows and columns rescaled
      load(kt);
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const float top = step_max(h);
        const int old = exps[ld_row + RPP * h];
        if (top * f[h] >= (float)(1 << kScaleTop)) set(h, top);
        // as the row's first lane, which never lies past its end, set it
        const int by = __shfl(old - exps[ld_row + RPP * h], lane & ~7, 64);
        if (ld_c == 0) moved[ld_row + RPP * h] = by;
        g[h] = fmaxf(ldexpf(g[h], by), split_store(buf, h));
      }
      load(min(kt + 1, kt1 - 1));
      lds_barrier();
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j][r] = ldexpf(acc[i][j][r], moved[out_row(i)] + moved[kBM + out_col(j, r)]);
    }
    h8 a[2][MI], w[2][NJ];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
        a[1 - p][i] =
            *reinterpret_cast<const h8 *>(&plane[buf][1 - p][(arow + 16 * i) * BK + rd_at]);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        w[p][j] =
            *reinterpret_cast<const h8 *>(&plane[buf][p][(kBM + bcol + 16 * j) * BK + rd_at]);
    }
    // the products, with the next step's split between them and the loads of
    // the one after
    trim(kt + 1);
    const int kb = min(min(kt + 2, kt1 - 1) * BK + 4 * ld_c, k - 4);
    float top = 0.0f;
    constexpr int kPer = 3 * MI * NJ / H;  // products per row of the split
    static_assert(kPer * H == 3 * MI * NJ, "products");
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const float top4 = split_store(1 - buf, h);
      top = fmaxf(top, top4);
      g[h] = fmaxf(g[h], top4);
      x[h] = *reinterpret_cast<const v4f *>(row[h] + kb);
#pragma unroll
      for (int u = h * kPer; u < (h + 1) * kPer; ++u) {
        const int q = u / (MI * NJ), j = u / MI % NJ, i = u % MI;  // a1 b0, a0 b1, a0 b0
        acc[i][j] =
            __builtin_amdgcn_mfma_f32_16x16x32_f16(w[q == 1][j], a[q == 0][i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                     // a product,
        __builtin_amdgcn_sched_group_barrier(0x2, (20 + kPer - 1) / kPer, 0);  // then vector work
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (__any(!(top < (float)(1 << kScaleTop))) && lane == 0) flag[1 - buf] = kt + 1;
    if ((kt + 2 - kt0) % kSteps == 0 && kt1 - kt - 2 >= kSteps) check();
  }
  check();
  // (a single lane's floats have no others beside them)
  if (__any(low < kLeast - 1 || k - kt0 * BK <= 4) && lane == 0) wide = 1;
  lds_barrier();  // every wave is done with the planes
  if (__builtin_amdgcn_readfirstlane(wide) != 0) {  // the steps over, at the same scales
#pragma unroll
    for (int h = 0; h < H; ++h) f[h] = __int_as_float((127 - exps[ld_row + RPP * h]) << 23);
    __bf16 *p3 = reinterpret_cast<__bf16 *>(&plane[0][0][0]);
    constexpr int kP3 = (kBM + kBN) * BK;  // 3 planes where 4 were
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    load(kt0);
#pragma unroll 1
    for (int kt = kt0; kt < kt1; ++kt) {
      trim(kt);
      lds_barrier();  // every wave is done with the step before
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const v4f y = x[h] * f[h];
        const Bf3x2 lo = split3x2(y[0], y[1]), hi = split3x2(y[2], y[3]);
        __bf16 *at = p3 + st_at + RPP * h * BK;
        *reinterpret_cast<u2 *>(at) = u2{lo.q0, hi.q0};
        *reinterpret_cast<u2 *>(at + kP3) = u2{lo.q1, hi.q1};
        *reinterpret_cast<u2 *>(at + 2 * kP3) = u2{lo.q2, hi.q2};
      }
      load(min(kt + 1, kt1 - 1));
      lds_barrier();
      bf8 a[3][MI], w[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          a[p][i] = *reinterpret_cast<const bf8 *>(p3 + p * kP3 + (arow + 16 * i) * BK + rd_at);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          w[p] = *reinterpret_cast<const bf8 *>(p3 + p * kP3 + (kBM + bcol + 16 * j) * BK + rd_at);
#pragma unroll
        for (int o = 2; o >= 0; --o)  // the small piece products first
#pragma unroll
          for (int p = o; p >= 0; --p)
#pragma unroll
            for (int i = 0; i < MI; ++i)
              acc[i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[o - p], a[p][i], acc[i][j], 0, 0, 0);
      }
    }
  }
  // to the operands' units
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[i][j][r] = ldexpf(acc[i][j][r], exps[out_row(i)] + exps[kBM + out_col(j, r)]);

  if constexpr (SK) {
    // Partials go out and come back in with device-coherent (agent-scope)
    // accesses, which write through and read past this XCD's L2.
    constexpr int kTileInts = kThreads * MI * NJ * 4;
    const int tile = blockIdx.y * gridDim.x + blockIdx.x;
    const int z = blockIdx.z;
    int *part = sk.ws + (size_t)tile * sk.splits * kTileInts;
    int *mine = part + (size_t)z * kTileInts;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          __hip_atomic_store(mine + ((i * NJ + j) * 4 + r) * kThreads + tid,
                             __float_as_int(acc[i][j][r]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    __shared__ int last;
    wait_vmcnt<0>();  // this thread's partial has reached the coherence point
    __syncthreads();
    if (tid == 0) last = atomicAdd(sk.cnt + tile, 1) == sk.splits - 1;
    __syncthreads();
    if (!last) return;
    // a split at a time, its loads in flight together (one value's splits in
    // turn waited for each load: 4 us per split)
    v4f sum[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) sum[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int o = 0; o < sk.splits; ++o) {
      const int *theirs = part + (size_t)o * kTileInts + tid;
      v4f y[MI][NJ];
      if (o != z) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              y[i][j][r] = __int_as_float(__hip_atomic_load(
                  theirs + ((i * NJ + j) * 4 + r) * kThreads, __ATOMIC_RELAXED,
                  __HIP_MEMORY_SCOPE_AGENT));
      } else {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) y[i][j] = acc[i][j];
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) sum[i][j] += y[i][j];
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = sum[i][j];
    if (tid == 0) sk.cnt[tile] = 0;
  }

#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r0 = m0 + out_row(i);
    if (r0 >= m) continue;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c0 = n0 + out_col(j, 0);
      float *out = dst + (size_t)r0 * dstr + c0;
      if (c0 + 4 <= n) {
        v4f y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = ep.apply(acc[i][j][r], r0, c0 + r, dstr);
        __builtin_memcpy(out, &y, 16);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (c0 + r < n) out[r] = ep.apply(acc[i][j][r], r0, c0 + r, dstr);
      }
    }
  }
}

// One launch of the split kernel: tiles of (64 WM) x (64 WN), `splits`
// workgroups per tile along z (1: no split-K).
template <int WM, int WN>
hipError_t launch_h2(float *dst, int dstr, const F32Segs &b, int mstr, const float *src,
                      int sstr, int m, int k, const F32Epilogue &ep, int splits,
                      hipStream_t stream) {
  const int n = b.end[b.nseg - 1];
  const dim3 grid((n + 64 * WN - 1) / (64 * WN), (m + 64 * WM - 1) / (64 * WM), splits);
  F32Split sk{splits, nullptr, nullptr};
  if (splits > 1) {
    const int tiles = (int)(grid.x * grid.y);
    const hipError_t e = split_workspace(
        stream, (size_t)tiles * splits * kThreads * WM * WN * 16, tiles, &sk.ws, &sk.cnt);
    if (e != hipSuccess) return e;
    gemm_h2_kernel<WM, WN, true><<<grid, kThreads, 0, stream>>>(dst, dstr, b, mstr, src, sstr,
                                                                m, k, ep, sk);
  } else {
    gemm_h2_kernel<WM, WN, false><<<grid, kThreads, 0, stream>>>(dst, dstr, b, mstr, src, sstr,
                                                                 m, k, ep, sk);
  }
  return hipGetLastError();
}

// Any shape, any alignment: one thread per output.
__global__ __launch_bounds__(kThreads) void gemm_f32_generic_kernel(
    float *__restrict__ dst, int dstr, const float *__restrict__ mat, int mstr,
    const float *__restrict__ src, int sstr, int m, int n, int k, F32Epilogue ep) {
  const int col = blockIdx.x * 64 + (threadIdx.x & 63);
  const int row = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (row >= m || col >= n) return;
  const float *a = src + (size_t)row * sstr;
  const float *b = mat + (size_t)col * mstr;
  float acc = 0.0f;
  for (int l = 0; l < k; ++l) acc = __builtin_fmaf(a[l], b[l], acc);
  dst[(size_t)row * dstr + col] = ep.apply(acc, row, col, dstr);
}

// The fp64 twin of the fp32 GEMM for the verification modes: each output is
// the fp64 sum, rounded once by the epilogue.  A workgroup computes a 32 x 64
// tile, each thread 2 x 4 outputs, over K in LDS chunks of 32.
constexpr int kF64M = 32, kF64N = 64, kF64K = 32;

__global__ __launch_bounds__(kThreads) void gemm_f64_kernel(
    float *__restrict__ dst, int dstr, const float *__restrict__ mat, int mstr,
    const float *__restrict__ src, int sstr, int m, int n, int k, F32Epilogue ep) {
  __shared__ float as[kF64M][kF64K + 1];
  __shared__ float bs[kF64N][kF64K + 1];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * kF64M, n0 = blockIdx.x * kF64N;
  const int tm = tid / 16, tn = tid % 16;  // outputs (m0 + 2 tm + i, n0 + tn + 16 j)
  double acc[2][4] = {};
  for (int k0 = 0; k0 < k; k0 += kF64K) {
    for (int i = tid; i < kF64M * kF64K; i += kThreads) {
      const int r = i / kF64K, c = i % kF64K;
      as[r][c] = (m0 + r < m && k0 + c < k) ? src[(size_t)(m0 + r) * sstr + k0 + c] : 0.0f;
    }
    for (int i = tid; i < kF64N * kF64K; i += kThreads) {
      const int r = i / kF64K, c = i % kF64K;
      bs[r][c] = (n0 + r < n && k0 + c < k) ? mat[(size_t)(n0 + r) * mstr + k0 + c] : 0.0f;
    }
    __syncthreads();
#pragma unroll 4
    for (int c = 0; c < kF64K; ++c) {
      const double x0 = as[2 * tm][c], x1 = as[2 * tm + 1][c];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double w = bs[tn + 16 * j][c];
        acc[0][j] = fma(x0, w, acc[0][j]);
        acc[1][j] = fma(x1, w, acc[1][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = m0 + 2 * tm + i;
    if (row >= m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + tn + 16 * j;
      if (col < n) dst[(size_t)row * dstr + col] = ep.apply_f64(acc[i][j], row, col, dstr);
    }
  }
}

// The fp32 GEMM's kernel: the split one by default, the fp32-MFMA one
// with GEMMA_HIP_GEMM_F32=mfma (read at every launch, so that one process
// can time or check both).
bool gemm_f32_split() {
  const char *e = getenv("GEMMA_HIP_GEMM_F32");
  return e == nullptr || strcmp(e, "mfma") != 0;
}

// Block tile of the fp32-MFMA kernel: 128x128 when that gives every CU at
// least two workgroups, else 64x64 (k/v, o and down at the gemma-3-4b
// prefill shapes leave most of the GPU idle at 128x128).
// GEMMA_HIP_GEMM_F32_TILE=128, 128x64 or 64 (read at every launch) forces a
// tile for either kernel.
enum Tile { kTile64, kTile128x64, kTile128 };
bool forced_tile(Tile *t) {
  const char *e = getenv("GEMMA_HIP_GEMM_F32_TILE");
  if (e == nullptr) return false;
  if (strcmp(e, "128") == 0) *t = kTile128;
  else if (strcmp(e, "128x64") == 0) *t = kTile128x64;
  else if (strcmp(e, "64") == 0) *t = kTile64;
  else return false;
  return true;
}

Tile f32_tile(int m, int n, const DeviceInfo &dev) {
  Tile t;
  if (forced_tile(&t)) return t;
  const long tiles128 = (long)((m + 127) / 128) * ((n + 127) / 128);
  return tiles128 >= 2L * dev.cus ? kTile128 : kTile64;
}

long tile_count(int m, int n, Tile t) {
  const int bm = t == kTile64 ? 64 : 128, bn = t == kTile128 ? 128 : 64;
  return (long)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
}

// Tile and split-K ways of the split kernel: the least of a time modelled from
// a sweep of the gemma-3 prompt and SigLIP shapes (each tile in 1, 2, 3, 4, 6
// and 8 splits; the model's choice is within 8% of the sweep's best).  A tile
// takes `lat` us a K step while its workgroups are alone on their CUs and
// `thr` us of a CU's time when `slots` share one; `ends` steps' time goes to its
// first loads and its stores.  Splitting K costs the partials' way through
// memory and the last workgroup's sum over them.  As measured, us, without and
// with splits: 512x2560x10240 (80 128x128 tiles) 160 -> 102 in 6, 2048x2048x2560
// (256) 83 -> 80 in 2, 64x1024x2048 (16 64x64 tiles) 34 -> 13 in 8, but
// 4096x4304x1152 (1088) 155 -> 165 in 2.  Each split keeps at least 6 K steps
// (192 floats); at most 16 splits, and partials of at most 5 128x128 tiles per
// CU (80 MiB).  Products of under 1.5 128x128 tiles per CU with 512 floats or
// more of K take two splits at least, whose sums are half as long: 4096x1152x588
// 38 -> 40 us, 2.8e-7 -> 2.0e-7 off the 64-bit sums (rms); 4096x1152x1152 62 ->
// 58, 3.8e-7 -> 2.7e-7.
// GEMMA_HIP_GEMM_F32_TILE forces the tile, GEMMA_HIP_GEMM_F32_SPLIT=s the
// splits (clamped to 1..min(16, K steps)); both are read at every launch.
struct H2Plan {
  Tile tile;
  int splits;
};
H2Plan h2_plan(int m, int n, int k, bool may_split, const DeviceInfo &dev) {
  struct Cost {
    Tile tile;
    int bm, bn, slots;
    double lat, thr, ends;
  };
  static constexpr Cost kCosts[] = {{kTile64, 64, 64, 4, 0.50, 0.33, 2},
                                    {kTile128x64, 128, 64, 3, 0.72, 0.56, 3},
                                    {kTile128, 128, 128, 2, 1.0, 0.87, 4}};
  constexpr double kSplitUs = 1.0, kPerSplitUs = 0.6, kPartialBytesPerUs = 9e6;
  const int nk = (k + 31) / 32;
  Tile only{};
  const bool one_tile = forced_tile(&only);
  const char *e = getenv("GEMMA_HIP_GEMM_F32_SPLIT");
  const int forced =
      !may_split ? 1 : e == nullptr ? 0 : std::max(1, std::min({atoi(e), nk, 16}));
  const int fewest = nk >= 16 && 2 * tile_count(m, n, kTile128) < 3L * dev.cus ? 2 : 1;
  H2Plan best{kTile64, fewest};
  double least = 1e300;
  for (const Cost &c : kCosts) {
    if (one_tile && c.tile != only) continue;
    if (one_tile) best.tile = c.tile;
    const long tiles = tile_count(m, n, c.tile);
    for (int s = forced ? forced : fewest; s <= (forced ? forced : 16); ++s) {
      const double partials = (double)tiles * s * c.bm * c.bn * 4;
      if (!forced && s > 1 && (nk < 6 * s || partials > 5.0 * dev.cus * 128 * 128 * 4)) break;
      const double wgs = (double)tiles * s / dev.cus, whole = std::ceil(wgs);
      const double steps = (nk + s - 1) / s + c.ends;
      // between the mean and the fullest CU's share: workgroups sharing a CU
      // run faster once the others have ended
      double us = steps * std::max(c.lat * std::ceil(wgs / c.slots), c.thr * (wgs + whole) / 2);
      if (s > 1) us += kSplitUs + kPerSplitUs * s + partials / kPartialBytesPerUs;
      if (us < least) {
        least = us;
        best = {c.tile, s};
      }
    }
  }
  return best;
}

hipError_t launch_h2_auto(float *dst, int dstr, const F32Segs &b, int mstr, const float *src,
                          int sstr, int m, int k, const F32Epilogue &ep, const DeviceInfo &dev,
                          hipStream_t stream) {
  // the split-K workspace is kept by stream, and may have to be allocated: not
  // for a handle of several streams, not under capture
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const bool may_split = stream_has_own_handle(stream) &&
                         hipStreamIsCapturing(stream, &cap) == hipSuccess &&
                         cap == hipStreamCaptureStatusNone;
  const H2Plan p = h2_plan(m, b.end[b.nseg - 1], k, may_split, dev);
  if (p.tile == kTile128)
    return launch_h2<2, 2>(dst, dstr, b, mstr, src, sstr, m, k, ep, p.splits, stream);
  if (p.tile == kTile128x64)
    return launch_h2<2, 1>(dst, dstr, b, mstr, src, sstr, m, k, ep, p.splits, stream);
  return launch_h2<1, 1>(dst, dstr, b, mstr, src, sstr, m, k, ep, p.splits, stream);
}

// float4 loads of both operands: K and the row strides multiples of 4
// floats, the bases 16-byte aligned.
bool f32_vec4(int k, int mstr, int sstr, const float *mat, const float *src) {
  return k % 4 == 0 && mstr % 4 == 0 && sstr % 4 == 0 && (uintptr_t)mat % 16 == 0 &&
         (uintptr_t)src % 16 == 0;
}

}  // namespace

hipError_t launch_gemm_f32(float *dst, int dstr, const float *mat, int mstr,
                           const float *src, int sstr, int m, int n, int k,
                           const F32Epilogue &ep, const DeviceInfo &dev, hipStream_t stream,
                           bool f64) {
  if (f64) {
    const dim3 grid((n + kF64N - 1) / kF64N, (m + kF64M - 1) / kF64M);
    gemm_f64_kernel<<<grid, kThreads, 0, stream>>>(dst, dstr, mat, mstr, src, sstr, m, n, k, ep);
    return hipGetLastError();
  }
  if (f32_vec4(k, mstr, sstr, mat, src)) {
    if (gemm_f32_split()) {
      const F32Segs b{{mat, nullptr, nullptr}, {n, n, n}, 1};
      return launch_h2_auto(dst, dstr, b, mstr, src, sstr, m, k, ep, dev, stream);
    }
    const Tile tile = f32_tile(m, n, dev);
    if (tile == kTile128) {
      const dim3 grid((n + 127) / 128, (m + 127) / 128);
      gemm_f32_kernel<2, 2><<<grid, kThreads, 0, stream>>>(dst, dstr, mat, mstr, src, sstr, m,
                                                          n, k, ep);
    } else if (tile == kTile128x64) {
      const dim3 grid((n + 63) / 64, (m + 127) / 128);
      gemm_f32_kernel<2, 1><<<grid, kThreads, 0, stream>>>(dst, dstr, mat, mstr, src, sstr, m,
                                                          n, k, ep);
    } else {
      const dim3 grid((n + 63) / 64, (m + 63) / 64);
      gemm_f32_kernel<1, 1><<<grid, kThreads, 0, stream>>>(dst, dstr, mat, mstr, src, sstr, m,
                                                          n, k, ep);
    }
  } else {
    const dim3 grid((n + 63) / 64, (m + 3) / 4);
    gemm_f32_generic_kernel<<<grid, kThreads, 0, stream>>>(dst, dstr, mat, mstr,
                                                           src, sstr, m, n, k, ep);
  }
  return hipGetLastError();
}

hipError_t launch_gemm_f32_segs(float *dst, int dstr, const F32Segs &b, int mstr,
                                const float *src, int sstr, int m, int k,
                                const F32Epilogue &ep, const DeviceInfo &dev, hipStream_t stream,
                                bool f64) {
  bool vec4 = true;
  for (int t = 0; t < b.nseg; ++t) vec4 = vec4 && f32_vec4(k, mstr, sstr, b.w[t], src);
  if (!f64 && vec4 && gemm_f32_split())
    return launch_h2_auto(dst, dstr, b, mstr, src, sstr, m, k, ep, dev, stream);
  // one launch per segment, the epilogue's column-indexed inputs shifted
  // to the segment's first column
  for (int t = 0; t < b.nseg; ++t) {
    const int first = t ? b.end[t - 1] : 0;
    F32Epilogue et = ep;
    if (et.bias != nullptr) et.bias += first;
    if (et.pos_q != nullptr) et.pos_q += first;
    if (et.pos_f != nullptr) et.pos_f += first;
    const hipError_t e = launch_gemm_f32(dst + first, dstr, b.w[t], mstr, src, sstr, m,
                                         b.end[t] - first, k, et, dev, stream, f64);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_gemm_f32(float *dst, int dstr, const float *mat, int mstr,
                           const float *src, int sstr, int m, int n, int k,
                           const float *bias, bool clamp,
                           const DeviceInfo &dev, hipStream_t stream) {
  F32Epilogue ep{};
  ep.bias = bias;
  ep.clamp = clamp;
  return launch_gemm_f32(dst, dstr, mat, mstr, src, sstr, m, n, k, ep, dev, stream, false);
}

}  // namespace gh
