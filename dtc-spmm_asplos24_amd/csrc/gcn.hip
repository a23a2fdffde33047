// Dense half of a GCN layer on gfx950: B = act(X) * W in bf16, written as
// the row-major bf16 B the SpMM gathers (b_dtype bfloat16).
//
// The reference's GCN forward (DTCSpMM_gcn, DTC-SpMM/DTCSpMM_kernel.cu:1033-1116)
// takes X W as a float32 tensor that the caller computed with a torch GEMM;
// here the product is one MFMA kernel whose prologue applies the previous
// layer's activation (ReLU) and the float32 -> bf16 cast while it loads X, and
// whose epilogue rounds to bf16 in the layout and precision the bf16-B SpMM
// reads -- no separate activation, cast or conversion pass over the
// M x F intermediates.
//
// The product is HBM-bound (X read once, B written once: 128 flop per byte at
// K = F = 256, against MI355X's 2.5 PFLOP/s over 8 TB/s = 312), so the
// kernel is built to read X once and keep W in L2:
//   * a workgroup computes 64 rows x 256 columns: 4 waves, 64 columns each
//     (4 MFMA column tiles), 4 row tiles of 16 each -- 64 accumulator VGPRs;
//   * X's 64 rows are staged in LDS as bf16, 128 columns of K at a time
//     (16 KB, rows padded by 16 bytes), shared by the four waves;
//   * W is packed once per call into MFMA fragment order (K/32 x F/16 groups
//     of 64 lanes x 8 bf16), so each B fragment is one contiguous 1 KB read,
//     served by L2 (W is 128 KB at K = F = 256);
//   * v_mfma_f32_16x16x32_bf16: lane l holds A[m = l % 16][k = 8 (l / 16) + j],
//     B[k = 8 (l / 16) + j][n = l % 16] and D[m = 4 (l / 16) + i][n = l % 16];
//   * the epilogue stages each wave's 16 x 64 tile through LDS and writes
//     whole 128-byte row segments.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>
#include <type_traits>

#include "dtc.h"
#include "dtc_internal.h"

namespace dtc {
namespace {

typedef __bf16 gbf16x8 __attribute__((ext_vector_type(8)));
typedef float gfloatx4 __attribute__((ext_vector_type(4)));

constexpr int kGemmRows = 64;         // rows per workgroup (128 measured slower: one wave per SIMD)
constexpr int kGemmCols = 256;        // columns per workgroup (4 waves x 64)
constexpr int kWaveCols = 64;         // columns per wave (4 MFMA column tiles)
constexpr int kKChunk = 128;          // K columns of X staged per LDS pass
constexpr int kXStride = kKChunk + 8; // LDS row stride in bf16 (16 bytes of padding)
constexpr int kColTiles = kWaveCols / 16;

// Packs W [K x F] (row-major bf16) into fragment order: group (s, t) for
// k-step s (32 rows of W) and column tile t (16 columns) holds, for lane l,
// W[32 s + 8 (l / 16) + j][16 t + l % 16], j = 0..7, as 8 consecutive bf16.
__global__ __launch_bounds__(256) void k_pack_w(const __bf16 *__restrict__ w, int32_t K, int32_t F,
                                                __bf16 *__restrict__ wp) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one (s, t, lane)
  const int64_t groups = (int64_t)(K / 32) * (F / 16);
  if (gid >= groups * 64) return;
  const int lane = (int)(gid & 63);
  const int64_t grp = gid >> 6;
  const int t = (int)(grp % (F / 16));
  const int s = (int)(grp / (F / 16));
  const int n = 16 * t + (lane & 15);
  const int k0 = 32 * s + 8 * (lane >> 4);
  gbf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = w[(int64_t)(k0 + j) * F + n];
  *reinterpret_cast<gbf16x8 *>(wp + gid * 8) = v;
}

template <bool XF32, bool RELU>
__device__ __forceinline__ __bf16 act(float x) {
  return (__bf16)(RELU ? fmaxf(x, 0.0f) : x);
}

// X[r0 .. r0 + ROWS)[kc .. kc + kw) (kw a multiple of 32, at most 128) is
// staged in two steps, so that the next chunk's loads are in flight while the
// current one is multiplied: load_x reads thread tid's pieces (8 consecutive
// elements of one row; piece idx = tid + 256 q, row idx / (kw / 8)) into
// registers, rows past M as zeros; store_x applies act, rounds to bf16 and
// writes them to LDS.
template <bool XF32, int ROWS>
struct XPieces {
  static constexpr int kPieces = ROWS * kKChunk / 8 / 256;  // per thread, at the widest chunk
  typename std::conditional<XF32, gfloatx4, gbf16x8>::type v[kPieces][XF32 ? 2 : 1];
};

template <bool XF32, int ROWS>
__device__ __forceinline__ void load_x(const void *__restrict__ x, int64_t r0, int32_t M, int32_t K,
                                       int kc, int kw, XPieces<XF32, ROWS> &xp) {
  const int per_row = kw / 8;
#pragma unroll
  for (int q = 0; q < XPieces<XF32, ROWS>::kPieces; ++q) {
    const int idx = threadIdx.x + 256 * q;
    const int r = idx / per_row;
    const int p = idx - r * per_row;
    const int64_t row = r0 + r;
    const bool ok = idx < ROWS * per_row && row < M;
    if constexpr (XF32) {
      const float *src = static_cast<const float *>(x) + (ok ? row * K + kc + 8 * p : 0);
      xp.v[q][0] = ok ? *reinterpret_cast<const gfloatx4 *>(src) : gfloatx4{0.f, 0.f, 0.f, 0.f};
      xp.v[q][1] = ok ? *reinterpret_cast<const gfloatx4 *>(src + 4) : gfloatx4{0.f, 0.f, 0.f, 0.f};
    } else {
      const __bf16 *src = static_cast<const __bf16 *>(x) + (ok ? row * K + kc + 8 * p : 0);
      gbf16x8 z;
#pragma unroll
      for (int j = 0; j < 8; ++j) z[j] = (__bf16)0.0f;
      xp.v[q][0] = ok ? *reinterpret_cast<const gbf16x8 *>(src) : z;
    }
  }
}

template <bool XF32, bool RELU, int ROWS>
__device__ __forceinline__ void store_x(int kw, const XPieces<XF32, ROWS> &xp, __bf16 *s_x) {
  const int per_row = kw / 8;
#pragma unroll
  for (int q = 0; q < XPieces<XF32, ROWS>::kPieces; ++q) {
    const int idx = threadIdx.x + 256 * q;
    if (idx >= ROWS * per_row) continue;  // a narrower last chunk (a guard, not a loop exit)
    const int r = idx / per_row;
    const int p = idx - r * per_row;
    gbf16x8 v;
    if constexpr (XF32) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = act<XF32, RELU>(xp.v[q][0][j]);
        v[4 + j] = act<XF32, RELU>(xp.v[q][1][j]);
      }
    } else {
      v = xp.v[q][0];
      if constexpr (RELU) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = act<XF32, RELU>((float)v[j]);
      }
    }
    *reinterpret_cast<gbf16x8 *>(s_x + r * kXStride + 8 * p) = v;
  }
}

// One 16 x 64 output tile (64 columns from col0, those below F; rows below
// M), staged row-major in LDS at s_o, written as whole row segments.  With a
// mask (the layer's input, laid out and typed as the output) each element is
// multiplied by mask > 0.
template <bool OF32>
__device__ __forceinline__ void write_tile(const void *s_o, int64_t r0, int col0, int32_t M, int32_t F,
                                           const void *mask, void *out) {
  typedef typename std::conditional<OF32, gfloatx4, gbf16x8>::type vec;
  constexpr int kVec = OF32 ? 4 : 8;            // elements per piece
  constexpr int kPerRow = kWaveCols / kVec;     // pieces per row
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < 16 * kPerRow / 64; ++h) {
    const int piece = h * 64 + lane;
    const int r = piece / kPerRow;
    const int p = piece % kPerRow;
    const int64_t row = r0 + r;
    vec v = static_cast<const vec *>(s_o)[piece];
    if (row >= M || col0 + kVec * p >= F) continue;
    const int64_t at = (row * F + col0) / kVec + p;
    if (mask) {
      const vec m = static_cast<const vec *>(mask)[at];
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        if constexpr (OF32) v[j] *= m[j] > 0.f ? 1.f : 0.f;
        else v[j] = (__bf16)((float)v[j] * ((float)m[j] > 0.f ? 1.f : 0.f));
      }
    }
    static_cast<vec *>(out)[at] = v;
  }
}

// ROWS rows (ROWS / 16 row tiles) per workgroup.  F: output columns, a
// multiple of 32; OF32: the bf16-rounded result stored as float32.  As the
// input gradient (X = dY float32, a mask, float32 output: 805 MB at 262,144 x
// 256) 163-185 us, 4.4-4.9 TB/s, the rate of a large copy; a cast, a GEMM, a
// compare, a product and a cast took 470.
template <bool XF32, bool RELU, int ROWS, bool OF32>
__global__ __launch_bounds__(256) void k_gcn_transform(const void *__restrict__ x,
                                                       const __bf16 *__restrict__ wp, int32_t M,
                                                       int32_t K, int32_t F,
                                                       const void *__restrict__ mask,
                                                       void *__restrict__ out) {
  constexpr int kRowTiles = ROWS / 16;
  __shared__ __attribute__((aligned(16))) __bf16 s_x[ROWS * kXStride];  // 34,816 bytes at 128 rows
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int64_t r0 = (int64_t)blockIdx.x * ROWS;
  const int col0 = blockIdx.y * kGemmCols + wave * kWaveCols;  // this wave's first column
  const bool active = col0 < F;
  const int ntile_f = F / 16;
  gfloatx4 acc[kRowTiles][kColTiles];
#pragma unroll
  for (int i = 0; i < kRowTiles; ++i)
#pragma unroll
    for (int c = 0; c < kColTiles; ++c) acc[i][c] = gfloatx4{0.f, 0.f, 0.f, 0.f};
  XPieces<XF32, ROWS> xp;
  load_x<XF32, ROWS>(x, r0, M, K, 0, min(kKChunk, K), xp);
  for (int kc = 0; kc < K; kc += kKChunk) {
    const int kw = min(kKChunk, K - kc);
    __syncthreads();  // the previous chunk's fragments are read
    store_x<XF32, RELU, ROWS>(kw, xp, s_x);
    __syncthreads();
    if (kc + kKChunk < K) load_x<XF32, ROWS>(x, r0, M, K, kc + kKChunk, min(kKChunk, K - kc - kKChunk), xp);
    if (active) {
      for (int ks = 0; ks < kw; ks += 32) {
        const int s = (kc + ks) / 32;
        gbf16x8 bfrag[kColTiles];
#pragma unroll
        for (int c = 0; c < kColTiles; ++c) {
          const int t = min(col0 / 16 + c, ntile_f - 1);  // past F (a multiple of 32): computed, not written
          bfrag[c] = *reinterpret_cast<const gbf16x8 *>(wp + (((int64_t)s * ntile_f + t) * 64 + lane) * 8);
        }
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i) {
          const gbf16x8 afrag = *reinterpret_cast<const gbf16x8 *>(
              s_x + (16 * i + (lane & 15)) * kXStride + ks + 8 * (lane >> 4));
#pragma unroll
          for (int c = 0; c < kColTiles; ++c)
            acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afrag, bfrag[c], acc[i][c], 0, 0, 0);
        }
      }
    }
  }
  // Epilogue: each wave stages a 16 x 64 tile (2 or 4 KB) in its own part of
  // s_x and writes it out as 16 rows of 128 or 256 bytes.
  __syncthreads();  // every wave is done reading X from s_x
  if (!active) return;
  typedef typename std::conditional<OF32, float, __bf16>::type oelem;
  oelem *s_o = reinterpret_cast<oelem *>(s_x) + wave * (16 * kWaveCols);
  static_assert(sizeof(s_x) >= 4 * 16 * kWaveCols * sizeof(oelem), "epilogue staging");
#pragma unroll
  for (int i = 0; i < kRowTiles; ++i) {
#pragma unroll
    for (int c = 0; c < kColTiles; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        s_o[(4 * (lane >> 4) + e) * kWaveCols + 16 * c + (lane & 15)] = (oelem)(__bf16)acc[i][c][e];
    wave_lds_sync();
    write_tile<OF32>(s_o, r0 + 16 * i, col0, M, F, mask, out);
    wave_lds_sync();
  }
}

// Packs W^T the same way, for the product dY W^T: group (s, t) for k-step s
// (32 columns of W) and output tile t (16 rows of W) holds, for lane l,
// W[16 t + l % 16][32 s + 8 (l / 16) + j]: 8 consecutive elements of a row.
__global__ __launch_bounds__(256) void k_pack_wt(const __bf16 *__restrict__ w, int32_t K, int32_t F,
                                                 __bf16 *__restrict__ wp) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one (s, t, lane)
  const int64_t groups = (int64_t)(F / 32) * (K / 16);
  if (gid >= groups * 64) return;
  const int lane = (int)(gid & 63);
  const int64_t grp = gid >> 6;
  const int t = (int)(grp % (K / 16));
  const int s = (int)(grp / (K / 16));
  const __bf16 *src = w + (int64_t)(16 * t + (lane & 15)) * F + 32 * s + 8 * (lane >> 4);
  gbf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = src[j];
  *reinterpret_cast<gbf16x8 *>(wp + gid * 8) = v;
}

// Partial dW = act(X)^T dY over a range of rows: each wave a 64 x 64 tile of
// dW for rows_per rows, the waves of a workgroup neighbouring tiles of the
// same rows.  The contraction runs over rows, so an MFMA operand needs 8 rows
// of one column per lane; instead of transposing through LDS, lane l reads 4
// consecutive columns (4 c .. 4 c + 3, c = l % 16) of the 8 rows m0 + 8 (l /
// 16) + j straight from memory (16-lane groups read 256 contiguous bytes)
// and MFMA tile t takes column t of every lane's four: tile (t, u) holds
// dW rows 4 c + t and columns 4 c + u of the wave's 64 x 64.  The next
// 32 rows are loaded while the current ones are converted and multiplied.
// Bound by its loads (X and dY read once from HBM, the waves' repeats of a row
// from L2): on X 262,144 x 256 float32 and dY 262,144 x 256, 537 MB, 162 us
// with the sum below, where a ReLU, a cast, a transposing copy and a batched
// GEMM took 390; on bf16 X 127.  Three waves per SIMD (168 registers) and four
// waves per workgroup measured 2-6% ahead of two and eight.
constexpr int kDwWaves = 4;
template <bool XF32, bool RELU>
__global__ __launch_bounds__(64 * kDwWaves, 3) void k_gcn_dw(const void *__restrict__ x_,
                                                          const float *__restrict__ dy, int32_t M,
                                                          int32_t K, int32_t F, int32_t tiles,
                                                          int32_t units, int32_t rows_per,
                                                          float *__restrict__ parts) {
  typedef typename std::conditional<XF32, float, __bf16>::type xelem;
  typedef xelem xvec __attribute__((ext_vector_type(4)));
  const xelem *x = static_cast<const xelem *>(x_);
  // Consecutive workgroups go to the 8 XCDs round robin; the grid is a
  // multiple of 8, and this gives every XCD a contiguous range of units, so
  // that the workgroups sharing rows share an L2.
  const int per_xcd = gridDim.x >> 3;
  const int block = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int unit = block * kDwWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;
  const int split = unit / tiles;
  const int tile = unit - split * tiles;
  const int nf = F / 64;
  const int k0 = tile / nf * 64;
  const int f0 = tile % nf * 64;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15;
  const int h = lane >> 4;
  const int64_t r0 = (int64_t)split * rows_per;
  const int64_t r1 = r0 + rows_per < M ? r0 + rows_per : M;
  const int kx = min(k0 + 4 * c, K - 4);  // columns past K (a multiple of 32) are computed, not written
  xvec xv[8];
  gfloatx4 yv[8];
  // Rows m0 + 8 h + j: a wave-uniform row base and one 32-bit lane offset
  // (25 K and 25 F are below 2^31: check_gradient_shape).
  const uint32_t xo = (uint32_t)(8 * h * K + kx), yo = (uint32_t)(8 * h * F + f0 + 4 * c);
  auto load = [&](int64_t m0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      xv[j] = *reinterpret_cast<const xvec *>(x + (m0 + j) * K + xo);
      yv[j] = *reinterpret_cast<const gfloatx4 *>(dy + (m0 + j) * F + yo);
    }
  };
  auto act_of = [](float v) { return (__bf16)(RELU && v < 0.f ? 0.f : v); };  // a NaN stays one
  gfloatx4 acc[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[t][u] = gfloatx4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](auto &&next) {
    gbf16x8 a[4], b[4];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        a[t][j] = act_of((float)xv[j][t]);
        b[t][j] = (__bf16)yv[j][t];
      }
    next();
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
  };
  int64_t m0 = r0;
  if (m0 + 32 <= r1) {
    load(m0);
    for (; m0 + 64 <= r1; m0 += 32) multiply([&] { load(m0 + 32); });
    multiply([] {});
    m0 += 32;
  }
  if (m0 < r1) {  // fewer than 32 rows left: zeros past them
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t row = m0 + 8 * h + j;
      xvec zx;
#pragma unroll
      for (int t = 0; t < 4; ++t) zx[t] = (xelem)0.f;
      xv[j] = row < r1 ? *reinterpret_cast<const xvec *>(x + row * K + kx) : zx;
      yv[j] = row < r1 ? *reinterpret_cast<const gfloatx4 *>(dy + row * F + f0 + 4 * c) : gfloatx4{0.f, 0.f, 0.f, 0.f};
    }
    multiply([] {});
  }
  // acc[t][u][i]: dW row k0 + 4 (4 h + i) + t, column f0 + 4 c + u
  float *dst = parts + (int64_t)split * K * F;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + 4 * (4 * h + i) + t;
      if (k >= K) continue;
      const gfloatx4 v = {acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
      *reinterpret_cast<gfloatx4 *>(dst + (int64_t)k * F + f0 + 4 * c) = v;
    }
}

// dW = bf16(sum of the partials), in a fixed order: 32 groups of 4 columns by
// 8 ranges of partials per workgroup, the ranges added through LDS.
__global__ __launch_bounds__(256) void k_gcn_dw_sum(const float *__restrict__ parts, int32_t splits,
                                                    int64_t count, __bf16 *__restrict__ dw) {
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
  __shared__ gfloatx4 s_sum[8][32];
  const int g = threadIdx.x & 31;
  const int part = threadIdx.x >> 5;
  const int64_t at = ((int64_t)blockIdx.x * 32 + g) * 4;
  gfloatx4 sum = {0.f, 0.f, 0.f, 0.f};
  if (at < count)
#pragma unroll 4
    for (int s = part; s < splits; s += 8) sum += *reinterpret_cast<const gfloatx4 *>(parts + s * count + at);
  s_sum[part][g] = sum;
  __syncthreads();
  if (part != 0 || at >= count) return;
#pragma unroll
  for (int s = 1; s < 8; ++s) sum += s_sum[s][g];
  bf4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = (__bf16)sum[j];
  *reinterpret_cast<bf4 *>(dw + at) = v;
}

// Rows per partial and number of partials of dW: about two waves per SIMD of
// 64 x 64 tiles, at least 128 rows each.
struct DwPlan {
  int32_t tiles, rows_per, splits;
};
DwPlan dw_plan(int32_t m, int32_t k, int32_t f) {
  DwPlan p;
  p.tiles = (int32_t)(ceil_div(k, 64) * (f / 64));
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>(2048 / p.tiles, ceil_div(m, 128)));
  p.rows_per = (int32_t)(ceil_div(ceil_div(std::max<int32_t>(m, 1), want), 32) * 32);
  p.splits = (int32_t)std::max<int64_t>(1, ceil_div(m, p.rows_per));
  return p;
}

dtc_status_t check_gcn_shape(int32_t m, int32_t k, int32_t f) {
  if (m < 0 || k <= 0 || f <= 0) return fail(DTC_ERROR_INVALID_VALUE, "M must be >= 0, K and F > 0");
  if (k % 32 != 0) return fail(DTC_ERROR_UNSUPPORTED, "K must be a multiple of 32");
  if (f % 64 != 0) return fail(DTC_ERROR_UNSUPPORTED, "F must be a multiple of 64");
  return DTC_SUCCESS;
}

// The gradients' kernels hold row offsets and tile counts in 32 bits and launch
// a thread per two of dW's elements, of which a launch takes fewer than 2^32.
dtc_status_t check_gradient_shape(int32_t m, int32_t k, int32_t f) {
  const dtc_status_t st = check_gcn_shape(m, k, f);
  if (st == DTC_SUCCESS && (int64_t)k * f >= (int64_t)1 << 31)
    return fail(DTC_ERROR_UNSUPPORTED, "K * F must be below 2^31 for the gradients");
  return st;
}

}  // namespace
}  // namespace dtc

using namespace dtc;

extern "C" {

dtc_status_t dtc_gcn_pack_weights(const void *w, int32_t k, int32_t f, void *w_packed,
                                  dtc_stream_t stream_) {
  clear_error();
  dtc_status_t st = check_gcn_shape(0, k, f);
  if (st != DTC_SUCCESS) return st;
  if (!w || !w_packed) return fail(DTC_ERROR_INVALID_VALUE, "W and the packed buffer are required");
  if (((uintptr_t)w_packed & 15) != 0) return fail(DTC_ERROR_INVALID_VALUE, "the packed buffer must be 16-byte aligned");
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  const int64_t threads = (int64_t)(k / 32) * (f / 16) * 64;
  k_pack_w<<<(unsigned)ceil_div(threads, 256), 256, 0, stream>>>(static_cast<const __bf16 *>(w), k, f,
                                                                static_cast<__bf16 *>(w_packed));
  DTC_LAUNCH_CHECK("gcn_pack_weights");
  return DTC_SUCCESS;
}

dtc_status_t dtc_gcn_transform(const void *x, int32_t x_dtype, int32_t relu, const void *w_packed,
                               int32_t m, int32_t k, int32_t f, void *out, dtc_stream_t stream_) {
  clear_error();
  dtc_status_t st = check_gcn_shape(m, k, f);
  if (st != DTC_SUCCESS) return st;
  if (x_dtype != DTC_GCN_X_FLOAT32 && x_dtype != DTC_GCN_X_BFLOAT16)
    return fail(DTC_ERROR_INVALID_VALUE, "x_dtype must be DTC_GCN_X_FLOAT32 or DTC_GCN_X_BFLOAT16");
  if (relu != 0 && relu != 1) return fail(DTC_ERROR_INVALID_VALUE, "relu must be 0 or 1");
  if (m == 0) return DTC_SUCCESS;
  if (!x || !w_packed || !out) return fail(DTC_ERROR_INVALID_VALUE, "X, packed W and the output are required");
  if (((uintptr_t)x & 15) || ((uintptr_t)w_packed & 15) || ((uintptr_t)out & 15))
    return fail(DTC_ERROR_INVALID_VALUE, "X, packed W and the output must be 16-byte aligned");
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  const __bf16 *wp = static_cast<const __bf16 *>(w_packed);
  __bf16 *o = static_cast<__bf16 *>(out);
  const dim3 grid((unsigned)ceil_div(m, kGemmRows), (unsigned)ceil_div(f, kGemmCols));
  auto launch = [&](auto kernel) { kernel<<<grid, 256, 0, stream>>>(x, wp, m, k, f, nullptr, o); };
  if (x_dtype == DTC_GCN_X_FLOAT32)
    relu ? launch(k_gcn_transform<true, true, kGemmRows, false>) : launch(k_gcn_transform<true, false, kGemmRows, false>);
  else
    relu ? launch(k_gcn_transform<false, true, kGemmRows, false>) : launch(k_gcn_transform<false, false, kGemmRows, false>);
  DTC_LAUNCH_CHECK("gcn_transform");
  return DTC_SUCCESS;
}

dtc_status_t dtc_gcn_input_grad(const float *dy, const void *w, const void *x, int32_t x_dtype, int32_t relu,
                                int32_t m, int32_t k, int32_t f, void *dx, void *workspace,
                                size_t workspace_bytes, dtc_stream_t stream_) {
  clear_error();
  dtc_status_t st = check_gradient_shape(m, k, f);
  if (st != DTC_SUCCESS) return st;
  if (x_dtype != DTC_GCN_X_FLOAT32 && x_dtype != DTC_GCN_X_BFLOAT16)
    return fail(DTC_ERROR_INVALID_VALUE, "x_dtype must be DTC_GCN_X_FLOAT32 or DTC_GCN_X_BFLOAT16");
  if (relu != 0 && relu != 1) return fail(DTC_ERROR_INVALID_VALUE, "relu must be 0 or 1");
  if (m == 0) return DTC_SUCCESS;
  if (!dy || !w || !dx || (relu && !x)) return fail(DTC_ERROR_INVALID_VALUE, "dY, W, dX and (for a ReLU) X are required");
  if (((uintptr_t)dy & 15) || ((uintptr_t)x & 15) || ((uintptr_t)dx & 15) || ((uintptr_t)workspace & 15))
    return fail(DTC_ERROR_INVALID_VALUE, "dY, X, dX and the workspace must be 16-byte aligned");
  const size_t need = (size_t)k * f * sizeof(__bf16);
  if (!workspace || workspace_bytes < need)
    return fail(DTC_ERROR_WORKSPACE, "the input gradient needs " + std::to_string(need) + " bytes of workspace");
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  __bf16 *wt = static_cast<__bf16 *>(workspace);
  const int64_t threads = (int64_t)(f / 32) * (k / 16) * 64;
  k_pack_wt<<<(unsigned)ceil_div(threads, 256), 256, 0, stream>>>(static_cast<const __bf16 *>(w), k, f, wt);
  DTC_LAUNCH_CHECK("gcn_pack_wt");
  const dim3 grid((unsigned)ceil_div(m, kGemmRows), (unsigned)ceil_div(k, kGemmCols));
  const void *mask = relu ? x : nullptr;
  if (x_dtype == DTC_GCN_X_FLOAT32)
    k_gcn_transform<true, false, kGemmRows, true><<<grid, 256, 0, stream>>>(dy, wt, m, f, k, mask, dx);
  else
    k_gcn_transform<true, false, kGemmRows, false><<<grid, 256, 0, stream>>>(dy, wt, m, f, k, mask, dx);
  DTC_LAUNCH_CHECK("gcn_input_grad");
  return DTC_SUCCESS;
}

dtc_status_t dtc_gcn_weight_grad_workspace_size(int32_t m, int32_t k, int32_t f, size_t *bytes) {
  clear_error();
  if (!bytes) return fail(DTC_ERROR_INVALID_VALUE, "bytes is NULL");
  dtc_status_t st = check_gradient_shape(m, k, f);
  if (st != DTC_SUCCESS) return st;
  *bytes = (size_t)dw_plan(m, k, f).splits * k * f * sizeof(float);
  return DTC_SUCCESS;
}

dtc_status_t dtc_gcn_weight_grad(const void *x, int32_t x_dtype, int32_t relu, const float *dy, int32_t m,
                                 int32_t k, int32_t f, void *dw, void *workspace, size_t workspace_bytes,
                                 dtc_stream_t stream_) {
  clear_error();
  dtc_status_t st = check_gradient_shape(m, k, f);
  if (st != DTC_SUCCESS) return st;
  if (x_dtype != DTC_GCN_X_FLOAT32 && x_dtype != DTC_GCN_X_BFLOAT16)
    return fail(DTC_ERROR_INVALID_VALUE, "x_dtype must be DTC_GCN_X_FLOAT32 or DTC_GCN_X_BFLOAT16");
  if (relu != 0 && relu != 1) return fail(DTC_ERROR_INVALID_VALUE, "relu must be 0 or 1");
  if (!dw || (m > 0 && (!x || !dy))) return fail(DTC_ERROR_INVALID_VALUE, "X, dY and dW are required");
  if (((uintptr_t)x & 15) || ((uintptr_t)dy & 15) || ((uintptr_t)dw & 7) || ((uintptr_t)workspace & 15))
    return fail(DTC_ERROR_INVALID_VALUE, "X, dY and the workspace must be 16-byte aligned, dW 8-byte");
  const DwPlan p = dw_plan(m, k, f);
  const size_t need = (size_t)p.splits * k * f * sizeof(float);
  if (!workspace || workspace_bytes < need)
    return fail(DTC_ERROR_WORKSPACE, "the weight gradient needs " + std::to_string(need) + " bytes of workspace");
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  float *parts = static_cast<float *>(workspace);
  const int32_t units = p.tiles * p.splits;
  const unsigned grid = (unsigned)(ceil_div(ceil_div(units, kDwWaves), 8) * 8);
  auto launch = [&](auto kernel) {
    kernel<<<grid, 64 * kDwWaves, 0, stream>>>(x, dy, m, k, f, p.tiles, units, p.rows_per, parts);
  };
  if (x_dtype == DTC_GCN_X_FLOAT32) relu ? launch(k_gcn_dw<true, true>) : launch(k_gcn_dw<true, false>);
  else relu ? launch(k_gcn_dw<false, true>) : launch(k_gcn_dw<false, false>);
  DTC_LAUNCH_CHECK("gcn_dw");
  const int64_t count = (int64_t)k * f;
  k_gcn_dw_sum<<<(unsigned)ceil_div(count, 128), 256, 0, stream>>>(parts, p.splits, count, static_cast<__bf16 *>(dw));
  DTC_LAUNCH_CHECK("gcn_dw_sum");
  return DTC_SUCCESS;
}

}  // extern "C"
