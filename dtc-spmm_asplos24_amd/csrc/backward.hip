// Gradient building blocks for C = A * B on gfx950.
//
// The reference binds its backward names to the forwards
// (DTC-SpMM/DTCSpMM.cpp:384-399) and so returns A * dY; these kernels supply
// the true gradients instead:
//   dB = A^T * dC  -> the CSR transpose here, then the ME-TCF build and the
//                     SpMM of the transpose;
//   dA = SDDMM     -> dA[e] = dC[row(e), :] . B[col(e), :] on A's pattern.
#include <algorithm>
#include <string>
#include <type_traits>

#include "dtc_internal.h"

namespace dtc {
namespace {

// out[e] = x[row(e)] . y[col(e)], edge-parallel: every wavefront takes 8
// consecutive edges at a time (CSR order), all 64 lanes reading VEC floats of
// each edge's two rows (one 1 KB row per edge at n = 256 and VEC = 4), so a
// hub row is spread over many wavefronts.  The row of an edge comes from
// edge_to_row when given, else from a binary search of rowptr (lanes 0-7,
// one edge each).  The 8 partial dot products are reduced together: three
// halving exchanges (4, 2, 1 values) then three plain butterfly steps.
constexpr int kSddmmEdges = 8;

// Y as bfloat16 (YBF = true): VEC bf16 per lane (8 bytes at VEC = 4), taken
// exactly and widened to float32 before the product.
template <int VEC, bool YBF>
struct YVec;
template <int VEC>
struct YVec<VEC, false> {
  typedef float type __attribute__((ext_vector_type(VEC)));
  __device__ static float at(const type &v, int i) { return v[i]; }
};
template <int VEC>
struct YVec<VEC, true> {
  typedef unsigned short type __attribute__((ext_vector_type(VEC)));
  __device__ static float at(const type &v, int i) {
    return __uint_as_float((uint32_t)v[i] << 16);
  }
};

template <int VEC, bool YBF>
__global__ __launch_bounds__(256) void k_sddmm(const int32_t *rowptr, const int32_t *col,
                                               const int32_t *e2r, int32_t M, int32_t nnz,
                                               const float *x, const void *y_, int32_t y_rows,
                                               int32_t n, float *out) {
  typedef float vfloat __attribute__((ext_vector_type(VEC)));
  typedef YVec<VEC, YBF> YV;
  typedef typename YV::type yvec;
  typedef typename std::conditional<YBF, unsigned short, float>::type yelem;
  const yelem *y = static_cast<const yelem *>(y_);
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  const int64_t groups = ((int64_t)nnz + kSddmmEdges - 1) / kSddmmEdges;
  for (int64_t g = wave; g < groups; g += nwaves) {
    const int64_t e0 = g * kSddmmEdges;
    // rows and columns of the 8 edges (lane k holds edge e0 + k)
    int my_row = 0, my_col = -1;
    if (lane < kSddmmEdges && e0 + lane < nnz) {
      const int e = (int)(e0 + lane);
      my_col = col[e];
      if (e2r) {
        my_row = e2r[e];
      } else {
        int lo = 0, hi = M;  // last row r with rowptr[r] <= e
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (rowptr[mid] <= e) lo = mid;
          else hi = mid;
        }
        my_row = lo;
      }
      if ((unsigned)my_row >= (unsigned)M) my_col = -1;  // defensive: never read outside x
    }
    // Branch-free loads: an edge without a valid column reads row 0 of x and
    // y (both exist: M >= 1 and y_rows >= 1 here) and is masked afterwards,
    // so all 16 row loads of a lane are in flight together.
    int rk[kSddmmEdges], jk[kSddmmEdges];
    bool ok[kSddmmEdges];
#pragma unroll
    for (int k = 0; k < kSddmmEdges; ++k) {
      rk[k] = __builtin_amdgcn_readlane(my_row, k);
      jk[k] = __builtin_amdgcn_readlane(my_col, k);
      ok[k] = (unsigned)jk[k] < (unsigned)y_rows;
      if (!ok[k]) rk[k] = jk[k] = 0;
    }
    float p[kSddmmEdges];
#pragma unroll
    for (int k = 0; k < kSddmmEdges; ++k) p[k] = 0.f;
    // bfloat16 y, all 8 edges in one row (the common case inside long rows):
    // x is loaded once, so a lane moves 16 + 8*8 bytes instead of 8*(16 + 8).
    // rk[] is wave-uniform, so this is a scalar branch; the general path is
    // left as it was rather than copying registers whose loads are still in
    // flight, which would make the loads wait on one another.  Not for
    // float32 y: there the second path costs registers (one wave fewer per
    // SIMD) and measured slower.
    bool one_row = YBF;
#pragma unroll
    for (int k = 1; k < kSddmmEdges; ++k) one_row = one_row && rk[k] == rk[0];
    if (one_row) {
      for (int c = lane * VEC; c < n; c += kWave * VEC) {
        const vfloat xv = *reinterpret_cast<const vfloat *>(x + (int64_t)rk[0] * n + c);
        yvec yv[kSddmmEdges];
#pragma unroll
        for (int k = 0; k < kSddmmEdges; ++k)
          yv[k] = *reinterpret_cast<const yvec *>(y + (int64_t)jk[k] * n + c);
#pragma unroll
        for (int k = 0; k < kSddmmEdges; ++k)
#pragma unroll
          for (int v = 0; v < VEC; ++v) p[k] += xv[v] * YV::at(yv[k], v);
      }
    } else {
      for (int c = lane * VEC; c < n; c += kWave * VEC) {
        vfloat xv[kSddmmEdges];
        yvec yv[kSddmmEdges];
#pragma unroll
        for (int k = 0; k < kSddmmEdges; ++k) {
          xv[k] = *reinterpret_cast<const vfloat *>(x + (int64_t)rk[k] * n + c);
          yv[k] = *reinterpret_cast<const yvec *>(y + (int64_t)jk[k] * n + c);
        }
#pragma unroll
        for (int k = 0; k < kSddmmEdges; ++k)
#pragma unroll
          for (int v = 0; v < VEC; ++v) p[k] += xv[k][v] * YV::at(yv[k], v);
      }
    }
#pragma unroll
    for (int k = 0; k < kSddmmEdges; ++k)
      if (!ok[k]) p[k] = 0.f;
    // halving exchanges: lanes keep the half of the values their bit selects
    const bool b5 = lane & 32, b4 = lane & 16, b3 = lane & 8;
    float q[4], t[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float send = b5 ? p[i] : p[i + 4];
      q[i] = (b5 ? p[i + 4] : p[i]) + __shfl_xor(send, 32, kWave);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float send = b4 ? q[i] : q[i + 2];
      t[i] = (b4 ? q[i + 2] : q[i]) + __shfl_xor(send, 16, kWave);
    }
    float v = (b3 ? t[1] : t[0]) + __shfl_xor(b3 ? t[0] : t[1], 8, kWave);
    v += __shfl_xor(v, 4, kWave);
    v += __shfl_xor(v, 2, kWave);
    v += __shfl_xor(v, 1, kWave);
    const int k = (lane >> 3) & 7;  // edge index this lane's sum belongs to
    if ((lane & 7) == 0 && e0 + k < nnz) out[e0 + k] = v;
  }
}

// The same by 16-lane groups, for operands that buffers can address (32-bit
// byte offsets; loads past an array's end return zero).  A wave takes 64
// consecutive edges, lane l holding the column and row of the l-th, and its
// lane groups 16 of them each, in steps of U edges per group: lane c of a group
// reads 16 bytes of a Y row per chunk (a group 256 contiguous bytes, an
// instruction four rows).  The rows of X that the edges span are staged in the
// wave's LDS, so a row is read once per wave and not once per edge; when they
// do not fit, fewer edges are taken at a time, and rows of hardly an edge each
// are read per edge.  The U sums over 16 lanes reduce together in
// data-parallel-primitive steps.
// Bound by the gathers of Y, 7 TB/s where it lies in the memory-side cache
// (uniform), 10-11 with hub columns in L2 (R-MAT).  Against the kernel above,
// which gives a row all 64 lanes and reads X per edge, us: 2^18-node R-MAT,
// 7.6M edges, float32 N = 64 496 -> 159, N = 69 509 -> 228, N = 128 521 -> 355,
// N = 192 564 -> 549, bf16 N = 128 400 -> 178, N = 256 432 -> 380; band 200,000
// N = 128 235 -> 85; uniform 262,144 of 8 per row N = 128 196 -> 174.  (X kept
// in registers while a lane group's row lasts, instead of LDS: 401 at N = 128;
// two steps' gathers in flight in turn: 357; several blocks of edges per wave
// with their columns loaded a block ahead: 359-361, and 20-30% slower on 0.5M
// edges.)
// NC: chunks per row (64 float32 or 128 bf16 columns each).  TAIL (float32): N
// is not a multiple of 4; the lane that crosses a row's end reads the row's
// last 4 columns instead and drops those its neighbour counts.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __uint_as_float(
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
constexpr int kDppRor = 0x120;  // + n: rotate each 16-lane row right by n lanes
constexpr int kDppRor8 = kDppRor + 8, kDppHalfMirror = 0x141, kDppXor1 = 0xB1, kDppXor2 = 0x4E;
constexpr int kDppBcast = 0x150;  // + n: lane n of each 16-lane row to the whole row
constexpr int kSddmmLds = 2048;   // floats of X staged per wave

// Edges per lane group and step.
template <int NC, bool YBF>
constexpr int sddmm_step() {
  return YBF ? (NC == 1 ? 4 : 2) : (NC == 1 ? 8 : 4);
}
template <int NC, bool YBF, bool TAIL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TAIL && NC == 3 ? 4 : 5))) void k_sddmm_groups(const int32_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ col,
                                                      const int32_t *__restrict__ e2r, int32_t M,
                                                      int32_t nnz, const float *__restrict__ x,
                                                      const void *__restrict__ y, int32_t y_rows,
                                                      int32_t n,
                                                      float *__restrict__ out) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int CW = YBF ? 8 : 4;         // columns per lane and chunk
  constexpr int XV = CW / 4;              // X vectors per chunk
  constexpr int XC = 16 * CW * NC;        // columns of a pass
  constexpr int U = sddmm_step<NC, YBF>();  // edges per group and step
  constexpr int kRows = kSddmmLds / XC;   // rows of X that fit
  constexpr uint32_t kOut = 0x80000000u;  // past every buffer: reads zero
  __shared__ __align__(16) float s_x[4][kSddmmLds];
  const int lane = lane_id();
  const int c = lane & 15;
  float *xs = s_x[wave_uniform(threadIdx.x >> 6)];
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave * 64 >= nnz) return;
  const int first = (int)(wave * 64);
  const int last = (int)min((int64_t)first + 64, (int64_t)nnz);  // exclusive
  const __amdgpu_buffer_rsrc_t xb =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x), 0, (int)((uint32_t)M * (uint32_t)n * 4u), 0x00020000);
  const __amdgpu_buffer_rsrc_t yb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void *>(y), 0, (int)((uint32_t)y_rows * (uint32_t)n * (YBF ? 2u : 4u)), 0x00020000);
  const uint32_t xstride = (uint32_t)n * 4u, ystride = (uint32_t)n * (YBF ? 2u : 4u);
  auto column = [&](int k) { return k * 16 * CW + c * CW; };
  auto load_ids = [&](int e0, int &j, int &r) {
    const int e = e0 + lane;
    j = r = -1;
    if (e < last) {
      j = col[e];
      if (e2r) {
        r = e2r[e];
      } else {
        int lo = 0, hi = M;  // last row r with rowptr[r] <= e
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (rowptr[mid] <= e) lo = mid;
          else hi = mid;
        }
        r = lo;
      }
    }
  };
  f4 yr[U][NC];  // 16 bytes of every edge's row and chunk
  auto load_y = [&](const int (&j)[U]) {
    uint32_t at[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int cl = column(k);
      at[k] = cl < n ? (uint32_t)(TAIL ? min(cl, n - 4) : cl) * (YBF ? 2u : 4u) : kOut;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t base = __umul24(min((uint32_t)j[u], (uint32_t)y_rows), ystride);
#pragma unroll
      for (int k = 0; k < NC; ++k)
        yr[u][k] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(yb, base + at[k], 0, 0));
    }
  };
  // X chunk k (its XV vectors) . Y chunk k of edge u: chains of four products,
  // the chains added in pairs (the kernel above, whose lanes have one chain each
  // at these widths, rounds as often; one chain of all a lane's products raised
  // the error at N = 128 from 7.3e-8 to 7.7e-8)
  auto dot = [&](int u, int k, const f4(&xv)[XV]) {
    float part[XV];
    if constexpr (YBF) {
#pragma unroll
      for (int v = 0; v < XV; ++v)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t two = __float_as_uint(yr[u][k][2 * v + i]);
          const float lo = __uint_as_float(two << 16), hi = __uint_as_float(two & 0xffff0000u);
          part[v] = i ? fmaf(xv[v][2], lo, part[v]) : xv[v][0] * lo;
          part[v] = fmaf(xv[v][2 * i + 1], hi, part[v]);
        }
      return part[0] + part[1];
    } else {
      const int at = column(k);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool own = !TAIL || min(at, n - 4) + i >= at;
        const float xi = own ? xv[0][i] : 0.f, yi = own ? yr[u][k][i] : 0.f;
        part[0] = i ? fmaf(xi, yi, part[0]) : xi * yi;
      }
      return part[0];
    }
  };
  // X of one row through memory (blocks that span many rows)
  auto dot_row = [&](int u, int row) {
    float sum = 0.f;
    const uint32_t base = __umul24(min((uint32_t)row, (uint32_t)M), xstride);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int at = column(k);
      const uint32_t o = at < n ? base + (uint32_t)(TAIL ? min(at, n - 4) : at) * 4u : kOut;
      f4 xv[XV];
#pragma unroll
      for (int v = 0; v < XV; ++v)
        xv[v] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(xb, o + 16 * v, 0, 0));
      sum = k ? sum + dot(u, k, xv) : dot(u, k, xv);
    }
    return sum;
  };
  // X from LDS: row at float offset ro
  auto dot_lds = [&](int u, int ro) {
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      f4 xv[XV];
      if constexpr (TAIL) {
        const int at = column(k);
        const int from = at < n ? min(at, n - 4) : at;
#pragma unroll
        for (int i = 0; i < 4; ++i) xv[0][i] = xs[ro + from + i];
      } else {
#pragma unroll
        for (int v = 0; v < XV; ++v) xv[v] = *reinterpret_cast<const f4 *>(xs + ro + column(k) + 4 * v);
      }
      sum = k ? sum + dot(u, k, xv) : dot(u, k, xv);
    }
    return sum;
  };
  for (int e0 = first; e0 < last;) {
    int my_col, my_row;
    load_ids(e0, my_col, my_row);
    // Edges (bit e - e0) with both rows: the others read zeros, which an
    // infinity or a NaN on the other side turns into NaN, and get 0 at the store.
    const uint64_t valid = __ballot((unsigned)my_col < (unsigned)y_rows && (unsigned)my_row < (unsigned)M);
    // Edges of this block: up to 64, fewer when their rows do not fit in LDS
    // (a multiple of a step's 4 U; with fewer than one step's, X is read per
    // edge).  Rows never decrease in a valid CSR; a block ends where they do.
    const int r_lo = __builtin_amdgcn_readlane(my_row, 0);
    const int left = min(64, last - e0);
    const int before = __shfl_up(my_row, 1, 64);  // lane 0: its own row
    const bool fits = lane < left && my_row >= before && my_row - r_lo < kRows;
    const uint64_t misfits = ~__ballot(fits) & (left == 64 ? ~0ull : (1ull << left) - 1);
    const int fit = misfits ? (int)__builtin_ctzll(misfits) : left;
    const bool staged = r_lo >= 0 && (fit == left || fit >= 4 * U);
    const int count = staged && fit < left ? fit / (4 * U) * (4 * U) : left;
    // edges per lane group: lane group g takes edges [g per, (g + 1) per)
    const int per = count == left ? 16 : count / 4;
    if (per != 16) {
      const int from = (lane >> 4) * per + (lane & 15);
      my_col = __shfl(my_col, from, 64);
      my_row = __shfl(my_row, from, 64);
    }
    if (staged) {
      const int r_hi = __builtin_amdgcn_readlane(my_row, (count - 1) / per * 16 + (count - 1) % per);
      const int need = (r_hi - r_lo + 1) * (XC / 4);  // vectors
      wave_lds_sync();  // the previous rows are read
#pragma unroll 1
      for (int i0 = 0; i0 < need; i0 += 128) {  // two vectors per lane and round
        f4 v[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int i = i0 + 64 * q + lane;
          const int rr = i / (XC / 4), cl = i % (XC / 4) * 4;
          const uint32_t base = __umul24(min((uint32_t)(r_lo + rr), (uint32_t)M), xstride);
          if constexpr (TAIL) {
#pragma unroll
            for (int w = 0; w < 4; ++w)
              v[q][w] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                  xb, cl + w < n ? base + (uint32_t)(cl + w) * 4u : kOut, 0, 0));
          } else {
            v[q] = __builtin_bit_cast(
                f4, __builtin_amdgcn_raw_buffer_load_b128(xb, cl < n ? base + (uint32_t)cl * 4u : kOut, 0, 0));
          }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
          if (i0 + 64 * q + lane < kSddmmLds / 4) *reinterpret_cast<f4 *>(xs + (i0 + 64 * q + lane) * 4) = v[q];
      }
      wave_lds_sync();
    }
    // Step s takes lanes U s .. U s + U - 1 of every 16-lane row, broadcast from
    // lanes 0 .. U - 1 after s rotations (a rolled loop: unrolled, the
    // compiler holds all sixteen edges' broadcasts in registers).
#pragma unroll 1
    for (int s = 0; U * s < per; ++s) {
      int j[U], r[U];
#define DTC_BCAST(u)                                                                 \
  if constexpr (u < U) {                                                              \
    j[u] = __builtin_amdgcn_update_dpp(0, my_col, kDppBcast + u, 0xf, 0xf, true);     \
    r[u] = __builtin_amdgcn_update_dpp(0, my_row, kDppBcast + u, 0xf, 0xf, true);     \
  }
      DTC_BCAST(0) DTC_BCAST(1) DTC_BCAST(2) DTC_BCAST(3)
      DTC_BCAST(4) DTC_BCAST(5) DTC_BCAST(6) DTC_BCAST(7)
#undef DTC_BCAST
      my_col = __builtin_amdgcn_update_dpp(0, my_col, kDppRor + 16 - U, 0xf, 0xf, true);
      my_row = __builtin_amdgcn_update_dpp(0, my_row, kDppRor + 16 - U, 0xf, 0xf, true);
      float p[U];
      load_y(j);
      if (staged) {
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = dot_lds(u, max(r[u] - r_lo, 0) * XC);  // (-1: no edge)
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = dot_row(u, r[u]);
      }
      // Halving exchanges with lanes c ^ 8, c ^ 7 and c ^ 2 while there are
      // sums to halve, then plain ones: lane c ends with edge c / (16 / U).
      const bool b3 = c & 8, b2 = c & 4, b1 = c & 2;
#pragma unroll
      for (int u = 0; u < U / 2; ++u)
        p[u] = (b3 ? p[u + U / 2] : p[u]) + dpp_f32<kDppRor8>(b3 ? p[u] : p[u + U / 2]);
      if constexpr (U >= 4) {
#pragma unroll
        for (int u = 0; u < U / 4; ++u)
          p[u] = (b2 ? p[u + U / 4] : p[u]) + dpp_f32<kDppHalfMirror>(b2 ? p[u] : p[u + U / 4]);
      } else {
        p[0] += dpp_f32<kDppHalfMirror>(p[0]);
      }
      if constexpr (U == 8) p[0] = (b1 ? p[1] : p[0]) + dpp_f32<kDppXor2>(b1 ? p[0] : p[1]);
      else p[0] += dpp_f32<kDppXor2>(p[0]);
      const float v = p[0] + dpp_f32<kDppXor1>(p[0]);
      const int eo = (lane >> 4) * per + U * s + c / (16 / U);
      if (c % (16 / U) == 0 && eo < count) out[e0 + eo] = (valid >> eo) & 1 ? v : 0.f;
    }
    e0 += count;
  }
}

__global__ void k_zero_f32(float *p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0.f;
}

__global__ __launch_bounds__(256) void k_gather(const float *in, const int32_t *idx,
                                                int32_t count, float *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) out[i] = in[idx[i]];
}

}  // namespace
}  // namespace dtc

using namespace dtc;

extern "C" {

dtc_status_t dtc_csr_transpose_workspace_size(int32_t num_rows, int32_t num_cols, int32_t nnz,
                                              size_t *bytes) {
  clear_error();
  if (!bytes) return fail(DTC_ERROR_INVALID_VALUE, "bytes is NULL");
  if (num_rows < 0 || num_cols < 0 || nnz < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "sizes must be >= 0");
  *bytes = transpose_workspace_bytes(nnz);
  return DTC_SUCCESS;
}

dtc_status_t dtc_csr_transpose(const int32_t *node_pointer, const int32_t *edge_list,
                               int32_t num_rows, int32_t num_cols, int32_t nnz,
                               int32_t *node_pointer_t, int32_t *edge_list_t, int32_t *perm,
                               void *workspace, size_t workspace_bytes, dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (num_rows < 0 || num_cols < 0 || nnz < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "sizes must be >= 0");
  if (!node_pointer || !node_pointer_t)
    return fail(DTC_ERROR_INVALID_VALUE, "row pointers are required");
  if (nnz > 0 && (!edge_list || !edge_list_t || !perm))
    return fail(DTC_ERROR_INVALID_VALUE, "edge arrays are required when nnz > 0");
  const size_t need = transpose_workspace_bytes(nnz);
  if (!workspace || workspace_bytes < need)
    return fail(DTC_ERROR_WORKSPACE, "transpose workspace needs " + std::to_string(need) + " bytes");
  return transpose_edges(node_pointer, edge_list, num_rows, num_cols, nnz, node_pointer_t,
                         edge_list_t, perm, workspace, stream);
}

dtc_status_t dtc_sddmm_csr(const int32_t *node_pointer, const int32_t *edge_list,
                           const int32_t *edge_to_row, int32_t num_rows, int32_t nnz,
                           const float *x, const void *y, int32_t y_dtype, int32_t y_rows,
                           int32_t n, float *out, dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (num_rows < 0 || nnz < 0 || y_rows < 0 || n <= 0)
    return fail(DTC_ERROR_INVALID_VALUE, "sizes must be >= 0 and N >= 1");
  if (y_dtype != DTC_B_FLOAT32 && y_dtype != DTC_B_BFLOAT16)
    return fail(DTC_ERROR_INVALID_VALUE, "y_dtype must be DTC_B_FLOAT32 or DTC_B_BFLOAT16");
  if (!node_pointer) return fail(DTC_ERROR_INVALID_VALUE, "node_pointer is NULL");
  if (nnz == 0 || num_rows == 0) return DTC_SUCCESS;
  if (!edge_list || !x || !y || !out) return fail(DTC_ERROR_INVALID_VALUE, "NULL argument");
  if (y_rows == 0) {  // every column is out of range: all zeros
    k_zero_f32<<<(unsigned)std::min<int64_t>(4096, ceil_div(nnz, 256)), 256, 0, stream>>>(out, nnz);
    DTC_LAUNCH_CHECK("zero");
    return DTC_SUCCESS;
  }
  const bool ybf = y_dtype == DTC_B_BFLOAT16;
  const int64_t lim = (int64_t)1 << 31;
  const bool buffers = ((int64_t)num_rows + 1) * n * 4 < lim && ((int64_t)y_rows + 1) * n * 4 < lim &&
                       num_rows < (1 << 24) - 1 && y_rows < (1 << 24) - 1 && n < (1 << 22);
  // Up to 192 float32 or 256 bf16 columns.  At 256 float32 columns the kernel
  // above, whose 64 lanes read whole 1 KB rows, is ahead where Y misses the
  // caches (R-MAT 2^18 764 against 847 us) and behind where it does not (block
  // model 60,000 566 against 430): it keeps the wide rows, the bf16 widths that
  // are no multiple of 8, and operands beyond 2 GiB.
  if (buffers && (ybf ? n % 8 == 0 && n <= 256 && (uintptr_t)y % 16 == 0 : n >= 4 && n <= 192)) {
    const unsigned grid = (unsigned)ceil_div(nnz, 256);
    const int chunks = (int)ceil_div(n, ybf ? 128 : 64);
    auto launch = [&](auto kernel) {
      kernel<<<grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_row, num_rows, nnz, x, y, y_rows, n, out);
    };
    if (ybf) chunks == 1 ? launch(k_sddmm_groups<1, true, false>) : launch(k_sddmm_groups<2, true, false>);
    else if (n % 4)
      chunks == 1   ? launch(k_sddmm_groups<1, false, true>)
      : chunks == 2 ? launch(k_sddmm_groups<2, false, true>)
                    : launch(k_sddmm_groups<3, false, true>);
    else
      chunks == 1   ? launch(k_sddmm_groups<1, false, false>)
      : chunks == 2 ? launch(k_sddmm_groups<2, false, false>)
                    : launch(k_sddmm_groups<3, false, false>);
    DTC_LAUNCH_CHECK("sddmm_groups");
    return DTC_SUCCESS;
  }
  const int64_t groups = ceil_div(nnz, kSddmmEdges);
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(1 << 16, ceil_div(groups, 4)));
  const bool v4 = n % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)y % (ybf ? 8 : 16) == 0;
  if (v4 && ybf)
    k_sddmm<4, true><<<grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_row, num_rows, nnz,
                                               x, y, y_rows, n, out);
  else if (v4)
    k_sddmm<4, false><<<grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_row, num_rows, nnz,
                                                x, y, y_rows, n, out);
  else if (ybf)
    k_sddmm<1, true><<<grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_row, num_rows, nnz,
                                               x, y, y_rows, n, out);
  else
    k_sddmm<1, false><<<grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_row, num_rows, nnz,
                                                x, y, y_rows, n, out);
  DTC_LAUNCH_CHECK("sddmm");
  return DTC_SUCCESS;
}

dtc_status_t dtc_gather_f32(const float *in, const int32_t *idx, int32_t count, float *out,
                            dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (count < 0) return fail(DTC_ERROR_INVALID_VALUE, "count must be >= 0");
  if (count == 0) return DTC_SUCCESS;
  if (!in || !idx || !out) return fail(DTC_ERROR_INVALID_VALUE, "NULL argument");
  k_gather<<<(unsigned)ceil_div(count, 256), 256, 0, stream>>>(in, idx, count, out);
  DTC_LAUNCH_CHECK("gather");
  return DTC_SUCCESS;
}

}  // extern "C"
