// ME-TCF SpMM on gfx950: C = A * B with A in 16 x 8 TC blocks.
//
// Work decomposition (one wavefront = one work unit, 4 waves per workgroup):
//   unit = (run of TC blocks, column tile of 16*VEC*NSUB output columns).
//   The unbalanced schedule uses one whole window per unit
//   (DTCSpMM_kernel.cu:811-944 launches one CTA per window); the balanced
//   schedule cuts the TC-block list into fixed chunks, each unit walking the
//   windows that start in its chunk and flushing on every window change, with
//   windows longer than a chunk cut and merged atomically
//   (DTCSpMM_kernel.cu:4730-4901 walks 64-block chunks and flushes on a
//   window change).
//
// Inner loop: 4 consecutive TC blocks of the window form one K = 32 group,
// which is exactly the K of v_mfma_f32_16x16x32_{bf16,f16}.  Lane l works on
// block g = l / 16 of the group and MFMA column q = l % 16:
//   * B operand: the lane gathers the 8 rows SparseAToX[8*(bb+g) + j] of B,
//     VEC consecutive floats each at column tile + q*VEC (one 16-lane group
//     reads 16*VEC*4 contiguous bytes of a row);
//   * A operand: the lane needs A_g[q][0..7], read from a per-wave LDS tile
//     built by scattering the stored values at their tile ids;
//   * C: lane l holds rows 4*(l/16) + i, i < 4, of its MFMA column, i.e. the
//     output columns tile + q*VEC + v for the v-th MFMA.
// What bounds it: the row gathers (the gather-only kernel of probe_gather.hip
// takes 3.24 of 3.73 ms on the 2^20-node R-MAT at N = 256, chunk 256 and 32-column
// tiles, 3.53 of 4.41 on the 232,965-row block model at N = 128, chunk 256 and
// 64-column tiles), then the float32 MFMAs, which do 16-row work on columns of
// one or two entries.  So the loop is built to leave one exposed latency per
// group, the gathers' own, few vector instructions around them, and five waves
// per SIMD to overlap one wave's MFMAs with the others' gathers (a second group
// in flight per wave at three to four waves per SIMD measured 10-35% slower).
// For FP32 the same group is fed as 8 steps of v_mfma_f32_16x16x4_f32 where
// step j pairs A_g[:, j] with B row j of block g.  The k order inside a
// group is a permutation shared by A and B, so every mapping sums the same
// products.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "dtc_internal.h"

// Workspace of dtc_spmm_balanced_noalloc, for callers that cannot allocate:
// a fixed device array, one copy per GPU, held until the process ends.  Host
// code never uses this name as an address (on the host it is a stand-in
// symbol); the device address comes from hipGetSymbolAddress, per device.
constexpr size_t kNoAllocScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace dtc {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr int kBlkH = 16;
constexpr int kBlkW = 8;
constexpr int kGroup = 4;                        // TC blocks per K=32 group
constexpr int kTileFloats = kGroup * kBlkH * kBlkW;  // 512

// Per-wave LDS floats of a kernel instance: the A tiles of one group, or the
// 16-row output tile of one window while it is merged with atomics.
template <int VEC, int NSUB>
constexpr int wave_lds_floats() {
  return kBlkH * 16 * VEC * NSUB > kTileFloats ? kBlkH * 16 * VEC * NSUB : kTileFloats;
}
// ... followed by 4 words of wave state (the balanced chunk index for the
// deterministic merge), kept in LDS rather than in registers: the flush
// that reads it runs at the walk loop's register peak.
template <int VEC, int NSUB>
constexpr int wave_lds_words() {
  return wave_lds_floats<VEC, NSUB>() + 4;
}
constexpr int kWavesPerBlock = 4;

struct SpmmParams {
  const int32_t *rwo;    // unbalanced: row window offsets [W + 1]
  const int32_t *rowid;  // balanced: window of every TC block [T]
  const uint8_t *tile;
  const int32_t *off;
  const int32_t *atox;
  const float *vals;  // TC-block order, NULL = all ones
  const void *B;      // float32, or bf16 for the bf16-B schemes
  float *C;
  int32_t num_windows;
  int32_t num_blocks;
  int32_t M;
  int32_t b_rows;
  int32_t N;
  int32_t nnz;         // entries of tile / vals
  int32_t n_ct;        // column tiles
  int32_t num_items;   // windows (unbalanced) or chunks (balanced)
  int32_t chunk;       // balanced: chunk length in TC blocks; unbalanced: windows per unit
  int32_t *queue;      // persistent work counter
  const int2 *runs;    // balanced: run [b, e) of every chunk, cut flags in the sign bits
  float *parts;        // balanced, deterministic merge: partial-tile slots (NULL: atomics)
  int32_t span;        // balanced cut span in TC blocks (a multiple of chunk)
  int32_t long_blocks; // unbalanced: windows of more blocks are shared out to the workgroup
  int32_t groups;      // workgroups per column tile
  int32_t long_groups; // unbalanced, tiles in turn: those of the part that takes the long windows
};

// Kernels take the arrays as restrict-qualified arguments: the compiler may
// then read the wave-uniform ones (block offsets, window ids) through the
// scalar cache, whose waits do not queue behind the B gathers.
#define SPMM_KERNEL_ARGS                                                                   \
  const int32_t *__restrict__ a_rwo, const int32_t *__restrict__ a_rowid,                  \
      const uint8_t *__restrict__ a_tile, const int32_t *__restrict__ a_off,               \
      const int32_t *__restrict__ a_atox, const float *__restrict__ a_vals,                \
      const void *__restrict__ a_B, float *__restrict__ a_C, SpmmParams a_p
#define SPMM_PARAMS_FROM_ARGS                                                              \
  SpmmParams {                                                                             \
    a_rwo, a_rowid, a_tile, a_off, a_atox, a_vals, a_B, a_C, a_p.num_windows,              \
        a_p.num_blocks, a_p.M, a_p.b_rows, a_p.N, a_p.nnz, a_p.n_ct, a_p.num_items,        \
        a_p.chunk, a_p.queue, a_p.runs, a_p.parts, a_p.span,                               \
        a_p.long_blocks, a_p.groups, a_p.long_groups                                       \
  }

template <int VEC>
struct VecType {
  typedef float type __attribute__((ext_vector_type(VEC)));
};
template <>
struct VecType<1> {
  typedef float type;
};

template <int VEC>
__device__ __forceinline__ float comp(const typename VecType<VEC>::type &x, int v) {
  if constexpr (VEC == 1) return x;
  else return x[v];
}

template <int VEC>
__device__ __forceinline__ typename VecType<VEC>::type vzero() {
  typename VecType<VEC>::type z;
  if constexpr (VEC == 1) z = 0.f;
  else
#pragma unroll
    for (int v = 0; v < VEC; ++v) z[v] = 0.f;
  return z;
}

// Schemes for B stored as bf16 (values taken exactly): A enters as three
// bf16 limbs (A3) or as one (A1); accumulation is float32 either way.
constexpr int kBf16B_A3 = 16;
constexpr int kBf16B_A1 = 17;
template <int PREC>
constexpr bool is_bf16b() {
  return PREC == kBf16B_A3 || PREC == kBf16B_A1;
}

template <int VEC>
struct BfVec {
  typedef __bf16 type __attribute__((ext_vector_type(VEC)));
};

// Register type of one lane's slice of one gathered B row.
template <int PREC, int VEC>
using breg_t = typename std::conditional<is_bf16b<PREC>(), typename BfVec<VEC>::type,
                                         typename VecType<VEC>::type>::type;

__device__ __forceinline__ float bf16_to_f32(__bf16 x) { return (float)x; }

// Limb split of x into bf16 terms, x = l0 + l1 (+ l2) + residual.
__device__ __forceinline__ void split2(float x, __bf16 &h, __bf16 &l) {
  h = (__bf16)x;
  l = (__bf16)(x - bf16_to_f32(h));
}
__device__ __forceinline__ void split3(float x, __bf16 &h, __bf16 &m, __bf16 &l) {
  h = (__bf16)x;
  const float r1 = x - bf16_to_f32(h);
  m = (__bf16)r1;
  l = (__bf16)(r1 - bf16_to_f32(m));
}

#define MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32((a), (b), (c), 0, 0, 0)
#define MFMA_BF16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16((a), (b), (c), 0, 0, 0)
#define MFMA_F16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_f16((a), (b), (c), 0, 0, 0)

// acc[s][v] += A_group * B_group for the columns of subtile s, component v.
template <int PREC, int VEC, int NSUB>
__device__ __forceinline__ void mfma_group(const float (&a)[8], const breg_t<PREC, VEC> (&breg)[NSUB][8],
                                           floatx4 (&acc)[NSUB][VEC], bool has_vals) {
  if constexpr (is_bf16b<PREC>()) {
    bf16x8 A0, A1, A2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __bf16 h, m, l;
      split3(a[j], h, m, l);
      A0[j] = h;
      A1[j] = m;
      A2[j] = l;
    }
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        bf16x8 Bv;
#pragma unroll
        for (int j = 0; j < 8; ++j) Bv[j] = breg[s][j][v];
        floatx4 c = acc[s][v];
        if (PREC == kBf16B_A3 && has_vals) {
          c = MFMA_BF16(A2, Bv, c);
          c = MFMA_BF16(A1, Bv, c);
        }
        acc[s][v] = MFMA_BF16(A0, Bv, c);
      }
  } else if constexpr (PREC == DTC_PRECISION_FP32) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int s = 0; s < NSUB; ++s)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[s][v] = MFMA_F32(a[j], comp<VEC>(breg[s][j], v), acc[s][v]);
  } else if constexpr (PREC == DTC_PRECISION_BF16) {
    bf16x8 A;
#pragma unroll
    for (int j = 0; j < 8; ++j) A[j] = (__bf16)a[j];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        bf16x8 Bv;
#pragma unroll
        for (int j = 0; j < 8; ++j) Bv[j] = (__bf16)comp<VEC>(breg[s][j], v);
        acc[s][v] = MFMA_BF16(A, Bv, acc[s][v]);
      }
  } else if constexpr (PREC == DTC_PRECISION_FP16) {
    halfx8 A;
#pragma unroll
    for (int j = 0; j < 8; ++j) A[j] = (_Float16)a[j];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        halfx8 Bv;
#pragma unroll
        for (int j = 0; j < 8; ++j) Bv[j] = (_Float16)comp<VEC>(breg[s][j], v);
        acc[s][v] = MFMA_F16(A, Bv, acc[s][v]);
      }
  } else if constexpr (PREC == DTC_PRECISION_BF16X3) {
    bf16x8 Ah, Al;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __bf16 h, l;
      split2(a[j], h, l);
      Ah[j] = h;
      Al[j] = l;
    }
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        bf16x8 Bh, Bl;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          __bf16 h, l;
          split2(comp<VEC>(breg[s][j], v), h, l);
          Bh[j] = h;
          Bl[j] = l;
        }
        floatx4 c = acc[s][v];
        if (has_vals) c = MFMA_BF16(Al, Bh, c);
        c = MFMA_BF16(Ah, Bl, c);
        c = MFMA_BF16(Ah, Bh, c);
        acc[s][v] = c;
      }
  } else {  // DTC_PRECISION_BF16X6
    bf16x8 A0, A1, A2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __bf16 h, m, l;
      split3(a[j], h, m, l);
      A0[j] = h;
      A1[j] = m;
      A2[j] = l;
    }
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        bf16x8 B0, B1, B2;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          __bf16 h, m, l;
          split3(comp<VEC>(breg[s][j], v), h, m, l);
          B0[j] = h;
          B1[j] = m;
          B2[j] = l;
        }
        floatx4 c = acc[s][v];
        if (has_vals) {
          c = MFMA_BF16(A2, B0, c);
          c = MFMA_BF16(A1, B1, c);
        }
        c = MFMA_BF16(A0, B2, c);
        if (has_vals) c = MFMA_BF16(A1, B0, c);
        c = MFMA_BF16(A0, B1, c);
        c = MFMA_BF16(A0, B0, c);
        acc[s][v] = c;
      }
  }
}

// Columns of this lane in every subtile: VEC consecutive ones from c[s].  The
// last tile's lanes past N - VEC are moved back so that every vector lies
// inside a row of B and C: they recompute (and store again, bit for bit) the
// columns of their neighbours, no load or store needs a mask, and N need not
// be a multiple of VEC (only N >= VEC).
template <int NSUB>
struct Cols {
  int c[NSUB];
};
template <int VEC, int NSUB>
__device__ __forceinline__ Cols<NSUB> lane_cols(int ct, int N) {
  Cols<NSUB> o;
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
    o.c[s] = min(ct * (16 * VEC * NSUB) + s * 16 * VEC + (lane_id() & 15) * VEC, N - VEC);
  return o;
}

// The arrays a wave reads, as buffer resources (WIDE = false): 32-bit byte
// offsets, one vector instruction per address, and loads past an array's
// end return zero, so the loop carries no 64-bit address arithmetic and no
// masks.  The host takes this form when every array is below 2 GiB and B
// has fewer than 2^24 rows of fewer than 2^24 bytes (fits_buffers); larger
// operands take 64-bit pointers (WIDE = true).
template <bool WIDE>
struct Bufs {};
template <>
struct Bufs<false> {
  __amdgpu_buffer_rsrc_t tile, vals, atox, b;
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buf(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
template <int PREC, bool WIDE, bool DENSE>
__device__ __forceinline__ Bufs<WIDE> make_bufs(const SpmmParams &p) {
  Bufs<WIDE> o;
  if constexpr (!WIDE) {
    constexpr uint32_t esz = is_bf16b<PREC>() ? 2 : 4;
    // whole 4-element vectors (kDense; the host checks their alignment, so the
    // last one lies in the same 16 bytes as an element of the array)
    const uint32_t n4 = ((uint32_t)p.nnz + 3u) & ~3u;
    o.tile = make_buf(p.tile, DENSE ? n4 : (uint32_t)p.nnz);
    o.vals = make_buf(p.vals, p.vals ? (DENSE ? n4 : (uint32_t)p.nnz) * 4u : 0u);
    o.atox = make_buf(p.atox, (uint32_t)p.num_blocks * (kBlkW * 4u));
    o.b = make_buf(p.B, (uint32_t)p.b_rows * ((uint32_t)p.N * esz));
  }
  return o;
}

// Block data of 64 consecutive blocks from sb, lane l holding block sb + l.
// Groups starting in the first kStageBlocks of them find their (up to 4)
// blocks and the following block's offset inside the stage.
constexpr int kStageBlocks = 56;
struct Stage {
  int sb;
  int off;  // TCblock_offset, clamped to the stored elements
  int wid;  // balanced schedule: window id, -1 at or past the run's end
};

template <bool BALANCED>
__device__ __forceinline__ Stage load_stage(const SpmmParams &p, int sb, int e) {
  Stage s;
  s.sb = sb;
  const int i = sb + lane_id();
  s.off = p.off[min(i, p.num_blocks)];
  s.wid = BALANCED && i < e ? p.rowid[i] : -1;
  return s;
}

// How the blocks are shared out (walk_blocks).
constexpr int kWindows = 0, kBalanced = 1, kSplit = 2;

// How a kernel reads its operands.
constexpr int kPtr = 0;    // 64-bit pointers (operands of any size)
constexpr int kBuf = 1;    // buffers, one element per lane
constexpr int kDense = 2;  // buffers, four consecutive elements per lane

// One K = 32 group: its wave-uniform position, and the per-lane metadata
// loaded one group ahead of its use.
struct Group {
  int bb;          // first block
  int nblk;        // blocks (1 .. 4)
  int w;           // window
  int o0, o1, o2, o3, o4;  // element offsets of its blocks; o4: its end
  int4 r0, r1;     // SparseAToX of block bb + lane / 16
  // Tile ids and values of the group's first elements.  Plain: elements
  // o0 + lane and o0 + 64 + lane (the second 64 are loaded only for groups
  // that have them).  Dense: elements (o0 & ~3) + 4 lane + k in byte k of
  // tile and in v<k>.
  int tile, tile2;
  float v0, v1, v2, v3;
};

// Loads of a group's metadata.  They are issued before the previous group's
// gathers and used after them, so their latency is never on the wave's path.
template <int MODE>
__device__ __forceinline__ void load_rows(const SpmmParams &p, const Bufs<MODE == kPtr> &bufs, Group &m) {
  const int blk = m.bb + (lane_id() >> 4);
  if constexpr (MODE == kPtr) {
    const int4 *ap = reinterpret_cast<const int4 *>(p.atox + (int64_t)min(blk, p.num_blocks - 1) * kBlkW);
    m.r0 = ap[0];
    m.r1 = ap[1];
  } else {
    const uint32_t ao = (uint32_t)blk * (kBlkW * 4u);
    m.r0 = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(bufs.atox, ao, 0, 0));
    m.r1 = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(bufs.atox, ao + 16, 0, 0));
  }
}

template <int MODE>
__device__ __forceinline__ void load_elems(const SpmmParams &p, const Bufs<MODE == kPtr> &bufs, bool has_vals,
                                           Group &m) {
  const int lane = lane_id();
  m.v0 = m.v1 = 1.0f;
  if constexpr (MODE == kDense) {
    m.v2 = m.v3 = 1.0f;
    const uint32_t e = (uint32_t)(m.o0 & ~3) + 4u * (uint32_t)lane;
    m.tile = (int)__builtin_amdgcn_raw_buffer_load_b32(bufs.tile, e, 0, 0);
    if (has_vals) {
      const floatx4 v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(bufs.vals, e * 4, 0, 0));
      m.v0 = v[0];
      m.v1 = v[1];
      m.v2 = v[2];
      m.v3 = v[3];
    }
  } else if constexpr (MODE == kBuf) {
    const uint32_t e = (uint32_t)(m.o0 + lane);
    m.tile = __builtin_amdgcn_raw_buffer_load_b8(bufs.tile, e, 0, 0);
    if (has_vals) m.v0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bufs.vals, e * 4, 0, 0));
    if (m.o4 - m.o0 > kWave) {
      m.tile2 = __builtin_amdgcn_raw_buffer_load_b8(bufs.tile, e + kWave, 0, 0);
      if (has_vals)
        m.v1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bufs.vals, (e + kWave) * 4, 0, 0));
    }
  } else {
    const int last = p.nnz - 1;
    const int e = m.o0 < p.nnz - lane ? m.o0 + lane : last;
    m.tile = p.tile[e];
    if (has_vals) m.v0 = p.vals[e];
    if (m.o4 - m.o0 > kWave) {
      const int e2 = e < p.nnz - kWave ? e + kWave : last;
      m.tile2 = p.tile[e2];
      if (has_vals) m.v1 = p.vals[e2];
    }
  }
}

template <int PREC, int VEC>
struct BElem {
  typedef typename std::conditional<is_bf16b<PREC>(), __bf16, float>::type type;
  // a row's vector: aligned to its element only (any N)
  typedef breg_t<PREC, VEC> type_u __attribute__((aligned(is_bf16b<PREC>() ? 8 : 4)));
};

// This lane's 8 rows of B through 64-bit pointers: loads from clamped
// addresses, zero where the row is not one of B's (or ok is false).
template <int PREC, int VEC, int NSUB>
__device__ __forceinline__ void gather_ptr(const SpmmParams &p, const int (&rows)[8], bool ok,
                                           const Cols<NSUB> &cols,
                                           breg_t<PREC, VEC> (&breg)[NSUB][8]) {
  typedef breg_t<PREC, VEC> vt;
  typedef typename BElem<PREC, VEC>::type et;
  const et *B = static_cast<const et *>(p.B);
  vt zero;
  if constexpr (VEC == 1) zero = (et)0.f;
  else
#pragma unroll
    for (int v = 0; v < VEC; ++v) zero[v] = (et)0.f;
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = ok && (unsigned)rows[j] < (unsigned)p.b_rows;
      const vt v = *reinterpret_cast<const typename BElem<PREC, VEC>::type_u *>(
          B + (int64_t)(in ? rows[j] : 0) * p.N + cols.c[s]);
      breg[s][j] = in ? v : zero;
    }
}

// B rows of the group into registers.  Lanes whose block lies past the group,
// and slots whose row is not one of B's, get zeros: through buffers, from
// byte offsets past B's end (its size is below 2^31).
template <int PREC, int VEC, int NSUB, bool WIDE>
__device__ __forceinline__ void gather_b(const SpmmParams &p, const Bufs<WIDE> &bufs, const Group &m,
                                         const Cols<NSUB> &cols, breg_t<PREC, VEC> (&breg)[NSUB][8]) {
  typedef breg_t<PREC, VEC> vt;
  const int rows[8] = {m.r0.x, m.r0.y, m.r0.z, m.r0.w, m.r1.x, m.r1.y, m.r1.z, m.r1.w};
  const bool ok = (lane_id() >> 4) < m.nblk;
  if constexpr (WIDE) {
    gather_ptr<PREC, VEC, NSUB>(p, rows, ok, cols, breg);
  } else {
    constexpr uint32_t esz = is_bf16b<PREC>() ? 2 : 4;
    const uint32_t stride = (uint32_t)p.N * esz;
    uint32_t base[NSUB];
#pragma unroll
    for (int s = 0; s < NSUB; ++s) base[s] = ok ? (uint32_t)cols.c[s] * esz : 0x80000000u;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t r = __umul24(min((uint32_t)rows[j], (uint32_t)p.b_rows), stride);
#pragma unroll
      for (int s = 0; s < NSUB; ++s) {
        const uint32_t o = r + base[s];
        constexpr int bytes = VEC * (int)esz;
        if constexpr (bytes == 16)
          breg[s][j] = __builtin_bit_cast(vt, __builtin_amdgcn_raw_buffer_load_b128(bufs.b, o, 0, 0));
        else if constexpr (bytes == 8)
          breg[s][j] = __builtin_bit_cast(vt, __builtin_amdgcn_raw_buffer_load_b64(bufs.b, o, 0, 0));
        else
          breg[s][j] = __builtin_bit_cast(vt, __builtin_amdgcn_raw_buffer_load_b32(bufs.b, o, 0, 0));
      }
    }
  }
}

// Dense 16x8 A tiles of the group in this wave's LDS, then this lane's
// operand A_g[q][0..7].  Element (block gg, row, slot) lies at float
// (slot / 4) * 256 + (16 gg + row) * 4 + slot % 4: lane 16 gg + row reads its
// two float4 with consecutive lanes on consecutive addresses (no bank
// conflicts).  Stored elements are added (LDS float atomics): a CSR with a
// repeated (row, column) pair puts several elements on one tile id, and the
// product must count each of them, as the CSR product does.
template <int MODE>
__device__ __forceinline__ void build_a(const SpmmParams &p, const Bufs<MODE == kPtr> &bufs, const Group &m,
                                        bool has_vals, float *lds, float (&a)[8]) {
  const int lane = lane_id();
  floatx4 *t4 = reinterpret_cast<floatx4 *>(lds);
  const floatx4 z4 = {0.f, 0.f, 0.f, 0.f};
  t4[lane] = z4;
  t4[kWave + lane] = z4;
  wave_lds_sync();
  auto add = [&](int e, int t, float v) {
    const int gg = (e >= m.o1) + (e >= m.o2) + (e >= m.o3);
    atomicAdd(&lds[((t & 4) << 6) | (gg << 6) | (((t >> 3) & 15) << 2) | (t & 3)], v);
  };
  if constexpr (MODE == kDense) {
    int e = (m.o0 & ~3) + 4 * lane;
    auto add4 = [&](int t, float v0, float v1, float v2, float v3) {
      if (e >= m.o0 && e < m.o4) add(e, t, v0);
      if (e + 1 >= m.o0 && e + 1 < m.o4) add(e + 1, t >> 8, v1);
      if (e + 2 >= m.o0 && e + 2 < m.o4) add(e + 2, t >> 16, v2);
      if (e + 3 < m.o4) add(e + 3, t >> 24, v3);
    };
    add4(m.tile, m.v0, m.v1, m.v2, m.v3);
    for (int first = (m.o0 & ~3) + 4 * kWave; first < m.o4; first += 4 * kWave) {  // more than 253 elements
      e += 4 * kWave;
      const int t = (int)__builtin_amdgcn_raw_buffer_load_b32(bufs.tile, (uint32_t)e, 0, 0);
      floatx4 v = {1.f, 1.f, 1.f, 1.f};
      if (has_vals)
        v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(bufs.vals, (uint32_t)e * 4u, 0, 0));
      add4(t, v[0], v[1], v[2], v[3]);
    }
  } else {
    int e = m.o0 + lane;
    if (e < m.o4) add(e, m.tile, m.v0);
    if (m.o4 - m.o0 > kWave) {
      e += kWave;
      if (e < m.o4) add(e, m.tile2, m.v1);
      for (e += kWave; e < m.o4; e += kWave) add(e, p.tile[e], has_vals ? p.vals[e] : 1.0f);
    }
  }
  wave_lds_sync();
  const floatx4 lo = t4[lane];
  const floatx4 hi = t4[kWave + lane];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    a[j] = lo[j];
    a[j + 4] = hi[j];
  }
  wave_lds_sync();
}

template <int VEC, int NSUB>
__device__ __forceinline__ void zero_acc(floatx4 (&acc)[NSUB][VEC]) {
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[s][v] = floatx4{0.f, 0.f, 0.f, 0.f};
}

// A row's vector in C: aligned to a float only (any N).
template <int VEC>
struct CVec {
  typedef typename VecType<VEC>::type type __attribute__((aligned(4)));
};

// lane_id(), recomputed where it is used: what is derived from it cannot be
// hoisted out of the walk loop, where the rarely run store paths' addresses
// would be held in registers (or scratch) across every group.
__device__ __forceinline__ int lane_here() {
  int lane = lane_id();
  asm volatile("" : "+v"(lane));
  return lane;
}

// First of this lane's four rows of C in window w, at column col.
template <bool WIDE>
__device__ __forceinline__ float *c_rows(const SpmmParams &p, int w, int lane, int col) {
  float *base = p.C + (int64_t)w * kBlkH * p.N;  // wave-uniform
  const int g = lane >> 4;
  if constexpr (WIDE) return base + (int64_t)(4 * g) * p.N + col;
  return reinterpret_cast<float *>(reinterpret_cast<char *>(base) + (uint32_t)(4 * g * p.N + col) * 4u);
}

// Writes the 16 rows of window w held in acc.
template <int VEC, int NSUB, bool WIDE>
__device__ __forceinline__ void store_window(const SpmmParams &p, int w, const Cols<NSUB> &cols,
                                             const floatx4 (&acc)[NSUB][VEC]) {
  typedef typename CVec<VEC>::type vfloat;
  if (w < 0) return;
  const int lane = lane_here();
  const int64_t left = p.M - (int64_t)w * kBlkH - 4 * (lane >> 4);  // rows from this lane's first on
#pragma unroll
  for (int s = 0; s < NSUB; ++s) {
    float *c = c_rows<WIDE>(p, w, lane, cols.c[s]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      vfloat out;
      if constexpr (VEC == 1) out = acc[s][0][i];
      else
#pragma unroll
        for (int v = 0; v < VEC; ++v) out[v] = acc[s][v][i];
      if (i < left) __builtin_nontemporal_store(out, reinterpret_cast<vfloat *>(c + (int64_t)i * p.N));
    }
  }
}

// Zeroes this wave's column tile of windows [w0, w1) (empty windows: no TC
// block writes them, so any wave may, at any time of the launch).
template <int VEC, int NSUB, bool WIDE>
__device__ __forceinline__ void zero_windows(const SpmmParams &p, int w0, int w1, const Cols<NSUB> &cols) {
  typedef typename CVec<VEC>::type vfloat;
  const vfloat z = vzero<VEC>();
  const int lane = lane_here();
#pragma unroll 1
  for (int w = max(w0, 0); w < w1; ++w) {
    const int64_t left = p.M - (int64_t)w * kBlkH - 4 * (lane >> 4);
#pragma unroll 1
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int s = 0; s < NSUB; ++s)
        if (i < left)
          __builtin_nontemporal_store(
              z, reinterpret_cast<vfloat *>(c_rows<WIDE>(p, w, lane, cols.c[s]) + (int64_t)i * p.N));
  }
}

// Adds the 16 rows of window w held in acc to C with atomics, through this
// wave's LDS: the tile is written in the accumulator layout and read back
// row-major, so that each atomic instruction covers 64 consecutive floats of
// a row (or two rows of a 32-column tile) instead of lanes 16 bytes apart
// spread over 4 rows -- a quarter of the cache lines per instruction.
// With the deterministic merge (p.parts set) the row-major tile is stored
// instead, whole, in a partial-tile slot: slot 2 c holds chunk c's share of
// its first window, slot 2 c + 1 of its last (`last_role`), each slot n_ct
// tiles of 16 x TW floats; k_balance_fixup sums them in chunk order.  The
// chunk index is the one run_unit left in the wave's LDS state word.
template <int VEC, int NSUB>
__device__ __forceinline__ void add_window_atomic(const SpmmParams &p, int w, int ct, const Cols<NSUB> &cols,
                                                  float *lds, const floatx4 (&acc)[NSUB][VEC],
                                                  bool last_role) {
  constexpr int TW = 16 * VEC * NSUB;  // tile width in floats
  const int lane = lane_here();
  const int g = lane >> 4;
  const int col0 = ct * TW;  // first column of the tile
#pragma unroll
  for (int s = 0; s < NSUB; ++s) {
    const int lc = cols.c[s] - col0;  // below 0: a moved-back lane's columns of the previous tile
#pragma unroll
    for (int v = 0; v < VEC; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lc + v >= 0) lds[(4 * g + i) * TW + lc + v] = acc[s][v][i];
  }
  wave_lds_sync();
  const int64_t N = p.N;
  if (p.parts) {
    const int item = wave_uniform(reinterpret_cast<const int *>(lds)[wave_lds_floats<VEC, NSUB>()]);
    const int slot = 2 * item + (last_role ? 1 : 0);
    float *dst = p.parts + ((int64_t)slot * p.n_ct + ct) * (kBlkH * TW);
#pragma unroll 1
    for (int k = 0; k < kBlkH * TW / 64; ++k) dst[k * 64 + lane] = lds[k * 64 + lane];
    wave_lds_sync();
    return;
  }
  // Rolled: at most two flushes per chunk take this path, and unrolling it
  // keeps every address live at once (twice the kernel's registers).
#pragma unroll 1
  for (int k = 0; k < kBlkH * TW / 64; ++k) {
    const int e = k * 64 + lane;
    const int r = e / TW;
    const int col = col0 + e % TW;
    const int64_t row = (int64_t)w * kBlkH + r;
    if (row >= 0 && row < p.M && col < p.N) unsafeAtomicAdd(p.C + row * N + col, lds[e]);
  }
  wave_lds_sync();
}

// The blocks of one work unit as ONE software pipeline over K = 32 groups,
// windows and all: groups never cross a window start (they are the groups a
// per-window loop would form), and when a group opens a new window the
// accumulators of the previous one are stored and cleared.
//   Balanced schedule: the blocks [b, e) of a chunk's run.  Window starts
//     come from the stage's window ids (one ballot per stage).  Windows
//     atomic_w0 / atomic_w1 (if >= 0) are merged with atomic adds (windows
//     cut at chunk boundaries), every other window is stored whole.
//   Unbalanced schedule: the windows [w0, w1), at most 63 of them; lane l
//     holds RowWindowOffset[w0 + l].
//   Split schedule: the blocks [b, e) of window w0, left in acc.
// Empty windows are zeroed by the wave that passes them: the gap before the
// unit's first block, the gaps between its windows, and after its last one.
//
// Per group i: the next group's position (scalar, from the stage held in
// registers: no load to wait for), its metadata loads, group i's gathers,
// the previous window's stores if the window changed, group i's A tile, the
// MFMAs.  Loads retire in order, so waiting for the gathers of group i also
// waits for the metadata of group i + 1, which was issued before them: one
// exposed memory latency per group, the gathers' own.
template <int PREC, int VEC, int NSUB, int SCHED, int MODE>
__device__ __forceinline__ void walk_blocks(const SpmmParams &p, int b, int e, int w0, int w1, int rwo,
                                            int ct, float *lds, int atomic_w0, int atomic_w1,
                                            floatx4 (&acc)[NSUB][VEC]) {
  constexpr bool BALANCED = SCHED == kBalanced;
  constexpr bool WIDE = MODE == kPtr;
  const bool has_vals = p.vals != nullptr;
  const Cols<NSUB> cols = lane_cols<VEC, NSUB>(ct, p.N);
  const Bufs<WIDE> bufs = make_bufs<PREC, WIDE, MODE == kDense>(p);
  zero_acc<VEC, NSUB>(acc);
  Group cur;
  int wi = 0, wend = 0;  // unbalanced: current window (relative to w0) and its end
  if constexpr (SCHED == kSplit) {
    wend = e;
  } else if constexpr (!BALANCED) {
    const int nw = w1 - w0;
    while (wi < nw && __builtin_amdgcn_readlane(rwo, wi) >= __builtin_amdgcn_readlane(rwo, wi + 1)) ++wi;
    if (wi == nw) {
      zero_windows<VEC, NSUB, WIDE>(p, w0, w1, cols);
      return;
    }
    b = __builtin_amdgcn_readlane(rwo, wi);
    wend = __builtin_amdgcn_readlane(rwo, wi + 1);
  }
  cur.bb = b;
  load_rows<MODE>(p, bufs, cur);  // needs no block offset: ahead of the stage's latency
  Stage st = load_stage<BALANCED>(p, b, e);
  Stage ahead = st;
  if (b + kStageBlocks < e) ahead = load_stage<BALANCED>(p, b + kStageBlocks, e);
  uint64_t starts = 0;
  auto find_starts = [&]() {
    if constexpr (BALANCED) {
      const int prev = __shfl_up(st.wid, 1, 64);
      starts = __ballot(st.wid != prev);  // bit 0 is never looked at
    }
  };
  // Position of the group that starts at block bb (inside the stage).
  auto place = [&](int bb, Group &m) {
    const int k = bb - st.sb;
    m.bb = bb;
    if constexpr (BALANCED) {
      m.nblk = 1 + (int)__builtin_ctzll((starts >> (k + 1)) | 8u);
      m.w = __builtin_amdgcn_readlane(st.wid, k);
    } else {
      m.nblk = min(kGroup, wend - bb);
      m.w = w0 + wi;
    }
    // Blocks past the group's end need no offset: an element below o4 lies
    // below their starts.
    m.o4 = min(__builtin_amdgcn_readlane(st.off, k + m.nblk), p.nnz);
    m.o0 = max(__builtin_amdgcn_readlane(st.off, k), 0);
    m.o1 = __builtin_amdgcn_readlane(st.off, k + 1);
    m.o2 = __builtin_amdgcn_readlane(st.off, k + 2);
    m.o3 = __builtin_amdgcn_readlane(st.off, k + 3);
  };
  find_starts();
  place(b, cur);
  load_elems<MODE>(p, bufs, has_vals, cur);
  int cw = cur.w;
  // pending empty windows [gap0, gap1): zeroed at one place in the loop
  int gap0 = w0;
  int gap1 = cw;
  if constexpr (BALANCED) {
    gap0 = (b > 0 ? wave_uniform(p.rowid[b - 1]) : -1) + 1;
    gap1 = min(cw, p.num_windows);
  }
  while (true) {
    // next group
    int bn = cur.bb + cur.nblk;
    bool more;
    if constexpr (BALANCED || SCHED == kSplit) {
      more = bn < e;
    } else {
      more = true;
      if (bn >= wend) {
        const int nw = w1 - w0;
        do {
          ++wi;
        } while (wi < nw && __builtin_amdgcn_readlane(rwo, wi) >= __builtin_amdgcn_readlane(rwo, wi + 1));
        more = wi < nw;
        if (more) {
          bn = __builtin_amdgcn_readlane(rwo, wi);
          wend = __builtin_amdgcn_readlane(rwo, wi + 1);
        }
      }
    }
    Group nxt = cur;  // the last group re-reads its own metadata
    if (more) {
      if ((unsigned)(bn - st.sb) >= (unsigned)kStageBlocks) {
        if ((unsigned)(bn - ahead.sb) < (unsigned)kStageBlocks) st = ahead;
        else st = load_stage<BALANCED>(p, bn, e);
        if (st.sb + kStageBlocks < e) ahead = load_stage<BALANCED>(p, st.sb + kStageBlocks, e);
        find_starts();
      }
      place(bn, nxt);
    }
    load_rows<MODE>(p, bufs, nxt);
    load_elems<MODE>(p, bufs, has_vals, nxt);
    breg_t<PREC, VEC> breg[NSUB][8];
    gather_b<PREC, VEC, NSUB, WIDE>(p, bufs, cur, cols, breg);
    // The previous window's stores go out after this group's gathers: loads
    // and stores retire through one in-order counter, so a store issued first
    // would hold up the wait for the gathers.
    if (SCHED != kSplit && cur.w != cw) {
      if (BALANCED && (cw == atomic_w0 || cw == atomic_w1))
        add_window_atomic<VEC, NSUB>(p, cw, ct, cols, lds, acc, cw != atomic_w0);
      else store_window<VEC, NSUB, WIDE>(p, cw, cols, acc);
      zero_acc<VEC, NSUB>(acc);
      gap0 = cw + 1;
      gap1 = min(cur.w, p.num_windows);
      cw = cur.w;
    }
    if (SCHED != kSplit && gap0 < gap1) {
      zero_windows<VEC, NSUB, WIDE>(p, gap0, gap1, cols);
      gap0 = gap1;
    }
    float a[8];
    build_a<MODE>(p, bufs, cur, has_vals, lds, a);
    mfma_group<PREC, VEC, NSUB>(a, breg, acc, has_vals);
    if (!more) break;
    cur = nxt;
  }
  if constexpr (SCHED == kSplit) return;  // the caller merges acc
  if (BALANCED && (cw == atomic_w0 || cw == atomic_w1))
    add_window_atomic<VEC, NSUB>(p, cw, ct, cols, lds, acc, cw != atomic_w0);
  else store_window<VEC, NSUB, WIDE>(p, cw, cols, acc);
  if constexpr (BALANCED) {
    if (e == p.num_blocks) zero_windows<VEC, NSUB, WIDE>(p, cw + 1, p.num_windows, cols);
  } else {
    zero_windows<VEC, NSUB, WIDE>(p, cw + 1, w1, cols);
  }
}

// End of window w whose block b is known: one ballot over the next 64 block
// ids covers most windows; longer ones finish with a wave-parallel search.
__device__ __forceinline__ int window_end_from(const int32_t *rowid, int b, int T, int w) {
  const int idx = b + lane_id();
  const uint64_t m = __ballot(idx >= T || rowid[idx] != w);
  if (m) return b + (int)__builtin_ctzll(m);
  return wave_lower_bound<int32_t>(rowid, b + 64, T, w + 1);
}

// Start of window w whose block b is known (the mirror image).
__device__ __forceinline__ int window_start_from(const int32_t *rowid, int b, int w) {
  if (b == 0) return 0;
  const int idx = b - 1 - lane_id();  // b-1, b-2, ..., b-64
  const uint64_t m = __ballot(idx < 0 || rowid[idx] != w);
  if (m) return b - (int)__builtin_ctzll(m);
  return wave_lower_bound<int32_t>(rowid, 0, b - 64, w);
}

template <int PREC, int VEC, int NSUB, int MODE>
__device__ __forceinline__ void run_unit(const SpmmParams &p, int item, int ct, float *lds) {
  floatx4 acc[NSUB][VEC];
  {
    // The chunk's run and the windows it merges atomically were worked out
    // by the preparation kernel (k_balance_prep).
    const int2 r = p.runs[item];
    const bool cut_first = r.x < 0;
    const bool cut_last = r.y < 0;
    const int b = cut_first ? ~r.x : r.x;
    const int e = cut_last ? ~r.y : r.y;
    if (b >= e) return;
    const int w_first = cut_first ? wave_uniform(p.rowid[b]) : -1;
    const int w_last = cut_last ? wave_uniform(p.rowid[e - 1]) : -1;
    if (p.parts && (cut_first || cut_last)) {
      reinterpret_cast<int *>(lds)[wave_lds_floats<VEC, NSUB>()] = item;
      wave_lds_sync();
    }
    walk_blocks<PREC, VEC, NSUB, kBalanced, MODE>(p, b, e, 0, 0, 0, ct, lds, w_first, w_last, acc);
  }
}

// Waves per SIMD the compiler must leave room for (its register budget), per
// instance: asked for these it keeps the accumulators out of the AGPRs and
// spills nothing in the loop; left to itself it stops one or two waves short.
// The unbalanced bf16x6 fits four (at three a band of 100,000 rows, N = 224, took
// 50 us against 43, R-MAT of 262,144, N = 128, 902 against 832); the other bf16x3
// and bf16x6 splits would spill and keep the default.  The balanced schedule over
// dense blocks spills at five (the same band, N = 512, 107 us against 94 at four).
template <int PREC, int VEC, int NSUB, bool BALANCED, int MODE>
constexpr int spmm_waves_per_eu() {
  if (PREC == DTC_PRECISION_BF16X6 && !BALANCED && VEC * NSUB == 4) return 4;
  if (PREC == DTC_PRECISION_BF16X3 || PREC == DTC_PRECISION_BF16X6) return 1;
  if (PREC == DTC_PRECISION_FP32 && BALANCED && MODE == kDense && VEC * NSUB == 4) return 4;
  if (is_bf16b<PREC>()) return VEC == 8 ? 4 : 5;
  return VEC * NSUB <= 2 ? 6 : VEC * NSUB == 4 ? 5 : 1;
}

// Window w by the workgroup's four waves: each takes a quarter of its groups,
// and their tiles are added through LDS in wave order (a fixed one: the result
// stays repeatable).  The window's serial chain of gathers becomes a quarter as
// long.
template <int PREC, int VEC, int NSUB, int MODE>
__device__ __forceinline__ void split_window(const SpmmParams &p, int w, int ct,
                                             float (*s_tile)[wave_lds_words<VEC, NSUB>()]) {
  constexpr int TW = 16 * VEC * NSUB;
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int b1 = max(0, min(wave_uniform(p.rwo[w + 1]), p.num_blocks));
  const int b0 = max(0, min(wave_uniform(p.rwo[w]), b1));
  const int per = (b1 - b0 + kGroup * kWavesPerBlock - 1) / (kGroup * kWavesPerBlock) * kGroup;  // blocks per wave
  const int b = min(b0 + wave * per, b1);
  const int e = min(b + per, b1);
  floatx4 acc[NSUB][VEC];
  if (b < e) walk_blocks<PREC, VEC, NSUB, kSplit, MODE>(p, b, e, w, w + 1, 0, ct, s_tile[wave], -1, -1, acc);
  else zero_acc<VEC, NSUB>(acc);
  const Cols<NSUB> cols = lane_cols<VEC, NSUB>(ct, p.N);
  const int g = lane >> 4;
#pragma unroll
  for (int s = 0; s < NSUB; ++s) {
    const int lc = cols.c[s] - ct * TW;  // below 0: a moved-back lane's columns of the previous tile
#pragma unroll
    for (int v = 0; v < VEC; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lc + v >= 0) s_tile[wave][(4 * g + i) * TW + lc + v] = acc[s][v][i];
  }
  __syncthreads();
  // 16 x TW sums, consecutive threads on consecutive columns
#pragma unroll
  for (int k = threadIdx.x; k < kBlkH * TW; k += 256) {
    const int col = ct * TW + k % TW;
    const int64_t row = (int64_t)w * kBlkH + k / TW;
    if (row < p.M && col < p.N) {
      const float sum = (s_tile[0][k] + s_tile[1][k]) + (s_tile[2][k] + s_tile[3][k]);
      __builtin_nontemporal_store(sum, p.C + row * p.N + col);
    }
  }
}

// The unbalanced schedule's unit: p.chunk consecutive windows per wave, except
// those of more than p.long_blocks blocks, which the workgroup's four waves
// then take together: one hub window is otherwise the whole launch (R-MAT of
// 761,088 rows, N = 48: a window of 5,585 blocks at 0.29 us each).
//
// With the column tiles one after another a hub window of the last tile would
// start late and outlast the launch, so a first part of the launch
// (p.long_groups workgroups a tile, the tiles side by side) takes the long
// windows of all tiles, and the second the others (R-MAT of 2^20 rows and 31.4 M
// entries, N = 128 4.54 -> 3.93 ms, 256 7.35 -> 5.74).  A workgroup of the first
// part looks at kLongGroups groups (one each took 60 us of a 2.56 ms launch
// without long windows, only to find none), one of each quarter: with group i of
// the first quarter the i-th from the end of the others, which in a power-law
// graph are light where it is heavy.
constexpr int kLongGroups = 4;
template <int PREC, int VEC, int NSUB, int MODE, bool IN_TURN>
__device__ __forceinline__ void run_windows(const SpmmParams &p, int group, int ct, bool long_part,
                                            float (*s_tile)[wave_lds_words<VEC, NSUB>()], uint32_t *s_long) {
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  // first window of the workgroup's share v & 3 (a wave's chunk) of its group v / 4
  auto first_window = [&](int v) {
    const int g = v < kWavesPerBlock ? group : (v / kWavesPerBlock + 1) * p.long_groups - 1 - group;
    return (g * kWavesPerBlock + v % kWavesPerBlock) * p.chunk;
  };
  auto blocks_before = [&](int w) { return max(0, min(p.rwo[min(w, p.num_windows)], p.num_blocks)); };
  if (!IN_TURN || !long_part) {
    const int g0 = group * kWavesPerBlock * p.chunk;  // the workgroup's windows (g0 < num_windows)
    const int g1 = min(g0 + kWavesPerBlock * p.chunk, p.num_windows);
    const int w0 = min(g0 + wave * p.chunk, g1);
    const int w1 = min(w0 + p.chunk, g1);
    // Lane l (at most 32): start of window w0 + l; lanes 62 and 63: the
    // workgroup's first block and end.  Offsets are clamped to the blocks
    // actually passed in.
    int rwo = blocks_before(lane == 62 ? g0 : lane == 63 ? g1 : min(w0 + lane, w1));
    // (Not for dense blocks: their windows are near their average -- a hub row
    // has one entry a column -- and the second walk's registers cost a band of
    // 45,312 rows, bf16x6, N = 240 2%: 27.9 against 28.5 us.)
    const bool any_long = MODE != kDense && __builtin_amdgcn_readlane(rwo, 63) -
                                                    __builtin_amdgcn_readlane(rwo, 62) > p.long_blocks;
    uint32_t longs = 0;  // this wave's long windows, a bit each
    if (any_long) {
      const int blocks = __shfl_down(rwo, 1, 64) - rwo;
      longs = (uint32_t)__ballot(w0 + lane < w1 && blocks > p.long_blocks);
    }
    if (any_long && lane == 0) s_long[wave] = longs;
    floatx4 acc[NSUB][VEC];
    for (int a = w0; a < w1;) {
      const int n = min(w1 - a, longs ? (int)__builtin_ctz(longs) : 32);  // windows up to the next long one
      if (n > 0)
        walk_blocks<PREC, VEC, NSUB, kWindows, MODE>(p, 0, __builtin_amdgcn_readlane(rwo, n), a, a + n, rwo, ct,
                                                     s_tile[wave], -1, -1, acc);
      if (!longs) break;
      a += n + 1;
      longs = n + 1 < 32 ? longs >> (n + 1) : 0;
      rwo = __shfl(rwo, lane + n + 1, 64);
    }
    if (!any_long || IN_TURN) return;  // workgroup-uniform
  } else {
#pragma unroll 1
    for (int k = 0; k < kLongGroups; ++k) {
      const int w = first_window(k * kWavesPerBlock + wave) + lane;
      const uint64_t longs = __ballot(lane < p.chunk && blocks_before(w + 1) - blocks_before(w) > p.long_blocks);
      if (lane == 0) s_long[k * kWavesPerBlock + wave] = (uint32_t)longs;
    }
  }
  __syncthreads();
  const int shares = IN_TURN ? kLongGroups * kWavesPerBlock : kWavesPerBlock;
  const int longs = (int)s_long[min(lane, shares - 1)];  // lane v: share v's
  for (int v = 0; v < shares; ++v) {
    for (uint32_t m = (uint32_t)__builtin_amdgcn_readlane(longs, v); m; m &= m - 1) {
      split_window<PREC, VEC, NSUB, MODE>(p, first_window(v) + (int)__builtin_ctz(m), ct, s_tile);
      __syncthreads();  // its tiles are read
    }
  }
}

// Group g of `groups` for a workgroup that would take group g in turn, the
// runs of 8 groups permuted: by the sum of the octal digits above the lowest.
// Workgroups go to the 8 XCDs round robin, and in a power-law graph the work
// falls with every bit set in a row's number, so groups in turn give one XCD
// the heavy ones of all runs: of an R-MAT matrix of 2^20 rows and 31.4 M
// entries 40% of the TC blocks go to one XCD and 1.7% to another in turn (18%
// and 6% with four tiles side by side), 12.9% and 12.0% so.  N = 48 4.71 -> 3.51
// ms, 128 8.45 -> 4.54, 256 16.4 -> 7.35.
__device__ __forceinline__ int spread_group(int g, int groups) {
  int turn = 0;
#pragma unroll
  for (int k = 3; k < 30; k += 3) turn += g >> k;  // (of which the low three bits count)
  return (g | 7) < groups ? (g & ~7) | ((g + turn) & 7) : g;
}

// Workgroup i serves column tile i % n_ct: workgroups are dispatched to the
// 8 XCDs round robin, so when n_ct divides 8 every XCD (and its L2) only
// sees one column tile of B.
template <int PREC, int VEC, int NSUB, bool BALANCED, int MODE>
__global__ __launch_bounds__(256) __attribute__((
    amdgpu_waves_per_eu(spmm_waves_per_eu<PREC, VEC, NSUB, BALANCED, MODE>()))) void spmm_kernel(SPMM_KERNEL_ARGS) {
  const SpmmParams p = SPMM_PARAMS_FROM_ARGS;
  __shared__ __attribute__((aligned(16))) float s_tile[kWavesPerBlock][wave_lds_words<VEC, NSUB>()];
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int ct = blockIdx.x % p.n_ct;
  const int group = blockIdx.x / p.n_ct;
  if constexpr (BALANCED) {
    const int item = group * kWavesPerBlock + wave;
    if (item >= p.num_items) return;
    run_unit<PREC, VEC, NSUB, MODE>(p, item, ct, s_tile[wave]);
  } else {
    __shared__ uint32_t s_long[kWavesPerBlock];
    run_windows<PREC, VEC, NSUB, MODE, false>(p, spread_group(group, p.groups), ct, false, s_tile, s_long);
  }
}

// The same with the column tiles one after another: workgroup i serves tile
// i / groups.  All XCDs then gather from the same column slice of B at a time; in
// the balanced schedule from two, half of B's columns apart: with one alone, where
// many gathers go to rows whose numbers are multiples of 16 (R-MAT as its
// generator labels it), few memory channels serve them.  2^20 rows, N = 256, ms,
// side by side, one and two slices at a time: 3.98, 4.50 and 4.22; with the
// numbers shuffled inside groups of 16 3.45, 3.20 and 3.16.  The unbalanced launch
// begins with the part that takes the long windows.
template <int PREC, int VEC, int NSUB, bool BALANCED, int MODE>
__global__ __launch_bounds__(256) __attribute__((
    amdgpu_waves_per_eu(spmm_waves_per_eu<PREC, VEC, NSUB, BALANCED, MODE>()))) void spmm_kernel_turn(SPMM_KERNEL_ARGS) {
  const SpmmParams p = SPMM_PARAMS_FROM_ARGS;
  __shared__ __attribute__((aligned(16))) float s_tile[kWavesPerBlock][wave_lds_words<VEC, NSUB>()];
  if constexpr (BALANCED) {
    const int wave = wave_uniform(threadIdx.x >> 6);
    const int pass = blockIdx.x / p.groups;
    const int group = blockIdx.x % p.groups;
    const int ct = !(group & 1) ? pass : pass < p.n_ct / 2 ? pass + (p.n_ct + 1) / 2 : pass - p.n_ct / 2;
    const int item = group * kWavesPerBlock + wave;
    if (item >= p.num_items) return;
    run_unit<PREC, VEC, NSUB, MODE>(p, item, ct, s_tile[wave]);
  } else {
    __shared__ uint32_t s_long[kLongGroups * kWavesPerBlock];
    const int long_wgs = p.long_groups * p.n_ct;
    const bool long_part = (int)blockIdx.x < long_wgs;
    const unsigned at = blockIdx.x - (long_part ? 0 : long_wgs), per = long_part ? p.n_ct : p.groups;
    const int q = at / per, r = at % per;
    const int group = spread_group(long_part ? q : r, long_part ? p.long_groups : p.groups);
    run_windows<PREC, VEC, NSUB, MODE, true>(p, group, long_part ? r : q, long_part, s_tile, s_long);
  }
}

// Unbalanced schedule for launches that cannot fill the GPU: one workgroup
// per (window, column tile).
template <int PREC, int VEC, int NSUB, int MODE>
__global__ __launch_bounds__(256) __attribute__((
    amdgpu_waves_per_eu(spmm_waves_per_eu<PREC, VEC, NSUB, false, MODE>()))) void spmm_kernel_split(SPMM_KERNEL_ARGS) {
  const SpmmParams p = SPMM_PARAMS_FROM_ARGS;
  __shared__ __attribute__((aligned(16))) float s_tile[kWavesPerBlock][wave_lds_words<VEC, NSUB>()];
  split_window<PREC, VEC, NSUB, MODE>(p, blockIdx.x / p.n_ct, blockIdx.x % p.n_ct, s_tile);  // grid: n_ct * num_windows
}

// Persistent variant of the balanced schedule: every wave pulls units from a
// global counter until the list is exhausted.
template <int PREC, int VEC, int NSUB, int MODE>
__global__ __launch_bounds__(256) __attribute__((
    amdgpu_waves_per_eu(spmm_waves_per_eu<PREC, VEC, NSUB, true, MODE>()))) void spmm_kernel_persistent(SPMM_KERNEL_ARGS) {
  const SpmmParams p = SPMM_PARAMS_FROM_ARGS;
  __shared__ __attribute__((aligned(16))) float s_tile[kWavesPerBlock][wave_lds_words<VEC, NSUB>()];
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int total = p.num_items * p.n_ct;
  while (true) {
    int u = 0;
    if (lane == 0) u = atomicAdd(p.queue, 1);
    u = __shfl(u, 0, 64);
    u = wave_uniform(u);
    if (u >= total) break;
    run_unit<PREC, VEC, NSUB, MODE>(p, u / p.n_ct, u % p.n_ct, s_tile[wave]);
  }
}

// Zeroes the rows of window w (one wave).
__device__ __forceinline__ void zero_window_rows(float *C, int64_t w, int32_t M, int32_t N) {
  const int lane = lane_id();
  const int64_t r0 = w * kBlkH;
  const int64_t r1 = (r0 + kBlkH < (int64_t)M) ? r0 + kBlkH : (int64_t)M;
  if (r0 >= r1) return;
  float *base = C + r0 * (int64_t)N;
  const int64_t count = (r1 - r0) * (int64_t)N;
  if ((N & 3) == 0 && ((uintptr_t)base & 15) == 0) {
    floatx4 *b4 = reinterpret_cast<floatx4 *>(base);
    const floatx4 z = {0.f, 0.f, 0.f, 0.f};
    for (int64_t idx = lane; idx < count / 4; idx += 64) b4[idx] = z;
  } else {
    for (int64_t idx = lane; idx < count; idx += 64) base[idx] = 0.f;
  }
}

constexpr int kNearSpan = 512;  // chunks up to this many blocks use the bounded scans

// Start of window w (the window of block c) if it lies at most `span` blocks
// before c, else -1.  All span/64 loads per lane are issued before the first
// ballot: one memory round trip instead of a search's chain.
__device__ __forceinline__ int window_start_near(const int32_t *rowid, int c, int w, int span) {
  const int lane = lane_id();
  int v[kNearSpan / 64];
#pragma unroll
  for (int k = 0; k < kNearSpan / 64; ++k) {
    const int idx = c - 1 - lane - 64 * k;  // c-1, c-2, ...; -2 marks the array's start
    v[k] = (64 * k < span && idx >= c - span) ? (idx >= 0 ? rowid[idx] : -2) : w;
  }
#pragma unroll
  for (int k = 0; k < kNearSpan / 64; ++k) {
    const uint64_t m = __ballot(v[k] != w);
    if (m) return c - 64 * k - (int)__builtin_ctzll(m);
  }
  return -1;
}

// End of window w (the window of block c) if it lies at most `span` blocks
// after c, else -1 (same single round of loads).
__device__ __forceinline__ int window_end_near(const int32_t *rowid, int c, int T, int w, int span) {
  const int lane = lane_id();
  int v[kNearSpan / 64 + 1];  // blocks c .. c + span
#pragma unroll
  for (int k = 0; k < kNearSpan / 64 + 1; ++k) {
    const int idx = c + lane + 64 * k;  // c, c+1, ...; -2 marks the array's end
    v[k] = (64 * k <= span && idx <= c + span) ? (idx < T ? rowid[idx] : -2) : w;
  }
#pragma unroll
  for (int k = 0; k < kNearSpan / 64 + 1; ++k) {
    const uint64_t m = __ballot(v[k] != w);
    if (m) return c + 64 * k + (int)__builtin_ctzll(m);
  }
  return -1;
}

// Balanced-schedule preparation.  Ownership rule, for chunks of `chunk` TC
// blocks and a cut span `span` (a multiple of chunk): a window of at most
// `span` blocks belongs whole to the chunk holding its first block (and may
// run past that chunk's end); a longer window is cut at the multiples of
// `span` into pieces, each belonging to the chunk holding its first block,
// and the pieces are merged with atomic adds.  The multiples of `span` are
// chunk boundaries, so a chunk's run can only begin with a cut piece (one that
// starts at the chunk's first block) and only end with one (the first piece
// of a long window that starts inside the chunk, which then runs past the
// chunk's end); every window in between is short and whole.  A larger span
// cuts fewer windows into fewer pieces (fewer atomic tiles written) at the
// price of longer work units.  Wave v, one per chunk:
//   * for chunk v ([c0, c1) = blocks [v*chunk, (v+1)*chunk)), writes the
//     chunk's run [b, e) to runs[v]: b = c0 unless the window or piece
//     holding c0 began earlier (then b = its end), e = c1 unless a window or
//     piece that begins inside the chunk runs past c1 (then e = its end); ~b
//     marks a cut first piece, ~e a cut last piece (b >= e: nothing to do);
//     and zeroes the rows of the cut windows that start in the chunk, since
//     no chunk stores them whole;
//   * (wave 0) resets the persistent work counter.
// The window searches run here, once per chunk, on an idle memory system
// instead of at the start of every SpMM wave.  Empty windows are zeroed by
// the SpMM waves themselves (walk_blocks): nothing else writes them.
__global__ __launch_bounds__(256) void k_balance_prep(const int32_t *rowid, int32_t T,
                                                      int32_t M, int32_t N,
                                                      int32_t chunk, int32_t span,
                                                      int32_t num_items, float *C,
                                                      int32_t *queue, int2 *runs,
                                                      int32_t zero_cut) {
  if (queue && blockIdx.x == 0 && threadIdx.x == 0) *queue = 0;
  const int lane = lane_id();
  const int64_t v = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (v >= num_items) return;
  const int c0 = (int)v * chunk;
  const int c1 = min(c0 + chunk, T);
  // Window extents: exact for spans above kNearSpan (searches); for smaller
  // spans only within `span` blocks of the boundary, -1 meaning farther --
  // which already makes the window longer than the span.
  const bool near = span <= kNearSpan;
  auto start_of = [&](int c, int w) {
    return wave_uniform(near ? window_start_near(rowid, c, w, span) : window_start_from(rowid, c, w));
  };
  auto end_of = [&](int c, int w) {
    return wave_uniform(near ? window_end_near(rowid, c, T, w, span)
                             : max(c + 1, window_end_from(rowid, c, T, w)));
  };
  // first multiple of span after x (a chunk boundary; no multiple of span
  // lies strictly inside a chunk)
  auto next_cut = [&](int x) { return (int)min<int64_t>(((int64_t)x / span + 1) * span, T); };
  auto is_long = [&](int ws, int we) { return ws < 0 || we < 0 || we - ws > span; };
  const int w0 = wave_uniform(rowid[c0]);
  const int ws0 = start_of(c0, w0);
  const int we0 = end_of(c0, w0);
  const bool first_long = is_long(ws0, we0);
  bool cut_first = false;
  int b;
  if (!first_long) {
    b = ws0 < c0 ? we0 : c0;
  } else {
    // the piece holding c0 starts at c0 when c0 is a multiple of span or the
    // window's first block; it ends at the next multiple of span or the
    // window's end (an unknown end lies more than span away: past the cut)
    const int pe = (we0 >= 0 && we0 < next_cut(c0)) ? we0 : next_cut(c0);
    if (c0 % span == 0 || ws0 == c0) {
      b = c0;
      cut_first = true;
    } else {
      b = pe;
    }
  }
  int e = c1;
  bool cut_last = false;
  int wl = -1, wsl = -1;
  if (b < c1 && c1 < T) {
    const int r_in = wave_uniform(rowid[c1 - 1]);
    const int r_out = wave_uniform(rowid[c1]);
    if (r_in == r_out) {  // a window crosses c1
      if (r_in == w0) {
        // the run's first window or piece runs past c1 (b == c0 here): a
        // short window whole, or the same piece as the one at c0
        e = first_long ? ((we0 >= 0 && we0 < next_cut(c0)) ? we0 : next_cut(c0)) : we0;
      } else {
        wl = r_in;  // starts inside the chunk: within span of c1
        wsl = start_of(c1, r_in);
        const int wel = end_of(c1, r_in);
        if (!is_long(wsl, wel)) {
          e = wel;
        } else {
          e = (wel >= 0 && wel < next_cut(wsl)) ? wel : next_cut(wsl);
          cut_last = true;
        }
      }
    }
  }
  if (b >= c1) {
    b = e = c1;
    cut_first = cut_last = false;
  }
  if (lane == 0) runs[v] = make_int2(cut_first ? ~b : b, cut_last ? ~e : e);
  if (!zero_cut) return;  // deterministic merge: k_balance_fixup writes cut windows whole
  if (cut_first && ws0 == c0) zero_window_rows(C, w0, M, N);
  if (cut_last) zero_window_rows(C, wl, M, N);
}

// Deterministic merge of cut windows, after the SpMM kernel: wave (chunk c,
// column tile ct) takes the one cut window that starts in chunk c, if any
// (a cut window is longer than the span, so no chunk holds the start of two),
// sums its partial tiles in chunk order -- chunk c's slot for the window's
// role there, then slot 2 c' of every chunk c' holding a later piece (the
// chunks at the multiples of span inside the window), where it is the first
// piece -- and stores the window's rows.  Tiles are row-major 16 x tw floats
// (tw = the SpMM's column-tile width).
__global__ __launch_bounds__(256) void k_balance_fixup(const int32_t *__restrict__ rowid,
                                                       SpmmParams p, int32_t tw) {
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int ct = blockIdx.x % p.n_ct;
  const int c = (blockIdx.x / p.n_ct) * kWavesPerBlock + wave;
  if (c >= p.num_items) return;
  const int2 r = p.runs[c];
  const bool cut_first = r.x < 0;
  const bool cut_last = r.y < 0;
  if (!cut_first && !cut_last) return;
  const int c0 = c * p.chunk;
  const int b = cut_first ? ~r.x : r.x;
  const int e = cut_last ? ~r.y : r.y;
  int w = -1, role = 0;
  if (cut_first) {  // the chunk's first window: cut, and starting at c0?
    const int wf = wave_uniform(rowid[b]);
    if (c0 == 0 || wave_uniform(rowid[c0 - 1]) != wf) w = wf;
  }
  if (w < 0 && cut_last) {  // the chunk's last window, starting inside the chunk?
    const int wl = wave_uniform(rowid[e - 1]);
    if (c0 == 0 || wave_uniform(rowid[c0 - 1]) != wl) {
      w = wl;
      role = 1;
    }
  }
  if (w < 0) return;
  const int we = wave_uniform(window_end_from(rowid, e - 1, p.num_blocks, w));
  // later pieces start at the multiples of span in (c0, we): chunks
  // first_later, first_later + step, ... (no multiple of span lies strictly
  // inside chunk c, so the first one after c0 is the first after the start)
  const int step = p.span / p.chunk;
  const int first_later = (int)(((int64_t)c0 / p.span + 1) * p.span / p.chunk);
  const int c_last = (we - 1) / p.chunk;
  const int64_t tile = (int64_t)kBlkH * tw;
  const int64_t slot_stride = (int64_t)p.n_ct * tile;
  const float *first = p.parts + ((int64_t)2 * c + role) * slot_stride + ct * tile;
  const float *later = p.parts + (int64_t)ct * tile;
  const int64_t N = p.N;
  for (int k = lane; k < kBlkH * tw; k += kWave) {
    float sum = first[k];
#pragma unroll 8
    for (int cc = first_later; cc <= c_last; cc += step) sum += later[(int64_t)2 * cc * slot_stride + k];
    const int64_t row = (int64_t)w * kBlkH + k / tw;
    const int col = ct * tw + k % tw;
    if (row < p.M && col < p.N) __builtin_nontemporal_store(sum, p.C + row * N + col);
  }
}

// ------------------------------------------------------------ host side

typedef void (*KernelFn)(const int32_t *, const int32_t *, const uint8_t *, const int32_t *,
                         const int32_t *, const float *, const void *, float *, SpmmParams);

struct Variant {
  int prec;  // DTC_PRECISION_* or a bf16-B scheme
  int vec;
  int nsub;
  int mode;  // kPtr, kBuf or kDense
};

// Launch schedules of a kernel instance.
constexpr int kRunWindows = 0, kRunBalanced = 1, kRunPersistent = 2, kRunSplit = 3;
constexpr int kRunWindowsTurn = 4, kRunBalancedTurn = 5;

template <int PREC, int VEC, int NSUB, int MODE>
KernelFn pick_schedule(int schedule) {
  switch (schedule) {
    case kRunWindows: return spmm_kernel<PREC, VEC, NSUB, false, MODE>;
    case kRunBalanced: return spmm_kernel<PREC, VEC, NSUB, true, MODE>;
    case kRunPersistent: return spmm_kernel_persistent<PREC, VEC, NSUB, MODE == kDense ? kBuf : MODE>;
    case kRunWindowsTurn: return spmm_kernel_turn<PREC, VEC, NSUB, false, MODE == kDense ? kBuf : MODE>;
    case kRunBalancedTurn: return spmm_kernel_turn<PREC, VEC, NSUB, true, MODE>;
    default: return spmm_kernel_split<PREC, VEC, NSUB, MODE>;
  }
}

template <int PREC, int VEC, int NSUB>
KernelFn pick_mode(const Variant &v, int schedule) {
  return v.mode == kDense ? pick_schedule<PREC, VEC, NSUB, kDense>(schedule)
                          : pick_schedule<PREC, VEC, NSUB, kBuf>(schedule);
}

template <int PREC>
KernelFn pick_shape(const Variant &v, int schedule) {
  if (v.mode == kPtr)
    return v.vec == 4 ? pick_schedule<PREC, 4, 1, kPtr>(schedule) : pick_schedule<PREC, 1, 1, kPtr>(schedule);
  if (v.vec == 4 && v.nsub == 2) return pick_mode<PREC, 4, 2>(v, schedule);
  if (v.vec == 4) return pick_mode<PREC, 4, 1>(v, schedule);
  if (v.vec == 2) return pick_mode<PREC, 2, 1>(v, schedule);
  return pick_mode<PREC, 1, 1>(v, schedule);
}

template <int PREC>
KernelFn pick_shape_bf16b(const Variant &v, int schedule) {
  if (v.mode == kPtr) return pick_schedule<PREC, 4, 1, kPtr>(schedule);
  if (v.vec == 8) return pick_mode<PREC, 8, 1>(v, schedule);
  return pick_mode<PREC, 4, 1>(v, schedule);
}

KernelFn pick_kernel(const Variant &v, int schedule) {
  switch (v.prec) {
    case DTC_PRECISION_FP32: return pick_shape<DTC_PRECISION_FP32>(v, schedule);
    case DTC_PRECISION_BF16: return pick_shape<DTC_PRECISION_BF16>(v, schedule);
    case DTC_PRECISION_FP16: return pick_shape<DTC_PRECISION_FP16>(v, schedule);
    case DTC_PRECISION_BF16X3: return pick_shape<DTC_PRECISION_BF16X3>(v, schedule);
    case kBf16B_A3: return pick_shape_bf16b<kBf16B_A3>(v, schedule);
    case kBf16B_A1: return pick_shape_bf16b<kBf16B_A1>(v, schedule);
    default: return pick_shape<DTC_PRECISION_BF16X6>(v, schedule);
  }
}

// How the kernels read these operands.  Buffers need 32-bit byte offsets
// (offsets of 2^31 and more lie past B's end) and 24-bit factors of a row's
// offset.  The dense form pays where groups hold more than one load's 64
// elements on average; it reads whole 4-element vectors, whose alignment
// keeps the last one in the same 16 bytes as an element of the array.
int operand_mode(int64_t b_rows, int64_t n, int64_t esz, int64_t nnz, int64_t num_blocks, const void *tile,
                 const void *vals) {
  const int64_t lim = (int64_t)1 << 31;
  const bool fits = (b_rows + 1) * n * esz < lim && b_rows < (1 << 24) - 1 && n * esz < (1 << 24) &&
                    nnz * 4 < lim - 64 && num_blocks * kBlkW * 4 < lim;
  if (!fits) return kPtr;
  const bool aligned = ((uintptr_t)tile & 3) == 0 && ((uintptr_t)vals & 15) == 0;
  return aligned && nnz > 16 * num_blocks ? kDense : kBuf;
}

// Kernel scheme and lane shape from the options, N and operand alignment.  An
// explicit vec must divide N and the base addresses; vec 0 takes any N of at
// least its width (unaligned vectors, the last lanes moved back: lane_cols).
// vec 0 for float32 B: 4 floats per lane (64-column tiles), less where N is
// narrower.
dtc_status_t resolve_shape(const dtc_spmm_options_t *opt, int32_t n, const void *b, const float *c,
                           bool balanced, bool dense, int64_t windows, bool unshared, bool short_windows,
                           bool few_entries, int mode, Variant *out) {
  const bool wide = mode == kPtr;
  const int prec = opt ? opt->precision : DTC_PRECISION_FP32;
  const int bdt = opt ? opt->b_dtype : DTC_B_FLOAT32;
  int vec = opt ? opt->vec : 0;
  int nsub = opt ? opt->subtiles : 0;
  out->mode = mode;
  if (bdt == DTC_B_BFLOAT16) {
    // bf16 B: 4 or 8 bf16 per lane (8 or 16 bytes), one subtile.
    if (vec != 0 && vec != 4 && vec != 8)
      return fail(DTC_ERROR_INVALID_VALUE, "vec must be 0, 4 or 8 for bfloat16 B");
    auto fits = [&](int v) {
      return n % v == 0 && ((uintptr_t)b % (2 * v)) == 0 && ((uintptr_t)c % (4 * v)) == 0;
    };
    // 128-column tiles where N fills more than half of one, in the unbalanced
    // schedule not for rows of few entries, whose windows leave a wave little to
    // overlap (us, 64 and 128 columns: band of 8 to a row, 200,000 rows, N = 256 55
    // and 84, uniform 200,000 of 8 142 and 164; band of 12, 10^6 rows, N = 128 208 and
    // 190, uniform 65,536 of 32 53 and 42).
    if (vec == 0) {
      if (!fits(4))
        return fail(DTC_ERROR_INVALID_VALUE,
                    "bfloat16 B needs N to be a multiple of 4 and 8-byte aligned B/C rows");
      vec = n > 64 && !few_entries ? 8 : 4;
    } else
    if (!fits(vec))
      return fail(DTC_ERROR_INVALID_VALUE,
                  "bfloat16 B needs N to be a multiple of 4 and 8-byte aligned B/C rows");
    out->prec = (prec == DTC_PRECISION_BF16) ? kBf16B_A1 : kBf16B_A3;
    out->vec = wide ? 4 : vec;
    out->nsub = 1;
    return DTC_SUCCESS;
  }
  if (bdt != DTC_B_FLOAT32) return fail(DTC_ERROR_INVALID_VALUE, "unknown b_dtype");
  if (vec != 0 && vec != 1 && vec != 2 && vec != 4)
    return fail(DTC_ERROR_INVALID_VALUE, "vec must be 0, 1, 2 or 4");
  if (nsub < 0 || nsub > 2) return fail(DTC_ERROR_INVALID_VALUE, "subtiles must be 0, 1 or 2");
  auto fits = [&](int v) {
    return n % v == 0 && ((uintptr_t)b % (4 * v)) == 0 && ((uintptr_t)c % (4 * v)) == 0;
  };
  if (vec != 0 && !fits(vec))
    return fail(DTC_ERROR_INVALID_VALUE,
                "vec " + std::to_string(vec) + " needs N and the B/C base addresses to be multiples of it");
  if (vec == 0) {
    vec = n <= 16 ? 1 : n <= 32 ? 2 : 4;
    // Where 64-column tiles would leave half of the last one empty: one of 128
    // (two subtiles) in the unbalanced schedule and for dense blocks (each tile
    // builds its A again), else three of 32 in the balanced one (N = 96, us: 46,000
    // blocks 40 against 47 and 55, 157,000 96 / 108 / 121, 1.08 M 476 / 526 / 539;
    // block model of 958,000 blocks of 13 382 / 397 / 372, band of 55 a block 66 and
    // 60).  128-column tiles also for wide B in the unbalanced schedule.  There not
    // where rows share columns without being dense, as hubs do, whose windows then
    // take longer (us with one and two subtiles: R-MAT of 25,568 rows, N = 84 220 and
    // 313, of 262,144 631 and 881, block model of 60,000, N = 320 1,218 and 1,465;
    // uniform 65,536 rows of 32, N = 84 111 and 84, 200,000 of 16, N = 260 755 and
    // 627), and for dense blocks not with the limb splits, whose registers cost waves
    // in windows of a group or two (band of 5 blocks a window, N = 224, bf16x3 37 and
    // 40, bf16x6 43 and 47; of 10, N = 512 72 and 63, 77 and 75), nor where wide B
    // leaves half of the last tile empty (N = 320 51 and 55, 384 62 and 58; the other
    // way round where columns are unshared: 30,000 rows of 16, N = 320 85 and 77,
    // of 8, N = 384 53 and 56).  Not where the wider tiles leave the chip short of
    // units either (uniform 20,000 of 30, N = 96 33 and 41, band of 5,000, N = 384 11.5
    // and 16.1).
    const bool half = n % 128 > 64 && n % 128 <= 96;
    if (nsub == 0 && balanced && half && n < 128 && !dense) vec = 2;
    if (nsub == 0 && balanced) nsub = half && dense ? 2 : 1;
    if (nsub == 0) {
      const bool limbs = prec == DTC_PRECISION_BF16X3 || prec == DTC_PRECISION_BF16X6;
      const bool two = mode == kDense ? !(limbs && short_windows) && (half || (n > 256 && (n - 1) % 128 >= 64))
                                      : half || (n > 256 && (n - 1) % 128 < 64);
      const bool fills = windows * ceil_div(n, 128) >= (mode == kDense ? 1024 : 4096);
      nsub = two && fills && (mode == kDense || unshared) ? 2 : 1;
    }
  }
  if (wide) vec = n >= 4 ? 4 : 1;
  if (nsub == 0 || wide || vec != 4) nsub = 1;
  out->prec = prec;
  out->vec = vec;
  out->nsub = nsub;
  return DTC_SUCCESS;
}

// Whether the unbalanced schedule splits each window over a workgroup's four
// waves: with at most one unit per SIMD (two when windows are long) the chip
// idles while every wave walks its window's groups one after another.
// Uniform matrices, 64-column tiles, us whole -> split: 128 windows of 57
// blocks 17 -> 6.6, of 162 42 -> 13; 512 windows at 1,024 units, of 62 blocks
// 19 -> 15.5, of 16 7.0 -> 7.5; at 2,048 units, of 62 28 -> 29, of 227 95 -> 85.
bool split_windows(int64_t windows, int64_t n_ct, int64_t num_blocks) {
  const int64_t units = windows * n_ct;
  return (units <= 1024 && num_blocks > 5 * windows) || (units <= 2048 && num_blocks > 96 * windows);
}

// Consecutive windows per unit of the unbalanced schedule: short windows are
// walked several to a wave, as one pipeline, while enough units remain.  For
// units of up to 32 columns only, where a window is little work: wider ones lose
// more by the longer chains, and in a band by rows of B that the workgroup's
// waves no longer read at the same time.  us, one window and several: uniform
// 2^20 rows of 4, N = 16 111 and 103, of 8, N = 32 194 and 188, of 4, N = 64 186
// and 197; band of 19 columns half filled, 500,001 rows, N = 100 105 and 117, of
// 25, 10^6 rows, N = 128 262 and 277; R-MAT of 2^20 rows of 4, N = 64 618 and 843.
int32_t windows_per_unit(int64_t windows, int64_t n_ct, int64_t num_blocks, int32_t columns) {
  int32_t k = 1;
  if (columns > 32) return k;
  while (k < 32 && 2 * k * num_blocks <= 32 * windows && windows * n_ct >= 2 * k * 16384) k *= 2;
  return k;
}

// Blocks from which the unbalanced schedule shares a window out to a workgroup:
// windows far longer than the others, whose chains would outlast the launch.
// (us, none shared / from 16 / 8 / 4 times the average on: R-MAT of 16 a row,
// 761,088 rows, N = 48 2,700 / 1,334 / 1,332 / 1,333; 262,144 of 32, N = 128
// 2,018 / 1,199 / 1,179 / 1,188; 20,000 of 40, N = 64 264 / 215 / 152 / 142;
// 25,568 of 40, N = 85 511 / 434 / 355 / 255; block model of 60,000 rows and hubs,
// N = 128 714 / 715 / 683 / 446.  From 64 or 256 blocks on instead of 128: within
// 1%.  Uniform matrices, whose windows are near their average, have none.)
int32_t long_window(int64_t windows, int64_t num_blocks) {
  return (int32_t)std::min<int64_t>(std::max<int64_t>(128, 4 * num_blocks / windows), INT32_MAX);
}

// Whether hardly any column has two entries in a window (of the least 8 entries
// a block, at most 8.25): uniform matrices; in power-law ones rows share the
// hubs' columns (8.3 to 13 entries a block).
bool unshared_columns(int64_t nnz, int64_t num_blocks) { return 4 * nnz <= 33 * num_blocks; }

// Whether windows hold about as many columns as random entries over all of B's
// rows would: x entries a row of B and window fall on (1 - e^-x) / x as many columns.
bool even_windows(int64_t nnz, int64_t num_blocks, int64_t windows, int64_t b_rows) {
  if (nnz <= 0 || windows <= 0 || b_rows <= 0) return false;
  const double x = (double)nnz / ((double)windows * (double)b_rows);
  return 4.0 * (double)nnz * (-std::expm1(-x) / x) <= 33.0 * (double)num_blocks;
}

// Whether the column tiles go one after another instead of side by side.  B
// beyond the 256 MB memory-side cache: one slice (or two) at a time, so that most
// of its gathers hit there.  (Two tiles of 256 MB each are no faster in turn,
// uniform 2^20 rows of 16, N = 128 1.24 and 1.29 ms; two of 512 are, N = 256 2.93
// and 2.53.)
bool tiles_in_turn(const SpmmParams &p, int64_t esz) {
  const int64_t b_bytes = (int64_t)p.b_rows * p.N * esz;
  return p.n_ct > 1 && b_bytes > (int64_t)(p.n_ct > 2 ? 256 : 512) << 20;
}

dtc_status_t check_common(const uint8_t *tile, const int32_t *off, const int32_t *atox,
                          int32_t num_blocks, int32_t nnz, int32_t num_nodes, const void *b,
                          int32_t b_rows, int32_t n, float *c, const dtc_spmm_options_t *opt) {
  if (num_nodes < 0 || b_rows < 0 || num_blocks < 0 || nnz < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "sizes must be >= 0");
  if (n <= 0) return fail(DTC_ERROR_INVALID_VALUE, "N (feature width) must be >= 1");
  if (!off) return fail(DTC_ERROR_INVALID_VALUE, "TCblock_offset is NULL");
  if (num_nodes > 0 && !c) return fail(DTC_ERROR_INVALID_VALUE, "C is NULL");
  if (b_rows > 0 && !b) return fail(DTC_ERROR_INVALID_VALUE, "B is NULL");
  if (num_blocks > 0) {
    if (!tile || !atox)
      return fail(DTC_ERROR_INVALID_VALUE, "TCblocktile_id and sparse_AToX_idx are required");
    if (nnz < 1) return fail(DTC_ERROR_INVALID_VALUE, "TC blocks without stored elements");
    if ((uintptr_t)atox % 16 != 0)
      return fail(DTC_ERROR_INVALID_VALUE, "sparse_AToX_idx must be 16-byte aligned");
  }
  const int prec = opt ? opt->precision : DTC_PRECISION_FP32;
  if (prec < DTC_PRECISION_FP32 || prec > DTC_PRECISION_BF16X6)
    return fail(DTC_ERROR_INVALID_VALUE, "unknown precision");
  if ((int64_t)num_nodes * n > ((int64_t)1 << 40))
    return fail(DTC_ERROR_UNSUPPORTED, "output too large");
  return DTC_SUCCESS;
}

// The default chunk by the block count alone, in TC blocks: the one that a cut
// span is measured against, and the one for a workspace that the chunks of
// resolve_chunk exceed (it is mostly longer than those, not always).
int long_chunk_blocks(int32_t num_blocks) {
  int c = 32;
  while (c < 512 && (int64_t)c * 2 * 8192 <= (int64_t)num_blocks) c *= 2;
  return c;
}

// Balanced chunk: options->chunk_blocks, or with 0 the power of two in [8, 256]
// that leaves some 550 * chunk units (chunks x 64-column tiles): a small launch
// is as long as one unit's chain, a large one pays for every unit's start and
// every cut window's merge.  Best and next chunks measured, us, R-MAT: 4,100
// blocks, N = 64 (8) 15 (16) 21; 18,700, N = 48 (8) 22 (32) 25, N = 192 (32) 33
// (16) 35; 46,000, N = 48 (16) 34 (32) 43, N = 256 (32) 70 (16) 73; 157,000, N =
// 64 (32) 71 (16) 77, N = 256 (64) 179 (32) 187; 432,000, N = 32 (32) 98 (64)
// 108, N = 128 (64) 240 (32) 246; 1.08 M, N = 128 (64) 565 (128) 586; block model
// of 958,000 blocks, N = 256 (128) 761 (64) 825.
// Dense blocks take longer chunks (more work a block, and windows of one length,
// most of which a short chunk cuts in two): half as many units per chunk beyond
// 11 entries a block, and beyond 24 at least 32 blocks unless the launch is small.
// Block model of 99,700 blocks of 12.5, N = 64, (32) 46 (16) 50; band of 55 a
// block, 53,000 blocks, N = 64 (32) 37 (16) 44, 106,000, N = 256 (32) 164 (64)
// 187, 8,750, N = 128 (8) 19.6 (16) 21.3.
// Where entries are spread like random ones, windows are of one length, and a
// shorter chunk cuts and merges every one of them: up to the average window's
// length the chunk doubles while it leaves 27 * chunk units of 64 columns.  us, chunk by the rule above and this:
// uniform 20,000 rows of 16, N = 128 (16) 34 (32) 23, bf16 B 31 and 18 (28 and 21
// with the chunk by block count); 30,000 of 30, N = 64 (16) 57 (64) 42; 65,536 of
// 32, N = 128 (32) 150 (64) 108; 16,384 of 60, N = 64 (16) 54 (64) 37 (128) 62;
// 4,096 of 16, N = 64 (8) 14.4 (16) 15.1, N = 128 (8) 19.6 (16) 15.8.
// nnz 0, windows 0: not known, the shortest chunk it could be.
constexpr int64_t kChunkUnits = 550;
int resolve_chunk(const dtc_spmm_options_t *opt, int32_t num_blocks, int32_t nnz, int32_t n, int64_t windows,
                  int64_t b_rows) {
  if (opt && opt->chunk_blocks > 0) return opt->chunk_blocks;
  if (opt && opt->cut_span_blocks != 0) return long_chunk_blocks(num_blocks);
  const bool dense = nnz > 24 * (int64_t)num_blocks;
  const int64_t k = !dense && nnz > 11 * (int64_t)num_blocks ? kChunkUnits / 2 : kChunkUnits;
  int c = dense && num_blocks >= 1 << 15 ? 32 : 8;
  const int64_t work = (int64_t)num_blocks * ceil_div(std::max(n, 1), 64);
  if (even_windows(nnz, num_blocks, windows, b_rows))
    while (c < 256 && c * windows < num_blocks && std::min<int64_t>(work * 64, (int64_t)num_blocks * n) > 64 * 108 * c * c)
      c *= 2;
  while (c < 256 && work > k * c * c) c *= 2;
  return c;
}

// Cut span of the balanced schedule: options->cut_span_blocks, a positive
// multiple of the chunk, or the chunk itself when 0.
dtc_status_t resolve_cut_span(const dtc_spmm_options_t *opt, int chunk, int *span) {
  const int s = opt ? opt->cut_span_blocks : 0;
  if (s < 0) return fail(DTC_ERROR_INVALID_VALUE, "cut_span_blocks must be >= 0");
  if (s > 0 && s % chunk != 0)
    return fail(DTC_ERROR_INVALID_VALUE, "cut_span_blocks must be a multiple of the chunk (" +
                                             std::to_string(chunk) + " blocks)");
  *span = s > 0 ? s : chunk;
  return DTC_SUCCESS;
}

// Balanced workspace: the persistent work counter, then one int2 run per
// chunk; with the deterministic merge, then two partial-tile slots per chunk
// of 16 rows x N floats (N rounded up to 128, a multiple of every
// column-tile width).  Without a chunk size, one run per block covers every
// chunk size.
constexpr size_t kQueueBytes = 256;
size_t balanced_workspace_bytes(int32_t num_blocks) {
  return kQueueBytes + sizeof(int2) * (size_t)std::max<int32_t>(num_blocks, 0);
}
int64_t num_chunks(int32_t num_blocks, int32_t chunk) {
  return ceil_div(std::max<int32_t>(num_blocks, 0), std::max<int32_t>(chunk, 1));
}
size_t balanced_parts_offset(int32_t num_blocks, int32_t chunk) {
  return align_up(kQueueBytes + sizeof(int2) * (size_t)num_chunks(num_blocks, chunk), 256);
}
size_t balanced_workspace_bytes_for(int32_t num_blocks, int32_t n, int32_t chunk, bool det) {
  if (!det) return kQueueBytes + sizeof(int2) * (size_t)num_chunks(num_blocks, chunk);
  const int64_t npad = ceil_div(std::max<int32_t>(n, 1), 128) * 128;
  return balanced_parts_offset(num_blocks, chunk) +
         (size_t)(2 * num_chunks(num_blocks, chunk)) * kBlkH * (size_t)npad * sizeof(float);
}

// The chunk for a workspace of this size: resolve_chunk's, or with the default
// the one by the block count alone where only that one fits.  `need`: the least
// workspace, which does not depend on how the windows are filled.
int fit_chunk(const dtc_spmm_options_t *opt, int32_t num_blocks, int32_t nnz, int32_t n, int32_t num_nodes,
              int32_t b_rows, size_t workspace_bytes, size_t *need) {
  const bool det = opt && opt->deterministic;
  auto bytes = [&](int chunk) { return balanced_workspace_bytes_for(num_blocks, n, chunk, det); };
  const int chunk = resolve_chunk(opt, num_blocks, nnz, n, ceil_div(num_nodes, kBlkH), b_rows);
  const int by_count = long_chunk_blocks(num_blocks);
  if (opt && (opt->chunk_blocks > 0 || opt->cut_span_blocks != 0)) {
    *need = bytes(chunk);
    return chunk;
  }
  *need = bytes(std::max(resolve_chunk(opt, num_blocks, nnz, n, 0, 0), by_count));
  return bytes(chunk) <= workspace_bytes ? chunk : std::max(chunk, by_count);
}

__global__ __launch_bounds__(256) void k_zero(float *c, int64_t count) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) c[i] = 0.f;
}

// C = 0 when B has no rows (every column of A is out of range).
dtc_status_t zero_output(float *c, int32_t m, int32_t n, hipStream_t stream) {
  const int64_t count = (int64_t)m * n;
  if (count == 0) return DTC_SUCCESS;
  const unsigned grid = (unsigned)std::min<int64_t>(65536, ceil_div(count, 256));
  k_zero<<<grid, 256, 0, stream>>>(c, count);
  DTC_LAUNCH_CHECK("zero_output");
  return DTC_SUCCESS;
}

}  // namespace
// TC-GNN's SpMM (DTCSpMM.cpp:97-115, DTCSpMM_kernel.cu:703-808 and
// :1566-1685), the comparison baseline without TC-block compaction.  Its
// format is ME-TCF's phase 1 only: blockPartition, edgeToColumn, edgeToRow.
// One unit per (row window, column tile); for every group of 4 blocks (32
// condensed columns) the wave rescans ALL of the window's edges, scattering
// those whose condensed column falls in the group into the LDS A tile and
// recording each condensed column's original column (TC-GNN's per-block
// sparse_AToX), then gathers B and runs the MFMAs as the ME-TCF kernels do.
// The rescans -- window edges times groups -- are what ME-TCF's compaction
// removes.
template <int VEC>
__global__ __launch_bounds__(256) void spmm_tcgnn_kernel(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const int32_t *__restrict__ e2c, const int32_t *__restrict__ e2r,
    const int32_t *__restrict__ bpart, const float *__restrict__ vals, int32_t W,
    SpmmParams p) {
  __shared__ __attribute__((aligned(16))) float s_tile[kWavesPerBlock][kTileFloats];
  __shared__ int32_t s_atox[kWavesPerBlock][kGroup * kBlkW];
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int ct = blockIdx.x % p.n_ct;
  const int w = (blockIdx.x / p.n_ct) * kWavesPerBlock + wave;
  if (w >= W) return;
  const Cols<1> cols = lane_cols<VEC, 1>(ct, p.N);
  const int64_t r0 = (int64_t)w * kBlkH;
  const int ws = wave_uniform(rowptr[min(r0, (int64_t)p.M)]);
  const int we = wave_uniform(rowptr[min(r0 + kBlkH, (int64_t)p.M)]);
  const int nb = wave_uniform(bpart[w]);
  float *tile = s_tile[wave];
  int32_t *atox = s_atox[wave];
  floatx4 acc[1][VEC];
  zero_acc<VEC, 1>(acc);
  const int g = lane >> 4;
  const int q = lane & 15;
  for (int k0 = 0; k0 < nb; k0 += kGroup) {
    floatx4 *t4 = reinterpret_cast<floatx4 *>(tile);
    const floatx4 z4 = {0.f, 0.f, 0.f, 0.f};
    t4[lane * 2] = z4;
    t4[lane * 2 + 1] = z4;
    if (lane < kGroup * kBlkW) atox[lane] = 0;  // padding slots gather row 0 times 0
    wave_lds_sync();
    for (int e = ws + lane; e < we; e += kWave) {
      const int c = e2c[e];
      const int gg = (c >> 3) - k0;
      if (gg >= 0 && gg < kGroup) {
        const int slot = c & (kBlkW - 1);
        atomicAdd(&tile[gg * (kBlkH * kBlkW) + (e2r[e] & (kBlkH - 1)) * kBlkW + slot],
                  vals ? vals[e] : 1.0f);  // repeated (row, column) pairs add up
        atox[gg * kBlkW + slot] = col[e];
      }
    }
    wave_lds_sync();
    float a[8];
    const floatx4 lo = t4[(g * (kBlkH * kBlkW) + q * kBlkW) / 4];
    const floatx4 hi = t4[(g * (kBlkH * kBlkW) + q * kBlkW) / 4 + 1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[j] = lo[j];
      a[j + 4] = hi[j];
    }
    int rows[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) rows[j] = atox[g * kBlkW + j];
    wave_lds_sync();
    breg_t<DTC_PRECISION_FP32, VEC> breg[1][8];
    gather_ptr<DTC_PRECISION_FP32, VEC, 1>(p, rows, g < nb - k0, cols, breg);
    mfma_group<DTC_PRECISION_FP32, VEC, 1>(a, breg, acc, true);
  }
  store_window<VEC, 1, true>(p, w, cols, acc);
}

}  // namespace dtc

using namespace dtc;

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept.
dtc_status_t noalloc_scratch(void **out) {
  int dev = 0;
  DTC_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(DTC_ERROR_UNSUPPORTED, "device ordinal " + std::to_string(dev) + " beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(DTC_ERROR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return DTC_SUCCESS;
}

}  // namespace

extern "C" {

dtc_status_t dtc_spmm_tcgnn(const int32_t *node_pointer, const int32_t *edge_list,
                            const int32_t *block_partition, const int32_t *edge_to_column,
                            const int32_t *edge_to_row, const float *values, int32_t num_nodes,
                            int32_t nnz, const float *b, int32_t b_rows, int32_t n, float *c,
                            const dtc_spmm_options_t *options, dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (num_nodes < 0 || nnz < 0 || b_rows < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "sizes must be >= 0");
  if (n <= 0) return fail(DTC_ERROR_INVALID_VALUE, "N (feature width) must be >= 1");
  if (options && (options->precision != DTC_PRECISION_FP32 || options->b_dtype != DTC_B_FLOAT32))
    return fail(DTC_ERROR_UNSUPPORTED, "the TC-GNN baseline runs float32 only");
  if (num_nodes == 0) return DTC_SUCCESS;
  if (!node_pointer || !block_partition || !c)
    return fail(DTC_ERROR_INVALID_VALUE, "node_pointer, block_partition and C are required");
  if (nnz > 0 && (!edge_list || !edge_to_column || !edge_to_row))
    return fail(DTC_ERROR_INVALID_VALUE, "edge arrays are required when nnz > 0");
  if (b_rows > 0 && !b) return fail(DTC_ERROR_INVALID_VALUE, "B is NULL");
  dtc_spmm_options_t o{};
  o.precision = DTC_PRECISION_FP32;
  o.vec = options ? options->vec : 0;
  o.subtiles = 1;
  Variant var;
  dtc_status_t st = resolve_shape(&o, n, b, c, false, false, 0, false, false, false, kBuf, &var);
  if (st != DTC_SUCCESS) return st;
  const int32_t W = (int32_t)ceil_div(num_nodes, kBlkH);
  if (b_rows == 0) return zero_output(c, num_nodes, n, stream);
  SpmmParams p{};
  p.B = b;
  p.C = c;
  p.M = num_nodes;
  p.b_rows = b_rows;
  p.N = n;
  p.n_ct = (int32_t)ceil_div(n, 16 * var.vec);
  const int64_t grid = (int64_t)p.n_ct * ceil_div(W, kWavesPerBlock);
  if (grid > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "grid too large");
  switch (var.vec) {
    case 4:
      spmm_tcgnn_kernel<4><<<(unsigned)grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_column,
                                                               edge_to_row, block_partition, values, W, p);
      break;
    case 2:
      spmm_tcgnn_kernel<2><<<(unsigned)grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_column,
                                                               edge_to_row, block_partition, values, W, p);
      break;
    default:
      spmm_tcgnn_kernel<1><<<(unsigned)grid, 256, 0, stream>>>(node_pointer, edge_list, edge_to_column,
                                                               edge_to_row, block_partition, values, W, p);
  }
  DTC_LAUNCH_CHECK("spmm_tcgnn");
  return DTC_SUCCESS;
}

dtc_status_t dtc_spmm_windows(const int32_t *row_window_offset, const uint8_t *tcblocktile_id,
                              const int32_t *tcblock_offset, const int32_t *sparse_atox,
                              const float *tcblock_values, int32_t num_windows,
                              int32_t num_blocks, int32_t nnz,
                              int32_t num_nodes, const void *b, int32_t b_rows, int32_t n,
                              float *c, const dtc_spmm_options_t *options,
                              dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  dtc_status_t st = check_common(tcblocktile_id, tcblock_offset, sparse_atox, num_blocks, nnz,
                                 num_nodes, b, b_rows, n, c, options);
  if (st != DTC_SUCCESS) return st;
  if (!row_window_offset) return fail(DTC_ERROR_INVALID_VALUE, "Rowwindow_offset is NULL");
  if (num_windows < 0 || num_blocks < 0 || nnz < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "num_windows, num_blocks and nnz must be >= 0");
  if (num_blocks > 0 && (!tcblocktile_id || !sparse_atox))
    return fail(DTC_ERROR_INVALID_VALUE, "TCblocktile_id and sparse_AToX_idx are required");
  if ((int64_t)num_windows * kBlkH < num_nodes)
    return fail(DTC_ERROR_INVALID_VALUE,
                "Rowwindow_offset has " + std::to_string(num_windows) + " windows, fewer than num_nodes/16");
  Variant var;
  const int esz = options && options->b_dtype == DTC_B_BFLOAT16 ? 2 : 4;
  const int mode = operand_mode(b_rows, n, esz, nnz, num_blocks, tcblocktile_id, tcblock_values);
  const bool unshared = unshared_columns(nnz, num_blocks);
  st = resolve_shape(options, n, b, c, false, false, num_windows, unshared, num_blocks <= 6 * (int64_t)num_windows,
                     nnz <= 160 * (int64_t)num_windows, mode, &var);
  if (st != DTC_SUCCESS) return st;
  // Only windows that hold output rows are processed.
  const int32_t W = (int32_t)std::min<int64_t>(num_windows, ceil_div(num_nodes, kBlkH));
  if (W == 0) return DTC_SUCCESS;
  if (b_rows == 0) return zero_output(c, num_nodes, n, stream);
  SpmmParams p{};
  p.rwo = row_window_offset;
  p.tile = tcblocktile_id;
  p.off = tcblock_offset;
  p.atox = sparse_atox;
  p.vals = tcblock_values;
  p.B = b;
  p.C = c;
  p.num_windows = W;
  p.M = num_nodes;
  p.b_rows = b_rows;
  p.N = n;
  p.n_ct = (int32_t)ceil_div(n, 16 * var.vec * var.nsub);
  p.num_blocks = num_blocks;
  p.nnz = nnz;
  const bool split = split_windows(W, p.n_ct, num_blocks);
  p.chunk = split ? 1 : windows_per_unit(W, p.n_ct, num_blocks, std::min(n, 16 * var.vec * var.nsub));
  p.num_items = (int32_t)ceil_div(W, p.chunk);
  // (Uniform 2^20 rows of 16, N = 256, ms, side by side and one after another: 3.10
  // and 2.56; R-MAT of 31.4 M entries 4.94 and 5.74, of 8 M, N = 128 1.29 and 2.02;
  // band of 400,000 rows, N = 260 0.304 and 0.337.)
  const bool turn = !split && unshared && tiles_in_turn(p, esz);
  p.long_blocks = long_window(W, num_blocks);
  KernelFn fn = pick_kernel(var, split ? kRunSplit : turn ? kRunWindowsTurn : kRunWindows);
  p.groups = split ? W : (int32_t)ceil_div(p.num_items, kWavesPerBlock);
  p.long_groups = turn ? (int32_t)ceil_div(p.groups, kLongGroups) : 0;
  const int64_t grid = (int64_t)p.n_ct * ((int64_t)p.groups + p.long_groups);
  if (grid > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "grid too large");
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, stream, p.rwo, p.rowid, p.tile, p.off,
                     p.atox, p.vals, p.B, p.C, p);
  DTC_LAUNCH_CHECK("spmm_windows");
  return DTC_SUCCESS;
}

dtc_status_t dtc_spmm_balanced_workspace_size(int32_t num_blocks, size_t *bytes) {
  clear_error();
  if (!bytes) return fail(DTC_ERROR_INVALID_VALUE, "bytes is NULL");
  if (num_blocks < 0) return fail(DTC_ERROR_INVALID_VALUE, "num_blocks must be >= 0");
  *bytes = balanced_workspace_bytes(num_blocks);
  return DTC_SUCCESS;
}

dtc_status_t dtc_spmm_balanced_workspace_size_ex(int32_t num_blocks, int32_t n,
                                                 const dtc_spmm_options_t *options, size_t *bytes) {
  clear_error();
  if (!bytes) return fail(DTC_ERROR_INVALID_VALUE, "bytes is NULL");
  if (num_blocks < 0) return fail(DTC_ERROR_INVALID_VALUE, "num_blocks must be >= 0");
  if (n < 0) return fail(DTC_ERROR_INVALID_VALUE, "N must be >= 0");
  if (options && options->chunk_blocks < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "chunk_blocks must be >= 0");
  const bool det = options && options->deterministic;
  // For every N up to this one: a narrower N can have shorter, i.e. more chunks.
  *bytes = 0;
  for (int64_t m = n;;) {
    const int64_t chunk = resolve_chunk(options, num_blocks, 0, (int32_t)m, 0, 0);
    *bytes = std::max(*bytes, balanced_workspace_bytes_for(num_blocks, (int32_t)m, (int32_t)chunk, det));
    if ((options && (options->chunk_blocks > 0 || options->cut_span_blocks != 0)) || chunk <= 8) break;
    m = kChunkUnits * (chunk / 2) * (chunk / 2) / num_blocks * 64;  // the widest with half the chunk
    if (m == 0) break;
  }
  return DTC_SUCCESS;
}

dtc_status_t dtc_spmm_balanced(const int32_t *tcblock_rowid, const uint8_t *tcblocktile_id,
                               const int32_t *tcblock_offset, const int32_t *sparse_atox,
                               const float *tcblock_values, int32_t num_blocks, int32_t nnz,
                               int32_t num_nodes, const void *b, int32_t b_rows, int32_t n,
                               float *c, const dtc_spmm_options_t *options, void *workspace,
                               size_t workspace_bytes, dtc_stream_t stream_) {
  clear_error();
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  dtc_status_t st = check_common(tcblocktile_id, tcblock_offset, sparse_atox, num_blocks, nnz,
                                 num_nodes, b, b_rows, n, c, options);
  if (st != DTC_SUCCESS) return st;
  if (num_blocks > 0 && (!tcblock_rowid || !tcblocktile_id || !sparse_atox))
    return fail(DTC_ERROR_INVALID_VALUE, "TCblock_rowid, TCblocktile_id and sparse_AToX_idx are required");
  Variant var;
  const int esz = options && options->b_dtype == DTC_B_BFLOAT16 ? 2 : 4;
  const int mode = operand_mode(b_rows, n, esz, nnz, num_blocks, tcblocktile_id, tcblock_values);
  st = resolve_shape(options, n, b, c, true, nnz > (num_blocks >= (1 << 19) ? 11 : 24) * (int64_t)num_blocks, 0, false,
                     false, false, mode, &var);
  if (st != DTC_SUCCESS) return st;
  const bool det = options && options->deterministic;
  size_t need = 0;
  const int chunk = fit_chunk(options, num_blocks, nnz, n, num_nodes, b_rows, workspace_bytes, &need);
  int span = chunk;
  st = resolve_cut_span(options, chunk, &span);
  if (st != DTC_SUCCESS) return st;
  const bool persistent = options && options->persistent;
  if (options && (options->deterministic < 0 || options->deterministic > 1))
    return fail(DTC_ERROR_INVALID_VALUE, "deterministic must be 0 or 1");
  const int32_t W = (int32_t)ceil_div(num_nodes, kBlkH);
  if (W == 0) return DTC_SUCCESS;
  if (num_blocks > 0 && (!workspace || workspace_bytes < need))
    return fail(DTC_ERROR_WORKSPACE,
                "balanced SpMM needs the workspace that dtc_spmm_balanced_workspace_size_ex reports (" +
                    std::to_string(need) + " bytes)");
  if (b_rows == 0 || num_blocks == 0) return zero_output(c, num_nodes, n, stream);
  SpmmParams p{};
  p.rowid = tcblock_rowid;
  p.tile = tcblocktile_id;
  p.off = tcblock_offset;
  p.atox = sparse_atox;
  p.vals = tcblock_values;
  p.B = b;
  p.C = c;
  p.num_windows = W;
  p.num_blocks = num_blocks;
  p.M = num_nodes;
  p.b_rows = b_rows;
  p.N = n;
  p.nnz = nnz;
  p.n_ct = (int32_t)ceil_div(n, 16 * var.vec * var.nsub);
  p.num_items = (int32_t)ceil_div(num_blocks, chunk);
  p.chunk = chunk;
  p.span = span;
  // (Chunks that keep windows up to a span whole run longer, and side by side they
  // lose nothing as labelled by the generator: spans of 256, ms, 3.93 against 4.04.)
  const bool turn = span == chunk && tiles_in_turn(p, esz);
  p.groups = (int32_t)ceil_div(p.num_items, kWavesPerBlock);
  p.queue = persistent ? static_cast<int32_t *>(workspace) : nullptr;
  int2 *runs = reinterpret_cast<int2 *>(static_cast<char *>(workspace) + kQueueBytes);
  p.runs = runs;
  p.parts = det ? reinterpret_cast<float *>(static_cast<char *>(workspace) +
                                            balanced_parts_offset(num_blocks, chunk))
                : nullptr;
  const int64_t prep_waves = p.num_items;
  k_balance_prep<<<(unsigned)ceil_div(prep_waves, kWavesPerBlock), 256, 0, stream>>>(
      tcblock_rowid, num_blocks, num_nodes, n, chunk, span, p.num_items, c, p.queue, runs, det ? 0 : 1);
  DTC_LAUNCH_CHECK("balance_prep");
  if (!persistent) {
    KernelFn fn = pick_kernel(var, turn ? kRunBalancedTurn : kRunBalanced);
    const int64_t grid = (int64_t)p.n_ct * p.groups;
    if (grid > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "grid too large");
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, stream, p.rwo, p.rowid, p.tile, p.off,
                     p.atox, p.vals, p.B, p.C, p);
  } else {
    int dev = 0, cus = 0;
    DTC_HIP_CHECK(hipGetDevice(&dev));
    DTC_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t units = (int64_t)p.num_items * p.n_ct;
    const int64_t grid = std::max<int64_t>(1, std::min<int64_t>(ceil_div(units, kWavesPerBlock),
                                                                (int64_t)cus * 8));
    KernelFn fn = pick_kernel(var, kRunPersistent);
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, stream, p.rwo, p.rowid, p.tile, p.off,
                     p.atox, p.vals, p.B, p.C, p);
  }
  DTC_LAUNCH_CHECK("spmm_balanced");
  if (det) {
    const int64_t grid = (int64_t)p.n_ct * ceil_div(p.num_items, kWavesPerBlock);
    k_balance_fixup<<<(unsigned)grid, 256, 0, stream>>>(tcblock_rowid, p, 16 * var.vec * var.nsub);
    DTC_LAUNCH_CHECK("balance_fixup");
  }
  return DTC_SUCCESS;
}

// dtc_spmm_balanced with the library's fixed scratch array as its workspace:
// no hipMalloc/hipFree and no allocating call.  Everything the kernels read
// from the scratch is written earlier in the same call (chunk runs and the
// persistent counter by the preparation kernel, partial tiles by the SpMM
// kernel), so nothing needs clearing between calls.
dtc_status_t dtc_spmm_balanced_noalloc(const int32_t *tcblock_rowid, const uint8_t *tcblocktile_id,
                                       const int32_t *tcblock_offset, const int32_t *sparse_atox,
                                       const float *tcblock_values, int32_t num_blocks, int32_t nnz,
                                       int32_t num_nodes, const void *b, int32_t b_rows, int32_t n,
                                       float *c, const dtc_spmm_options_t *options,
                                       dtc_stream_t stream) {
  clear_error();
  if (num_blocks < 0 || n < 0) return fail(DTC_ERROR_INVALID_VALUE, "num_blocks and N must be >= 0");
  if (options && options->chunk_blocks < 0)
    return fail(DTC_ERROR_INVALID_VALUE, "chunk_blocks must be >= 0");
  dtc_spmm_options_t o{};
  if (options) o = *options;
  size_t need = 0;
  const int chunk = fit_chunk(options, num_blocks, nnz, n, num_nodes, b_rows, kNoAllocScratchBytes, &need);
  o.chunk_blocks = chunk;
  if (need > kNoAllocScratchBytes)
    return fail(DTC_ERROR_UNSUPPORTED,
                "this SpMM needs " + std::to_string(need) + " bytes of workspace, more than the " +
                    std::to_string(kNoAllocScratchBytes) +
                    " bytes of the allocation-free entry point; use dtc_spmm_balanced with a workspace");
  void *ws = nullptr;
  dtc_status_t st = noalloc_scratch(&ws);
  if (st != DTC_SUCCESS) return st;
  return dtc_spmm_balanced(tcblock_rowid, tcblocktile_id, tcblock_offset, sparse_atox, tcblock_values,
                           num_blocks, nnz, num_nodes, b, b_rows, n, c, &o, ws, kNoAllocScratchBytes,
                           stream);
}

}  // extern "C"
