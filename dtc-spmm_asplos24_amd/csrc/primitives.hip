// Device-wide building blocks for the ME-TCF build on gfx950 (wave64):
// reduce-then-scan prefix sums and a stable LSD radix sort of
// (uint64 key, int32 value) pairs whose per-tile ranking uses wave ballots.
#include <string>

#include "seg_sort.h"

namespace dtc {

// ------------------------------------------------------------------ status

static thread_local std::string g_last_error;

dtc_status_t fail(dtc_status_t st, const std::string &msg) {
  g_last_error = msg;
  return st;
}
void clear_error() { g_last_error.clear(); }

// -------------------------------------------------------------------- scan

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

struct LoadI32 {
  const int32_t *p;
  __device__ __forceinline__ int operator()(int64_t i) const { return p[i]; }
};

template <class Key>
struct LoadKeyChange {
  const Key *k;
  __device__ __forceinline__ int operator()(int64_t i) const {
    return (i == 0 || k[i] != k[i - 1]) ? 1 : 0;
  }
};

template <class Load>
__global__ __launch_bounds__(kScanThreads) void scan_reduce_kernel(Load load, int64_t n,
                                                                    int32_t *partials) {
  __shared__ int smem[4];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int sum = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k * kScanThreads + threadIdx.x;
    if (i < n) sum += load(i);
  }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = smem[0] + smem[1] + smem[2] + smem[3];
}

// Exclusive scan of partials[0..m) in place, one workgroup.
__global__ __launch_bounds__(kScanThreads) void scan_partials_kernel(int32_t *partials,
                                                                      int64_t m) {
  __shared__ int smem[4];
  int carry = 0;
  for (int64_t base = 0; base < m; base += kScanTile) {
    int v[kScanItems];
    int local = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      const int64_t i = base + (int64_t)threadIdx.x * kScanItems + k;
      v[k] = i < m ? partials[i] : 0;
      local += v[k];
    }
    int total;
    const int inc = block256_inclusive_sum(local, smem, total);
    int run = carry + inc - local;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      const int64_t i = base + (int64_t)threadIdx.x * kScanItems + k;
      if (i < m) partials[i] = run;
      run += v[k];
    }
    carry += total;
  }
}

template <class Load>
__global__ __launch_bounds__(kScanThreads) void scan_downsweep_kernel(
    Load load, int32_t *out, int64_t n, const int32_t *partials, int inclusive) {
  __shared__ int smem[4];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int v[kScanItems];
  int local = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    v[k] = i < n ? load(i) : 0;
    local += v[k];
  }
  int total;
  const int inc = block256_inclusive_sum(local, smem, total);
  int run = partials[blockIdx.x] + inc - local;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (inclusive) run += v[k];
    if (i < n) out[i] = run;
    if (!inclusive) run += v[k];
  }
}

size_t scan_workspace_bytes(int64_t n) {
  return align_up(sizeof(int32_t) * (size_t)std::max<int64_t>(1, ceil_div(n, kScanTile)), 256);
}

template <class Load>
static dtc_status_t scan_impl(Load load, int32_t *out, int64_t n, bool inclusive, void *ws,
                              hipStream_t stream) {
  if (n <= 0) return DTC_SUCCESS;
  const int64_t tiles = ceil_div(n, kScanTile);
  if (tiles > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "scan too large");
  int32_t *partials = static_cast<int32_t *>(ws);
  scan_reduce_kernel<Load><<<(unsigned)tiles, kScanThreads, 0, stream>>>(load, n, partials);
  DTC_LAUNCH_CHECK("scan_reduce");
  scan_partials_kernel<<<1, kScanThreads, 0, stream>>>(partials, tiles);
  DTC_LAUNCH_CHECK("scan_partials");
  scan_downsweep_kernel<Load>
      <<<(unsigned)tiles, kScanThreads, 0, stream>>>(load, out, n, partials, inclusive ? 1 : 0);
  DTC_LAUNCH_CHECK("scan_downsweep");
  return DTC_SUCCESS;
}

dtc_status_t scan_i32(const int32_t *in, int32_t *out, int64_t n, bool inclusive, void *ws,
                      hipStream_t stream) {
  return scan_impl(LoadI32{in}, out, n, inclusive, ws, stream);
}

dtc_status_t scan_key_changes(const uint64_t *keys, int32_t *out, int64_t n, void *ws,
                              hipStream_t stream) {
  return scan_impl(LoadKeyChange<uint64_t>{keys}, out, n, true, ws, stream);
}

dtc_status_t scan_key_changes_u32(const uint32_t *keys, int32_t *out, int64_t n, void *ws,
                                  hipStream_t stream) {
  return scan_impl(LoadKeyChange<uint32_t>{keys}, out, n, true, ws, stream);
}

// -------------------------------------------------------------- radix sort

constexpr int kSortThreads = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kRadix = 256;

// Tile maps: tile t covers [start, start + len) of the key array, and the
// count of digit d in it lives at hist[hbase + d * hstride].
//   PlainTiles: tiles of kSortTile keys over the whole array, hist laid out
//     [digit][tile], so one exclusive scan of hist gives every (digit, tile)
//     its first output position;
//   SegTiles: the array is a sequence of segments (segment w' = [csb[w'],
//     csb[w'+1])), each cut into its own tiles (tile t belongs to segment
//     tw[t], segment w' owns tiles [tb[w'], tb[w'+1])), hist laid out
//     [segment][digit][tile of the segment]: the same scan then gives
//     csb[w'] + (entries of w' with a smaller digit) + (entries of digit d in
//     earlier tiles of w'), i.e. each pass sorts every segment on its own.
struct PlainTiles {
  int64_t n;
  int ntiles;
  __device__ __forceinline__ bool valid(int) const { return true; }
  __device__ __forceinline__ void get(int t, int64_t &start, int &len, int64_t &hbase,
                                      int &hstride) const {
    start = (int64_t)t * kSortTile;
    len = (int)min<int64_t>(kSortTile, n - start);
    hbase = t;
    hstride = ntiles;
  }
};

struct SegTiles {
  const int32_t *tw, *tb, *csb;
  const int32_t *ntot;  // number of tiles (the grid may be larger)
  __device__ __forceinline__ bool valid(int t) const { return t < *ntot; }
  __device__ __forceinline__ void get(int t, int64_t &start, int &len, int64_t &hbase,
                                      int &hstride) const {
    const int w = tw[t];
    const int t0 = tb[w];
    const int tl = t - t0;
    start = (int64_t)csb[w] + (int64_t)tl * kSortTile;
    len = (int)min<int64_t>(kSortTile, (int64_t)csb[w + 1] - start);
    hbase = (int64_t)t0 * kRadix + tl;
    hstride = tb[w + 1] - t0;
  }
};

// Digit counts of one tile.
template <class Key, class Tiles>
__global__ __launch_bounds__(kSortThreads) void radix_hist_kernel(const Key *keys, int shift,
                                                                   int32_t *hist, Tiles tiles) {
  __shared__ int cnt[kRadix];
  if (!tiles.valid(blockIdx.x)) {  // past the last tile: the scanned tail reads zeros
    hist[(int64_t)blockIdx.x * kRadix + threadIdx.x] = 0;
    return;
  }
  cnt[threadIdx.x] = 0;
  __syncthreads();
  int64_t start, hbase;
  int len, hstride;
  tiles.get(blockIdx.x, start, len, hbase, hstride);
  Key kreg[kSortItems];  // all loads in flight before the first count
#pragma unroll
  for (int k = 0; k < kSortItems; ++k)
    kreg[k] = keys[start + min(k * kSortThreads + (int)threadIdx.x, len - 1)];
#pragma unroll
  for (int k = 0; k < kSortItems; ++k)
    if (k * kSortThreads + (int)threadIdx.x < len)
      atomicAdd(&cnt[(int)((kreg[k] >> shift) & (kRadix - 1))], 1);
  __syncthreads();
  hist[hbase + (int64_t)threadIdx.x * hstride] = cnt[threadIdx.x];
}

// Stable scatter: element i of the tile goes to offsets[d][tile] + (number of
// earlier elements of the tile with the same digit d).  Tiles are 4,096
// keys.  Wave w owns the tile's elements [1024 w, 1024 w + 1024), taken in 16
// rounds of 64 in index order, so index order is wave-major, then round,
// then lane.  Each wave
// ranks its own elements without workgroup barriers: inside a round the rank
// among equal digits comes from eight ballots (one per digit bit) and a
// popcount, added to the wave's running count of the digit (per-wave LDS
// counters).  Then, once per tile, the four waves' counts give each digit's
// per-wave prefixes and the tile's digit-sorted layout (a scan over the 256
// digits), and the tile is laid out in LDS in digit order and written out so
// that consecutive threads store consecutive elements of one digit's run
// (~16 keys on average: runs, not 4,096 scattered 12-byte writes; with
// 2,048-key tiles the runs of ~8 keys made the scatter 1.5x slower than a
// pass whose few digits give long runs).
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kWaveItems = kSortTile / kSortWaves;  // 1,024 elements per wave

//
// In gives the key and the value words of element i, the first kComputed of
// them from i alone; Out takes them at their place.  Keys and words go through
// the same LDS buffer one after another (a 16 KB buffer instead of one for each
// keeps four to six workgroups on a CU instead of two).
template <class Key>
struct PairIn {
  typedef Key key_type;
  static constexpr int kWords = 1, kComputed = 0;
  const Key *k;
  const int32_t *v;
  __device__ __forceinline__ void tile(int64_t, int, int32_t *, int *) const {}
  __device__ __forceinline__ Key key(int64_t i) const { return k[i]; }
  __device__ __forceinline__ int32_t word(int, int64_t i, int, const int32_t *) const { return v[i]; }
};
template <class Key>
struct PairOut {
  Key *k;
  int32_t *v;
  __device__ __forceinline__ void key(int64_t i, Key x) const { k[i] = x; }
  __device__ __forceinline__ void word(int, int64_t i, int32_t x) const { v[i] = x; }
};

template <class In, class Out, class Tiles>
__global__ __launch_bounds__(kSortThreads) void radix_scatter_kernel(In in, Out out, int shift,
                                                                      const int32_t *offsets,
                                                                      Tiles tiles) {
  typedef typename In::key_type Key;
  constexpr int NW = In::kWords;
  __shared__ int s_off[kRadix];             // global position of the tile's first element of digit d
  __shared__ int s_loc[kRadix];             // local position of the same element
  __shared__ int s_wcnt[kSortWaves][kRadix];  // per-wave digit counts, then per-wave prefixes
  __shared__ int s_scan[kSortWaves];
  __shared__ Key s_keys[kSortTile];
  int32_t *s_word = reinterpret_cast<int32_t *>(s_keys);
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  if (!tiles.valid(blockIdx.x)) return;  // workgroup-uniform
  int64_t start, hbase;
  int len, hstride;
  tiles.get(blockIdx.x, start, len, hbase, hstride);
  const int wbase = wave * kWaveItems;  // tile-relative
  // All of the wave's keys and values are loaded up front (one memory
  // latency for the whole tile).
  Key kreg[kSortItems];
  int32_t vreg[NW][kSortItems];
  in.tile(start, len, s_word, s_scan);
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int i = wbase + r * 64 + lane;
    kreg[r] = i < len ? in.key(start + i) : (Key)0;
#pragma unroll
    for (int w = In::kComputed; w < NW; ++w)
      vreg[w][r] = i < len ? in.word(w, start + i, i, s_word) : 0;
  }
  s_off[tid] = offsets[hbase + (int64_t)tid * hstride];
#pragma unroll
  for (int k = 0; k < kRadix / 64; ++k) s_wcnt[wave][k * 64 + lane] = 0;
  wave_lds_sync();
  int lrank[kSortItems];  // rank among the wave's earlier elements of the same digit
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const bool valid = wbase + r * 64 + lane < len;
    const int d = (int)((kreg[r] >> shift) & (kRadix - 1));
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const bool b = (d >> bit) & 1;
      const uint64_t m = __ballot(b);
      peers &= b ? m : ~m;
    }
    const int rank = __popcll(peers & lt_mask);
    lrank[r] = valid ? s_wcnt[wave][d] + rank : 0;
    wave_lds_sync();
    if (valid && rank == 0) s_wcnt[wave][d] += __popcll(peers);
    wave_lds_sync();
  }
  __syncthreads();
  // per digit d = tid: the waves' exclusive prefixes, and the tile's count of d
  int cnt = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    const int c = s_wcnt[w][tid];
    s_wcnt[w][tid] = cnt;
    cnt += c;
  }
  // exclusive scan of the 256 digit counts: the digit-sorted local layout
  const int inc = wave_inclusive_sum(cnt);
  if (lane == 63) s_scan[wave] = inc;
  __syncthreads();
  int pre = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) pre += w < wave ? s_scan[w] : 0;
  s_loc[tid] = pre + inc - cnt;
  __syncthreads();
  // lrank: place in the tile's layout; pos: place in the output of the element
  // that this thread writes
  int pos[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    if (wbase + r * 64 + lane < len) {
      const int d = (int)((kreg[r] >> shift) & (kRadix - 1));
      lrank[r] += s_loc[d] + s_wcnt[wave][d];
      s_keys[lrank[r]] = kreg[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int j = r * kSortThreads + tid;
    if (j < len) {
      const Key key = s_keys[j];
      const int d = (int)((key >> shift) & (kRadix - 1));
      pos[r] = s_off[d] + (j - s_loc[d]);
      out.key(pos[r], key);
    }
  }
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
      if (wbase + r * 64 + lane < len)
        s_word[lrank[r]] = w < In::kComputed
                               ? in.word(w, start + wbase + r * 64 + lane, 0, nullptr)
                               : vreg[w][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
      if (r * kSortThreads + tid < len) out.word(w, pos[r], s_word[r * kSortThreads + tid]);
  }
}

size_t radix_sort_workspace_bytes(int64_t n) {
  const int64_t ntiles = std::max<int64_t>(1, ceil_div(n, kSortTile));
  return align_up(sizeof(int32_t) * (size_t)(ntiles * kRadix), 256) +
         scan_workspace_bytes(ntiles * kRadix);
}

dtc_status_t radix_sort_pairs(uint64_t *keys0, int32_t *vals0, uint64_t *keys1,
                              int32_t *vals1, int64_t n, int key_bits, bool *result_in_1,
                              void *ws, hipStream_t stream) {
  *result_in_1 = false;
  if (n <= 1 || key_bits <= 0) return DTC_SUCCESS;
  const int64_t ntiles = ceil_div(n, kSortTile);
  if (ntiles * kRadix > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "sort too large");
  Carver c(ws);
  int32_t *hist = c.take<int32_t>((size_t)(ntiles * kRadix));
  void *scan_ws = c.take<char>(scan_workspace_bytes(ntiles * kRadix));
  uint64_t *kin = keys0, *kout = keys1;
  int32_t *vin = vals0, *vout = vals1;
  bool in_1 = false;
  const PlainTiles tiles{n, (int)ntiles};
  for (int shift = 0; shift < key_bits; shift += 8) {
    radix_hist_kernel<uint64_t, PlainTiles>
        <<<(unsigned)ntiles, kSortThreads, 0, stream>>>(kin, shift, hist, tiles);
    DTC_LAUNCH_CHECK("radix_hist");
    dtc_status_t st = scan_i32(hist, hist, ntiles * kRadix, false, scan_ws, stream);
    if (st != DTC_SUCCESS) return st;
    radix_scatter_kernel<<<(unsigned)ntiles, kSortThreads, 0, stream>>>(
        PairIn<uint64_t>{kin, vin}, PairOut<uint64_t>{kout, vout}, shift, hist, tiles);
    DTC_LAUNCH_CHECK("radix_scatter");
    std::swap(kin, kout);
    std::swap(vin, vout);
    in_1 = !in_1;
  }
  *result_in_1 = in_1;
  return DTC_SUCCESS;
}

size_t seg_radix_sort_workspace_bytes(int64_t n, int64_t segments) {
  const int64_t ntiles = std::max<int64_t>(1, ceil_div(n, kSortTile) + segments);
  return align_up(sizeof(int32_t) * (size_t)(ntiles * kRadix), 256) +
         scan_workspace_bytes(ntiles * kRadix);
}

int64_t seg_radix_tile_size() { return kSortTile; }

dtc_status_t seg_radix_sort_pairs_u32(uint32_t *keys0, int32_t *vals0, uint32_t *keys1,
                                      int32_t *vals1, int key_bits, const int32_t *tw,
                                      const int32_t *tb, const int32_t *csb,
                                      const int32_t *ntiles_dev, int64_t ntiles,
                                      bool *result_in_1, void *ws, hipStream_t stream) {
  *result_in_1 = false;
  if (ntiles <= 0 || key_bits <= 0) return DTC_SUCCESS;
  if (ntiles * kRadix > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "sort too large");
  Carver c(ws);
  int32_t *hist = c.take<int32_t>((size_t)(ntiles * kRadix));
  void *scan_ws = c.take<char>(scan_workspace_bytes(ntiles * kRadix));
  uint32_t *kin = keys0, *kout = keys1;
  int32_t *vin = vals0, *vout = vals1;
  bool in_1 = false;
  const SegTiles tiles{tw, tb, csb, ntiles_dev};
  for (int shift = 0; shift < key_bits; shift += 8) {
    radix_hist_kernel<uint32_t, SegTiles>
        <<<(unsigned)ntiles, kSortThreads, 0, stream>>>(kin, shift, hist, tiles);
    DTC_LAUNCH_CHECK("radix_hist");
    dtc_status_t st = scan_i32(hist, hist, ntiles * kRadix, false, scan_ws, stream);
    if (st != DTC_SUCCESS) return st;
    radix_scatter_kernel<<<(unsigned)ntiles, kSortThreads, 0, stream>>>(
        PairIn<uint32_t>{kin, vin}, PairOut<uint32_t>{kout, vout}, shift, hist, tiles);
    DTC_LAUNCH_CHECK("radix_scatter");
    std::swap(kin, kout);
    std::swap(vin, vout);
    in_1 = !in_1;
  }
  *result_in_1 = in_1;
  return DTC_SUCCESS;
}

// ------------------------------------------------------------ CSR transpose
//
// Stable sort of the edges by column, carrying (edge, row).  The first pass
// reads the columns themselves and makes edge and row on the way, the last one
// writes the transposed arrays, so that an edge moves 4 + 12 bytes in the first
// pass and 12 + 12 in each other one.  12.2 M edges of 60,000 columns: check and
// counts 19 us, passes 103 and 86 (3.4 TB/s: runs of 16 elements), counts 21,
// row pointer 14; with 64-bit keys, a kernel that made them and one that looked
// every edge's row up at the end it took 420 us.

// Edges in CSR order.  The row of every edge of the tile: each row that starts
// in the tile marks its first entry (a later one overrides an empty one before
// it), and an entry's row is the largest mark up to it.
struct EdgeIn {
  typedef uint32_t key_type;
  static constexpr int kWords = 2, kComputed = 1;
  const int32_t *col, *rowptr;
  int32_t M;
  __device__ __forceinline__ void tile(int64_t start, int len, int32_t *s_row, int *s_scan) const {
    const int tid = threadIdx.x, lane = tid & 63;
    const int4 none = make_int4(0, 0, 0, 0);
    int4 *mine = reinterpret_cast<int4 *>(s_row) + tid * (kSortItems / 4);
#pragma unroll
    for (int k = 0; k < kSortItems / 4; ++k) mine[k] = none;
    // rows of the tile's first and last entry: the last r with rowptr[r] <= e
    const int e0 = (int)start, e1 = (int)start + len - 1;
    const int r0 = wave_lower_bound<int32_t>(rowptr, 0, M + 1, e0 + 1) - 1;
    const int r1 = wave_lower_bound<int32_t>(rowptr, r0 + 1, M + 1, e1 + 1) - 1;
    __syncthreads();
    for (int64_t r = (int64_t)r0 + 1 + tid; r <= r1; r += kSortThreads)
      atomicMax(&s_row[rowptr[r] - e0], (int)r);
    __syncthreads();
    int m[kSortItems];
    int top = r0;
#pragma unroll
    for (int k = 0; k < kSortItems / 4; ++k) {
      const int4 v = mine[k];
      m[4 * k] = top = max(top, v.x);
      m[4 * k + 1] = top = max(top, v.y);
      m[4 * k + 2] = top = max(top, v.z);
      m[4 * k + 3] = top = max(top, v.w);
    }
    int up = top;  // largest mark of this and the lower lanes
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int t = __shfl_up(up, d, kWave);
      if (lane >= d) up = max(up, t);
    }
    if (lane == kWave - 1) s_scan[tid >> 6] = up;
    int below = __shfl_up(up, 1, kWave);
    if (lane == 0) below = r0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w)
      if (w < (tid >> 6)) below = max(below, s_scan[w]);
#pragma unroll
    for (int k = 0; k < kSortItems / 4; ++k)
      mine[k] = make_int4(max(m[4 * k], below), max(m[4 * k + 1], below), max(m[4 * k + 2], below),
                          max(m[4 * k + 3], below));
    __syncthreads();
  }
  __device__ __forceinline__ uint32_t key(int64_t i) const { return (uint32_t)col[i]; }
  __device__ __forceinline__ int32_t word(int w, int64_t i, int j, const int32_t *s_row) const {
    return w == 0 ? (int32_t)i : s_row[j];
  }
};
struct EdgePairIn {
  typedef uint32_t key_type;
  static constexpr int kWords = 2, kComputed = 0;
  const uint32_t *k;
  const int32_t *edge, *row;
  __device__ __forceinline__ void tile(int64_t, int, int32_t *, int *) const {}
  __device__ __forceinline__ uint32_t key(int64_t i) const { return k[i]; }
  __device__ __forceinline__ int32_t word(int w, int64_t i, int, const int32_t *) const {
    return w == 0 ? edge[i] : row[i];
  }
};
struct EdgePairOut {
  uint32_t *k;
  int32_t *edge, *row;
  __device__ __forceinline__ void key(int64_t i, uint32_t x) const { k[i] = x; }
  __device__ __forceinline__ void word(int w, int64_t i, int32_t x) const {
    if (w == 0) edge[i] = x;
    else row[i] = x;
  }
};

__global__ void transpose_flags_kernel(int32_t *f) {
  if (threadIdx.x == 0 && blockIdx.x == 0) f[0] = 0;
}

// The digit counts of the first pass together with the checks of the CSR: 1
// row pointer decreases, 2 column outside [0, K), 4 its ends.
__global__ __launch_bounds__(kSortThreads) void transpose_check_kernel(
    const int32_t *rowptr, const int32_t *col, int32_t M, int32_t K, int32_t nnz, int32_t ntiles,
    int32_t *hist, int32_t *flags) {
  __shared__ int cnt[kRadix];
  const int64_t tid = (int64_t)blockIdx.x * kSortThreads + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kSortThreads;
  int f = 0;
  for (int64_t r = tid; r < M; r += stride)
    if (rowptr[r] > rowptr[r + 1]) f |= 1;
  if (tid == 0 && (rowptr[0] != 0 || rowptr[M] != nnz)) f |= 4;
  if ((int)blockIdx.x < ntiles) {  // workgroup-uniform
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t start = (int64_t)blockIdx.x * kSortTile;
    const int len = (int)min<int64_t>(kSortTile, nnz - start);
    int c[kSortItems];
#pragma unroll
    for (int k = 0; k < kSortItems; ++k)
      c[k] = col[start + min(k * kSortThreads + (int)threadIdx.x, len - 1)];
#pragma unroll
    for (int k = 0; k < kSortItems; ++k) {
      if (c[k] < 0 || c[k] >= K) f |= 2;
      if (k * kSortThreads + (int)threadIdx.x < len) atomicAdd(&cnt[c[k] & (kRadix - 1)], 1);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
  }
  if (f) atomicOr(flags, f);
}

// rowptr_t[c] = edges of columns below c.
__global__ __launch_bounds__(kSortThreads) void transpose_rowptr_kernel(const uint32_t *keys,
                                                                        int32_t nnz, int32_t K,
                                                                        int32_t *rowptr_t) {
  const int64_t i = (int64_t)blockIdx.x * kSortThreads + threadIdx.x;
  if (i <= K) rowptr_t[i] = lower_bound_dev<uint32_t>(keys, 0, nnz, (uint32_t)i);
}

struct TransposeWs {
  int32_t *flags, *hist;
  uint32_t *keys[2];
  int32_t *edge, *row;  // of the passes between the first and the last
  int32_t *edge1, *row1;
  void *scan;
  size_t bytes;
};

static TransposeWs carve_transpose(void *ws, int64_t nnz) {
  Carver c(ws);
  TransposeWs t;
  const size_t n = (size_t)std::max<int64_t>(nnz, 1);
  const int64_t counts = ceil_div((int64_t)n, kSortTile) * kRadix;
  t.flags = c.take<int32_t>(64);
  for (int i = 0; i < 2; ++i) t.keys[i] = c.take<uint32_t>(n);
  t.edge = c.take<int32_t>(n);
  t.row = c.take<int32_t>(n);
  t.edge1 = c.take<int32_t>(n);
  t.row1 = c.take<int32_t>(n);
  t.hist = c.take<int32_t>((size_t)counts);
  t.scan = c.take<char>(scan_workspace_bytes(counts));
  t.bytes = c.used();
  return t;
}

size_t transpose_workspace_bytes(int64_t nnz) { return carve_transpose(nullptr, nnz).bytes; }

dtc_status_t transpose_edges(const int32_t *rowptr, const int32_t *col, int32_t M, int32_t K,
                             int32_t nnz, int32_t *rowptr_t, int32_t *col_t, int32_t *perm,
                             void *workspace, hipStream_t stream) {
  const TransposeWs t = carve_transpose(workspace, nnz);
  const int64_t ntiles = ceil_div(nnz, kSortTile);
  if (ntiles * kRadix > INT32_MAX) return fail(DTC_ERROR_UNSUPPORTED, "sort too large");
  transpose_flags_kernel<<<1, 64, 0, stream>>>(t.flags);
  DTC_LAUNCH_CHECK("flags_init");
  const unsigned check = (unsigned)std::max<int64_t>(std::max<int64_t>(ntiles, 1),
                                                     std::min<int64_t>(1024, ceil_div(M, kSortThreads)));
  transpose_check_kernel<<<check, kSortThreads, 0, stream>>>(rowptr, col, M, K, nnz, (int32_t)ntiles,
                                                             t.hist, t.flags);
  DTC_LAUNCH_CHECK("transpose_check");
  int32_t flags = 0;
  DTC_HIP_CHECK(hipMemcpyAsync(&flags, t.flags, 4, hipMemcpyDeviceToHost, stream));
  DTC_HIP_CHECK(hipStreamSynchronize(stream));
  if (flags)
    return fail(DTC_ERROR_INVALID_CSR, "invalid CSR for transpose (flags " + std::to_string(flags) + ")");
  int key_bits = 1;
  while (key_bits < 31 && (int64_t(1) << key_bits) < K) ++key_bits;
  const PlainTiles tiles{nnz, (int)ntiles};
  int at = 0;  // keys[at]: the passes' keys so far
  for (int shift = 0; shift < key_bits && nnz > 0; shift += 8) {
    const bool last = shift + 8 >= key_bits;
    uint32_t *kin = t.keys[at], *kout = t.keys[at ^ 1];
    int32_t *ein = at ? t.edge1 : t.edge, *rin = at ? t.row1 : t.row;
    const EdgePairOut out = {kout, last ? perm : at ? t.edge : t.edge1,
                             last ? col_t : at ? t.row : t.row1};
    if (shift > 0) {
      radix_hist_kernel<uint32_t, PlainTiles>
          <<<(unsigned)ntiles, kSortThreads, 0, stream>>>(kin, shift, t.hist, tiles);
      DTC_LAUNCH_CHECK("radix_hist");
    }
    dtc_status_t st = scan_i32(t.hist, t.hist, ntiles * kRadix, false, t.scan, stream);
    if (st != DTC_SUCCESS) return st;
    if (shift == 0)
      radix_scatter_kernel<<<(unsigned)ntiles, kSortThreads, 0, stream>>>(
          EdgeIn{col, rowptr, M}, out, shift, t.hist, tiles);
    else
      radix_scatter_kernel<<<(unsigned)ntiles, kSortThreads, 0, stream>>>(
          EdgePairIn{kin, ein, rin}, out, shift, t.hist, tiles);
    DTC_LAUNCH_CHECK("radix_scatter");
    at ^= 1;
  }
  transpose_rowptr_kernel<<<(unsigned)ceil_div((int64_t)K + 1, kSortThreads), kSortThreads, 0,
                            stream>>>(t.keys[at], nnz, K, rowptr_t);
  DTC_LAUNCH_CHECK("transpose_rowptr");
  return DTC_SUCCESS;
}

}  // namespace dtc

extern "C" {

const char *dtc_status_string(dtc_status_t status) {
  switch (status) {
    case DTC_SUCCESS: return "success";
    case DTC_ERROR_INVALID_VALUE: return "invalid value";
    case DTC_ERROR_UNSUPPORTED: return "unsupported";
    case DTC_ERROR_WORKSPACE: return "workspace too small";
    case DTC_ERROR_INVALID_CSR: return "invalid CSR";
    case DTC_ERROR_HIP: return "HIP error";
    case DTC_ERROR_INCONSISTENT: return "inconsistent blockPartition";
  }
  return "unknown status";
}

const char *dtc_last_error(void) { return dtc::g_last_error.c_str(); }

int32_t dtc_version(void) { return 10000; }

}  // extern "C"
