// Device-side graph construction: edge list -> CSR (+ CSC for directed
// graphs) and the seeded generators, on the GPU, with the same result as the
// host build (host_graph.cpp) bit for bit: self-loops dropped, optional
// symmetrization, rows sorted by (column, weight), optional dedup keeping the
// minimum weight.
//
// Reference: DAWN::Matrix::coo2Csr / coo2Csr_Weighted (src/matrix.cpp:28-82:
// row counts, prefix sum, copy of the row-sorted COO), DAWN::Matrix::
// transpose / transpose_Weighted (matrix.cpp:3-26: a sort of the COO by
// (row, column[, value])), DAWN::IO::readGraph* (src/io.cpp:2-192: 0-based
// entries, self-loops dropped, both directions for undirected graphs),
// DAWN::Graph::createGraph (src/graph.cpp:9-77).
//
// Pipeline, on the graph's stream:
//   emit     one 64-bit key per directed entry, u << vb | v (vb = bits of
//            n), and its weight; a self-loop becomes the key ~0, which sorts
//            after every real key, and is counted.
//   sort     stable LSD radix sort, 8-bit digits over the 2*vb key bits
//            (own kernels: per-tile digit counts, a device-wide exclusive
//            scan of the counts in digit-major order, and a scatter that
//            ranks each tile in LDS by wave ballots and writes it out in
//            digit runs).  Weighted graphs first sort the entry indices by
//            weight, so that equal keys come out weight-ascending.
//   compact  the first entry of each run of equal keys (dedup) or every
//            entry: column and weight in place, row offsets from the row
//            boundaries; for directed graphs the transposed keys v << vb | u
//            of the kept entries, sorted the same way, give the in-edge CSC.
// Heavy-vertex chunk lists come from the device offsets (count, scan,
// write), as the host build does from its offsets.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"

namespace dawn {

int validate_csr(const dawn_csr* csr);

namespace {

constexpr int kRsPer = 16;                 // keys per thread per tile
constexpr int kRsTile = kBlock * kRsPer;   // 4096 keys per workgroup
constexpr int kScanPer = 16;
constexpr int kScanTile = kBlock * kScanPer;
constexpr uint64_t kSentinel = ~0ull;

// ---- counter-based random numbers (the host generators' draws) -----------

__device__ __forceinline__ uint64_t d_splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ uint64_t d_rng(uint64_t seed, uint64_t stream, uint64_t index) {
  return d_splitmix64(d_splitmix64(seed * 0xD1B54A32D192ED03ull + stream) ^
                      (index * 0x9E3779B97F4A7C15ull));
}

__device__ __forceinline__ uint32_t d_bounded32(uint64_t r, uint32_t range) {
  return (uint32_t)(((r >> 32) * (uint64_t)range) >> 32);
}

// Streams of the host generators (host_graph.cpp).
enum : uint64_t { kStPairU = 1, kStPairV = 2, kStWeight = 3, kStRmat = 4, kStExtra = 5 };

// ---- workgroup scans ------------------------------------------------------

__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t x) {
  const int l = lane_id();
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (l >= o) x += y;
  }
  return x;
}

// Exclusive scan of one value per thread over the workgroup (kBlock
// threads); *total receives the sum.  Every thread must call it.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t* total) {
  __shared__ uint32_t s_w[kBlock / kWave];
  const int w = threadIdx.x / kWave;
  const uint32_t inc = wave_incl_scan_u32(x);
  if (lane_id() == kWave - 1) s_w[w] = inc;
  __syncthreads();
  uint32_t base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kBlock / kWave; i++) {
    if (i < w) base += s_w[i];
    tot += s_w[i];
  }
  __syncthreads();  // s_w is reused by the next call
  *total = tot;
  return base + inc - x;
}

// Sum of each tile of kScanTile values.
__global__ void __launch_bounds__(kBlock) scan_sums_kernel(const uint32_t* in, int64_t n,
                                                           uint32_t* sums) {
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  uint32_t x = 0;
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    if (i < n) x += in[i];
  }
  uint32_t tot;
  (void)block_excl_scan(x, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Exclusive scan of each tile in place, plus the tile's offset.
__global__ void __launch_bounds__(kBlock) scan_tiles_kernel(uint32_t* data, int64_t n,
                                                            const uint32_t* tile_off) {
  __shared__ uint32_t s[kScanTile];
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    s[r * kBlock + threadIdx.x] = i < n ? data[i] : 0u;
  }
  __syncthreads();
  uint32_t loc[kScanPer], x = 0;
#pragma unroll
  for (int j = 0; j < kScanPer; j++) {
    loc[j] = x;
    x += s[threadIdx.x * kScanPer + j];
  }
  uint32_t tot;
  const uint32_t base = block_excl_scan(x, &tot) + (tile_off ? tile_off[blockIdx.x] : 0u);
#pragma unroll
  for (int j = 0; j < kScanPer; j++) s[threadIdx.x * kScanPer + j] = base + loc[j];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    if (i < n) data[i] = s[r * kBlock + threadIdx.x];
  }
}

// Device-wide exclusive scan of n uint32 values in place (sum < 2^32).
struct ScanTemp {
  std::vector<DevBuf<uint32_t>*> levels;
  ~ScanTemp() {
    for (auto* b : levels) delete b;
  }
};

int excl_scan(uint32_t* data, int64_t n, hipStream_t s, ScanTemp& t, size_t level = 0) {
  if (n <= 0) return DAWN_OK;
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  if (tiles == 1) {
    scan_tiles_kernel<<<1, kBlock, 0, s>>>(data, n, nullptr);
    DAWN_HIP(hipGetLastError());
    return DAWN_OK;
  }
  if (t.levels.size() <= level) t.levels.push_back(new DevBuf<uint32_t>());
  DevBuf<uint32_t>& sums = *t.levels[level];
  DAWN_TRY(sums.alloc((size_t)tiles));
  scan_sums_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(data, n, sums.p);
  DAWN_HIP(hipGetLastError());
  DAWN_TRY(excl_scan(sums.p, tiles, s, t, level + 1));
  scan_tiles_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(data, n, sums.p);
  DAWN_HIP(hipGetLastError());
  return DAWN_OK;
}

// ---- LSD radix sort ---------------------------------------------------------

// Digit counts of each tile, digit-major: hist[d * tiles + tile].
__global__ void __launch_bounds__(kBlock) rs_hist_kernel(const uint64_t* keys, int64_t N,
                                                         int shift, int64_t tiles,
                                                         uint32_t* hist) {
  __shared__ uint32_t s_cnt[256];
  s_cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)blockIdx.x * kRsTile;
#pragma unroll
  for (int r = 0; r < kRsPer; r++) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    if (i < N) atomicAdd(&s_cnt[(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * tiles + blockIdx.x] = s_cnt[threadIdx.x];
}

// One stable scatter pass: the tile is ranked in LDS (key order within a
// digit = index order), then written out digit run by digit run.
// offs = scanned counts: offs[d * tiles + tile] = output position of the
// tile's first key of digit d.  A wave ranks a segment of its own against its
// own digit counts, so that the workgroup meets four times a tile instead of
// three times a round (33.5 M keys: 231 -> 137 us a pass; moving them takes 113
// at the copy's rate).
template <bool VALS>
__global__ void __launch_bounds__(kBlock) rs_scatter_kernel(const uint64_t* kin,
                                                            const int32_t* vin, uint64_t* kout,
                                                            int32_t* vout, int64_t N, int shift,
                                                            int64_t tiles, const uint32_t* offs) {
  constexpr int kWaves = kBlock / kWave;
  static_assert(kBlock == 256 && kRsTile == kRsPer * kBlock, "a thread per digit, kRsPer rounds a wave");
  __shared__ uint64_t s_key[kRsTile];
  __shared__ int32_t s_val[VALS ? kRsTile : 1];
  __shared__ uint32_t s_start[256], s_gbase[256];
  __shared__ uint32_t s_wcnt[kWaves][256];  // counts, then first positions
  const int tid = threadIdx.x;
  const int wv = tid / kWave;
  const int64_t t0 = (int64_t)blockIdx.x * kRsTile;
  const int nt = (int)min<int64_t>(kRsTile, N - t0);
  const int seg = wv * (kRsTile / kWaves) + lane_id();
  uint64_t k[kRsPer];
  int32_t v[kRsPer];
  uint32_t rank[kRsPer];  // within the wave's keys of that digit
#pragma unroll
  for (int r = 0; r < kRsPer; r++) k[r] = seg + r * kWave < nt ? kin[t0 + seg + r * kWave] : 0ull;
  if (VALS) {
#pragma unroll
    for (int r = 0; r < kRsPer; r++) v[r] = seg + r * kWave < nt ? vin[t0 + seg + r * kWave] : 0;
  }
  const uint32_t base = offs[(int64_t)tid * tiles + blockIdx.x];
#pragma unroll
  for (int w = 0; w < kWaves; w++) s_wcnt[w][tid] = 0;
  __syncthreads();
  const uint64_t below = lanes_below_mask();
#pragma unroll
  for (int r = 0; r < kRsPer; r++) {
    const uint32_t d = (uint32_t)(k[r] >> shift) & 255u;
    const bool valid = seg + r * kWave < nt;
    uint64_t eq = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      eq &= bit ? m : ~m;
    }
    const uint32_t at = (uint32_t)__popcll(eq & below);
    const uint32_t had = s_wcnt[wv][d];
    wave_lds_sync();
    if (valid && at == 0) s_wcnt[wv][d] = had + (uint32_t)__popcll(eq);
    wave_lds_sync();
    rank[r] = had + at;
  }
  __syncthreads();
  uint32_t c[kWaves], sum = 0, tot;
#pragma unroll
  for (int w = 0; w < kWaves; w++) {
    c[w] = sum;
    sum += s_wcnt[w][tid];
  }
  const uint32_t st = block_excl_scan(sum, &tot);
  s_start[tid] = st;
  s_gbase[tid] = base;
#pragma unroll
  for (int w = 0; w < kWaves; w++) s_wcnt[w][tid] = st + c[w];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRsPer; r++) {
    if (seg + r * kWave >= nt) continue;
    const uint32_t pos = s_wcnt[wv][(uint32_t)(k[r] >> shift) & 255u] + rank[r];
    s_key[pos] = k[r];
    if (VALS) s_val[pos] = v[r];
  }
  __syncthreads();
#pragma unroll 4
  for (int i = tid; i < nt; i += kBlock) {
    const uint64_t key = s_key[i];
    const uint32_t dg = (uint32_t)(key >> shift) & 255u;
    const int64_t pos = (int64_t)s_gbase[dg] + (i - s_start[dg]);
    kout[pos] = key;
    if (VALS) vout[pos] = s_val[i];
  }
}

struct SortTemp {
  DevBuf<uint32_t> hist;
  ScanTemp scan;
};

// Stable LSD radix sort of N keys on their low `bits` bits, with optional
// int32 payload; ping-pongs between (k0, v0) and (k1, v1).  *in1 tells
// which buffer holds the result.
int radix_sort(uint64_t* k0, uint64_t* k1, int32_t* v0, int32_t* v1, int64_t N, int bits,
               hipStream_t s, SortTemp& t, bool* in1) {
  *in1 = false;
  if (N <= 1 || bits <= 0) return DAWN_OK;
  const int64_t tiles = (N + kRsTile - 1) / kRsTile;
  DAWN_TRY(t.hist.alloc((size_t)tiles * 256));
  bool cur1 = false;
  for (int shift = 0; shift < bits; shift += 8) {
    const uint64_t* ki = cur1 ? k1 : k0;
    uint64_t* ko = cur1 ? k0 : k1;
    const int32_t* vi = cur1 ? v1 : v0;
    int32_t* vo = cur1 ? v0 : v1;
    rs_hist_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(ki, N, shift, tiles, t.hist.p);
    DAWN_HIP(hipGetLastError());
    DAWN_TRY(excl_scan(t.hist.p, tiles * 256, s, t.scan));
    if (v0)
      rs_scatter_kernel<true><<<(unsigned)tiles, kBlock, 0, s>>>(ki, vi, ko, vo, N, shift, tiles,
                                                                 t.hist.p);
    else
      rs_scatter_kernel<false><<<(unsigned)tiles, kBlock, 0, s>>>(ki, nullptr, ko, nullptr, N,
                                                                  shift, tiles, t.hist.p);
    DAWN_HIP(hipGetLastError());
    cur1 = !cur1;
  }
  *in1 = cur1;
  return DAWN_OK;
}

// ---- emission of directed entries -----------------------------------------

// Generator / edge-list parameters of one emit launch.
struct EmitArgs {
  int kind;             // 0 edge list, 1 ER, 2 RMAT, 3 grid
  int32_t n;
  int64_t count;        // pairs
  int symmetrize;
  int weighted;
  int vb;               // key bits of a vertex id
  uint64_t seed;
  int32_t wmin, wmax;
  // ER / grid
  int32_t side;
  int64_t horiz, grid_edges;
  // RMAT
  int32_t scale;
  uint64_t ta, tb, tc;
  // edge list
  const int32_t* u;
  const int32_t* v;
  const int32_t* w;
  // out
  uint64_t* keys;
  int32_t* wts;
  unsigned long long* selfloops;
  unsigned int* bad;    // edge list: an id out of range or a negative weight
};

__device__ __forceinline__ int32_t d_weight(const EmitArgs& a, int64_t i) {
  const uint32_t range = (uint32_t)((int64_t)a.wmax - a.wmin + 1);
  return a.wmin + (int32_t)d_bounded32(d_rng(a.seed, kStWeight, (uint64_t)i), range);
}

// Pair i of the generator or edge list (the host generators' formulas).
__device__ __forceinline__ void d_pair(const EmitArgs& a, int64_t i, int32_t& u, int32_t& v,
                                       int32_t& w) {
  w = 1;
  if (a.kind == 0) {
    u = a.u[i];
    v = a.v[i];
    if (a.w) w = a.w[i];
    return;
  }
  if (a.kind == 1) {
    u = (int32_t)d_bounded32(d_rng(a.seed, kStPairU, (uint64_t)i), (uint32_t)a.n);
    v = (int32_t)d_bounded32(d_rng(a.seed, kStPairV, (uint64_t)i), (uint32_t)a.n);
  } else if (a.kind == 2) {
    uint32_t uu = 0, vv = 0;
    uint64_t r = 0;
    for (int32_t l = 0; l < a.scale; l++) {
      if ((l & 1) == 0) r = d_rng(a.seed, kStRmat, (uint64_t)i * 16 + (uint64_t)(l >> 1));
      const uint64_t x = (l & 1) ? (r >> 32) : (r & 0xffffffffull);
      uint32_t ub, vbit;
      if (x < a.ta) { ub = 0; vbit = 0; }
      else if (x < a.tb) { ub = 0; vbit = 1; }
      else if (x < a.tc) { ub = 1; vbit = 0; }
      else { ub = 1; vbit = 1; }
      uu = (uu << 1) | ub;
      vv = (vv << 1) | vbit;
    }
    u = (int32_t)uu;
    v = (int32_t)vv;
  } else {
    if (i < a.horiz) {
      const int64_t r = i / (a.side - 1), c = i % (a.side - 1);
      u = (int32_t)(r * a.side + c);
      v = u + 1;
    } else if (i < a.grid_edges) {
      const int64_t j = i - a.horiz;
      const int64_t r = j / a.side, c = j % a.side;
      u = (int32_t)(r * a.side + c);
      v = u + a.side;
    } else {
      const int64_t j = i - a.grid_edges;
      u = (int32_t)d_bounded32(d_rng(a.seed, kStExtra, (uint64_t)(2 * j)), (uint32_t)a.n);
      v = (int32_t)d_bounded32(d_rng(a.seed, kStExtra, (uint64_t)(2 * j + 1)), (uint32_t)a.n);
    }
  }
  if (a.weighted) w = d_weight(a, i);
}

// Entries of pair i at 2i, 2i+1 (symmetrized) or i.
__global__ void __launch_bounds__(kBlock) emit_kernel(EmitArgs a) {
  unsigned long long loops = 0;
  unsigned bad = 0;
  const int per = a.symmetrize ? 2 : 1;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < a.count;
       i += (int64_t)gridDim.x * kBlock) {
    int32_t u, v, w;
    d_pair(a, i, u, v, w);
    if (a.kind == 0 && (u < 0 || u >= a.n || v < 0 || v >= a.n || w < 0)) {
      bad = 1;
      u = v = 0;  // recorded as a self-loop; the call fails
    }
    uint64_t k0 = kSentinel, k1 = kSentinel;
    if (u != v) {
      k0 = ((uint64_t)u << a.vb) | (uint64_t)v;
      k1 = ((uint64_t)v << a.vb) | (uint64_t)u;
    } else {
      loops += 1;
    }
    a.keys[per * i] = k0;
    if (a.weighted) a.wts[per * i] = w;
    if (per == 2) {
      a.keys[2 * i + 1] = k1;
      if (a.weighted) a.wts[2 * i + 1] = w;
    }
  }
  loops = wave_sum_u64(loops);
  if (lane_id() == 0 && loops) atomicAdd(a.selfloops, loops);
  if (bad) atomicOr(a.bad, 1u);
}

// Weight-first order: keys sorted by weight carry their index; gather the
// entries in that order.
__global__ void iota_kernel(int32_t* p, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = (int32_t)i;
}

__global__ void weight_keys_kernel(const int32_t* w, uint64_t* k, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    k[i] = (uint64_t)(uint32_t)w[i];
}

__global__ void gather_kernel(const int32_t* perm, const uint64_t* kin, const int32_t* win,
                              uint64_t* kout, int32_t* wout, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t p = perm[i];
    kout[i] = kin[p];
    wout[i] = win[p];
  }
}

// ---- compaction -------------------------------------------------------------

__device__ __forceinline__ bool is_head(const uint64_t* keys, int64_t i, int dedup) {
  return !dedup || i == 0 || keys[i] != keys[i - 1];
}

// Kept entries per tile of kScanTile.
__global__ void __launch_bounds__(kBlock) cmp_count_kernel(const uint64_t* keys, int64_t E,
                                                           int dedup, uint32_t* cnt) {
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  uint32_t x = 0;
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + threadIdx.x;
    if (i < E && is_head(keys, i, dedup)) x++;
  }
  uint32_t tot;
  (void)block_excl_scan(x, &tot);
  if (threadIdx.x == 0) cnt[blockIdx.x] = tot;
}

// Writes the kept entries (column = low vb bits, weight) at their ranks and
// the row offsets at the row boundaries; with tkeys, also the transposed
// keys (column << vb | row) and weights of the kept entries (in-edge CSC).
// A wave reads and writes 64 consecutive entries at a time, ranked by ballots
// (33.5 M keys: 16 consecutive ones a thread took 712 us, this 116).
__global__ void __launch_bounds__(kBlock) cmp_write_kernel(
    const uint64_t* keys, const int32_t* w, int64_t E, int dedup, int vb, const uint32_t* tile_off,
    int32_t n, int64_t m, int32_t* col, int32_t* w_out, int32_t* row_ptr, uint64_t* tkeys,
    int32_t* tw) {
  constexpr int kWaves = kBlock / kWave, kGroups = kScanPer * kWaves;
  static_assert(kGroups <= kWave, "one wave scans the groups");
  __shared__ uint32_t s_at[kGroups];  // heads of a group of 64 entries, then their first rank
  const int tid = threadIdx.x, lane = lane_id(), wv = tid / kWave;
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  const uint64_t vmask = (1ull << vb) - 1;
  uint64_t key[kScanPer], prev[kScanPer];
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + tid;
    key[r] = i < E ? keys[i] : 0ull;
    prev[r] = lane == 0 && i > 0 && i < E ? keys[i - 1] : 0ull;
  }
  uint64_t heads[kScanPer];
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + tid;
    const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)key[r], 1);
    const uint32_t hi = (uint32_t)__shfl_up((int)(uint32_t)(key[r] >> 32), 1);
    if (lane != 0) prev[r] = (uint64_t)hi << 32 | lo;
    heads[r] = __ballot(i < E && (!dedup || i == 0 || key[r] != prev[r]));
    if (lane == 0) s_at[r * kWaves + wv] = (uint32_t)__popcll(heads[r]);
  }
  __syncthreads();
  if (wv == 0) {
    const uint32_t x = lane < kGroups ? s_at[lane] : 0u;
    const uint32_t inc = wave_incl_scan_u32(x);
    if (lane < kGroups) s_at[lane] = tile_off[blockIdx.x] + inc - x;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t i = t0 + r * kBlock + tid;
    if (i >= E) continue;
    const int32_t u = (int32_t)(key[r] >> vb);
    if ((heads[r] >> lane) & 1ull) {
      const uint32_t pos = s_at[r * kWaves + wv] + (uint32_t)__popcll(heads[r] & lanes_below_mask());
      const int32_t v = (int32_t)(key[r] & vmask);
      const int32_t uprev = i == 0 ? -1 : (int32_t)(prev[r] >> vb);
      col[pos] = v;
      if (w_out) w_out[pos] = w[i];
      if (tkeys) {
        tkeys[pos] = ((uint64_t)v << vb) | (uint64_t)u;
        if (tw) tw[pos] = w[i];
      }
      if (u != uprev)
        for (int32_t x = uprev + 1; x <= u; x++) row_ptr[x] = (int32_t)pos;
    }
    if (i == E - 1)
      for (int32_t x = u + 1; x <= n; x++) row_ptr[x] = (int32_t)m;
  }
}

__global__ void fill_i32_kernel(int32_t* p, int64_t N, int32_t value) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = value;
}

// Sorted keys [0, E) -> CSR arrays (allocated here) on the device.
int compact(const uint64_t* keys, const int32_t* w, int64_t E, int dedup, int vb, int32_t n,
            hipStream_t s, SortTemp& t, int32_t** row_ptr, int32_t** col, int32_t** w_out,
            int64_t* m_out, uint64_t* tkeys, int32_t* tw) {
  auto dalloc = [](int32_t** p, size_t count) -> int {
    DAWN_HIP(hipMalloc((void**)p, sizeof(int32_t) * std::max<size_t>(count, 1)));
    return DAWN_OK;
  };
  DAWN_TRY(dalloc(row_ptr, (size_t)n + 1));
  int64_t m = 0;
  const int64_t tiles = (E + kScanTile - 1) / kScanTile;
  DevBuf<uint32_t> cnt;
  if (E > 0) {
    DAWN_TRY(cnt.alloc((size_t)tiles));
    cmp_count_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(keys, E, dedup, cnt.p);
    DAWN_HIP(hipGetLastError());
    uint32_t last = 0;
    DAWN_HIP(hipMemcpyAsync(&last, cnt.p + tiles - 1, sizeof last, hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    DAWN_TRY(excl_scan(cnt.p, tiles, s, t.scan));
    uint32_t off = 0;
    DAWN_HIP(hipMemcpyAsync(&off, cnt.p + tiles - 1, sizeof off, hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    m = (int64_t)off + last;
  }
  if (m > (int64_t)INT32_MAX) return DAWN_ERR_OVERFLOW;
  DAWN_TRY(dalloc(col, (size_t)m));
  if (w) DAWN_TRY(dalloc(w_out, (size_t)m));
  if (E > 0) {
    cmp_write_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(keys, w, E, dedup, vb, cnt.p, n, m, *col,
                                                        w ? *w_out : nullptr, *row_ptr, tkeys, tw);
  } else {
    fill_i32_kernel<<<grid_for((int64_t)n + 1), kBlock, 0, s>>>(*row_ptr, (int64_t)n + 1, 0);
  }
  DAWN_HIP(hipGetLastError());
  DAWN_HIP(hipStreamSynchronize(s));
  *m_out = m;
  return DAWN_OK;
}

// ---- degrees and chunk lists -------------------------------------------------

// Per tile of kScanTile rows: rows of at least `heavy` entries (hv), their
// chunks beyond the first (ex); over all rows the largest degree and the
// number of empty rows.
__global__ void __launch_bounds__(kBlock) row_count_kernel(const int32_t* rp, int32_t n, int heavy,
                                                           int chunk, uint32_t* hv, uint32_t* ex,
                                                           unsigned* max_deg, unsigned* empty) {
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  uint32_t h = 0, x = 0, z = 0;
  int32_t big = 0;
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t v = t0 + r * kBlock + threadIdx.x;
    if (v >= n) continue;
    const int32_t d = rp[v + 1] - rp[v];
    big = max(big, d);
    z += d == 0;
    if (d < heavy) continue;
    h++;
    x += (uint32_t)((d - 1) / chunk);
  }
  uint32_t th, tx, tz;
  (void)block_excl_scan(h, &th);
  (void)block_excl_scan(x, &tx);
  (void)block_excl_scan(z, &tz);
  for (int o = 32; o >= 1; o >>= 1) big = max(big, __shfl_xor(big, o));
  if (lane_id() == 0 && big) atomicMax(max_deg, (unsigned)big);
  if (threadIdx.x == 0) {
    hv[blockIdx.x] = th;
    ex[blockIdx.x] = tx;
    if (tz) atomicAdd(empty, tz);
  }
}

// The lists: first chunks of the heavy rows in row order, then the others,
// row by row.  hv / ex: the tiles' first positions.
__global__ void __launch_bounds__(kBlock) row_chunks_kernel(const int32_t* rp, int32_t n, int heavy,
                                                            int chunk, const uint32_t* hv,
                                                            const uint32_t* ex, int32_t* cv,
                                                            int32_t* cb, int32_t* ce) {
  constexpr int kWaves = kBlock / kWave, kGroups = kScanPer * kWaves;
  static_assert(kGroups <= kWave, "one wave scans the groups");
  __shared__ uint32_t s_h[kGroups], s_x[kGroups];
  const int tid = threadIdx.x, lane = lane_id(), wv = tid / kWave;
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  int32_t beg[kScanPer], deg[kScanPer];
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const int64_t v = t0 + r * kBlock + tid;
    beg[r] = v < n ? rp[v] : 0;
    deg[r] = v < n ? rp[v + 1] - beg[r] : -1;
  }
  uint32_t at_h[kScanPer], at_x[kScanPer];  // within the group of 64 rows
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    const bool in = deg[r] >= heavy;
    const uint64_t m = __ballot(in);
    const uint32_t x = in ? (uint32_t)((deg[r] - 1) / chunk) : 0u;
    const uint32_t inc = wave_incl_scan_u32(x);
    at_h[r] = (uint32_t)__popcll(m & lanes_below_mask());
    at_x[r] = inc - x;
    if (lane == kWave - 1) {
      s_h[r * kWaves + wv] = (uint32_t)__popcll(m);
      s_x[r * kWaves + wv] = inc;
    }
  }
  __syncthreads();
  if (wv == 0) {
    const uint32_t h = lane < kGroups ? s_h[lane] : 0u, x = lane < kGroups ? s_x[lane] : 0u;
    const uint32_t ih = wave_incl_scan_u32(h), ix = wave_incl_scan_u32(x);
    if (lane < kGroups) {
      s_h[lane] = hv[blockIdx.x] + ih - h;
      s_x[lane] = ex[blockIdx.x] + ix - x;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kScanPer; r++) {
    if (deg[r] < heavy) continue;
    const int32_t v = (int32_t)(t0 + r * kBlock + tid), end = beg[r] + deg[r];
    const uint32_t h = s_h[r * kWaves + wv] + at_h[r];
    cv[h] = v;
    cb[h] = beg[r];
    ce[h] = deg[r] > chunk ? beg[r] + chunk : end;
    uint32_t x = s_x[r * kWaves + wv] + at_x[r];
    for (int64_t k = (int64_t)beg[r] + chunk; k < end; k += chunk, x++) {
      cv[x] = v;
      cb[x] = (int32_t)k;
      ce[x] = (int32_t)min(k + chunk, (int64_t)end);
    }
  }
}

// ---- hub-first order ---------------------------------------------------------

// Sort keys: the degree counted down from the largest, the vertex above it.
__global__ void order_keys_kernel(const int32_t* rp, int32_t n, int32_t max_deg, uint64_t* keys,
                                  uint32_t* rest) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    keys[v] = (uint64_t)v << 32 | (uint32_t)(max_deg - (rp[v + 1] - rp[v]));
    rest[v] = 1u;
  }
}

__global__ void order_hubs_kernel(const uint64_t* keys, int32_t k, int32_t* perm, int32_t* inv,
                                  uint32_t* rest) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < k;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t v = (int32_t)(keys[i] >> 32);
    perm[v] = (int32_t)i;
    inv[i] = v;
    rest[v] = 0u;
  }
}

// after: the scanned `rest`, the rank of a vertex among those that are no hubs.
__global__ void order_rest_kernel(const uint32_t* after, int32_t n, int32_t k, int32_t* perm, int32_t* inv) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    if ((v + 1 < n ? after[v + 1] : (uint32_t)(n - k)) == after[v]) continue;  // a hub
    perm[v] = k + (int32_t)after[v];
    inv[k + after[v]] = (int32_t)v;
  }
}

__global__ void order_degrees_kernel(const int32_t* rp, const int32_t* inv, int32_t n, uint32_t* out) {
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r <= n;
       r += (int64_t)gridDim.x * blockDim.x)
    out[r] = r < n ? (uint32_t)(rp[inv[r] + 1] - rp[inv[r]]) : 0u;
}

int key_bits(int32_t n) {
  int b = 1;
  while (b < 31 && (1ll << b) < (int64_t)n) b++;
  return b;
}

int weight_bits(int32_t wmax) {
  int b = 1;
  while (b < 31 && (1ll << b) <= (int64_t)wmax) b++;
  return b;
}

// Builds the device graph from one emit launch.
int build_device(EmitArgs ea, int dedup, int32_t wmax_bound, dawn_graph** out) {
  if (!out) return DAWN_ERR_INVALID_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    (void)hipGetLastError();
    return DAWN_ERR_NO_DEVICE;
  }
  const int32_t n = ea.n;
  const int per = ea.symmetrize ? 2 : 1;
  const int64_t N = ea.count * per;
  if (N > (int64_t)INT32_MAX) return DAWN_ERR_OVERFLOW;
  dawn_graph* g = new dawn_graph();
  auto fail = [&](int rc) {
    dawn_graph_destroy(g);
    return rc;
  };
  g->n = n;
  g->directed = ea.symmetrize ? 0 : 1;
  g->weighted = ea.weighted ? 1 : 0;
  if (hipGetDevice(&g->device) != hipSuccess) return fail(DAWN_ERR_HIP);
  if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess)
    return fail(DAWN_ERR_HIP);
  hipStream_t s = g->stream;
  int rc = DAWN_OK;
  {
    SortTemp t;
    DevBuf<uint64_t> ka, kb;
    DevBuf<int32_t> wa, wb, perm;
    DevBuf<unsigned long long> loops;
    DevBuf<unsigned int> bad;
    if ((rc = ka.alloc((size_t)N)) || (rc = kb.alloc((size_t)N))) return fail(rc);
    if (ea.weighted && ((rc = wa.alloc((size_t)N)) || (rc = wb.alloc((size_t)N)))) return fail(rc);
    if ((rc = loops.alloc(1)) || (rc = bad.alloc(1))) return fail(rc);
    if (hipMemsetAsync(loops.p, 0, sizeof(unsigned long long), s) != hipSuccess ||
        hipMemsetAsync(bad.p, 0, sizeof(unsigned int), s) != hipSuccess)
      return fail(DAWN_ERR_HIP);
    ea.vb = key_bits(n);
    ea.keys = ka.p;
    ea.wts = ea.weighted ? wa.p : nullptr;
    ea.selfloops = loops.p;
    ea.bad = bad.p;
    if (ea.count > 0) {
      emit_kernel<<<grid_for(ea.count, kBlock, 65536u), kBlock, 0, s>>>(ea);
      if (hipGetLastError() != hipSuccess) return fail(DAWN_ERR_HIP);
    }
    unsigned long long h_loops = 0;
    unsigned int h_bad = 0;
    if (hipMemcpyAsync(&h_loops, loops.p, sizeof h_loops, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipMemcpyAsync(&h_bad, bad.p, sizeof h_bad, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return fail(DAWN_ERR_HIP);
    if (h_bad) return fail(DAWN_ERR_INVALID_ARG);
    const int64_t E = N - (int64_t)h_loops * per;  // entries before the sentinels
    uint64_t* keys = ka.p;
    int32_t* wts = ea.weighted ? wa.p : nullptr;
    bool in1 = false;
    if (ea.weighted && N > 1) {
      // Weight-first: entry indices sorted by weight, then the entries
      // gathered in that order, so the stable key sort leaves equal keys
      // weight-ascending (dedup keeps the minimum, as the host build).
      if ((rc = perm.alloc((size_t)N))) return fail(rc);
      DevBuf<int32_t> perm2;
      if ((rc = perm2.alloc((size_t)N))) return fail(rc);
      weight_keys_kernel<<<grid_for(N, kBlock, 65536u), kBlock, 0, s>>>(wa.p, kb.p, N);
      iota_kernel<<<grid_for(N, kBlock, 65536u), kBlock, 0, s>>>(perm.p, N);
      // kb holds the weight keys; ka keeps the entry keys for the gather.
      DevBuf<uint64_t> kc;
      if ((rc = kc.alloc((size_t)N))) return fail(rc);
      if ((rc = radix_sort(kb.p, kc.p, perm.p, perm2.p, N, weight_bits(wmax_bound), s, t, &in1)))
        return fail(rc);
      const int32_t* order = in1 ? perm2.p : perm.p;
      gather_kernel<<<grid_for(N, kBlock, 65536u), kBlock, 0, s>>>(order, ka.p, wa.p, kb.p, wb.p, N);
      if (hipGetLastError() != hipSuccess) return fail(DAWN_ERR_HIP);
      // Sort (kb, wb) by key, ping-ponging with (ka, wa).
      if ((rc = radix_sort(kb.p, ka.p, wb.p, wa.p, N, 2 * ea.vb, s, t, &in1))) return fail(rc);
      keys = in1 ? ka.p : kb.p;
      wts = in1 ? wa.p : wb.p;
    } else {
      if ((rc = radix_sort(ka.p, kb.p, nullptr, nullptr, N, 2 * ea.vb, s, t, &in1))) return fail(rc);
      keys = in1 ? kb.p : ka.p;
    }
    // Directed graphs: the kept entries' transposed keys go to the free
    // key buffer, for the in-edge CSC.
    uint64_t* tk = nullptr;
    int32_t* tw = nullptr;
    if (g->directed) {
      tk = keys == ka.p ? kb.p : ka.p;
      if (ea.weighted) tw = wts == wa.p ? wb.p : wa.p;
    }
    int64_t m = 0;
    if ((rc = compact(keys, wts, E, dedup, ea.vb, n, s, t, &g->row_ptr, &g->col,
                      &g->weight, &m, tk, tw)))
      return fail(rc);
    g->m = m;
    if (g->directed) {
      // tk/tw hold m transposed entries in (row, column, weight) order;
      // sort them by (column, row) into the free buffers.
      uint64_t* tk2 = tk == ka.p ? kb.p : ka.p;
      int32_t* tw2 = ea.weighted ? (tw == wa.p ? wb.p : wa.p) : nullptr;
      if ((rc = radix_sort(tk, tk2, tw, tw2, m, 2 * ea.vb, s, t, &in1))) return fail(rc);
      const uint64_t* ck = in1 ? tk2 : tk;
      const int32_t* cw = ea.weighted ? (in1 ? tw2 : tw) : nullptr;
      int64_t m2 = 0;
      if ((rc = compact(ck, cw, m, 0, ea.vb, n, s, t, &g->in_row_ptr, &g->in_col,
                        &g->in_weight, &m2, nullptr, nullptr)))
        return fail(rc);
    } else {
      g->in_row_ptr = g->row_ptr;
      g->in_col = g->col;
      g->in_weight = g->weight;
    }
  }
  // Host copies of the offsets (degrees for the drivers) and degree stats.
  g->h_row_ptr.resize((size_t)n + 1);
  if (hipMemcpy(g->h_row_ptr.data(), g->row_ptr, sizeof(int32_t) * ((size_t)n + 1),
                hipMemcpyDeviceToHost) != hipSuccess)
    return fail(DAWN_ERR_HIP);
  if (g->directed) {
    g->h_in_row_ptr.resize((size_t)n + 1);
    if (hipMemcpy(g->h_in_row_ptr.data(), g->in_row_ptr, sizeof(int32_t) * ((size_t)n + 1),
                  hipMemcpyDeviceToHost) != hipSuccess)
      return fail(DAWN_ERR_HIP);
  }
  // Degree statistics come with the chunk lists: largest degrees and empty rows.
  (void)tuned_knobs_for(g, &g->knobs);
  g->own_knobs = g->knobs;
  RowStats out_rows, in_rows;
  if ((rc = build_chunks(g, &out_rows, &in_rows))) return fail(rc);
  g->max_out_degree = out_rows.max_deg;
  g->max_in_degree = in_rows.max_deg;
  g->zero_in = in_rows.empty;
  *out = g;
  return DAWN_OK;
}

EmitArgs base_args(int kind, int32_t n, int64_t count, int symmetrize, int weighted, uint64_t seed,
                   int32_t wmin, int32_t wmax) {
  EmitArgs a{};
  a.kind = kind;
  a.n = n;
  a.count = count;
  a.symmetrize = symmetrize;
  a.weighted = weighted;
  a.seed = seed;
  a.wmin = wmin;
  a.wmax = wmax;
  return a;
}

bool weights_ok(int32_t weighted, int32_t wmin, int32_t wmax) {
  return !weighted || (wmin >= 0 && wmax >= wmin);
}

}  // namespace

int hub_order_device(const dawn_graph* g, int32_t k, int32_t* perm, int32_t* inv) {
  const int32_t n = g->n;
  hipStream_t s = g->stream;
  SortTemp t;
  DevBuf<uint64_t> ka, kb;
  DevBuf<uint32_t> rest;
  DAWN_TRY(ka.alloc((size_t)n));
  DAWN_TRY(kb.alloc((size_t)n));
  DAWN_TRY(rest.alloc((size_t)n));
  const unsigned grid = grid_for(n);
  order_keys_kernel<<<grid, kBlock, 0, s>>>(g->row_ptr, n, g->max_out_degree, ka.p, rest.p);
  DAWN_HIP(hipGetLastError());
  bool in1 = false;
  DAWN_TRY(radix_sort(ka.p, kb.p, nullptr, nullptr, n, weight_bits(g->max_out_degree), s, t, &in1));
  order_hubs_kernel<<<grid_for(k), kBlock, 0, s>>>(in1 ? kb.p : ka.p, k, perm, inv, rest.p);
  DAWN_HIP(hipGetLastError());
  DAWN_TRY(excl_scan(rest.p, n, s, t.scan));
  order_rest_kernel<<<grid, kBlock, 0, s>>>(rest.p, n, k, perm, inv);
  DAWN_HIP(hipGetLastError());
  DAWN_HIP(hipStreamSynchronize(s));
  return DAWN_OK;
}

int permuted_offsets_device(const int32_t* rp, const int32_t* inv, int32_t n, hipStream_t s, int32_t* out) {
  ScanTemp t;
  order_degrees_kernel<<<grid_for((int64_t)n + 1), kBlock, 0, s>>>(rp, inv, n, (uint32_t*)out);
  DAWN_HIP(hipGetLastError());
  DAWN_TRY(excl_scan((uint32_t*)out, (int64_t)n + 1, s, t));
  DAWN_HIP(hipStreamSynchronize(s));
  return DAWN_OK;
}

int chunk_list_device(const int32_t* rp, int32_t n, int heavy, int chunk, hipStream_t s, int32_t** dv,
                      int32_t** db, int32_t** de, int64_t* count, int64_t* rows, RowStats* stats) {
  const int64_t tiles = (n + (int64_t)kScanTile - 1) / kScanTile;
  // Per tile: heavy rows, further chunks; then the largest degree, the empty rows.
  DevBuf<uint32_t> cnt;
  std::vector<uint32_t> h((size_t)tiles * 2 + 2);
  const size_t bytes = sizeof(uint32_t) * h.size();
  DAWN_TRY(cnt.alloc(h.size()));
  DAWN_HIP(hipMemsetAsync(cnt.p, 0, bytes, s));
  row_count_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(rp, n, heavy, chunk, cnt.p, cnt.p + tiles,
                                                      cnt.p + 2 * tiles, cnt.p + 2 * tiles + 1);
  DAWN_HIP(hipGetLastError());
  DAWN_HIP(hipMemcpyAsync(h.data(), cnt.p, bytes, hipMemcpyDeviceToHost, s));
  DAWN_HIP(hipStreamSynchronize(s));
  uint64_t at = 0;
  for (int64_t i = 0; i < 2 * tiles; i++) {
    if (i == tiles) *rows = (int64_t)at;
    const uint32_t x = h[i];
    h[i] = (uint32_t)at;
    at += x;  // at most m
  }
  *count = (int64_t)at;
  if (stats) *stats = RowStats{(int32_t)h[2 * tiles], (int64_t)h[2 * tiles + 1]};
  for (int32_t** p : {dv, db, de}) {
    const hipError_t e = hipMalloc((void**)p, sizeof(int32_t) * std::max<uint64_t>(at, 1));
    if (e != hipSuccess) {
      *p = nullptr;
      set_hip_error(e, "hipMalloc", __FILE__, __LINE__);
      return e == hipErrorOutOfMemory ? DAWN_ERR_OUT_OF_MEMORY : DAWN_ERR_HIP;
    }
  }
  if (at) {
    DAWN_HIP(hipMemcpyAsync(cnt.p, h.data(), sizeof(uint32_t) * 2 * (size_t)tiles, hipMemcpyHostToDevice, s));
    row_chunks_kernel<<<(unsigned)tiles, kBlock, 0, s>>>(rp, n, heavy, chunk, cnt.p, cnt.p + tiles, *dv,
                                                         *db, *de);
    DAWN_HIP(hipGetLastError());
  }
  DAWN_HIP(hipStreamSynchronize(s));
  return DAWN_OK;
}

}  // namespace dawn

using namespace dawn;

extern "C" {

int dawn_graph_from_edges(int32_t n, int64_t count, const int32_t* u, const int32_t* v,
                          const int32_t* w, int32_t symmetrize, int32_t dedup, dawn_graph** out) {
  if (!out || n <= 0 || count < 0 || (count > 0 && (!u || !v))) return DAWN_ERR_INVALID_ARG;
  // Host arrays are staged on the device; device arrays are read in place.
  DevBuf<int32_t> du, dv, dw;
  const int32_t *pu = u, *pv = v, *pw = w;
  int32_t wmax = 0;
  if (count > 0 && !is_device_pointer(u)) {
    DAWN_TRY(du.alloc((size_t)count));
    DAWN_TRY(dv.alloc((size_t)count));
    DAWN_HIP(hipMemcpy(du.p, u, sizeof(int32_t) * count, hipMemcpyHostToDevice));
    DAWN_HIP(hipMemcpy(dv.p, v, sizeof(int32_t) * count, hipMemcpyHostToDevice));
    pu = du.p;
    pv = dv.p;
  }
  if (w && count > 0) {
    std::vector<int32_t> hw;
    const int32_t* wh = w;
    if (is_device_pointer(w)) {
      hw.resize((size_t)count);
      DAWN_HIP(hipMemcpy(hw.data(), w, sizeof(int32_t) * count, hipMemcpyDeviceToHost));
      wh = hw.data();
    } else {
      DAWN_TRY(dw.alloc((size_t)count));
      DAWN_HIP(hipMemcpy(dw.p, w, sizeof(int32_t) * count, hipMemcpyHostToDevice));
      pw = dw.p;
    }
    for (int64_t i = 0; i < count; i++) wmax = std::max(wmax, wh[i]);
  }
  EmitArgs a = base_args(0, n, count, symmetrize ? 1 : 0, w ? 1 : 0, 0, 0, 0);
  a.u = pu;
  a.v = pv;
  a.w = pw;
  return build_device(a, dedup ? 1 : 0, std::max(wmax, 1), out);
}

int dawn_graph_gen_er(int32_t n, double avg_degree, uint64_t seed, int32_t weighted, int32_t wmin,
                      int32_t wmax, dawn_graph** out) {
  if (!out || n <= 1 || avg_degree < 0 || !weights_ok(weighted, wmin, wmax))
    return DAWN_ERR_INVALID_ARG;
  const int64_t M = (int64_t)std::llround((double)n * avg_degree / 2.0);
  EmitArgs a = base_args(1, n, M, 1, weighted ? 1 : 0, seed, wmin, wmax);
  return build_device(a, 1, std::max(wmax, 1), out);
}

int dawn_graph_gen_rmat(int32_t scale, int32_t edge_factor, double ra, double rb, double rc,
                        uint64_t seed, int32_t weighted, int32_t wmin, int32_t wmax,
                        dawn_graph** out) {
  if (!out || scale < 1 || scale > 30 || edge_factor < 1 || ra < 0 || rb < 0 || rc < 0 ||
      ra + rb + rc > 1.0 || !weights_ok(weighted, wmin, wmax))
    return DAWN_ERR_INVALID_ARG;
  const int32_t n = (int32_t)(1u << scale);
  const int64_t M = (int64_t)edge_factor << scale;
  EmitArgs a = base_args(2, n, M, 1, weighted ? 1 : 0, seed, wmin, wmax);
  a.scale = scale;
  a.ta = (uint64_t)std::llround(ra * 4294967296.0);
  a.tb = (uint64_t)std::llround((ra + rb) * 4294967296.0);
  a.tc = (uint64_t)std::llround((ra + rb + rc) * 4294967296.0);
  return build_device(a, 1, std::max(wmax, 1), out);
}

int dawn_graph_gen_grid(int32_t side, double extra_fraction, uint64_t seed, int32_t weighted,
                        int32_t wmin, int32_t wmax, dawn_graph** out) {
  if (!out || side < 2 || side > 46340 || extra_fraction < 0 || !weights_ok(weighted, wmin, wmax))
    return DAWN_ERR_INVALID_ARG;
  const int32_t n = side * side;
  const int64_t horiz = (int64_t)side * (side - 1);
  const int64_t grid_edges = 2 * horiz;
  const int64_t extra = (int64_t)std::llround(extra_fraction * (double)grid_edges);
  EmitArgs a = base_args(3, n, grid_edges + extra, 1, weighted ? 1 : 0, seed, wmin, wmax);
  a.side = side;
  a.horiz = horiz;
  a.grid_edges = grid_edges;
  return build_device(a, 1, std::max(wmax, 1), out);
}

int dawn_graph_download(const dawn_graph* g, dawn_csr* out) {
  if (!g || !out) return DAWN_ERR_INVALID_ARG;
  DAWN_HIP(hipSetDevice(g->device));
  const size_t n = (size_t)g->n, m = (size_t)g->m;
  int32_t* rp = (int32_t*)std::malloc(sizeof(int32_t) * (n + 1));
  int32_t* cc = (int32_t*)std::malloc(sizeof(int32_t) * std::max<size_t>(m, 1));
  int32_t* ww = g->weighted ? (int32_t*)std::malloc(sizeof(int32_t) * std::max<size_t>(m, 1)) : nullptr;
  if (!rp || !cc || (g->weighted && !ww)) {
    std::free(rp);
    std::free(cc);
    std::free(ww);
    return DAWN_ERR_OUT_OF_MEMORY;
  }
  hipError_t e = hipMemcpy(rp, g->row_ptr, sizeof(int32_t) * (n + 1), hipMemcpyDeviceToHost);
  if (e == hipSuccess && m) e = hipMemcpy(cc, g->col, sizeof(int32_t) * m, hipMemcpyDeviceToHost);
  if (e == hipSuccess && m && ww)
    e = hipMemcpy(ww, g->weight, sizeof(int32_t) * m, hipMemcpyDeviceToHost);
  if (e != hipSuccess) {
    std::free(rp);
    std::free(cc);
    std::free(ww);
    set_hip_error(e, "hipMemcpy", __FILE__, __LINE__);
    return DAWN_ERR_HIP;
  }
  out->n = g->n;
  out->m = g->m;
  out->directed = g->directed;
  out->weighted = g->weighted;
  out->row_ptr = rp;
  out->col = cc;
  out->weight = ww;
  return DAWN_OK;
}

}  // extern "C"
