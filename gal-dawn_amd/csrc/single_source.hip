// Single-source frontier engine: unweighted DAWN (BOVM) and int32 min-plus
// DAWN (SOVM) on one HIP device.
//
// Reference: DAWN::BFS_GPU (src/algorithm/gpu/bfs.cu:9-129) and
// DAWN::SSSP_GPU (src/algorithm/gpu/sssp.cu:18-157); CPU semantics
// DAWN::BFS_CPU (src/algorithm/cpu/bfs.cpp:23-185) and DAWN::SSSP_CPU
// (src/algorithm/cpu/sssp.cpp:23-199).
//
// Layout in HBM (per graph, reused across calls; k: launch of the step kernel,
// counted from 0 per traversal):
//   dist   int32[n]         distances (INF = unreached): the caller's buffer when
//                           it is device memory, else the workspace's
//   q      int32[2][n]      frontier queue read by launch k in slot k&1: vertices
//                           of out-degree 1 to hchunk
//   hq     int2[2][hcap]    (vertex, first edge) of every hchunk-edge chunk of the
//                           frontier's other vertices
//   bm     uint32[3][words] frontier bitmap read by launch k in slot k%3
//   slots  SsSlot[4]        queue lengths and counters of that frontier in slot k%4
//   state  SsState[4]       step / done / mode / rule state in slot k%4
// Launch k reads slot k, writes slot k+1 and clears slot k+2.  Every step but a
// pull writes BOTH the queue and the bitmap of the new level, so the three modes
// are interchangeable from step to step with no conversion:
//   PUSH    queue in: wave-balanced edge expansion (chunks of the heavy
//           vertices one wave each, the others 1 to 64 per wave by LDS scan)
//   PULL    bitmap in: unvisited vertices scan in-edges (CSC) with early exit
//   BITMAP  bitmap in: dense scan of the frontier bitmap, top-down expansion
// The step loop is one kernel per step: every workgroup makes the same
// decision from the last level's counters, then all expand the level; runs
// of levels with few edges are walked by one workgroup within one launch.
// The launch that finds the frontier empty writes the final state, with the
// traversal's counts and device time, to pinned host memory, so a call is its
// launches and one wait.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "sched.hpp"

namespace dawn {

// Counters (frontier vertices, their out-edges, GAPBS scout; min-plus also the
// smallest frontier distance, as the largest INF - distance, and the out-edges
// of deferred vertices) are added per workgroup into one of kStripes stripes,
// each on its own 128-byte line, so the atomics of the workgroups spread over
// 64 addresses; the next launch sums them, one stripe per lane.
constexpr int kStripes = 64;
constexpr int kStripeU64 = 16;  // 128 bytes per stripe
static_assert(kStripes == kWave, "one stripe per lane is summed");
struct SsSlot {
  unsigned long long part[kStripes][kStripeU64];
  unsigned qlen, hqlen;  // queue entries, heavy-chunk entries
  unsigned pad[30];
};
constexpr int kSsSlots = 4;

struct SsState {
  SchedState s;
  int32_t launches;                   // step launches that did something
  int32_t pad;
  long long mode_steps[DAWN_NUM_MODES];
  unsigned long long reached, edges;  // vertices reached, their out-edges (set when done)
  long long t0, t1;                   // device clock at the first and the last launch
  long long delta, thr;               // min-plus: advance per step (0: none), threshold
};

struct SsArgs {
  int32_t n;
  int32_t source;
  int64_t words;  // bitmap words per slot
  const int32_t* row_ptr;
  const int32_t* col;
  const int32_t* w;
  const int32_t* in_row_ptr;
  const int32_t* in_col;
  const int32_t* in_w;
  int32_t* dist;
  int32_t* q;        // 2 * n
  int2* hq;          // 2 * hcap
  int64_t hcap;      // >= 2 m / hchunk: every heavy vertex's chunks fit
  int32_t hchunk;    // edges per heavy chunk; longer lists are cut
  int32_t heavy;     // degree from which the static chunk lists hold a vertex
  uint32_t* bm;      // 3 * words
  const int32_t* oc_v;  // static out-edge chunks (BITMAP steps)
  const int32_t* oc_beg;
  const int32_t* oc_end;
  int64_t num_oc;
  SsSlot* slots;             // kSsSlots
  unsigned long long* tot;   // reach counts: workgroups done, then a pair of parts each
  SsState* st;               // kSsSlots
  SsState* host;             // pinned: the final state (null: not written)
  const unsigned long long* wsum;  // kWsumBlocks parts of the sum of the weights
  double delta_scale;        // threshold advance per unit of that sum
};

// Everything a step launch needs but its number.
struct SsRun {
  SsArgs a;
  SchedParams p;
  SchedTrace tr;   // recording only (else null)
  int32_t force;   // >= 0: every step in this mode
  int32_t small;   // runs of small levels may be walked within a launch
};

// Threads per workgroup of the step kernels, and workgroups per launch (two
// per CU).  Every workgroup that found something reserves its queue ranges
// with atomics on one address each, about 12 ns apiece in turn: 4096
// workgroups of 256 threads spent up to 50 us of a step on them, and an
// idle launch of 4096 workgroups takes 4.4 us, of 512 less than half.
constexpr int kSsBlock = 1024;
constexpr unsigned kSsGrid = 512;
constexpr int kSsWaves = kSsBlock / kWave;
// Queue entries a workgroup stages in LDS before reserving global space.
constexpr int kStageCap = 8192;
// Queue length of a level whose queue was not written (a pull step writes
// the bitmap only): a top-down step that follows reads the bitmap instead.
constexpr unsigned kNoQueue = 0xFFFFFFFFu;

struct SsWorkspace {
  int32_t n = 0;
  DevBuf<int32_t> dist, q;  // dist: only for outputs that are not device memory
  DevBuf<int2> hq;
  int64_t hcap = 0;
  DevBuf<uint32_t> bm;
  DevBuf<SsSlot> slots;
  DevBuf<unsigned long long> tot;
  DevBuf<SsState> st;
  DevBuf<unsigned long long> wsum;  // min-plus: parts of the sum of the weights
  DevBuf<float> trace_feat;    // recording only
  DevBuf<int32_t> trace_mode;
  SsState* h_state = nullptr;  // pinned
  int32_t last_launches[2] = {0, 0};  // step launches the last traversal (per kind) took
  hipEvent_t ev0 = nullptr, ev1 = nullptr;  // recording only
};

void ss_workspace_free(SsWorkspace* ws) {
  if (!ws) return;
  if (ws->h_state) (void)hipHostFree(ws->h_state);
  if (ws->ev0) (void)hipEventDestroy(ws->ev0);
  if (ws->ev1) (void)hipEventDestroy(ws->ev1);
  delete ws;
}

namespace {

// Four columns of an edge list, read by one load at any 4-byte offset.
struct __attribute__((packed, aligned(4))) Cols4 {
  int32_t c[4];
};

__device__ __forceinline__ bool test_bit(const uint32_t* bm, int32_t v) {
  return (bm[v >> 5] >> (v & 31)) & 1u;
}

// Largest j in [0, kWave) with off[j] <= e (off non-decreasing, off[0] <= e).
__device__ __forceinline__ int owner_of(const int* off, int e) {
  int j = 0;
#pragma unroll
  for (int o = kWave / 2; o >= 1; o >>= 1)
    if (off[j + o] <= e) j += o;
  return j;
}

// A thread's counts of the level it finds.
struct Acc {
  unsigned fv = 0, zero = 0;  // vertices, those without out-edges
  unsigned long long fe = 0;  // their out-edges
  unsigned long long de = 0;  // min-plus: out-edges of deferred vertices
  unsigned near = 0;          // min-plus: largest INF - distance of a frontier vertex
  __device__ void add(int d) {
    fv += 1;
    zero += d == 0;
    fe += (unsigned)d;
  }
  __device__ void dist(int32_t d) { near = max(near, (unsigned)(kInf - d)); }
};

// Edges per heavy chunk: two rounds of a wave.
constexpr int kHeavyChunk = 128;

// Chunks of a vertex of out-degree d.
__device__ __forceinline__ int chunks_of(const SsArgs& a, int d) {
  return (d + a.hchunk - 1) / a.hchunk;
}

// Writes the heavy-chunk entries of vertex u (degree d, first edge rb) from
// slot `at` on: entries first, first + step, ...
__device__ __forceinline__ void put_chunks(const SsArgs& a, int2* hq, unsigned at, int32_t u,
                                           int rb, int d, int first, int step) {
  const int k = chunks_of(a, d);
  for (int i = first; i < k; i += step) hq[at + i] = make_int2(u, rb + i * a.hchunk);
}

// Heavy-chunk entries of the wave's lanes with d > hchunk: lists of up to
// eight entries by their own lane, longer ones by the whole wave in turn (a
// hub's hundreds of entries written by one lane took longer than the step's
// edges).  *len is the counter to reserve from, in LDS or global memory.
// Called by all 64 lanes.
__device__ __forceinline__ void wave_put_chunks(const SsArgs& a, int2* hq, unsigned* len,
                                                int32_t u, int rb, int d) {
  const int k = d > a.hchunk ? chunks_of(a, d) : 0;
  unsigned at = 0;
  if (k) at = atomicAdd(len, (unsigned)k);
  if (k && k <= 8) put_chunks(a, hq, at, u, rb, d, 0, 1);
  uint64_t hm = __ballot(k > 8);
  while (hm) {
    const int l = __ffsll((unsigned long long)hm) - 1;
    hm &= hm - 1;
    put_chunks(a, hq, __shfl(at, l), __shfl(u, l), __shfl(rb, l), __shfl(d, l), lane_id(), kWave);
  }
}

// Exclusive scan of one int per thread over a kSsBlock-thread workgroup.
// scratch: kSsWaves ints of LDS; *total receives the sum.
__device__ __forceinline__ int ss_scan(int x, int* scratch, int* total) {
  const int l = lane_id(), w = threadIdx.x / kWave;
  int inc = x;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (l >= o) inc += y;
  }
  if (l == kWave - 1) scratch[w] = inc;
  __syncthreads();
  int before = 0, sum = 0;
#pragma unroll
  for (int i = 0; i < kSsWaves; i++) {
    const int t = scratch[i];
    if (i < w) before += t;
    sum += t;
  }
  __syncthreads();
  *total = sum;
  return before + inc - x;
}

// Where a launch puts the new level.
struct SsOut {
  SsSlot* slot;
  int32_t* q;
  int2* hq;
};
__device__ __forceinline__ SsOut out_of(const SsArgs& a, int k) {
  return {a.slots + ((k + 1) % kSsSlots), a.q + (int64_t)((k + 1) & 1) * a.n,
          a.hq + (int64_t)((k + 1) & 1) * a.hcap};
}

// Workgroup-level staging of a step's outputs: the vertices found in the
// step, with their out-degrees (read beside the atomic that found them), and
// the level's counters.  Waves reserve LDS slots with LDS atomics; flush()
// splits the staged vertices into the light queue and heavy chunks, and
// reserves each global range once per workgroup: a global counter that every
// wave bumps serialises at one address.  Vertices beyond the LDS capacity go
// straight to the global queues, wave by wave.
struct SsStage {
  int32_t v[kStageCap];
  uint16_t d[kStageCap];  // out-degree, 65535 for any larger one
  unsigned n;             // slots reserved (may pass kStageCap)
  unsigned odd;           // staged vertices that are not light: no edges, or heavy
  unsigned base[2];       // global positions of the workgroup's ranges
  int scan[kSsWaves];
  unsigned long long tot[5];
  __device__ void init() {
    if (threadIdx.x < 5) tot[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) n = odd = 0u;
    __syncthreads();
  }
  // Records a vertex of out-degree deg found in the step (each vertex once
  // per level).  Called by all 64 lanes of a wave.
  __device__ void append(const SsArgs& a, const SsOut& o, bool pred, int32_t x, int deg, Acc& acc) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int leader = __ffsll((unsigned long long)m) - 1;
    const unsigned cnt = (unsigned)__popcll(m);
    unsigned b = 0;
    if (lane_id() == leader) b = atomicAdd(&n, cnt);
    b = __shfl(b, leader);
    const unsigned idx = b + (unsigned)__popcll(m & lanes_below_mask());
    const bool in = pred && idx < (unsigned)kStageCap;
    if (in) {
      v[idx] = x;
      d[idx] = (uint16_t)min(deg, 65535);
    }
    if (pred) acc.add(deg);
    const uint64_t om = __ballot(in && (deg == 0 || deg > a.hchunk));
    if (om && lane_id() == leader) atomicAdd(&odd, (unsigned)__popcll(om));
    if (b + cnt > (unsigned)kStageCap) spill(a, o, pred && !in, x, deg);
  }
  __device__ void spill(const SsArgs& a, const SsOut& o, bool pred, int32_t x, int deg) {
    const bool light = pred && deg > 0 && deg <= a.hchunk;
    const int at = wave_append(&o.slot->qlen, light);
    if (light) o.q[at] = x;
    const bool heavy = pred && deg > a.hchunk;
    wave_put_chunks(a, o.hq, &o.slot->hqlen, x, heavy ? a.row_ptr[x] : 0, heavy ? deg : 0);
  }
  // Every thread, once, at the end of the step kernel.  The staged order is
  // kept: vertices found together are neighbours in the next queue, so the
  // lanes that expand them read neighbouring rows and distances (queue
  // entries interleaved by thread made push steps on a 2048^2 grid 2-3x
  // slower).
  template <bool MP>
  __device__ void flush(const SsArgs& a, const SsOut& o, Acc& acc) {
    __syncthreads();
    const unsigned cnt = n < (unsigned)kStageCap ? n : (unsigned)kStageCap;
    const bool all_light = odd == 0;
    if (cnt && all_light) {  // block-uniform
      if (threadIdx.x == 0) base[0] = atomicAdd(&o.slot->qlen, cnt);
    } else if (cnt) {
      int nl = 0, nh = 0, tl, th;
      for (unsigned i = threadIdx.x; i < cnt; i += kSsBlock) {
        int g = d[i];
        if (g == 65535) g = a.row_ptr[v[i] + 1] - a.row_ptr[v[i]];
        if (g > a.hchunk) nh += chunks_of(a, g);
        else if (g > 0) nl += 1;
      }
      (void)ss_scan(nl, scan, &tl);
      (void)ss_scan(nh, scan, &th);
      if (threadIdx.x == 0) {
        base[0] = tl ? atomicAdd(&o.slot->qlen, (unsigned)tl) : 0u;
        base[1] = th ? atomicAdd(&o.slot->hqlen, (unsigned)th) : 0u;
      }
    }
    if (__ballot(acc.fv != 0 || acc.near != 0)) {  // beside the reservation
      const unsigned long long c =
          wave_sum_u64((unsigned long long)acc.fv | ((unsigned long long)acc.zero << 32));
      const unsigned long long fe = wave_sum_u64(acc.fe);
      const unsigned long long de = MP ? wave_sum_u64(acc.de) : 0ull;
      const int near = MP ? wave_max_i32((int)acc.near) : 0;
      if (lane_id() == 0) {
        atomicAdd(&tot[0], c & 0xFFFFFFFFull);
        atomicAdd(&tot[1], fe);
        atomicAdd(&tot[2], fe + (c >> 32));  // scout: max(degree, 1)
        if (near) atomicMax(&tot[3], (unsigned long long)near);
        if (de) atomicAdd(&tot[4], de);
      }
    }
    __syncthreads();
    if (threadIdx.x < 5 && tot[threadIdx.x]) {
      unsigned long long* part = o.slot->part[blockIdx.x % kStripes];
      if (threadIdx.x == 3) atomicMax(&part[3], tot[3]);
      else atomicAdd(&part[threadIdx.x], tot[threadIdx.x]);
    }
    if (cnt && all_light) {
      for (unsigned i = threadIdx.x; i < cnt; i += kSsBlock) o.q[base[0] + i] = v[i];
    } else if (cnt) {
      int32_t* q_out = o.q + base[0];
      for (unsigned i0 = 0; i0 < cnt; i0 += kSsBlock) {
        const unsigned i = i0 + threadIdx.x;
        int rb = 0, g = 0;
        int32_t x = 0;
        if (i < cnt) {
          x = v[i];
          g = d[i];
          if (g > a.hchunk) {
            rb = a.row_ptr[x];
            g = a.row_ptr[x + 1] - rb;
          }
        }
        const bool light = g > 0 && g <= a.hchunk;
        int tr;
        const int ol = ss_scan(light ? 1 : 0, scan, &tr);
        if (light) q_out[ol] = x;
        q_out += tr;
        wave_put_chunks(a, o.hq, &base[1], x, rb, g > a.hchunk ? g : 0);
      }
    }
  }
};

// LDS of one wave's batch of vertices: scanned out-degrees, first edges, tail
// distances; for frontiers read from the bitmap also its words and their
// scanned bit counts.
template <bool DU>
struct PushLds {
  int off[kSsWaves][kWave];
  int beg[kSsWaves][kWave];
  int du[DU ? kSsWaves : 1][kWave];
  int woff[kSsWaves][kWave];
  uint32_t word[kSsWaves][kWave];
};

__device__ __forceinline__ int wave_incl_scan(int x) {
  const int l = lane_id();
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int y = __shfl_up(x, o);
    if (l >= o) x += y;
  }
  return x;
}

// Edge lists of up to 64 vertices (one per lane: first edge, out-degree, tail
// distance), walked as one by the wave: LDS degree scan, two edges per lane
// and round.  edge(du0, du1, e0, e1) handles edges e0 and e1 (-1: none) in one
// wave-uniform call.
template <bool DU, class F>
__device__ __forceinline__ void wave_edges(PushLds<DU>& s, int beg, int deg, int du, F&& edge) {
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  int* off = s.off[wv];
  int* begs = s.beg[wv];
  int* dus = s.du[DU ? wv : 0];
  const int inc = wave_incl_scan(deg);
  const int total = __shfl(inc, kWave - 1);
  off[lane] = inc - deg;
  begs[lane] = beg - (inc - deg);
  if (DU) dus[lane] = du;
  wave_lds_sync();
  for (int e = lane; e - lane < total; e += 2 * kWave) {
    const int e1 = e + kWave;
    const int j0 = owner_of(off, e), j1 = owner_of(off, e1);
    edge(DU ? dus[j0] : 0, DU ? dus[j1] : 0, e < total ? begs[j0] + e : -1,
         e1 < total ? begs[j1] + e1 : -1);
  }
  wave_lds_sync();
}

// Out-edges of the frontier queue of launch k, spread over the waves of the
// grid: a wave takes the heavy chunks one by one, and of the light queue 1 to
// 64 vertices at a time (as few as the grid's waves need to cover the queue).
// With DU, vertices at distance thr or more are not expanded: defer(yes, u,
// its distance, its out-degree), wave-uniform too.  Bound by the latency of
// the dependent loads per edge (column, then its distance): with whole
// workgroups taking 256 queue entries each, a frontier of a few thousand
// vertices ran on a few CUs and a hub's list on one (RMAT scale 22, 10.2 M
// edges of 3133 vertices: 29.7 ms, now 0.25 ms; scale 20, 1.03 M edges of 434:
// 6.9 ms, now 0.18 ms, where the atomics on the few bitmap words of the hubs
// bound it).
template <bool DU, class F, class D>
__device__ __forceinline__ void push_edges(const SsArgs& a, PushLds<DU>& s, int k, unsigned qn,
                                           unsigned hn, int32_t thr, F&& edge, D&& defer) {
  const int32_t* q_in = a.q + (int64_t)(k & 1) * a.n;
  const int2* hq_in = a.hq + (int64_t)(k & 1) * a.hcap;
  const int lane = lane_id();
  const int64_t wid = (int64_t)blockIdx.x * kSsWaves + threadIdx.x / kWave;
  const int64_t nw = (int64_t)gridDim.x * kSsWaves;
  for (int64_t c = wid; c < hn; c += nw) {  // wave-uniform
    const int2 h = hq_in[c];
    const int end = min(h.y + a.hchunk, a.row_ptr[h.x + 1]);
    const int du = DU ? a.dist[h.x] : 0;
    if (DU && du >= thr) {  // once per vertex: by its first chunk
      const int rb = a.row_ptr[h.x];
      defer(lane == 0 && h.y == rb, h.x, du, a.row_ptr[h.x + 1] - rb);
      continue;
    }
    for (int kb = h.y; kb < end; kb += 2 * kWave) {
      const int k0 = kb + lane, k1 = k0 + kWave;
      edge(du, du, k0 < end ? k0 : -1, k1 < end ? k1 : -1);
    }
  }
  int64_t per = (qn + nw - 1) / nw;
  per = per < 1 ? 1 : per > kWave ? kWave : per;
  for (int64_t c = wid * per; c < qn; c += nw * per) {  // wave-uniform
    int beg = 0, deg = 0, du = 0;
    int32_t u = 0;
    if (lane < per && c + lane < qn) {
      u = q_in[c + lane];
      beg = a.row_ptr[u];
      deg = a.row_ptr[u + 1] - beg;
      if (DU) du = a.dist[u];
    }
    if (DU) {
      const bool later = deg > 0 && du >= thr;
      defer(later, u, du, deg);
      if (later) deg = 0;
    }
    wave_edges<DU>(s, beg, deg, du, edge);
  }
}

// Position of the r-th set bit of x (r < popcount).
__device__ __forceinline__ int select_bit(uint32_t x, int r) {
  int at = 0;
#pragma unroll
  for (int w = 16; w >= 1; w >>= 1) {
    const int c = __popc((x >> at) & ((1u << w) - 1u));
    if (r >= c) {
      r -= c;
      at += w;
    }
  }
  return at;
}

// Out-edges of the frontier bitmap, in vertex order: a wave takes up to 64
// consecutive words (fewer, so that the words are spread over the grid's
// waves), 64 of their set bits at a time.  Neighbouring vertices are expanded
// together, so their rows, columns and heads' distances share lines, where a
// queue of some hundred thousand vertices, in the order they were found,
// moves most of a line per access (2048^2 grid, min-plus: a traversal with its dense
// steps in vertex order 1.61 ms, all by the queue 1.98).
// Vertices of out-degree >= heavy go by the graph's static out-edge chunks, a
// wave each.
template <bool DU, class F, class D>
__device__ __forceinline__ void bitmap_edges(const SsArgs& a, PushLds<DU>& s, const uint32_t* bm_in,
                                             int32_t thr, F&& edge, D&& defer) {
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  const int64_t wid = (int64_t)blockIdx.x * kSsWaves + wv;
  const int64_t nw = (int64_t)gridDim.x * kSsWaves;
  int64_t per = (a.words + nw - 1) / nw;
  per = per > kWave ? kWave : per;
  int* woff = s.woff[wv];
  uint32_t* word = s.word[wv];
  for (int64_t w0 = wid * per; w0 < a.words; w0 += nw * per) {  // wave-uniform
    const uint32_t x = lane < per && w0 + lane < a.words ? bm_in[w0 + lane] : 0u;
    if (!__ballot(x != 0)) continue;
    const int inc = wave_incl_scan(__popc(x));
    const int total = __shfl(inc, kWave - 1);
    woff[lane] = inc - __popc(x);
    word[lane] = x;
    wave_lds_sync();
    for (int i0 = 0; i0 < total; i0 += kWave) {
      const int i = i0 + lane;
      int beg = 0, deg = 0, du = 0;
      int32_t u = 0;
      if (i < total) {
        const int j = owner_of(woff, i);
        u = (int32_t)((w0 + j) * 32 + select_bit(word[j], i - woff[j]));
        beg = a.row_ptr[u];
        deg = a.row_ptr[u + 1] - beg;
        if (DU) du = a.dist[u];
      }
      if (DU) {
        const bool later = deg > 0 && du >= thr;
        defer(later, u, du, deg);
        if (later) deg = 0;
      }
      if (deg >= a.heavy) deg = 0;
      wave_edges<DU>(s, beg, deg, du, edge);
    }
    wave_lds_sync();
  }
  // 64 chunks are probed at once, one per lane, as most are not in the
  // frontier; a grid apart, as a hub's chunks are neighbours in the list.
  for (int64_t c0 = wid; c0 < a.num_oc; c0 += nw * kWave) {  // wave-uniform
    const int32_t mine = c0 + lane * nw < a.num_oc ? a.oc_v[c0 + lane * nw] : -1;
    uint64_t m = __ballot(mine >= 0 && test_bit(bm_in, mine));
    while (m) {
      const int l = __ffsll((unsigned long long)m) - 1;
      m &= m - 1;
      const int du = DU ? a.dist[__shfl(mine, l)] : 0;
      if (DU && du >= thr) continue;
      const int end = a.oc_end[c0 + l * nw];
      for (int e = a.oc_beg[c0 + l * nw] + lane; e - lane < end; e += 2 * kWave)
        edge(du, du, e < end ? e : -1, e + kWave < end ? e + kWave : -1);
    }
  }
}

// Clears what the next launch writes: its bitmap slot and its counters.
__device__ __forceinline__ void clear_next(const SsArgs& a, int k) {
  const int64_t gs = (int64_t)gridDim.x * blockDim.x;
  const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t* bm_nx = a.bm + (int64_t)((k + 2) % 3) * a.words;
  for (int64_t i = gt; i < a.words; i += gs) bm_nx[i] = 0u;
  unsigned long long* p = reinterpret_cast<unsigned long long*>(a.slots + ((k + 2) % kSsSlots));
  for (int64_t i = gt; i < (int64_t)(sizeof(SsSlot) / 8); i += gs) p[i] = 0ull;
}

// ---------------------------------------------------------------- kernels ---

// Initial distances, bitmaps, counters; for BOVM also level 0 = {source}
// (GAPBS starts scout_count at out_degree(source), test/gabps/bfs.cc:140).
__global__ void __launch_bounds__(kBlock) ss_fill_kernel(SsArgs a, int bovm) {
  const int64_t gs = (int64_t)gridDim.x * kBlock;
  const int64_t gt = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int32_t s = a.source;
  auto value = [&](int64_t v) { return bovm && v == s ? 0 : kInf; };
  if (((uintptr_t)a.dist & 15) == 0) {
    const int64_t n4 = a.n / 4;
    for (int64_t i = gt; i < n4; i += gs)
      reinterpret_cast<int4*>(a.dist)[i] =
          make_int4(value(4 * i), value(4 * i + 1), value(4 * i + 2), value(4 * i + 3));
    for (int64_t v = 4 * n4 + gt; v < a.n; v += gs) a.dist[v] = value(v);
  } else {
    for (int64_t v = gt; v < a.n; v += gs) a.dist[v] = value(v);
  }
  for (int64_t i = gt; i < 3 * a.words; i += gs)
    a.bm[i] = bovm && i == s >> 5 ? 1u << (s & 31) : 0u;
  if (blockIdx.x != 0) return;
  unsigned long long* p = reinterpret_cast<unsigned long long*>(a.slots);
  for (int i = threadIdx.x; i < (int)(kSsSlots * sizeof(SsSlot) / 8); i += kBlock) p[i] = 0ull;
  if (threadIdx.x == 0) a.tot[0] = 0ull;
  __syncthreads();
  SsState st{};
  st.t0 = wall_clock64();
  if (bovm) {
    const int rb = a.row_ptr[s], d = a.row_ptr[s + 1] - rb;
    if (d > a.hchunk) put_chunks(a, a.hq, 0, s, rb, d, threadIdx.x, kBlock);
    if (threadIdx.x == 0) {
      a.q[0] = s;
      SsSlot& c = a.slots[0];
      c.part[0][0] = 1ull;
      c.part[0][1] = c.part[0][2] = (unsigned)d;
      if (d > a.hchunk) c.hqlen = (unsigned)chunks_of(a, d);
      else c.qlen = 1;
      st.s.scout = d;
    }
  }
  if (threadIdx.x == 0) {
    st.s.e2c = a.row_ptr[a.n];
    st.s.force_mode = -1;
    st.s.source = s;
    st.s.last_mode = DAWN_MODE_PUSH;
    a.st[0] = st;
  }
}

// Sum of the edge weights, in one part per workgroup (once per graph).
constexpr int kWsumBlocks = 512;
__global__ void __launch_bounds__(kBlock) ss_wsum_kernel(const int32_t* w, int64_t m,
                                                         unsigned long long* out) {
  __shared__ unsigned long long s_t[kBlock / kWave];
  unsigned long long t = 0;
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < m; k += (int64_t)kWsumBlocks * kBlock)
    t += (unsigned)w[k];
  t = wave_sum_u64(t);
  if (lane_id() == 0) s_t[threadIdx.x / kWave] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kBlock / kWave; i++) t += s_t[i];
    out[blockIdx.x] = t;
  }
}

// Level 1 for min-plus, as SSSP_CPU::SSSP initialises it
// (src/algorithm/cpu/sssp.cpp:40-46): every listed out-edge of the source
// writes its weight in row order (a later duplicate overwrites an earlier
// one), the distinct neighbours form the first frontier, distance[source]
// = 0, and the source is never relaxed afterwards.  One workgroup: each
// neighbour's slot first takes -1 - (its last listed edge) by atomicMin,
// then that edge alone replaces it by its weight (weights are >= 0, so no
// other edge of the neighbour matches).  A hub source's list in one thread
// took 100k dependent round trips.
__global__ void __launch_bounds__(kSsBlock) sssp_seed_kernel(SsArgs a) {
  __shared__ unsigned s_len[2], s_near;
  __shared__ unsigned long long s_c[3], s_wsum;
  const int32_t s = a.source;
  const int32_t b = a.row_ptr[s], e = a.row_ptr[s + 1];
  if (threadIdx.x < 2) s_len[threadIdx.x] = 0u;
  if (threadIdx.x < 3) s_c[threadIdx.x] = 0ull;
  if (threadIdx.x == 3) {
    s_near = 0u;
    s_wsum = 0ull;
  }
  for (int32_t k = b + threadIdx.x; k < e; k += kSsBlock) atomicMin(&a.dist[a.col[k]], -1 - k);
  __syncthreads();
  for (int32_t k = b + threadIdx.x; k < e; k += kSsBlock) {
    const int32_t v = a.col[k];
    if (__hip_atomic_load(&a.dist[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != -1 - k) continue;
    __hip_atomic_store(&a.dist[v], a.w[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v == s) continue;
    atomicMax(&s_near, (unsigned)(kInf - a.w[k]));
    atomicOr(&a.bm[v >> 5], 1u << (v & 31));
    const int rb = a.row_ptr[v], d = a.row_ptr[v + 1] - rb;
    if (d > a.hchunk)
      put_chunks(a, a.hq, atomicAdd(&s_len[1], (unsigned)chunks_of(a, d)), v, rb, d, 0, 1);
    else if (d > 0)
      a.q[atomicAdd(&s_len[0], 1u)] = v;
    atomicAdd(&s_c[0], 1ull);
    atomicAdd(&s_c[1], (unsigned long long)d);
    atomicAdd(&s_c[2], (unsigned long long)(d > 0 ? d : 1));
  }
  if (threadIdx.x < kWsumBlocks) {
    const unsigned long long x = wave_sum_u64(a.wsum[threadIdx.x]);
    if (lane_id() == 0) atomicAdd(&s_wsum, x);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  __hip_atomic_store(&a.dist[s], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  SsSlot& c = a.slots[0];
  for (int i = 0; i < 3; i++) c.part[0][i] = s_c[i];
  c.part[0][3] = s_near;
  c.qlen = s_len[0];
  c.hqlen = s_len[1];
  SsState& st = a.st[0];
  st.s.step = 1;
  st.s.scout = (long long)s_c[2];
  if (a.delta_scale > 0) st.delta = max(1ll, (long long)ceil(a.delta_scale * (double)s_wsum));
}

// A head that may join the new level: BOVM if unreached, min-plus if the path
// over this edge is shorter than its distance.
struct Head {
  int32_t v, nd, deg;
  bool cand, join;
};

// First half: the head's distance is compared; the second half's accesses
// (which need no answer from each other) are the atomicMin (min-plus), the
// atomicOr on the level's bitmap, whose first setter joins the vertex to the
// level, and its out-degree.  A min-plus head whose distance another edge
// has lowered below nd meanwhile may still be joined here: that edge's tail
// was expanded in this step too, so the head belongs to the next frontier.
template <bool MP>
__device__ __forceinline__ Head head_of(const SsArgs& a, int lv, int32_t src, int e, int du) {
  Head h{0, lv, 0, false, false};
  if (e >= 0) {
    h.v = a.col[e];
    if (MP) h.nd = minplus(du, a.w[e]);
    h.cand = MP ? h.v != src : true;
  }
  return h;
}
template <bool MP>
__device__ __forceinline__ void test_head(const SsArgs& a, Head& h) {
  if (h.cand) h.cand = MP ? h.nd < a.dist[h.v] : a.dist[h.v] == kInf;
}
template <bool MP>
__device__ __forceinline__ void join_head(const SsArgs& a, Head& h, uint32_t* bm_out, Acc& acc) {
  if (!h.cand) return;
  const uint32_t bit = 1u << (h.v & 31);
  if (MP) atomicMin(&a.dist[h.v], h.nd);
  const uint32_t old = atomicOr(&bm_out[h.v >> 5], bit);
  h.deg = a.row_ptr[h.v + 1] - a.row_ptr[h.v];
  h.join = (old & bit) == 0;
  if (MP) acc.dist(h.nd);
  else if (h.join) a.dist[h.v] = h.nd;
}

// Counters of a completed level.
struct SsLevel {
  unsigned long long fv, fe, scout;
  unsigned qlen, hqlen;
};

// What a step launch decides, in LDS; the same in every workgroup.
struct SsCtl {
  SsState st;  // state of the step to run (s.step = the level to discover)
  SsLevel c;   // level s.step - 1
  int run;     // 0: nothing left, 1: all workgroups expand, 2: one walks small levels
  int fresh;   // run 0: this launch found the frontier empty
  float x[8];
};

// Levels of at most kSmallEdges out-edges (and so at most as many vertices
// found behind them) are walked by one workgroup, one after the other, within
// a launch: a level costs about 4 us of dependent accesses there, and 9-12 us
// as a step of its own (launch, decision, reservation of queue ranges, the
// same accesses).  A level of 4000 edges takes one workgroup about 20 us, the
// grid 12.  kSmallLevels bounds a launch on paths (about 20 ms).
constexpr int kSmallEdges = 2048;
constexpr int kSmallLevels = 4096;
// Min-plus: frontiers of at least n / kMpDense vertices are read from the bitmap.
constexpr unsigned long long kMpDense = 32;

// Whether the level with counters c may be walked by one workgroup under
// `mode`: its queue exists and holds every vertex with out-edges.
__device__ __forceinline__ bool small_level(const SsLevel& c, int mode) {
  return mode == DAWN_MODE_PUSH && c.qlen != kNoQueue && c.fe <= kSmallEdges && c.fv <= kSmallEdges;
}

// Mode of the step after the level with counters c, by the rule or the
// forced policy; keeps the rule state current.  The learned network's choice
// is made by the caller (it needs the workgroup).  Min-plus has no rule of
// the reference: it pushes, in vertex order from the bitmap once the frontier
// is dense enough for its vertices to share lines (from n / 32 on: 2048^2 grid
// 1.61 ms, by the queue alone 1.98, by the bitmap alone 1.76; random graphs
// within 3% of each other).  A pull relaxes every edge of the graph per step
// and was never faster (2048^2 grid: 3.6 ms; RMAT scale 18: 14.5 against 0.7).
template <bool MP>
__device__ inline int ss_rule_mode(const SsRun& r, SchedState& s, const SsLevel& c) {
  if (r.force >= 0) return r.force;
  if (r.p.policy == DAWN_POLICY_PUSH) return DAWN_MODE_PUSH;
  if (r.p.policy == DAWN_POLICY_PULL) return DAWN_MODE_PULL;
  if (r.p.policy == DAWN_POLICY_BITMAP) return DAWN_MODE_BITMAP;
  if (MP) return c.fv * kMpDense >= (unsigned long long)r.p.n ? DAWN_MODE_BITMAP : DAWN_MODE_PUSH;
  LevelCounters lc{};
  lc.fv = c.fv;
  lc.fe = c.fe;
  lc.scout = c.scout;
  return sched_fixed_mode(s, lc, r.p);
}

__device__ __forceinline__ bool learned(const SsRun& r) {
  return r.p.policy == DAWN_POLICY_LEARNED && r.p.mlp && r.force < 0;
}

// A frontier without a queue (after a pull step) is expanded top-down from
// its bitmap.
__device__ __forceinline__ int queue_mode(int mode, const SsLevel& c) {
  return mode == DAWN_MODE_PUSH && c.qlen == kNoQueue ? DAWN_MODE_BITMAP : mode;
}

__device__ __forceinline__ void ss_advance(SchedState& s, const SsLevel& c, int mode) {
  s.step += 1;
  s.mode = mode;
  s.last_mode = mode;
  s.work_fv += c.fv;  // the level this step expands
  s.work_fe += c.fe;
}

// Every workgroup decides from the same state and counters: a launch of its
// own for the decision cost 4-5 us per step.  Called by all threads; the
// result is in ctl after the last barrier.
template <bool MP>
__device__ inline void ss_decide(const SsRun& r, int k, SsCtl& ctl) {
  const SsArgs& a = r.a;
  if (threadIdx.x < kWave) {
    const SsSlot& slot = a.slots[k % kSsSlots];
    SsState st = a.st[k % kSsSlots];
    unsigned long long fv = slot.part[lane_id()][0], fe = slot.part[lane_id()][1],
                       sc = slot.part[lane_id()][2];
    const unsigned qlen = slot.qlen, hqlen = slot.hqlen;
    unsigned near = 0;
    unsigned long long de = 0;
    if (MP) {
      near = (unsigned)wave_max_i32((int)slot.part[lane_id()][3]);
      de = wave_sum_u64(slot.part[lane_id()][4]);
    }
    fv = wave_sum_u64(fv);
    fe = wave_sum_u64(fe);
    sc = wave_sum_u64(sc);
    if (threadIdx.x == 0) {
      const SsLevel c{fv, fe, sc, qlen, hqlen};
      ctl.c = c;
      ctl.run = 0;
      ctl.fresh = 0;
      if (!st.s.done) {
        if (c.fv == 0) {
          st.s.done = 1;
          st.s.levels = st.s.step;  // levels 0..step-1 are non-empty
          ctl.fresh = 1;
        } else {
          const SchedState before = st.s;
          const int mode = ss_rule_mode<MP>(r, st.s, c);
          st.launches += 1;
          if (MP) {
            st.s.work_fe -= de;  // counted with the frontier, not expanded
            if (st.delta > 0) st.thr = max(st.thr, (long long)(kInf - near)) + st.delta;
          }
          // Small levels are pushed whatever the network would say.
          ctl.run = r.small && small_level(c, learned(r) ? DAWN_MODE_PUSH : mode) ? 2 : 1;
          if (ctl.run == 1 && (learned(r) || r.tr.feat)) {
            LevelCounters lc{};
            lc.fv = c.fv;
            lc.fe = c.fe;
            float x[8];
            sched_features(lc, before.step + 1, r.p, before, x);
            for (int i = 0; i < 8; i++) ctl.x[i] = x[i];
          }
          ss_advance(st.s, c, ctl.run == 2 ? DAWN_MODE_PUSH : queue_mode(mode, c));
        }
      }
      ctl.st = st;
    }
  }
  __syncthreads();
  if (ctl.run == 1 && learned(r)) {
    const int m = queue_mode(sched_mlp_mode(ctl.x, r.p), ctl.c);
    if (threadIdx.x == 0) ctl.st.s.mode = ctl.st.s.last_mode = m;
    __syncthreads();
  }
  if (threadIdx.x == 0 && ctl.run) ctl.st.mode_steps[ctl.st.s.mode] += 1;
}

// LDS of the small-level walk: the level's vertices (min-plus: their slots in
// a hash table that also holds their distances), then the scanned
// out-degrees, first edges and distances of the level being expanded.
template <bool MP>
struct SmallLds {
  static constexpr int kTab = MP ? 2 * kSmallEdges : 1;
  int32_t q[kSmallEdges];
  int off[kSmallEdges];
  int beg[kSmallEdges];
  int du[MP ? kSmallEdges : 1];
  int32_t tab_v[kTab];
  int32_t tab_d[kTab];
  int scan[kSsWaves];
  unsigned n, zero, hq, hn, near;
};

// Slot of v in the level's table (at most half full); *first: v was not there.
template <bool MP>
__device__ __forceinline__ unsigned tab_insert(SmallLds<MP>& s, int32_t v, bool* first) {
  constexpr unsigned kTab = SmallLds<MP>::kTab;
  unsigned h = ((unsigned)v * 2654435761u) % kTab;
  for (;;) {
    const int32_t old = atomicCAS(&s.tab_v[h], -1, v);
    if (old == -1 || old == v) {
      *first = old == -1;
      return h;
    }
    h = (h + 1) % kTab;
  }
}

// Walks levels in one workgroup, from level ctl.st.s.step on, until a level
// is empty, too large, or the rule leaves PUSH; then writes the last level's
// queue, bitmap bits and counters as a step of the whole grid would have left
// them.  A level's edges are spread over the threads by one scan of its
// vertices' out-degrees, so a level is one chain of three dependent accesses:
// offsets, columns, and one atomicMin on the distance, whose old value tells
// a first arrival (hop counts only grow) or an improvement.  The frontier
// bitmap stays out of the loop: min-plus keeps the level's distinct vertices,
// with their distances, in an LDS table.
template <bool MP>
__device__ inline void small_levels(const SsRun& run, int k, SmallLds<MP>& s, SsCtl& ctl) {
  constexpr int kPer = kSmallEdges / kSsBlock;
  const SsArgs& a = run.a;
  const int t = threadIdx.x;
  const int32_t src = ctl.st.s.source;
  const SsOut o = out_of(a, k);
  auto clear_table = [&]() {
    if (MP)
      for (int i = t; i < SmallLds<MP>::kTab; i += kSsBlock) {
        s.tab_v[i] = -1;
        s.tab_d[i] = kInf;
      }
  };
  {  // The level's vertices: the light queue and the first chunk of each heavy one.
    const int32_t* q_in = a.q + (int64_t)(k & 1) * a.n;
    const int2* hq_in = a.hq + (int64_t)(k & 1) * a.hcap;
    const unsigned qn = ctl.c.qlen, hn = ctl.c.hqlen;
    if (t == 0) s.n = 0u;
    clear_table();
    __syncthreads();
    for (unsigned i = t; i < qn + hn; i += kSsBlock) {
      int32_t v;
      if (i < qn) {
        v = q_in[i];
      } else {
        const int2 h = hq_in[i - qn];
        v = h.y == a.row_ptr[h.x] ? h.x : -1;
      }
      if (v < 0) continue;
      if (MP) {
        bool first;
        const unsigned h = tab_insert(s, v, &first);
        s.tab_d[h] = a.dist[v];
        v = (int32_t)h;
      }
      s.q[atomicAdd(&s.n, 1u)] = v;
    }
    __syncthreads();
  }
  for (int it = 0;; it++) {
    const unsigned cnt = s.n;
    int32_t v[kPer];
    int rb[kPer], d[kPer], du[MP ? kPer : 1], sum = 0;
#pragma unroll
    for (int r = 0; r < kPer; r++) {
      const unsigned i = (unsigned)(t * kPer + r);
      v[r] = -1;
      rb[r] = d[r] = 0;
      if (i < cnt) {
        v[r] = MP ? s.tab_v[s.q[i]] : s.q[i];
        if (MP) du[r] = s.tab_d[s.q[i]];
        rb[r] = a.row_ptr[v[r]];
        d[r] = a.row_ptr[v[r] + 1] - rb[r];
      }
    }
#pragma unroll
    for (int r = 0; r < kPer; r++) sum += d[r];
    if (t == 0) s.zero = 0u;
    int total;
    int off = ss_scan(sum, s.scan, &total);
    if (t == 0) s.n = 0u;
    clear_table();
    if (it > 0) {  // the level just found: go on, or leave it to the grid?
      int z = 0;
#pragma unroll
      for (int r = 0; r < kPer; r++) z += v[r] >= 0 && d[r] == 0;
      if (z) atomicAdd(&s.zero, (unsigned)z);
      __syncthreads();
      if (t == 0) {
        const SsLevel c{cnt, (unsigned long long)total, (unsigned long long)total + s.zero, cnt, 0u};
        ctl.c = c;
        if (cnt == 0) {
          ctl.st.s.done = 1;
          ctl.st.s.levels = ctl.st.s.step;
          ctl.run = 0;
          ctl.fresh = 1;
        } else {
          SchedState next = ctl.st.s;
          const int mode = ss_rule_mode<MP>(run, next, c);
          if (it < kSmallLevels && small_level(c, learned(run) ? DAWN_MODE_PUSH : mode)) {
            ss_advance(next, c, DAWN_MODE_PUSH);
            ctl.st.s = next;
            ctl.st.mode_steps[DAWN_MODE_PUSH] += 1;
          } else {
            ctl.run = 1;
          }
        }
      }
      __syncthreads();
      if (ctl.run != 2) {
        if (ctl.run == 1) {  // hand over
          uint32_t* bm_out = a.bm + (int64_t)((k + 1) % 3) * a.words;
          if (t == 0) s.hq = s.hn = s.near = 0u;
          // Dealt out wave by wave, so that the chunk lists of neighbouring
          // hubs are written by different waves.
#pragma unroll
          for (int r = 0; r < kPer; r++) s.off[t * kPer + r] = v[r];
          __syncthreads();
          for (int r = 0; r < kPer; r++) {
            const int32_t x = s.off[r * kSsBlock + lane_id() * kSsWaves + t / kWave];
            int xb = 0, xd = 0;
            if (x >= 0) {
              xb = a.row_ptr[x];
              xd = a.row_ptr[x + 1] - xb;
              atomicOr(&bm_out[x >> 5], 1u << (x & 31));
            }
            if (xd > 0 && xd <= a.hchunk) o.q[atomicAdd(&s.hq, 1u)] = x;
            wave_put_chunks(a, o.hq, &s.hn, x, xb, xd);
          }
          if (MP) {
            unsigned near = 0;
#pragma unroll
            for (int r = 0; r < kPer; r++)
              if (v[r] >= 0) near = max(near, (unsigned)(kInf - du[r]));
            if (near) atomicMax(&s.near, near);
          }
          __syncthreads();
          if (t == 0) {
            if (MP) o.slot->part[0][3] = s.near;
            o.slot->part[0][0] = ctl.c.fv;
            o.slot->part[0][1] = ctl.c.fe;
            o.slot->part[0][2] = ctl.c.scout;
            o.slot->qlen = s.hq;
            o.slot->hqlen = s.hn;
          }
        }
        return;
      }
    }
    // Expand level step - 1 into level step.
    const int lv = ctl.st.s.step;
#pragma unroll
    for (int r = 0; r < kPer; r++) {
      const int i = t * kPer + r;
      s.off[i] = off;
      s.beg[i] = rb[r] - off;
      if (MP) s.du[i] = du[r];
      off += d[r];
    }
    __syncthreads();
    int32_t hv[kPer], nd[kPer], old[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++) {
      const int e = t + r * kSsBlock;
      hv[r] = -1;
      nd[r] = lv;
      if (e < total) {
        int j = 0;  // the last entry that starts at or before e
#pragma unroll
        for (int w = kSmallEdges / 2; w >= 1; w >>= 1)
          if (s.off[j + w] <= e) j += w;
        const int ke = s.beg[j] + e;
        hv[r] = a.col[ke];
        if (MP) {
          nd[r] = minplus(s.du[j], a.w[ke]);
          if (hv[r] == src || nd[r] == kInf) hv[r] = -1;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < kPer; r++) {
      old[r] = -1;
      if (hv[r] >= 0) old[r] = atomicMin(&a.dist[hv[r]], nd[r]);
    }
#pragma unroll
    for (int r = 0; r < kPer; r++) {
      bool f = old[r] > nd[r];
      if (MP && f) {
        const unsigned h = tab_insert(s, hv[r], &f);
        atomicMin(&s.tab_d[h], nd[r]);
        hv[r] = (int32_t)h;
      }
      const int at = wave_append(&s.n, f);
      if (f) s.q[at] = hv[r];
    }
    __syncthreads();
  }
}

// The final state, once, to the host (one thread): BOVM's levels are
// disjoint, so its expanded levels are the vertices reached.
template <bool MP>
__device__ inline void ss_finish(const SsArgs& a, SsCtl& ctl) {
  if (!MP) {
    ctl.st.reached = ctl.st.s.work_fv;
    ctl.st.edges = ctl.st.s.work_fe;
  }
  ctl.st.t1 = wall_clock64();
  if (a.host) {
    *a.host = ctl.st;
    __threadfence_system();
  }
}

// Min-plus, after the step launches up to launch k: vertices reached and
// their out-edges, if the traversal is done.  Each workgroup writes its part;
// the last one to count itself in (one atomic each: several same-address
// atomics per workgroup took longer than the pass) sums them for the host.
constexpr unsigned kReachBlocks = 256;
__global__ void __launch_bounds__(kSsBlock) ss_reach_kernel(SsArgs a, int k) {
  __shared__ unsigned long long s_t[2];
  __shared__ unsigned s_last;
  if (!a.st[k % kSsSlots].s.done) return;
  if (threadIdx.x < 2) s_t[threadIdx.x] = 0ull;
  __syncthreads();
  unsigned long long cnt = 0, edges = 0;
  const int64_t gs = (int64_t)gridDim.x * kSsBlock;
  for (int64_t v0 = (int64_t)blockIdx.x * kSsBlock + threadIdx.x; v0 < a.n; v0 += 4 * gs) {
    int d[4], g[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int64_t v = min(v0 + j * gs, (int64_t)a.n - 1);
      d[j] = a.dist[v];
      g[j] = a.row_ptr[v + 1] - a.row_ptr[v];
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (v0 + j * gs < a.n && d[j] != kInf) {
        cnt += 1;
        edges += (unsigned)g[j];
      }
  }
  cnt = wave_sum_u64(cnt);
  edges = wave_sum_u64(edges);
  if (lane_id() == 0 && cnt) {
    atomicAdd(&s_t[0], cnt);
    atomicAdd(&s_t[1], edges);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    a.tot[1 + 2 * blockIdx.x] = s_t[0];
    a.tot[2 + 2 * blockIdx.x] = s_t[1];
    __threadfence();
    s_last = atomicAdd(&a.tot[0], 1ull) + 1 == gridDim.x;
  }
  __syncthreads();
  if (!s_last || threadIdx.x >= kWave) return;
  __threadfence();
  cnt = edges = 0;
  for (unsigned b = threadIdx.x; b < gridDim.x; b += kWave) {
    cnt += __hip_atomic_load(&a.tot[1 + 2 * b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    edges += __hip_atomic_load(&a.tot[2 + 2 * b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  cnt = wave_sum_u64(cnt);
  edges = wave_sum_u64(edges);
  if (threadIdx.x != 0) return;
  a.host->reached = cnt;
  a.host->edges = edges;
  __threadfence_system();
}

// Unreached vertices look for a tail in the frontier bitmap; each vertex is
// written only by its own lane.
__device__ __forceinline__ void pull_bfs(const SsArgs& a, int lv, const uint32_t* bm_in,
                                         uint32_t* bm_out, Acc& acc) {
  const int lane = lane_id();
  const int64_t wstride = (int64_t)gridDim.x * kSsBlock;
  for (int64_t base = (int64_t)blockIdx.x * kSsBlock + (threadIdx.x & ~(kWave - 1)); base < a.n;
       base += wstride) {
    const int32_t v = (int32_t)(base + lane);
    int beg = 0, deg = 0;
    if (v < a.n && a.dist[v] == kInf) {
      beg = a.in_row_ptr[v];
      deg = a.in_row_ptr[v + 1] - beg;
    }
    bool found = false;
    // Rounds of four in-edges per lane (columns by one 16-byte load, probed
    // two by two), until every lane has found a frontier tail or run out;
    // of a heavy vertex only the first two rounds, the rest by the whole
    // wave.  Bound by requests (each lane reads its own list and probes a
    // word per edge), so probes past the first hit cost: 128 edges of a
    // heavy vertex probed at once made a sparse step on RMAT scale 22 60%
    // slower than 64.
    const int lim = deg < kHeavyDegree ? deg : 8;
    for (int j = 0; __ballot(!found && j < lim); j += 4) {
      if (!found && j < lim) {
        const int32_t* p = a.in_col + beg + j;
        Cols4 u;
        if (j + 4 <= deg) {
          u = *reinterpret_cast<const Cols4*>(p);
        } else {
          const int r = deg - 1 - j;  // 0..2: repeat the last column
          u = {{p[0], p[min(1, r)], p[r], p[r]}};
        }
        const bool f0 = test_bit(bm_in, u.c[0]), f1 = test_bit(bm_in, u.c[1]);
        found = f0 || f1;
        if (!found) {
          const bool f2 = test_bit(bm_in, u.c[2]), f3 = test_bit(bm_in, u.c[3]);
          found = f2 || f3;
        }
      }
    }
    uint64_t hm = __ballot(!found && deg >= kHeavyDegree);
    while (hm) {
      const int l = __ffsll((unsigned long long)hm) - 1;
      hm &= hm - 1;
      const int hb = __shfl(beg, l), he = hb + __shfl(deg, l);
      bool f = false;
      for (int k0 = hb + 8; k0 < he; k0 += kWave) {
        const int k = k0 + lane;
        const bool h = k < he && test_bit(bm_in, a.in_col[k]);
        if (__ballot(h)) { f = true; break; }
      }
      if (lane == l) found = f;
    }
    if (found) a.dist[v] = lv;
    const uint64_t fm = __ballot(found);
    if (lane == 0) {
      bm_out[base >> 5] = (uint32_t)fm;
      bm_out[(base >> 5) + 1] = (uint32_t)(fm >> 32);
    }
    if (found) acc.add(a.row_ptr[v + 1] - a.row_ptr[v]);  // bitmap only: no queue entries
  }
}

__device__ __forceinline__ void pull_minplus(const SsArgs& a, int32_t src, const uint32_t* bm_in,
                                             uint32_t* bm_out, Acc& acc) {
  const int lane = lane_id();
  // Every vertex takes the minimum over its in-edges from frontier
  // vertices; each vertex is written only by its own lane.
  const int64_t wstride = (int64_t)gridDim.x * kSsBlock;
  for (int64_t base = ((int64_t)(threadIdx.x / kWave) * gridDim.x + blockIdx.x) * kWave; base < a.n;
       base += wstride) {
    const int32_t v = (int32_t)(base + lane);
    const bool cand = v < a.n && v != src;
    int beg = 0, deg = 0;
    int32_t cur = kInf;
    if (cand) {
      beg = a.in_row_ptr[v];
      deg = a.in_row_ptr[v + 1] - beg;
      cur = a.dist[v];
    }
    int32_t best = cur;
    const bool light = cand && deg < kHeavyDegree;
    const int maxd = wave_max_i32(light ? deg : 0);
    for (int j = 0; j < maxd; j++) {
      if (light && j < deg) {
        const int32_t u = a.in_col[beg + j];
        if (test_bit(bm_in, u)) {
          long long nd = (long long)a.dist[u] + a.in_w[beg + j];
          if (nd < best) best = (int32_t)nd;
        }
      }
    }
    uint64_t hm = __ballot(cand && deg >= kHeavyDegree);
    while (hm) {
      const int l = __ffsll((unsigned long long)hm) - 1;
      hm &= hm - 1;
      const int hb = __shfl(beg, l), he = hb + __shfl(deg, l);
      int32_t hbest = kInf;
      for (int k = hb + lane; k < he; k += kWave) {
        const int32_t u = a.in_col[k];
        if (test_bit(bm_in, u)) {
          long long nd = (long long)a.dist[u] + a.in_w[k];
          if (nd < hbest) hbest = (int32_t)nd;
        }
      }
      for (int o = 32; o >= 1; o >>= 1) hbest = min(hbest, __shfl_xor(hbest, o));
      if (lane == l && hbest < best) best = hbest;
    }
    const bool found = cand && best < cur;
    if (found) {
      a.dist[v] = best;
      acc.dist(best);
    }
    const uint64_t fm = __ballot(found);
    if (lane == 0) {
      bm_out[base >> 5] = (uint32_t)fm;
      bm_out[(base >> 5) + 1] = (uint32_t)(fm >> 32);
    }
    if (found) acc.add(a.row_ptr[v + 1] - a.row_ptr[v]);  // bitmap only: no queue entries
  }
}

// One step of the traversal: BOVM (discovers level lv) or min-plus
// (GOVM/GOVMP semantics: relaxes the out-edges of the vertices whose distance
// dropped in the previous step).  k: the launch's number modulo 12.
//
// Min-plus relaxes in rough distance order: a step expands the frontier
// vertices below a threshold that moves on by delta every step (and past the
// smallest frontier distance), and leaves the others in the frontier.  The
// fixed point is the same; vertices whose distance would still drop are
// mostly not expanded too early.  delta = 2 x mean weight / mean degree, about
// the distance the shortest paths' front covers per hop: in a CPU count the
// steps stay as many as without (2048^2 grid with weights in [1, 1000]: 79 ->
// 80; random graphs of degree 4-32: 27-35, the same) and the relaxations per
// edge fall from 2.7-5.5 to 1.3-1.8; half of it takes 1.5-2x the steps, twice
// of it saves almost no relaxations.  On skewed graphs (RMAT: 16 steps, 4.5
// relaxations per edge) it takes 59 steps for 3.7, so graphs with a vertex of
// more than 16 times the mean degree use no threshold.
template <bool MP>
__global__ void __launch_bounds__(kSsBlock, 8) ss_step_kernel(SsRun run, int k) {
  __shared__ SsCtl ctl;
  __shared__ union {
    struct {
      SsStage sg;
      PushLds<MP> push;
    } wide;
    SmallLds<MP> small;
  } lds;
  const SsArgs& a = run.a;
  ss_decide<MP>(run, k, ctl);
  if (ctl.run != 0) clear_next(a, k);
  if (ctl.run != 1) {  // uniform over the grid: nothing left, or small levels
    if (blockIdx.x != 0) return;
    if (ctl.run == 2) {
      small_levels<MP>(run, k, lds.small, ctl);
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      if (ctl.fresh) ss_finish<MP>(a, ctl);
      a.st[(k + 1) % kSsSlots] = ctl.st;
    }
    return;
  }
  const int lv = ctl.st.s.step, mode = ctl.st.s.mode;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.st[(k + 1) % kSsSlots] = ctl.st;
    if (run.tr.mode && lv < kTraceMax) {
      run.tr.mode[lv] = mode;
      for (int i = 0; i < 8; i++) run.tr.feat[lv * 8 + i] = ctl.x[i];
    }
  }
  const int32_t src = a.source;
  const uint32_t* bm_in = a.bm + (int64_t)(k % 3) * a.words;
  uint32_t* bm_out = a.bm + (int64_t)((k + 1) % 3) * a.words;
  const SsOut o = out_of(a, k);
  SsStage& sg = lds.wide.sg;
  sg.init();
  Acc acc;
  // A frontier vertex at or beyond the threshold stays in the frontier, but for
  // one without a distance (its edge from the source weighs INT32_MAX): no path
  // goes on from it, and it would never get below.
  const int32_t thr = MP && ctl.st.delta > 0 ? (int32_t)min(ctl.st.thr, (long long)kInf) : kInf;
  auto defer = [&](bool yes, int32_t u, int du, int deg) {
    const uint32_t bit = 1u << (u & 31);
    yes = yes && du != kInf;
    const bool first = yes && (atomicOr(&bm_out[u >> 5], bit) & bit) == 0;
    if (yes) acc.dist(du);
    if (first) acc.de += (unsigned)deg;
    sg.append(a, o, first, u, deg, acc);
  };
  auto edge = [&](int du0, int du1, int e0, int e1) {
    Head h0 = head_of<MP>(a, lv, src, e0, du0), h1 = head_of<MP>(a, lv, src, e1, du1);
    test_head<MP>(a, h0);
    test_head<MP>(a, h1);
    join_head<MP>(a, h0, bm_out, acc);
    join_head<MP>(a, h1, bm_out, acc);
    sg.append(a, o, h0.join, h0.v, h0.deg, acc);
    sg.append(a, o, h1.join, h1.v, h1.deg, acc);
  };
  if (mode == DAWN_MODE_PUSH) {
    push_edges<MP>(a, lds.wide.push, k, ctl.c.qlen, ctl.c.hqlen, thr, edge, defer);
  } else if (mode == DAWN_MODE_BITMAP) {  // (min-plus: GOVMP shape)
    bitmap_edges<MP>(a, lds.wide.push, bm_in, thr, edge, defer);
  } else {
    // PULL: the bitmap only, no queue entries.
    if (blockIdx.x == 0 && threadIdx.x == 0) o.slot->qlen = kNoQueue;
    if constexpr (MP) pull_minplus(a, src, bm_in, bm_out, acc);
    else pull_bfs(a, lv, bm_in, bm_out, acc);
  }
  sg.flush<MP>(a, o, acc);
}

int ensure_ss(dawn_graph* g) {
  if (!g->ss) g->ss = new SsWorkspace();
  SsWorkspace* ws = g->ss;
  if (ws->n == g->n && ws->st.p) return DAWN_OK;
  ws->n = g->n;
  ws->hcap = 2 * (g->m / kHeavyChunk) + 1;
  DAWN_TRY(ws->q.alloc((size_t)2 * g->n));
  DAWN_TRY(ws->hq.alloc((size_t)2 * ws->hcap));
  DAWN_TRY(ws->bm.alloc((size_t)3 * (((int64_t)g->n + 63) / 64 * 2)));
  DAWN_TRY(ws->slots.alloc(kSsSlots));
  DAWN_TRY(ws->tot.alloc(1 + 2 * kReachBlocks));
  if (!ws->h_state) DAWN_HIP(hipHostMalloc((void**)&ws->h_state, sizeof(SsState)));
  return ws->st.alloc(kSsSlots);
}

// Launch arguments that depend on the graph and the call alone.
SsRun make_run(const dawn_graph* g, int32_t source, int32_t policy) {
  SsRun r{};
  SsArgs& a = r.a;
  a.n = g->n;
  a.source = source;
  a.words = ((int64_t)g->n + 63) / 64 * 2;
  a.row_ptr = g->row_ptr;
  a.col = g->col;
  a.w = g->weight;
  a.in_row_ptr = g->in_row_ptr;
  a.in_col = g->in_col;
  a.in_w = g->in_weight;
  a.oc_v = g->oc_v;
  a.oc_beg = g->oc_beg;
  a.oc_end = g->oc_end;
  a.num_oc = g->num_oc;
  a.heavy = g->knobs.heavy_degree;
  SchedParams& p = r.p;
  p.n = g->n;
  p.m = g->m;
  p.policy = policy;
  p.alpha = 15;
  p.beta = 18;
  p.batched = 0;
  p.allow_pull = 1;
  p.avg_degree = g->n ? (float)((double)g->m / g->n) : 0.f;
  p.max_degree = (float)g->max_out_degree;
  const double avg = p.avg_degree;
  a.delta_scale = g->m > 0 && g->max_out_degree <= 16 * avg ? 2.0 / (avg * (double)g->m) : 0.0;
  r.force = -1;
  r.small = 1;
  return r;
}

// The graph's workspace.
void use_workspace(SsRun& r, const SsWorkspace* ws) {
  SsArgs& a = r.a;
  a.dist = ws->dist.p;
  a.q = ws->q.p;
  a.hq = ws->hq.p;
  a.hcap = ws->hcap;
  a.hchunk = kHeavyChunk;
  a.bm = ws->bm.p;
  a.slots = ws->slots.p;
  a.tot = ws->tot.p;
  a.st = ws->st.p;
}

unsigned ss_grid(const dawn_graph* g) { return grid_for(std::max<int64_t>(g->n, 1), kSsBlock, kSsGrid); }

int ss_start(const SsRun& r, int kind, hipStream_t s) {
  ss_fill_kernel<<<grid_for(std::max<int64_t>(3 * r.a.words, r.a.n / 4)), kBlock, 0, s>>>(r.a, kind == 0);
  if (kind) sssp_seed_kernel<<<1, kSsBlock, 0, s>>>(r.a);
  DAWN_HIP(hipGetLastError());
  return DAWN_OK;
}

void ss_step(const SsRun& r, int kind, int64_t k, unsigned grid, hipStream_t s) {
  if (kind == 0) ss_step_kernel<false><<<grid, kSsBlock, 0, s>>>(r, (int)(k % 12));
  else ss_step_kernel<true><<<grid, kSsBlock, 0, s>>>(r, (int)(k % 12));
}

// A whole traversal: the first `first` step launches, then more (twice as
// many each time) while the frontier is not empty, one wait after each set.
// A launch past the end costs 2-4 us, a wait too many about 15 us.  h: the
// final state; without a pinned r.a.host it is copied from the device.  reach:
// count the vertices reached (min-plus).
int ss_traverse(const dawn_graph* g, const SsRun& r, int kind, int first, bool reach, hipStream_t s,
                SsState* h) {
  // Forced min-plus pulls look at every vertex in every step, a wave at a time;
  // their waves are spread over four times the workgroups (random graph of
  // 20,000 vertices: 441 us on 20 CUs, 357 on 79).
  const unsigned grid = kind == 1 && r.p.policy == DAWN_POLICY_PULL
                            ? grid_for(std::max<int64_t>(g->n, 1), kSsBlock / 4, kSsGrid)
                            : ss_grid(g);
  const bool pinned = r.a.host != nullptr;
  h->s.done = 0;
  DAWN_TRY(ss_start(r, kind, s));
  const int64_t limit = (int64_t)g->n + 2;
  int64_t k = 0;
  for (int K = first;; K = std::min(64, k == first ? 4 : 2 * K)) {
    for (int i = 0; i < K; i++, k++) ss_step(r, kind, k, grid, s);
    if (reach) ss_reach_kernel<<<grid_for(g->n, kSsBlock, kReachBlocks), kSsBlock, 0, s>>>(r.a, (int)(k % 12));
    DAWN_HIP(hipGetLastError());
    if (!pinned)
      DAWN_HIP(hipMemcpyAsync(h, r.a.st + k % kSsSlots, sizeof(SsState), hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    if (h->s.done) return DAWN_OK;
    if (k > limit) return DAWN_ERR_HIP;  // step bound exceeded
  }
}

// Statistics of a finished traversal.
int ss_stats(const dawn_graph* g, const SsState& h, dawn_stats* stats) {
  int khz = 0;
  DAWN_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, g->device));
  stats->device_ms += khz > 0 ? (double)(h.t1 - h.t0) / khz : 0.0;
  stats->vertices_reached += (int64_t)h.reached;
  stats->edges_reached += (int64_t)h.edges;
  stats->batches += 1;
  stats->frontier_edges += (int64_t)h.s.work_fe;
  for (int m = 0; m < DAWN_NUM_MODES; m++) {
    stats->steps += h.mode_steps[m];
    stats->mode_steps[m] += h.mode_steps[m];
  }
  return DAWN_OK;
}

}  // namespace

// Runs one single-source traversal.  kind 0: BOVM, 1: min-plus.
int run_single_source(dawn_graph* g, int kind, int32_t source, int32_t* dist_out, int32_t policy,
                      dawn_stats* stats) {
  if (!g || source < 0 || source >= g->n) return DAWN_ERR_INVALID_ARG;
  if (kind == 1 && !g->weighted) return DAWN_ERR_NOT_WEIGHTED;
  if (g->h_row_ptr[source] == g->h_row_ptr[source + 1]) return DAWN_ERR_ISOLATED_SOURCE;
  std::lock_guard<std::mutex> guard(g->lock);
  DAWN_HIP(hipSetDevice(g->device));
  DAWN_TRY(ensure_ss(g));
  SsWorkspace* ws = g->ss;
  const bool direct = in_place(g->device, dist_out);
  if (!direct) DAWN_TRY(ws->dist.alloc(g->n));
  SsRun r = make_run(g, source, policy);
  use_workspace(r, ws);
  if (direct) r.a.dist = dist_out;
  r.a.host = ws->h_state;
  if (kind == 1 && !ws->wsum.p) {
    DAWN_TRY(ws->wsum.alloc(kWsumBlocks));
    ss_wsum_kernel<<<kWsumBlocks, kBlock, 0, g->stream>>>(g->weight, g->m, ws->wsum.p);
    DAWN_HIP(hipGetLastError());
  }
  r.a.wsum = ws->wsum.p;
  // The single-source network (trained on single-source steps); without
  // one the learned policy takes the fixed rule.  Min-plus: the fixed rule.
  r.p.mlp = kind == 0 ? sched_single_mlp_device(g->device, &r.p.mlp_norm) : nullptr;
  if (kind == 1 && policy == DAWN_POLICY_LEARNED) r.p.policy = DAWN_POLICY_FIXED;
  // Launches before the first look at the done flag: the knob, else what the
  // last traversal of this kind on the graph took (and the one that finds
  // the frontier empty).
  int K = g->knobs.ss_chunk > 0 ? g->knobs.ss_chunk : 8;
  if (g->knobs.ss_chunk <= 0 && ws->last_launches[kind] > 0) K = std::min(256, ws->last_launches[kind]);
  DAWN_TRY(ss_traverse(g, r, kind, K, kind == 1 && stats, g->stream, ws->h_state));
  ws->last_launches[kind] = ws->h_state->launches + 1;
  if (stats) DAWN_TRY(ss_stats(g, *ws->h_state, stats));
  if (dist_out && !direct) {
    DAWN_HIP(hipMemcpyAsync(dist_out, ws->dist.p, sizeof(int32_t) * g->n, hipMemcpyDefault, g->stream));
    DAWN_HIP(hipStreamSynchronize(g->stream));
  }
  return DAWN_OK;
}

// ---- per-step mode timings (scheduler training data) ------------------------
//
// Every mode discovers the same levels (the frontier of level l is the set
// of vertices at hop distance l, whatever the modes of the steps before), so
// a step starts from the same state in every run: one BOVM traversal per
// mode with that mode forced, each step launched on its own with HIP events
// around the step kernel, gives the time of every mode at every step
// (minimum over `repeats` traversals); one traversal under `policy` gives
// the step features and the policy's choices.

namespace {

// One traversal from r.a.source, step by step.  times: kernel time of each
// step (steps 1..levels).
int ss_stepwise(dawn_graph* g, SsWorkspace* ws, const SsRun& r, std::vector<float>* times, int* levels) {
  hipStream_t s = g->stream;
  const unsigned grid = ss_grid(g);
  DAWN_TRY(ss_start(r, 0, s));
  times->clear();
  for (int64_t k = 0; k <= (int64_t)g->n + 1; k++) {
    DAWN_HIP(hipEventRecord(ws->ev0, s));
    ss_step(r, 0, k, grid, s);
    DAWN_HIP(hipGetLastError());
    DAWN_HIP(hipEventRecord(ws->ev1, s));
    DAWN_HIP(hipMemcpyAsync(ws->h_state, ws->st.p + (k + 1) % kSsSlots, sizeof(SsState),
                            hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    if (ws->h_state->s.done) {
      *levels = ws->h_state->s.levels;
      return DAWN_OK;
    }
    float ms = 0.f;
    DAWN_HIP(hipEventElapsedTime(&ms, ws->ev0, ws->ev1));
    times->push_back(ms);
  }
  return DAWN_ERR_HIP;  // step bound exceeded
}

}  // namespace

int run_ss_record(dawn_graph* g, const int32_t* sources, int32_t S, int32_t repeats,
                  float* features, float* times_ms, int32_t* chosen, int32_t max_rows,
                  int32_t* rows_out, int32_t policy) {
  if (!g || S < 0 || (S > 0 && !sources) || repeats < 1 || !rows_out || max_rows < 0)
    return DAWN_ERR_INVALID_ARG;
  if (g->weighted) return DAWN_ERR_UNSUPPORTED;
  *rows_out = 0;
  std::lock_guard<std::mutex> guard(g->lock);
  DAWN_HIP(hipSetDevice(g->device));
  DAWN_TRY(ensure_ss(g));
  SsWorkspace* ws = g->ss;
  DAWN_TRY(ws->dist.alloc(g->n));
  DAWN_TRY(ws->trace_feat.alloc((size_t)kTraceMax * 8));
  DAWN_TRY(ws->trace_mode.alloc(kTraceMax));
  if (!ws->ev0) DAWN_HIP(hipEventCreate(&ws->ev0));
  if (!ws->ev1) DAWN_HIP(hipEventCreate(&ws->ev1));
  int32_t rows = 0;
  std::vector<float> t, feat;
  std::vector<int32_t> modes;
  for (int32_t i = 0; i < S && rows < max_rows; i++) {
    int64_t src = sources[i] % (int64_t)g->n;
    if (src < 0) src += g->n;
    if (g->h_row_ptr[src] == g->h_row_ptr[src + 1]) continue;  // isolated: no traversal
    SsRun r = make_run(g, (int32_t)src, policy);
    use_workspace(r, ws);
    r.p.mlp = sched_single_mlp_device(g->device, &r.p.mlp_norm);
    r.tr = SchedTrace{ws->trace_feat.p, ws->trace_mode.p};
    r.small = 0;  // every level a step of its own
    // The policy's run: features and choices of steps 1..levels.
    int levels = 0;
    DAWN_TRY(ss_stepwise(g, ws, r, &t, &levels));
    const int nrec = std::min(levels + 1, kTraceMax);
    modes.assign(nrec, 0);
    feat.assign((size_t)nrec * 8, 0.f);
    DAWN_HIP(hipMemcpy(modes.data(), ws->trace_mode.p, sizeof(int32_t) * nrec, hipMemcpyDeviceToHost));
    DAWN_HIP(hipMemcpy(feat.data(), ws->trace_feat.p, sizeof(float) * 8 * nrec, hipMemcpyDeviceToHost));
    // Every mode forced, minimum over the repeats.
    std::vector<float> best((size_t)levels * DAWN_NUM_MODES, 1e30f);
    for (int m = 0; m < DAWN_NUM_MODES; m++)
      for (int rep = 0; rep < repeats; rep++) {
        int lv = 0;
        r.force = m;
        DAWN_TRY(ss_stepwise(g, ws, r, &t, &lv));
        if (lv != levels || (int)t.size() != levels) return DAWN_ERR_HIP;  // modes must agree
        for (int k = 0; k < levels; k++)
          best[(size_t)k * DAWN_NUM_MODES + m] = std::min(best[(size_t)k * DAWN_NUM_MODES + m], t[k]);
      }
    for (int k = 1; k <= levels && k < nrec && rows < max_rows; k++, rows++) {
      for (int j = 0; j < 8; j++) features[(size_t)rows * 8 + j] = feat[(size_t)k * 8 + j];
      for (int m = 0; m < DAWN_NUM_MODES; m++)
        times_ms[(size_t)rows * DAWN_NUM_MODES + m] = best[(size_t)(k - 1) * DAWN_NUM_MODES + m];
      if (chosen) chosen[rows] = modes[k];
    }
  }
  *rows_out = rows;
  return DAWN_OK;
}

// ---- allocation-free BOVM traversal (dawn_bfs_noalloc) --------------------
//
// For callers that cannot allocate device memory (serving loops, harnesses
// that forbid hipMalloc): the single-source BOVM traversal on a fixed
// scratch region instead of the graph's workspace.  The region is the
// file-scope device array `scratch` below, sized for graphs of up to
// kNoAllocMaxN vertices (57 MB); the code object carries it, so each GPU
// the library runs on holds its own copy until the process ends.  Host code
// never passes the array's name to a kernel (in host code it is a stand-in,
// not a device address): once per device, with that device current, the
// first call takes its device address from hipGetSymbolAddress and keeps it
// per device; every kernel argument and copy uses that address.
//
// Every call re-initialises what it reads.  Calls on one GPU share the array,
// so the calls of a process are serialised per device by a lock (two calls
// that overlapped on one GPU would race).  The final state is copied from the
// device (pinned memory would have to be allocated), after sets of step
// launches.  The single-source scheduler network is used only if it is
// already on the device (installing it allocates); otherwise the learned
// policy falls back to the fixed rule, as when no network is set.

constexpr int32_t kNoAllocMaxN = 1 << 22;
constexpr int kNoAllocMaxDevices = 64;

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
constexpr int64_t kNoAllocWords = ((int64_t)kNoAllocMaxN + 63) / 64 * 2;
constexpr size_t kNaDist = 0;
constexpr size_t kNaQ = align256(kNaDist + sizeof(int32_t) * (size_t)kNoAllocMaxN);
constexpr size_t kNaHq = align256(kNaQ + sizeof(int32_t) * 2 * (size_t)kNoAllocMaxN);
constexpr int64_t kNoAllocHeavy = 1 << 18;  // heavy-chunk entries per level
constexpr size_t kNaBm = align256(kNaHq + sizeof(int2) * 2 * (size_t)kNoAllocHeavy);
constexpr size_t kNaSlots = align256(kNaBm + sizeof(uint32_t) * 3 * (size_t)kNoAllocWords);
constexpr size_t kNaTot = align256(kNaSlots + sizeof(SsSlot) * kSsSlots);
constexpr size_t kNaState = align256(kNaTot + sizeof(unsigned long long));
constexpr size_t kNoAllocBytes = align256(kNaState + sizeof(SsState) * kSsSlots);

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

std::mutex g_noalloc_lock[kNoAllocMaxDevices];
unsigned char* g_noalloc_base[kNoAllocMaxDevices] = {};  // device address of `scratch`

}  // namespace

int run_bfs_noalloc(dawn_graph* g, int32_t source, int32_t* dist_out, int32_t policy,
                    dawn_stats* stats) {
  if (!g || source < 0 || source >= g->n) return DAWN_ERR_INVALID_ARG;
  if (g->n > kNoAllocMaxN) {
    set_error("dawn_bfs_noalloc: the graph has more vertices than the scratch region holds "
              "(at most 4194304)");
    return DAWN_ERR_SCRATCH_LIMIT;
  }
  if (g->device < 0 || g->device >= kNoAllocMaxDevices) return DAWN_ERR_UNSUPPORTED;
  if (g->h_row_ptr[source] == g->h_row_ptr[source + 1]) return DAWN_ERR_ISOLATED_SOURCE;
  std::lock_guard<std::mutex> device_guard(g_noalloc_lock[g->device]);
  std::lock_guard<std::mutex> guard(g->lock);
  DAWN_HIP(hipSetDevice(g->device));
  unsigned char* base = g_noalloc_base[g->device];
  if (!base) {
    DAWN_HIP(hipGetSymbolAddress((void**)&base, HIP_SYMBOL(scratch)));
    if (!base) return DAWN_ERR_HIP;
    g_noalloc_base[g->device] = base;
  }
  SsRun r = make_run(g, source, policy);
  SsArgs& a = r.a;
  a.dist = (int32_t*)(base + kNaDist);
  a.q = (int32_t*)(base + kNaQ);
  a.hq = (int2*)(base + kNaHq);
  a.hcap = kNoAllocHeavy;
  // Chunks long enough that the heavy lists of any graph fit the region.
  a.hchunk = kHeavyChunk;
  while (2 * (g->m / a.hchunk) + 1 > kNoAllocHeavy) a.hchunk *= 2;
  a.bm = (uint32_t*)(base + kNaBm);
  a.slots = (SsSlot*)(base + kNaSlots);
  a.tot = (unsigned long long*)(base + kNaTot);
  a.st = (SsState*)(base + kNaState);
  r.p.mlp = sched_single_mlp_if_present(g->device, &r.p.mlp_norm);
  const int K = g->knobs.ss_chunk > 0 ? g->knobs.ss_chunk : 8;
  const auto t0 = std::chrono::steady_clock::now();
  SsState h{};
  DAWN_TRY(ss_traverse(g, r, 0, K, false, g->stream, &h));
  const double ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (stats) {
    dawn_stats st{};
    DAWN_TRY(ss_stats(g, h, &st));
    stats->device_ms += ms;
    stats->vertices_reached += st.vertices_reached;
    stats->edges_reached += st.edges_reached;
    stats->batches += 1;
    stats->steps += st.steps;
    for (int m = 0; m < DAWN_NUM_MODES; m++) stats->mode_steps[m] += st.mode_steps[m];
  }
  if (dist_out) {
    DAWN_HIP(hipMemcpyAsync(dist_out, a.dist, sizeof(int32_t) * g->n, hipMemcpyDefault, g->stream));
    DAWN_HIP(hipStreamSynchronize(g->stream));
  }
  return DAWN_OK;
}

}  // namespace dawn

extern "C" int dawn_bfs_noalloc(const dawn_graph* g, int32_t source, int32_t* dist,
                                int32_t policy, dawn_stats* stats) {
  return dawn::run_bfs_noalloc(const_cast<dawn_graph*>(g), source, dist, policy, stats);
}

