// Many independent graphs of uneven size in one persistent launch.
//
// Replaces, for a batch of graphs, the reference's host loop of per-source
// launches (DAWN::MSSP_GPU::run, src/algorithm/gpu/mssp.cu:26-43 and
// run_Weighted :53-102): here every (graph, source block) is a task in a
// device work queue, and each workgroup pops tasks with one atomic and runs
// the whole traversal inside the workgroup (barriers are workgroup-local, so
// no grid-wide synchronisation exists and every workgroup exits once the
// task counter passes the last task).
//
// Unweighted task: all sources of one graph (or a share of them) as lanes of
// one field per vertex, level-synchronous BOVM with the fields in LDS, pushed
// and pulled (run_lds).  Graphs too large for a workgroup's LDS (more than 1.2
// million vertices), and those whose sources would be several tasks in LDS and
// are done sooner as one where tasks wait for a CU (memory_faster: small graphs
// and graphs of many levels), keep words of up to 64 lanes in memory, sparse BOVM:
//   Q_l = [(v, lanes that reached v at level l)]
//   expand: for (u, f) in Q_l, w in N(u): nv = f & ~seen[w]; if nv,
//           atomicOr(next[w], nv); the first writer appends w to `touched`
//   commit: for w in touched: nw = next[w] & ~seen[w]; next[w] = 0;
//           seen[w] |= nw; dist[b][w] = l+1 for b in nw; Q_{l+1} += (w, nw)
// Weighted task: one source, int32 min-plus (the fixed point of GOVM,
// src/algorithm/cpu/sssp.cpp:141-199, from the reference's seeding), with its
// state in LDS up to 134,000 vertices (run_weighted_lds).  Larger graphs by
// near-far relaxation in memory: vertices whose distance dropped are relaxed next if
// it is below a threshold (near), else set aside (far); when no near vertex
// is left the threshold moves past the smallest far distance by delta and
// the far pile is split.  Relaxing in distance order re-relaxes far fewer
// edges than plain frontier relaxation (CPU count on the 4.1M-edge ER graph
// of the uneven workload: 5.7 -> 1.2 relaxations per edge); atomicMin
// relaxations in place in the output row.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "common.hpp"

namespace dawn {

// Device memory by type: through a plain pointer that was itself read from
// memory the compiler emits flat loads, which also wait for the LDS.
typedef const int32_t __attribute__((address_space(1)))* GlobalInts;

struct BatchGraph {
  int32_t n;
  int32_t weighted;
  int64_t m;
  GlobalInts row_ptr;
  GlobalInts col;
  GlobalInts w;
  GlobalInts in_row_ptr;  // in-edges (the CSR for undirected graphs)
  GlobalInts in_col;
  int64_t dist_off;  // first output row of this graph
  int32_t max_deg;   // largest out-degree
  int32_t pad;
};

struct BatchTask {
  int32_t graph;
  int32_t lane0;   // first source index within the graph's block
  int32_t lanes;   // sources in this task (1 for weighted)
  int32_t bits;    // unweighted: log2 of the bits per vertex in LDS, -1: state in memory
};

struct BatchArgs {
  const BatchGraph* graphs;
  const BatchTask* tasks;
  int32_t num_tasks;
  int32_t spg;               // sources per graph
  const int32_t* sources;    // num_graphs * spg (already reduced mod n)
  int32_t* dist;
  unsigned* task_counter;
  unsigned long long* levels_total;
  int32_t* graph_levels;     // per unweighted graph: levels of its longest task
  const unsigned long long* wsum;  // per graph: sum of edge weights (weighted)
  // Per-workgroup scratch, sized for the largest graph (max_n).
  int64_t max_n;
  uint64_t* seen;      // [grid][max_n]
  uint64_t* next;      // [grid][max_n]
  int32_t* qv;         // [grid][2][max_n]
  uint64_t* qw;        // [grid][2][max_n]
  int32_t* touched;    // [grid][max_n]
  uint8_t* stage;      // [grid][stage_cap]: arrival levels that are not in LDS
  int64_t stage_cap;
  int32_t* lds_q;      // [grid][max_lds_n]: vertex queue of the LDS tasks
  int2* entries;       // [grid][max_lds_n]: expanded queue entries of the LDS tasks
  int64_t max_lds_n;
};

namespace {

// Threads per workgroup of the persistent kernels.  A task (one graph's
// traversal) runs inside one workgroup, and the LDS that holds its state is a
// CU's whole, so one workgroup is resident per CU and its own waves are all
// that hides a step's latency: as many as a workgroup can have, 16, four per
// SIMD, which leaves each thread 128 registers.
constexpr int kBatchBlock = 1024;

template <int BS>
__device__ __forceinline__ int owner(const int* off, int e) {
  int lo = 0, hi = BS - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= e) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The owners of 4 x 64 consecutive edges from e0 on (wave-uniform), edge
// e0 + 64 r + lane in o[r]; past the end the last edge, e[r].  First the
// owners of the range's two ends, a ballot over BS/64 segments and one inside,
// then each lane searches between those: 4 probes at a mean degree of 16
// instead of 10, and without branches, so that the four searches interleave
// and the loads that follow are all in flight (one weighted source of RMAT-17:
// relaxations 5.1 ms -> 3.2 ms).
template <int BS>
__device__ __forceinline__ int wave_owner(const int* off, int e) {
  constexpr int S = BS / kWave;
  const int seg = __popcll(__ballot(off[lane_id() * S] <= e)) - 1;
  const uint64_t in = __ballot(off[seg * S + lane_id() % S] <= e);
  return seg * S + __popcll(in & ((1ull << S) - 1)) - 1;
}
template <int BS>
__device__ __forceinline__ void owners4(const int* off, int e0, int edges, int (&e)[4], int (&o)[4]) {
  const int lo = __builtin_amdgcn_readfirstlane(wave_owner<BS>(off, e0));
  const int hi = __builtin_amdgcn_readfirstlane(wave_owner<BS>(off, min(e0 + 4 * kWave, edges) - 1));
#pragma unroll
  for (int r = 0; r < 4; r++) {
    e[r] = min(e0 + r * kWave + lane_id(), edges - 1);
    o[r] = lo;
  }
  for (int step = hi > lo ? 1 << (31 - __clz(hi - lo)) : 0; step; step >>= 1) {
    int to[4], at[4];
#pragma unroll
    for (int r = 0; r < 4; r++) to[r] = min(o[r] + step, hi);
#pragma unroll
    for (int r = 0; r < 4; r++) at[r] = off[to[r]];
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = at[r] <= e[r] ? to[r] : o[r];
  }
}

// Exclusive scan of one int per thread over a BS-thread workgroup.
// scratch: BS/kWave ints of LDS; *total receives the sum.
template <int BS>
__device__ __forceinline__ int scan_bs(int x, int* scratch, int* total) {
  const int l = lane_id();
  const int w = threadIdx.x / kWave;
  int inc = x;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    int y = __shfl_up(inc, o);
    if (l >= o) inc += y;
  }
  if (l == kWave - 1) scratch[w] = inc;
  __syncthreads();
  int base = 0, sum = 0;
#pragma unroll
  for (int i = 0; i < BS / kWave; i++) {
    const int s = scratch[i];
    if (i < w) base += s;
    sum += s;
  }
  __syncthreads();
  *total = sum;
  return base + inc - x;
}

// Appends through an LDS counter (one workgroup owns the list).
__device__ __forceinline__ int lds_append(unsigned* s_count, bool pred) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return -1;
  const int leader = __ffsll((unsigned long long)m) - 1;
  unsigned base = 0;
  if (lane_id() == leader) base = atomicAdd(s_count, (unsigned)__popcll(m));
  base = __shfl(base, leader);
  return pred ? (int)(base + (unsigned)__popcll(m & lanes_below_mask())) : -1;
}

// Stage entry of a level that does not fit 16 bits (written to its row).
constexpr uint16_t kStaged = 0xFFFF;
constexpr int32_t kStageLanes = 8;  // tasks with their state in memory: lanes that stage their levels

// atomicOr on a lane word of type LT; sub-word types go through the
// aligned 32-bit word that holds them.  Returns the old value of *p.
template <typename LT>
__device__ __forceinline__ LT atomic_or_lanes(LT* p, LT v) {
  if constexpr (sizeof(LT) == 8) {
    return (LT)atomicOr((unsigned long long*)p, (unsigned long long)v);
  } else if constexpr (sizeof(LT) == 4) {
    return (LT)atomicOr((unsigned*)p, (unsigned)v);
  } else {
    const uintptr_t ad = (uintptr_t)p;
    const int sh = (int)(ad & 3) * 8;
    const unsigned old = atomicOr((unsigned*)(ad & ~(uintptr_t)3), (unsigned)v << sh);
    return (LT)(old >> sh);
  }
}

// LT: the narrowest unsigned type holding the task's lanes (8 sources per
// graph: one byte per vertex).  The per-vertex state (seen, next, queue
// words) is probed and OR-ed at random per scanned edge, so its footprint
// decides how much of it the caches hold: at 8 bytes per vertex the
// workgroups' state spilled out of L2 and the Infinity Cache, and the
// kernel moved about 100 GB for 512 graphs of 14 M vertices.
template <int BS, typename LT>
__device__ void run_unweighted(const BatchArgs& a, const BatchGraph& G, const BatchTask& T,
                               LT* seen, LT* next, int32_t* qv, LT* qw,
                               int32_t* touched, int* s_off, int* s_beg, uint64_t* s_f,
                               int* s_scan, unsigned* s_cnt) {
  const int32_t n = G.n;
  const int64_t mn = a.max_n;
  // Lane b of the task is source lane0 + b of the graph: row drow + b * n.
  int32_t* drow = a.dist + G.dist_off + (int64_t)T.lane0 * n;
  const LT lanemask = (LT)(T.lanes >= 64 ? ~0ull : ((1ull << T.lanes) - 1));
  // Tasks of at most kStageLanes lanes stage each arrival level in stage[v][b]
  // (16 bits; kStaged marks a level that did not fit, written to its row at
  // once) and write the rows in one coalesced pass at the end, instead of
  // 4-byte stores scattered over the rows as vertices are reached.
  constexpr bool kStage = sizeof(LT) == 1;
  static_assert(!kStage || kStageLanes == 8, "a byte of lanes");
  uint16_t* stage = reinterpret_cast<uint16_t*>(a.stage + (int64_t)blockIdx.x * a.stage_cap);
  for (int32_t v = threadIdx.x; v < n; v += blockDim.x) {
    seen[v] = (LT)~lanemask;
    next[v] = 0;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s_cnt[0] = 0;  // |Q_0|
    for (int i = 0; i < T.lanes; i++) {
      const int32_t s = a.sources[(int64_t)T.graph * a.spg + T.lane0 + i];
      const LT bit = (LT)(1ull << i);
      if ((seen[s] & lanemask) == 0) {
        qv[s_cnt[0]] = s;
        qw[s_cnt[0]] = 0;
        s_cnt[0]++;
      }
      seen[s] |= bit;
      if constexpr (kStage) stage[(int64_t)s * 8 + i] = 0;
      else drow[(int64_t)i * n + s] = 0;
    }
    // Words of the level-0 entries.
    for (unsigned j = 0; j < s_cnt[0]; j++) qw[j] = seen[qv[j]] & lanemask;
  }
  __syncthreads();
  unsigned qn = s_cnt[0];
  int par = 0;
  int level = 0;
  while (qn > 0) {
    const int32_t* qv_in = qv + (int64_t)par * mn;
    const LT* qw_in = qw + (int64_t)par * mn;
    int32_t* qv_out = qv + (int64_t)(par ^ 1) * mn;
    LT* qw_out = qw + (int64_t)(par ^ 1) * mn;
    if (threadIdx.x == 0) s_cnt[1] = 0;  // |touched|
    __syncthreads();
    // Expand Q_level with workgroup edge balancing (LDS degree scan).
    for (unsigned c0 = 0; c0 < qn; c0 += BS) {
      const unsigned i = c0 + threadIdx.x;
      int beg = 0, deg = 0;
      uint64_t f = 0;
      if (i < qn) {
        const int32_t u = qv_in[i];
        beg = G.row_ptr[u];
        deg = G.row_ptr[u + 1] - beg;
        f = qw_in[i];
      }
      int total;
      const int off = scan_bs<BS>(deg, s_scan, &total);
      s_off[threadIdx.x] = off;
      s_beg[threadIdx.x] = beg;
      s_f[threadIdx.x] = f;
      __syncthreads();
      for (int e0 = 0; e0 < total; e0 += BS) {
        const int e = e0 + threadIdx.x;
        bool first = false;
        int32_t w = 0;
        if (e < total) {
          const int j = owner<BS>(s_off, e);
          w = G.col[s_beg[j] + (e - s_off[j])];
          const LT nv = (LT)(s_f[j] & ~(uint64_t)seen[w]);
          if (nv) first = atomic_or_lanes<LT>(&next[w], nv) == 0;
        }
        const int slot = lds_append(&s_cnt[1], first);
        if (first) touched[slot] = w;
      }
      __syncthreads();
    }
    // Commit the touched vertices into Q_{level+1} and the distance rows.
    if (threadIdx.x == 0) s_cnt[2] = 0;
    __syncthreads();
    const unsigned tn = s_cnt[1];
    const int32_t lv = level + 1;
    for (unsigned t0 = 0; t0 < tn; t0 += BS) {
      const unsigned t = t0 + threadIdx.x;
      bool isf = false;
      int32_t w = 0;
      LT nw = 0;
      if (t < tn) {
        w = touched[t];
        const LT nx = next[w];
        next[w] = 0;
        nw = (LT)(nx & ~seen[w]);
        if (nw) {
          seen[w] = (LT)(seen[w] | nw);
          isf = true;
          uint64_t bits = (uint64_t)nw;
          while (bits) {
            const int b = __ffsll((unsigned long long)bits) - 1;
            bits &= bits - 1;
            if constexpr (kStage) {
              if (lv < (int32_t)kStaged) {
                stage[(int64_t)w * 8 + b] = (uint16_t)lv;
                continue;
              }
              stage[(int64_t)w * 8 + b] = kStaged;
            }
            drow[(int64_t)b * n + w] = lv;
          }
        }
      }
      const int slot = lds_append(&s_cnt[2], isf);
      if (isf) {
        qv_out[slot] = w;
        qw_out[slot] = nw;
      }
    }
    __syncthreads();
    qn = s_cnt[2];
    par ^= 1;
    level = lv;
    __syncthreads();
  }
  // Rows: staged levels, INF for lanes that never arrived (one thread per
  // vertex, so each row store of a wave covers 64 consecutive vertices).
  for (int32_t v = threadIdx.x; v < n; v += blockDim.x) {
    const uint64_t got = (uint64_t)(LT)(seen[v] & lanemask);
    if constexpr (kStage) {
      const uint4 q = *reinterpret_cast<const uint4*>(stage + (int64_t)v * 8);
      const uint32_t hw[4] = {q.x, q.y, q.z, q.w};
      for (int b = 0; b < T.lanes; b++) {
        const uint32_t l = (hw[b >> 1] >> (16 * (b & 1))) & 0xFFFFu;
        if (!((got >> b) & 1)) drow[(int64_t)b * n + v] = kInf;
        else if (l != kStaged) drow[(int64_t)b * n + v] = (int32_t)l;
      }
    } else {
      uint64_t miss = (uint64_t)(LT)(~seen[v] & lanemask);
      while (miss) {
        const int b = __ffsll((unsigned long long)miss) - 1;
        miss &= miss - 1;
        drow[(int64_t)b * n + v] = kInf;
      }
    }
  }
  if (threadIdx.x == 0) {
    atomicAdd(a.levels_total, (unsigned long long)level);
    atomicMax(&a.graph_levels[T.graph], level);
  }
}

// ---- unweighted tasks with their state in LDS -----------------------------
//
// A graph's traversal probes and updates its per-vertex lane words at random
// per scanned edge; in memory each probe moved a line (512 graphs, 8 sources:
// 41 GB, 18.7 ms).  Here a vertex has a field in a workgroup's LDS: for L > 1
// lanes (1 << bits) 2L bits, A (lanes that have reached it) in the low half
// and B (lanes that arrive at the level being found) in the high half, so that
// one LDS atomic marks an arrival in both; for one lane A alone, as its queue
// entries need no B.  Per level:
//   gather  the queue's vertices give their B bits, offsets and degrees to
//           the entry list; B is cleared
//   pull    of the lanes whose frontier holds more than 1 / kPullShare of the
//           graph's edges, if there are more edges than a push takes in one
//           round (counting them per lane costs more than that round): every
//           vertex that misses one of them ORs its in-neighbours' A bits until
//           it has found them all (a lane that an in-neighbour has and the
//           vertex lacks arrived there one level ago, or the vertex would have
//           it); they enter A afterwards.  Without that bound 1500 grids of 150
//           vertices, 16 sources each, took 2.2 times as long, 1500 random graphs
//           of 150 vertices and degree 16 1.4 times
//   push    of the other lanes: short lists by a thread per entry, else the
//           entries' edges spread over the threads (LDS degree scan), four
//           edges in flight per thread: bits new in A arrive; the first
//           arrival at a vertex in the level appends it to the queue
// Arrival levels are staged in a byte per vertex and lane, in LDS where they
// fit beside the fields (in memory, the scattered bytes of 256 workgroups are
// most of the batch's traffic), and written as rows at the end.
constexpr int kLdsWords = 37800;  // 151,200 bytes
constexpr int kMaxBits = 4;       // up to 16 lanes per task
constexpr int kPullShare = 8;
constexpr int kSerialDeg = 12;    // largest out-degree of graphs whose lists threads walk alone
constexpr uint32_t kStaged8 = 0xFFu;  // stage entry of a level that does not fit (in its row)

// Lanes per vertex (log2) of a task of `lanes` sources on n vertices whose
// fields fit the LDS, or -1.  A task's entries hold degree and lanes in 32
// bits, so graphs with a larger degree than 65535 take one lane.
inline int64_t lds_field_words(int64_t n, int bits) { return (n * (bits ? 2 << bits : 1) + 31) / 32; }
inline int lds_bits(int64_t n, int lanes, int32_t max_deg) {
  int b = 0;
  while ((1 << b) < lanes) b++;
  return b <= kMaxBits && (b == 0 || max_deg < 65536) && lds_field_words(n, b) <= kLdsWords ? b : -1;
}

// Bytes of arrival levels that a task of `lanes` sources keeps in memory
// (BatchArgs::stage); bits as in BatchTask.
inline int64_t stage_bytes(int64_t n, int lanes, int bits) {
  if (bits < 0) return lanes <= kStageLanes ? n * kStageLanes * (int64_t)sizeof(uint16_t) : 0;
  const bool in_lds = lds_field_words(n, bits) * 4 + (n << bits) <= (int64_t)kLdsWords * 4;
  return in_lds ? 0 : n << bits;
}

struct LdsTask {
  alignas(16) uint32_t W[kLdsWords];
  unsigned lane_edges[1 << kMaxBits];
};

// Four columns of an edge list, read by one load at any 4-byte offset.
struct __attribute__((packed, aligned(4))) Cols4 {
  int32_t c[4];
};
// The columns at p, of which r + 1 >= 1 are there (the last one repeated).
__device__ __forceinline__ Cols4 cols_at(GlobalInts p, int r) {
  if (r >= 3) return *(const Cols4*)(const int32_t*)p;
  return Cols4{{p[0], p[min(1, r)], p[r], p[r]}};
}

// p[i .. i + 3] by a 32-bit offset from a base in scalar registers.
__device__ __forceinline__ Cols4 four_at(GlobalInts p, uint32_t i) {
  return *(const Cols4*)((const char*)(const int32_t*)p + i * 4u);
}

// sources, lanes, bits: of the task.  gstage: levels that do not fit the LDS.
// levels(v, b) afterwards: kInf, or the level, by any thread.
template <int BS, typename Out>
__device__ int run_lds(const BatchGraph& G, const int32_t* sources, int32_t lanes, int bits, int32_t* drow,
                       uint8_t* gstage, LdsTask& s, int32_t* qv, int2* ent, int* s_off, int* s_beg,
                       uint32_t* s_f, int* s_scan, unsigned* s_cnt, uint32_t* s_red, Out out) {
  const int32_t n = G.n;
  const int t = threadIdx.x;
  const bool one = bits == 0;
  const int L = 1 << bits, fw = one ? 0 : bits + 1, fpw = 5 - fw;  // log2 field width, fields per word
  const uint32_t fmask = (1u << L) - 1u;
  uint32_t bmask = 0;  // the B halves of a word
  if (!one)
    for (int k = 0; k < 32; k += 2 * L) bmask |= fmask << (k + L);
  const int words = (int)((((int64_t)n << fw) + 31) >> 5);
  uint8_t* lstage = reinterpret_cast<uint8_t*>(s.W + words);
  const bool in_lds = (int64_t)words * 4 + (int64_t)n * L <= (int64_t)kLdsWords * 4;
  auto word_of = [&](int32_t v) { return v >> fpw; };
  auto shift_of = [&](int32_t v) { return (v & ((1 << fpw) - 1)) << fw; };
  auto mark = [&](uint32_t nv) { return one ? nv : nv | nv << L; };
  auto put_level = [&](int32_t v, uint32_t bits, int32_t lv) {
    for (; bits; bits &= bits - 1) {
      const int b = __ffs(bits) - 1;
      const uint8_t x = (uint8_t)min((uint32_t)lv, kStaged8);
      const int64_t at = (int64_t)v * L + b;
      if (in_lds) lstage[at] = x;
      else gstage[at] = x;
      if (x == kStaged8) drow[(int64_t)b * n + v] = lv;
    }
  };
  for (int i = t; i < words; i += BS) s.W[i] = 0u;
  if (t == 0) s_cnt[0] = 0u;
  __syncthreads();
  if (t < lanes) {
    const int32_t v = sources[t];
    const uint32_t bit = 1u << t;
    const uint32_t old = atomicOr(&s.W[word_of(v)], mark(bit) << shift_of(v)) >> shift_of(v);
    put_level(v, bit, 0);
    if (!(old & fmask)) qv[atomicAdd(&s_cnt[0], 1u)] = v;
  }
  __syncthreads();
  int level = 0;
  for (;; level++) {
    const unsigned qn = s_cnt[0];
    if (qn == 0) break;
    const int32_t lv = level + 1;
    // Gather: entries of the frontier, its edges, its live lanes.
    if (t == 0) {
      s_red[0] = 0u;
      s_cnt[1] = 0u;
    }
    __syncthreads();
    unsigned fe = 0;  // at most m < 2^31
    uint32_t live = 0;
    // B is cleared at the queue's vertices, or in all words if those are fewer:
    // levels of a few vertices leave the words alone.  A thread's first entry
    // stays in a register.
    const bool few = qn <= (unsigned)words;
    int2 mine = make_int2(0, 0);
    for (unsigned i = t; i < qn; i += BS) {
      const int32_t v = qv[i];
      uint32_t f = 1u;
      if (!one) {
        uint32_t* w = &s.W[word_of(v)];
        const int at = shift_of(v) + L;
        f = ((few ? atomicAnd(w, ~(fmask << at)) : *w) >> at) & fmask;
      }
      const int rb = G.row_ptr[v], d = G.row_ptr[v + 1] - rb;
      const int2 e2 = make_int2(rb, one ? d : d | (int)(f << 16));
      if (i < (unsigned)BS) mine = e2;
      else ent[i] = e2;
      fe += (unsigned)d;
      live |= f;
    }
    for (int o = 32; o >= 1; o >>= 1) {
      fe += (unsigned)__shfl_xor((int)fe, o);
      live |= (uint32_t)__shfl_xor((int)live, o);
    }
    if (lane_id() == 0) {
      if (fe) atomicAdd(&s_cnt[1], fe);
      if (live) atomicOr(&s_red[0], live);
    }
    __syncthreads();
    live = s_red[0];
    auto entry = [&](unsigned i) { return i < (unsigned)BS ? mine : ent[i]; };  // of this thread
    uint32_t pull = 0;  // lanes to pull
    if (s_cnt[1] > 4u * BS && (unsigned long long)s_cnt[1] * kPullShare > (unsigned long long)G.m) {
      // The frontier's edges lane by lane: the lanes with many are pulled
      // (a lane with few would make every vertex scan its whole list).
      if (one) {
        pull = 1u;
      } else {
        if (t < 1 << kMaxBits) s.lane_edges[t] = 0u;
        __syncthreads();
        for (int b0 = 0; b0 < lanes; b0 += 4) {
          unsigned c[4] = {0, 0, 0, 0};
          for (unsigned i = t; i < qn; i += BS) {
            const unsigned df = (unsigned)entry(i).y;
#pragma unroll
            for (int b = 0; b < 4; b++) c[b] += (df >> (16 + b0 + b)) & 1u ? df & 0xFFFFu : 0u;
          }
#pragma unroll
          for (int b = 0; b < 4; b++) {
            for (int o = 32; o >= 1; o >>= 1) c[b] += (unsigned)__shfl_xor((int)c[b], o);
            if (lane_id() == 0 && c[b] && b0 + b < lanes) atomicAdd(&s.lane_edges[b0 + b], c[b]);
          }
        }
        __syncthreads();
        for (int b = 0; b < lanes; b++)
          if ((unsigned long long)s.lane_edges[b] * kPullShare > (unsigned long long)G.m) pull |= 1u << b;
      }
    }
    if (!one && !few)
      for (int i = t; i < words; i += BS) s.W[i] &= ~bmask;
    if (t == 0) s_cnt[0] = 0u;
    __syncthreads();
    if (pull) {
      // Four vertices a thread: their offsets, then the first four edges of
      // each, are in flight together (one at a time, a chain of three reads
      // from memory each: 65 sources of 65,536 vertices and 0.5 M edges 375 us,
      // 331 with four); what that leaves goes on vertex by vertex.
      constexpr int V = 4;
      auto field = [&](int32_t u) { return s.W[word_of(u)] >> shift_of(u); };
      const bool by_four = G.m >= V && G.m < kSourcesMaxM;
      for (int32_t v0 = 0; v0 < n; v0 += V * BS) {
        uint32_t miss[V], got[V];
        int beg[V], deg[V];
#pragma unroll
        for (int r = 0; r < V; r++) {
          const int32_t v = v0 + r * BS + t;
          miss[r] = v < n ? pull & ~(s.W[word_of(v)] >> shift_of(v)) : 0u;
          got[r] = 0u;
        }
        if (!__ballot((miss[0] | miss[1] | miss[2] | miss[3]) != 0)) continue;
#pragma unroll
        for (int r = 0; r < V; r++) {
          const int32_t v = miss[r] ? v0 + r * BS + t : 0;
          beg[r] = G.in_row_ptr[v];
          deg[r] = G.in_row_ptr[v + 1];
        }
#pragma unroll
        for (int r = 0; r < V; r++) deg[r] = miss[r] ? deg[r] - beg[r] : 0;
        int done = 0;  // edges looked at
        if (by_four) {
          Cols4 u[V];
          int k0[V];
#pragma unroll
          for (int r = 0; r < V; r++) {
            k0[r] = min(deg[r] > 0 ? beg[r] : 0, (int)G.m - V);
            u[r] = four_at(G.in_col, (uint32_t)k0[r]);
          }
#pragma unroll
          for (int r = 0; r < V; r++)
#pragma unroll
            for (int c = 0; c < 4; c++)
              got[r] |= k0[r] + c >= beg[r] && k0[r] + c < beg[r] + deg[r] ? field(u[r].c[c]) : 0u;
          done = 4;
        }
#pragma unroll
        for (int r = 0; r < V; r++) {
          const int lim = deg[r] < 64 ? deg[r] : 16;
          for (int j = done; j < lim && (got[r] & miss[r]) != miss[r]; j += 4) {
            const Cols4 u = cols_at(G.in_col + beg[r] + j, deg[r] - 1 - j);
            got[r] |= field(u.c[0]) | field(u.c[1]) | field(u.c[2]) | field(u.c[3]);
          }
          // The rest of long lists by the whole wave, four edges per lane.
          uint64_t hm = __ballot(deg[r] >= 64 && (got[r] & miss[r]) != miss[r]);
          while (hm) {
            const int l = __ffsll((unsigned long long)hm) - 1;
            hm &= hm - 1;
            const int hb = __shfl(beg[r], l), he = hb + __shfl(deg[r], l);
            const uint32_t want = (uint32_t)__shfl((int)miss[r], l);
            uint32_t g = (uint32_t)__shfl((int)got[r], l);
            for (int k0 = hb + 16; k0 < he && (g & want) != want; k0 += 4 * kWave) {
              const int k = k0 + 4 * lane_id();
              uint32_t x = 0;
              if (k < he) {
                const Cols4 u = cols_at(G.in_col + k, he - 1 - k);
                x = field(u.c[0]) | field(u.c[1]) | field(u.c[2]) | field(u.c[3]);
              }
              for (int o = 32; o >= 1; o >>= 1) x |= (uint32_t)__shfl_xor((int)x, o);
              g |= x;
            }
            if (lane_id() == l) got[r] = g;
          }
        }
#pragma unroll
        for (int r = 0; r < V; r++) {
          const int32_t v = v0 + r * BS + t;
          got[r] &= miss[r];
          if (got[r]) {
            if (!one) atomicOr(&s.W[word_of(v)], got[r] << (shift_of(v) + L));
            put_level(v, got[r], lv);
          }
          const int slot = lds_append(&s_cnt[0], got[r] != 0);
          if (got[r]) qv[slot] = v;
        }
      }
      __syncthreads();
      if (one) {
        const unsigned found = s_cnt[0];
        for (unsigned i = t; i < found; i += BS) atomicOr(&s.W[word_of(qv[i])], 1u << shift_of(qv[i]));
      } else {
        for (int i = t; i < words; i += BS) s.W[i] |= (s.W[i] & bmask) >> L;
      }
      __syncthreads();
      if (!(live & ~pull)) continue;
    }
    // Push the lanes that were not pulled (their bits are disjoint from the
    // pulled lanes').  Four heads at a time: their words, the atomics on those
    // that lack a lane, then one reservation of queue slots for the wave.
    auto visit = [&](const int32_t (&w)[4], const uint32_t (&f)[4]) {
      uint32_t nv[4], old[4];
      bool first[4];
#pragma unroll
      for (int r = 0; r < 4; r++)
        nv[r] = __hip_atomic_load(&s.W[word_of(w[r])], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
      for (int r = 0; r < 4; r++) nv[r] = f[r] & ~(nv[r] >> shift_of(w[r]));
#pragma unroll
      for (int r = 0; r < 4; r++)
        old[r] = nv[r] ? atomicOr(&s.W[word_of(w[r])], mark(nv[r]) << shift_of(w[r])) >> shift_of(w[r])
                       : 0u;
      uint64_t m[4];
      unsigned cnt = 0;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        nv[r] &= ~old[r];
        first[r] = nv[r] != 0 && (one || ((old[r] >> L) & fmask) == 0);
        m[r] = __ballot(first[r]);
        cnt += (unsigned)__popcll(m[r]);
      }
      if (!__ballot((nv[0] | nv[1] | nv[2] | nv[3]) != 0)) return;
      unsigned at = 0;
      if (cnt && lane_id() == 0) at = atomicAdd(&s_cnt[0], cnt);
#pragma unroll
      for (int r = 0; r < 4; r++) put_level(w[r], nv[r], lv);
      at = __shfl(at, 0);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (first[r]) qv[at + (unsigned)__popcll(m[r] & lanes_below_mask())] = w[r];
        at += (unsigned)__popcll(m[r]);
      }
    };
    if (G.max_deg <= kSerialDeg) {
      // Short lists: a thread walks its own entry's, four columns per load.
      for (unsigned c0 = t & ~(kWave - 1); c0 < qn; c0 += BS) {  // wave-uniform
        const unsigned i = c0 + lane_id();
        int2 e2 = make_int2(0, 0);
        if (i < qn) e2 = entry(i);
        const uint32_t f = (one ? 1u : (uint32_t)e2.y >> 16) & ~pull;
        const int d = !f ? 0 : one ? e2.y : e2.y & 0xFFFF;
        const int most = wave_max_i32(d);
        for (int j = 0; j < most; j += 4) {
          Cols4 u{{0, 0, 0, 0}};
          if (j < d) u = cols_at(G.col + e2.x + j, d - 1 - j);
          const uint32_t fr[4] = {j < d ? f : 0u, j + 1 < d ? f : 0u, j + 2 < d ? f : 0u,
                                  j + 3 < d ? f : 0u};
          visit(u.c, fr);
        }
      }
      __syncthreads();
      continue;
    }
    for (unsigned c0 = 0; c0 < qn; c0 += BS) {
      const unsigned i = c0 + t;
      int2 e2 = make_int2(0, 0);
      if (i < qn) e2 = entry(i);
      const uint32_t f0 = (one ? 1u : (uint32_t)e2.y >> 16) & ~pull;
      int total;
      const int off = scan_bs<BS>(!f0 ? 0 : one ? e2.y : e2.y & 0xFFFF, s_scan, &total);
      s_off[t] = off;
      s_beg[t] = e2.x - off;
      s_f[t] = f0;
      __syncthreads();
      for (int e0 = __builtin_amdgcn_readfirstlane(t / kWave) * 4 * kWave; e0 < total; e0 += 4 * BS) {
        int e[4], o[4];
        int32_t w[4];
        uint32_t f[4];
        owners4<BS>(s_off, e0, total, e, o);
#pragma unroll
        for (int r = 0; r < 4; r++) w[r] = G.col[s_beg[o[r]] + e[r]];
#pragma unroll
        for (int r = 0; r < 4; r++) f[r] = s_f[o[r]];
#pragma unroll
        for (int r = 0; r < 4; r++) f[r] = e0 + r * kWave + lane_id() < total ? f[r] : 0u;
        visit(w, f);
      }
      __syncthreads();
    }
  }
  out([&](int32_t v, int b) -> int32_t {
    if (!((s.W[word_of(v)] >> (shift_of(v) + b)) & 1u)) return kInf;
    const int64_t at = (int64_t)v * L + b;
    const uint32_t l = in_lds ? lstage[at] : gstage[at];
    return l == kStaged8 ? drow[(int64_t)b * n + v] : (int32_t)l;
  });
  return level;
}

template <int BS>
__device__ void lds_task(const BatchArgs& a, const BatchGraph& G, const BatchTask& T, LdsTask& s,
                         int32_t* qv, int2* ent, int* s_off, int* s_beg, uint32_t* s_f, int* s_scan,
                         unsigned* s_cnt, uint32_t* s_red) {
  const int32_t n = G.n;
  int32_t* drow = a.dist + G.dist_off + (int64_t)T.lane0 * n;
  // Rows: a row store of a wave covers 64 consecutive vertices.
  const int levels = run_lds<BS>(
      G, a.sources + (int64_t)T.graph * a.spg + T.lane0, T.lanes, T.bits, drow,
      a.stage + (int64_t)blockIdx.x * a.stage_cap, s, qv, ent, s_off, s_beg, s_f, s_scan, s_cnt, s_red,
      [&](auto level_of) {
        for (int32_t v = threadIdx.x; v < n; v += BS)
          for (int b = 0; b < T.lanes; b++) drow[(int64_t)b * n + v] = level_of(v, b);
      });
  if (threadIdx.x == 0) {
    atomicAdd(a.levels_total, (unsigned long long)levels);
    atomicMax(&a.graph_levels[T.graph], levels);
  }
}

// One weighted source.  The reference's initialisation
// (src/algorithm/cpu/sssp.cpp:40-46): listed out-edges of the source write
// their weight in row order, the distinct neighbours form the first
// frontier, distance[source] = 0, the source is never relaxed.  Then
// near-far relaxation to the same fixed point.  flags[v], one byte: kNear
// (v is in the near queue, cleared when v is taken out to be relaxed) and
// kFar (v is in the far pile).  A byte per vertex instead of two 32-bit
// words keeps more of the task's randomly probed state in the caches; a
// relaxation clears kNear and then reads dist[u] at the L2, so an
// improvement that found kNear still set is relaxed with its new value.
constexpr unsigned kNear = 1u, kFar = 2u;

__device__ __forceinline__ unsigned flags_or(uint8_t* f, unsigned bits) {
  const uintptr_t ad = (uintptr_t)f;
  const int sh = (int)(ad & 3) * 8;
  return (atomicOr((unsigned*)(ad & ~(uintptr_t)3), bits << sh) >> sh) & 0xFFu;
}
__device__ __forceinline__ void flags_clear(uint8_t* f, unsigned bits) {
  const uintptr_t ad = (uintptr_t)f;
  const int sh = (int)(ad & 3) * 8;
  atomicAnd((unsigned*)(ad & ~(uintptr_t)3), ~(bits << sh));
}

template <int BS>
__device__ void run_weighted(const BatchArgs& a, const BatchGraph& G, const BatchTask& T,
                             uint8_t* flags, int32_t* qv, int32_t* far,
                             int* s_off, int* s_beg, int* s_du, int* s_scan, unsigned* s_cnt,
                             int* s_red) {
  const int32_t n = G.n;
  const int64_t mn = a.max_n;
  const int32_t src = a.sources[(int64_t)T.graph * a.spg + T.lane0];
  int32_t* dist = a.dist + G.dist_off + (int64_t)T.lane0 * n;
  // delta: twice the mean edge weight over the mean degree (on the uneven
  // workload's weighted graphs, scales 1-8 measured within 10%, 2 best).
  const double avg_w = G.m > 0 ? (double)a.wsum[T.graph] / (double)G.m : 1.0;
  const double avg_deg = n > 0 ? (double)G.m / (double)n : 1.0;
  const long long delta = (long long)fmax(1.0, 2.0 * avg_w / fmax(avg_deg, 1.0));
  for (int32_t v = threadIdx.x; v < n; v += blockDim.x) {
    dist[v] = kInf;
    flags[v] = 0;
  }
  __syncthreads();
  // s_cnt: [0] near queue length, [1] next near length, [3] far length,
  // [4] next far length.
  if (threadIdx.x == 0) {
    const int32_t b = G.row_ptr[src], e = G.row_ptr[src + 1];
    for (int32_t k = b; k < e; k++) dist[G.col[k]] = G.w[k];
    dist[src] = 0;
    int32_t dmin = kInf;
    for (int32_t k = b; k < e; k++)
      if (G.col[k] != src) dmin = min(dmin, dist[G.col[k]]);
    const long long thr = (long long)dmin + delta;
    unsigned c = 0, f = 0;
    for (int32_t k = b; k < e; k++) {
      const int32_t v = G.col[k];
      if (v == src || flags[v]) continue;
      if (dist[v] < thr) {
        flags[v] = (uint8_t)kNear;
        qv[c++] = v;
      } else {
        flags[v] = (uint8_t)kFar;
        far[f++] = v;
      }
    }
    s_cnt[0] = c;
    s_cnt[3] = f;
    s_red[1] = (int)min(thr, (long long)kInf);
  }
  __syncthreads();
  unsigned qn = s_cnt[0];
  long long thr = s_red[1];
  int par = 0, fpar = 0;
  uint32_t steps = 0;
  for (;;) {
    while (qn > 0) {
      const int32_t* q_in = qv + (int64_t)par * mn;
      int32_t* q_out = qv + (int64_t)(par ^ 1) * mn;
      int32_t* f_out = far + (int64_t)fpar * mn;
      steps++;
      if (threadIdx.x == 0) s_cnt[1] = 0;
      __syncthreads();
      for (unsigned c0 = 0; c0 < qn; c0 += BS) {
        const unsigned i = c0 + threadIdx.x;
        int beg = 0, deg = 0, du = 0;
        if (i < qn) {
          const int32_t u = q_in[i];
          beg = G.row_ptr[u];
          deg = G.row_ptr[u + 1] - beg;
          flags_clear(flags + u, kNear);
          du = __hip_atomic_load(dist + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        int total;
        const int off = scan_bs<BS>(deg, s_scan, &total);
        s_off[threadIdx.x] = off;
        s_beg[threadIdx.x] = beg;
        s_du[threadIdx.x] = du;
        __syncthreads();
        for (int e0 = 0; e0 < total; e0 += BS) {
          const int e = e0 + threadIdx.x;
          bool add_near = false, add_far = false;
          int32_t v = 0;
          if (e < total) {
            const int j = owner<BS>(s_off, e);
            const int k = s_beg[j] + (e - s_off[j]);
            v = G.col[k];
            // The weight and the head's distance in flight together: opaque to
            // the compiler, which in the kernel with tasks of every kind read
            // one after the other (a source of RMAT-18: 41.6 ms, 38.8 so).
            int32_t wk = G.w[k], dv = dist[v];
            asm volatile("" : "+v"(wk), "+v"(dv));
            const int32_t nd = minplus(s_du[j], wk);
            if (v != src && nd < dv) {
              const int32_t old = atomicMin(&dist[v], nd);
              if (nd < old) {
                if ((long long)nd < thr) add_near = !(flags_or(flags + v, kNear) & kNear);
                else add_far = !(flags_or(flags + v, kFar) & kFar);
              }
            }
          }
          const int slot = lds_append(&s_cnt[1], add_near);
          if (add_near) q_out[slot] = v;
          const int fslot = lds_append(&s_cnt[3], add_far);
          if (add_far) f_out[fslot] = v;
        }
        __syncthreads();
      }
      qn = s_cnt[1];
      par ^= 1;
      __syncthreads();
    }
    const unsigned fn = s_cnt[3];
    if (fn == 0) break;
    // No near vertex left: the threshold moves past the smallest far
    // distance, and the far pile splits into near and the next far pile.
    // An entry whose distance dropped below the old threshold was relaxed
    // as a near vertex already and leaves the pile.
    const int32_t* f_in = far + (int64_t)fpar * mn;
    int32_t* f_next = far + (int64_t)(fpar ^ 1) * mn;
    int32_t* q_out = qv + (int64_t)par * mn;
    int32_t lmin = kInf;
    for (unsigned i = threadIdx.x; i < fn; i += BS) {
      const int32_t d = dist[f_in[i]];
      if ((long long)d >= thr) lmin = min(lmin, d);
    }
    lmin = min(lmin, __shfl_xor(lmin, 32));
    for (int o = 16; o >= 1; o >>= 1) lmin = min(lmin, __shfl_xor(lmin, o));
    if (threadIdx.x == 0) s_red[0] = kInf;
    __syncthreads();
    if (lane_id() == 0) atomicMin(&s_red[0], lmin);
    __syncthreads();
    const long long old_thr = thr;
    const int32_t fmin = s_red[0];
    thr = fmin == kInf ? old_thr : (long long)fmin + delta;
    if (threadIdx.x == 0) {
      s_cnt[1] = 0;
      s_cnt[4] = 0;
    }
    __syncthreads();
    for (unsigned c0 = 0; c0 < fn; c0 += BS) {
      const unsigned i = c0 + threadIdx.x;
      bool to_near = false, keep = false;
      int32_t v = 0;
      if (i < fn) {
        v = f_in[i];
        const long long d = dist[v];
        if (d < old_thr) {
          flags_clear(flags + v, kFar);  // relaxed as a near vertex already
        } else if (d < thr) {
          flags_clear(flags + v, kFar);
          to_near = !(flags_or(flags + v, kNear) & kNear);
        } else {
          keep = true;
        }
      }
      const int slot = lds_append(&s_cnt[1], to_near);
      if (to_near) q_out[slot] = v;
      const int kslot = lds_append(&s_cnt[4], keep);
      if (keep) f_next[kslot] = v;
    }
    __syncthreads();
    qn = s_cnt[1];
    if (threadIdx.x == 0) s_cnt[3] = s_cnt[4];
    fpar ^= 1;
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(a.levels_total, (unsigned long long)steps);
}

// ---- weighted tasks with LDS state ----------------------------------------
//
// Label-correcting relaxation to the same fixed point, with everything that
// is probed at random per edge in LDS and no queues: what is to be expanded is
// marked at the vertex, and every step scans the marks.
//
// Graphs of up to kDistN vertices keep the distances there (DL): a word
// 2 d + mark, all ones for a vertex not reached.  An improvement is one
// unsigned minimum with 2 nd + 1: it sets the mark, and an equal distance
// changes nothing.  Larger graphs keep the distances in the output row and in
// LDS a mark bit and a byte, d <= base + byte * 2^qs, 255 for none known: an
// edge whose path is no shorter than that bound cannot improve the vertex and
// touches no memory.  Bytes are stored without an atomic: of two improvements
// the larger may stay, which only makes the bound looser and the vertex later.
// When the bytes to come leave the lower half of the range, base moves up to
// the smallest and all are rewritten (rebase).
//
// Graphs without hubs move the threshold by delta after every step (rolling:
// few steps, 1.0-1.8 relaxations per edge); graphs with hubs exhaust what is
// below it first (1.3 to 1.7 per edge where rolling takes 3.4).  delta, in mean
// weights over the mean degree: 2 where the distances are in LDS and a step
// costs about what its relaxations do (1: grids of up to 37,000 vertices 26%
// slower, RMAT 13%); 1 (hubs: 1/2) where a relaxation may go to memory (2:
// random graphs 33% slower, grids 7%, RMAT-17 13%).
//
// Measured, 512 graphs of 1,000 to 130,000 vertices, 8 sources each (1.7 G
// edges to relax once): 45.0 ms with queues, marks and distances in memory and
// one edge per thread in flight.  What bounds it now is the instructions of a
// relaxation (RMAT-17, one CU: 2 G relaxations/s of 60 VALU and 15 LDS
// operations per wave and edge) and, for small graphs, the step's scan (3 us).
constexpr int64_t kDistN = kSourcesDistN;  // words, rounded up to four
static_assert(kDistN + 3 <= kLdsWords, "distances");
constexpr int64_t kBoundN = kSourcesN;     // a byte and a bit per vertex
constexpr int64_t kSerialM = 4;            // edges of one load
constexpr int64_t kLdsM = kSourcesMaxM;    // edges reached by 32-bit byte offsets
static_assert((kBoundN + 3) / 4 + (kBoundN + 31) / 32 <= kLdsWords, "bounds and marks");
enum { kWeightedMemory = -1, kWeightedDist = 0, kWeightedBound = 1 };  // BatchTask::bits

// p[i] by a 32-bit offset from a base in scalar registers.
__device__ __forceinline__ int32_t at32(GlobalInts p, uint32_t i) {
  return *(GlobalInts)((const char __attribute__((address_space(1)))*)p + i * 4u);
}

// Of two distances, kInf for none, in 32 bits (both are >= 0).
__device__ __forceinline__ int32_t plus_sat(int32_t a, int32_t b) {
  return (int32_t)min((uint32_t)a + (uint32_t)b, (uint32_t)kInf);
}

// One source.  dist: its row (DL: not touched, the words are left in s.W).
// Returns the steps taken.
template <int BS, bool DL>
__device__ uint32_t run_weighted_lds(const BatchGraph& G, int32_t src, unsigned long long wsum,
                                     int32_t* dist, LdsTask& s, int* s_off, int* s_beg, int* s_du,
                                     int* s_scan, int* s_red) {
  // Vertices per thread: quads at a stride of BS quads, or words of 32 in order.
  constexpr int kQuads = (int)((kDistN + 4 * BS - 1) / (4 * BS));
  constexpr int kWords = (int)(((kBoundN + 31) / 32 + BS - 1) / BS);
  static_assert(kQuads * 4 <= 64, "a bit each");
  const int32_t n = G.n;
  const int t = threadIdx.x;
  uint32_t* word = s.W;                               // DL
  uint8_t* key = reinterpret_cast<uint8_t*>(s.W);     // otherwise
  const int nb = (n + 31) / 32, n4 = (n + 3) / 4;
  uint32_t* pend = s.W + n4;
  const double avg_w = G.m > 0 ? (double)wsum / (double)G.m : 1.0;
  const double avg_deg = n > 0 ? (double)G.m / (double)n : 1.0;
  const bool roll = G.max_deg <= 16 * avg_deg;
  const double delta = fmax(1.0, ceil((DL ? 2.0 : roll ? 1.0 : 0.5) * avg_w / fmax(avg_deg, 1.0)));
  int qs = 0;  // two or three units to a delta
  while (!DL && qs < 22 && (double)(2ll << qs) < delta * (2.0 / 3)) qs++;
  const long long step_k = DL ? (long long)delta : (long long)ceil(delta / (double)(1 << qs));
  uint32_t base = 0;
  auto get = [&](int32_t v) {
    return __hip_atomic_load((int32_t*)((char*)dist + (uint32_t)v * 4u), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  };
  auto put = [&](int32_t v, int32_t d) {
    __hip_atomic_store(dist + v, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto key_of = [&](int32_t v) {
    return (uint32_t)__hip_atomic_load(key + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto units = [&](int32_t d) {  // smallest k >= 0 with d <= base + k * 2^qs, at most 255
    return (uint32_t)d <= base ? 0u : min(((uint32_t)d - base + (1u << qs) - 1u) >> qs, 255u);
  };
  auto improved = [&](int32_t v, int32_t d) {
    __hip_atomic_store(key + v, (uint8_t)units(d), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    atomicOr(&pend[v >> 5], 1u << (v & 31));
  };
  for (int32_t v = t; v < (DL ? n4 * 4 : n); v += BS) {
    if (DL) word[v] = ~0u;
    else dist[v] = kInf, key[v] = 255;
  }
  if (!DL)
    for (int i = t; i < nb; i += BS) pend[i] = 0u;
  __syncthreads();
  // Reference initialisation (sssp.cpp:40-46), all edges at once: a
  // neighbour's slot first takes a tag of its last listed edge, then that edge
  // alone replaces it by its weight.  Tags are even (DL: the words of marked
  // vertices are odd) or negative (weights are >= 0).
  const int32_t sb = G.row_ptr[src], se = G.row_ptr[src + 1];
  for (int32_t k = sb + t; k < se; k += BS) {
    if (DL) atomicMin(&word[G.col[k]], (uint32_t)(kInf - k) * 2u);
    else atomicMin(&dist[G.col[k]], -1 - k);
  }
  __syncthreads();
  for (int32_t k = sb + t; k < se; k += BS) {
    const int32_t v = G.col[k], w = G.w[k];
    if (DL) {
      if (word[v] == (uint32_t)(kInf - k) * 2u) word[v] = (uint32_t)w * 2u + 1u;
    } else if (get(v) == -1 - k) {
      put(v, w);
      if (v != src && w != kInf) improved(v, w);
    }
  }
  __syncthreads();
  if (t == 0) {
    if (DL) word[src] = 0u;
    else put(src, 0), key[src] = 0;
  }
  // Four relaxations in flight: the keys, atomics on those that may improve.
  auto relax = [&](const int32_t (&v)[4], const int32_t (&nd)[4]) {
    if (DL) {
#pragma unroll
      for (int r = 0; r < 4; r++)
        atomicMin(&word[v[r]], (uint32_t)nd[r] * 2u + 1u);
      return;
    }
    bool may[4];
    uint32_t k[4];
    int32_t old[4];
#pragma unroll
    for (int r = 0; r < 4; r++) k[r] = key_of(v[r]);
#pragma unroll
    for (int r = 0; r < 4; r++)
      may[r] = (uint32_t)nd[r] < (k[r] == 255u ? (uint32_t)kInf : base + (k[r] << qs));
#pragma unroll
    for (int r = 0; r < 4; r++)
      old[r] = may[r] ? atomicMin((int32_t*)((char*)dist + (uint32_t)v[r] * 4u), nd[r]) : -1;
    // Opaque to the compiler, which else moves each comparison, and with it
    // the wait for its atomic, up before the next atomic.
#pragma unroll
    for (int r = 0; r < 4; r++) asm volatile("" : "+v"(old[r]));
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (nd[r] < old[r]) improved(v[r], nd[r]);
  };
  long long thr = -1;  // set by the first pass, which selects nothing
  uint32_t steps = 0;
  for (;;) {
    if (t == 0) s_red[0] = kInf;
    __syncthreads();
    // What is to be expanded with a key of at most thr, and the smallest key
    // of the rest.
    uint64_t quads = 0;
    uint32_t sel[kWords];
    int count = 0;
    int32_t least = kInf;
    if (DL) {
      const uint32_t lim = thr < 0 ? 0u : (uint32_t)min(thr, (long long)kInf - 1) * 2u + 1u;
      uint32_t lm = ~0u;
#pragma unroll
      for (int r = 0; r < kQuads; r++) {
        const int q = r * BS + t;
        if (q < n4) {
          const uint4 x = reinterpret_cast<const uint4*>(word)[q];
          const uint32_t y[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const bool marked = y[c] & 1u, in = marked && y[c] <= lim;
            quads |= (uint64_t)in << (r * 4 + c);
            if (marked && !in) lm = min(lm, y[c]);
          }
        }
      }
      count = __popcll(quads);
      least = (int32_t)(lm >> 1);  // all ones (not reached): kInf
    } else {
#pragma unroll
      for (int r = 0; r < kWords; r++) {
        const int i = t * kWords + r;
        uint32_t x = i < nb ? pend[i] : 0u;
        sel[r] = 0u;
        while (x) {
          const int b = __ffs(x) - 1;
          x &= x - 1;
          const int32_t k = (int32_t)key_of(i * 32 + b);
          if ((long long)k <= thr) sel[r] |= 1u << b;
          else least = min(least, k);
        }
        count += __popc(sel[r]);
      }
    }
    least = wave_min_i32(least);
    if (lane_id() == 0 && least != kInf) atomicMin(&s_red[0], least);
    int total;
    int pos = scan_bs<BS>(count, s_scan, &total);
    if (total == 0) {
      const int32_t fm = s_red[0];  // scan_bs has synchronised
      __syncthreads();
      if (fm == kInf) break;
      if (!DL && fm > 127) {
        // Rebase.  Unknown bytes are set from the distances; where only such
        // are to come, base moves to the smallest of their distances.
        uint32_t shift = (uint32_t)(fm - 1);
        if (fm == 255) {
          int32_t dm = kInf;
          for (int i = t; i < nb; i += BS)
            for (uint32_t x = pend[i]; x; x &= x - 1) dm = min(dm, get(i * 32 + __ffs(x) - 1));
          dm = wave_min_i32(dm);
          if (t == 0) s_red[0] = kInf;
          __syncthreads();
          if (lane_id() == 0) atomicMin(&s_red[0], dm);
          __syncthreads();
          dm = s_red[0];
          shift = (uint32_t)dm <= base ? 0u : ((uint32_t)dm - base) >> qs;
        }
        base += shift << qs;
        for (int32_t v = t; v < n; v += BS) {
          const uint32_t k = key[v];
          if (k != 255u) {
            key[v] = (uint8_t)(k > shift ? k - shift : 0u);
          } else {
            const int32_t d = get(v);
            if (d != kInf) key[v] = (uint8_t)units(d);
          }
        }
        thr = -1;
        __syncthreads();
      } else {
        thr = (long long)fm + step_k;
      }
      continue;
    }
    steps++;
    for (int w0 = 0; w0 < total; w0 += BS) {
      // The next BS of them, off the marks before their distances are read:
      // a later improvement marks them again.  No other thread is at this
      // thread's marks here.
      if (DL) {
        for (; quads && pos < w0 + BS; quads &= quads - 1, pos++) {
          const int b = __ffsll((unsigned long long)quads) - 1;
          const int32_t v = ((b >> 2) * BS + t) * 4 + (b & 3);
          s_beg[pos - w0] = v;
          s_du[pos - w0] = (int32_t)(word[v] >> 1);
          word[v] &= ~1u;
        }
      } else {
#pragma unroll
        for (int r = 0; r < kWords; r++) {
          const uint32_t before = sel[r];
          for (; sel[r] && pos < w0 + BS; sel[r] &= sel[r] - 1, pos++)
            s_beg[pos - w0] = (t * kWords + r) * 32 + __ffs(sel[r]) - 1;
          if (before != sel[r]) pend[t * kWords + r] &= ~(before ^ sel[r]);
        }
      }
      __syncthreads();
      int beg = 0, deg = 0, du = 0;
      if (w0 + t < total) {
        const int32_t u = s_beg[t];
        beg = at32(G.row_ptr, (uint32_t)u);
        deg = at32(G.row_ptr, (uint32_t)u + 1u) - beg;
        du = DL ? s_du[t] : get(u);
      }
      if (G.max_deg <= kSerialDeg && G.m >= kSerialM) {
        // A thread per vertex, four edges by one load; what the load holds of
        // other rows is relaxed at no distance.
        const int most = wave_max_i32(deg), end = beg + deg;
        for (int j = 0; j < most; j += 4) {
          const int k0 = min(j < deg ? beg + j : 0, (int)G.m - 4);  // kSerialM <= m < kLdsM
          const Cols4 u = four_at(G.col, k0), w = four_at(G.w, k0);
          int32_t v[4], nd[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            v[r] = u.c[r];
            nd[r] = plus_sat(k0 + r >= beg + j && k0 + r < end ? du : kInf, w.c[r]);
          }
          relax(v, nd);
        }
      } else {
        int edges;
        const int off = scan_bs<BS>(deg, s_scan, &edges);
        s_off[t] = off;
        s_beg[t] = beg - off;
        if (!DL) s_du[t] = du;
        __syncthreads();
        for (int e0 = __builtin_amdgcn_readfirstlane(t / kWave) * 4 * kWave; e0 < edges; e0 += 4 * BS) {
          int e[4], o[4], k[4], du[4];
          int32_t v[4], nd[4];
          owners4<BS>(s_off, e0, edges, e, o);
#pragma unroll
          for (int r = 0; r < 4; r++) k[r] = s_beg[o[r]] + e[r], du[r] = s_du[o[r]];
#pragma unroll
          for (int r = 0; r < 4; r++) du[r] = e0 + r * kWave + lane_id() < edges ? du[r] : kInf;
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] = at32(G.col, k[r]), nd[r] = at32(G.w, k[r]);
#pragma unroll
          for (int r = 0; r < 4; r++) nd[r] = plus_sat(du[r], nd[r]);
          relax(v, nd);
        }
      }
      __syncthreads();
    }
    if (roll) thr = DL || thr <= 191 ? thr + step_k : -1;  // -1: towards a rebase
  }
  return steps;
}

template <int BS, bool DL>
__device__ void weighted_task(const BatchArgs& a, const BatchGraph& G, const BatchTask& T, LdsTask& s,
                              int* s_off, int* s_beg, int* s_du, int* s_scan, int* s_red) {
  int32_t* dist = a.dist + G.dist_off + (int64_t)T.lane0 * G.n;
  const uint32_t steps =
      run_weighted_lds<BS, DL>(G, a.sources[(int64_t)T.graph * a.spg + T.lane0], a.wsum[T.graph], dist, s,
                               s_off, s_beg, s_du, s_scan, s_red);
  if (DL)
    for (int32_t v = threadIdx.x; v < G.n; v += BS) dist[v] = (int32_t)(s.W[v] >> 1);
  if (threadIdx.x == 0) atomicAdd(a.levels_total, (unsigned long long)steps);
}

// Sum of the edge weights of each weighted graph (the near-far delta):
// kWsumParts workgroups per graph, one atomic each.
constexpr int kWsumParts = 4;
__global__ void __launch_bounds__(kBlock) wsum_kernel(const BatchGraph* graphs,
                                                      unsigned long long* out) {
  __shared__ unsigned long long s_t;
  const BatchGraph G = graphs[blockIdx.x / kWsumParts];
  const int part = blockIdx.x % kWsumParts;
  if (threadIdx.x == 0) s_t = 0ull;
  __syncthreads();
  unsigned long long t = 0;
  if (G.weighted)
    for (int64_t k = (int64_t)part * kBlock + threadIdx.x; k < G.m; k += (int64_t)kWsumParts * kBlock)
      t += (unsigned)G.w[k];
  t = wave_sum_u64(t);
  if (lane_id() == 0 && t) atomicAdd(&s_t, t);
  __syncthreads();
  if (threadIdx.x == 0 && s_t) atomicAdd(&out[blockIdx.x / kWsumParts], s_t);
}

// KIND: the tasks of the batch are all unweighted (0), all weighted (1), mixed
// (2) or all unweighted with their state in memory (3); with one kind alone the
// compiler keeps the registers the others would take (mixed: 105 scalar and 14
// vector spills).
template <int BS, int KIND>
__global__ void __launch_bounds__(BS) batch_kernel(BatchArgs a) {
  __shared__ int s_off[BS];
  __shared__ int s_beg[BS];
  __shared__ uint32_t s_lf[BS];
  __shared__ int s_scan[BS / kWave];
  __shared__ unsigned s_cnt[5];
  __shared__ int s_red[2];
  __shared__ int s_task;
  __shared__ uint32_t s_or[1];
  __shared__ LdsTask s_lds;
  // The tasks with their state in memory use the LDS for what is left of theirs.
  uint64_t* s_f = reinterpret_cast<uint64_t*>(s_lds.W);
  const int64_t mn = a.max_n;
  uint64_t* seen = a.seen + (int64_t)blockIdx.x * mn;
  uint64_t* next = a.next + (int64_t)blockIdx.x * mn;
  int32_t* qv = a.qv + (int64_t)blockIdx.x * 2 * mn;
  uint64_t* qw = a.qw + (int64_t)blockIdx.x * 2 * mn;
  int32_t* touched = a.touched + (int64_t)blockIdx.x * mn;
  for (;;) {
    if (threadIdx.x == 0) s_task = (int)atomicAdd(a.task_counter, 1u);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_task);  // uniform: T and G in scalar registers
    __syncthreads();
    if (t >= a.num_tasks) break;  // every workgroup leaves once the queue is empty
    const BatchTask T = a.tasks[t];
    const BatchGraph G = a.graphs[T.graph];
    if (KIND == 1 || (KIND == 2 && G.weighted)) {
      if (T.bits == kWeightedDist)
        weighted_task<BS, true>(a, G, T, s_lds, s_off, s_beg, (int*)s_lf, s_scan, s_red);
      else if (T.bits == kWeightedBound)
        weighted_task<BS, false>(a, G, T, s_lds, s_off, s_beg, (int*)s_lf, s_scan, s_red);
      else
        run_weighted<BS>(a, G, T, (uint8_t*)next, qv, (int32_t*)qw, s_off, s_beg,
                         (int*)s_f, s_scan, s_cnt, s_red);
    } else {
      if (KIND != 3 && T.bits >= 0)
        lds_task<BS>(a, G, T, s_lds, a.lds_q + (int64_t)blockIdx.x * a.max_lds_n,
                    a.entries + (int64_t)blockIdx.x * a.max_lds_n, s_off, s_beg, s_lf, s_scan, s_cnt, s_or);
      else if (T.lanes <= kStageLanes)
        run_unweighted<BS, uint8_t>(a, G, T, (uint8_t*)seen, (uint8_t*)next, qv, (uint8_t*)qw,
                                    touched, s_off, s_beg, s_f, s_scan, s_cnt);
      else if (T.lanes <= 16)
        run_unweighted<BS, uint16_t>(a, G, T, (uint16_t*)seen, (uint16_t*)next, qv, (uint16_t*)qw,
                                     touched, s_off, s_beg, s_f, s_scan, s_cnt);
      else if (T.lanes <= 32)
        run_unweighted<BS, uint32_t>(a, G, T, (uint32_t*)seen, (uint32_t*)next, qv, (uint32_t*)qw,
                                     touched, s_off, s_beg, s_f, s_scan, s_cnt);
      else
        run_unweighted<BS, uint64_t>(a, G, T, seen, next, qv, qw, touched, s_off, s_beg, s_f,
                                     s_scan, s_cnt);
    }
    __syncthreads();
  }
}

// Many sources of one weighted graph, a workgroup each at a time.
struct SourcesArgs {
  BatchGraph G;
  const int32_t* sources;
  int32_t count;
  int32_t* rows;            // [count][n], or null
  int32_t* scratch;         // without rows and with more than kDistN vertices: [grid][n]
  unsigned* counter;
  unsigned long long* acc;  // per source: distance sum, vertices reached, their out-degrees, steps
  const unsigned long long* wsum;
};

template <int BS, bool DL>
__global__ void __launch_bounds__(BS) sources_kernel(SourcesArgs a) {
  __shared__ int s_off[BS];
  __shared__ int s_beg[BS];
  __shared__ int s_du[BS];
  __shared__ int s_scan[BS / kWave];
  __shared__ int s_red[1];
  __shared__ int s_next;
  __shared__ unsigned long long s_acc[3];
  __shared__ LdsTask s_lds;
  const int t = threadIdx.x;
  const int32_t n = a.G.n;
  for (;;) {
    if (t == 0) s_next = (int)atomicAdd(a.counter, 1u);
    if (t < 3) s_acc[t] = 0ull;
    __syncthreads();
    const int i = __builtin_amdgcn_readfirstlane(s_next);
    __syncthreads();
    if (i >= a.count) break;  // every workgroup leaves once the sources are taken
    int32_t* row = a.rows ? a.rows + (int64_t)i * n : DL ? nullptr : a.scratch + (int64_t)blockIdx.x * n;
    const uint32_t steps = run_weighted_lds<BS, DL>(a.G, a.sources[i], *a.wsum, row, s_lds, s_off, s_beg,
                                                    s_du, s_scan, s_red);
    unsigned long long sum = 0, edges = 0;
    unsigned reached = 0;
    for (int32_t v = t; v < n; v += BS) {
      const int32_t d = DL ? (int32_t)(s_lds.W[v] >> 1)
                           : __hip_atomic_load(row + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (DL && row) row[v] = d;
      if (d != kInf) {
        sum += (unsigned)d;
        reached++;
        edges += (unsigned)(a.G.row_ptr[v + 1] - a.G.row_ptr[v]);
      }
    }
    sum = wave_sum_u64(sum);
    edges = wave_sum_u64(edges);
    const unsigned long long many = wave_sum_u64(reached);
    if (lane_id() == 0) {
      atomicAdd(&s_acc[0], sum);
      atomicAdd(&s_acc[1], many);
      atomicAdd(&s_acc[2], edges);
    }
    __syncthreads();
    if (t < 4) a.acc[(int64_t)i * 4 + t] = t < 3 ? s_acc[t] : steps;
    __syncthreads();
  }
}

// The same unweighted: levels in LDS (n <= kSourcesN), one lane.
static_assert((kSourcesN + 31) / 32 * 4 + kSourcesN <= (int64_t)kLdsWords * 4, "a bit and a level each");
struct BfsSourcesArgs {
  BatchGraph G;
  const int32_t* sources;
  int32_t count;
  int32_t* rows;            // [count][n], or null
  int32_t* scratch;         // without rows: [grid][n], for levels beyond a byte
  int32_t write;            // rows are written: to `rows`, else each over the last in `scratch`
  int32_t* qv;              // [grid][n]
  int2* ent;                // [grid][n]
  unsigned* counter;
  unsigned long long* acc;  // as above, levels for steps
};

template <int BS>
__global__ void __launch_bounds__(BS) bfs_sources_kernel(BfsSourcesArgs a) {
  __shared__ int s_off[BS];
  __shared__ int s_beg[BS];
  __shared__ uint32_t s_lf[BS];
  __shared__ int s_scan[BS / kWave];
  __shared__ unsigned s_cnt[5];
  __shared__ uint32_t s_or[1];
  __shared__ int s_next;
  __shared__ unsigned long long s_acc[3];
  __shared__ LdsTask s_lds;
  const int t = threadIdx.x;
  const int32_t n = a.G.n;
  for (;;) {
    if (t == 0) s_next = (int)atomicAdd(a.counter, 1u);
    if (t < 3) s_acc[t] = 0ull;
    __syncthreads();
    const int i = __builtin_amdgcn_readfirstlane(s_next);
    __syncthreads();
    if (i >= a.count) break;  // every workgroup leaves once the sources are taken
    int32_t* row = a.rows ? a.rows + (int64_t)i * n : a.scratch + (int64_t)blockIdx.x * n;
    const int levels = run_lds<BS>(
        a.G, a.sources + i, 1, 0, row, nullptr, s_lds, a.qv + (int64_t)blockIdx.x * n,
        a.ent + (int64_t)blockIdx.x * n, s_off, s_beg, s_lf, s_scan, s_cnt, s_or, [&](auto level_of) {
          unsigned long long sum = 0;
          unsigned reached = 0, edges = 0;  // m < 2^31
          for (int32_t v = t; v < n; v += BS) {
            const int32_t d = level_of(v, 0);
            if (a.write) row[v] = d;
            if (d != kInf) {
              sum += (unsigned)d;
              reached++;
              edges += (unsigned)(a.G.row_ptr[v + 1] - a.G.row_ptr[v]);
            }
          }
          sum = wave_sum_u64(sum);
          const unsigned long long many = wave_sum_u64((unsigned long long)reached);
          const unsigned long long es = wave_sum_u64((unsigned long long)edges);
          if (lane_id() == 0) {
            atomicAdd(&s_acc[0], sum);
            atomicAdd(&s_acc[1], many);
            atomicAdd(&s_acc[2], es);
          }
        });
    __syncthreads();
    if (t < 4) a.acc[(int64_t)i * 4 + t] = t < 3 ? s_acc[t] : (unsigned long long)levels;
    __syncthreads();
  }
}

}  // namespace

constexpr int32_t kSourcesLaunch = 1 << 16;  // sources of one launch

// Sources (reduced mod n) a workgroup each, for graphs whose state fits its
// LDS; the engines of lanes say when.  compute_rows: unweighted rows are
// computed without an output too (dawn_mssp).  acc: per source the distance sum, the
// vertices reached, their out-degrees, the steps (levels); device time in *ms.
int run_sources_lds(dawn_graph* g, SourcesWorkspace* ws, const int32_t* sources, int32_t S, int32_t* dist,
                    bool compute_rows, std::vector<unsigned long long>& acc, double* ms) {
  if (g->n > kSourcesN || g->m >= kSourcesMaxM) return DAWN_ERR_UNSUPPORTED;
  const bool dl = g->n <= kDistN;
  // Rows go to the caller's device memory itself; with bounds in LDS the
  // distances are lowered there, in plain memory of the device only.
  const bool direct = g->weighted && !dl ? in_place(g->device, dist) : is_device_pointer(dist);
  int cus = 0;
  DAWN_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
  hipStream_t s = g->stream;
  // Other rows are copied, in blocks of a workgroup per CU.
  const int32_t per = std::min<int32_t>(S, dist && !direct ? cus : kSourcesLaunch);
  const int grid = std::max(1, std::min<int>(per, cus));
  const size_t gn = (size_t)grid * g->n;
  const BatchGraph G{g->n, g->weighted, g->m, (GlobalInts)g->row_ptr, (GlobalInts)g->col,
                     (GlobalInts)g->weight, (GlobalInts)g->in_row_ptr, (GlobalInts)g->in_col, 0,
                     g->max_out_degree, 0};
  DAWN_TRY(ws->counter.alloc(1));
  DAWN_TRY(ws->sources.alloc((size_t)per));
  DAWN_TRY(ws->acc.alloc((size_t)per * 4));
  if (dist && !direct) DAWN_TRY(ws->rows.alloc((size_t)per * g->n));
  else if (!dist && !(g->weighted && dl)) DAWN_TRY(ws->rows.alloc(gn));
  for (hipEvent_t* e : {&ws->ev0, &ws->ev1})
    if (!*e) DAWN_HIP(hipEventCreate(e));
  if (!g->weighted) {
    DAWN_TRY(ws->queue.alloc(gn));
    DAWN_TRY(ws->entries.alloc(gn));
  } else if (!ws->wsum.p) {
    DAWN_TRY(ws->graph.alloc(sizeof(BatchGraph)));
    DAWN_TRY(ws->wsum.alloc(1));
    DAWN_HIP(hipMemcpyAsync(ws->graph.p, &G, sizeof(BatchGraph), hipMemcpyHostToDevice, s));
    DAWN_HIP(hipMemsetAsync(ws->wsum.p, 0, sizeof(unsigned long long), s));
    wsum_kernel<<<kWsumParts, kBlock, 0, s>>>((const BatchGraph*)ws->graph.p, ws->wsum.p);
    DAWN_HIP(hipGetLastError());
  }
  acc.resize((size_t)S * 4);
  *ms = 0;
  for (int32_t b0 = 0; b0 < S; b0 += per) {
    const int32_t count = std::min(per, S - b0);
    int32_t* rows = !dist ? nullptr : direct ? dist + (int64_t)b0 * g->n : ws->rows.p;
    DAWN_HIP(hipMemcpyAsync(ws->sources.p, sources + b0, sizeof(int32_t) * (size_t)count,
                            hipMemcpyHostToDevice, s));
    DAWN_HIP(hipEventRecord(ws->ev0, s));
    DAWN_HIP(hipMemsetAsync(ws->counter.p, 0, sizeof(unsigned), s));
    if (g->weighted) {
      const SourcesArgs a{G, ws->sources.p, count, rows, ws->rows.p, ws->counter.p, ws->acc.p, ws->wsum.p};
      if (dl) sources_kernel<kBatchBlock, true><<<grid, kBatchBlock, 0, s>>>(a);
      else sources_kernel<kBatchBlock, false><<<grid, kBatchBlock, 0, s>>>(a);
    } else {
      const BfsSourcesArgs a{G, ws->sources.p, count, rows, ws->rows.p, dist || compute_rows,
                             ws->queue.p, ws->entries.p, ws->counter.p, ws->acc.p};
      bfs_sources_kernel<kBatchBlock><<<grid, kBatchBlock, 0, s>>>(a);
    }
    DAWN_HIP(hipGetLastError());
    DAWN_HIP(hipEventRecord(ws->ev1, s));
    DAWN_HIP(hipMemcpyAsync(acc.data() + (size_t)b0 * 4, ws->acc.p,
                            sizeof(unsigned long long) * 4 * (size_t)count, hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    if (dist && !direct) {
      DAWN_HIP(hipMemcpy(dist + (int64_t)b0 * g->n, ws->rows.p, sizeof(int32_t) * (size_t)count * g->n,
                         hipMemcpyDefault));
      DAWN_HIP(hipStreamSynchronize(nullptr));  // rows that are no host memory
    }
    float x = 0.f;
    DAWN_HIP(hipEventElapsedTime(&x, ws->ev0, ws->ev1));
    *ms += x;
  }
  return DAWN_OK;
}

namespace {

// Unweighted tasks of the uneven batch.  The sources of a graph share one task
// as lanes of a field, except on the largest graphs, whose tasks would be the
// batch's critical path, and where fewer lanes keep the fields and staged
// levels in LDS (kSpan*: lanes x vertices; graphs with hubs pull most of their
// edges once for all lanes and take more, deep ones pay for their levels in
// every task).  512 graphs of 1k-130k vertices, 8 sources: one task per graph
// 4.6 ms, at most 65,536 lanes x vertices 3.6, at most 116,000 with the levels
// in LDS 2.6.
constexpr int64_t kSpanFlat = 116000, kSpan = 262144;
constexpr int32_t kHubDeg = 1024;
constexpr int64_t kSplit2 = 500000, kSplit1 = 2000000;

// Graphs of many levels of few edges each: as batches have found it, before
// that those of hardly more edges than vertices (paths, trees, road maps).  A
// level takes a task 3-4 us whatever its lanes, so their tasks take as many
// lanes as fit: 300 trees of 20,000 vertices and some 1000 levels, 16 sources,
// take 22 ms as four tasks of 4 lanes, 10 as one of 16.  Grids of 20,000
// vertices have 285 edges a level and are not among them (four tasks 4.9 ms,
// one in memory 13.1).
bool deep(const dawn_graph* g) {
  const int64_t levels = g->batch_levels.load(std::memory_order_relaxed);
  return levels ? g->m < 128 * levels : g->m * 5 <= 13 * (int64_t)g->n;
}

// Lanes per task with its state in LDS, 0: it does not fit.
int32_t lds_lanes(const dawn_graph* g, int32_t spg) {
  int32_t per = std::min(spg, 1 << kMaxBits);
  if (g->m >= kSplit1) per = 1;
  else if (g->m >= kSplit2) per = std::max(1, spg / 2);
  const int64_t span = deep(g) || g->max_out_degree > kHubDeg ? kSpan : kSpanFlat;
  while (per > 1 && (lds_bits(g->n, per, g->max_out_degree) < 0 || g->n * (int64_t)per > span))
    per = (per + 1) / 2;
  return lds_bits(g->n, per, g->max_out_degree) < 0 ? 0 : per;
}

// Whether `k` tasks of a graph in LDS take longer than one of up to 64 lanes in
// memory, where tasks wait for a CU anyway.  Measured on 1500 graphs, LDS over
// memory: four tasks, random graphs of degree 4 with 2000, 6000 and 8000 edges
// 1.5, 1.09 and 0.93, paths of 150 and 1000 vertices 2.4 and 2.6; two tasks,
// random graphs with 600, 2000 and 3000 edges 1.3, 1.06 and 0.98.
bool memory_faster(const dawn_graph* g, int32_t k) {
  return k > 1 && (deep(g) || g->m <= (k > 2 ? 8000 : 2500));
}

}  // namespace

void sources_workspace_free(SourcesWorkspace* ws) {
  if (!ws) return;
  for (hipEvent_t e : {ws->ev0, ws->ev1})
    if (e) (void)hipEventDestroy(e);
  delete ws;
}

}  // namespace dawn

using namespace dawn;

extern "C" int dawn_batch_mssp(dawn_graph* const* graphs, int32_t num_graphs,
                               const int32_t* sources, int32_t spg, int32_t* dist,
                               const int64_t* dist_offsets, dawn_stats* stats) {
  if (!graphs || num_graphs <= 0 || !sources || spg <= 0 || spg > 64 || !dist_offsets)
    return DAWN_ERR_INVALID_ARG;
  const int device = graphs[0]->device;
  int64_t total = 0;
  // Largest graphs of the tasks that keep state in memory, and in LDS.
  int64_t max_n = 0, max_lds_n = 0, stage_cap = 0;
  std::vector<BatchGraph> hg(num_graphs);
  std::vector<BatchTask> ht;
  std::vector<int32_t> hs((size_t)num_graphs * spg);
  int cus = 0;
  DAWN_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  int64_t tasks = 0;  // with their state in LDS where it fits
  for (int32_t i = 0; i < num_graphs; i++) {
    const dawn_graph* g = graphs[i];
    if (!g || g->device != device || g->n <= 0) return DAWN_ERR_INVALID_ARG;
    const int32_t per = g->weighted ? 1 : lds_lanes(g, spg);
    tasks += per ? (spg + per - 1) / per : 1;
  }
  const bool queued = tasks > cus;
  for (int32_t i = 0; i < num_graphs; i++) {
    const dawn_graph* g = graphs[i];
    hg[i] = BatchGraph{g->n, g->weighted, g->m, (GlobalInts)g->row_ptr, (GlobalInts)g->col,
                       (GlobalInts)g->weight, (GlobalInts)g->in_row_ptr, (GlobalInts)g->in_col,
                       dist_offsets[i], g->max_out_degree, 0};
    total = std::max<int64_t>(total, dist_offsets[i] + (int64_t)spg * g->n);
    for (int32_t j = 0; j < spg; j++) {
      int64_t s = sources[(int64_t)i * spg + j] % (int64_t)g->n;
      if (s < 0) s += g->n;
      hs[(size_t)i * spg + j] = (int32_t)s;
      if (stats && g->h_row_ptr[s] == g->h_row_ptr[s + 1]) stats->skipped_sources += 1;
    }
    if (g->weighted) {
      const int state = g->m >= kLdsM || g->n > kBoundN ? kWeightedMemory
                        : g->n <= kDistN                ? kWeightedDist
                                                        : kWeightedBound;
      for (int32_t j = 0; j < spg; j++) ht.push_back(BatchTask{i, j, 1, state});
      if (state == kWeightedMemory) max_n = std::max<int64_t>(max_n, g->n);
    } else {
      int32_t per = lds_lanes(g, spg);
      const bool memory = per == 0 || (queued && memory_faster(g, (spg + per - 1) / per));
      if (memory) {  // lanes as wide as 64
        per = g->m >= kSplit1 ? 1 : g->m >= kSplit2 ? std::max(1, spg / 2) : spg;
        max_n = std::max<int64_t>(max_n, g->n);
      } else {
        max_lds_n = std::max<int64_t>(max_lds_n, g->n);
      }
      for (int32_t j = 0; j < spg; j += per) {
        const int32_t lanes = std::min(per, spg - j);
        const int bits = memory ? -1 : lds_bits(g->n, lanes, g->max_out_degree);
        stage_cap = std::max(stage_cap, stage_bytes(g->n, lanes, bits));  // a last task may have fewer lanes
        ht.push_back(BatchTask{i, j, lanes, bits});
      }
    }
  }
  // The long tasks start early: graphs of short lists take many levels (a
  // grid of 131,000 vertices 2.8 ms), the others go by their edges.
  auto cost = [&](const BatchTask& x) {
    const BatchGraph& g = hg[x.graph];
    return (g.weighted ? 0 : (g.max_deg <= kSerialDeg ? 5 : 1) * x.lanes) * (int64_t)g.n + g.m;
  };
  std::stable_sort(ht.begin(), ht.end(),
                   [&](const BatchTask& x, const BatchTask& y) { return cost(x) > cost(y); });
  DAWN_HIP(hipSetDevice(device));
  // One workgroup per CU: as many as are resident at once.
  const int grid = std::max(1, std::min<int>((int)ht.size(), cus));

  // One allocation for everything, cut at 256-byte offsets.
  stage_cap = (stage_cap + 255) / 256 * 256;
  DevBuf<unsigned char> mem;
  DevBuf<int32_t> dout;
  size_t bytes = 0;
  auto cut = [&](size_t count, size_t size) {
    const size_t at = bytes;
    bytes += (count * size + 255) / 256 * 256;
    return at;
  };
  const size_t g1 = (size_t)grid, mx = (size_t)max_n, lx = (size_t)max_lds_n;
  const size_t o_graphs = cut(hg.size(), sizeof(BatchGraph)), o_tasks = cut(ht.size(), sizeof(BatchTask));
  const size_t o_src = cut(hs.size(), sizeof(int32_t));
  const size_t o_cnt = cut(1, sizeof(unsigned)), o_lev = cut(1, sizeof(unsigned long long));
  const size_t o_glev = cut(hg.size(), sizeof(int32_t)), o_levels_end = bytes;
  const size_t o_wsum = cut(hg.size(), sizeof(unsigned long long)), o_zero_end = bytes;
  const size_t o_seen = cut(g1 * mx, sizeof(uint64_t)), o_next = cut(g1 * mx, sizeof(uint64_t));
  const size_t o_q = cut(g1 * 2 * mx, sizeof(int32_t)), o_qw = cut(g1 * 2 * mx, sizeof(uint64_t));
  const size_t o_touch = cut(g1 * mx, sizeof(int32_t)), o_stage = cut(g1 * (size_t)stage_cap, 1);
  const size_t o_ldsq = cut(g1 * lx, sizeof(int32_t)), o_ent = cut(g1 * lx, sizeof(int2));
  DAWN_TRY(mem.alloc(bytes));
  bool any_weighted = false;
  bool all_weighted = true;
  for (const BatchGraph& x : hg) {
    any_weighted = any_weighted || x.weighted;
    all_weighted = all_weighted && x.weighted;
  }
  // Weighted tasks lower the distances in the rows: in plain memory of the
  // device only.
  const bool direct = any_weighted ? in_place(device, dist) : is_device_pointer(dist);
  int32_t* out = dist;
  if (!direct) {
    DAWN_TRY(dout.alloc((size_t)total));
    out = dout.p;
  }
  hipStream_t s = graphs[0]->stream;
  unsigned char* const M = mem.p;
  DAWN_HIP(hipMemcpyAsync(M + o_graphs, hg.data(), sizeof(BatchGraph) * hg.size(), hipMemcpyHostToDevice, s));
  DAWN_HIP(hipMemcpyAsync(M + o_tasks, ht.data(), sizeof(BatchTask) * ht.size(), hipMemcpyHostToDevice, s));
  DAWN_HIP(hipMemcpyAsync(M + o_src, hs.data(), sizeof(int32_t) * hs.size(), hipMemcpyHostToDevice, s));
  DAWN_HIP(hipMemsetAsync(M + o_cnt, 0, o_zero_end - o_cnt, s));
  BatchArgs a{};
  a.graphs = (const BatchGraph*)(M + o_graphs);
  a.tasks = (const BatchTask*)(M + o_tasks);
  a.num_tasks = (int32_t)ht.size();
  a.spg = spg;
  a.sources = (const int32_t*)(M + o_src);
  a.dist = out;
  a.task_counter = (unsigned*)(M + o_cnt);
  a.levels_total = (unsigned long long*)(M + o_lev);
  a.wsum = (const unsigned long long*)(M + o_wsum);
  a.graph_levels = (int32_t*)(M + o_glev);
  a.max_n = max_n;
  a.seen = (uint64_t*)(M + o_seen);
  a.next = (uint64_t*)(M + o_next);
  a.qv = (int32_t*)(M + o_q);
  a.qw = (uint64_t*)(M + o_qw);
  a.touched = (int32_t*)(M + o_touch);
  a.stage = M + o_stage;
  a.stage_cap = stage_cap;
  a.lds_q = (int32_t*)(M + o_ldsq);
  a.entries = (int2*)(M + o_ent);
  a.max_lds_n = max_lds_n;
  hipEvent_t e0, e1;
  DAWN_HIP(hipEventCreate(&e0));
  DAWN_HIP(hipEventCreate(&e1));
  DAWN_HIP(hipEventRecord(e0, s));
  if (any_weighted) wsum_kernel<<<num_graphs * kWsumParts, kBlock, 0, s>>>(a.graphs, (unsigned long long*)(M + o_wsum));
  if (!any_weighted && max_lds_n == 0) batch_kernel<kBatchBlock, 3><<<grid, kBatchBlock, 0, s>>>(a);
  else if (!any_weighted) batch_kernel<kBatchBlock, 0><<<grid, kBatchBlock, 0, s>>>(a);
  else if (all_weighted) batch_kernel<kBatchBlock, 1><<<grid, kBatchBlock, 0, s>>>(a);
  else batch_kernel<kBatchBlock, 2><<<grid, kBatchBlock, 0, s>>>(a);
  DAWN_HIP(hipGetLastError());
  DAWN_HIP(hipEventRecord(e1, s));
  DAWN_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  DAWN_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  std::vector<unsigned char> lev(o_levels_end - o_lev);
  DAWN_HIP(hipMemcpy(lev.data(), M + o_lev, lev.size(), hipMemcpyDeviceToHost));
  unsigned long long levels = 0;
  std::memcpy(&levels, lev.data(), sizeof levels);
  for (int32_t i = 0; i < num_graphs; i++) {
    int32_t most = 0;
    std::memcpy(&most, lev.data() + (o_glev - o_lev) + sizeof(int32_t) * (size_t)i, sizeof most);
    if (most > graphs[i]->batch_levels.load(std::memory_order_relaxed))
      graphs[i]->batch_levels.store(most, std::memory_order_relaxed);
  }
  if (dist && !direct && !is_device_pointer(dist)) {
    DAWN_HIP(hipMemcpy(dist, out, sizeof(int32_t) * (size_t)total, hipMemcpyDeviceToHost));
  } else if (dist && !direct) {  // what lies between the graphs' rows stays
    for (int32_t i = 0; i < num_graphs; i++)
      DAWN_HIP(hipMemcpyAsync(dist + dist_offsets[i], out + dist_offsets[i],
                              sizeof(int32_t) * (size_t)spg * hg[i].n, hipMemcpyDefault, s));
    DAWN_HIP(hipStreamSynchronize(s));
  }
  if (stats) {
    stats->device_ms += ms;
    stats->steps += (int64_t)levels;
    stats->batches += (int64_t)ht.size();
  }
  return DAWN_OK;
}
