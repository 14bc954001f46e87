// Batched weighted multi-source shortest paths: int32 min-plus over up to 64
// sources at once on one HIP device.
//
// Replaces the per-source weighted loops of the reference,
// DAWN::MSSP_GPU::run_Weighted (src/algorithm/gpu/mssp.cu:53-102) and
// DAWN::APSP_GPU::run_Weighted (src/algorithm/gpu/apsp.cu:9-60) (and the
// CPU MSSP, whose weighted sparse step GOVM reads distance[j] for the queue
// index, src/algorithm/cpu/sssp.cpp:157; not reproduced): the sources of a
// batch share every frontier step.  Per source the result is the reference
// SSSP's (SSSP_CPU::SSSP, sssp.cpp:23-80): the source's listed out-edges
// seed their weight in row order (a later duplicate overwrites an earlier
// one), the source itself is never relaxed, and the distances are the
// fixed point of min-plus relaxation from that state.
//
// Layout in HBM (per graph, reused across batches):
//   dist   int32[n][L]   L = 8, 16, 32 or 64 lanes (the smallest power of
//                        two >= the batch's sources, at least 8), so one
//                        vertex's distances of all lanes share cache lines
//   act    u32[3][n]     lanes of v improved in a step (step k reads k % 3,
//                        writes k + 1 and clears what step k - 1 read; u64
//                        for 64 lanes)
//   q      int32[3][n]   vertices with any improved lane, in the same order
// One kernel a step, launched with its number k: every workgroup derives the
// mode from the frontier's size, the queue lengths rotate over four slots, so
// nothing is decided, swapped or cleared between steps (four kernels a step,
// two of them idle, cost 30 us of each).  The host launches a chunk of steps
// and reads whether the frontier emptied.
//
// A group of L / 4 threads holds a vertex's record, four lanes a thread, so
// that a wave's 16-byte loads cover whole lines (a thread per record took 64
// lines an instruction: 285 us per pull step of a 2048 x 2048 grid, 16 lanes,
// the L1's rate).  Push: a group per queued vertex relaxes its edges four at a
// time; improved lanes are OR-ed into act[k + 1], the first improvement appends
// the vertex (staged per workgroup in LDS).  Edge lists of heavy vertices go by
// chunks, a wave each.
//
// Graphs small enough for a workgroup's LDS take another route (by_workgroup).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.hpp"

namespace dawn {

namespace {

constexpr int kWChunk = 32;       // steps per wait before a traversal's depth is known
constexpr int kWStageCap = 4096;  // next-queue entries a workgroup stages in LDS
// Vertices per workgroup of a step: what a pull may append stays within half of
// kWStageCap (past it every wave's append is an atomic on one address: with
// 4096 vertices to 2048 entries a step of a 2048 x 2048 grid took 0.8 ms).
constexpr int kWSpan = 2048;
constexpr int kWSlots = 4, kWSlotPad = 32;  // queue lengths, a line each

struct WState {
  int32_t steps;       // steps taken
  int32_t pull_steps;  // of those, pulled
  int32_t done;
  int32_t pad[29];
  unsigned qlen[kWSlots * kWSlotPad];
};

// Pull when the frontier holds at least n / kWPullDiv vertices (policy
// FIXED / LEARNED); PUSH and PULL policies force one mode.  Measured, 16 lanes,
// n/16, n/8, n/5: 2048 x 2048 10.6, 10.1, 9.9 ms; ER 1,000,000 3.2, 3.0, 2.9;
// RMAT-18 2.3, 2.4, 3.0; RMAT-20 6.4, 6.3, 6.9.
constexpr int64_t kWPullDiv = 8;

struct WBatch {
  int32_t nlanes;
  int32_t pad;
  int32_t src[64];
};

struct WArgs {
  int32_t n;
  int32_t policy;
  const int32_t* row_ptr;
  const int32_t* col;
  const int32_t* w;
  const int32_t* in_row_ptr;  // in-edges (CSC; the CSR for undirected graphs)
  const int32_t* in_col;
  const int32_t* in_w;
  const int32_t* hc_v;        // in-edge chunks of vertices of in-degree >= heavy
  const int32_t* hc_beg;
  const int32_t* hc_end;
  int64_t num_hc;
  const int32_t* oc_v;        // the same of out-edges
  const int32_t* oc_beg;
  const int32_t* oc_end;
  int64_t num_oc;
  int32_t heavy;
  int32_t* dist;        // [n][L]
  uint64_t* act;        // [3][n]
  int32_t* q;           // [3][n]
  WState* st;
  const WBatch* batch;
};

// Masks of a batch's lanes: 32 bits where they suffice (2048 x 2048, 16 lanes:
// 10.1 ms with 64, 9.3 with 32: the masks are read once per edge).
template <int L>
using WMask = std::conditional_t<(L <= 32), unsigned int, unsigned long long>;
template <int L>
__device__ __forceinline__ WMask<L>* w_act(const WArgs& a, int slot) {
  return reinterpret_cast<WMask<L>*>(a.act) + (int64_t)slot * a.n;
}

template <int L>
__global__ void w_fill_kernel(WArgs a) {
  const int64_t gs = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t quads = (int64_t)a.n * L / 4;
  for (int64_t i = t0; i < quads; i += gs)
    reinterpret_cast<int4*>(a.dist)[i] = make_int4(kInf, kInf, kInf, kInf);
  for (int64_t i = t0; i < 3 * (int64_t)a.n; i += gs) w_act<L>(a, 0)[i] = 0;
  uint32_t* st = reinterpret_cast<uint32_t*>(a.st);
  if (t0 < (int64_t)(sizeof(WState) / 4)) st[t0] = 0u;
}

// Reference initialisation, one workgroup per source lane (each owns its
// column of dist): of the listed out-edges to a neighbour the last gives its
// weight (first a tag, -1 - edge, whose minimum is that edge's), then
// dist[source] = 0; the out-neighbours other than the source form the first
// frontier.  Isolated sources keep an empty frontier (row INF except the
// source), as MSSP skips them.
template <int L>
__global__ void __launch_bounds__(kBlock) w_seed_kernel(WArgs a) {
  const int b = blockIdx.x;
  if (b >= a.batch->nlanes) return;
  const int32_t s = a.batch->src[b];
  const int32_t beg = a.row_ptr[s], end = a.row_ptr[s + 1];
  auto at = [&](int32_t v) { return a.dist + (int64_t)v * L + b; };
  for (int32_t k = beg + threadIdx.x; k < end; k += kBlock) atomicMin(at(a.col[k]), -1 - k);
  __syncthreads();
  for (int32_t k = beg + threadIdx.x; k < end; k += kBlock) {
    int32_t* p = at(a.col[k]);
    if (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == -1 - k)
      __hip_atomic_store(p, a.w[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(at(s), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int32_t k = beg + threadIdx.x; k < end; k += kBlock) {
    const int32_t v = a.col[k];
    if (v == s) continue;
    const WMask<L> old = atomicOr(&w_act<L>(a, 0)[v], (WMask<L>)1 << b);
    if (old == 0) a.q[atomicAdd(&a.st->qlen[0], 1u)] = v;
  }
}

// Of two distances, kInf for none (both are >= 0).
__device__ __forceinline__ int32_t w_plus(int32_t x, int32_t y) {
  return (int32_t)min((uint32_t)x + (uint32_t)y, (uint32_t)kInf);
}

__device__ __forceinline__ bool w_pulls(unsigned qn, int32_t n, int32_t policy) {
  if (policy == DAWN_POLICY_PULL) return true;
  return policy != DAWN_POLICY_PUSH && (int64_t)qn * kWPullDiv >= (int64_t)n;
}

// OR over the groups of VL threads; every thread of a group receives it.
template <int VL>
__device__ __forceinline__ uint64_t group_or(uint64_t x) {
#pragma unroll
  for (int o = 1; o < VL; o <<= 1) {
    uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)x, o), hi = 0;
    if (VL == 16) hi = (uint32_t)__shfl_xor((int)(uint32_t)(x >> 32), o);
    x |= (uint64_t)hi << 32 | lo;
  }
  return x;
}

constexpr int kRound = 4;  // edges in flight per group

// Step k.  A pull, for large frontiers: every vertex v takes, per source lane
// b, the minimum of dist[u][b] + w over its in-edges (u, w) whose tail improved
// lane b in the last step, and stores the lanes that improve with plain stores
// (v's record is written by v's group only; a concurrent reader of it sees the
// old or the new value of each lane, both path lengths, so the fixed point is
// unchanged).  Vertices of in-degree >= heavy are done by in-edge chunks, a
// wave each, merged with atomicMin.
template <int L, bool Wide>
__global__ void __launch_bounds__(kBlock) w_step_kernel(WArgs a, int k) {
  constexpr int VL = L / 4;          // threads per record
  constexpr int VW = kWave / VL;     // records per wave
  if (a.st->done) return;  // set by an earlier step, or by this one where qn == 0
  const unsigned qn = a.st->qlen[(k % kWSlots) * kWSlotPad];
  if (qn == 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) a.st->done = 1;
    return;
  }
  const bool pull = w_pulls(qn, a.n, a.policy);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.st->qlen[((k + 2) % kWSlots) * kWSlotPad] = 0u;
    a.st->steps = k + 1;
    a.st->pull_steps += pull;
  }
  const int32_t* q_in = a.q + (int64_t)(k % 3) * a.n;
  int32_t* q_out = a.q + (int64_t)((k + 1) % 3) * a.n;
  using Mask = WMask<L>;
  const Mask* act_in = w_act<L>(a, k % 3);
  Mask* act_out = w_act<L>(a, (k + 1) % 3);
  unsigned* qlen_out = &a.st->qlen[((k + 1) % kWSlots) * kWSlotPad];
  const int64_t t0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t threads = (int64_t)gridDim.x * kBlock;
  // The masks step k - 1 read: by its queue, or all where that held many.
  if (k > 0) {
    Mask* clr = w_act<L>(a, (k + 2) % 3);
    const int32_t* q_prev = a.q + (int64_t)((k + 2) % 3) * a.n;
    const unsigned pn = a.st->qlen[((k + kWSlots - 1) % kWSlots) * kWSlotPad];
    if ((int64_t)pn * 16 >= a.n) {
      for (int64_t i = t0; i < a.n; i += threads) clr[i] = 0;
    } else {
      for (int64_t i = t0; i < pn; i += threads) clr[q_prev[i]] = 0;
    }
  }
  __shared__ LdsQueue<kWStageCap> s_q;
  if (threadIdx.x == 0) s_q.init();
  __syncthreads();
  const int lane = lane_id();
  const int sub = lane % VL, grp = lane / VL;
  const int64_t wave = t0 / kWave, nwaves = threads / kWave;
  auto quad = [&](int32_t v) { return reinterpret_cast<int4*>(a.dist + (int64_t)v * L) + sub; };
  // This thread's lanes of a mask; inactive lanes' distances count as kInf.
  auto bits4 = [&](Mask m) { return (unsigned)(m >> (4 * sub)) & 15u; };
  auto masked = [&](int4 d, unsigned m) {
    return make_int4(m & 1 ? d.x : kInf, m & 2 ? d.y : kInf, m & 4 ? d.z : kInf, m & 8 ? d.w : kInf);
  };
  if (!pull) {
    // kRound edges of this group's vertex (v < 0: none), whose distances are du.
    auto relax = [&](const int32_t (&v)[kRound], const int32_t (&wt)[kRound], int4 du) {
      int4 dv[kRound];
      int32_t old[kRound][4], nd[kRound][4];
#pragma unroll
      for (int r = 0; r < kRound; r++) dv[r] = v[r] >= 0 ? *quad(v[r]) : make_int4(0, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < kRound; r++) {
        nd[r][0] = w_plus(du.x, wt[r]), nd[r][1] = w_plus(du.y, wt[r]);
        nd[r][2] = w_plus(du.z, wt[r]), nd[r][3] = w_plus(du.w, wt[r]);
        int32_t* p = reinterpret_cast<int32_t*>(quad(v[r]));
        old[r][0] = nd[r][0] < dv[r].x ? atomicMin(p, nd[r][0]) : -1;
        old[r][1] = nd[r][1] < dv[r].y ? atomicMin(p + 1, nd[r][1]) : -1;
        old[r][2] = nd[r][2] < dv[r].z ? atomicMin(p + 2, nd[r][2]) : -1;
        old[r][3] = nd[r][3] < dv[r].w ? atomicMin(p + 3, nd[r][3]) : -1;
      }
      // Opaque to the compiler, which else moves each comparison, and with it
      // the wait for its atomic, up before the next atomic.
#pragma unroll
      for (int r = 0; r < kRound; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) asm volatile("" : "+v"(old[r][c]));
      Mask was[kRound], imp[kRound];
#pragma unroll
      for (int r = 0; r < kRound; r++) {
        unsigned x = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) x |= (nd[r][c] < old[r][c] ? 1u : 0u) << c;
        imp[r] = (Mask)group_or<VL>((uint64_t)x << (4 * sub));
        was[r] = 1;
        if (sub == 0 && imp[r]) was[r] = atomicOr(&act_out[v[r]], imp[r]);
      }
#pragma unroll
      for (int r = 0; r < kRound; r++) asm volatile("" : "+v"(was[r]));
#pragma unroll
      for (int r = 0; r < kRound; r++)
        s_q.append(sub == 0 && imp[r] != 0 && was[r] == 0, v[r], qlen_out, q_out);
    };
    for (int64_t i0 = wave * VW; i0 < qn; i0 += nwaves * VW) {  // wave-uniform
      const int64_t i = i0 + grp;
      int32_t u = 0;
      int beg = 0, deg = 0;
      int4 du = make_int4(kInf, kInf, kInf, kInf);
      if (i < qn) {
        u = q_in[i];
        beg = a.row_ptr[u];
        deg = a.row_ptr[u + 1] - beg;
        const unsigned m = bits4(act_in[u]);
        du = masked(*quad(u), m);
        if (deg >= a.heavy) deg = 0;
      }
      const int most = wave_max_i32(deg);
      for (int j = 0; j < most; j += kRound) {
        int32_t v[kRound], wt[kRound];
#pragma unroll
        for (int r = 0; r < kRound; r++) v[r] = j + r < deg ? a.col[beg + j + r] : -1;
#pragma unroll
        for (int r = 0; r < kRound; r++) wt[r] = j + r < deg ? a.w[beg + j + r] : 0;
        relax(v, wt, du);
      }
    }
    // Heavy vertices by out-edge chunks: a wave looks at 64 chunks, then takes
    // the active ones, kRound edges per group at a time.  The 64 lie a grid
    // apart: few neighbouring ones would leave most waves without any and the
    // others with 64 in turn (3000 vertices of degree 50, 64 sources, pushed: 6.8
    // ms, so 0.72; RMAT-17, 64 sources, by the rule 6.1 and 3.4).
    for (int64_t c0 = wave; c0 < a.num_oc; c0 += nwaves * kWave) {  // wave-uniform
      const int64_t c = c0 + lane * nwaves;
      uint64_t hot = __ballot(c < a.num_oc && act_in[a.oc_v[c < a.num_oc ? c : 0]] != 0);
      for (; hot; hot &= hot - 1) {
        const int64_t hc = c0 + (__ffsll((unsigned long long)hot) - 1) * nwaves;
        const int32_t u = a.oc_v[hc];
        const int kb = a.oc_beg[hc], ke = a.oc_end[hc];
        const int4 du = masked(*quad(u), bits4(act_in[u]));
        for (int j = kb; j < ke; j += kRound * VW) {
          int32_t v[kRound], wt[kRound];
#pragma unroll
          for (int r = 0; r < kRound; r++) v[r] = j + r * VW + grp < ke ? a.col[j + r * VW + grp] : -1;
#pragma unroll
          for (int r = 0; r < kRound; r++) wt[r] = j + r * VW + grp < ke ? a.w[j + r * VW + grp] : 0;
          relax(v, wt, du);
        }
      }
    }
  } else {
    // Minima over kRound in-edges (u < 0: none) of this thread's lanes.
    auto gather = [&](const int32_t (&u)[kRound], const int32_t (&wt)[kRound], int4& best) {
      unsigned m[kRound];
      int4 du[kRound];
#pragma unroll
      for (int r = 0; r < kRound; r++) m[r] = u[r] >= 0 ? bits4(act_in[u[r]]) : 0u;
#pragma unroll
      for (int r = 0; r < kRound; r++)
        du[r] = m[r] ? *quad(u[r]) : make_int4(kInf, kInf, kInf, kInf);
#pragma unroll
      for (int r = 0; r < kRound; r++) {
        const int4 d = masked(du[r], m[r]);
        best.x = min(best.x, w_plus(d.x, wt[r])), best.y = min(best.y, w_plus(d.y, wt[r]));
        best.z = min(best.z, w_plus(d.z, wt[r])), best.w = min(best.w, w_plus(d.w, wt[r]));
      }
    };
    // Lanes of best below dv, moved there.
    auto take = [](const int4& best, int4& dv) {
      unsigned x = 0;
      if (best.x < dv.x) dv.x = best.x, x |= 1;
      if (best.y < dv.y) dv.y = best.y, x |= 2;
      if (best.z < dv.z) dv.z = best.z, x |= 4;
      if (best.w < dv.w) dv.w = best.w, x |= 8;
      return x;
    };
    if constexpr (Wide) {
      // Records of 64 lanes, or of 32 where heavy vertices hold the edges: a
      // group takes a vertex, list and all (the minima of 64 vertices would
      // take 32 or 64 registers and leave two or three waves per SIMD to the
      // heavy vertices: RMAT-20, 64 sources, 23 -> 32 ms, 32 sources 13 -> 18;
      // without heavy vertices, 2048 x 2048, 32 sources, 28 -> 22).  Which
      // vertices have a tail that improved is found first, a thread each, unless
      // most will have one: most of a step's vertices often have none, and a
      // group waits on three accesses for each (1000 x 1000 with shortcuts, 33
      // sources, all steps pulled: 16.3 -> 10.8 ms, by the rule 10.4 -> 10.1;
      // RMAT-20 of degree 8, 64 sources, pulled 16.3 -> 11.4).  A wave looks at 64
      // vertices, or as many as give every wave some (random graph of 65,536,
      // degree 8, 64 sources: 2.3 ms by 64 vertices, 1.3 so).
      // A group takes two vertices at a time, without branches, so that both
      // chains are in flight (2048 x 2048, 64 sources, pulled 3.24 -> 2.82 s, by the
      // rule 3.13 -> 2.72; random graph of 1,000,000, degree 12, 16.7 -> 15.8 ms;
      // RMAT-20 18.2 -> 18.0).  An edge past a list's end reads the list's first
      // one; a group that has a first vertex and no second reads the edge at the
      // lists' start of the wave's first vertex, which is not past the first's.
      const bool dense = (int64_t)qn * 4 >= a.n;
      const int64_t each = (a.n + nwaves - 1) / nwaves;
      const int span = (int)min((int64_t)kWave, (each + 2 * VW - 1) / (2 * VW) * (2 * VW));
      for (int64_t v0 = wave * span; v0 < a.n; v0 += nwaves * span) {  // wave-uniform
        int vbeg = 0, vdeg = 0;
        if (lane < span && v0 + lane < a.n) {
          vbeg = a.in_row_ptr[v0 + lane];
          vdeg = a.in_row_ptr[v0 + lane + 1] - vbeg;
          if (vdeg >= a.heavy) vdeg = 0;
        }
        bool hot = dense && vdeg > 0;
        for (int j = 0; __ballot(!hot && j < vdeg); j += kRound) {
          int32_t u[kRound];
          Mask m[kRound];
#pragma unroll
          for (int r = 0; r < kRound; r++) u[r] = !hot && j + r < vdeg ? a.in_col[vbeg + j + r] : -1;
#pragma unroll
          for (int r = 0; r < kRound; r++) m[r] = u[r] >= 0 ? act_in[u[r]] : (Mask)0;
#pragma unroll
          for (int r = 0; r < kRound; r++) hot |= m[r] != 0;
        }
        uint64_t todo = __ballot(hot);
        while (todo) {  // 2 VW of them at a time
          int at[2] = {-1, -1}, beg[2], deg[2];
          int32_t v[2];
          int4 best[2];
#pragma unroll
          for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int q = 0; q < VW; q++) {
              if (grp == q && todo) at[h] = __ffsll((unsigned long long)todo) - 1;
              todo &= todo - 1;
            }
            const int from = at[h] < 0 ? 0 : at[h];
            beg[h] = __shfl(vbeg, from);
            const int len = __shfl(vdeg, from);
            deg[h] = at[h] < 0 ? 0 : len;
            v[h] = (int32_t)v0 + from;
            best[h] = make_int4(kInf, kInf, kInf, kInf);
          }
          for (int j = 0; j < max(deg[0], deg[1]); j += kRound) {
            int32_t u[2][kRound], wt[2][kRound];
            unsigned m[2][kRound];
            int4 du[2][kRound];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int r = 0; r < kRound; r++) {
                const int k = beg[h] + (j + r < deg[h] ? j + r : 0);
                u[h][r] = a.in_col[k];
                wt[h][r] = a.in_w[k];
              }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int r = 0; r < kRound; r++) {
                const Mask x = act_in[u[h][r]];
                m[h][r] = j + r < deg[h] ? bits4(x) : 0u;
              }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int r = 0; r < kRound; r++) du[h][r] = *quad(m[h][r] ? u[h][r] : v[h]);
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int r = 0; r < kRound; r++) {
                const int4 d = masked(du[h][r], m[h][r]);
                int4& b = best[h];
                b.x = min(b.x, w_plus(d.x, wt[h][r])), b.y = min(b.y, w_plus(d.y, wt[h][r]));
                b.z = min(b.z, w_plus(d.z, wt[h][r])), b.w = min(b.w, w_plus(d.w, wt[h][r]));
              }
          }
#pragma unroll
          for (int h = 0; h < 2; h++) {
            unsigned x = 0;
            if (min(min(best[h].x, best[h].y), min(best[h].z, best[h].w)) != kInf) {
              int4 dv = *quad(v[h]);
              x = take(best[h], dv);
              if (x) *quad(v[h]) = dv;
            }
            const uint64_t imp = group_or<VL>((uint64_t)x << (4 * sub));
            if (sub == 0 && imp) act_out[v[h]] = (Mask)imp;  // v's own slot (heavy vertices are not here)
            s_q.append(sub == 0 && imp != 0, v[h], qlen_out, q_out);
          }
        }
      }
    } else {
      // Light vertices, 64 a wave: a thread per vertex reads its list, kRound
      // edges at a time, and their tails' masks; then the groups, VW vertices at
      // a time, read the records.  Without branches (a tail that did not improve
      // gives way to the vertex's own record, read below in any case), so that a
      // stage's loads are all in flight (16 vertices a wave, list and records by
      // the group: 390 us for 2048 x 2048, a chain of six latencies each).
      for (int64_t v0 = wave * kWave; v0 < a.n; v0 += nwaves * kWave) {  // wave-uniform
        int beg = 0, deg = 0;
        if (v0 + lane < a.n) {
          beg = a.in_row_ptr[v0 + lane];
          deg = a.in_row_ptr[v0 + lane + 1] - beg;
          if (deg >= a.heavy) deg = 0;
        }
        int4 best[VL];
#pragma unroll
        for (int q = 0; q < VL; q++) best[q] = make_int4(kInf, kInf, kInf, kInf);
        auto vertex = [&](int q) { return (int32_t)min(v0 + q * VW + grp, (int64_t)a.n - 1); };
        const int most = wave_max_i32(deg);
        bool any = false;
        for (int j = 0; j < most; j += kRound) {
          int32_t u[kRound], wt[kRound];
          Mask m[kRound];
#pragma unroll
          for (int r = 0; r < kRound; r++) {
            const int k = j + r < deg ? beg + j + r : 0;
            u[r] = a.in_col[k];
            wt[r] = a.in_w[k];
          }
#pragma unroll
          for (int r = 0; r < kRound; r++) m[r] = act_in[u[r]];
          Mask seen = 0;
#pragma unroll
          for (int r = 0; r < kRound; r++) {
            m[r] = j + r < deg ? m[r] : (Mask)0;
            seen |= m[r];
          }
          if (!__ballot(seen != 0)) continue;
          any = true;
#pragma unroll
          for (int q = 0; q < VL; q += 2) {
            int4 du[2][kRound];
            int32_t w2[2][kRound];
            unsigned m2[2][kRound];
#pragma unroll
            for (int h = 0; h < 2; h++) {
              const int from = (q + h) * VW + grp;
#pragma unroll
              for (int r = 0; r < kRound; r++) {
                m2[h][r] = bits4((uint32_t)__shfl((int)(uint32_t)m[r], from));
                w2[h][r] = __shfl(wt[r], from);
                const int32_t t = __shfl(u[r], from);
                du[h][r] = *quad(m2[h][r] ? t : vertex(q + h));
              }
            }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int r = 0; r < kRound; r++) {
                const int4 d = masked(du[h][r], m2[h][r]);
                int4& b = best[q + h];
                b.x = min(b.x, w_plus(d.x, w2[h][r])), b.y = min(b.y, w_plus(d.y, w2[h][r]));
                b.z = min(b.z, w_plus(d.z, w2[h][r])), b.w = min(b.w, w_plus(d.w, w2[h][r]));
              }
          }
        }
        if (!any) continue;
#pragma unroll
        for (int q = 0; q < VL; q += 2) {
          int4 dv[2];
#pragma unroll
          for (int h = 0; h < 2; h++) dv[h] = *quad(vertex(q + h));
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int4 b = best[q + h];
            const int32_t v = vertex(q + h);
            const bool in = v0 + (q + h) * VW + grp < a.n;
            const unsigned x = in ? take(b, dv[h]) : 0u;
            if (x) *quad(v) = dv[h];
            const uint64_t imp = group_or<VL>((uint64_t)x << (4 * sub));
            if (sub == 0 && imp) act_out[v] = (Mask)imp;  // v's own slot (heavy vertices are not here)
            s_q.append(sub == 0 && imp != 0, v, qlen_out, q_out);
          }
        }
      }
    }
    for (int64_t hc = wave; hc < a.num_hc; hc += nwaves) {  // wave-uniform
      const int32_t v = a.hc_v[hc];
      const int kb = a.hc_beg[hc], ke = a.hc_end[hc];
      int4 best = make_int4(kInf, kInf, kInf, kInf);
      for (int j = kb; j < ke; j += kRound * VW) {
        int32_t u[kRound], wt[kRound];
#pragma unroll
        for (int r = 0; r < kRound; r++) u[r] = j + r * VW + grp < ke ? a.in_col[j + r * VW + grp] : -1;
#pragma unroll
        for (int r = 0; r < kRound; r++) wt[r] = j + r * VW + grp < ke ? a.in_w[j + r * VW + grp] : 0;
        gather(u, wt, best);
      }
      for (int o = VL; o < kWave; o <<= 1) {
        best.x = min(best.x, __shfl_xor(best.x, o)), best.y = min(best.y, __shfl_xor(best.y, o));
        best.z = min(best.z, __shfl_xor(best.z, o)), best.w = min(best.w, __shfl_xor(best.w, o));
      }
      unsigned x = 0;
      if (grp == 0 && min(min(best.x, best.y), min(best.z, best.w)) != kInf) {
        int32_t* p = reinterpret_cast<int32_t*>(quad(v));
        const int4 dv = *quad(v);
        if (best.x < dv.x && best.x < atomicMin(p, best.x)) x |= 1;
        if (best.y < dv.y && best.y < atomicMin(p + 1, best.y)) x |= 2;
        if (best.z < dv.z && best.z < atomicMin(p + 2, best.z)) x |= 4;
        if (best.w < dv.w && best.w < atomicMin(p + 3, best.w)) x |= 8;
      }
      const uint64_t imp = group_or<VL>((uint64_t)x << (4 * sub));
      bool append = false;
      if (lane == 0 && imp) append = atomicOr(&act_out[v], (Mask)imp) == 0;
      s_q.append(append, v, qlen_out, q_out);
    }
  }
  s_q.flush(qlen_out, q_out);
}

// Distance rows (lane b at out + b * stride) and per-lane sums: a workgroup
// stages 256 / 128 vertices x L lanes in LDS (one contiguous read, records at
// an odd stride), then wave w writes the rows of lanes w, w + 4, ... segment by
// segment.  Sums stay in registers, per thread and lane, until the end
// (reduced per 64 vertices they took 395 us of a 2048 x 2048 grid's 16 lanes).
// acc: [0..63] distance sums, [64..127] reached vertices, [128..191] sum of
// out-degrees of reached vertices, per lane.
template <int L>
__global__ void __launch_bounds__(kBlock) w_final_kernel(WArgs a, int32_t* out, int64_t stride,
                                                         unsigned long long* acc) {
  constexpr int T = L <= 32 ? 256 : 128;  // vertices per tile
  constexpr int W = kBlock / kWave, B = L / W;
  __shared__ int32_t s_tile[T * (L + 1)];
  __shared__ int32_t s_deg[T];
  const int nl = a.batch->nlanes;
  const int lane = lane_id();
  const int wv = threadIdx.x / kWave;
  unsigned long long sum[B], edges[B];
  unsigned reached[B];
#pragma unroll
  for (int r = 0; r < B; r++) sum[r] = edges[r] = 0, reached[r] = 0;
  for (int64_t b0 = (int64_t)blockIdx.x * T; b0 < a.n; b0 += (int64_t)gridDim.x * T) {
    const int cnt = (int)std::min<int64_t>(T, a.n - b0);  // block-uniform
    const int4* src = reinterpret_cast<const int4*>(a.dist + b0 * L);
    __syncthreads();
    for (int i = threadIdx.x; i < cnt * (L / 4); i += kBlock) {
      const int4 x = src[i];
      int32_t* p = s_tile + (i / (L / 4)) * (L + 1) + i % (L / 4) * 4;
      p[0] = x.x, p[1] = x.y, p[2] = x.z, p[3] = x.w;
    }
    for (int i = threadIdx.x; i < cnt; i += kBlock) s_deg[i] = a.row_ptr[b0 + i + 1] - a.row_ptr[b0 + i];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < B; r++) {
      const int bl = r * W + wv;
      if (bl >= nl) continue;
      for (int i = lane; i < cnt; i += kWave) {
        const int32_t d = s_tile[i * (L + 1) + bl];
        if (out) out[(int64_t)bl * stride + b0 + i] = d;
        if (d != kInf) {
          sum[r] += (unsigned)d;
          reached[r]++;
          edges[r] += (unsigned)s_deg[i];
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < B; r++) {
    const int bl = r * W + wv;
    const unsigned long long s1 = wave_sum_u64(sum[r]), s2 = wave_sum_u64(reached[r]), s3 = wave_sum_u64(edges[r]);
    if (lane == 0 && bl < nl) {
      if (s1) atomicAdd(&acc[bl], s1);
      if (s2) atomicAdd(&acc[64 + bl], s2);
      if (s3) atomicAdd(&acc[128 + bl], s3);
    }
  }
}

__global__ void w_zero_kernel(unsigned long long* p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}

}  // namespace

struct WmsWorkspace {
  int32_t n = 0;
  int32_t lanes = 0;
  DevBuf<int32_t> dist, q, rows;
  DevBuf<uint64_t> act;
  DevBuf<WState> st;
  DevBuf<WBatch> batch;
  DevBuf<unsigned long long> sums;
  WState* h_state = nullptr;
  WBatch* h_batch = nullptr;
  int32_t last_steps = 0;  // steps the last batch took
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

void wms_workspace_free(WmsWorkspace* ws) {
  if (!ws) return;
  if (ws->h_state) (void)hipHostFree(ws->h_state);
  if (ws->h_batch) (void)hipHostFree(ws->h_batch);
  for (hipEvent_t e : {ws->ev0, ws->ev1})
    if (e) (void)hipEventDestroy(e);
  delete ws;
}

namespace {

int ensure_wms(dawn_graph* g, int L) {
  if (!g->wms) g->wms = new WmsWorkspace();
  WmsWorkspace* ws = g->wms;
  if (ws->n == g->n && ws->lanes == L) return DAWN_OK;
  ws->n = ws->lanes = 0;  // set once every buffer is in place
  ws->dist.release();
  ws->rows.release();
  DAWN_TRY(ws->dist.alloc((size_t)g->n * L));
  DAWN_TRY(ws->act.alloc((size_t)3 * g->n));
  DAWN_TRY(ws->q.alloc((size_t)3 * g->n));
  DAWN_TRY(ws->st.alloc(1));
  DAWN_TRY(ws->batch.alloc(1));
  DAWN_TRY(ws->sums.alloc(3 * 64));
  if (!ws->h_state) DAWN_HIP(hipHostMalloc((void**)&ws->h_state, sizeof(WState)));
  if (!ws->h_batch) DAWN_HIP(hipHostMalloc((void**)&ws->h_batch, sizeof(WBatch)));
  for (hipEvent_t* e : {&ws->ev0, &ws->ev1})
    if (!*e) DAWN_HIP(hipEventCreate(e));
  ws->n = g->n;
  ws->lanes = L;
  return DAWN_OK;
}

template <int L>
int run_w(dawn_graph* g, const int32_t* sources, int32_t S, int32_t* dist, int64_t* sums,
          int32_t policy, dawn_stats* stats) {
  DAWN_TRY(ensure_wms(g, L));
  WmsWorkspace* ws = g->wms;
  hipStream_t s = g->stream;
  const bool dist_dev = dist && is_device_pointer(dist);
  if (dist && !dist_dev) DAWN_TRY(ws->rows.alloc((size_t)L * g->n));
  WArgs a{};
  a.n = g->n;
  a.policy = policy;
  a.row_ptr = g->row_ptr;
  a.col = g->col;
  a.w = g->weight;
  a.in_row_ptr = g->in_row_ptr;
  a.in_col = g->in_col;
  a.in_w = g->in_weight;
  a.hc_v = g->hc_v;
  a.hc_beg = g->hc_beg;
  a.hc_end = g->hc_end;
  a.num_hc = g->num_hc;
  a.oc_v = g->oc_v;
  a.oc_beg = g->oc_beg;
  a.oc_end = g->oc_end;
  a.num_oc = g->num_oc;
  a.heavy = g->knobs.heavy_degree;
  a.dist = ws->dist.p;
  a.act = ws->act.p;
  a.q = ws->q.p;
  a.st = ws->st.p;
  a.batch = ws->batch.p;
  const unsigned fill_grid = grid_for((int64_t)g->n * L);
  const unsigned step_grid = (unsigned)std::max<int64_t>(1024, (g->n + kWSpan - 1) / kWSpan);
  const unsigned fin_grid = 1024;
  const bool wide = g->num_hc * 64 > g->n;  // heavy vertices hold many of the edges

  // Steps per wait: what the last batch took and the one that finds the
  // frontier empty, so that one read of the done flag usually suffices.
  const int chunk = ws->last_steps > 0 ? std::min(256, ws->last_steps + 1) : kWChunk;

  float total_ms = 0.f;
  std::vector<unsigned long long> h_sums(3 * 64);
  for (int32_t b0 = 0; b0 < S; b0 += L) {
    const int32_t lanes = std::min<int32_t>(L, S - b0);
    WBatch& hb = *ws->h_batch;
    std::memset(&hb, 0, sizeof hb);
    hb.nlanes = lanes;
    for (int i = 0; i < lanes; i++) {
      int64_t v = sources[b0 + i] % (int64_t)g->n;
      if (v < 0) v += g->n;
      hb.src[i] = (int32_t)v;
      if (stats && g->h_row_ptr[v] == g->h_row_ptr[v + 1]) stats->skipped_sources += 1;
    }
    DAWN_HIP(hipMemcpyAsync(ws->batch.p, ws->h_batch, sizeof(WBatch), hipMemcpyHostToDevice, s));
    DAWN_HIP(hipEventRecord(ws->ev0, s));
    w_fill_kernel<L><<<fill_grid, kBlock, 0, s>>>(a);
    w_seed_kernel<L><<<(unsigned)lanes, kBlock, 0, s>>>(a);
    int64_t launched = 0;
    for (;;) {
      for (int i = 0; i < chunk; i++) {
        const int k = (int)(launched + i);
        if (wide) w_step_kernel<L, L >= 32><<<step_grid, kBlock, 0, s>>>(a, k);
        else w_step_kernel<L, L >= 64><<<step_grid, kBlock, 0, s>>>(a, k);
      }
      launched += chunk;
      DAWN_HIP(hipMemcpyAsync(ws->h_state, ws->st.p, sizeof(WState), hipMemcpyDeviceToHost, s));
      DAWN_HIP(hipStreamSynchronize(s));
      if (ws->h_state->done) break;
      if (launched > (int64_t)g->n + 2 * chunk) return DAWN_ERR_HIP;
    }
    int32_t* out = dist ? (dist_dev ? dist + (int64_t)b0 * g->n : ws->rows.p) : nullptr;
    w_zero_kernel<<<1, 64, 0, s>>>(ws->sums.p, 3 * 64);
    w_final_kernel<L><<<fin_grid, kBlock, 0, s>>>(a, out, g->n, ws->sums.p);
    DAWN_HIP(hipGetLastError());
    DAWN_HIP(hipEventRecord(ws->ev1, s));
    DAWN_HIP(hipMemcpyAsync(h_sums.data(), ws->sums.p, sizeof(unsigned long long) * 3 * 64,
                            hipMemcpyDeviceToHost, s));
    DAWN_HIP(hipStreamSynchronize(s));
    float ms = 0.f;
    DAWN_HIP(hipEventElapsedTime(&ms, ws->ev0, ws->ev1));
    total_ms += ms;
    if (dist && !dist_dev)
      DAWN_HIP(hipMemcpy(dist + (int64_t)b0 * g->n, ws->rows.p, sizeof(int32_t) * (size_t)lanes * g->n,
                         hipMemcpyDeviceToHost));
    for (int i = 0; i < lanes; i++)
      if (sums) sums[b0 + i] = (int64_t)h_sums[i];
    ws->last_steps = ws->h_state->steps;
    if (stats) {
      for (int i = 0; i < lanes; i++) {
        stats->vertices_reached += (int64_t)h_sums[64 + i];
        stats->edges_reached += (int64_t)h_sums[128 + i];
      }
      stats->batches += 1;
      stats->steps += ws->h_state->steps;
      stats->mode_steps[DAWN_MODE_PUSH] += ws->h_state->steps - ws->h_state->pull_steps;
      stats->mode_steps[DAWN_MODE_PULL] += ws->h_state->pull_steps;
    }
  }
  if (stats) stats->device_ms += total_ms;
  return DAWN_OK;
}

}  // namespace

// Graphs whose state fits a workgroup's LDS: every source in a workgroup of
// its own (batch.hip), 256 at a time, instead of 64 lanes that share steps.
// Measured (ms, workgroups / lanes):
//   random graph of 16,384, degree 8: 1 source 0.24 / 0.36, 64 0.26 / 0.58, 256 0.28 / 2.3
//   random graph of 32,768, degree 16: 1 source 0.52 / 0.59, 64 0.55 / 0.99, 256 0.58 / 4.1
//   random graph of 37,000, degree 20: 8 sources - / 0.68, 16 0.63 / 0.78, 64 0.64 / 1.4
//   random graph of 30,000, degree 100: 8 sources - / 0.87, 16 1.19 / 1.10, 32 1.28 / 1.59
//   RMAT-14, 0.43 M edges: 1 source 0.52 / 0.32, 16 0.55 / 0.48, 32 0.55 / 0.58, 64 0.57 / 0.82
//   RMAT-15, 0.88 M edges: 8 sources - / 0.45, 16 0.97 / 0.54, 32 0.99 / 0.73, 64 0.99 / 1.20
//   grid 190 x 190: 1 source 2.0 / 3.5, 64 2.0 / 6.6
//   random graph of 65,536, degree 8: 64 sources - / 1.15, 65 1.13 / 1.84, 256 1.67 / 4.7
//   random graph of 130,000, degree 3: 64 sources - / 1.27, 65 1.56 / 2.10, 256 2.0 / 5.1
//   RMAT-16, 1.8 M edges: 64 sources - / 1.83, 65 2.99 / 1.97, 128 3.5 / 3.7, 256 3.7 / 7.3
//   grid 360 x 360: 64 sources - / 21, 65 8.3 / 27, 256 8.4 / 83
// The lines suit graphs without hubs; with hubs the lanes are the better up to
// some 48 sources, a fixed 0.2 to 0.4 ms that the rule leaves there.
// With the distances in LDS (up to kSourcesDistN vertices) the lines are
// kSourcesM edges and kSourcesS sources; with bounds there and distances in
// memory, more sources than one batch of lanes.  A forced mode is one of the
// lanes' steps, and knobs set by hand are theirs.
constexpr int64_t kSourcesM = 600000;
constexpr int32_t kSourcesS = 16;

static bool by_workgroup(const dawn_graph* g, int32_t S, int32_t policy) {
  if (g->lanes_only() || (policy != DAWN_POLICY_FIXED && policy != DAWN_POLICY_LEARNED)) return false;
  if (g->n > kSourcesN || g->m >= kSourcesMaxM) return false;
  return g->n <= kSourcesDistN ? g->m <= kSourcesM || S >= kSourcesS : S > 64;
}

static int run_lanes(dawn_graph* g, const int32_t* sources, int32_t S, int32_t* dist, int64_t* sums,
                     int32_t policy, dawn_stats* stats) {
  const int32_t per = std::min<int32_t>(S, 64);
  if (per <= 8) return run_w<8>(g, sources, S, dist, sums, policy, stats);
  if (per <= 16) return run_w<16>(g, sources, S, dist, sums, policy, stats);
  if (per <= 32) return run_w<32>(g, sources, S, dist, sums, policy, stats);
  return run_w<64>(g, sources, S, dist, sums, policy, stats);
}

// Weighted multi-source traversal: a workgroup per source, or batches of up to
// 64 sources.
int run_wmsbfs(dawn_graph* g, const int32_t* sources, int32_t S, int32_t* dist, int64_t* sums,
               int32_t policy, dawn_stats* stats) {
  if (!g || !g->weighted || S < 0 || (S > 0 && !sources) || g->n <= 0) return DAWN_ERR_INVALID_ARG;
  if (S == 0) return DAWN_OK;
  std::lock_guard<std::mutex> guard(g->lock);
  DAWN_HIP(hipSetDevice(g->device));
  if (by_workgroup(g, S, policy)) {
    if (!g->sources) g->sources = new SourcesWorkspace();
    std::vector<int32_t> src(S);
    for (int32_t i = 0; i < S; i++) {
      int64_t v = sources[i] % (int64_t)g->n;
      if (v < 0) v += g->n;
      src[i] = (int32_t)v;
    }
    std::vector<unsigned long long> acc;
    double ms = 0;
    const int rc = run_sources_lds(g, g->sources, src.data(), S, dist, false, acc, &ms);
    if (rc == DAWN_ERR_OUT_OF_MEMORY) {  // nothing has run yet: the lanes try
      sources_workspace_free(g->sources);
      g->sources = nullptr;
      (void)hipGetLastError();
      return run_lanes(g, sources, S, dist, sums, policy, stats);
    }
    if (rc != DAWN_OK) return rc;
    int64_t steps = 0;
    for (int32_t i = 0; i < S; i++) {
      const unsigned long long* x = acc.data() + (size_t)i * 4;
      if (sums) sums[i] = (int64_t)x[0];
      if (!stats) continue;
      if (g->h_row_ptr[src[i]] == g->h_row_ptr[src[i] + 1]) stats->skipped_sources += 1;
      stats->vertices_reached += (int64_t)x[1];
      stats->edges_reached += (int64_t)x[2];
      // Batches of 64 sources, as the lanes count them: the steps of one are
      // those of its longest source.
      steps = std::max<int64_t>(i % 64 ? steps : 0, (int64_t)x[3]);
      if (i % 64 != 63 && i != S - 1) continue;
      stats->steps += steps;
      stats->mode_steps[DAWN_MODE_PUSH] += steps;
      stats->batches += 1;
    }
    if (stats) stats->device_ms += ms;
    return DAWN_OK;
  }
  return run_lanes(g, sources, S, dist, sums, policy, stats);
}

}  // namespace dawn
