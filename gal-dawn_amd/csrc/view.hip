// Hub-first vertex order for the batched unweighted engine (no counterpart
// in the reference, whose vertices keep their file order).
//
// The dense pull gathers the frontier record of every in-neighbour, and on
// skewed graphs most gathers hit the few vertices of largest out-degree.
// Scattered over the vertex range, each such record shares its cache line
// with cold vertices; placed first, the hot records fill whole lines and a
// few MB of L2 / Infinity Cache hold them.  The view renumbers the k
// vertices of largest out-degree to [0, k) (descending degree, ties by id)
// and keeps every other vertex in its original order after them, so the
// distance pass, which writes rows in the original order, still reads
// almost contiguous records.  Results are identical (the order only moves
// work in memory); the engine maps sources in and rows out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "common.hpp"

namespace dawn {

namespace {

// Row r of the new adjacency = row inv[r] of the old one, columns mapped
// through perm, the hubs (new ids below k) first: a pull finds most lanes at
// them and leaves the row.  One wave per row, 64 edges at a time, placed by
// ballots: hubs from the front, then the others.
__global__ void view_copy_kernel(int32_t n, int32_t k, const int32_t* old_rp, const int32_t* old_col,
                                 const int32_t* new_rp, int32_t* new_col, const int32_t* inv,
                                 const int32_t* perm) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t nwaves = (int64_t)gridDim.x * blockDim.x / kWave;
  for (int64_t r = wave; r < n; r += nwaves) {
    const int32_t o = inv[r];
    const int32_t b = old_rp[o], deg = old_rp[o + 1] - b, nb = new_rp[r];
    if (deg <= kWave) {
      const int32_t c = lane < deg ? perm[old_col[b + lane]] : 0;
      const uint64_t in = __ballot(lane < deg), hub = __ballot(lane < deg && c < k);
      const uint64_t mine = c < k ? hub : in & ~hub;
      const int at = (c < k ? 0 : __popcll(hub)) + __popcll(mine & lanes_below_mask());
      if (lane < deg) new_col[nb + at] = c;
      continue;
    }
    int hubs = 0;
    for (int j = lane; j - lane < deg; j += kWave)  // wave-uniform
      hubs += __popcll(__ballot(j < deg && perm[old_col[b + (j < deg ? j : 0)]] < k));
    int front = 0, back = hubs;
    for (int j = lane; j - lane < deg; j += kWave) {
      const int32_t c = j < deg ? perm[old_col[b + j]] : 0;
      const uint64_t in = __ballot(j < deg), hub = __ballot(j < deg && c < k), rest = in & ~hub;
      const int at = c < k ? front + __popcll(hub & lanes_below_mask()) : back + __popcll(rest & lanes_below_mask());
      if (j < deg) new_col[nb + at] = c;
      front += __popcll(hub);
      back += __popcll(rest);
    }
  }
}

void free_ptr(int32_t*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

}  // namespace

void ms_view_free(dawn_graph* g) {
  MsView* v = g->view;
  if (!v) return;
  (void)hipSetDevice(g->device);
  if (v->in_row_ptr == v->row_ptr) v->in_row_ptr = nullptr;
  if (v->in_col == v->col) v->in_col = nullptr;
  if (v->oc_v == v->hc_v) v->oc_v = v->oc_beg = v->oc_end = nullptr;
  for (int32_t** p : {&v->row_ptr, &v->col, &v->in_row_ptr, &v->in_col, &v->perm, &v->hc_v,
                      &v->hc_beg, &v->hc_end, &v->oc_v, &v->oc_beg, &v->oc_end})
    free_ptr(*p);
  delete v;
  g->view = nullptr;
}

// Builds the view if the knobs ask for one and the graph is large enough
// for cache placement to matter; returns DAWN_OK with g->view == null
// otherwise.
int ms_view_ensure(dawn_graph* g) {
  if (!g->knobs.hub_order || g->n < kViewMinVertices) {
    ms_view_free(g);
    return DAWN_OK;
  }
  if (g->view) return DAWN_OK;
  const int32_t n = g->n;
  const int32_t k = std::max<int32_t>(1, n / 16);
  MsView* view = new MsView();
  view->k = k;
  g->view = view;
  auto fail = [&](int rc) {
    ms_view_free(g);
    return rc;
  };
  auto dalloc = [&](int32_t** p, int64_t count) -> int {
    const hipError_t e = hipMalloc((void**)p, sizeof(int32_t) * std::max<int64_t>(count, 1));
    if (e == hipSuccess) return DAWN_OK;
    *p = nullptr;
    set_hip_error(e, "hipMalloc", __FILE__, __LINE__);
    return e == hipErrorOutOfMemory ? DAWN_ERR_OUT_OF_MEMORY : DAWN_ERR_HIP;
  };
  DevBuf<int32_t> inv;
  int rc;
  if ((rc = dalloc(&view->perm, n)) || (rc = inv.alloc((size_t)n)) ||
      (rc = hub_order_device(g, k, view->perm, inv.p)))
    return fail(rc);
  view->h_perm.resize(n);
  auto relabel = [&](const int32_t* old_rp, const int32_t* old_col, int32_t** rp_out,
                     int32_t** col_out) -> int {
    DAWN_TRY(dalloc(rp_out, (int64_t)n + 1));
    DAWN_TRY(dalloc(col_out, g->m));
    DAWN_TRY(permuted_offsets_device(old_rp, inv.p, n, g->stream, *rp_out));
    view_copy_kernel<<<2048, kBlock, 0, g->stream>>>(n, k, old_rp, old_col, *rp_out, *col_out, inv.p,
                                                     view->perm);
    DAWN_HIP(hipGetLastError());
    return DAWN_OK;
  };
  rc = relabel(g->row_ptr, g->col, &view->row_ptr, &view->col);
  if (!rc && g->directed) rc = relabel(g->in_row_ptr, g->in_col, &view->in_row_ptr, &view->in_col);
  if (!rc && (hipMemcpyAsync(view->h_perm.data(), view->perm, sizeof(int32_t) * (size_t)n,
                             hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
              hipStreamSynchronize(g->stream) != hipSuccess))
    rc = DAWN_ERR_HIP;
  if (rc) return fail(rc);
  if (!g->directed) {
    view->in_row_ptr = view->row_ptr;
    view->in_col = view->col;
  }
  const int heavy = g->knobs.heavy_degree, chunk = g->knobs.pull_chunk;
  if ((rc = chunk_list_device(view->in_row_ptr, n, heavy, chunk, g->stream, &view->hc_v, &view->hc_beg,
                              &view->hc_end, &view->num_hc, &view->num_hv, nullptr)))
    return fail(rc);
  if (g->directed) {
    int64_t num_ov = 0;
    if ((rc = chunk_list_device(view->row_ptr, n, heavy, chunk, g->stream, &view->oc_v, &view->oc_beg,
                                &view->oc_end, &view->num_oc, &num_ov, nullptr)))
      return fail(rc);
  } else {
    view->oc_v = view->hc_v;
    view->oc_beg = view->hc_beg;
    view->oc_end = view->hc_end;
    view->num_oc = view->num_hc;
  }
  return DAWN_OK;
}

}  // namespace dawn
