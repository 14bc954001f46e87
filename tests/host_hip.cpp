// The library's host code on stand-ins for the HIP runtime: device memory is
// host memory, kernels are not run (their arguments can be looked at), and
// allocations can be made to fail from a chosen one on.  The definitions here
// come before the runtime's own, as the program is searched first.
//
//   host_hip list                 the operations
//   host_hip memory <operation>   from every allocation of the operation on,
//                                 memory is short: the call and the one after
//                                 it say so, the next one works, nothing leaks
//   host_hip managed              a traversal that lowers distances in its rows
//                                 is not given rows in managed memory
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "dawn_capi.h"

namespace {
long g_allocs = 0, g_fail_from = -1, g_failed = 0, g_live = 0;
hipError_t g_last = hipSuccess;  // kept until hipGetLastError, as the runtime does
std::map<const void*, size_t> g_blocks;
const void* g_managed = nullptr;  // a buffer of managed memory
long g_seen_managed = 0;          // launches of 1024 threads whose first argument holds its address

hipError_t give(void** p, size_t bytes) {
  if (g_fail_from >= 0 && g_allocs++ >= g_fail_from) {
    g_failed++;
    *p = nullptr;
    return g_last = hipErrorOutOfMemory;
  }
  *p = std::calloc(bytes ? bytes : 1, 1);
  g_blocks[*p] = bytes;
  g_live++;
  return hipSuccess;
}
hipError_t take(void* p) {
  if (!p) return hipSuccess;
  if (!g_blocks.erase(p)) std::abort();  // not allocated, or freed twice
  std::free(p);
  g_live--;
  return hipSuccess;
}
bool on_device(const void* p) {
  auto it = g_blocks.upper_bound(p);
  if (it == g_blocks.begin()) return false;
  --it;
  return (const char*)p < (const char*)it->first + (it->second ? it->second : 1);
}
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;
}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 100000;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipMalloc(void** p, size_t bytes) { return give(p, bytes); }
hipError_t hipFree(void* p) { return take(p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return give(p, bytes); }
hipError_t hipHostFree(void* p) { return take(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof *a);
  if (p && p == g_managed) a->type = hipMemoryTypeManaged;
  else if (on_device(p)) a->type = hipMemoryTypeDevice;
  else return g_last = hipErrorInvalidValue;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)8, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)8, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return *e = (hipGraphExec_t)8, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)8, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  return g_grid = g, g_block = b, g_shared = sh, g_stream = s, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
  return *g = g_grid, *b = g_block, *sh = g_shared, *s = g_stream, hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3 block, void** args, size_t, hipStream_t) {
  if (g_managed && block.x == 1024)  // their argument structs hold more than 128 bytes
    for (int i = 0; i < 128; i += 8) g_seen_managed += !std::memcmp((const char*)args[0] + i, &g_managed, 8);
  return hipSuccess;
}
}

namespace {
struct Ring {  // a ring of n vertices
  std::vector<int32_t> rp, col, w;
  dawn_csr csr{};
  Ring(int32_t n, bool weighted) {
    for (int32_t v = 0; v < n; v++) {
      rp.push_back(2 * v);
      col.insert(col.end(), {(v + n - 1) % n, (v + 1) % n});
      w.insert(w.end(), {3, 3});
    }
    rp.push_back(2 * n);
    csr.n = n;
    csr.m = 2 * (int64_t)n;
    csr.row_ptr = rp.data();
    csr.col = col.data();
    csr.weight = weighted ? w.data() : nullptr;
    csr.weighted = weighted;
  }
};

struct Op {
  int32_t n;
  bool weighted;
  std::function<int(dawn_graph*)> call;
};

int mssp(dawn_graph* g, int32_t n, int32_t count, int32_t policy, bool out) {
  std::vector<int32_t> src((size_t)count), rows(out ? (size_t)count * n : 0);
  for (int32_t i = 0; i < count; i++) src[i] = i % n;
  std::vector<int64_t> sums((size_t)count);
  return dawn_mssp(g, src.data(), count, out ? rows.data() : nullptr, sums.data(), policy, nullptr);
}

std::map<std::string, Op> ops() {
  auto one = [](bool w) {
    return [w](dawn_graph* g) {
      dawn_stats st{};
      std::vector<int32_t> d(300);
      return w ? dawn_sssp(g, 0, d.data(), DAWN_POLICY_FIXED, &st) : dawn_bfs(g, 0, d.data(), DAWN_POLICY_FIXED, &st);
    };
  };
  auto many = [](int32_t n, int32_t count, int32_t policy, bool out) {
    return [=](dawn_graph* g) { return mssp(g, n, count, policy, out); };
  };
  auto batch = [](dawn_graph* g) {
    const int32_t src[3] = {0, 1, 2};
    const int64_t at = 0;
    std::vector<int32_t> d(900);
    return dawn_batch_mssp(&g, 1, src, 3, d.data(), &at, nullptr);
  };
  return {
      {"bfs", {300, false, one(false)}},
      {"sssp", {300, true, one(true)}},
      {"weighted_lanes_8", {300, true, many(300, 5, DAWN_POLICY_PUSH, true)}},
      {"weighted_lanes_64", {300, true, many(300, 70, DAWN_POLICY_PUSH, true)}},
      {"weighted_workgroups", {300, true, many(300, 70, DAWN_POLICY_FIXED, true)}},
      {"lanes", {300, false, many(300, 130, DAWN_POLICY_PUSH, true)}},
      {"lanes_hub_order", {66000, false, many(66000, 3, DAWN_POLICY_PUSH, false)}},
      {"workgroups", {300, false, many(300, 70, DAWN_POLICY_FIXED, true)}},
      {"workgroups_no_rows", {300, false, many(300, 70, DAWN_POLICY_FIXED, false)}},
      {"batch", {300, false, batch}},
      {"batch_weighted", {300, true, batch}},
  };
}

int fail(const char* what, long k, int rc) {
  std::printf("allocation %ld: %s (status %d)\n", k, what, rc);
  return 1;
}

int memory(const Op& op) {
  const Ring r(op.n, op.weighted);
  int usual = 0;
  for (long k = -1;; k++) {
    const long before = g_live;
    dawn_graph* g = nullptr;
    g_fail_from = -1;
    if (dawn_graph_create(&r.csr, &g)) return fail("the graph", k, 0);
    if (k < 0) {
      usual = op.call(g);
      if (usual == DAWN_ERR_OUT_OF_MEMORY) return fail("out of memory without a shortage", k, usual);
    } else {
      g_allocs = g_failed = 0;
      g_fail_from = k;
      const int first = op.call(g);
      const bool hit = g_failed > 0;
      if (hit && first != DAWN_ERR_OUT_OF_MEMORY) return fail("the shortage is not reported", k, first);
      if (hit) {
        const int second = op.call(g);
        if (second != DAWN_ERR_OUT_OF_MEMORY) return fail("the second call passes over what is missing", k, second);
        g_fail_from = -1;
        const int third = op.call(g);
        if (third != usual) return fail("the call after the shortage differs", k, third);
      }
      if (!hit) {
        dawn_graph_destroy(g);
        std::printf("%ld allocations\n", k);
        return k > 0 ? 0 : 1;
      }
    }
    dawn_graph_destroy(g);
    if (g_live != before) return fail("memory is lost", k, (int)(g_live - before));
  }
}

// Weighted sources a workgroup each on more vertices than their distances fit
// the LDS for, as a call of their own and in a batch: the kernel lowers them in
// the rows by atomics.
int managed() {
  constexpr int32_t n = 40000, most = 65;
  const Ring r(n, true);
  dawn_graph* g = nullptr;
  if (dawn_graph_create(&r.csr, &g)) return 1;
  int bad = 0;
  for (const bool batch : {false, true}) {
    const int32_t count = batch ? 3 : most;
    const int64_t first = batch ? 5 : 0;  // a batch's rows may lie anywhere in the buffer
    std::vector<int32_t> src((size_t)count, 1), rows((size_t)(first + (int64_t)count * n), 7);
    g_managed = rows.data();
    g_seen_managed = 0;
    const int rc = batch ? dawn_batch_mssp(&g, 1, src.data(), count, rows.data(), &first, nullptr)
                         : dawn_mssp(g, src.data(), count, rows.data(), nullptr, DAWN_POLICY_FIXED, nullptr);
    g_managed = nullptr;
    std::printf("status %d, %ld launches hold the rows, entries %d %d\n", rc, g_seen_managed, rows[first], rows.back());
    // The kernels did not run: the entries are those of fresh memory.
    bad |= rc || g_seen_managed || rows[first] != 0 || rows.back() != 0 || (first && rows[first - 1] != 7);
  }
  dawn_graph_destroy(g);
  return bad;
}
}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "list") {
    for (const auto& o : ops()) std::printf("%s\n", o.first.c_str());
    return 0;
  }
  if (what == "memory" && argc > 2) return memory(ops().at(argv[2]));
  if (what == "managed") return managed();
  return 2;
}
