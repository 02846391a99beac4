// ML::HIP driver layer: thin C wrappers over the HIP runtime/module API, one per function the
// reference binds from libcuda (src/ml/cuda/driver.cr:20-50). See include/ml_hip_driver.h.
#include "ml_hip_driver.h"

#include "internal.h"

#include <hip/hip_runtime_api.h>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

// ---- graphs of a few kernels in a row ----------------------------------------------------------------------------------
// hipGraphLaunch takes 16 us of host time whatever is in the graph, and leaves the device idle for 5 us between one graph and the
// next; a plain launch takes 2.8 and leaves less than 1 (graphs of empty kernels, one to four of them, back to back: 16.2 to 18.4 us; one
// kernel of 22.6 us 27.7, two 50.3). A decode step of one runner is two to four kernels one after the other, so a graph that is a chain
// of up to CHAIN_MOST of this library's kernels and nothing else is launched as those kernels. Anything else - longer chains (a step of many layers captured as
// one graph, whose one idle gap is a small part of it), other nodes, branches, other modules' kernels, instantiation flags - goes through hipGraphLaunch.
// Two launches of one executable on two streams are not ordered by hipGraphLaunch either (graphs of two kernels of 8.7 ms on one workgroup, one executable on two
// streams 18.0 ms, on one stream twice 34.7).
namespace {
constexpr size_t CHAIN_MOST = 5;   // 14 us of launches
struct Chain {
  hipGraph_t graph = nullptr;   // a copy of the program's graph: the parameters below are its
  std::vector<hipKernelNodeParams> kernels;
  ~Chain() {
    if (graph) (void)hipGraphDestroy(graph);
  }
};
std::mutex g_chain_mu;
std::unordered_map<void*, std::shared_ptr<const Chain>> g_chains;   // by executable graph, until that is destroyed
std::unordered_map<void*, std::shared_ptr<std::mutex>> g_launching;   // by stream, while a graph is being launched on it

// Held while a graph is launched: a chain's kernels follow each other whole among the graphs that several threads launch on one stream, as single enqueues
// would. A mutex for each stream, so that a launch that waits for room in its queue holds up no other stream's.
class StreamLock {
 public:
  explicit StreamLock(void* stream) : stream_(stream) {
    {
      std::lock_guard<std::mutex> lk(g_chain_mu);
      std::shared_ptr<std::mutex>& m = g_launching[stream];
      if (!m) m = std::make_shared<std::mutex>();
      mutex_ = m;
    }
    mutex_->lock();
  }
  ~StreamLock() {
    mutex_->unlock();
    std::lock_guard<std::mutex> lk(g_chain_mu);
    if (mutex_.use_count() == 2) g_launching.erase(stream_);   // the table's and this one: nobody else waits
  }
  StreamLock(const StreamLock&) = delete;
  StreamLock& operator=(const StreamLock&) = delete;

 private:
  void* stream_;
  std::shared_ptr<std::mutex> mutex_;
};

// The chain a graph is, or null.
std::shared_ptr<const Chain> chain_of(hipGraph_t graph) {
  auto c = std::make_shared<Chain>();
  size_t n = 0, edges = 0;
  if (hipGraphGetNodes(graph, nullptr, &n) != hipSuccess || n == 0 || n > CHAIN_MOST) return nullptr;
  if (hipGraphClone(&c->graph, graph) != hipSuccess) {
    c->graph = nullptr;
    return nullptr;
  }
  std::vector<hipGraphNode_t> nodes(n);
  if (hipGraphGetNodes(c->graph, nodes.data(), &n) != hipSuccess || n != nodes.size()) return nullptr;
  if (hipGraphGetEdges(c->graph, nullptr, nullptr, &edges) != hipSuccess || edges != n - 1) return nullptr;
  std::vector<hipGraphNode_t> from(n), to(n);
  if (edges && (hipGraphGetEdges(c->graph, from.data(), to.data(), &edges) != hipSuccess || edges != n - 1)) return nullptr;
  from.resize(edges);
  to.resize(edges);
  auto count = [](const std::vector<hipGraphNode_t>& v, hipGraphNode_t x) {
    size_t k = 0;
    for (hipGraphNode_t y : v) k += y == x;
    return k;
  };
  hipGraphNode_t at = nullptr;
  for (hipGraphNode_t x : nodes) {
    if (count(from, x) > 1 || count(to, x) > 1) return nullptr;
    if (count(to, x) == 0) at = x;   // n - 1 edges, at most one into and out of a node: one start, or a circle beside it
  }
  for (size_t k = 0; k < n; k++) {
    hipGraphNodeType type;
    hipKernelNodeParams p = {};
    if (!at || hipGraphNodeGetType(at, &type) != hipSuccess || type != hipGraphNodeTypeKernel ||
        hipGraphKernelNodeGetParams(at, &p) != hipSuccess || !p.func || !p.kernelParams || p.extra || !cogni_internal_is_kernel(p.func))
      return nullptr;
    c->kernels.push_back(p);
    hipGraphNode_t next = nullptr;
    for (size_t e = 0; e < edges; e++)
      if (from[e] == at) next = to[e];
    at = next;
  }
  return at ? nullptr : c;
}
}   // namespace

extern "C" {

void cogni_internal_drop_chains(void) {
  std::unordered_map<void*, std::shared_ptr<const Chain>> gone;   // (destroyed outside the lock)
  std::lock_guard<std::mutex> lk(g_chain_mu);
  gone.swap(g_chains);
}

int mlhip_init(uint32_t flags) { return (int)hipInit(flags); }

int mlhip_device_get(int32_t* device, int32_t ordinal) {
  hipDevice_t d = 0;
  hipError_t e = hipDeviceGet(&d, ordinal);
  if (e == hipSuccess && device) *device = (int32_t)d;
  return (int)e;
}

int mlhip_device_get_name(char* name, int32_t len, int32_t device) {
  hipError_t e = hipDeviceGetName(name, len, (hipDevice_t)device);
  if (e == hipSuccess && name && len > 0 && name[0] == '\0') {   // some containers expose no marketing name
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) std::snprintf(name, (size_t)len, "AMD %s", prop.gcnArchName);
  }
  return (int)e;
}

int mlhip_device_compute_capability(int32_t* major, int32_t* minor, int32_t device) {
  int a = 0, b = 0;
  hipError_t e = hipDeviceComputeCapability(&a, &b, (hipDevice_t)device);
  if (e == hipSuccess) {
    if (major) *major = a;
    if (minor) *minor = b;
  }
  return (int)e;
}

int mlhip_device_get_arch(char* name, int32_t len, int32_t device) {
  if (!name || len <= 0) return (int)hipErrorInvalidValue;
  hipDeviceProp_t prop;
  hipError_t e = hipGetDeviceProperties(&prop, device);
  if (e != hipSuccess) return (int)e;
  std::strncpy(name, prop.gcnArchName, (size_t)len - 1);
  name[len - 1] = '\0';
  return 0;
}

int mlhip_device_get_cu_clock(int32_t* compute_units, int32_t* clock_khz, int32_t device) {
  int cu = 0, clk = 0;
  hipError_t e = hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) return (int)e;
  e = hipDeviceGetAttribute(&clk, hipDeviceAttributeClockRate, device);
  if (e != hipSuccess) return (int)e;
  if (compute_units) *compute_units = cu;
  if (clock_khz) *clock_khz = clk;
  return 0;
}

int mlhip_ctx_create(mlhip_context* ctx, uint32_t /*flags*/, int32_t device) {
  hipError_t e = hipSetDevice(device);
  if (e != hipSuccess) return (int)e;
  if (ctx) *ctx = reinterpret_cast<void*>((intptr_t)device + 1);  // non-null token for the primary context
  return 0;
}

int mlhip_ctx_destroy(mlhip_context /*ctx*/) { return 0; }

int mlhip_module_load_data(mlhip_module* mod, const void* image) {
  return (int)hipModuleLoadData(reinterpret_cast<hipModule_t*>(mod), image);
}

int mlhip_module_unload(mlhip_module mod) { return (int)hipModuleUnload((hipModule_t)mod); }

int mlhip_module_get_function(mlhip_function* fn, mlhip_module mod, const char* name) {
  return (int)hipModuleGetFunction(reinterpret_cast<hipFunction_t*>(fn), (hipModule_t)mod, name);
}

int mlhip_func_get_attribute(int32_t* value, int32_t attrib, mlhip_function fn) {
  int v = 0;
  hipError_t e = hipFuncGetAttribute(&v, (hipFunction_attribute)attrib, (hipFunction_t)fn);
  if (e == hipSuccess && value) *value = v;
  return (int)e;
}

int mlhip_stream_create(mlhip_stream* stream, uint32_t flags) {
  return (int)hipStreamCreateWithFlags(reinterpret_cast<hipStream_t*>(stream), flags);
}

int mlhip_stream_destroy(mlhip_stream stream) { return (int)hipStreamDestroy((hipStream_t)stream); }

int mlhip_stream_synchronize(mlhip_stream stream) { return (int)hipStreamSynchronize((hipStream_t)stream); }

int mlhip_stream_begin_capture(mlhip_stream stream, int32_t mode) {
  return (int)hipStreamBeginCapture((hipStream_t)stream, (hipStreamCaptureMode)mode);
}

int mlhip_stream_end_capture(mlhip_stream stream, mlhip_graph* graph) {
  return (int)hipStreamEndCapture((hipStream_t)stream, reinterpret_cast<hipGraph_t*>(graph));
}

int mlhip_graph_instantiate(mlhip_graph_exec* exec, mlhip_graph graph, uint64_t flags) {
  const hipError_t e = hipGraphInstantiateWithFlags(reinterpret_cast<hipGraphExec_t*>(exec), (hipGraph_t)graph, (unsigned long long)flags);
  if (e != hipSuccess) return (int)e;
  std::shared_ptr<const Chain> c = flags == 0 ? chain_of((hipGraph_t)graph) : nullptr;
  std::lock_guard<std::mutex> lk(g_chain_mu);
  if (c) g_chains[*exec] = std::move(c);
  else g_chains.erase(*exec);
  return 0;
}

int mlhip_graph_upload(mlhip_graph_exec exec, mlhip_stream stream) {
  return (int)hipGraphUpload((hipGraphExec_t)exec, (hipStream_t)stream);
}

int32_t mlhip_graph_exec_kernels(mlhip_graph_exec exec) {
  std::lock_guard<std::mutex> lk(g_chain_mu);
  const auto it = g_chains.find(exec);
  return it == g_chains.end() ? 0 : (int32_t)it->second->kernels.size();
}

int mlhip_graph_launch(mlhip_graph_exec exec, mlhip_stream stream) {
  const StreamLock whole(stream);
  std::shared_ptr<const Chain> c;
  {
    std::lock_guard<std::mutex> lk(g_chain_mu);
    if (auto it = g_chains.find(exec); it != g_chains.end()) c = it->second;
  }
  if (c) {
    for (const hipKernelNodeParams& k : c->kernels)
      if (hipError_t e = hipModuleLaunchKernel((hipFunction_t)k.func, k.gridDim.x, k.gridDim.y, k.gridDim.z, k.blockDim.x, k.blockDim.y, k.blockDim.z,
                                               k.sharedMemBytes, (hipStream_t)stream, k.kernelParams, nullptr);
          e != hipSuccess)
        return (int)e;
    return 0;
  }
  return (int)hipGraphLaunch((hipGraphExec_t)exec, (hipStream_t)stream);
}

int mlhip_graph_destroy(mlhip_graph graph) { return (int)hipGraphDestroy((hipGraph_t)graph); }

int mlhip_graph_exec_destroy(mlhip_graph_exec exec) {
  std::shared_ptr<const Chain> c;   // (destroyed outside the lock)
  {
    std::lock_guard<std::mutex> lk(g_chain_mu);
    if (auto it = g_chains.find(exec); it != g_chains.end()) {
      c = std::move(it->second);
      g_chains.erase(it);
    }
  }
  return (int)hipGraphExecDestroy((hipGraphExec_t)exec);
}

int mlhip_mem_alloc(mlhip_deviceptr* dptr, size_t bytesize) {
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytesize);
  if (e == hipSuccess && dptr) *dptr = (mlhip_deviceptr)(uintptr_t)p;
  return (int)e;
}

int mlhip_mem_free(mlhip_deviceptr dptr) { return (int)hipFree((void*)(uintptr_t)dptr); }

int mlhip_memcpy_htod(mlhip_deviceptr dst, const void* src, size_t bytesize) {
  return (int)hipMemcpyHtoD((hipDeviceptr_t)(uintptr_t)dst, const_cast<void*>(src), bytesize);
}

int mlhip_memcpy_dtoh(void* dst, mlhip_deviceptr src, size_t bytesize) {
  return (int)hipMemcpyDtoH(dst, (hipDeviceptr_t)(uintptr_t)src, bytesize);
}

int mlhip_memcpy_dtod(mlhip_deviceptr dst, mlhip_deviceptr src, size_t bytesize) {
  return (int)hipMemcpyDtoD((hipDeviceptr_t)(uintptr_t)dst, (hipDeviceptr_t)(uintptr_t)src, bytesize);
}

int mlhip_launch_kernel(mlhip_function fn, uint32_t grid_x, uint32_t grid_y, uint32_t grid_z, uint32_t block_x,
                        uint32_t block_y, uint32_t block_z, uint32_t shared_mem_bytes, mlhip_stream stream,
                        void** kernel_params, void** extra) {
  return (int)hipModuleLaunchKernel((hipFunction_t)fn, grid_x, grid_y, grid_z, block_x, block_y, block_z,
                                    shared_mem_bytes, (hipStream_t)stream, kernel_params, extra);
}

int mlhip_ctx_synchronize(void) { return (int)hipDeviceSynchronize(); }

int mlhip_event_create(mlhip_event* ev) { return (int)hipEventCreate(reinterpret_cast<hipEvent_t*>(ev)); }

int mlhip_event_record(mlhip_event ev, mlhip_stream stream) {
  return (int)hipEventRecord((hipEvent_t)ev, (hipStream_t)stream);
}

int mlhip_event_synchronize(mlhip_event ev) { return (int)hipEventSynchronize((hipEvent_t)ev); }

int mlhip_event_elapsed_ms(float* ms, mlhip_event start, mlhip_event stop) {
  return (int)hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop);
}

int mlhip_event_destroy(mlhip_event ev) { return (int)hipEventDestroy((hipEvent_t)ev); }

const char* mlhip_error_string(int code) { return hipGetErrorName((hipError_t)code); }

}  // extern "C"
