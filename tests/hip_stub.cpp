// Stand-in for the HIP runtime calls that libfem_amd makes, for tests of its host code without a GPU: device memory is
// host memory under a settable limit, kernels and streams do nothing. Load it with RTLD_GLOBAL before the library.
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {
std::mutex mu;
std::map<void *, size_t> blocks;
size_t used = 0, limit = size_t(1) << 40;
int lastError = 0, launches = 0, graphLaunches = 0, graphNodes = 0, graphs = 0;
struct Dim3 {
  unsigned x, y, z;
};
}  // namespace

extern "C" {

void stub_limit(size_t bytes) { limit = bytes; }
size_t stub_used() { return used; }
int stub_launches() { return launches; }             // kernels launched directly
int stub_graph_launches() { return graphLaunches; }  // graphs launched
int stub_graph_nodes() { return graphNodes; }        // kernel nodes recorded
int stub_graphs() { return graphs; }                 // executable graphs alive

int hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  if (used + n > limit) return lastError = 2;  // hipErrorOutOfMemory
  *p = std::calloc(n ? n : 1, 1);
  blocks[*p] = n;
  used += n;
  return 0;
}
int hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.find(p);
  if (it == blocks.end()) return p ? 1 : 0;
  used -= it->second;
  blocks.erase(it);
  std::free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(n ? n : 1, 1)) ? 0 : 2; }
int hipHostFree(void *p) { return std::free(p), 0; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return std::memcpy(d, s, n), 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return std::memcpy(d, s, n), 0; }
int hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *) { return std::memset(d, v, n), 0; }
int hipGetLastError() {
  const int e = lastError;
  return lastError = 0, e;
}
const char *hipGetErrorString(int e) { return e ? "error" : "no error"; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { return *s = &mu, 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamIsCapturing(void *, int *status) { return *status = 0, 0; }
int hipEventCreate(void **e) { return *e = &mu, 0; }
int hipEventCreateWithFlags(void **e, unsigned) { return *e = &mu, 0; }
int hipEventDestroy(void *) { return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventQuery(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1, 0; }
int hipLaunchKernel(const void *, Dim3, Dim3, void **, size_t, void *) { return launches++, 0; }
int hipGraphCreate(void **g, unsigned) { return *g = &mu, 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphAddKernelNode(void **n, void *, void *const *, size_t, const void *) { return *n = &mu, graphNodes++, 0; }
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) { return *e = &mu, graphs++, 0; }
int hipGraphLaunch(void *, void *) { return graphLaunches++, 0; }
int hipGraphExecDestroy(void *) { return graphs--, 0; }
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void *) { return 0; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *n, void **s) {
  *g = *b = Dim3{1, 1, 1};
  *n = 0;
  *s = nullptr;
  return 0;
}
}
