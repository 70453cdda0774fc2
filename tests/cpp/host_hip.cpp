// The part of the HIP runtime that this package's libraries call, on host memory and without a device: allocations are
// host allocations, copies and fills are done at once, a kernel launch is written to a log and computes nothing.  Tests
// load it in front of libespdl_dl.so / libespdl_hip.so (tests/host_hip.py), so that what the host side does around the
// launches - their order, their sizes, attributes, graphs, allocations - can be looked at without a GPU.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

struct Launch {
    const void *func;
    unsigned grid[3], block[3];
    unsigned lds;
    unsigned long long thread;
};

struct Node {
    hipKernelNodeParams params;
};

struct Graph {
    std::vector<Node *> nodes;
};

std::mutex g_mutex;
std::vector<Launch> g_log;
std::map<const void *, std::string> g_names;
std::map<const void *, int> g_lds_limit;
std::map<std::string, long> g_calls;
Graph *g_capture = nullptr;
std::atomic<int> g_delay_us{0};
void *g_no_params[1] = {nullptr};

thread_local dim3 t_grid, t_block;
thread_local size_t t_lds;
thread_local hipStream_t t_stream;

void called(const char *name)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    g_calls[name]++;
}

} // namespace

#define EXPORT extern "C" __attribute__((visibility("default")))

// --- what a test asks ---
EXPORT void host_hip_clear()
{
    std::lock_guard<std::mutex> lock(g_mutex);
    g_log.clear();
    g_calls.clear();
}
EXPORT void host_hip_delay(int us) { g_delay_us = us; }
EXPORT long host_hip_calls(const char *name)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    return g_calls[name];
}
EXPORT int host_hip_launches()
{
    std::lock_guard<std::mutex> lock(g_mutex);
    return (int)g_log.size();
}
// name of the kernel; sizes = grid x, y, z, block x, y, z, dynamic LDS bytes, LDS limit set for the kernel (0: never)
EXPORT const char *host_hip_launch(int i, unsigned *sizes, unsigned long long *thread)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    const Launch &l = g_log[(size_t)i];
    for (int k = 0; k < 3; k++) {
        sizes[k] = l.grid[k];
        sizes[3 + k] = l.block[k];
    }
    sizes[6] = l.lds;
    sizes[7] = (unsigned)(g_lds_limit.count(l.func) ? g_lds_limit[l.func] : 0);
    *thread = l.thread;
    return g_names[l.func].c_str();
}

// --- kernels ---
EXPORT void **__hipRegisterFatBinary(const void *) { return g_no_params; }
EXPORT void __hipUnregisterFatBinary(void **) {}
EXPORT void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
EXPORT void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, dim3 *, dim3 *, int *)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    g_names[host] = device;
}
EXPORT hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    t_grid = grid;
    t_block = block;
    t_lds = lds;
    t_stream = stream;
    return hipSuccess;
}
EXPORT hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream)
{
    *grid = t_grid;
    *block = t_block;
    *lds = t_lds;
    *stream = t_stream;
    return hipSuccess;
}
EXPORT hipError_t hipLaunchKernel(const void *func, dim3 grid, dim3 block, void **, size_t lds, hipStream_t)
{
    if (g_delay_us > 0)
        std::this_thread::sleep_for(std::chrono::microseconds(g_delay_us));
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_capture) {
        Node *node = new Node();
        node->params.func = const_cast<void *>(func);
        node->params.gridDim = grid;
        node->params.blockDim = block;
        node->params.sharedMemBytes = (unsigned)lds;
        node->params.kernelParams = g_no_params;
        g_capture->nodes.push_back(node);
        return hipSuccess;
    }
    g_log.push_back({func, {grid.x, grid.y, grid.z}, {block.x, block.y, block.z}, (unsigned)lds,
                     (unsigned long long)std::hash<std::thread::id>()(std::this_thread::get_id())});
    return hipSuccess;
}
EXPORT hipError_t hipFuncSetAttribute(const void *func, hipFuncAttribute attr, int value)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    if (attr == hipFuncAttributeMaxDynamicSharedMemorySize)
        g_lds_limit[func] = value;
    return hipSuccess;
}
EXPORT hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
    *n = 2;
    return hipSuccess;
}

// --- device ---
EXPORT hipError_t hipGetDevice(int *device)
{
    *device = 0;
    return hipSuccess;
}
EXPORT hipError_t hipDeviceGetAttribute(int *value, hipDeviceAttribute_t attr, int)
{
    *value = attr == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
    return hipSuccess;
}
EXPORT hipError_t hipGetLastError() { return hipSuccess; }
EXPORT const char *hipGetErrorString(hipError_t) { return "host"; }
EXPORT hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }

// --- memory ---
EXPORT hipError_t hipMalloc(void **p, size_t bytes)
{
    called("hipMalloc");
    *p = aligned_alloc(256, (bytes + 255) & ~(size_t)255);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
EXPORT hipError_t hipFree(void *p)
{
    free(p);
    return hipSuccess;
}
EXPORT hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    called("hipHostMalloc");
    *p = aligned_alloc(256, (bytes + 255) & ~(size_t)255);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
EXPORT hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
EXPORT hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind)
{
    memcpy(dst, src, bytes);
    return hipSuccess;
}
EXPORT hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    memcpy(dst, src, bytes);
    return hipSuccess;
}
EXPORT hipError_t hipMemcpy2DAsync(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t height,
                                   hipMemcpyKind, hipStream_t)
{
    for (size_t y = 0; y < height; y++)
        memcpy(static_cast<char *>(dst) + y * dpitch, static_cast<const char *>(src) + y * spitch, width);
    return hipSuccess;
}
EXPORT hipError_t hipMemset(void *dst, int value, size_t bytes)
{
    memset(dst, value, bytes);
    return hipSuccess;
}
EXPORT hipError_t hipMemsetAsync(void *dst, int value, size_t bytes, hipStream_t)
{
    memset(dst, value, bytes);
    return hipSuccess;
}
EXPORT hipError_t hipMemset2DAsync(void *dst, size_t pitch, int value, size_t width, size_t height, hipStream_t)
{
    for (size_t y = 0; y < height; y++)
        memset(static_cast<char *>(dst) + y * pitch, value, width);
    return hipSuccess;
}

// --- streams, events ---
EXPORT hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(new char);
    return hipSuccess;
}
EXPORT hipError_t hipStreamDestroy(hipStream_t s)
{
    delete reinterpret_cast<char *>(s);
    return hipSuccess;
}
EXPORT hipError_t hipStreamSynchronize(hipStream_t)
{
    called("hipStreamSynchronize");
    return hipSuccess;
}
EXPORT hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status)
{
    *status = g_capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
EXPORT hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = nullptr;
    return hipSuccess;
}
EXPORT hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
EXPORT hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
EXPORT hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}

// --- graphs: a capture is one chain of kernel nodes ---
EXPORT hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    g_capture = new Graph();
    return hipSuccess;
}
EXPORT hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *graph)
{
    *graph = reinterpret_cast<hipGraph_t>(g_capture);
    g_capture = nullptr;
    return hipSuccess;
}
EXPORT hipError_t hipGraphGetNodes(hipGraph_t graph, hipGraphNode_t *nodes, size_t *n)
{
    const Graph *g = reinterpret_cast<Graph *>(graph);
    for (size_t i = 0; nodes && i < g->nodes.size(); i++)
        nodes[i] = reinterpret_cast<hipGraphNode_t>(g->nodes[i]);
    *n = g->nodes.size();
    return hipSuccess;
}
EXPORT hipError_t hipGraphGetEdges(hipGraph_t graph, hipGraphNode_t *from, hipGraphNode_t *to, size_t *n)
{
    const Graph *g = reinterpret_cast<Graph *>(graph);
    *n = g->nodes.empty() ? 0 : g->nodes.size() - 1;
    for (size_t i = 0; from && i < *n; i++) {
        from[i] = reinterpret_cast<hipGraphNode_t>(g->nodes[i]);
        to[i] = reinterpret_cast<hipGraphNode_t>(g->nodes[i + 1]);
    }
    return hipSuccess;
}
EXPORT hipError_t hipGraphNodeGetType(hipGraphNode_t, hipGraphNodeType *type)
{
    *type = hipGraphNodeTypeKernel;
    return hipSuccess;
}
EXPORT hipError_t hipGraphKernelNodeGetParams(hipGraphNode_t node, hipKernelNodeParams *params)
{
    *params = reinterpret_cast<Node *>(node)->params;
    return hipSuccess;
}
EXPORT hipError_t hipGraphInstantiate(hipGraphExec_t *exec, hipGraph_t graph, hipGraphNode_t *, char *, size_t)
{
    called("hipGraphInstantiate");
    *exec = reinterpret_cast<hipGraphExec_t>(graph);
    return hipSuccess;
}
EXPORT hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    called("hipGraphLaunch");
    return hipSuccess;
}
EXPORT hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
EXPORT hipError_t hipGraphDestroy(hipGraph_t graph)
{
    Graph *g = reinterpret_cast<Graph *>(graph);
    for (Node *node : g->nodes)
        delete node;
    delete g;
    return hipSuccess;
}
