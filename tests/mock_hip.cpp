// Host-only stand-in for the HIP runtime calls of libquickfock.so: memory is
// malloc, kernels do nothing, and every kernel launch is recorded with the
// launches it waits for, through streams, events and graphs.  Tests load it in
// front of the real runtime (mock_hip.py) and check the order and the buffers
// of a build's launches without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {

struct Kernel {
    std::string name;
    std::vector<void*> args;   // the arguments that are pointers, by position (null: not read)
    dim3 grid;
};
struct Op {
    Kernel k;
    std::set<int> deps;        // earlier operations it waits for
};
struct Node {
    Kernel k;
    std::vector<int> deps;     // of the same graph
};
struct Graph {
    std::vector<Node> nodes;
};

std::map<const void*, std::string> names;
std::vector<Op> ops;
std::map<void*, std::set<int>> stream_last;   // what the next operation of a stream waits for
std::map<void*, std::set<int>> event_at;
std::map<void*, int> capturing;                // id of the capture a stream takes part in
std::map<void*, int> event_capture;
std::vector<void*> streams;                    // created and not destroyed
std::string text;
int execs = 0;             // instantiated graphs
hipError_t last_error = hipSuccess;
std::string fail_name;
int fail_after = -1, failed = 0;

// true where the test asked this call to fail
bool fails(const char* fn)
{
    if (fail_after < 0 || fail_name != fn) return false;
    if (fail_after-- > 0) return false;
    ++failed;
    last_error = hipErrorInvalidValue;
    return true;
}

Kernel kernel(const void* f, void** args, dim3 grid)
{
    Kernel k;
    k.name = names.count(f) ? names[f] : "?";
    k.grid = grid;
    // position of the global slot buffer, where the kernel has one
    const char* const fams[] = {"fock_coop_kernel", "fused_coop_kernel", "grad_coop_kernel", "fused_grad_coop_kernel"};
    const int at[] = {4, 5, 4, 5};
    int pos = -1;
    for (int x = 0; x < 4; ++x)
        if (k.name.find(fams[x]) != std::string::npos) pos = at[x];
    for (int x = 0; x <= pos; ++x) k.args.push_back(x == pos ? *(void**)args[x] : nullptr);
    return k;
}

struct Call {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
} call;

}  // namespace

#define MOCK extern "C" __attribute__((visibility("default")))
#define MAY_FAIL                                       \
    do {                                               \
        if (fails(__func__)) return hipErrorInvalidValue; \
    } while (0)

// ---- the test's side
MOCK void mock_clear() { ops.clear(); stream_last.clear(); event_at.clear(); }
// makes the call after `after` more of its name fail; how many have since
MOCK void mock_fail(const char* fn, int after)
{
    fail_name = fn;
    fail_after = after;
    failed = 0;
}
MOCK int mock_failed() { return failed; }
MOCK int mock_execs() { return execs; }
// begins capture `id` on a stream, or (0) ends the one it takes part in
MOCK void mock_capture(void* s, int id)
{
    if (id) {
        capturing[s] = id;
        return;
    }
    const int was = capturing.count(s) ? capturing[s] : 0;
    for (auto it = capturing.begin(); it != capturing.end();) it = it->second == was ? capturing.erase(it) : ++it;
}
MOCK int mock_streams() { return (int)streams.size(); }
// one line per launch: index, name, grid, slot buffer (0: none), indices it waits for
MOCK const char* mock_log()
{
    text.clear();
    for (size_t i = 0; i < ops.size(); ++i) {
        char b[64];
        std::snprintf(b, sizeof b, " %u %zu", ops[i].k.grid.x, ops[i].k.args.empty() ? (size_t)0 : (size_t)ops[i].k.args.back());
        text += std::to_string(i) + " " + ops[i].k.name + b;
        for (int d : ops[i].deps) text += " " + std::to_string(d);
        text += "\n";
    }
    return text.c_str();
}
// what the next operation of a stream would wait for
MOCK const char* mock_stream(void* s)
{
    text.clear();
    for (int d : stream_last[s]) text += std::to_string(d) + " ";
    return text.c_str();
}

// ---- kernels
MOCK void** __hipRegisterFatBinary(const void*)
{
    static void* module;
    return &module;
}
MOCK void __hipUnregisterFatBinary(void**) {}
MOCK void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    names[f] = name;
}
MOCK void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
MOCK hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    call = {g, b, lds, s};
    return hipSuccess;
}
MOCK hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s)
{
    *g = call.grid;
    *b = call.block;
    *lds = call.lds;
    *s = call.s;
    return hipSuccess;
}
MOCK hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s)
{
    MAY_FAIL;
    ops.push_back({kernel(f, args, grid), stream_last[s]});
    stream_last[s] = {(int)ops.size() - 1};
    return hipSuccess;
}

// ---- streams and events
MOCK hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    MAY_FAIL;
    *s = (hipStream_t) new char;
    streams.push_back(*s);
    return hipSuccess;
}
MOCK hipError_t hipStreamDestroy(hipStream_t s)
{
    for (size_t k = 0; k < streams.size(); ++k)
        if (streams[k] == s) streams.erase(streams.begin() + k--);
    delete (char*)s;
    return hipSuccess;
}
MOCK hipError_t hipStreamSynchronize(hipStream_t) { MAY_FAIL; return hipSuccess; }
MOCK hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st)
{
    *st = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
MOCK hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus* st, unsigned long long* id)
{
    hipStreamIsCapturing(s, st);
    if (id) *id = capturing.count(s) ? capturing[s] : 0;
    return hipSuccess;
}
MOCK hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
MOCK hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t) new Graph; return hipSuccess; }
MOCK hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    MAY_FAIL;
    *e = (hipEvent_t) new char;
    return hipSuccess;
}
MOCK hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
MOCK hipError_t hipEventDestroy(hipEvent_t e) { delete (char*)e; return hipSuccess; }
MOCK hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
MOCK hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
MOCK hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    MAY_FAIL;
    event_at[e] = stream_last[s];
    event_capture[e] = capturing.count(s) ? capturing[s] : 0;
    return hipSuccess;
}
MOCK hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    MAY_FAIL;
    // a stream outside takes part in a capture by its first wait; one of another capture, or a
    // captured one that waits for work outside it, is an error
    const int mine = capturing.count(s) ? capturing[s] : 0, theirs = event_capture[e];
    if (mine && mine != theirs) return last_error = hipErrorStreamCaptureIsolation;
    if (theirs) capturing[s] = theirs;
    stream_last[s].insert(event_at[e].begin(), event_at[e].end());
    return hipSuccess;
}

// ---- graphs
MOCK hipError_t hipGraphCreate(hipGraph_t* g, unsigned) { MAY_FAIL; *g = (hipGraph_t) new Graph; return hipSuccess; }
MOCK hipError_t hipGraphDestroy(hipGraph_t g) { delete (Graph*)g; return hipSuccess; }
MOCK hipError_t hipGraphAddKernelNode(hipGraphNode_t* out, hipGraph_t g, const hipGraphNode_t* deps, size_t n,
                                      const hipKernelNodeParams* p)
{
    MAY_FAIL;
    Graph& x = *(Graph*)g;
    Node node{kernel(p->func, p->kernelParams, p->gridDim), {}};
    for (size_t k = 0; k < n; ++k) node.deps.push_back((int)(size_t)deps[k] - 1);
    x.nodes.push_back(node);
    *out = (hipGraphNode_t)x.nodes.size();
    return hipSuccess;
}
MOCK hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    MAY_FAIL;
    *e = (hipGraphExec_t) new Graph(*(Graph*)g);
    ++execs;
    return hipSuccess;
}
MOCK hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
    delete (Graph*)e;
    --execs;
    return hipSuccess;
}
MOCK hipError_t hipGraphExecKernelNodeSetParams(hipGraphExec_t e, hipGraphNode_t n, const hipKernelNodeParams* p)
{
    MAY_FAIL;
    ((Graph*)e)->nodes[(size_t)n - 1].k = kernel(p->func, p->kernelParams, p->gridDim);
    return hipSuccess;
}
MOCK hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s)
{
    MAY_FAIL;
    const Graph& x = *(Graph*)e;
    const int base = (int)ops.size();
    const std::set<int> before = stream_last[s];
    std::set<int> all;
    for (const Node& n : x.nodes) {
        Op op{n.k, {}};
        for (int d : n.deps) op.deps.insert(base + d);
        if (n.deps.empty()) op.deps = before;
        all.insert((int)ops.size());
        ops.push_back(op);
    }
    if (!all.empty()) stream_last[s] = all;   // a stream goes on when the whole graph is done
    return hipSuccess;
}

// ---- memory, device, errors
std::map<void*, size_t> device;   // allocations not yet freed
MOCK hipError_t hipMalloc(void** p, size_t n)
{
    MAY_FAIL;
    *p = std::malloc(n ? n : 1);
    device[*p] = n;
    return hipSuccess;
}
MOCK hipError_t hipFree(void* p) { device.erase(p); std::free(p); return hipSuccess; }
MOCK long long mock_bytes()
{
    long long n = 0;
    for (auto& d : device) n += (long long)d.second;
    return n;
}
MOCK hipError_t hipHostMalloc(void** p, size_t n, unsigned) { MAY_FAIL; *p = std::malloc(n ? n : 1); return hipSuccess; }
MOCK hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
MOCK hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { MAY_FAIL; std::memcpy(to, from, n); return hipSuccess; }
MOCK hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(to, from, n, k); }
MOCK hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
MOCK hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = std::calloc(1, 64u << 20);
    *p = scratch;
    return hipSuccess;
}
MOCK hipError_t hipSetDevice(int) { return hipSuccess; }
MOCK hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
MOCK hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
MOCK hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 0; return hipSuccess; }
MOCK hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) { std::memset(p, 0, sizeof *p); return hipSuccess; }
MOCK hipError_t hipDeviceSynchronize() { MAY_FAIL; return hipSuccess; }
MOCK const char* hipGetErrorString(hipError_t) { return "mock"; }
MOCK hipError_t hipGetLastError()
{
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
