// Where a launcher puts its kernel: on a stream, as a node into a HIP graph, or
// as new arguments into a node of an instantiated one.
#pragma once
#include <hip/hip_runtime.h>

namespace qf {

struct LaunchTo {
    hipStream_t stream = nullptr;
    // building: a new node follows deps, becomes `node`, and the next one through
    // the same target follows it (a class of two kernels runs them in order, as on
    // a stream)
    hipGraph_t graph = nullptr;
    const hipGraphNode_t* deps = nullptr;
    int ndeps = 0;
    hipGraphExec_t exec = nullptr;          // updating: `node` of this graph takes the new arguments
    hipGraphNode_t node = nullptr;
    hipError_t err = hipSuccess;            // of building and updating: the first one

    LaunchTo(hipStream_t s) : stream(s) {}
    LaunchTo(hipGraph_t g, const hipGraphNode_t* after, int n) : graph(g), deps(after), ndeps(n) {}
    LaunchTo(hipGraphExec_t x, hipGraphNode_t n) : exec(x), node(n) {}
    LaunchTo(const LaunchTo&) = delete;     // deps may point to `node`
    LaunchTo& operator=(const LaunchTo&) = delete;

    template <class... Params, class... Args>
    void operator()(void (*kernel)(Params...), dim3 grid, dim3 block, size_t lds, const Args&... args)
    {
        if (!graph && !exec)
            hipLaunchKernelGGL(kernel, grid, block, (unsigned)lds, stream, Params(args)...);
        else
            node_of(kernel, grid, block, lds, Params(args)...);
    }

private:
    template <class... Params>
    void node_of(void (*kernel)(Params...), dim3 grid, dim3 block, size_t lds, Params... params)
    {
        if (err != hipSuccess) return;
        void* list[] = {(void*)&params...};
        hipKernelNodeParams p{};
        p.func = (void*)kernel;
        p.gridDim = grid;
        p.blockDim = block;
        p.sharedMemBytes = (unsigned)lds;
        p.kernelParams = list;
        if (exec) {
            err = hipGraphExecKernelNodeSetParams(exec, node, &p);
            return;
        }
        hipGraphNode_t added = nullptr;
        err = hipGraphAddKernelNode(&added, graph, ndeps ? deps : nullptr, ndeps, &p);
        if (err != hipSuccess) return;
        node = added;
        deps = &node;
        ndeps = 1;
    }
};

}  // namespace qf
