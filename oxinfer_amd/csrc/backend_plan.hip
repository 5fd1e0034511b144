// A recorded run of device-pointer ops that replays with one call: the matmul side of the reference's DecodePlan
// (src/gpu_decode.rs:572-587; the CUDA backend builds a fixed launch list per graph once and re-issues it every token,
// src/cuda_decode.rs:1044-1049). Here the list is a HIP graph captured from the library's own launches: between
// oxhip_plan_begin and oxhip_plan_end every oxhip_dev_* call on the plan's stream is recorded instead of run, and
// oxhip_plan_replay submits all of them at once, so a token pays one host call for its whole chain of launches.
//
// What makes the library's launches recordable: nothing in a warmed call allocates, frees, synchronizes or clears memory
// with a memset (arrival counters return to zero inside the kernels that use them; the few clears there are go through a
// fill kernel). Scratch that grows on first use (a stream's K-slice rows, an MoE layer's pass buffers, packed GEMM
// activations) must exist before recording starts: run the chain once on the same stream first. A call that would have to
// allocate while recording fails the recording (oxhip_plan_end reports it), and nothing is replayable then.
//
// A short plan of the library's own kernels is replayed launch by launch, from the list that the finished graph holds: the submission
// of a graph costs the stream 5 us of its own, 8 behind an ordinary launch, where a launch from the list costs the device what a
// graph's node does and the host 2.45 us, which it has while the kernels before it run. See DIRECT_MAX.
#include <dlfcn.h>

#include <unordered_map>

#include "backend.hpp"

using namespace oxhip;

struct oxhip_plan {
    oxhip_ctx* ctx = nullptr;
    hipStream_t stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool recording = false;
    size_t nodes = 0;
    uint64_t streamed0 = 0;  // the stream's count of weight bytes when the recording began
    std::vector<hipKernelNodeParams> direct;  // the launches in order (arguments live in `graph`); empty: the graph is submitted
};

// The longest plan that goes out launch by launch, and the weight bytes per launch that it has to stream at least. 16 kernels of
// 8 us (4, 2): 148.7 us as a graph, 143.6 this way (84.7, 79.7; 54.1, 47.9), behind a copy kernel 153.0 and 145.3; two Q4_K_M
// layers at one token 114.2 -> 106.5 us, one layer of 1536 / 4096 in MLX 4-bit 36.8 -> 31.5, three of them 92.1 -> 92.5. The gain
// does not grow with the plan, while the host's share does, so longer plans stay one submission. A chain with hardly any matrix
// in it would be bound by the host (24 quantizations: 48.6 us as a graph, 55.3 this way), so it stays one too.
constexpr size_t DIRECT_MAX = 24;
constexpr uint64_t DIRECT_BYTES = 1 << 20;

static uint64_t streamed_on(oxhip_ctx* c, hipStream_t s) {
    std::lock_guard<std::mutex> lk(c->smu);
    auto it = c->per_stream.find(s);
    return it == c->per_stream.end() ? 0 : it->second->streamed.load();
}

// Whether a kernel is this library's (its symbol lies in the library's own image). The caller's are left to the graph: a node does not
// tell everything that its launch asked for (a cooperative kernel's reads as an ordinary one, which could never pass its grid barrier).
static bool own_kernel(const void* symbol) {
    Dl_info k{}, here{};
    return dladdr(symbol, &k) && dladdr(reinterpret_cast<const void*>(&oxhip_plan_begin), &here) && k.dli_fbase == here.dli_fbase;
}

// The launches of a graph that is one chain of this library's kernels; empty for any other graph.
static std::vector<hipKernelNodeParams> chain_of(hipGraph_t g) {
    size_t n = 0, ne = 0;
    if (hipGraphGetNodes(g, nullptr, &n) != hipSuccess || !n || n > DIRECT_MAX || hipGraphGetEdges(g, nullptr, nullptr, &ne) != hipSuccess || ne != n - 1) return {};
    std::vector<hipGraphNode_t> nodes(n), from(ne + 1), to(ne + 1);
    if (hipGraphGetNodes(g, nodes.data(), &n) != hipSuccess || (ne && hipGraphGetEdges(g, from.data(), to.data(), &ne) != hipSuccess)) return {};
    std::unordered_map<hipGraphNode_t, hipGraphNode_t> next;
    std::set<hipGraphNode_t> entered;
    for (size_t i = 0; i < ne; i++)
        if (!next.emplace(from[i], to[i]).second || !entered.insert(to[i]).second) return {};
    hipGraphNode_t at = nullptr;
    for (hipGraphNode_t v : nodes)
        if (!entered.count(v)) at = v;  // (n - 1 edges, each into a node of its own: one start)
    std::vector<hipKernelNodeParams> out;
    while (at && out.size() < n) {
        hipGraphNodeType type;
        hipKernelNodeParams k{};
        if (hipGraphNodeGetType(at, &type) != hipSuccess || type != hipGraphNodeTypeKernel || hipGraphKernelNodeGetParams(at, &k) != hipSuccess || !k.func ||
            !own_kernel(k.func) || !k.kernelParams || k.extra) {
            (void)hipGetLastError();
            return {};
        }
        out.push_back(k);
        auto it = next.find(at);
        at = it == next.end() ? nullptr : it->second;
    }
    if (out.size() != n) out.clear();
    return out;
}

extern "C" {

oxhip_plan* oxhip_plan_begin(oxhip_ctx* c, void* stream) {
    if (!c || !stream) {
        set_error("plan_begin: needs a context and a stream of its own (not the null stream)");
        return nullptr;
    }
    if (hipSetDevice(c->device) != hipSuccess) {
        set_error("plan_begin: hipSetDevice failed");
        return nullptr;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    // thread-local mode: other threads of the process may go on allocating while this one records
    hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) {
        set_error(std::string("plan_begin: hipStreamBeginCapture: ") + hipGetErrorString(e));
        return nullptr;
    }
    {
        std::lock_guard<std::mutex> lk(c->smu);
        c->record_failed.erase(s);
    }
    auto* p = new oxhip_plan();
    p->streamed0 = streamed_on(c, s);
    p->ctx = c;
    p->stream = s;
    p->recording = true;
    return p;
}

int oxhip_plan_end(oxhip_plan* p) {
    if (!p || !p->recording) {
        set_error("plan_end: no recording in progress");
        return 0;
    }
    p->recording = false;
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(p->stream, &g);
    bool refused;
    {
        std::lock_guard<std::mutex> lk(p->ctx->smu);
        refused = p->ctx->record_failed.erase(p->stream) != 0;
    }
    if (refused) {  // a recorded call declined because it would have had to allocate: its launches are missing from the graph
        if (g) (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        set_error("plan_end: a recorded call needed scratch that did not exist yet (run the chain once on this stream before recording)");
        return 0;
    }
    if (e != hipSuccess || !g) {
        (void)hipGetLastError();
        set_error(std::string("plan_end: the recording was invalidated (a recorded call allocated, synchronized or failed): ") + hipGetErrorString(e));
        return 0;
    }
    size_t n = 0;
    (void)hipGraphGetNodes(g, nullptr, &n);
    if (!n) {
        (void)hipGraphDestroy(g);
        set_error("plan_end: nothing was recorded on the plan's stream");
        return 0;
    }
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        set_error(std::string("plan_end: hipGraphInstantiate: ") + hipGetErrorString(e));
        return 0;
    }
    p->graph = g;
    p->exec = x;
    p->nodes = n;
    if (streamed_on(p->ctx, p->stream) - p->streamed0 >= n * DIRECT_BYTES) p->direct = chain_of(g);
    return 1;
}

size_t oxhip_plan_launches(const oxhip_plan* p) { return p ? p->nodes : 0; }

int oxhip_plan_one_by_one(const oxhip_plan* p) { return p && !p->direct.empty(); }

int oxhip_plan_replay(oxhip_plan* p, void* stream) {
    if (!p || !p->exec) {
        set_error("plan_replay: the plan holds no finished recording");
        return 0;
    }
    HIP_TRY(hipSetDevice(p->ctx->device), "hipSetDevice");
    hipStream_t s = stream ? static_cast<hipStream_t>(stream) : p->stream;
    std::lock_guard<std::mutex> lk(p->ctx->replay_mu);  // whichever way they go out: a submission would split another plan's launches
    if (p->direct.empty() || stream_recording(s)) {  // (into a recording: as ever)
        HIP_TRY(hipGraphLaunch(p->exec, s), "plan_replay: hipGraphLaunch");
        return 1;
    }
    for (size_t i = 0; i < p->direct.size(); i++) {
        const hipKernelNodeParams& k = p->direct[i];
        const hipError_t e = hipLaunchKernel(k.func, k.gridDim, k.blockDim, k.kernelParams, k.sharedMemBytes, s);
        if (e != hipSuccess) {
            set_error("plan_replay: launch " + std::to_string(i + 1) + " of " + std::to_string(p->direct.size()) + ": " + hipGetErrorString(e));
            return 0;
        }
    }
    return 1;
}

void oxhip_plan_free(oxhip_plan* p) {
    if (!p) return;
    if (p->ctx) (void)hipSetDevice(p->ctx->device);
    if (p->recording) {  // abandon the recording
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(p->stream, &g);
        if (g) (void)hipGraphDestroy(g);
        (void)hipGetLastError();
    }
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    delete p;
}

}  // extern "C"
