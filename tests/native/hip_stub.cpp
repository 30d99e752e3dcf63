// A HIP runtime for the host code of libqiw on the CPU: device memory is host memory, copies
// happen at once, and kernel launches are recorded instead of run.  Linked with the library's
// own objects (tests/hip_stub.py), so that what the host code launches, captures and replays
// can be checked without a GPU.  Freed device memory stays mapped and is never handed out
// again, so its addresses stay recognizable in a launch's arguments.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "qiw.h"
#include "qiw_device.h"

namespace {

struct Launch {
    std::string name;
    unsigned grid[3], block[3];
    size_t lds;
    std::string args;  // bytes of the kernel's first argument, of evaluators and bookkeeping
};
struct Graph {
    std::vector<Launch> launches;
};

std::map<const void *, std::string> g_names;
std::map<char *, std::pair<size_t, bool>> g_mem;  // block: bytes, freed
std::vector<Launch> g_run;                        // launches in stream order, replayed ones among them
Graph *g_capture = nullptr;
int g_captures = 0;
size_t g_live = 0, g_peak = 0, g_copies = 0;

size_t arg_bytes(const std::string &n) {
    auto has = [&](const char *s) { return n.find(s) != std::string::npos; };
    if (has("k_eval_arcs_t")) return sizeof(ArcArgs);
    if (has("k_eval_sarcs_t") || has("k_eval_flat_t")) return sizeof(EvalArgs);
    if (has("k_eval_vec_t")) return sizeof(VecArgs);
    if (has("k_eval_mfma_t")) return sizeof(MfmaArgs);
    if (has("k_eval_block")) return sizeof(BlockArgs);
    if (has("finalize_corr")) return sizeof(CorrFinalizeArgs);
    if (has("reduce_finalize")) return sizeof(FinalizeArgs);
    return 0;
}

struct Config {
    dim3 grid, block;
    size_t lds = 0;
    hipStream_t stream = nullptr;
};
Config g_config;

void *take(size_t bytes) {
    char *p = (char *)std::calloc(1, bytes ? bytes : 1);
    if (!p) return nullptr;
    g_mem[p] = {bytes, false};
    g_live += bytes;
    g_peak = g_live > g_peak ? g_live : g_peak;
    return p;
}
hipError_t give(void *q) {
    auto it = g_mem.find((char *)q);
    if (it == g_mem.end() || it->second.second) return hipErrorInvalidValue;
    it->second.second = true;
    g_live -= it->second.first;
    return hipSuccess;
}
// 0: inside a live block, 1: inside a freed one, 2: neither
int where(const char *p) {
    auto it = g_mem.upper_bound(const_cast<char *>(p));
    if (it == g_mem.begin()) return 2;
    --it;
    return p < it->first + it->second.first ? (it->second.second ? 1 : 0) : 2;
}

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    g_config.grid = grid;
    g_config.block = block;
    g_config.lds = lds;
    g_config.stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *st) {
    *grid = g_config.grid;
    *block = g_config.block;
    *lds = g_config.lds;
    *st = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t) {
    Launch l;
    l.name = g_names[f];
    l.grid[0] = grid.x, l.grid[1] = grid.y, l.grid[2] = grid.z;
    l.block[0] = block.x, l.block[1] = block.y, l.block[2] = block.z;
    l.lds = lds;
    if (const size_t n = arg_bytes(l.name)) l.args.assign((const char *)args[0], n);
    (g_capture ? g_capture->launches : g_run).push_back(l);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) { return (*p = take(bytes)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return p ? give(p) : hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    return (*p = std::calloc(1, bytes ? bytes : 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) {
    if (n) std::memcpy(to, from, n);
    ++g_copies;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
    if (n) std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *scratch = take(QIW_NOALLOC_SCRATCH_BYTES);
    *p = scratch;
    return scratch ? hipSuccess : hipErrorOutOfMemory;
}

hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error of the CPU runtime"; }
hipError_t hipStreamCreate(hipStream_t *s) {
    *s = (hipStream_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free((void *)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return g_capture ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free((void *)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capture = new Graph;
    ++g_captures;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = (hipGraph_t)g_capture;
    g_capture = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t) new Graph(*(Graph *)g);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    const Graph &g = *(Graph *)e;
    g_run.insert(g_run.end(), g.launches.begin(), g.launches.end());
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    delete (Graph *)e;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete (Graph *)g;
    return hipSuccess;
}

// ---- what the tests read ----
void stub_clear(void) {
    g_run.clear();
    g_captures = 0;
    g_copies = 0;
    g_peak = g_live;
}
int stub_captures(void) { return g_captures; }
size_t stub_copies(void) { return g_copies; }
size_t stub_peak_bytes(void) { return g_peak; }
int stub_launches(void) { return (int)g_run.size(); }
const char *stub_name(int i) { return g_run[i].name.c_str(); }
// grid x y z, block x y z, LDS bytes
void stub_shape(int i, int64_t *out) {
    const Launch &l = g_run[i];
    for (int k = 0; k < 3; ++k) out[k] = l.grid[k], out[3 + k] = l.block[k];
    out[6] = (int64_t)l.lds;
}
int stub_args(int i, const char **bytes) {
    *bytes = g_run[i].args.data();
    return (int)g_run[i].args.size();
}
// pointers in the arguments of launch i into device memory that has been freed
int stub_freed_args(int i) {
    const std::string &a = g_run[i].args;
    int n = 0;
    for (size_t o = 0; o + 8 <= a.size(); o += 8) {
        char *p;
        std::memcpy(&p, a.data() + o, 8);
        n += where(p) == 1;
    }
    return n;
}

}  // extern "C"
