// A HIP runtime without a GPU, for tests of the library's host code on the CPU.
//
// Loaded (RTLD_GLOBAL) before libclm_hip.so, whose runtime calls then resolve here.  Device memory
// is host memory that remembers its device; kernels are logged by name and do not run, but for the
// two that clear words and the one that reads words back, so that status words are what a test
// plants (fake_plant).  Anything that reaches memory or a stream of another device than it should
// is counted (fake_misplaced).
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Block {
    size_t bytes;
    int device;
};
struct Plant {
    std::string kernel;
    int arg;
    uint32_t word;
};
struct Launch {
    std::string kernel;
    std::vector<void *> words;  // of the watched argument
};

int g_devices = 1, g_device = 0, g_misplaced = 0;
bool g_capturing = false;
size_t g_allocated = 0;
std::map<char *, Block> g_blocks;
std::map<hipStream_t, int> g_streams;
std::map<const void *, std::string> g_names;
std::vector<Plant> g_plants;
std::vector<Launch> g_log;
std::vector<Plant> g_watches;  // (word: how many words of the argument)
struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} g_call;

int device_of(const void *p) {
    auto it = g_blocks.upper_bound((char *)p);
    if (it == g_blocks.begin()) return -1;
    --it;
    return (char *)p < it->first + it->second.bytes ? it->second.device : -1;
}
int stream_device(hipStream_t s) {
    auto it = g_streams.find(s);
    return it == g_streams.end() ? -1 : it->second;
}
void check(hipStream_t s, const void *p) {
    const int d = device_of(p), e = stream_device(s);
    if (d >= 0 && e >= 0 && d != e) ++g_misplaced;
}

}  // namespace

extern "C" {

// -- what a test asks -----------------------------------------------------------------
void fake_devices(int n) { g_devices = n; }
int fake_misplaced() { return g_misplaced; }
size_t fake_allocated() { return g_allocated; }
void fake_plant(const char *kernel, int arg, uint32_t word) { g_plants.push_back({kernel, arg, word}); }
void fake_watch(const char *kernel, int arg, int words) {
    g_watches.push_back({kernel, arg, (uint32_t)words});
}
void fake_clear_log() { g_log.clear(); }
int fake_launches() { return (int)g_log.size(); }
const char *fake_launch(int k) { return g_log[k].kernel.c_str(); }
void *fake_word(int k, int w) { return w < (int)g_log[k].words.size() ? g_log[k].words[w] : nullptr; }

// -- the runtime ------------------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_call = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = g_call.grid;
    *block = g_call.block;
    *shared = g_call.shared;
    *stream = g_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t stream) {
    const std::string &name = g_names[f];
    if (stream_device(stream) >= 0 && stream_device(stream) != g_device) ++g_misplaced;
    Launch l{name, {}};
    for (const Plant &w : g_watches)
        if (name.find(w.kernel) != std::string::npos) {
            l.words.resize(w.word);
            std::memcpy(l.words.data(), args[w.arg], sizeof(void *) * w.word);
        }
    g_log.push_back(l);
    if (g_capturing) return hipSuccess;
    if (name.find("k_fill_multi") != std::string::npos) {
        struct List {
            int *p[8];
            int n[8];
            int count;
        } list;
        std::memcpy(&list, args[0], sizeof(list));
        for (int k = 0; k < list.count; ++k) {
            check(stream, list.p[k]);
            std::memset(list.p[k], 0, sizeof(int) * (size_t)list.n[k]);
        }
    } else if (name.find("k_fill_int") != std::string::npos) {
        int *p = *(int **)args[0];
        check(stream, p);
        for (int k = 0; k < *(int *)args[1]; ++k) p[k] = *(int *)args[2];
    } else if (name.find("k_read_back") != std::string::npos) {
        struct List {
            const uint32_t *p[4];
            int n[4];
            int count;
        } list;
        std::memcpy(&list, args[0], sizeof(list));
        uint32_t *dst = *(uint32_t **)args[1];
        for (int k = 0; k < list.count; dst += list.n[k++])
            if (list.n[k]) {
                check(stream, list.p[k]);
                std::memcpy(dst, list.p[k], sizeof(uint32_t) * list.n[k]);
            }
    }
    for (size_t k = 0; k < g_plants.size(); ++k)
        if (name.find(g_plants[k].kernel) != std::string::npos) {
            **(uint32_t **)args[g_plants[k].arg] |= g_plants[k].word;
            g_plants.erase(g_plants.begin() + k);
            break;
        }
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
    *n = g_devices;
    return hipSuccess;
}
hipError_t hipSetDevice(int device) {
    if (device < 0 || device >= g_devices) return hipErrorInvalidDevice;
    g_device = device;
    return hipSuccess;
}
hipError_t hipGetDevice(int *device) {
    *device = g_device;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeWarpSize ? 64 : 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes) {
    *p = std::calloc(bytes, 1);  // (untouched pages take no memory)
    if (!*p) return hipErrorOutOfMemory;
    g_blocks[(char *)*p] = {bytes, g_device};
    g_allocated += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    auto it = g_blocks.find((char *)p);
    if (it == g_blocks.end()) return hipErrorInvalidValue;
    g_allocated -= it->second.bytes;
    g_blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = std::calloc(bytes, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t stream) {
    check(stream, dst);
    check(stream, src);
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int v, size_t bytes, hipStream_t stream) {
    check(stream, dst);
    std::memset(dst, v, bytes);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)std::malloc(1);
    g_streams[*s] = g_device;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    g_streams.erase(s);
    std::free((void *)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t s) { return stream_device(s); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    g_capturing = false;
    *g = (hipGraph_t)&g_call;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t)&g_call;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    g_log.push_back({"graph", {}});
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)&g_call;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 20;
    return hipSuccess;
}

}  // extern "C"
