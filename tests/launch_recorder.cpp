// The HIP runtime calls of libbbhx_hip.so, recorded instead of made: loaded with
// RTLD_GLOBAL before the library, in a process of its own, these definitions take the
// place of the runtime's, so that a host without a GPU can look at the grids of its
// launches. Device memory is host memory, of which pages are there once written.

#include <sys/mman.h>

#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

struct dim3 {
    unsigned x, y, z;
};

namespace {

struct Launch {
    int kernel;
    dim3 grid, block;
    int64_t arg[32];  // 8 bytes at each of the first arguments, if they were asked for
};

struct State {
    std::vector<std::pair<const void*, std::string>> kernels;
    std::vector<Launch> launches;
    std::string args_of;  // kernel (a part of its name) whose first nargs arguments are kept
    int nargs = 0;
};

State& state()
{
    static State s;
    return s;
}

dim3 g_grid, g_block;
size_t g_shared;
void* g_stream;

int take(void** p, size_t bytes)
{
    *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return *p == MAP_FAILED ? 2 : 0;
}

}  // namespace

extern "C" {

// what the tests ask for
void recorder_clear(const char* args_of, int nargs)
{
    state().launches.clear();
    state().args_of = args_of;
    state().nargs = nargs;
}
int recorder_count() { return (int)state().launches.size(); }
const char* recorder_kernel(int i) { return state().kernels[state().launches[i].kernel].second.c_str(); }
void recorder_grid(int i, uint64_t* out)
{
    const Launch& l = state().launches[i];
    const unsigned v[6] = {l.grid.x, l.grid.y, l.grid.z, l.block.x, l.block.y, l.block.z};
    for (int k = 0; k < 6; k++) out[k] = v[k];
}
int64_t recorder_arg(int i, int k) { return state().launches[i].arg[k]; }

// what the library calls
void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    state().kernels.emplace_back(host, name);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, void* stream)
{
    g_grid = grid;
    g_block = block;
    g_shared = shared;
    g_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, void** stream)
{
    *grid = g_grid;
    *block = g_block;
    *shared = g_shared;
    *stream = g_stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, void*)
{
    Launch l{};
    l.kernel = -1;
    for (size_t k = 0; k < state().kernels.size(); k++)
        if (state().kernels[k].first == f) l.kernel = (int)k;
    if (l.kernel < 0) return 1;
    l.grid = grid;
    l.block = block;
    if (state().kernels[l.kernel].second.find(state().args_of) != std::string::npos)
        for (int k = 0; k < state().nargs && k < 32; k++) std::memcpy(&l.arg[k], args[k], 8);
    state().launches.push_back(l);
    return 0;
}
int hipGetLastError() { return 0; }
int hipMalloc(void** p, size_t bytes) { return take(p, bytes); }
int hipFree(void*) { return 0; }
int hipMemcpy(void* to, const void* from, size_t bytes, int)
{
    std::memcpy(to, from, bytes);
    return 0;
}
int hipMemcpyAsync(void* to, const void* from, size_t bytes, int kind, void*) { return hipMemcpy(to, from, bytes, kind); }
int hipGetSymbolAddress(void** p, const void*) { return take(p, size_t(1) << 30); }
int hipGetDevice(int* d)
{
    *d = 0;
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return take(s, 1); }
int hipStreamIsCapturing(void*, int* status)
{
    *status = 0;
    return 0;
}
int hipEventCreate(void** e) { return take(e, 1); }
int hipEventCreateWithFlags(void** e, unsigned) { return take(e, 1); }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*)
{
    *ms = 0.0f;
    return 0;
}

}
