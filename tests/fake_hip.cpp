// fake_hip.cpp -- the HIP runtime calls of libgofann_hip.so, without a GPU.
//
// Loaded with RTLD_GLOBAL before the library, these definitions take the
// place of libamdhip64's: device memory is host memory under a settable
// limit, a kernel launch is recorded (name, grid, LDS, stream) and not run.
// So the host side of an entry point (placement, scratch, refusals) can be
// checked on a machine without a GPU.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string name;
    unsigned grid;
    size_t lds;
    const void* stream;
};

constexpr int kCus = 256;
constexpr size_t kLds = 160 * 1024;

std::map<const void*, std::string>& names()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::map<void*, size_t> g_blocks;
std::vector<Launch> g_launches;
size_t g_used = 0, g_limit = SIZE_MAX;
int g_waves = 16;                     // resident one-wave workgroups per CU by registers
const void* g_capturing = nullptr;    // the stream that is being captured
bool g_capture_broken = false;
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;

// What the runtime does with a call that a capture in global mode forbids.
bool forbidden()
{
    if (g_capturing == nullptr || g_mode == hipStreamCaptureModeRelaxed) return false;
    g_capture_broken = true;
    return true;
}
}  // namespace

extern "C" {

void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_used() { return g_used; }
void fake_waves(int waves) { g_waves = waves; }
void fake_capture(const void* stream)
{
    g_capturing = stream;
    g_capture_broken = false;
}
int fake_capture_broken() { return g_capture_broken ? 1 : 0; }
void fake_clear() { g_launches.clear(); }
int fake_launches() { return static_cast<int>(g_launches.size()); }
const char* fake_name(int i) { return g_launches[i].name.c_str(); }
unsigned fake_grid(int i) { return g_launches[i].grid; }

void** __hipRegisterFatBinary(const void*)
{
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*)
{
    if (std::strstr(name, "gofann")) names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
static Config g_config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    g_config = Config{grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = g_config.grid;
    *block = g_config.block;
    *lds = g_config.lds;
    *stream = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t lds, hipStream_t stream)
{
    const auto it = names().find(f);
    g_launches.push_back(Launch{it == names().end() ? "?" : it->second, grid.x, lds, stream});
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(static_cast<void*>(p), 0, sizeof(*p));
    p->multiProcessorCount = kCus;
    p->sharedMemPerBlock = kLds;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = static_cast<int>(kLds);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*)
{
    std::memset(static_cast<void*>(a), 0, sizeof(*a));
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void*, int, size_t lds)
{
    *blocks = std::min<int>(g_waves, lds ? static_cast<int>(kLds / lds) : g_waves);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static uint64_t word;
    *p = &word;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes)
{
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    if (bytes > g_limit - std::min(g_used, g_limit)) return hipErrorOutOfMemory;
    *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
    g_blocks[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    g_used -= g_blocks[p];
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st)
{
    *st = g_capturing && s == g_capturing ? hipStreamCaptureStatusActive
                                          : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* mode)
{
    std::swap(*mode, g_mode);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error of the stand-in runtime"; }
}
