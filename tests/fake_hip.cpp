// A stand-in for the HIP runtime on the CPU, for tests of what the library's
// host code does when an allocation fails or the device answers late.  Device
// memory is host memory.  Kernels do nothing, but for what the host waits for:
// the last kernel of a step reports (when the stream is next waited for, as
// late as a device may) and the pressure pass of a PCISPH correction answers
// its flag.  The positions of the arguments read here are those of the
// kernels' signatures in csrc/lps_kernels.hip.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "lps_common.h"

namespace {
std::map<const void*, std::string> g_names;
struct Config { dim3 grid, block; size_t shared; hipStream_t stream; } g_config;
int g_fail_in = -1;          // allocations until the one that fails (-1: none)
int g_plain_its = 4, g_seeded_its = 4;  // corrections of a step without and with the seed
bool g_seeded = false;
uint32_t g_overflow_cells = 0;  // cells the next step needs, as a grid overflow (0: it succeeds)
uint32_t g_cell_cap = 0;
uint32_t g_null_launches = 0;
hipError_t g_last = hipSuccess;  // as the runtime keeps it: the last error, until it is asked for
size_t g_bytes = 0;
std::map<void*, size_t> g_sizes;
StepReport* g_report = nullptr;
StepReport g_now{0u, 0u, 0u};

hipError_t failed(hipError_t e) { return g_last = e; }

template <class T>
T arg(void** args, int k) { return *static_cast<T*>(args[k]); }

void need(void** args, int first, int last) {
    for (int k = first; k <= last; k++)
        if (!arg<void*>(args, k)) g_null_launches++;
}
void finish_step(StepReport* r) {
    if (!r) return;
    g_report = r;
    g_now.status = g_overflow_cells ? LPS_ERR_GRID_OVERFLOW : 0u;
    g_now.cells_needed = g_overflow_cells;
    if (!g_overflow_cells) g_now.steps_ok++;
    g_overflow_cells = 0;
    g_seeded = false;
}
}  // namespace

extern "C" {
void fake_fail_malloc(int in) { g_fail_in = in; }
void fake_iterations(int plain, int seeded) { g_plain_its = plain; g_seeded_its = seeded; }
void fake_leave_error() { failed(hipErrorInvalidValue); }
void fake_overflow(uint32_t cells) { g_overflow_cells = cells; }
uint32_t fake_null_launches() { return g_null_launches; }
size_t fake_bytes() { return g_bytes; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
    g_config = Config{grid, block, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
    *grid = g_config.grid;
    *block = g_config.block;
    *shared = g_config.shared;
    *s = g_config.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    const std::string& n = g_names[f];
    auto is = [&](const char* part) { return n.find(part) != std::string::npos; };
    if (is("k_grid_one")) {
        g_cell_cap = arg<uint32_t>(args, 4);
    } else if (is("k_sort_one")) {
        g_cell_cap = arg<uint32_t>(args, 4);
        if (g_overflow_cells) static_cast<SceneGrid**>(args[1])[1]->cells = g_overflow_cells - 1u;
        need(args, 6, 6);
        if (g_cell_cap) need(args, 7, 8);  // with no cells it reports an overflow and stops
    } else if (is("k_keys")) {
        need(args, 0, 0);
        if (g_cell_cap) need(args, 3, 5);
    } else if (is("k_reorder")) {
        need(args, 2, 16);
    } else if (is("k_density_t")) {  // its neighbour lists
        for (int k = 0; k < 2; k++)
            if (!static_cast<void**>(args[10])[k]) g_null_launches++;
    } else if (is("k_mlp_seed")) {
        g_seeded = true;
    } else if (is("k_pci_pressure")) {
        const int k = (int)arg<uint32_t>(args, 17), its = g_seeded ? g_seeded_its : g_plain_its;
        if (k <= its) {
            volatile uint32_t* flag = arg<uint32_t*>(args, is("k_pci_pressure_t") ? 22 : 21);
            flag[1] = (uint32_t)k;
            flag[2] = 0u;
            flag[3] = 1u;
            flag[4] = 1u;
            flag[0] = k == its ? 1u : 0u;
        }
    } else if (is("k_pressure_sph_t")) {
        finish_step(static_cast<StepReport**>(args[9])[9]);
    } else if (is("k_integrate")) {
        finish_step(arg<StepReport*>(args, 17));
    }
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (g_fail_in >= 0 && g_fail_in-- == 0) return failed(hipErrorOutOfMemory);
    *p = std::calloc(n, 1);
    g_sizes[*p] = n;
    g_bytes += n;
    return *p ? hipSuccess : failed(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
    g_bytes -= g_sizes[p];
    g_sizes.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return failed(hipErrorInvalidSymbol); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(&g_config); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) {  // a context ends
    g_report = nullptr;
    g_now = StepReport{0u, 0u, 0u};
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    if (g_report) *g_report = g_now;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return failed(hipErrorNotSupported); }
}
