// Host-side check of a compiled segment's staging (csrc/provider.hip, csrc/runtime.hip) without a GPU: this program defines
// the HIP runtime functions that libsharplight_hip.so calls -- two devices, streams whose work runs only when something
// waits for them, a last-error slot that keeps an error until it is read, device memory as host memory -- and drives
// segments through the C API. argv[1] names the scenario; exit status 0 if it holds. The only kernels that run are the
// staging copy and, on request, a gather that raises the device's error record.
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <deque>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "../include/sharplight_hip.h"

namespace {
struct Stream {
    int device;
    std::deque<std::function<void()>> work;
    void drain()
    {
        for (; !work.empty(); work.pop_front()) work.front()();
    }
};
int g_device = 0;
uint32_t g_record[2][8];             // the error record of each device
std::map<const void*, std::string>& kernels()  // (filled by the library's initialisers, before this program's)
{
    static std::map<const void*, std::string> m;
    return m;
}
hipError_t g_last = hipSuccess;
bool g_refuse_host_malloc = false;   // hipHostMalloc fails
bool g_refuse_copies = false;        // launches of the staging copy fail
bool g_bad_gather = false;           // the next gather raises its error
struct Call {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
std::vector<Call> g_calls;
std::set<Stream*> g_streams;
std::map<void*, size_t> g_blocks;     // allocations and their bytes; g_pinned: those of host memory
std::set<void*> g_pinned;

hipError_t done(hipError_t e)
{
    if (e != hipSuccess) g_last = e;
    return e;
}
Stream* stream(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*)
{
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels()[host] = name; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    g_calls.push_back({grid, block, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s)
{
    *grid = g_calls.back().grid, *block = g_calls.back().block, *lds = g_calls.back().lds, *s = g_calls.back().stream;
    g_calls.pop_back();
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s)
{
    const std::string name = kernels()[f];
    Stream* st = stream(s);
    if (name.find("copy_staged") != std::string::npos) {  // (dst, src, bytes, err_dst, err_src)
        if (g_refuse_copies) return done(hipErrorLaunchFailure);
        uint8_t *dst = *static_cast<uint8_t**>(args[0]), *src = *static_cast<uint8_t**>(args[1]);
        const size_t n = *static_cast<size_t*>(args[2]);
        uint32_t *ed = *static_cast<uint32_t**>(args[3]), *es = *static_cast<uint32_t**>(args[4]);
        if (st->device != g_device || (es && es != g_record[st->device])) {
            printf("a staging copy of device %d launched from device %d\n", st->device, g_device);
            exit(1);
        }
        st->work.push_back([=] {
            memcpy(dst, src, n);
            if (ed) memcpy(ed, es, 32);
        });
    } else if (name.find("gather") != std::string::npos && g_bad_gather) {
        g_bad_gather = false;
        st->work.push_back([=] {
            const uint32_t r[8] = {1, 12, 0, 10};  // kErrGatherIndex, id 12 of 10 rows
            memcpy(g_record[st->device], r, sizeof r);
        });
    }
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = g_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    g_device = d;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "planted error"; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    *p = g_record[g_device];
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n)
{
    *p = aligned_alloc(256, (n + 511) / 256 * 256);
    g_blocks[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    g_blocks.erase(p);
    g_pinned.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (g_refuse_host_malloc) return done(hipErrorOutOfMemory);
    const hipError_t e = hipMalloc(p, n);
    g_pinned.insert(*p);
    return e;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    Stream* st = new Stream{g_device, {}};
    g_streams.insert(st);
    *s = reinterpret_cast<hipStream_t>(st);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    g_streams.erase(stream(s));
    delete stream(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    stream(s)->drain();
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st)
{
    *st = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)  // pageable: not before the stream's work
{
    stream(st)->drain();
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
}

namespace {
#define EXPECT(cond)                                            \
    do {                                                        \
        if (!(cond)) {                                          \
            printf("line %d: %s [%s]\n", __LINE__, #cond, slhip_last_error()); \
            exit(1);                                            \
        }                                                       \
    } while (0)

// y = rows of a [10, 64] table.
const char* kGather = "value 0 f32 10 64\nvalue 1 i32 T\nvalue 2 f32 T 64\ninput 1\nweight 0\noutput 2\nnode Gather 0,1 -> 2\n";
const int32_t kIds[4] = {1, 2, 3, 4};

slhip_segment compile()
{
    slhip_segment s = nullptr;
    EXPECT(slhip_segment_compile(kGather, 4, &s) == SLHIP_OK);
    return s;
}
int set_ids(slhip_segment s) { return slhip_segment_set_input(s, 1, kIds, sizeof kIds); }
int run(slhip_segment s) { return slhip_segment_execute(s, 4); }
int output(slhip_segment s)
{
    float y[4 * 64];
    return slhip_segment_get_output(s, 2, y, sizeof y);
}
void destroy(slhip_segment s) { EXPECT(slhip_segment_destroy(s) == SLHIP_OK); }

// Closing one segment leaves the error that another one's run has raised.
void close_keeps_the_error_of_another()
{
    slhip_segment a = compile(), b = compile();
    EXPECT(set_ids(a) == SLHIP_OK && run(a) == SLHIP_OK && output(a) == SLHIP_OK);
    EXPECT(set_ids(b) == SLHIP_OK);
    g_bad_gather = true;
    EXPECT(run(b) == SLHIP_OK);
    for (Stream* s : g_streams) s->drain();  // b's run has ended
    destroy(a);
    EXPECT(output(b) == SLHIP_ERR_INDEX);
    EXPECT(output(b) == SLHIP_OK);
    destroy(b);
}

// A thread whose current device is another one sets inputs and reads outputs, and stays on its device.
void another_current_device()
{
    slhip_segment s = compile();
    g_device = 1;
    EXPECT(set_ids(s) == SLHIP_OK && g_device == 1);
    g_device = 0;
    EXPECT(run(s) == SLHIP_OK);
    g_device = 1;
    EXPECT(output(s) == SLHIP_OK && g_device == 1);
    g_device = 0;
    g_bad_gather = true;
    EXPECT(run(s) == SLHIP_OK);
    g_device = 1;
    EXPECT(output(s) == SLHIP_ERR_INDEX && g_device == 1);
    g_device = 0;
    g_bad_gather = true;
    EXPECT(run(s) == SLHIP_OK);
    g_device = 1;
    EXPECT(set_ids(s) == SLHIP_ERR_INDEX && g_device == 1);
    destroy(s);
}

// Without staging memory the runtime's copies are taken, and the refused allocation is no later call's error.
void staging_memory_refused()
{
    g_refuse_host_malloc = true;
    slhip_segment s = compile();
    EXPECT(set_ids(s) == SLHIP_OK);
    EXPECT(run(s) == SLHIP_OK);
    EXPECT(output(s) == SLHIP_OK);
    destroy(s);
}

// An input that is still to be copied stays in place when reading an output fails before it has waited.
void failed_output_keeps_the_inputs()
{
    const char* add = "value 0 f32 T 64\nvalue 1 f32 T 64\nvalue 2 f32 T 64\ninput 0\ninput 1\noutput 2\nnode Add 0,1 -> 2\n";
    slhip_segment s = nullptr;
    EXPECT(slhip_segment_compile(add, 1, &s) == SLHIP_OK);
    float in[2][64], y[64];
    for (int i = 0; i < 64; i++) in[0][i] = 1.0f, in[1][i] = 2.0f;
    EXPECT(slhip_segment_set_input(s, 0, in[0], sizeof in[0]) == SLHIP_OK);
    EXPECT(slhip_segment_execute(s, 1) == SLHIP_OK);
    g_refuse_copies = true;
    EXPECT(slhip_segment_get_output(s, 2, y, sizeof y) != SLHIP_OK);
    g_refuse_copies = false;
    EXPECT(slhip_segment_set_input(s, 1, in[1], sizeof in[1]) == SLHIP_OK);
    EXPECT(slhip_segment_get_output(s, 2, y, sizeof y) == SLHIP_OK);  // (runs what is queued)
    int held = 0;  // device blocks that begin with the first input's rows
    for (const auto& b : g_blocks)
        if (b.second >= sizeof in[0] && memcmp(b.first, in[0], sizeof in[0]) == 0 && g_pinned.count(b.first) == 0) held++;
    EXPECT(held == 1);
    destroy(s);
}
}  // namespace

int main(int argc, char** argv)
{
    const std::map<std::string, void (*)()> scenarios = {
        {"close_keeps_the_error_of_another", close_keeps_the_error_of_another},
        {"another_current_device", another_current_device},
        {"staging_memory_refused", staging_memory_refused},
        {"failed_output_keeps_the_inputs", failed_output_keeps_the_inputs},
    };
    const auto it = scenarios.find(argc > 1 ? argv[1] : "");
    if (it == scenarios.end()) return 2;
    it->second();
    puts("ok");
    return 0;
}
