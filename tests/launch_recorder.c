/* The part of the HIP runtime that libsubstation_amd.so calls, without a GPU: kernels are not run, their names and grids are kept.
 * Loaded in front of the library (tests/launches.py), so that a test on the CPU can ask what a call would launch. */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } Dim;

static struct { const void* stub; const char* name; } kernels[4096];
static int n_kernels;
static char* text;
static size_t used, room;
static struct { Dim grid, block; size_t shared; void* stream; } next;
static long events;

const char* recorder_text(void) { return text ? text : ""; }
void recorder_clear(void) { used = 0; if (text) text[0] = 0; }
long recorder_events(void) { return events; }

void** __hipRegisterFatBinary(const void* data) { static void* handle; (void)data; return &handle; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* stub, char* name, const char* device_name, unsigned threads, void* tid, void* bid,
                           void* block, void* grid, int* w) {
    (void)m; (void)name; (void)threads; (void)tid; (void)bid; (void)block; (void)grid; (void)w;
    if (n_kernels < (int)(sizeof(kernels) / sizeof(kernels[0]))) { kernels[n_kernels].stub = stub; kernels[n_kernels++].name = device_name; }
}
void __hipRegisterVar(void** m, void* var, char* host, const char* device, int ext, size_t size, int constant, int global) {
    (void)m; (void)var; (void)host; (void)device; (void)ext; (void)size; (void)constant; (void)global;
}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void* stream) {
    next.grid = grid; next.block = block; next.shared = shared; next.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* shared, void** stream) {
    *grid = next.grid; *block = next.block; *shared = next.shared; *stream = next.stream;
    return 0;
}
int hipLaunchKernel(const void* stub, Dim grid, Dim block, void** args, size_t shared, void* stream) {
    const char* name = "unknown kernel";
    (void)block; (void)args; (void)shared; (void)stream;
    for (int i = 0; i < n_kernels; ++i) if (kernels[i].stub == stub) name = kernels[i].name;
    if (used + strlen(name) + 64 > room) {
        char* more = realloc(text, room = 2 * room + strlen(name) + 4096);
        if (!more) abort();
        text = more;
    }
    used += (size_t)sprintf(text + used, "%s %u %u %u\n", name, grid.x, grid.y, grid.z);
    return 0;
}
int hipMalloc(void** p, size_t n) { *p = NULL; return posix_memalign(p, 4096, n ? n : 1) ? 2 : 0; }
int hipFree(void* p) { free(p); return 0; }
int hipMemcpy(void* to, const void* from, size_t n, int kind) { (void)kind; memcpy(to, from, n); return 0; }
int hipMemset(void* p, int v, size_t n) { memset(p, v, n); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int attribute, int device) { (void)attribute; (void)device; *v = 100000; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { (void)e; return "recorder"; }
int hipGetSymbolAddress(void** p, const void* symbol) { (void)symbol; return hipMalloc(p, 4 << 20); }
int hipStreamIsCapturing(void* stream, int* status) { (void)stream; *status = 0; return 0; }
int hipStreamSynchronize(void* stream) { (void)stream; return 0; }
int hipThreadExchangeStreamCaptureMode(int* mode) { (void)mode; return 0; }
int hipEventCreate(void** e) { *e = &events; ++events; return 0; }
int hipEventDestroy(void* e) { (void)e; return 0; }
int hipEventRecord(void* e, void* stream) { (void)e; (void)stream; return 0; }
int hipEventSynchronize(void* e) { (void)e; return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 0; return 0; }
