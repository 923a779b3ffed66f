/* The HIP entry points that libash_hip.so calls, for tests of its host side on a CPU:
 * nothing runs on a device, a launch and a wait go to the test (stand_in_device.py),
 * which does what the device would do, later, or not at all. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
    uint32_t x, y, z;
} dim3_t;

/* 0, or the error of the launch / the wait */
static int (*on_launch)(const char* kernel, uintptr_t stream, void** args);
static int (*on_wait)(uintptr_t stream);
static int (*on_host_malloc)(size_t bytes);

void stand_in_connect(int (*launch)(const char*, uintptr_t, void**), int (*wait)(uintptr_t),
                      int (*host_malloc)(size_t)) {
    on_launch = launch;
    on_wait = wait;
    on_host_malloc = host_malloc;
}

static __thread int last_error;
static int failed(int error) {
    if (error) last_error = error;
    return error;
}

int hipGetLastError(void) {
    const int error = last_error;
    last_error = 0;
    return error;
}
const char* hipGetErrorString(int error) { return error ? "refused by the test" : "no error"; }

enum { kMostKernels = 4096 };
static struct {
    const void* stub;
    const char* name;
} kernels[kMostKernels];
static int num_kernels;

void** __hipRegisterFatBinary(const void* data) {
    static void* handle;
    (void)data;
    return &handle;
}
void __hipUnregisterFatBinary(void** modules) { (void)modules; }
void __hipRegisterFunction(void** modules, const void* stub, char* device_name, const char* name,
                           unsigned threads, void* a, void* b, void* c, void* d, void* e) {
    (void)modules, (void)device_name, (void)threads, (void)a, (void)b, (void)c, (void)d, (void)e;
    if (num_kernels == kMostKernels) abort();
    kernels[num_kernels].stub = stub;
    kernels[num_kernels++].name = name;
}
void __hipRegisterVar(void** modules, void* var, char* host, char* device, int ext, size_t size,
                      int constant, int global) {
    (void)modules, (void)var, (void)host, (void)device, (void)ext, (void)size, (void)constant, (void)global;
}

static __thread struct {
    dim3_t grid, block;
    size_t shared;
    void* stream;
} call;

int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t shared, void* stream) {
    call.grid = grid;
    call.block = block;
    call.shared = shared;
    call.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* shared, void** stream) {
    *grid = call.grid;
    *block = call.block;
    *shared = call.shared;
    *stream = call.stream;
    return 0;
}
int hipLaunchKernel(const void* stub, dim3_t grid, dim3_t block, void** args, size_t shared, void* stream) {
    (void)grid, (void)block, (void)shared;
    for (int k = 0; k < num_kernels; ++k) {
        if (kernels[k].stub == stub) return failed(on_launch(kernels[k].name, (uintptr_t)stream, args));
    }
    abort();
}

int hipStreamSynchronize(void* stream) { return failed(on_wait((uintptr_t)stream)); }
int hipDeviceSynchronize(void) { return failed(on_wait((uintptr_t)-1)); }
/* the devices that there are, the one that is current, and the stream of one that is captured */
static int num_devices = 1, current_device, capturing_device = -1;
static void* capturing_stream;
void stand_in_capture(int devices, int current, int device, void* stream) {
    num_devices = devices;
    current_device = current;
    capturing_device = device;
    capturing_stream = stream;
}
int stand_in_current_device(void) { return current_device; }
/* (the default stream is the current device's) */
int hipStreamIsCapturing(void* stream, int* status) {
    *status = capturing_device >= 0 && stream == capturing_stream && (stream != NULL || current_device == capturing_device);
    return 0;
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
    (void)flags;
    const int error = on_host_malloc(bytes);
    if (error) return failed(error);
    *p = aligned_alloc(256, (bytes + 255) / 256 * 256);
    return *p == NULL ? failed(2) : 0;
}
int hipMemcpyAsync(void* to, const void* from, size_t bytes, int kind, void* stream) {
    (void)kind, (void)stream;
    memcpy(to, from, bytes);
    return 0;
}
int hipGetDevice(int* device) {
    *device = current_device;
    return 0;
}
int hipSetDevice(int device) {
    if (device < 0 || device >= num_devices) return failed(101);
    current_device = device;
    return 0;
}
int hipDeviceGetAttribute(int* value, int attribute, int device) {
    (void)attribute, (void)device;
    *value = 256;
    return 0;
}
int hipFuncSetAttribute(const void* stub, int attribute, int value) {
    (void)stub, (void)attribute, (void)value;
    return 0;
}
int hipGetSymbolAddress(void** p, const void* symbol) {
    (void)p, (void)symbol;
    return failed(1);
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* groups, const void* stub, int threads, size_t shared) {
    (void)stub, (void)threads, (void)shared;
    *groups = 2;
    return 0;
}
int hipPointerGetAttributes(void* attributes, const void* p) {
    (void)attributes, (void)p;
    return failed(1);
}

const char* stand_in_kernel(int k) { return k < num_kernels ? kernels[k].name : NULL; }
