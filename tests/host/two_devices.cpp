// A HIP runtime of two devices without any: host memory, launches that are checked and written down instead of run.  Loaded
// ahead of libet_amd.so it answers the calls that the library makes, so that what the launchers do per device, per stream
// and per thread can be tested where there is no GPU.  Kernels need the opt-in to more than 64 KB of LDS on each device,
// and a launch takes a function of its stream's device, as the runtime documents.
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace {
constexpr int OK = 0, INVALID_VALUE = 1, INVALID_DEVICE = 101, INVALID_HANDLE = 400;
struct Stream {
    int device;
};
struct Function {
    const void *symbol;
    int device;
};
struct Launch {
    int device;
    unsigned block, lds;
    void *third; // the third parameter's eight bytes (two_devices_third)
};
std::mutex lock;
std::map<std::pair<const void *, int>, int> allowed; // (kernel, device) -> dynamic LDS
std::map<std::pair<const void *, int>, Function *> functions;
std::vector<Launch> launches; // the first few thousand
Launch latest;
bool refuse_lds = false; // the opt-in to large LDS fails
unsigned third_lds = 0; // launches with that much LDS have at least three parameters, others may have one
unsigned char symbols[2][1 << 16]; // a device variable's stand-in on either device
thread_local int current = 0, last_error = OK;

int fail(int e) {
    if (e != OK)
        last_error = e;
    return e;
}
int device_of(void *stream) { return stream ? static_cast<Stream *>(stream)->device : current; }
bool lds_allowed(const void *symbol, int device, size_t lds) { return lds <= 64 * 1024 || allowed[{symbol, device}] >= (int)lds; }
struct Dim {
    unsigned x, y, z;
};
} // namespace

extern "C" {
// ---- what the tests ask
void two_devices_stream(int device, void **stream) { *stream = new Stream{device}; }
int two_devices_launches() {
    std::lock_guard<std::mutex> l(lock);
    return (int)launches.size();
}
void two_devices_refuse(int on) { refuse_lds = on; }
void two_devices_third(unsigned lds) { third_lds = lds; }
void two_devices_clear() {
    std::lock_guard<std::mutex> l(lock);
    launches.clear();
}
void two_devices_launch(int i, int *device, unsigned *block, unsigned *lds) {
    std::lock_guard<std::mutex> l(lock);
    *device = launches[i].device;
    *block = launches[i].block;
    *lds = launches[i].lds;
}
// whose copy of a device variable the launch was handed as its third parameter; -1: nobody's
int two_devices_variable_of(int i) {
    std::lock_guard<std::mutex> l(lock);
    const unsigned char *p = static_cast<unsigned char *>(launches[i].third);
    for (int d = 0; d < 2; d++)
        if (p >= symbols[d] && p < symbols[d] + sizeof(symbols[d]))
            return d;
    return -1;
}
// One thread launches the plan again and again while this one sets a key, to two values in turn.  Returns how often a launch
// that began after the key was set did not have the value's threads a workgroup.  (A few seconds at most: on one processor
// the two threads hardly meet.)
int two_devices_race(int (*set)(const char *, int), int (*run)(const void *, void *, const void *, int, int, void *),
                     const void *plan, void *x, int rows, const char *key, const int *values, const unsigned *threads, int times) {
    std::atomic<bool> stop{false};
    std::atomic<int> done{0};
    std::thread runs([&] {
        for (; !stop; done++)
            run(plan, x, x, rows, 1, nullptr);
    });
    int wrong = 0;
    const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(5);
    for (int i = 0; i < times && std::chrono::steady_clock::now() < end; i++) {
        set(key, values[i & 1]);
        const int before = done;
        while (done < before + 2) // (the first of them may have begun earlier)
            std::this_thread::yield();
        std::lock_guard<std::mutex> l(lock);
        wrong += latest.block != threads[i & 1];
    }
    stop = true;
    runs.join();
    return wrong;
}

// ---- the runtime
int hipGetDevice(int *d) { return *d = current, OK; }
int hipSetDevice(int d) { return d < 0 || d > 1 ? fail(INVALID_DEVICE) : (current = d, OK); }
int hipStreamGetDevice(void *s, int *d) { return *d = device_of(s), OK; }
int hipGetLastError() {
    const int e = last_error;
    last_error = OK;
    return e;
}
const char *hipGetErrorString(int) { return "refused by the two devices"; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, OK; } // (compute units)
int hipDeviceSynchronize() { return OK; }
int hipStreamSynchronize(void *) { return OK; }
int hipStreamCreate(void **s) { return two_devices_stream(current, s), OK; }
int hipStreamDestroy(void *s) { return delete static_cast<Stream *>(s), OK; }
int hipMalloc(void **p, size_t n) { return posix_memalign(p, 256, n ? n : 1) ? fail(2) : OK; }
int hipFree(void *p) { return free(p), OK; }
int hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipHostFree(void *p) { return hipFree(p); }
int hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, OK; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return memcpy(d, s, n), OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return memcpy(d, s, n), OK; }
int hipGetSymbolAddress(void **p, const void *) { return *p = symbols[current], OK; }
int hipFuncSetAttribute(const void *symbol, int, int value) {
    std::lock_guard<std::mutex> l(lock);
    if (refuse_lds)
        return fail(INVALID_VALUE);
    allowed[{symbol, current}] = value;
    return OK;
}
int hipGetFuncBySymbol(void **fn, const void *symbol) {
    std::lock_guard<std::mutex> l(lock);
    Function *&f = functions[{symbol, current}];
    if (!f)
        f = new Function{symbol, current};
    *fn = f;
    return OK;
}
int hipModuleLaunchKernel(void *fn, unsigned, unsigned, unsigned, unsigned bx, unsigned, unsigned, unsigned lds, void *stream,
                          void **params, void **) {
    const Function *f = static_cast<Function *>(fn);
    std::lock_guard<std::mutex> l(lock);
    if (f->device != device_of(stream))
        return fail(INVALID_HANDLE);
    if (!lds_allowed(f->symbol, f->device, lds))
        return fail(INVALID_VALUE);
    void *third = nullptr;
    if (lds && lds == third_lds)
        memcpy(&third, params[2], sizeof(third));
    latest = {f->device, bx, lds, third};
    if (launches.size() < 4096)
        launches.push_back(latest);
    return OK;
}
// (finds its device by itself: not written down)
int hipLaunchKernel(const void *symbol, Dim, Dim, void **, size_t lds, void *stream) {
    std::lock_guard<std::mutex> l(lock);
    return lds_allowed(symbol, device_of(stream), lds) ? OK : fail(INVALID_VALUE);
}
static thread_local struct {
    Dim grid, block;
    size_t lds;
    void *stream;
} call;
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void *stream) {
    call = {grid, block, lds, stream};
    return OK;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *lds, void **stream) {
    *grid = call.grid;
    *block = call.block;
    *lds = call.lds;
    *stream = call.stream;
    return OK;
}
}
