// A stand-in for the part of the HIP runtime that copies through staging buffers use: several GPUs, streams that hold their
// copies back until somebody waits for them, and the runtime's rule that an event is recorded on a stream of its own GPU. The only kernel that
// is launched here is the library's copy of bytes (source, destination, 16-byte units, bytes, ...).
// Loaded in front of the library by test_staging.py; no GPU is involved.
#include <cstdlib>
#include <cstring>
#include <vector>

namespace {
struct Copy {
    void* dst;
    const void* src;
    size_t bytes;
};
struct Stream {
    int device;
    std::vector<Copy> queue;
    void run() {
        for (const Copy& c : queue) std::memcpy(c.dst, c.src, c.bytes);
        queue.clear();
    }
};
struct Event {
    int device;
    Stream* on;
};
constexpr int kDevices = 3;
Stream g_null[kDevices] = {{0, {}}, {1, {}}, {2, {}}};
int g_current = 0, g_fail_records = 0, g_pinned = 0, g_capturing = 0, g_copies = 0, g_launches = 0, g_memory_of = 0, g_error = 0;
Stream* of(void* s) { return s ? static_cast<Stream*>(s) : &g_null[g_current]; }
constexpr int kInvalidHandle = 400, kNotReady = 600, kInvalidDevice = 101;
}  // namespace

extern "C" {
int hipGetDevice(int* d) { return *d = g_current, 0; }
int hipSetDevice(int d) { return d < 0 || d >= kDevices ? kInvalidDevice : (g_current = d, 0); }
int hipStreamGetDevice(void* s, int* d) { return *d = of(s)->device, 0; }
int hipStreamIsCapturing(void*, int* status) { return *status = g_capturing, 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), ++g_pinned, 0; }
int hipHostFree(void* p) { return std::free(p), --g_pinned, 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = new Event{g_current, nullptr}, 0; }
int hipEventDestroy(void* e) { return delete static_cast<Event*>(e), 0; }
int hipEventRecord(void* e, void* s) {
    if (g_fail_records > 0) return --g_fail_records, kInvalidHandle;
    if (static_cast<Event*>(e)->device != of(s)->device) return kInvalidHandle;
    return static_cast<Event*>(e)->on = of(s), 0;
}
int hipEventQuery(void* e) { return static_cast<Event*>(e)->on && !static_cast<Event*>(e)->on->queue.empty() ? kNotReady : 0; }
int hipEventSynchronize(void* e) {
    if (static_cast<Event*>(e)->on) static_cast<Event*>(e)->on->run();
    return 0;
}
int hipMemcpyAsync(void* dst, const void* src, size_t n, int, void* s) { return of(s)->queue.push_back({dst, src, n}), ++g_copies, 0; }
struct Dim3 {
    unsigned x, y, z;
};
int hipLaunchKernel(const void*, Dim3, Dim3, void** args, size_t, void* s) {
    of(s)->queue.push_back({*static_cast<void**>(args[1]), *static_cast<void**>(args[0]), *static_cast<size_t*>(args[3])});
    return ++g_launches, 0;
}
struct Attribute {  // hipPointerAttribute_t
    int type, device;
    void *device_pointer, *host_pointer;
    int managed;
    unsigned flags;
};
int hipPointerGetAttributes(Attribute* a, const void*) {  // (device memory of one of the GPUs, or host memory)
    *a = Attribute{};
    return a->type = g_memory_of < 0 ? 1 : 2, a->device = g_memory_of, 0;
}
int hipStreamSynchronize(void* s) { return of(s)->run(), 0; }
int hipGetLastError() {
    const int e = g_error;
    return g_error = 0, e;
}

void fake_fail_records(int n) { g_fail_records = n; }
void fake_capture(int on) { g_capturing = on; }
void* fake_stream(int device) { return new Stream{device, {}}; }
int fake_pinned() { return g_pinned; }
void fake_memory_of(int device) { g_memory_of = device; }  // what the program's pointers are: a GPU's, -1: pinned host memory
void fake_error(int e) { g_error = e; }                    // left by a call of the program's own
int fake_copies() { return g_copies; }
int fake_launches() { return g_launches; }
}
