// A HIP runtime without a GPU, for tests of the library's host side: memory is
// host memory, a stream is a queue of copies that run when somebody waits for
// them (the latest time the real one allows), kernels are not run but recorded.
// Loaded with RTLD_GLOBAL before libhydrogen.so, it takes the place of the real
// runtime in that process.
#include <unistd.h>

#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>

namespace {

constexpr int kOk = 0, kInvalid = 1, kNotSupported = 801;
constexpr int kHostToDevice = 1, kDeviceToHost = 2;
constexpr int kUnregistered = 0, kHost = 1, kDevice = 2;      // hipMemoryType

std::recursive_mutex mu;

struct Op {
    void* dst;
    const void* src;
    size_t bytes;
};
struct Stream {
    std::deque<Op> queue;
    size_t done = 0;
    void run(size_t upto) {
        for (; done < upto && !queue.empty(); ++done, queue.pop_front())
            std::memcpy(queue.front().dst, queue.front().src, queue.front().bytes);
    }
    size_t total() const { return done + queue.size(); }
};
struct Event {
    Stream* s = nullptr;
    size_t upto = 0;
};

std::map<char*, size_t> pinned, device;
std::map<const void*, std::string> kernels;
std::map<std::string, std::pair<int, int>> failing;          // function -> calls until it fails, its code
std::string launches, watch_name;
int watch_index = 0, watch_value = -1, last_error = kOk;
long direct_copies = 0, syncs = 0;
unsigned event_delay_us = 0;

const size_t* find(const std::map<char*, size_t>& m, const void* p) {
    auto it = m.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
    if (it == m.begin()) return nullptr;
    --it;
    return static_cast<const char*>(p) < it->first + it->second ? &it->second : nullptr;
}

// the error `fn` is to fail with now, if any
int injected(const char* fn) {
    auto it = failing.find(fn);
    if (it == failing.end() || --it->second.first > 0) return kOk;
    const int code = it->second.second;
    failing.erase(it);
    return last_error = code;
}

int allocate(std::map<char*, size_t>& m, void** p, size_t bytes, const char* fn) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int e = injected(fn)) return e;
    *p = std::calloc(bytes ? bytes : 1, 1);
    m[static_cast<char*>(*p)] = bytes;
    return kOk;
}
int release(std::map<char*, size_t>& m, void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    m.erase(static_cast<char*>(p));
    std::free(p);
    return kOk;
}

Stream null_stream;
Stream* of(void* s) { return s ? static_cast<Stream*>(s) : &null_stream; }

}  // namespace

extern "C" {

// ---- what the tests set and ask
void fake_fail(const char* fn, int nth, int code) { failing[fn] = {nth, code}; }
void fake_event_delay(unsigned us) { event_delay_us = us; }
const char* fake_launches() { return launches.c_str(); }
void fake_clear() { launches.clear(); direct_copies = syncs = 0; watch_value = -1; }
// remembers the int argument `index` of the last launch of a kernel whose name holds `name`
void fake_watch(const char* name, int index) { watch_name = name; watch_index = index; }
int fake_watched() { return watch_value; }
// copies to or from the caller's own pinned or device memory (not of 2 MB, the
// size of the library's slots)
long fake_direct_copies() { return direct_copies; }
// waits for a stream
long fake_syncs() { return syncs; }
int fake_last_error() { return last_error; }
void fake_set_last_error(int e) { last_error = e; }

// ---- kernels
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    kernels[host] = name;
}
struct Dim { unsigned x, y, z; };
static thread_local struct { Dim grid, block; size_t shared; void* stream; } config;
int __hipPushCallConfiguration(Dim g, Dim b, size_t shared, void* s) { config = {g, b, shared, s}; return kOk; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* shared, void** s) {
    *g = config.grid; *b = config.block; *shared = config.shared; *s = config.stream;
    return kOk;
}
int hipLaunchKernel(const void* f, Dim, Dim, void** args, size_t, void* s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int e = injected("hipLaunchKernel")) return e;
    const std::string& name = kernels[f];
    launches += name + "\n";
    if (name.find("k_copy_out") != std::string::npos)          // (to, from, 16-byte units): the one that is run
        of(s)->queue.push_back({*static_cast<void**>(args[0]), *static_cast<const void**>(args[1]),
                                *static_cast<const unsigned*>(args[2]) * size_t(16)});
    if (!watch_name.empty() && name.find(watch_name) != std::string::npos)
        watch_value = *static_cast<const int*>(args[watch_index]);
    return kOk;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return kOk; }
int hipGetSymbolAddress(void** p, const void*) { static char scratch[1 << 20]; *p = scratch; return kOk; }

// ---- the device, errors
int hipGetDevice(int* d) { *d = 0; return kOk; }
int hipSetDevice(int) { return kOk; }
int hipGetDeviceCount(int* n) { *n = 1; return kOk; }
int hipGetDevicePropertiesR0600(void*, int) { return kNotSupported; }
const char* hipGetErrorString(int e) { return e ? "fake error" : "no error"; }
int hipGetLastError() { const int e = last_error; last_error = kOk; return e; }

// ---- memory
int hipMalloc(void** p, size_t bytes) { return allocate(device, p, bytes, "hipMalloc"); }
int hipFree(void* p) { return release(device, p); }
int hipHostMalloc(void** p, size_t bytes, unsigned) { return allocate(pinned, p, bytes, "hipHostMalloc"); }
int hipHostFree(void* p) { return release(pinned, p); }
int hipPointerGetAttributes(void* attributes, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int e = injected("hipPointerGetAttributes")) return e;
    *static_cast<int*>(attributes) = find(pinned, p) ? kHost : find(device, p) ? kDevice : kUnregistered;
    return kOk;
}

// ---- streams and events
int hipStreamCreateWithFlags(void** s, unsigned) { *s = new Stream; return kOk; }
int hipStreamDestroy(void* s) { of(s)->run(size_t(-1)); delete of(s); return kOk; }
int hipStreamSynchronize(void* s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    ++syncs;
    if (const int e = injected("hipStreamSynchronize")) return e;
    of(s)->run(size_t(-1));
    return kOk;
}
int hipStreamWaitEvent(void*, void* e, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (static_cast<Event*>(e)->s) static_cast<Event*>(e)->s->run(static_cast<Event*>(e)->upto);
    return kOk;
}
int hipEventCreateWithFlags(void** e, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int r = injected("hipEventCreateWithFlags")) return r;
    *e = new Event;
    return kOk;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { delete static_cast<Event*>(e); return kOk; }
int hipEventRecord(void* e, void* s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *static_cast<Event*>(e) = {of(s), of(s)->total()};
    return kOk;
}
int hipEventSynchronize(void* e) {
    if (event_delay_us) usleep(event_delay_us);
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int r = injected("hipEventSynchronize")) return r;
    if (static_cast<Event*>(e)->s) static_cast<Event*>(e)->s->run(static_cast<Event*>(e)->upto);
    return kOk;
}
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 1.0f; return kOk; }

int hipMemcpyAsync(void* dst, const void* src, size_t bytes, int kind, void* s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (const int e = injected("hipMemcpyAsync")) return e;
    const void* host = kind == kHostToDevice ? src : kind == kDeviceToHost ? dst : nullptr;
    of(s)->queue.push_back({dst, src, bytes});
    if (host && !find(pinned, host)) of(s)->run(size_t(-1));   // pageable memory: the call waits
    const size_t* size = !host ? nullptr : find(pinned, host) ? find(pinned, host) : find(device, host);
    if (size && *size != (size_t(2) << 20)) ++direct_copies;   // not one of the library's 2 MB slots
    return kOk;
}
int hipMemcpy(void* dst, const void* src, size_t bytes, int) { std::memcpy(dst, src, bytes); return kOk; }
int hipMemsetAsync(void* p, int v, size_t bytes, void* s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    of(s)->run(size_t(-1));
    std::memset(p, v, bytes);
    return kOk;
}

// ---- graphs: captured launches are recorded as they are made
int hipStreamBeginCapture(void*, int) { return kOk; }
int hipStreamEndCapture(void*, void** g) { static char graph; *g = &graph; return kOk; }
int hipGraphInstantiate(void** x, void* g, void*, char*, size_t) { *x = g; return kOk; }
int hipGraphLaunch(void*, void*) { return kOk; }
int hipGraphDestroy(void*) { return kOk; }
int hipGraphExecDestroy(void*) { return kOk; }

}  // extern "C"
