// A stand-in for the HIP runtime under which libqe_amd.so's host code runs
// without a GPU: every kernel launch is recorded instead of made.  Loaded with
// RTLD_GLOBAL before the library, so the library's HIP symbols resolve here.
// One line per event, in the order the calls were made:
//   launch <thread> <stream> <grid x y z> <block x> <dynamic LDS> <mangled kernel name>
//   free <thread> <address>
// A device of 256 compute units, no error ever, no stream in capture until
// recorder_set_capturing says so.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <time.h>

#include <atomic>
#include <condition_variable>
#include <map>
#include <mutex>
#include <string>

struct Dim {
    uint32_t x, y, z;
};
typedef void* Stream;

namespace {
std::mutex g_mutex;
std::condition_variable g_opened;
std::string g_log;
std::map<const void*, std::string> g_names;
std::map<Stream, bool> g_capturing;
Stream g_gate = nullptr;      // launches on this stream wait ...
bool g_gate_closed = false;   // ... while this holds
std::atomic<int> g_waiting{0};
int g_pause_us = 0;
std::atomic<int> g_threads{0};
thread_local int t_id = -1;
thread_local struct {
    Dim grid, block;
    size_t lds;
    Stream stream;
} t_config;

int thread_id() {
    if (t_id < 0) t_id = g_threads++;
    return t_id;
}
// a pause after each launch, so that a second thread gets in between two of them
void pause() {
    if (g_pause_us <= 0) return;
    timespec t{0, 1000L * g_pause_us};
    nanosleep(&t, nullptr);
}
}  // namespace

extern "C" {

void recorder_reset(int pause_us) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_log.clear();
    g_capturing.clear();
    g_pause_us = pause_us;
}
void recorder_set_capturing(Stream s, int on) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_capturing[s] = on != 0;
}
// Launches on `s` are recorded, then wait until recorder_open.
void recorder_close(Stream s) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_gate = s;
    g_gate_closed = true;
}
void recorder_open() {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_gate_closed = false;
    g_opened.notify_all();
}
int recorder_waiting() { return g_waiting; }
// Copies the log; returns its whole length.
size_t recorder_log(char* out, size_t n) {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (n > 0) snprintf(out, n, "%s", g_log.c_str());
    return g_log.size();
}

void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, Stream s) {
    t_config = {grid, block, lds, s};
    return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* lds, Stream* s) {
    *grid = t_config.grid;
    *block = t_config.block;
    *lds = t_config.lds;
    *s = t_config.stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim grid, Dim block, void**, size_t lds, Stream s) {
    char head[160];
    snprintf(head, sizeof(head), "launch %d %p %u %u %u %u %zu ", thread_id(), s, grid.x, grid.y, grid.z, block.x, lds);
    {
        std::unique_lock<std::mutex> lock(g_mutex);
        g_log += head + g_names[f] + "\n";
        if (g_gate_closed && s == g_gate) {
            ++g_waiting;
            g_opened.wait(lock, [] { return !g_gate_closed; });
            --g_waiting;
        }
    }
    pause();
    return 0;
}
int hipMalloc(void** p, size_t) {
    static std::atomic<uintptr_t> next{uintptr_t(1) << 40};
    *p = reinterpret_cast<void*>(next.fetch_add(uintptr_t(1) << 30));
    return 0;
}
int hipFree(void* p) {
    char line[64];
    snprintf(line, sizeof(line), "free %d %p\n", thread_id(), p);
    std::lock_guard<std::mutex> lock(g_mutex);
    g_log += line;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;
    return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "no error"; }
int hipStreamIsCapturing(Stream s, int* status) {
    std::lock_guard<std::mutex> lock(g_mutex);
    *status = g_capturing.count(s) != 0 && g_capturing[s] ? 1 : 0;
    return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
    *p = reinterpret_cast<void*>(uintptr_t(1) << 45);
    return 0;
}

}  // extern "C"
