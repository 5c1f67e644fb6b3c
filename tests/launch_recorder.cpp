// HIP entry points that record kernel launches instead of making them, for CPU
// tests of the library's dispatch.  Loaded RTLD_GLOBAL before librsfa.so, so the
// library binds to these (tests/launch_recorder.py).  The device: 256 CUs, never
// capturing unless told so; occupancies and the counters' address are the test's.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string> kernels;
std::string lines;
std::map<std::string, int> occupancy;  // by part of the kernel's name
int capturing = 0;
char scratch[4096];      // address of the library's no-allocation buffer
char counters[1 << 21];  // what hipMalloc hands out
struct Config {
    unsigned grid[3], block[3];
    size_t lds;
    void* stream;
} config;

const char* area(uint64_t a) {
    if (a >= (uint64_t)scratch && a < (uint64_t)(scratch + sizeof(scratch))) return "scratch";
    if (a >= (uint64_t)counters && a < (uint64_t)(counters + sizeof(counters))) return "allocated";
    return "none";
}
}  // namespace

extern "C" {
struct Dim3 {
    unsigned x, y, z;
};

const char* recorder_lines() { return lines.c_str(); }
void recorder_clear() { lines.clear(); }
void recorder_occupancy(const char* part, int wgs) { occupancy[part] = wgs; }
void recorder_capturing(int on) { capturing = on; }

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[fn] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* stream) {
    config = Config{{g.x, g.y, g.z}, {b.x, b.y, b.z}, lds, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** stream) {
    *g = Dim3{config.grid[0], config.grid[1], config.grid[2]};
    *b = Dim3{config.block[0], config.block[1], config.block[2]};
    *lds = config.lds;
    *stream = config.stream;
    return 0;
}
int hipGetDevice(int* dev) { return *dev = 0; }
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* fn, int, size_t) {
    *n = 1;
    for (const auto& o : occupancy)
        if (kernels[fn].find(o.first) != std::string::npos) *n = o.second;
    return 0;
}
int hipMalloc(void** p, size_t n) {
    if (n > sizeof(counters)) return 2;
    *p = counters;
    return 0;
}
int hipFree(void*) { return 0; }
int hipMemset(void*, int, size_t) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void** p, const void*) {
    *p = scratch;
    return 0;
}
int hipStreamIsCapturing(void*, int* status) {
    *status = capturing;
    return 0;
}
// One line per launch: kernel, workgroups, threads, whether blocks go in pairs, and
// where the counters it gets lie.  clear_words takes their address first, the
// attention kernels take a struct by value that holds both.
int hipLaunchKernel(const void* fn, Dim3 grid, Dim3 block, void** args, size_t, void*) {
    const std::string name = kernels.count(fn) ? kernels[fn] : "?";
    uint64_t ticket;
    int32_t pairs = 0;
    const bool clear = name.find("clear_words") != std::string::npos;
    memcpy(&ticket, (const char*)args[0] + (clear ? 0 : RECORDER_TICKET_OFFSET), sizeof(ticket));
    if (!clear) memcpy(&pairs, (const char*)args[0] + RECORDER_PAIRS_OFFSET, sizeof(pairs));
    char tail[96];
    snprintf(tail, sizeof(tail), " %u %u %d %s\n", grid.x, block.x, pairs, area(ticket));
    lines += name + tail;
    return 0;
}
}
