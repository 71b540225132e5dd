// launch_recorder.cpp — stands in for the HIP runtime where the library launches kernels, so that the
// launches of a call can be seen without a GPU: loaded before libsapient_hip.so with global symbols, it
// takes the library's kernel registrations and launches, refuses what HIP refuses (a launch of 2^32 or more
// work-items in x, an empty or oversized grid or block) and keeps the rest as lines
// "kernel grid.x grid.y block.x". Nothing is run, so pointers may be any address.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::string& lines() {
    static std::string s;
    return s;
}
}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string s = d ? d : name;
    std::free(d);
    // "void sph::(anonymous namespace)::kernel<...>(...)" -> "kernel<...>"
    const std::string ns = "(anonymous namespace)::";
    const size_t at = s.find(ns);
    if (at != std::string::npos) s = s.substr(at + ns.size());
    for (size_t p; (p = s.find(ns)) != std::string::npos;) s.erase(p, ns.size());
    int depth = 0;
    size_t end = 0;
    for (; end < s.size() && (depth > 0 || s[end] != '('); ++end) depth += s[end] == '<' ? 1 : s[end] == '>' ? -1 : 0;
    s.resize(end);
    for (size_t p; (p = s.find(' ')) != std::string::npos;) s.erase(p, 1);
    names()[host] = s;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
    const uint64_t threads = (uint64_t)b.x * b.y * b.z;
    if (g.x == 0 || g.y == 0 || g.z == 0 || threads == 0 || threads > 1024 || g.x > INT32_MAX || g.y > 65536 || g.z > 65536 ||
        (uint64_t)g.x * b.x > UINT32_MAX)
        return hipErrorInvalidConfiguration;
    lines() += names()[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " + std::to_string(b.x) + "\n";
    return hipSuccess;
}

// What the launchers ask of the runtime beside: an MI355X, no capture.
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    if (a != hipDeviceAttributeMultiprocessorCount) return hipErrorInvalidValue;
    *v = 256;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

// The launches since the last call of this.
const char* take_launches() {
    static std::string out;
    out = lines();
    lines().clear();
    return out.c_str();
}
}
