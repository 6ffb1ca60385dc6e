// A stand-in for the HIP runtime on the CPU: device memory is host memory, no
// kernel runs.  Linked into a test program ahead of the library, it takes the
// library's calls; one or two allocations can be made to fail, and every launch and
// copy is checked: a pointer a kernel gets must be null or lie in memory that
// is allocated at that time, and what a launch's other arguments need must be
// there.  Host C++ only.
#pragma once

#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace stand_in {

inline std::map<char*, size_t> live;                       // allocated now
inline std::map<const void*, std::string>& kernels() {     // demangled, by host function (the library's
    static std::map<const void*, std::string> k;           // constructors fill it, before this program's run)
    return k;
}
inline std::vector<std::string> faults;
inline long allocs = 0, launches = 0, fail_at[2] = {-1, -1};     // the allocations that fail (from 1)

inline hipError_t get(void** p, size_t n) {
    *p = nullptr;
    ++allocs;
    if (allocs == fail_at[0] || allocs == fail_at[1]) return hipErrorOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    live[(char*)*p] = n;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t drop(void* p) {
    if (!p) return hipSuccess;
    if (!live.erase((char*)p)) faults.push_back("free of memory that is not allocated");
    else free(p);
    return hipSuccess;
}
// bytes from p to the end of its allocation, -1 if it is in none
inline long room(const void* p) {
    auto it = live.upper_bound((char*)p);
    if (it == live.begin()) return -1;
    --it;
    const long off = (const char*)p - it->first;
    return off <= (long)it->second ? (long)it->second - off : -1;
}
inline void need(const void* p, size_t n, const std::string& what) {
    if (room(p) < (long)n) faults.push_back(what);
}
inline void copy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    if (k == hipMemcpyHostToDevice) need(d, n, "copy to device memory that is not there");
    if (k == hipMemcpyDeviceToHost) need(s, n, "copy from device memory that is not there");
    if (faults.empty()) memcpy(d, s, n);
}

// the types of a demangled kernel's parameters
inline std::vector<std::string> parameters(const std::string& f) {
    int depth = 0;
    size_t open = f.rfind(')');
    for (size_t i = open; i-- > 0;) {           // the list that ends the name
        if (f[i] == ')') ++depth;
        if (f[i] == '(' && depth-- == 0) { open = i; break; }
    }
    std::vector<std::string> out(1);
    depth = 0;
    for (size_t i = open + 1; i < f.rfind(')'); ++i) {
        if (f[i] == '<' || f[i] == '(') ++depth;
        if (f[i] == '>' || f[i] == ')') --depth;
        if (f[i] == ',' && depth == 0) out.emplace_back();
        else out.back() += f[i];
    }
    return out;
}

inline void launch(const void* fn, void** args) {
    ++launches;
    const std::string& name = kernels()[fn];
    const std::vector<std::string> p = parameters(name);
    const auto ptr = [&](size_t i) { return *(char**)args[i]; };
    const auto num = [&](size_t i) { return *(int*)args[i]; };
    for (size_t i = 0; i < p.size(); ++i)
        if (p[i].back() == '*' && ptr(i) && room(ptr(i)) < 0)
            faults.push_back(name + ": argument " + std::to_string(i) + " is not allocated");
    const auto is = [&](const char* k) { return name.find(k) != std::string::npos; };
    // what may be null in some launches and not in others
    if (is("::output_kernel(") && ptr(6) && !(ptr(9) && ptr(10))) faults.push_back(name + ": targets without dY or loss");
    if (is("::pbuild4_kernel<") && num(11) > 0) {
        need(ptr(9), 16 * (size_t)num(11), name + ": programs are not staged");
        need(ptr(10), 16 * (size_t)num(11), name + ": programs do not fit");
    }
}

}  // namespace stand_in

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return stand_in::get(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return stand_in::get(p, n); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipFree(void* p) { return stand_in::drop(p); }
hipError_t hipHostFree(void* p) { return stand_in::drop(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { stand_in::copy(d, s, n, k); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    stand_in::copy(d, s, n, k);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    stand_in::need(d, n, "clearing device memory that is not there");
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    stand_in::launch(f, args);
    return hipSuccess;
}
static struct { dim3 g, b; size_t m; hipStream_t s; } stand_in_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
    stand_in_call = {g, b, m, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = stand_in_call.g; *b = stand_in_call.b; *m = stand_in_call.m; *s = stand_in_call.s;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    stand_in::kernels()[fn] = d ? d : name;
    free(d);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {      // (a macro: the versioned name)
    memset((void*)p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 4; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }
}
