// The stand-in runtime of hip_mock.cpp with a record of what is launched: each kernel's
// (demangled) name as it is queued, "null workspace" after a lane-layout kernel that was
// given none, and a capture by the caller that can be switched on. Test infrastructure only.
#include <hip/hip_runtime.h>

#include <cxxabi.h>

#include <string>
#include <vector>

#include "kwgpu_internal.h"

#define __hipRegisterFunction base_register_function
#define hipLaunchKernel base_launch_kernel
#include "hip_mock.cpp"
#undef __hipRegisterFunction
#undef hipLaunchKernel

static std::map<const void*, std::string>& kernel_names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::vector<std::string> g_launched;
bool g_caller_captures = false;

extern "C" {
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, uint3*,
                           uint3*, dim3*, dim3*, int*) {
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string s = d ? d : name;
    std::free(d);
    s = s.substr(0, s.rfind('('));                      // no arguments,
    if (s.compare(0, 5, "void ") == 0) s = s.substr(5);  // no return type,
    const size_t at = s.find("(anonymous namespace)::");
    kernel_names()[host] = at == std::string::npos ? s : s.substr(at + 23);  // no namespace
}
hipError_t hipLaunchKernel(const void* host, dim3 g, dim3 b, void** args, size_t shm, hipStream_t s) {
    const std::string& name = kernel_names()[host];
    g_launched.push_back(name);
    if (name.find("fd1d_lane") == 0 && !static_cast<const kwgpu::FdBatch*>(args[0])->ws)
        g_launched.push_back("null workspace");
    return base_launch_kernel(host, g, b, args, shm, s);
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
    *st = g_caller_captures || g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
}
