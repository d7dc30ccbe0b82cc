// Which kernel a conv's launch takes, with how many workgroups and how much LDS, without a device: the runtime's entry points and the direct-dispatch
// layer are taken by the functions below (an executable's definitions come before a library's).
// Reads lines "alone|packed|transformed|group|refused|refused_group C K H W R S stride pad tile_hint small flags times" (flags: bits of the job id), calls
// each layer that often and prints a line: the plan's workgroups, then "kernel grid dynamic_lds allowed_lds" per launch, separated by ';'.
// packed, transformed: held by launch packing until all are in; group: each call has the layer twice.  refused: the runtime refuses the launch
// (hipErrorInvalidValue); printed is what the call returned.

#include "../../paella_amd/csrc/hip/direct_dispatch.h"
#include "paella_ops.h"

#include <cxxabi.h>

#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <map>
#include <sstream>
#include <string>

namespace {

std::map<const void*, std::string>& names() {  // filled while the libraries are loaded, before main
    static std::map<const void*, std::string> m;
    return m;
}
std::map<const void*, int> g_allowed_lds;
std::string g_out;
bool g_refuse = false;
hipError_t g_last_error = hipSuccess;
char g_queue;  // its address is the one direct queue's handle

struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_call;

void note(const void* kernel, dim3 grid, size_t lds) {
    std::string name = names()[kernel];
    if (char* plain = abi::__cxa_demangle(name.c_str(), nullptr, nullptr, nullptr)) {
        name = plain;
        std::free(plain);
    }
    const std::string unnamed = "(anonymous namespace)::";  // reduced to its own name and template arguments
    for (size_t at; (at = name.find(unnamed)) != std::string::npos;) name.erase(at, unnamed.size());
    if (name.rfind("void ", 0) == 0) name = name.substr(5);
    name = name.substr(0, name.find('('));
    for (size_t at; (at = name.find(' ')) != std::string::npos;) name.erase(at, 1);
    std::ostringstream s;
    s << (g_out.empty() ? "" : ";") << name << ' ' << grid.x << ' ' << lds << ' ' << g_allowed_lds[kernel];
    g_out += s.str();
}

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host_function, char*, const char* device_name, unsigned, void*, void*, void*, void*, int*) {
    names()[host_function] = device_name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    g_call = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = g_call.grid;
    *block = g_call.block;
    *lds = g_call.lds;
    *stream = g_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 grid, dim3, void**, size_t lds, hipStream_t) {
    note(kernel, grid, lds);
    return g_last_error = g_refuse ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* kernel, hipFuncAttribute what, int value) {
    if (what == hipFuncAttributeMaxDynamicSharedMemorySize) g_allowed_lds[kernel] = value;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes*, const void*) { return hipErrorNoDevice; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last_error;
    g_last_error = hipSuccess;
    return e;
}

int paella_direct_queue_shared(void** queue) {
    *queue = &g_queue;
    return 0;
}
}

namespace paella {
int g_direct_queue_count = 1;
DirectQueue* direct_queue_lookup_slow(void* handle) { return handle == &g_queue ? reinterpret_cast<DirectQueue*>(&g_queue) : nullptr; }
bool direct_queue_ordered(const DirectQueue*) { return false; }
const DirectKernel* direct_kernel(const void* host_function) { return reinterpret_cast<const DirectKernel*>(host_function); }
void direct_dispatch(DirectQueue*, const DirectKernel* kernel, dim3 grid, dim3, unsigned lds, const void*, size_t, size_t) { note(kernel, grid, lds); }
uint64_t direct_shared_min_waiting() { return 1; }
}  // namespace paella

int main() {
    alignas(16) static float memory[4];  // operands are not looked at
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string route;
        paella_conv_desc d = {};
        int hint = 0, small = -1, times = 1;
        unsigned flags = 0;
        if (!(in >> route >> d.C >> d.K >> d.H >> d.W >> d.R >> d.S >> d.stride_h >> d.pad_h >> hint >> small >> flags >> times)) return 1;
        d.stride_w = d.stride_h;
        d.pad_w = d.pad_h;
        d.dil_h = d.dil_w = d.groups = 1;
        d.act = PAELLA_ACT_RELU;
        paella_conv_plan plan;
        if (paella_conv2d_plan(&d, 0, hint, &plan)) return 1;
        if (small >= 0) plan.small = small;
        g_refuse = route.rfind("refused", 0) == 0;
        const bool packed = route == "packed" || route == "transformed", group = route.find("group") != std::string::npos;
        const paella_conv_operands member = {&plan, memory, memory, memory, nullptr, nullptr, memory, memory};
        const paella_conv_operands members[2] = {member, member};
        void* const stream = packed ? &g_queue : nullptr;
        if (packed && paella_pack_enable(1)) return 1;
        for (int i = 0; i < times; ++i) {
            const uint32_t job = (uint32_t)(i + 1) | flags;
            const int rc = group ? paella_conv2d_launch_group(members, 2, stream, job, nullptr)
                           : route == "transformed"
                               ? paella_conv2d_launch_transformed(&plan, memory, memory, memory, PAELLA_ACT_RELU, memory, memory, nullptr, nullptr, memory,
                                                                  memory, stream, job, nullptr)
                               : paella_conv2d_launch(&plan, memory, memory, memory, nullptr, nullptr, memory, memory, stream, job, nullptr);
            if (g_refuse) g_out = "returned " + std::to_string(rc);
            else if (rc) return 1;
        }
        if (packed && paella_pack_enable(0)) return 1;
        std::printf("%u %s\n", plan.dims.grid, g_out.c_str());
        g_out.clear();
        g_allowed_lds.clear();
    }
    return 0;
}
