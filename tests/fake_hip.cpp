// The HIP runtime's entry points that the library calls, as a recorder: nothing is launched.  Loaded in front of the
// library with global visibility, so that its calls end here.
#include <stddef.h>
#include <stdint.h>

#include <set>
#include <string>

struct Dim3 {
    uint32_t x, y, z;
};
static std::set<const void*> large;  // kernels that may use more than 64 KiB
static int attributes, launches, refused, grid_y;
static thread_local Dim3 config_grid, config_block;
static thread_local size_t config_lds;
static thread_local void* config_stream;

extern "C" {
int hipGetDevice(int* device) { return *device = 0; }
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void** address, const void*) {
    *address = reinterpret_cast<void*>(uintptr_t(1) << 32);
    return 0;
}
int hipFuncSetAttribute(const void* kernel, int, int) {
    ++attributes;
    large.insert(kernel);
    return 0;
}
int hipLaunchKernel(const void* kernel, Dim3 grid, Dim3, void**, size_t lds, void*) {
    ++launches;
    grid_y = (int)grid.y;
    refused += lds > 64 * 1024 && large.count(kernel) == 0;
    return 0;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
    config_grid = grid, config_block = block, config_lds = lds, config_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
    *grid = config_grid, *block = config_block, *lds = config_lds, *stream = config_stream;
    return 0;
}
int fake_attributes() { return attributes; }
int fake_launches() { return launches; }
int fake_grid_y() { return grid_y; }  // of the last launch
int fake_refused() { return refused; }  // launches with more LDS than their kernel was allowed
}
