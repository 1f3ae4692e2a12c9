// The HIP runtime's calls that the EXL3 linears reach, accepted and counted in place of the runtime's own (loaded with
// global symbols ahead of the library): what a call asks the runtime for beside launches, on a host without a device.
#include <cstddef>

extern "C" {
int counted_launches = 0;
int counted_others = 0;
int __hipPushCallConfiguration(...) { return 0; }
int __hipPopCallConfiguration(...) { return 0; }
int hipLaunchKernel(const void*, ...) { return ++counted_launches, 0; }
int hipFuncSetAttribute(const void*, int, int) { return ++counted_others, 0; }
int hipGetSymbolAddress(void** at, const void*) { return ++counted_others, *at = reinterpret_cast<void*>(size_t{1} << 40), 0; }
int hipGetDevice(int* device) { return *device = 0, 0; }
int hipGetLastError() { return 0; }
}
