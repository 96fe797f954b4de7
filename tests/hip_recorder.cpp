// The part of the HIP runtime's interface that the library's host code calls, without a device: launches are written down instead of
// run, allocations hand out addresses that nobody reads.  Loaded in front of the library, in a process of its own
// (tests/test_host_dispatch.py), so that the host side of a call can be looked at on any machine.
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct dim3 {
  uint32_t x, y, z;
};

struct Launch {
  const char* name;       // mangled name of the kernel
  uint32_t grid, block;   // along x
  unsigned char arg0[120]; // the first argument (GemmArgs, or PadCopy)
  unsigned char arg1[48]; // the second (PadCopy, or Touch, which ends a NormedGemm)
};

static std::map<const void*, std::string> names;
static std::vector<Launch> launches;
static uintptr_t next_address = uintptr_t(1) << 40;
static struct {
  dim3 grid, block;
  size_t shared;
  void* stream;
} config;

extern "C" {

void recorder_reset() { launches.clear(); }
int recorder_count() { return (int)launches.size(); }
const Launch* recorder_launch(int i) { return &launches[i]; }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
  names[host] = device;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, void* stream) {
  config = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, void** stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return 0;
}
int hipLaunchKernel(const void* host, dim3 grid, dim3 block, void** args, size_t, void*) {
  Launch l = {names[host].c_str(), grid.x, block.x, {}, {}};
  const bool copy = std::strstr(l.name, "pad_copy_kernel") != nullptr;
  if (copy) {
    std::memcpy(l.arg0, args[0], 48);
    std::memcpy(l.arg1, args[1], 48);
  } else if (std::strstr(l.name, "gemm") != nullptr && std::strstr(l.name, "reduce") == nullptr) {
    std::memcpy(l.arg0, args[0], sizeof(l.arg0));
    if (std::strstr(l.name, "5Touch") != nullptr) std::memcpy(l.arg1, args[1], 40);
    if (std::strstr(l.name, "gemm_normed") != nullptr) std::memcpy(l.arg1, static_cast<unsigned char*>(args[0]) + 200, 40);
  }
  launches.push_back(l);
  return 0;
}
int hipMalloc(void** p, size_t bytes) {
  *p = reinterpret_cast<void*>(next_address);
  next_address += (bytes + 4095) / 4096 * 4096;
  return 0;
}
int hipFree(void*) { return 0; }
int hipGetDevice(int* device) { return *device = 0; }
int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipDeviceGetAttribute(int* value, int, int) {
  *value = 256;  // (only the number of compute units is asked for)
  return 0;
}
int hipGetDevicePropertiesR0600(void*, int) { return 1; }
int hipGetSymbolAddress(void** p, const void*) {
  *p = reinterpret_cast<void*>(uintptr_t(1) << 39);
  return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "recorded"; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipMemcpy(void*, const void*, size_t, int) { return 0; }
int hipMemset(void*, int, size_t) { return 0; }

}  // extern "C"
