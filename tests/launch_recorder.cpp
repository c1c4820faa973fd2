// The HIP runtime functions libxla_amd_qmm.so calls, as stand-ins that note each launch and start nothing: loaded in
// front of the library (tests/launch_recorder.py), they show without a GPU which kernels a call launches and how.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {
struct Dim {
  uint32_t x, y, z;
};
struct Configuration {
  Dim grid, block;
  size_t lds;
  void* stream;
};
std::map<const void*, std::string> names;      // host handle of a kernel -> its device name
std::map<const void*, int> lds_limit;          // ... -> the dynamic LDS it was allowed
std::vector<Configuration> pending;
std::string notes;                             // one line per launch
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, Dim*, Dim*, int*) {
  names[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void* stream) {
  pending.push_back({grid, block, lds, stream});
  return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* lds, void** stream) {
  const Configuration c = pending.back();
  pending.pop_back();
  *grid = c.grid; *block = c.block; *lds = c.lds; *stream = c.stream;
  return 0;
}
int hipGetDevice(int* device) { *device = 0; return 0; }
int hipDeviceGetAttribute(int* value, int, int) { *value = 256; return 0; }  // (compute units: all that is asked for)
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "error"; }
int hipGetSymbolAddress(void** address, const void*) { *address = (void*)0x10000; return 0; }
int hipFuncSetAttribute(const void* kernel, int, int value) { lds_limit[kernel] = value; return 0; }
int hipLaunchKernel(const void* kernel, Dim grid, Dim block, void** args, size_t lds, void*) {
  // the first eight 8-byte words of the first argument: pointers and sizes where it is a struct of arguments
  uint64_t words[8];
  memcpy(words, args[0], sizeof(words[0]));
  const bool whole = names[kernel].find("QmmRowMajorArgs") != std::string::npos;
  if (whole) memcpy(words, args[0], sizeof(words));
  char line[1024];
  int at = snprintf(line, sizeof(line), "%s %u %u %u %u %u %u %zu %d", names[kernel].c_str(), grid.x, grid.y, grid.z,
                    block.x, block.y, block.z, lds, lds_limit.count(kernel) ? lds_limit[kernel] : 64 * 1024);
  for (int i = 0; i < (whole ? 8 : 1); ++i) at += snprintf(line + at, sizeof(line) - at, " %llu", (unsigned long long)words[i]);
  notes += line;
  notes += '\n';
  return 0;
}
// The launches since the last call.
const char* take_notes() {
  static std::string out;
  out.swap(notes);
  notes.clear();
  return out.c_str();
}
}
