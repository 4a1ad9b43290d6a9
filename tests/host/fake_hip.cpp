// A HIP runtime without a GPU for the dispatch tests: the calls that the library makes to load its code objects and
// launch kernels, recorded by kernel name. Loaded with global visibility before libnspeech_rocm.so, whose HIP
// references then bind to these definitions. No kernel runs and no pointer is read.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <string>

namespace {
int g_lds = 163840, g_cus = 256, g_occupancy = 1;
std::string g_log, g_out;
}  // namespace

extern "C" {

void fake_hip_set(int lds, int cus, int occupancy) {
  g_lds = lds;
  g_cus = cus;
  g_occupancy = occupancy;
}

// The launches since the last call: "name gx gy gz block lds n" lines, n the tile argument of the conv's record kernels
// (their fourth), 0 for others.
const char* fake_hip_take_log(void) {
  g_out.swap(g_log);
  g_log.clear();
  return g_out.c_str();
}

hipError_t hipGetDevice(int* dev) {
  *dev = 0;
  return hipSuccess;
}

hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}

hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? g_lds : a == hipDeviceAttributeMultiprocessorCount ? g_cus : 0;
  return hipSuccess;
}

hipError_t hipModuleLoadData(hipModule_t* m, const void*) {
  *m = (hipModule_t)&g_lds;
  return hipSuccess;
}

hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
  *f = (hipFunction_t)strdup(name);
  return hipSuccess;
}

hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) {
  *n = g_occupancy;
  return hipSuccess;
}

hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned,
                                 unsigned, unsigned lds, hipStream_t, void** params, void**) {
  const char* name = (const char*)f;
  const bool tiles = !std::strncmp(name, "nsrk_conv1d_pr_", 15) || !std::strncmp(name, "nsrk_conv1d_ps", 14);
  char line[256];
  std::snprintf(line, sizeof(line), "%s %u %u %u %u %u %d\n", name, gx, gy, gz, bx, lds, tiles ? *(const int*)params[3] : 0);
  g_log += line;
  return hipSuccess;
}

hipError_t hipGetLastError(void) { return hipSuccess; }

const char* hipGetErrorString(hipError_t) { return "fake"; }

hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = &g_lds;
  return hipSuccess;
}

}  // extern "C"
