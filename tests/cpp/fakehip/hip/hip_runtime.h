// The few runtime calls that tuvok_amd/csrc/devmem.cpp makes, over host memory with a
// limit: for devmem_check.cpp, which runs without a GPU.
#pragma once
#include <cstddef>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
struct hipDeviceProp_t {
  size_t totalGlobalMem;
};
hipError_t hipMalloc(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipGetDevice(int* device);
hipError_t hipSetDevice(int device);
hipError_t hipDeviceSynchronize();
hipError_t hipGetLastError();
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int device);
