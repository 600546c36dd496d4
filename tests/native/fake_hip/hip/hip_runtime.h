// The part of the HIP runtime that the block pool calls, on the host.
#pragma once
#include <cstddef>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
hipError_t hipMalloc(void **p, size_t bytes);
hipError_t hipFree(void *p);
hipError_t hipGetDevice(int *device);
hipError_t hipGetLastError();
