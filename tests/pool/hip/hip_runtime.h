// The few runtime calls the block pool makes, over a device of fixed size that
// exists only as bookkeeping: what is allocated, the error the last call left,
// and a hook that runs while a thread waits for the device.
#pragma once
#include <stddef.h>
#include <stdint.h>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidValue = 1 };
typedef void* hipStream_t;
const char* hipGetErrorString(hipError_t e);
hipError_t hipMalloc(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipGetDevice(int* dev);
hipError_t hipDeviceSynchronize();
hipError_t hipGetLastError();
hipError_t hipMemGetInfo(size_t* free_b, size_t* total_b);
