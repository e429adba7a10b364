// TEST INFRASTRUCTURE ONLY: see hip_runtime.h.
#pragma once
#include "hip_runtime.h"

hipError_t hipExtLaunchKernel(const void* kernel, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s,
                              hipEvent_t start, hipEvent_t stop, int flags);
