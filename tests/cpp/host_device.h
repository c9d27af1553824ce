// Knobs of host_device.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

extern std::atomic<int> g_copy_us;    // what every copy waits before it touches its bytes
extern std::atomic<int> g_mallocs;    // hipMalloc calls so far
extern std::atomic<int> g_malloc_us;  // what each takes
extern std::atomic<bool> g_no_threads;  // the process has reached its limit of threads
