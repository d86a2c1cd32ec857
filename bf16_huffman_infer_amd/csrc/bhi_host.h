// Host-side helpers shared by the C-ABI entry points: error reporting, and the order of launches.
#pragma once
#include <hip/hip_runtime.h>
#include <mutex>
#include "../../include/bhi.h"

// Records `msg` as the calling thread's last error and returns `code`.
int bhi_fail(int code, const char* msg);

// Fetches the status of the launch just enqueued; 0 or a positive hipError_t.
int bhi_launch_status(const char* what);

// Held while a call enqueues launches that hand data to each other in a workspace.  Callers' threads may share a
// stream and with it the workspace: only calls whose launches follow one another in the stream are ordered by it.
std::mutex& bhi_launches_mutex();
