// Held while the kernels of one product are enqueued that pass numbers on in the caller's workspace.  One workspace serves a stream for all threads of a process, and a
// stream runs what it is given in order, but between the launches of one thread's product another's must not get in.
#pragma once
#include <mutex>

std::mutex& workspace_lock();      // matmul_library.hip
