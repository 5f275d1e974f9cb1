// A host stand-in for the HIP runtime and the library's kernels, so that the runtime's own code
// (runtime.cpp, evaluator.cpp, server.cpp, autotune.cpp) runs without a GPU.
//
// A stream is a queue of operations that run only when something waits for them: a synchronization,
// an event wait, or a step the test takes. Copies move their bytes when they run, as a DMA would, so
// staging memory reused too early shows as wrong bytes. Kernels do nothing, except that the upload
// kernel copies. Device memory is reserved address space, touched only by copies.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <vector>

namespace model {

struct Copy {
    size_t bytes;
    bool kernel;  // by the upload kernel, else by a copy command
};
extern std::vector<Copy> uploads;       // host-to-device copies queued so far
extern uint64_t launches;               // kernel launches so far
extern bool refuse_launch;              // the next kernel launch is refused (and the flag cleared)
extern float elapsed_ms;                // what hipEventElapsedTime reports
extern uint64_t records_while_capturing;  // event records on a stream that a caller captures
extern uint64_t destroyed_graphs;       // executable graphs destroyed so far
extern size_t free_bytes;               // what hipMemGetInfo reports

extern uint64_t ip_launches, ip_finish_launches;  // of the inner product, and of the one inside the finish
extern std::function<void()> on_launch;  // called at every kernel launch
extern std::function<void(size_t)> on_malloc;  // called with the bytes of every device allocation

void kernel();                          // one launch: counted, or refused
void queue_copy(void* dst, const void* src, size_t bytes, hipStream_t s);
void set_capturing(hipStream_t s, bool on);  // a capture by the caller, begun or ended
size_t pending(hipStream_t s);          // operations queued on s that have not run
bool step(hipStream_t s);               // runs one (false: none could)
size_t mapped();                        // device bytes held by hipMalloc and hipMallocAsync

}  // namespace model
