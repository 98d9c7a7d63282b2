// mr_hostio.h -- the host-memory side of the trace entry points: device and
// pinned buffers kept between calls, and result copies into the caller's
// (pageable) arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <memory>
#include <vector>

namespace mr {

// Runs f(0) .. f(n - 1) on up to `threads` threads, this one among them.
// f must not throw.
void parallel_for(int64_t n, int threads, const std::function<void(int64_t)> &f);

// Threads worth using for `bytes` of host memory traffic.
int copy_threads(size_t bytes);

// What one host-memory call works with: a stream, a device buffer and pinned
// chunks.  Calls that overlap (other threads) each hold a stage of their own.
struct HostStage;

// A stage of the device that is current, whose device buffer holds at least
// `bytes`; null with *err set when an allocation fails.  Returned to the pool
// when the pointer dies.
struct StageReturn {
    void operator()(HostStage *s) const;
};
using StagePtr = std::unique_ptr<HostStage, StageReturn>;
StagePtr acquire_stage(size_t bytes, hipError_t *err);

hipStream_t stage_stream(const HostStage &s);
char *stage_device(const HostStage &s);

// One caller array and where its bytes start in the stage's device buffer.
struct HostPiece {
    char *host;
    size_t offset, bytes;
};

// Copies the pieces (ascending, non-overlapping offsets) into or out of the
// stage's device buffer, through the pinned chunks; both return when the
// copies are done, copy_out after everything enqueued on the stage's stream.
hipError_t copy_in(HostStage &s, const std::vector<HostPiece> &pieces);
hipError_t copy_out(HostStage &s, const std::vector<HostPiece> &pieces);

// Frees the larger device buffers of the stages not in use (the last field
// handle of the process died).
void trim_idle_stages();

// Frees every stage not in use.
void drop_idle_stages();

}  // namespace mr
