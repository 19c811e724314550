// host_copy.h -- large results from device memory to a caller's ordinary
// (pageable) host memory.
//
// The runtime's own copy into pageable memory runs on one thread, which also
// takes the page faults of a fresh array: 10 GB/s for the 226 MB of fields of
// a 192^3 lattice.  Here several threads each keep two 2 MiB pinned buffers,
// one being filled by the device while the other is copied out, so that the
// faults and the copies of different parts run side by side.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>

namespace lbf {

// The pinned buffers and events of one GPU (32 MiB), shared by every object
// of the process that holds one and released with the last of them.
class HostStage;

// Copies `bytes` from device memory to dst, ordered after the work queued on
// s (a created stream), and returns when dst is complete.  Works on the
// stream's device, whichever is current.  `stage` is the caller's handle for
// that device, taken on the first large copy and kept; any number of threads,
// each with its own handle, may copy at once.  dst may also be pinned or device
// memory.
hipError_t copy_to_host(std::shared_ptr<HostStage>& stage, void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace lbf
