// Copies of large device arrays into the caller's pageable memory.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <vector>

namespace hlb {

struct HostSegment {
  void* dst;         // caller's memory
  const void* src;   // device memory
  size_t bytes;
};

// Copies the segments in order on `stream` and returns when all of them are
// in place (hipSuccess or the first error).
hipError_t copy_to_host(const std::vector<HostSegment>& segments, hipStream_t stream);

// The pinned staging memory is shared by the process: allocated by the first
// large copy and given back with the last user (one acquire and one release
// per solver).
void staging_acquire();
void staging_release();

}  // namespace hlb
