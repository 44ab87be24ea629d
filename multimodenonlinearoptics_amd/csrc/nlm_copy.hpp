// nlm_copy.hpp -- copies between the device and host memory (nlm_copy.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <string>

int set_err(int kind, const std::string& msg);

// Copies to and from a caller's pageable memory (nlm_copy.hip).  nlm_to_host returns
// when every item is in place (items with a null host pointer are skipped) and the
// stream's work before it is done; nlm_to_device when `host` may be reused.
struct HostCopy {
  void* host;
  const void* dev;
  size_t bytes;
};
int nlm_to_host(const HostCopy* items, int n, hipStream_t s);
int nlm_to_device(void* dev, const void* host, size_t bytes, hipStream_t s);
