// plb_xfer.hpp -- chunked copies between the caller's arrays and device
// layouts (plb_xfer.hip).
#pragma once

#include <functional>
#include <vector>

#include "plb_internal.hpp"

namespace plb {

// Enqueues, on the copy's stream, the kernel that fills (read-backs) or takes
// (writes) the slot of nodes first .. first + m - 1: `item` bytes per node
// and array, the arrays one after the other.
using ChunkKernel = std::function<int(int64_t first, int64_t m, void* slot)>;

// Every array holds n items; returns when all of it has arrived.
int download(int device, hipStream_t s, int64_t n, size_t item, const std::vector<char*>& arrays,
             const ChunkKernel& kernel);
int upload(int device, hipStream_t s, int64_t n, size_t item, const void* array, const ChunkKernel& kernel);

// Whether p lies in page-locked memory that kernels reach by the same pointer.
bool page_locked(const void* p);

// +1 for a context that is created, -1 for one that goes: the kept slots go with the last.
void xfer_context(int add);

}  // namespace plb
