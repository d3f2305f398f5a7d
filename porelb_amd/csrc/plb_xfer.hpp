// plb_xfer.hpp -- chunked copies between the caller's arrays and device
// layouts (plb_xfer.hip).
#pragma once

#include "plb_internal.hpp"

namespace plb {

// Enqueues, on the copy's stream, the kernel that fills (read-backs) or takes
// (writes) the slot of nodes first .. first + m - 1: `item` bytes per node
// and array, the arrays one after the other.
// Refers to the caller's function object for the length of the copy.
class ChunkKernel {
public:
    template <typename F>
    ChunkKernel(const F& f)
        : object_(&f), call_([](const void* o, int64_t first, int64_t m, void* slot) { return (*(const F*)o)(first, m, slot); })
    {
    }
    int operator()(int64_t first, int64_t m, void* slot) const { return call_(object_, first, m, slot); }

private:
    const void* object_;
    int (*call_)(const void*, int64_t, int64_t, void*);
};

// The caller's arrays, one for each of the parts that the kernels lay out.
struct Arrays {
    char* at[Q - 1];
    size_t n = 0;
    Arrays() = default;
    Arrays(void* one) { add(one); }
    void add(void* a) { at[n++] = (char*)a; }
};

// Every array holds n items; returns when all of it has arrived.
int download(int device, hipStream_t s, int64_t n, size_t item, const Arrays& arrays, const ChunkKernel& kernel);
int upload(int device, hipStream_t s, int64_t n, size_t item, const void* array, const ChunkKernel& kernel);

// Whether p lies in page-locked memory that kernels reach by the same pointer.
bool page_locked(const void* p);

// +1 for a context that is created, -1 for one that goes: the kept slots go with the last.
void xfer_context(int add);

}  // namespace plb
