// Device buffers and streams of one preparation step, released together.
#pragma once

#include <algorithm>
#include <vector>

#include "dgraph.hpp"

namespace blest {

struct Scratch {
    std::vector<void*> ptrs;
    template <class T>
    T* alloc(size_t count) {
        void* p = nullptr;
        BLEST_HIP(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)));
        ptrs.push_back(p);
        return static_cast<T*>(p);
    }
    ~Scratch() {
        for (void* p : ptrs) (void)hipFree(p);
    }
};

struct StreamGuard {
    hipStream_t s = nullptr;
    ~StreamGuard() {
        if (s) {
            (void)hipStreamSynchronize(s);
            (void)hipStreamDestroy(s);
        }
    }
};

// Waits for a stream that outlives the step, so that the step's buffers are free to go.
struct StreamDrain {
    hipStream_t s;
    ~StreamDrain() { (void)hipStreamSynchronize(s); }
};

inline dim3 grid_for(uint64_t items, unsigned block = 256) {
    return dim3(unsigned(std::max<uint64_t>(1, std::min<uint64_t>((items + block - 1) / block, 65536))));
}

template <class T>
T read_one(const T* d, hipStream_t s) {
    T v{};
    BLEST_HIP(hipMemcpyAsync(&v, d, sizeof(T), hipMemcpyDeviceToHost, s));
    BLEST_HIP(hipStreamSynchronize(s));
    return v;
}

}  // namespace blest
