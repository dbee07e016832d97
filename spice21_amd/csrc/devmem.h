// Device memory owned by one object.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "internal.h"

namespace s21 {

struct DevMem {
    void* p = nullptr;
    size_t bytes = 0;  // of the memory at p: a failed allocation leaves none
    DevMem() {}
    DevMem(const DevMem&) = delete;
    DevMem& operator=(const DevMem&) = delete;
    ~DevMem() { clear(); }
    void clear() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    void alloc(size_t b) {
        clear();
        if (!b) return;
        void* q = nullptr;
        const hipError_t e = hipMalloc(&q, b);
        if (e != hipSuccess) fail(S21_DEVICE, std::string("HIP: ") + hipGetErrorString(e));
        p = q;
        bytes = b;
    }
    // Memory of b bytes, kept from before where it has that size.
    void keep(size_t b) {
        if (bytes != b) alloc(b);
    }
    template <typename V>
    V* as() const {
        return (V*)p;
    }
};

}  // namespace s21
