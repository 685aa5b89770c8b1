// Host staging of a plan's own host calls.  Host code without HIP.
#pragma once
#include <cstddef>
#include <new>

namespace mtk {

// n floats, 8-byte aligned, pinned or, where that cannot be had, ordinary
// memory (copies then stage and wait inside the runtime).  Pinned: get(bytes) ->
// memory or null, put(memory).
template <typename Pinned> struct Staging {
    float *p = nullptr;
    bool pinned = false;
    Staging() = default;
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;
    void alloc(size_t n) {
        release();
        p = (float *)Pinned::get(sizeof(float) * n);
        pinned = p != nullptr;
        if (!p) p = (float *)::operator new(sizeof(float) * n);
    }
    void release() {
        if (p && pinned) Pinned::put(p);
        if (p && !pinned) ::operator delete(p);
        p = nullptr;
    }
    ~Staging() { release(); }
};

}  // namespace mtk
