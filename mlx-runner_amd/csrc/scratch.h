// Device scratch kept between calls: buffers that grow to the largest size asked for.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stddef.h>

namespace mlxr {

// p holds at least `need` elements afterwards; its contents are not kept. On an error there is no buffer.
template <typename T>
hipError_t scratch_grow(T*& p, size_t& have, size_t need, hipStream_t s) {
    if (need <= have) return hipSuccess;
    if (p) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(p);
        p = nullptr;
        have = 0;
    }
    if (hipError_t e = hipMalloc(reinterpret_cast<void**>(&p), need * sizeof(T))) {
        p = nullptr;
        return e;
    }
    have = need;
    return hipSuccess;
}

// The same, its first `zeroed` elements (counters that every launch leaves at zero) cleared when the buffer is
// new: on the stream whose launches count in it, which nothing else orders after a clear on another one (it is
// a non-blocking stream). A buffer that could not be cleared is not kept.
template <typename T>
hipError_t scratch_grow_zeroed(T*& p, size_t& have, size_t need, size_t zeroed, hipStream_t s) {
    if (need <= have) return hipSuccess;
    if (hipError_t e = scratch_grow(p, have, need, s)) return e;
    hipError_t e = hipMemsetAsync(p, 0, zeroed * sizeof(T), s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        (void)hipFree(p);
        p = nullptr;
        have = 0;
    }
    return e;
}

}  // namespace mlxr
