// broadcast_plan.hpp -- dims and index arithmetic of broadcast_to: plain C++
// (constexpr, so that the kernels and the host share it).
#pragma once

#include <cstddef>
#include <cstdint>

namespace tlhip {

// broadcast_to: target dims and, per target dim, the input stride (0 where
// the input has size 1 or no dim)
struct BcastDims {
    int nd = 0;
    int64_t shape[8] = {};
    int64_t xstride[8] = {};
};

// Dims of 1 dropped, neighbours that advance together (or both repeat)
// merged: fewer divisions per element, longer inner rows.
constexpr BcastDims bcast_merge(const BcastDims& full) {
    BcastDims b;
    for (int i = 0; i < full.nd; i++) {
        if (full.shape[i] == 1) continue;
        if (b.nd && (full.xstride[i] ? b.xstride[b.nd - 1] == full.xstride[i] * full.shape[i] : b.xstride[b.nd - 1] == 0)) {
            b.shape[b.nd - 1] *= full.shape[i];
            b.xstride[b.nd - 1] = full.xstride[i];
            continue;
        }
        b.shape[b.nd] = full.shape[i];
        b.xstride[b.nd++] = full.xstride[i];
    }
    if (!b.nd) {
        b.nd = 1;
        b.shape[0] = 1;
    }
    return b;
}

// Whether the 16-byte kernel (V elements per thread) takes merged dims of
// `total` elements on 16-byte aligned tensors: the innermost dim a multiple of
// V and either contiguous or repeated, every other stride a multiple of V, and
// at most 2^32 - 256 vectors, which bounds every extent it counts in 32 bits
// (the innermost in vectors).
constexpr bool bcast_wide_ok(const BcastDims& b, int64_t total, int V) {
    const int l = b.nd - 1;
    bool ok = total >= 4096 && total / V <= 0xffffff00ll && b.shape[l] % V == 0 && b.xstride[l] <= 1;
    for (int i = 0; i < l; i++) ok = ok && (b.xstride[l] == 0 || b.xstride[i] % V == 0);
    return ok;
}

// Input element that target elements V g .. V g + V - 1 start at (wide form).
constexpr size_t bcast_wide_src(const BcastDims& b, uint32_t g, int V) {
    const int l = b.nd - 1;
    const uint32_t per = (uint32_t)(b.shape[l] / V);   // (the extent itself may pass 32 bits)
    size_t src = (size_t)(g % per) * V * b.xstride[l];
    uint32_t rem = g / per;
    for (int i = l - 1; i >= 0; i--) {
        const uint32_t sh = (uint32_t)b.shape[i];
        src += (size_t)(rem % sh) * b.xstride[i];
        rem /= sh;
    }
    return src;
}

// Input element of target element g (one element per thread).
constexpr int64_t bcast_src(const BcastDims& b, int64_t g) {
    int64_t src = 0;
    for (int i = b.nd - 1; i >= 0; i--) {
        src += g % b.shape[i] * b.xstride[i];
        g /= b.shape[i];
    }
    return src;
}

}  // namespace tlhip
