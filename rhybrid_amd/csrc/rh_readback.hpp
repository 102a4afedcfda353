// Grid arrays to the caller's memory: the planes of an SoA array on the device
// become interleaved doubles on the host (the layout of the reference's
// user-data arrays, src/hybrid.h), cell by cell.
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>

namespace rh {

// A context's pinned staging ring: READBACK_SLOTS slots of READBACK_SLOT_BYTES,
// allocated and freed with the context.
constexpr int READBACK_SLOTS = 4;
constexpr size_t READBACK_SLOT_BYTES = size_t(1) << 20;

template <typename Real, int DIM>
inline void interleave(const Real* __restrict__ planes, size_t stride, size_t n, double* __restrict__ out) {
    for (size_t i = 0; i < n; ++i)
        for (int l = 0; l < DIM; ++l) out[i * DIM + l] = (double)planes[l * stride + i];
}

template <typename Real>
inline void interleave(const Real* planes, size_t stride, size_t n, int dim, double* out) {
    if (dim == 3) interleave<Real, 3>(planes, stride, n, out);
    else if (dim == 1) interleave<Real, 1>(planes, stride, n, out);
    else
        for (size_t i = 0; i < n; ++i)
            for (int l = 0; l < dim; ++l) out[i * dim + l] = (double)planes[l * stride + i];
}

// Bound by the host, which first touches the caller's array here (it is
// usually new): the array goes over in chunks through the pinned ring, copied
// by the device while earlier chunks are converted out of the cache.
// cellRhoQi, cellJi and faceB of 128x96x96 take 5.8 ms, 9.4 in one piece each
// through pageable memory; of 16^3 60 us against 90.  (Converted by up to
// eight threads the large box takes 4.3 to 9.3 ms and a 68x80x20 box up to
// 3 ms instead of 0.6: starting and waking threads costs milliseconds now and
// then.)
// copy(c, first cell, cells) enqueues chunk c's planes into slot
// c % READBACK_SLOTS; wait(c) returns when they are there.  Both may throw.
template <typename Real, typename Copy, typename Wait>
void readback(size_t nc, int dim, double* data, const Real* const* slot, size_t chunk, Copy&& copy, Wait&& wait) {
    const size_t chunks = (nc + chunk - 1) / chunk;
    auto cells = [&](size_t c) { return std::min(chunk, nc - c * chunk); };
    for (size_t c = 0; c < std::min(chunks, (size_t)READBACK_SLOTS); ++c) copy(c, c * chunk, cells(c));
    for (size_t c = 0; c < chunks; ++c) {
        wait(c);
        interleave<Real>(slot[c % READBACK_SLOTS], chunk, cells(c), dim, data + c * chunk * dim);
        const size_t n = c + READBACK_SLOTS;  // into the slot that is free now
        if (n < chunks) copy(n, n * chunk, cells(n));
    }
}

// A context's staging ring for every array it reads back.  Host threads may
// read arrays of one context side by side: a read holds the ring, and the
// events of its slots, until its last chunk is converted, and the others wait
// for it (they would share the one stream and its copy engine anyway).
class ReadbackRing {
public:
    void* mem = nullptr;  // READBACK_SLOTS * READBACK_SLOT_BYTES

    // copy(c, to, stride, first cell, cells) enqueues chunk c's planes to `to`,
    // `stride` values apart; wait(c) as above.
    template <typename Real, typename Copy, typename Wait>
    void read(size_t nc, int dim, double* data, Copy&& copy, Wait&& wait) {
        std::lock_guard<std::mutex> held(mu);
        const size_t chunk = std::min(nc, READBACK_SLOT_BYTES / (dim * sizeof(Real)));
        Real* slot[READBACK_SLOTS];
        for (int q = 0; q < READBACK_SLOTS; ++q)
            slot[q] = reinterpret_cast<Real*>(static_cast<char*>(mem) + q * READBACK_SLOT_BYTES);
        readback<Real>(
            nc, dim, data, slot, chunk,
            [&](size_t c, size_t first, size_t n) { copy(c, slot[c % READBACK_SLOTS], chunk, first, n); }, wait);
    }

private:
    std::mutex mu;
};

}  // namespace rh
