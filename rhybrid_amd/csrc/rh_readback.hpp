// Grid arrays to the caller's memory: the planes of an SoA array on the device
// become interleaved doubles on the host (the layout of the reference's
// user-data arrays, src/hybrid.h), cell by cell.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <system_error>
#include <thread>
#include <vector>

namespace rh {

// A context's pinned staging ring: READBACK_SLOTS slots of READBACK_SLOT_BYTES,
// allocated and freed with the context.
constexpr int READBACK_SLOTS = 4;
constexpr size_t READBACK_SLOT_BYTES = size_t(1) << 20;
// Most threads of one read-back, the caller's own included, and the values
// that give each of them enough to do (a thread costs about 20 us to start).
constexpr int READBACK_THREADS = 8;
constexpr size_t READBACK_VALUES_PER_THREAD = size_t(1) << 17;

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

// Bound by the host: the doubles are first touched here (the caller's array is
// usually new, so the kernel clears its pages too), which one thread does at
// about 5 GB/s.  The array goes over in chunks through the pinned ring, copied
// by the device while earlier chunks are converted by up to eight threads.
// faceB of 128x96x96 (28 MB of doubles) takes 1.4 ms, 3.0 to 4.6 in one piece
// through pageable memory; of 160x128x128 3.9 against 8.0 (16 threads and
// slots of half the size: the same within the noise).  A small array is
// converted by the caller alone (16^3: 22 us against 31).
// copy(slot, offset of the first cell, cells): enqueues a chunk's planes into
// the slot; wait(slot): until it is there.  Both may throw.
template <typename Real, typename Copy, typename Wait>
void readback(size_t nc, int dim, double* data, const Real* const* slot, size_t chunk, Copy&& copy, Wait&& wait) {
    const size_t chunks = (nc + chunk - 1) / chunk;
    auto cells = [&](size_t c) { return std::min(chunk, nc - c * chunk); };
    auto convert = [&](size_t c) {
        interleave<Real>(slot[c % READBACK_SLOTS], chunk, cells(c), dim, data + c * chunk * dim);
    };
    std::atomic<size_t> next{0}, ready{0};  // chunks handed out, chunks on the host
    std::atomic<bool> stop{false};
    std::vector<std::atomic<bool>> done(chunks);
    for (auto& d : done) d.store(false, std::memory_order_relaxed);
    auto work = [&] {
        for (;;) {
            const size_t c = next.fetch_add(1, std::memory_order_relaxed);
            if (c >= chunks) return;
            while (ready.load(std::memory_order_acquire) <= c) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            convert(c);
            done[c].store(true, std::memory_order_release);
        }
    };
    const size_t most = std::min({(size_t)READBACK_THREADS, chunks, nc * dim / READBACK_VALUES_PER_THREAD,
                                  (size_t)std::max(1u, std::thread::hardware_concurrency())});
    std::vector<std::thread> threads;
    struct Join {  // also on the way out of an error
        std::vector<std::thread>& t;
        std::atomic<bool>& stop;
        ~Join() {
            stop.store(true, std::memory_order_relaxed);
            for (auto& q : t) q.join();
        }
    };
    {
        Join join{threads, stop};
        for (size_t c = 0; c < std::min(chunks, (size_t)READBACK_SLOTS); ++c) copy(c, c * chunk, cells(c));
        threads.reserve(most);
        try {
            for (size_t t = 1; t < most; ++t) threads.emplace_back(work);
        } catch (const std::system_error&) {  // as many threads as there are
        }
        for (size_t c = 0; c < chunks; ++c) {
            wait(c);
            ready.store(c + 1, std::memory_order_release);
            if (threads.empty()) {
                convert(c);
                done[c].store(true, std::memory_order_relaxed);
            }
            // the slots whose chunks are converted take the next ones
            const size_t n = c + READBACK_SLOTS;
            if (n < chunks) {
                while (!done[n - READBACK_SLOTS].load(std::memory_order_acquire)) std::this_thread::yield();
                copy(n, n * chunk, cells(n));
            }
        }
        if (!threads.empty()) work();
        for (size_t c = 0; c < chunks; ++c)
            while (!done[c].load(std::memory_order_acquire)) std::this_thread::yield();
    }
}

}  // namespace rh
