// Two host threads reading through one ReadbackRing: each must get its own
// array.  The "device" puts a chunk into its slot when it is asked for, and a
// wait lets the other thread run before the chunk is converted, so that a ring
// used by both at once returns mixed values.
#include <chrono>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <thread>
#include <vector>

#include "../rhybrid_amd/csrc/rh_readback.hpp"

template <typename Real>
static bool reads_own(rh::ReadbackRing& ring, size_t nc, int dim, Real first) {
    std::vector<Real> dev(nc * dim);
    for (size_t i = 0; i < dev.size(); ++i) dev[i] = first + (Real)(i % 4099);
    std::vector<double> out(nc * dim, -1.0);
    ring.read<Real>(
        nc, dim, out.data(),
        [&](size_t, Real* to, size_t stride, size_t at, size_t n) {
            for (int l = 0; l < dim; ++l) std::memcpy(to + l * stride, dev.data() + l * nc + at, n * sizeof(Real));
        },
        [](size_t) { std::this_thread::sleep_for(std::chrono::milliseconds(1)); });
    for (size_t n = 0; n < nc; ++n)
        for (int l = 0; l < dim; ++l)
            if (out[n * dim + l] != (double)dev[l * nc + n]) return false;
    return true;
}

int main() {
    std::vector<char> mem(rh::READBACK_SLOTS * rh::READBACK_SLOT_BYTES);
    rh::ReadbackRing ring;
    ring.mem = mem.data();
    int bad[2] = {0, 0};
    std::thread a([&] { for (int r = 0; r < 4; ++r) bad[0] += !reads_own<float>(ring, 700001, 3, 1.0f); });
    std::thread b([&] { for (int r = 0; r < 100; ++r) bad[1] += !reads_own<double>(ring, 900, 1, 100000.0); });
    a.join();
    b.join();
    // a read that fails gives the ring back
    bool threw = false;
    try {
        double x = 0.0;
        ring.read<float>(1, 1, &x, [](size_t, float*, size_t, size_t, size_t) { throw std::runtime_error("copy"); },
                         [](size_t) {});
    } catch (const std::runtime_error&) {
        threw = true;
    }
    const bool after = reads_own<float>(ring, 1000, 3, 5.0f);
    const bool ok = !bad[0] && !bad[1] && threw && after;
    std::printf(ok ? "ok\n" : "%d and %d reads mixed\n", bad[0], bad[1]);
    return !ok;
}
