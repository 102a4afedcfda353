// readback() against a plain loop: array sizes about the chunk's multiples, one
// to more chunks than slots, and an error thrown by a copy or a wait, which must
// reach the caller.
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <vector>

#include "../rhybrid_amd/csrc/rh_readback.hpp"

template <typename Real>
static bool run(size_t nc, int dim, size_t chunk, int fail_copy, int fail_wait) {
    std::vector<Real> dev(nc * dim), ring(rh::READBACK_SLOTS * chunk * dim);
    for (size_t i = 0; i < dev.size(); ++i) dev[i] = (Real)(0.37 * (double)(i % 100003) - 11.0);
    Real* slot[rh::READBACK_SLOTS];
    for (int q = 0; q < rh::READBACK_SLOTS; ++q) slot[q] = ring.data() + q * chunk * dim;
    std::vector<double> out(nc * dim, -1e300);
    int copies = 0, waits = 0;
    bool threw = false;
    try {
        rh::readback<Real>(
            nc, dim, out.data(), slot, chunk,
            [&](size_t c, size_t first, size_t n) {
                if (copies++ == fail_copy) throw std::runtime_error("copy");
                for (int l = 0; l < dim; ++l)
                    std::memcpy(slot[c % rh::READBACK_SLOTS] + l * chunk, dev.data() + l * nc + first, n * sizeof(Real));
            },
            [&](size_t) {
                if (waits++ == fail_wait) throw std::runtime_error("wait");
            });
    } catch (const std::runtime_error&) {
        threw = true;
    }
    const int chunks = (int)((nc + chunk - 1) / chunk);
    const bool fails = (fail_copy >= 0 && fail_copy < chunks) || (fail_wait >= 0 && fail_wait < chunks);
    if (threw != fails) return false;
    if (threw) return true;
    for (size_t n = 0; n < nc; ++n)
        for (int l = 0; l < dim; ++l)
            if (out[n * dim + l] != (double)dev[l * nc + n]) return false;
    return copies == chunks && waits == chunks;
}

int main() {
    int bad = 0;
    for (int dim : {1, 3, 4})
        for (size_t nc : {size_t(1), size_t(999), size_t(1000), size_t(1001), size_t(3999), size_t(4000), size_t(4001), size_t(9500)}) {
            bad += !run<float>(nc, dim, 1000, -1, -1);
            bad += !run<double>(nc, dim, 1000, -1, -1);
            bad += !run<float>(nc, dim, nc, -1, -1);
        }
    // the sizes of production arrays
    for (size_t nc : {size_t(1) << 18, (size_t(1) << 20) + 77}) {
        bad += !run<float>(nc, 3, 87381, -1, -1);
        bad += !run<double>(nc, 1, 100000, -1, -1);
        for (int f : {0, 3, 5}) {
            bad += !run<float>(nc, 3, 87381, f, -1);
            bad += !run<float>(nc, 3, 87381, -1, f);
        }
    }
    std::printf(bad ? "%d failed\n" : "ok\n", bad);
    return bad != 0;
}
