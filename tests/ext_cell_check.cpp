// put_ext_cell / take_ext_cell: every extended cell and every x that a stored
// particle can have comes back bit for bit, with the cell; a removed
// particle's mark stays a mark.
#include <cstdio>
#include <cstring>
#include <limits>

#include "../rhybrid_amd/csrc/rh_geom.hpp"

template <typename Real>
static int check() {
    using L = std::numeric_limits<Real>;
    const Real xs[] = {Real(0), -Real(0), L::denorm_min(), L::min(), Real(0.25), Real(0.5), Real(1) - L::epsilon() / 2, Real(1)};
    int bad = 0;
    for (const Real x : xs)
        for (int e = 0; e < 512; ++e) {
            Real y = x;
            const uint8_t low = rh::put_ext_cell(e, y);
            const int back = rh::take_ext_cell(low, y);
            bad += back != e || std::memcmp(&x, &y, sizeof(x)) != 0;
        }
    Real gone = Real(-1);
    (void)rh::take_ext_cell((uint8_t)216, gone);
    return bad + (gone != Real(-1));
}

int main() {
    const int bad = check<float>() + check<double>();
    std::printf(bad ? "%d wrong\n" : "ok\n", bad);
    return bad != 0;
}
