// strip_bands.hpp -- how many bands of rows the strip kernel cuts a mesh
// into (kernels_apply.hip).  Host arithmetic only, without HIP.
#pragma once
#include <algorithm>
#include <cstdint>

namespace sipg_internal {

// Bands per strip for nstrip strips of dimy rows on a device that holds res
// workgroups at once.  A wave costs its rows and about one more for the
// first row's latency and the band's outer rows, and the workgroups run in
// rounds of what the device holds: the fewest bands (at most one per four
// rows, and one block sum per workgroup within max_sums while there are
// several bands) that minimise rounds x (rows per wave + 1.25).
//
// Within a number of rounds more bands only shorten the waves, so one
// candidate per number of rounds decides: the fewest bands that need the
// rows per wave of as many bands as those rounds hold.  At most max_sums /
// res of them (17) and 0.1 us a call, where trying every count took 25 us on
// the 8 x 65536 mesh, on every launch: back-to-back applies at degree 1 on
// 7 x 4096 elements 6.6 -> 4.5 us, on 16 x 1024 4.4 -> 3.6.
inline int strip_bands(int64_t nstrip, int dimy, int64_t res, int64_t max_sums) {
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>((dimy + (int64_t)3) / 4, max_sums / nstrip));
    const int64_t last = (nstrip * most + res - 1) / res;
    int best = 1;
    int64_t cost = INT64_MAX;                                     // four times rounds x (rows per wave + 1.25)
    for (int64_t r = (nstrip + res - 1) / res; r <= last; ++r) {
        const int64_t held = std::min(most, r * res / nstrip);
        const int64_t rows = ((dimy + held - 1) / held + 3) / 4;  // of each wave
        const int64_t nb = (dimy + 4 * rows - 1) / (4 * rows);
        const int64_t c = (nstrip * nb + res - 1) / res * (4 * rows + 5);
        if (c < cost) {
            cost = c;
            best = (int)nb;
        }
    }
    return best;
}

}  // namespace sipg_internal
