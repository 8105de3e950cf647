// How the DC correlations of a block of steps are divided over launches and
// waves (host arithmetic only, no HIP).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace tbg {

// A launch takes `ne` energies (the last one what is left): `tiles` tiles of
// (current, unit of VU states, 16 energies), each over `nz` splits of `split`
// rows, a wave per tile and split.  About 16 waves a compute unit over all
// tiles, and no more tiles in a launch than that, so that neither the grid
// nor the partial sums (4 KB per tile, split and state of a unit) grow with
// the number of energies.  nz is a multiple of 32: 4 waves a workgroup on 8
// XCDs.
struct DcSplit {
    int ne, tiles;
    int64_t split, nz;
};

inline DcSplit dc_split(int K, int VU, int n_en, int64_t n_pad, int num_cus) {
    DcSplit d;
    const int units = K / VU, et = (n_en + 15) / 16;
    const int most = std::max(1, 16 * num_cus / (2 * units));
    const int launches = (et + most - 1) / most;
    const int each = (et + launches - 1) / launches;   // in even shares
    d.ne = std::min(n_en, 16 * each);
    d.tiles = 2 * units * each;
    const int64_t want = std::max<int64_t>(32, (16 * (int64_t)num_cus / d.tiles + 31) / 32 * 32);
    d.split = std::max<int64_t>(64, ((n_pad + want - 1) / want + 63) / 64 * 64);
    d.nz = ((n_pad + d.split - 1) / d.split + 31) / 32 * 32;
    return d;
}

// Device bytes that a DC run allocates after it has chosen how many states it
// keeps: the quasi-eigenstates and their two currents, the phase table, the
// partial sums of their norms (`chunks` rows) and of the correlations, and
// these themselves; 64 MB for what is small.
inline size_t dc_bytes(const DcSplit& d, int K, int VU, int n_en, int64_t n_pad, int T,
                       int chunks) {
    const size_t nq = (size_t)n_en * K;
    return 16 * (size_t)n_pad * nq * 3 + 16 * (size_t)T * (n_en + 15) + 24 * (size_t)chunks * nq +
           4096 * (size_t)d.nz * d.tiles * VU + 32 * (size_t)T * nq + ((size_t)64 << 20);
}

}  // namespace tbg
