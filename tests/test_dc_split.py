"""The division of a DC run's correlations over launches and waves, at its
edges, on the CPU (plain C++, no GPU)."""
import os
import subprocess

from tbplas_amd import build

CODE = r"""
#include <cstdio>
#include "tbg_dc_split.h"
// 0 where the division covers every energy and every row, in range
static int bad(int K, int VU, int n_en, int64_t n_pad, int cus) {
    const tbg::DcSplit d = tbg::dc_split(K, VU, n_en, n_pad, cus);
    const int units = K / VU;
    if (d.ne < 1 || d.ne > n_en || (d.ne < n_en && d.ne % 16)) return 1;
    if (d.tiles != 2 * units * ((d.ne + 15) / 16)) return 2;
    if (d.tiles > 16 * cus && d.tiles > 2 * units) return 3;
    if (d.nz < 32 || d.nz % 32 || d.split < 64 || d.split % 64) return 4;
    if (d.nz * d.split < n_pad) return 5;
    // threads of a launch, and its partial sums in a GiB or two
    if (d.nz / 4 * d.tiles * 256 >= (1ll << 31)) return 6;
    if ((double)d.nz * d.tiles * VU * 4096 > 2.5e9 && d.tiles > 2 * units) return 7;
    // one launch with about 16 waves a unit where the tiles are no more
    const int all = 2 * units * ((n_en + 15) / 16);
    if (all <= 16 * cus && (d.ne != n_en || d.tiles != all)) return 8;
    return 0;
}
int main() {
    long n = 0;
    for (int cus : {1, 3, 4, 32, 38, 64, 228, 256, 304})
        for (int K = 1; K <= 32; ++K)
            for (int VU : {1, 2}) {
                if (K % VU) continue;
                const int edge = 16 * cus / (2 * (K / VU)) * 16;   // energies of one launch
                for (int base : {1, 2, 15, 16, 17, 33, 1024, 1025, 4096, 4097, 65536, 1 << 20,
                                 edge - 16, edge - 1, edge, edge + 1, edge + 16, 2 * edge,
                                 2 * edge + 1})
                    for (int64_t n_pad : {(int64_t)64, (int64_t)128, (int64_t)2048,
                                          (int64_t)507904, (int64_t)1 << 28}) {
                        if (base < 1) continue;
                        const int r = bad(K, VU, base, n_pad, cus);
                        if (r) {
                            std::printf("%d: K %d VU %d n_en %d n_pad %lld cus %d\n", r, K, VU,
                                        base, (long long)n_pad, cus);
                            return 1;
                        }
                        ++n;
                    }
            }
    std::printf("%ld\n", n);
    // 8 complex128 states, 4097 energies, 8192 steps, 130,000 rows: the sums
    // take more than half a GiB beside the energies' vectors
    const tbg::DcSplit d = tbg::dc_split(8, 1, 4097, 130048, 256);
    std::printf("%zu %lld %d\n", tbg::dc_bytes(d, 8, 1, 4097, 130048, 8192, 508), (long long)d.nz,
                d.tiles);
}
"""


def test_every_energy_and_row_is_covered(tmp_path):
    """Many energies times states: more tiles than waves fit the chip made
    the number of splits 0, and the split a division by it."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(CODE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", build.CSRC, str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    first, second = r.stdout.splitlines()
    assert int(first) > 10000
    total, nz, tiles = (int(x) for x in second.split())
    nq = 8 * 4097
    vectors = 3 * 130048 * nq * 16
    sums = 508 * nq * 3 * 8 + nz * tiles * 256 * 16 + 8192 * 2 * nq * 16 + 8192 * 4112 * 16
    assert sums > 2 ** 29
    assert 0 <= total - vectors - sums < 2 ** 27
