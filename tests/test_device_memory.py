"""Device memory that a run can do with less of, on the CPU: compiled against
a stand-in for the HIP runtime whose allocations fail beyond a budget and
leave their error for the next check, as HIP does."""
import subprocess

import pytest

from tbplas_amd import build

STAND_IN = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "tbg_engine.h"

static size_t budget = 0, used = 0;
static std::map<void*, size_t> blocks;
static hipError_t last = hipSuccess;
hipError_t hipMalloc(void** p, size_t n) {
    if (used + n > budget) return last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    blocks[*p] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    used -= blocks.at(p);
    blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
namespace tbg {
void launch_fill_zero(void*, size_t, hipStream_t) { TBG_HIP(hipGetLastError()); }
}
"""

KEPT = r"""
int main(int, char** v) {
    const int free_buffers = std::atoi(v[1]), steps = std::atoi(v[2]), room = std::atoi(v[3]),
              most = std::atoi(v[4]);
    try {
        tbg_handle h;
        tbg::Engine<double> e;
        e.h = &h;
        e.vbytes = 1000;
        budget = 2000 + 1000 * (size_t)free_buffers;
        e.X.alloc(1000);
        e.Y.alloc(1000);
        e.keep_history(steps, (size_t)room * 1000, most);
        if (hipGetLastError() != hipSuccess) return 2;
        std::printf("%d %zu\n", e.hist(), used / 1000);
    } catch (const tbg::Error& e) {
        std::printf("%s\n", e.msg.c_str());
        return 1;
    }
}
"""

RING = r"""
#include <cstring>
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
int main() {
    // a closed chain of 4096 rows in tiles of 64
    const int n = 4096;
    std::vector<int> cols(n * 2), sw(n / 64, 2);
    std::vector<double> vals(n * 2, 0.5);
    std::vector<int64_t> soff;
    for (int s = 0; s <= n / 64; ++s) soff.push_back(s * 128);
    for (int r = 0; r < n; ++r) {
        cols[soff[r >> 6] + (r & 63)] = (r + 1) % n;
        cols[soff[r >> 6] + 64 + (r & 63)] = (r + n - 1) % n;
    }
    tbg_handle h;
    h.resident = 1;
    h.num_cus = 16;
    h.max_lds = 163840;
    tbg_ham H;
    H.n = n;
    H.nslices = n / 64;
    H.padded = n * 2;
    H.real_vals = true;
    H.cols.borrow(cols.data(), cols.size() * 4);
    H.vals.borrow(vals.data(), vals.size() * 8);
    H.slice_w.borrow(sw.data(), sw.size() * 4);
    H.slice_off.borrow(soff.data(), soff.size() * 8);
    for (int t = 0; t <= n; t += 64) H.tiles.push_back(t);
    size_t need = 0;
    {
        budget = 1 << 30;
        auto R = tbg::build_ring(&h, tbg::BlockSrc{cols.data(), vals.data(), sw.data(),
                                                   soff.data(), n / 64, n * 2, n, 8},
                                 {H.tiles}, 8, 1, 1, 20, true);
        if (!R || R->depth < 1) return 1;
        need = R->bytes();
    }
    if (used != 0) return 2;
    for (size_t b : {(size_t)0, need / 4, need / 2, need - 1}) {
        budget = b;
        if (tbg::get_ring(&h, &H, 8, 1, 1, 20)) return 3;
        if (used != 0 || !H.rings.empty() || hipGetLastError() != hipSuccess) return 4;
    }
    budget = need;
    return tbg::get_ring(&h, &H, 8, 1, 1, 20) && H.rings.size() == 1 ? 0 : 5;
}
"""

SCRATCH = r"""
#include "tbg_csr.h"
int main() {
    budget = 1000;
    {
        tbg::Scratch w(900);               // at once, and what is beyond it
        tbg::DevBuf a, b, c;
        w.give(a, 100);
        w.give(b, 300);
        if (used != 900 || a.owned || b.owned || (char*)b.p != (char*)a.p + 256) return 1;
        w.give(c, 90);
        if (!a.p || used != 900) return 2;
        tbg::DevBuf d;
        try {
            w.give(d, 400);
            return 3;
        } catch (const tbg::Error& e) {
            if (e.code != TBG_EOOM) return 4;
        }
    }
    if (used != 0) return 5;
    {
        tbg::Scratch w(1200);              // 700 of it are needed at a time
        tbg::DevBuf a;
        w.give(a, 200);
        for (int i = 0; i < 2; ++i) {
            tbg::DevBuf b;
            w.give(b, 500);
            if (used != 700) return 6;
        }
        if (hipGetLastError() != hipSuccess) return 7;
    }
    return used == 0 ? 0 : 8;
}
"""

SUMS = r"""
int main() {
    for (int have : {1, 2, 3, 7, 8, 15, 16, 40}) {
        tbg_handle h;
        tbg::Engine<double> e;
        e.h = &h;
        budget = 800 * (size_t)have;
        e.part.alloc(800);
        e.keep_sums();
        const int want = have >= 16 ? 16 : have >= 8 ? 8 : have >= 4 ? 4 : have >= 2 ? 2 : 1;
        if (e.part_steps != want || used != 800 * (size_t)want || e.part_stride != 100) return 1;
        if (hipGetLastError() != hipSuccess) return 2;
    }
}
"""

UNITS = r"""
int main() {
    for (size_t have = 0; have < 40; ++have)
        for (int most = 1; most <= 24; ++most) {
            budget = have * 10;
            int64_t want = most;           // by halves, rounded up
            while (want > 1 && (size_t)want > have) want = (want + 1) / 2;
            tbg::DevBuf d;
            try {
                const int64_t got = tbg::alloc_units(d, 10, most);
                if (have == 0 || got != want || d.bytes != 10 * (size_t)got || used != d.bytes)
                    return 1;
            } catch (const tbg::Error& e) {
                if (have > 0 || e.code != TBG_EOOM || used != 0) return 2;
            }
            if (hipGetLastError() != hipSuccess) return 3;
        }
}
"""


def _compile(main, d, more=()):
    src, out = d / "t.cpp", d / "t"
    src.write_text(STAND_IN + main)
    subprocess.run(["g++", "-std=c++17", "-O0", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", build.CSRC, str(src), "-o", str(out), *more],
                   check=True)
    return str(out)


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return _compile(KEPT, tmp_path_factory.mktemp("kept"))


@pytest.mark.parametrize("free,steps,room,most,kept", [
    (99, 500, 99, 16, 16), (99, 500, 99, 8, 8), (99, 500, 99, 7, 4), (99, 500, 99, 1, 1),
    (99, 500, 14, 16, 8), (99, 500, 7, 16, 8), (99, 500, 6, 16, 4), (99, 500, 0, 16, 1),
    (99, 1, 99, 16, 1), (99, 2, 99, 16, 2), (99, 8, 99, 16, 8), (99, 9, 99, 16, 16),
    # the allocations fail where the free memory promised more
    (15, 500, 99, 16, 16), (14, 500, 99, 16, 8), (6, 500, 99, 16, 4), (2, 500, 99, 16, 2),
    (1, 500, 99, 16, 2), (0, 500, 99, 16, 1)])
def test_as_many_states_as_memory_gives(exe, free, steps, room, most, kept):
    """The states a DC run keeps (Engine::keep_history): kept - 2 buffers
    beside the two of the engine, and a spare one."""
    r = subprocess.run([exe, str(free), str(steps), str(room), str(most)], capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stdout
    assert r.stdout.split() == [str(kept), str(kept + 1 if kept > 1 else 2)]


def test_no_memory_for_resident_tables(tmp_path):
    """The run takes other passes then, and the next one tries again."""
    exe = _compile(RING, tmp_path, ["-x", "c++", build.CSRC + "/tbg_ring.hip", "-lpthread",
                                    "-Wl,--unresolved-symbols=ignore-all"])
    assert subprocess.run([exe]).returncode == 0


def test_scratch_at_once_or_one_by_one(tmp_path):
    r = subprocess.run([_compile(SCRATCH, tmp_path)])
    assert r.returncode == 0


def test_sums_of_as_many_steps_as_memory_gives(tmp_path):
    r = subprocess.run([_compile(SUMS, tmp_path)])
    assert r.returncode == 0


def test_scratch_by_halves(tmp_path):
    r = subprocess.run([_compile(UNITS, tmp_path)])
    assert r.returncode == 0
