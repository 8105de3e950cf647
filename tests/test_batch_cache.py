"""Which batches' tables a handle keeps between runs, on the CPU (plain C++,
no GPU): within a bound, the least recently used gone first, and none longer
than its Hamiltonians."""
import subprocess

from tbplas_amd import build

CODE = r"""
#include <cassert>
#include "tbg_batch_cache.h"
static int live = 0;
namespace tbg { struct Ring { Ring() { ++live; } ~Ring() { --live; } }; }
using namespace tbg;
static std::shared_ptr<Ring> ring() { return std::make_shared<Ring>(); }
int main() {
    BatchCache c;
    BatchShares a, b;
    {
        BatchShares h1, h2;                 // a batch of two Hamiltonians
        auto t = c.add("1|2", ring(), 10, 100);
        h1.join(t);
        h2.join(t);
        assert(c.find("1|2") == t && t->ring() && live == 1);
        {
            BatchShares h3;                 // one in another batch too
            auto u = c.add("1|3", ring(), 10, 100);
            h1.join(u);
            h3.join(u);
            assert(live == 2);
        }
        assert(live == 1 && !c.find("1|3") && c.find("1|2") == t && c.kept.size() == 1);
    }
    assert(live == 0 && !c.find("1|2") && c.kept.empty());
    // a run that goes on holds its tables itself
    {
        auto r = ring();
        {
            BatchShares h;
            h.join(c.add("4", r, 10, 100));
        }
        assert(live == 1);
    }
    assert(live == 0);
    // within 100 bytes, the last used kept; more than that alone
    a.join(c.add("a", ring(), 40, 100));
    a.join(c.add("b", ring(), 40, 100));
    assert(c.find("a"));
    a.join(c.add("c", ring(), 40, 100));
    assert(live == 2 && c.find("a") && !c.find("b") && c.find("c"));
    b.join(c.add("d", ring(), 500, 100));
    assert(live == 1 && c.find("d") && c.kept.size() == 1);
    // tiles that do not fit are remembered, without a bound on bytes to end it
    for (int i = 0; i < 5000; ++i) b.join(c.add("n" + std::to_string(i), nullptr, 0, 100));
    assert(c.find("n4999") && !c.find("n4999")->ring() && c.kept.size() <= 1024);
    assert(b.of.size() <= 1025 && live == 0);
    // the handle closed before its Hamiltonians
    {
        BatchShares h;
        {
            BatchCache d;
            h.join(d.add("x", ring(), 1, 100));
        }
        assert(live == 1);
    }
    assert(live == 0);
}
"""


def test_kept_tables(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(CODE)
    subprocess.run(["g++", "-std=c++17", "-O0", "-UNDEBUG", "-I", build.CSRC, str(src), "-o",
                    str(exe), "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
