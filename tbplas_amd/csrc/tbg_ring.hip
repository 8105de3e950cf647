// Resident passes of the Chebyshev recurrence: host tables and launch.
//
// A tile pass (tbg_block.hip) keeps two vectors of a tile in LDS, which
// limits it to five terms on about 900 rows of 64 bytes, and while a tile
// computes its workgroup's compute unit reads nothing.  A resident pass
// takes the states of a run in groups of 16 bytes a row (two complex64
// states or one complex128): one workgroup owns a row block for one group,
// holds only v_{m-1} of the block and its halo rings in LDS, and v_{m-2},
// the entries of the matrix and the step output in registers (512 KB a
// compute unit against 160 KB of LDS).  A block with its rings has up to
// 4096 rows, two fit a compute unit, and a pass is half or all of a time
// step of 20 terms: nothing is read or written in between.
//
// The blocks are made here, on the host, from the caller's spatial tiles:
// tiles (or runs of a tile's rows) are merged along the matrix' own
// couplings into compact blocks sized for the LDS, then each block's rings
// are found, sorted by layout row (coalesced loads), and its tables written
// (positions in the block, 16 bits, and values).  Blocks are independent,
// so the work is spread over the host's cores.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>

#include "tbg_ring.h"

namespace tbg {

namespace {

// Up to 16 host threads for the whole of a build: started for each of its five
// phases they took 0.2 to 0.7 of the 1.8 to 3.4 ms that the tables of 8,000 to
// 33,000 rows took.  Between two phases they look for the next one for a
// while, then sleep.
class Team {
public:
    explicit Team(int want) {
        try {
            for (int t = 1; t < want; ++t) {
                threads_.emplace_back([this, t] { serve(t); });
                ++size_;
            }
        } catch (...) {   // no more threads: the ones that started do the work
        }
    }
    ~Team() {
        {
            std::lock_guard<std::mutex> g(mu_);
            stop_ = true;
            phase_.fetch_add(1, std::memory_order_release);
        }
        cv_.notify_all();
        for (auto& t : threads_) t.join();
    }
    Team(const Team&) = delete;
    Team& operator=(const Team&) = delete;

    // f(i, thread) for i < n, at least `grain` of them a thread; the first
    // exception is rethrown here.
    template <typename F>
    void run(int64_t n, int64_t grain, F&& f) {
        grain = std::max<int64_t>(grain, 1);
        const int nt = (int)std::max<int64_t>(1, std::min<int64_t>(size_, n / grain));
        const int64_t step = std::max<int64_t>(1, std::min<int64_t>(grain, n / (4 * nt) + 1));
        std::atomic<int64_t> next{0};
        std::exception_ptr err;
        std::mutex err_mu;
        const std::function<void(int)> work = [&](int th) {
            if (th >= nt) return;
            try {
                for (;;) {
                    const int64_t a = next.fetch_add(step);
                    if (a >= n) break;
                    for (int64_t i = a; i < std::min(n, a + step); ++i) f(i, th);
                }
            } catch (...) {
                std::lock_guard<std::mutex> g(err_mu);
                if (!err) err = std::current_exception();
                next.store(n);
            }
        };
        if (nt > 1) {
            {
                std::lock_guard<std::mutex> g(mu_);
                work_ = &work;
                busy_.store(size_ - 1, std::memory_order_relaxed);
                phase_.fetch_add(1, std::memory_order_release);
            }
            cv_.notify_all();
        }
        work(0);
        if (nt > 1)
            while (busy_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
        if (err) std::rethrow_exception(err);
    }

private:
    void serve(int th) {
        for (unsigned seen = 0;;) {
            for (int spin = 0; spin < 4000 && phase_.load(std::memory_order_acquire) == seen; ++spin)
                std::this_thread::yield();
            {
                std::unique_lock<std::mutex> g(mu_);
                cv_.wait(g, [&] { return phase_.load(std::memory_order_relaxed) != seen; });
                seen = phase_.load(std::memory_order_relaxed);
                if (stop_) return;
            }
            (*work_)(th);
            busy_.fetch_sub(1, std::memory_order_release);
        }
    }
    std::vector<std::thread> threads_;
    int size_ = 1;
    std::mutex mu_;
    std::condition_variable cv_;
    std::atomic<unsigned> phase_{0};
    std::atomic<int> busy_{0};
    const std::function<void(int)>* work_ = nullptr;
    bool stop_ = false;
};

constexpr int kHostThreads = 16;

struct Csr {   // the sliced-ELL matrix on the host
    std::vector<int> cols, sw;
    std::vector<int64_t> soff;
    std::vector<unsigned char> vals;
    int width(int r) const { return sw[r >> 6]; }
    int64_t elem(int r, int j) const { return soff[r >> 6] + (int64_t)j * 64 + (r & 63); }
};

// Per-thread marks over the rows (zeroed pages are only touched where used).
struct Marks {
    int *mark = nullptr, *loc = nullptr;
    int stamp = 0;
    ~Marks() {
        std::free(mark);
        std::free(loc);
    }
    void need(int64_t n) {
        if (mark) return;
        mark = (int*)std::calloc((size_t)n, sizeof(int));
        loc = (int*)std::calloc((size_t)n, sizeof(int));
        if (!mark || !loc) throw std::bad_alloc();
    }
};

// rows = owned rows + rings 1 .. depth (each sorted); ends[k]; false when
// more than cap rows.
bool grow(const Csr& A, Marks& mk, std::vector<int>& rows, int depth, int64_t cap,
          std::vector<int>& ends) {
    const int st = ++mk.stamp;
    for (size_t q = 0; q < rows.size(); ++q) {
        mk.mark[rows[q]] = st;
        mk.loc[rows[q]] = (int)q;
    }
    ends.assign(1, (int)rows.size());
    size_t from = 0;
    for (int k = 1; k <= depth; ++k) {
        const size_t to = rows.size();
        for (size_t q = from; q < to; ++q) {
            const int r = rows[q], w = A.width(r);
            for (int j = 0; j < w; ++j) {
                const int c = A.cols[A.elem(r, j)];
                if (mk.mark[c] != st) {
                    mk.mark[c] = st;
                    rows.push_back(c);
                }
            }
        }
        std::sort(rows.begin() + to, rows.end());
        for (size_t q = to; q < rows.size(); ++q) mk.loc[rows[q]] = (int)q;
        ends.push_back((int)rows.size());
        if ((int64_t)rows.size() > cap) return false;
        from = to;
    }
    return true;
}

struct Block {
    std::vector<int> rows, ends;
    std::vector<uint16_t> pos;   // of each computed row's entries, in the block
    int seg = 0, w = 0;
};

// The positions in block b (as grown, its rows marked) of the entries of the
// rows that a pass computes: those of a row of ring q lie in the rings up to
// q + 1, which the pass holds one term earlier (false: they do not).  W a row,
// or b.w columns of them for wide rows; places beyond a row's entries hold
// the row itself (with a value of zero).
bool positions(const Csr& A, const Marks& mk, Block& b, int depth, int W) {
    const int nC = b.ends[depth - 1];
    const size_t ww = W ? W : b.w;
    b.pos.resize(nC * ww);
    int ring = 0;
    for (int l = 0; l < nC; ++l) {
        while (l >= b.ends[ring]) ++ring;
        const int r = b.rows[l], w = A.width(r);
        const int end = b.ends[ring + 1];
        for (int j = 0; j < (int)ww; ++j) {
            int pos = l;
            if (j < w) {
                const int c = A.cols[A.elem(r, j)];
                pos = mk.loc[c];
                if (mk.mark[c] != mk.stamp || pos >= end) return false;
            }
            b.pos[W ? l * ww + j : (size_t)j * nC + l] = (uint16_t)pos;
        }
    }
    return true;
}

// A compact piece of a caller's tile, from which blocks are made.
struct Atom {
    std::vector<int> rows;
    int seg = 0;
};

// Rows r0 .. r1 of a tile in k x k pieces of about equal size: k runs of
// rows (strips, where the rows follow a lattice), each cut across by the
// distance from one of its ends (breadth first along the couplings).
void split_tile(const Csr& A, Marks& mk, int64_t r0, int64_t r1, int k, int seg,
                std::vector<Atom>& out) {
    for (int q = 0; q < k; ++q) {
        const int a = (int)(r0 + (r1 - r0) * q / k), b = (int)(r0 + (r1 - r0) * (q + 1) / k);
        std::vector<int> order;
        int from = a;
        for (int sweep = 0; sweep < 2; ++sweep) {   // the second from the farthest row
            const int st = ++mk.stamp;
            order.clear();
            auto visit = [&](int r) {
                mk.mark[r] = st;
                order.push_back(r);
            };
            visit(from);
            for (size_t head = 0, next = a; order.size() < (size_t)(b - a); ++head) {
                if (head == order.size()) {         // another component
                    while (mk.mark[next] == st) ++next;
                    visit((int)next);
                }
                const int r = order[head];
                for (int j = 0, w = A.width(r); j < w; ++j) {
                    const int c = A.cols[A.elem(r, j)];
                    if (c >= a && c < b && mk.mark[c] != st) visit(c);
                }
            }
            from = order.back();
        }
        for (int p = 0; p < k; ++p) {
            const size_t n = order.size();
            Atom at;
            at.seg = seg;
            at.rows.assign(order.begin() + n * p / k, order.begin() + n * (p + 1) / k);
            if (at.rows.empty()) continue;
            std::sort(at.rows.begin(), at.rows.end());
            out.push_back(std::move(at));
        }
    }
}

}  // namespace

std::shared_ptr<Ring> build_ring(tbg_handle* h, const BlockSrc& src,
                                 const std::vector<std::vector<int64_t>>& segs, int real_bytes,
                                 int V, int groups, int terms, bool real_vals) {
    const int unit_bytes = V * 2 * real_bytes;
    // (a plane is addressed with 32-bit byte offsets)
    if ((uint64_t)src.nslices * 64 * unit_bytes > kRingPlane) return nullptr;
    const int64_t n = src.nrows;
    const size_t vsz = src.vsz;
    Csr A;
    A.cols.resize((size_t)src.padded);
    A.sw.resize((size_t)src.nslices);
    A.soff.resize((size_t)src.nslices + 1);
    A.vals.resize((size_t)src.padded * vsz);
    auto down = [&](void* dst, const void* from, size_t bytes) {
        if (bytes) TBG_HIP(hipMemcpyAsync(dst, from, bytes, hipMemcpyDeviceToHost, h->stream));
    };
    down(A.cols.data(), src.cols, A.cols.size() * sizeof(int));
    down(A.vals.data(), src.vals, A.vals.size());
    down(A.sw.data(), src.sw, A.sw.size() * sizeof(int));
    down(A.soff.data(), src.soff, A.soff.size() * sizeof(int64_t));
    TBG_HIP(hipStreamSynchronize(h->stream));

    int64_t covered = 0;
    int wmax = 0;
    for (const auto& t : segs) {
        covered += t.back() - t.front();
        for (int64_t s = t.front() >> 6; s <= (t.back() - 1) >> 6; ++s)
            wmax = std::max(wmax, A.sw[s]);
    }
    if (covered < 1 || wmax < 1) return nullptr;
    const int W = wmax <= 3 ? 3 : wmax <= 4 ? 4 : 0;
    const int nr = ring_rows(real_bytes, V, real_vals, W);
    const int nro = ring_owned(real_bytes, V, real_vals, W);
    std::vector<Marks> marks(kHostThreads);
    const int64_t cores = std::max(1u, std::thread::hardware_concurrency());
    Team team((int)std::min({(int64_t)kHostThreads, cores, covered / 256 + 1}));

    // growth of a block per ring, from a few tiles: side(k) = side(0) + k c
    // with side = sqrt(rows)
    double growth = 0.0;
    {
        int cnt = 0;
        std::vector<int> rows, ends;
        marks[0].need(n);
        for (const auto& t : segs) {
            const size_t nt = t.size() - 1;
            const size_t step = std::max<size_t>(1, nt * segs.size() / 8);
            for (size_t i = nt / 2 % step; i < nt; i += step) {
                rows.clear();
                for (int64_t r = t[i]; r < t[i + 1]; ++r) rows.push_back((int)r);
                const int d = std::min(terms, 8);
                grow(A, marks[0], rows, d, n + 1, ends);
                if (ends.back() * 2 < t.back() - t.front() || cnt == 0) {
                    growth += (std::sqrt((double)ends.back()) - std::sqrt((double)ends[0])) / d;
                    ++cnt;
                }
            }
        }
        growth /= std::max(cnt, 1);
    }

    // Depth and owned rows: the least estimated cycles of a step.  A row of
    // three entries costs a compute unit about 0.9 cycles a term (LDS: its
    // entries, its own value twice); bytes pass at about 16 a cycle (of
    // tables that several groups read, two thirds come from L2); with two
    // workgroups a compute unit most of the lesser of the two hides behind
    // the other; a launch takes about 5000.  A sample too small to fill the
    // chip with full blocks gets one workgroup a compute unit, which is alone
    // there, rather than two with more halo between them, and two only where
    // one would be too large (us a step, one / two a unit: 131k rows, one
    // complex128 state 24 / 31; 65k rows 21 / 31; 32k rows, four states
    // 26 / 44; 131k rows, four complex64 states 40 / 54).  One pass a step
    // against two (ms a step): 8.4M rows, four complex64 groups 2.68 / 2.07;
    // 0.9M rows, eight complex128 groups 0.72 / 0.54; 4.2M rows, one
    // complex128 group 0.38 / 0.32; 0.5M rows, six complex64 groups (15
    // terms) 0.29 / 0.32; 0.2M rows, twelve complex128 groups 0.32 / 0.30.
    const int64_t cap = std::min<int64_t>((int64_t)nr * kRingLanes,
                                          (int64_t)h->max_lds / kRingPerCu / unit_bytes);
    const int64_t own_cap = (int64_t)nro * kRingLanes;
    const double row_cost = 0.18 * ((W ? W : wmax) + 2);
    const double fill = 0.85;   // blocks are not squares: room for their rings
    int depth = 0;
    int64_t target = 0;
    double best = 0.0;
    for (int passes = 1; passes <= 8; ++passes) {
        const int d = (terms + passes - 1) / passes;
        if (d > kRingMax || (passes > 1 && d < 3)) continue;
        const double side = std::sqrt(fill * cap) - growth * d;
        if (side < 8.0) continue;
        const double cus = (double)h->num_cus, rows = (double)covered * groups;
        const double most = std::min<double>((double)own_cap, side * side);
        // a small sample: one workgroup a compute unit, or two
        double own = std::max(64.0, rows / (0.84 * cus));
        int each = 1;
        if (own > most) {
            own = rows / (0.84 * kRingPerCu * cus);
            each = kRingPerCu;
        }
        if (own > most) {
            own = most;
            each = 0;
        }
        double comp = 0.0;
        for (int k = 0; k < d; ++k) {
            const double s = std::sqrt(own) + growth * k;
            comp += std::max(row_cost * s * s, 300.0);
        }
        const double all = std::pow(std::sqrt(own) + growth * d, 2);
        const double table = 8.0 + (W ? W : wmax) * (double)vsz;
        const double bytes = all * (4.0 + unit_bytes * (passes > 1 ? 2 : 1)) +
                             all * (groups > 1 ? table / 3.0 : table) +
                             own * unit_bytes * (passes > 1 ? 4 : 3);
        const double mem = bytes / 16.0 + 2000.0;
        const double pair = std::max(comp, mem) + 0.4 * std::min(comp, mem);
        const double cost =
            passes * (5000.0 + (each == 1   ? comp + mem
                                : each == 2 ? 2.0 * pair
                                            : rows / (0.9 * own * cus) * pair));
        if (best == 0.0 || cost < best) {
            best = cost;
            depth = d;
            target = (int64_t)own;
        }
    }
    if (depth == 0) return nullptr;

    // atoms: runs of a tile's rows no longer than a fraction of the target
    std::vector<Atom> atoms;
    {
        std::vector<std::pair<int, int64_t>> tiles;   // (segment, first row's place)
        for (size_t sg = 0; sg < segs.size(); ++sg)
            for (size_t i = 0; i + 1 < segs[sg].size(); ++i) tiles.emplace_back((int)sg, (int64_t)i);
        std::vector<std::vector<Atom>> cut(tiles.size());
        const double piece = std::max(24.0, target / 8.0);
        team.run((int64_t)tiles.size(), 16, [&](int64_t i, int th) {
            marks[th].need(n);
            const auto& t = segs[tiles[i].first];
            const int64_t a = t[tiles[i].second], b = t[tiles[i].second + 1];
            const int k = std::max(1, (int)std::lround(std::sqrt((b - a) / piece)));
            split_tile(A, marks[th], a, b, k, tiles[i].first, cut[i]);
        });
        for (auto& c : cut)
            for (auto& a : c) atoms.push_back(std::move(a));
    }
    const int na = (int)atoms.size();
    std::vector<int> atom_of((size_t)n, -1);
    team.run(na, 64, [&](int64_t i, int) {
        for (int r : atoms[i].rows) atom_of[r] = (int)i;
    });
    std::vector<std::vector<std::pair<int, int>>> nbr((size_t)na);   // (atom, couplings)
    team.run(na, 64, [&](int64_t i, int) {
        auto& v = nbr[i];
        for (int r : atoms[i].rows)
            for (int j = 0, w = A.width(r); j < w; ++j) {
                const int t = atom_of[A.cols[A.elem(r, j)]];
                if (t == (int)i || t < 0) continue;
                size_t q = 0;
                while (q < v.size() && v[q].first != t) ++q;
                if (q == v.size()) v.emplace_back(t, 0);
                ++v[q].second;
            }
    });
    // grow each block from the first free atom by the neighbour with the
    // most couplings to it (most of its own couplings first among equals)
    std::vector<std::vector<int>> groups_of;
    {
        std::vector<char> used((size_t)na, 0);
        std::vector<int> link((size_t)na, 0), cand;
        for (int i = 0; i < na; ++i) {
            if (used[i]) continue;
            std::vector<int> blk{i};
            used[i] = 1;
            int64_t rows = (int64_t)atoms[i].rows.size();
            cand.clear();
            auto join = [&](int a) {
                for (const auto& e : nbr[a]) {
                    if (used[e.first]) continue;
                    if (link[e.first] == 0) cand.push_back(e.first);
                    link[e.first] += e.second;
                }
            };
            join(i);
            for (;;) {
                int bi = -1;
                double bv = 0.0;
                for (size_t q = 0; q < cand.size(); ++q) {
                    const int c = cand[q];
                    const int64_t sz = (int64_t)atoms[c].rows.size();
                    if (used[c] || rows + sz > target) continue;
                    const double v = link[c] / std::sqrt((double)sz);
                    if (bi < 0 || v > bv * 1.02 || (v > bv * 0.98 && c < bi)) {
                        bi = c;
                        bv = v;
                    }
                }
                if (bi < 0) break;
                used[bi] = 1;
                blk.push_back(bi);
                rows += (int64_t)atoms[bi].rows.size();
                join(bi);
            }
            for (int c : cand) link[c] = 0;
            std::sort(blk.begin(), blk.end());
            groups_of.push_back(std::move(blk));
        }
    }
    // small leftovers go to their neighbours, where these have room
    {
        std::vector<int> owner((size_t)na, -1), rows_of(groups_of.size(), 0);
        for (size_t b = 0; b < groups_of.size(); ++b)
            for (int at : groups_of[b]) {
                owner[at] = (int)b;
                rows_of[b] += (int)atoms[at].rows.size();
            }
        std::vector<int> by_size(groups_of.size());
        for (size_t b = 0; b < by_size.size(); ++b) by_size[b] = (int)b;
        std::stable_sort(by_size.begin(), by_size.end(),
                         [&](int x, int y) { return rows_of[x] < rows_of[y]; });
        const int64_t most = std::min<int64_t>(own_cap, target + target / 25);
        for (int b : by_size) {
            if (rows_of[b] * 5 > target * 3) break;
            std::vector<std::pair<int, int>> moves;
            std::vector<std::pair<int, int>> added;   // (block, rows)
            for (int at : groups_of[b]) {
                int to = -1, link = 0;
                for (const auto& e : nbr[at]) {
                    const int o = owner[e.first];
                    if (o == b || atoms[e.first].seg != atoms[at].seg || e.second <= link) continue;
                    int64_t r = rows_of[o] + (int64_t)atoms[at].rows.size();
                    for (const auto& x : added)
                        if (x.first == o) r += x.second;
                    if (r > most) continue;
                    to = o;
                    link = e.second;
                }
                if (to < 0) break;
                moves.emplace_back(at, to);
                added.emplace_back(to, (int)atoms[at].rows.size());
            }
            if (moves.size() < groups_of[b].size()) continue;
            for (const auto& m : moves) {
                owner[m.first] = m.second;
                groups_of[m.second].push_back(m.first);
                rows_of[m.second] += (int)atoms[m.first].rows.size();
            }
            groups_of[b].clear();
            rows_of[b] = 0;
        }
        std::vector<std::vector<int>> kept;
        for (auto& g : groups_of)
            if (!g.empty()) {
                std::sort(g.begin(), g.end());
                kept.push_back(std::move(g));
            }
        groups_of = std::move(kept);
    }
    std::stable_sort(groups_of.begin(), groups_of.end(),
                     [&](const std::vector<int>& x, const std::vector<int>& y) {
                         return atoms[x[0]].seg < atoms[y[0]].seg;
                     });

    // rings and tables, split where a block does not fit
    const int64_t ng = (int64_t)groups_of.size();
    std::vector<std::vector<Block>> made((size_t)ng);
    std::atomic<bool> fits{true}, sound{true};
    team.run(ng, 4, [&](int64_t i, int th) {
        Marks& mk = marks[th];
        mk.need(n);
        std::vector<std::vector<int>> todo(1);
        for (int a : groups_of[i])
            todo[0].insert(todo[0].end(), atoms[a].rows.begin(), atoms[a].rows.end());
        std::sort(todo[0].begin(), todo[0].end());
        while (!todo.empty() && fits) {
            Block b;
            b.rows = todo.back();
            todo.pop_back();
            b.seg = atoms[groups_of[i][0]].seg;
            const size_t n0 = b.rows.size();
            if ((int64_t)n0 > own_cap || !grow(A, mk, b.rows, depth, cap, b.ends)) {
                if (n0 < 16) {
                    fits = false;
                    return;
                }
                b.rows.resize(n0);
                todo.emplace_back(b.rows.begin() + n0 / 2, b.rows.end());
                todo.emplace_back(b.rows.begin(), b.rows.begin() + n0 / 2);
                continue;
            }
            for (int r : b.rows) b.w = std::max(b.w, A.width(r));
            if (!positions(A, mk, b, depth, W)) {
                sound = false;
                return;
            }
            made[i].push_back(std::move(b));
        }
    });
    TBG_REQUIRE(sound, "internal: resident-pass table out of range");
    if (!fits) return nullptr;
    auto R = std::make_shared<Ring>();
    std::vector<Block*> blocks;
    for (auto& v : made)
        for (auto& b : v) blocks.push_back(&b);
    const int nb = (int)blocks.size();
    std::vector<RingMeta> meta((size_t)nb);
    std::vector<int> ends((size_t)nb * (depth + 1));
    int64_t nrow = 0, ntab = 0, nent = 0, computed = 0;
    R->seg_block.clear();
    for (int b = 0; b < nb; ++b) {
        while ((int)R->seg_block.size() <= blocks[b]->seg) R->seg_block.push_back(b);
        const Block& k = *blocks[b];
        RingMeta& m = meta[b];
        const int nC = k.ends[depth - 1];
        m.offR = nrow;
        m.offT = ntab;
        m.offE = nent;
        m.w = k.w;
        m.pad = nC;
        nrow += k.ends[depth];
        ntab += W ? nC : 0;
        nent += W ? 0 : (int64_t)nC * k.w;
        computed += nC;
        for (int q = 0; q <= depth; ++q) ends[(size_t)b * (depth + 1) + q] = k.ends[q];
        R->rows_max = std::max(R->rows_max, k.ends[depth]);
        R->owned_max = std::max(R->owned_max, k.ends[0]);
    }
    while (R->seg_block.size() < segs.size() + 1) R->seg_block.push_back(nb);
    const int shift = unit_bytes == 16 ? 4 : 3;
    TBG_REQUIRE(unit_bytes == 16 || unit_bytes == 8, "internal: unit of another size");
    // the tables one behind the other, copied at once (pages that the threads
    // touch first, no zeros before)
    struct Part {
        size_t bytes, at;
    } part[5] = {{meta.size() * sizeof(RingMeta), 0},
                 {ends.size() * sizeof(int), 0},
                 {(size_t)nrow * sizeof(int), 0},
                 {(size_t)(W ? ntab * 4 : nent) * sizeof(uint16_t), 0},
                 {(size_t)(W ? ntab * W : nent) * vsz, 0}};
    size_t total = 0;
    for (Part& p : part) {
        p.at = total;
        total += (p.bytes + 255) / 256 * 256;
    }
    const std::unique_ptr<unsigned char[]> buf(new unsigned char[total]);
    std::memcpy(buf.get() + part[0].at, meta.data(), part[0].bytes);
    std::memcpy(buf.get() + part[1].at, ends.data(), part[1].bytes);
    int* const rows = reinterpret_cast<int*>(buf.get() + part[2].at);
    unsigned char* const idx = buf.get() + part[3].at;
    unsigned char* const vals = buf.get() + part[4].at;
    team.run(nb, 4, [&](int64_t b, int) {
        const Block& k = *blocks[b];
        const RingMeta& m = meta[b];
        std::memcpy(rows + m.offR, k.rows.data(), k.rows.size() * sizeof(int));
        if (!W) std::memcpy(idx + m.offE * 2, k.pos.data(), k.pos.size() * 2);
        const int ww = W ? W : m.w;
        for (int l = 0; l < m.pad; ++l) {
            const int r = k.rows[l], w = A.width(r);
            for (int j = 0; j < ww; ++j) {
                const int64_t av = W ? (m.offT + l) * W + j : m.offE + (int64_t)j * m.pad + l;
                if (j < w) std::memcpy(vals + av * vsz, A.vals.data() + A.elem(r, j) * vsz, vsz);
                else std::memset(vals + av * vsz, 0, vsz);
            }
            if (W) {
                const uint16_t* p = k.pos.data() + (size_t)l * W;
                const uint32_t word[2] = {(uint32_t)p[0] << shift | (uint32_t)p[2] << 18,
                                          (uint32_t)p[1] << shift |
                                              (W > 3 ? (uint32_t)p[3] << 18 : 0u)};
                std::memcpy(idx + (m.offT + l) * 8, word, 8);
            }
        }
    });
    R->depth = depth;
    R->width = W;
    R->nblocks = nb;
    R->rows_lane = nr;
    R->owned_lane = nro;
    R->halo = (double)computed / (double)covered;
    R->sched[0] = 0;
    for (const Part& p : part) R->sched[0] += (int64_t)p.bytes;
    R->sched[1] = nrow;
    R->sched[2] = computed;
    R->sched[3] = covered;
    R->all.alloc(total);
    DevBuf* const to[5] = {&R->meta, &R->ends, &R->rows, &R->idx, &R->vals};
    for (int i = 0; i < 5; ++i)
        to[i]->borrow(R->all.as<unsigned char>() + part[i].at, part[i].bytes);
    TBG_HIP(hipMemcpyAsync(R->all.p, buf.get(), total, hipMemcpyHostToDevice, h->stream));
    TBG_HIP(hipStreamSynchronize(h->stream));
    return R;
}

std::string ring_key(int real_bytes, int V, int groups) {
    return std::to_string(real_bytes) + "|" + std::to_string(V) + "|" + std::to_string(groups) +
           "|";
}

std::shared_ptr<Ring> get_ring(tbg_handle* h, const tbg_ham* H, int real_bytes, int V, int groups,
                               int terms) {
    if (!h->resident || H->tiles.size() < 2) return nullptr;
    if (terms > kRingMax) terms = 20;    // a long series: any depth divides it well
    const std::string key = ring_key(real_bytes, V, groups) + std::to_string(terms);
    for (const auto& kv : H->rings)
        if (kv.first == key) return kv.second;
    BlockSrc src;
    src.cols = H->cols.as<int>();
    src.vals = H->vals.p;
    src.sw = H->slice_w.as<int>();
    src.soff = H->slice_off.as<int64_t>();
    src.nslices = H->nslices;
    src.padded = H->padded;
    src.nrows = H->n;
    src.vsz = H->vals.bytes / (size_t)std::max<int64_t>(H->padded, 1);
    std::shared_ptr<Ring> R;
    if (!with_memory([&] {
            R = build_ring(h, src, {H->tiles}, real_bytes, V, groups, terms, H->real_vals);
        }))
        return nullptr;   // (tried again by the next run)
    H->rings.emplace_back(key, R);
    if (H->rings.size() > 2) H->rings.erase(H->rings.begin());
    return R;
}

template <typename R>
void launch_ring(const RingArgs<R>& a, const Ring& r, int V, bool real_vals, hipStream_t s) {
    if (a.T < 1 || a.T > r.depth || a.depth != r.depth || r.depth > kRingMax)
        throw Error{TBG_EINVAL, "internal: more terms in a pass than the tables' rings allow"};
    if (r.rows_lane != ring_rows(sizeof(R), V, real_vals, r.width) ||
        r.owned_lane != ring_owned(sizeof(R), V, real_vals, r.width) ||
        r.rows_max > r.rows_lane * kRingLanes || r.owned_max > r.owned_lane * kRingLanes ||
        (uint64_t)a.plane * sizeof(typename CplxT<R>::T) > kRingPlane)
        throw Error{TBG_EINVAL, "internal: resident pass beyond its workgroup"};
    if ((a.q1 == nullptr) != (a.q2 == nullptr) || a.acc == nullptr || a.p1 == nullptr ||
        (!a.first && a.p0 == nullptr) || (a.q1 != nullptr && a.part != nullptr))
        throw Error{TBG_EINVAL, "internal: resident pass without its vectors"};
#define TBG_RING_RV(VV)                                                        \
    do {                                                                       \
        if (real_vals) launch_ring_rt<R, VV, true>(a, r, s);                   \
        else launch_ring_rt<R, VV, false>(a, r, s);                            \
    } while (0)
    if constexpr (sizeof(R) == 4) {
        if (V == 2) {
            TBG_RING_RV(2);
            return;
        }
    }
    if (V != 1) throw Error{TBG_EINVAL, "internal: unsupported vectors per lane"};
    TBG_RING_RV(1);
#undef TBG_RING_RV
}
template void launch_ring<float>(const RingArgs<float>&, const Ring&, int, bool, hipStream_t);
template void launch_ring<double>(const RingArgs<double>&, const Ring&, int, bool, hipStream_t);

void prepare_ring(int max_lds) {
    allow_ring_lds<float, 1, true>(max_lds);
    allow_ring_lds<float, 1, false>(max_lds);
    allow_ring_lds<float, 2, true>(max_lds);
    allow_ring_lds<float, 2, false>(max_lds);
    allow_ring_lds<double, 1, true>(max_lds);
    allow_ring_lds<double, 1, false>(max_lds);
}

}  // namespace tbg
