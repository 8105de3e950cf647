// Resident-pass tables of batches between their runs (host code, no HIP).
#pragma once

#include <stddef.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

namespace tbg {

struct Ring;

// The tables of one batch, shared by the handle that made them and by the
// batch's Hamiltonians; a Hamiltonian may be closed from another thread.
class BatchTables {
public:
    BatchTables(std::string key, std::shared_ptr<Ring> ring, size_t bytes)
        : key(std::move(key)), bytes(bytes), ring_(std::move(ring)) {}
    const std::string key;
    const size_t bytes;
    bool gone() const {
        std::lock_guard<std::mutex> g(mu_);
        return gone_;
    }
    // (null also for tiles that do not fit)
    std::shared_ptr<Ring> ring() const {
        std::lock_guard<std::mutex> g(mu_);
        return ring_;
    }
    void give_back() {
        std::shared_ptr<Ring> last;   // (freed outside the lock)
        std::lock_guard<std::mutex> g(mu_);
        gone_ = true;
        last.swap(ring_);
    }

private:
    mutable std::mutex mu_;
    std::shared_ptr<Ring> ring_;
    bool gone_ = false;
};

typedef std::vector<std::shared_ptr<BatchTables>> BatchList;

inline void drop_gone(BatchList& v) {
    v.erase(std::remove_if(v.begin(), v.end(),
                           [](const std::shared_ptr<BatchTables>& t) { return t->gone(); }),
            v.end());
}

// A Hamiltonian's batches: their tables go with it.
struct BatchShares {
    BatchList of;
    BatchShares() = default;
    BatchShares(const BatchShares&) = delete;
    BatchShares& operator=(const BatchShares&) = delete;
    ~BatchShares() {
        for (auto& t : of) t->give_back();
    }
    void join(const std::shared_ptr<BatchTables>& t) {
        drop_gone(of);
        of.push_back(t);
    }
};

// A handle's batches.  As the tables of single Hamiltonians do, a batch's
// live as long as its Hamiltonians; but a batch is not an object that a
// program closes, so that all batches together keep at most `limit` bytes
// (the last one used may be larger): the one not used for the longest time
// goes first.
struct BatchCache {
    BatchList kept;   // the last one used is the last
    std::shared_ptr<BatchTables> find(const std::string& key) {
        drop_gone(kept);
        for (size_t i = 0; i < kept.size(); ++i)
            if (kept[i]->key == key) {
                std::rotate(kept.begin() + i, kept.begin() + i + 1, kept.end());
                return kept.back();
            }
        return nullptr;
    }
    std::shared_ptr<BatchTables> add(const std::string& key, std::shared_ptr<Ring> ring,
                                     size_t bytes, size_t limit) {
        auto t = std::make_shared<BatchTables>(key, std::move(ring), bytes);
        kept.push_back(t);
        size_t sum = 0;
        for (auto& k : kept) sum += k->bytes;
        while (kept.size() > 1 && (sum > limit || kept.size() > 1024)) {
            sum -= kept.front()->bytes;
            kept.front()->give_back();
            kept.erase(kept.begin());
        }
        return t;
    }
};

}  // namespace tbg
