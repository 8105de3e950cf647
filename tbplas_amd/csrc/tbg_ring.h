// Resident passes: up to a whole time step of Chebyshev terms per launch on
// row blocks that stay in LDS and registers (tables in tbg_ring.hip, kernel
// in tbg_ring_pass.h).
#pragma once

#include <memory>
#include <string>
#include <vector>

#include "tbg_block.h"
#include "tbg_prop.h"

namespace tbg {

constexpr int kRingMax = 32;      // terms of one resident pass at most
constexpr int kRingLanes = 512;   // lanes of a workgroup (two on a compute unit:
constexpr int kRingPerCu = 2;     // 128 registers a lane)
// byte offset beyond every plane, which has less than kRingPlane bytes
constexpr unsigned kRingNowhere = 0xffffff00u;
constexpr uint64_t kRingPlane = 0xfffffe00u;

// Rows per lane of a resident pass: a lane keeps v_{m-2}, the table (two
// words of positions and the values) and, of its owned rows, the output in
// about 96 of its 128 registers.
constexpr int ring_rows(int real_bytes, int V, bool real_vals, int W) {
    const int unit = V * 2 * real_bytes / 4;
    const int table = W == 0 ? 0 : 2 + W * (real_vals ? 1 : 2) * real_bytes / 4;
    const int rows = 2 * 100 / (3 * unit + 2 * table);
    const int most = unit == 4 ? 8 : 10;
    return rows > most ? most : rows;
}
constexpr int ring_owned(int real_bytes, int V, bool real_vals, int W) {
    return (ring_rows(real_bytes, V, real_vals, W) + 1) / 2;
}

// One row block: rows[offR ..] lists the owned rows, then the halo rings
// (ring k = neighbours of the rings before it, in layout order within the
// ring); ends[b * (depth + 1) + k] = rows of the block and its first k
// rings.  The tables of the rows that a pass computes (all but the last
// ring) start at row offT (packed tables) or at entry offE (wide rows).
struct RingMeta {
    int64_t offR, offT, offE;
    int w, pad;
};

// Tables of a matrix for resident passes of up to depth terms.
//   w <= 4: idx = two words per row with the positions of four entries (in
//   the low 18 bits the byte offset of entries 0 and 1, in the high 14 the
//   row of entries 2 and 3), vals = w values per row;
//   w > 4 (width 0): idx and vals column-major per block, offE + j * nC + l.
struct Ring {
    int depth = 0;
    int width = 0;           // 3, 4, or 0 for wide rows
    int nblocks = 0;
    int rows_lane = 0, owned_lane = 0;   // rows per lane it may have
    int rows_max = 0;        // widest block with all its rings
    int owned_max = 0;
    double halo = 0.0;       // rows computed per row owned, first term
    std::vector<int> seg_block;
    // what one pass of depth terms must move: table bytes, rows loaded,
    // rows computed in the first term, rows owned
    int64_t sched[4] = {0, 0, 0, 0};
    DevBuf all, meta, ends, rows, idx, vals;   // (the others are parts of all)
    size_t bytes() const { return all.bytes; }
};

// Vectors per lane (states of one workgroup) for Kp slots: 16-byte units
// where the slot count allows, so that a unit is one LDS access.
template <typename R>
inline int ring_vectors(int Kp) {
    return sizeof(R) == 4 && Kp % 2 == 0 ? 2 : 1;
}

// Tables for passes of `terms` terms (capped) over the tiles of `segs`, for
// `groups` groups of V states of real_bytes-byte reals; null where the blocks cannot
// be made (a row with too wide a halo).
std::shared_ptr<Ring> build_ring(tbg_handle* h, const BlockSrc& src,
                                 const std::vector<std::vector<int64_t>>& segs, int real_bytes,
                                 int V, int groups, int terms, bool real_vals);

// What tables are made for, as a cache key that starts with everything but
// the terms.
std::string ring_key(int real_bytes, int V, int groups);

// The tables of H for groups of V states of real_bytes-byte reals (built on
// first use, the last few kept on H), or null when the handle does not ask
// for resident passes, H has no tiles, no block fits, or there is no memory
// for the tables.
std::shared_ptr<Ring> get_ring(tbg_handle* h, const tbg_ham* H, int real_bytes, int V, int groups,
                               int terms);

template <typename R>
struct RingArgs {
    const void* p0;          // v_{m-2} (not read by a first pass)
    const void* p1;          // v_{m-1}
    void* q1;                // last two terms of the owned rows (null: the
    void* q2;                // pass ends the step)
    void* acc;               // step output
    int64_t plane;           // complex elements of one group's states
    int depth, T, groups, first;
    // v_m = i ai H v_{m-1} + v_{m-2}: of the first term and of the others,
    // forward and backward.  exp(-i H tau): ai = -1, -2.  Chebyshev
    // polynomials T_m run as u_m = (-i)^m T_m, which obey the same
    // recurrence; bit t of turn: term t enters the output as c_t i u.
    R ai[2][2];
    int poly;
    unsigned turn;
    R c0[2];                 // c_0 per coefficient class (first pass)
    R c[kRingMax][2];        // coefficients of the pass's terms per class
    uint64_t bwd_mask, cls_mask;
    int* counter;            // first pass: bumped once when non-null
    const void* psi0;        // with part: dot and norm; without psi0: norm
    double* part;            // [block][nv], nv = 3 values per slot
    int nv;
};

template <typename R>
void launch_ring(const RingArgs<R>& a, const Ring& r, int V, bool real_vals, hipStream_t s);

// instances (tbg_ring_*.hip)
template <typename R, int V, bool RV>
void launch_ring_rt(const RingArgs<R>& a, const Ring& r, hipStream_t s);
template <typename R, int V, bool RV>
void allow_ring_lds(int bytes);
void prepare_ring(int max_lds);

}  // namespace tbg
