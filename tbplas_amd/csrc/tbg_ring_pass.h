// The resident-pass kernel.  See tbg_ring.hip for the tables.
#pragma once

#include <algorithm>
#include <type_traits>

#include "tbg_ring.h"
#include "tbg_vec.h"

namespace tbg {

typedef __amdgpu_buffer_rsrc_t BufRsrc;
typedef unsigned buf_u2 __attribute__((ext_vector_type(2)));
typedef unsigned buf_u3 __attribute__((ext_vector_type(3)));
typedef unsigned buf_u4 __attribute__((ext_vector_type(4)));

// A buffer of `bytes` bytes at p (the same for every lane); loads beyond it
// return zeros.  Only a load's lane offset is compared with `bytes`, its
// scalar offset is not: the loads here have a scalar offset of 0, and what
// comes before a group of rows is taken off the buffer (buffer_from).
__device__ __forceinline__ BufRsrc buffer_of(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
// The part of that buffer from byte `skip` on, empty when it ends before:
// scalar arithmetic, and the lanes' offsets are the same for every group.
__device__ __forceinline__ BufRsrc buffer_from(const void* p, unsigned bytes, unsigned skip) {
    const unsigned s = skip < bytes ? skip : bytes;
    return buffer_of(static_cast<const unsigned char*>(p) + s, bytes - s);
}

// The W <= 4 entries of one row: positions in the block and values.  Rows
// are addressed as a scalar base (that of their group) plus one 32-bit
// offset a lane, so that no lane holds addresses.
template <typename R, bool RV, int W>
struct RingRow {
    static constexpr int VB = W * (int)(RV ? sizeof(R) : 2 * sizeof(R));   // value bytes
    static constexpr int NW = VB / 4 > 0 ? VB / 4 : 1;
    buf_u2 c;
    unsigned v[NW];
    // row r0 + lane of the tables of `rows` rows
    __device__ __forceinline__ void load(const void* idx_, const void* vals_, unsigned rows,
                                         unsigned r0, unsigned lane) {
        const BufRsrc idx = buffer_from(idx_, rows * 8u, r0 * 8u);
        const BufRsrc vals = buffer_from(vals_, rows * (unsigned)VB, r0 * (unsigned)VB);
        c = __builtin_amdgcn_raw_buffer_load_b64(idx, lane * 8u, 0, 0);
#pragma unroll
        for (int q = 0; q + 4 <= NW; q += 4) {
            const buf_u4 t =
                __builtin_amdgcn_raw_buffer_load_b128(vals, lane * VB + q * 4u, 0, 0);
            v[q] = t.x;
            v[q + 1] = t.y;
            v[q + 2] = t.z;
            v[q + 3] = t.w;
        }
        constexpr int q = NW / 4 * 4;
        if constexpr (NW % 4 == 3) {
            const buf_u3 t =
                __builtin_amdgcn_raw_buffer_load_b96(vals, lane * VB + q * 4u, 0, 0);
            v[q] = t.x;
            v[q + 1] = t.y;
            v[q + 2] = t.z;
        } else if constexpr (NW % 4 == 2) {
            const buf_u2 t =
                __builtin_amdgcn_raw_buffer_load_b64(vals, lane * VB + q * 4u, 0, 0);
            v[q] = t.x;
            v[q + 1] = t.y;
        }
    }
    // LDS byte offset of entry j's row (units of 2^SH bytes): entries 0 and 1
    // lie scaled in the low 18 bits of the two words, 2 and 3 unscaled in
    // the high 14
    template <int SH>
    __device__ __forceinline__ unsigned at(int j) const {
        const unsigned w = j % 2 ? c.y : c.x;
        return j < 2 ? w & 0x3ffffu : (w >> 18) << SH;
    }
    __device__ __forceinline__ HVal<R, RV> val(int j) const {
        constexpr int E = (int)(RV ? sizeof(R) : 2 * sizeof(R)) / 4;
        HVal<R, RV> h;
        __builtin_memcpy(&h, &v[j * E], E * 4);
        return h;
    }
};

// The unit of row `row` of a plane (of less than 4 GiB): a scalar base and a
// 32-bit offset a lane, so that no lane holds addresses.
template <typename R, int V>
__device__ __forceinline__ Vec<R, V> unit_at(const void* plane, int row) {
    return vld<R, V>(reinterpret_cast<const unsigned char*>(plane) +
                         (unsigned)row * (unsigned)sizeof(Vec<R, V>), 0);
}

// Stores the unit of row `row`, or nothing for row -1 (beyond the buffer).
template <typename R, int V>
__device__ __forceinline__ void unit_to(BufRsrc plane, int row, const Vec<R, V>& o) {
    const unsigned at = row < 0 ? kRingNowhere : (unsigned)row * (unsigned)sizeof(Vec<R, V>);
    R t[2 * V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        t[2 * v] = o.re[v];
        t[2 * v + 1] = o.im[v];
    }
    if constexpr (sizeof(o) == 16) {
        buf_u4 u;
        __builtin_memcpy(&u, t, 16);
        __builtin_amdgcn_raw_buffer_store_b128(u, plane, at, 0, 0);
    } else {
        buf_u2 u;
        __builtin_memcpy(&u, t, 8);
        __builtin_amdgcn_raw_buffer_store_b64(u, plane, at, 0, 0);
    }
}

// The unit at LDS byte offset o.  The dynamic LDS is all the LDS that the
// kernel has, so it starts at offset 0 and the offset is the address.
template <typename R, int V>
__device__ __forceinline__ Vec<R, V> lds_unit(unsigned o) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    Vec<R, V> x;
    static_assert(sizeof(x) == 8 || sizeof(x) == 16, "units of 8 or 16 bytes");
    R t[2 * V];
    if constexpr (sizeof(x) == 16) {
        const u4 q = *(const __attribute__((address_space(3))) u4*)o;
        __builtin_memcpy(t, &q, 16);
    } else {
        const u2 q = *(const __attribute__((address_space(3))) u2*)o;
        __builtin_memcpy(t, &q, 8);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        x.re[v] = t[2 * v];
        x.im[v] = t[2 * v + 1];
    }
    return x;
}

// One workgroup's pass over one row block for one group of V states.
//
// Where things are: v_{m-1} of the block and its rings in LDS (16 bytes a
// row, gathered by position), v_{m-2}, the matrix entries and the output of
// a lane's rows (NR rows, rows l = i NT + lane) in registers.  A term forms
// v_m over v_{m-2} in the registers, then, between two barriers, exchanges
// it with v_{m-1} in LDS.  The rows are ordered by ring, so the rows still
// needed at a term are a prefix; the term loop runs in stretches of equal
// rows per lane, each unrolled, so that all register indices are constant.
//
// What bounds it: LDS (W gathers, one read and one write of 16 bytes a row
// and term) and the vector ALU (27 instructions for two complex64 states of
// three real entries), of which the exchange's share does not overlap
// within a workgroup; two workgroups a compute unit fill each other's
// gaps.  Reading the entries from L2 at every term instead of holding them
// (which allows 5120 rows a block) took 122 against 92 ms for 256 steps of
// one complex128 state on 4.2M orbitals: its tables then miss L2 at every
// term; 16-wave workgroups, one a compute unit, 113 (both before the loads
// lost their branches, which took the 92 to 81).
template <typename R, int V, bool RV, int W, bool POLY, int NT, int NR, int NRO>
struct RingPass {
    using C = typename CplxT<R>::T;
    using VT = Vec<R, V>;
    VT prev[NR], acc[NRO];
    RingRow<R, RV, W> tab[W > 0 ? NR : 1];   // the entries of the lane's rows
    R ai[V];
    const uint16_t* idx;           // wide rows (W = 0)
    const unsigned char* vals;
    unsigned char* lds;
    int tid, wide, pad;

    __device__ __forceinline__ void gather(VT* x, const RingRow<R, RV, W>& e) const {
        constexpr int SH = V * sizeof(C) == 16 ? 4 : 3;
#pragma unroll
        for (int j = 0; j < W; ++j) x[j] = lds_unit<R, V>(e.template at<SH>(j));
    }
    // One term on the rows l < na, ceil(na / NT) = N: only the last of a
    // lane's N rows may be beyond na (what it computes there, from a row of
    // a later ring or from zeros, is never read).  Every polynomial runs as
    // v_m = i a H v_{m-1} + v_{m-2} with a power of two a (RingArgs), so one
    // fma a component rounds as the product and the sum apart would.
    template <int N>
    __device__ __forceinline__ void term(const R* cc, const R* ci, int na) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            VT s = vzero<R, V>();
            if constexpr (W > 0) {
                VT x[W > 0 ? W : 1];
                // (the offsets are taken from the words anew each term)
                asm volatile("" : "+v"(tab[i].c.x), "+v"(tab[i].c.y));
                gather(x, tab[i]);
#pragma unroll
                for (int j = 0; j < W; ++j) mac<R, V, RV>(s, tab[i].val(j), x[j]);
            } else {
                const int l = i == N - 1 ? min(i * NT + tid, na - 1) : i * NT + tid;
                s = row_sum<R, V, RV>(
                    wide, vals, [&](int j) { return (int)idx[j * pad + l]; },
                    [&](int j) { return j * pad + l; },
                    [&](int c) { return vld<R, V>(lds, (int64_t)c * V); });
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                prev[i].re[v] = fma(-ai[v], s.im[v], prev[i].re[v]);
                prev[i].im[v] = fma(ai[v], s.re[v], prev[i].im[v]);
                // formed here, not where it is stored
                asm volatile("" : "+v"(prev[i].re[v]), "+v"(prev[i].im[v]));
            }
            if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        // the output (rows beyond the owned ones are not stored): o += c v,
        // or c i v (the product with the zero part adds nothing)
#pragma unroll
        for (int i = 0; i < (N < NRO ? N : NRO); ++i) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                acc[i].re[v] = fma(cc[v], prev[i].re[v], acc[i].re[v]);
                acc[i].im[v] = fma(cc[v], prev[i].im[v], acc[i].im[v]);
                if (POLY) {
                    acc[i].re[v] = fma(-ci[v], prev[i].im[v], acc[i].re[v]);
                    acc[i].im[v] = fma(ci[v], prev[i].re[v], acc[i].im[v]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int l = i * NT + tid;
            if (i < N - 1 || l < na) {
                const VT old = vld<R, V>(lds, (int64_t)l * V);
                vst<R, V>(lds, (int64_t)l * V, prev[i]);
                prev[i] = old;
            }
            if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }
    // terms t .. while they have N rows per lane, then N - 1, ..
    template <int N>
    __device__ __forceinline__ void terms(const RingArgs<R>& a, const int* ends, const int* cl,
                                          const bool* bw, int& t, int& na) {
        while (t < a.T && na > (N - 1) * NT) {
            const int na_next = ends[t + 1 < a.T ? a.T - 2 - t : 0];
            R cc[V], ci[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const bool turn = POLY && ((a.turn >> t) & 1u) != 0;
                cc[v] = turn ? R(0) : a.c[t][cl[v]];
                ci[v] = turn ? a.c[t][cl[v]] : R(0);
            }
            term<N>(cc, ci, na);
#pragma unroll
            for (int v = 0; v < V; ++v) {
                ai[v] = a.ai[1][bw[v]];
            }
            na = na_next;
            ++t;
        }
        if constexpr (N > 1) terms<N - 1>(a, ends, cl, bw, t, na);
    }
};

template <typename R, int V, bool RV, int W, bool POLY, int NT, int NR, int NRO>
__global__ void __launch_bounds__(NT, 4)
k_ring(RingArgs<R> a, const RingMeta* __restrict__ meta_, const int* __restrict__ ends_,
       const int* __restrict__ rows_, const uint16_t* idx_, const unsigned char* vals_) {
    using C = typename CplxT<R>::T;
    using VT = Vec<R, V>;
    extern __shared__ __align__(16) unsigned char tbg_ring_smem[];
    unsigned char* lds = tbg_ring_smem;
    if (a.counter != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *a.counter += 1;
    const int wg = remap_chunk(blockIdx.x, gridDim.x);
    const int b = wg / a.groups, g = wg - b * a.groups;
    const RingMeta m = meta_[b];
    const int* ends = ends_ + (int64_t)b * (a.depth + 1);
    const int nL = ends[a.T], nC = ends[a.T - 1], n0 = ends[0];
    const int tid = threadIdx.x;
    // the layout row of row i NT + lane of the block (beyond the block: row 0)
    auto layout_row = [&](int i, unsigned lane) {
        return (int)__builtin_amdgcn_raw_buffer_load_b32(
            buffer_from(rows_ + m.offR, (unsigned)nL * 4u, i * NT * 4u), lane * 4u, 0, 0);
    };
    RingPass<R, V, RV, W, POLY, NT, NR, NRO> P;
    P.lds = lds;
    P.tid = tid;
    P.wide = m.w;
    P.pad = m.pad;
    P.idx = idx_ + (W ? m.offT * 4 : m.offE);
    P.vals = vals_ + (W ? m.offT * W : m.offE) * (RV ? sizeof(R) : sizeof(C));
    const C* p1 = reinterpret_cast<const C*>(a.p1) + g * a.plane;
    const C* p0 = reinterpret_cast<const C*>(a.p0) + g * a.plane;
    C* accp = reinterpret_cast<C*>(a.acc) + g * a.plane;
    int cl[V];
    bool bw[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        cl[v] = (int)((a.cls_mask >> (g * V + v)) & 1ull);
        bw[v] = ((a.bwd_mask >> (g * V + v)) & 1ull) != 0;
    }
    // v_{m-1} of every row to LDS, v_{m-2} and the output to registers.
    // No branches around single loads (lanes beyond the block read row 0; a
    // block of few rows skips the upper half): with one each, every load
    // waited for the one before, and this phase took 36,000 of a block's
    // 75,000 cycles (8.4M rows, four complex64 groups: 334 ms for 128 steps,
    // 265 without; 4.2M rows, one complex128 state: 96 and 81 for 256).  All
    // loads at once, the entries first, or v_{m-1} loaded straight to LDS
    // measured 0 to 8% slower; so did a workgroup that takes several groups
    // in turn and keeps the entries (they come from L2, and fewer, longer
    // workgroups balance worse).
    {
        int row[NR];
        unsigned ln = tid;   // (a copy: no offset made from it outlives the loads)
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int i = 0; i < NR; ++i) row[i] = layout_row(i, ln);
        constexpr int HB = (NR + 1) / 2;
#pragma unroll
        for (int hb = 0; hb < NR; hb += HB) {
            if (hb * NT >= nL) break;
            VT x[HB];
#pragma unroll
            for (int q = 0; q < HB && hb + q < NR; ++q) x[q] = unit_at<R, V>(p1, row[hb + q]);
#pragma unroll
            for (int q = 0; q < HB && hb + q < NR; ++q) {
                const int i = hb + q;
                vst<R, V>(lds, (int64_t)(i * NT + tid) * V, x[q]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!a.first) {
#pragma unroll
            for (int i = 0; i < NR; ++i) P.prev[i] = unit_at<R, V>(p0, row[i]);
#pragma unroll
            for (int i = 0; i < NRO; ++i) P.acc[i] = unit_at<R, V>(accp, row[i]);
        } else {
#pragma unroll
            for (int i = 0; i < NR; ++i) P.prev[i] = vzero<R, V>();
        }
    }
    if constexpr (W > 0) {
        unsigned ln = tid;
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int i = 0; i < NR; ++i)
            P.tab[i].load(P.idx, P.vals, (unsigned)P.pad, i * NT, ln);
    }
    if (a.first) {
        R c0[V];
#pragma unroll
        for (int v = 0; v < V; ++v) c0[v] = a.c0[cl[v]];
#pragma unroll
        for (int i = 0; i < NRO; ++i) {
            P.acc[i] = vzero<R, V>();
            axpy<R, V>(P.acc[i], c0, vld<R, V>(lds, (int64_t)(i * NT + tid) * V));
        }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) {
        P.ai[v] = a.ai[0][bw[v]];
    }
    int t = 0, na = nC;
    P.template terms<NR>(a, ends, cl, bw, t, na);
    // owned rows: the output, the last two terms (the last one in LDS, where
    // the same lane wrote it) and the epilogue's sums.  No branches here
    // either: the stores of lanes without a row go nowhere.
    double dre[V], dim_[V], nrm[V];
#pragma unroll
    for (int v = 0; v < V; ++v) { dre[v] = 0.0; dim_[v] = 0.0; nrm[v] = 0.0; }
    {
        int at[NRO];
#pragma unroll
        for (int i = 0; i < NRO; ++i) at[i] = layout_row(i, tid);
        const unsigned bytes = (unsigned)(a.plane * (int64_t)sizeof(C));
        const BufRsrc accb = buffer_of(accp, bytes);
#pragma unroll
        for (int i = 0; i < NRO; ++i) at[i] = i * NT + tid < n0 ? at[i] : -1;
#pragma unroll
        for (int i = 0; i < NRO; ++i) unit_to<R, V>(accb, at[i], P.acc[i]);
        if (a.q1 != nullptr) {
            const BufRsrc q1 = buffer_of(reinterpret_cast<C*>(a.q1) + g * a.plane, bytes);
            const BufRsrc q2 = buffer_of(reinterpret_cast<C*>(a.q2) + g * a.plane, bytes);
#pragma unroll
            for (int i = 0; i < NRO; ++i) {
                unit_to<R, V>(q1, at[i], P.prev[i]);
                unit_to<R, V>(q2, at[i], vld<R, V>(lds, (int64_t)(i * NT + tid) * V));
            }
        } else if (a.part != nullptr) {
            VT p[NRO];
#pragma unroll
            for (int i = 0; i < NRO; ++i) p[i] = vzero<R, V>();
            if (a.psi0 != nullptr) {
                const C* psi0 = reinterpret_cast<const C*>(a.psi0) + g * a.plane;
#pragma unroll
                for (int i = 0; i < NRO; ++i) p[i] = unit_at<R, V>(psi0, max(at[i], 0));
            }
#pragma unroll
            for (int i = 0; i < NRO; ++i) {
                if (i * NT + tid < n0) {
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const double pr = p[i].re[v], pi = p[i].im[v];
                        const double orr = P.acc[i].re[v], oi = P.acc[i].im[v];
                        dre[v] = fma(pr, orr, fma(pi, oi, dre[v]));
                        dim_[v] = fma(pr, oi, fma(-pi, orr, dim_[v]));
                        nrm[v] = fma(orr, orr, fma(oi, oi, nrm[v]));
                    }
                }
            }
        }
    }
    if (a.part != nullptr) {
        // butterfly over the wave, then the waves in order (the barrier: LDS
        // is read above)
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                dre[v] += __shfl_xor(dre[v], o);
                dim_[v] += __shfl_xor(dim_[v], o);
                nrm[v] += __shfl_xor(nrm[v], o);
            }
        }
        constexpr int NW = NT / 64;
        double* red = reinterpret_cast<double*>(lds);   // [NW][3 V]
        __syncthreads();
        if ((tid & 63) == 0) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                red[(tid >> 6) * 3 * V + v * 3 + 0] = dre[v];
                red[(tid >> 6) * 3 * V + v * 3 + 1] = dim_[v];
                red[(tid >> 6) * 3 * V + v * 3 + 2] = nrm[v];
            }
        }
        __syncthreads();
        if (tid < 3 * V) {
            double s = red[tid];
            for (int wv = 1; wv < NW; ++wv) s += red[wv * 3 * V + tid];
            a.part[(int64_t)b * a.nv + g * 3 * V + tid] = s;
        }
    }
}

template <typename R, int V, bool RV, int W, bool POLY>
static void launch_ring_w(const RingArgs<R>& a, const Ring& r, hipStream_t s) {
    // every lane has its rows' places, used or not
    constexpr size_t lds = (size_t)ring_rows(sizeof(R), V, RV, W) * kRingLanes * V *
                           sizeof(typename CplxT<R>::T);
    static_assert(lds >= (kRingLanes / 64) * 3 * V * sizeof(double), "the sums' place");
    hipLaunchKernelGGL((k_ring<R, V, RV, W, POLY, kRingLanes, ring_rows(sizeof(R), V, RV, W), ring_owned(sizeof(R), V, RV, W)>),
                       dim3(r.nblocks * a.groups), dim3(kRingLanes), lds, s, a, r.meta.as<RingMeta>(),
                       r.ends.as<int>(), r.rows.as<int>(), r.idx.as<uint16_t>(),
                       r.vals.as<unsigned char>());
    TBG_HIP(hipGetLastError());
}

template <typename R, int V, bool RV, int W>
static void launch_ring_v(const RingArgs<R>& a, const Ring& r, hipStream_t s) {
    if (a.poly) launch_ring_w<R, V, RV, W, true>(a, r, s);
    else launch_ring_w<R, V, RV, W, false>(a, r, s);
}

template <typename R, int V, bool RV>
void launch_ring_rt(const RingArgs<R>& a, const Ring& r, hipStream_t s) {
    switch (r.width) {
        case 3: launch_ring_v<R, V, RV, 3>(a, r, s); break;
        case 4: launch_ring_v<R, V, RV, 4>(a, r, s); break;
        default: launch_ring_v<R, V, RV, 0>(a, r, s); break;
    }
}

template <typename R, int V, bool RV, int W>
static void allow_ring_w(int bytes) {
    constexpr int NR = ring_rows(sizeof(R), V, RV, W), NRO = ring_owned(sizeof(R), V, RV, W);
    auto one = [&](const void* fn) {
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) !=
            hipSuccess)
            (void)hipGetLastError();
    };
    one(reinterpret_cast<const void*>(&k_ring<R, V, RV, W, false, kRingLanes, NR, NRO>));
    one(reinterpret_cast<const void*>(&k_ring<R, V, RV, W, true, kRingLanes, NR, NRO>));
}

template <typename R, int V, bool RV>
void allow_ring_lds(int bytes) {
    allow_ring_w<R, V, RV, 3>(bytes);
    allow_ring_w<R, V, RV, 4>(bytes);
    allow_ring_w<R, V, RV, 0>(bytes);
}

}  // namespace tbg
