// AC and DC conductivity correlation drivers and their kernels, plus the
// block-diagonal concatenation used by batched runs.
//
// AC (tbplas/fortran/tbpm.f90:193-351): the 3K states J_x psi0, J_y psi0 and
// psi0 of K samples are propagated together as one SpMM; the Fermi and
// one-minus-Fermi polynomials run in the same launches through per-vector
// coefficient classes.  After each step one kernel forms the four current
// correlations <psi2| J_a psi1_b> with the current operators stored on the
// Hamiltonian's structure.
//
// DC (tbpm.f90:497-718): phase 1 propagates psi(+t) and psi(-t) together
// (per-vector sign of the time step) and accumulates the quasi-eigenstates in
// FP64 in the same pass as the DOS correlation; phase 2 propagates J_a psi0
// and correlates with J_a |QE_i>/|<psi0|QE_i>|, which the reference
// recomputes every step (tbpm.f90:677-697) but is time independent and is
// formed once here.
#include <cmath>

#include "tbg_cond.h"
#include "tbg_dc_split.h"

namespace tbg {

static unsigned nblk(int64_t n, int bs = 256) {
    return (unsigned)std::max<int64_t>(1, (n + bs - 1) / bs);
}

// ---------------------------------------------------------------------------
// Batch concatenation
// ---------------------------------------------------------------------------
__global__ void k_add_i64(const int64_t* src, int64_t n, int64_t add, int64_t* dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] + add;
}
__global__ void k_add_i32(const int* src, int64_t n, int add, int* dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] + add;
}

// Real values widened to complex (imaginary part 0) for a batch that mixes
// real and complex Hamiltonians.
template <typename R>
__global__ void k_real_to_cplx(const R* src, int64_t n, typename CplxT<R>::T* dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        typename CplxT<R>::T o;
        o.x = src[i];
        o.y = R(0);
        dst[i] = o;
    }
}

void concat_hams(tbg_handle* h, int n, const tbg_ham* const* hams, Concat& out) {
    int64_t ns = 0, ne = 0;
    bool all_real = true;
    for (int i = 0; i < n; ++i) {
        ns += hams[i]->nslices;
        ne += hams[i]->padded;
        all_real = all_real && hams[i]->real_vals;
    }
    TBG_REQUIRE(ns * 64 < (int64_t(1) << 31), "batch too large for 32-bit columns");
    const bool f32 = hams[0]->precision == TBG_FP32;
    const size_t cb = f32 ? sizeof(float2) : sizeof(double2);
    const size_t vb = all_real ? cb / 2 : cb;
    out.real_vals = all_real ? 1 : 0;
    out.nslices = ns;
    out.cols.alloc((size_t)std::max<int64_t>(ne, 1) * sizeof(int));
    out.vals.alloc((size_t)std::max<int64_t>(ne, 1) * vb);
    out.soff.alloc((size_t)(ns + 1) * sizeof(int64_t));
    out.sw.alloc((size_t)std::max<int64_t>(ns, 1) * sizeof(int));
    int64_t s0 = 0, e0 = 0;
    for (int i = 0; i < n; ++i) {
        const tbg_ham* H = hams[i];
        if (H->padded > 0) {
            hipLaunchKernelGGL(k_add_i32, dim3(nblk(H->padded)), dim3(256), 0, h->stream,
                               H->cols.as<int>(), H->padded, (int)(s0 * 64),
                               out.cols.as<int>() + e0);
            TBG_HIP(hipGetLastError());
            char* dst = reinterpret_cast<char*>(out.vals.p) + e0 * vb;
            if (H->real_vals && !all_real) {
                if (f32)
                    hipLaunchKernelGGL(k_real_to_cplx<float>, dim3(nblk(H->padded)), dim3(256), 0,
                                       h->stream, H->vals.as<float>(), H->padded,
                                       reinterpret_cast<float2*>(dst));
                else
                    hipLaunchKernelGGL(k_real_to_cplx<double>, dim3(nblk(H->padded)), dim3(256), 0,
                                       h->stream, H->vals.as<double>(), H->padded,
                                       reinterpret_cast<double2*>(dst));
                TBG_HIP(hipGetLastError());
            } else {
                TBG_HIP(hipMemcpyAsync(dst, H->vals.p, (size_t)H->padded * vb,
                                       hipMemcpyDeviceToDevice, h->stream));
            }
        }
        hipLaunchKernelGGL(k_add_i64, dim3(nblk(H->nslices + 1)), dim3(256), 0, h->stream,
                           H->slice_off.as<int64_t>(), H->nslices + 1, e0,
                           out.soff.as<int64_t>() + s0);
        TBG_HIP(hipGetLastError());
        TBG_HIP(hipMemcpyAsync(out.sw.as<int>() + s0, H->slice_w.p, (size_t)H->nslices * sizeof(int),
                               hipMemcpyDeviceToDevice, h->stream));
        s0 += H->nslices;
        e0 += H->padded;
    }
    TBG_HIP(hipStreamSynchronize(h->stream));
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------
// Four current correlations per sample s: slots s (psi1_x), K+s (psi1_y),
// 2K+s (psi2).  part[c][s][q][re, im], q = xx, xy, yx, yy (tbpm.f90:284-291).
template <typename R>
__global__ void __launch_bounds__(256)
k_accorr(const int* __restrict__ cols, const typename CplxT<R>::T* __restrict__ jx,
         const typename CplxT<R>::T* __restrict__ jy, const int64_t* __restrict__ soff,
         const int* __restrict__ sw, const int64_t* __restrict__ chunk,
         const typename CplxT<R>::T* __restrict__ X, Lay lay, int K, double* __restrict__ part) {
    __shared__ double sh[256 * 8];
    const int c = remap_chunk(blockIdx.x, gridDim.x);
    const int64_t r0 = chunk[c] * 64, r1 = chunk[c + 1] * 64;
    const int ng = 256 / K;
    const int s = threadIdx.x % K, grp = threadIdx.x / K;
    double d[8];
    for (int q = 0; q < 8; ++q) d[q] = 0.0;
    if (grp < ng) {
        for (int64_t r = r0 + grp; r < r1; r += ng) {
            const int64_t sl = r >> 6;
            const int lr = (int)(r & 63);
            const int64_t off = soff[sl];
            const int w = sw[sl];
            R w0r = 0, w0i = 0, w1r = 0, w1i = 0, w2r = 0, w2i = 0, w3r = 0, w3i = 0;
            for (int j = 0; j < w; ++j) {
                const int64_t e = off + (int64_t)j * 64 + lr;
                const int col = cols[e];
                const auto a = jx[e];
                const auto b = jy[e];
                const auto u = X[lay.at(col, s)];
                const auto v = X[lay.at(col, K + s)];
                w0r = fma(a.x, u.x, fma(-a.y, u.y, w0r)); w0i = fma(a.x, u.y, fma(a.y, u.x, w0i));
                w1r = fma(b.x, u.x, fma(-b.y, u.y, w1r)); w1i = fma(b.x, u.y, fma(b.y, u.x, w1i));
                w2r = fma(a.x, v.x, fma(-a.y, v.y, w2r)); w2i = fma(a.x, v.y, fma(a.y, v.x, w2i));
                w3r = fma(b.x, v.x, fma(-b.y, v.y, w3r)); w3i = fma(b.x, v.y, fma(b.y, v.x, w3i));
            }
            const auto p = X[lay.at(r, 2 * K + s)];
            const double pr = p.x, pi = p.y;
            const double wr[4] = {w0r, w1r, w2r, w3r}, wi[4] = {w0i, w1i, w2i, w3i};
            for (int q = 0; q < 4; ++q) {
                d[2 * q + 0] = fma(pr, wr[q], fma(pi, wi[q], d[2 * q + 0]));
                d[2 * q + 1] = fma(pr, wi[q], fma(-pi, wr[q], d[2 * q + 1]));
            }
        }
    }
    for (int q = 0; q < 8; ++q) sh[threadIdx.x * 8 + q] = d[q];
    __syncthreads();
    if (threadIdx.x < K * 8) {
        const int s2 = threadIdx.x / 8, q = threadIdx.x % 8;
        double acc = 0.0;
        for (int g = 0; g < ng; ++g) acc += sh[(g * K + s2) * 8 + q];
        part[(int64_t)c * 8 * K + s2 * 8 + q] = acc;
    }
}

// The DC run keeps the outputs of S (up to 16) steps and works on them at
// once: the quasi-eigenstates are read and written, and the vectors Y read,
// once per S steps instead of at every step.  With 28 energies of 8 states
// on 0.5M orbitals the quasi-eigenstates are 1.9 GB and Y 3.8 GB: a step's
// update took 786 us and its correlations 637 us, both at 5 TB/s; 16 steps
// together take 1119 and 1134 us.
constexpr int kDcSteps = 16;
struct DcStates {
    const void* p[kDcSteps];   // states after the block's steps
};

// FP64 vectors of K states for several energies: state s of row r for energy
// e at e * K * n_pad + lay.at(r, s), laid out as the first K slots of the
// run's states are (QLay::lin: those K slots are the first K * n_pad
// elements of a state buffer, slots K .. 2K the next), else row by row.
struct QLay {
    Lay lay{1};
    int64_t stride = 0;
    bool lin = false;
    __host__ __device__ __forceinline__ int64_t at(int64_t e, int64_t r, int s) const {
        return e * stride + lay.at(r, s);
    }
};

static QLay q_layout(const Lay& x, int K, int64_t n_pad) {
    QLay q;
    q.stride = K * n_pad;
    q.lin = x.sh >= 0 && K % x.unit() == 0;
    q.lay = q.lin ? Lay(K, x.sh, x.plane) : Lay(K);
    return q;
}

// QE(e, r, s) initialised to psi0 (FP64, tbpm.f90:600-603); psi0 is in the
// caller's row order, layout row r holds caller row perm[r].
__global__ void k_qe_init(const double2* __restrict__ psi0, int64_t n, int K, int64_t n_pad,
                          const int* __restrict__ perm, QLay ql, int n_en,
                          double2* __restrict__ qe) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pad * K) return;
    const int s = (int)(i / n_pad);
    const int64_t r = i - s * n_pad;
    const int64_t c = r < n ? (perm ? (int64_t)perm[r] : r) : 0;
    const double2 v = r < n ? psi0[(int64_t)s * n + c] : make_double2(0.0, 0.0);
    for (int e = blockIdx.y; e < n_en; e += gridDim.y) qe[ql.at(e, r, s)] = v;
}

// The quasi-eigenstate update (tbpm.f90:616-638) of `count` steps, the last
// of them step *counter: QE_e += W(t) (P(t, e) psi(t) + conj(P(t, e)) psi(-t))
// in the order of the steps, with pw(t, e) = W(t) P(t, e).  A thread keeps
// EC energies of one state of one row in registers over the block's steps;
// pw's rows are `pitch` (a multiple of EC) wide, zeros behind the n_en.
// Bound by HBM: QE read and written, the states once per EC energies: 16
// steps at 28 energies of 8 FP32 states, 0.5M orbitals, move 5.9 GB in 1119
// us (5.3 TB/s; 16 single steps took 12.6 ms).  EC = 16 holds 64 registers
// of sums; fewer would read the states more often.
template <typename R, bool LIN, int EC>
__global__ void __launch_bounds__(256)
k_qe(DcStates xs, int count, Lay lay, int K, int64_t n_pad, QLay ql, double2* __restrict__ qe,
     int n_en, int pitch, const double2* __restrict__ pw, const int* __restrict__ counter) {
    using C = typename CplxT<R>::T;
    const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (m >= n_pad * K) return;
    const int e0 = blockIdx.y * EC;
    const int ne = min(EC, n_en - e0);
    int64_t ip, iq, io;   // psi(t), psi(-t) and the energies' vectors
    if constexpr (LIN) {
        ip = io = m;
        iq = m + n_pad * K;
    } else {
        const int64_t r = m / K;
        const int s = (int)(m - r * K);
        ip = lay.at(r, s);
        iq = lay.at(r, K + s);
        io = ql.lay.at(r, s);
    }
    double2* out = qe + (int64_t)e0 * ql.stride + io;
    double2 v[EC];
#pragma unroll
    for (int e = 0; e < EC; ++e)
        v[e] = e < ne ? out[e * ql.stride] : make_double2(0.0, 0.0);
    const double2* w = pw + (int64_t)(*counter - count) * pitch + e0;
    for (int j = 0; j < count; ++j, w += pitch) {
        const C* X = reinterpret_cast<const C*>(xs.p[j]);
        const C p = X[ip], q = X[iq];
        const double pr = p.x, pi = p.y, qr = q.x, qi = q.y;
#pragma unroll
        for (int e = 0; e < EC; ++e) {
            // a step's share is summed before it is added: one rounding of
            // the size of QE a step
            const double2 P = w[e];
            v[e].x += fma(P.y, qi, fma(P.x, qr, fma(-P.y, pi, P.x * pr)));
            v[e].y += fma(-P.y, qr, fma(P.x, qi, fma(P.y, pr, P.x * pi)));
        }
    }
#pragma unroll
    for (int e = 0; e < EC; ++e)
        if (e < ne) out[e * ql.stride] = v[e];
}

// Per quasi-eigenstate q = e*K + s: <psi0_s|QE_q> (re, im) and |QE_q|^2.
// Grid x: chunks; part[c][q][3].
__global__ void __launch_bounds__(256)
k_qe_stats(const int64_t* __restrict__ chunk, const double2* __restrict__ qe, QLay ql, int64_t nq,
           int K, const double2* __restrict__ psi0, int64_t n, const int* __restrict__ perm,
           double* __restrict__ part) {
    __shared__ double sh[4][3];
    const int64_t r0 = chunk[blockIdx.x] * 64,
                  r1 = std::min<int64_t>(chunk[blockIdx.x + 1] * 64, n);
    for (int64_t q = blockIdx.y; q < nq; q += gridDim.y) {
    const int s = (int)(q % K);
    double d[3] = {0.0, 0.0, 0.0};
    for (int64_t r = r0 + threadIdx.x; r < r1; r += 256) {
        const double2 v = qe[ql.at(q / K, r, s)];
        const double2 z = psi0[(int64_t)s * n + (perm ? (int64_t)perm[r] : r)];
        d[0] = fma(z.x, v.x, fma(z.y, v.y, d[0]));
        d[1] = fma(z.x, v.y, fma(-z.y, v.x, d[1]));
        d[2] = fma(v.x, v.x, fma(v.y, v.y, d[2]));
    }
    for (int o = 1; o < 64; o <<= 1)
        for (int k = 0; k < 3; ++k) d[k] += __shfl_xor(d[k], o);
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; ++k) sh[threadIdx.x >> 6][k] = d[k];
    __syncthreads();
    if (threadIdx.x < 3)
        part[((int64_t)blockIdx.x * nq + q) * 3 + threadIdx.x] =
            ((sh[0][threadIdx.x] + sh[1][threadIdx.x]) + sh[2][threadIdx.x]) + sh[3][threadIdx.x];
    __syncthreads();
    }
}

// Sum partial rows part[c][nv] over all chunks -> out[nv] (one thread per
// value, by 32s: what it leaves in |<psi0|QE>| all correlations share).
__global__ void k_sum_rows(const double* __restrict__ part, int nchunks, int64_t nv,
                           double* __restrict__ out) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nv) return;
    double acc = 0.0;
    for (int c0 = 0; c0 < nchunks; c0 += 32) {
        double s = 0.0;
        for (int c = c0; c < min(c0 + 32, nchunks); ++c) s += part[(int64_t)c * nv + q];
        acc += s;
    }
    out[q] = acc;
}

// |QE(e, r, s) / div(e, s)|^2 in the caller's row order:
// out[(s * n_en + e) * n + perm[r]] (tbpm.f90:820-825, one sample per state
// s).
__global__ void k_qe_abs2(const double2* __restrict__ qe, QLay ql, int64_t n, int K, int n_en,
                          const double* __restrict__ div, const int* __restrict__ perm,
                          double* __restrict__ out) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t c = perm ? (int64_t)perm[r] : r;
    for (int64_t q = blockIdx.y; q < (int64_t)n_en * K; q += gridDim.y) {
        const int64_t e = q / K, s = q - e * K;
        const double2 v = qe[ql.at(e, r, (int)s)];
        const double x = v.x / div[q], y = v.y / div[q];
        out[(s * n_en + e) * n + c] = x * x + y * y;
    }
}

// Y_a(e, r, s) = sum_j J_a[r,j] (QE(e, col, s) / div(e, s)), a = x, y
// (tbpm.f90:680-684), both currents from one gather.
template <typename R>
__global__ void __launch_bounds__(256)
k_dc_y(const int* __restrict__ cols, const typename CplxT<R>::T* __restrict__ jx,
       const typename CplxT<R>::T* __restrict__ jy, const int64_t* __restrict__ soff,
       const int* __restrict__ sw, int64_t n_pad, const double2* __restrict__ qe, QLay ql, int K,
       int n_en, const double* __restrict__ div, double2* __restrict__ Y) {
    const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (m >= n_pad * K) return;
    const int unit = ql.lay.unit();    // consecutive threads: a row's unit, then the next row
    const int64_t g = m / (n_pad * unit), in = m - g * n_pad * unit;
    const int64_t r = in / unit;
    const int s = (int)(g * unit + (in - r * unit));
    const int64_t off = soff[r >> 6] + (r & 63);
    const int w = sw[r >> 6];
    for (int e = blockIdx.y; e < n_en; e += gridDim.y) {
    const double dv = div[(int64_t)e * K + s];
    double xr = 0.0, xi = 0.0, yr = 0.0, yi = 0.0;
    for (int j = 0; j < w; ++j) {
        const int64_t o = off + (int64_t)j * 64;
        const double2 v = qe[ql.at(e, cols[o], s)];
        const auto a = jx[o];
        const auto b = jy[o];
        const double vr = v.x / dv, vi = v.y / dv;
        const double ar = a.x, ai = a.y, br = b.x, bi = b.y;
        xr = ar * vr - ai * vi + xr;
        xi = ar * vi + ai * vr + xi;
        yr = br * vr - bi * vi + yr;
        yi = br * vi + bi * vr + yi;
    }
    Y[ql.at(e, r, s)] = make_double2(xr, xi);
    Y[ql.at((int64_t)n_en + e, r, s)] = make_double2(yr, yi);
    }
}

// The DC correlations of `count` <= 16 steps at the energies e0 .. e0 + ne of
// n_en (DcSplit): for each current a, state s: part[z][tile][v][j][e] =
// sum_{rows of split z} conj(X_j(aK + s)) Y_a(e0 + e, s), a 16 x ne product
// over the rows on the FP64 matrix cores (complex: four
// v_mfma_f64_16x16x4f64 per four rows).  A wave owns one tile (current, unit
// of VU states, 16 energies) and one split of the rows and reads both
// operands as it multiplies: lane i + 16 k holds step i and energy i of row
// k, neighbouring rows of a step or an energy are contiguous.  Bound by HBM:
// Y once per 16 steps (3.8 GB at 28 energies, 8 states, 0.5M rows: 1134 us,
// where 16 single steps on the vector ALU took 10.2 ms).
typedef double dc_d4 __attribute__((ext_vector_type(4)));
template <typename R, int VU>
__global__ void __launch_bounds__(256)
k_dcdot(DcStates xs, int count, Lay lay, int K, int64_t n_pad, const double2* __restrict__ Y,
        QLay ql, int n_en, int e0, int ne, int64_t split, double2* __restrict__ part) {
    using C = typename CplxT<R>::T;
    const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4;
    const int et = (ne + 15) / 16, units = K / VU, tiles = 2 * units * et;
    // blocks b, b + 8, ...: one XCD; the tiles of the same rows follow each
    // other there, for they read the same lines of states and of Y
    const int xcd = blockIdx.x % 8, b = blockIdx.x / 8, tile = b % tiles;
    const int64_t z = (int64_t)(b / tiles * 8 + xcd) * 4 + (threadIdx.x >> 6);
    const int a = tile / (units * et), u = tile / et % units;
    const int e = e0 + min((tile % et) * 16 + i, ne - 1);
    const int64_t r0 = z * split, r1 = min(r0 + split, n_pad);
    const C* X = reinterpret_cast<const C*>(xs.p[min(i, count - 1)]);
    const double2* Yp = Y + ((int64_t)a * n_en + e) * ql.stride;
    dc_d4 re[VU], im[VU];
#pragma unroll
    for (int v = 0; v < VU; ++v) {
        re[v] = dc_d4{0.0, 0.0, 0.0, 0.0};
        im[v] = dc_d4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll 4
    for (int64_t rb = r0; rb < r1; rb += 4) {   // (n_pad and split: multiples of 64)
        const int64_t r = rb + k;
        C x[VU];
        double2 y[VU];
        const int64_t ix = lay.at(r, a * K + u * VU), iy = ql.lay.at(r, u * VU);
        if constexpr (VU == 2 && sizeof(R) == 4) {
            const float4 t = *reinterpret_cast<const float4*>(X + ix);
            x[0] = make_float2(t.x, t.y);
            x[1] = make_float2(t.z, t.w);
        } else {
#pragma unroll
            for (int v = 0; v < VU; ++v) x[v] = X[ix + v];
        }
#pragma unroll
        for (int v = 0; v < VU; ++v) y[v] = Yp[iy + v];
#pragma unroll
        for (int v = 0; v < VU; ++v) {
            const double xr = x[v].x, xi = x[v].y;
            re[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(xr, y[v].x, re[v], 0, 0, 0);
            im[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(xr, y[v].y, im[v], 0, 0, 0);
            re[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi, y[v].y, re[v], 0, 0, 0);
            im[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(-xi, y[v].x, im[v], 0, 0, 0);
        }
    }
    // D[step][energy] sits in lane energy + 16 (step % 4), element step / 4
    double2* out = part + (z * tiles + tile) * VU * 256;
#pragma unroll
    for (int v = 0; v < VU; ++v)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            out[v * 256 + (k + 4 * q) * 16 + i] = make_double2(re[v][q], im[v][q]);
}

// The splits' sums, step j of the block to row *counter - count + 1 + j of
// out: out[row][a nq + e K + s].  Added by eights, eights of eights and so on:
// in one chain, the up to 2432 sums of a run with few tiles brought complex128
// correlations 5 to 40% further from exact ones than the single steps were.
template <int VU>
__global__ void __launch_bounds__(256)
k_dcsum(const double2* __restrict__ part, int nz, int count, int K, int n_en, int e0, int ne,
        const int* __restrict__ counter, double2* __restrict__ out) {
    const int et = (ne + 15) / 16, units = K / VU;
    const int tile = blockIdx.x, v = blockIdx.y, o = threadIdx.x, j = o >> 4;
    const int a = tile / (units * et), u = tile / et % units, el = (tile % et) * 16 + (o & 15);
    if (j >= count || el >= ne) return;
    const int e = e0 + el;
    auto add = [](double2& a, const double2& b) {
        a.x += b.x;
        a.y += b.y;
    };
    const double2 zero = make_double2(0.0, 0.0);
    double2 t = zero, s1 = zero, s2 = zero;
    const double2* q = part + ((int64_t)tile * VU + v) * 256 + o;
    const int64_t next = (int64_t)gridDim.x * VU * 256;
    for (int z = 0; z < nz; z += 8) {   // (nz: a multiple of 32)
        double2 p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = q[(z + k) * next];
#pragma unroll
        for (int w = 1; w < 8; w *= 2)
#pragma unroll
            for (int k = 0; k < 8; k += 2 * w) add(p[k], p[k + w]);
        add(s1, p[0]);
        if ((z & 56) == 56) {
            add(s2, s1);
            s1 = zero;
            if ((z & 504) == 504) {
                add(t, s2);
                s2 = zero;
            }
        }
    }
    add(s2, s1);
    add(t, s2);
    const int64_t nq = (int64_t)n_en * K;
    out[(int64_t)(*counter - count + 1 + j) * 2 * nq + a * nq + (int64_t)e * K + u * VU + v] = t;
}

// Dynamic polarisation, per sample s: slots s (psi1), K+s (psi2):
// part[c][s] = Im sum_r conj(psi2_r) rho_r psi1_r, rho_r = e^{i q.r_r}
// (inner_prod(psi2, density_q .pMul. psi1), tbpm.f90:455-478).
template <typename R>
__global__ void __launch_bounds__(256)
k_rhocorr(const int64_t* __restrict__ chunk, const typename CplxT<R>::T* __restrict__ X, Lay lay,
          int K, const double2* __restrict__ rho, double* __restrict__ part) {
    __shared__ double sh[256];
    const int c = remap_chunk(blockIdx.x, gridDim.x);
    const int64_t r0 = chunk[c] * 64, r1 = chunk[c + 1] * 64;
    const int ng = 256 / K;
    const int s = threadIdx.x % K, grp = threadIdx.x / K;
    double d = 0.0;
    if (grp < ng) {
        for (int64_t r = r0 + grp; r < r1; r += ng) {
            const auto a = X[lay.at(r, s)];
            const auto b = X[lay.at(r, K + s)];
            const double2 q = rho[r];
            const double ar = a.x, ai = a.y;
            const double wr = q.x * ar - q.y * ai, wi = q.x * ai + q.y * ar;
            d = fma((double)b.x, wi, fma(-(double)b.y, wr, d));
        }
    }
    sh[threadIdx.x] = d;
    __syncthreads();
    if (threadIdx.x < K) {
        double acc = 0.0;
        for (int g = 0; g < ng; ++g) acc += sh[g * K + threadIdx.x];
        part[(int64_t)c * K + threadIdx.x] = acc;
    }
}

// Slots [0, K) of X times conj(rho) per layout row (density(-q) .pMul. wf0).
template <typename R>
__global__ void k_rho_conj_mul(typename CplxT<R>::T* __restrict__ X, Lay lay, int K,
                               const double2* __restrict__ rho, int64_t n_pad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pad * K) return;
    const int64_t r = i / K;
    const int s = (int)(i - r * K);
    auto v = X[lay.at(r, s)];
    const double2 q = rho[r];
    const double vr = v.x, vi = v.y;
    v.x = (R)(q.x * vr + q.y * vi);
    v.y = (R)(q.x * vi - q.y * vr);
    X[lay.at(r, s)] = v;
}

// ---------------------------------------------------------------------------
// Drivers
// ---------------------------------------------------------------------------
static bool broken(double n, double ref, double thr) {
    const double d = std::fabs(n - ref);
    return std::isnan(d) || !std::isfinite(d) || d > thr;
}

static int chunks_for(tbg_handle* h, int64_t nslices) { return chunk_target(h, nslices); }

template <typename R>
void corr_ac_impl(tbg_handle* h, const tbg_ham* H, const double* bes, int nb, const double* cF,
                  int nF, const double* cO, int nO, const double* psi0, int K, int T,
                  int chk_step, double chk_thr, double* corr, int* fail_step) {
    using C = typename CplxT<R>::T;
    Engine<R> e;
    e.init(h, view_of(H), {0, H->nslices}, 3 * K, chunks_for(h, H->nslices), H, nullptr, nb - 1,
           std::max(nF, nO) - 1);
    e.keep_sums();
    const int Kp = e.Kp;
    const hipStream_t st = h->stream;
    DevBuf psi(e.vbytes);
    launch_fill_zero(psi.p, e.vbytes, st);
    launch_pack<R>(psi0, K, H->n, psi.p, e.lay, 0, H->perm_ptr(), st);
    // psi1_x = J_x psi0, psi1_y = J_y psi0, psi2 = psi0 (tbpm.f90:279-281)
    launch_spmv<R>(H, H->jx.p, psi.p, e.lay, 0, e.X.p, e.lay, 0, K, st);
    launch_spmv<R>(H, H->jy.p, psi.p, e.lay, 0, e.X.p, e.lay, K, K, st);
    launch_pack<R>(psi0, K, H->n, e.X.p, e.lay, 2 * K, H->perm_ptr(), st);
    // Fermi operators: class 0 = 1 - F on psi1, class 1 = F on psi2.
    uint64_t cls = 0;
    for (int k = 2 * K; k < 3 * K; ++k) cls |= 1ull << k;
    const StepPoly fp = cheb_poly(cO, nO, cF, nF);
    {
        TimingHold hold(h);
        e.step(fp, 0, cls, 0, nullptr, nullptr);
    }
    // norm_ref of psi2 (tbpm.f90:306) and per-step norms of every slot.
    const int nvn = 3 * Kp;
    DevBuf nbuf((size_t)T * nvn * sizeof(double));
    DevBuf abuf((size_t)T * 8 * K * sizeof(double));
    TBG_HIP(hipMemsetAsync(abuf.p, 0, (size_t)T * 8 * K * sizeof(double), st));
    DevBuf counter(sizeof(int));
    TBG_HIP(hipMemsetAsync(counter.p, 0, sizeof(int), st));
    launch_dotnorm<R>(e.plan, e.X.p, e.X.p, e.lay, Kp, e.part.template as<double>(), st);
    launch_reduce(e.part.template as<double>(), nvn, e.plan.inst_chunk_dev.template as<int>(), 1,
                  nbuf.as<double>(), 0, counter.as<int>(), 0, st);
    const StepPoly sp = time_poly(bes, nb);
    const int64_t astride = (int64_t)e.plan.nchunks * 8 * K;
    DevBuf apart;
    e.part_steps = (int)alloc_units(apart, (size_t)astride * sizeof(double), e.part_steps);
    auto reduce_corr = [&](int steps) {
        if (steps > 0)
            launch_reduce(apart.as<double>(), 8 * K, e.plan.inst_chunk_dev.template as<int>(), 1,
                          abuf.as<double>(), 0, counter.as<int>(), 0, st, steps, astride);
    };
    auto after = [&]() {
        timed_launch(h, kTimeAcCorr, [&] {
            hipLaunchKernelGGL(k_accorr<R>, dim3(e.plan.nchunks), dim3(256), 0, st,
                               H->cols.as<int>(), H->jx.as<C>(), H->jy.as<C>(),
                               H->slice_off.as<int64_t>(), H->slice_w.as<int>(),
                               e.plan.chunk.template as<int64_t>(), e.X.template as<C>(), e.lay, K,
                               apart.as<double>() + e.part_at * astride);
        });
        e.add_sums(nvn, 1, nbuf.as<double>(), 0, counter.as<int>());
        if (e.part_at == 0) reduce_corr(e.part_steps);
    };
    auto rest = [&]() {
        reduce_corr(e.part_at);
        e.add_rest(nvn, 1, nbuf.as<double>(), 0, counter.as<int>());
    };
    // t = 2..T (tbpm.f90:308-345); t = 1 is never stored.
    if (T >= 2) e.run(T - 1, sp, 0, 0, F_NORM, nullptr, counter.as<int>(), after, rest);
    std::vector<double> ha((size_t)T * 8 * K), hn((size_t)T * nvn);
    TBG_HIP(hipMemcpyAsync(ha.data(), abuf.p, ha.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    TBG_HIP(hipMemcpyAsync(hn.data(), nbuf.p, hn.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    TBG_HIP(hipStreamSynchronize(st));
    std::vector<double> out((size_t)K * 4 * T * 2);
    for (int s = 0; s < K; ++s)
        for (int q = 0; q < 4; ++q)
            for (int t = 0; t < T; ++t)
                for (int ri = 0; ri < 2; ++ri)
                    out[(((size_t)s * 4 + q) * T + t) * 2 + ri] = ha[(size_t)t * 8 * K + s * 8 + 2 * q + ri];
    TBG_HIP(hipMemcpyAsync(corr, out.data(), out.size() * sizeof(double), hipMemcpyHostToDevice, st));
    TBG_HIP(hipStreamSynchronize(st));
    // Check at loop index chk_step on psi2 after chk_step-2 steps.
    if (chk_step >= 2 && chk_step <= T) {
        for (int s = 0; s < K; ++s) {
            const int slot = 2 * K + s;
            const double ref = hn[slot * 3 + 2];
            const double nn = hn[(size_t)(chk_step - 2) * nvn + slot * 3 + 2];
            if (broken(nn, ref, chk_thr)) {
                if (fail_step) *fail_step = chk_step;
                throw Error{TBG_ENORM, "wave function norm broken at step " +
                                           std::to_string(chk_step) + " (state " +
                                           std::to_string(s) + "); check the Hermiticity of the "
                                           "Hamiltonian or increase the rescale factor"};
            }
        }
    }
}

// tbpm_dyn_pol (tbpm.f90:355-493) on caller states: per q-point, psi1 =
// (1 - F)(H) (density(-q) .pMul. psi0) and psi2 = F(H) psi0, propagated
// together; corr(s, q, t) = Im <psi2 | density(q) .pMul. psi1> at t = 1
// (before any step) .. T.  Norm check at loop index chk_step (2..T) on
// psi2 after chk_step-2 steps against its norm after the Fermi operator.
template <typename R>
void dyn_pol_impl(tbg_handle* h, const tbg_ham* H, const double* bes, int nb, const double* cF,
                  int nF, const double* cO, int nO, const double* psi0, int K, int T,
                  const double* q_points, int n_q, const double* pos, int chk_step,
                  double chk_thr, double* corr, int* fail_step) {
    using C = typename CplxT<R>::T;
    const hipStream_t st = h->stream;
    Engine<R> e;
    e.init(h, view_of(H), {0, H->nslices}, 2 * K, chunks_for(h, H->nslices), H, nullptr, nb - 1,
           std::max(nF, nO) - 1);
    const int Kp = e.Kp;
    const int64_t n = H->n, n_pad = e.n_pad;
    uint64_t cls = 0;
    for (int k = K; k < 2 * K; ++k) cls |= 1ull << k;
    const StepPoly fp = cheb_poly(cO, nO, cF, nF);
    const StepPoly sp = time_poly(bes, nb);
    const int nvn = 3 * Kp;
    DevBuf rho((size_t)n_pad * sizeof(double2)), rho_in((size_t)n * sizeof(double2));
    DevBuf nbuf((size_t)T * nvn * sizeof(double));
    DevBuf cbuf((size_t)T * K * sizeof(double));
    DevBuf counter(sizeof(int));
    std::vector<double> hr((size_t)n * 2), hc((size_t)T * K), hn((size_t)T * nvn);
    std::vector<double> out((size_t)K * n_q * T);
    auto corr_now = [&]() {
        hipLaunchKernelGGL(k_rhocorr<R>, dim3(e.plan.nchunks), dim3(256), 0, st,
                           e.plan.chunk.template as<int64_t>(), e.X.template as<C>(), e.lay, K,
                           rho.as<double2>(), e.part.template as<double>());
        launch_reduce(e.part.template as<double>(), K, e.plan.inst_chunk_dev.template as<int>(),
                      1, cbuf.as<double>(), 0, counter.as<int>(), 0, st);
    };
    auto after = [&]() {
        launch_reduce(e.part.template as<double>(), nvn, e.epi_range(), 1, nbuf.as<double>(), 0,
                      counter.as<int>(), 0, st);
        corr_now();
    };
    for (int iq = 0; iq < n_q; ++iq) {
        // density(q) = e^{i q.r} per orbital (funcs.f90:125-149), caller order
        const double* q = q_points + (size_t)iq * 3;
        for (int64_t j = 0; j < n; ++j) {
            const double pw = q[0] * pos[j * 3 + 0] + q[1] * pos[j * 3 + 1] + q[2] * pos[j * 3 + 2];
            hr[j * 2 + 0] = std::cos(pw);
            hr[j * 2 + 1] = std::sin(pw);
        }
        TBG_HIP(hipMemcpyAsync(rho_in.p, hr.data(), hr.size() * sizeof(double),
                               hipMemcpyHostToDevice, st));
        launch_fill_zero(rho.p, rho.bytes, st);
        launch_pack<double>(rho_in.as<double>(), 1, n, rho.p, 1, 0, H->perm_ptr(), st);
        // psi1 = (1 - F) density(-q) psi0 in slots [0, K), psi2 = F psi0 in [K, 2K)
        launch_fill_zero(e.X.p, e.vbytes, st);
        launch_pack<R>(psi0, K, n, e.X.p, e.lay, 0, H->perm_ptr(), st);
        launch_pack<R>(psi0, K, n, e.X.p, e.lay, K, H->perm_ptr(), st);
        hipLaunchKernelGGL(k_rho_conj_mul<R>, dim3(nblk(n_pad * K)), dim3(256), 0, st,
                           e.X.template as<C>(), e.lay, K, rho.as<double2>(), n_pad);
        TBG_HIP(hipGetLastError());
        {
            TimingHold hold(h);
            e.step(fp, 0, cls, 0, nullptr, nullptr);
        }
        TBG_HIP(hipMemsetAsync(counter.p, 0, sizeof(int), st));
        launch_dotnorm<R>(e.plan, e.X.p, e.X.p, e.lay, Kp, e.part.template as<double>(), st);
        launch_reduce(e.part.template as<double>(), nvn, e.plan.inst_chunk_dev.template as<int>(),
                      1, nbuf.as<double>(), 0, counter.as<int>(), 0, st);
        corr_now();   // t = 1 (tbpm.f90:459-466)
        if (T >= 2) e.run(T - 1, sp, 0, 0, F_NORM, nullptr, counter.as<int>(), after);
        TBG_HIP(hipMemcpyAsync(hc.data(), cbuf.p, hc.size() * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        TBG_HIP(hipMemcpyAsync(hn.data(), nbuf.p, hn.size() * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        TBG_HIP(hipStreamSynchronize(st));
        for (int s = 0; s < K; ++s)
            for (int t = 0; t < T; ++t) out[((size_t)s * n_q + iq) * T + t] = hc[(size_t)t * K + s];
        if (chk_step >= 2 && chk_step <= T) {
            for (int s = 0; s < K; ++s) {
                const int slot = K + s;
                const double ref = hn[slot * 3 + 2];
                const double nn = hn[(size_t)(chk_step - 2) * nvn + slot * 3 + 2];
                if (broken(nn, ref, chk_thr)) {
                    if (fail_step) *fail_step = chk_step;
                    throw Error{TBG_ENORM, "wave function norm broken at step " +
                                               std::to_string(chk_step) + " (state " +
                                               std::to_string(s) + ", q-point " +
                                               std::to_string(iq) + "); check the Hermiticity "
                                               "of the Hamiltonian or increase the rescale factor"};
                }
            }
        }
    }
    TBG_HIP(hipMemcpyAsync(corr, out.data(), out.size() * sizeof(double), hipMemcpyHostToDevice,
                           st));
    TBG_HIP(hipStreamSynchronize(st));
}

template <typename R>
void corr_dc_impl(tbg_handle* h, const tbg_ham* H, const double* bes, int nb, const double* psi0,
                  int K, int T, double t_step, const double* energies, const int64_t* en_inds,
                  int n_en, int chk_step, double chk_thr, double* dos_corr, double* dc_corr,
                  int* fail_step, double* qe_abs2) {
    using C = typename CplxT<R>::T;
    const hipStream_t st = h->stream;
    Engine<R> e;
    e.init(h, view_of(H), {0, H->nslices}, 2 * K, chunks_for(h, H->nslices), H, nullptr, nb - 1);
    e.keep_sums();
    const int Kp = e.Kp;
    const int64_t n = H->n, n_pad = e.n_pad;
    const int64_t nq = (int64_t)n_en * K;
    DevBuf psi(e.vbytes);
    launch_fill_zero(psi.p, e.vbytes, st);
    launch_pack<R>(psi0, K, n, psi.p, e.lay, 0, H->perm_ptr(), st);
    launch_pack<R>(psi0, K, n, e.X.p, e.lay, 0, H->perm_ptr(), st);
    launch_pack<R>(psi0, K, n, e.X.p, e.lay, K, H->perm_ptr(), st);
    const QLay ql = q_layout(e.lay, K, n_pad);
    const bool pairs = sizeof(R) == 4 && ql.lin && ql.lay.sh == 1;
    const int VU = pairs ? 2 : 1;
    DcSplit ds{};
    // the kept states leave room for all that follows
    if (nq > 0) {
        ds = dc_split(K, VU, n_en, n_pad, h->num_cus);
        const size_t rest = dc_bytes(ds, K, VU, n_en, n_pad, T, e.plan.nchunks);
        size_t room = 0, total = 0;
        TBG_HIP(hipMemGetInfo(&room, &total));
        e.keep_history(T, room > rest ? (room - rest) / 2 : 0, h->kept_steps);
    }
    uint64_t bwd = 0;
    for (int k = K; k < 2 * K; ++k) bwd |= 1ull << k;
    const unsigned nbm = nblk(n_pad * K), ny = (unsigned)std::min(n_en, 32768),
                   nyq = (unsigned)std::min<int64_t>(nq, 32768);
    // energies a thread of k_qe keeps, in even chunks
    const int chunks = std::max((n_en + 15) / 16, 1), even = (n_en + chunks - 1) / chunks;
    const int ec = even <= 2 ? 2 : even <= 8 ? 8 : 16;
    const int nec = (n_en + ec - 1) / ec, pitch = nec * ec;
    DevBuf qe((size_t)std::max<int64_t>(n_pad * nq, 1) * sizeof(double2));
    if (nq > 0)
        hipLaunchKernelGGL(k_qe_init, dim3(nbm, ny), dim3(256), 0, st,
                           reinterpret_cast<const double2*>(psi0), n, K, n_pad, H->perm_ptr(), ql,
                           n_en, qe.as<double2>());
    // W(t) P(t, e): phases exp(i E t dt) and the Hanning window
    // (tbpm.f90:625-629).
    std::vector<double> ptab((size_t)T * std::max(pitch, 1) * 2, 0.0);
    const double pi = 3.14159265358979323846;
    for (int t = 1; t <= T; ++t) {
        const double W = 0.5 * (1 + std::cos(pi * t / T));
        for (int i = 0; i < n_en; ++i) {
            const double th = energies[en_inds[i]] * t * t_step;
            ptab[((size_t)(t - 1) * pitch + i) * 2 + 0] = W * std::cos(th);
            ptab[((size_t)(t - 1) * pitch + i) * 2 + 1] = W * std::sin(th);
        }
    }
    DevBuf dptab(ptab.size() * sizeof(double));
    TBG_HIP(hipMemcpyAsync(dptab.p, ptab.data(), ptab.size() * sizeof(double), hipMemcpyHostToDevice, st));
    const int nvn = 3 * Kp;
    DevBuf nbuf((size_t)(T + 1) * nvn * sizeof(double));
    DevBuf counter(sizeof(int));
    TBG_HIP(hipMemsetAsync(counter.p, 0, sizeof(int), st));
    launch_dotnorm<R>(e.plan, e.X.p, e.X.p, e.lay, Kp, e.part.template as<double>(), st);
    launch_reduce(e.part.template as<double>(), nvn, e.plan.inst_chunk_dev.template as<int>(), 1,
                  nbuf.as<double>(), 0, counter.as<int>(), 0, st);
    const StepPoly sp = time_poly(bes, nb);
    std::vector<double> hn((size_t)(T + 1) * nvn);   // <psi0|psi(t)> and |psi(t)|^2 per slot
    // Check at t == chk_step on psi(+-) after chk_step-1 steps vs <psi0|psi0>
    // (tbpm.f90:608-611, 772-775).
    auto check_norms = [&]() {
        if (chk_step < 1 || chk_step > T) return;
        for (int k = 0; k < 2 * K; ++k) {
            const double ref = hn[k * 3 + 2];
            const double nn = hn[(size_t)(chk_step - 1) * nvn + k * 3 + 2];
            if (broken(nn, ref, chk_thr)) {
                if (fail_step) *fail_step = chk_step;
                throw Error{TBG_ENORM, "wave function norm broken at step " +
                                           std::to_string(chk_step) +
                                           "; check the Hermiticity of the Hamiltonian or "
                                           "increase the rescale factor"};
            }
        }
    };
    // the states of the last `count` of the `done` steps enqueued or captured
    // (whole rounds of the buffers), the run's input being state `base`
    int done = 0, base = 0;
    auto kept = [&](int count) {
        DcStates xs;
        for (int j = 0; j < kDcSteps; ++j)
            xs.p[j] = e.history(base + done - count + 1 + std::min(j, count - 1));
        return xs;
    };
    auto qe_update = [&](int count) {
        const DcStates xs = kept(count);
        // (y: the energies of a launch whose grid stays within 65535)
        for (int y = 0; y < nec; y += 32768) {
            const dim3 grid(nbm, (unsigned)std::min(nec - y, 32768));
            const int e0 = y * ec;
#define TBG_QE(LIN, EC)                                                                     \
    hipLaunchKernelGGL((k_qe<R, LIN, EC>), grid, dim3(256), 0, st, xs, count, e.lay, K, n_pad, \
                       ql, qe.as<double2>() + e0 * ql.stride, n_en - e0, pitch,              \
                       dptab.as<double2>() + e0, counter.as<int>())
            timed_launch(h, kTimeQe, [&] {
                if (ql.lin) {
                    if (ec == 2) TBG_QE(true, 2);
                    else if (ec == 8) TBG_QE(true, 8);
                    else TBG_QE(true, 16);
                } else {
                    if (ec == 2) TBG_QE(false, 2);
                    else if (ec == 8) TBG_QE(false, 8);
                    else TBG_QE(false, 16);
                }
                TBG_HIP(hipGetLastError());
            });
        }
#undef TBG_QE
    };
    auto after1 = [&]() {
        e.add_sums(nvn, 1, nbuf.as<double>(), 0, counter.as<int>());
        ++done;
        if (nq > 0 && done % e.hist() == 0) qe_update(e.hist());
    };
    e.run(T, sp, bwd, 0, F_DOT | F_NORM, psi.p, counter.as<int>(), after1,
          [&]() { e.add_rest(nvn, 1, nbuf.as<double>(), 0, counter.as<int>()); });
    if (nq > 0 && done % e.hist() != 0) qe_update(done % e.hist());
    TBG_HIP(hipMemcpyAsync(hn.data(), nbuf.p, hn.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    // |QE| and a = |<psi0|QE>| (tbpm.f90:642-647, 667): the currents act on
    // QE / |QE| / (a / |QE|) = QE / a.
    std::vector<double> div(std::max<int64_t>(nq, 1));
    DevBuf ddiv(div.size() * sizeof(double));
    if (nq > 0) {
        DevBuf qpart((size_t)e.plan.nchunks * nq * 3 * sizeof(double));
        DevBuf qsum((size_t)nq * 3 * sizeof(double));
        std::vector<double> hs((size_t)nq * 3);
        hipLaunchKernelGGL(k_qe_stats, dim3(e.plan.nchunks, nyq), dim3(256), 0, st,
                           e.plan.chunk.template as<int64_t>(), qe.as<double2>(), ql, nq, K,
                           reinterpret_cast<const double2*>(psi0), n, H->perm_ptr(),
                           qpart.as<double>());
        TBG_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_sum_rows, dim3(nblk(nq * 3)), dim3(256), 0, st, qpart.as<double>(),
                           e.plan.nchunks, nq * 3, qsum.as<double>());
        TBG_HIP(hipGetLastError());
        TBG_HIP(hipMemcpyAsync(hs.data(), qsum.p, hs.size() * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        TBG_HIP(hipStreamSynchronize(st));
        for (int64_t q = 0; q < nq; ++q)
            div[q] = qe_abs2 != nullptr ? std::sqrt(hs[q * 3 + 2])
                                        : std::hypot(hs[q * 3 + 0], hs[q * 3 + 1]);
        TBG_HIP(hipMemcpyAsync(ddiv.p, div.data(), nq * sizeof(double), hipMemcpyHostToDevice, st));
        if (qe_abs2 != nullptr) {   // quasi-eigenstates: done after normalising
            hipLaunchKernelGGL(k_qe_abs2, dim3(nblk(n), nyq), dim3(256), 0, st,
                               qe.as<double2>(), ql, n, K, n_en, ddiv.as<double>(),
                               H->perm_ptr(), qe_abs2);
            TBG_HIP(hipGetLastError());
            TBG_HIP(hipStreamSynchronize(st));
            check_norms();
            return;
        }
    }
    // Y_a = J_a (QE / a), time independent.
    DevBuf Y((size_t)std::max<int64_t>(n_pad * 2 * nq, 1) * sizeof(double2));
    if (nq > 0) {
        hipLaunchKernelGGL(k_dc_y<R>, dim3(nbm, ny), dim3(256), 0, st, H->cols.as<int>(),
                           H->jx.as<C>(), H->jy.as<C>(), H->slice_off.as<int64_t>(),
                           H->slice_w.as<int>(), n_pad, qe.as<double2>(), ql, K, n_en,
                           ddiv.as<double>(), Y.as<double2>());
        TBG_HIP(hipGetLastError());
    }
    qe.release();
    // Phase 2: J_x psi0, J_y psi0 propagated forward (tbpm.f90:655-697).
    e.drop_graph();
    launch_fill_zero(e.X.p, e.vbytes, st);
    launch_spmv<R>(H, H->jx.p, psi.p, e.lay, 0, e.X.p, e.lay, 0, K, st);
    launch_spmv<R>(H, H->jy.p, psi.p, e.lay, 0, e.X.p, e.lay, K, K, st);
    const int64_t nq2 = 2 * nq;
    DevBuf cbuf((size_t)std::max<int64_t>(T * nq2 * 2, 1) * sizeof(double));
    TBG_HIP(hipMemsetAsync(counter.p, 0, sizeof(int), st));
    DevBuf dpart;
    if (nq2 > 0) dpart.alloc((size_t)ds.nz * ds.tiles * VU * 256 * sizeof(double2));
    auto correlate = [&](int count) {
        const DcStates xs = kept(count);
        for (int e0 = 0; e0 < n_en; e0 += ds.ne) {
            const int ne = std::min(ds.ne, n_en - e0);
            const int tiles = 2 * (K / VU) * ((ne + 15) / 16);
            timed_launch(h, kTimeDcDot, [&] {
                const dim3 grid((unsigned)(ds.nz / 4 * tiles));
                if (pairs) {
                    if constexpr (sizeof(R) == 4)
                        hipLaunchKernelGGL((k_dcdot<R, 2>), grid, dim3(256), 0, st, xs, count,
                                           e.lay, K, n_pad, Y.as<double2>(), ql, n_en, e0, ne,
                                           ds.split, dpart.as<double2>());
                } else {
                    hipLaunchKernelGGL((k_dcdot<R, 1>), grid, dim3(256), 0, st, xs, count, e.lay,
                                       K, n_pad, Y.as<double2>(), ql, n_en, e0, ne, ds.split,
                                       dpart.as<double2>());
                }
                TBG_HIP(hipGetLastError());
            });
            const dim3 grid((unsigned)tiles, VU);
            if (pairs)
                hipLaunchKernelGGL(k_dcsum<2>, grid, dim3(256), 0, st, dpart.as<double2>(),
                                   (int)ds.nz, count, K, n_en, e0, ne, counter.as<int>(),
                                   cbuf.as<double2>());
            else
                hipLaunchKernelGGL(k_dcsum<1>, grid, dim3(256), 0, st, dpart.as<double2>(),
                                   (int)ds.nz, count, K, n_en, e0, ne, counter.as<int>(),
                                   cbuf.as<double2>());
            TBG_HIP(hipGetLastError());
        }
    };
    base = e.cur;
    done = 0;
    if (nq2 > 0) correlate(1);   // t = 1, unpropagated
    auto after2 = [&]() {
        ++done;
        if (nq2 > 0 && done % e.hist() == 0) correlate(e.hist());
    };
    if (T >= 2) e.run(T - 1, sp, 0, 0, 0, nullptr, counter.as<int>(), after2);
    if (nq2 > 0 && done % e.hist() != 0) correlate(done % e.hist());
    std::vector<double> hc((size_t)T * nq2 * 2);
    if (nq2 > 0)
        TBG_HIP(hipMemcpyAsync(hc.data(), cbuf.p, hc.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    TBG_HIP(hipStreamSynchronize(st));
    std::vector<double> od((size_t)K * T * 2), oc((size_t)K * 2 * std::max(n_en, 0) * T * 2);
    for (int s = 0; s < K; ++s)
        for (int t = 0; t < T; ++t)
            for (int ri = 0; ri < 2; ++ri)
                od[((size_t)s * T + t) * 2 + ri] = hn[(size_t)(t + 1) * nvn + s * 3 + ri];
    for (int s = 0; s < K; ++s)
        for (int a = 0; a < 2; ++a)
            for (int i = 0; i < n_en; ++i)
                for (int t = 0; t < T; ++t)
                    for (int ri = 0; ri < 2; ++ri)
                        oc[((((size_t)s * 2 + a) * n_en + i) * T + t) * 2 + ri] =
                            hc[(size_t)t * nq2 * 2 + (a * nq + (int64_t)i * K + s) * 2 + ri];
    TBG_HIP(hipMemcpyAsync(dos_corr, od.data(), od.size() * sizeof(double), hipMemcpyHostToDevice, st));
    if (!oc.empty())
        TBG_HIP(hipMemcpyAsync(dc_corr, oc.data(), oc.size() * sizeof(double), hipMemcpyHostToDevice, st));
    TBG_HIP(hipStreamSynchronize(st));
    check_norms();
}

template void corr_ac_impl<float>(tbg_handle*, const tbg_ham*, const double*, int, const double*,
                                  int, const double*, int, const double*, int, int, int, double,
                                  double*, int*);
template void corr_ac_impl<double>(tbg_handle*, const tbg_ham*, const double*, int, const double*,
                                   int, const double*, int, const double*, int, int, int, double,
                                   double*, int*);
template void dyn_pol_impl<float>(tbg_handle*, const tbg_ham*, const double*, int, const double*,
                                  int, const double*, int, const double*, int, int, const double*,
                                  int, const double*, int, double, double*, int*);
template void dyn_pol_impl<double>(tbg_handle*, const tbg_ham*, const double*, int,
                                   const double*, int, const double*, int, const double*, int, int,
                                   const double*, int, const double*, int, double, double*, int*);
template void corr_dc_impl<float>(tbg_handle*, const tbg_ham*, const double*, int, const double*,
                                  int, int, double, const double*, const int64_t*, int, int, double,
                                  double*, double*, int*, double*);
template void corr_dc_impl<double>(tbg_handle*, const tbg_ham*, const double*, int, const double*,
                                   int, int, double, const double*, const int64_t*, int, int,
                                   double, double*, double*, int*, double*);

}  // namespace tbg
