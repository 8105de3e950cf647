// Kubo-Bastin Hall conductivity moments (KPM): mu_mn of tbpm_kbdc
// (tbplas/fortran/tbpm.f90:836-960), and the Haydock recursion
// coefficients of ldos_haydock (tbpm.f90:964-1024, Haydock_coef
// propagation.f90:85-155), on the device.
//
// For each state psi: W_j = J_b T_j(H~) psi (j < N, b = x or y), P_i =
// T_i(H~) J_x psi (i < N) and mu(i, j) = g_i g_j <P_i | W_j> with the Jackson
// weights g (kpm.f90:8-29).  The Chebyshev vectors (T_j = 2 H~ T_{j-1} -
// T_{j-2}, in place over T_{j-2}) and the current of each come from one
// kernel (k_hall_term); the N x N Gram matrix P^H W is formed
// per block of up to 256 rows of mu on the FP64 matrix cores (k_gram: a
// complex product as four real 16x16x4 MFMAs, the long n dimension split
// over workgroups and summed in a fixed order by k_gram_sum).  Complex128
// only: the moments are sums of N^2 products that complex64 would leave at
// ~1e-7 of their size.
#include <cmath>
#include <type_traits>
#include <vector>

#include "tbg_engine.h"

namespace tbg {

namespace {

// One Chebyshev term and one current from one gather of x: out[r] = alpha
// (H~ x)[r] - prev[r] (alpha = 2; first: (H~ x)[r]; out may be prev) unless
// out is null, and with CUR w[r] = (J x)[r].  A thread per row; neighbouring
// rows stay on one XCD from launch to launch.  Bound by the matrix and the
// vectors in L2 and the Infinity Cache and by the chain column number ->
// gather -> store: 4.9 us with the current and 4.4 us without at 200,000
// rows of three complex entries (a term and an SpMV launch took 5.4 + 5.8
// and 5.4 us; the SpMV read x and the column numbers again).
template <bool RV, bool CUR>
__global__ void __launch_bounds__(256)
k_hall_term(const int* __restrict__ cols, const void* __restrict__ vals,
            const double2* __restrict__ jb, const int64_t* __restrict__ soff,
            const int* __restrict__ sw, int64_t nslices, const double2* x, const double2* prev,
            double2* out, double2* __restrict__ w, int first) {
    const int lane = threadIdx.x & 63;
    const int sl = __builtin_amdgcn_readfirstlane(
        remap_chunk(blockIdx.x, gridDim.x) * 4 + (int)(threadIdx.x >> 6));
    if (sl >= nslices) return;
    const int64_t r = (int64_t)sl * 64 + lane, off = soff[sl] + lane;
    const int width = sw[sl];
    const bool term = out != nullptr;
    double2 p = make_double2(0.0, 0.0);
    if (term && !first) p = prev[r];
    double hr = 0.0, hi = 0.0, jr = 0.0, ji = 0.0;
    auto entries = [&](auto count, int j0) {
        constexpr int E = decltype(count)::value;
        int c[E];
        double2 h[E], q[E], v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int64_t o = off + (int64_t)(j0 + e) * 64;
            c[e] = cols[o];
            h[e] = q[e] = make_double2(0.0, 0.0);
            if (term) {
                if constexpr (RV) h[e].x = reinterpret_cast<const double*>(vals)[o];
                else h[e] = reinterpret_cast<const double2*>(vals)[o];
            }
            if constexpr (CUR) q[e] = jb[o];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = x[c[e]];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if constexpr (RV) {
                hr = fma(h[e].x, v[e].x, hr);
                hi = fma(h[e].x, v[e].y, hi);
            } else {
                hr = fma(-h[e].y, v[e].y, fma(h[e].x, v[e].x, hr));
                hi = fma(h[e].y, v[e].x, fma(h[e].x, v[e].y, hi));
            }
            if constexpr (CUR) {
                jr = fma(-q[e].y, v[e].y, fma(q[e].x, v[e].x, jr));
                ji = fma(q[e].y, v[e].x, fma(q[e].x, v[e].y, ji));
            }
        }
    };
    int j = 0;
    for (; j + 4 <= width; j += 4) entries(std::integral_constant<int, 4>{}, j);
    switch (width - j) {
        case 3: entries(std::integral_constant<int, 3>{}, j); break;
        case 2: entries(std::integral_constant<int, 2>{}, j); break;
        case 1: entries(std::integral_constant<int, 1>{}, j); break;
        default: break;
    }
    if (term) {
        const double al = first ? 1.0 : 2.0;
        out[r] = make_double2(fma(al, hr, -p.x), fma(al, hi, -p.y));
    }
    if constexpr (CUR) w[r] = make_double2(jr, ji);
}

// Gram matrix of the Hall moments on the FP64 matrix cores:
// part[z][m][j] = sum_{k in split z} conj(P[m][k]) W[j][k] for m < rows,
// j < N, with P and W column-major (column m of P at P + m * np).  A
// workgroup (4 waves) owns a 128 x 64 tile of the output and one split of
// k; it stages 8 rows of k of both operands in LDS (two buffers, one
// barrier a stage) and each wave accumulates a 64 x 32 sub-tile as 4 x 2
// blocks of v_mfma_f64_16x16x4f64: re += Pr Wr + Pi Wi, im += Pr Wi - Pi Wr.
// 128 x 64 with 64 x 32 a wave needs 6 LDS reads for 32 MFMAs where 32 x 32
// needed 4 (twice as wide) for 16, and its staged columns serve 1.5 times the
// products: 256 x 2048 moments of 200,000 rows in 12.5 ms, 67 TFLOP/s, 93% of
// what a large complex128 library product reaches on the same card (64 x 64
// tiles: 13.5 to 14.4 ms).
// Operand layout of the instruction: lane i + 16 k holds A[i][k] and
// B[k][i]; the result D[i][j] sits in lane j + 16 (i % 4), element i / 4
// (checked on the device with known operands).
constexpr int kGramM = 128, kGramN = 64;   // output rows / columns per workgroup
constexpr int kGramK = 8;                  // rows of k per LDS stage
constexpr int kGramLd = kGramK + 1;   // LDS stride in complex values from one operand
                                       // column to the next: 36 banks, so the 16
                                       // lanes of an operand read land on distinct
                                       // groups of four
constexpr int kGramPerCu = 2;          // workgroups a CU holds (registers)
typedef double gram_d4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256, kGramPerCu)
k_gram(const double2* __restrict__ P, const double2* __restrict__ W, int64_t np, int rows,
       int N, int64_t kchunk, double2* __restrict__ part) {
    __shared__ double2 lds[2][kGramM + kGramN][kGramLd];   // [P columns, W columns][k]
    // an XCD's workgroups: the tiles of one split first, so that they read
    // the same rows of P and W at about the same time
    const int tm = (rows + kGramM - 1) / kGramM, tn = (N + kGramN - 1) / kGramN;
    const int b = remap_chunk(blockIdx.x, gridDim.x);
    const int m0 = b % tm * kGramM, j0 = b / tm % tn * kGramN, z = b / (tm * tn);
    const int64_t kb = z * kchunk;
    const int64_t ke = kb + kchunk < np ? kb + kchunk : np;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = (w >> 1) * 64, wn = (w & 1) * 32;
    const int li = lane & 15, lk = lane >> 4;
    gram_d4 cre[4][2], cim[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            cre[a][c] = gram_d4{0.0, 0.0, 0.0, 0.0};
            cim[a][c] = gram_d4{0.0, 0.0, 0.0, 0.0};
        }
    // The next stage's operands are loaded into registers while the MFMAs
    // of this one run, then stored to the other LDS buffer.  Columns past
    // the end repeat the last one: their results are not stored.
    constexpr int Q = (kGramM + kGramN) / 32;
    const int sk = t & 7, sm = t >> 3;
    const double2* src[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = sm + 32 * q;
        src[q] = (c < kGramM ? P + (int64_t)min(m0 + c, rows - 1) * np
                             : W + (int64_t)min(j0 + c - kGramM, N - 1) * np) + sk;
    }
    double2 nx[Q];
    auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            nx[q] = k0 + sk < ke ? src[q][k0] : make_double2(0.0, 0.0);
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int q = 0; q < Q; ++q) lds[buf][sm + 32 * q][sk] = nx[q];
    };
    if (kb < ke) {
        fetch(kb);
        put(0);
    }
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = kb; k0 < ke; k0 += kGramK, buf ^= 1) {
        const bool more = k0 + kGramK < ke;
        if (more) fetch(k0 + kGramK);
#pragma unroll
        for (int kk = 0; kk < kGramK; kk += 4) {
            double2 A[4], Bv[2];
#pragma unroll
            for (int a = 0; a < 4; ++a) A[a] = lds[buf][wm + 16 * a + li][kk + lk];
#pragma unroll
            for (int c = 0; c < 2; ++c) Bv[c] = lds[buf][kGramM + wn + 16 * c + li][kk + lk];
            // sixteen independent accumulators between two products into
            // the same one; each gets its products in the order re: Pr Wr,
            // Pi Wi and im: Pr Wi, -Pi Wr
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    cre[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[a].x, Bv[c].x, cre[a][c],
                                                                     0, 0, 0);
                    cim[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[a].x, Bv[c].y, cim[a][c],
                                                                     0, 0, 0);
                }
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    cre[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[a].y, Bv[c].y, cre[a][c],
                                                                     0, 0, 0);
                    cim[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(-A[a].y, Bv[c].x, cim[a][c],
                                                                     0, 0, 0);
                }
        }
        if (more) put(buf ^ 1);
        __syncthreads();
    }
    double2* out = part + (int64_t)z * rows * N;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + wm + 16 * a + lk + 4 * v;
                const int j = j0 + wn + 16 * c + li;
                if (m < rows && j < N)
                    out[(int64_t)m * N + j] = make_double2(cre[a][c][v], cim[a][c][v]);
            }
}

// mu(i0 + m, j) = g_{i0 + m} g_j sum_z part[z][m][j] in the order z = 0, 1,
// ... (the reference's g(:) * g(j) * corr_mu(:, j)), at i si + j sj of mu.
__global__ void k_gram_sum(const double2* __restrict__ part, int nsplit, int rows, int N,
                           const double* __restrict__ g, int i0, double2* __restrict__ mu,
                           int64_t si, int64_t sj) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)rows * N) return;
    const int m = (int)(q / N), j = (int)(q % N);
    double re = 0.0, im = 0.0;
    for (int z = 0; z < nsplit; ++z) {
        const double2 v = part[(int64_t)z * rows * N + q];
        re += v.x;
        im += v.y;
    }
    const double w = g[i0 + m] * g[j];
    mu[(i0 + m) * si + j * sj] = make_double2(w * re, w * im);
}

// Haydock step i on one vector (Kp = 1): buf -= a_i cur + b_{i-1} prev with
// a_i = dots[3i] + i dots[3i+1] and b_{i-1} = sqrt(nrm[3(i-1)+2]) read on
// the device (axpbypz, propagation.f90:144).
__global__ void k_lz_update(double2* __restrict__ buf, const double2* __restrict__ cur,
                            const double2* __restrict__ prev, int64_t np,
                            const double* __restrict__ dots, const double* __restrict__ nrm,
                            int i) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= np) return;
    const double ar = dots[3 * i], ai = dots[3 * i + 1];
    const double b = i > 0 ? sqrt(nrm[3 * (i - 1) + 2]) : 0.0;
    const double2 c = cur[r], p = prev[r];
    double2 v = buf[r];
    v.x = v.x - (ar * c.x - ai * c.y) - b * p.x;
    v.y = v.y - (ar * c.y + ai * c.x) - b * p.y;
    buf[r] = v;
}

// buf /= b_i = sqrt(nrm[3i+2]) (propagation.f90:146)
__global__ void k_lz_scale(double2* __restrict__ buf, int64_t np, const double* __restrict__ nrm,
                           int i) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= np) return;
    const double b = sqrt(nrm[3 * i + 2]);
    double2 v = buf[r];
    v.x = v.x / b;
    v.y = v.y / b;
    buf[r] = v;
}

}  // namespace

void haydock_impl(tbg_handle* h, const tbg_ham* H, const double* psi0, int K, int depth,
                  double rescale, double* coefa, double* coefb) {
    const hipStream_t st = h->stream;
    Engine<double> e;
    e.init(h, view_of(H), {0, H->nslices}, 1, chunk_target(h, H->nslices), nullptr);
    TBG_REQUIRE(e.Kp == 1, "internal: one state per Haydock launch");
    const int64_t n = H->n, np = e.n_pad;
    const size_t vb = (size_t)np * sizeof(double2);
    DevBuf v0(vb), v1(vb), v2(vb);
    DevBuf dots((size_t)depth * 3 * sizeof(double)), nrm((size_t)depth * 3 * sizeof(double));
    double* part = e.part.template as<double>();
    const int* range = e.plan.inst_chunk_dev.template as<int>();
    const unsigned nb = (unsigned)((np + 255) / 256);
    std::vector<double> hd((size_t)depth * 3), hn((size_t)depth * 3);
    for (int s = 0; s < K; ++s) {
        void* cur = v0.p;
        void* prev = v1.p;
        void* buf = v2.p;
        launch_fill_zero(cur, vb, st);
        launch_fill_zero(prev, vb, st);
        launch_pack<double>(psi0 + (size_t)s * n * 2, 1, n, cur, 1, 0, H->perm_ptr(), st);
        for (int i = 0; i < depth; ++i) {
            TermArgs a = e.base_args(0, 0);   // buf = rescale H~ cur  (amv)
            a.pin = cur;
            a.pout = buf;
            a.ar[0] = a.ar[1] = rescale;
            a.ai[0] = a.ai[1] = 0.0;
            launch_term<double>(F_STORE, a, e.plan.nchunks, st);
            launch_dotnorm<double>(e.plan, cur, buf, 1, 1, part, st);   // a_i = <cur|buf>
            launch_reduce(part, 3, range, 1, dots.as<double>(), 0, nullptr, i, st);
            hipLaunchKernelGGL(k_lz_update, dim3(nb), dim3(256), 0, st,
                               reinterpret_cast<double2*>(buf),
                               reinterpret_cast<const double2*>(cur),
                               reinterpret_cast<const double2*>(prev), np, dots.as<double>(),
                               nrm.as<double>(), i);
            TBG_HIP(hipGetLastError());
            launch_dotnorm<double>(e.plan, buf, buf, 1, 1, part, st);   // b_i = |buf|
            launch_reduce(part, 3, range, 1, nrm.as<double>(), 0, nullptr, i, st);
            hipLaunchKernelGGL(k_lz_scale, dim3(nb), dim3(256), 0, st,
                               reinterpret_cast<double2*>(buf), np, nrm.as<double>(), i);
            TBG_HIP(hipGetLastError());
            void* t = prev;
            prev = cur;
            cur = buf;
            buf = t;
        }
        TBG_HIP(hipMemcpyAsync(hd.data(), dots.p, hd.size() * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        TBG_HIP(hipMemcpyAsync(hn.data(), nrm.p, hn.size() * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        TBG_HIP(hipStreamSynchronize(st));
        for (int i = 0; i < depth; ++i) {
            coefa[((size_t)s * depth + i) * 2 + 0] = hd[(size_t)i * 3 + 0];
            coefa[((size_t)s * depth + i) * 2 + 1] = hd[(size_t)i * 3 + 1];
            coefb[(size_t)s * depth + i] = std::sqrt(hn[(size_t)i * 3 + 2]);
        }
    }
}

void hall_mu_impl(tbg_handle* h, const tbg_ham* H, const double* psi0, int K, int N, int dir,
                  bool rows_first, double* mu) {
    const hipStream_t st = h->stream;
    const int64_t n = H->n, np = H->nslices * 64;
    const size_t vb = (size_t)np * sizeof(double2);
    // Jackson kernel (kpm.f90:20-27)
    std::vector<double> g(N);
    g[0] = 0.5;
    const double q = M_PI / N, cotq = std::cos(q) / std::sin(q);
    for (int k = 1; k < N; ++k) g[k] = ((N - k) * std::cos(q * k) + cotq * std::sin(q * k)) / N;
    DevBuf dg(g.size() * sizeof(double));
    TBG_HIP(hipMemcpyAsync(dg.p, g.data(), g.size() * sizeof(double), hipMemcpyHostToDevice, st));
    const int B = std::min(N, 256);
    DevBuf W((size_t)N * vb), Pb((size_t)B * vb), T0(vb), T1(vb), psi(vb);
    auto col = [&](DevBuf& m, int j) {
        return reinterpret_cast<double2*>(reinterpret_cast<char*>(m.p) + (size_t)j * vb);
    };
    // out = T_m from x = T_{m-1} and prev = T_{m-2} (null: m = 1); w = J x
    auto step = [&](const double2* x, const double2* prev, double2* out, const void* J,
                    double2* w) {
        const dim3 grid((unsigned)((H->nslices + 3) / 4));
#define TBG_HALL(RV, CUR)                                                                     \
    hipLaunchKernelGGL((k_hall_term<RV, CUR>), grid, dim3(256), 0, st, H->cols.as<int>(),      \
                       H->vals.p, reinterpret_cast<const double2*>(J),                         \
                       H->slice_off.as<int64_t>(), H->slice_w.as<int>(), H->nslices, x, prev,  \
                       out, w, prev == nullptr ? 1 : 0)
        if (H->real_vals) {
            if (J) TBG_HALL(true, true);
            else TBG_HALL(true, false);
        } else {
            if (J) TBG_HALL(false, true);
            else TBG_HALL(false, false);
        }
#undef TBG_HALL
        TBG_HIP(hipGetLastError());
    };
    // The k split of the Gram blocks: rounds of resident workgroups times the
    // rows of k of each, plus about 200 rows' worth for its start and its
    // partial sums; among equals the finest (the last round ends together).
    // 8, 16 and 24 splits of the size above take the same 12.5 ms.
    auto split_of = [&](int rows) {
        const int64_t tiles = (int64_t)((rows + kGramM - 1) / kGramM) * ((N + kGramN - 1) / kGramN);
        const int64_t slots = (int64_t)kGramPerCu * h->num_cus;
        int64_t best = 1, cost = 0;
        for (int64_t s = 1; s <= 64 && s * 4 * kGramK <= std::max<int64_t>(np, 4 * kGramK); ++s) {
            const int64_t c = (tiles * s + slots - 1) / slots * ((np + s - 1) / s + 200);
            if (s == 1 || c <= cost) {
                best = s;
                cost = c;
            }
        }
        return best;
    };
    // The partial sums of as many splits (of B rows; a last block of fewer
    // rows has more) as the vectors leave memory for: 200 MB at the size
    // above, 4 GB for 20,000 moments.
    const int tail = N % B ? N % B : B;
    const int64_t units = std::max(split_of(B), (split_of(tail) * tail + B - 1) / B);
    DevBuf gpart;
    const int64_t gcols = alloc_units(gpart, (size_t)B * N * sizeof(double2), units) * B;
    for (int s = 0; s < K; ++s) {
        double2* cur = T0.as<double2>();   // T_j
        double2* oth = T1.as<double2>();   // T_{j-1}; T_{j+1} is formed in place over it
        const double2* x = psi.as<double2>();
        launch_fill_zero(psi.p, vb, st);
        launch_pack<double>(psi0 + (size_t)s * n * 2, 1, n, psi.p, 1, 0, H->perm_ptr(), st);
        // W_j = J_b T_j psi (tbpm.f90:892-922)
        const void* jb = dir == 1 ? H->jx.p : H->jy.p;
        for (int j = 0; j < N; ++j) {
            const double2* prev = j == 0 ? nullptr : j == 1 ? psi.as<double2>() : oth;
            step(x, prev, j + 1 < N ? oth : nullptr, jb, col(W, j));
            std::swap(cur, oth);
            x = cur;
        }
        // P_i = T_i J_x psi in blocks of B columns, mu[i0.., :] = P^H W
        double2* mus = reinterpret_cast<double2*>(mu) + (size_t)s * N * N;
        const double2* p0 = nullptr;   // P_{i-2}
        const double2* p1 = nullptr;   // P_{i-1}
        for (int i = 0; i < N; ++i) {
            double2* pi = col(Pb, i % B);
            if (i == 0) step(psi.as<double2>(), nullptr, nullptr, H->jx.p, pi);
            else step(p1, p0, pi, nullptr, nullptr);
            p0 = p1;
            p1 = pi;
            if (i % B == B - 1 || i == N - 1) {
                const int i0 = i - i % B, rows = i % B + 1;
                const int64_t want = std::min(split_of(rows), gcols / rows);
                const int64_t kchunk = ((np + want - 1) / want + kGramK - 1) / kGramK * kGramK;
                const int64_t nsplit = (np + kchunk - 1) / kchunk;
                const dim3 grid((unsigned)(nsplit * ((N + kGramN - 1) / kGramN) *
                                           ((rows + kGramM - 1) / kGramM)));
                timed_launch(h, kTimeGram, [&] {
                    hipLaunchKernelGGL(k_gram, grid, dim3(256), 0, st, Pb.as<double2>(),
                                       W.as<double2>(), np, rows, N, kchunk,
                                       gpart.as<double2>());
                    TBG_HIP(hipGetLastError());
                });
                const int64_t nq = (int64_t)rows * N;
                hipLaunchKernelGGL(k_gram_sum, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0,
                                   st, gpart.as<double2>(), (int)nsplit, rows, N,
                                   dg.as<double>(), i0, mus, rows_first ? (int64_t)N : 1,
                                   rows_first ? 1 : (int64_t)N);
                TBG_HIP(hipGetLastError());
            }
        }
    }
    TBG_HIP(hipStreamSynchronize(st));
}

}  // namespace tbg
