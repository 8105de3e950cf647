"""Resident passes (up to a whole time step per launch on blocks held in LDS
and registers) against one term per pass on the same Hamiltonian: states bit
for bit, correlations to the grouping of their FP64 sums (1e-13, sums of at
most a few thousand partials of size <= 1)."""
import math

import numpy as np
import pytest

import oracle
import tbplas_amd as tb
from tbplas_amd import tbpm
from conftest import golden, tau_of

pytestmark = pytest.mark.gpu


@pytest.fixture
def handle(gpu):
    h = tb._lib.Handle(0)
    yield h
    h.close()


def _sample(L1, L2, field=0.0, vac=0.02, W=0.6, seed=11):
    v = tb.random_vacancies(2 * L1 * L2, vac, seed) if vac else None
    s = tb.make_graphene_sample(L1, L2, vacancies=v)
    if W:
        tb.add_anderson_disorder(s, W, seed + 1)
    if field:
        s.set_magnetic_field(field, 0)
    s.rescale_ham(9.0)
    return s, oracle.build_ham_csr(s.orb_eng, s.hop_i, s.hop_j, s.hop_v)


def _states(n, K, seed=21):
    return tb.states.random_states(n, tb.states.sample_seeds(seed, K))


def _agree(h, H, bes, psi, T=9):
    """Resident passes on, then off: steps, a long series and C(t)."""
    coef = np.cos(np.arange(75) * 0.7) / (1.0 + np.arange(75))
    res = {}
    for on in (True, False):
        h.set_blocking(False)
        h.set_resident(on)
        h.set_kernel_timing(True)
        steps = [tbpm.cheb_step(H, bes, psi, fwd) for fwd in (True, False)]
        h.set_kernel_timing(False)
        assert any(k.startswith("ring") for k in h.kernel_times()) == on
        res[on] = steps + [tbpm.cheb_poly(H, coef, psi),
                           tbpm.corr_dos(H, bes, psi, T, chk_thr=1e-4)]
    for a, b in zip(res[True][:3], res[False][:3]):
        np.testing.assert_array_equal(a, b)
    assert np.max(np.abs(res[True][3] - res[False][3])) < 1e-13
    return res[True][3]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("K", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("L1,L2,field,W,tile", [
    (5, 4, 0.0, 0.0, 0.5),        # blocks that wrap around the sample
    (48, 31, 0.0, 0.6, 0.9),      # four entries a row
    (40, 52, 30.0, 0.0, 1.7),     # three complex entries a row
    (33, 47, 30.0, 0.6, 30.0)])   # one tile: split into blocks
def test_states_bitwise(handle, prec, K, L1, L2, field, W, tile):
    s, (ip, ix, dt) = _sample(L1, L2, field, 0.02 if L1 > 8 else 0.0, W)
    order, tiles = s.tile_order(tile, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision=prec, handle=handle, order=order,
                         tiles=tiles)
    bes = tbpm.bessel_series(tau_of(s), 1e-15)
    psi = _states(s.num_orb, K)
    c = _agree(handle, H, bes, psi)
    ref = oracle.orc_tbpm_dos(ip, ix, dt, bes, psi[:1], 9)
    assert np.max(np.abs(c[:1] - ref)) < (1e-12 if prec == "fp64" else 2e-5)
    H.close()


@pytest.mark.parametrize("nterms", [3, 4, 22, 34, 60])
def test_series_lengths(handle, nterms):
    """Passes of uneven length: short series, one term over a pass, more
    terms than one pass may have."""
    s, (ip, ix, dt) = _sample(60, 60)
    order, tiles = s.tile_order(1.3, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision="fp64", handle=handle, order=order,
                         tiles=tiles)
    tau = {3: 0.2, 4: 0.4, 22: 3.2, 34: 9.0, 60: 27.0}[nterms]
    bes = np.array([float(x) for x in tbpm.bessel_series(tau, 1e-30)[:nterms]])
    psi = _states(s.num_orb, 2)
    _agree(handle, H, bes, psi, T=3)
    H.close()


@pytest.mark.parametrize("prec,K,tile", [("fp32", 8, 4.8), ("fp64", 8, 3.2), ("fp64", 1, 7.5),
                                         ("fp32", 12, 3.8), ("fp32", 64, 1.5), ("fp32", 1, 16.0)])
def test_large_blocks(handle, prec, K, tile):
    """262,144 orbitals: blocks at the limits of a workgroup's LDS and
    registers, several per compute unit."""
    s, (ip, ix, dt) = _sample(300, 437, vac=0.0, W=0.0)
    order, tiles = s.tile_order(tile, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision=prec, handle=handle, order=order,
                         tiles=tiles)
    _agree(handle, H, tbpm.bessel_series(tau_of(s), 1e-15), _states(s.num_orb, K), T=5)
    H.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_wide_rows_and_scattered_tiles(handle, prec):
    """A random sparse Hermitian matrix (rows of ~9 entries) with tiles that
    are not spatial: every ring reaches the whole matrix."""
    rng = np.random.default_rng(31)
    n, m = 700, 2800
    hi, hj = rng.integers(0, n, m), rng.integers(0, n, m)
    keep = hi != hj
    hi, hj = hi[keep], hj[keep]
    hv = (rng.normal(size=len(hi)) + 1j * rng.normal(size=len(hi))) * 0.05
    ip, ix, dt = oracle.build_ham_csr(rng.uniform(-0.2, 0.2, n), hi, hj, hv)
    order = rng.permutation(n).astype(np.int64)
    H = tbpm.Hamiltonian(n, ip, ix, dt, precision=prec, handle=handle, order=order,
                         tiles=np.r_[np.arange(0, n, 32), n].astype(np.int64))
    bes = tbpm.bessel_series(math.pi, 1e-14)
    psi = _states(n, 3, seed=24)
    c = _agree(handle, H, bes, psi)
    ref = oracle.orc_tbpm_dos(ip, ix, dt, bes, psi, 9)
    assert np.max(np.abs(c - ref)) < (1e-12 if prec == "fp64" else 2e-5)
    H.close()


@pytest.mark.parametrize("prec,K", [("fp64", 1), ("fp32", 3), ("fp32", 4)])
def test_batch(handle, prec, K):
    """Uneven instances, one of them complex; correlations stay per instance."""
    hams, psis, refs = [], [], []
    bes = None
    for i, (L1, L2) in enumerate([(9, 14), (30, 22), (5, 5), (41, 17)]):
        s, (ip, ix, dt) = _sample(L1, L2, 25.0 if i == 3 else 0.0, 0.02 * (i % 2), 0.3 * i,
                                  seed=40 + i)
        bes = tbpm.bessel_series(tau_of(s), 1e-15)
        order, tiles = s.tile_order(0.8, return_tiles=True)
        hams.append(tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision=prec, handle=handle,
                                     order=order, tiles=tiles))
        psis.append(_states(s.num_orb, K, seed=400 + i))
        refs.append(oracle.orc_tbpm_dos(ip, ix, dt, bes, psis[-1], 20))
    handle.set_resident(True)
    out = tbpm.corr_dos_batch(hams, bes, psis, 20, chk_thr=1e-4)
    again = tbpm.corr_dos_batch(hams, bes, psis, 20, chk_thr=1e-4)
    for o, a, r in zip(out, again, refs):
        np.testing.assert_array_equal(o, a)
        assert np.max(np.abs(o - r)) < (1e-12 if prec == "fp64" else 2e-5)
    for H in hams:
        H.close()


def test_batch_tables_go_with_the_hamiltonians(gpu, handle):
    """Closing a batch's Hamiltonians gives its tables back (some 16 MB for
    the 183,000 orbitals here; the pages of other allocations may stay)."""
    s, csr = _sample(214, 214, vac=0.0)
    order, tiles = s.tile_order(2.4, return_tiles=True)
    bes, psi = tbpm.bessel_series(tau_of(s), 1e-15), _states(s.num_orb, 1)
    handle.set_resident(True)

    def free():
        gpu.cuda.synchronize()
        gpu.cuda.empty_cache()
        return gpu.cuda.mem_get_info()[0]

    def batch():
        hams = [tbpm.Hamiltonian(s.num_orb, *csr, precision="fp64", handle=handle, order=order,
                                 tiles=tiles) for _ in range(2)]
        out = tbpm.corr_dos_batch(hams, bes, [psi, psi], 4)
        with_tables = free()
        for H in hams:
            H.close()
        return out, with_tables

    first, _ = batch()
    before = free()
    for _ in range(3):
        out, with_tables = batch()
        np.testing.assert_array_equal(out, first)
    assert with_tables < before - 16e6
    assert free() >= before - 4e6


@pytest.mark.parametrize("what", ["ac", "dc"])
def test_conductivity_fixtures(handle, what):
    """The reference's AC and DC correlations on its own states."""
    g = golden(f"ref_{what}.npz")
    n = len(g["indptr"]) - 1
    handle.set_resident(True)
    H = tbpm.Hamiltonian(n, g["indptr"], g["indices"], g["hop"], g["dx"], g["dy"],
                         cur_scale=float(g["rescale"]), precision="fp64", handle=handle,
                         tiles=np.r_[np.arange(0, n, 32), n].astype(np.int64))
    if what == "ac":
        cF, cO = (tbpm.fermi_cheb_coef(2 ** 15, float(g["beta_re"]), float(g["mu_re"]), om, 1e-12)
                  for om in (False, True))
        avg = np.mean(tbpm.corr_ac(H, g["bes"], cF, cO, g["psi0"], int(g["T"])), axis=0)
        ref = g["corr"]
        assert np.max(np.abs(avg - ref)) < 1e-11 * max(1.0, np.max(np.abs(ref)))
    else:
        dos, dc = tbpm.corr_dc(H, g["bes"], g["psi0"], int(g["T"]), float(g["t_step"]),
                               g["energies"], g["en_inds"])
        ne = len(g["en_inds"])
        assert np.max(np.abs(dos.mean(axis=0) - g["dos"])) < 1e-12
        assert np.max(np.abs(dc.mean(axis=0) - g["dc"][:, :ne])) < \
            1e-10 * max(1.0, np.max(np.abs(g["dc"])))
    H.close()


@pytest.mark.parametrize("prec,other", [("fp64", "fp32"), ("fp32", "fp64")])
@pytest.mark.parametrize("K", [1, 3])
def test_layout_queries_in_the_other_precision(handle, prec, other, K):
    """What a run would look like in the other precision does not change what
    runs: odd state counts have the same groups in both."""
    s, (ip, ix, dt) = _sample(31, 24)
    order, tiles = s.tile_order(1.3, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision=prec, handle=handle, order=order,
                         tiles=tiles)
    bes = np.array([float(x) for x in tbpm.bessel_series(math.pi, 1e-30)[:21]])
    psi = _states(s.num_orb, K)
    handle.set_resident(True)
    for query in (H.blocking_info, H.blocking_launch, H.blocking_bytes):
        theirs, ours = query(K, other), query(K)
        assert theirs and ours
    got = tbpm.corr_dos(H, bes, psi, 6, chk_thr=1e-4)
    handle.set_resident(False)
    handle.set_blocking(False)
    assert np.max(np.abs(got - tbpm.corr_dos(H, bes, psi, 6, chk_thr=1e-4))) < 1e-13
    H.close()


def test_graph_replay_and_timing(handle):
    """Replayed steps equal launched ones; the step counter and the norm
    check work with resident passes."""
    s, (ip, ix, dt) = _sample(40, 40)
    order, tiles = s.tile_order(1.0, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, dt, precision="fp32", handle=handle, order=order,
                         tiles=tiles)
    bes = tbpm.bessel_series(tau_of(s), 1e-15)
    psi = _states(s.num_orb, 4)
    handle.set_resident(True)
    out = []
    for graph in (True, True, False):
        handle.set_graph(graph)
        out.append(tbpm.corr_dos(H, bes, psi, 70, chk_thr=1e-4))
    np.testing.assert_array_equal(out[0], out[1])
    np.testing.assert_array_equal(out[0], out[2])
    with pytest.raises(tb._lib.NormError):
        tbpm.corr_dos(H, bes, psi, 20, chk_step=10, chk_thr=1e-30)
    H.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 2e-4)])
@pytest.mark.parametrize("resident", [True, False])
@pytest.mark.parametrize("T,n_en,K", [(1, 1, 1), (2, 3, 2), (7, 16, 3), (16, 2, 4), (17, 17, 2),
                                      (33, 9, 5), (50, 33, 1)])
def test_dc_step_blocks_vs_oracle(handle, prec, tol, resident, T, n_en, K):
    """The quasi-eigenstates and the DC correlations are summed over blocks
    of up to 16 kept steps: block lengths and remainders, energies around the
    16 of a tile, states in planes and row by row.  Tolerances as in the
    other comparisons of corr_dc with the oracle; the chosen energies keep
    |<psi0|QE>| away from zero in both."""
    s, _ = _sample(9, 14)
    ip, ix, hop, dx, dy = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    bes = tbpm.bessel_series(tau_of(s), 1e-14)
    psi = _states(s.num_orb, K)
    t_step = 2 * math.pi / 18.0
    en = np.linspace(-2.6, 2.6, 64)
    inds = np.unique(np.linspace(3, 60, n_en).astype(int))
    assert len(inds) == n_en
    handle.set_blocking(False)
    handle.set_resident(resident)
    order, tiles = s.tile_order(1.3, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, hop, dx, dy, cur_scale=9.0, precision=prec,
                         handle=handle, order=order if resident else None,
                         tiles=tiles if resident else None)
    d, c = tbpm.corr_dc(H, bes, psi, T, t_step, en, inds)
    rd, rc = oracle.orc_tbpm_dccond(ip, ix, hop, dx, dy, 9.0, bes, psi, T, t_step, en, inds)
    assert np.max(np.abs(d - rd)) < tol
    assert np.max(np.abs(c - rc)) < tol * max(1.0, np.max(np.abs(rc)))
    g = tbpm.quasi_eigenstates(H, bes, psi, T, t_step, list(en[inds]))
    r = oracle.orc_quasi_eigenstates(ip, ix, hop, bes, psi, T, t_step, list(en[inds]))
    assert np.max(np.abs(g - r)) < tol * max(1.0, np.max(r))
    H.close()


def test_dc_more_energies_than_grid_rows(handle):
    """1,050,000 energies are 65,625 groups of 16, more than a grid's 65,535
    rows: the same numbers over and over (1e-12 of the largest: sums of 64
    rows in another grouping)."""
    s, _ = _sample(4, 8, vac=0.0)
    ip, ix, hop, dx, dy = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    bes = tbpm.bessel_series(tau_of(s), 1e-14)
    psi = _states(s.num_orb, 1)
    en = np.linspace(-2.6, 2.6, 16)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, hop, dx, dy, cur_scale=9.0, precision="fp64",
                         handle=handle)
    few = tbpm.corr_dc(H, bes, psi, 2, 2 * math.pi / 18.0, en, np.arange(16))[1]
    many = tbpm.corr_dc(H, bes, psi, 2, 2 * math.pi / 18.0, en, np.arange(1_050_000) % 16)[1]
    many = many.reshape(1, 2, -1, 16, 2)
    assert np.max(np.abs(many - few[:, :, None])) < 1e-12 * max(1.0, np.max(np.abs(few)))
    H.close()


def test_dc_sums_round_as_trees(handle):
    """After one step the window is zero, QE is psi0 and the correlation is
    |J psi0|^2 / |psi0|^2 of 24,000 positive terms.  Against 80-bit sums: a
    chain of n equal terms leaves sqrt(n / 3) roundings of 2^-53 / sqrt(3),
    0.64e-16 of the sum each.  The partial sums of 384 splits, by eights, and
    of 94 chunks, by 32s, leave chains of 3 to 32: 2.1e-16 together, allowed
    twice; one after the other they leave 7e-16 and 4e-16, and more where
    terms of one size round alike."""
    s, _ = _sample(100, 120, 20.0, 0.0, 0.0)
    ip, ix, hop, dx, dy = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, hop, dx, dy, cur_scale=9.0, precision="fp64",
                         handle=handle)
    bes = tbpm.bessel_series(tau_of(s), 1e-14)
    err = []
    for psi in _states(s.num_orb, 24):
        c = tbpm.corr_dc(H, bes, psi[None], 1, 2 * math.pi / 18.0, np.array([0.1]), np.arange(1))[1]
        z = psi.astype(np.clongdouble)
        for a, d in enumerate((dx, dy)):
            j = np.add.reduceat(hop.astype(np.clongdouble) * d * 9.0 * z[ix], ip[:-1])
            want = np.sum(np.abs(j) ** 2) / np.sum(np.abs(z) ** 2)
            err.append(float((np.clongdouble(c[0, a, 0, 0]) - want).real / want))
    assert np.sqrt(np.mean(np.square(err))) < 4.2e-16
    H.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("resident", [True, False])
@pytest.mark.parametrize("T", [7, 16, 37])
def test_dc_kept_steps(handle, prec, resident, T):
    """Runs that keep 1, 2, 4 or 8 states (less memory) give what runs that
    keep 16 give: the same quasi-eigenstates bit for bit (each is summed step
    by step in every block length), and correlations to the grouping of the
    rows (1e-12 of the largest)."""
    s, _ = _sample(9, 14)
    ip, ix, hop, dx, dy = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    bes = tbpm.bessel_series(tau_of(s), 1e-14)
    psi = _states(s.num_orb, 3)
    en = np.linspace(-2.6, 2.6, 18)
    handle.set_blocking(False)
    handle.set_resident(resident)
    order, tiles = s.tile_order(1.3, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, hop, dx, dy, cur_scale=9.0, precision=prec,
                         handle=handle, order=order if resident else None,
                         tiles=tiles if resident else None)
    res = {}
    for most in (16, 8, 5, 2, 1):
        handle.set_kept_steps(most)
        d, c = tbpm.corr_dc(H, bes, psi, T, 2 * math.pi / 18.0, en, np.arange(18))
        res[most] = d, c, tbpm.quasi_eigenstates(H, bes, psi, T, 2 * math.pi / 18.0, list(en))
    d16, c16, q16 = res[16]
    for d, c, q in res.values():
        np.testing.assert_array_equal(d, d16)
        np.testing.assert_array_equal(q, q16)
        assert np.max(np.abs(c - c16)) < 1e-12 * max(1.0, np.max(np.abs(c16)))
    for bad in (0, 17):
        with pytest.raises(tb._lib.TBGError):
            handle.set_kept_steps(bad)
    H.close()


@pytest.mark.parametrize("prec,resident,K,n_en", [
    ("fp64", True, 32, 1024), ("fp64", True, 32, 1025), ("fp64", False, 32, 2100),
    ("fp32", True, 32, 2049), ("fp64", False, 8, 4097)])
def test_dc_many_energies(handle, prec, resident, K, n_en):
    """More energies than one launch takes (its tiles of a current, a state
    and 16 energies are at most 16 a compute unit; 1024 energies of 32 states
    on 256 units): the same numbers as runs over parts of the energies, of
    which each sum is independent (1e-12 of the largest: sums of 128 rows in
    another grouping)."""
    s, _ = _sample(6, 9, vac=0.0)
    ip, ix, hop, dx, dy = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    bes = tbpm.bessel_series(tau_of(s), 1e-14)
    psi = _states(s.num_orb, K)
    en = np.linspace(-2.6, 2.6, n_en)
    handle.set_blocking(False)
    handle.set_resident(resident)
    order, tiles = s.tile_order(1.3, return_tiles=True)
    H = tbpm.Hamiltonian(s.num_orb, ip, ix, hop, dx, dy, cur_scale=9.0, precision=prec,
                         handle=handle, order=order if resident else None,
                         tiles=tiles if resident else None)
    run = [tbpm.corr_dc(H, bes, psi, 3, 2 * math.pi / 18.0, en, inds)
           for inds in (np.arange(n_en), np.arange(7), np.arange(n_en - 19, n_en))]
    assert np.all(np.isfinite(run[0][1]))
    np.testing.assert_array_equal(run[0][0], run[1][0])
    for part, got in ((run[1][1], run[0][1][:, :, :7]), (run[2][1], run[0][1][:, :, -19:])):
        assert np.max(np.abs(got - part)) < 1e-12 * max(1.0, np.max(np.abs(part)))
    H.close()


@pytest.mark.parametrize("resident", [True, False])
@pytest.mark.parametrize("cuts", [[1] * 5, [15, 1, 16, 17], [16, 33], [3, 40, 5], [64], [2, 2, 2]])
def test_sums_kept_over_steps_equal_sums_of_single_steps(handle, resident, cuts):
    """The partial sums of up to 16 steps are added by one launch: a run cut
    anywhere (graphs of any length, rests) has the rows of a run whose steps
    are launched and summed one by one, bit for bit."""
    s, csr = _sample(12, 17)
    order, tiles = s.tile_order(1.0, return_tiles=True)
    handle.set_blocking(False)
    handle.set_resident(resident)
    H = tbpm.Hamiltonian(s.num_orb, *csr, precision="fp64", handle=handle, order=order,
                         tiles=tiles)
    bes, psi, T = tbpm.bessel_series(tau_of(s), 1e-14), _states(s.num_orb, 2), sum(cuts)
    run = tbpm.DosRun(H, bes, psi, T)
    for c in cuts:
        run.advance(c)
    got = run.result()
    run.close()
    handle.set_graph(False)
    single = tbpm.DosRun(H, bes, psi, T)
    for _ in range(T):
        single.advance(1)
    want = single.result()
    single.close()
    np.testing.assert_array_equal(got, want)
    H.close()
