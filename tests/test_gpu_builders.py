"""GPU CSR assembly, rescale and Peierls phases: bit-exact against the oracle
restatements of the reference builders (sample.pyx:18-257, sample.py:375-391)."""
import numpy as np
import pytest

import oracle
import tbplas_amd as tb
from conftest import golden

pytestmark = pytest.mark.gpu


def _samples():
    rng = np.random.default_rng(42)
    out = []
    s = tb.make_graphene_sample(16)
    out.append(("pristine16", s))
    s = tb.make_graphene_sample(9, 7, pbc=(False, False))
    out.append(("open9x7", s))
    n0 = 2 * 20 * 20
    s = tb.make_graphene_sample(20, vacancies=tb.random_vacancies(n0, 0.03, 1))
    tb.add_anderson_disorder(s, 1.0, 2)
    s.orb_eng[::7] = 0.0
    out.append(("vac_anderson20", s))
    s = tb.make_graphene_sample(12)
    s.set_magnetic_field(20.0, 0)
    out.append(("peierls12", s))
    s = tb.make_graphene_sample(2)       # wrapped duplicates (both directions)
    out.append(("tiny2", s))
    s = tb.make_graphene_sample(1, 3)    # self-hops and multiple duplicates
    out.append(("tiny1x3", s))
    for name, s in out:
        s.hop_v = s.hop_v * np.exp(1j * rng.uniform(-0.3, 0.3, s.num_hop)) if name == "open9x7" else s.hop_v
    return out


@pytest.mark.parametrize("idx", range(6))
def test_build_ham_dxy_bit_exact(gpu, idx):
    name, s = _samples()[idx]
    s.rescale_ham(9.0)
    got = s.build_ham_dxy()
    ref = oracle.build_ham_dxy_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v, s.dr)
    for g, r in zip(got, ref):
        assert g.dtype == r.dtype
        np.testing.assert_array_equal(g, r, err_msg=name)


@pytest.mark.parametrize("idx", range(6))
def test_build_ham_csr_canonical_bit_exact(gpu, idx):
    name, s = _samples()[idx]
    s.rescale_ham(9.0)
    m = s.build_ham_csr()
    ip, ix, dt = oracle.build_ham_csr(s.orb_eng, s.hop_i, s.hop_j, s.hop_v)
    np.testing.assert_array_equal(m.indptr.astype(np.int64), ip, err_msg=name)
    np.testing.assert_array_equal(m.indices.astype(np.int64), ix, err_msg=name)
    np.testing.assert_array_equal(m.data, dt, err_msg=name)


def test_builders_golden_fixture(gpu):
    g = golden("graphene4.npz")
    s = tb.Sample(g["orb_eng"], g["orb_pos"], g["hop_i"], g["hop_j"], g["hop_v"], g["dr"])
    ip, ix, h, dx, dy = s.build_ham_dxy()
    np.testing.assert_array_equal(ip, g["dxy_indptr"])
    np.testing.assert_array_equal(ix, g["dxy_indices"])
    np.testing.assert_array_equal(h, g["dxy_hop"])
    np.testing.assert_array_equal(dx, g["dxy_dx"])
    np.testing.assert_array_equal(dy, g["dxy_dy"])
    m = s.build_ham_csr()
    np.testing.assert_array_equal(m.indices, g["csr_indices"])
    np.testing.assert_array_equal(m.data, g["csr_data"])


def test_get_rescale_bit_exact(gpu):
    for name, s in _samples():
        assert s.get_rescale() == oracle.get_rescale_loop(s.orb_eng, s.hop_i, s.hop_j, s.hop_v), name


def test_rescale_ham_none_uses_estimate(gpu):
    s = tb.make_graphene_sample(8)
    s.rescale_ham()
    assert s.rescale == pytest.approx(8.1, abs=1e-12)
    assert np.allclose(np.abs(s.hop_v), 2.7 / s.rescale)


@pytest.mark.parametrize("gauge", [0, 1, 2])
def test_peierls_bit_exact(gpu, gauge):
    s = tb.make_graphene_sample(10)
    ref = oracle.set_mag_field_loop(s.hop_i, s.hop_j, s.hop_v, s.dr, s.orb_pos, 20.0, gauge)
    s.set_magnetic_field(20.0, gauge)
    np.testing.assert_array_equal(s.hop_v, ref)


def test_builder_rejects_bad_indices(gpu):
    s = tb.make_graphene_sample(4)
    s.hop_j = s.hop_j.copy()
    s.hop_j[3] = s.num_orb + 5
    from tbplas_amd._lib import TBGError
    with pytest.raises(TBGError):
        s.build_ham_dxy()
    with pytest.raises(TBGError):
        s.build_ham_csr()


def test_large_sample_properties(gpu):
    """At 1024x1024 (2.1M orbitals): sorted insertion-order rows equal the
    canonical rows, every row has 3 entries, values are the rescaled hop."""
    s = tb.make_graphene_sample(1024)
    s.rescale_ham(9.0)
    ip, ix, h, dx, dy = [t.cpu().numpy() for t in s.build_ham_dxy_device()]
    cp, cx, cd = [t.cpu().numpy() for t in s.build_ham_csr_device()]
    np.testing.assert_array_equal(ip, cp)
    assert np.all(np.diff(ip) == 3)
    rows = np.repeat(np.arange(s.num_orb), 3)
    order = np.lexsort((ix, rows))
    np.testing.assert_array_equal(ix[order], cx)
    np.testing.assert_array_equal(h[order], cd)
    assert np.all(cd == s.hop_v[0])
    # dx is antisymmetric: the pair (r, c) and (c, r) carry opposite signs
    assert abs(np.sum(dx)) < 1e-6 and abs(np.sum(dy)) < 1e-6


@pytest.mark.parametrize("at", [0, 1, 255, 256, -2, -1])
def test_fill_refuses_an_indptr_of_other_hops(gpu, at):
    """The comparison of the caller's indptr with the hops' own, at the edges
    of its blocks and ends; the unchanged one passes."""
    import ctypes
    import torch
    s = tb.make_graphene_sample(17, 31)
    s.init_orb_eng()
    L, h = tb._lib, tb._lib.default_handle(0)
    d = tb.sample._DevHops(s, 0, with_dr=True)
    n, m = s.num_orb, s.num_hop
    ip = torch.empty(n + 1, dtype=torch.int64, device="cuda:0")
    nnz = ctypes.c_int64(0)
    hops = [L.ptr(x) for x in (d.orb_eng, d.hop_i, d.hop_j)]
    for csr in (False, True):
        if csr:
            L.check(L.lib().tbg_ham_csr_count(h.ptr, n, m, *hops, L.ptr(d.hop_v), L.ptr(ip),
                                              ctypes.byref(nnz)))
        else:
            L.check(L.lib().tbg_ham_dxy_count(h.ptr, n, m, *hops, 1e-5, L.ptr(ip),
                                              ctypes.byref(nnz)))
        ix = torch.empty(nnz.value, dtype=torch.int64, device="cuda:0")
        v = torch.empty(nnz.value, dtype=torch.complex128, device="cuda:0")
        x, y = (torch.empty(nnz.value, dtype=torch.float64, device="cuda:0") for _ in range(2))

        def fill():
            if csr:
                return L.lib().tbg_ham_csr_fill(h.ptr, n, m, *hops, L.ptr(d.hop_v), L.ptr(ip),
                                                L.ptr(ix), L.ptr(v))
            return L.lib().tbg_ham_dxy_fill(h.ptr, n, m, *hops, L.ptr(d.hop_v), L.ptr(d.dr), 1e-5,
                                            L.ptr(ip), L.ptr(ix), L.ptr(v), L.ptr(x), L.ptr(y))
        assert fill() == 0
        ip[at] += 1
        torch.cuda.synchronize()
        with pytest.raises(L.TBGError, match="does not match the hop list"):
            L.check(fill())
