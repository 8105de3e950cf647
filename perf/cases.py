"""The work this framework is measured on.

Every case is one call that a TBPM user makes on honeycomb samples, through
the package's public entry points: a DOS run, a batch of DOS runs, a
propagated wave function, an AC or DC conductivity run, the Kubo-Bastin
moments, and the assembly of the Hamiltonian.  The Hamiltonian is prepared as
``Solver`` prepares it (assembled on the GPU, rows in square tiles of the
library's rule, the library's untuned launch shape), so a pass is the
propagation itself: the initial states go in as host arrays, the correlations
come back as host arrays.

``prepare`` builds the sample arrays, the Hamiltonian and the random-phase
states; ``run`` makes the call; ``exact`` states the same result in 64 bits
with plain torch (exact k-space propagation for pristine periodic samples,
gather-and-add Chebyshev series otherwise).
"""
import math

import numpy as np
import torch

import tbplas_amd as tb
from tbplas_amd import tbpm, tune

RESCALE = 9.0            # eV; |E| <= 3 * 2.7 + W / 2
HOP = -2.7               # eV
A0 = 0.246               # nm
KT = 8.617333262e-5 * 300.0
FERMI_FFT = 2 ** 15


# -- the cases -------------------------------------------------------------
def _case(kind, prec, l1, l2, states, steps, name=None, vac=0.0, anderson=0.0, field=0.0,
          energies=0, instances=0, frames=0):
    c = {"kind": kind, "prec": prec, "l1": l1, "l2": l2, "states": states, "steps": steps,
         "vac": vac, "anderson": anderson, "field": field, "energies": energies,
         "instances": instances, "frames": frames}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest sample anyone tries first: launches and host calls only
        _case("dos", "fp64", 31, 33, 1, 512, "dos_tiny_f64"),
        # 131,072 orbitals, one state at full precision: latency per step
        _case("dos", "fp64", 256, 256, 1, 1024, "dos_latency_f64"),
        # the default precision and state count on a large sample
        _case("dos", "fp64", 1448, 1448, 1, 256, "dos_one_f64"),
        # eight samples of a random average at full precision, an odd size
        # with on-site disorder (four entries a row)
        _case("dos", "fp64", 701, 643, 8, 128, "dos_k8_f64", vac=0.01, anderson=0.8),
        # the headline: 8,388,608 orbitals, eight complex64 states
        _case("dos", "fp32", 2048, 2048, 8, 128, "dos_large_f32"),
        # disorder ensembles: instances of uneven size in one run
        _case("batch", "fp32", 128, 512, 4, 128, "batch_f32", anderson=1.0, vac=0.01,
              instances=12),
        # a wave packet followed in time, frames kept
        _case("psi_t", "fp64", 384, 517, 1, 192, "psi_t_f64", anderson=0.5, frames=6),
        # optical conductivity, complex64, four samples a run
        _case("ac", "fp32", 512, 512, 4, 256, "ac_f32"),
        # optical conductivity at full precision: a ragged sample with
        # vacancies in a magnetic field (complex hoppings), three samples
        _case("ac", "fp64", 389, 211, 3, 128, "ac_f64", vac=0.01, field=20.0),
        # DC conductivity of a disordered sample in a field; the energies
        # are those of a window of +-0.5 eV at this number of steps
        _case("dc", "fp32", 512, 500, 8, 256, "dc_f32", vac=0.01, anderson=1.0, field=20.0,
              energies=28),
        # Hall moments of the reference's example: 200,000 orbitals, B = 100 T
        _case("hall", "fp64", 500, 200, 1, 2048, "hall_f64", field=100.0),
        # assembly of both forms of the Hamiltonian from host arrays
        _case("assembly", "fp64", 1024, 1021, 0, 0, "assembly", anderson=0.3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["dos", "dos", "dos", "batch", "psi_t", "ac", "dc", "hall", "assembly"])
    prec = rng.choice(["fp64", "fp32"])
    vac = rng.choice([0.0, 0.01])
    anderson = rng.choice([0.0, round(rng.uniform(0.1, 1.0), 2)])
    field = rng.choice([0.0, 0.0, round(rng.uniform(5.0, 100.0), 1)])

    def lattice(lo, hi):
        l1 = _log(rng, lo, hi)
        return l1, max(lo, min(hi, int(l1 * rng.uniform(0.6, 1.6))))

    def steps(lo, hi, n, vectors, most):
        """Steps within the cost of the largest case (orbital-vector-steps)."""
        return max(8, min(_log(rng, lo, hi), int(most / (n * vectors))))

    if kind == "dos":
        states = rng.choice([1, 1, 2, 3, 4, 5, 8, 8, 16])
        l1, l2 = lattice(24, 1400)
        t = steps(64, 1024, 2 * l1 * l2, states, 1.5e9)
        return _case(kind, prec, l1, l2, states, t, vac=vac, anderson=anderson, field=field)
    if kind == "batch":
        lo, hi = sorted((_log(rng, 32, 400), _log(rng, 64, 500)))
        inst = rng.randint(2, 12)
        states = rng.choice([1, 2, 4, 8])
        t = steps(64, 512, inst * 2 * lo * hi, states, 1e9)
        return _case(kind, prec, lo, hi + 1, states, t, vac=vac, anderson=anderson,
                     field=0.0, instances=inst)
    if kind == "psi_t":
        l1, l2 = lattice(32, 900)
        t = steps(32, 512, 2 * l1 * l2, 1, 2e8)
        return _case(kind, prec, l1, l2, 1, t, vac=vac, anderson=anderson, field=field,
                     frames=rng.randint(1, 8))
    if kind == "ac":
        l1, l2 = lattice(32, 600)
        states = rng.choice([1, 2, 3, 4])
        t = steps(32, 512, 2 * l1 * l2, 3 * states, 6e8)
        return _case(kind, prec, l1, l2, states, t, vac=vac, anderson=anderson, field=field)
    if kind == "dc":
        l1, l2 = lattice(32, 500)
        states = rng.choice([1, 2, 4, 8])
        t = steps(32, 512, 2 * l1 * l2, 4 * states, 1e9)
        return _case(kind, prec, l1, l2, states, t, vac=vac, anderson=anderson, field=field,
                     energies=rng.choice([1, 5, rng.randint(2, 40), max(1, t // 9)]))
    if kind == "hall":
        l1, l2 = lattice(40, 320)
        return _case(kind, "fp64", l1, l2, rng.choice([1, 1, 2]),
                     min(_log(rng, 100, 1500), int(2.5e8 / (2 * l1 * l2))),
                     vac=vac, anderson=anderson, field=field)
    l1, l2 = lattice(64, 1100)
    return _case(kind, "fp64", l1, l2, 0, 0, anderson=anderson, field=field)


# -- inputs ----------------------------------------------------------------
def _lattice(case, seed, l1=None, l2=None):
    """Arrays of a periodic honeycomb sample in eV: orbital (ia, ib, io), per
    cell the A-B bond and the two B-A bonds to the next cells; vacancies
    removed, on-site energies in U[-W/2, W/2], Peierls phases in the Landau
    gauge."""
    l1, l2 = l1 or case["l1"], l2 or case["l2"]
    rng = np.random.default_rng(seed)
    ia, ib = (x.reshape(-1) for x in np.indices((l1, l2)))
    cell = ia * l2 + ib
    a1, a2 = A0 * np.array([1.0, 0.0]), A0 * np.array([0.5, math.sqrt(0.75)])
    tau = (a1 + a2) / 3.0
    n = 2 * l1 * l2
    pos = np.zeros((n, 3))
    pos[0::2, :2] = ia[:, None] * a1 + ib[:, None] * a2
    pos[1::2, :2] = pos[0::2, :2] + tau
    hop_i, hop_j, dr = np.empty((l1 * l2, 3), np.int64), np.empty((l1 * l2, 3), np.int64), \
        np.zeros((l1 * l2, 3, 3))
    hop_i[:, 0], hop_j[:, 0], dr[:, 0, :2] = 2 * cell, 2 * cell + 1, tau
    hop_i[:, 1], hop_j[:, 1] = 2 * cell + 1, 2 * ((ia + 1) % l1 * l2 + ib)
    hop_i[:, 2], hop_j[:, 2] = 2 * cell + 1, 2 * (ia * l2 + (ib + 1) % l2)
    dr[:, 1, :2], dr[:, 2, :2] = a1 - tau, a2 - tau
    hop_i, hop_j, dr = hop_i.reshape(-1), hop_j.reshape(-1), dr.reshape(-1, 3)
    hop_v = np.full(len(hop_i), HOP, dtype=np.complex128)
    if case["field"]:
        # e B / hbar in 1/nm^2 for B in tesla
        y = pos[hop_i, 1] + 0.5 * dr[:, 1]
        hop_v *= np.exp(1j * (1.519267447e-3 * case["field"]) * dr[:, 0] * y)
    eng = np.zeros(n)
    if case["anderson"]:
        eng = rng.uniform(-0.5 * case["anderson"], 0.5 * case["anderson"], n)
        eng[np.abs(eng) < 1e-3] = 1e-3      # every orbital keeps its diagonal entry
    if case["vac"]:
        keep = np.ones(n, bool)
        keep[rng.choice(n, max(1, int(case["vac"] * n)), replace=False)] = False
        new = np.cumsum(keep) - 1
        bond = keep[hop_i] & keep[hop_j]
        eng, pos = eng[keep], pos[keep]
        hop_i, hop_j, hop_v, dr = new[hop_i[bond]], new[hop_j[bond]], hop_v[bond], dr[bond]
    return eng, pos, hop_i, hop_j, hop_v, dr


def _sizes(case):
    """Edges of a batch's instances, spread from l1 to l2."""
    k = case["instances"]
    return [int(round(case["l1"] * (case["l2"] / case["l1"]) ** (i / max(1, k - 1))))
            for i in range(k)]


def _phases(n, states, seed):
    """(states, n) complex128 random-phase states of unit norm, on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    phi = torch.rand((states, n), generator=g, device="cuda", dtype=torch.float64)
    return torch.polar(torch.full_like(phi, 1.0 / math.sqrt(n)), 2.0 * math.pi * phi)


def _packet(pos, eng_seed):
    """A Gaussian wave packet in the middle of the sample, with a momentum."""
    rng = np.random.default_rng(eng_seed)
    xy = pos[:, :2]
    mid = 0.5 * (xy.min(axis=0) + xy.max(axis=0))
    w = 0.12 * (xy.max(axis=0) - xy.min(axis=0)).min()
    k = rng.uniform(-4.0, 4.0, 2)
    z = np.exp(-((xy - mid) ** 2).sum(axis=1) / (2 * w * w) + 1j * (xy @ k))
    return z / np.linalg.norm(z)


def _bessel(tau):
    """exp(-i x tau) as a Chebyshev series: J_m(tau) down to 1e-15, by the
    trapezoid rule on Bessel's integral."""
    th = (np.arange(256) + 0.5) * (math.pi / 256)
    j = [float(np.mean(np.cos(m * th - tau * np.sin(th)))) for m in range(40)]
    return np.array(j[:next(m for m in range(4, 40) if abs(j[m]) <= 1e-15)])


def _fermi(one_minus):
    """Jackson-damped Chebyshev coefficients of the (one-minus) Fermi
    function at 300 K, mu = 0, to 1e-12."""
    x = np.cos(2.0 * math.pi * np.arange(FERMI_FFT) / FERMI_FFT)
    f = 1.0 / (1.0 + np.exp(np.clip(x * (RESCALE / KT), -700, 700)))
    f = 1.0 - f if one_minus else f
    n = FERMI_FFT // 2
    k = np.arange(n)
    q = math.pi / n
    g = ((n - k) * np.cos(q * k) + np.sin(q * k) / math.tan(q)) / n
    g[0] = 0.5
    c = g * np.fft.fft(f).real[:n] / n
    return c[:int(np.nonzero(np.abs(c) > 1e-12)[0][-1]) + 1]


def _tau(case):
    """Time step times the rescaling factor (AC: half a step)."""
    return 0.5 * math.pi if case["kind"] == "ac" else math.pi


def _energies(case):
    """The energy grid of a DC run and the indices nearest to zero."""
    t = case["steps"]
    en = np.array([RESCALE * i / t - RESCALE for i in range(2 * t)])
    k = min(case["energies"], 2 * t)
    first = max(0, min(2 * t - k, t - k // 2))
    return en, np.arange(first, first + k, dtype=np.int64)


def _frames(case):
    return np.unique(np.linspace(0, case["steps"], case["frames"] + 1).round().astype(np.int64))


# -- what a program holds before the call -----------------------------------
def _hamiltonian(case, arrays, vectors, current=False, tiled=True):
    eng, pos, hop_i, hop_j, hop_v, dr = arrays
    s = tb.Sample(eng.copy(), pos, hop_i, hop_j, hop_v.copy(), dr)
    s.rescale_ham(RESCALE)
    if current:
        ip, ix, hv, dx, dy = s.build_ham_dxy_device()
    else:
        (ip, ix, hv), dx, dy = s.build_ham_csr_device(), None, None
    order = tiles = None
    if tiled:
        rule = tb.ac_tile_nm if case["kind"] == "ac" else tb.auto_tile_nm
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        edge = rule(vectors, case["prec"], n_orb=s.num_orb, cus=cus)
        order, tiles = s.tile_order(edge, return_tiles=True)
    return tbpm.Hamiltonian(s.num_orb, ip, ix, hv, dx, dy, cur_scale=s.rescale,
                            precision=case["prec"], order=order, tiles=tiles)


def _vectors(case):
    return {"ac": 3, "dc": 2}.get(case["kind"], 1) * case["states"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "assembly":
        return {"case": case, "sample": tb.Sample(*_lattice(case, seed))}
    st = {"case": case, "bes": _bessel(_tau(case))}
    if kind == "batch":
        hs, ps = [], []
        for i, l in enumerate(_sizes(case)):
            hs.append(_hamiltonian(case, _lattice(case, seed * 64 + i, l, l), _vectors(case)))
            ps.append(_phases(hs[-1].n, case["states"], seed * 64 + i).cpu().numpy())
        st.update(hams=hs, psi=ps)
        st["shape"] = hs
    else:
        arrays = _lattice(case, seed)
        st["H"] = _hamiltonian(case, arrays, _vectors(case), current=kind in ("ac", "dc", "hall"),
                               tiled=kind not in ("psi_t", "hall"))
        st["shape"] = st["H"]
        if kind == "psi_t":
            st["psi"] = _packet(arrays[1], seed)
        else:
            st["psi"] = _phases(len(arrays[0]), case["states"], seed).cpu().numpy()
    if kind == "ac":
        st["fermi"] = (_fermi(False), _fermi(True))
    return st


def run(st):
    case = st["case"]
    kind, t = case["kind"], case["steps"]
    thr = 1e-4 if case["prec"] == "fp32" else 1e-9
    if kind == "assembly":
        s = st["sample"]
        return list(s.build_ham_csr_device()) + list(s.build_ham_dxy_device())
    if kind not in ("psi_t", "hall"):
        # the launch shape a program sets for its run, as Solver does
        # (gpu['autotune'] off)
        tune.apply(st["shape"], _vectors(case), st["bes"], False)
    if kind == "dos":
        return tbpm.corr_dos(st["H"], st["bes"], st["psi"], t, chk_thr=thr)
    if kind == "batch":
        return tbpm.corr_dos_batch(st["hams"], st["bes"], st["psi"], t, chk_thr=thr)
    if kind == "psi_t":
        return tbpm.psi_t(st["H"], st["bes"], st["psi"], _frames(case), t, chk_thr=thr)
    if kind == "ac":
        return tbpm.corr_ac(st["H"], st["bes"], *st["fermi"], st["psi"], t, chk_thr=thr)
    if kind == "dc":
        en, inds = _energies(case)
        return tbpm.corr_dc(st["H"], st["bes"], st["psi"], t, math.pi / RESCALE, en, inds,
                            chk_thr=thr)
    return tbpm.hall_mu(st["H"], st["psi"], t, 1)


# -- what a pass cannot do without --------------------------------------------
def work(case):
    """Inputs and outputs once; the arithmetic of every series term (a
    product with each entry of a row, the recurrence, the sum)."""
    kind, t, k = case["kind"], case["steps"], case["states"]
    n = 2 * case["l1"] * case["l2"]
    if kind == "batch":
        n = sum(2 * l * l for l in _sizes(case))
    entries = (3 + (1 if case["anderson"] else 0)) * n
    real = not case["field"]
    size = 8 if case["prec"] == "fp32" else 16
    if kind == "assembly":
        # hop arrays and on-site energies read, two CSR forms written
        return {"bytes": n * 8 + 1.5 * n * (16 + 16 + 24) + 2 * 8 * (n + 1) + entries * (24 + 40),
                "flops": 0}
    matrix = entries * (4 + (size // 2 if real else size))
    per_term = k * (entries * (4 if real else 8) + 10 * n)
    terms = len(_bessel(_tau(case))) - 1
    states = 16 * n * k
    if kind in ("dos", "batch"):
        return {"bytes": matrix + states + 16 * k * (t + 1) * max(1, case["instances"]),
                "flops": t * (terms * per_term + 12 * n * k)}
    if kind == "psi_t":
        return {"bytes": matrix + states + 16 * n * len(_frames(case)),
                "flops": t * terms * per_term}
    if kind == "ac":
        fermi = len(_fermi(False)) - 1
        return {"bytes": matrix + entries * 2 * size + states + 64 * k * t,
                "flops": 3 * (fermi + (t - 1) * terms) * per_term +
                (t - 1) * k * (32 * entries + 32 * n)}
    if kind == "dc":
        e = min(case["energies"], 2 * t)
        return {"bytes": matrix + entries * 2 * size + states + 16 * k * t * (1 + 2 * e),
                "flops": 4 * t * terms * per_term + t * k * n * (e * 32 + 8)}
    # Hall: two recurrences, one current per vector, one N x N product
    return {"bytes": matrix + entries * 2 * size + states + 16 * k * t * t,
            "flops": k * t * (2 * entries * 8 + entries * 8 + 8 * n) + 8.0 * k * t * t * n}


# -- the same results in 64 bits ----------------------------------------------
class _Matrix:
    """H / RESCALE and the currents as padded rows on the GPU."""

    def __init__(self, arrays, current=False):
        eng, _, hop_i, hop_j, hop_v, dr = arrays
        n = len(eng)
        row = np.concatenate([np.arange(n), hop_i, hop_j])
        col = np.concatenate([np.arange(n), hop_j, hop_i])
        val = np.concatenate([eng.astype(np.complex128), hop_v, hop_v.conj()]) / RESCALE
        o = np.argsort(row, kind="stable")
        row, col, val = row[o], col[o], val[o]
        first = np.searchsorted(row, np.arange(n))
        slot = np.arange(len(row)) - first[row]
        self.w = int(slot.max()) + 1
        cols = np.repeat(np.arange(n)[:, None], self.w, axis=1)
        vals = np.zeros((n, self.w), np.complex128)
        cols[row, slot], vals[row, slot] = col, val
        self.cols = torch.from_numpy(np.ascontiguousarray(cols.T)).cuda()
        self.vals = self._dev(vals if np.any(vals.imag) else vals.real)
        if current:
            d = np.concatenate([np.zeros((n, 3)), dr, -dr])[o]
            self.j = []
            for x in range(2):
                z = np.zeros((n, self.w), np.complex128)
                z[row, slot] = 1j * RESCALE * val * d[:, x]
                self.j.append(self._dev(z))

    @staticmethod
    def _dev(v):
        return torch.from_numpy(np.ascontiguousarray(v.T)).cuda()[:, :, None]

    def mul(self, x, vals=None):
        """x (n, K)"""
        vals = self.vals if vals is None else vals
        y = vals[0] * x[self.cols[0]]
        for j in range(1, self.w):
            y += vals[j] * x[self.cols[j]]
        return y

    def series(self, x, coef, a1, a, b):
        """sum_m c_m v_m, v_1 = a1 H v_0, v_m = a H v_{m-1} + b v_{m-2};
        coef (terms,) or (terms, K)"""
        u, v = x, a1 * self.mul(x)
        out = coef[0] * u + coef[1] * v
        for c in coef[2:]:
            u, v = v, a * self.mul(v) + b * u
            out += c * v
        return out

    def step(self, x, bes, sign=1.0):
        """exp(-i H tau sign) x"""
        c = [bes[0]] + [2.0 * j for j in bes[1:]]
        return self.series(x, c, -1j * sign, -2j * sign, 1.0)


def _dot(a, b):
    return (a.conj() * b).sum(dim=0)


def _kspace(case, psi):
    """C(t) of a pristine periodic sample from its Bloch bands."""
    l1, l2, t = case["l1"], case["l2"], case["steps"]
    k1 = torch.arange(l1, device="cuda", dtype=torch.float64)[:, None] * (2 * math.pi / l1)
    k2 = torch.arange(l2, device="cuda", dtype=torch.float64)[None, :] * (2 * math.pi / l2)
    one = torch.ones((), device="cuda", dtype=torch.float64)
    f = (HOP / RESCALE) * (1.0 + torch.polar(one, -k1) + torch.polar(one, -k2))
    e = f.abs()
    ph = torch.where(e > 1e-14, f / e.clamp_min(1e-300), torch.ones_like(f)).reshape(-1)
    e = e.reshape(-1)
    cell = psi.reshape(-1, l1, l2, 2)
    ws = []
    for s in range(len(psi)):
        u = torch.fft.fft2(cell[s, :, :, 0], norm="ortho").reshape(-1)
        v = torch.fft.fft2(cell[s, :, :, 1], norm="ortho").reshape(-1) * ph
        p, m = (0.5 * (u + v).abs() ** 2), (0.5 * (u - v).abs() ** 2)
        ws.append((p + m, p - m))
    even, odd = (torch.stack([w[q] for w in ws]) for q in range(2))
    times = torch.arange(t + 1, device="cuda", dtype=torch.float64) * math.pi
    out = torch.zeros((len(psi), t + 1), device="cuda", dtype=torch.complex128)
    for a in range(0, len(e), 1 << 19):
        arg = e[a:a + (1 << 19), None] * times
        out += torch.complex(even[:, a:a + (1 << 19)] @ torch.cos(arg),
                             -(odd[:, a:a + (1 << 19)] @ torch.sin(arg)))
    return out


def _dos(m, psi, bes, t):
    x0 = psi.T.contiguous()
    out, x = [_dot(x0, x0)], x0
    for _ in range(t):
        x = m.step(x, bes)
        out.append(_dot(x0, x))
    return torch.stack(out, dim=1)


def _ac(case, arrays, psi, bes):
    m, k = _Matrix(arrays, True), case["states"]
    x0 = psi.T.contiguous()
    x = torch.cat([m.mul(x0, m.j[0]), m.mul(x0, m.j[1]), x0], dim=1)
    f, g = _fermi(False), _fermi(True)
    coef = np.zeros((max(len(f), len(g)), 3 * k))
    coef[:len(g), :2 * k], coef[:len(f), 2 * k:] = g[:, None], f[:, None]
    x = m.series(x, torch.from_numpy(coef).cuda(), 1.0, 2.0, -1.0)
    out = torch.zeros((k, 4, case["steps"]), device="cuda", dtype=torch.complex128)
    for t in range(1, case["steps"]):
        x = m.step(x, bes)
        u, p = x[:, :2 * k].contiguous(), x[:, 2 * k:]
        wx, wy = m.mul(u, m.j[0]), m.mul(u, m.j[1])
        for q, w in enumerate((wx[:, :k], wy[:, :k], wx[:, k:], wy[:, k:])):
            out[:, q, t] = _dot(p, w)
    return out


def _dc(case, arrays, psi, bes):
    m, k, t = _Matrix(arrays, True), case["states"], case["steps"]
    en, inds = _energies(case)
    e = torch.from_numpy(en[inds]).cuda()
    x0 = psi.T.contiguous()
    dos = torch.zeros((k, t), device="cuda", dtype=torch.complex128)
    qe = [x0.clone() for _ in inds]
    p, q = x0, x0
    for s in range(1, t + 1):
        p, q = m.step(p, bes), m.step(q, bes, -1.0)
        dos[:, s - 1] = _dot(x0, p)
        w = 0.5 * (1.0 + math.cos(math.pi * s / t))
        ph = torch.polar(torch.ones_like(e), e * (s * math.pi / RESCALE))
        for i in range(len(qe)):
            qe[i] += (w * ph[i]) * p + (w * ph[i].conj()) * q
    out = torch.zeros((k, 2, len(inds), t), device="cuda", dtype=torch.complex128)
    for i in range(len(qe)):
        qe[i] = qe[i] / torch.sqrt(_dot(qe[i], qe[i]).real)
        qe[i] = qe[i] / _dot(x0, qe[i]).abs()
    for a in range(2):
        y = [m.mul(v, m.j[a]) for v in qe]
        x = m.mul(x0, m.j[a])
        for s in range(t):
            if s:
                x = m.step(x, bes)
            for i in range(len(y)):
                out[:, a, i, s] = _dot(x, y[i])
    return dos, out


def _hall(case, arrays, psi):
    m, n_k = _Matrix(arrays, True), case["steps"]
    i = torch.arange(n_k, device="cuda", dtype=torch.float64)
    q = math.pi / n_k
    g = ((n_k - i) * torch.cos(q * i) + torch.sin(q * i) / math.tan(q)) / n_k
    g[0] = 0.5
    res = []
    for s in range(len(psi)):
        def rows(x, after=None):
            u = torch.empty((n_k, len(x)), device="cuda", dtype=torch.complex128)
            a, b = x, m.mul(x)
            for r in range(n_k):
                u[r] = (a if after is None else m.mul(a, after))[:, 0]
                a, b = b, 2.0 * m.mul(b) - a
            return u
        x0 = psi[s][:, None].contiguous()
        p, w = rows(m.mul(x0, m.j[0])), rows(x0, m.j[0])
        res.append(g[:, None] * (p.conj() @ w.T) * g)
    return torch.stack(res)


def _assembly(arrays):
    eng, _, hop_i, hop_j, hop_v, dr = arrays
    n, m = len(eng), len(hop_i)

    def csr(diag, sort_cols):
        d = np.nonzero(diag)[0]
        row = np.concatenate([d, hop_i, hop_j])
        col = np.concatenate([d, hop_j, hop_i])
        val = np.concatenate([eng[d].astype(np.complex128), hop_v, hop_v.conj()])
        dxy = np.concatenate([np.zeros((len(d), 3)), dr, -dr])
        key = col if sort_cols else np.concatenate([np.full(len(d), -1), 2 * np.arange(m),
                                                    2 * np.arange(m) + 1])
        o = np.lexsort((key, row))
        ptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int64)
        return ptr, col[o], val[o], dxy[o]

    ip, ix, hv, _ = csr(eng != 0, True)
    jp, jx, jv, d = csr(np.abs(eng) >= 1e-5, False)
    return [ip, ix, hv, jp, jx, jv, np.ascontiguousarray(d[:, 0]), np.ascontiguousarray(d[:, 1])]


def exact(case, seed):
    kind = case["kind"]
    if kind == "assembly":
        return _assembly(_lattice(case, seed))
    if kind == "batch":
        bes = _bessel(math.pi)
        out = []
        for i, l in enumerate(_sizes(case)):
            arrays = _lattice(case, seed * 64 + i, l, l)
            psi = _phases(len(arrays[0]), case["states"], seed * 64 + i)
            out.append(_dos(_Matrix(arrays), psi, bes, case["steps"]).cpu().numpy())
        return out
    n, terms = 2 * case["l1"] * case["l2"], case["steps"] * 20
    pristine = not (case["vac"] or case["anderson"] or case["field"])
    if kind == "dos" and pristine:
        return _kspace(case, _phases(n, case["states"], seed)).cpu().numpy()
    if n * _vectors(case) * terms * (2 if kind == "dc" else 1) > 1.2e11:
        return None          # over 20 seconds as plain gathers
    arrays = _lattice(case, seed)
    if kind == "psi_t":
        m, bes, frames = _Matrix(arrays), _bessel(math.pi), _frames(case)
        x, out = torch.from_numpy(_packet(arrays[1], seed))[:, None].cuda(), []
        for t in range(case["steps"] + 1):
            if t:
                x = m.step(x, bes)
            if t in frames:
                out.append(x[:, 0].cpu())
        return torch.stack(out).numpy()
    psi = _phases(len(arrays[0]), case["states"], seed)
    if kind == "hall":
        return _hall(case, arrays, psi).cpu().numpy()
    bes = _bessel(_tau(case))
    if kind == "dos":
        return _dos(_Matrix(arrays), psi, bes, case["steps"]).cpu().numpy()
    if kind == "ac":
        return _ac(case, arrays, psi, bes).cpu().numpy()
    return tuple(x.cpu().numpy() for x in _dc(case, arrays, psi, bes))
