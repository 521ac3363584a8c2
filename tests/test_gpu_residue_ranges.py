"""Residue arithmetic on rows that span a wide range over the aux functions (run with -m gpu).

Pair energies, each judged by its own size against the matrix kernel of the same precision
(FERRIC_HIP_TILE selects either), whose error follows sum |B||B| of the pair itself. The rows of
an occupied orbital lie on the aux functions of its site and decay from there, so that a
pair's products are small beside the rows' largest elements.

Tolerance, FP64: products off by at most 2^-50 (root mean square over a, b), which the sum
over nvir^2 of them, with nvir independent roundings at least, takes to 2^-49 nvir^-1/2
= 1.4e-16 of the energy at 160 virtuals; four such deviations and the matrix kernel's own
2^-52: 1e-15. MIXED: 2^-24 instead of 2^-50 on either side, 2 x 4 x 2^-23 nvir^-1/2: 8e-8.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import Precision, _lib, rimp2  # noqa: E402
from ferric_amd import unrestricted as un  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402

NOCC, NVIR = 24, 160
BAR = {Precision.FP64: 1e-15, Precision.MIXED: 8e-8}


@pytest.fixture(autouse=True)
def residue_route(monkeypatch):
    monkeypatch.setenv("FERRIC_HIP_TILE", "256")  # whatever is faster at these sizes


@pytest.fixture
def timing():
    _lib.lib().fh_set_timing(1)
    yield
    _lib.lib().fh_set_timing(0)


def _chain(weight, per, naux=None, seed=1):
    """b of orbitals on a line, `per` aux functions a site, weight(|i - site|); zero rows up to
    naux."""
    rng = np.random.default_rng(seed)
    d = np.abs(np.arange(NOCC)[:, None] - np.arange(NOCC)[None, :])
    w = weight(d.astype(float))
    b = rng.standard_normal((NOCC, per, NOCC, NVIR)) * w[:, None, :, None] * np.sqrt(0.0081 / per)
    b = b.reshape(NOCC * per, NOCC * NVIR)
    if naux:
        b = np.concatenate([b, np.zeros((naux - len(b), NOCC * NVIR))])
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, NOCC)),
                          np.sort(rng.uniform(0.12, 5.0, NVIR))])
    return b, eps


def _against_matrix(b, eps, precision, monkeypatch):
    t = torch.from_numpy(b).cuda()
    pe = estimate_pair_energies_from_b_ov(t, eps, NOCC, NVIR, precision=precision)
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    pm = estimate_pair_energies_from_b_ov(t, eps, NOCC, NVIR, precision=precision)
    bar = BAR[precision] * np.abs(pm.e_os)
    assert np.all(np.abs(pe.e_os - pm.e_os) <= bar)
    assert np.all(np.abs(pe.e_ss - pm.e_ss) <= 2 * bar)
    return pe, pm


@pytest.mark.parametrize("naux", [1008, 4608])
def test_short_chain(naux, monkeypatch):
    """Orbitals that reach three sites: the products of pairs six sites apart are e^-6 of the
    nearest ones'."""
    print("residue ranges, reach", naux, flush=True)
    b, eps = _chain(lambda d: np.where(d <= 3, np.exp(-d), 0.0), 42, naux)
    _against_matrix(b, eps, Precision.FP64, monkeypatch)


def _tile():
    return _lib.last_timing()["tile"]


@pytest.mark.parametrize("precision", [Precision.FP64, Precision.MIXED])
@pytest.mark.parametrize("weight", ["e^-d", "e^-d/2", "(1+d)^-3", "halves 1e-3", "halves 1e-6",
                                    "halves 1e-9", "halves 1e-12"])
def test_rows_past_the_range_take_the_matrix_kernel(weight, precision, monkeypatch, timing):
    """Chains without an end, and even and odd orbitals on the two halves of the aux functions
    with tails on the other one: the matrix kernel's energies bit for bit where the route is
    its (and it has to be, for the steepest), its accuracy otherwise."""
    print("residue ranges", weight, precision, flush=True)
    f = {"e^-d": lambda d: np.exp(-d), "e^-d/2": lambda d: np.exp(-0.5 * d),
         "(1+d)^-3": lambda d: (1.0 + d) ** -3.0}.get(weight)
    if f:
        b, eps = _chain(f, 42)
    else:
        b, eps = _chain(lambda d: np.ones_like(d), 42)
        tail = np.where(np.arange(len(b))[:, None] * 2 // len(b) == np.arange(NOCC) % 2, 1.0,
                        float(weight.split()[1]))
        b *= np.repeat(tail, NVIR, axis=1)
    t = torch.from_numpy(b).cuda()
    estimate_pair_energies_from_b_ov(t, eps, NOCC, NVIR, precision=precision)
    matrix = _tile() == 64
    pe, pm = _against_matrix(b, eps, precision, monkeypatch)
    if weight in ("e^-d", "halves 1e-6", "halves 1e-9", "halves 1e-12"):
        assert matrix
    if matrix:
        assert np.array_equal(pe.e_os, pm.e_os) and np.array_equal(pe.e_ss, pm.e_ss)


@pytest.mark.parametrize("precision", [Precision.FP64, Precision.MIXED])
def test_ordinary_rows_stay(precision, timing):
    """Normal rows, hot aux functions, rows of different size, zero rows and a zero orbital, and
    a non-finite row, which is not judged."""
    for kind in ("normal", "hot", "sizes", "zeros", "nan"):
        b, eps = _chain(lambda d: np.ones_like(d), 42)
        rng = np.random.default_rng(8)
        if kind == "hot":
            b[::37] *= 20.0
        if kind == "sizes":
            b *= 2.0 ** rng.integers(-20, 21, NOCC * NVIR)
        if kind == "zeros":
            b[:, rng.integers(0, NOCC * NVIR, 300)] = 0.0
            b[:, 5 * NVIR:6 * NVIR] = 0.0
        if kind == "nan":
            b[5, 7] = np.nan
        print("residue ranges, ordinary", kind, precision, flush=True)
        estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, NOCC, NVIR,
                                         precision=precision)
        assert _tile() == 256


@pytest.mark.parametrize("tail", [1e-6, 1e-12])
def test_other_entries(tail, monkeypatch, timing):
    """The opposite-spin block of two channels on the two halves, and a density and an energy
    whose orbitals lie on either: the matrix kernels' results bit for bit."""
    print("residue ranges, entries", tail, flush=True)
    b, eps = _chain(lambda d: np.ones_like(d), 60)
    half = np.where(np.arange(len(b)) * 2 // len(b) == 0, 1.0, tail)[:, None]
    a, c = un.SpinChannel(b * half, eps, NOCC, NVIR), un.SpinChannel(b * half[::-1], eps, NOCC,
                                                                   NVIR)
    mixed = torch.from_numpy(np.concatenate([(b * half)[:, :12 * NVIR],
                                             (b * half[::-1])[:, 12 * NVIR:]], axis=1)).cuda()

    def results():
        out = [un.u_opposite_spin(a, c)]
        tiles = [_tile()]
        sc, oo, vv = rimp2.mp2_density(mixed, eps, NOCC, NVIR)
        tiles.append(_tile())
        return out + [sc.e_os, sc.e_ss, np.asarray(oo), np.asarray(vv)], tiles

    got, tiles = results()
    assert tiles == [64, 64]
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    want, _ = results()
    assert all(np.array_equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("weight", [lambda d: np.exp(-d), lambda d: np.ones_like(d)],
                         ids=["wide", "ordinary"])
def test_mixed_out_of_range_is_refused_on_either_route(weight):
    """max|B| past sqrt(FLT_MAX / 64) = 2.3e18."""
    print("residue ranges, refused", flush=True)
    b, eps = _chain(weight, 42)
    with pytest.raises(_lib.RangeError):
        estimate_pair_energies_from_b_ov(torch.from_numpy(b * 1e21).cuda(), eps, NOCC, NVIR,
                                         precision=Precision.MIXED)


@pytest.mark.parametrize("scale", [1e-120, 1e-30, 1e30, 1e120])
def test_scaled_rows(scale, monkeypatch, timing):
    """A scale of B by itself moves no digits; where the squares leave the range of the test, or
    come near its ends, the matrix kernel's bits (at 1e120 the energies themselves overflow)."""
    print("residue ranges, scale", scale, flush=True)
    b, eps = _chain(lambda d: np.ones_like(d), 42)
    t = torch.from_numpy(b * scale).cuda()
    pe = estimate_pair_energies_from_b_ov(t, eps, NOCC, NVIR)
    if 1e-60 < scale < 1e60:
        assert _tile() == 256
        _against_matrix(b * scale, eps, Precision.FP64, monkeypatch)
        return
    assert _tile() == 64
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    pm = estimate_pair_energies_from_b_ov(t, eps, NOCC, NVIR)
    assert np.array_equal(pe.e_os, pm.e_os, equal_nan=True)
    assert np.array_equal(pe.e_ss, pm.e_ss, equal_nan=True)
