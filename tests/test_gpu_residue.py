"""The residue-arithmetic pair kernels (run with -m gpu).

Shapes at the edges of the tiling: two orbitals to a tile with an odd one left
over, a tile exactly full, one block past it (two tiles), three tiles, one Q
panel, one row in the last panel, the largest aux count, more workgroups than
items. The pair energies are held to the oracle and to the matrix kernel of the
same precision (FERRIC_HIP_TILE selects it). Tolerance: each g is off by at most
its rounding to FP64 plus 2^-(beta + 1) of the two rows' ranges per term, below
the matrix kernel's own naux 2^-53 sum |B||B|; 1e-12 of the largest pair is the
bar of the other FP64 pair-energy tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import Precision, _lib, rimp2, synthetic  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402

SHAPES = [
    (60, 65, 700, 0),    # two orbitals a tile, 5 blocks each
    (41, 128, 400, 0),   # two orbitals fill a tile, the last group alone
    (14, 145, 1200, 2),  # one orbital a tile, frozen core
    (13, 256, 430, 0),   # a full tile
    (18, 257, 1500, 0),  # two tiles, 9 and 8 blocks
    (9, 300, 4608, 0),   # the largest aux count, several workgroups to an item
    (43, 513, 65, 0),    # three tiles, one row in the second panel
    (46, 200, 60, 1),    # one panel
]


def _problem(nocc, nvir, naux, seed=77, spread=True):
    rng = np.random.default_rng(seed + nocc * 1000 + nvir)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    if spread:  # rows of very different size, within a row and from row to row
        b[::37] *= 20.0
        b[5::11] *= 1e-6
        b *= 2.0 ** rng.integers(-3, 4, nocc * nvir)
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    return b, eps


def _args(b, eps, nocc, frozen):
    return np.concatenate([np.full(frozen, -11.2), eps]), frozen, frozen + nocc


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_fp64_pairs_at_the_edges(shape, oracle_mod, monkeypatch):
    nocc, nvir, naux, frozen = shape
    print("residue pairs", shape, flush=True)
    b, eps = _problem(nocc, nvir, naux)
    e, fo, nt = _args(b, eps, nocc, frozen)
    t = torch.from_numpy(b).cuda()
    pe = estimate_pair_energies_from_b_ov(t, e, nocc, nvir, fo, nt)
    w_os, w_ss = oracle_mod.pair_energies(b, eps, nocc, nvir)
    top = np.max(np.abs(w_os))
    assert np.max(np.abs(pe.e_os - w_os)) <= 1e-12 * top
    assert np.max(np.abs(pe.e_ss - w_ss)) <= 1e-12 * top
    assert np.array_equal(pe.e_os, pe.e_os.T)
    again = estimate_pair_energies_from_b_ov(t, e, nocc, nvir, fo, nt)
    assert np.array_equal(pe.e_os, again.e_os) and np.array_equal(pe.e_ss, again.e_ss)
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    pm = estimate_pair_energies_from_b_ov(t, e, nocc, nvir, fo, nt)
    assert np.max(np.abs(pe.e_os - pm.e_os)) <= 1e-12 * top
    assert np.max(np.abs(pe.e_ss - pm.e_ss)) <= 1e-12 * top


@pytest.mark.parametrize("shape", [(41, 65, 900), (24, 160, 800), (13, 257, 700)],
                         ids=lambda s: "-".join(map(str, s)))
def test_mixed_pairs_against_the_rounded_operand(shape, oracle_mod):
    """MIXED in ten moduli: the FP64 pair energies of the FP32-rounded B. Y keeps at
    least 32 bits below a row's largest value (4.5 sigma here), so g is off by at
    most 2 naux 2^-33 (4.5 sigma)^2 = 2^-27.7 of the diagonal g and, against the typical
    off-diagonal |g| (naux^1/2 times smaller), by 2^-27.7 naux^1/2 < 1.4e-7; twice that in
    the energy."""
    nocc, nvir, naux = shape
    print("residue mixed pairs", shape, flush=True)
    b, eps = _problem(nocc, nvir, naux, spread=False)
    pe = estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, nocc, nvir,
                                          precision=Precision.MIXED)
    br = b.astype(np.float32).astype(np.float64)
    w_os, w_ss = oracle_mod.pair_energies(br, eps, nocc, nvir)
    top = np.max(np.abs(w_os))
    assert np.max(np.abs(pe.e_os - w_os)) <= 2.8e-7 * top
    assert np.max(np.abs(pe.e_ss - w_ss)) <= 2.8e-7 * top


def test_fp64_energy_kappa_rows_and_storage(oracle_mod):
    """The energy entry (a workspace past the fixed array of the no-allocation
    entry): row partials, kappa, FP32 storage, frozen core."""
    nocc, nvir, naux, frozen = 20, 230, 3800, 1
    print("residue energy", nocc, nvir, naux, flush=True)
    b, eps = _problem(nocc, nvir, naux, spread=False)
    b = b.astype(np.float32).astype(np.float64)
    e, fo, nt = _args(b, eps, nocc, frozen)
    t = torch.from_numpy(b).cuda()
    sc, rows = rimp2.spin_components(t, e, nocc, nvir, fo, nt, row_partials=True)
    want = oracle_mod.spin_components_blas(b, eps, nocc, nvir, nthreads=16)
    bos, bss = oracle_mod.energy_bound(b, eps, nocc, nvir, 0, nocc)
    assert abs(sc.e_os - want[0]) <= min(1e-10, bos) and abs(sc.e_ss - want[1]) <= min(1e-10, bss)
    assert abs(rows[:, 0].sum() - sc.e_os) <= 1e-12 * abs(sc.e_os)
    s32 = rimp2.spin_components(t.float(), e, nocc, nvir, fo, nt)
    assert (s32.e_os, s32.e_ss) == (sc.e_os, sc.e_ss)
    sk = rimp2.spin_components(t, e, nocc, nvir, fo, nt, 1.45)
    wk = oracle_mod.spin_components_blas(b, eps, nocc, nvir, kappa=1.45, nthreads=16)
    assert abs(sk.e_os - wk[0]) <= 1e-10 and abs(sk.e_ss - wk[1]) <= 1e-10


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_row_marks_its_pairs_only(bad):
    nocc, nvir, naux = 14, 209, 560
    print("residue non-finite", bad, flush=True)
    b, eps = _problem(nocc, nvir, naux, spread=False)
    good = estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, nocc, nvir)
    b[17, 3 * nvir + 150] = bad
    pe = estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, nocc, nvir)
    hit = np.zeros((nocc, nocc), dtype=bool)
    hit[3, :] = hit[:, 3] = True
    assert np.all(np.isnan(pe.e[hit]))
    assert np.array_equal(pe.e_os[~hit], good.e_os[~hit])


def test_pool_ceiling_falls_back_to_the_matrix_kernel():
    p = synthetic.decane_scale()
    print("residue pool ceiling", flush=True)
    t = torch.from_numpy(p.b_ov).cuda()
    ref = estimate_pair_energies_from_b_ov(t, p.eps, p.nocc, p.nvir)
    lib = _lib.lib()
    lib.fh_release_workspace()
    before = _lib.stats()["fail_pool_full"]
    try:
        assert lib.fh_set_pool_limit(100 << 20) == 0  # the matrix kernel needs 71 MB
        pe = estimate_pair_energies_from_b_ov(t, p.eps, p.nocc, p.nvir)
    finally:
        lib.fh_set_pool_limit(0)
    assert _lib.stats()["fail_pool_full"] == before
    assert np.max(np.abs(pe.e - ref.e)) <= 1e-12 * np.max(np.abs(ref.e))


@pytest.mark.parametrize("shape", [(9, 150, 8, 145, 1500), (12, 272, 7, 400, 900),
                                   (3, 256, 4, 513, 4000)], ids=lambda s: "-".join(map(str, s)))
def test_opposite_spin_rectangle(shape, oracle_mod, monkeypatch):
    """Uneven channels: one tile a side, two, and one against three."""
    from ferric_amd import unrestricted as un
    na, va, nb, vb, naux = shape
    print("residue rectangle", shape, flush=True)
    ba, ea = _problem(na, va, naux, seed=3)
    bb, eb = _problem(nb, vb, naux, seed=4)
    g = torch.from_numpy
    ca = un.SpinChannel(g(ba).cuda(), ea, na, va)
    cb = un.SpinChannel(g(bb).cuda(), eb, nb, vb)
    e = un.u_opposite_spin(ca, cb)
    want = oracle_mod.u_opposite_spin((ba, ea, na, va, 0, na), (bb, eb, nb, vb, 0, nb),
                                      nthreads=16)
    assert abs(e - want) <= 1e-12 * abs(want)
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    assert abs(e - un.u_opposite_spin(ca, cb)) <= 1e-12 * abs(want)
