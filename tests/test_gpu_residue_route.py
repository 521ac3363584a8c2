"""The residue kernels wherever they can run, and the rule that chooses them (run with -m gpu).

FERRIC_HIP_TILE=256 takes them at the shapes of test_gpu_residue, some of which the rule gives
to the matrix kernels, which are faster there; the tolerances are those of that file.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import Precision, _lib  # noqa: E402
from ferric_amd import unrestricted as un  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402
from tests.test_gpu_residue import SHAPES, _args, _problem  # noqa: E402


@pytest.fixture(autouse=True)
def timing():
    _lib.set_timing(True)
    yield
    _lib.set_timing(False)


def _tile():
    return _lib.last_timing()["tile"]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_fp64_pairs(shape, oracle_mod, monkeypatch):
    nocc, nvir, naux, frozen = shape
    print("residue route, pairs", shape, flush=True)
    monkeypatch.setenv("FERRIC_HIP_TILE", "256")
    b, eps = _problem(nocc, nvir, naux)
    e, fo, nt = _args(b, eps, nocc, frozen)
    pe = estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), e, nocc, nvir, fo, nt)
    assert _tile() == 256
    w_os, w_ss = oracle_mod.pair_energies(b, eps, nocc, nvir)
    top = np.max(np.abs(w_os))
    assert np.max(np.abs(pe.e_os - w_os)) <= 1e-12 * top
    assert np.max(np.abs(pe.e_ss - w_ss)) <= 1e-12 * top


@pytest.mark.parametrize("shape", [(41, 65, 900), (24, 160, 800), (13, 257, 700)],
                         ids=lambda s: "-".join(map(str, s)))
def test_mixed_pairs(shape, oracle_mod, monkeypatch):
    nocc, nvir, naux = shape
    print("residue route, mixed", shape, flush=True)
    monkeypatch.setenv("FERRIC_HIP_TILE", "256")
    b, eps = _problem(nocc, nvir, naux, spread=False)
    pe = estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, nocc, nvir,
                                          precision=Precision.MIXED)
    assert _tile() == 256
    br = b.astype(np.float32).astype(np.float64)
    w_os, w_ss = oracle_mod.pair_energies(br, eps, nocc, nvir)
    top = np.max(np.abs(w_os))
    assert np.max(np.abs(pe.e_os - w_os)) <= 2.8e-7 * top
    assert np.max(np.abs(pe.e_ss - w_ss)) <= 2.8e-7 * top


@pytest.mark.parametrize("shape", [(9, 150, 8, 145, 1500), (12, 272, 7, 400, 900),
                                   (3, 256, 4, 513, 4000), (5, 65, 4, 66, 60)],
                         ids=lambda s: "-".join(map(str, s)))
def test_opposite_spin(shape, oracle_mod, monkeypatch):
    na, va, nb, vb, naux = shape
    print("residue route, rectangle", shape, flush=True)
    monkeypatch.setenv("FERRIC_HIP_TILE", "256")
    ba, ea = _problem(na, va, naux, seed=3)
    bb, eb = _problem(nb, vb, naux, seed=4)
    g = torch.from_numpy
    e = un.u_opposite_spin(un.SpinChannel(g(ba).cuda(), ea, na, va),
                           un.SpinChannel(g(bb).cuda(), eb, nb, vb))
    assert _tile() == 256
    want = oracle_mod.u_opposite_spin((ba, ea, na, va, 0, na), (bb, eb, nb, vb, 0, nb),
                                      nthreads=16)
    assert abs(e - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("precision, shape, tile", [
    (Precision.FP64, (70, 208, 889), 256), (Precision.FP64, (16, 512, 1000), 256),
    (Precision.FP64, (9, 371, 1363), 64), (Precision.FP64, (46, 200, 60), 64),
    (Precision.MIXED, (24, 208, 742), 256), (Precision.MIXED, (23, 491, 177), 64),
], ids=str)
def test_rule(precision, shape, tile):
    """Shapes where one side is faster by 10% or more."""
    nocc, nvir, naux = shape
    print("residue route, rule", shape, flush=True)
    b, eps = _problem(nocc, nvir, naux, spread=False)
    estimate_pair_energies_from_b_ov(torch.from_numpy(b).cuda(), eps, nocc, nvir,
                                     precision=precision)
    assert _tile() == tile
