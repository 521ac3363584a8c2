"""Residue arithmetic on rows that span a wide range over the aux functions (run with -m gpu).

Pair energies, each judged by its own size against the matrix kernel of the same precision
(FERRIC_HIP_TILE selects it), whose error follows sum |B||B| of the pair itself. The rows of
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

from ferric_amd import Precision  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402

NOCC, NVIR = 24, 160
BAR = {Precision.FP64: 1e-15, Precision.MIXED: 8e-8}


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
