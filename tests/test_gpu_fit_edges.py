"""The domain-fit kernel at the edges of its blocks (run with -m gpu).

Domains and virtuals of one, one short of, exactly and one past a 16-wide block, more
columns than a workgroup holds at once, the whole aux set per pair; against numpy's
solve. Tolerance: V is the identity plus a Gram matrix of norm about one, condition below
10, so both solves are within a few D 2^-53 of the truth; 1e-12 of the block's largest is
the bar of the other domain-fit tests.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import KernelError, synthetic  # noqa: E402
from ferric_amd.dlpno import domain_fit_pair_blocks, pno_pair_energies  # noqa: E402

SHAPES = [(1, 1), (15, 16), (16, 17), (17, 15), (33, 100), (129, 40), (70, 200), (300, 33)]


def _problem(naux, nvir, nocc=3):
    rng = np.random.default_rng(naux * 1000 + nvir)
    w = rng.standard_normal((naux, naux)) / math.sqrt(naux)
    return rng.standard_normal((naux, nocc * nvir)), np.eye(naux) + w @ w.T / 4.0


@pytest.mark.parametrize("naux,nvir", SHAPES)
def test_blocks(naux, nvir):
    print("fit edges", naux, nvir, flush=True)
    a, v = _problem(naux, nvir)
    xyz, cen = np.zeros((naux, 3)), np.zeros((3, 3))
    pairs = [(0, 0), (0, 2), (1, 2)]
    j, d = domain_fit_pair_blocks(torch.from_numpy(a).cuda(), torch.from_numpy(v).cuda(), xyz,
                                  cen, 3, nvir, 1.0, pairs)
    assert d == naux
    w = np.linalg.solve(v, a)
    for k, (p, q) in enumerate(pairs):
        want = a[:, p * nvir:(p + 1) * nvir].T @ w[:, q * nvir:(q + 1) * nvir]
        assert np.max(np.abs(j[k].cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("at", [0, 15, 16, 40])
def test_indefinite_metric_is_refused_at_any_column(at):
    print("fit indefinite", at, flush=True)
    a, v = _problem(41, 5)
    v[at, at] = -1.0
    with pytest.raises(KernelError):
        domain_fit_pair_blocks(torch.from_numpy(a).cuda(), torch.from_numpy(v).cuda(),
                               np.zeros((41, 3)), np.zeros((3, 3)), 3, 5, 1.0, [(0, 1)])


def test_fits_after_pno_truncation():
    """The call once gave NaN in some blocks when a PNO truncation had run before it in the
    process."""
    print("fit after pno", flush=True)
    p = synthetic.decane_scale()
    pairs = [(i, j) for i in range(12) for j in range(i, 12)]
    pno_pair_energies(torch.from_numpy(p.b_ov).cuda(), p.eps, p.nocc, p.nvir, 0, p.nocc, pairs,
                      1e-6)
    a, v, xyz, cen, _ = synthetic.local_fit_chain(nocc=40, nvir=100, aux_per_site=12)
    j, _ = domain_fit_pair_blocks(torch.from_numpy(a).cuda(), torch.from_numpy(v).cuda(), xyz,
                                  cen, 40, 100, 6.0)
    assert bool(torch.isfinite(j).all())
