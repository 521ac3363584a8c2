"""Domain fits with several workgroups to a pair (run with -m gpu).

At and one below the domain sizes and pair counts where that route begins, uneven domains in
one batch, more columns than one turn of a workgroup holds. Against numpy's solve, with the
tolerance of test_gpu_fit_edges (V is the identity plus a Gram matrix of norm about one,
condition below 10; a few D 2^-53); and bit for bit against one workgroup to a pair, which
FERRIC_FIT_BATCH selects by the pairs of a batch (the operations and their order are the same).
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import KernelError, dlpno  # noqa: E402


def _problem(naux, nvir, nocc):
    rng = np.random.default_rng(naux * 1000 + nvir)
    w = rng.standard_normal((naux, naux)) / math.sqrt(naux)
    return rng.standard_normal((naux, nocc * nvir)), np.eye(naux) + w @ w.T / 4.0


def _fit(a, v, nocc, nvir, pairs, spread=0.0, radius=1.0):
    naux = len(v)
    xyz, cen = np.zeros((naux, 3)), np.zeros((nocc, 3))
    xyz[:, 0] = spread * np.arange(naux) / naux
    cen[:, 0] = spread * np.arange(nocc) / max(1, nocc - 1)
    j, d = dlpno.domain_fit_pair_blocks(torch.from_numpy(a).cuda(), torch.from_numpy(v).cuda(),
                                        xyz, cen, nocc, nvir, radius, pairs)
    return j.cpu().numpy(), d, xyz[:, 0], cen[:, 0]


def _check(j, a, v, nvir, pairs, x, c, radius=1.0):
    for k, (p, q) in enumerate(pairs):
        d = np.flatnonzero((np.abs(x - c[p]) <= radius) | (np.abs(x - c[q]) <= radius))
        want = a[d, p * nvir:(p + 1) * nvir].T @ np.linalg.solve(v[np.ix_(d, d)],
                                                                  a[d, q * nvir:(q + 1) * nvir])
        assert np.max(np.abs(j[k] - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("naux,nvir,npairs", [(399, 20, 2), (400, 20, 64), (400, 20, 65),
                                              (413, 170, 3), (999, 5, 66), (1000, 5, 66)])
def test_sizes(naux, nvir, npairs):
    print("fit large", naux, nvir, npairs, flush=True)
    nocc = 11
    a, v = _problem(naux, nvir, nocc)
    pairs = [(i, j) for i in range(nocc) for j in range(i, nocc)][:npairs]
    j, d, x, c = _fit(a, v, nocc, nvir, pairs)
    assert d == naux
    _check(j[::9], a, v, nvir, pairs[::9], x, c)


def test_both_routes_bit_for_bit(monkeypatch):
    """66 pairs of up to 430 aux functions, the domains of between 215 and 430."""
    print("fit large, routes", flush=True)
    nocc, nvir, naux = 11, 33, 620
    a, v = _problem(naux, nvir, nocc)
    pairs = [(i, j) for i in range(nocc) for j in range(i, nocc)]
    one, d, x, c = _fit(a, v, nocc, nvir, pairs, spread=6.0, radius=1.04)
    assert 400 <= d < 500
    _check(one[::7], a, v, nvir, pairs[::7], x, c, 1.04)
    monkeypatch.setenv("FERRIC_FIT_BATCH", "33")
    several, _, _, _ = _fit(a, v, nocc, nvir, pairs, spread=6.0, radius=1.04)
    assert np.array_equal(one, several)


@pytest.mark.parametrize("at", [0, 17, 431])
@pytest.mark.parametrize("bad", [np.nan, -1.0])
def test_refusals(at, bad):
    print("fit large, refusal", at, bad, flush=True)
    a, v = _problem(432, 7, 3)
    v[at, at] = bad
    with pytest.raises(KernelError, match=rf"not positive definite \(Cholesky info {at + 1}\)"):
        _fit(a, v, 3, 7, [(0, 1), (1, 2)])
