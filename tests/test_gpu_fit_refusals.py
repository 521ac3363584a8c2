"""Domain fits refuse a metric that is not finite and positive definite (run with -m gpu).

The error names the first bad pivot, from 1, as LAPACK's potrf does. Positions: the first and
last row of a block of 16, inside one, and the last row of a domain that ends inside a block.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import _lib, dlpno  # noqa: E402

NAUX, NOCC, NVIR = 37, 2, 20


def _fit(v):
    rng = np.random.default_rng(4)
    a = torch.from_numpy(rng.standard_normal((NAUX, NOCC * NVIR))).cuda()
    j, d = dlpno.domain_fit_pair_blocks(a, torch.from_numpy(v).cuda(), np.zeros((NAUX, 3)),
                                        np.zeros((NOCC, 3)), NOCC, NVIR, 1.0, [(0, 1)])
    assert d == NAUX
    return a.cpu().numpy(), j.cpu().numpy()[0]


def _metric():
    x = 0.3 * np.arange(NAUX)
    return np.exp(-(x[:, None] - x[None, :]) ** 2 / 4.0) + 0.5 * np.eye(NAUX)


def test_good_metric():
    a, j = _fit(_metric())
    want = a[:, :NVIR].T @ np.linalg.solve(_metric(), a[:, NVIR:])
    assert np.max(np.abs(j - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 0.0, -3.0])
@pytest.mark.parametrize("at", [0, 15, 16, 20, 36])
def test_diagonal(at, bad):
    print("fit diagonal", at, bad, flush=True)
    v = _metric()
    v[at, at] = bad
    with pytest.raises(_lib.KernelError,
                       match=rf"not positive definite \(Cholesky info {at + 1}\)"):
        _fit(v)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [(1, 0), (15, 3), (16, 15), (20, 18), (36, 2)])
def test_off_diagonal(at, bad):
    print("fit off diagonal", at, bad, flush=True)
    v = _metric()
    v[at] = v[at[::-1]] = bad
    with pytest.raises(_lib.KernelError,
                       match=rf"not positive definite \(Cholesky info {at[0] + 1}\)"):
        _fit(v)
