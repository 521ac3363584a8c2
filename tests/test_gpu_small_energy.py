"""The one-launch energy at the edges of its range (run with -m gpu).

One element, both tile sides full and just short, the most items, the largest aux count
and one past it (the packed kernels), frozen core, kappa and row partials, against the
oracle to its rounding bound and 1e-10; and the packed kernels (FERRIC_HIP_TILE holds the
call to them) to the sum of both bounds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import rimp2  # noqa: E402

SHAPES = [(1, 1, 1, 0), (5, 19, 84, 0), (22, 24, 77, 1), (3, 25, 16, 0), (6, 63, 255, 2),
          (10, 64, 256, 0), (10, 64, 257, 0)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("kappa", [None, 1.45])
def test_edges(shape, kappa, oracle_mod, monkeypatch):
    nocc, nvir, naux, frozen = shape
    print("small energy", shape, kappa, flush=True)
    rng = np.random.default_rng(nvir)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    act = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    eps = np.concatenate([np.full(frozen, -11.2), act])
    t = torch.from_numpy(b).cuda()
    args = (t, eps, nocc, nvir, frozen, frozen + nocc, kappa)
    sc, rows = rimp2.spin_components(*args, row_partials=True)
    kw = {} if kappa is None else {"kappa": kappa}
    want = oracle_mod.spin_components_blas(b, act, nocc, nvir, nthreads=16, **kw)
    bos, bss = oracle_mod.energy_bound(b, act, nocc, nvir, 0, nocc)
    assert abs(sc.e_os - want[0]) <= min(1e-10, bos) and abs(sc.e_ss - want[1]) <= min(1e-10, bss)
    assert abs(rows[:, 0].sum() - sc.e_os) <= 1e-12 * abs(sc.e_os)
    again = rimp2.spin_components(*args)
    assert (again.e_os, again.e_ss) == (sc.e_os, sc.e_ss)
    monkeypatch.setenv("FERRIC_HIP_TILE", "32" if nvir <= 24 else "64")
    pk = rimp2.spin_components(*args)
    assert abs(pk.e_os - sc.e_os) <= 2 * bos and abs(pk.e_ss - sc.e_ss) <= 2 * bss
