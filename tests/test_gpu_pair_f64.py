"""The direct-load FP64 pair kernel at the edges of its tiles (run with -m gpu).

Virtuals that end in one, two, three and four blocks of the last tile (a narrow last tile
has its own wave layout), one tile and several, an odd and an even number of panels,
kappa, against the oracle's FP64 components: to its rounding bound and 1e-10.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import rimp2  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402

SHAPES = [(1, 25, 1), (3, 48, 17), (4, 64, 16), (5, 65, 40), (4, 96, 33), (3, 100, 100),
          (3, 113, 24), (6, 129, 8), (2, 209, 130)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("kappa", [None, 1.45])
def test_tile_edges(shape, kappa, oracle_mod, monkeypatch):
    nocc, nvir, naux = shape
    print("pair f64", shape, kappa, flush=True)
    monkeypatch.setenv("FERRIC_HIP_TILE", "64")
    rng = np.random.default_rng(nvir)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    t = torch.from_numpy(b).cuda()
    sc, rows = rimp2.spin_components(t, eps, nocc, nvir, 0, nocc, kappa, row_partials=True)
    kw = {} if kappa is None else {"kappa": kappa}
    want = oracle_mod.spin_components_blas(b, eps, nocc, nvir, nthreads=16, **kw)
    bos, bss = oracle_mod.energy_bound(b, eps, nocc, nvir, 0, nocc)
    assert abs(sc.e_os - want[0]) <= min(1e-10, bos) and abs(sc.e_ss - want[1]) <= min(1e-10, bss)
    assert abs(rows[:, 0].sum() - sc.e_os) <= 1e-12 * abs(sc.e_os)
    if kappa is None:
        pe = estimate_pair_energies_from_b_ov(t, eps, nocc, nvir)
        w_os, w_ss = oracle_mod.pair_energies(b, eps, nocc, nvir)
        assert np.max(np.abs(pe.e_os - w_os)) <= 1e-12 * np.max(np.abs(w_os))
        assert np.max(np.abs(pe.e_ss - w_ss)) <= 1e-12 * np.max(np.abs(w_os))
