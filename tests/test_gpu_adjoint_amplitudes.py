"""The FP64 adjoint over whole amplitudes (run with -m gpu).

Sizes at the edges of its tiles and panels, K slices, both pair kernels, against dense
FP64 host arithmetic; the row-by-row path, which a pool ceiling selects, against the
same. Tolerance: Gamma and dE/deps are sums of at most nov = 3965 and nocc^2 nvir
products of amplitudes exact to about 1e-13 of the largest; 1e-11 of the largest result
is the bar of the other FP64 adjoint tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import _lib, rimp2  # noqa: E402

SHAPES = [
    (1, 1, 1),       # one element
    (3, 17, 40),     # less than a tile each way
    (8, 16, 64),     # one tile exactly, no padding
    (5, 26, 65),     # two (i, a) past a tile, one Q past a tile
    (16, 47, 200),   # K of 47 panels in two slices
    (61, 65, 700),   # residue pass, two orbitals a tile
    (14, 145, 1200), # residue pass, three flushes and a remainder
]


def _problem(nocc, nvir, naux):
    rng = np.random.default_rng(9 + nvir)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    return b, eps


def _host(b, eps, nocc, nvir, c_os, c_ss):
    g = (b.T @ b).reshape(nocc, nvir, nocc, nvir)
    eo, ev = eps[:nocc], eps[nocc:]
    t = g / (eo[:, None, None, None] - ev[None, :, None, None] + eo[None, None, :, None]
             - ev[None, None, None, :])
    u = (c_os + c_ss) * t - c_ss * t.transpose(0, 3, 2, 1)
    w = t * u
    gam = 4.0 * b @ u.reshape(nocc * nvir, -1).T
    deps = np.concatenate([-2 * w.sum((1, 2, 3)), 2 * w.sum((0, 2, 3))])
    return (g * u).sum(), gam, deps


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_edges(shape, dtype):
    nocc, nvir, naux = shape
    print("adjoint amplitudes", shape, dtype, flush=True)
    b, eps = _problem(nocc, nvir, naux)
    if dtype == torch.float32:
        b = b.astype(np.float32).astype(np.float64)
    t = torch.from_numpy(b).cuda().to(dtype)
    sc, e, gam, deps = rimp2.energy_adjoint(t, eps, nocc, nvir, 0, nocc, 1.2, 0.4)
    w_e, w_g, w_d = _host(b, eps, nocc, nvir, 1.2, 0.4)
    assert abs(e - w_e) <= 1e-11 * abs(w_e)
    assert np.max(np.abs(gam.cpu().numpy() - w_g)) <= 1e-11 * np.max(np.abs(w_g))
    assert np.max(np.abs(deps - w_d)) <= 1e-11 * np.max(np.abs(w_d))
    again = rimp2.energy_adjoint(t, eps, nocc, nvir, 0, nocc, 1.2, 0.4)
    assert torch.equal(gam, again[2]) and np.array_equal(deps, again[3])


def test_pool_ceiling_runs_the_rows():
    nocc, nvir, naux = 24, 100, 300
    print("adjoint pool ceiling", flush=True)
    b, eps = _problem(nocc, nvir, naux)
    t = torch.from_numpy(b).cuda()
    w_e, w_g, w_d = _host(b, eps, nocc, nvir, 1.0, 1.0)
    lib = _lib.lib()
    lib.fh_release_workspace()
    before = _lib.stats()["fail_pool_full"]
    try:
        assert lib.fh_set_pool_limit(40 << 20) == 0  # the amplitudes alone are 46 MB
        _, e, gam, deps = rimp2.energy_adjoint(t, eps, nocc, nvir, 0, nocc)
    finally:
        lib.fh_set_pool_limit(0)
    assert _lib.stats()["fail_pool_full"] == before
    assert abs(e - w_e) <= 1e-11 * abs(w_e)
    assert np.max(np.abs(gam.cpu().numpy() - w_g)) <= 1e-11 * np.max(np.abs(w_g))
    assert np.max(np.abs(deps - w_d)) <= 1e-11 * np.max(np.abs(w_d))
