"""The tiling and amplitude routes of the MP2 densities at their edges (run with -m gpu).

Against P from dense FP64 amplitudes on the host. Tolerance: the amplitudes are within
1e-13 of their block's largest (an FP64 product of naux terms and one division), and the two
sums of up to nocc^2 nvir = 1.6e6 like-signed terms on the diagonal differ by a few
2^-53 sqrt(1.6e6) = 1.4e-13; 1e-11 of the largest element is the bar of the other density
tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import rimp2  # noqa: E402

SHAPES = [
    (3, 17, 40),     # one tile each, fewer slices than the reducing groups
    (5, 64, 33),     # the tile exactly full
    (65, 66, 90),    # both densities two tiles, the second nearly empty
    (61, 65, 700),   # amplitudes from the residue pass: two orbitals a tile
    (14, 145, 1200), # one orbital a tile
    (18, 257, 1500), # two tiles
]


def _host(b, eps, nocc, nvir, c_os, c_ss):
    g = (b.T @ b).reshape(nocc, nvir, nocc, nvir).transpose(0, 2, 1, 3)
    eo, ev = eps[:nocc], eps[nocc:]
    t = g / (eo[:, None, None, None] + eo[None, :, None, None] - ev[None, None, :, None]
             - ev[None, None, None, :])
    u = (c_os + c_ss) * t - c_ss * t.swapaxes(2, 3)
    tv = t.transpose(2, 0, 1, 3).reshape(nvir, -1)
    uv = u.transpose(2, 0, 1, 3).reshape(nvir, -1)
    return -(t.reshape(nocc, -1) @ u.reshape(nocc, -1).T), tv @ uv.T


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_tiles_and_routes(shape, monkeypatch):
    nocc, nvir, naux = shape
    print("density route", shape, flush=True)
    rng = np.random.default_rng(5 + nvir)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    t = torch.from_numpy(b).cuda()
    w_oo, w_vv = _host(b, eps, nocc, nvir, 1.2, 0.4)
    for tile in (None, "64"):  # "64" holds the amplitude pass to the matrix kernel
        if tile:
            monkeypatch.setenv("FERRIC_HIP_TILE", tile)
        _, p_oo, p_vv = rimp2.mp2_density(t, eps, nocc, nvir, 0, nocc, 1.2, 0.4)
        assert np.max(np.abs(p_oo - w_oo)) <= 1e-11 * np.max(np.abs(w_oo))
        assert np.max(np.abs(p_vv - w_vv)) <= 1e-11 * np.max(np.abs(w_vv))
