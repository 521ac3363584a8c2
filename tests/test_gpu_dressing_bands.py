"""Dressed bands of few aux rows (run with -m gpu): the first product has another form from 24
rows and 2 to 64 left columns on. Against numpy in FP64; sums of nao^2 naux products: 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import dressing  # noqa: E402


@pytest.mark.parametrize("naux", [1, 23, 24, 25])
@pytest.mark.parametrize("nleft", [1, 2, 64, 65])
def test_band(naux, nleft):
    print("dressing band", naux, nleft, flush=True)
    nao, nright = 90, 33
    rng = np.random.default_rng(naux * 100 + nleft)
    j3 = rng.standard_normal((naux, nao, nao))
    j3 += j3.transpose(0, 2, 1)  # integrals: symmetric in the two functions
    m = rng.standard_normal((naux, naux))
    cl, cr = rng.standard_normal((nao, nleft)), rng.standard_normal((nao, nright))
    g = [torch.from_numpy(x).cuda() for x in (j3, m, cl, cr)]
    got = dressing.stream_dressed_mo_band(*g).cpu().numpy()
    want = m @ np.einsum("qmn,mi,na->qia", j3, cl, cr, optimize=True).reshape(naux, -1)
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))
