"""The two forms of the first dressing product (run with -m gpu): 64 and 65 columns on the
left, against float64 numpy. Tolerance: three chained products of 70, 70 and 31 terms with
entries near one, each within n 2^-53 of its absolute sum: 1e-13 of the largest element
times ten."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import dressing  # noqa: E402


@pytest.mark.parametrize("nleft", [1, 64, 65])
def test_left_widths(nleft):
    print("dressing nleft", nleft, flush=True)
    rng = np.random.default_rng(nleft)
    naux, nao, nright = 31, 70, 9
    j3 = rng.standard_normal((naux, nao, nao))
    j3 += j3.transpose(0, 2, 1)
    m, cl, cr = (rng.standard_normal(s) for s in ((naux, naux), (nao, nleft), (nao, nright)))
    got = dressing.stream_dressed_mo_band(*(torch.from_numpy(x).cuda() for x in (j3, m, cl, cr)),
                                          (3, 29)).cpu().numpy()
    y = np.einsum("qml,mr->qlr", j3 @ cl, cr).reshape(naux, -1)
    want = (m @ y)[3:29]
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))
