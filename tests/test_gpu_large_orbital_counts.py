"""Energies past the pinned buffer of results and orbital energies (run with -m gpu).

It holds 8192 doubles, of which a call takes 2 + 3 nocc + nvir. The last shape of each kind
that fits and the first that does not, against dense FP64 arithmetic in torch. One product
per element at naux = 1, two at 2; 4e6 to 7e7 compensated energy terms of one sign: 1e-13.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import rimp2  # noqa: E402


@pytest.mark.parametrize("shape", [(2729, 1, 2), (2731, 1, 2), (1, 8187, 1), (1, 8190, 1)],
                         ids=lambda s: "-".join(map(str, s)))
def test_energy(shape):
    nocc, nvir, naux = shape
    print("orbital counts", shape, flush=True)
    rng = np.random.default_rng(nocc)
    b = rng.standard_normal((naux, nocc * nvir))
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    t = torch.from_numpy(b).cuda()
    sc = rimp2.spin_components(t, eps, nocc, nvir)
    e = torch.from_numpy(eps).cuda()
    g = t.t().contiguous() @ t  # (ia, jb), i = j or a = b: the exchange term is the same
    if nocc == 1:
        d = 2 * e[0] - e[1:][:, None] - e[1:][None, :]
    else:
        d = e[:nocc][:, None] + e[:nocc][None, :] - 2 * e[nocc]
    want = float((g * g / d).sum())
    assert abs(sc.e_os - want) <= 1e-13 * abs(want)
    assert abs(sc.e_ss) <= 1e-13 * abs(want)
