"""Host-pointer entries against the device-tensor ones (run with -m gpu).

The same kernels on the same B: equal bit for bit. The shapes take the residue
kernel; in the last one its scratch of column maxima is larger than the beta B.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import unrestricted as un  # noqa: E402


def _channel(nocc, nvir, naux, seed):
    rng = np.random.default_rng(seed)
    b = rng.standard_normal((naux, nocc * nvir)) * np.sqrt(0.09 / naux)
    eps = np.concatenate([np.sort(rng.uniform(-1.2, -0.35, nocc)),
                          np.sort(rng.uniform(0.12, 5.0, nvir))])
    return b, eps


@pytest.mark.parametrize("shape", [(21, 229, 20, 230, 960), (12, 272, 7, 400, 900),
                                   (64, 144, 1, 150, 1000)], ids=lambda s: "-".join(map(str, s)))
def test_opposite_spin_host_arrays(shape, oracle_mod):
    na, va, nb, vb, naux = shape
    print("opposite spin, host arrays", shape, flush=True)
    ba, ea = _channel(na, va, naux, 5)
    bb, eb = _channel(nb, vb, naux, 6)
    host = un.u_opposite_spin(un.SpinChannel(ba, ea, na, va), un.SpinChannel(bb, eb, nb, vb))
    dev = un.u_opposite_spin(un.SpinChannel(torch.from_numpy(ba).cuda(), ea, na, va),
                             un.SpinChannel(torch.from_numpy(bb).cuda(), eb, nb, vb))
    assert host == dev
    want = oracle_mod.u_opposite_spin((ba, ea, na, va, 0, na), (bb, eb, nb, vb, 0, nb),
                                      nthreads=16)
    assert abs(host - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("shape", [(21, 229, 960), (13, 257, 1500)],
                         ids=lambda s: "-".join(map(str, s)))
def test_same_spin_host_arrays(shape):
    no, nv, naux = shape
    print("same spin, host arrays", shape, flush=True)
    b, e = _channel(no, nv, naux, 7)
    assert un.u_same_spin(un.SpinChannel(b, e, no, nv)) == un.u_same_spin(
        un.SpinChannel(torch.from_numpy(b).cuda(), e, no, nv))
