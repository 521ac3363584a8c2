"""FP64 energies at the most aux functions that the 32-bit row offsets of the 64-wide kernel
reach, and one more (run with -m gpu).

One occupied orbital, 25 virtuals (64-wide tiles), 1.7 GB of B. Against the products in chunks
of 2^16 aux functions. Tolerance: a chain of n = 8.4e6 additions to sums that grow to |g| is
off by about 0.3 2^-53 n^1/2 = 1e-13 of it, four such deviations, twice that in the energy:
1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import rimp2  # noqa: E402


@pytest.mark.parametrize("naux", [8388592, 8388593])
def test_energy(naux):
    print("long aux", naux, flush=True)
    nvir = 25
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    b = torch.randn(naux, nvir, device="cuda", dtype=torch.float64, generator=g)
    b *= naux ** -0.5
    eps = np.concatenate([[-0.6], np.linspace(0.2, 4.0, nvir)])
    sc = rimp2.spin_components(b, eps, 1, nvir)
    k = torch.zeros(nvir, nvir, device="cuda", dtype=torch.float64)
    for part in b.split(1 << 16):
        k += part.t().contiguous() @ part
    e = torch.from_numpy(eps).cuda()
    d = 2 * e[0] - e[1:][:, None] - e[1:][None, :]
    want = float((k * k / d).sum())
    assert abs(sc.e_os - want) <= 1e-12 * abs(want)
    assert abs(sc.e_ss) <= 1e-12 * abs(want)
