"""The workspace of routes that have another behind them (run with -m gpu).

A pool ceiling that holds the start of the faster route but not all of it, and ceilings
set after a call that took it: the call is made by the other route, is not counted as a
failure, and gives that route's results. Tolerances as in test_gpu_adjoint_amplitudes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from ferric_amd import Precision, _lib, batched, rimp2, synthetic  # noqa: E402
from ferric_amd.dlpno import estimate_pair_energies_from_b_ov  # noqa: E402
from tests.test_gpu_adjoint_amplitudes import _host, _problem  # noqa: E402

SHAPE = (24, 100, 300)


@pytest.fixture
def pool():
    lib = _lib.lib()
    lib.fh_release_workspace()
    lib.fh_reset_stats()
    yield lib
    lib.fh_set_pool_limit(0)
    lib.fh_release_workspace()


def _gradient(precision=Precision.FP64):
    b, eps = _problem(*SHAPE)
    t = torch.from_numpy(b).cuda()
    return rimp2.energy_adjoint(t, eps, SHAPE[0], SHAPE[1], 0, SHAPE[0], precision=precision)


def _check(res):
    b, eps = _problem(*SHAPE)
    w_e, w_g, w_d = _host(b, eps, SHAPE[0], SHAPE[1], 1.0, 1.0)
    _, e, gam, deps = res
    assert abs(e - w_e) <= 1e-11 * abs(w_e)
    assert np.max(np.abs(gam.cpu().numpy() - w_g)) <= 1e-11 * np.max(np.abs(w_g))
    assert np.max(np.abs(deps - w_d)) <= 1e-11 * np.max(np.abs(w_d))


def test_ceiling_between_the_amplitudes_and_the_operand(pool):
    """88 MB for all of it, 81 for the amplitudes, B by Q and the K slices."""
    whole = _gradient()
    peak = _lib.stats()["pool_peak_bytes"]
    pool.fh_release_workspace()
    assert pool.fh_set_pool_limit(peak - 1) == 0
    rows = _gradient()
    _check(rows)
    _check(whole)
    assert _lib.stats()["fail_pool_full"] == 0
    _check(_gradient())  # and with what the first one left behind


def test_ceiling_after_an_amplitude_call(pool):
    _gradient()
    assert pool.fh_set_pool_limit(40 << 20) == 0  # the amplitudes alone are 46 MB
    _check(_gradient())
    assert _lib.stats()["fail_pool_full"] == 0


@pytest.mark.parametrize("precision", [Precision.BF16X3, Precision.INT8X4])
def test_ceiling_after_a_residue_call(pool, precision):
    """Another kind of call under the ceiling that it needs by itself, beside the 2 doubles a
    pair that the pair energies keep on any route (14 kB at 41 occupied)."""
    want = _gradient(precision)
    peak = _lib.stats()["pool_peak_bytes"]
    p = synthetic.decane_scale()
    estimate_pair_energies_from_b_ov(torch.from_numpy(p.b_ov).cuda(), p.eps, p.nocc, p.nvir)
    assert _lib.stats()["pool_peak_bytes"] > 4 * peak
    assert pool.fh_set_pool_limit(peak + 16 * (41 * 42 // 2)) == 0
    got = _gradient(precision)
    assert got[1] == want[1] and torch.equal(got[2], want[2])
    assert _lib.stats()["fail_pool_full"] == 0


@pytest.mark.parametrize("precision, ceiling", [(Precision.BF16X3, 15080208),
                                                (Precision.INT8X4, 40767696),
                                                (Precision.FP64, 25606928)])
def test_sums_of_one_row_at_a_time(pool, precision, ceiling):
    """The bytes of the slots with the sums of one row. The energies and dE/deps are the same
    compensated sums in another order: 1e-14; Gamma is not touched by it."""
    if precision == Precision.FP64:
        assert pool.fh_set_pool_limit(40 << 20) == 0  # the amplitudes alone are 46 MB
    want = _gradient(precision)
    assert ceiling < _lib.stats()["pool_peak_bytes"] < 1.2 * ceiling
    pool.fh_release_workspace()
    assert pool.fh_set_pool_limit(ceiling) == 0
    got = _gradient(precision)
    assert _lib.stats()["fail_pool_full"] == 0
    assert torch.equal(got[2], want[2])
    assert abs(got[1] - want[1]) <= 1e-14 * abs(want[1])
    assert np.max(np.abs(got[3] - want[3])) <= 1e-14 * np.max(np.abs(want[3]))


def test_a_call_past_the_ceiling_is_refused_as_before(pool):
    _gradient()
    assert pool.fh_set_pool_limit(8 << 20) == 0  # the row path needs 27 MB
    with pytest.raises(_lib.PoolFullError):
        _gradient()
    assert _lib.stats()["fail_pool_full"] == 1


def test_batched_graph_after_slots_were_given_back(pool):
    """The captured graphs hold workspace pointers: a residue call grows the operand slot that
    they read, a ceiling makes the next call free it, and the domains' energies stay the same
    bit for bit."""
    rng = np.random.default_rng(2)
    nocc, nvir, naux = np.array([3, 5, 8]), np.array([40, 90, 130]), np.array([100, 200, 333])
    size = nocc * nvir * naux
    b = torch.from_numpy(rng.standard_normal(int(size.sum())) * 0.02).cuda()
    eps = torch.from_numpy(np.concatenate(
        [np.concatenate([np.linspace(-1.2, -0.4, o), np.linspace(0.2, 4.0, v)])
         for o, v in zip(nocc, nvir)])).cuda()
    offs = np.concatenate([[0], np.cumsum(size)[:-1]])
    eoff = np.concatenate([[0], np.cumsum(nocc + nvir)[:-1]])

    def run():
        return batched.domain_energies(b, eps, nocc, nvir, naux, offs, eoff,
                                       precision=Precision.BF16X3)

    want = run()
    assert all(np.array_equal(x, y) for x, y in zip(want, run()))
    small = _lib.stats()["pool_peak_bytes"]
    p = synthetic.decane_scale()
    t = torch.from_numpy(p.b_ov).cuda()
    for _ in range(2):
        estimate_pair_energies_from_b_ov(t, p.eps, p.nocc, p.nvir)
        assert all(np.array_equal(x, y) for x, y in zip(want, run()))
        assert pool.fh_set_pool_limit(small + (64 << 20)) == 0
        _gradient(Precision.BF16X3)
        assert all(np.array_equal(x, y) for x, y in zip(want, run()))
        assert pool.fh_set_pool_limit(0) == 0
