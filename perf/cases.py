"""The work a user has this library do, as timed cases over its public entry points.

``listed()`` names twelve cases from the smallest call (water in cc-pVDZ) to the
100/900/3600 workload; ``draw(rng)`` gives further cases of the same kinds with
sizes spread over the ranges between them. ``prepare`` makes a case's inputs on
the device from a seed, ``run`` is one pass as a user's program makes it,
``work`` the bytes and operations the pass cannot do without, and ``exact`` the
same results from plain torch or numpy in 64 bits.

Kinds:

* ``energy``   the closed-shell spin components of a resident B (any precision)
* ``job``      three-centre integrals -> dressed B -> spin components, the order
               of one RI-MP2 single point
* ``gradient`` energy and adjoint, through the autograd function
* ``density``  the MP2 one-particle densities P_oo, P_vv
* ``ump2``     the three blocks of an open-shell energy
* ``dlpno``    a local-MP2 energy in its default configuration: pair energies, the pair
               screen and the sum over the retained pairs
* ``domains``  many small independent pair domains in one call
* ``fits``     domain-local fits of pair blocks and their pair energies
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ferric_amd import batched, dlpno, dressing, rimp2, unrestricted
from ferric_amd._lib import Precision
from ferric_amd.autograd import ri_mp2_energy

DEV = "cuda"


def listed():
    return [
        # One point of a potential-energy scan of a small molecule: water in cc-pVDZ. A call this
        # small is launches, transfers and waits.
        {"name": "energy_water", "kind": "energy", "precision": "fp64", "store": "f64",
         "nocc": 5, "nvir": 19, "naux": 84, "frozen": 0, "kappa": 0.0},
        # The energy of a medium molecule (decane in a double-zeta basis) in the default precision.
        {"name": "energy_decane", "kind": "energy", "precision": "fp64", "store": "f64",
         "nocc": 41, "nvir": 209, "naux": 960, "frozen": 0, "kappa": 0.0},
        # The same call under the reference's mixed precision setting, on a larger molecule.
        {"name": "energy_mixed", "kind": "energy", "precision": "mixed", "store": "f64",
         "nocc": 60, "nvir": 450, "naux": 1800, "frozen": 10, "kappa": 0.0},
        # The largest single energy: the 100/900/3600 workload in the mode its headline uses.
        {"name": "energy_large_int8x4", "kind": "energy", "precision": "int8x4", "store": "f32",
         "nocc": 100, "nvir": 900, "naux": 3600, "frozen": 0, "kappa": 0.0},
        # A whole FP64 single point after the SCF: integrals dressed into B, then the energy.
        {"name": "job_fp64", "kind": "job", "precision": "fp64", "nocc": 60, "nvir": 450,
         "naux": 1800},
        # One geometry step's SCS-MP2 gradient intermediates, in FP64 ...
        {"name": "gradient_decane", "kind": "gradient", "precision": "fp64", "nocc": 41,
         "nvir": 209, "naux": 960, "frozen": 0},
        # ... and for a larger molecule in the INT8X4 mode.
        {"name": "gradient_int8x4", "kind": "gradient", "precision": "int8x4", "nocc": 60,
         "nvir": 450, "naux": 1800, "frozen": 0},
        # Unrelaxed densities of an orbital-optimised or property run.
        {"name": "density_decane", "kind": "density", "nocc": 41, "nvir": 209, "naux": 960},
        # An open-shell cation of the same size: both same-spin blocks and the opposite-spin one.
        {"name": "ump2_cation", "kind": "ump2", "precision": "fp64", "nocc_a": 21, "nvir_a": 229,
         "nocc_b": 20, "nvir_b": 230, "naux": 960},
        # A local-MP2 energy of a chain molecule: every pair's energy, and the pairs the default
        # 1e-5 Eh screen keeps.
        {"name": "dlpno_chain", "kind": "dlpno", "nocc": 100, "nvir": 200, "per_site": 24},
        # The pair domains of a large molecule, uneven in every dimension.
        {"name": "domains_512", "kind": "domains", "precision": "fp64", "ndom": 512, "shapes": 1005},
        # Aux fits local to each pair's domain, and the pair energies of the fitted blocks.
        {"name": "fits_chain", "kind": "fits", "nocc": 40, "nvir": 100, "per_site": 12,
         "radius": 6.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["energy", "energy", "energy", "job", "gradient", "gradient", "density",
                       "ump2", "dlpno", "domains", "fits"])
    if kind == "energy":
        # An aux basis holds about 2.5 to 4.5 functions per orbital; frozen cores and the
        # kappa regulariser belong to FP64 runs, storage in FP32 to reduced ones too.
        precision = rng.choice(["fp64", "fp64", "fp64", "mixed", "int8x4", "bf16x3", "fp32"])
        nocc, nvir = _log(rng, 4, 90), _log(rng, 12, 560)
        return {"kind": kind, "precision": precision, "store": rng.choice(["f64", "f32"]),
                "nocc": nocc, "nvir": nvir, "naux": int((nocc + nvir) * rng.uniform(2.5, 4.0)),
                "frozen": rng.choice([0, 0, 1, 7]),
                "kappa": rng.choice([0.0, 0.0, 1.45]) if precision == "fp64" else 0.0}
    if kind == "job":
        nocc, nvir = _log(rng, 5, 60), _log(rng, 20, 450)
        return {"kind": kind, "precision": rng.choice(["fp64", "int8x4"]), "nocc": nocc,
                "nvir": nvir, "naux": int((nocc + nvir) * rng.uniform(2.5, 3.6))}
    if kind == "gradient":
        nocc, nvir = _log(rng, 4, 60), _log(rng, 15, 450)
        return {"kind": kind, "precision": rng.choice(["fp64", "int8x4", "bf16x3"]),
                "nocc": nocc, "nvir": nvir, "naux": int((nocc + nvir) * rng.uniform(2.5, 3.6)),
                "frozen": rng.choice([0, 0, 3])}
    if kind == "density":
        nocc, nvir = _log(rng, 4, 48), _log(rng, 15, 260)
        return {"kind": kind, "nocc": nocc, "nvir": nvir,
                "naux": int((nocc + nvir) * rng.uniform(2.5, 4.0))}
    if kind == "ump2":
        na, nv = _log(rng, 4, 50), _log(rng, 16, 350)
        nb = max(2, na - rng.choice([1, 1, 2, 3]))
        return {"kind": kind, "precision": rng.choice(["fp64", "fp64", "int8x4"]), "nocc_a": na,
                "nvir_a": nv, "nocc_b": nb, "nvir_b": nv + na - nb,
                "naux": int((na + nv) * rng.uniform(2.5, 4.0))}
    if kind == "dlpno":
        return {"kind": kind, "nocc": _log(rng, 8, 100), "nvir": _log(rng, 30, 200),
                "per_site": rng.randint(12, 26)}
    if kind == "domains":
        return {"kind": kind, "precision": rng.choice(["fp64", "fp64", "bf16x3"]),
                "ndom": _log(rng, 16, 600), "shapes": rng.randrange(1, 1 << 20)}
    return {"kind": "fits", "nocc": _log(rng, 8, 48), "nvir": _log(rng, 20, 120),
            "per_site": rng.randint(6, 14), "radius": rng.choice([4.5, 6.0, 9.0, 12.5])}


# ---- inputs ---------------------------------------------------------------------------------


def _precision(case):
    return {"fp64": Precision.FP64, "fp32": Precision.FP32, "mixed": Precision.MIXED,
            "bf16x3": Precision.BF16X3, "int8x4": Precision.INT8X4}[case["precision"]]


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 64 + salt)
    return g


def _energies(rng, nocc, nvir, frozen=0):
    core = np.sort(rng.uniform(-11.3, -11.1, frozen))
    occ = np.sort(rng.uniform(-1.2, -0.35, nocc))
    vir = np.sort(np.exp(rng.uniform(math.log(0.12), math.log(5.0), nvir)))
    return np.concatenate([core, occ, vir])


def _b(seed, salt, naux, nocc, nvir, dtype=torch.float64):
    """A fitted tensor: normal entries, one aux row in a hundred much larger, as the diffuse
    s functions of a fitting basis are."""
    b = torch.randn(naux, nocc * nvir, device=DEV, dtype=dtype, generator=_gen(seed, salt))
    b *= math.sqrt(0.09 / naux)
    b[::100] *= 4.0
    return b


def _shapes(case):
    rng = np.random.default_rng(case["shapes"])
    n = case["ndom"]
    nocc = rng.integers(2, 13, n)
    nvir = np.rint(np.exp(rng.uniform(math.log(20), math.log(240), n))).astype(np.int64)
    naux = np.rint(np.exp(rng.uniform(math.log(80), math.log(720), n))).astype(np.int64)
    sizes = naux * nocc * nvir
    b_off = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    e_off = np.concatenate([[0], np.cumsum(nocc + nvir)[:-1]]).astype(np.int64)
    return nocc, nvir, naux, b_off, e_off


def _chain_b(seed, nocc, nvir, per_site, reach=3):
    """B of localized occupied orbitals on a line: orbital i lives on the aux rows of the sites
    within ``reach``, decaying as exp(-distance)."""
    b = torch.randn(nocc, per_site, nocc, nvir, device=DEV, dtype=torch.float64,
                    generator=_gen(seed, 1))
    site = torch.arange(nocc, device=DEV)
    d = (site[:, None] - site[None, :]).abs()
    w = torch.where(d <= reach, torch.exp(-d.double()), torch.zeros((), device=DEV).double())
    b *= w[:, None, :, None]
    b *= math.sqrt(0.0081 / per_site)
    return b.reshape(nocc * per_site, nocc * nvir).contiguous()


def _line(nocc):
    c = np.zeros((nocc, 3))
    c[:, 0] = 2.5 * np.arange(nocc)
    return c


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 7])
    s = {"case": case}
    if kind == "energy":
        s["eps"] = _energies(rng, case["nocc"], case["nvir"], case["frozen"])
        s["b"] = _b(seed, 1, case["naux"], case["nocc"], case["nvir"],
                    torch.float32 if case["store"] == "f32" else torch.float64)
    elif kind == "job":
        nocc, nvir, naux = case["nocc"], case["nvir"], case["naux"]
        nao = nocc + nvir
        s["eps"] = _energies(rng, nocc, nvir)
        j3 = torch.randn(naux, nao, nao, device=DEV, dtype=torch.float64, generator=_gen(seed, 1))
        s["j3"] = j3 + j3.transpose(1, 2)
        s["j3"] *= math.sqrt(0.09 / naux / nao)
        c = torch.randn(nao, nao, device=DEV, dtype=torch.float64, generator=_gen(seed, 2))
        c *= nao ** -0.25
        s["c_occ"], s["c_vir"] = c[:, :nocc].contiguous(), c[:, nocc:].contiguous()
        m = torch.randn(naux, naux, device=DEV, dtype=torch.float64, generator=_gen(seed, 3))
        s["m"] = (m + m.t()) * (0.3 / math.sqrt(naux))
        s["m"].diagonal().add_(1.0)
    elif kind == "gradient":
        s["eps"] = torch.from_numpy(_energies(rng, case["nocc"], case["nvir"], case["frozen"]))
        s["b"] = _b(seed, 1, case["naux"], case["nocc"], case["nvir"])
    elif kind == "density":
        s["eps"] = _energies(rng, case["nocc"], case["nvir"])
        s["b"] = _b(seed, 1, case["naux"], case["nocc"], case["nvir"])
    elif kind == "ump2":
        for k, t in enumerate("ab"):
            no, nv = case["nocc_" + t], case["nvir_" + t]
            s[t] = unrestricted.SpinChannel(_b(seed, 1 + k, case["naux"], no, nv),
                                            _energies(rng, no, nv), no, nv)
    elif kind == "dlpno":
        s["b"] = _chain_b(seed, case["nocc"], case["nvir"], case["per_site"])
        s["eps"] = _energies(rng, case["nocc"], case["nvir"])
        s["centers"] = _line(case["nocc"])
    elif kind == "domains":
        nocc, nvir, naux, b_off, e_off = s["shapes"] = _shapes(case)
        s["b"] = torch.randn(int((nocc * nvir * naux).sum()), device=DEV, dtype=torch.float64,
                             generator=_gen(seed, 1))
        scale = torch.from_numpy(np.sqrt(0.09 / naux)).to(DEV)
        s["b"] *= scale.repeat_interleave(torch.from_numpy(nocc * nvir * naux).to(DEV))
        s["eps"] = torch.from_numpy(np.concatenate(
            [_energies(rng, int(o), int(v)) for o, v in zip(nocc, nvir)])).to(DEV)
    else:
        nocc, nvir, per = case["nocc"], case["nvir"], case["per_site"]
        naux = nocc * per
        xs = np.repeat(2.5 * np.arange(nocc), per) + rng.uniform(-0.8, 0.8, naux)
        s["xyz"] = np.zeros((naux, 3))
        s["xyz"][:, 0] = xs
        s["xyz"][:, 1] = rng.uniform(-0.3, 0.3, naux)
        s["centers"] = _line(nocc)
        x = torch.from_numpy(xs).to(DEV)
        s["v"] = torch.exp(-(x[:, None] - x[None, :]) ** 2 / 4.0)
        s["v"].diagonal().add_(0.5)
        a = torch.randn(naux, nocc, nvir, device=DEV, dtype=torch.float64, generator=_gen(seed, 1))
        w = torch.exp(-(x[:, None] - torch.from_numpy(s["centers"][:, 0]).to(DEV)).abs() / 2.5)
        s["a"] = (a * (0.1 * w)[:, :, None]).reshape(naux, nocc * nvir).contiguous()
        s["eps"] = _energies(rng, nocc, nvir)
        s["pairs"] = [(i, j) for i in range(nocc) for j in range(i, nocc)]
    return s


# ---- one pass -------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "energy":
        fz, no = case["frozen"], case["nocc"]
        sc = rimp2.spin_components(s["b"], s["eps"], no, case["nvir"], fz, fz + no,
                                   case["kappa"] or None, _precision(case))
        return sc.e_os, sc.e_ss, sc.e_total
    if kind == "job":
        b = dressing.stream_dressed_mo_band(s["j3"], s["m"], s["c_occ"], s["c_vir"])
        sc = rimp2.spin_components(b, s["eps"], case["nocc"], case["nvir"],
                                   precision=_precision(case))
        return {"b": b, "e": [sc.e_os, sc.e_ss, sc.e_total]}
    if kind == "gradient":
        b = s["b"].detach().requires_grad_()
        eps = s["eps"].detach().requires_grad_()
        e_os, e_ss = ri_mp2_energy(b, eps, case["nocc"], case["nvir"], case["frozen"],
                                   precision=_precision(case))
        (1.2 * e_os + e_ss / 3.0).backward()
        return {"e": [e_os.detach(), e_ss.detach()], "b": b.grad, "eps": eps.grad}
    if kind == "density":
        sc, p_oo, p_vv = rimp2.mp2_density(s["b"], s["eps"], case["nocc"], case["nvir"])
        return {"e": [sc.e_os, sc.e_ss], "oo": p_oo, "vv": p_vv}
    if kind == "ump2":
        return unrestricted.u_mp2_components(s["a"], s["b"], _precision(case))
    if kind == "dlpno":
        no, nv = case["nocc"], case["nvir"]
        pe = dlpno.estimate_pair_energies_from_b_ov(s["b"], s["eps"], no, nv)
        dom = dlpno.build_pair_domains_by_energy(s["centers"], pe, 1e-5)
        sc, diag = dlpno.dlpno_mp2_from_b_ov(s["b"], s["eps"], no, nv, 0, no, dom,
                                             pair_energies=pe)
        return {"os": pe.e_os, "ss": pe.e_ss, "e": [sc.e_os, sc.e_ss], "n": diag.n_pairs}
    if kind == "domains":
        return batched.domain_energies(s["b"], s["eps"], *s["shapes"], precision=_precision(case))
    j, dmax = dlpno.domain_fit_pair_blocks(s["a"], s["v"], s["xyz"], s["centers"], case["nocc"],
                                           case["nvir"], case["radius"], s["pairs"])
    e_os, e_ss = dlpno.pair_energies_from_blocks(j, s["pairs"], s["eps"], case["nocc"],
                                                 case["nvir"])
    return {"j": j, "dmax": dmax, "os": e_os, "ss": e_ss}


# ---- what a pass cannot do without ------------------------------------------------------------


def _pairs(nocc, nvir, naux):
    """FLOP of the unique occupied pairs' products (a multiply-add is two)."""
    return float(nocc) * (nocc + 1) * nvir * nvir * naux


def work(case):
    kind = case["kind"]
    if kind == "energy":
        no, nv, na = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": na * no * nv * (4.0 if case["store"] == "f32" else 8.0),
                "flops": _pairs(no, nv, na)}
    if kind == "job":
        no, nv, na = case["nocc"], case["nvir"], case["naux"]
        n = no + nv
        return {"bytes": 8.0 * (na * n * n + n * n + na * na + na * no * nv),
                "flops": 2.0 * na * n * n * no + 2.0 * na * n * no * nv
                + 2.0 * na * na * no * nv + _pairs(no, nv, na)}
    if kind == "gradient":
        # the forward energy, then the adjoint: its amplitudes once more (none are kept between
        # the two calls) and two updates of Gamma per pair
        no, nv, na = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": 8.0 * 2 * na * no * nv, "flops": 4.0 * _pairs(no, nv, na)}
    if kind == "density":
        no, nv, na = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": 8.0 * (na * no * nv + no * no + nv * nv),
                "flops": _pairs(no, nv, na) + float(no) * no * nv ** 3 + float(no) ** 3 * nv * nv}
    if kind == "ump2":
        a, b, va, vb, na = (case[k] for k in ("nocc_a", "nocc_b", "nvir_a", "nvir_b", "naux"))
        return {"bytes": 8.0 * na * (a * va + b * vb),
                "flops": _pairs(a, va, na) + _pairs(b, vb, na) + 2.0 * a * b * va * vb * na}
    if kind == "dlpno":
        no, nv = case["nocc"], case["nvir"]
        na = no * case["per_site"]
        return {"bytes": 8.0 * (na * no * nv + 2 * no * no), "flops": _pairs(no, nv, na)}
    if kind == "domains":
        nocc, nvir, naux, _, _ = _shapes(case)
        return {"bytes": 8.0 * float((nocc * nvir * naux).sum()),
                "flops": float((nocc * (nocc + 1.0) * nvir ** 2 * naux).sum())}
    no, nv, per = case["nocc"], case["nvir"], case["per_site"]
    w = 2 * case["radius"] / 2.5
    pairs = no * (no + 1) / 2
    flops = 0.0
    for k in range(no):  # the no - k pairs k sites apart
        d = min(no, w + min(k, w)) * per
        flops += (no - k) * (d ** 3 / 3 + 2.0 * d * d * nv + 2.0 * d * nv * nv)
    return {"bytes": 8.0 * (no * per * no * nv + (no * per) ** 2 + pairs * nv * nv),
            "flops": flops}


# ---- the same results in plain torch or numpy, 64 bits -------------------------------------------------


def _blocks(b, nocc, nvir):
    return b.double().reshape(b.shape[0], nocc, nvir).permute(1, 0, 2).contiguous()


def _denominators(eps, nocc, nvir, frozen=0):
    e = torch.as_tensor(eps, device=DEV, dtype=torch.float64)
    return e[frozen:frozen + nocc], e[frozen + nocc:frozen + nocc + nvir]


def _row(bi, i, ei, ev):
    """g and D of the pairs (i, j >= i)."""
    n, naux, nvir = bi.shape
    g = (bi[i].t().contiguous() @ bi[i:].permute(1, 0, 2).reshape(naux, -1))
    g = g.reshape(nvir, n - i, nvir).permute(1, 0, 2).contiguous()
    d = (ei[i] + ei[i:])[:, None, None] - ev[None, :, None] - ev[None, None, :]
    return g, d


def _energy_exact(b, eps, nocc, nvir, frozen=0, kappa=0.0, matrix=False):
    bi = _blocks(b, nocc, nvir)
    ei, ev = _denominators(eps, nocc, nvir, frozen)
    e_os = e_ss = torch.zeros((), dtype=torch.float64, device=DEV)
    p_os, p_ss = torch.zeros(2, nocc, nocc, dtype=torch.float64, device=DEV)
    for i in range(nocc):
        g, d = _row(bi, i, ei, ev)
        w = 1.0 / d
        if kappa:
            w = w * (1.0 - torch.exp(kappa * d)) ** 2
        f = torch.full((nocc - i,), 2.0, dtype=torch.float64, device=DEV)
        f[0] = 1.0
        o = f * (g * g * w).sum((1, 2))
        s = f * (g * (g - g.transpose(1, 2)) * w).sum((1, 2))
        e_os, e_ss = e_os + o.sum(), e_ss + s.sum()
        p_os[i, i:] = p_os[i:, i] = o
        p_ss[i, i:] = p_ss[i:, i] = s
    return (e_os, e_ss, p_os, p_ss) if matrix else (e_os, e_ss)


def _amplitudes(b, eps, nocc, nvir, frozen=0):
    bi = _blocks(b, nocc, nvir)
    ei, ev = _denominators(eps, nocc, nvir, frozen)
    t = torch.empty(nocc, nocc, nvir, nvir, dtype=torch.float64, device=DEV)
    for i in range(nocc):
        g, d = _row(bi, i, ei, ev)
        g = g / d
        t[i, i:] = g
        t[i:, i] = g.transpose(1, 2)
    return bi, t


def _gradient_exact(b, eps, nocc, nvir, frozen, c_os, c_ss):
    bi = _blocks(b, nocc, nvir)
    ei, ev = _denominators(eps, nocc, nvir, frozen)
    naux = bi.shape[1]
    gam = torch.zeros_like(bi)
    d_occ, d_vir = torch.zeros_like(ei), torch.zeros_like(ev)
    e_os = e_ss = torch.zeros((), dtype=torch.float64, device=DEV)
    flat = bi.permute(1, 0, 2).reshape(naux, nocc * nvir)
    for i in range(nocc):
        g = (bi[i].t().contiguous() @ flat).reshape(nvir, nocc, nvir).permute(1, 0, 2).contiguous()
        d = (ei[i] + ei)[:, None, None] - ev[None, :, None] - ev[None, None, :]
        t = g / d
        x = t.transpose(1, 2)
        tt = (c_os + c_ss) * t - c_ss * x
        e_os, e_ss = e_os + (g * t).sum(), e_ss + (g * (t - x)).sum()
        gam[i] = 4.0 * flat @ tt.permute(0, 2, 1).reshape(nocc * nvir, nvir)
        # E = sum_ij sum_ab g (t~): dE/deps_p = -sum t t~ dD/deps_p; each pair holds i and j
        q = t * tt
        d_occ[i] -= 2.0 * q.sum()
        d_vir += 2.0 * q.sum((0, 1))
    grad = gam.permute(1, 0, 2).reshape(naux, nocc * nvir)
    de = torch.cat([torch.zeros(frozen, dtype=torch.float64, device=DEV), d_occ, d_vir])
    return e_os, e_ss, grad, de


def _same_spin(ch):
    bi = _blocks(ch.b, ch.nocc, ch.nvir)
    ei, ev = _denominators(ch.eps, ch.nocc, ch.nvir)
    e = torch.zeros((), dtype=torch.float64, device=DEV)
    for i in range(ch.nocc):
        g, d = _row(bi, i, ei, ev)
        e = e + 0.5 * ((g - g.transpose(1, 2)) ** 2 / d).sum()  # i = j is antisymmetrised to ...
        e = e - 0.25 * ((g[0] - g[0].t()) ** 2 / d[0]).sum()    # ... half the weight
    return e


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "energy":
        o, e = _energy_exact(s["b"], s["eps"], case["nocc"], case["nvir"], case["frozen"],
                             case["kappa"])
        return o, e, o + e
    if kind == "job":
        no, nv, na = case["nocc"], case["nvir"], case["naux"]
        n = no + nv
        half = (s["j3"].reshape(na * n, n) @ s["c_occ"]).reshape(na, n, no)
        mo = torch.stack([h.t().contiguous() @ s["c_vir"] for h in half])
        b = s["m"] @ mo.reshape(na, no * nv)
        o, e = _energy_exact(b, s["eps"], no, nv)
        return {"b": b, "e": [o, e, o + e]}
    if kind == "gradient":
        o, e, g, d = _gradient_exact(s["b"], s["eps"], case["nocc"], case["nvir"], case["frozen"],
                                     1.2, 1.0 / 3.0)
        return {"e": [o, e], "b": g, "eps": d}
    if kind == "density":
        no, nv = case["nocc"], case["nvir"]
        o, e = _energy_exact(s["b"], s["eps"], no, nv)
        _, t = _amplitudes(s["b"], s["eps"], no, nv)
        tt = 2.0 * t - t.transpose(2, 3)
        # P_ij = -sum_k,ab t_ik t~_jk; P_ab = sum_ij,c t_ij^ac t~_ij^bc
        oo = -t.reshape(no, -1) @ tt.reshape(no, -1).t().contiguous()
        vv = torch.zeros(nv, nv, dtype=torch.float64, device=DEV)
        for i in range(no):
            vv += (t[i].permute(1, 0, 2).reshape(nv, -1)
                   @ tt[i].permute(1, 0, 2).reshape(nv, -1).t().contiguous())
        return {"e": [o, e], "oo": oo, "vv": vv}
    if kind == "ump2":
        a, b = s["a"], s["b"]
        ba, bb = _blocks(a.b, a.nocc, a.nvir), _blocks(b.b, b.nocc, b.nvir)
        ea, va = _denominators(a.eps, a.nocc, a.nvir)
        eb, vb = _denominators(b.eps, b.nocc, b.nvir)
        flat = bb.permute(1, 0, 2).reshape(ba.shape[1], -1)
        os = torch.zeros((), dtype=torch.float64, device=DEV)
        for i in range(a.nocc):
            g = (ba[i].t().contiguous() @ flat).reshape(a.nvir, b.nocc, b.nvir)
            os = os + (g * g / (ea[i] + eb[None, :, None] - va[:, None, None]
                                - vb[None, None, :])).sum()
        return _same_spin(a), _same_spin(b), os
    if kind == "dlpno":
        no, nv = case["nocc"], case["nvir"]
        _, _, os, ss = _energy_exact(s["b"], s["eps"], no, nv, matrix=True)
        keep = (os + ss).abs().triu() >= 1e-5
        keep.fill_diagonal_(True)
        return {"os": os, "ss": ss, "e": [os[keep].sum(), ss[keep].sum()], "n": int(keep.sum())}
    if kind == "domains":
        os, ss = [], []
        for no, nv, na, bo, eo in zip(*(v.tolist() for v in s["shapes"])):
            b = s["b"][bo:bo + na * no * nv].reshape(na, no * nv)
            o, e = _energy_exact(b, s["eps"][eo:eo + no + nv], no, nv)
            os.append(o)
            ss.append(e)
        return torch.stack(os), torch.stack(ss)
    no, nv = case["nocc"], case["nvir"]
    a, v, x, c = s["a"].cpu().numpy(), s["v"].cpu().numpy(), s["xyz"], s["centers"]
    ei, ev = (t.cpu().numpy() for t in _denominators(s["eps"], no, nv))
    near = ((x[:, None, :] - c[None, :, :]) ** 2).sum(-1) <= case["radius"] ** 2
    j, os, ss, dmax = [], [], [], 0
    for i, k in s["pairs"]:
        d = np.flatnonzero(near[:, i] | near[:, k])
        dmax = max(dmax, d.size)
        ai, aj = a[d, i * nv:(i + 1) * nv], a[d, k * nv:(k + 1) * nv]
        g = ai.T @ np.linalg.solve(v[np.ix_(d, d)], aj)
        den = ei[i] + ei[k] - ev[:, None] - ev[None, :]
        f = 1.0 if i == k else 2.0
        j.append(g)
        os.append(f * (g * g / den).sum())
        ss.append(f * (g * (g - g.T) / den).sum())
    return {"j": np.stack(j), "dmax": dmax, "os": np.array(os), "ss": np.array(ss)}
