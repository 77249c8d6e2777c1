"""The FP32 functors at the edges of their kernel: the i-counts where the number of i-lanes per
wave changes (1912/1913 ... 63872/63873) and the smallest, the j-counts where it does (32/33 ...
512/513), j-counts around a tile (512) and its remainders, an i-array that is accumulated into,
against the FP64 sums.

Tolerance, in units of u = 2^-24: a coordinate difference carries 3 (difference of the high parts, of
the low parts, their sum), |r|^2 6 and three for its sums, 1/r half of that and at most 2 of its own (a
Newton step on the hardware estimate), its cube three times 6.5 and 2, the mass 1, the products 3, the
component 3 again: 29.  The four pairs of a quad are added in FP32: 3; the quads in FP64, rounded once
at the end: |error| <= 33 u sum_j |term_j|, 48 u with a margin for the second order, the moments' own
roundings and the value accumulated into.  Neighbour numbers and ids are whole numbers and equal to
the oracle's."""
import numpy as np
import pytest

from gplum_amd import abi, gpu

pytestmark = pytest.mark.gpu

TOL = 48 * 2.0 ** -24
EPS2 = np.float32(1e-10)


def scales(epi, pos, mass, r_out=None):
    """Per i: sum_j m / r^2 and sum_j m / r (r clamped at r_out for EP-EP)."""
    a, p = np.zeros(len(epi)), np.zeros(len(epi))
    for k in range(len(pos)):
        r2 = ((epi["pos"] - pos[k]) ** 2).sum(1) + EPS2
        if r_out is not None:
            r2 = np.maximum(r2, np.maximum(epi["r_out"], r_out[k]) ** 2)
        a += mass[k] / r2
        p += mass[k] / np.sqrt(r2)
    return a, p


def check(force, start, a64, p64, sa, sp):
    err_a = np.abs(force["acc"].astype(np.float64) - start["acc"] - a64).max(1)
    err_p = np.abs(force["phi"].astype(np.float64) - start["phi"] - p64)
    assert np.all(err_a <= TOL * (sa + np.abs(start["acc"]).max(1)))
    assert np.all(err_p <= TOL * (sp + np.abs(start["phi"])))


@pytest.mark.parametrize("ni,nj", [(1, 0), (1, 513), (3, 1), (4, 255), (5, 511), (9, 512), (130, 1025), (1912, 1029),
                                   (1913, 1029), (3824, 300), (3825, 300), (15968, 130), (15969, 600), (31936, 70),
                                   (31937, 70), (63872, 65), (63873, 65), (41, 4), (129, 32), (129, 33), (65, 64), (65, 65),
                                   (33, 128), (33, 129), (17, 256), (17, 257), (9, 513)])
def test_functors_at_kernel_edges(oracle_lib, ni, nj):
    rng = np.random.default_rng(ni + nj)
    n = max(ni, nj)
    pos = np.array([1.0, 0.2, 0.01]) + rng.normal(0, 2e-3, (n, 3))
    epi, epj = np.zeros(ni, dtype=abi.EPI), np.zeros(nj, dtype=abi.EPJ)
    for a in (epi, epj):
        a["pos"] = pos[:len(a)]
        a["id_local"] = np.arange(len(a))
        a["r_out"] = rng.uniform(1e-4, 3e-4, n)[:len(a)]
        a["r_search"] = 2.5 * a["r_out"]
    epj["mass"] = rng.uniform(0.5e-12, 2e-12, nj)
    start = abi.cleared_force(ni)
    start["acc"] = rng.normal(0, 1e-9, (ni, 3))
    print("EP-EP", ni, nj, flush=True)
    f_gpu, f_orc = start.copy(), start.copy()
    gpu.calc_force_epep(epi, epj, f_gpu, EPS2)
    oracle_lib.epep_f32(epi, epj, f_orc, EPS2)
    assert np.array_equal(f_gpu["neighbor"], f_orc["neighbor"])
    a64, p64 = oracle_lib.epep_f64(epi, epj, EPS2)
    check(f_gpu, start, a64, p64, *scales(epi, epj["pos"], epj["mass"], epj["r_out"]))
    # super-particles a few hundredths away, of extent 1e-3
    far = np.array([1.0, 0.2, 0.01]) + rng.choice([-1.0, 1.0], (nj, 3)) * rng.uniform(0.02, 0.05, (nj, 3))
    for dt, name in ((abi.SPJ_QUAD, "quad"), (abi.SPJ_MONO, "mono")):
        print("EP-SP", name, ni, nj, flush=True)
        spj = np.zeros(nj, dtype=dt)
        spj["pos"] = far
        spj["mass"] = rng.uniform(0.5e-11, 2e-11, nj)
        if name == "quad":
            spj["quad"] = spj["mass"][:, None] * rng.uniform(-1e-6, 1e-6, (nj, 6))
        f = start.copy()
        getattr(gpu, "calc_force_epsp_" + name)(epi, spj, f, EPS2)
        a64, p64 = getattr(oracle_lib, "epsp_%s_f64" % name)(epi, spj, EPS2)
        check(f, start, a64, p64, *scales(epi, far, spj["mass"]))
        assert np.array_equal(f["neighbor"], start["neighbor"])
