"""The FP32 functors where they change to one i-particle per lane (1500 (entries + 16) i-particles),
and the split of their work over lanes: neighbour data equal to the oracle's FP32 kernel, sums within
rounding of the FP64 ones, and the same values however the work is split.

Tolerances, in units of u = 2^-24, from the operations of a pair.  A coordinate difference carries 3
(the difference of the high parts, of the low parts, their sum), so |r|^2 6 and three more for its
sums, 1/r half of that and at most 2 of its own (a Newton step on the hardware estimate, with the
residual exact), its cube three times 6.5 and 2, the mass 1, the products 3, the component 3 again: 29.  The four
pairs of a quad add 3; quads are added in FP64 and the result is rounded once: at most 33 for each
pair's size, 48 with a margin for the second order and the EP-SP moments' own roundings.  Two splits
of the same list differ by FP64 roundings (2^-49 of the largest possible sum covers 203 terms) before
the last one to FP32: at most that and one unit in the last place."""
import ctypes

import numpy as np
import pytest

from gplum_amd import abi, gpu

pytestmark = pytest.mark.gpu

EPS2 = np.float32(1e-10)


def lists(ni, nj):
    rng = np.random.default_rng([ni, nj])
    n = max(ni, nj)
    pos = np.array([1.0, 0.2, 0.01]) + rng.normal(0, 2e-3, (n, 3))
    epi, epj = np.zeros(ni, dtype=abi.EPI), np.zeros(nj, dtype=abi.EPJ)
    for a in (epi, epj):
        a["pos"] = pos[:len(a)]
        a["id_local"] = np.arange(len(a))
        a["r_out"] = rng.uniform(1e-4, 3e-4, n)[:len(a)]
        a["r_search"] = 2.5 * a["r_out"]
    epj["mass"] = rng.uniform(0.5e-12, 2e-12, nj)
    spj = np.zeros(nj, dtype=abi.SPJ_QUAD)
    spj["pos"] = np.array([1.0, 0.2, 0.01]) + rng.choice([-1.0, 1.0], (nj, 3)) * rng.uniform(0.02, 0.05, (nj, 3))
    spj["mass"] = rng.uniform(0.5e-11, 2e-11, nj)
    spj["quad"] = spj["mass"][:, None] * rng.uniform(-1e-6, 1e-6, (nj, 6))
    return epi, epj, spj


def close(force, a64, p64, epi, pos, mass, r_out=0.0):
    d2 = ((epi["pos"][:, None] - pos[None]) ** 2).sum(2) + float(EPS2)
    if np.ndim(r_out):
        d2 = np.maximum(d2, np.maximum(epi["r_out"][:, None], r_out[None]) ** 2)
    tol = 48 * 2.0 ** -24
    assert np.all(np.abs(force["acc"] - a64).max(1) <= tol * (mass / d2).sum(1))
    assert np.all(np.abs(force["phi"] - p64) <= tol * (mass / np.sqrt(d2)).sum(1))


@pytest.mark.parametrize("ni,nj", [(24000, 0), (25499, 1), (25500, 1), (30000, 4), (30001, 4), (36255, 8), (70499, 31), (70500, 31),
                                   (120001, 63), (420000, 263), (1048576, 3)])
def test_wide_rule_edges(oracle_lib, ni, nj):
    epi, epj, spj = lists(ni, nj)
    print("EP-EP", ni, nj, flush=True)
    f, ref = abi.cleared_force(ni), abi.cleared_force(ni)
    gpu.calc_force_epep(epi, epj, f, EPS2)
    oracle_lib.epep_f32(epi, epj, ref, EPS2)
    assert np.array_equal(f["neighbor"], ref["neighbor"])
    a64, p64 = oracle_lib.epep_f64(epi, epj, EPS2)
    part = slice(max(0, ni - 20000), ni)                 # (the sizes of all terms would be large arrays)
    close(f[part], a64[part], p64[part], epi[part], epj["pos"], epj["mass"], epj["r_out"])
    print("EP-SP", ni, nj, flush=True)
    q = abi.cleared_force(ni)
    gpu.calc_force_epsp_quad(epi, spj, q, EPS2)
    a64, p64 = oracle_lib.epsp_quad_f64(epi, spj, EPS2)
    close(q[part], a64[part], p64[part], epi[part], spj["pos"], spj["mass"])


def test_same_values_however_split():
    # 1048576 to 1 i-particles against the same list (all relative to the first): other numbers of
    # i-lanes and j-lanes, and with 1048576 one i-particle per lane and no j-lanes
    epi, epj, spj = lists(1048576, 203)
    want = None
    for ni in (1048576, 70000, 20000, 9000, 4500, 2100, 1000, 300, 7, 1):
        out = []
        for call, j in ((gpu.calc_force_epep, epj), (gpu.calc_force_epsp_quad, spj)):
            f = abi.cleared_force(ni)
            call(epi[:ni], j, f, EPS2)
            out.append(f)
        if want is None:
            want = out
        for f, w in zip(out, want):
            assert np.array_equal(f["neighbor"], w["neighbor"][:ni])
            worst = 0.0
            for k in ("acc", "phi"):
                a, b = f[k], w[k][:ni]
                most = 2.0 ** -49 * (epj["mass"].sum() + spj["mass"].sum()) / 1e-8      # no pair is nearer than 1e-4
                last = np.spacing(np.maximum(np.abs(a), np.abs(b)))
                worst = max(worst, ((np.abs(a.astype(np.float64) - b) - most) / last).max())
            print("%d i-particles: %.2f units in the last place" % (ni, worst))
            assert worst <= 1.0


def test_many_particles_against_one_entry_cost_their_bytes():
    # such a call reads the i-particles and reads and writes the forces, 112 bytes per i-particle; plain
    # copies of both arrays move 160.  Half as long again as the copies leaves room for what a kernel
    # needs beside its bytes; sums over lanes that hold no entry took nearly three times as long
    ni = 1048576
    epi, epj, _ = lists(ni, 1)
    gpu.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")               # the runtime that the library is linked with
    vp, bufs = ctypes.c_void_p, []

    def device(nbytes, src=None):
        p = vp()
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
        bufs.append(p)
        if src is not None:
            assert hip.hipMemcpy(p, vp(src.ctypes.data), ctypes.c_size_t(nbytes), 1) == 0
        return p
    force_h = abi.cleared_force(ni)
    e, j, f = (device(a.nbytes, a) for a in (epi, epj, force_h))
    e2, f2 = device(epi.nbytes), device(force_h.nbytes)
    t0, t1 = vp(), vp()
    assert hip.hipEventCreate(ctypes.byref(t0)) == 0 and hip.hipEventCreate(ctypes.byref(t1)) == 0

    def force():
        gpu.check(gpu.lib().gplum_calc_force_epep_noalloc(e, ni, j, 1, f, EPS2, None))

    def copies():
        for dst, src, n in ((e2, e, epi.nbytes), (f2, f, force_h.nbytes)):
            assert hip.hipMemcpyAsync(dst, src, ctypes.c_size_t(n), 3, None) == 0
    best = {}
    for fn in (force, copies, force, copies):
        for _ in range(5):
            fn()
            assert hip.hipEventRecord(t0, None) == 0
            for _ in range(20):
                fn()
            assert hip.hipEventRecord(t1, None) == 0 and hip.hipEventSynchronize(t1) == 0
            ms = ctypes.c_float()
            assert hip.hipEventElapsedTime(ctypes.byref(ms), t0, t1) == 0
            best[fn] = min(best.get(fn, np.inf), ms.value / 20)
    print("1048576 x 1: %.1f us, copies %.1f us" % (1e3 * best[force], 1e3 * best[copies]))
    for p in bufs:
        assert hip.hipFree(p) == 0
    assert best[force] < 1.5 * best[copies]
