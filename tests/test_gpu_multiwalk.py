"""MultiWalk dispatch and retrieve (list and index form, quadrupole and monopole) with ragged walks,
enough of them that each split of a workgroup over i-lanes (2 to 64) is taken: walk by walk
against the oracle, the neighbour data equal to its FP32 kernel's, the sums within rounding of its
FP64 ones.  Walks of one i-particle, of none, of a workgroup's and one more or less; EP or SP
lists that are empty, longer than a tile, or both empty; nodes with second moments.

Tolerance as for the functors (the same pairs, quads and FP64 sums): 48 2^-24 of the sum of the term
sizes of both lists.  A walk by itself takes another split than among others: FP64 roundings and
one unit in the last place."""
import ctypes

import numpy as np
import pytest

from gplum_amd import abi, gpu

pytestmark = pytest.mark.gpu

EPS2 = np.float32(1e-10)
N_EPJ, N_SPJ = 5000, 3000
# i-lanes: number of walks, their i-particles (from, to)
SPLITS = {2: (5, 20, 130), 4: (24, 85, 120), 8: (40, 98, 125), 16: (150, 100, 125), 32: (270, 66, 126), 64: (540, 3, 120)}


def i_lanes(n_epi, n_list):
    """The rule of the split: the most i-lanes that leave each list's quads a j-lane, or enough
    workgroups of 2 i-particles per i-lane."""
    for li in (64, 32, 16, 8, 4):
        groups = sum(-(-n // (2 * li)) for n in n_epi)
        if li * (sum(n_list) // len(n_list)) <= 2048 or groups >= (240 if li <= 8 else 500):
            return li
    return 2


def world(rng, quad):
    epj = np.zeros(N_EPJ, dtype=abi.EPJ)
    epj["id_local"] = epj["id"] = np.arange(N_EPJ)
    epj["pos"] = np.array([1.0, 0.2, 0.01]) + rng.normal(0, 2e-3, (N_EPJ, 3))
    epj["r_out"] = rng.uniform(1e-4, 3e-4, N_EPJ)
    epj["r_search"] = 2.5 * epj["r_out"]
    epj["mass"] = rng.uniform(0.5e-12, 2e-12, N_EPJ)
    spj = np.zeros(N_SPJ, dtype=abi.SPJ_QUAD if quad else abi.SPJ_MONO)
    spj["pos"] = np.array([1.0, 0.2, 0.01]) + rng.choice([-1.0, 1.0], (N_SPJ, 3)) * rng.uniform(0.02, 0.05, (N_SPJ, 3))
    spj["mass"] = rng.uniform(0.5e-11, 2e-11, N_SPJ)
    if quad:
        spj["quad"] = spj["mass"][:, None] * rng.uniform(-1e-5, 1e-5, (N_SPJ, 6))
    return epj, spj


def walks(rng, lanes, epj):
    """(i-particles, EP indices, SP indices) per walk."""
    n_walk, lo, hi = SPLITS[lanes]
    out = []
    for w in range(n_walk):
        ni, nj, ns = int(rng.integers(lo, hi + 1)), int(rng.integers(470, 760)), int(rng.integers(300, 560))
        if w < 3:
            ni = 2 * lanes + w - 1                       # a workgroup's i-particles, one less and one more
        ni, nj, ns = {3: (1, nj, ns), 4: (ni, 0, ns)}.get(w, (ni, nj, ns))
        if n_walk > 20:
            ni, nj, ns = {5: (ni, nj, 0), 6: (ni, 0, 0), 7: (0, nj, ns), 8: (ni, 3, 1), 9: (ni, 512, 513)}.get(w, (ni, nj, ns))
        idj = rng.choice(N_EPJ, nj, replace=False).astype(np.int32)
        epi = np.zeros(ni, dtype=abi.EPI)
        # i-particles: some of the EP list and some that are not in it
        src = epj[np.concatenate([idj[:ni // 2], rng.choice(N_EPJ, ni - len(idj[:ni // 2]), replace=False)]).astype(int)]
        for k in ("id_local", "pos", "r_out", "r_search"):
            epi[k] = src[k]
        out.append((epi, idj, rng.choice(N_SPJ, ns, replace=False).astype(np.int32)))
    return out


def table(arrays):
    return (ctypes.c_void_p * len(arrays))(*[a.ctypes.data for a in arrays])


def counts(arrays):
    return (ctypes.c_int * len(arrays))(*[len(a) for a in arrays])


def dispatch(form, quad, ww, epj, spj, tag=0):
    L, mono, nw = gpu.lib(), "" if quad else "_mono", len(ww)
    epi = [w[0] for w in ww]
    force = [abi.cleared_force(len(e)) for e in epi]
    if form == "index":
        j, s = [w[1] for w in ww], [w[2] for w in ww]
        gpu.check(getattr(L, "gplum_multiwalk_dispatch_index" + mono)(
            tag, nw, table(epi), counts(epi), table(j), counts(j), table(s), counts(s), abi.ptr(epj), len(epj), abi.ptr(spj),
            len(spj), 1))
    else:
        j, s = [np.ascontiguousarray(epj[w[1]]) for w in ww], [np.ascontiguousarray(spj[w[2]]) for w in ww]
        gpu.check(getattr(L, "gplum_multiwalk_dispatch" + mono)(tag, nw, table(epi), counts(epi), table(j), counts(j), table(s),
                                                              counts(s)))
    gpu.check(L.gplum_multiwalk_retrieve(tag, nw, counts(epi), table(force)))
    return force


def sizes(x, pos, mass, clamp=None):
    r2 = ((x[:, None] - pos[None]) ** 2).sum(2) + float(EPS2)
    if clamp is not None:
        r2 = np.maximum(r2, clamp)
    return (mass / r2).sum(1), (mass / np.sqrt(r2)).sum(1)


@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("form", ["list", "index"])
@pytest.mark.parametrize("lanes", sorted(SPLITS))
def test_walks_match_oracle(oracle_lib, lanes, form, quad):
    rng = np.random.default_rng([lanes, quad])
    epj, spj = world(rng, quad)
    ww = walks(rng, lanes, epj)
    assert i_lanes([len(w[0]) for w in ww], [len(w[1]) + len(w[2]) for w in ww]) == lanes
    print("%d walks, %d i-particles" % (len(ww), sum(len(w[0]) for w in ww)), flush=True)
    L = gpu.lib()
    L.gplum_multiwalk_set_eps2.argtypes = [ctypes.c_float]
    gpu.check(L.gplum_multiwalk_set_eps2(EPS2))
    try:
        force = dispatch(form, quad, ww, epj, spj)
        alone = [dispatch(form, quad, [w], epj, spj, tag=1)[0] for w in ww[:5]]
    finally:
        gpu.check(L.gplum_multiwalk_set_eps2(0.0))
    sp64 = oracle_lib.epsp_quad_f64 if quad else oracle_lib.epsp_mono_f64
    tol, worst = 48 * 2.0 ** -24, 0.0
    for k, ((epi, idj, ids), f) in enumerate(zip(ww, force)):
        if len(epi) == 0:
            continue
        j, s = np.ascontiguousarray(epj[idj]), np.ascontiguousarray(spj[ids])
        ref = abi.cleared_force(len(epi))
        oracle_lib.epep_f32(epi, j, ref, EPS2)
        assert np.array_equal(f["neighbor"], ref["neighbor"]), k
        a, p = oracle_lib.epep_f64(epi, j, EPS2)
        b, q = sp64(epi, s, EPS2)
        ja, jp = sizes(epi["pos"], j["pos"], j["mass"], np.maximum(epi["r_out"][:, None], j["r_out"][None]) ** 2)
        sa, sp = sizes(epi["pos"], s["pos"], s["mass"])
        ea, ep = np.abs(f["acc"] - (a + b)).max(1), np.abs(f["phi"] - (p + q))
        assert np.all(ea <= tol * (ja + sa)) and np.all(ep <= tol * (jp + sp)), k
        if len(idj) + len(ids):
            worst = max(worst, (ea / (ja + sa)).max(), (ep / (jp + sp)).max())
        if k < len(alone):
            assert np.array_equal(alone[k]["neighbor"], f["neighbor"])
            for name, most in (("acc", ja + sa), ("phi", jp + sp)):
                most = 2.0 ** -49 * (most[:, None] if name == "acc" else most)
                last = np.spacing(np.maximum(np.abs(f[name]), np.abs(alone[k][name])))
                assert np.all(np.abs(f[name].astype(np.float64) - alone[k][name]) <= last + most)
    print("largest error: %.2f 2^-24 of the term sizes" % (worst * 2.0 ** 24))
