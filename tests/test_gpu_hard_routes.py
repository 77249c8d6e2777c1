"""Clusters of 2 to 4 bodies whose steps are not powers of two, under a dt_tree and dt_min that
are: the lane-per-term path takes them, not the LDS path that large clusters need.  The results of
both are the same bits, so the path shows in the time: about 0.5 of the LDS path's on one
cluster (a chain of block steps; the launch is a small part of it), the same where the LDS path
is taken; 0.75 lies between.  And batches that mix such clusters with others, through each entry
point, against the oracle bit for bit."""
import numpy as np
import pytest

from gplum_amd import gpu, ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 4])
def test_steps_off_the_grid_keep_the_lane_per_term_path(oracle_lib, n):
    # small step criteria: a chain of hundreds of block steps
    kw = dict(eta=0.0005, eta_sun=0.0005, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -4, dt_min=2.0 ** -24, gamma=0.1)
    p = gpu.params(**kw)
    pp, off = ic.clusters(1, seed=5, size_min=n, size_max=n, m_hi=1e-9)
    ic.cluster_acc0(pp, off)
    oracle_lib.cluster_prepare(oracle_lib.params(**kw), pp, off)
    pp["dt"] = 0.75 * 2.0 ** -11
    best, out, steps = {}, {}, 0
    for lds in (False, True):
        best[lds] = np.inf
        for _ in range(5):
            got = pp.copy()
            _, steps, ms = gpu.hard_integrate(p, got, off, lane_per_particle=lds)
            best[lds] = min(best[lds], ms)
        out[lds] = got.tobytes()
    print("%d bodies, %d block steps: %.3f us per step, LDS path %.3f" % (n, steps, 1e3 * best[False] / steps,
                                                                         1e3 * best[True] / steps))
    assert out[False] == out[True]
    assert steps > 100
    assert best[False] < 0.75 * best[True]


@pytest.mark.parametrize("mode", ["batch", "per cluster", "graph"])
def test_mixed_steps_match_oracle(oracle_lib, mode):
    kw = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -4, dt_min=2.0 ** -13, gamma=0.1,
              collision=1)
    parts, off = [], [0]
    for k, n in enumerate((2, 3, 4, 5, 17, 33, 1) * 4):
        pp, _ = ic.clusters(1, seed=[91, k], size_min=n, size_max=n, m_hi=1e-8)
        if n > 1:
            ic.cluster_acc0(pp, [0, n])
        pp["id"] += off[-1]
        pp["f"] = 100.0
        parts.append(pp)
        off.append(off[-1] + n)
    pp, off = np.concatenate(parts), np.array(off)
    oracle_lib.cluster_prepare(oracle_lib.params(**kw), pp, off)
    for a, b in zip(off[:-1:2], off[1::2]):          # every other cluster, one of its members
        pp["dt"][a + (b - a) // 2] *= 0.75
    ref, got = pp.copy(), pp.copy()
    nc, ed, steps = oracle_lib.hermite_clusters(oracle_lib.params(**kw), ref, off)
    if mode == "graph":
        ed_g, steps_g, _, mismatches = gpu.hard_integrate_graph(gpu.params(**kw), got, off, replays=3)
        assert mismatches == 0
    else:
        ed_g, steps_g, _ = gpu.hard_integrate(gpu.params(**kw), got, off, persistent=mode == "batch")
    print("%s: %d block steps (oracle %d), %d collisions" % (mode, steps_g, steps, nc))
    fields = ("pos", "vel", "acc_d", "jerk_d", "acc_s", "jerk_s", "phi_s", "mass", "r_planet", "dt", "time", "id", "flags")
    assert [f for f in fields if got[f].tobytes() != ref[f].tobytes()] == []
    assert steps_g == steps and ed_g == ed and nc > 0
