"""The size classes of the batched Hermite against the oracle, bit for bit, at the edges of
each class: one wave (up to 16 members; 2 to 4 on the lane-per-term path until a merger), 256
threads (up to 32), 512 threads (up to 64, the last size whose hard forces are summed
sequentially), 512 threads with a wave per body (up to 256) and the global-memory path.
Both sides use the same operations in the same order, so no difference is allowed."""
import numpy as np
import pytest

from gplum_amd import gpu, ic

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "acc_d", "jerk_d", "acc_s", "jerk_s", "phi_s", "mass", "r_planet", "dt", "time", "id", "flags")


def clusters_of(sizes, seed, m_hi, f):
    parts, off = [], [0]
    for k, n in enumerate(sizes):
        pp, _ = ic.clusters(1, seed=[seed, k], size_min=n, size_max=n, m_hi=m_hi)
        if n > 1:
            ic.cluster_acc0(pp, [0, n])
        pp["id"] += off[-1]
        pp["f"] = f
        parts.append(pp)
        off.append(off[-1] + n)
    return np.concatenate(parts), np.array(off)


@pytest.mark.parametrize("merging", [False, True])
@pytest.mark.parametrize("sizes", [(1, 2, 3, 4, 5, 6, 7, 8, 9, 15, 16, 17), (16, 17, 18, 31, 32, 33, 34),
                                   (63, 64, 65, 66, 100), (127, 128, 129, 130), (192, 193, 255, 256, 257)])
def test_size_classes_match_oracle(oracle_lib, sizes, merging):
    # a coarse smallest step bounds the oracle's time on the large clusters
    kw = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -4, dt_min=2.0 ** -13, gamma=0.1,
              collision=int(merging))
    pp, off = clusters_of(sizes, 41 + int(merging), 1e-8 if merging else 1e-9, 100.0 if merging else 1.0)
    oracle_lib.cluster_prepare(oracle_lib.params(**kw), pp, off)
    ref, got = pp.copy(), pp.copy()
    nc, ed, steps = oracle_lib.hermite_clusters(oracle_lib.params(**kw), ref, off)
    ed_g, steps_g, ms = gpu.hard_integrate(gpu.params(**kw), got, off)
    print("sizes %s: %d block steps (oracle %d), %d collisions, %.2f ms" % (sizes, steps_g, steps, nc, ms))
    bad = [(n, f) for n, a, b in zip(sizes, off[:-1], off[1:]) for f in FIELDS
           if got[f][a:b].tobytes() != ref[f][a:b].tobytes()]
    assert bad == []
    assert steps_g == steps and ed_g == ed
    assert np.allclose(got["phi_d"], ref["phi_d"], rtol=1e-13, atol=0.0)
    assert not merging or nc > 0


@pytest.mark.parametrize("merging", [False, True])
@pytest.mark.parametrize("dt_tree,dt_scale", [(2.0 ** -4, 1.0), (2.0 ** -4, 0.75), (3 * 2.0 ** -6, 1.0), (3 * 2.0 ** -6, 2.0 / 3)])
def test_step_grids_match_oracle(oracle_lib, dt_tree, dt_scale, merging):
    # steps that are powers of two and steps that are not (of a dt_tree that is none, or given)
    kw = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=dt_tree, dt_min=dt_tree * 2.0 ** -9, gamma=0.1,
              collision=int(merging))
    pp, off = clusters_of((2, 3, 4, 5) * 8, 57, 1e-8 if merging else 1e-9, 100.0 if merging else 1.0)
    oracle_lib.cluster_prepare(oracle_lib.params(**kw), pp, off)
    pp["dt"] *= dt_scale
    ref, got = pp.copy(), pp.copy()
    nc, ed, steps = oracle_lib.hermite_clusters(oracle_lib.params(**kw), ref, off)
    ed_g, steps_g, _ = gpu.hard_integrate(gpu.params(**kw), got, off)
    print("%d block steps (oracle %d), %d collisions" % (steps_g, steps, nc))
    assert [f for f in FIELDS if got[f].tobytes() != ref[f].tobytes()] == []
    assert steps_g == steps and ed_g == ed
