"""The tree of up to 8192 particles, built by one workgroup, against the level kernels on the
same particles (tree_coop_min = 1 asks for them): nodes, moments and groups are the same, so
every particle's force and neighbour data are the same bits.  Rings, and rings with a clump that
reaches the deepest level; and a tree above the limit that gets deeper than the one before."""
import numpy as np
import pytest

from gplum_amd import gpu, ic

pytestmark = pytest.mark.gpu

KW = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -6, dt_min=2.0 ** -20, gamma=0.1)


def particles(n, clump):
    pp = ic.disk(n, 3e-7 / n, 0.95, 1.05, seed=n)
    if clump:
        k = min(n // 2, 200)
        pp["pos"][:k] = pp["pos"][k] + np.random.default_rng(n).uniform(-1e-6, 1e-6, (k, 3))
        pp["vel"][:k] = pp["vel"][k]
    return pp


def forces(system, pp):
    system.set_particles(pp)
    system.set_radii()
    system.soft_force(initial=True)
    return system.particles().tobytes()


@pytest.mark.parametrize("group", [64, 256])
@pytest.mark.parametrize("n", [2, 9, 64, 65, 1000, 8191, 8192])
def test_same_bits_as_the_level_kernels(n, group):
    for clump in (False, True):
        if clump and n < 9:
            continue
        pp = particles(n, clump)
        p = gpu.params(n_group_limit=group, **KW)
        small, levels = gpu.System(p, pp), gpu.System(p, pp)
        small.set_forecast("off")
        levels.set_forecast("off")
        levels.set_tuning(n_group_limit=group, tree_coop_min=1)
        print("n %d group %d clump %d" % (n, group, clump), flush=True)
        assert forces(small, pp) == forces(levels, pp)


def test_deeper_tree_above_the_limit():
    p = gpu.params(n_group_limit=64, **KW)
    flat, deep = particles(9000, False), particles(9000, True)
    s, fresh = gpu.System(p, flat), gpu.System(p, deep)
    s.set_forecast("off")
    fresh.set_forecast("off")
    forces(s, flat)
    assert forces(s, deep) == forces(fresh, deep)
