"""Trees with small leaves around the particle number up to which one workgroup builds them (3584 +
1024 n_leaf_limit, 8192 at most): the same bits as the level kernels, which a tree_coop_min of the
particle number asks for, and the rule's choice takes no longer than they do.  (One workgroup takes
1.4 times as long for 8192 particles in leaves of 1 and 1.18 times in leaves of 2; that tree_coop_min
also splits the root with a workgroup, up to 1.04 times, and 1.1 is above that.)"""
import numpy as np
import pytest

from gplum_amd import gpu, ic

pytestmark = pytest.mark.gpu

KW = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -6, dt_min=2.0 ** -20, gamma=0.1)


def pair_of_systems(n, leaf):
    pp = ic.disk(n, 3e-7 / n, 0.95, 1.05, seed=n)
    p = gpu.params(n_group_limit=64, n_leaf_limit=leaf, **KW)
    out = []
    for coop in (0, n):
        s = gpu.System(p, pp)
        s.set_forecast("off")
        s.set_tuning(n_group_limit=64, tree_coop_min=coop)
        s.set_radii()
        s.soft_force(initial=True)
        out.append(s)
    return out


@pytest.mark.parametrize("leaf,n", [(1, 4608), (1, 4609), (2, 5632), (2, 5633), (3, 6657), (4, 7680), (4, 7681), (5, 8192)])
def test_same_bits_at_the_line(leaf, n):
    rule, levels = pair_of_systems(n, leaf)
    assert rule.particles().tobytes() == levels.particles().tobytes()


@pytest.mark.parametrize("leaf", [1, 2, 8])
def test_rule_is_no_slower_than_the_level_kernels(leaf):
    for n in (4500, 8192):
        systems = pair_of_systems(n, leaf)
        best = [np.inf, np.inf]
        for _ in range(6):
            for k, s in enumerate(systems):
                s.reset_stats(True)
                for _ in range(5):
                    s.soft_force(initial=True)
                best[k] = min(best[k], s.stats()["tree_ms"] / 5)
        print("leaves of %d, %d particles: rule %.0f us, level kernels %.0f us" % (leaf, n, 1e3 * best[0], 1e3 * best[1]))
        assert best[0] <= 1.1 * best[1]
