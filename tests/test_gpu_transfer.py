"""Particles to the device and back: every field of every particle unchanged, byte for byte, at
sizes around a workgroup and around a transfer (2^18 particles), and what initialize() fills
in (time, counters, a missing radius and enlargement).  Copies only, so no difference is
allowed; the radius is one pow, compared to its last digit."""
import math

import numpy as np
import pytest

from gplum_amd import abi, gpu, ic

pytestmark = pytest.mark.gpu

KW = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -6, dt_min=2.0 ** -20, gamma=0.1)


@pytest.mark.parametrize("n", [1, 7, 256, 257, 2 ** 18 - 1, 2 ** 18, 2 ** 18 + 3])
def test_round_trip(n):
    rng = np.random.default_rng(n)
    pp = np.frombuffer(rng.bytes(n * abi.PARTICLE.itemsize), dtype=abi.PARTICLE).copy()
    pp["id"] = rng.permutation(n)
    S = gpu.System(gpu.params(**KW))
    for _ in range(2):
        S.set_particles(pp, 0.0)
        assert S.particles().tobytes() == pp.tobytes()


def test_initialize_fills_in():
    pp = ic.disk(3000, 1e-10, 0.9, 1.1, seed=5)
    kw = dict(KW, collision=1)
    bare = pp.copy()
    bare["r_planet"][::2] = 0.0
    bare["f"][::3] = 0.0
    bare["time"], bare["flags"], bare["n_cluster"] = 3.0, 5, 9
    S = gpu.System(gpu.params(**kw))
    S.set_particles(bare, 0.5)
    S.initialize()
    out = S.particles()
    out = out[np.argsort(out["id"])]
    src = bare[np.argsort(bare["id"])]
    p = gpu.params(**kw)
    want = np.array([r if r > 0 else math.pow(0.75 * m / (math.pi * p.dens), 1.0 / 3.0)
                     for r, m in zip(src["r_planet"], src["mass"])])
    np.testing.assert_allclose(out["r_planet"], want, rtol=4e-16)
    assert np.array_equal(out["f"], np.where(src["f"] == 0.0, p.increase_factor, src["f"]))
    assert np.all(out["time"] == 0.5)
