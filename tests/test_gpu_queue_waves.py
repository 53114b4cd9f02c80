"""Arm queues run by numbers of waves that are no multiple of 8 (workgroups of 3 or 10 waves, every
small waves_per_cu): every chunk is some wave's, also those just after the waves' first ones.  Edges of
one state, nearly all in collision, so a chunk that no wave takes shows as free edges; and edges of
many states in a queue of many chunks per wave."""
import numpy as np
import pytest

from helpers import O, backend, gpu_edges, near_home, scenes

pytestmark = pytest.mark.gpu


def _scene(kind, rng):
    if kind == "held_boxes":  # workgroups of 10 waves
        return scenes.mixed_arms(rng=rng, n_modes=24)
    desc = scenes.quad_arms(rng=rng)
    al = desc.dh[..., 2]
    C = np.zeros(desc.dh.shape[:2] + (12,))  # the DH joints as chain joints: workgroups of 3 waves
    C[..., 0], C[..., 3] = 1.0, desc.dh[..., 1]
    C[..., 5], C[..., 6] = np.cos(al), -np.sin(al)
    C[..., 9], C[..., 10], C[..., 11] = np.sin(al), np.cos(al), desc.dh[..., 0]
    desc.joint_fixed = C
    return desc


@pytest.mark.parametrize("waves_per_cu", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("kind", ["chain", "held_boxes"])
def test_every_chunk_is_taken(kind, waves_per_cu):
    rng = np.random.default_rng(7)
    desc = _scene(kind, rng)
    B = backend()
    sc, o = B.Scene(desc), O.Scene(desc)
    for n, states, q in ((1500, 3, None), (4200, 40, 0.4)):
        a = scenes.uniform_configs(rng, desc, n) if q is None else near_home(rng, desc, n, q)
        b = np.clip(a + rng.normal(0, 0.05, a.shape), desc.limits[0], desc.limits[1])
        N = np.full(n, states, np.int32)
        modes = rng.integers(0, 24, n).astype(np.int32) if kind == "held_boxes" else None
        ref = o.check_edges(a, b, 0.05, N=N, modes=modes)
        for g, t in ((1, 1), (1, 4), (2, 16)):
            tune = B.make_tune(slots_per_pass=g, slots_per_ticket=t, waves_per_cu=waves_per_cu)
            got = gpu_edges(sc, a, b, 0.05, N=N, modes=modes, tune=tune)
            assert np.array_equal(got, ref), (n, g, t, int(np.sum(got != ref)))


@pytest.mark.parametrize("seed,n_arms,n", [(737, 3, 30000), (195, 5, 5200), (1, 6, 20000)])
def test_edges_that_collide_near_their_start(seed, n_arms, n):
    # arms in contact around the home pose: waves hold slots of edges that others are finding in collision
    rng = np.random.default_rng(seed)
    desc = scenes.quad_arms(rng=rng, n_arms=n_arms, dof=7, n_boxes=50)
    sc, o = backend().Scene(desc), O.Scene(desc)
    a = near_home(rng, desc, n, 0.1)
    b = np.clip(a + 0.3 * rng.lognormal(0, 1, (n, 1)) * rng.uniform(-1, 1, a.shape), desc.limits[0], desc.limits[1])
    ref = o.check_edges(a, b, 0.05)
    assert ref.mean() < 0.5
    for _ in range(2):
        assert np.array_equal(gpu_edges(sc, a, b, 0.05), ref)
