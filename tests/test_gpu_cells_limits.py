"""The cell table of plane scenes at the ends of its range, against the oracle: the largest number of
obstacles, all of them undecided in one cell; plane edges of more passes than the queue holds."""
import numpy as np
import pytest

from helpers import O, backend, gpu_configs, gpu_edges, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["disks", "planar"])
@pytest.mark.parametrize("no", [65534, 65535])
def test_all_obstacles_undecided_in_a_cell(kind, no):
    ang = np.linspace(-np.pi, np.pi, 40)
    if kind == "disks":  # one point, many times over: undecided around the robot's radius
        desc = scenes.disks_scene([0.1], 2, np.array([[-1.0] * 2, [1.0] * 2]),
                                  rects=[(np.zeros(2), np.zeros(2))] * no)
        q = [(r * np.cos(t), r * np.sin(t)) for t in ang for r in (0.0999, 0.1, 0.1001, 0.101)]
    else:  # undecided between the robot's half width and its half diagonal
        desc = scenes.planar_boxes(rng=np.random.default_rng(0), n_robots=1, n_obstacles=no)
        desc.robot_half[:] = [[0.05, 0.2]]
        desc.obstacle_pose[:], desc.obstacle_half[:] = 0.0, 0.0
        q = [(r * np.cos(t), r * np.sin(t), 0.7) for t in ang for r in (0.04, 0.06, 0.1, 0.15, 0.19, 0.21)]
    q = np.array(q)
    ref = O.Scene(desc).check_configs(q)
    assert 0.2 < ref.mean() < 0.9
    assert np.array_equal(gpu_configs(backend().Scene(desc), q), ref)


@pytest.mark.parametrize("rd,nr", [(2, 2), (2, 5), (3, 2)])
@pytest.mark.parametrize("incl", [False, True])
def test_queue_of_edges_beyond_its_passes(rd, nr, incl):
    # one slot per pass, 40,000 states: every slot holds the states 16,384 apart as well
    rng = np.random.default_rng(rd + nr)
    lim = np.array([[-2.0] * (nr * rd), [2.0] * (nr * rd)])
    desc = scenes.disks_scene([0.01] * nr, rd, lim, spheres=[(np.full(rd, 1.9), 0.002)])
    B = backend()
    sc, o = B.Scene(desc), O.Scene(desc)
    n = 24
    a = rng.uniform(-1.5, 1.5, (n, nr * rd))
    b = a + rng.uniform(-0.3, 0.3, a.shape)
    at = rng.uniform(0, 1, n)  # robot 0 meets the sphere somewhere along every other edge
    for i in range(0, n, 2):
        d = rng.uniform(-0.05, 0.05, rd)
        a[i, :rd], b[i, :rd] = 1.9 - at[i] * d, 1.9 + (1 - at[i]) * d
    N = np.full(n, 40000, np.int32)
    N[3], N[4] = 16386, 16387
    S = np.where(np.arange(n) % 3 == 0, 7, 0).astype(np.int32)
    ref = o.check_edges(a, b, 0.01, N=N, N_start=S, include_endpoints=incl)
    assert 0 < ref.sum() < n
    tune = B.make_tune(slots_per_pass=1, use_graph=0)
    assert np.array_equal(gpu_edges(sc, a, b, 0.01, tune=tune, N=N, N_start=S, incl=incl), ref)
