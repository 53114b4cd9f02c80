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


def _spread(desc, how):
    """Obstacles of a plane scene with one far off, a long wall, or half of them moved away."""
    disks = desc.kind == "disks"
    pos = desc.rect_center if disks else desc.obstacle_pose
    if how == "far":
        pos[0, :2] = [500.0, 300.0]
    elif how == "groups":
        pos[::2, 0] += 300.0
    else:
        pos[0, :2] = [0.0, 2.3]
        if disks:
            desc.rect_size[0] = [120.0, 0.1]
        else:
            desc.obstacle_half[0], desc.obstacle_pose[0, 2] = [60.0, 0.05], 0.0


@pytest.mark.parametrize("how", ["far", "wall", "groups"])
@pytest.mark.parametrize("kind,nr", [("disks", 1), ("disks", 2), ("disks", 3), ("disks", 5), ("planar", 1), ("planar", 4),
                                     ("planar", 5), ("planar", 9)])
@pytest.mark.parametrize("no", [12, 70])
def test_scenes_spread_wide(how, kind, nr, no):
    # few obstacles leave the table few tests, many make the scene give it up
    rng = np.random.default_rng(no + nr)
    desc = (scenes.planar_disks(rng=rng, n_robots=nr, n_rects=no) if kind == "disks" else
            scenes.planar_boxes(rng=rng, n_robots=nr, n_obstacles=no))
    if kind == "planar":
        desc.robot_half *= 0.4
    else:
        desc.robot_radius = desc.robot_radius * 0.5
    _spread(desc, how)
    sc, o = backend().Scene(desc), O.Scene(desc)
    n = 5000
    a = rng.uniform(desc.limits[0], desc.limits[1], (n, desc.dim))
    b = a + rng.normal(0, 0.15, a.shape)
    for mask in (0xFFFFFFFF, 0b1):
        assert np.array_equal(gpu_configs(sc, a, mask=mask), o.check_configs(a, mask=mask)), mask
        assert np.array_equal(gpu_edges(sc, a, b, 0.02, mask=mask), o.check_edges(a, b, 0.02, mask=mask)), mask
