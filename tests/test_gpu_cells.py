"""Plane scenes by cell table against the oracle: robot counts on both sides of the kernels' bounds,
cells with more open obstacles than a record holds, obstacles of zero size and far apart, states on
cell borders, outside the grid, with huge yaws and non-finite coordinates, robot masks, and scenes
that have no table (no obstacles, negative sizes, far from the origin)."""
import numpy as np
import pytest

from helpers import O, backend, gpu_configs, gpu_edges, scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _check(desc, q, a, b, res=0.02):
    sc, o = backend().Scene(desc), O.Scene(desc)
    for mask in (0xFFFFFFFF, 0b10):
        assert np.array_equal(gpu_configs(sc, q, mask=mask), o.check_configs(q, mask=mask)), mask
        assert np.array_equal(gpu_edges(sc, a, b, res, mask=mask), o.check_edges(a, b, res, mask=mask)), mask


def _inputs(rng, desc, n, step, per):
    D = desc.dim
    q = 1.3 * rng.uniform(desc.limits[0], desc.limits[1], size=(n, D))
    q[:n // 4, 0::per] = np.round(q[:n // 4, 0::per] * 16) / 16  # borders of cells and obstacles
    q[0] = 0.0
    q[1, per % D], q[2, 0], q[3, 1] = np.nan, np.inf, -1e9
    a = rng.uniform(desc.limits[0], desc.limits[1], size=(n, D))
    return q, a, a + rng.normal(0, step, a.shape)


@pytest.mark.parametrize("nr", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("no", [0, 1, 60])
def test_planar(nr, no):
    rng = np.random.default_rng(100 * nr + no)
    desc = scenes.planar_boxes(rng=rng, n_robots=nr, n_obstacles=no)
    desc.robot_half *= rng.uniform(0.05, 1.0)
    if no > 30:
        desc.obstacle_pose[:30, :2] = desc.obstacle_pose[0, :2] + rng.normal(0, 0.1, (30, 2))  # a pile
        desc.obstacle_half[30:33] = 0.0
    q, a, b = _inputs(rng, desc, 6000, 0.2, 3)
    q[5:400, 2] *= 10.0 ** rng.uniform(0, 9, 395)
    _check(desc, q, a, b)


@pytest.mark.parametrize("nr", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rd", [2, 3])
def test_disks(nr, rd):
    rng = np.random.default_rng(10 * nr + rd)
    lim = np.array([[-2.0] * (nr * rd), [2.0] * (nr * rd)])
    desc = scenes.disks_scene(
        rng.uniform(0.0, 0.2, nr), rd, lim,
        spheres=[(rng.uniform(-2, 2, rd), r) for r in np.concatenate([[0.0], rng.uniform(0, 0.3, 12)])],
        rects=[(rng.uniform(-2, 2, rd), s) for s in rng.uniform(0.0, 0.5, (15, rd))]
        + [(np.zeros(rd) + 0.01 * k, np.full(rd, 0.4)) for k in range(9)])
    q, a, b = _inputs(rng, desc, 6000, 0.3, rd)
    _check(desc, q, a, b)


def test_scenes_without_a_table():
    rng = np.random.default_rng(4)
    desc = scenes.planar_boxes(rng=rng, n_robots=2, n_obstacles=20)
    q, a, b = _inputs(rng, desc, 3000, 0.2, 3)
    desc.obstacle_half[3] *= -1.0
    _check(desc, q, a, b)
    desc.obstacle_half[3] *= -1.0
    desc.obstacle_pose[4, 0] = 3e5
    _check(desc, q, a, b)


def _batch(rng, desc, n):
    a = rng.uniform(desc.limits[0], desc.limits[1], size=(n, desc.dim))
    step = np.exp(rng.normal(np.log(0.3), 1.2, (n, 1)))
    return a, a + step * rng.uniform(-1, 1, a.shape)


# edges per wave 1, 2, 4, 8, 16 change at multiples of 4,000; the last wave is partly filled
@pytest.mark.parametrize("n", [1, 63, 7999, 8000, 16001, 32003, 64005])
@pytest.mark.parametrize("kind,nr", [("disks", 2), ("disks", 3), ("planar", 2), ("planar", 5)])
def test_batches(n, kind, nr):
    rng = np.random.default_rng(n + nr)
    desc = (scenes.planar_disks(rng=rng, n_robots=nr, n_rects=6) if kind == "disks" else
            scenes.planar_boxes(rng=rng, n_robots=nr, n_obstacles=12))
    sc, o = backend().Scene(desc), O.Scene(desc)
    a, b = _batch(rng, desc, n)
    if n > 100:
        a[5, 1], b[6] = np.nan, a[6]
    assert np.array_equal(gpu_edges(sc, a, b, 0.01), o.check_edges(a, b, 0.01))
    N = rng.integers(2, 90, n).astype(np.int32)
    S = (rng.uniform(size=n) * N * 0.5).astype(np.int32)
    M = np.where(rng.uniform(size=n) < 0.3, -1, S + rng.integers(0, 40, n)).astype(np.int32)
    for incl in (False, True):
        assert np.array_equal(gpu_edges(sc, a, b, 0.05, N=N, N_start=S, N_max=M, incl=incl),
                              o.check_edges(a, b, 0.05, N=N, N_start=S, N_max=M, include_endpoints=incl))


# 1,024 states: the most that a wave takes on its own; 200 edges of 60,000: more items than the list
# holds; 3 of 3,000,000: the largest share of the list
@pytest.mark.parametrize("n,states", [(9, 1026), (9, 1027), (40, 20000), (200, 60000), (3, 3000000)])
def test_long_edges(n, states):
    rng = np.random.default_rng(states)
    desc = scenes.disks_scene([0.1, 0.05], 2, np.array([[-2.0] * 4, [2.0] * 4]),
                              spheres=[(np.array([0.3, 0.2]), 0.1)], rects=[(np.array([-0.9, 0.5]), np.array([0.2, 0.3]))])
    sc, o = backend().Scene(desc), O.Scene(desc)
    a = rng.uniform(-2, 2, (n, 4))
    b = a.copy()
    b[:, 0] = a[:, 0] + 0.5
    b[:, 1:] += 0.2 * rng.uniform(-1, 1, (n, 3))
    N = np.full(n, states, np.int32)
    N[::4] = 50
    ref = o.check_edges(a, b, 0.01, N=N)
    ta, tb, tN = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), torch.from_numpy(N).cuda()
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    plan = backend().EdgePlan(sc, sc.edge_batch(ta, tb, out, 0.01, N=tN), keep=(ta, tb, tN, out))
    for _ in range(4):  # the counters go from run to run
        out.fill_(9)
        plan.run()
        assert np.array_equal(out.cpu().numpy().astype(bool), ref)
