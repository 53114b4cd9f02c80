"""The cell table of plane scenes at the ends of its range, against the oracle: the largest number of
obstacles, all of them undecided in one cell."""
import numpy as np
import pytest

from helpers import O, backend, gpu_configs, scenes

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
