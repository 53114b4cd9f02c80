"""The self-collision screen of arm batches and the chunks of short queues, against the oracle: batch
sizes on both sides of the screen's thresholds and of a wave's chunk, DH and chain joints, prismatic
joints, modes with few active arms and held boxes, robot masks, windows, non-finite coordinates, and
batches whose states are mostly free (the screen stops early)."""
import numpy as np
import pytest

from arm_bruteforce import tiny_arm_scene
from helpers import O, backend, gpu_configs, gpu_edges, near_home, scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _edges(rng, desc, n, sigma):
    a = scenes.uniform_configs(rng, desc, n) if sigma is None else near_home(rng, desc, n, sigma)
    b = np.clip(a + rng.normal(0, 0.2, a.shape), desc.limits[0], desc.limits[1])
    return a, b


@pytest.mark.parametrize("n", [1535, 1536, 1537, 4111, 70001])
@pytest.mark.parametrize("n_arms,dof,sigma", [(4, 7, None), (1, 8, None), (3, 2, 0.5), (2, 6, 0.1)])
def test_screen_edges(n, n_arms, dof, sigma):
    rng = np.random.default_rng(n + 10 * n_arms)
    desc = scenes.quad_arms(rng=rng, n_arms=n_arms, dof=dof, n_boxes=12)
    sc, o = backend().Scene(desc), O.Scene(desc)
    a, b = _edges(rng, desc, n, sigma)
    a[5, 1] = np.nan  # not coordinate 0, where it makes the length of the edge undefined
    b[6] = a[6]  # no interior state
    assert np.array_equal(gpu_edges(sc, a, b, 0.1), o.check_edges(a, b, 0.1))


@pytest.mark.parametrize("chain", [False, True])
def test_screen_masks_modes_windows(chain):
    rng = np.random.default_rng(5)
    desc = scenes.mixed_arms(n_modes=40, n_arms=5, dof=6, n_boxes=12, rng=rng)
    if chain:
        al = desc.dh[..., 2]
        C = np.zeros(desc.dh.shape[:2] + (12,))
        C[..., 0], C[..., 3] = 1.0, desc.dh[..., 1]
        C[..., 5], C[..., 6] = np.cos(al), -np.sin(al)
        C[..., 9], C[..., 10], C[..., 11] = np.sin(al), np.cos(al), desc.dh[..., 0]
        desc.joint_fixed = C
    sc, o = backend().Scene(desc), O.Scene(desc)
    n = 3000
    a, b = _edges(rng, desc, n, 0.6)
    modes = rng.integers(0, 40, n).astype(np.int32)
    N = np.maximum(2, (np.max(np.abs(b - a), axis=1) / 0.05).astype(np.int64) + 1).astype(np.int32)
    S = (rng.uniform(size=n) * N * 0.5).astype(np.int32)
    M = np.where(rng.uniform(size=n) < 0.3, -1, S + rng.integers(0, 10, n)).astype(np.int32)
    for mask in (0xFFFFFFFF, 0b10110, 0b01000, 0):
        assert np.array_equal(gpu_edges(sc, a, b, 0.05, modes=modes, mask=mask),
                              o.check_edges(a, b, 0.05, modes=modes, mask=mask)), mask
    for incl in (False, True):
        ref = o.check_edges(a, b, 0.05, N=N, N_start=S, N_max=M, include_endpoints=incl, modes=modes)
        assert np.array_equal(gpu_edges(sc, a, b, 0.05, N=N, N_start=S, N_max=M, incl=incl, modes=modes), ref)


@pytest.mark.parametrize("n", [49151, 49152, 50001])
@pytest.mark.parametrize("sigma", [None, 0.1])
def test_screen_configs(n, sigma):
    rng = np.random.default_rng(n)
    desc = scenes.mixed_arms(n_modes=16, n_arms=3, dof=6, n_boxes=10, rng=rng)
    sc, o = backend().Scene(desc), O.Scene(desc)
    q, _ = _edges(rng, desc, n, sigma)
    q[3, 2], q[n - 1, 1] = np.inf, np.nan
    modes = rng.integers(0, 16, n).astype(np.int32)
    bad = modes.copy()
    bad[7] = 99  # a mode the scene does not have counts as a collision
    ref = o.check_configs(q, modes=modes)
    got = gpu_configs(sc, q, modes=bad)
    assert not got[7]
    assert np.array_equal(np.delete(got, 7), np.delete(ref, 7))
    assert np.array_equal(gpu_configs(sc, q, modes=modes, mask=0b010), o.check_configs(q, modes=modes, mask=0b010))


def test_screen_prismatic():
    rng = np.random.default_rng(31)
    desc = tiny_arm_scene(rng, scenes, chain=True, prism=0.4)
    sc, o = backend().Scene(desc), O.Scene(desc)
    q = rng.uniform(1.1 * desc.limits[0], 1.1 * desc.limits[1], size=(60000, desc.dim))  # some beyond travel
    assert np.array_equal(gpu_configs(sc, q), o.check_configs(q))
    a, b = q[:5000], q[5000:10000]
    assert np.array_equal(gpu_edges(sc, a, b, 0.1), o.check_edges(a, b, 0.1))


def test_long_edges_at_one_slot_per_pass():
    # 17,000 states: more passes than the queue holds
    rng = np.random.default_rng(2)
    desc = scenes.quad_arms(rng=rng, n_arms=2, dof=3, n_boxes=0)
    sc, o = backend().Scene(desc), O.Scene(desc)
    a = near_home(rng, desc, 6, 0.3)
    b = a + 0.17 * np.sign(rng.normal(size=a.shape))
    assert np.array_equal(gpu_edges(sc, a, b, 1e-5), o.check_edges(a, b, 1e-5))


# records of arm edges: rows as one run of words (strided, indexed, odd and misaligned rows not), a
# wave's last edges missing, every coordinate count up to the largest, batches beyond one pass of the grid
@pytest.mark.parametrize("n_arms,dof,n", [(1, 1, 70), (1, 7, 2000), (2, 3, 1), (3, 6, 65), (8, 8, 3001), (2, 1, 270001)])
@pytest.mark.parametrize("layout", ["rows", "columns", "offset", "index"])
def test_records(n_arms, dof, n, layout):
    rng = np.random.default_rng(n + dof)
    desc = scenes.quad_arms(rng=rng, n_arms=n_arms, dof=dof, n_boxes=3)
    sc, o = backend().Scene(desc), O.Scene(desc)
    D = desc.dim
    a, b = _edges(rng, desc, n, 0.3)
    if D > 1 and n > 8:
        a[5, 1] = np.nan  # skipped in the length, a collision at every state
    ref = o.check_edges(a, b, 0.1)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    kw = {}
    if layout == "columns":
        ta, tb = ta.t().contiguous().t(), tb.t().contiguous().t()
    elif layout == "offset":  # 8 bytes past a 16-byte word
        ta, tb = (torch.cat([t.new_zeros(1), t.flatten()])[1:].view(n, D) for t in (ta, tb))
    elif layout == "index":
        perm = torch.randperm(n, device="cuda")
        inv = torch.argsort(perm).to(torch.int32)
        ta, tb, kw = ta[perm], tb[perm], dict(idx1=inv, idx2=inv)
    out = torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    sc.check_edges_device(sc.edge_batch(ta, tb, out, 0.1, **kw))
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), ref.astype(np.uint8))
