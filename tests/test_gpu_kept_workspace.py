"""One-shot batches (mrcc_check_edges) on one scene from several host threads and streams at once: the
scene keeps one workspace, which one call at a time holds; the others allocate their own.  Batches of
different sizes, growing and shrinking, a batch in error among them, and one beyond the size that is kept."""
import threading

import numpy as np
import pytest

from helpers import O, backend, near_home, scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_threads_and_sizes():
    B = backend()
    rng = np.random.default_rng(12)
    desc = scenes.quad_arms(rng=rng, n_arms=2, dof=6, n_boxes=20)
    sc, o = B.Scene(desc), O.Scene(desc)
    jobs = []
    for n in (40, 9000, 700, 20000, 1, 3000):
        a = near_home(rng, desc, n, 0.5)
        b = np.clip(a + rng.normal(0, 0.2, a.shape), desc.limits[0], desc.limits[1])
        jobs.append((a, b, o.check_edges(a, b, 0.05)))
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for turn in range(8):
                a, b, ref = jobs[(k + turn) % len(jobs)]
                ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
                out = torch.full((len(a),), 7, dtype=torch.uint8, device="cuda")
                kw = {}
                if turn % 3 == 2:  # N_start beyond N: the call reports it, the edge counts as a collision
                    ns = torch.zeros(len(a), dtype=torch.int32, device="cuda")
                    ns[0] = 1 << 20
                    kw = dict(N_start=ns)
                st.synchronize()
                try:
                    sc.check_edges_device(sc.edge_batch(ta, tb, out, 0.05, **kw))
                    failed = False
                except B._lib.MrccError:
                    failed = True
                got = out.cpu().numpy().astype(bool)
                want = ref.copy()
                want[0] &= not kw
                if failed != bool(kw) or not np.array_equal(got, want):
                    bad.append((k, turn, failed, int(np.sum(got != want))))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_beyond_the_kept_size():
    B = backend()
    rng = np.random.default_rng(3)
    desc = scenes.planar_boxes(rng=rng, n_robots=2, n_obstacles=20)
    sc, o = B.Scene(desc), O.Scene(desc)
    n = 1200000  # queue of 72 bytes an edge
    a = rng.uniform(desc.limits[0], desc.limits[1], (n, 6))
    b = a + rng.normal(0, 0.02, a.shape)
    tune = B.make_tune(slots_per_pass=8)
    m = 4000
    ref = o.check_edges(a[-m:], b[-m:], 0.01)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    for k in (n, m, n):
        out = torch.full((k,), 7, dtype=torch.uint8, device="cuda")
        sc.check_edges_device(sc.edge_batch(ta[-k:], tb[-k:], out, 0.01), tune)
        assert np.array_equal(out[-m:].cpu().numpy().astype(bool), ref)
