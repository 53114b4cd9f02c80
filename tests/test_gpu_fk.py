"""Link frames against the oracle, bit for bit: every joint count (shared over a quad's lanes), arm
counts and row counts that leave a wave's last items empty, results that are not 16-byte aligned, and
rows given by column."""
import ctypes

import numpy as np
import pytest

from helpers import O, backend, pkg, scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_arms,dof", [(1, 1), (3, 2), (2, 3), (5, 4), (1, 5), (3, 6), (4, 7), (7, 8)])
@pytest.mark.parametrize("n", [1, 37])
@pytest.mark.parametrize("offset", [0, 1])
def test_frames(n_arms, dof, n, offset):
    rng = np.random.default_rng(10 * n_arms + dof)
    desc = scenes.quad_arms(rng=rng, n_arms=n_arms, dof=dof, n_boxes=2)
    sc, o = backend().Scene(desc), O.Scene(desc)
    D = desc.dim
    Q = rng.uniform(-3, 3, size=(n, D))
    q = torch.from_numpy(Q).cuda()
    if offset:
        q = q.t().contiguous().t()
    buf = torch.full((n * D * 12 + 2,), np.nan, dtype=torch.float64, device="cuda")
    out = buf[offset:]
    pkg._lib.check(pkg.lib().mrcc_arm_fk(sc.handle, ctypes.c_void_p(q.data_ptr()), n, q.stride(0), q.stride(1),
                                         ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(0)))
    torch.cuda.synchronize()
    got = out[:n * D * 12].cpu().numpy().reshape(n, D, 12)
    for r in range(n):
        assert np.array_equal(got[r], o.arm_fk(Q[r]).reshape(D, 12)), r
    assert torch.isnan(buf[:offset]).all() and torch.isnan(out[n * D * 12:]).all()
