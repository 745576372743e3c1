"""The training pass in tiles of 64 rows, one workgroup per tile up to one per compute unit: the
gradient against the CPU reference where tiles can go wrong (a single row, a wave's 16 rows, a full
tile, one row more, more tiles than workgroups), and the same bits twice (the shares are added in a
fixed order).

Tolerance: FP32 sums in another order can move a BF16 rounding of an activation or of a gradient by
one spacing, 2^-8 of it; three layers of them stay below 3 * 2^-8 = 1.2e-2 of a block's largest
gradient (bar 2e-2), and the loss, a mean of unrounded outputs, below 1e-3."""
import numpy as np
import pytest

import crm_mlp
import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 64, 65, 64 * 256 + 1])
def test_gradient_of_a_ragged_batch(n):
    import torch
    rng = np.random.default_rng(n)
    p = (crm_mlp.init_params(5) + rng.normal(0, 0.02, crm_mlp.NPARAM)).astype(np.float32)
    mean, scale, oscale = rng.normal(0, 0.5, 9), rng.uniform(0.5, 2.0, 9), rng.uniform(0.5, 2.0, 6)
    X = rng.normal(0, 1.5, (n, 9)).astype(np.float32)
    T = rng.normal(0, 1.0, (n, 6)).astype(np.float32)
    m = crm_mlp.CrmMlp(0)
    try:
        m.set_params(p)
        m.set_norm(mean, scale, oscale)
        x, t = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
        g, loss = m.grad(x, t)
        again, loss2 = m.grad(x, t)
    finally:
        m.close()
    assert loss == loss2 and np.array_equal(g, again)
    f32 = [a.astype(np.float32) for a in (mean, scale, oscale)]
    want, gw = mlp_ref.loss_grad(p, X, T, *f32, "bf16")
    assert abs(loss - want) <= 1e-3 * abs(want)
    offs = np.cumsum([0, 9 * 128, 128, 128 * 128, 128, 128 * 128, 128, 128 * 6, 6])
    for b in range(8):
        e, w = g[offs[b]:offs[b + 1]], gw[offs[b]:offs[b + 1]]
        assert np.abs(e - w).max() <= 2e-2 * np.abs(w).max(), b
