"""GPU: the launch shape never changes a system's bits.

The layer pass runs on 16 x 16, 16 x 32 or 16 x 64 tiles and, with few
workgroups, the WFS and layer passes run in the split form (the WFSs or layers
of a tile over several thread groups).  Which form runs depends on how many
systems a call holds, so all of them have to give the same bits: terms are
added in loop order and p.Ap is summed per 16 x 16 nodes in one order.  All
calls go through the C ABI (maos_amd.tomo)."""
import numpy as np
import pytest

from maos_amd import configs, tomo, workload

pytestmark = pytest.mark.gpu

CFGS = {
    "ngs8": lambda: configs.small8(),
    "ngs10": lambda: configs.batch_member(10.0, 3, 4),
    "lgs20": lambda: configs.batch_member(20.0, 4, 4),
    "lgs30": lambda: configs.large30(),
}


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("name", list(CFGS))
def test_tile_rows_and_split_bit_exact(name, mode):
    """Twelve systems in one call (above the split form's bound on all but the
    smallest system, which the tuned choice of two systems per workgroup keeps
    out of it) against the same systems one, two and three at a time, on every
    layer tile shape: identical solutions and residuals."""
    cfg = CFGS[name]()
    r = tomo.Recon(cfg)
    n = 12
    grads = np.stack([workload.make_inputs(cfg, r, 70 + s) for s in range(n)])
    g = tomo.GpuTomo(r, nbatch=n, maxit=4)
    g.precision(mode)
    g.tune_set(2, 2, 0, 16)
    ref = g.tomo_batch(grads)
    rr = g.residuals(n)
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    for rows in (0, 16, 32, 64):
        g.tune_set(0, 0, 0, rows)
        x = g.tomo_batch(grads)
        assert np.array_equal(x, ref) and np.array_equal(g.residuals(n), rr), "12 systems, %d rows" % rows
    for k in (1, 2, 3):
        h = tomo.GpuTomo(r, nbatch=k, maxit=4)
        h.precision(mode)
        for rows in (0, 16, 32, 64):
            h.tune_set(0, 0, 0, rows)
            x = h.tomo_batch(grads[:k])
            assert np.array_equal(x, ref[:k]), "%d systems, %d rows" % (k, rows)
            assert np.array_equal(h.residuals(k), rr[:k])
        h.close()
    g.close()
    r.close()
