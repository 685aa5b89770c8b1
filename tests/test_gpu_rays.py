"""GPU: ray paths of the tomography operators.

Where a layer's rays fall a whole number of nodes from its grid, rounding
leaves some of them at fraction 1 of the node before; such plans take the
matched kernels too, with the generic kernels' values.
"""
import numpy as np
import pytest

from maos_amd import configs, tomo, workload
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _fit30():
    c = configs.large30()
    return configs.with_fit_dirs(c, configs.fit_for(c))


WHOLE = {
    "lgs20_w4_l4": lambda: configs.batch_member(20.0, 4, 4),
    "lgs10_w3_l3": lambda: configs.batch_member(10.0, 3, 3),
    "large30_fit": _fit30,
}


@pytest.mark.parametrize("name", list(WHOLE))
def test_whole_node_offsets_are_matched(name):
    """L and R against the oracle: FP64 sums of FP32 inputs, coefficients and
    fractions, each rounded by 6e-8 (bar 1e-6); the solve to its gate."""
    cfg = WHOLE[name]()
    r = tomo.Recon(cfg)
    g, o = tomo.GpuTomo(r, maxit=10), Oracle(r, nthread=8)
    print("case", cfg["name"], g.info(), flush=True)
    assert g.info()["matched"] == 1
    x = np.random.default_rng(5).standard_normal(r.nx)
    assert rel(g.L(x), o.tomo_l(x)) < 1e-6
    grad = workload.make_inputs(cfg, r, 7)
    assert rel(g.R(grad), o.tomo_r(grad)) < 1e-6
    xs, _, _ = g.tomo(grad)
    assert rel(xs, o.solve(grad, 10)[0]) < 1e-4


def test_off_grid_rays_stay_generic():
    """Rays at a ratio other than 1 keep the generic kernels."""
    assert tomo.GpuTomo(tomo.Recon(configs.lgs8_flat())).info()["matched"] == 0
