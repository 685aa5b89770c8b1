"""GPU: the FP64 solve's ray gathers (precision mode 4).

HX' takes a table of two rays a node and axis where every node has at most
two, and lists where one has more (layers coarser than the rays: a cone
narrows the ray spacing).  WFSs and layers are taken three at a time and GP's
entries four at a time, so the counts below are around those: remainders of
one, two and none, with and without TT removal in the LHS.  Both sides are
FP64: a sum of at most some hundred terms in another order, 1e-12 relative
L2."""
import numpy as np
import pytest

from maos_amd import configs, tomo, workload
from oracle.oracle import Oracle
from parity_util import rel

pytestmark = pytest.mark.gpu

CASES = {
    "w1_l1": lambda: configs.batch_member(8.0, 1, 1),
    "w2_l3": lambda: configs.batch_member(8.0, 2, 3),
    "w3_l4": lambda: configs.batch_member(10.0, 3, 4),
    "w4_l5": lambda: configs.batch_member(8.0, 4, 5),
    "w4_l2_flat": lambda: configs.lgs8_flat(),
    "w5_l2_split0": lambda: configs.batch_member(8.0, 5, 2, recon_split=0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_gathers64(name):
    cfg = CASES[name]()
    r = tomo.Recon(cfg)
    g = tomo.GpuTomo(r, maxit=2)
    g.precision(4)
    o = Oracle(r, nthread=4)
    x = np.random.default_rng(11).standard_normal(r.nx)
    grad = workload.make_inputs(cfg, r, 12)
    el, er = rel(g.L(x), o.tomo_l(x)), rel(g.R(grad), o.tomo_r(grad))
    print("L %.3e R %.3e" % (el, er), flush=True)
    assert el < 1e-12 and er < 1e-12
    g.close()
