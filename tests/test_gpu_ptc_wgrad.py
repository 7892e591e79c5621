"""The weight gradients on the BF16 matrix cores (Ls a multiple of 4, more than 32 channel
products per 8 x 8 group): one to five 4-slice runs per site (a 16-point group is one site,
several, or straddles them), point counts that are no multiple of 16, more than eight
channels (several groups of tiles) and odd counts (half filled tiles).  The last two stay
on the general kernel: Ls = 6, and too few channels.

Bar: 1e-4 relative against the FP64 oracle, the bar of the network's other gradient tests:
the layers' FP32 error, 2e-5, enters the two factors and the loss's residual.
"""
import numpy as np
import pytest

import ptc_oracle as po
import dwf_amd
from dwf_amd import lattice
from dwf_amd.ptc import ParallelTransportNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,Ls,ch", [((2, 2, 2, 2), 4, (1, 8, 8, 1)),
                                        ((6, 2, 2, 2), 4, (1, 5, 7, 1)),
                                        ((2, 2, 2, 6), 12, (1, 9, 8, 1)),
                                        ((2, 2, 4, 2), 16, (1, 6, 6, 1)),
                                        ((2, 4, 2, 2), 20, (1, 15, 13, 1)),
                                        ((4, 4, 4, 8), 8, (1, 7, 5, 1)),
                                        ((2, 2, 2, 4), 6, (1, 5, 7, 1)),
                                        ((2, 2, 2, 6), 4, (1, 9, 10, 1))])
def test_gradient(dims, Ls, ch):
    print("case ptc wgrad", dims, Ls, ch, flush=True)
    U = lattice.random_gauge(dims, 0.4, 31)
    op = dwf_amd.AFopr_Domainwall_5din_eo(dims, Ls, 0.05, 1.6, 1.0, 0.0, (1, 1, 1, -1), "float")
    op.set_config(U)
    net = ParallelTransportNet(op, ch)
    net.set_weights((0.2 * np.random.default_rng(32).standard_normal(net.nw)).astype(np.float32))
    b, x = op.new_field(), op.new_field()
    op.convert(b, lattice.random_spinor5(dims, Ls, 33))
    op.convert(x, lattice.random_spinor5(dims, Ls, 34))
    loss, grad = net.loss_grad([b], [x])
    lo, go = po.loss_grad(po.Lattice(dims, U, Ls), net.get_weights().astype(np.float64), ch,
                          [(op.reverse(b), op.reverse(x))])
    assert abs(loss - lo) / lo < 1e-5
    assert np.linalg.norm(grad - go) / np.linalg.norm(go) < 1e-4
