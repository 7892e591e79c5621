"""The network layers on the BF16 matrix cores (three-part split of the transports):
channel counts from 9 to 16 (weights of a layer too large for LDS, five to eight row
tiles, odd counts on both sides), Ls = 16 (a tile is one site, shifts by lane) and Ls that
straddle sites, and inputs scaled far down and up.

Bar: 2e-5 relative against the FP64 oracle with the same bfloat16 weights, the bar of the
network's other tests: the parts add up to the FP32 transport exactly, so only the FP32
accumulation rounds, 11 x 16 x 8 terms per layer of 6e-8 each, over four layers; the layers
are linear, so the scale of the input does not enter (its smallest part, 2^-24 of 1e-25,
is still a normal bfloat16).
"""
import numpy as np
import pytest

import ptc_oracle as po
import dwf_amd
from dwf_amd import lattice
from dwf_amd.ptc import ParallelTransportNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,Ls,ch", [((2, 2, 2, 4), 16, (1, 10, 16, 1)),
                                        ((2, 2, 2, 4), 16, (1, 11, 13, 3, 1)),
                                        ((2, 4, 2, 2), 6, (1, 15, 9, 1)),
                                        ((2, 2, 4, 2), 5, (1, 12, 14, 1)),
                                        ((4, 2, 2, 2), 20, (1, 5, 2, 1))])
@pytest.mark.parametrize("scale", [1.0, 1e-25, 1e15])
def test_forward(dims, Ls, ch, scale):
    print("case ptc split", dims, Ls, ch, scale, flush=True)
    U = lattice.random_gauge(dims, 0.4, 21)
    op = dwf_amd.AFopr_Domainwall_5din_eo(dims, Ls, 0.05, 1.6, 1.0, 0.0, (1, 1, 1, -1), "float")
    op.set_config(U)
    net = ParallelTransportNet(op, ch)
    net.set_weights((0.2 * np.random.default_rng(22).standard_normal(net.nw)).astype(np.float32))
    x = scale * lattice.random_spinor5(dims, Ls, 23)
    fi, fo = op.new_field(), op.new_field()
    op.convert(fi, x)
    net.apply(fo, fi)
    want = po.apply(po.Lattice(dims, U, Ls), net.get_weights().astype(np.float64), ch,
                    op.reverse(fi))
    got = op.reverse(fo)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-5
