"""The two weight-gradient kernels on the same layers: DWF_PTC_KERNEL=valu-wgrad changes only
the weight gradients, so the one-channel layers, which stay on the general kernel, agree bit
for bit, and the 8 -> 8 layer shows the difference of the two kernels alone.

The target is uncorrelated with the input and large beside the network's output, so a
gradient element is a sum of N = 3 x points products of random sign.  Bars: each kernel rounds
partial sums of tens of products in FP32, errors of 6e-8 of a partial sum with random signs,
so both are within a few 1e-7 of the sum's size and their difference is below 5e-7; its mean
over the n = 11 x 64 x 16 elements of one part, which only errors of one sign leave, is below
six times 5e-7 / sqrt(n) = 3e-8.
"""
import numpy as np
import pytest

import dwf_amd
from dwf_amd import lattice
from dwf_amd.ptc import ParallelTransportNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,Ls", [((4, 4, 4, 8), 16), ((8, 8, 8, 16), 8)])
def test_both_forms_of_one_layer(dims, Ls, monkeypatch):
    print("case ptc wgrad forms", dims, Ls, flush=True)
    ch = (1, 8, 8, 1)
    op = dwf_amd.AFopr_Domainwall_5din_eo(dims, Ls, 0.05, 1.6, 1.0, 0.0, (1, 1, 1, -1), "float")
    op.set_config(np.tile(lattice.random_gauge((2, 2, 2, 2), 0.4, 41),
                          (1, lattice.volume(dims) // 16, 1)))
    net = ParallelTransportNet(op, ch)
    net.set_weights((0.2 * np.random.default_rng(42).standard_normal(net.nw)).astype(np.float32))
    b, x = op.new_field(), op.new_field()
    op.convert(b, lattice.random_spinor5(dims, Ls, 43))
    op.convert(x, 1e6 * lattice.random_spinor5(dims, Ls, 44))
    grads = []
    for kernel in ("", "valu-wgrad"):
        monkeypatch.setenv("DWF_PTC_KERNEL", kernel)
        grads.append(net.loss_grad([b], [x])[1])
    n1, n2 = 11 * 8 * 32, 11 * 64 * 32
    first, middle, last = ([g[s] for g in grads] for s in
                           (slice(0, n1), slice(n1, n1 + n2), slice(n1 + n2, None)))
    assert np.array_equal(*first) and np.array_equal(*last)
    d = (middle[0] - middle[1]) / np.sqrt(np.mean(middle[1] ** 2))
    assert d.any()
    print("  difference", np.sqrt(np.mean(d ** 2)), "mean", d[0::2].mean(), d[1::2].mean())
    assert np.sqrt(np.mean(d ** 2)) < 5e-7
    assert abs(d[0::2].mean()) < 3e-8 and abs(d[1::2].mean()) < 3e-8
